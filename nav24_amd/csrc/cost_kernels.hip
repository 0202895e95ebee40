// cost_kernels.hip — differentiable robust reprojection cost (include/nav_ba_cost.h).
//
// Hand-written adjoint of C = sum rho(|z - pi_d(T X)|^2) for a batch of
// problems sharing one pinhole + radial-tangential camera.  The observation
// structure is uploaded once (point-major order, tiles of whole points that
// never span two problems, camera-major index lists); each evaluation runs
//   k_cg_obs    one lane per observation: cost term and its adjoint; the
//               point gradient is summed per point from LDS in fixed order,
//               cost and intrinsic gradients per tile, and the pose gradient
//               term of each observation goes to a buffer;
//   k_cg_cam    one workgroup per camera: its observations' pose terms in
//               camera-major order (fixed order);
//   k_cg_final  per-problem costs and the intrinsic gradient over the tiles.
// The forward (cost only) skips the adjoint and the second kernel.
// T = double or float: the projection and residual are FP64 either way, the
// adjoint runs in T; tile partials and the final sums are FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/nav_ba_cost.h"
#include "ba_device.hpp"

namespace navcost {

using navba::block_sum;
using navba::kWave;
using navba::wave_sum;

constexpr int kTileObs = 256;  // observations per tile (whole points; one larger point has a tile of its own)
constexpr int kThreads = 256;
constexpr int kPoseThreads = 64;  // one pose per thread: a wave per workgroup spreads few poses over the CUs

struct CostProblem {
    int n_obs, n_tiles, n_cam, n_pt, n_prob;
    int robust;
    double delta;
    const int* o_cam;      // point-major, caller (global) camera index
    const int* o_pt;       // point-major, caller (global) point index
    const double* uv_d;    // 2 per observation (FP64 for both compute types: the residual is FP64)
    const int* pt_list;    // unique points with observations, ascending
    const int* pt_ptr;     // [n_pts_used + 1]
    const int* tile_obs;   // [n_tiles + 1]
    const int* tile_pt;    // [n_tiles + 1] range in pt_list
    const int* tile_prob;  // [n_tiles]
    const int* prob_tile0; // [n_prob + 1]
    const int* cam_ptr;    // [n_cam + 1] camera-major lists
    const int* cam_obs;    // positions in point-major order
};

template <typename T>
struct ObsGrad {
    double cost;  // the robust term, from the FP64 residual
    T gX[3];
    T gpose[6];
    T gintr[8];
};

template <typename T>
__device__ __forceinline__ T sqrt_t(T v) { return sqrt(v); }

// Cost term of one observation and, if kGrad, its adjoint.  The projection
// and residual are formed in FP64 whatever T is: the residual is a difference
// of two pixel coordinates of a few hundred pixels, and in FP32 that
// cancellation alone left the cost of an FP32 problem 6.6e-4 off its FP64
// value (FP64 issues at the FP32 rate on gfx950 without packed math, so the
// forward costs the same).  The adjoint then runs in T.
template <typename T, bool kGrad>
__device__ __forceinline__ void obs_term(const T* __restrict__ Tcw, const T* __restrict__ X, const T in[8], double u,
                                         double v, int robust, double delta, ObsGrad<T>& g) {
    const double R0 = Tcw[0], R1 = Tcw[1], R2 = Tcw[2], R3 = Tcw[3], R4 = Tcw[4], R5 = Tcw[5];
    const double R6 = Tcw[6], R7 = Tcw[7], R8 = Tcw[8];
    const double x0 = X[0], x1 = X[1], x2 = X[2];
    const double Xc0 = R0 * x0 + R1 * x1 + R2 * x2 + (double)Tcw[9];
    const double Xc1 = R3 * x0 + R4 * x1 + R5 * x2 + (double)Tcw[10];
    const double Xc2 = R6 * x0 + R7 * x1 + R8 * x2 + (double)Tcw[11];
    const double iz = 1.0 / Xc2;
    const double x = Xc0 * iz, y = Xc1 * iz;
    const double fx = in[0], fy = in[1], cx = in[2], cy = in[3], k1 = in[4], k2 = in[5], p1 = in[6], p2 = in[7];
    const double r2 = x * x + y * y;
    const double rad = 1.0 + k1 * r2 + k2 * r2 * r2;
    const double xy = x * y;
    const double xd = x * rad + 2.0 * p1 * xy + p2 * (r2 + 2.0 * x * x);
    const double yd = y * rad + p1 * (r2 + 2.0 * y * y) + 2.0 * p2 * xy;
    const double e0 = u - (fx * xd + cx);
    const double e1 = v - (fy * yd + cy);
    const double s = e0 * e0 + e1 * e1;
    double w;
    const double d2 = delta * delta;
    if (!robust || s <= d2) {
        g.cost = s;
        w = 1.0;
    } else {
        const double r = sqrt(s);
        g.cost = 2.0 * delta * r - d2;
        w = delta / r;
    }
    if (!kGrad) return;
    // the adjoint in T from the FP64 forward values
    const T tx = (T)x, ty = (T)y, tr2 = (T)r2, trad = (T)rad, txy = (T)xy, tiz = (T)iz;
    const T tk1 = in[4], tk2 = in[5], tp1 = in[6], tp2 = in[7], tfx = in[0], tfy = in[1];
    const T gpu = (T)(-2.0 * w * e0), gpv = (T)(-2.0 * w * e1);  // d C / d (projected u, v)
    g.gintr[0] = gpu * (T)xd;
    g.gintr[1] = gpv * (T)yd;
    g.gintr[2] = gpu;
    g.gintr[3] = gpv;
    const T gxd = gpu * tfx, gyd = gpv * tfy;
    g.gintr[4] = (gxd * tx + gyd * ty) * tr2;
    g.gintr[5] = (gxd * tx + gyd * ty) * tr2 * tr2;
    g.gintr[6] = gxd * T(2) * txy + gyd * (tr2 + T(2) * ty * ty);
    g.gintr[7] = gxd * (tr2 + T(2) * tx * tx) + gyd * T(2) * txy;
    const T kr = tk1 + T(2) * tk2 * tr2;
    const T dxdx = trad + T(2) * tx * tx * kr + T(2) * tp1 * ty + T(6) * tp2 * tx;
    const T dxdy = T(2) * txy * kr + T(2) * tp1 * tx + T(2) * tp2 * ty;
    const T dydx = dxdy;
    const T dydy = trad + T(2) * ty * ty * kr + T(6) * tp1 * ty + T(2) * tp2 * tx;
    const T gx = gxd * dxdx + gyd * dydx;
    const T gy = gxd * dxdy + gyd * dydy;
    const T gc0 = gx * tiz, gc1 = gy * tiz, gc2 = -(gx * tx + gy * ty) * tiz;  // d C / d Xc
    // world point: R^T gc
    g.gX[0] = Tcw[0] * gc0 + Tcw[3] * gc1 + Tcw[6] * gc2;
    g.gX[1] = Tcw[1] * gc0 + Tcw[4] * gc1 + Tcw[7] * gc2;
    g.gX[2] = Tcw[2] * gc0 + Tcw[5] * gc1 + Tcw[8] * gc2;
    // pose, left perturbation: d Xc / d omega = -[Xc]x, d Xc / d upsilon = I
    const T tc0 = (T)Xc0, tc1 = (T)Xc1, tc2 = (T)Xc2;
    g.gpose[0] = tc1 * gc2 - tc2 * gc1;
    g.gpose[1] = tc2 * gc0 - tc0 * gc2;
    g.gpose[2] = tc0 * gc1 - tc1 * gc0;
    g.gpose[3] = gc0;
    g.gpose[4] = gc1;
    g.gpose[5] = gc2;
}

// One workgroup per tile.  part[t] = {cost, d/d intrinsics (8)} of the tile (FP64).
template <typename T, bool kGrad>
__global__ __launch_bounds__(kThreads) void k_cg_obs(CostProblem P, const T* __restrict__ Tcw,
                                                     const T* __restrict__ X, const T* __restrict__ intr,
                                                     T* __restrict__ gpo, T* __restrict__ gX,
                                                     double* __restrict__ part) {
    __shared__ T sh[3][kTileObs];
    __shared__ double red[kThreads / kWave];
    __shared__ T redp[kThreads / kWave][3];
    const int t = blockIdx.x;
    const int o0 = P.tile_obs[t], o1 = P.tile_obs[t + 1];
    const int q0 = P.tile_pt[t], q1 = P.tile_pt[t + 1];
    T in[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) in[k] = intr[k];
    double cost = 0.0, gi[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    T gp[3] = {T(0), T(0), T(0)};
    for (int a = o0 + (int)threadIdx.x; a < o1; a += kThreads) {
        const int c = P.o_cam[a], q = P.o_pt[a];
        const double* uv = P.uv_d + 2 * (size_t)a;
        ObsGrad<T> g;
        obs_term<T, kGrad>(Tcw + 12 * (size_t)c, X + 3 * (size_t)q, in, uv[0], uv[1], P.robust, P.delta, g);
        cost += g.cost;
        if (kGrad) {
#pragma unroll
            for (int k = 0; k < 8; ++k) gi[k] += (double)g.gintr[k];
#pragma unroll
            for (int k = 0; k < 6; ++k) gpo[6 * (size_t)a + k] = g.gpose[k];
            gp[0] += g.gX[0]; gp[1] += g.gX[1]; gp[2] += g.gX[2];
        }
    }
    if (kGrad && gX) {  // uniform: gX is a kernel argument
        if (o1 - o0 <= kTileObs) {
            // one observation per lane: per-point sums in fixed order from LDS
            sh[0][threadIdx.x] = gp[0]; sh[1][threadIdx.x] = gp[1]; sh[2][threadIdx.x] = gp[2];
            __syncthreads();
            for (int i = q0 + (int)threadIdx.x; i < q1; i += kThreads) {
                T s0 = T(0), s1 = T(0), s2 = T(0);
                for (int a = P.pt_ptr[i]; a < P.pt_ptr[i + 1]; ++a) {
                    s0 += sh[0][a - o0]; s1 += sh[1][a - o0]; s2 += sh[2][a - o0];
                }
                const int q = P.pt_list[i];
                gX[3 * (size_t)q] = s0; gX[3 * (size_t)q + 1] = s1; gX[3 * (size_t)q + 2] = s2;
            }
        } else {
            // one point with more than kTileObs observations
            const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const T v = wave_sum(gp[k]);
                if (lane == 0) redp[wid][k] = v;
            }
            __syncthreads();
            if (threadIdx.x < 3) {
                T s = T(0);
                for (int i = 0; i < kThreads / kWave; ++i) s += redp[i][threadIdx.x];
                gX[3 * (size_t)P.pt_list[q0] + threadIdx.x] = s;
            }
        }
    }
    const double cs = block_sum<double, kThreads>(cost, red);
    if (threadIdx.x == 0) part[9 * (size_t)t] = cs;
    if (kGrad) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            __syncthreads();
            const double v = block_sum<double, kThreads>(gi[k], red);
            if (threadIdx.x == 0) part[9 * (size_t)t + 1 + k] = v;
        }
    }
}

// One workgroup per camera: d C / d xi in fixed order over its observations.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_cg_cam(CostProblem P, const T* __restrict__ gpo, T* __restrict__ gpose) {
    __shared__ double red[kThreads / kWave];
    const int c = blockIdx.x;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    for (int k = P.cam_ptr[c] + (int)threadIdx.x; k < P.cam_ptr[c + 1]; k += kThreads) {
        const int a = P.cam_obs[k];
#pragma unroll
        for (int j = 0; j < 6; ++j) acc[j] += (double)gpo[6 * (size_t)a + j];
    }
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        __syncthreads();
        const double v = block_sum<double, kThreads>(acc[j], red);
        if (threadIdx.x == 0) gpose[6 * (size_t)c + j] = (T)v;
    }
}

// Workgroup p < n_prob: cost of problem p over its tiles; workgroup n_prob:
// the total cost and the intrinsic gradient over all tiles (fixed order).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_cg_final(CostProblem P, const double* __restrict__ part, int grad,
                                                       T* __restrict__ cost, T* __restrict__ total,
                                                       T* __restrict__ gintr) {
    __shared__ double red[kThreads / kWave];
    const int pr = blockIdx.x;
    if (pr < P.n_prob) {
        double s = 0.0;
        for (int t = P.prob_tile0[pr] + (int)threadIdx.x; t < P.prob_tile0[pr + 1]; t += kThreads)
            s += part[9 * (size_t)t];
        const double v = block_sum<double, kThreads>(s, red);
        if (threadIdx.x == 0) cost[pr] = (T)v;
        return;
    }
    if (total) {
        double s = 0.0;
        for (int t = threadIdx.x; t < P.n_tiles; t += kThreads) s += part[9 * (size_t)t];
        const double v = block_sum<double, kThreads>(s, red);
        if (threadIdx.x == 0) *total = (T)v;
    }
    if (!grad || !gintr) return;
    for (int k = 0; k < 8; ++k) {
        double s = 0.0;
        for (int t = threadIdx.x; t < P.n_tiles; t += kThreads) s += part[9 * (size_t)t + 1 + k];
        const double v = block_sum<double, kThreads>(s, red);
        if (threadIdx.x == 0) gintr[k] = (T)v;
    }
}

// ---- pose tangents ----------------------------------------------------------
// Coefficients of exp on SE3 at th2 = |omega|^2 and their derivatives:
//   a = sin t / t, b = (1 - cos t) / t^2, c = (t - sin t) / t^3,
//   db = b'(t) / t = (a - 2 b) / t^2,  dc = c'(t) / t = (b - 3 c) / t^2.
// Below th2 = 0.25 their Taylor series (seven terms, truncation below 1e-17):
// the closed forms cancel there.  FP64 for both compute types.
struct ExpCoef { double a, b, c, db, dc; };

__device__ __forceinline__ ExpCoef exp_coef(double t2) {
    ExpCoef k;
    if (t2 < 0.25) {
        // sum_j (-t2)^j / (2j + s)!, s = 1, 2, 3; and the two derivatives,
        // sum_j (-1)^(j+1) 2 (j + 1) t2^j / (2j + 2 + s)!, s = 2, 3
        k.a = 1.0 + t2 * (-1.0 / 6 + t2 * (1.0 / 120 + t2 * (-1.0 / 5040 + t2 * (1.0 / 362880 + t2 * (-1.0 / 39916800 + t2 * (1.0 / 6227020800.0))))));
        k.b = 0.5 + t2 * (-1.0 / 24 + t2 * (1.0 / 720 + t2 * (-1.0 / 40320 + t2 * (1.0 / 3628800 + t2 * (-1.0 / 479001600 + t2 * (1.0 / 87178291200.0))))));
        k.c = 1.0 / 6 + t2 * (-1.0 / 120 + t2 * (1.0 / 5040 + t2 * (-1.0 / 362880 + t2 * (1.0 / 39916800 + t2 * (-1.0 / 6227020800.0 + t2 * (1.0 / 1307674368000.0))))));
        k.db = -2.0 / 24 + t2 * (4.0 / 720 + t2 * (-6.0 / 40320 + t2 * (8.0 / 3628800 + t2 * (-10.0 / 479001600 + t2 * (12.0 / 87178291200.0 + t2 * (-14.0 / 20922789888000.0))))));
        k.dc = -2.0 / 120 + t2 * (4.0 / 5040 + t2 * (-6.0 / 362880 + t2 * (8.0 / 39916800 + t2 * (-10.0 / 6227020800.0 + t2 * (12.0 / 1307674368000.0 + t2 * (-14.0 / 355687428096000.0))))));
    } else {
        const double t = sqrt(t2), s = sin(t), co = cos(t);
        k.a = s / t;
        k.b = (1.0 - co) / t2;
        k.c = (t - s) / (t2 * t);
        k.db = (k.a - 2.0 * k.b) / t2;
        k.dc = (k.b - 3.0 * k.c) / t2;
    }
    return k;
}

__device__ __forceinline__ void cross3(const double x[3], const double y[3], double r[3]) {
    r[0] = x[1] * y[2] - x[2] * y[1];
    r[1] = x[2] * y[0] - x[0] * y[2];
    r[2] = x[0] * y[1] - x[1] * y[0];
}

__device__ __forceinline__ double dot3(const double x[3], const double y[3]) {
    return x[0] * y[0] + x[1] * y[1] + x[2] * y[2];
}

// v + p (w x v) + q (w x (w x v)): exp's rotation with (a, b), its V matrix
// (the left Jacobian of SO3) with (b, c), V's transpose with (-b, c).
__device__ __forceinline__ void rot3(const double w[3], double p, double q, const double v[3], double r[3]) {
    double wv[3], wwv[3];
    cross3(w, v, wv);
    cross3(w, wv, wwv);
#pragma unroll
    for (int i = 0; i < 3; ++i) r[i] = v[i] + p * wv[i] + q * wwv[i];
}

// T = exp(xi) T_cw, one pose per thread.  Launch bound: a few hundred
// operations and at most 144 bytes per pose.  As torch operations the map and
// its derivative were about 230 launches of a gradient step; with these two
// kernels a step of BACost takes 260 us instead of 1970 on 64 scenes of
// 5 000 points (1 280 poses, float) and 168 instead of 1800 on one of 700
// (double).
template <typename T>
__global__ void k_se3_left(int n, const T* __restrict__ xi, const T* __restrict__ Tcw, T* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    double w[3], u[3], t[3], col[3], r[3], v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        w[i] = (double)xi[6 * (size_t)c + i];
        u[i] = (double)xi[6 * (size_t)c + 3 + i];
        t[i] = (double)Tcw[12 * (size_t)c + 9 + i];
    }
    const ExpCoef k = exp_coef(dot3(w, w));
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int i = 0; i < 3; ++i) col[i] = (double)Tcw[12 * (size_t)c + 3 * i + j];
        rot3(w, k.a, k.b, col, r);
#pragma unroll
        for (int i = 0; i < 3; ++i) out[12 * (size_t)c + 3 * i + j] = (T)r[i];
    }
    rot3(w, k.a, k.b, t, r);
    rot3(w, k.b, k.c, u, v);
#pragma unroll
    for (int i = 0; i < 3; ++i) out[12 * (size_t)c + 9 + i] = (T)(r[i] + v[i]);
}

// g_xi = J_l(xi)^T g.  With p = V u, a step d of omega turns T by J d (J = V)
// and moves its translation, seen from the left, by (dV) u - (J d) x p, so
//   g_upsilon -> V^T g_u
//   g_omega   -> V^T (g_w - p x g_u) + grad_omega (g_u . V u),
// the last term from V u = u + b w x u + c (w (w.u) - |w|^2 u).
template <typename T>
__global__ void k_tangent_grad(int n, const T* __restrict__ xi, const T* __restrict__ g, T* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    double w[3], u[3], gw[3], gu[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        w[i] = (double)xi[6 * (size_t)c + i];
        u[i] = (double)xi[6 * (size_t)c + 3 + i];
        gw[i] = (double)g[6 * (size_t)c + i];
        gu[i] = (double)g[6 * (size_t)c + 3 + i];
    }
    const double t2 = dot3(w, w);
    const ExpCoef k = exp_coef(t2);
    double p[3], pg[3], ug[3], a[3], ru[3], rw[3];
    rot3(w, k.b, k.c, u, p);
    cross3(p, gu, pg);
    cross3(u, gu, ug);
#pragma unroll
    for (int i = 0; i < 3; ++i) a[i] = gw[i] - pg[i];
    rot3(w, -k.b, k.c, a, rw);
    rot3(w, -k.b, k.c, gu, ru);
    const double wug = dot3(w, ug), wu = dot3(w, u), gw0 = dot3(gu, w), gu0 = dot3(gu, u);
    const double s = k.db * wug + k.dc * (gw0 * wu - t2 * gu0) - 2.0 * k.c * gu0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        out[6 * (size_t)c + i] = (T)(rw[i] + k.b * ug[i] + k.c * (gu[i] * wu + u[i] * gw0) + s * w[i]);
        out[6 * (size_t)c + 3 + i] = (T)ru[i];
    }
}

template <typename T>
__global__ void k_zero(T* p, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = T(0);
}

}  // namespace navcost

using namespace navcost;

struct nav_ba_cost_handle {
    int device = 0;
    std::string err;
    bool prepared = false;
    CostProblem P{};
    std::vector<void*> bufs;
    void* gpo = nullptr;
    size_t gpo_bytes = 0;
    double* part = nullptr;
};

namespace {

void free_all(nav_ba_cost_handle* h) {
    for (void* p : h->bufs) (void)hipFree(p);
    h->bufs.clear();
    if (h->gpo) (void)hipFree(h->gpo);
    h->gpo = nullptr;
    h->gpo_bytes = 0;
    h->part = nullptr;
}

template <class V>
int up(nav_ba_cost_handle* h, const V& v, const typename V::value_type** out) {
    void* p = nullptr;
    const size_t bytes = std::max<size_t>(sizeof(typename V::value_type) * v.size(), 256);
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) { h->err = std::string("hipMalloc: ") + hipGetErrorString(e); return NAV_BA_HIP_ERROR; }
    h->bufs.push_back(p);
    if (!v.empty() && hipMemcpy(p, v.data(), sizeof(typename V::value_type) * v.size(), hipMemcpyHostToDevice) != hipSuccess) {
        h->err = "hipMemcpy failed";
        return NAV_BA_HIP_ERROR;
    }
    *out = (const typename V::value_type*)p;
    return NAV_BA_OK;
}

int32_t launch_status(nav_ba_cost_handle* h) {
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) return NAV_BA_OK;
    h->err = std::string("launch: ") + hipGetErrorString(e);
    return NAV_BA_HIP_ERROR;
}

template <typename T>
int32_t eval_t(nav_ba_cost_handle* h, const T* Tcw, const T* X, const T* intr, T* total, T* cost, T* gpose, T* gX,
               T* gintr, hipStream_t s) {
    const CostProblem& P = h->P;
    const bool grad = gpose || gX || gintr;
    T* gpo = (T*)h->gpo;
    if (grad && gX) hipLaunchKernelGGL(k_zero<T>, dim3(256), dim3(256), 0, s, gX, (size_t)3 * P.n_pt);
    if (P.n_tiles > 0) {
        if (grad)  // gX may be null: the per-point sums are then skipped
            hipLaunchKernelGGL((k_cg_obs<T, true>), dim3(P.n_tiles), dim3(kThreads), 0, s, P, Tcw, X, intr, gpo, gX,
                               h->part);
        else
            hipLaunchKernelGGL((k_cg_obs<T, false>), dim3(P.n_tiles), dim3(kThreads), 0, s, P, Tcw, X, intr,
                               (T*)nullptr, (T*)nullptr, h->part);
    }
    if (grad && gpose && P.n_cam > 0)
        hipLaunchKernelGGL(k_cg_cam<T>, dim3(P.n_cam), dim3(kThreads), 0, s, P, (const T*)gpo, gpose);
    hipLaunchKernelGGL(k_cg_final<T>, dim3(P.n_prob + 1), dim3(kThreads), 0, s, P, (const double*)h->part,
                       grad ? 1 : 0, cost, total, gintr);
    return launch_status(h);
}

// T = exp(xi) T_cw, then the evaluation there.
template <typename T>
int32_t eval_tangent_t(nav_ba_cost_handle* h, const T* xi, const T* Tcw, const T* X, const T* intr, T* Tout, T* total,
                       T* cost, T* gpose, T* gX, T* gintr, hipStream_t s) {
    const int n = h->P.n_cam;
    if (n > 0)
        hipLaunchKernelGGL(k_se3_left<T>, dim3((n + kPoseThreads - 1) / kPoseThreads), dim3(kPoseThreads), 0, s, n, xi,
                           Tcw, Tout);
    return eval_t<T>(h, Tout, X, intr, total, cost, gpose, gX, gintr, s);
}

template <typename T>
int32_t tangent_grad_t(int n, const T* xi, const T* g, T* out, hipStream_t s) {
    hipLaunchKernelGGL(k_tangent_grad<T>, dim3((n + kPoseThreads - 1) / kPoseThreads), dim3(kPoseThreads), 0, s, n, xi, g,
                       out);
    return hipGetLastError() == hipSuccess ? NAV_BA_OK : NAV_BA_HIP_ERROR;
}

}  // namespace

extern "C" {

int32_t nav_ba_cost_create(nav_ba_cost_handle** out, int32_t device) {
    if (!out) return NAV_BA_BAD_ARG;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || device < 0 || device >= n) return NAV_BA_NO_DEVICE;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return NAV_BA_NO_DEVICE;
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return NAV_BA_NO_DEVICE;
    nav_ba_cost_handle* h = new nav_ba_cost_handle();
    h->device = device;
    *out = h;
    return NAV_BA_OK;
}

void nav_ba_cost_destroy(nav_ba_cost_handle* h) {
    if (!h) return;
    (void)hipSetDevice(h->device);
    (void)hipDeviceSynchronize();
    free_all(h);
    delete h;
}

const char* nav_ba_cost_last_error(const nav_ba_cost_handle* h) { return h ? h->err.c_str() : "null handle"; }

int32_t nav_ba_cost_prepare(nav_ba_cost_handle* h, const nav_ba_problem* probs, int32_t n_probs, int32_t robust,
                            double huber_delta) {
    if (!h) return NAV_BA_BAD_ARG;
    h->err.clear();
    h->prepared = false;
    if (!probs || n_probs <= 0) { h->err = "no problems"; return NAV_BA_BAD_ARG; }
    if (hipSetDevice(h->device) != hipSuccess) { h->err = "hipSetDevice"; return NAV_BA_HIP_ERROR; }
    (void)hipDeviceSynchronize();
    free_all(h);
    std::vector<int> cam_off(n_probs + 1, 0), pt_off(n_probs + 1, 0);
    size_t no = 0;
    for (int p = 0; p < n_probs; ++p) {
        const nav_ba_problem& q = probs[p];
        if (q.n_cam < 0 || q.n_pt < 0 || q.n_obs < 0 || (q.n_obs > 0 && (!q.obs_cam || !q.obs_pt || !q.obs_uv))) {
            h->err = "invalid problem " + std::to_string(p);
            return NAV_BA_BAD_ARG;
        }
        for (int i = 0; i < q.n_obs; ++i)
            if (q.obs_cam[i] < 0 || q.obs_cam[i] >= q.n_cam || q.obs_pt[i] < 0 || q.obs_pt[i] >= q.n_pt) {
                h->err = "observation index out of range in problem " + std::to_string(p);
                return NAV_BA_BAD_ARG;
            }
        cam_off[p + 1] = cam_off[p] + q.n_cam;
        pt_off[p + 1] = pt_off[p] + q.n_pt;
        no += (size_t)q.n_obs;
    }
    if (no > (size_t)0x7fffffff) { h->err = "too many observations"; return NAV_BA_TOO_LARGE; }
    const int nc = cam_off[n_probs], np = pt_off[n_probs];
    std::vector<int> gcam(no), gpt(no);
    std::vector<double> guv(2 * no);
    {
        size_t k = 0;
        for (int p = 0; p < n_probs; ++p)
            for (int i = 0; i < probs[p].n_obs; ++i, ++k) {
                gcam[k] = cam_off[p] + probs[p].obs_cam[i];
                gpt[k] = pt_off[p] + probs[p].obs_pt[i];
                guv[2 * k] = probs[p].obs_uv[2 * (size_t)i];
                guv[2 * k + 1] = probs[p].obs_uv[2 * (size_t)i + 1];
            }
    }
    // point-major order (point, camera, input order): two stable counting sorts
    std::vector<int> byc(no), ord(no);
    {
        std::vector<int> off(nc + 1, 0);
        for (size_t i = 0; i < no; ++i) off[gcam[i] + 1]++;
        for (int c = 0; c < nc; ++c) off[c + 1] += off[c];
        for (size_t i = 0; i < no; ++i) byc[off[gcam[i]]++] = (int)i;
        std::vector<int> poff(np + 1, 0);
        for (size_t i = 0; i < no; ++i) poff[gpt[i] + 1]++;
        for (int q = 0; q < np; ++q) poff[q + 1] += poff[q];
        for (size_t k = 0; k < no; ++k) { const int i = byc[k]; ord[poff[gpt[i]]++] = i; }
    }
    std::vector<int> o_cam(no), o_pt(no);
    std::vector<double> uv_d(2 * no);
    for (size_t k = 0; k < no; ++k) {
        const int i = ord[k];
        o_cam[k] = gcam[i]; o_pt[k] = gpt[i];
        uv_d[2 * k] = guv[2 * (size_t)i]; uv_d[2 * k + 1] = guv[2 * (size_t)i + 1];
    }
    // unique points, tiles of whole points per problem
    std::vector<int> pt_list, pt_ptr{0}, tile_obs{0}, tile_pt{0}, tile_prob, prob_tile0{0};
    {
        size_t k = 0;
        for (int p = 0; p < n_probs; ++p) {  // a problem's points, hence observations, are contiguous
            while (k < no && o_pt[k] < pt_off[p + 1]) {
                const int q = o_pt[k];
                size_t e = k;
                while (e < no && o_pt[e] == q) ++e;
                pt_list.push_back(q);
                pt_ptr.push_back((int)e);
                k = e;
            }
        }
        int i = 0;
        const int nu = (int)pt_list.size();
        for (int p = 0; p < n_probs; ++p) {
            while (i < nu && pt_list[i] < pt_off[p + 1]) {
                int j = i;
                while (j < nu && pt_list[j] < pt_off[p + 1] && pt_ptr[j + 1] - pt_ptr[i] <= kTileObs) ++j;
                if (j == i) j = i + 1;
                tile_obs.push_back(pt_ptr[j]);
                tile_pt.push_back(j);
                tile_prob.push_back(p);
                i = j;
            }
            prob_tile0.push_back((int)tile_prob.size());
        }
    }
    std::vector<int> cam_ptr(nc + 1, 0), cam_obs(no);
    for (size_t k = 0; k < no; ++k) cam_ptr[o_cam[k] + 1]++;
    for (int c = 0; c < nc; ++c) cam_ptr[c + 1] += cam_ptr[c];
    {
        std::vector<int> pos(cam_ptr.begin(), cam_ptr.end() - 1);
        for (size_t k = 0; k < no; ++k) cam_obs[pos[o_cam[k]]++] = (int)k;
    }
    CostProblem& P = h->P;
    P = CostProblem{};
    P.n_obs = (int)no; P.n_tiles = (int)tile_prob.size(); P.n_cam = nc; P.n_pt = np; P.n_prob = n_probs;
    P.robust = robust ? 1 : 0;
    P.delta = huber_delta;
    int st;
    if ((st = up(h, o_cam, &P.o_cam)) || (st = up(h, o_pt, &P.o_pt)) || (st = up(h, uv_d, &P.uv_d)) ||
        (st = up(h, pt_list, &P.pt_list)) || (st = up(h, pt_ptr, &P.pt_ptr)) ||
        (st = up(h, tile_obs, &P.tile_obs)) || (st = up(h, tile_pt, &P.tile_pt)) ||
        (st = up(h, tile_prob, &P.tile_prob)) || (st = up(h, prob_tile0, &P.prob_tile0)) ||
        (st = up(h, cam_ptr, &P.cam_ptr)) || (st = up(h, cam_obs, &P.cam_obs)))
        return st;
    void* part = nullptr;
    if (hipMalloc(&part, sizeof(double) * 9 * std::max<size_t>(tile_prob.size(), 1)) != hipSuccess) {
        h->err = "hipMalloc part";
        return NAV_BA_HIP_ERROR;
    }
    h->bufs.push_back(part);
    h->part = (double*)part;
    h->gpo_bytes = sizeof(double) * 6 * std::max<size_t>(no, 1);
    if (hipMalloc(&h->gpo, h->gpo_bytes) != hipSuccess) { h->err = "hipMalloc gpo"; return NAV_BA_HIP_ERROR; }
    h->prepared = true;
    return NAV_BA_OK;
}

int32_t nav_ba_cost_sizes(const nav_ba_cost_handle* h, int32_t* n_cam, int32_t* n_pt, int32_t* n_obs,
                          int32_t* n_problems) {
    if (!h || !h->prepared) return NAV_BA_NOT_PREPARED;
    if (n_cam) *n_cam = h->P.n_cam;
    if (n_pt) *n_pt = h->P.n_pt;
    if (n_obs) *n_obs = h->P.n_obs;
    if (n_problems) *n_problems = h->P.n_prob;
    return NAV_BA_OK;
}

int32_t nav_ba_cost_eval(nav_ba_cost_handle* h, int32_t dtype, const void* T_cw, const void* X, const void* intr,
                         void* cost, void* g_pose, void* g_X, void* g_intr, void* stream) {
    if (!h) return NAV_BA_BAD_ARG;
    if (!h->prepared) { h->err = "evaluation before nav_ba_cost_prepare"; return NAV_BA_NOT_PREPARED; }
    if (!T_cw || !X || !intr || !cost) { h->err = "null state or cost pointer"; return NAV_BA_BAD_ARG; }
    if (hipSetDevice(h->device) != hipSuccess) { h->err = "hipSetDevice"; return NAV_BA_HIP_ERROR; }
    hipStream_t s = (hipStream_t)stream;
    if (dtype == NAV_BA_COST_F64)
        return eval_t<double>(h, (const double*)T_cw, (const double*)X, (const double*)intr, nullptr, (double*)cost,
                              (double*)g_pose, (double*)g_X, (double*)g_intr, s);
    if (dtype == NAV_BA_COST_F32)
        return eval_t<float>(h, (const float*)T_cw, (const float*)X, (const float*)intr, nullptr, (float*)cost,
                             (float*)g_pose, (float*)g_X, (float*)g_intr, s);
    h->err = "unknown dtype";
    return NAV_BA_BAD_ARG;
}

int32_t nav_ba_cost_eval_tangent(nav_ba_cost_handle* h, int32_t dtype, const void* xi, const void* T_cw,
                                 const void* X, const void* intr, void* T, void* total, void* cost, void* g_pose,
                                 void* g_X, void* g_intr, void* stream) {
    if (!h) return NAV_BA_BAD_ARG;
    if (!h->prepared) { h->err = "evaluation before nav_ba_cost_prepare"; return NAV_BA_NOT_PREPARED; }
    if (!xi || !T_cw || !X || !intr || !T || !total || !cost) {
        h->err = "null state or cost pointer";
        return NAV_BA_BAD_ARG;
    }
    if (hipSetDevice(h->device) != hipSuccess) { h->err = "hipSetDevice"; return NAV_BA_HIP_ERROR; }
    hipStream_t s = (hipStream_t)stream;
    if (dtype == NAV_BA_COST_F64)
        return eval_tangent_t<double>(h, (const double*)xi, (const double*)T_cw, (const double*)X, (const double*)intr,
                                      (double*)T, (double*)total, (double*)cost, (double*)g_pose, (double*)g_X,
                                      (double*)g_intr, s);
    if (dtype == NAV_BA_COST_F32)
        return eval_tangent_t<float>(h, (const float*)xi, (const float*)T_cw, (const float*)X, (const float*)intr,
                                     (float*)T, (float*)total, (float*)cost, (float*)g_pose, (float*)g_X,
                                     (float*)g_intr, s);
    h->err = "unknown dtype";
    return NAV_BA_BAD_ARG;
}

int32_t nav_ba_cost_tangent_grad(int32_t device, int32_t dtype, int32_t n, const void* xi, const void* g_pose,
                                 void* g_xi, void* stream) {
    if (n < 0 || (n > 0 && (!xi || !g_pose || !g_xi)) || (dtype != NAV_BA_COST_F64 && dtype != NAV_BA_COST_F32))
        return NAV_BA_BAD_ARG;
    if (n == 0) return NAV_BA_OK;
    int was = 0;
    if (hipGetDevice(&was) != hipSuccess) return NAV_BA_HIP_ERROR;
    if (was != device && hipSetDevice(device) != hipSuccess) return NAV_BA_HIP_ERROR;
    hipStream_t s = (hipStream_t)stream;
    const int32_t st = dtype == NAV_BA_COST_F64
                           ? tangent_grad_t<double>(n, (const double*)xi, (const double*)g_pose, (double*)g_xi, s)
                           : tangent_grad_t<float>(n, (const float*)xi, (const float*)g_pose, (float*)g_xi, s);
    if (was != device && hipSetDevice(was) != hipSuccess) return NAV_BA_HIP_ERROR;
    return st;
}

}  // extern "C"
