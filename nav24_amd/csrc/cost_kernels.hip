// cost_kernels.hip — differentiable robust reprojection cost (include/nav_ba_cost.h).
//
// Hand-written adjoint of C = sum rho(|z - pi_d(T X)|^2) for a batch of
// problems sharing one pinhole + radial-tangential camera.  The observation
// structure is uploaded once, in two orders: point-major, in tiles of whole
// points and groups of consecutive tiles that never span two problems, and
// camera-major, in chunks of one camera's observations.  Each evaluation runs
//   k_cg_obs    one workgroup per group: cost terms and their adjoint, a lane
//               per observation of a tile; the point gradient is summed per
//               point from LDS in fixed order, the cost per tile, the intrinsic
//               gradients per group; in the same launch one workgroup per camera
//               chunk: its pose gradient, from the terms formed again in
//               camera-major order; and zeros for the points without observations;
//   k_cg_final  per-problem costs and the total over the tiles, the intrinsic
//               gradient over the groups, the pose gradients over the chunks
//               (fixed order).
// The forward (cost only) is k_cg_cost, one workgroup per tile: the same sums per
// tile, so the same costs.
// T = double or float: the projection and residual are FP64 either way, the
// adjoint runs in T; partial and final sums are FP64.
// Forming an observation's terms twice costs less than one pass that writes six
// pose terms per observation (72 MB at 3 M observations, float) for a second one
// to gather.
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

constexpr int kTileObs = 256;  // observations per tile (whole points; one larger point has a tile of its own)
constexpr int kThreads = 256;
// Sums over the workgroup come once per group or chunk, so these are long where
// there are many observations.  Groups are as short as keeps them to kGroups, up to
// kGroupTiles tiles (gradients of 0.8, 1.0 and 3.2 M observations: 26.7, 31.0 and
// 63 us; with at least kGroups of them, 31.8, 37.4 and 64; with twice as many, 31.8,
// 37.1 and 66.5).  Chunks are as long as
// leaves kChunks of them, up to kChunkMax observations.
constexpr int kXcds = 8;
constexpr int kGroups = 2048;
constexpr int kChunks = 1024;
constexpr int kGroupTiles = 8;
constexpr int kChunkMax = 4096;
constexpr int kPoseThreads = 64;  // one pose per thread: a wave per workgroup spreads few poses over the CUs

struct CostProblem {
    int n_obs, n_tiles, n_groups, n_chunks, n_unseen, n_cam, n_pt, n_prob;
    int robust;
    double delta;
    const int* o_cam;      // point-major, caller (global) camera index
    const int* o_pt;       // point-major, caller (global) point index
    const double2* uv;     // point-major (FP64 for both compute types: the residual is FP64)
    const int* pt_list;    // unique points with observations, ascending
    const int* pt_ptr;     // [n_pts_used + 1]
    const int* tile_obs;   // [n_tiles + 1]
    const int* tile_pt;    // [n_tiles + 1] range in pt_list
    const int* group_tile; // [n_groups + 1]
    const int* prob_tile0; // [n_prob + 1]
    const int* c_pt;       // camera-major, caller (global) point index
    const double2* c_uv;   // camera-major
    const int* chunk_cam;  // [n_chunks]
    const int* chunk_ptr;  // [n_chunks + 1] range of camera-major observations
    const int* cam_chunk0; // [n_cam + 1]
    const int* unseen;     // [n_unseen] points without observations
};

template <typename T>
struct ObsGrad {
    double cost;  // the robust term, from the FP64 residual
    T gX[3];
    T gpose[6];
    T gintr[8];
};

// What of an observation's terms a caller wants: the cost, with the gradients
// to point and intrinsics, or the gradient to the pose alone.
enum Want { kCost = 0, kPointSide = 1, kPoseSide = 2 };

// Cost term of one observation and, unless kCost, its adjoint.  The projection
// and residual are formed in FP64 whatever T is: the residual is a difference
// of two pixel coordinates of a few hundred pixels, and in FP32 that
// cancellation alone left the cost of an FP32 problem 6.6e-4 off its FP64
// value (FP64 issues at the FP32 rate on gfx950 without packed math, so the
// forward costs the same).  The adjoint then runs in T.  TP is the type of the
// poses: T where they are the caller's, FP64 where they come from k_se3_left (a
// pose of ~10 m rounded to float is half a micrometre off, which near a camera's
// plane is the whole error of the gradients).
template <typename T, Want kWant, typename TP>
__device__ __forceinline__ void obs_term(const TP* __restrict__ Tcw, const T* __restrict__ X, const T in[8], double u,
                                         double v, int robust, double delta, ObsGrad<T>& g) {
    const double R0 = Tcw[0], R1 = Tcw[1], R2 = Tcw[2], R3 = Tcw[3], R4 = Tcw[4], R5 = Tcw[5];
    const double R6 = Tcw[6], R7 = Tcw[7], R8 = Tcw[8];
    const double x0 = X[0], x1 = X[1], x2 = X[2];
    const double Xc0 = R0 * x0 + R1 * x1 + R2 * x2 + (double)Tcw[9];
    const double Xc1 = R3 * x0 + R4 * x1 + R5 * x2 + (double)Tcw[10];
    const double Xc2 = R6 * x0 + R7 * x1 + R8 * x2 + (double)Tcw[11];
    const double iz = navba::recip<double>(Xc2);  // the division's bits on 40 scenes, 1 % of a gradient faster
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
    if (kWant == kCost) return;
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
    g.gX[0] = (T)R0 * gc0 + (T)R3 * gc1 + (T)R6 * gc2;
    g.gX[1] = (T)R1 * gc0 + (T)R4 * gc1 + (T)R7 * gc2;
    g.gX[2] = (T)R2 * gc0 + (T)R5 * gc1 + (T)R8 * gc2;
    // pose, left perturbation: d Xc / d omega = -[Xc]x, d Xc / d upsilon = I
    const T tc0 = (T)Xc0, tc1 = (T)Xc1, tc2 = (T)Xc2;
    g.gpose[0] = tc1 * gc2 - tc2 * gc1;
    g.gpose[1] = tc2 * gc0 - tc0 * gc2;
    g.gpose[2] = tc0 * gc1 - tc1 * gc0;
    g.gpose[3] = gc0;
    g.gpose[4] = gc1;
    g.gpose[5] = gc2;
}

typedef double dbl4 __attribute__((ext_vector_type(4)));

// Sum over the two (four) lanes that differ in bit 4 (and 5) of their index, in each of them.
__device__ __forceinline__ double sum_quarters(double v) {
    const long long b = __double_as_longlong(v);
    const auto l1 = __builtin_amdgcn_permlane16_swap((unsigned)b, (unsigned)b, false, false);
    const auto h1 = __builtin_amdgcn_permlane16_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    const double s = __longlong_as_double(((long long)h1[0] << 32) | l1[0]) +
                     __longlong_as_double(((long long)h1[1] << 32) | l1[1]);
    const long long c = __double_as_longlong(s);
    const auto l2 = __builtin_amdgcn_permlane32_swap((unsigned)c, (unsigned)c, false, false);
    const auto h2 = __builtin_amdgcn_permlane32_swap((unsigned)(c >> 32), (unsigned)(c >> 32), false, false);
    return __longlong_as_double(((long long)h2[0] << 32) | l2[0]) +
           __longlong_as_double(((long long)h2[1] << 32) | l2[1]);
}

// Sum of a value per lane over the wave, in every lane: a matrix instruction with
// a second operand of ones (16 row sums of four lanes each, four to a lane), then
// within lanes and over the lanes' quarters, half the instructions of a sum by
// lane moves.
__device__ __forceinline__ double wave_total(double v) {
    const dbl4 r = __builtin_amdgcn_mfma_f64_16x16x4f64(v, 1.0, dbl4{0.0, 0.0, 0.0, 0.0}, 0, 0, 0);
    return sum_quarters((r[0] + r[1]) + (r[2] + r[3]));
}

// Sums of N values per lane over the workgroup, in a fixed order: value q in
// thread q < N.
template <int N>
__device__ __forceinline__ double block_sums(const double v[N], double (*red)[N]) {
    const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const double s = wave_total(v[q]);
        if (lane == 0) red[wid][q] = s;
    }
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x < N)
        for (int i = 0; i < kThreads / kWave; ++i) s += red[i][threadIdx.x];
    return s;
}

// Item of workgroup b of n: workgroups b = x (mod kXcds) run on one XCD and take
// consecutive items, so the points and poses that these share stay in its L2.
__device__ __forceinline__ int xcd_band(int b, int n) {
    const int x = b % kXcds, lo = n / kXcds, more = n % kXcds;
    return x * lo + min(x, more) + b / kXcds;
}

// A tile's cost from its lanes' in LDS, by one wave; both kernels form it so.
__device__ __forceinline__ double tile_total(const double c[kThreads]) {
    static_assert(kThreads == 4 * kWave, "four values a lane");
    const int l = threadIdx.x % kWave;
    return wave_total((c[l] + c[l + kWave]) + (c[l + 2 * kWave] + c[l + 3 * kWave]));
}

// The cost alone: one workgroup per tile, its cost to tile_cost; eight workgroups
// per CU.  Bound by memory and the FP64 operations of the terms.  64 scenes of
// 5 000 points (3.16 M observations), with the final sums: 25.2 us in FP64 and 21.3
// in FP32; one workgroup per group of tiles 28.5 and 25.2, and without the bound on
// registers 25.4 and 23.8.
template <typename T, typename TP>
__global__ __launch_bounds__(kThreads, 8) void k_cg_cost(CostProblem P, const TP* __restrict__ Tcw,
                                                      const T* __restrict__ X, const T* __restrict__ intr,
                                                      double* __restrict__ tile_cost) {
    __shared__ double lane_cost[kThreads];
    const int tid = threadIdx.x, t = xcd_band(blockIdx.x, P.n_tiles);
    T in[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) in[k] = intr[k];
    const int o1 = P.tile_obs[t + 1];
    double cost = 0.0;
    for (int a = P.tile_obs[t] + tid; a < o1; a += kThreads) {
        const double2 uv = P.uv[a];
        ObsGrad<T> g;
        obs_term<T, kCost>(Tcw + 12 * (size_t)P.o_cam[a], X + 3 * (size_t)P.o_pt[a], in, uv.x, uv.y, P.robust, P.delta, g);
        cost += g.cost;
    }
    lane_cost[tid] = cost;
    __syncthreads();
    if (tid >= kWave) return;
    const double s = tile_total(lane_cost);
    if (tid == 0) tile_cost[t] = s;
}

// Workgroups 0 .. n_groups - 1: the tiles' costs to tile_cost, part[q n_groups +
// group] = d / d intrinsics[q] (FP64); the next n_chunks (if gpart): gpart[6 chunk
// + j]; then those that clear the unseen points' gradients.  Bound by the FP64
// operations of the terms and by memory together: 24 bytes per observation in one
// order and 20 in the other.  64 scenes of 5 000 points, with the final sums: 67 us
// in FP64 and 63 in FP32 (68 at FP64 poses), before 220 and 191 (a gather of six
// stored pose terms per observation, and one workgroup's sums over all tiles).
template <typename T, typename TP>
__global__ __launch_bounds__(kThreads, 4) void k_cg_obs(CostProblem P, const TP* __restrict__ Tcw,
                                                        const T* __restrict__ X, const T* __restrict__ intr,
                                                        T* __restrict__ gX, double* __restrict__ tile_cost,
                                                        double* __restrict__ part, double* __restrict__ gpart) {
    __shared__ T sh[2][3][kTileObs];
    __shared__ double lane_cost[kGroupTiles][kThreads];
    __shared__ double red[kThreads / kWave][8];
    __shared__ double redc[kThreads / kWave][6];
    const int tid = threadIdx.x;
    T in[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) in[k] = intr[k];
    int b = blockIdx.x;
    if (b < P.n_groups) {
        b = xcd_band(b, P.n_groups);
        double acc[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] = 0.0;
        const int t0 = P.group_tile[b], t1 = P.group_tile[b + 1];
        int o0 = P.tile_obs[t0], c = 0, q = 0;
        double2 uv;
        // the lane's first observation of tile t, loaded while the tile before is worked on
        auto load = [&](int a, int o1) {
            if (a < o1) {
                c = P.o_cam[a];
                q = P.o_pt[a];
                uv = P.uv[a];
            }
        };
        load(o0 + tid, P.tile_obs[t0 + 1]);
        for (int t = t0; t < t1; ++t) {
            const int o1 = P.tile_obs[t + 1];
            const bool one = o1 - o0 > kTileObs;  // one point with more than kTileObs observations
            // the point that this thread sums, loaded before the terms are formed
            int q0 = 0, n_sum = 0, pt = 0, a0 = 0, a1 = 0;
            auto point = [&](int p) {
                pt = P.pt_list[p];
                a0 = P.pt_ptr[p];
                a1 = P.pt_ptr[p + 1];
            };
            if (gX) {
                q0 = P.tile_pt[t];
                n_sum = 3 * (P.tile_pt[t + 1] - q0);
                if (tid < n_sum) point(q0 + tid / 3);
            }
            double cost = 0.0;
            T gp[3] = {T(0), T(0), T(0)};
            for (int a = o0 + tid; a < o1; a += kThreads) {
                const TP* Tc = Tcw + 12 * (size_t)c;
                const T* Xq = X + 3 * (size_t)q;
                const double u = uv.x, v = uv.y;
                if (a + kThreads < o1) load(a + kThreads, o1);
                ObsGrad<T> g;
                obs_term<T, kPointSide>(Tc, Xq, in, u, v, P.robust, P.delta, g);
                cost += g.cost;
#pragma unroll
                for (int k = 0; k < 8; ++k) acc[k] += (double)g.gintr[k];
                gp[0] += g.gX[0]; gp[1] += g.gX[1]; gp[2] += g.gX[2];
            }
            if (t + 1 < t1) load(o1 + tid, P.tile_obs[t + 2]);
            lane_cost[t - t0][tid] = cost;
            T (*st)[kTileObs] = sh[(t - t0) & 1];  // written again two tiles, hence a barrier, later
            if (gX) {  // uniform: gX is a kernel argument
#pragma unroll
                for (int k = 0; k < 3; ++k) st[k][tid] = gp[k];
                __syncthreads();
            }
            // per-point sums in fixed order, a thread per point and component
            for (int i = tid; i < n_sum; i += kThreads) {
                if (i != tid) point(q0 + i / 3);
                const T* v = st[i % 3];
                T s = T(0);
                if (one) {  // 256 lanes' sums: in FP64, as a serial sum of so many loses bits in float
                    double d = 0.0;
                    for (int a = 0; a < kThreads; ++a) d += (double)v[a];
                    s = (T)d;
                } else {
                    int a = a0 - o0;
                    const int e = a1 - o0;
                    for (; a + 4 <= e; a += 4) {
                        const T v0 = v[a], v1 = v[a + 1], v2 = v[a + 2], v3 = v[a + 3];
                        s = (((s + v0) + v1) + v2) + v3;
                    }
                    for (; a < e; ++a) s += v[a];
                }
                gX[3 * (size_t)pt + i % 3] = s;
            }
            o0 = o1;
        }
        if (!gX) __syncthreads();
        // after the last tile: a sum per tile within the loop cost 4 % of a gradient
        for (int t = t0 + tid / kWave; t < t1; t += kThreads / kWave) {
            const double s = tile_total(lane_cost[t - t0]);
            if (tid % kWave == 0) tile_cost[t] = s;
        }
        const double s = block_sums<8>(acc, red);
        if (tid < 8) part[(size_t)tid * P.n_groups + b] = s;
        return;
    }
    b -= P.n_groups;
    if (gpart) {
        if (b < P.n_chunks) {
            b = xcd_band(b, P.n_chunks);
            double acc[6] = {0, 0, 0, 0, 0, 0};
            const TP* Tc = Tcw + 12 * (size_t)P.chunk_cam[b];
            const int k1 = P.chunk_ptr[b + 1];
            int k = P.chunk_ptr[b] + tid, q = 0;
            double2 uv;
            if (k < k1) {
                q = P.c_pt[k];
                uv = P.c_uv[k];
            }
            for (; k < k1; k += kThreads) {
                const T* Xq = X + 3 * (size_t)q;
                const double u = uv.x, v = uv.y;
                if (k + kThreads < k1) {
                    q = P.c_pt[k + kThreads];
                    uv = P.c_uv[k + kThreads];
                }
                ObsGrad<T> g;
                obs_term<T, kPoseSide>(Tc, Xq, in, u, v, P.robust, P.delta, g);
#pragma unroll
                for (int j = 0; j < 6; ++j) acc[j] += (double)g.gpose[j];
            }
            const double s = block_sums<6>(acc, redc);
            if (tid < 6) gpart[6 * (size_t)b + tid] = s;
            return;
        }
        b -= P.n_chunks;
    }
    const int i = b * kThreads + tid;
    if (gX && i < P.n_unseen)
#pragma unroll
        for (int k = 0; k < 3; ++k) gX[3 * (size_t)P.unseen[i] + k] = T(0);
}

// This thread's share of a sum over v[i0 .. i1), sixteen loads in flight: the
// partial sums come from other XCDs, a microsecond away.
__device__ __forceinline__ double strided_sum(const double* __restrict__ v, int i0, int i1) {
    constexpr int kLoads = 16;
    double s = 0.0;
    for (int i = i0 + (int)threadIdx.x; i < i1; i += kLoads * kThreads) {
        double x[kLoads];
#pragma unroll
        for (int k = 0; k < kLoads; ++k) x[k] = v[min(i + k * kThreads, i1 - 1)];
#pragma unroll
        for (int k = 0; k < kLoads; ++k) s += i + k * kThreads < i1 ? x[k] : 0.0;
    }
    return s;
}

// Workgroup p < n_prob: cost of problem p over its tiles; then one for the total
// over all tiles (if asked for), eight for the intrinsic gradient over the groups
// (likewise); the others: pose gradients over the cameras' chunks, a thread per
// entry (all in a fixed order).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_cg_final(CostProblem P, const double* __restrict__ tile_cost,
                                                       const double* __restrict__ part, T* __restrict__ cost,
                                                       T* __restrict__ total, T* __restrict__ gintr,
                                                       const double* __restrict__ gpart, T* __restrict__ gpose) {
    __shared__ double red[kThreads / kWave];
    int b = blockIdx.x;
    auto sum = [&](const double* v, int i0, int i1, T* out) {
        const double s = block_sum<double, kThreads>(strided_sum(v, i0, i1), red);
        if (threadIdx.x == 0) *out = (T)s;
    };
    if (b < P.n_prob) return sum(tile_cost, P.prob_tile0[b], P.prob_tile0[b + 1], cost + b);
    b -= P.n_prob;
    if (total && b-- == 0) return sum(tile_cost, 0, P.n_tiles, total);
    if (gintr && b < 8) return sum(part + (size_t)b * P.n_groups, 0, P.n_groups, gintr + b);
    if (gintr) b -= 8;
    const int i = b * kThreads + (int)threadIdx.x;
    if (i >= 6 * P.n_cam) return;
    const int c = i / 6, j = i % 6;
    double s = 0.0;
    for (int k = P.cam_chunk0[c]; k < P.cam_chunk0[c + 1]; ++k) s += gpart[6 * (size_t)k + j];
    gpose[i] = (T)s;
}

// ---- pose tangents ----------------------------------------------------------
// Coefficients of exp on SE3 at th2 = |omega|^2 and their derivatives:
//   a = sin t / t, b = (1 - cos t) / t^2, c = (t - sin t) / t^3,
//   db = b'(t) / t = (a - 2 b) / t^2,  dc = c'(t) / t = (b - 3 c) / t^2.
// Below th2 = 0.25 their Taylor series (seven terms, truncation below 5e-17):
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

// T = exp(xi) T_cw, one pose per thread; out64: the same before its rounding to
// T, for the cost to be evaluated at (null where T is FP64: out serves).  Launch
// bound: a few hundred operations and at most 240 bytes per pose.  As torch operations the map and
// its derivative were about 230 launches of a gradient step; with these two
// kernels a step of BACost (64 scenes of 5 000 points, 1 280 poses, float) went
// from 1970 us to 260, on one scene of 700 (double) from 1800 to 168.
template <typename T>
__global__ void k_se3_left(int n, const T* __restrict__ xi, const T* __restrict__ Tcw, T* __restrict__ out,
                           double* __restrict__ out64) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    double w[3], u[3], t[3], col[3], r[3], v[3];
    auto put = [&](int e, double x) {
        out[12 * (size_t)c + e] = (T)x;
        if (out64) out64[12 * (size_t)c + e] = x;
    };
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
        for (int i = 0; i < 3; ++i) put(3 * i + j, r[i]);
    }
    rot3(w, k.a, k.b, t, r);
    rot3(w, k.b, k.c, u, v);
#pragma unroll
    for (int i = 0; i < 3; ++i) put(9 + i, r[i] + v[i]);
}

// g_xi = J_l(xi)^T g.  With p = V u, a step d of omega turns T by J d (J = V)
// and moves its translation, seen from the left, by (dV) u - (J d) x p, so
//   g_upsilon -> V^T g_u
//   g_omega   -> V^T (g_w - p x g_u) + grad_omega (g_u . V u),
// the last term from V u = u + b w x u + c (w (w.u) - |w|^2 u).
// The result is rounded to T and then multiplied by scale.
template <typename T>
__device__ __forceinline__ void tangent_grad_row(int c, const T* __restrict__ xi, const T* __restrict__ g, T scale,
                                                 T* __restrict__ out) {
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
        out[6 * (size_t)c + i] = (T)(rw[i] + k.b * ug[i] + k.c * (gu[i] * wu + u[i] * gw0) + s * w[i]) * scale;
        out[6 * (size_t)c + 3 + i] = (T)ru[i] * scale;
    }
}

template <typename T>
__global__ void k_tangent_grad(int n, const T* __restrict__ xi, const T* __restrict__ g, T* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < n) tangent_grad_row<T>(c, xi, g, T(1), out);
}

// The three gradients of a cost times the incoming gradient: poses (b_pose
// workgroups), points (four entries per thread), intrinsics.  Launch bound; as a
// kernel for the poses and three products it was four launches, 20 us of a
// step's host time.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_backward(int n, long long nx, const T* __restrict__ xi,
                                                       const T* __restrict__ gp, const T* __restrict__ gX,
                                                       const T* __restrict__ gi, const T* __restrict__ scale,
                                                       T* __restrict__ out_xi, T* __restrict__ out_X,
                                                       T* __restrict__ out_i, int b_pose, int b_pt) {
    const T s = *scale;
    int b = blockIdx.x;
    if (b < b_pose) {
        const int c = b * kThreads + threadIdx.x;
        if (c < n) tangent_grad_row<T>(c, xi, gp, s, out_xi);
        return;
    }
    b -= b_pose;
    if (b < b_pt) {
        const long long i0 = 4LL * kThreads * b + threadIdx.x;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const long long i = i0 + q * kThreads;
            if (i < nx) out_X[i] = gX[i] * s;
        }
        return;
    }
    if (threadIdx.x < 8) out_i[threadIdx.x] = gi[threadIdx.x] * s;
}

}  // namespace navcost

using namespace navcost;

struct nav_ba_cost_handle {
    int device = 0;
    std::string err;
    bool prepared = false;
    CostProblem P{};
    std::vector<void*> bufs;
    double* tile_cost = nullptr;  // [n_tiles]
    double* part = nullptr;   // [8][n_groups]
    double* gpart = nullptr;  // [n_chunks][6]
    double* pose = nullptr;   // [n_cam][12] exp(xi) T_cw in FP64, where the caller's type is float
};

namespace {

void free_all(nav_ba_cost_handle* h) {
    for (void* p : h->bufs) (void)hipFree(p);
    h->bufs.clear();
    h->tile_cost = h->part = h->gpart = h->pose = nullptr;
}

// A prepare's arrays and scratch in one allocation; arrays up to kPackBytes go in
// one copy (a copy of its own costs the host 18 us whatever its size up to there).
class Upload {
public:
    template <class V>
    void add(const V& v, const typename V::value_type** out) {
        a_.push_back(Array{v.data(), sizeof(typename V::value_type) * v.size(), reinterpret_cast<const void**>(out)});
    }
    void scratch(size_t bytes, double** out) {
        a_.push_back(Array{nullptr, bytes, reinterpret_cast<const void**>(const_cast<const double**>(out))});
    }
    int flush(nav_ba_cost_handle* h) {
        constexpr size_t kPackBytes = 64 << 10;
        std::stable_partition(a_.begin(), a_.end(), [](const Array& a) { return a.src && a.bytes <= kPackBytes; });
        std::vector<size_t> at(a_.size());
        size_t total = 0, packed = 0;
        for (size_t k = 0; k < a_.size(); ++k) {
            at[k] = total;
            total += (std::max<size_t>(a_[k].bytes, 1) + 255) & ~size_t(255);
            if (a_[k].src && a_[k].bytes <= kPackBytes) packed = total;
        }
        void* d = nullptr;
        const hipError_t e = hipMalloc(&d, std::max<size_t>(total, 256));
        if (e != hipSuccess) { h->err = std::string("hipMalloc: ") + hipGetErrorString(e); return NAV_BA_HIP_ERROR; }
        h->bufs.push_back(d);
        std::vector<char> pack(packed);
        bool ok = true;
        for (size_t k = 0; k < a_.size(); ++k) {
            *a_[k].dst = static_cast<char*>(d) + at[k];
            if (!a_[k].src || a_[k].bytes == 0) continue;
            if (at[k] < packed) std::memcpy(pack.data() + at[k], a_[k].src, a_[k].bytes);
            else ok = ok && hipMemcpy(static_cast<char*>(d) + at[k], a_[k].src, a_[k].bytes, hipMemcpyHostToDevice) == hipSuccess;
        }
        if (packed > 0) ok = ok && hipMemcpy(d, pack.data(), packed, hipMemcpyHostToDevice) == hipSuccess;
        if (!ok) { h->err = "hipMemcpy failed"; return NAV_BA_HIP_ERROR; }
        return NAV_BA_OK;
    }

private:
    struct Array { const void* src; size_t bytes; const void** dst; };  // src null: scratch
    std::vector<Array> a_;
};

int32_t launch_status(nav_ba_cost_handle* h) {
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) return NAV_BA_OK;
    h->err = std::string("launch: ") + hipGetErrorString(e);
    return NAV_BA_HIP_ERROR;
}

template <typename T, typename TP>
int32_t eval_t(nav_ba_cost_handle* h, const TP* Tcw, const T* X, const T* intr, T* total, T* cost, T* gpose, T* gX,
               T* gintr, hipStream_t s) {
    const CostProblem& P = h->P;
    const bool grad = gpose || gX || gintr;
    const int unseen = gX ? (P.n_unseen + kThreads - 1) / kThreads : 0;
    const int blocks = P.n_groups + (gpose ? P.n_chunks : 0) + unseen;
    if (grad && blocks > 0)  // a null gX or gpose skips its part
        hipLaunchKernelGGL((k_cg_obs<T, TP>), dim3(blocks), dim3(kThreads), 0, s, P, Tcw, X, intr, gX, h->tile_cost,
                           h->part, gpose ? h->gpart : nullptr);
    if (!grad && P.n_tiles > 0)
        hipLaunchKernelGGL((k_cg_cost<T, TP>), dim3(P.n_tiles), dim3(kThreads), 0, s, P, Tcw, X, intr, h->tile_cost);
    const int finals = P.n_prob + (total ? 1 : 0) + (gintr ? 8 : 0) + (gpose ? (6 * P.n_cam + kThreads - 1) / kThreads : 0);
    hipLaunchKernelGGL(k_cg_final<T>, dim3(finals), dim3(kThreads), 0, s, P, (const double*)h->tile_cost,
                       (const double*)h->part, cost, total, gintr, (const double*)h->gpart, gpose);
    return launch_status(h);
}

// T = exp(xi) T_cw, then the evaluation there, at the poses before their rounding to T.
template <typename T>
int32_t eval_tangent_t(nav_ba_cost_handle* h, const T* xi, const T* Tcw, const T* X, const T* intr, T* Tout, T* total,
                       T* cost, T* gpose, T* gX, T* gintr, hipStream_t s) {
    const int n = h->P.n_cam;
    double* pose = sizeof(T) < sizeof(double) ? h->pose : nullptr;
    if (n > 0)
        hipLaunchKernelGGL(k_se3_left<T>, dim3((n + kPoseThreads - 1) / kPoseThreads), dim3(kPoseThreads), 0, s, n, xi,
                           Tcw, Tout, pose);
    if (pose) return eval_t<T, double>(h, pose, X, intr, total, cost, gpose, gX, gintr, s);
    return eval_t<T, T>(h, Tout, X, intr, total, cost, gpose, gX, gintr, s);
}

template <typename T>
int32_t tangent_grad_t(int n, const T* xi, const T* g, T* out, hipStream_t s) {
    hipLaunchKernelGGL(k_tangent_grad<T>, dim3((n + kPoseThreads - 1) / kPoseThreads), dim3(kPoseThreads), 0, s, n, xi, g,
                       out);
    return hipGetLastError() == hipSuccess ? NAV_BA_OK : NAV_BA_HIP_ERROR;
}

// Null outputs are skipped.
template <typename T>
int32_t backward_t(int n, long long nx, const T* xi, const T* gp, const T* gX, const T* gi, const T* scale, T* out_xi,
                   T* out_X, T* out_i, hipStream_t s) {
    const int b_pose = out_xi ? (n + kThreads - 1) / kThreads : 0;
    const int b_pt = out_X ? (int)((nx + 4 * kThreads - 1) / (4 * kThreads)) : 0;
    const int blocks = b_pose + b_pt + (out_i ? 1 : 0);
    if (blocks == 0) return NAV_BA_OK;
    hipLaunchKernelGGL(k_backward<T>, dim3(blocks), dim3(kThreads), 0, s, n, nx, xi, gp, gX, gi, scale, out_xi, out_X,
                       out_i, b_pose, b_pt);
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
    // Both orders, a problem at a time (its cameras and points are contiguous, and
    // its part of every array stays in the cache): point-major (point, camera, input
    // order) by two stable counting sorts, camera-major from it by a third.
    std::vector<int> o_cam(no), o_pt(no), c_pt(no), cam_ptr(nc + 1, 0);
    std::vector<double2> uv(no), c_uv(no);
    {
        std::vector<int> byc, off, poff;
        size_t o0 = 0;
        for (int p = 0; p < n_probs; ++p) {
            const nav_ba_problem& q = probs[p];
            const int m = q.n_obs, c0 = cam_off[p], p0 = pt_off[p];
            off.assign(q.n_cam + 1, 0);
            poff.assign(q.n_pt + 1, 0);
            for (int i = 0; i < m; ++i) {
                off[q.obs_cam[i] + 1]++;
                poff[q.obs_pt[i] + 1]++;
            }
            for (int c = 0; c < q.n_cam; ++c) off[c + 1] += off[c];
            for (int c = 0; c < q.n_pt; ++c) poff[c + 1] += poff[c];
            for (int c = 0; c < q.n_cam; ++c) cam_ptr[c0 + c + 1] = (int)o0 + off[c + 1];
            byc.resize(m);
            for (int i = 0; i < m; ++i) byc[off[q.obs_cam[i]]++] = i;
            for (int k = 0; k < m; ++k) {
                const int i = byc[k];
                const size_t at = o0 + poff[q.obs_pt[i]]++;
                o_cam[at] = c0 + q.obs_cam[i];
                o_pt[at] = p0 + q.obs_pt[i];
                uv[at] = double2{q.obs_uv[2 * (size_t)i], q.obs_uv[2 * (size_t)i + 1]};
            }
            for (int c = 0; c < q.n_cam; ++c) off[c] = cam_ptr[c0 + c];
            for (size_t k = o0; k < o0 + m; ++k) {
                const int at = off[o_cam[k] - c0]++;
                c_pt[at] = o_pt[k];
                c_uv[at] = uv[k];
            }
            o0 += m;
        }
    }
    // unique points, tiles of whole points per problem
    std::vector<int> pt_list, pt_ptr{0}, tile_obs{0}, tile_pt{0}, prob_tile0{0};
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
                i = j;
            }
            prob_tile0.push_back((int)tile_pt.size() - 1);
        }
    }
    // groups of consecutive tiles of one problem
    auto groups_of = [&](int per) {
        long long n = 0;
        for (int p = 0; p < n_probs; ++p) n += (prob_tile0[p + 1] - prob_tile0[p] + per - 1) / per;
        return n;
    };
    int per_group = 1;
    while (per_group < kGroupTiles && groups_of(per_group) > kGroups) ++per_group;
    std::vector<int> group_tile{0};
    for (int p = 0; p < n_probs; ++p) {
        for (int t = prob_tile0[p]; t < prob_tile0[p + 1];) {
            t = std::min(t + per_group, prob_tile0[p + 1]);
            group_tile.push_back(t);
        }
    }
    // chunks of the camera-major order
    const int chunk = std::min<int>(kChunkMax, std::max<int>(1, (int)(no / ((size_t)kChunks * kThreads))) * kThreads);
    std::vector<int> chunk_cam, chunk_ptr{0}, cam_chunk0{0};
    for (int c = 0; c < nc; ++c) {
        for (int k = cam_ptr[c]; k < cam_ptr[c + 1];) {
            k = std::min(cam_ptr[c + 1] - k, chunk) + k;
            chunk_cam.push_back(c);
            chunk_ptr.push_back(k);
        }
        cam_chunk0.push_back((int)chunk_cam.size());
    }
    std::vector<int> unseen;
    for (int q = 0, i = 0; q < np; ++q) {
        if (i < (int)pt_list.size() && pt_list[i] == q) ++i;
        else unseen.push_back(q);
    }
    CostProblem& P = h->P;
    P = CostProblem{};
    P.n_obs = (int)no; P.n_tiles = prob_tile0.back(); P.n_groups = (int)group_tile.size() - 1; P.n_chunks = (int)chunk_cam.size();
    P.n_unseen = (int)unseen.size();
    P.n_cam = nc; P.n_pt = np; P.n_prob = n_probs;
    P.robust = robust ? 1 : 0;
    P.delta = huber_delta;
    Upload u;
    u.add(o_cam, &P.o_cam); u.add(o_pt, &P.o_pt); u.add(uv, &P.uv);
    u.add(pt_list, &P.pt_list); u.add(pt_ptr, &P.pt_ptr); u.add(tile_obs, &P.tile_obs); u.add(tile_pt, &P.tile_pt);
    u.add(group_tile, &P.group_tile); u.add(prob_tile0, &P.prob_tile0);
    u.add(c_pt, &P.c_pt); u.add(c_uv, &P.c_uv);
    u.add(chunk_cam, &P.chunk_cam); u.add(chunk_ptr, &P.chunk_ptr); u.add(cam_chunk0, &P.cam_chunk0);
    u.add(unseen, &P.unseen);
    u.scratch(sizeof(double) * P.n_tiles, &h->tile_cost);
    u.scratch(sizeof(double) * 8 * P.n_groups, &h->part);
    u.scratch(sizeof(double) * 6 * P.n_chunks, &h->gpart);
    u.scratch(sizeof(double) * 12 * nc, &h->pose);
    const int st = u.flush(h);
    if (st != NAV_BA_OK) return st;
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
        return eval_t<double, double>(h, (const double*)T_cw, (const double*)X, (const double*)intr, nullptr, (double*)cost,
                              (double*)g_pose, (double*)g_X, (double*)g_intr, s);
    if (dtype == NAV_BA_COST_F32)
        return eval_t<float, float>(h, (const float*)T_cw, (const float*)X, (const float*)intr, nullptr, (float*)cost,
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

int32_t nav_ba_cost_backward(int32_t device, int32_t dtype, int32_t n_cam, int32_t n_pt, const void* xi,
                             const void* g_pose, const void* g_X, const void* g_intr, const void* g, void* out_xi,
                             void* out_X, void* out_intr, void* stream) {
    if (n_cam < 0 || n_pt < 0 || !g || (dtype != NAV_BA_COST_F64 && dtype != NAV_BA_COST_F32)) return NAV_BA_BAD_ARG;
    if ((out_xi && n_cam > 0 && (!xi || !g_pose)) || (out_X && n_pt > 0 && !g_X) || (out_intr && !g_intr))
        return NAV_BA_BAD_ARG;
    int was = 0;
    if (hipGetDevice(&was) != hipSuccess) return NAV_BA_HIP_ERROR;
    if (was != device && hipSetDevice(device) != hipSuccess) return NAV_BA_HIP_ERROR;
    hipStream_t s = (hipStream_t)stream;
    const long long nx = 3LL * n_pt;
    const int32_t st =
        dtype == NAV_BA_COST_F64
            ? backward_t<double>(n_cam, nx, (const double*)xi, (const double*)g_pose, (const double*)g_X,
                                 (const double*)g_intr, (const double*)g, (double*)out_xi, (double*)out_X,
                                 (double*)out_intr, s)
            : backward_t<float>(n_cam, nx, (const float*)xi, (const float*)g_pose, (const float*)g_X,
                                (const float*)g_intr, (const float*)g, (float*)out_xi, (float*)out_X, (float*)out_intr, s);
    if (was != device && hipSetDevice(was) != hipSuccess) return NAV_BA_HIP_ERROR;
    return st;
}

}  // extern "C"
