// chol_kernels.hip — FP64 dense Cholesky of the reduced camera system and the
// two triangular solves (the factorisation g2o's LinearSolverEigen performs at
// BE_GraphOptim.cpp:43; here a plain LL^T, which for S + lambda I > 0 gives the
// same step as LDL^T).
//
// One problem: right-looking, 64x64 tiles, the matrix padded with the identity
// to a tile multiple, one launch per block column k.  Each diagonal tile is
// factored together with the inverse of its factor, M_k = L_kk^-1, so that
//   panel    L_ik = A_ik M_k^T                      (a 64x64x64 product),
//   forward  y_k = M_k (g_k - sum_{j<k} L_kj y_j)   (matrix-vector),
//   backward x_k = M_k^T (y_k - sum_{m>k} L_mk^T x_m)
// need no substitution chains.  On the reduced systems of the 60-keyframe
// problem (n = 348, condition 4e6, lambda 1e-4 .. 1e-10) this changes the step
// by at most 4e-13 relative against a substitution-based factorisation.
// Launch k: workgroup (i, j), k < j <= i, forms L_ik (and L_jk) from the
// updated A_ik, A_jk and M_k, then updates A_ij -= L_ik L_jk^T; workgroups
// (i, k+1) store L_ik, and workgroup (k+1, k+1) factors its freshly updated
// tile, inverts it and runs that tile's forward step.  The factor goes to a
// separate buffer, so no workgroup overwrites a tile another one still reads;
// the diagonal factors L_kk themselves are never stored (only M_k is used).
// All products run on FP64 MFMA (v_mfma_f64_16x16x4).
// Measured (rocprofv3, average per launch, launch included): 28 tiles, step
// 23.8 -> 15.6 us (14.9 without the zero tiles), first tile 18 -> 12.6 us, backward 28 launches of 4.2 -> 7 of
// 9.5 us; 6 tiles, step 21.6 -> 14.2 us, against a factorisation of the diagonal
// tile by pivots (31 k cycles of the step's 55 k; square roots, a column per
// pivot through LDS), operands staged through LDS and a launch per tile in the
// backward step.  A step's floor is its launch (about 2 us), one round trip to
// memory and the chain of the diagonal tile.
#include "ba_kernels.h"

namespace navba {

typedef double dbl4 __attribute__((ext_vector_type(4)));

// One FP64 16x16x4 matrix FMA of a wave, D = A B + C, with A[i][k] in lane
// i + 16k, B[k][j] in lane j + 16k and D[i][j] in element i / 4 of lane
// j + 16 (i % 4) (checked on gfx950 against a host product).
__device__ __forceinline__ dbl4 mfma16x16x4(double a, double b, dbl4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Index of the calling wave in its workgroup, as a scalar (wave-uniform
// branches and block indices stay on the scalar unit).
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// Orders the LDS accesses of one wave around a hand-off between its lanes
// (the wave's LDS instructions execute in program order).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// The value of v in lane l (l wave-uniform), as a uniform double.
__device__ __forceinline__ double lane_value(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffff), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Reciprocal: the hardware's estimate (relative error e below 2^-24) and one
// step of third order, r (1 + e + e^2).
__device__ __forceinline__ double fast_rcp(double d) {
    const double r = __builtin_amdgcn_rcp(d);
    const double e = fma(-d, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// Four products of 4x4 blocks, D_b = A_b B_b (b = 0..3), with A[i][k] in lane
// i + 4b + 16k, B[k][j] in lane j + 4b + 16k and D[i][j] in lane j + 4b + 16i
// (checked on gfx950 against a host product).
__device__ __forceinline__ double mfma4x4x4(double a, double b) {
    return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, 0.0, 0, 0, 0);
}

// LDL^T of a symmetric 16x16 tile and the inverse of its unit factor, by one
// wave in registers.  acc holds the tile in the matrix instruction's result
// layout (element v of lane (i, k) = l & 15, l >> 4: row 4 v + k, column i);
// by symmetry acc[p] is then the column panel 4p..4p+3 in the layout of an
// operand (lane (i, k): row i, column 4p + k), so a panel needs no data
// movement.  Per panel p of four columns:
//   the 4x4 diagonal block's LDL^T and the inverse N of its unit factor, the
//     same in every lane from ten lane reads;
//   W = A_p N^T as four 4x4 blocks, L_p = W D^-1, acc -= W L_p^T;
//   Z, which starts as the identity and ends as the inverse: Z_p = N Z_p,
//     Z -= L_p Z_p for the rows below.
// dv[p] = the reciprocal pivot of column 4p + k in lane (i, k).  Returns false
// if a pivot was not positive and finite (its values are then arbitrary), the
// same in every lane.
// A solve by substitution in 4x4 blocks instead of the inverse was no more
// accurate over 512 ill-conditioned windows (the same quantiles of the pose and
// cost errors against the oracle) and 4 us slower on the largest window.
__device__ __forceinline__ bool tile16_ldl(dbl4 acc, dbl4& Z, double dv[4]) {
    const int lane = threadIdx.x & 63, i = lane & 15, k = lane >> 4, i4 = lane & 3;
#pragma unroll
    for (int v = 0; v < 4; ++v) Z[v] = (4 * v + k == i) ? 1.0 : 0.0;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const double a = acc[p];
        const int q = 4 * p;
        const double a00 = lane_value(a, q), a10 = lane_value(a, q + 1), a11 = lane_value(a, q + 17),
                     a20 = lane_value(a, q + 2), a21 = lane_value(a, q + 18), a30 = lane_value(a, q + 3),
                     a31 = lane_value(a, q + 19), a22 = lane_value(a, q + 34), a32 = lane_value(a, q + 35),
                     a33 = lane_value(a, q + 51);
        const double i0 = fast_rcp(a00);
        const double l10 = a10 * i0, l20 = a20 * i0, l30 = a30 * i0;
        const double d1 = fma(-l10, a10, a11), t21 = fma(-l20, a10, a21), t31 = fma(-l30, a10, a31);
        const double i1 = fast_rcp(d1);
        const double l21 = t21 * i1, l31 = t31 * i1;
        const double d2 = fma(-l21, t21, fma(-l20, a20, a22)), t32 = fma(-l31, t21, fma(-l30, a20, a32));
        const double i2 = fast_rcp(d2);
        const double l32 = t32 * i2;
        const double d3 = fma(-l32, t32, fma(-l31, t31, fma(-l30, a30, a33)));
        const double i3 = fast_rcp(d3);
        // N, unit lower, element (i & 3, k) in lane (i, k)
        const double n20 = fma(l21, l10, -l20), n31 = fma(l32, l21, -l31);
        const double n30 = fma(-l32, n20, fma(l31, l10, -l30));
        double nv = i4 == k ? 1.0 : 0.0;
        if (i4 == 1 && k == 0) nv = -l10;
        if (i4 == 2 && k == 0) nv = n20;
        if (i4 == 2 && k == 1) nv = -l21;
        if (i4 == 3 && k == 2) nv = -l32;
        if (i4 == 3 && k == 1) nv = n31;
        if (i4 == 3 && k == 0) nv = n30;
        dv[p] = k == 0 ? i0 : k == 1 ? i1 : k == 2 ? i2 : i3;
        if (p < 3) {
            const double w = mfma4x4x4(nv, a);  // W[i][k]
            const double zp = mfma4x4x4(nv, Z[p]);  // row 4p + k, column i of N Z_p
            const double lp = w * dv[p];
            acc = mfma16x16x4(-w, lp, acc);
            Z = mfma16x16x4(i >= q + 4 ? -lp : 0.0, zp, Z);
            Z[p] = zp;
        } else {
            Z[p] = mfma4x4x4(nv, Z[p]);
        }
    }
    bool good = true;
#pragma unroll
    for (int p = 0; p < 4; ++p) good = good && dv[p] > 0.0 && isfinite(dv[p]);
    return __all(good);
}

// Sum over the four lanes (i, 0..3), in each of them: row pairs, then halves.
__device__ __forceinline__ double sum_over_k(double v) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
    const auto l1 = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h1 = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    const double s = __longlong_as_double(((long long)h1[0] << 32) | l1[0]) +
                     __longlong_as_double(((long long)h1[1] << 32) | l1[1]);
    const long long c = __double_as_longlong(s);
    const unsigned lo2 = (unsigned)c, hi2 = (unsigned)(c >> 32);
    const auto l2 = __builtin_amdgcn_permlane32_swap(lo2, lo2, false, false);
    const auto h2 = __builtin_amdgcn_permlane32_swap(hi2, hi2, false, false);
    return __longlong_as_double(((long long)h2[0] << 32) | l2[0]) +
           __longlong_as_double(((long long)h2[1] << 32) | l2[1]);
}

// 16-column stages of diagonal tile i that hold rows of the n-row system (the
// last tile's padding rows beyond are the identity and are not factored).
__device__ __forceinline__ int tile_stages(int n, int i) { return min(4, (n - 64 * i + 15) >> 4); }

// ---------------------------------------------------------------- diagonal tiles
// A diagonal tile is factored by one workgroup of four waves, its 16x16 blocks
// in registers: wave w holds the blocks (w, 0..w), block (w, j) in operand
// layout (element p of lane (i, k): row i, column 4 p + k).  With A and B
// swapped, the matrix instruction returns a product's transpose, which is that
// same layout, so a block goes through solve and update without data movement.
// Stage s (two barriers):
//   wave s    LDL^T of block (s, s) and the inverse Z_s of its unit factor
//             (tile16_ldl); the other waves, whose blocks are done, meanwhile
//             form R_sw = sum_{w<=k<s} L_sk M_kw, wave w owning block column w
//             of the inverse, which needs only its own blocks M_kw;
//   barrier   Z_s, the reciprocal pivots;
//   wave i>s  W_is = A_is Z_s^T (= L_is D_s), shared through LDS; barrier;
//             A_ij -= W_is D_s^-1 W_js^T, s < j <= i: wave s + 1 needs one block
//             before it goes on;
//   wave w<s  M_sw = -Z_s R_sw;
//   wave 0    the right-hand side, carried like a block row whose 16 rows are
//             all g: z_s = Z_s g_s, g_j -= W_js D_s^-1 z_s.
// The tile's factor in LL^T form is L D^1/2, its inverse M = D^-1/2 (unit
// inverse), its forward result y = D^-1/2 z; M and y are scaled on the way out.
// Bound by the chain through the four blocks (about 3 k cycles each).
struct DiagLds {
    double Z[4][16 * 17];  // [row][17]: read along rows and columns without bank conflicts
    double W[6][256];      // W_is in lane order, block i (i - 1) / 2 + s
    double dinv[64];       // reciprocal pivots
    double sd[64];         // their square roots
    double g[64];          // right-hand side
};

// Inverse tiles: M row-major (64x64, for the backward step), then its lower
// 16x16 blocks (b, c) at kInvPack + 256 (b (b + 1) / 2 + c) in the order in
// which k_chol_step's lanes read them: entry (j, 4 k + e) at 4 (j + 16 k) + e.
constexpr int kInvPack = 4096;
static_assert(kInvTile == kInvPack + 10 * 256, "inverse tile size");

__device__ __forceinline__ double fast_sqrt(double d) {  // by rsq and two Goldschmidt steps; d > 0
    double H = __builtin_amdgcn_rsq(d), g = d * H;
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const double e = fma(-g, H, 1.0);
        g = fma(0.5 * g, e, g);
        H = fma(0.5 * H, e, H);
    }
    return g;
}

// Block (b, c) of the inverse, m in result layout, its rows scaled by sd.
__device__ __forceinline__ void inv_store(double* __restrict__ Li, int b, int c, dbl4 m, const double* sd) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
    double* pk = Li + kInvPack + 256 * (b * (b + 1) / 2 + c) + 64 * (r16 >> 2) + (r16 & 3);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = 4 * v + kq;
        const double x = m[v] * sd[16 * b + r];
        Li[(16 * b + r) * 64 + 16 * c + r16] = x;
        pk[4 * r] = x;
    }
}

// a: the calling wave's blocks; D.g is written (a barrier follows before it is
// read); nst: stages that hold rows of the system.  Li and y receive the
// tile's inverse and forward result.  idle(h), h = 0, 1: other work for one wave
// each, called where the chain does not wait for that wave.  Returns false in the wave that met a
// pivot which is not positive and finite.
template <class Idle>
__device__ __forceinline__ bool diag_factor(dbl4 a[4], DiagLds& D, int nst, double* __restrict__ Li,
                                            double* __restrict__ y, Idle idle) {
    const int lane = threadIdx.x & 63, w = wave_id(), r16 = lane & 15, kq = lane >> 4;
    const dbl4 zero = {0.0, 0.0, 0.0, 0.0};
    bool good = true;
    dbl4 m[4], gt[4], zs = zero;  // m[i]: block (i, w) of the unit inverse, result layout
    auto clear = [&](int b, int c) {  // a block above the diagonal
#pragma unroll
        for (int v = 0; v < 4; ++v) Li[(16 * b + 4 * v + kq) * 64 + 16 * c + r16] = 0.0;
    };
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        dbl4 R = zero;
        if (w == s) {
            double dv[4] = {1.0, 1.0, 1.0, 1.0};
            if (s < nst) {
                good = tile16_ldl(a[s], m[s], dv);
            } else {  // padding rows: the identity
#pragma unroll
                for (int v = 0; v < 4; ++v) m[s][v] = (4 * v + kq == r16) ? 1.0 : 0.0;
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) D.Z[s][17 * (4 * v + kq) + r16] = m[s][v];
            if (r16 < 4) {
                const double d = r16 == 0 ? dv[0] : r16 == 1 ? dv[1] : r16 == 2 ? dv[2] : dv[3];
                D.dinv[16 * s + 4 * r16 + kq] = d;
                D.sd[16 * s + 4 * r16 + kq] = fast_sqrt(d);
            }
        } else if (w < s) {
            inv_store(Li, s - 1, w, m[s - 1], D.sd);
#pragma unroll
            for (int k = 0; k < s; ++k)
                if (k >= w) {
                    const double* W = D.W[s * (s - 1) / 2 + k];
#pragma unroll
                    for (int p = 0; p < 4; ++p)
                        R = mfma16x16x4(W[64 * p + lane] * D.dinv[16 * k + 4 * p + kq], m[k][p], R);
                }
        }
        if (s == 1 && w == 0) idle(0);
        if (s == 2 && w == 1) idle(1);
        if (s == 3 && w < 2) {
            clear(w, 1 + w);
            clear(w, 2 + w);
            if (w == 0) clear(0, 3);
            else clear(2, 3);
        }
        if (w == 0 && s > 0) {
            if (r16 == 0)
#pragma unroll
                for (int v = 0; v < 4; ++v) y[16 * (s - 1) + 4 * v + kq] = zs[v] * D.sd[16 * (s - 1) + 4 * v + kq];
        }
        __syncthreads();
        if (w == 0 && s == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int p = 0; p < 4; ++p) gt[j][p] = D.g[16 * j + 4 * p + kq];
        }
        double zt[4], dk[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            zt[p] = D.Z[s][17 * r16 + 4 * p + kq];
            dk[p] = D.dinv[16 * s + 4 * p + kq];
        }
        dbl4 wv = zero;
        if (w > s) {
#pragma unroll
            for (int p = 0; p < 4; ++p) wv = mfma16x16x4(zt[p], a[s][p], wv);
#pragma unroll
            for (int p = 0; p < 4; ++p) D.W[w * (w - 1) / 2 + s][64 * p + lane] = wv[p];
        }
        if (s < 3) __syncthreads();
        if (w > s) {
#pragma unroll
            for (int j = s + 1; j < 4; ++j)
                if (j <= w) {
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        const double x = j == w ? wv[p] : D.W[j * (j - 1) / 2 + s][64 * p + lane];
                        a[j] = mfma16x16x4(-x, wv[p] * dk[p], a[j]);
                    }
                }
        }
        if (w == 0) {
            zs = zero;
#pragma unroll
            for (int p = 0; p < 4; ++p) zs = mfma16x16x4(zt[p], gt[s][p], zs);
#pragma unroll
            for (int j = s + 1; j < 4; ++j)
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    gt[j] = mfma16x16x4(-D.W[j * (j - 1) / 2 + s][64 * p + lane], zs[p] * dk[p], gt[j]);
        }
        if (w < s) {
            m[s] = zero;
#pragma unroll
            for (int p = 0; p < 4; ++p) m[s] = mfma16x16x4(-zt[p], R[p], m[s]);
        }
    }
    inv_store(Li, 3, w, m[3], D.sd);
    if (w == 0 && r16 == 0)
#pragma unroll
        for (int v = 0; v < 4; ++v) y[48 + 4 * v + kq] = zs[v] * D.sd[48 + 4 * v + kq];
    return good;
}

__global__ __launch_bounds__(256) void k_chol_first(const double* __restrict__ S, double* __restrict__ Li, int lda, int n,
                                                    const double* __restrict__ g, double* __restrict__ y, LMDev* lm) {
    __shared__ DiagLds D;
    const int lane = threadIdx.x & 63, w = wave_id(), r16 = lane & 15, kq = lane >> 4;
    dbl4 a[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (j <= w)
#pragma unroll
            for (int p = 0; p < 4; ++p) a[j][p] = S[(size_t)(16 * w + r16) * lda + 16 * j + 4 * p + kq];
    if (threadIdx.x < 64) D.g[threadIdx.x] = g[threadIdx.x];
    if (lm->phase == kPhaseDone) return;  // a step launched after the solve has finished
    if (!diag_factor(a, D, tile_stages(n, 0), Li, y, [](int) {}) && lane == 0) atomicOr(&lm->fail, 1);
}

// Four consecutive doubles of a row.
__device__ __forceinline__ void load4(double v[4], const double* __restrict__ p) {
    const double2 a = reinterpret_cast<const double2*>(p)[0], b = reinterpret_cast<const double2*>(p)[1];
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    v[3] = b.y;
}

// W = A_k M_k^T for the calling wave's 16 rows: va[4 g + e] of lane (i, k) is
// entry (i, 16 g + 4 k + e) of the rows (the order of a product's terms is
// free, so each lane takes 32 contiguous bytes), vm the blocks of M_k in the
// same order.  W in operand layout: element 4 b + v, column 16 b + 4 v + k.
__device__ __forceinline__ void panel_rows(const double va[16], const double vm[40], dbl4 W[4]) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        W[b] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int g = 0; g <= b; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                W[b] = mfma16x16x4(vm[4 * (b * (b + 1) / 2 + g) + e], va[4 * g + e], W[b]);
    }
}

constexpr int kCus = 256;  // compute units of the device

// One launch per tile column k; workgroup (i, j), k < j <= i, four waves, wave w
// the rows 16 w.. of the tile.  Operands come from memory straight into
// registers in the order the matrix instructions take them, L_ik stays there
// (panel_rows), and only L_jk, which every wave needs, goes through LDS: one
// barrier.  (M_k through LDS too, loaded once instead of by each wave, cost a
// second barrier and 2 k cycles.)  Workgroup (k+1, k+1) goes on to factor its tile
// and is the launch's critical path: wave 0 starts the first block's
// factorisation while the others still update theirs, L is stored by waves that
// the chain does not wait for, and its waves take priority over those that share
// its compute unit.
__global__ __launch_bounds__(256, 2) void k_chol_step(double* __restrict__ S, double* __restrict__ Lm,
                                                      double* __restrict__ Li, int lda, int n, int k,
                                                      const double* __restrict__ g, double* __restrict__ y,
                                                      double* __restrict__ fsum, LMDev* lm) {
    __shared__ double Wj[4][16][64];  // [rows 16 b][element][lane]
    __shared__ double ys[64];
    __shared__ int nz[4];
    __shared__ DiagLds D;
    // Workgroups past the 256th share the first ones' compute units, so up to twice
    // that many the critical one (index 0) goes last among the 256: alone.
    // (300-camera loop, 378 to 276 workgroups: 22.1 and 19.6 -> 17.3 us a step.)
    const int at = gridDim.x > kCus && gridDim.x < 2 * kCus ? kCus - 1 : 0, b = blockIdx.x;
    const int idx = b == at ? 0 : b < at ? b + 1 : b;
    int ii = (int)((sqrtf(8.0f * idx + 1.0f) - 1.0f) * 0.5f);  // to one; then exactly
    while ((ii + 1) * (ii + 2) / 2 <= idx) ++ii;
    while (ii * (ii + 1) / 2 > idx) --ii;
    const int jj = idx - ii * (ii + 1) / 2;
    const int i = k + 1 + ii, j = k + 1 + jj;
    const bool same = (i == j), diag = idx == 0, panel = j == k + 1;
    if (diag) __builtin_amdgcn_s_setprio(3);
    // every global load of the launch in flight at once (no other workgroup
    // writes any of them)
    const int lane = threadIdx.x & 63, w = wave_id(), r16 = lane & 15, kq = lane >> 4;
    double vm[40], vi[16], vj[16];
    const double* Ai = S + (size_t)(64 * i + 16 * w + r16) * lda + 64 * k + 4 * kq;
    const double* Aj = S + (size_t)(64 * j + 16 * w + r16) * lda + 64 * k + 4 * kq;
    const double* Mk = Li + (size_t)kInvTile * k + kInvPack + 4 * lane;
#pragma unroll
    for (int q = 0; q < 4; ++q) load4(vi + 4 * q, Ai + 16 * q);
#pragma unroll
    for (int q = 0; q < 10; ++q) load4(vm + 4 * q, Mk + 256 * q);
    if (!same) {
#pragma unroll
        for (int q = 0; q < 4; ++q) load4(vj + 4 * q, Aj + 16 * q);
    }
    dbl4 cur[4];
    double* Aij = S + (size_t)(64 * i + 16 * w) * lda + 64 * j;
    if (diag) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (b <= w)
#pragma unroll
                for (int v = 0; v < 4; ++v) cur[b][v] = Aij[(size_t)r16 * lda + 16 * b + 4 * v + kq];
    } else {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) cur[b][v] = Aij[(size_t)(4 * v + kq) * lda + 16 * b + r16];
    }
    // the forward step: y_k, and sum_{t<k} L_it y_t of the earlier launches (one
    // workgroup per launch adds its term, so the order is fixed)
    const double yk = panel && w == 0 ? y[64 * k + lane] : 0.0;
    double f0 = 0.0;
    if (panel && k > 0) f0 = diag ? (w == 1 ? fsum[64 * i + lane] : 0.0) : (kq == 0 ? fsum[64 * i + 16 * w + r16] : 0.0);
    const double gi = diag && w == 1 ? g[64 * i + lane] : 0.0;
    if (lm->phase == kPhaseDone) return;  // a step launched after the solve has finished (loads in flight meanwhile)
    if (!diag) {
        // A zero A_ik or A_jk (cameras that share no points, and no fill) leaves the
        // tile as it is: the workgroup ends here and leaves the matrix cores to the
        // others.  28 tiles of a 300-camera loop, where 55 of the 378 tiles take part
        // in the first step: 422 -> 412 us for the 27 steps, the same bits.
        bool zi = true, zj = true;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            zi = zi && vi[q] == 0.0;
            zj = zj && (same || vj[q] == 0.0);
        }
        const int some = (__any(!zi) ? 1 : 0) | (__any(same ? !zi : !zj) ? 2 : 0);
        if (lane == 0) nz[w] = some;
        __syncthreads();
        const int all = nz[0] | nz[1] | nz[2] | nz[3];
        if (!(all & 1) || (!panel && !(all & 2))) {
            if (panel) {  // L_ik = 0; its term of the forward sum too
                if (k == 0 && kq == 0) fsum[64 * i + 16 * w + r16] = 0.0;
                double* L = Lm + (size_t)(64 * i + 16 * w + r16) * lda + 64 * k + kq;
#pragma unroll
                for (int p = 0; p < 16; ++p) L[4 * p] = 0.0;
            }
            return;
        }
    }
    if (w == 0) ys[lane] = yk;
    auto share = [&](const dbl4 W[4]) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) Wj[w][4 * b + v][lane] = W[b][v];
    };
    dbl4 Wi[4];
    panel_rows(vi, vm, Wi);  // L_ik
    __builtin_amdgcn_sched_barrier(0);  // what follows would lengthen the operands' lives
    if (!same) {
        dbl4 Wr[4];
        panel_rows(vj, vm, Wr);  // L_jk
        share(Wr);
    } else {
        share(Wi);
    }
    __syncthreads();
    if (diag) {
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (b <= w)
#pragma unroll
                for (int p = 0; p < 16; ++p) cur[b] = mfma16x16x4(-Wj[b][p][lane], Wi[p >> 2][p & 3], cur[b]);
        if (w == 1) {
            // the tile's right-hand side, a row per lane
            double f[4] = {gi - f0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int p = 0; p < 16; ++p)
#pragma unroll
                for (int q = 0; q < 4; ++q) f[q] = fma(-Wj[kq][p][r16 + 16 * q], ys[4 * p + q], f[q]);
            D.g[lane] = (f[0] + f[1]) + (f[2] + f[3]);
        }
        // two waves store L_ik while the chain goes on without them
        auto store_l = [&](int half) {
            double* L = Lm + (size_t)(64 * i + 32 * half + r16) * lda + 64 * k + kq;
#pragma unroll
            for (int p = 0; p < 32; ++p) L[(size_t)(16 * (p >> 4)) * lda + 4 * (p & 15)] = Wj[2 * half + (p >> 4)][p & 15][lane];
        };
        if (!diag_factor(cur, D, tile_stages(n, i), Li + (size_t)kInvTile * i, y + 64 * i, store_l) && lane == 0)
            atomicOr(&lm->fail, 1);
        return;
    }
    if (panel) {
        double f = f0;  // + L_ik y_k
#pragma unroll
        for (int p = 0; p < 16; ++p) f = fma(Wi[p >> 2][p & 3], ys[4 * p + kq], f);
        f = sum_over_k(f);
        if (kq == 0) fsum[64 * i + 16 * w + r16] = f;
        double* L = Lm + (size_t)(64 * i + 16 * w + r16) * lda + 64 * k + kq;
#pragma unroll
        for (int p = 0; p < 16; ++p) L[4 * p] = Wi[p >> 2][p & 3];
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int p = 0; p < 16; ++p) cur[b] = mfma16x16x4(-Wi[p >> 2][p & 3], Wj[b][p][lane], cur[b]);
    // a diagonal tile keeps its upper triangle (never used; left unchanged so
    // that it does not drift over the trials of a solve)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 16 * w + 4 * v + kq;
            if (!same || r >= 16 * b + r16) Aij[(size_t)(4 * v + kq) * lda + 16 * b + r16] = cur[b][v];
        }
}

// Backward step x = L^-T y for up to kBackSingleMax tiles in one workgroup of
// 512 threads, tile by tile
// from the last.  The right-hand sides r (the forward result) are held in LDS
// and updated in place:
//   x_k  = M_k^T r_k      (64x64 product, 8 partial sums per entry),
//   r_i -= L_ki^T x_k     (all columns left of tile k: 128 per pass, 4 partial
//                          sums per column);
// r_k is final when step k starts (every later step has subtracted its
// term), and x_k takes its place in LDS.  The L_ki loads of a step's first
// pass are issued before x_k is formed.  One workgroup keeps the tile chain
// inside one launch.  dp = 0 when the factorisation failed.  The same
// workgroup then forms the candidate poses from x (the camera update of the
// problem's one window) and the camera part of x'(lambda x + b).
constexpr int kBackThreads = 512;

// NP: 128-column passes of the widest update (64 (nt - 1) columns), so that
// the L loads of a step fit in registers.
constexpr int kBackPassMax = (64 * (kBackSingleMax - 1) + 127) / 128;

template <int NP>
__global__ __launch_bounds__(kBackThreads) void k_chol_back(DevProblem P, const double* __restrict__ Lm,
                                                            const double* __restrict__ Li, int lda, int nt,
                                                            const double* __restrict__ y, double* __restrict__ dp,
                                                            const LMDev* lm, const PoseQT* __restrict__ pose,
                                                            const double* __restrict__ Hc, PoseQT* __restrict__ pn,
                                                            CamRT* __restrict__ cn, double* __restrict__ red_scale) {
    extern __shared__ double rs[];  // [64 nt]
    __shared__ double part[8][64];
    __shared__ double red[4][128 * NP];
    __shared__ double xk[64];
    __shared__ double shs[kBackThreads / kWave];
    const int tid = threadIdx.x, n = 64 * nt;
    // the camera inputs (pose, b_p) of the first kBackThreads cameras load
    // while the solve runs
    const CamIn cin = camera_inputs(P, pose, Hc, max(0, min(tid, P.n_cam - 1)));
    if (lm->phase == kPhaseDone) return;
    const int fail = lm->fail;
    if (fail) {
        for (int i = tid; i < n; i += kBackThreads) dp[i] = 0.0;
    } else {
    const int c = tid & 63, grp = tid >> 6;   // x_k: entry c, rows grp + 8u
    const int pc = tid & 127, mq = tid >> 7;  // updates: column pc of each pass, rows 16 mq + u
    // M_k of the next step is loaded during the current one
    double mv[8];
    {
        const double* Mk = Li + (size_t)kInvTile * (nt - 1);
#pragma unroll
        for (int u = 0; u < 8; ++u) mv[u] = Mk[(grp + 8 * u) * 64 + c];
    }
    for (int i = tid; i < n; i += kBackThreads) rs[i] = y[i];
    __syncthreads();
    for (int k = nt - 1; k >= 0; --k) {
        const int ncols = 64 * k;
        const double* Lk = Lm + (size_t)(64 * k) * lda;
        // every L_ki load of the step, all passes, before x_k is formed
        double lv[NP][16];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const int col = 128 * q + pc;
            if (col < ncols) {
#pragma unroll
                for (int u = 0; u < 16; ++u) lv[q][u] = Lk[(size_t)(16 * mq + u) * lda + col];
            }
        }
        {
            double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
            for (int u = 0; u < 8; u += 4) {
                s0 += mv[u] * rs[64 * k + grp + 8 * u];
                s1 += mv[u + 1] * rs[64 * k + grp + 8 * u + 8];
                s2 += mv[u + 2] * rs[64 * k + grp + 8 * u + 16];
                s3 += mv[u + 3] * rs[64 * k + grp + 8 * u + 24];
            }
            part[grp][c] = (s0 + s1) + (s2 + s3);
        }
        if (k > 0) {
            const double* Mk = Li + (size_t)kInvTile * (k - 1);
#pragma unroll
            for (int u = 0; u < 8; ++u) mv[u] = Mk[(grp + 8 * u) * 64 + c];
        }
        __syncthreads();
        if (tid < 64) {
            const double x = ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid])) +
                             ((part[4][tid] + part[5][tid]) + (part[6][tid] + part[7][tid]));
            xk[tid] = x;
            rs[64 * k + tid] = x;  // r_k is not read again
            dp[64 * k + tid] = x;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const int col = 128 * q + pc;
            if (col < ncols) {
                double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
                for (int u = 0; u < 16; u += 4) {
                    s0 += lv[q][u] * xk[16 * mq + u];
                    s1 += lv[q][u + 1] * xk[16 * mq + u + 1];
                    s2 += lv[q][u + 2] * xk[16 * mq + u + 2];
                    s3 += lv[q][u + 3] * xk[16 * mq + u + 3];
                }
                red[mq][col] = (s0 + s1) + (s2 + s3);
            }
        }
        __syncthreads();
        for (int col = tid; col < ncols; col += kBackThreads)
            rs[col] -= (red[0][col] + red[1][col]) + (red[2][col] + red[3][col]);
        __syncthreads();
    }
    }
    const double lambda = lm->lambda;
    double sc = 0.0;
    for (int c = tid; c < P.n_cam; c += kBackThreads)
        sc += camera_candidate(c == tid ? cin : camera_inputs(P, pose, Hc, c), lambda, fail, c,
                               [&](int f, int i) { return rs[6 * f + i]; }, pn, cn);
    const double s = block_sum<double, kBackThreads>(sc, shs);
    if (tid == 0) red_scale[0] = s;
}

// Backward step for many tiles (more than kBackSingleMax): one launch per group
// of up to kBackGroup tiles k1, k1 - 1, .., from the last, so the reads of the
// factor spread over the chip.  The right-hand sides r of the tiles still to
// solve live in y (the forward result) and are updated in place: every
// workgroup of a launch forms the group's x (M_k^T r_k and the updates within
// the group, recomputed by each workgroup instead of waiting for one); the last
// workgroup writes them to dp, workgroup i below the group subtracts their terms
// L_ki^T x_k from r_i.  The group's r are only read during its launch, and final
// when it starts.  dp = 0 when the factorisation failed.
constexpr int kBackGroup = 4;

__global__ __launch_bounds__(kBackThreads) void k_chol_back_group(const double* __restrict__ Lm,
                                                                  const double* __restrict__ Li, int lda, int nt,
                                                                  int k1, int cnt, double* __restrict__ y,
                                                                  double* __restrict__ dp, const LMDev* lm) {
    __shared__ double part[kBackGroup - 1][8][64];
    __shared__ double xs[kBackGroup][64];
    __shared__ double rs[kBackGroup][64];
    const int tid = threadIdx.x, c = tid & 63, grp = tid >> 6;  // column c, rows grp + 8 u of every tile
    const int k0 = k1 - cnt + 1, i = blockIdx.x;  // i == k0 writes the group's x, i < k0 updates r_i
    // every load before its first use: M_k, r_k and the group's own tiles L_kh, h < k
    double mv[kBackGroup][8], gv[kBackGroup][kBackGroup][8];
#pragma unroll
    for (int q = 0; q < kBackGroup; ++q) {
        if (q >= cnt) continue;
        const double* M = Li + (size_t)kInvTile * (k1 - q) + grp * 64 + c;
#pragma unroll
        for (int u = 0; u < 8; ++u) mv[q][u] = M[512 * u];
#pragma unroll
        for (int h = q + 1; h < kBackGroup; ++h) {
            if (h >= cnt) continue;
            const double* L = Lm + (size_t)(64 * (k1 - q) + grp) * lda + 64 * (k1 - h) + c;
#pragma unroll
            for (int u = 0; u < 8; ++u) gv[q][h][u] = L[(size_t)(8 * u) * lda];
        }
    }
    if (grp < cnt) rs[grp][c] = y[64 * (k1 - grp) + c];
    if (lm->phase == kPhaseDone) return;  // a step launched after the solve has finished
    if (lm->fail) {
        if (k1 == nt - 1) {  // this launch has a workgroup for every tile
            if (i < k0) {
                if (tid < 64) dp[64 * i + tid] = 0.0;
            } else if (grp < cnt) {
                dp[64 * (k1 - grp) + c] = 0.0;
            }
        }
        return;
    }
    double lv[kBackGroup][8];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kBackGroup; ++q) {
        if (q < cnt) {
            double s0 = 0.0, s1 = 0.0;
#pragma unroll
            for (int u = 0; u < 8; u += 2) {
                s0 = fma(mv[q][u], rs[q][grp + 8 * u], s0);
                s1 = fma(mv[q][u + 1], rs[q][grp + 8 * u + 8], s1);
            }
            part[0][grp][c] = s0 + s1;
            if (i < k0) {  // the tile L_ki of the update, while the chain goes on
                const double* L = Lm + (size_t)(64 * (k1 - q) + grp) * lda + 64 * i + c;
#pragma unroll
                for (int u = 0; u < 8; ++u) lv[q][u] = L[(size_t)(8 * u) * lda];
            }
            __syncthreads();
            if (tid < 64) {
                const double x = ((part[0][0][tid] + part[0][1][tid]) + (part[0][2][tid] + part[0][3][tid])) +
                                 ((part[0][4][tid] + part[0][5][tid]) + (part[0][6][tid] + part[0][7][tid]));
                xs[q][tid] = x;
                if (i == k0) dp[64 * (k1 - q) + tid] = x;
            }
            __syncthreads();
            if (q + 1 < cnt) {
#pragma unroll
                for (int h = q + 1; h < kBackGroup; ++h) {
                    if (h >= cnt) continue;
                    double t0 = 0.0, t1 = 0.0;
#pragma unroll
                    for (int u = 0; u < 8; u += 2) {
                        t0 = fma(gv[q][h][u], xs[q][grp + 8 * u], t0);
                        t1 = fma(gv[q][h][u + 1], xs[q][grp + 8 * u + 8], t1);
                    }
                    part[h - 1][grp][c] = t0 + t1;
                }
                __syncthreads();
                if (grp > q && grp < cnt) {
                    const double (*pt)[64] = part[grp - 1];
                    rs[grp][c] -= ((pt[0][c] + pt[1][c]) + (pt[2][c] + pt[3][c])) +
                                  ((pt[4][c] + pt[5][c]) + (pt[6][c] + pt[7][c]));
                }
                __syncthreads();
            }
        }
    }
    if (i == k0) return;
    double s0 = 0.0, s1 = 0.0;
#pragma unroll
    for (int q = 0; q < kBackGroup; ++q) {
        if (q >= cnt) continue;
#pragma unroll
        for (int u = 0; u < 8; u += 2) {
            s0 = fma(lv[q][u], xs[q][grp + 8 * u], s0);
            s1 = fma(lv[q][u + 1], xs[q][grp + 8 * u + 8], s1);
        }
    }
    __syncthreads();  // part is free (the last step's sums are read)
    part[0][grp][c] = s0 + s1;
    __syncthreads();
    if (tid < 64)
        y[64 * i + tid] -= ((part[0][0][tid] + part[0][1][tid]) + (part[0][2][tid] + part[0][3][tid])) +
                           ((part[0][4][tid] + part[0][5][tid]) + (part[0][6][tid] + part[0][7][tid]));
}

// ---------------------------------------------------------------- per-window systems
// One workgroup (512 threads) per running window, and for a single problem of
// at most 30 free cameras: the window's reduced system (n = 6 nb unknowns) is
// summed from the Schur rows' partials straight into LDS, factored there as
// S = L D L^T (L unit lower, no square roots: a reciprocal's chain is shorter)
// and solved.  The system lies in LDS as 16x16 tiles of the lower triangle,
// the operand size of the FP64 matrix instruction; the right-hand side is row n
// below the matrix, so the forward step is part of the panel solve.
// Per tile column k, with M_k the inverse of the diagonal tile's unit factor:
//   solve    W_ik = A_ik M_k^T (= L_ik D_k) for the rows i > k, one tile per
//            wave at a time;
//   chain    wave 0: A_{k+1,k+1} -= W D^-1 W^T, then the tile's LDL^T and
//            M_{k+1} in registers (tile16_ldl);
//   update   meanwhile, waves 1..7: A_ij -= W_ik D_k^-1 W_jk^T for the other
//            tiles, k < j <= i.
// Two barriers per tile column.  The backward step x_k = M_k^T D_k^-1 (z_k -
// sum_{i>k} W_ik^T x_i) runs over the waves with one barrier per tile column;
// then the window's candidate poses are formed from the step in LDS (the
// camera update, fused).  Bound by the chain through the diagonal tiles (four
// pivots at a time, about 3.3 k cycles per tile) and, in the first columns of
// a large window, by the updates' matrix instructions.  A pivot that is not
// positive and finite marks the window failed (dp = 0, lm.fail = 1), as the
// tiled path does.
// Measured (rocprofv3, average per launch): one 30-camera window 82 -> 48 us, one
// 8-camera window 16.4 -> 13.5, 24 windows 80 -> 47, 512 windows 84 -> 51,
// against a right-looking form in 6x6 blocks on the vector units, one wave
// factoring a block column per barrier.  Of the 120 k cycles of a 28-camera
// window the load takes 32 k (one round trip to memory a chunk of the rows), the
// eleven columns 60 k, the backward step 13 k.
constexpr int kBS = 37;  // stride of a 6x6 block in LDS (k_chol_blocks)
constexpr int kSmallThreads = 512;
constexpr int kSmallWaves = kSmallThreads / kWave;

// Lower-triangular 6x6 Cholesky and inverse of the block at a (row-major 6x6,
// lower part read), result L written back to a (lower part) and M = L^-1 to m
// (full 6x6, upper part zero); y <- M y.  Returns false on a bad pivot.
__device__ __forceinline__ bool diag_factor(double* a, double* m, double* y) {
    double l[6][6], inv[6];
    bool ok_all = true;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        double d = a[6 * j + j];
#pragma unroll
        for (int k = 0; k < j; ++k) d -= l[j][k] * l[j][k];
        const bool ok = (d > 0.0) && isfinite(d);
        ok_all = ok_all && ok;
        d = ok ? d : 1.0;
        double r = __builtin_amdgcn_rsq(d);
        r = r * (1.5 - 0.5 * d * r * r);
        r = r * (1.5 - 0.5 * d * r * r);
        l[j][j] = d * r;
        inv[j] = r;
#pragma unroll
        for (int i = j + 1; i < 6; ++i) {
            double v = a[6 * i + j];
#pragma unroll
            for (int k = 0; k < j; ++k) v -= l[i][k] * l[j][k];
            l[i][j] = v * r;
        }
    }
    double M[6][6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
#pragma unroll
        for (int i = 0; i < 6; ++i) M[i][j] = 0.0;
        M[j][j] = inv[j];
#pragma unroll
        for (int i = j + 1; i < 6; ++i) {
            double v = 0.0;
#pragma unroll
            for (int k = j; k < i; ++k) v += l[i][k] * M[k][j];
            M[i][j] = -v * inv[i];
        }
    }
    double yn[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k <= i; ++k) v += M[i][k] * y[k];
        yn[i] = v;
    }
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        y[i] = yn[i];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            if (j <= i) a[6 * i + j] = l[i][j];
            m[6 * i + j] = M[i][j];
        }
    }
    return ok_all;
}

// LDS of one window's system: n rows of the matrix and the right-hand side as
// row n, in tiles of the lower triangle row by row, the last tile row with
// only the rows it has; then the reciprocal pivots, the solution and a row of
// 16 per wave.  Tile rows are 17 doubles apart: 16 lanes reading one row or
// one column touch 16 bank pairs, and an element's offset stays linear in its
// indices, so a lane keeps one offset per operand layout and the four elements
// are immediate offsets (with an exclusive-or swizzle instead, the address
// arithmetic cost more than the products).  The last tile row is read as if it
// had 16 rows: what lies behind it belongs to the same buffer, and results of
// those rows are never stored.
constexpr int kTileStride = 17;
constexpr int kTileSize = 16 * kTileStride;
struct WinTiles {
    int nt, nc, last, tail;        // tile rows, tile columns, rows of the last tile row, columns of the last tile column
    int dinv, x, xw, total;        // offsets in doubles
    __host__ __device__ explicit WinTiles(int n) {
        nt = (n >> 4) + 1;
        nc = (n + 15) >> 4;
        last = (n & 15) + 1;
        tail = n - 16 * (nc - 1);
        dinv = kTileSize * (nt * (nt - 1) / 2) + kTileStride * last * nc;
        dinv += dinv & 1;
        x = dinv + 16 * nc;
        xw = x + 16 * nc;
        total = xw + 16 * kSmallWaves + kTileSize;  // a whole tile may be read from the last one's place
    }
    __device__ __forceinline__ int tile(int i, int j) const {
        return (kTileSize / 2) * (i * (i + 1)) + (i == nt - 1 ? kTileStride * last : kTileSize) * j;
    }
};

// One S row f of the window, by one wave.  Lanes 0..53 take three slots of 18
// 16-byte pairs at a time, so a lane's entry (i, c), (i, c + 1) of the 6x6
// block is the same in every step; lanes 54..56 take the three pairs of the
// right-hand side's coefficient in the first.  NP = steps for the row's slots.
struct SRow {
    int lf, ns, nch, cols;  // row, slots, chunks; lane s: window camera of slot s
    const double* item;     // partial sums of its first chunk; the chunks lie 36 ns + 6 apart
};

template <int NP>
__device__ __forceinline__ void row_load(double2 v[NP], const SRow& r, int ch, int lane) {
    const double2* p = reinterpret_cast<const double2*>(r.item + (size_t)ch * (36 * r.ns + 6));
    const int i0 = lane < 54 ? lane : 18 * r.ns + min(lane - 54, 2), end = 18 * r.ns + 2;
    const int step = lane < 54 ? 54 : 0;
#pragma unroll
    for (int u = 0; u < NP; ++u) v[u] = p[min(i0 + step * u, end)];
}

// This lane's two values of the row's Hpp (packed) and b: of its entries of
// the diagonal block, or of its pair of the coefficient.
__device__ __forceinline__ double2 row_h(const double* __restrict__ hc, int lane) {
    const int i = lane / 3, c = 2 * (lane - 3 * i);
    const int e = lane < 18 ? sym6(i, c) : 21 + 2 * min(max(lane - 54, 0), 2);
    return double2{hc[e], hc[lane < 18 ? sym6(i, c + 1) : e + 1]};
}

template <int NP>
__device__ __forceinline__ void row_add(double2 v[NP], const double2 x[NP]) {
#pragma unroll
    for (int u = 0; u < NP; ++u) {
        v[u].x += x[u].x;
        v[u].y += x[u].y;
    }
}

// The row's entries of the system's lower triangle from its sums: S_ff = Hpp +
// lambda I - sum on the diagonal block (slot 0), S_gf = -sum^T below it, g_f =
// b_f - coefficient in row n.  rowat[3 g + c / 2]: byte offset of row 6 g + c
// of the system in its first tile, the top bit set in the last tile row (whose
// tiles are shorter) and kNoRow for the slots that are not stored here: three
// integer operations a pair find its place, where a closed form took thirty.
constexpr unsigned kNoRow = 0x40000000u;

template <int NP>
__device__ __forceinline__ void row_store(const double2 v[NP], const SRow& r, double2 hh, double lambda,
                                          const WinTiles& L, double* sm, const unsigned* rowat, int n, int lane) {
    const int so = lane / 18, pr = lane - 18 * so;
    const int i = pr / 3, c = 2 * (pr - 3 * i);
    const int C = 6 * r.lf + i, ic = C >> 4, cc = C & 15;
    const bool diag = lane < 18;
    if (diag || (lane >= 54 && lane < 57)) {
        // two neighbours (row, D), (row, D + 1), D even: of the diagonal block, or of row n
        const int row = diag ? C : n, D = 6 * r.lf + (diag ? c : 2 * (lane - 54)), ir = row >> 4;
        const int T = (kTileSize / 2) * (ir * (ir + 1)) + (ir == L.nt - 1 ? kTileStride * L.last : kTileSize) * (D >> 4);
        double* d = sm + T + kTileStride * (row & 15) + (D & 15);
        if (row >= D) d[0] = hh.x + (row == D ? lambda : 0.0) - v[0].x;
        if (row > D) d[1] = hh.y + (row == D + 1 ? lambda : 0.0) - v[0].y;
    }
    const unsigned full = 8u * (kTileSize * ic + cc), cut = 8u * (kTileStride * L.last * ic + cc) - 0x80000000u;
    const unsigned spare = 8u * L.xw;  // where the pairs that are not stored go
    // lane s: the byte offset in rowat of slot s's camera; lanes without a slot, and
    // slot 0, name the camera past the last one, whose rows are not stored
    const int g = 12 * ((lane > 0 && lane < r.ns) ? r.cols : kSmallMaxN / 6);
    const int from = 4 * (lane < 54 ? so : kSmallMaxN / 6), half = 2 * c;
    const char* at0 = reinterpret_cast<const char*>(rowat);
#pragma unroll
    for (int u = 0; u < NP; ++u) {
        const unsigned at = *reinterpret_cast<const unsigned*>(at0 + (__builtin_amdgcn_ds_bpermute(from + 12 * u, g) + half));
        const unsigned o = min(at + ((int)at < 0 ? cut : full), spare);
        double* d = reinterpret_cast<double*>(reinterpret_cast<char*>(sm) + o);
        d[0] = -v[u].x;
        d[kTileStride] = -v[u].y;  // the row is even: the next one is in the tile
    }
}

__global__ __launch_bounds__(kSmallThreads) void k_chol_small(DevProblem P, const double* __restrict__ spart,
                                                              const double* __restrict__ Hc,
                                                              double* __restrict__ dp, LMDev* lm,
                                                              const PoseQT* __restrict__ pose, PoseQT* __restrict__ pn,
                                                              CamRT* __restrict__ cn, double* __restrict__ red_scale) {
    static_assert(kSmallMaxN <= 180, "four S rows per wave, of at most 30, 22, 14 and 6 slots");
    extern __shared__ __align__(16) double sm[];
    __shared__ double ssum[kSmallWaves];
    __shared__ unsigned rowat[3 * (kSmallMaxN / 6 + 1)];
    __shared__ int bad;
    const int win = P.win_chol_order[blockIdx.x];
    if (!running(lm, win)) return;
    const int fc0 = P.win_fc0[win];
    const int nb = P.win_fc0[win + 1] - fc0;
    const int n = 6 * nb;
    const WinTiles L(n);
    const int g0 = 6 * fc0;
    const int tid = threadIdx.x;
    const int lane = tid & 63, i16 = lane & 15, k4 = lane >> 4;
    const int wid = wave_id();
    const double lambda = lm[win].lambda;
    const int fail0 = lm[win].fail;
    const int cam0 = P.win_cam0[win], cam1 = P.win_cam0[win + 1];
    CamIn cin;  // the inputs of this thread's first camera, loaded while the system is solved
    if (nb > 0) {
    // ---- the system, summed from the Schur rows' partials.  A row of at most 30
    // slots is one column group, whose chunk items lie back to back (36 doubles
    // per slot, then 6).  Wave w takes the rows w, 15 - w, 16 + w and 31 - w
    // (about the same number of slots for every wave), all four rows' first
    // chunks in flight at once.  Blocks without co-visibility stay zero.
    SRow row[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int lf = q == 0 ? wid : q == 1 ? 15 - wid : q == 2 ? 16 + wid : 31 - wid;
        row[q] = SRow{lf, 0, 0, 0, spart};
        if (lf < nb) {
            const int f = fc0 + lf;
            const int c0 = P.colptr[f];
            row[q].ns = P.colptr[f + 1] - c0;
            row[q].nch = P.row_nchunks[f];
            row[q].item = spart + P.row_pofs0[f];
            if (lane < row[q].ns) row[q].cols = P.colcam[c0 + lane] - fc0;
        }
    }
    auto clear = [&]() {  // while the loads are in flight
        double2* z = reinterpret_cast<double2*>(sm);
        for (int q = tid; q < L.total / 2; q += kSmallThreads) z[q] = double2{0.0, 0.0};
        if (tid < 3 * (kSmallMaxN / 6 + 1)) {
            const int R = 2 * tid, ir = R >> 4;  // row 6 g + c = 2 (3 g + c / 2)
            const unsigned o = 8u * ((kTileSize / 2) * ir * (ir + 1) + kTileStride * (R & 15));
            rowat[tid] = R < n ? o | (ir == L.nt - 1 ? 0x80000000u : 0u) : kNoRow;
        }
        if (tid == 0) bad = 0;
        __syncthreads();
    };
    const double* hc = Hc + 28 * (size_t)fc0;
    if (nb <= kSmallWaves) {
        // one row of at most eight slots per wave: its chunks six at a time
        constexpr int kCh = 6;
        double2 v[3], x[kCh][3], h0;
        if (row[0].ns) {
            h0 = row_h(hc + 28 * row[0].lf, lane);
            row_load<3>(v, row[0], 0, lane);
#pragma unroll
            for (int u = 0; u < kCh; ++u) row_load<3>(x[u], row[0], min(1 + u, row[0].nch - 1), lane);
        }
        clear();
        if (row[0].ns) {
            for (int ch = 1; ch < row[0].nch; ch += kCh) {
#pragma unroll
                for (int u = 0; u < kCh; ++u)
                    if (ch + u < row[0].nch) row_add<3>(v, x[u]);
                if (ch + kCh < row[0].nch)
#pragma unroll
                    for (int u = 0; u < kCh; ++u) row_load<3>(x[u], row[0], min(ch + kCh + u, row[0].nch - 1), lane);
            }
            row_store<3>(v, row[0], h0, lambda, L, sm, rowat, n, lane);
        }
    } else {
        double2 v0[10], v1[8], v2[5], v3[2], h[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) h[q] = row_h(hc + 28 * min(row[q].lf, nb - 1), lane);
        row_load<10>(v0, row[0], 0, lane);  // nb > 8: every wave has this row
        if (row[1].ns) row_load<8>(v1, row[1], 0, lane);
        if (row[2].ns) row_load<5>(v2, row[2], 0, lane);
        if (row[3].ns) row_load<2>(v3, row[3], 0, lane);
        clear();
        const int most = max(max(row[0].nch, row[1].nch), max(row[2].nch, row[3].nch));
        for (int ch = 1; ch < most; ++ch) {
            {
                double2 x0[10];
                if (ch < row[0].nch) {
                    row_load<10>(x0, row[0], ch, lane);
                    row_add<10>(v0, x0);
                }
            }
            double2 x1[8], x2[5], x3[2];
            if (ch < row[1].nch) row_load<8>(x1, row[1], ch, lane);
            if (ch < row[2].nch) row_load<5>(x2, row[2], ch, lane);
            if (ch < row[3].nch) row_load<2>(x3, row[3], ch, lane);
            if (ch < row[1].nch) row_add<8>(v1, x1);
            if (ch < row[2].nch) row_add<5>(v2, x2);
            if (ch < row[3].nch) row_add<2>(v3, x3);
        }
        row_store<10>(v0, row[0], h[0], lambda, L, sm, rowat, n, lane);
        if (row[1].ns) row_store<8>(v1, row[1], h[1], lambda, L, sm, rowat, n, lane);
        if (row[2].ns) row_store<5>(v2, row[2], h[2], lambda, L, sm, rowat, n, lane);
        if (row[3].ns) row_store<2>(v3, row[3], h[3], lambda, L, sm, rowat, n, lane);
    }
    __syncthreads();
    // the diagonal tiles' upper halves
    for (int d = wid; d < L.nc; d += kSmallWaves) {
        double* T = sm + L.tile(d, d);
        const int rows = d == L.nc - 1 ? L.tail : 16;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int r = 4 * v + k4;
            if (r > i16 && r < rows) T[kTileStride * i16 + r] = T[kTileStride * r + i16];
        }
    }
    __syncthreads();
    // ---- factorisation and forward step
    double* dinv = sm + L.dinv;
    double* x = sm + L.x;
    const int nt = L.nt, nc = L.nc, last = L.last;
    const bool split = nt > nc;  // the right-hand side has a tile row of its own
    // this lane's places in a tile: operand element (i, 4t + k) at oop + 4t,
    // result element (4v + k, i) at ores + 4v rows
    const int oop = kTileStride * i16 + k4, ores = kTileStride * k4 + i16;
    constexpr int kV = 4 * kTileStride;
    // a tile row's result; the last one has fewer rows
    auto put = [&](double* T, const dbl4& r, bool full) {
        if (full) {
#pragma unroll
            for (int v = 0; v < 4; ++v) T[v * kV] = r[v];
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (4 * v + k4 < last) T[v * kV] = r[v];
        }
    };
    // wave 0's part of column k: the diagonal tile (updated by column k - 1),
    // its factor and inverse; M_k takes the tile's place
    auto chain = [&](int k) {
        double* T = sm + L.tile(k, k) + ores;
        dbl4 acc, Z;
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] = T[v * kV];
        if (k > 0) {
            const double* w = sm + L.tile(k, k - 1) + oop;
            const double* d = dinv + 16 * (k - 1) + k4;
            double wv[4], dk[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                wv[t] = w[4 * t];
                dk[t] = d[4 * t];
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) acc = mfma16x16x4(wv[t] * -dk[t], wv[t], acc);
        }
        const int rows = k == nc - 1 ? L.tail : 16;
        if (rows < 16) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 4 * v + k4;
                if (r == rows) T[v * kV] = acc[v];  // the right-hand side's row
                acc[v] = (r < rows && i16 < rows) ? acc[v] : (r == i16 ? 1.0 : 0.0);  // identity past the end
            }
        }
        double dv[4];
        if (!tile16_ldl(acc, Z, dv) && lane == 0) bad = 1;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (4 * v + k4 < rows) T[v * kV] = Z[v];
            if (i16 == 0) dinv[16 * k + 4 * v + k4] = dv[v];
        }
    };
    if (wid == 0) chain(0);
    __syncthreads();
    for (int k = 0; k < nc; ++k) {
        // solve: W_ik = A_ik M_k^T in place for the tile rows i > k
        if (k + 1 + wid < nt) {
            double m[4];
            const double* M = sm + L.tile(k, k) + oop;
#pragma unroll
            for (int t = 0; t < 4; ++t) m[t] = M[4 * t];
            for (int i = k + 1 + wid; i < nt; i += kSmallWaves) {
                double* A = sm + L.tile(i, k);
                double a[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) a[t] = A[oop + 4 * t];
                dbl4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int t = 0; t < 4; ++t) acc = mfma16x16x4(a[t], m[t], acc);
                wave_sync();
                put(A + ores, acc, i < nt - 1);
            }
        }
        __syncthreads();
        if (k + 1 >= nc) break;
        if (wid == 0) {
            __builtin_amdgcn_s_setprio(3);
            chain(k + 1);
            __builtin_amdgcn_s_setprio(0);
        } else {
            // update of the tiles (i, j), k < j <= i, beyond the chain's: whole tile
            // rows, the longest first, wave w the rows nt - w and nt - 15 + w; two
            // tiles at a time
            double dk[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) dk[t] = -dinv[16 * k + 4 * t + k4];
#pragma unroll 1
            for (int h = 0; h < 2; ++h) {
                const int i = h ? nt - 15 + wid : nt - wid;
                if (i < k + 2) continue;
                const bool full = i < nt - 1;
                const int jend = min(i, nc - 1), step = full ? kTileSize : kTileStride * last;
                double a[4];
                const double* W = sm + L.tile(i, k) + oop;
                double* C = sm + L.tile(i, k + 1) + ores;
#pragma unroll
                for (int t = 0; t < 4; ++t) a[t] = W[4 * t] * dk[t];
                int j = k + 1;
                for (; j < jend; j += 2) {
                    const double* B0 = sm + L.tile(j, k) + oop;
                    const double* B1 = sm + L.tile(j + 1, k) + oop;
                    double b0[4], b1[4];
                    dbl4 c0, c1;
#pragma unroll
                    for (int t = 0; t < 4; ++t) b0[t] = B0[4 * t];
#pragma unroll
                    for (int v = 0; v < 4; ++v) c0[v] = C[v * kV];
#pragma unroll
                    for (int t = 0; t < 4; ++t) b1[t] = B1[4 * t];
#pragma unroll
                    for (int v = 0; v < 4; ++v) c1[v] = C[step + v * kV];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        c0 = mfma16x16x4(a[t], b0[t], c0);
                        c1 = mfma16x16x4(a[t], b1[t], c1);
                    }
                    put(C, c0, full);
                    put(C + step, c1, full);
                    C += 2 * step;
                }
                if (j == jend) {
                    const double* B0 = sm + L.tile(j, k) + oop;
                    double b0[4];
                    dbl4 c0;
#pragma unroll
                    for (int t = 0; t < 4; ++t) b0[t] = B0[4 * t];
#pragma unroll
                    for (int v = 0; v < 4; ++v) c0[v] = C[v * kV];
#pragma unroll
                    for (int t = 0; t < 4; ++t) c0 = mfma16x16x4(a[t], b0[t], c0);
                    put(C, c0, full);
                }
            }
        }
        __syncthreads();
    }
    if (cam0 + tid < cam1) cin = camera_inputs(P, pose, Hc, cam0 + tid);
    if (bad) {
        for (int q = tid; q < n; q += kSmallThreads) dp[g0 + q] = 0.0;
        if (tid == 0) lm[win].fail = 1;
    } else {
        // ---- backward step.  The solved right-hand side z = D^-1 of row n; its part
        // in the last diagonal tile (whose inverse lies above it) is solved here.
        const double* yrow = sm + L.tile(nt - 1, 0) + kTileStride * (last - 1);
        const int ystep = kTileStride * last;
        for (int q = tid; q < 16 * (split ? nc : nc - 1); q += kSmallThreads)
            x[q] = yrow[(q >> 4) * ystep + (q & 15)] * dinv[q];
        if (!split && wid == kSmallWaves - 1) {
            const double* M = sm + L.tile(nc - 1, nc - 1) + oop;
            const double* y = yrow + (nc - 1) * ystep + k4;
            double p = 0.0;
#pragma unroll
            for (int t = 0; t < 4; ++t) p = fma(M[4 * t], 4 * t + k4 < L.tail ? y[4 * t] : 0.0, p);
            p = sum_over_k(p);
            if (k4 == 0) x[16 * (nc - 1) + i16] = i16 < L.tail ? p * dinv[16 * (nc - 1) + i16] : 0.0;
        }
        __syncthreads();
        // Every wave forms x_k = M_k^T s_k (the same values) and then updates its
        // share to the left, s_j -= D_j^-1 W_kj^T x_k: four products per lane, summed
        // over the lanes of a column.  At most two tiles a wave; everything but s_k is
        // loaded ahead of x_k.
        static_assert(kSmallMaxN <= 16 * (2 * kSmallWaves + 1), "two tiles to the left per wave");
        double* xk = sm + L.xw + 16 * wid;
        double m[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) m[t] = 4 * t + k4 < L.tail ? sm[L.tile(nc - 1, nc - 1) + ores + t * kV] : 0.0;
        for (int k = nc - 1; k >= 0; --k) {
            const int rows = k == nc - 1 ? L.tail : 16;
            double s4[4], w[2][4], xd[2], dd[2];
#pragma unroll
            for (int t = 0; t < 4; ++t) s4[t] = x[16 * k + 4 * t + k4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int j = min(wid + kSmallWaves * h, k);
                const double* W = sm + L.tile(k, j) + ores;
#pragma unroll
                for (int t = 0; t < 4; ++t) w[h][t] = 4 * t + k4 < rows ? W[t * kV] : 0.0;
                xd[h] = x[16 * j + i16];
                dd[h] = dinv[16 * j + i16];
            }
            double p = sum_over_k(fma(s4[0], m[0], s4[1] * m[1]) + fma(s4[2], m[2], s4[3] * m[3]));
            p = i16 < rows ? p : 0.0;
            if (k4 == 0) xk[i16] = p;
            if (k > 0) {  // the next step's inverse
                const double* M = sm + L.tile(k - 1, k - 1) + ores;
#pragma unroll
                for (int t = 0; t < 4; ++t) m[t] = M[t * kV];
            }
            wave_sync();
            double xs[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) xs[t] = xk[4 * t + k4];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int j = wid + kSmallWaves * h;
                if (j >= k) continue;
                const double u = sum_over_k(fma(xs[0], w[h][0], xs[1] * w[h][1]) + fma(xs[2], w[h][2], xs[3] * w[h][3]));
                if (k4 == 0) x[16 * j + i16] = fma(-u, dd[h], xd[h]);
            }
            __syncthreads();  // s_k has been read by every wave, s_j (j < k) updated
            if (wid == 0 && k4 == 0 && i16 < rows) {
                x[16 * k + i16] = p;
                dp[g0 + 16 * k + i16] = p;
            }
        }
    }
    } else if (cam0 + tid < cam1) {
        cin = camera_inputs(P, pose, Hc, cam0 + tid);
    }
    __syncthreads();
    // candidate poses of the window's cameras from the step in LDS, and their
    // part of x'(lambda x + b): the camera update (k_update_cam), with the same
    // threads and the same sum
    const int fail = (nb > 0 && bad) ? 1 : fail0;
    double sc = 0.0;
    if (tid < 256)
        for (int c = cam0 + tid; c < cam1; c += 256)
            sc += camera_candidate(c == cam0 + tid ? cin : camera_inputs(P, pose, Hc, c), lambda, fail, c,
                                   [&](int f, int i) { return sm[L.x + 6 * (f - fc0) + i]; }, pn, cn);
    const double s = block_sum<double, 256>(sc, ssum);
    if (tid == 0) red_scale[win] = s;
}

size_t cholesky_small_smem(const DevProblem& P) {
    return sizeof(double) * (size_t)WinTiles(std::max(6 * P.max_win_fc, 6)).total;
}

// One workgroup per window, largest windows first: with the largest window's
// LDS a CU may hold one workgroup, and the small windows then fill in behind
// the large ones (P.win_chol_order).
void launch_cholesky_small(const DevProblem& P, const DevState& cur, const DevState& cand, const DevWork& W,
                           hipStream_t st) {
    hipLaunchKernelGGL(k_chol_small, dim3(P.n_win), dim3(kSmallThreads), cholesky_small_smem(P), st, P,
                       (const double*)W.spart, (const double*)W.Hc, W.dp, W.lm, (const PoseQT*)cur.pose, cand.pose,
                       cand.cam, W.red_scale);
}

int prepare_cholesky_small(const DevProblem& P) {
    const size_t smem = cholesky_small_smem(P);
    if (smem > 160 * 1024) return -1;
    return hipFuncSetAttribute((const void*)k_chol_small, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) ==
                   hipSuccess ? 0 : -1;
}

// ---------------------------------------------------------------- one mid-size problem, on request
// One workgroup (512 threads) factors the whole system in 6x6 camera blocks,
// the per-window algorithm with the matrix in global memory (it stays
// in the L2 of the CU's XCD: 490 KB at 58 free cameras).  The lower block
// triangle is packed column by column (block (I, J), J <= I, at
// J nb - J(J-1)/2 + (I - J)) and entry-major (entry e of block b at
// e * nblk + b), so the threads of a trailing update, which own consecutive
// blocks, read and write consecutive addresses.  The panel column of the
// current step is staged in LDS.  One CU runs the whole chain of nb block
// steps through L2 (3.5 us per step at 11 free cameras, against 530 us in all
// at 58 and 349 us for the tiles there), so the per-window kernel in LDS
// replaced it for small systems; it stays as a switch for tests and sizes
// between 31 and 128 free cameras.
__device__ __forceinline__ int colstart(int J, int nb) { return J * nb - J * (J - 1) / 2; }

// (I, J) of packed block b; J found from the column starts
__device__ __forceinline__ void block_ij(int b, int nb, int& I, int& J) {
    const double B = 2.0 * nb + 1.0;
    int j = (int)((B - sqrt(B * B - 8.0 * b)) * 0.5);
    if (j < 0) j = 0;
    while (j > 0 && colstart(j, nb) > b) --j;
    while (j + 1 < nb && colstart(j + 1, nb) <= b) ++j;
    J = j;
    I = j + (b - colstart(j, nb));
}

__global__ __launch_bounds__(kSmallThreads) void k_chol_blocks(const double* __restrict__ S, int lda, int nb,
                                                               const double* __restrict__ g,
                                                               double* __restrict__ Lg, double* __restrict__ dp,
                                                               LMDev* lm) {
    extern __shared__ double sm[];
    __shared__ double xk[6];
    __shared__ int bad;
    if (lm->phase == kPhaseDone) return;
    const int n = 6 * nb;
    const int nblk = nb * (nb + 1) / 2;
    double* Pn = sm;                                      // (nb - 1) * kBS: panel column L_IK, I > K
    double* Mb = sm + (size_t)(nb > 1 ? nb - 1 : 1) * kBS;  // nb * kBS: M_K = L_KK^-1
    double* yv = Mb + (size_t)nb * kBS;                   // n
    double* dg = yv + n;                                  // kBS: diagonal block being factored
    const int tid = threadIdx.x;
    for (int idx = tid; idx < nblk * 36; idx += kSmallThreads) {
        const int b = idx / 36, e = idx - 36 * (idx / 36);
        int I, J;
        block_ij(b, nb, I, J);
        const int r = e / 6, c = e - 6 * (e / 6);
        Lg[(size_t)e * nblk + b] = S[(size_t)(6 * I + r) * lda + 6 * J + c];
    }
    for (int i = tid; i < n; i += kSmallThreads) yv[i] = g[i];
    if (tid == 0) bad = 0;
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int e = 0; e < 36; ++e) dg[e] = Lg[(size_t)e * nblk];
        if (!diag_factor(dg, Mb, yv)) bad = 1;
#pragma unroll
        for (int e = 0; e < 36; ++e) Lg[(size_t)e * nblk] = dg[e];
    }
    __syncthreads();
    for (int K = 0; K < nb; ++K) {
        // panel: L_IK = A_IK M_K^T into Lg and LDS, y_I -= L_IK y_K
        const int rows = 6 * (nb - K - 1);
        const double* M = Mb + K * kBS;
        const int cK = colstart(K, nb);
        for (int t = tid; t < rows; t += kSmallThreads) {
            const int I = K + 1 + t / 6, r = t - 6 * (t / 6);
            const int bIK = cK + (I - K);
            double a[6], o[6];
#pragma unroll
            for (int c = 0; c < 6; ++c) a[c] = Lg[(size_t)(6 * r + c) * nblk + bIK];
            double yr = 0.0;
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                double v = 0.0;
#pragma unroll
                for (int m = 0; m <= c; ++m) v += a[m] * M[6 * c + m];
                o[c] = v;
                yr += v * yv[6 * K + c];
            }
            double* prow = Pn + (I - K - 1) * kBS + 6 * r;
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                Lg[(size_t)(6 * r + c) * nblk + bIK] = o[c];
                prow[c] = o[c];
            }
            yv[6 * I + r] -= yr;
        }
        __syncthreads();
        // trailing update: the trailing blocks are the packed tail from column K+1
        const int rem = nb - K - 1;
        const int nupd = rem * (rem + 1) / 2;
        const int base = K + 1 < nb ? colstart(K + 1, nb) : 0;
        for (int q = tid; q < nupd; q += kSmallThreads) {
            int I, J;
            block_ij(base + q, nb, I, J);
            const double* A = Pn + (I - K - 1) * kBS;
            const double* B = Pn + (J - K - 1) * kBS;
            double acc[36];
#pragma unroll
            for (int e = 0; e < 36; ++e) acc[e] = Lg[(size_t)e * nblk + base + q];
            double bm[36];
#pragma unroll
            for (int e = 0; e < 36; ++e) bm[e] = B[e];
#pragma unroll
            for (int r = 0; r < 6; ++r) {
                double ar[6];
#pragma unroll
                for (int m = 0; m < 6; ++m) ar[m] = A[6 * r + m];
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    double v = acc[6 * r + c];
#pragma unroll
                    for (int m = 0; m < 6; ++m) v -= ar[m] * bm[6 * c + m];
                    acc[6 * r + c] = v;
                }
            }
            if (q == 0) {  // block (K+1, K+1): factor it now, through LDS
#pragma unroll
                for (int e = 0; e < 36; ++e) dg[e] = acc[e];
            } else {
#pragma unroll
                for (int e = 0; e < 36; ++e) Lg[(size_t)e * nblk + base + q] = acc[e];
            }
        }
        if (tid == 0 && nupd > 0) {
            const int J = K + 1;
            double yk[6];
#pragma unroll
            for (int i = 0; i < 6; ++i) yk[i] = yv[6 * J + i];
            if (!diag_factor(dg, Mb + J * kBS, yk)) bad = 1;
#pragma unroll
            for (int i = 0; i < 6; ++i) yv[6 * J + i] = yk[i];
#pragma unroll
            for (int e = 0; e < 36; ++e) Lg[(size_t)e * nblk + base] = dg[e];
        }
        __syncthreads();
    }
    if (bad) {
        for (int i = tid; i < n; i += kSmallThreads) dp[i] = 0.0;
        if (tid == 0) lm->fail = 1;
        return;
    }
    for (int K = nb - 1; K >= 0; --K) {
        if (tid < 6) {
            const double* M = Mb + K * kBS;
            double v = 0.0;
            for (int m = tid; m < 6; ++m) v += M[6 * m + tid] * yv[6 * K + m];
            xk[tid] = v;
        }
        __syncthreads();
        if (tid < 6) {
            yv[6 * K + tid] = xk[tid];
            dp[6 * K + tid] = xk[tid];
        }
        for (int t = tid; t < 6 * K; t += kSmallThreads) {
            const int J = t / 6, c = t - 6 * (t / 6);
            const int bKJ = colstart(J, nb) + (K - J);
            double v = 0.0;
#pragma unroll
            for (int r = 0; r < 6; ++r) v += Lg[(size_t)(6 * r + c) * nblk + bKJ] * xk[r];
            yv[t] -= v;
        }
        __syncthreads();
    }
}

size_t cholesky_blocks_smem(int nb) {
    return sizeof(double) * ((size_t)(nb > 1 ? nb - 1 : 1) * kBS + (size_t)nb * kBS + 6 * (size_t)nb + kBS);
}

int prepare_cholesky(const DevProblem& P) {
    if (!P.use_blocks) {
        // the tiled path's backward step holds the right-hand sides in LDS
        const size_t smem = sizeof(double) * (size_t)std::max(P.n_pad, 64);
        if (smem + 9 * 1024 > 160 * 1024) return -1;
        const void* kerns[] = {(const void*)k_chol_back<1>, (const void*)k_chol_back<2>, (const void*)k_chol_back<3>,
                               (const void*)k_chol_back<4>, (const void*)k_chol_back<kBackPassMax>};
        for (const void* kf : kerns)
            if (hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) return -1;
        return 0;
    }
    const size_t smem = cholesky_blocks_smem(P.n_fc);
    if (smem > 160 * 1024) return -1;
    return hipFuncSetAttribute((const void*)k_chol_blocks, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) ==
                   hipSuccess ? 0 : -1;
}

void launch_cholesky_solve(const DevProblem& P, const DevState& cur, const DevState& cand, const DevWork& W,
                           hipStream_t st) {
    if (P.n_fc == 0) return;
    const int nt = P.nt, lda = P.n_pad;
    if (P.use_blocks) {
        hipLaunchKernelGGL(k_chol_blocks, dim3(1), dim3(kSmallThreads), cholesky_blocks_smem(P.n_fc), st,
                           (const double*)W.S, lda, P.n_fc, (const double*)W.g, W.Lm, W.dp, W.lm);
        return;
    }
    hipLaunchKernelGGL(k_chol_first, dim3(1), dim3(256), 0, st, (const double*)W.S, W.Li, lda, P.n,
                       (const double*)W.g, W.y, W.lm);
    for (int k = 0; k + 1 < nt; ++k) {
        const int rem = nt - k - 1;
        hipLaunchKernelGGL(k_chol_step, dim3(rem * (rem + 1) / 2), dim3(256), 0, st, W.S, W.Lm, W.Li, lda, P.n, k,
                           (const double*)W.g, W.y, W.fsum, W.lm);
    }
    if (nt <= kBackSingleMax) {
        const int np = std::max(1, (64 * (nt - 1) + 127) / 128);
        auto kern = np == 1 ? k_chol_back<1> : np == 2 ? k_chol_back<2> : np == 3 ? k_chol_back<3>
                  : np == 4 ? k_chol_back<4> : k_chol_back<kBackPassMax>;
        hipLaunchKernelGGL(kern, dim3(1), dim3(kBackThreads), sizeof(double) * (size_t)lda, st, P,
                           (const double*)W.Lm, (const double*)W.Li, lda, nt, (const double*)W.y, W.dp,
                           (const LMDev*)W.lm, (const PoseQT*)cur.pose, (const double*)W.Hc, cand.pose, cand.cam,
                           W.red_scale);
    } else {
        for (int k1 = nt - 1; k1 >= 0; k1 -= kBackGroup) {
            const int cnt = std::min(kBackGroup, k1 + 1);
            hipLaunchKernelGGL(k_chol_back_group, dim3(k1 - cnt + 2), dim3(kBackThreads), 0, st, (const double*)W.Lm,
                               (const double*)W.Li, lda, nt, k1, cnt, W.y, W.dp, (const LMDev*)W.lm);
        }
    }
}

}  // namespace navba
