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
// The tile products run on FP64 MFMA (v_mfma_f64_16x16x4); the chain through
// the pivots runs in registers.  The backward step is a single launch.
#include "ba_kernels.h"

namespace navba {

typedef double TileLds[64][65];

// A 64x64 tile through registers, 16 elements per thread: fetch issues the
// global loads, put writes LDS (several fetches can be in flight before the
// first put).
__device__ __forceinline__ void tile_fetch(double v[16], const double* __restrict__ src, int lda) {
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int idx = threadIdx.x + 256 * s;
        v[s] = src[(size_t)(idx >> 6) * lda + (idx & 63)];
    }
}

__device__ __forceinline__ void tile_put(TileLds& T, const double v[16]) {
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int idx = threadIdx.x + 256 * s;
        T[idx >> 6][idx & 63] = v[s];
    }
}

__device__ __forceinline__ void tile_load(TileLds& T, const double* __restrict__ src, int lda) {
    double v[16];
    tile_fetch(v, src, lda);
    tile_put(T, v);
}

__device__ __forceinline__ void tile_store(const TileLds& T, double* __restrict__ dst, int lda) {
    double v[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int idx = threadIdx.x + 256 * s;
        v[s] = T[idx >> 6][idx & 63];
    }
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int idx = threadIdx.x + 256 * s;
        dst[(size_t)(idx >> 6) * lda + (idx & 63)] = v[s];
    }
}

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

// M[C..C+15][C..C+15] = L^-1 of the 16x16 diagonal block of the factor in A
// (lower triangle, rpiv = 1 / diag), by one wave: its two 8x8 diagonal blocks
// by substitution (one lane per column), then M21 = -M22 (L21 M11) on FP64
// MFMA (8x8 products, zero padded to 16x16).  The block's upper right 8x8
// quarter is not written (it must already hold zeros).
__device__ __forceinline__ void wave_inv16(const TileLds& A, const double* rpiv, TileLds& M, int C) {
    const int lane = threadIdx.x & 63;
    const int r16 = lane & 15, kq = lane >> 4, r8 = lane & 7;
    const int R = C + 8;
    if (lane < 16) {
        const int b = C + 8 * (lane >> 3), j = lane & 7;
        double d[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) d[i] = (i == j) ? rpiv[b + j] : 0.0;
#pragma unroll
        for (int i = 1; i < 8; ++i) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < i; ++k) s += A[b + i][b + k] * d[k];  // d[k] = 0 for k < j
            if (i > j) d[i] = -s * rpiv[b + i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) M[b + i][b + j] = d[i];
    }
    wave_sync();
    // T = L21 M11 (8x8): rows i = 4v + kq < 8, columns r16 < 8 of the 16x16
    // product (operand rows and columns 8..15 zero; row 8 + r8 read instead)
    const bool in = r16 < 8;
    dbl4 t = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m0 = 0; m0 < 8; m0 += 4) {
        const double va = A[R + r8][C + m0 + kq], vb = M[C + m0 + kq][C + r16];
        t = mfma16x16x4(in ? va : 0.0, in ? vb : 0.0, t);
    }
    if (in) {
        M[R + kq][C + r16] = t[0];
        M[R + 4 + kq][C + r16] = t[1];
    }
    wave_sync();
    dbl4 u = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m0 = 0; m0 < 8; m0 += 4) {
        const double va = M[R + r8][R + m0 + kq], vb = M[R + m0 + kq][C + r16];
        u = mfma16x16x4(in ? va : 0.0, in ? vb : 0.0, u);
    }
    wave_sync();
    if (in) {
        M[R + kq][C + r16] = -u[0];
        M[R + 4 + kq][C + r16] = -u[1];
    }
    wave_sync();
}

// 16x16 block product of one wave, acc += X[xr.., xc..] Y[yr.., yc..]; the
// result's element v in lane (r16, kq) is row 4v + kq, column r16.
__device__ __forceinline__ dbl4 blk_mul(const TileLds& X, int xr, int xc, const TileLds& Y, int yr, int yc, dbl4 acc) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
    double a[4], b[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        a[kk] = X[xr + r16][xc + 4 * kk + kq];
        b[kk] = Y[yr + 4 * kk + kq][yc + r16];
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) acc = mfma16x16x4(a[kk], b[kk], acc);
    return acc;
}

// Block (r, c) of M (16x16) <- sign * acc, in the layout of blk_mul.
__device__ __forceinline__ void blk_put(TileLds& M, int r, int c, dbl4 acc, double sign) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
#pragma unroll
    for (int v = 0; v < 4; ++v) M[16 * r + 4 * v + kq][16 * c + r16] = sign * acc[v];
}

// Block (i, j) of the tile inverse, M_ij = -M_ii T_ij, where block (i, j) of M
// holds T_ij = sum_{j<=k<i} L_ik M_kj (one wave; in place).
__device__ __forceinline__ void blk_finish(TileLds& M, int i, int j) {
    const dbl4 z = {0.0, 0.0, 0.0, 0.0};
    const dbl4 t = blk_mul(M, 16 * i, 16 * i, M, 16 * i, 16 * j, z);
    wave_sync();
    blk_put(M, i, j, t, -1.0);
}

// Block (i, j) of M += L_ik M_kj (or = when first), one wave.
__device__ __forceinline__ void blk_term(const TileLds& A, TileLds& M, int i, int k, int j, bool first) {
    const int lane = threadIdx.x & 63, r16 = lane & 15, kq = lane >> 4;
    dbl4 acc = {0.0, 0.0, 0.0, 0.0};
    if (!first) {
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] = M[16 * i + 4 * v + kq][16 * j + r16];
    }
    acc = blk_mul(A, 16 * i, 16 * k, M, 16 * k, 16 * j, acc);
    wave_sync();
    blk_put(M, i, j, acc, 1.0);
}

// The value of v in lane l (l wave-uniform), as a uniform double.
__device__ __forceinline__ double lane_value(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffff), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// In-LDS Cholesky of the SPD tile A (64x64, 256 threads) and the inverse of
// its factor: the lower triangle of A becomes L, rpiv[j] = 1 / L_jj and
// M = L^-1 (upper triangle zero).  The strict upper triangle of A's four
// 16x16 diagonal blocks is left with scratch values, the rest of A's upper
// triangle is unchanged.  Wave w owns columns 16w..16w+15, lane l row l.
// Four stages, one barrier between stages; in stage s:
//   waves w >= s apply panel s-1 (final since the last barrier) to their
//     columns, rows 16w.., on FP64 MFMA (16x16 blocks, K = 16, in place);
//   wave s then factors its 16 columns in registers.  Pivot j: 1/sqrt(d_j)
//     by rsq and two Goldschmidt steps; the next pivot is formed from
//     wave-uniform values read before this pivot's column update,
//     d_{j+1} = a_{j+1,j+1} - (a_{j+1,j} / sqrt(d_j))^2, so that the chain
//     through the pivots holds no cross-lane step; columns j+1 and j+2 are
//     updated with uniform multipliers, the others with the scaled column
//     broadcast through `scratch` (16 x 64 doubles of LDS, not M);
//   wave s-1, whose panel is final, forms the inverse's block row s-1 in 16x16
//     blocks, M_ii = L_ii^-1 and M_ij = -M_ii T_ij, and adds its terms to
//     the sums T_mj = sum_{j<=k<m} L_mk M_kj of the rows below (kept in M's
//     blocks (m, j)); stage 0's idle waves clear M's upper triangle.
// After the last stage wave 3 forms block row 3.  A pivot that is not
// positive and finite is replaced by 1 (the values stay finite); the return
// value, the same in every thread, says whether one was.
__device__ __forceinline__ bool tile_potrf_inv(TileLds& A, double* rpiv, double* scratch, TileLds& M, int nst) {
    const int lane = threadIdx.x & 63, w = wave_id();
    const int r16 = lane & 15, kq = lane >> 4;
    const int c0 = 16 * w;
    double (*cb)[64] = reinterpret_cast<double (*)[64]>(scratch);
    bool bad = false;
    for (int s = 0; s < nst; ++s) {
        if (s == 0 && w > 0) {
            for (int idx = (int)threadIdx.x - 64; idx < 4096; idx += 192) {
                const int i = idx >> 6, j = idx & 63;
                if ((j >> 3) > (i >> 3)) M[i][j] = 0.0;
            }
        }
        if (s == 0 && w >= nst) {
            // identity padding rows (the last tile of the system): their part of
            // the factor is the identity already in A; M's rows are the identity
            for (int idx = lane; idx < 16 * 64; idx += kWave) {
                const int i = c0 + (idx >> 6), j = idx & 63;
                if ((j >> 3) <= (i >> 3)) M[i][j] = (i == j) ? 1.0 : 0.0;
            }
            if (lane < 16) rpiv[c0 + lane] = 1.0;
        }
        if (s > 0 && w == s - 1) {
            // block row s-1 of the inverse and its terms of the rows below
            wave_inv16(A, rpiv, M, 16 * w);
            for (int j = 0; j < w; ++j) blk_finish(M, w, j);
            for (int m = w + 1; m < nst; ++m)
                for (int j = 0; j <= w; ++j) blk_term(A, M, m, w, j, j == w);
        }
        if (s > 0 && w >= s && w < nst) {
            const int p = 16 * (s - 1);
            double bv[4], av[4][4];
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) bv[kk] = A[c0 + r16][p + 4 * kk + kq];
#pragma unroll
            for (int bi = 0; bi < 4; ++bi)
                if (bi >= w)
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) av[bi][kk] = A[16 * bi + r16][p + 4 * kk + kq];
#pragma unroll
            for (int bi = 0; bi < 4; ++bi) {
                if (bi >= w) {
                    dbl4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int kk = 0; kk < 4; ++kk) acc = mfma16x16x4(av[bi][kk], bv[kk], acc);
#pragma unroll
                    for (int v = 0; v < 4; ++v) A[16 * bi + 4 * v + kq][c0 + r16] -= acc[v];
                }
            }
        }
        if (w == s) {
            wave_sync();
            double x[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) x[c] = A[lane][c0 + c];
            double rp[16];
            double d = lane_value(x[0], c0);
            double a1 = lane_value(x[0], c0 + 1), a2 = lane_value(x[0], c0 + 2), ad = lane_value(x[1], c0 + 1);
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const bool ok = (d > 0.0) && isfinite(d);
                bad |= !ok;
                d = ok ? d : 1.0;
                double H = __builtin_amdgcn_rsq(d);
                double g = d * H;
#pragma unroll
                for (int it = 0; it < 2; ++it) {
                    const double e = fma(-g, H, 1.0);
                    const double gh = 0.5 * g, Hh = 0.5 * H;
                    g = fma(gh, e, g);
                    H = fma(Hh, e, H);
                }
                rp[j] = H;
                const double l1 = a1 * H, l2 = a2 * H;
                const double dn = fma(-l1, l1, ad);
                x[j] = (lane == c0 + j) ? g : x[j] * H;
                if (j + 3 < 16) cb[j][lane] = x[j];
                if (j + 1 < 16) x[j + 1] = fma(-x[j], l1, x[j + 1]);
                if (j + 2 < 16) x[j + 2] = fma(-x[j], l2, x[j + 2]);
                if (j + 1 < 16) {
                    d = dn;
                    a1 = (j + 2 < 16) ? lane_value(x[j + 1], c0 + j + 2) : 0.0;
                    a2 = (j + 3 < 16) ? lane_value(x[j + 1], c0 + j + 3) : 0.0;
                    ad = (j + 2 < 16) ? lane_value(x[j + 2], c0 + j + 2) : 0.0;
                }
                if (j + 3 < 16) {
                    wave_sync();
#pragma unroll
                    for (int c = j + 3; c < 16; ++c) x[c] = fma(-x[j], cb[j][c0 + c], x[c]);
                }
            }
            if (lane >= c0) {
#pragma unroll
                for (int c = 0; c < 16; ++c) A[lane][c0 + c] = x[c];
            }
            if (lane == 0) {
#pragma unroll
                for (int j = 0; j < 16; ++j) rpiv[c0 + j] = rp[j];
            }
        }
        if (s < nst - 1) __syncthreads();
    }
    bad = __syncthreads_or(bad);
    if (w == nst - 1) {
        wave_inv16(A, rpiv, M, 16 * w);
        for (int j = 0; j < w; ++j) blk_finish(M, w, j);
    }
    __syncthreads();
    return bad;
}

// acc[b] = block (wave, b) of X Y^T in 16x16 blocks; with kTriY, Y is lower
// triangular and the zero part of the sum is skipped.
template <bool kTriY>
__device__ __forceinline__ void tile_mfma_nt(const TileLds& X, const TileLds& Y, dbl4 acc[4]) {
    const int lane = threadIdx.x & 63, w = wave_id(), r16 = lane & 15, kq = lane >> 4;
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m0 = 0; m0 < 64; m0 += 4) {
        const double a = X[16 * w + r16][m0 + kq];
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (!kTriY || m0 < 16 * b + 16) acc[b] = mfma16x16x4(a, Y[16 * b + r16][m0 + kq], acc[b]);
    }
}

// B <- B M^T (the panel solve B L^-T with M = L^-1 lower triangular, in LDS).
__device__ __forceinline__ void tile_right_mul_t(TileLds& B, const TileLds& M) {
    dbl4 acc[4];
    tile_mfma_nt<true>(B, M, acc);
    const int lane = threadIdx.x & 63, w = wave_id(), r16 = lane & 15, kq = lane >> 4;
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) B[16 * w + 4 * v + kq][16 * b + r16] = acc[b][v];
    __syncthreads();
}

// out = B v for a 64x64 tile B in LDS and a 64-vector v in global memory
// (four threads per row, summed by DPP in a fixed order).
__device__ __forceinline__ void tile_gemv(const TileLds& B, const double* __restrict__ v, double* __restrict__ out) {
    const int tid = threadIdx.x;
    const int r = tid >> 2, q = tid & 3;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
    for (int m = q; m < 64; m += 16) {
        s0 += B[r][m] * v[m];
        s1 += B[r][m + 4] * v[m + 4];
        s2 += B[r][m + 8] * v[m + 8];
        s3 += B[r][m + 12] * v[m + 12];
    }
    double s = (s0 + s1) + (s2 + s3);
    s += dpp_move<0xB1>(s);
    s += dpp_move<0x4E>(s);
    if (q == 0) out[r] = s;
}

// y_k = M_k (g_k - sum_{j<=k-1} L_kj y_j).  The products L_kj y_j were formed
// by the workgroups that computed L_kj (tile_gemv into fpart[k][j], 64 values
// each); the nterms of them are summed here in a fixed order, so the row block
// of the factor is not read again.  M_k is in LDS.
__device__ __forceinline__ void tile_forward(const TileLds& M, const double* __restrict__ fpart, int nterms,
                                             const double* __restrict__ g, double* __restrict__ y, double* rv) {
    const int tid = threadIdx.x;
    const int r = tid >> 2, q = tid & 3;
    {
        double s0 = 0.0, s1 = 0.0;
        int j = q;
        for (; j + 4 < nterms; j += 8) {
            s0 += fpart[64 * j + r];
            s1 += fpart[64 * (j + 4) + r];
        }
        if (j < nterms) s0 += fpart[64 * j + r];
        double s = s0 + s1;
        s += dpp_move<0xB1>(s);
        s += dpp_move<0x4E>(s);
        if (q == 0) rv[r] = g[r] - s;
    }
    __syncthreads();
    double s0 = 0.0, s1 = 0.0;
    for (int m = q; m < 64; m += 8) {  // M[r][m] = 0 for m > r
        s0 += M[r][m] * rv[m];
        s1 += M[r][m + 4] * rv[m + 4];
    }
    double s = s0 + s1;
    s += dpp_move<0xB1>(s);
    s += dpp_move<0x4E>(s);
    if (q == 0) y[r] = s;
    __syncthreads();
}

// 16-column stages of diagonal tile i that hold rows of the n-row system (the
// last tile's padding rows beyond are the identity and are not factored).
__device__ __forceinline__ int tile_stages(int n, int i) { return min(4, (n - 64 * i + 15) >> 4); }

__global__ __launch_bounds__(256) void k_chol_first(const double* __restrict__ S, double* __restrict__ Lm,
                                                    double* __restrict__ Li, int lda, int n, const double* __restrict__ g,
                                                    double* __restrict__ y, LMDev* lm) {
    __shared__ TileLds A;
    __shared__ TileLds M;
    __shared__ double scratch[16 * 64];
    __shared__ double rv[64];
    __shared__ double rpiv[64];
    tile_load(A, S, lda);
    if (lm->phase == kPhaseDone) return;  // a step launched after the solve has finished
    __syncthreads();
    if (tile_potrf_inv(A, rpiv, scratch, M, tile_stages(n, 0)) && threadIdx.x == 0) atomicOr(&lm->fail, 1);
    tile_store(M, Li, 64);
    tile_forward(M, nullptr, 0, g, y, rv);
}

__global__ __launch_bounds__(256) void k_chol_step(double* __restrict__ S, double* __restrict__ Lm,
                                                   double* __restrict__ Li, int lda, int n, int k,
                                                   const double* __restrict__ g, double* __restrict__ y,
                                                   double* __restrict__ fpart, int nt, LMDev* lm) {
    __shared__ TileLds Mk;
    __shared__ TileLds Bi;
    __shared__ TileLds Bj;
    __shared__ double rv[64];
    __shared__ double rpiv[64];
    const int idx = blockIdx.x;
    int ii = (int)((sqrt(8.0 * idx + 1.0) - 1.0) * 0.5);
    while ((ii + 1) * (ii + 2) / 2 <= idx) ++ii;
    while (ii * (ii + 1) / 2 > idx) --ii;
    const int jj = idx - ii * (ii + 1) / 2;
    const int i = k + 1 + ii, j = k + 1 + jj;
    const bool same = (i == j);
    // every global load of the launch in flight at once: M_k, A_ik, A_jk and
    // the tile A_ij to update (no other workgroup writes any of them)
    const int lane = threadIdx.x & 63, w = wave_id(), r16 = lane & 15, kq = lane >> 4;
    double* Aij = S + (size_t)(64 * i) * lda + 64 * j;
    double vm[16], vi[16], vj[16], cur[4][4];
    tile_fetch(vm, Li + (size_t)4096 * k, 64);
    tile_fetch(vi, S + (size_t)(64 * i) * lda + 64 * k, lda);
    if (!same) tile_fetch(vj, S + (size_t)(64 * j) * lda + 64 * k, lda);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int v = 0; v < 4; ++v) cur[b][v] = Aij[(size_t)(16 * w + 4 * v + kq) * lda + 16 * b + r16];
    if (lm->phase == kPhaseDone) return;  // a step launched after the solve has finished (loads in flight meanwhile)
    tile_put(Mk, vm);
    tile_put(Bi, vi);
    if (!same) tile_put(Bj, vj);
    __syncthreads();
    tile_right_mul_t(Bi, Mk);  // L_ik
    if (!same) tile_right_mul_t(Bj, Mk);  // L_jk
    if (j == k + 1) {
        tile_store(Bi, Lm + (size_t)(64 * i) * lda + 64 * k, lda);
        tile_gemv(Bi, y + 64 * k, fpart + ((size_t)i * nt + k) * 64);  // L_ik y_k for the forward step of tile i
    }
    dbl4 acc[4];
    tile_mfma_nt<false>(Bi, same ? Bi : Bj, acc);
    if (same && i == k + 1) {
        // Mk is free (the last product that read it ended with a barrier): it
        // takes the updated tile to factor, Bj its inverse
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) Mk[16 * w + 4 * v + kq][16 * b + r16] = cur[b][v] - acc[b][v];
        __syncthreads();
        if (tile_potrf_inv(Mk, rpiv, &Bi[0][0], Bj, tile_stages(n, i)) && threadIdx.x == 0) atomicOr(&lm->fail, 1);
        tile_store(Bj, Li + (size_t)4096 * i, 64);
        __syncthreads();  // fpart[i][k] (written above by this workgroup) is read back by the forward step
        tile_forward(Bj, fpart + (size_t)i * nt * 64, k + 1, g + 64 * i, y + 64 * i, rv);
    } else {
        // a diagonal tile keeps its upper triangle (never read; left unchanged
        // so that it does not drift over the trials of a solve)
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (!same || 16 * w + 4 * v + kq >= 16 * b + r16)
                    Aij[(size_t)(16 * w + 4 * v + kq) * lda + 16 * b + r16] = cur[b][v] - acc[b][v];
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
        const double* Mk = Li + (size_t)4096 * (nt - 1);
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
            const double* Mk = Li + (size_t)4096 * (k - 1);
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

// Backward step for many tiles (more than kBackSingleMax): one launch per tile
// k from the last, so the reads of the factor spread over k + 1 CUs.  The
// right-hand sides r of the tiles still to solve live in y (the forward
// result) and are updated in place: every workgroup of launch k forms
// x_k = M_k^T r_k (a 64x64 product, recomputed by each workgroup instead of
// waiting for one); workgroup k writes it to dp, workgroup i < k subtracts
// L_ki^T x_k from r_i.  r_k is only read during launch k, and final when it
// starts (launches j > k subtracted their terms).  dp = 0 when the
// factorisation failed.
__global__ __launch_bounds__(256) void k_chol_back_tile(const double* __restrict__ Lm, const double* __restrict__ Li,
                                                   int lda, int nt, int k, double* __restrict__ y,
                                                   double* __restrict__ dp, const LMDev* lm) {
    __shared__ double part[4][64];
    __shared__ double xk[64];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int i = blockIdx.x;  // 0..k: i == k writes x_k, i < k updates r_i
    // every global load of the launch is issued before the first use: the
    // L_ki column slice (independent of x_k), M_k, r_k and the failure flag
    double lv[16];
    if (i < k) {
        const double* L = Lm + (size_t)(64 * k) * lda + 64 * i + lane;
#pragma unroll
        for (int t = 0; t < 16; ++t) lv[t] = L[(size_t)(wid + 4 * t) * lda];
    }
    double mv[16], rv[16];
    {
        const double* Mk = Li + (size_t)4096 * k;
        const double* rk = y + 64 * k;
#pragma unroll
        for (int t = 0; t < 16; ++t) {  // rows r = wid + 4t; M_k[r][c] = 0 for r < c
            mv[t] = Mk[(wid + 4 * t) * 64 + lane];
            rv[t] = rk[wid + 4 * t];
        }
    }
    if (lm->phase == kPhaseDone) return;  // a step launched after the solve has finished
    const int fail = lm->fail;
    if (fail) {
        if (k == nt - 1 && tid < 64) dp[64 * i + tid] = 0.0;  // launch nt-1 has one workgroup per tile
        return;
    }
    // x_k[c] = sum_r M_k[r][c] r_k[r]: lanes over c, waves over r
    {
        double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0;
#pragma unroll
        for (int t = 0; t < 16; t += 4) {
            t0 += mv[t] * rv[t];
            t1 += mv[t + 1] * rv[t + 1];
            t2 += mv[t + 2] * rv[t + 2];
            t3 += mv[t + 3] * rv[t + 3];
        }
        part[wid][lane] = (t0 + t1) + (t2 + t3);
    }
    __syncthreads();
    if (wid == 0) xk[lane] = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
    __syncthreads();
    if (i == k) {
        if (tid < 64) dp[64 * k + tid] = xk[tid];
        return;
    }
    // r_i[c] -= sum_m L[64k + m][64i + c] x_k[m]: lanes over c, waves over m = wid + 4t
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
#pragma unroll
    for (int t = 0; t < 16; t += 4) {
        s0 += lv[t] * xk[wid + 4 * t];
        s1 += lv[t + 1] * xk[wid + 4 * t + 4];
        s2 += lv[t + 2] * xk[wid + 4 * t + 8];
        s3 += lv[t + 3] * xk[wid + 4 * t + 12];
    }
    __syncthreads();
    part[wid][lane] = (s0 + s1) + (s2 + s3);
    __syncthreads();
    if (wid == 0) y[64 * i + lane] -= (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
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
    hipLaunchKernelGGL(k_chol_first, dim3(1), dim3(256), 0, st, (const double*)W.S, W.Lm, W.Li, lda, P.n,
                       (const double*)W.g, W.y, W.lm);
    for (int k = 0; k + 1 < nt; ++k) {
        const int rem = nt - k - 1;
        hipLaunchKernelGGL(k_chol_step, dim3(rem * (rem + 1) / 2), dim3(256), 0, st, W.S, W.Lm, W.Li, lda, P.n, k,
                           (const double*)W.g, W.y, W.fpart, nt, W.lm);
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
        for (int k = nt - 1; k >= 0; --k)
            hipLaunchKernelGGL(k_chol_back_tile, dim3(k + 1), dim3(256), 0, st, (const double*)W.Lm,
                               (const double*)W.Li, lda, nt, k, W.y, W.dp, (const LMDev*)W.lm);
    }
}

}  // namespace navba
