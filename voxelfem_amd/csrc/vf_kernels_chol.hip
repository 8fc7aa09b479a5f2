// vf_kernels_chol.hip -- direct solve of the coarsest multigrid level on the device (FP64).
//
// The reference factors the reduced coarsest operator with CHOLMOD (TensorProductSimulator.hh:1198-1230)
// after every stiffness update. Here the reduced operator (fixed and detached DoFs removed, natural node
// order, so its half-bandwidth is about 3 (nny nnz + nnz + 1)) is stored as 64 x 64 blocks of its lower
// band and factored by a blocked right-looking band Cholesky A = L L^T:
//   for each block column k: L_kk^-1 from A_kk, L_ik = A_ik L_kk^-T for the kb blocks below, A_ij -= L_ik L_jk^T for
//   the trailing triangle of the band.
// The work is O(n bw^2) instead of the O(n^3) of a dense factorisation. For the solves, the explicit dense
// lower-triangular X = L^-1 is formed block row by block row, so a coarse solve x = X^T (X b) is two bandwidth-bound
// triangular matrix-vector products instead of a chain of small sequential triangular solves.
// One launch per block column (k_band_step) does all of that (two on wide bands): the chain of block columns is what bounds the
// factorisation, so nothing that the next diagonal block does not need sits between two links of it.
#include "vf_internal.hpp"

namespace vf {
namespace {

constexpr int NB = 64;        // block size
constexpr int BB = NB * NB;   // doubles per block
constexpr int TPB = 256;

// block (I, I-q) of the band, row-major inside the block
__device__ __forceinline__ double *bandblk(double *B, int kb, int I, int q) { return B + ((size_t)I * (kb + 1) + q) * BB; }
__device__ __forceinline__ const double *bandblk(const double *B, int kb, int I, int q) {
    return B + ((size_t)I * (kb + 1) + q) * BB;
}

// ---- assembly of the lower band from the cached coarsest element matrices (one work-item per
//      (row DoF, neighbour slot)); rows/cols of fixed or detached DoFs are absent (red[] < 0).
// Batched forms (blockIdx.z = system): every array argument advances by its z stride per system.
__global__ void __launch_bounds__(TPB) k_band_assemble(Grid g, const double *__restrict__ Ke, const int *__restrict__ red,
                                                       int kb, double *__restrict__ B, size_t zKe, size_t zRed,
                                                       size_t zB) {
    Ke += blockIdx.z * zKe;
    red += blockIdx.z * zRed;
    B += blockIdx.z * zB;
    const long t = (long)blockIdx.x * TPB + threadIdx.x;
    if (t >= (long)g.nnodes * 27 * 3) return;
    const int row = (int)(t % (3L * g.nnodes)), slot = (int)(t / (3L * g.nnodes));
    const int rr = red[row];
    if (rr < 0) return;
    const int n = row / 3, a = row % 3;
    const int nz = g.nn[2], ix = n / (g.nn[1] * nz), iy = (n / nz) % g.nn[1], iz = n % nz;
    const int off[3] = {slot / 9 - 1, (slot / 3) % 3 - 1, slot % 3 - 1};
    const int id[3] = {ix, iy, iz};
    for (int d = 0; d < 3; ++d)
        if ((unsigned)(id[d] + off[d]) >= (unsigned)g.nn[d]) return;
    const int m = ((ix + off[0]) * g.nn[1] + iy + off[1]) * nz + iz + off[2];
    int lo[3], hi[3];
    for (int d = 0; d < 3; ++d) {
        lo[d] = max(max(id[d] - 1, id[d] + off[d] - 1), 0);
        hi[d] = min(min(id[d], id[d] + off[d]), g.ne[d] - 1);
    }
    double Bv[3] = {0, 0, 0};
    for (int ex = lo[0]; ex <= hi[0]; ++ex)
        for (int ey = lo[1]; ey <= hi[1]; ++ey)
            for (int ez = lo[2]; ez <= hi[2]; ++ez) {
                const int ln = 4 * (ix - ex) + 2 * (iy - ey) + (iz - ez);
                const int lm = 4 * (ix + off[0] - ex) + 2 * (iy + off[1] - ey) + (iz + off[2] - ez);
                const double *K = Ke + (size_t)((ex * g.ne[1] + ey) * g.ne[2] + ez) * 576;
                for (int c = 0; c < 3; ++c) Bv[c] += K[(3 * ln + a) * 24 + 3 * lm + c];
            }
    for (int c = 0; c < 3; ++c) {
        const int cc = red[3 * m + c];
        if (cc < 0 || cc > rr) continue;  // lower triangle only
        const int I = rr / NB, J = cc / NB;
        bandblk(B, kb, I, I - J)[(rr % NB) * NB + cc % NB] = Bv[c];
    }
}

// identity on the padding rows of the last diagonal block
__global__ void k_band_pad(int n, int nb, int kb, double *B) {
    const int i = n + threadIdx.x;
    if (i < nb * NB) bandblk(B, kb, nb - 1, 0)[(i % NB) * NB + i % NB] = 1.0;
}
// batched: system z holds n[z] unknowns in nb blocks; identity on every row from n[z] on (grid: nb x systems)
__global__ void k_band_pad_b(const int *__restrict__ n, int nb, int kb, double *B, size_t zB) {
    B += blockIdx.y * zB;
    const int i = blockIdx.x * NB + threadIdx.x;
    if (i >= n[blockIdx.y] && i < nb * NB) bandblk(B, kb, blockIdx.x, 0)[(i % NB) * NB + i % NB] = 1.0;
}

// FP64 MFMA 16x16x4 operand layout: A[i][k] at lane i + 16 k, B[k][j] at lane j + 16 k, result D[4 v + l / 16][l % 16]
// in element v of lane l (the FP64 form interleaves the four result rows of a lane, unlike the FP32 16x16 forms).
typedef double dx4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ dx4 mfma(double a, double b, dx4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
// row stride of 64 x 64 blocks in LDS: the sixteen lanes served at once (one entry of sixteen rows) meet no bank twice
constexpr int LS = 66;

// 1/d to full precision: the hardware estimate x (24 bits) corrected by its residual e = 1 - d x to third order,
// x (1 + e + e^2); a fraction of the latency of a division, which would bound the chain of pivots
__device__ __forceinline__ double recip(double d) {
    const double x = __builtin_amdgcn_rcp(d), e = __builtin_fma(-d, x, 1.0);
    return __builtin_fma(x, __builtin_fma(e, e, e), x);
}
// d^-1/2 the same way: x (1 + e / 2 + 3 e^2 / 8) with e = 1 - d x^2
__device__ __forceinline__ double rsqrt_full(double d) {
    const double x = __builtin_amdgcn_rsq(d), e = __builtin_fma(-(d * x), x, 1.0);
    return __builtin_fma(x, e * __builtin_fma(0.375, e, 0.5), x);
}
__device__ __forceinline__ double lane_value(double v, int lane) {  // lane is uniform
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
template <int J>
__device__ __forceinline__ double row_bcast(double v) {  // lane J of the lane's DPP row of sixteen
    return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + J, 0xf, 0xf, true);
}
__device__ __forceinline__ double even_lane(double v) {  // quad_perm [0, 0, 2, 2]
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0xA0, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0xA0, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// One elimination step of the wavefront's 16 x 16 block (see chol16): rows J and J + 1 leave the rows below, one after the
// other as far as rounding goes (row J with pivot p00, then row J + 1 less m = p01 / p00 times row J, with pivot
// s = p11 - m p01), so the step is as stable as two of Cholesky's. (Through the adjugate of the 2 x 2 pivot, with one
// reciprocal of its determinant, the combinations cancel when the pivot is nearly singular: stiff pieces in 1e-9 void
// were solved to 8e-4 in place of 1e-5, or refused.) The old columns and the pivots come from the lanes that hold them. One wavefront
// alone is bound by the instructions it issues one after the other, so two rows go per step, and A and Y share one array.
template <int J>
__device__ __forceinline__ void chol16_step(double (&a)[4], int r, int part, double (&piv)[2], bool &ok) {
    constexpr int h = J / 4, i0 = J % 4;
    const double p00 = lane_value(a[i0], J + 16 * h), p01 = lane_value(a[i0], J + 1 + 16 * h),
                 p11 = lane_value(a[i0 + 1], J + 1 + 16 * h);
    const double c0 = __shfl(a[i0], r + 16 * h, 64), c1 = __shfl(a[i0 + 1], r + 16 * h, 64);
    const double ip = recip(p00), m = p01 * ip, s = __builtin_fma(-m, p01, p11), is = -recip(s);
    const bool below = r > J + 1;
    const double g = below ? -(c0 * ip) : 0.0, w = below ? __builtin_fma(-m, c0, c1) : 0.0;
    // only the last product waits for the second reciprocal
    double u[4], v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const double rj = row_bcast<J>(a[i]);
        u[i] = __builtin_fma(g, rj, a[i]);
        v[i] = w * __builtin_fma(-m, rj, row_bcast<J + 1>(a[i]));
    }
    if (part == h) {  // columns J, J + 1 of Y start here: rows J, J + 1 of it are (1, 0), (0, 1)
        u[i0] = g;
        u[i0 + 1] = 0.0;
        v[i0] = -(w * m);
        v[i0 + 1] = w;
    }
    ok = ok && p00 > 0 && s > 0;
    if ((r >> 1) == J / 2) {
        piv[0] = r & 1 ? s : p00;
        piv[1] = r & 1 ? -m : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = __builtin_fma(is, v[i], u[i]);
}
// U = L^-1 of the 16 x 16 symmetric block whose lower triangle is at S (row stride LS), by one wavefront: lane l holds
// columns 4 (l / 16) .. + 3 of row l % 16. Eliminating two rows at a time turns [A | I] into [.. | Y]; after the step at J
// the columns up to J + 1 of A are not used again and hold those of Y instead. Row J + 1 of Y still lacks its part
// -m of row J, which is added at the end; U = D^-1/2 Y with the pivots D. Writes U (zero above its diagonal) to X (row
// stride LS).
__device__ __forceinline__ bool chol16(const double *S, double *X, int l) {
    const int r = l & 15, part = l >> 4, c0 = 4 * part;
    double a[4], piv[2] = {1.0, 0.0};
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = S[max(r, c0 + i) * LS + min(r, c0 + i)];
    chol16_step<0>(a, r, part, piv, ok);
    chol16_step<2>(a, r, part, piv, ok);
    chol16_step<4>(a, r, part, piv, ok);
    chol16_step<6>(a, r, part, piv, ok);
    chol16_step<8>(a, r, part, piv, ok);
    chol16_step<10>(a, r, part, piv, ok);
    chol16_step<12>(a, r, part, piv, ok);
    chol16_step<14>(a, r, part, piv, ok);
    const double scale = rsqrt_full(piv[0]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = c0 + i;
        const double y = c == r ? 1.0 : c < (r & ~1) ? a[i] : 0.0;  // row r of Y
        X[r * LS + c] = scale * __builtin_fma(piv[1], even_lane(y), y);
    }
    return ok;
}
// D (16 x 16) = P Q^T (NT) or P Q (NN) over K = 16 columns of P, both in LDS with row stride LS, added to acc
__device__ __forceinline__ dx4 mul16_nt(const double *P, const double *Q, dx4 acc, int li, int lk) {
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mfma(P[li * LS + 4 * s + lk], Q[li * LS + 4 * s + lk], acc);
    return acc;
}
__device__ __forceinline__ dx4 mul16_nn(const double *P, const double *Q, dx4 acc, int li, int lk) {
#pragma unroll
    for (int s = 0; s < 4; ++s) acc = mfma(P[li * LS + 4 * s + lk], Q[(4 * s + lk) * LS + li], acc);
    return acc;
}
// X = L^-1 of the 64 x 64 block whose lower triangle is in S, by a workgroup of four wavefronts, in 16 x 16 blocks.
// Step p: wavefront 0 updates diagonal block p and inverts its factor (the serial chain) while the others update the
// remaining tiles with panel p - 1 and form the sums T_pj = sum_m L_pm X_mj of row p of the inverse (in the unused blocks
// above the diagonal of S); then the panel L_ip = S_ip U_p^T below and the row X_pj = -U_p T_pj take one wavefront each.
// The upper triangle of X is zeroed. Returns false (in wavefront 0) on a non-positive pivot.
__device__ __forceinline__ bool potrf_inverse(double *S, double *X, int t) {
    const int w = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63, li = l & 15, lk = l >> 4;
    auto blk = [](double *M, int i, int j) { return M + (16 * i) * LS + 16 * j; };
    auto put = [&](double *D, dx4 v, double sign) {
#pragma unroll
        for (int q = 0; q < 4; ++q) D[(4 * q + lk) * LS + li] = sign * v[q];
    };
    auto trail = [&](int i, int j, int p) {  // S_ij -= L_ip L_jp^T
        const dx4 v = mul16_nt(blk(S, i, p), blk(S, j, p), dx4{0, 0, 0, 0}, li, lk);
        double *D = blk(S, i, j);
#pragma unroll
        for (int q = 0; q < 4; ++q) D[(4 * q + lk) * LS + li] -= v[q];
    };
    bool ok = true;
    for (int e = t; e < 6 * 256; e += TPB) {  // the blocks above the diagonal
        const int q = e >> 8, i = q < 3 ? 0 : q < 5 ? 1 : 2, j = q < 3 ? q + 1 : q < 5 ? q - 1 : 3;
        X[(16 * i + ((e >> 4) & 15)) * LS + 16 * j + (e & 15)] = 0.0;
    }
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
        if (w == 0) {
            if (p) trail(p, p, p - 1);
            __builtin_amdgcn_wave_barrier();
            ok = chol16(blk(S, p, p), blk(X, p, p), l) && ok;
        } else if (p) {
            int q = 0;
            for (int j = p; j < 4; ++j)
                for (int i = j + (j == p); i < 4; ++i)
                    if (q++ % 3 == w - 1) trail(i, j, p - 1);
            for (int j = 0; j < p; ++j)
                if (q++ % 3 == w - 1) {
                    dx4 v = {0, 0, 0, 0};
#pragma unroll 1
                    for (int m = j; m < p; ++m) v = mul16_nn(blk(S, p, m), blk(X, m, j), v, li, lk);
                    put(blk(S, j, p), v, 1.0);
                }
        }
        __syncthreads();
        if (w < 3) {
            if (w < p) {
                put(blk(X, p, w), mul16_nn(blk(X, p, p), blk(S, w, p), dx4{0, 0, 0, 0}, li, lk), -1.0);
            } else {
                double *D = blk(S, w + 1, p);
                put(D, mul16_nt(D, blk(X, p, p), dx4{0, 0, 0, 0}, li, lk), 1.0);
            }
        }
        __syncthreads();
    }
    return ok;
}

// writes X = L^-1 of diagonal block k from LDS to Linv (64 x 64, row-major)
__device__ __forceinline__ void store_linv(const double *sX, double *__restrict__ Linv, int k, int t) {
    double *Lk = Linv + (size_t)k * BB;
    for (int e = t; e < BB; e += TPB) Lk[e] = sX[(e / NB) * LS + e % NB];
}

// ---- the first diagonal block (grid: systems)
__global__ void __launch_bounds__(TPB) k_band_first(int kb, const double *__restrict__ B, double *__restrict__ Linv,
                                                    int *__restrict__ flag, size_t zB, size_t zL) {
    B += blockIdx.x * zB;
    Linv += blockIdx.x * zL;
    __shared__ double sA[NB * LS], sX[NB * LS];
    const int t = threadIdx.x;
    const double *D = bandblk(B, kb, 0, 0);
    double v[BB / TPB];
#pragma unroll
    for (int q = 0; q < BB / TPB; ++q) v[q] = D[q * TPB + t];
#pragma unroll
    for (int q = 0; q < BB / TPB; ++q) sA[(q * TPB + t) / NB * LS + t % NB] = v[q];
    __syncthreads();
    if (!potrf_inverse(sA, sX, t) && t == 0) atomicOr(flag + blockIdx.x, 1);
    store_linv(sX, Linv, 0, t);
}

// L = A Linv^T for one 64 x 64 block A of the panel, into LDS and, where wanted, to Lp (leading dimension ld): wavefront
// w forms rows 16 w .. (Linv is lower triangular, so column tile j needs the first 16 (j + 1) terms only)
__device__ __forceinline__ void panel_put(dx4 v, int j, double *sL, double *__restrict__ Lp, size_t ld, int w, int li, int lk) {
#pragma unroll
    for (int q = 0; q < 4; ++q) sL[(16 * w + 4 * q + lk) * LS + 16 * j + li] = v[q];
    if (Lp)
#pragma unroll
        for (int q = 0; q < 4; ++q) Lp[(size_t)(16 * w + 4 * q + lk) * ld + 16 * j + li] = v[q];
}
__device__ __forceinline__ void panel_block(const double *__restrict__ A, const double *__restrict__ Lk, double *sL,
                                            double *__restrict__ Lp, size_t ld, int w, int li, int lk) {
    double a[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) a[s] = A[(16 * w + li) * NB + 4 * s + lk];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        dx4 v = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 4 * (j + 1); ++s) v = mfma(a[s], Lk[(16 * j + li) * NB + 4 * s + lk], v);
        panel_put(v, j, sL, Lp, ld, w, li, lk);
    }
}
// the same with A in sP (replaced by L; each wavefront touches its own rows only) and Linv in sL
__device__ __forceinline__ void panel_rows(double *sP, const double *sL, double *__restrict__ Lp, size_t ld, int w, int li,
                                           int lk) {
    double a[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) a[s] = sP[(16 * w + li) * LS + 4 * s + lk];
    dx4 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = dx4{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 16; ++s)
#pragma unroll
        for (int j = s / 4; j < 4; ++j) v[j] = mfma(a[s], sL[(16 * j + li) * LS + 4 * s + lk], v[j]);
#pragma unroll
    for (int j = 0; j < 4; ++j) panel_put(v[j], j, sP, Lp, ld, w, li, lk);
}

// ---- L_{k+a,k} of the whole panel, for wide bands (grid: systems x m)
__global__ void __launch_bounds__(TPB) k_band_panel(int k, int nb, int kb, const double *__restrict__ B,
                                                    const double *__restrict__ Linv, double *__restrict__ XT, size_t zB,
                                                    size_t zL, size_t zX, const int *__restrict__ nbz) {
    const size_t ld = (size_t)nb * NB;
    const int z = blockIdx.x, a = blockIdx.y + 1, I = k + a;
    if (nbz) nb = min(nb, nbz[z]);
    if (I >= nb) return;
    __shared__ double sL[NB * LS];
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
    panel_block(bandblk(B + z * zB, kb, I, a), Linv + z * zL + (size_t)k * BB, sL,
                XT + z * zX + (size_t)I * NB * ld + (size_t)k * NB, ld, w, l & 15, l >> 4);
}
// a 64 x 64 block of the panel from there into LDS
__device__ __forceinline__ void load_panel(const double *__restrict__ Lp, size_t ld, double *sL, int t) {
    double v[BB / TPB];
#pragma unroll
    for (int q = 0; q < BB / TPB; ++q) v[q] = Lp[(size_t)((q * TPB + t) / NB) * ld + t % NB];
#pragma unroll
    for (int q = 0; q < BB / TPB; ++q) sL[(q * TPB + t) / NB * LS + t % NB] = v[q];
}

// ---- everything that block column k allows once Linv_k is known (grid: systems x roles):
//   roles 0 .. m (m + 1) / 2 - 1, m = min(kb, nb - 1 - k): the pair (a, b), 1 <= b <= a <= m, forms L_{k+a,k} and
//     L_{k+b,k} from the panel (each pair for itself: the products cost less than a launch between panel and update;
//     PANEL: k_band_panel has formed them, see band_steps) and subtracts their product from A_{k+a,k+b}. Pairs with b = 1 store L_{k+a,k} in the lower block triangle of XT,
//     which nothing else uses. Role 0 is the pair (1, 1), which goes on to invert the factor of diagonal block k + 1:
//     that is the chain from launch to launch;
//   the roles after them: strips of 16 CT columns of block row k of X, X_kJ = -Linv_k sum_q L_{k,k-q} X_{k-q,J}
//     (J < k), X_kk = Linv_k, and their transposes into XT. They are off the chain and fill the chip beside it. CT = 1
//     spreads a row over four times the workgroups; CT = 4 reads each band block a quarter as often.
// 4131 unknowns, kb = 5: 61 launches of 16.3 us against 183 of 13.0 (panel), 13.1 (update) and 52.2 us (diagonal block)
// and 61 of 14.8 us for the rows of X: 1.01 against 5.66 ms. Of the 16 us the loads take 1.7, the panel 1.7, the update
// 1.9, the diagonal block 8.6 (four 16 x 16 factors of 1.4 us one after the other) and the launch the rest.
template <int CT, bool PANEL>
__global__ void __launch_bounds__(TPB) k_band_step(int k, int nb, int kb, double *__restrict__ B, double *__restrict__ Linv,
                                                   double *__restrict__ X, double *__restrict__ XT, int *__restrict__ flag,
                                                   size_t zB, size_t zL, size_t zX, const int *__restrict__ nbz) {
    const size_t ld = (size_t)nb * NB;  // leading dimension of X and XT (the padded size)
    const int mPairs = min(kb, nb - 1 - k), npairs = mPairs * (mPairs + 1) / 2;
    const int z = blockIdx.x;
    if (nbz) nb = min(nb, nbz[z]);
    if (k >= nb) return;
    B += z * zB;
    Linv += z * zL;
    X += z * zX;
    XT += z * zX;
    __shared__ double sP[NB * LS], sQ[NB * LS];
    const int t = threadIdx.x, w = t >> 6, l = t & 63, li = l & 15, lk = l >> 4;
    const double *Lk = Linv + (size_t)k * BB;
    int role = blockIdx.y;
    if (role < npairs) {
        int a = 1;
        while (role >= a) { role -= a; ++a; }
        const int b = role + 1, I = k + a, J = k + b;
        if (I >= nb) return;
        double *Aij = bandblk(B, kb, I, a - b), *Lp = XT + (size_t)I * NB * ld + (size_t)k * NB;
        if (a == b) {
            // both operands of the panel product go through LDS, requested at once with the block to update: this is
            // the path of the chain, which waits for one round of loads. Of A_II only the tiles on and below the
            // diagonal are needed: tile q = w, w + 4, w + 8 of the ten goes to wavefront w
            constexpr uint64_t tr = 0x3323213210, tc = 0x3221110000;  // row and column of tile q, a nibble each
            const double *A = bandblk(B, kb, I, a);
            double va[16], vl[16], old[3][4];
            if (!PANEL) {
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    va[q] = A[q * TPB + t];
                    vl[q] = Lk[q * TPB + t];
                }
            }
            const int wu = __builtin_amdgcn_readfirstlane(w);
            int ti[3], tj[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int id = min(wu + 4 * q, 9);
                ti[q] = (int)(tr >> (4 * id)) & 15;
                tj[q] = (int)(tc >> (4 * id)) & 15;
#pragma unroll
                for (int v = 0; v < 4; ++v) old[q][v] = Aij[(16 * ti[q] + 4 * v + lk) * NB + 16 * tj[q] + li];
            }
            if (PANEL) {
                load_panel(Lp, ld, sP, t);
            } else {
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    sP[(q * TPB + t) / NB * LS + t % NB] = va[q];
                    sQ[(q * TPB + t) / NB * LS + t % NB] = vl[q];
                }
                __syncthreads();
                panel_rows(sP, sQ, a == 1 ? Lp : nullptr, ld, w, li, lk);
            }
            __syncthreads();
            dx4 v[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) v[q] = dx4{0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < 16; ++s)  // the sums side by side: a product waits for the one before it in its sum
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    v[q] = mfma(sP[(16 * ti[q] + li) * LS + 4 * s + lk], sP[(16 * tj[q] + li) * LS + 4 * s + lk], v[q]);
            if (a != 1) {
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    if (wu + 4 * q <= 9)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            Aij[(16 * ti[q] + 4 * e + lk) * NB + 16 * tj[q] + li] = old[q][e] - v[q][e];
                return;
            }
            __syncthreads();  // the panel block in sP has been read by every wavefront
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (wu + 4 * q <= 9)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        sP[(16 * ti[q] + 4 * e + lk) * LS + 16 * tj[q] + li] = old[q][e] - v[q][e];
            __syncthreads();
            if (!potrf_inverse(sP, sQ, t) && t == 0) atomicOr(flag + z, 1);
            store_linv(sQ, Linv, k + 1, t);
            return;
        }
        double old[4][4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) old[j][q] = Aij[(16 * w + 4 * q + lk) * NB + 16 * j + li];
        if (PANEL) {
            load_panel(Lp, ld, sP, t);
            load_panel(XT + (size_t)J * NB * ld + (size_t)k * NB, ld, sQ, t);
        } else {
            panel_block(bandblk(B, kb, I, a), Lk, sP, b == 1 ? Lp : nullptr, ld, w, li, lk);
            panel_block(bandblk(B, kb, J, b), Lk, sQ, nullptr, ld, w, li, lk);
        }
        __syncthreads();
        dx4 v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = dx4{0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const double x = sP[(16 * w + li) * LS + 4 * s + lk];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = mfma(x, sQ[(16 * j + li) * LS + 4 * s + lk], v[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) Aij[(16 * w + 4 * q + lk) * NB + 16 * j + li] = old[j][q] - v[j][q];
        return;
    }
    // ---- a strip of block row k of X
    constexpr int CW = 16 * CT;
    role -= npairs;
    const int J = role / (NB / CW), cs = role % (NB / CW) * CW, col0 = J * NB + cs;
    if (J > k) return;
    double *Xr = X + (size_t)k * NB * ld + col0, *XTr = XT + (size_t)col0 * ld + (size_t)k * NB;
    if (J == k) {
        for (int e = t; e < NB * CW; e += TPB) {
            Xr[(size_t)(e / CW) * ld + e % CW] = Lk[(e / CW) * NB + cs + e % CW];
            XTr[(size_t)(e / NB) * ld + e % NB] = Lk[(e % NB) * NB + cs + e / NB];
        }
        return;
    }
    dx4 v[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) v[j] = dx4{0, 0, 0, 0};
    const int qmax = min(kb, k - J);
    for (int q = 1; q <= qmax; ++q) {
        const double *Lb = XT + (size_t)(k * NB + 16 * w + li) * ld + (size_t)(k - q) * NB + lk;
        const double *Xb = X + ((size_t)(k - q) * NB + lk) * ld + col0 + li;
        double a[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) a[s] = Lb[4 * s];
#pragma unroll
        for (int j = 0; j < CT; ++j) {
            double b[16];
#pragma unroll
            for (int s = 0; s < 16; ++s) b[s] = Xb[(size_t)(4 * s) * ld + 16 * j];
#pragma unroll
            for (int s = 0; s < 16; ++s) v[j] = mfma(a[s], b[s], v[j]);
        }
    }
    // the sum goes through LDS once, so that every wavefront sees all 64 of its rows as the K dimension of Linv_k T
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) sP[(16 * w + 4 * q + lk) * LS + 16 * j + li] = v[j][q];
    __syncthreads();
    double a[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) a[s] = Lk[(16 * w + li) * NB + 4 * s + lk];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        dx4 o = {0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 16; ++s) o = mfma(a[s], sP[(4 * s + lk) * LS + 16 * j + li], o);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            Xr[(size_t)(16 * w + 4 * q + lk) * ld + 16 * j + li] = -o[q];
            XTr[(size_t)(16 * j + li) * ld + 16 * w + 4 * q + lk] = -o[q];
        }
    }
}

// ---- coarse solves x = X^T (X b) over nsys independent systems (blockIdx.y = system z; nsys = 1 for a single structure):
// system z owns n[z] (or n0) reduced unknowns; its DoF i is component f % 3 of node f / 3 + z * nodeStride of the level
// vector, f = redToFull[z * redStride + i]; its factors X, XT (leading dimension ld) start at z * ld * ld.
// skip (optional): systems with skip[z] == 2 are left out (their x stays zero).
struct CoarseSys {
    const int *n;  // per system, or null: n0
    int n0, ld;
    const int *redToFull;
    size_t redStride, nodeStride;
    const int *skip;
    __device__ __forceinline__ int count(int z) const { return n ? n[z] : n0; }
    __device__ __forceinline__ bool out(int z) const { return skip && skip[z] == 2; }
};
// in = the reduced right-hand sides, zero up to the next multiple of 64 (in and out: the products below read whole
// blocks), and the level vector x cleared in the same launch (grid: enough for both)
template <typename T>
__global__ void __launch_bounds__(TPB) k_cgather(CoarseSys c, int N, size_t nx, const T *__restrict__ b, T *__restrict__ x,
                                                 double *__restrict__ in, double *__restrict__ out) {
    const int z = blockIdx.y, i = blockIdx.x * TPB + threadIdx.x;
    for (size_t e = (size_t)z * gridDim.x * TPB + i; e < nx; e += (size_t)gridDim.x * gridDim.y * TPB) x[e] = T(0);
    if (i >= c.ld || c.out(z)) return;
    const int n = c.count(z);
    double v = 0.0;
    if (i < n) {
        const int f = c.redToFull[z * c.redStride + i];
        v = (double)b[(size_t)(f % 3) * N + f / 3 + z * c.nodeStride];
    }
    in[(size_t)z * c.ld + i] = v;
    if (i >= n) out[(size_t)z * c.ld + i] = 0.0;
}
// this lane's part of sum_j R[j] v[j] over [c0, c1), both multiples of 64; eight loads of sixteen bytes in flight, without
// which a row's serial loop, and not the memory, bounds the product: 4131 unknowns 21.5 -> 12.0 us per triangular product
// (5.7 TB/s of the triangle), 8280 unknowns 75 -> 50.7 us (5.4 TB/s), eight structures of up to 7623 125 -> 101 us
__device__ __forceinline__ double row_part(const double *__restrict__ R, const double *__restrict__ v, int c0, int c1, int lane) {
    double s[4] = {0, 0, 0, 0};
    int j = c0 + 2 * lane;
    for (; j + 384 < c1; j += 512) {
        double2 r[4], w[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            r[q] = *reinterpret_cast<const double2 *>(R + j + 128 * q);
            w[q] = *reinterpret_cast<const double2 *>(v + j + 128 * q);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] += r[q].x * w[q].x + r[q].y * w[q].y;
    }
    for (; j < c1; j += 128) {
        const double2 r = *reinterpret_cast<const double2 *>(R + j), w = *reinterpret_cast<const double2 *>(v + j);
        s[0] += r.x * w.x + r.y * w.y;
    }
    return (s[0] + s[1]) + (s[2] + s[3]);
}
// rows w and n - 1 - w of a triangular product by wavefront w, so that every wavefront reads about the same amount; a row
// reads whole 64-column blocks (X is zero above its diagonal inside them)
template <typename F>
__device__ __forceinline__ void triangle_rows(int n, F &&row) {
    const int w = blockIdx.x * (TPB / 64) + (threadIdx.x >> 6);
    if (2 * w >= n) return;
    row(w);
    if (n - 1 - w != w) row(n - 1 - w);
}
__device__ __forceinline__ double wave_sum(double s) {
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
}
__global__ void __launch_bounds__(TPB) k_trmv_lower(CoarseSys c, const double *__restrict__ X, const double *__restrict__ b,
                                                    double *__restrict__ y) {
    const int z = blockIdx.y, lane = threadIdx.x & 63;
    if (c.out(z)) return;
    X += (size_t)z * c.ld * c.ld;
    b += (size_t)z * c.ld;
    y += (size_t)z * c.ld;
    triangle_rows(c.count(z), [&](int r) {
        const double s = wave_sum(row_part(X + (size_t)r * c.ld, b, 0, (r / NB + 1) * NB, lane));
        if (lane == 0) y[r] = s;
    });
}
// x = XT y, scattered to the level vector
template <typename T>
__global__ void __launch_bounds__(TPB) k_trmv_upper(CoarseSys c, int N, const double *__restrict__ XT,
                                                    const double *__restrict__ y, T *__restrict__ x) {
    const int z = blockIdx.y, lane = threadIdx.x & 63;
    if (c.out(z)) return;
    XT += (size_t)z * c.ld * c.ld;
    y += (size_t)z * c.ld;
    const int n = c.count(z), end = (n + NB - 1) / NB * NB;
    triangle_rows(n, [&](int r) {
        const double s = wave_sum(row_part(XT + (size_t)r * c.ld, y, r / NB * NB, end, lane));
        if (lane == 0) {
            const int f = c.redToFull[z * c.redStride + r];
            x[(size_t)(f % 3) * N + f / 3 + z * c.nodeStride] = (T)s;
        }
    });
}

template <typename T>
__global__ void __launch_bounds__(TPB) k_cfill(size_t n, T *x, T v) {
    const size_t i = (size_t)blockIdx.x * TPB + threadIdx.x;
    if (i < n) x[i] = v;
}

inline unsigned nblk(long count) { return (unsigned)((count + TPB - 1) / TPB); }

}  // namespace

size_t band_storage(int n, int kb) {
    const int nb = (n + NB - 1) / NB;
    return (size_t)nb * (kb + 1) * BB;
}

void band_cholesky_inverse(const Grid &g, const double *Ke, const int *red, int n, int kb, double *B, double *Linv,
                           double *X, double *XT, int *flag, hipStream_t s) {
    // fill kernels rather than memsets: the sequence may be captured into a HIP graph
    launch_fill<double>(band_storage(n, kb), B, 0.0, s);
    hipLaunchKernelGGL(k_band_assemble, dim3(nblk((long)g.nnodes * 81)), dim3(TPB), 0, s, g, Ke, red, kb, B, 0, 0, 0);
    band_factor_inverse(n, kb, B, Linv, X, XT, flag, s);
}

// the launches of the factorization and the inverse for nsys systems (see k_band_step). Both rules compare with the
// workgroups that run at once, two on every CU (as many as the LDS holds). Rows of X with more narrow strips than that take
// the wide ones, which read each band block a quarter as often: whole runs with narrow strips only / wide only / this rule,
// in ms: a 64 x 32 x 32 solve 4.20 / 5.18 / 4.22, forty layers of 160 x 80 x 80 in batches 257.2 / 250.1 / 249.9. With more
// pairs than that, the panel gets a launch of its own instead of being formed again by every pair: 14739 unknowns, kb = 14
// 15.4 either way (16.8 with the panel launch always), 24843, kb = 93 104 -> 88 ms, 23409, kb = 122 187 -> 142 ms (the
// separate launches and vector-unit products before k_band_step: 162).
static void band_steps(int nsys, const int *nbz, int nb, int kb, double *B, double *Linv, double *X, double *XT, int *flags,
                       size_t zB, size_t zL, size_t zX, hipStream_t s) {
    const long room = 2L * cu_count();
    hipLaunchKernelGGL(k_band_first, dim3(nsys), dim3(TPB), 0, s, kb, B, Linv, flags, zB, zL);
    for (int k = 0; k < nb; ++k) {
        const int m = std::min(kb, nb - 1 - k), pairs = m * (m + 1) / 2;
        const bool panel = (long)nsys * pairs > room;
        if (panel) hipLaunchKernelGGL(k_band_panel, dim3(nsys, m), dim3(TPB), 0, s, k, nb, kb, B, Linv, XT, zB, zL, zX, nbz);
        const bool narrow = (long)nsys * (k + 1) * 4 <= room;
        const dim3 grid(nsys, pairs + (narrow ? 4 : 1) * (k + 1));
        auto step = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, dim3(TPB), 0, s, k, nb, kb, B, Linv, X, XT, flags, zB, zL, zX, nbz);
        };
        if (narrow) panel ? step(k_band_step<1, true>) : step(k_band_step<1, false>);
        else panel ? step(k_band_step<4, true>) : step(k_band_step<4, false>);
    }
    VF_HIP(hipGetLastError());
}

void band_factor_inverse(int n, int kb, double *B, double *Linv, double *X, double *XT, int *flag, hipStream_t s) {
    const int nb = (n + NB - 1) / NB;
    launch_fill<int>(1, flag, 0, s);
    if (nb * NB > n) hipLaunchKernelGGL(k_band_pad, dim3(1), dim3(NB), 0, s, n, nb, kb, B);
    band_steps(1, nullptr, nb, kb, B, Linv, X, XT, flag, 0, 0, 0, s);
}

void band_cholesky_inverse_batched(const Grid &g, const double *Ke, size_t keStride, const int *red, size_t redStride,
                                   int nsys, const int *n, const int *nbz, int nb, int kb, double *B, double *Linv,
                                   double *X, double *XT, int *flags, hipStream_t s) {
    if (nsys < 1 || nsys > 65535 || nb < 1) throw std::runtime_error("batched band Cholesky: bad system count or size");
    const size_t ld = (size_t)nb * NB, zB = band_storage(nb * NB, kb), zL = (size_t)nb * BB, zX = ld * ld;
    launch_fill<double>(zB * nsys, B, 0.0, s);
    launch_fill<int>(nsys, flags, 0, s);
    hipLaunchKernelGGL(k_band_assemble, dim3(nblk((long)g.nnodes * 81), 1, nsys), dim3(TPB), 0, s, g, Ke, red, kb, B,
                       keStride, redStride, zB);
    hipLaunchKernelGGL(k_band_pad_b, dim3(nb, nsys), dim3(NB), 0, s, n, nb, kb, B, zB);
    band_steps(nsys, nbz, nb, kb, B, Linv, X, XT, flags, zB, zL, zX, s);
}

template <typename T>
static void coarse_apply(int nsys, const CoarseSys &c, int most, const double *X, const double *XT, int nnodes, int ncomp,
                         const T *b, T *x, double *tmp_in, double *tmp_out, hipStream_t s) {
    const dim3 gr((unsigned)((most + 2 * (TPB / 64) - 1) / (2 * (TPB / 64))), nsys);
    hipLaunchKernelGGL(k_cgather<T>, dim3(nblk(c.ld), nsys), dim3(TPB), 0, s, c, nnodes, (size_t)ncomp * nnodes, b, x, tmp_in,
                       tmp_out);
    hipLaunchKernelGGL(k_trmv_lower, gr, dim3(TPB), 0, s, c, X, tmp_in, tmp_out);
    hipLaunchKernelGGL(k_trmv_upper<T>, gr, dim3(TPB), 0, s, c, nnodes, XT, tmp_out, x);
    VF_HIP(hipGetLastError());
}

template <typename T>
void launch_coarse_chol_apply_batched(int nsys, const int *n, int ld, const double *X, const double *XT,
                                      const int *redToFull, size_t redStride, int nnodes, size_t nodeStride, const T *b,
                                      T *x, double *tmp_in, double *tmp_out, hipStream_t s, const int *skip) {
    const CoarseSys c{n, 0, ld, redToFull, redStride, nodeStride, skip};
    coarse_apply<T>(nsys, c, ld, X, XT, nnodes, 3, b, x, tmp_in, tmp_out, s);
}
template void launch_coarse_chol_apply_batched<double>(int, const int *, int, const double *, const double *,
                                                       const int *, size_t, int, size_t, const double *, double *,
                                                       double *, double *, hipStream_t, const int *);
template void launch_coarse_chol_apply_batched<float>(int, const int *, int, const double *, const double *,
                                                      const int *, size_t, int, size_t, const float *, float *,
                                                      double *, double *, hipStream_t, const int *);

template <typename T>
void launch_coarse_chol_apply(int nred, const double *X, const double *XT, const int *redToFull, int nnodes,
                              const T *b, T *x, double *tmp_in, double *tmp_out, hipStream_t s, int ncomp) {
    if (nred == 0) {  // nothing to solve
        hipLaunchKernelGGL(k_cfill<T>, dim3(nblk((long)ncomp * nnodes)), dim3(TPB), 0, s, (size_t)ncomp * nnodes, x, T(0));
        VF_HIP(hipGetLastError());
        return;
    }
    const CoarseSys c{nullptr, nred, (nred + NB - 1) / NB * NB, redToFull, 0, 0, nullptr};
    coarse_apply<T>(1, c, nred, X, XT, nnodes, ncomp, b, x, tmp_in, tmp_out, s);
}

template void launch_coarse_chol_apply<double>(int, const double *, const double *, const int *, int, const double *,
                                               double *, double *, double *, hipStream_t, int);
template void launch_coarse_chol_apply<float>(int, const double *, const double *, const int *, int, const float *,
                                              float *, double *, double *, hipStream_t, int);

}  // namespace vf
