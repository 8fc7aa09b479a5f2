// vf_kernels_ops.hip -- level operators of the multigrid hierarchy on gfx950:
// matrix-free fine K u, level-1 on-the-fly Galerkin operator, assembled 27-point block rows,
// multicolour block Gauss-Seidel and the grid transfers.
//
// Thread mapping: one work-item per output node, z (the contiguous index) fastest, so a
// 64-wide wavefront reads 64 consecutive doubles of each component plane. Element matrices
// (K0, the eight coarsened K0s) are indexed with compile-time offsets from a uniform pointer,
// which the compiler turns into scalar loads shared by the whole wavefront.
#include "vf_internal.hpp"

#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>

namespace vf {
namespace {

constexpr int TPB = 256;

__device__ __forceinline__ int eidx(const Grid &g, int ex, int ey, int ez) { return (ex * g.ne[1] + ey) * g.ne[2] + ez; }

template <typename T>
__device__ __forceinline__ void store_out(T *y, const T *b, int N, int n, const T f[3], int mode, uint8_t dm) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        T v;
        if (mode == AM_SET) v = f[c];
        else if (mode == AM_ADD) v = y[c * N + n] + f[c];
        else if (mode == AM_SUB) v = y[c * N + n] - f[c];
        else v = b[c * N + n] - f[c];
        if (dm & (1 << c)) v = T(0);
        y[c * N + n] = v;
    }
}

// Gather the 3x3x3 neighbourhood of node (ix,iy,iz); out-of-grid values read as zero.
template <typename T>
__device__ __forceinline__ void gather27(const Grid &g, const T *__restrict__ u, int ix, int iy, int iz,
                                         T un[27][3]) {
    const int N = g.nnodes, sx = g.nn[1] * g.nn[2], sy = g.nn[2];
    const int n = (ix * g.nn[1] + iy) * g.nn[2] + iz;
#pragma unroll
    for (int dx = -1; dx <= 1; ++dx)
#pragma unroll
        for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
            for (int dz = -1; dz <= 1; ++dz) {
                const int s = (dx + 1) * 9 + (dy + 1) * 3 + (dz + 1);
                const bool ok = (unsigned)(ix + dx) < (unsigned)g.nn[0] && (unsigned)(iy + dy) < (unsigned)g.nn[1] &&
                                (unsigned)(iz + dz) < (unsigned)g.nn[2];
                const int m = n + dx * sx + dy * sy + dz;
#pragma unroll
                for (int c = 0; c < 3; ++c) un[s][c] = ok ? u[c * N + m] : T(0);
            }
}

// neighbour slot of local node m of the element whose local index of the centre node is (i,j,k)
__device__ __forceinline__ constexpr int slot_of(int m, int i, int j, int k) {
    return (((m >> 2) & 1) - i + 1) * 9 + (((m >> 1) & 1) - j + 1) * 3 + ((m & 1) - k + 1);
}

template <typename T>
__device__ __forceinline__ void inv3_apply(const T M[9], const T r[3], T out[3]) {
    const T c00 = M[4] * M[8] - M[5] * M[7];
    const T c01 = M[5] * M[6] - M[3] * M[8];
    const T c02 = M[3] * M[7] - M[4] * M[6];
    const T det = M[0] * c00 + M[1] * c01 + M[2] * c02;
    const T id = T(1) / det;
    const T i00 = c00 * id, i01 = (M[2] * M[7] - M[1] * M[8]) * id, i02 = (M[1] * M[5] - M[2] * M[4]) * id;
    const T i10 = c01 * id, i11 = (M[0] * M[8] - M[2] * M[6]) * id, i12 = (M[2] * M[3] - M[0] * M[5]) * id;
    const T i20 = c02 * id, i21 = (M[1] * M[6] - M[0] * M[7]) * id, i22 = (M[0] * M[4] - M[1] * M[3]) * id;
    out[0] = i00 * r[0] + i01 * r[1] + i02 * r[2];
    out[1] = i10 * r[0] + i11 * r[1] + i12 * r[2];
    out[2] = i20 * r[0] + i21 * r[1] + i22 * r[2];
}

// u_n += update from (b - S') and M (MultigridSolver.hh:347-378): block solve for free nodes,
// sequential masked point updates for partially constrained nodes.
template <typename T>
__device__ __forceinline__ void gs_update(T *u, int N, int n, const T bms[3], const T M[9], uint8_t dm, int forward) {
    T ud[3];
    if (dm) {
        ud[0] = ud[1] = ud[2] = T(0);
        auto point = [&](int i) {
            const T fr = (dm & (1 << i)) ? T(0) : T(1);
            ud[i] = (bms[i] - (M[3 * i] * ud[0] + M[3 * i + 1] * ud[1] + M[3 * i + 2] * ud[2])) * (fr / M[4 * i]);
        };
        // no index that is only known at run time: the arrays stay in registers
        if (forward) {
            point(0);
            point(1);
            point(2);
        } else {
            point(2);
            point(1);
            point(0);
        }
    } else {
        inv3_apply(M, bms, ud);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) u[c * N + n] += ud[c];
}

// ------------------------------------------------------------------ fine level (K0, E)
// Sum over the 8 incident elements of E_e * K0[:, 3 ln + c]^T u_e (K0 symmetric, column access
// as in TPSStencils.hh:453-471); optionally also the diagonal block M = sum E_e K0[3ln.., 3ln..].
template <typename T, bool WANT_M>
__device__ __forceinline__ void fine_row(const Grid &g, const T *__restrict__ K0, const T *__restrict__ E, int ix,
                                         int iy, int iz, const T un[27][3], T f[3], T M[9]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int i = (e >> 2) & 1, j = (e >> 1) & 1, k = e & 1;
        const int ex = ix - i, ey = iy - j, ez = iz - k;
        const bool ok = (unsigned)ex < (unsigned)g.ne[0] && (unsigned)ey < (unsigned)g.ne[1] &&
                        (unsigned)ez < (unsigned)g.ne[2];
        if (!ok) continue;
        const T Ee = E[eidx(g, ex, ey, ez)];
        const int ln = 4 * i + 2 * j + k;
        T a0 = 0, a1 = 0, a2 = 0;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int s = slot_of(m, i, j, k);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const T um = un[s][d];
                const int row = (3 * m + d) * 24 + 3 * ln;
                a0 += K0[row + 0] * um;
                a1 += K0[row + 1] * um;
                a2 += K0[row + 2] * um;
            }
        }
        f[0] += Ee * a0;
        f[1] += Ee * a1;
        f[2] += Ee * a2;
        if (WANT_M) {
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int c2 = 0; c2 < 3; ++c2) M[3 * c + c2] += Ee * K0[(3 * ln + c) * 24 + 3 * ln + c2];
        }
    }
}

template <typename T, int MODE>
__global__ void __launch_bounds__(TPB) k_fine_apply(Grid g, const T *__restrict__ K0, const T *__restrict__ E,
                                                    const T *__restrict__ u, T *__restrict__ y,
                                                    const T *__restrict__ b, const uint8_t *__restrict__ dmask) {
    const int nz = g.nn[2], slab = g.ydet * nz;
    const int t = blockIdx.x * TPB + threadIdx.x;
    if (t >= g.nn[0] * slab) return;
    const int ix = t / slab, r = t - ix * slab, iy = r / nz, iz = r - iy * nz;
    const int n = (ix * g.nn[1] + iy) * nz + iz;
    T un[27][3];
    gather27(g, u, ix, iy, iz, un);
    T f[3] = {0, 0, 0};
    T M[9];
    fine_row<T, false>(g, K0, E, ix, iy, iz, un, f, M);
    store_out(y, b, g.nnodes, n, f, MODE, dmask ? dmask[n] : uint8_t(0));
}

// Rows of detached nodes of an AM_SET product are zero (TPSStencils.hh:717-727).
template <typename T>
__global__ void __launch_bounds__(TPB) k_zero_detached(Grid g, T *__restrict__ y) {
    const int nz = g.nn[2], rows = g.nn[1] - g.ydet, slab = rows * nz;
    const int t = blockIdx.x * TPB + threadIdx.x;
    if (t >= g.nn[0] * slab) return;
    const int ix = t / slab, r = t - ix * slab, iy = g.ydet + r / nz, iz = r % nz;
    const int n = (ix * g.nn[1] + iy) * nz + iz;
    y[n] = T(0);
    y[g.nnodes + n] = T(0);
    y[2 * g.nnodes + n] = T(0);
}

template <typename T>
__global__ void __launch_bounds__(TPB) k_fine_gs(Grid g, const T *__restrict__ K0, const T *__restrict__ E,
                                                 T *__restrict__ u, const T *__restrict__ b,
                                                 const uint8_t *__restrict__ dmask, int cx, int cy, int cz,
                                                 int forward) {
    const int mx = (g.nn[0] - cx + 1) / 2, my = (g.ydet - cy + 1) / 2, mz = (g.nn[2] - cz + 1) / 2;
    const int t = blockIdx.x * TPB + threadIdx.x;
    if (t >= mx * my * mz) return;
    const int jx = t / (my * mz), r = t - jx * my * mz, jy = r / mz, jz = r - jy * mz;
    const int ix = 2 * jx + cx, iy = 2 * jy + cy, iz = 2 * jz + cz;
    const int N = g.nnodes, n = (ix * g.nn[1] + iy) * g.nn[2] + iz;
    const uint8_t dm = dmask ? dmask[n] : uint8_t(0);
    if (dm == 7) return;
    T un[27][3];
    gather27(g, u, ix, iy, iz, un);
    T f[3] = {0, 0, 0};
    T M[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    fine_row<T, true>(g, K0, E, ix, iy, iz, un, f, M);
    const T bms[3] = {b[n] - f[0], b[N + n] - f[1], b[2 * N + n] - f[2]};
    gs_update(u, N, n, bms, M, dm, forward);
}

// ------------------------------------------------------------------ level 1 (fine E, Chat)
// Coarse element e with centre-node local index ln: Ke = sum_fi E_f Chat_fi (MultigridSolver.hh:483-491).
template <typename T, bool WANT_M, bool COLS>
__device__ __forceinline__ void l1_row(const Grid &gc, const Grid &gf, const T *__restrict__ Chat,
                                       const T *__restrict__ Ef, int ix, int iy, int iz, const T un[27][3], T f[3],
                                       T M[9]) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int i = (e >> 2) & 1, j = (e >> 1) & 1, k = e & 1;
        const int ex = ix - i, ey = iy - j, ez = iz - k;
        const bool ok = (unsigned)ex < (unsigned)gc.ne[0] && (unsigned)ey < (unsigned)gc.ne[1] &&
                        (unsigned)ez < (unsigned)gc.ne[2];
        if (!ok) continue;
        const int ln = 4 * i + 2 * j + k;
        T ue[24];
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int d = 0; d < 3; ++d) ue[3 * m + d] = un[slot_of(m, i, j, k)][d];
        const int fbase = eidx(gf, 2 * ex, 2 * ey, 2 * ez);
#pragma unroll
        for (int fi = 0; fi < 8; ++fi) {
            const T Efi = Ef[fbase + ((fi >> 2) & 1) * gf.ne[1] * gf.ne[2] + ((fi >> 1) & 1) * gf.ne[2] + (fi & 1)];
            const T *C = Chat + fi * 576;
            T a0 = 0, a1 = 0, a2 = 0;
#pragma unroll
            for (int bb = 0; bb < 24; ++bb) {
                if (COLS) {  // Ke[:, 3ln+c]^T u (smoother form, MultigridSolver.hh:310-314)
                    a0 += C[bb * 24 + 3 * ln + 0] * ue[bb];
                    a1 += C[bb * 24 + 3 * ln + 1] * ue[bb];
                    a2 += C[bb * 24 + 3 * ln + 2] * ue[bb];
                } else {     // Ke[3ln+c, :] u (operator form, MultigridSolver.hh:488-491)
                    a0 += C[(3 * ln + 0) * 24 + bb] * ue[bb];
                    a1 += C[(3 * ln + 1) * 24 + bb] * ue[bb];
                    a2 += C[(3 * ln + 2) * 24 + bb] * ue[bb];
                }
            }
            f[0] += Efi * a0;
            f[1] += Efi * a1;
            f[2] += Efi * a2;
            if (WANT_M) {
#pragma unroll
                for (int c = 0; c < 3; ++c)
#pragma unroll
                    for (int c2 = 0; c2 < 3; ++c2) M[3 * c + c2] += Efi * C[(3 * ln + c) * 24 + 3 * ln + c2];
            }
        }
    }
}

template <typename T, int MODE>
__global__ void __launch_bounds__(TPB) k_l1_apply(Grid gc, Grid gf, const T *__restrict__ Chat,
                                                  const T *__restrict__ Ef, const T *__restrict__ u,
                                                  T *__restrict__ y, const T *__restrict__ b,
                                                  const uint8_t *__restrict__ dmask) {
    const int nz = gc.nn[2], slab = gc.ydet * nz;
    const int t = blockIdx.x * TPB + threadIdx.x;
    if (t >= gc.nn[0] * slab) return;
    const int ix = t / slab, r = t - ix * slab, iy = r / nz, iz = r - iy * nz;
    const int n = (ix * gc.nn[1] + iy) * nz + iz;
    T un[27][3];
    gather27(gc, u, ix, iy, iz, un);
    T f[3] = {0, 0, 0};
    T M[9];
    l1_row<T, false, false>(gc, gf, Chat, Ef, ix, iy, iz, un, f, M);
    store_out(y, b, gc.nnodes, n, f, MODE, dmask ? dmask[n] : uint8_t(0));
}

template <typename T>
__global__ void __launch_bounds__(TPB) k_l1_gs(Grid gc, Grid gf, const T *__restrict__ Chat,
                                               const T *__restrict__ Ef, T *__restrict__ u, const T *__restrict__ b,
                                               const uint8_t *__restrict__ dmask, int cx, int cy, int cz,
                                               int forward) {
    const int mx = (gc.nn[0] - cx + 1) / 2, my = (gc.ydet - cy + 1) / 2, mz = (gc.nn[2] - cz + 1) / 2;
    const int t = blockIdx.x * TPB + threadIdx.x;
    if (t >= mx * my * mz) return;
    const int jx = t / (my * mz), r = t - jx * my * mz, jy = r / mz, jz = r - jy * mz;
    const int ix = 2 * jx + cx, iy = 2 * jy + cy, iz = 2 * jz + cz;
    const int N = gc.nnodes, n = (ix * gc.nn[1] + iy) * gc.nn[2] + iz;
    const uint8_t dm = dmask ? dmask[n] : uint8_t(0);
    if (dm == 7) return;
    T un[27][3];
    gather27(gc, u, ix, iy, iz, un);
    T f[3] = {0, 0, 0};
    T M[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    l1_row<T, true, true>(gc, gf, Chat, Ef, ix, iy, iz, un, f, M);
    const T bms[3] = {b[n] - f[0], b[N + n] - f[1], b[2 * N + n] - f[2]};
    gs_update(u, N, n, bms, M, dm, forward);
}

// ---- level-1 K u element by element in the Walsh basis (reflection-symmetric element matrix).
// With the Walsh basis W[l, k] = prod_{axes a in k} s_a(l) (s_a(l) = +-1 the side of local node l along a,
// per displacement component), the child matrices Chat_fi = R_fi Chat_0 R_fi (R_fi: reflection across the
// axes of fi, which permutes the nodes and flips the reflected displacement components) become sign flips
// of Chat_0 in that basis, so the coarse element matrix sum_fi E_fi Chat_fi reads
//   (W^T K_E W)[(k, a), (k', c)] = Cw[(k, a), (k', c)] Ehat[k ^ k' ^ e_a ^ e_c],
//   Cw = W^T Chat_0 W,  Ehat[d] = sum_fi (-1)^popcount(d & fi) E_fi,  e_a = the bit of axis a,
// and K_E u_E = W (Cw o Ehat) W^T u_E / 64 costs about 800 operations for all 24 outputs instead of
// 8 x 576 for the child products (W W^T = 8 I; the 1/64 is folded into the table Cw).
// In FP32 only, where it is bound by the same issue as the rows of l1_row_sep and reads the moduli and the iterate fewer
// times: residuals in us, this / those, 128 x 64 x 64 elements 13 / 11, 256 x 128 x 128 38 / 35, 384 x 192 x 192 98 / 103,
// 512 x 256 x 256 235 / 286 (FP64 384 x 192 x 192: 310 / 180). The tuner takes the faster.
// A workgroup owns a tile of WX x WY x WZ nodes, evaluates every element touching it into LDS and sums
// each owned node's eight element contributions in a fixed order (no atomics: deterministic).
constexpr int WX = 4, WY = 8, WZ = 8, WNT = WX * WY * WZ;
constexpr int WEX = WX + 1, WEY = WY + 1, WEZ = WZ + 1, WNE = WEX * WEY * WEZ;
static_assert(WNT == TPB, "one owned node per work-item");

// v: the element's nodal values [l][a] on entry, K_E v on exit
template <typename T>
__device__ __forceinline__ void l1_walsh_element(const T *__restrict__ Cw, const T Ef8[8], T v[8][3]) {
    T Eh[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) Eh[i] = Ef8[i];
    // Ehat = H E (H[d][fi] = (-1)^popcount(d & fi)), and w = W^T v, one axis at a time
#pragma unroll
    for (int bit = 4; bit >= 1; bit >>= 1)
#pragma unroll
        for (int lo = 0; lo < 8; ++lo) {
            if (lo & bit) continue;
            const int hi = lo | bit;
            const T e0 = Eh[lo], e1 = Eh[hi];
            Eh[lo] = e0 + e1;
            Eh[hi] = e0 - e1;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const T x0 = v[lo][a], x1 = v[hi][a];
                v[lo][a] = x0 + x1;
                v[hi][a] = x1 - x0;
            }
        }
    // out[k][a] = sum_d Ehat[d] sum_c Cw[(k, a), (k', c)] w[k'][c] with k' = k ^ d ^ e_a ^ e_c; rows and
    // columns of the constant mode k = 0 vanish (rigid translations)
    T out[8][3];
#pragma unroll
    for (int a = 0; a < 3; ++a) out[0][a] = T(0);
#pragma unroll
    for (int k = 1; k < 8; ++k)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            T acc = T(0);
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                T inner = T(0);
                bool any = false;
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int kp = k ^ d ^ (4 >> a) ^ (4 >> c);
                    if (kp == 0) continue;
                    inner += Cw[(3 * k + a) * 24 + 3 * kp + c] * v[kp][c];
                    any = true;
                }
                if (any) acc += Eh[d] * inner;
            }
            out[k][a] = acc;
        }
    // back to the nodes: v = W out
#pragma unroll
    for (int bit = 4; bit >= 1; bit >>= 1)
#pragma unroll
        for (int lo = 0; lo < 8; ++lo) {
            if (lo & bit) continue;
            const int hi = lo | bit;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const T x0 = out[lo][a], x1 = out[hi][a];
                out[lo][a] = x0 - x1;
                out[hi][a] = x0 + x1;
            }
        }
#pragma unroll
    for (int l = 0; l < 8; ++l)
#pragma unroll
        for (int a = 0; a < 3; ++a) v[l][a] = out[l][a];
}

// y (mode) K u over the nodes of rows below ydet (detached rows are left to the launcher); grid: one
// workgroup per node tile
template <typename T, int MODE>
__global__ void __launch_bounds__(TPB) k_l1_apply_w(Grid gc, Grid gf, const T *__restrict__ Cw,
                                                    const T *__restrict__ Ef, const T *__restrict__ u,
                                                    T *__restrict__ y, const T *__restrict__ b,
                                                    const uint8_t *__restrict__ dmask, int ntY, int ntZ) {
    __shared__ T sY[WNE * 24];
    const int N = gc.nnodes, sx = gc.nn[1] * gc.nn[2], sy = gc.nn[2];
    const int fz = gf.ne[2], fyz = gf.ne[1] * gf.ne[2];
    const int tz = blockIdx.x % ntZ, r0 = blockIdx.x / ntZ, ty = r0 % ntY, tx = r0 / ntY;
    const int x0 = tx * WX, y0 = ty * WY, z0 = tz * WZ;
    const int t = threadIdx.x;
    for (int el = t; el < WNE; el += TPB) {
        const int lx = el / (WEY * WEZ), rr = el - lx * WEY * WEZ, ly = rr / WEZ, lz = rr - ly * WEZ;
        const int ex = x0 - 1 + lx, ey = y0 - 1 + ly, ez = z0 - 1 + lz;
        T v[8][3];
        if ((unsigned)ex < (unsigned)gc.ne[0] && (unsigned)ey < (unsigned)gc.ne[1] && (unsigned)ez < (unsigned)gc.ne[2]) {
            const int n0 = (ex * gc.nn[1] + ey) * gc.nn[2] + ez;
            T Ef8[8];
            const int fb = eidx(gf, 2 * ex, 2 * ey, 2 * ez);
#pragma unroll
            for (int l = 0; l < 8; ++l) {
                const int nm = n0 + ((l >> 2) & 1) * sx + ((l >> 1) & 1) * sy + (l & 1);
#pragma unroll
                for (int a = 0; a < 3; ++a) v[l][a] = u[(size_t)a * N + nm];
                Ef8[l] = Ef[fb + ((l >> 2) & 1) * fyz + ((l >> 1) & 1) * fz + (l & 1)];
            }
            l1_walsh_element(Cw, Ef8, v);
        } else {
#pragma unroll
            for (int l = 0; l < 8; ++l)
#pragma unroll
                for (int a = 0; a < 3; ++a) v[l][a] = T(0);
        }
#pragma unroll
        for (int l = 0; l < 8; ++l)
#pragma unroll
            for (int a = 0; a < 3; ++a) sY[el * 24 + 3 * l + a] = v[l][a];
    }
    __syncthreads();
    const int ox = t / (WY * WZ), orr = t - ox * WY * WZ, oy = orr / WZ, oz = orr - oy * WZ;
    const int ix = x0 + ox, iy = y0 + oy, iz = z0 + oz;
    if (ix >= gc.nn[0] || iy >= gc.ydet || iz >= gc.nn[2]) return;
    T f[3] = {0, 0, 0};
#pragma unroll
    for (int l = 0; l < 8; ++l) {
        // the element with this node at local corner l: local element coordinates (o + 1 - bit)
        const int el = ((ox + 1 - ((l >> 2) & 1)) * WEY + (oy + 1 - ((l >> 1) & 1))) * WEZ + (oz + 1 - (l & 1));
#pragma unroll
        for (int a = 0; a < 3; ++a) f[a] += sY[el * 24 + 3 * l + a];
    }
    const int n = (ix * gc.nn[1] + iy) * gc.nn[2] + iz;
    store_out(y, b, N, n, f, MODE, dmask ? dmask[n] : uint8_t(0));
}

template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ double dpp_get(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// Level-1 node row from the fine moduli of an isotropic box element, by sum factorisation. The element matrix is a sum of
// products of 1D integrals over the axes, and so is its Galerkin coarsening: with I_pq(o) = sum over the 4 x 4 x 4 fine
// elements around the node of E times the integral of d_p phi_0 d_q phi_o over the element (phi the coarse shape
// functions of the node and of its neighbour at offset o), the 3 x 3 block of neighbour o is
//   B_cc = mu (I_xx + I_yy + I_zz) + (lambda + mu) I_cc,   B_cd = lambda I_cd + mu I_dc,
// and I_pq contracts E axis by axis with one of four functionals of the four fine cells along the axis: M (phi phi),
// D (phi' phi'), G (phi_0' phi_o), T (phi_0 phi_o'). Up to constant factors (kept in L1Coef), for cells c0 c1 | c2 c3:
//   o = -1: M = c0 + c1, D = -M, G = 3 c0 + c1, T = -(c0 + 3 c1);   o = +1: mirrored, G and T of opposite sign;
//   o = 0: M = (c0 + 7 c1 + 7 c2 + c3) / 2, D = c0 + c1 + c2 + c3, G = T = c0 + 3 c1 - 3 c2 - c3.
// That is about 840 operations per half row, in place of 2592 for the eight children's dense rows.
// A node has two work-items, one per side along x (h = 0 low, h = 1 high): each contracts its side's 2 x 4 x 4 cells with
// the neighbours of the outer and the centre plane, in x-mirrored order when h = 1 (which negates the x component of u and
// of the row), and the two rows are added with a lane exchange. The halves of a wavefront take one side each, so that
// neighbouring lanes read neighbouring nodes (interleaved lanes: residual 215 instead of 194 us in FP64).
// Bound by the latency of three rounds of moduli and, on the largest level, by reading the moduli once per colour; the
// nine sums and one layer's contractions fit three (FP64) and five (FP32) wavefronts per SIMD. Level 1 of 384 x 192 x 192:
// a sweep of eight colours 665 -> 537 us in FP64 and 420 -> 253 us in FP32, the residual 326 -> 194 and 98 -> 103 us; of
// 256 x 128 x 128: 303 -> 193 and 196 -> 100 us, 110 -> 58 and 38 -> 36 us (before: dense child rows with two work-items
// per node, and the residual element by element in the Walsh basis).
template <typename T>
struct L1CoefT {
    T mu[3], lm[3], cm[3], r;
};
template <typename T, int DL>
struct Ax4 {  // functionals of four cells at offset DL
    static __host__ __device__ __forceinline__ T M(T a, T b, T c, T d) {
        return DL < 0 ? a + b : DL > 0 ? c + d : T(0.5) * (a + d) + T(3.5) * (b + c);
    }
    static __host__ __device__ __forceinline__ T D(T a, T b, T c, T d) { return DL < 0 ? -(a + b) : DL > 0 ? -(c + d) : (a + b) + (c + d); }
    static __host__ __device__ __forceinline__ T G(T a, T b, T c, T d) {
        return DL < 0 ? T(3) * a + b : DL > 0 ? -(c + T(3) * d) : (a + T(3) * b) - (T(3) * c + d);
    }
    static __host__ __device__ __forceinline__ T T_(T a, T b, T c, T d) {
        return DL < 0 ? -(a + T(3) * b) : DL > 0 ? T(3) * c + d : (a + T(3) * b) - (T(3) * c + d);
    }
};
// one offset's weights I, its neighbour's values u, and the sums they are added to: V[c] += B_cc u_c, and without the
// scale of their pair of axes Q[xy, yx, xz, zx, yz, zy] += (I_dc + lambda / mu I_cd) u_d
template <typename T>
struct L1Sums {
    T V[3], Q[6];
};
template <typename T>
__device__ __forceinline__ void l1_offset(const L1CoefT<T> &k, T xx, T yy, T zz, T xy, T yx, T xz, T zx, T yz, T zy,
                                          const T u[3], L1Sums<T> &s) {
    const T S = k.mu[0] * xx + k.mu[1] * yy + k.mu[2] * zz;
    s.V[0] += (S + k.lm[0] * xx) * u[0];
    s.V[1] += (S + k.lm[1] * yy) * u[1];
    s.V[2] += (S + k.lm[2] * zz) * u[2];
    s.Q[0] += (yx + k.r * xy) * u[1];
    s.Q[1] += (xy + k.r * yx) * u[0];
    s.Q[2] += (zx + k.r * xz) * u[2];
    s.Q[3] += (xz + k.r * zx) * u[0];
    s.Q[4] += (zy + k.r * yz) * u[2];
    s.Q[5] += (yz + k.r * zy) * u[1];
}
// the half row's part of the offsets (., DY, DZ): Z fields Z*[x][y] of the cells contracted along z
template <typename T, int DY, int DZ, bool WANT_M>
__device__ __forceinline__ void l1_line(const L1CoefT<T> &k, const T (&ZM)[2][4], const T (&ZD)[2][4], const T (&ZG)[2][4],
                                        const T (&ZT)[2][4], const T uo[3], const T uc[3], L1Sums<T> &s, T M[6]) {
    using Y = Ax4<T, DY>;
    T mm[2], dm[2], gm[2], tm[2], md[2], mt[2], gt[2], mg[2], tg[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        mm[x] = Y::M(ZM[x][0], ZM[x][1], ZM[x][2], ZM[x][3]);
        dm[x] = DY ? -mm[x] : Y::D(ZM[x][0], ZM[x][1], ZM[x][2], ZM[x][3]);
        gm[x] = Y::G(ZM[x][0], ZM[x][1], ZM[x][2], ZM[x][3]);
        tm[x] = DY ? Y::T_(ZM[x][0], ZM[x][1], ZM[x][2], ZM[x][3]) : gm[x];
        md[x] = DZ ? -mm[x] : Y::M(ZD[x][0], ZD[x][1], ZD[x][2], ZD[x][3]);
        mt[x] = Y::M(ZT[x][0], ZT[x][1], ZT[x][2], ZT[x][3]);
        gt[x] = Y::G(ZT[x][0], ZT[x][1], ZT[x][2], ZT[x][3]);
        mg[x] = DZ ? Y::M(ZG[x][0], ZG[x][1], ZG[x][2], ZG[x][3]) : mt[x];
        tg[x] = Y::T_(ZG[x][0], ZG[x][1], ZG[x][2], ZG[x][3]);
    }
    // x: cells o (outer), i (inner)
    auto mo = [](const T *w) { return w[0] + w[1]; };               // outer plane: M, -D
    auto go = [](const T *w) { return T(3) * w[0] + w[1]; };        // G
    auto t3 = [](const T *w) { return w[0] + T(3) * w[1]; };        // -T; centre plane: G, T
    auto mc = [](const T *w) { return T(0.5) * w[0] + T(3.5) * w[1]; };  // centre plane: M (D as mo)
    l1_offset(k, -mo(mm), mo(dm), mo(md), go(tm), -t3(gm), go(mt), -t3(mg), mo(gt), mo(tg), uo, s);
    const T xx = mo(mm), yy = mc(dm), zz = mc(md), xy = t3(tm), yx = t3(gm), xz = t3(mt), zx = t3(mg), yz = mc(gt), zy = mc(tg);
    l1_offset(k, xx, yy, zz, xy, yx, xz, zx, yz, zy, uc, s);
    if (WANT_M && DY == 0 && DZ == 0) {
        const T S = k.mu[0] * xx + k.mu[1] * yy + k.mu[2] * zz;
        M[0] = S + k.lm[0] * xx;
        M[1] = S + k.lm[1] * yy;
        M[2] = S + k.lm[2] * zz;
        M[3] = k.cm[0] * (T(1) + k.r) * xy;  // G = T at the node itself
        M[4] = k.cm[1] * (T(1) + k.r) * xz;
        M[5] = k.cm[2] * (T(1) + k.r) * yz;
    }
}
// keeps what is derived from `at` behind the sums so far: the compiler would otherwise request every layer's operands
// first and hold them all
template <typename T>
__device__ __forceinline__ void l1_pin(unsigned &at, L1Sums<T> &s) {
    asm volatile("" : "+v"(at), "+v"(s.V[0]), "+v"(s.V[1]), "+v"(s.V[2]), "+v"(s.Q[0]), "+v"(s.Q[1]), "+v"(s.Q[2]),
                 "+v"(s.Q[3]), "+v"(s.Q[4]), "+v"(s.Q[5]));
}
template <typename T>
struct Vec2;
template <>
struct Vec2<float> { using t = float2; };
template <>
struct Vec2<double> { using t = double2; };

template <typename T, bool WANT_M>
__device__ __forceinline__ void l1_row_sep(const Grid &gc, const Grid &gf, const L1CoefT<T> &k, const T *__restrict__ Ef,
                                           const T *__restrict__ u, int ix, int iy, int iz, int h, T f[3], T M[6]) {
    const int N = gc.nnodes, sy = gc.nn[2], sx = gc.nn[1] * sy;
    const int fz = gf.ne[2], fyz = gf.ne[1] * gf.ne[2];
    const int n = ix * sx + iy * sy + iz;
    const T hs = h ? T(-1) : T(1);
    const bool xin = h ? ix < gc.ne[0] : ix > 0;
    const int fx0 = h ? 2 * ix + 1 : 2 * ix - 2, fxs = h ? -fyz : fyz;
    L1Sums<T> s;
#pragma unroll
    for (int c = 0; c < 3; ++c) s.V[c] = s.Q[c] = s.Q[3 + c] = T(0);
    const int ox = h ? sx : -sx;
    const T *__restrict__ u1 = u + N, *__restrict__ u2 = u + (size_t)2 * N;
    // the six values of a line (fixed offsets along y and z) of the two planes, requested one line ahead; a neighbour
    // outside the grid has weight zero and reads the node itself
    T nxt[6];
    auto request = [&](unsigned nn, int dy, int dz) {
        const bool in = (unsigned)(iy + dy) < (unsigned)gc.nn[1] && (unsigned)(iz + dz) < (unsigned)gc.nn[2];
        const unsigned mc = in ? nn + dy * sy + dz : nn, mo = xin ? mc + ox : mc;
        nxt[0] = u[mo];
        nxt[1] = u1[mo];
        nxt[2] = u2[mo];
        nxt[3] = u[mc];
        nxt[4] = u1[mc];
        nxt[5] = u2[mc];
    };
    request(n, -1, -1);
    auto line = [&](auto DYc, auto DZc, const T(&ZM)[2][4], const T(&ZD)[2][4], const T(&ZG)[2][4], const T(&ZT)[2][4]) {
        constexpr int DY = decltype(DYc)::value, DZ = decltype(DZc)::value;
        T uo[3] = {hs * nxt[0], nxt[1], nxt[2]}, uc[3] = {hs * nxt[3], nxt[4], nxt[5]};
        if (DY < 1 || DZ < 1) {
            unsigned nn = n;
            l1_pin(nn, s);
            request(nn, DY < 1 ? DY + 1 : -1, DY < 1 ? DZ : DZ + 1);
        }
        l1_line<T, DY, DZ, WANT_M>(k, ZM, ZD, ZG, ZT, uo, uc, s, M);
    };
    auto layer = [&](auto DZc) {
        constexpr int DZ = decltype(DZc)::value;
        using Z = Ax4<T, DZ>;
        // cells E[x: outer, inner][y][z], zero outside the grid; read again for each layer, since holding
        // them would cost the registers of a wavefront per SIMD
        unsigned eb = (unsigned)(fx0 * fyz);
        l1_pin(eb, s);
        T E[2][4][4];
#pragma unroll
        for (int zz = 0; zz < 2; ++zz)
#pragma unroll
            for (int yy = 0; yy < 2; ++yy) {
                const int ey = iy - 1 + yy, ez = iz - 1 + zz;
                const bool ok = xin && (unsigned)ey < (unsigned)gc.ne[1] && (unsigned)ez < (unsigned)gc.ne[2];
                const unsigned at = ok ? eb + (unsigned)(2 * ey * fz + 2 * ez) : 0u;  // element counts fit 31 bits
                if ((DZ < 0 && zz == 1) || (DZ > 0 && zz == 0)) continue;  // only the cells shared with the neighbour
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 2; ++y) {
                        // rows of fine elements are even in number and length, so a pair along z is aligned
                        const auto v = *reinterpret_cast<const typename Vec2<T>::t *>(Ef + (at + (ok ? (unsigned)(x * fxs + y * fz) : 0u)));
                        E[x][2 * yy + y][2 * zz] = ok ? v.x : T(0);
                        E[x][2 * yy + y][2 * zz + 1] = ok ? v.y : T(0);
                    }
            }
        T ZM[2][4], ZD[2][4], ZG[2][4], ZT[2][4];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                T *e = E[x][y];
                if (DZ > 0) e[0] = e[1] = T(0);
                if (DZ < 0) e[2] = e[3] = T(0);
                ZM[x][y] = Z::M(e[0], e[1], e[2], e[3]);
                ZD[x][y] = Z::D(e[0], e[1], e[2], e[3]);
                ZG[x][y] = Z::G(e[0], e[1], e[2], e[3]);
                ZT[x][y] = DZ ? Z::T_(e[0], e[1], e[2], e[3]) : ZG[x][y];
            }
        line(std::integral_constant<int, -1>(), DZc, ZM, ZD, ZG, ZT);
        __builtin_amdgcn_sched_barrier(0);
        line(std::integral_constant<int, 0>(), DZc, ZM, ZD, ZG, ZT);
        __builtin_amdgcn_sched_barrier(0);
        line(std::integral_constant<int, 1>(), DZc, ZM, ZD, ZG, ZT);
        __builtin_amdgcn_sched_barrier(0);
    };
    layer(std::integral_constant<int, -1>());
    layer(std::integral_constant<int, 0>());
    layer(std::integral_constant<int, 1>());
    f[0] = hs * (s.V[0] + k.cm[0] * s.Q[0] + k.cm[1] * s.Q[2]);
    f[1] = s.V[1] + k.cm[0] * s.Q[1] + k.cm[2] * s.Q[4];
    f[2] = s.V[2] + k.cm[1] * s.Q[3] + k.cm[2] * s.Q[5];
#pragma unroll
    for (int a = 0; a < 3; ++a) f[a] += __shfl_xor(f[a], 32, 64);  // the other work-item of the pair
    if (WANT_M) {
        M[3] *= hs;
        M[4] *= hs;
#pragma unroll
        for (int q = 0; q < 6; ++q) M[q] += __shfl_xor(M[q], 32, 64);
    }
}

template <typename T>
__global__ void __launch_bounds__(TPB, sizeof(T) == 8 ? 2 : 4) k_l1_gs_sep(Grid gc, Grid gf, L1CoefT<T> k, const T *__restrict__ Ef,
                                                   T *__restrict__ u, const T *__restrict__ b,
                                                   const uint8_t *__restrict__ dmask, int cx, int cy, int cz, int forward) {
    const int mx = (gc.nn[0] - cx + 1) / 2, my = (gc.ydet - cy + 1) / 2, mz = (gc.nn[2] - cz + 1) / 2;
    const int t = xcd_remap(blockIdx.x, gridDim.x) * (TPB / 2) + threadIdx.x / 64 * 32 + threadIdx.x % 32,
              h = threadIdx.x >> 5 & 1;
    if (t >= mx * my * mz) return;  // both work-items of a pair
    const int jx = t / (my * mz), r = t - jx * my * mz, jy = r / mz, jz = r - jy * mz;
    const int ix = 2 * jx + cx, iy = 2 * jy + cy, iz = 2 * jz + cz;
    const int N = gc.nnodes, n = (ix * gc.nn[1] + iy) * gc.nn[2] + iz;
    const uint8_t dm = dmask ? dmask[n] : uint8_t(0);
    if (dm == 7) return;  // both work-items of a pair
    T f[3], S[6];
    l1_row_sep<T, true>(gc, gf, k, Ef, u, ix, iy, iz, h, f, S);
    if (h) return;
    const T bms[3] = {b[n] - f[0], b[N + n] - f[1], b[2 * N + n] - f[2]};
    const T M[9] = {S[0], S[3], S[4], S[3], S[1], S[5], S[4], S[5], S[2]};
    gs_update(u, N, n, bms, M, dm, forward);
}

// y (mode) K u over the nodes of rows below ydet, two work-items per node
template <typename T, int MODE>
__global__ void __launch_bounds__(TPB, sizeof(T) == 8 ? 2 : 4) k_l1_apply_sep(Grid gc, Grid gf, L1CoefT<T> k, const T *__restrict__ Ef,
                                                      const T *__restrict__ u, T *__restrict__ y, const T *__restrict__ b,
                                                      const uint8_t *__restrict__ dmask) {
    const int nz = gc.nn[2], slab = gc.ydet * nz;
    const int t = xcd_remap(blockIdx.x, gridDim.x) * (TPB / 2) + threadIdx.x / 64 * 32 + threadIdx.x % 32,
              h = threadIdx.x >> 5 & 1;
    if (t >= gc.nn[0] * slab) return;
    const int ix = t / slab, r = t - ix * slab, iy = r / nz, iz = r - iy * nz;
    const int n = (ix * gc.nn[1] + iy) * nz + iz;
    T f[3], M[6];
    l1_row_sep<T, false>(gc, gf, k, Ef, u, ix, iy, iz, h, f, M);
    if (!h) store_out(y, b, gc.nnodes, n, f, MODE, dmask ? dmask[n] : uint8_t(0));
}

// ------------------------------------------------------------------ assembled block rows
// LANE nodes (one in FP64, two neighbours of a z-row in FP32: eight bytes of every block entry) are worked on by the
// sixteen lanes of one DPP row: lane p holds neighbour slots p and p + 16 (27 in all), so the nodes' 243 block entries
// and 81 neighbour values each are requested at once, in one round of loads, and the rows are summed by four DPP
// exchanges without LDS. A colour pass over a small level is bound by that one memory round; over a large level it
// streams the interleaved rows.
// Time per colour, averaged over the block levels of a hierarchy: 64 x 32 x 32 FP64 10.4 -> 4.3 us, 176 x 88 x 72 FP64
// 13.6 -> 7.5 us, 208 x 112 x 96 FP64 16.2 -> 9.9 us (before: four work-items per node). In FP32 one node per row of lanes
// reads four bytes a lane, which no level of 100,000 nodes or more can be streamed with: sweeps and residuals of
// 97 x 49 x 49 nodes 105 and 77 us with one node, 71 and 44 with two, of 193 x 97 x 97 nodes 655 and 610, 454 and 429 (FP64
// 839 and 820 us, 4.2 TB/s).
// sum over the sixteen lanes of a DPP row, the same in every lane
template <typename T>
__device__ __forceinline__ T row16_sum(T v) {
    v += dpp_get<0xB1>(v);   // quad_perm [1, 0, 3, 2]
    v += dpp_get<0x4E>(v);   // quad_perm [2, 3, 0, 1]
    v += dpp_get<0x141>(v);  // row_half_mirror
    v += dpp_get<0x140>(v);  // row_mirror
    return v;
}

// tile and workgroup of the two-launch sweep: 27 of the 32 rows of lanes hold a node at the first colour
constexpr int BP_TY = 4, BP_TZ = 12, BP_NT = 512;

constexpr int RL = 16;          // lanes per node
constexpr int RN16 = TPB / RL;  // rows of lanes per workgroup
constexpr int DIAG_LANE = 13;   // the lane that holds the nodes' own slot

// A row's results are written by lane 13 (its first node) and lane 12 (its second): which node is this lane's, if any
template <typename T>
__device__ __forceinline__ int lane_node(int p) {
    return p == DIAG_LANE ? 0 : BlockRows<T>::LANE == 2 && p == DIAG_LANE - 1 ? 1 : BlockRows<T>::LANE;
}

// LANE neighbouring nodes of a z-row of one colour: the first one's coordinates and index, how many there are
struct LaneNodes {
    int ix, iy, iz, n, count;
    size_t at;  // entry 0 of slot 0 of their block rows
};
template <typename T>
__device__ __forceinline__ bool lane_nodes(const Grid &g, size_t base, int c, int row, LaneNodes &r) {
    constexpr int LANE = BlockRows<T>::LANE;
    const int cx = (c >> 2) & 1, cy = (c >> 1) & 1, cz = c & 1;
    const int mx = (g.nn[0] - cx + 1) / 2, my = (g.ydet - cy + 1) / 2, mz = (g.nn[2] - cz + 1) / 2;
    const int mq = BlockRows<T>::row_nodes(g, cz) / LANE;
    if (row >= mx * my * mq) return false;
    const int jx = row / (my * mq), q = row - jx * my * mq, jy = q / mq, jz = (q - jy * mq) * LANE;
    r.ix = 2 * jx + cx;
    r.iy = 2 * jy + cy;
    r.iz = 2 * jz + cz;
    r.n = (r.ix * g.nn[1] + r.iy) * g.nn[2] + r.iz;
    r.count = min(LANE, mz - jz);
    r.at = BlockRows<T>::offset(g, base, c, jx, jy, jz);
    return true;
}

// row f = sum_s B_s u_s and, with WANT_M, diagonal block M of node lane_node(p) of the nodes r
template <typename T, bool WANT_M>
__device__ __forceinline__ void block_row16(const Grid &g, const T *__restrict__ blocks, int p, const LaneNodes &r,
                                            const T *__restrict__ u, T f[3], T M[9]) {
    using R = BlockRows<T>;
    const int N = g.nnodes, sy = g.nn[2], sx = g.nn[1] * sy;
    T B[2][9][R::LANE], un[2][R::LANE][3];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const bool real = p + RL * h < 27;
        const int s = real ? p + RL * h : 26;  // the idle lanes of the second half repeat slot 26 with u = 0
        const int q = (s * 171) >> 9;          // s / 3
        const int dx = ((s * 57) >> 9) - 1, dy = q - 3 * (dx + 1) - 1, dz = s - 3 * q - 1;
        const bool okxy = real && (unsigned)(r.ix + dx) < (unsigned)g.nn[0] && (unsigned)(r.iy + dy) < (unsigned)g.nn[1];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const T *e = blocks + (r.at + R::entry(k, s));
            if constexpr (R::LANE == 2) {
                const float2 v = *reinterpret_cast<const float2 *>(e);
                B[h][k][0] = v.x;
                B[h][k][1] = v.y;
            } else {
                B[h][k][0] = *e;
            }
        }
#pragma unroll
        for (int e = 0; e < R::LANE; ++e) {
            const bool ok = okxy && (unsigned)(r.iz + 2 * e + dz) < (unsigned)g.nn[2];
            const int m = ok ? r.n + dx * sx + dy * sy + dz + 2 * e : r.n;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const T v = u[(size_t)c * N + m];
                un[h][e][c] = ok ? v : T(0);
            }
        }
    }
    const bool second = lane_node<T>(p) == 1;
#pragma unroll
    for (int e = 0; e < R::LANE; ++e)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            T acc = B[0][3 * a][e] * un[0][e][0];
            acc += B[0][3 * a + 1][e] * un[0][e][1];
            acc += B[0][3 * a + 2][e] * un[0][e][2];
#pragma unroll
            for (int c = 0; c < 3; ++c) acc += B[1][3 * a + c][e] * un[1][e][c];
            acc = row16_sum(acc);
            f[a] = e == 0 || second ? acc : f[a];
        }
    if (WANT_M)
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            M[k] = B[0][k][0];
            if constexpr (R::LANE == 2) {
                const T v = dpp_get<0xE5>(B[0][k][1]);  // quad_perm [1, 1, 2, 3]: lane 12 takes lane 13's
                M[k] = second ? v : M[k];
            }
        }
}

// grid.y = colour class (the rows are stored by class)
template <typename T, int MODE>
__global__ void __launch_bounds__(TPB) k_block_apply(Grid g, const T *__restrict__ blocks, const T *__restrict__ u,
                                                     T *__restrict__ y, const T *__restrict__ b,
                                                     const uint8_t *__restrict__ dmask) {
    const int p = threadIdx.x % RL, e = lane_node<T>(p);
    LaneNodes r;
    if (!lane_nodes<T>(g, BlockRows<T>::class_base(g, blockIdx.y), blockIdx.y, blockIdx.x * RN16 + threadIdx.x / RL, r))
        return;
    T f[3];
    block_row16<T, false>(g, blocks, p, r, u, f, nullptr);
    const int n = r.n + 2 * e;
    if (e < r.count) store_out(y, b, g.nnodes, n, f, MODE, dmask ? dmask[n] : uint8_t(0));
}

// One colour of the block Gauss-Seidel sweep; the lanes that hold the diagonal blocks update the nodes.
template <typename T>
__global__ void __launch_bounds__(TPB) k_block_gs(Grid g, const T *__restrict__ blocks, T *__restrict__ u,
                                                  const T *__restrict__ b, const uint8_t *__restrict__ dmask,
                                                  size_t base, int colour, int forward) {
    const int p = threadIdx.x % RL, e = lane_node<T>(p), N = g.nnodes;
    LaneNodes r;
    if (!lane_nodes<T>(g, base, colour, blockIdx.x * RN16 + threadIdx.x / RL, r)) return;
    // requested with the rows, so that the update waits for no second round
    const int n = r.n + 2 * e;
    uint8_t dm = 7;
    T bn[3] = {0, 0, 0};
    if (e < r.count) {
        dm = dmask ? dmask[n] : uint8_t(0);
#pragma unroll
        for (int c = 0; c < 3; ++c) bn[c] = b[(size_t)c * N + n];
    }
    T f[3], M[9];
    block_row16<T, true>(g, blocks, p, r, u, f, M);
    if (dm != 7) {
        const T bms[3] = {bn[0] - f[0], bn[1] - f[1], bn[2] - f[2]};
        gs_update(u, N, n, bms, M, dm, forward);
    }
}

// One x-parity of the colour sweep in one launch (a sweep is two): the four colours of a parity only see the other
// parity's planes and each other, so a workgroup takes a (y, z) tile of one plane, holds its values in LDS and applies the
// four in-plane colours in order, each on the tile grown by the halo that the later colours read ((1,3), (1,2), (0,1),
// (0,0) nodes in (y, z); the neighbouring tiles recompute it from the same inputs). Sixteen lanes per node as in
// block_row16, and a node for every row of lanes at each of the four positions: all block rows are requested before the
// first colour, the off-plane part of the sums is taken as they arrive, and what a colour waits for is only three values
// from LDS (a lane has at most one slot in the plane: s = 9 .. 17 are lanes 9 .. 15 and 0, 1). Bound by latency: about
// 3.5 us of launch, one round of loads and four colours, 9 us against 15 for four colour launches. Requested one colour
// ahead instead of all at once (tiles of 4 x 8): 12 us, where all at once took 10.
// uin: the planes of this parity before the sweep, unb: the neighbour planes, uout (!= uin): receives this parity's
// planes, every node. zin bit 0 / 1: uin / unb is zero.
template <typename T, int TY, int TZ, int NT, bool FWD>
__global__ void __launch_bounds__(NT) k_block_gs_plane(Grid g, typename BlockRows<T>::Bases bases,
                                                       const T *__restrict__ blocks, const T *__restrict__ uin,
                                                       const T *__restrict__ unb, T *__restrict__ uout,
                                                       const T *__restrict__ b, const uint8_t *__restrict__ dmask,
                                                       int parity, int ntY, int ntZ, int zin) {
    constexpr int HY = 2, HZ = 4, RY = TY + 2 * HY, RZ = TZ + 2 * HZ, CS = RY * RZ;
    static_assert(TY % 2 == 0 && TZ % 2 == 0 && (TY / 2 + 1) * (TZ / 2 + 3) <= NT / RL, "one node per row of lanes");
    __shared__ T su[3 * CS], sb[3 * CS];
    const int N = g.nnodes, nx = g.nn[0], ny = g.nn[1], nz = g.nn[2];
    const int ix = parity + 2 * blockIdx.y, tz = blockIdx.x % ntZ, ty = blockIdx.x / ntZ;
    const int y0 = ty * ny / ntY, y1 = (ty + 1) * ny / ntY, z0 = tz * nz / ntZ, z1 = (tz + 1) * nz / ntZ;
    const int t = threadIdx.x, p = t % RL, row = t / RL;
    // this lane's two neighbour slots (see block_row16)
    int off[2], dy[2], dz[2], slot[2];
    bool okx[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const bool real = p + RL * h < 27;
        const int s = real ? p + RL * h : 26, q = (s * 171) >> 9;
        const int dx = ((s * 57) >> 9) - 1;
        slot[h] = s;
        dy[h] = q - 3 * (dx + 1) - 1;
        dz[h] = s - 3 * q - 1;
        okx[h] = real && dx != 0 && (unsigned)(ix + dx) < (unsigned)nx && !(zin & 2);
        off[h] = (dx * ny + dy[h]) * nz + dz[h];
    }
    const int hp = p < 2 ? 1 : 0;  // the slot in the plane
    const bool inplane = p < 2 || p >= 9;
    T B[4][2][9], un[4][2][3];
    int li[4];
    bool act[4], okp[4];
    uint8_t dm[4];
#pragma unroll
    for (int pos = 0; pos < 4; ++pos) {
        const int sub = FWD ? pos : 3 - pos, cy = (sub >> 1) & 1, cz = sub & 1, hy = pos < 2 ? 1 : 0, hz = 3 - pos;
        int ya = max(y0 - hy, 0), za = max(z0 - hz, 0);
        const int yb = min(y1 + hy, g.ydet), zb = min(z1 + hz, nz);
        ya += (ya & 1) != cy;
        za += (za & 1) != cz;
        const int nr = yb > ya ? (yb - ya + 1) / 2 : 0, nc = zb > za ? (zb - za + 1) / 2 : 0, ncs = max(nc, 1);
        act[pos] = row < nr * nc;
        const int wr = row / ncs;
        const int iy = act[pos] ? ya + 2 * wr : cy, iz = act[pos] ? za + 2 * (row - wr * ncs) : cz;
        const int n = (ix * ny + iy) * nz + iz;
        const int col = 4 * parity + sub;
        const size_t bo = BlockRows<T>::offset(g, bases.at[col], col, ix >> 1, iy >> 1, iz >> 1);
        li[pos] = act[pos] ? (iy - y0 + HY) * RZ + iz - z0 + HZ : HY * RZ + HZ;
        dm[pos] = 7;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool ok = (unsigned)(iy + dy[h]) < (unsigned)ny && (unsigned)(iz + dz[h]) < (unsigned)nz;
#pragma unroll
            for (int k = 0; k < 9; ++k) B[pos][h][k] = act[pos] ? blocks[bo + BlockRows<T>::entry(k, slot[h])] : T(0);
#pragma unroll
            for (int c = 0; c < 3; ++c) un[pos][h][c] = act[pos] && okx[h] && ok ? unb[(size_t)c * N + n + off[h]] : T(0);
            if (h == hp) okp[pos] = inplane && ok;
        }
        if (p == DIAG_LANE && act[pos]) dm[pos] = dmask ? dmask[n] : uint8_t(0);
    }
    for (int w = t; w < 3 * CS; w += NT) {
        const int c = w / CS, q = w - c * CS, ly = q / RZ, lz = q - ly * RZ, gy = y0 - HY + ly, gz = z0 - HZ + lz;
        const bool in = (unsigned)gy < (unsigned)ny && (unsigned)gz < (unsigned)nz;
        const size_t m = (size_t)c * N + ((size_t)ix * ny + gy) * nz + gz;
        sb[w] = in ? b[m] : T(0);
        su[w] = in && !(zin & 1) ? uin[m] : T(0);
    }
    T acc[4][3];
#pragma unroll
    for (int pos = 0; pos < 4; ++pos)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            T v = T(0);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int c = 0; c < 3; ++c) v += B[pos][h][3 * a + c] * un[pos][h][c];
            acc[pos][a] = v;
        }
    const int lo = (hp ? dy[1] : dy[0]) * RZ + (hp ? dz[1] : dz[0]);
    __syncthreads();
#pragma unroll
    for (int pos = 0; pos < 4; ++pos) {
        if (act[pos]) {  // whole rows of sixteen lanes
            T v[3], f[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) v[c] = okp[pos] ? su[c * CS + li[pos] + lo] : T(0);
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                T s = acc[pos][a];
#pragma unroll
                for (int c = 0; c < 3; ++c) s += (hp ? B[pos][1][3 * a + c] : B[pos][0][3 * a + c]) * v[c];
                f[a] = row16_sum(s);
            }
            if (p == DIAG_LANE && dm[pos] != 7) {
                const T bms[3] = {sb[li[pos]] - f[0], sb[CS + li[pos]] - f[1], sb[2 * CS + li[pos]] - f[2]};
                gs_update(su, CS, li[pos], bms, B[pos][0], dm[pos], FWD ? 1 : 0);
            }
        }
        __syncthreads();
    }
    const int OY = y1 - y0, OZ = z1 - z0;
    for (int w = t; w < 3 * TY * TZ; w += NT) {
        const int c = w / (TY * TZ), q = w - c * TY * TZ, oy = q / TZ, oz = q - oy * TZ;
        if (oy < OY && oz < OZ)
            uout[(size_t)c * N + ((size_t)ix * ny + y0 + oy) * nz + z0 + oz] = su[c * CS + (oy + HY) * RZ + oz + HZ];
    }
}

// ------------------------------------------------------------------ cached element matrices
template <typename T, int MODE>
__global__ void __launch_bounds__(TPB) k_elem_apply(Grid g, const T *__restrict__ Ke, const T *__restrict__ u,
                                                    T *__restrict__ y) {
    const int t = blockIdx.x * TPB + threadIdx.x;
    if (t >= g.nnodes) return;
    const int nz = g.nn[2], ix = t / (g.nn[1] * nz), iy = (t / nz) % g.nn[1], iz = t % nz;
    T un[27][3];
    gather27(g, u, ix, iy, iz, un);
    T f[3] = {0, 0, 0};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int i = (e >> 2) & 1, j = (e >> 1) & 1, k = e & 1;
        const int ex = ix - i, ey = iy - j, ez = iz - k;
        if (!((unsigned)ex < (unsigned)g.ne[0] && (unsigned)ey < (unsigned)g.ne[1] && (unsigned)ez < (unsigned)g.ne[2]))
            continue;
        const int ln = 4 * i + 2 * j + k;
        const T *K = Ke + (size_t)eidx(g, ex, ey, ez) * 576;
#pragma unroll
        for (int m = 0; m < 8; ++m)
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const T um = un[slot_of(m, i, j, k)][d];
#pragma unroll
                for (int c = 0; c < 3; ++c) f[c] += K[(3 * ln + c) * 24 + 3 * m + d] * um;
            }
    }
    store_out(y, (const T *)nullptr, g.nnodes, t, f, MODE, uint8_t(0));
}

// ------------------------------------------------------------------ transfers
// r_c(n) = sum_{o in {-1,0,1}^3} prod_d (1 - |o_d|/2) r_f(2n + o) over active fine nodes
// (MultigridSolver.hh:214-275); every detached coarse row is zeroed. The weights are separable, so a
// work-item owns one coarse (y, z) column and marches along x through its chunk of coarse planes: each
// fine plane's 3x3 in-plane sum is formed once and serves the coarse planes on both sides of it.
// xc (optional): the coarse iterate, zeroed in the same pass (the cycle starts the coarse level from zero)
template <typename T>
__global__ void __launch_bounds__(TPB) k_restrict(Grid gf, Grid gc, const T *__restrict__ rf, T *__restrict__ rc,
                                                  T *__restrict__ xc, int xchunk) {
    const int ncy = gc.nn[1], ncz = gc.nn[2];
    const int t = blockIdx.x * TPB + threadIdx.x;
    if (t >= ncy * ncz) return;
    const int cy = t / ncz, cz = t - cy * ncz;
    const int cx0 = blockIdx.y * xchunk, cx1 = min(cx0 + xchunk, gc.nn[0]);
    const bool act = cy < gc.ydet;
    const int Nf = gf.nnodes, Nc = gc.nnodes, nfy = gf.nn[1], nfz = gf.nn[2];
    auto plane = [&](int fx, T out[3]) {
        out[0] = out[1] = out[2] = T(0);
        if (!act || (unsigned)fx >= (unsigned)gf.nn[0]) return;
#pragma unroll
        for (int oy = -1; oy <= 1; ++oy) {
            const int fy = 2 * cy + oy;
            if ((unsigned)fy >= (unsigned)gf.ydet) continue;
#pragma unroll
            for (int oz = -1; oz <= 1; ++oz) {
                const int fz = 2 * cz + oz;
                if ((unsigned)fz >= (unsigned)nfz) continue;
                const T w = T((oy ? 0.5 : 1.0) * (oz ? 0.5 : 1.0));
                const int m = (fx * nfy + fy) * nfz + fz;
                out[0] += w * rf[m];
                out[1] += w * rf[Nf + m];
                out[2] += w * rf[2 * Nf + m];
            }
        }
    };
    T prev[3];
    plane(2 * cx0 - 1, prev);
    for (int cx = cx0; cx < cx1; ++cx) {
        T a[3], b[3];
        plane(2 * cx, a);
        plane(2 * cx + 1, b);
        const int n = (cx * ncy + cy) * ncz + cz;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            rc[(size_t)c * Nc + n] = T(0.5) * prev[c] + a[c] + T(0.5) * b[c];
            if (xc) xc[(size_t)c * Nc + n] = T(0);
            prev[c] = b[c];
        }
    }
}

// x_f (+)= P x_c, trilinear (MultigridSolver.hh:162-212). accumulate: active fine rows only
// (accum_interpolation); otherwise every fine row is overwritten (interpolation). A work-item owns one
// fine (y, z) column and marches along x through its chunk of coarse elements: the bilinear (y, z)
// interpolant of each coarse plane is formed once and serves the fine planes on both sides of it.
template <typename T>
__global__ void __launch_bounds__(TPB) k_interpolate(Grid gf, Grid gc, const T *__restrict__ xc, T *__restrict__ xf,
                                                     int accumulate, int xchunk) {
    const int nfy = gf.nn[1], nfz = gf.nn[2];
    const int rows = accumulate ? gf.ydet : nfy;
    const int t = blockIdx.x * TPB + threadIdx.x;
    if (t >= rows * nfz) return;
    const int fy = t / nfz, fz = t - fy * nfz;
    const int ncy = gc.nn[1], ncz = gc.nn[2], Nc = gc.nnodes, Nf = gf.nnodes;
    // coarse rows / columns of the (y, z) interpolant and their weights (the second index is clamped
    // where its weight is zero)
    const int cy = min(fy >> 1, gc.ne[1]), cz = min(fz >> 1, gc.ne[2]);
    const bool oy = fy & 1, oz = fz & 1;
    const T wy1 = oy ? T(0.5) : T(0), wy0 = oy ? T(0.5) : T(1);
    const T wz1 = oz ? T(0.5) : T(0), wz0 = oz ? T(0.5) : T(1);
    const int cy1 = oy ? cy + 1 : cy, cz1 = oz ? cz + 1 : cz;
    const int o00 = cy * ncz + cz, o01 = cy * ncz + cz1, o10 = cy1 * ncz + cz, o11 = cy1 * ncz + cz1;
    auto inplane = [&](int cx, T out[3]) {
        const int pb = cx * ncy * ncz;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T *p = xc + (size_t)c * Nc + pb;
            out[c] = wy0 * (wz0 * p[o00] + wz1 * p[o01]) + wy1 * (wz0 * p[o10] + wz1 * p[o11]);
        }
    };
    auto put = [&](int fx, const T v[3]) {
        const size_t n = ((size_t)fx * nfy + fy) * nfz + fz;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (accumulate) xf[(size_t)c * Nf + n] += v[c];
            else xf[(size_t)c * Nf + n] = v[c];
        }
    };
    const int ne0 = gc.ne[0];
    const int e0 = blockIdx.y * xchunk, e1 = min(e0 + xchunk, ne0);
    T a[3];
    inplane(e0, a);
    for (int e = e0; e < e1; ++e) {
        T b[3];
        inplane(e + 1, b);
        put(2 * e, a);
        const T h[3] = {T(0.5) * (a[0] + b[0]), T(0.5) * (a[1] + b[1]), T(0.5) * (a[2] + b[2])};
        put(2 * e + 1, h);
        a[0] = b[0];
        a[1] = b[1];
        a[2] = b[2];
    }
    if (e1 == ne0) put(2 * ne0, a);  // the last fine plane, on the last coarse plane
}

inline unsigned nblocks(long count) { return (unsigned)((count + TPB - 1) / TPB); }


}  // namespace

// ------------------------------------------------------------------ launchers
#define VF_DISPATCH_MODE(KERNEL, T, mode, grid, ...)                                                        \
    switch (mode) {                                                                                         \
    case AM_SET: hipLaunchKernelGGL((KERNEL<T, AM_SET>), grid, dim3(TPB), 0, s, __VA_ARGS__); break;         \
    case AM_ADD: hipLaunchKernelGGL((KERNEL<T, AM_ADD>), grid, dim3(TPB), 0, s, __VA_ARGS__); break;         \
    case AM_SUB: hipLaunchKernelGGL((KERNEL<T, AM_SUB>), grid, dim3(TPB), 0, s, __VA_ARGS__); break;         \
    default: hipLaunchKernelGGL((KERNEL<T, AM_RESIDUAL>), grid, dim3(TPB), 0, s, __VA_ARGS__); break;        \
    }

template <typename T>
void launch_zero_detached(const Grid &g, T *y, hipStream_t s) {
    if (g.ydet >= g.nn[1]) return;
    const long cz = (long)g.nn[0] * (g.nn[1] - g.ydet) * g.nn[2];
    hipLaunchKernelGGL(k_zero_detached<T>, dim3(nblocks(cz)), dim3(TPB), 0, s, g, y);
    VF_HIP(hipGetLastError());
}

template <typename T>
void launch_fine_apply(const Grid &g, const T *K0, const T *E, const T *u, T *y, const T *b, const uint8_t *dmask,
                       int mode, hipStream_t s) {
    const long count = (long)g.nn[0] * g.ydet * g.nn[2];
    if (count > 0) { VF_DISPATCH_MODE(k_fine_apply, T, mode, dim3(nblocks(count)), g, K0, E, u, y, b, dmask); }
    if (mode == AM_SET && g.ydet < g.nn[1]) {
        const long cz = (long)g.nn[0] * (g.nn[1] - g.ydet) * g.nn[2];
        hipLaunchKernelGGL(k_zero_detached<T>, dim3(nblocks(cz)), dim3(TPB), 0, s, g, y);
    }
    VF_HIP(hipGetLastError());
}

// Every block of every child's matrix against the rows' formulas (see l1_row_sep) with that child's modulus alone
bool l1_rows_factorise(const L1Coef &k, const double *Chat) {
    // F[q][o + 1][cell]: functional q (M, D, G, T) at offset o of one of the four cells along an axis
    double F[4][3][4];
    auto fill = [&](auto A, int o) {
        using Ax = decltype(A);
        for (int cell = 0; cell < 4; ++cell) {
            const double c0 = cell == 0, c1 = cell == 1, c2 = cell == 2, c3 = cell == 3;
            F[0][o + 1][cell] = Ax::M(c0, c1, c2, c3);
            F[1][o + 1][cell] = Ax::D(c0, c1, c2, c3);
            F[2][o + 1][cell] = Ax::G(c0, c1, c2, c3);
            F[3][o + 1][cell] = Ax::T_(c0, c1, c2, c3);
        }
    };
    fill(Ax4<double, -1>(), -1);
    fill(Ax4<double, 0>(), 0);
    fill(Ax4<double, 1>(), 1);
    double most = 0;
    for (int i = 0; i < 8 * 576; ++i) most = std::max(most, std::fabs(Chat[i]));
    for (int fi = 0; fi < 8; ++fi)
        for (int l = 0; l < 8; ++l)
            for (int m = 0; m < 8; ++m) {
                double W[3][3];
                for (int p = 0; p < 3; ++p)
                    for (int q = 0; q < 3; ++q) {
                        W[p][q] = 1;
                        for (int a = 0; a < 3; ++a) {
                            const int bl = (l >> (2 - a)) & 1, bm = (m >> (2 - a)) & 1, bf = (fi >> (2 - a)) & 1;
                            W[p][q] *= F[p == q ? (a == p ? 1 : 0) : a == p ? 2 : a == q ? 3 : 0][bm - bl + 1][bl ? bf : 2 + bf];
                        }
                    }
                const double S = k.mu[0] * W[0][0] + k.mu[1] * W[1][1] + k.mu[2] * W[2][2];
                for (int c = 0; c < 3; ++c)
                    for (int d = 0; d < 3; ++d) {
                        const double v = c == d ? S + k.lm[c] * W[c][c] : k.cm[c + d - 1] * (W[d][c] + k.ratio * W[c][d]);
                        if (!(std::fabs(v - Chat[fi * 576 + (3 * l + c) * 24 + 3 * m + d]) <= 1e-13 * most)) return false;
                    }
            }
    return true;
}

template <typename T>
static L1CoefT<T> l1_coef(const L1Coef &c) {
    L1CoefT<T> r;
    for (int q = 0; q < 3; ++q) {
        r.mu[q] = (T)c.mu[q];
        r.lm[q] = (T)c.lm[q];
        r.cm[q] = (T)c.cm[q];
    }
    r.r = (T)c.ratio;
    return r;
}

template <typename T>
void launch_l1_apply(const Grid &gc, const Grid &gf, const T *Chat, const L1Coef &sep, const float *Cw, const T *Ef,
                     const T *u, T *y, const T *b, const uint8_t *dmask, int mode, bool reflect, hipStream_t s) {
    const long count = (long)gc.nn[0] * gc.ydet * gc.nn[2];
    if (count > 0 && reflect && Cw) {
        if constexpr (std::is_same<T, float>::value) {
            const int ntX = (gc.nn[0] + WX - 1) / WX, ntY = (gc.ydet + WY - 1) / WY, ntZ = (gc.nn[2] + WZ - 1) / WZ;
            const long tiles = (long)ntX * ntY * ntZ;
            if (tiles > INT_MAX) throw std::runtime_error("grid too large for the level-1 product");
            VF_DISPATCH_MODE(k_l1_apply_w, T, mode, dim3((unsigned)tiles), gc, gf, Cw, Ef, u, y, b, dmask, ntY, ntZ);
        } else {
            throw std::runtime_error("the Walsh-basis level-1 product is single precision");
        }
    } else if (count > 0 && reflect) {
        VF_DISPATCH_MODE(k_l1_apply_sep, T, mode, dim3(nblocks(2 * count)), gc, gf, l1_coef<T>(sep), Ef, u, y, b, dmask);
    } else if (count > 0) {
        VF_DISPATCH_MODE(k_l1_apply, T, mode, dim3(nblocks(count)), gc, gf, Chat, Ef, u, y, b, dmask);
    }
    if (mode == AM_SET && gc.ydet < gc.nn[1]) {
        const long cz = (long)gc.nn[0] * (gc.nn[1] - gc.ydet) * gc.nn[2];
        hipLaunchKernelGGL(k_zero_detached<T>, dim3(nblocks(cz)), dim3(TPB), 0, s, gc, y);
    }
    VF_HIP(hipGetLastError());
}

// rows of lanes that a colour's active nodes take
template <typename T>
static long block_lane_rows(const Grid &g, int color) {
    const long mx = (g.nn[0] - ((color >> 2) & 1) + 1) / 2, my = (g.ydet - ((color >> 1) & 1) + 1) / 2;
    return mx * my * (BlockRows<T>::row_nodes(g, color & 1) / BlockRows<T>::LANE);
}

template <typename T>
void launch_block_apply(const Grid &g, const T *blocks, const T *u, T *y, const T *b, const uint8_t *dmask, int mode,
                        hipStream_t s) {
    const long most = block_lane_rows<T>(g, 0);
    if (most > 0)
        VF_DISPATCH_MODE(k_block_apply, T, mode, dim3((unsigned)((most + RN16 - 1) / RN16), 8), g, blocks, u, y, b, dmask);
    if (mode == AM_SET && g.ydet < g.nn[1]) {
        const long cz = (long)g.nn[0] * (g.nn[1] - g.ydet) * g.nn[2];
        hipLaunchKernelGGL(k_zero_detached<T>, dim3(nblocks(cz)), dim3(TPB), 0, s, g, y);
    }
    VF_HIP(hipGetLastError());
}

template <typename T>
void launch_elem_apply(const Grid &g, const T *Ke, const T *u, T *y, int mode, hipStream_t s) {
    if (mode == AM_SET) hipLaunchKernelGGL((k_elem_apply<T, AM_SET>), dim3(nblocks(g.nnodes)), dim3(TPB), 0, s, g, Ke, u, y);
    else if (mode == AM_ADD) hipLaunchKernelGGL((k_elem_apply<T, AM_ADD>), dim3(nblocks(g.nnodes)), dim3(TPB), 0, s, g, Ke, u, y);
    else if (mode == AM_SUB) hipLaunchKernelGGL((k_elem_apply<T, AM_SUB>), dim3(nblocks(g.nnodes)), dim3(TPB), 0, s, g, Ke, u, y);
    else throw std::runtime_error("residual mode unsupported on cached element matrices");
    VF_HIP(hipGetLastError());
}

static inline long color_count(const Grid &g, int cx, int cy, int cz) {
    const long mx = (g.nn[0] - cx + 1) / 2, my = (g.ydet - cy + 1) / 2, mz = (g.nn[2] - cz + 1) / 2;
    return (mx > 0 && my > 0 && mz > 0) ? mx * my * mz : 0;
}

template <typename T>
void launch_fine_gs(const Grid &g, const T *K0, const T *E, T *u, const T *b, const uint8_t *dmask, int color,
                    int forward, hipStream_t s) {
    const int cx = (color >> 2) & 1, cy = (color >> 1) & 1, cz = color & 1;
    const long count = color_count(g, cx, cy, cz);
    if (!count) return;
    hipLaunchKernelGGL(k_fine_gs<T>, dim3(nblocks(count)), dim3(TPB), 0, s, g, K0, E, u, b, dmask, cx, cy, cz, forward);
    VF_HIP(hipGetLastError());
}

template <typename T>
void launch_l1_gs(const Grid &gc, const Grid &gf, const T *Chat, const L1Coef &sep, const T *Ef, T *u, const T *b,
                  const uint8_t *dmask, int color, int forward, bool reflect, hipStream_t s) {
    const int cx = (color >> 2) & 1, cy = (color >> 1) & 1, cz = color & 1;
    const long count = color_count(gc, cx, cy, cz);
    if (!count) return;
    if (reflect)
        hipLaunchKernelGGL(k_l1_gs_sep<T>, dim3(nblocks(2 * count)), dim3(TPB), 0, s, gc, gf, l1_coef<T>(sep), Ef, u, b,
                           dmask, cx, cy, cz, forward);
    else
        hipLaunchKernelGGL(k_l1_gs<T>, dim3(nblocks(count)), dim3(TPB), 0, s, gc, gf, Chat, Ef, u, b, dmask, cx, cy,
                           cz, forward);
    VF_HIP(hipGetLastError());
}

template <typename T>
void launch_block_gs(const Grid &g, const T *blocks, T *u, const T *b, const uint8_t *dmask, int color, int forward,
                     hipStream_t s) {
    const long rows = block_lane_rows<T>(g, color);
    if (rows <= 0) return;
    hipLaunchKernelGGL(k_block_gs<T>, dim3((unsigned)((rows + RN16 - 1) / RN16)), dim3(TPB), 0, s, g, blocks, u, b, dmask,
                       BlockRows<T>::class_base(g, color), color, forward);
    VF_HIP(hipGetLastError());
}

// A workgroup holds a compute unit with its registers, so a launch is one latency long while every workgroup has a unit of
// its own, and the halo (27 + 24 + 14 + 12 nodes for a tile of 12 per colour) costs nothing; beyond that the eight colour
// launches are faster. Sweeps in us, two launches / eight (FP64, FP32): 27x15x13 (112 workgroups) 16.7 / 28.3, 16.0 / 30.4;
// 33x17x17 (170) 18.7 / 28.6, 17.4 / 32.3; 41x21x21 (252) 23.6 / 29.2, 19.0 / 31.6; 45x23x19 (276) 37.7 / 29.6, 28.5 / 31.8;
// 65x33x33 (891) 76 / 50, 57 / 44.
bool block_gs_planes(const Grid &g) {
    const int ntY = (g.nn[1] + BP_TY - 1) / BP_TY, ntZ = (g.nn[2] + BP_TZ - 1) / BP_TZ;
    return (long)ntY * ntZ * ((g.nn[0] + 1) / 2) <= cu_count();
}

template <typename T>
void launch_block_gs_plane(const Grid &g, const T *blocks, const T *uin, const T *unb, T *uout, const T *b,
                           const uint8_t *dmask, int parity, int forward, hipStream_t s, int zin) {
    if (uin == uout) throw std::runtime_error("the two-launch sweep needs distinct input and output vectors");
    const int planes = (g.nn[0] - parity + 1) / 2;
    if (planes <= 0) return;
    const int ntY = (g.nn[1] + BP_TY - 1) / BP_TY, ntZ = (g.nn[2] + BP_TZ - 1) / BP_TZ;
    if (forward)
        hipLaunchKernelGGL((k_block_gs_plane<T, BP_TY, BP_TZ, BP_NT, true>), dim3(ntY * ntZ, planes), dim3(BP_NT), 0, s, g,
                           BlockRows<T>::bases(g), blocks, uin, unb, uout, b, dmask, parity, ntY, ntZ, zin);
    else
        hipLaunchKernelGGL((k_block_gs_plane<T, BP_TY, BP_TZ, BP_NT, false>), dim3(ntY * ntZ, planes), dim3(BP_NT), 0, s, g,
                           BlockRows<T>::bases(g), blocks, uin, unb, uout, b, dmask, parity, ntY, ntZ, zin);
    VF_HIP(hipGetLastError());
}

// x-chunks of a marching transfer: about TARGET workgroups in all, at least MINLEN planes per chunk; a
// small level (fewer than TARGET workgroups even at one plane each), whose launch is latency-bound, gets
// one plane per workgroup
static inline int transfer_chunks(unsigned planeBlocks, int len, int minLen) {
    constexpr unsigned TARGET = 2048;
    if ((long)planeBlocks * len <= (long)TARGET) return std::max(1, std::min(len, 65535));
    int c = (int)std::max(1u, TARGET / std::max(1u, planeBlocks));
    c = std::min(c, std::max(1, len / minLen));
    return std::max(1, std::min(c, 65535));
}
template <typename T>
void launch_restrict(const Grid &gf, const Grid &gc, const T *rf, T *rc, hipStream_t s, T *xzero) {
    if (gf.nn[0] != 2 * gc.nn[0] - 1 || gf.nn[1] != 2 * gc.nn[1] - 1 || gf.nn[2] != 2 * gc.nn[2] - 1)
        throw std::runtime_error("restriction: the fine grid is not the refinement of the coarse grid");
    const unsigned pb = nblocks((long)gc.nn[1] * gc.nn[2]);
    const int chunks = transfer_chunks(pb, gc.nn[0], 4);
    const int xchunk = (gc.nn[0] + chunks - 1) / chunks;
    const int nch = (gc.nn[0] + xchunk - 1) / xchunk;
    hipLaunchKernelGGL(k_restrict<T>, dim3(pb, nch), dim3(TPB), 0, s, gf, gc, rf, rc, xzero, xchunk);
    VF_HIP(hipGetLastError());
}

template <typename T>
void launch_interpolate(const Grid &gf, const Grid &gc, const T *xc, T *xf, int accumulate, hipStream_t s) {
    if (gf.nn[0] != 2 * gc.nn[0] - 1 || gf.nn[1] != 2 * gc.nn[1] - 1 || gf.nn[2] != 2 * gc.nn[2] - 1)
        throw std::runtime_error("interpolation: the fine grid is not the refinement of the coarse grid");
    const long count = (long)(accumulate ? gf.ydet : gf.nn[1]) * gf.nn[2];
    if (!count || gc.ne[0] < 1) return;
    const unsigned pb = nblocks(count);
    const int chunks = transfer_chunks(pb, gc.ne[0], 2);
    const int xchunk = (gc.ne[0] + chunks - 1) / chunks;
    const int nch = (gc.ne[0] + xchunk - 1) / xchunk;
    hipLaunchKernelGGL(k_interpolate<T>, dim3(pb, nch), dim3(TPB), 0, s, gf, gc, xc, xf, accumulate, xchunk);
    VF_HIP(hipGetLastError());
}

#define VF_INST(T)                                                                                                     \
    template void launch_zero_detached<T>(const Grid &, T *, hipStream_t);                                             \
    template void launch_fine_apply<T>(const Grid &, const T *, const T *, const T *, T *, const T *, const uint8_t *,  \
                                       int, hipStream_t);                                                              \
    template void launch_l1_apply<T>(const Grid &, const Grid &, const T *, const L1Coef &, const float *, const T *,    \
                                     const T *, T *, const T *, const uint8_t *, int, bool, hipStream_t);              \
    template void launch_block_apply<T>(const Grid &, const T *, const T *, T *, const T *, const uint8_t *, int,       \
                                        hipStream_t);                                                                  \
    template void launch_elem_apply<T>(const Grid &, const T *, const T *, T *, int, hipStream_t);                     \
    template void launch_fine_gs<T>(const Grid &, const T *, const T *, T *, const T *, const uint8_t *, int, int,      \
                                    hipStream_t);                                                                      \
    template void launch_l1_gs<T>(const Grid &, const Grid &, const T *, const L1Coef &, const T *, T *, const T *,    \
                                  const uint8_t *, int, int, bool, hipStream_t);                                                        \
    template void launch_block_gs_plane<T>(const Grid &, const T *, const T *, const T *, T *, const T *,               \
                                           const uint8_t *, int, int, hipStream_t, int);                               \
    template void launch_block_gs<T>(const Grid &, const T *, T *, const T *, const uint8_t *, int, int, hipStream_t); \
    template void launch_restrict<T>(const Grid &, const Grid &, const T *, T *, hipStream_t, T *);                   \
    template void launch_interpolate<T>(const Grid &, const Grid &, const T *, T *, int, hipStream_t);

VF_INST(double)
VF_INST(float)

}  // namespace vf
