// vf_kernels_walsh.hip -- element-centric fine K u in the Walsh (Hadamard) basis of the Q1 element.
//
// With W[k][m] = prod_a s_a(m)^{k_a} (s_a(m) = -1 or +1 for the low or high side of axis a; k, m in
// {0,1}^3, index 4x+2y+z), the element stiffness of an axis-aligned box with an orthotropic (in
// particular isotropic) elasticity tensor is K0 = (1/64) W^T Khat W where Khat = W K0 W^T has only 48
// nonzero entries: Khat[(k,d),(k,d)] and Khat[(k,d),(k ^ e_d ^ e_c, c)] for c != d with k_d != k_c
// (the monomials of the element's displacement basis are orthogonal under 2-point Gauss integration).
// One element product y_e = E_e K0 u_e therefore costs two 3-stage butterflies per component, 48 products with the
// Khat entries and 24 scalings by E_e, instead of the 576 multiply-adds of the dense 24 x 24 product
// (TPSStencils.hh:453-471); along the march below half of the butterflies are shared with the neighbouring
// element, which leaves 72 + 48 additions. The host verifies the sparsity
// on the actual K0 and selects this kernel only where it holds.
//
// Work layout: a workgroup owns a (y,z) tile of 16 x 16 element columns and marches along x. The node plane ahead
// is staged in LDS; each work-item reads the four corners of its column's face, takes the y and z stages of the
// butterflies on that face once (the plane's transformed values serve the element ahead and the one behind), forms the x
// stage and the products, and adds the two elements' contributions to a plane while they are still transformed, so that
// the y and z stages back are taken once per plane as well. The corner values of the four (y,z)-neighbouring columns
// are then added along z between lanes and along y through LDS, with one barrier a step. The tile's outer element
// row/column only serves its neighbours: a tile owns 15 x 15 node columns. Every node value is summed in the same order
// whatever the tiling, so results are deterministic.
//
// Measured against one with both butterflies per element, all corners through LDS, two barriers a step and the addresses
// formed in the loop (577 vector instructions a step, now 267), in us, K u / residual: 65x33x33 FP64 9.2 / 9.3 -> 7.1 /
// 7.1; 209x113x97 FP64 54.3 / 55.9 -> 41.7 / 43.0, FP32 36.6 / 37.4 -> 28.1 / 27.3; 257x129x129 FP64 85.6 / 111.9 -> 64.9 /
// 99.1, FP32 58.5 / 60.9 -> 45.1 / 45.0; 385x193x193 FP64 268 / 394 -> 249 / 322, FP32 173 / 227 -> 148 / 198. At the
// largest, K u is bound by neither the vector units (about 45%) nor the bytes (3.2 TB/s, 3.9 moved): requesting the planes two steps
// ahead costs registers that spill, and waiting for all of a step's loads before the next ones are requested changes
// nothing.
#include "vf_internal.hpp"

#include <algorithm>
#include <climits>

namespace vf {
namespace {

template <typename T>
using CT = __attribute__((address_space(4))) T;

constexpr int TE = 16;       // element columns per tile side
constexpr int TN = TE - 1;   // node columns owned per tile side
constexpr int RN = TE + 1;   // node columns staged per tile side
constexpr int NTW = TE * TE; // work-items

__device__ __forceinline__ constexpr int bitof(int a) { return 1 << (2 - a); }

// Rows of Khat coupled by its off-diagonal entries: (k, d) with (k ^ e_d ^ e_c, c) for c != d, k_d != k_c. They
// form 14 groups of one to three rows (listed as k * 3 + d), closed under the coupling, so the product can be
// formed one group at a time in place.
struct WalshGroup {
    int n;
    int r[3];
};
__device__ constexpr WalshGroup kWalshGroups[14] = {
    {1, {0, 0, 0}},   {1, {1, 0, 0}},   {1, {2, 0, 0}},    {2, {3, 14, 0}},  {2, {4, 8, 0}},
    {3, {5, 7, 12}},  {2, {6, 13, 0}},  {3, {9, 16, 20}},  {2, {10, 15, 0}}, {2, {11, 18, 0}},
    {2, {17, 19, 0}}, {1, {21, 0, 0}},  {1, {22, 0, 0}},   {1, {23, 0, 0}}};

// the y and z stages of the butterflies of one face (node 2j+k), forward (m -> index) and backward
template <typename T, bool FWD>
__device__ __forceinline__ void face_butterfly(T f[4][3]) {
#pragma unroll
    for (int bb = 2; bb > 0; bb >>= 1)
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            if (m & bb) continue;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const T lo = f[m][d], hi = f[m | bb][d];
                f[m][d] = FWD ? lo + hi : lo - hi;
                f[m | bb][d] = FWD ? hi - lo : lo + hi;
            }
        }
}

// z -> E Khat z / 64 of one element, [index][component], in place
template <typename T>
__device__ __forceinline__ void walsh_product(const T *__restrict__ C, T Ee, T v[8][3]) {
    // zh[k][d] = E (Khat[(k,d),(k,d)] z[k][d] + sum_{c != d, k_d != k_c} Khat[(k,d),(k^e_d^e_c,c)] z[..][c]) / 64,
    // group by group: a group's rows only read the group's own entries, so they are overwritten after the group
    // (the temporaries are one group, not a second 24-entry array)
#pragma unroll
    for (int gi = 0; gi < 14; ++gi) {
        const WalshGroup grp = kWalshGroups[gi];
        T out[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            if (q >= grp.n) continue;
            const int k = grp.r[q] / 3, d = grp.r[q] % 3;
            // coefficients of row group k (nine values, loaded through an opaque pointer so they are not
            // hoisted out of the element loop and spilled)
            const T *Cg = C + 16 * k;
            asm volatile("" : "+s"(Cg));
            const CT<T> *Ck = (const CT<T> *)Cg;
            T acc = Ck[3 * d + d] * v[k][d];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                if (c == d) continue;
                const int kd = (k & bitof(d)) ? 1 : 0, kc = (k & bitof(c)) ? 1 : 0;
                if (kd == kc) continue;
                acc += Ck[3 * d + c] * v[k ^ bitof(d) ^ bitof(c)][c];
            }
            out[q] = Ee * acc;
        }
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            if (q >= grp.n) continue;
            v[grp.r[q] / 3][grp.r[q] % 3] = out[q];
        }
    }
}

// base plus a byte offset: a scalar base and a 32-bit lane offset are one addressing mode of the global loads
template <typename U>
__device__ __forceinline__ const U *at(const U *base, unsigned off) {
    return reinterpret_cast<const U *>(reinterpret_cast<const char *>(base) + off);
}
template <typename U>
__device__ __forceinline__ U *at(U *base, unsigned off) {
    return reinterpret_cast<U *>(reinterpret_cast<char *>(base) + off);
}

// v of the next lane of its sixteen (the last one: 0)
__device__ __forceinline__ float next_lane(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x101, 0xf, 0xf, true));  // row_shl:1
}
__device__ __forceinline__ double next_lane(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x101, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x101, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// dotp (SET mode, optional): per-workgroup partial sums of <u, y> over the owned nodes, in a fixed order.
template <typename T, int MODE>
__global__ void __launch_bounds__(NTW, sizeof(T) == 8 ? 3 : 5) k_ku_walsh(Grid g, const T *__restrict__ C, const T *__restrict__ E,
                                                  const T *__restrict__ u, T *__restrict__ y, const T *__restrict__ b,
                                                  const uint8_t *__restrict__ dmask, int ntZ, int xchunk,
                                                  double *__restrict__ dotp) {
    __shared__ T su[2][3 * RN * RN];  // node planes, double-buffered
    __shared__ T sp[2][3 * NTW];      // per element column: the plane's sums at its low-y edge, double-buffered
    __shared__ double sred[NTW / 64];
    const int N = g.nnodes, nx = g.nn[0], ny = g.nn[1], nz = g.nn[2];
    const int tiles = gridDim.x;
    const int logical = xcd_remap(blockIdx.x + blockIdx.y * tiles, tiles * gridDim.y);
    const int tile = logical % tiles, chunk = logical / tiles;
    const int tz = tile % ntZ, ty = tile / ntZ;
    const int sy = TN * ty - 1, sz = TN * tz - 1;  // first element (and staged node) of the tile
    const int x0 = chunk * xchunk, x1 = min(x0 + xchunk, nx);
    const int t = threadIdx.x, ly = t / TE, lz = t - ly * TE;
    const int ey = sy + ly, ez = sz + lz;
    const bool elemOk = (unsigned)ey < (unsigned)g.ne[1] && (unsigned)ez < (unsigned)g.ne[2];
    const int Y = ey + 1, Z = ez + 1;  // node owned by this work-item
    const bool owner = ly < TN && lz < TN && Y < g.ydet && Z < nz;

    // Node planes are fetched one step ahead into registers (per component PF values per work-item) and written to LDS at
    // the start of the next step, so the global-load latency overlaps a whole step of compute. Every access is a plane's
    // base in scalar registers and a byte offset inside the plane, found once: address arithmetic inside the march took
    // more vector instructions (a third of them products, at a quarter of the rate) than the element's own.
    constexpr int FACE = RN * RN, PF = (FACE + NTW - 1) / NTW;
    const size_t nplane = (size_t)ny * nz, eplane = (size_t)g.ne[1] * g.ne[2];
    unsigned po[PF];
    bool pok[PF];
#pragma unroll
    for (int q = 0; q < PF; ++q) {
        const int w = t + q * NTW, ry = w / RN, rz = w - ry * RN, gy = sy + ry, gz = sz + rz;
        pok[q] = w < FACE && (unsigned)gy < (unsigned)ny && (unsigned)gz < (unsigned)nz;
        po[q] = pok[q] ? (unsigned)(((size_t)gy * nz + gz) * sizeof(T)) : 0u;
    }
    const unsigned no = owner ? (unsigned)(((size_t)Y * nz + Z) * sizeof(T)) : 0u;
    const unsigned eo = elemOk ? (unsigned)(((size_t)ey * g.ne[2] + ez) * sizeof(T)) : 0u;
    T pf[PF][3];
    auto fetch_plane = [&](int ix) {
        const bool in = (unsigned)ix < (unsigned)nx;  // uniform
        const T *up = u + (in ? ix : 0) * nplane;
#pragma unroll
        for (int q = 0; q < PF; ++q) {
            pf[q][0] = pf[q][1] = pf[q][2] = T(0);
            if (in && pok[q]) {
#pragma unroll
                for (int c = 0; c < 3; ++c) pf[q][c] = *at(up + (size_t)c * N, po[q]);
            }
        }
    };
    auto store_plane = [&](int buf) {
#pragma unroll
        for (int q = 0; q < PF; ++q) {
            const int w = t + q * NTW;
            if ((q + 1) * NTW <= FACE || w < FACE) {
#pragma unroll
                for (int c = 0; c < 3; ++c) su[buf][c * FACE + w] = pf[q][c];
            }
        }
    };
    auto fetch_E = [&](int ex) {
        T v = T(0);
        if ((unsigned)ex < (unsigned)g.ne[0] && elemOk) v = *at(E + ex * eplane, eo);
        return v;
    };
    auto read_face = [&](int buf, T f[4][3]) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = q >> 1, k = q & 1;
#pragma unroll
            for (int c = 0; c < 3; ++c) f[q][c] = su[buf][c * RN * RN + (ly + j) * RN + lz + k];
        }
    };

    T zold[4][3], carry[4][3];  // of the node plane behind: transformed values, transformed contributions so far
    T fin[3] = {0, 0, 0};       // plane being finished: its sums at the high-y edge
    T bv[3] = {0, 0, 0};        // and the right-hand side, or u for the dot product, at the owned node
    uint8_t dm = 0;
    double dacc = 0;  // <u, y> over the owned nodes (SET mode with dotp)
#pragma unroll
    for (int q = 0; q < 4; ++q) carry[q][0] = carry[q][1] = carry[q][2] = T(0);
    // node plane ix: corners (j,k) of the elements at (ly+1-j, lz+1-k) that hold node (Y, Z), summed along z, then y
    auto finish = [&](int ix, int buf) {
        T *yp = y + ix * nplane;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const T f = fin[c] + sp[buf][c * NTW + t + TE];
            T out = MODE == AM_RESIDUAL ? bv[c] - f : f;
            if (dm & (1 << c)) out = T(0);
            *at(yp + (size_t)c * N, no) = out;
            if (MODE == AM_SET && dotp) dacc += (double)out * (double)bv[c];
        }
    };
    fetch_plane(x0 - 1);
    store_plane((x0 + 1) & 1);
    fetch_plane(x0);
    T Enext = fetch_E(x0 - 1);
    __syncthreads();
    read_face((x0 + 1) & 1, zold);
    face_butterfly<T, true>(zold);
    for (int ex = x0 - 1; ex < x1; ++ex) {
        // element plane ex: node planes ex (face i = 0, transformed in zold) and ex + 1 (face i = 1)
        const int buf = (ex + 1) & 1;
        store_plane(buf);     // plane ex + 1, fetched during the previous step
        fetch_plane(ex + 2);  // consumed by the next step
        const T Ee = Enext;
        Enext = fetch_E(ex + 1);
        // The only barrier of a step: plane ex + 1 and the edge sums of plane ex - 1 are in LDS. Both buffers alternate, so
        // what is overwritten in this step was last read before this barrier's predecessor.
        __syncthreads();
        if (ex > x0 && owner) finish(ex - 1, buf ^ 1);
        if (owner && ex >= x0) {  // right-hand side and mask of plane ex, which the next step finishes
            if (dmask) dm = *at(dmask + ex * nplane, no / (unsigned)sizeof(T));
            const T *src = (MODE == AM_RESIDUAL ? b : u) + ex * nplane;
            if (MODE == AM_RESIDUAL || dotp) {
#pragma unroll
                for (int c = 0; c < 3; ++c) bv[c] = *at(src + (size_t)c * N, no);
            }
        }
        T f[4][3], v[8][3];
        read_face(buf, f);
        face_butterfly<T, true>(f);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                v[q][c] = zold[q][c] + f[q][c];
                v[4 + q][c] = f[q][c] - zold[q][c];
                zold[q][c] = f[q][c];
            }
        walsh_product<T>(C, Ee, v);
        T w[4][3];  // plane ex: this element and the one behind, transformed
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                w[q][c] = carry[q][c] + (v[q][c] - v[4 + q][c]);
                carry[q][c] = v[q][c] + v[4 + q][c];
            }
        if (ex >= x0) {  // uniform
            face_butterfly<T, false>(w);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                fin[c] = w[3][c] + next_lane(w[2][c]);
                sp[buf][c * NTW + t] = w[1][c] + next_lane(w[0][c]);
            }
        }
    }
    __syncthreads();
    if (owner) finish(x1 - 1, x1 & 1);
    if (MODE == AM_SET && dotp) {
        for (int o = 32; o > 0; o >>= 1) dacc += __shfl_xor(dacc, o, 64);
        if ((t & 63) == 0) sred[t >> 6] = dacc;
        __syncthreads();
        if (t == 0) {
            double r = 0;
            for (int i = 0; i < NTW / 64; ++i) r += sred[i];
            dotp[logical] = r;  // chunk-major: the partials of one x-chunk are contiguous
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(256) k_zero_rows_w(Grid g, T *__restrict__ y) {
    const int nz = g.nn[2], rows = g.nn[1] - g.ydet, slab = rows * nz;
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= g.nn[0] * slab) return;
    const int ix = t / slab, r = t - ix * slab, iy = g.ydet + r / nz, iz = r % nz;
    const int n = (ix * g.nn[1] + iy) * nz + iz;
    y[n] = T(0);
    y[g.nnodes + n] = T(0);
    y[(size_t)2 * g.nnodes + n] = T(0);
}

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

}  // namespace

// Four workgroups per compute unit, no more than run at once: a second round costs more than it hides, e.g. in FP64
// (K u, us) 66 against 74 at 256x128x128 elements, 146 against 151 at 320x160x160. Where an FP64 field alone no longer fits
// the 256 MB last-level cache the launch is bound by HBM and the other way round: as many as asked for 249 against 259 at
// 384x192x192, 405 / 416 at 448x224x224, 673 / 732 at 512x256x256 (residuals 324 / 332, 512 / 521, 902 / 909); in FP32 the
// cap stays the better one (512x256x256: 404 against 445).
static int walsh_xchunk_of(const Grid &g, const void *kern, int alignX, size_t word) {
    const int tiles = cdiv(g.ydet, TN) * cdiv(g.nn[2], TN);
    const bool hbm = word == sizeof(double) && (size_t)3 * g.nnodes * word > (size_t)256 << 20;
    const int chunks0 = plane_chunks(tiles, g.nn[0], 4 * cu_count(), hbm ? INT_MAX : resident_workgroups(kern, NTW));
    int xchunk = cdiv(g.nn[0], chunks0);
    if (alignX > 0) {  // the largest divisor of alignX not above xchunk: no x-chunk straddles a multiple of alignX
        int best = 1;
        for (int d = 1; d <= alignX && d <= xchunk; ++d)
            if (alignX % d == 0) best = d;
        xchunk = best;
    }
    return xchunk;
}
int walsh_xchunk(const Grid &g, int mode, int alignX) {
    const void *kern = mode == AM_RESIDUAL ? (const void *)k_ku_walsh<double, AM_RESIDUAL> : (const void *)k_ku_walsh<double, AM_SET>;
    return walsh_xchunk_of(g, kern, alignX, sizeof(double));
}

size_t walsh_partials(const Grid &g) { return (size_t)cdiv(g.ydet, TN) * cdiv(g.nn[2], TN) * g.nn[0]; }

template <typename T>
void launch_fine_apply_walsh(const Grid &g, const T *C, const T *E, const T *u, T *y, const T *b,
                             const uint8_t *dmask, int mode, hipStream_t s, double *dotPartials, double *dotOut,
                             int alignX, size_t dotCapacity) {
    if (mode != AM_SET && mode != AM_RESIDUAL) throw std::runtime_error("Walsh K u supports the SET and RESIDUAL modes");
    if (dotOut && (mode != AM_SET || !dotPartials)) throw std::runtime_error("the fused <u, K u> needs SET mode and partials");
    if (dotOut && g.ydet <= 0) launch_fill<double>(1, dotOut, 0.0, s);
    if (g.ydet > 0) {
        // tiles cover node columns [TN*t, TN*t + TN); rows beyond ydet are skipped by the owners
        const int ntY = cdiv(g.ydet, TN), ntZ = cdiv(g.nn[2], TN);
        const int tiles = ntY * ntZ;
        const void *kern = mode == AM_RESIDUAL ? (const void *)k_ku_walsh<T, AM_RESIDUAL> : (const void *)k_ku_walsh<T, AM_SET>;
        const int xchunk = walsh_xchunk_of(g, kern, alignX, sizeof(T));
        const int chunks = cdiv(g.nn[0], xchunk);
        if (chunks > 65535) throw std::runtime_error("grid too large for the Walsh K u");
        if (dotOut && (size_t)tiles * chunks > dotCapacity)
            throw std::runtime_error("Walsh K u: " + std::to_string((size_t)tiles * chunks) +
                                     " partial sums do not fit the buffer of " + std::to_string(dotCapacity));
        const dim3 grid(tiles, chunks);
        if (mode == AM_RESIDUAL)
            hipLaunchKernelGGL((k_ku_walsh<T, AM_RESIDUAL>), grid, dim3(NTW), 0, s, g, C, E, u, y, b, dmask, ntZ, xchunk,
                               nullptr);
        else
            hipLaunchKernelGGL((k_ku_walsh<T, AM_SET>), grid, dim3(NTW), 0, s, g, C, E, u, y, b, dmask, ntZ, xchunk,
                               dotOut ? dotPartials : nullptr);
        if (dotOut) launch_final_sum(dotPartials, (int)(grid.x * grid.y), dotOut, s);
    }
    if (mode == AM_SET && g.ydet < g.nn[1]) {
        const long cz = (long)g.nn[0] * (g.nn[1] - g.ydet) * g.nn[2];
        hipLaunchKernelGGL(k_zero_rows_w<T>, dim3((unsigned)((cz + 255) / 256)), dim3(256), 0, s, g, y);
    }
    VF_HIP(hipGetLastError());
}

template void launch_fine_apply_walsh<double>(const Grid &, const double *, const double *, const double *, double *,
                                              const double *, const uint8_t *, int, hipStream_t, double *, double *,
                                              int, size_t);
template void launch_fine_apply_walsh<float>(const Grid &, const float *, const float *, const float *, float *,
                                             const float *, const uint8_t *, int, hipStream_t, double *, double *, int,
                                             size_t);

}  // namespace vf
