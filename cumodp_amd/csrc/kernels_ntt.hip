// kernels_ntt.hip -- stand-alone NTT and elementwise kernels for gfx950.
//
// Replaces the reference's one-stage-per-launch radix-2 Stockham passes
// (src/stockham.cu:75-397, src/list_stockham.cu:108-576, src/fft_aux.cu:70-322)
// with:
//   * k_ntt_lds / k_col_fwd + k_row_out / k_col_ntt -- natural-order
//     transforms (the multiplies are in mul_mx.hip).
#include <algorithm>

#include "internal.h"
#include "ntt_core.h"

namespace cm {

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous range of logical blocks so that neighbouring column tiles (which
// share 128-byte lines) meet in the same L2.
CM_DEV int xcd_remap(int b, int nb) {
    if (nb & 7) return b;
    return (b & 7) * (nb >> 3) + (b >> 3);
}

// ---------------------------------------------------------------------------
// natural-order forward DFT of rows inside one workgroup
// ---------------------------------------------------------------------------
template <int LOGL, int C>
__global__ __launch_bounds__((Tile<LOGL, C, false>::T)) void k_ntt_lds(
    u32 *__restrict__ X, int64_t m, const u32 *__restrict__ lv, Mod md, u32 sc) {
    using TL = Tile<LOGL, C, false>;
    __shared__ u32 lds[TL::LDS_WORDS];
    const int L = TL::L;
    const int64_t r0 = (int64_t)blockIdx.x * C;
    constexpr int PER = TL::WORDS / TL::T;
    u32 xa[PER];
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = threadIdx.x + r * TL::T, c = idx >> LOGL, i = idx & (L - 1);
        xa[r] = (r0 + c < m) ? X[(r0 + c) * L + i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = threadIdx.x + r * TL::T, c = idx >> LOGL, i = idx & (L - 1);
        lds[TL::addr(c, i)] = xa[r];
    }
    __syncthreads();
    cm_tile_dif<TL>(lds, lv, md);
#pragma unroll
    for (int c = 0; c < C; ++c) {
        if (r0 + c >= m) break;
        for (int i = threadIdx.x; i < L; i += TL::T) {
            u32 v = lds[TL::addr(c, (int)cm_brev(i, LOGL))];
            if (sc) v = cm_mul_tw(v, sc, md.p, md.np);
            X[(r0 + c) * L + i] = v;
        }
    }
}

// ---------------------------------------------------------------------------
// four-step pieces: an n-word array viewed as 2^k1 rows x 2^k2 columns
// ---------------------------------------------------------------------------
// Forward column transforms (DIF, bit-reversed rows) in place, followed by the
// outer twiddle w_n^(i2 * k1).  grid.x: column tiles, grid.y: arrays.
template <int LOGL1, int C>
__global__ __launch_bounds__((Tile<LOGL1, C, true>::T))
__attribute__((amdgpu_waves_per_eu(8, 8))) void k_col_fwd(
    u32 *__restrict__ X0, int64_t stride, int logn2, const u32 *__restrict__ lv,
    const u32 *__restrict__ olo, const u32 *__restrict__ ohi, Mod md) {
    using TL = Tile<LOGL1, C, true>;
    __shared__ u32 lds[TL::LDS_WORDS];
    u32 *X = X0 + (int64_t)blockIdx.y * stride;
    const int64_t n2 = (int64_t)1 << logn2;
    const int c0 = xcd_remap(blockIdx.x, gridDim.x) * C;
    constexpr int PER = TL::WORDS / TL::T;
    u32 xa[PER];
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = threadIdx.x + r * TL::T, i = idx / C, c = idx % C;
        xa[r] = X[i * n2 + c0 + c];
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) lds[TL::phys(threadIdx.x + r * TL::T)] = xa[r];
    __syncthreads();
    cm_tile_dif<TL>(lds, lv, md);
    constexpr int LOM = (1 << kOuterLoBits) - 1;
    for (int idx = threadIdx.x; idx < TL::WORDS; idx += TL::T) {
        const int i = idx / C, c = idx % C;
        const u32 e = (u32)(c0 + c) * cm_brev(i, LOGL1);
        X[i * n2 + c0 + c] = cm_mul_tw(
            cm_mont_lazy(lds[TL::phys(idx)], olo[e & LOM], md.p, md.np),
            ohi[e >> kOuterLoBits], md.p, md.np);
    }
}

// Row transforms for the natural-order stand-alone DFT: the workgroup takes
// the CR rows whose frequency index k1 = brev(row) is consecutive, and writes
// Y[k1 + k2 * n1] (out of place).  grid.y: arrays.
template <int LOGL2, int CR>
__global__ __launch_bounds__((Tile<LOGL2, CR, false>::T)) void k_row_out(
    const u32 *__restrict__ X0, u32 *__restrict__ Y0, int64_t stride, int logn1,
    const u32 *__restrict__ lv, Mod md, u32 sc) {
    using TL = Tile<LOGL2, CR, false>;
    __shared__ u32 lds[TL::LDS_WORDS];
    const u32 *X = X0 + (int64_t)blockIdx.y * stride;
    u32 *Y = Y0 + (int64_t)blockIdx.y * stride;
    const int L = TL::L;
    const int64_t n1 = (int64_t)1 << logn1;
    const int k10 = blockIdx.x * CR;
    constexpr int PER = TL::WORDS / TL::T;
    u32 xa[PER];
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = threadIdx.x + r * TL::T, c = idx >> LOGL2, i = idx & (L - 1);
        xa[r] = X[(int64_t)cm_brev(k10 + c, logn1) * L + i];
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = threadIdx.x + r * TL::T, c = idx >> LOGL2, i = idx & (L - 1);
        lds[TL::addr(c, i)] = xa[r];
    }
    __syncthreads();
    cm_tile_dif<TL>(lds, lv, md);
    for (int idx = threadIdx.x; idx < TL::WORDS; idx += TL::T) {
        const int k2 = idx / CR, c = idx % CR;
        u32 v = lds[TL::addr(c, (int)cm_brev(k2, LOGL2))];
        if (sc) v = cm_mul_tw(v, sc, md.p, md.np);
        Y[k10 + c + k2 * n1] = v;
    }
}

// Natural-order column transforms DFT_m (x) I_ncols of a row-major
// 2^LOGM x ncols array, in place (the column half of the bivariate DFT,
// src/list_stockham.cu:1193-1201); output scaled by sc when sc != 0.
template <int LOGM, int C>
__global__ __launch_bounds__((Tile<LOGM, C, true>::T)) void k_col_ntt(
    u32 *__restrict__ X0, int64_t ncols, int64_t bstride, const u32 *__restrict__ lv, Mod md,
    u32 sc) {
    using TL = Tile<LOGM, C, true>;
    __shared__ u32 lds[TL::LDS_WORDS];
    u32 *X = X0 + (int64_t)blockIdx.y * bstride;   // grid.y: arrays bstride words apart
    const int64_t c0 = (int64_t)blockIdx.x * C;
    constexpr int PER = TL::WORDS / TL::T;
    u32 xa[PER];
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = threadIdx.x + r * TL::T, i = idx / C, c = idx % C;
        xa[r] = (c0 + c < ncols) ? X[i * ncols + c0 + c] : 0u;
    }
#pragma unroll
    for (int r = 0; r < PER; ++r) lds[TL::phys(threadIdx.x + r * TL::T)] = xa[r];
    __syncthreads();
    md = cm_rebind(md);
    cm_tile_dif<TL>(lds, lv, md);
    for (int idx = threadIdx.x; idx < TL::WORDS; idx += TL::T) {
        const int i = idx / C, c = idx % C;
        if (c0 + c >= ncols) continue;
        u32 v = lds[TL::phys((int)cm_brev(i, LOGM) * C + c)];
        if (sc) v = cm_mul_tw(v, sc, md.p, md.np);
        X[i * ncols + c0 + c] = v;
    }
}

// ---------------------------------------------------------------------------
// elementwise kernels
// ---------------------------------------------------------------------------
__global__ void k_pointwise(u32 *__restrict__ Y, const u32 *__restrict__ X, int64_t n, u32 p,
                            u32 pinv, u32 r2) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        Y[i] = cm_mont(cm_mont(Y[i], X[i], p, pinv), r2, p, pinv);
}

__global__ void k_scale(u32 *__restrict__ X, int64_t n, u32 a, u32 aq, u32 p) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        X[i] = cm_shoup(X[i], a, aq, p);
}

// W[j] = w^j: each thread raises w to its index by square-and-multiply on
// Montgomery residues (wm = w * 2^32 mod p, one = 2^32 mod p).
__global__ void k_powers(u32 *__restrict__ W, int64_t n, u32 wm, u32 one, u32 p, u32 pinv) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        u32 r = one, x = wm;
        for (u64 e = (u64)i; e; e >>= 1) {
            if (e & 1) r = cm_mont(r, x, p, pinv);
            x = cm_mont(x, x, p, pinv);
        }
        W[i] = cm_mont(r, 1u, p, pinv);
    }
}

__global__ void k_fill(u32 *__restrict__ X, int64_t n, u32 v) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        X[i] = v;
}

static int ew_blocks(int64_t n) {
    int64_t b = (n + 255) / 256;
    return (int)(b < 8192 ? (b < 1 ? 1 : b) : 8192);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static Mod mod_of(const Family *fam) { return Mod{fam->p, fam->np}; }

// Montgomery form of the output scale `scale` (0 when scale == 1: no scaling)
static u32 scale_mont(u32 scale, u32 p) { return scale % p == 1u ? 0u : cm_host_mont(scale % p, p); }

// Pointwise constant of an N = 2^logn multiply: the Montgomery form of
// 2^32 / N mod p (see cm_tile_multiply).
u32 mul_scale(int logn, u32 p) {
    u32 ninv = cm_host_inv(cm_host_pow(2, logn, p), p);
    return cm_host_mont(cm_host_mul(cm_host_r1(p), ninv, p), p);
}

template <int LOGL>
static constexpr int rows_per_wg() { return LOGL >= 10 ? 1 : (1 << (LOGL >= 10 ? 0 : 10 - LOGL)); }

template <int LOGL>
static hipError_t ntt_lds_t(u32 *X, int64_t m, const u32 *lv, u32 sc, const Family *fam,
                            hipStream_t s) {
    constexpr int C = rows_per_wg<LOGL>();
    using TL = Tile<LOGL, C, false>;
    const int64_t nb = (m + C - 1) / C;
    ProfScope ps(kProfNttLds, s);
    hipLaunchKernelGGL((k_ntt_lds<LOGL, C>), dim3((unsigned)nb), dim3(TL::T), 0, s, X, m, lv,
                       mod_of(fam), sc);
    return hipGetLastError();
}

hipError_t launch_ntt_lds(int k, u32 *X, int64_t m, bool inverse, u32 scale, const Family *fam,
                          hipStream_t s) {
    if (m <= 0) return hipSuccess;
    const u32 *lv = inverse ? fam->lvi : fam->lv;
    const u32 sc = scale_mont(scale, fam->p);
    switch (k) {
#define CM_CASE(K) case K: return ntt_lds_t<K>(X, m, lv, sc, fam, s);
        CM_CASE(4) CM_CASE(5) CM_CASE(6) CM_CASE(7) CM_CASE(8) CM_CASE(9) CM_CASE(10)
        CM_CASE(11) CM_CASE(12) CM_CASE(13)
#undef CM_CASE
    }
    return hipErrorInvalidValue;
}

// column tile width: C columns x 2^LOGL1 rows <= 16384 words (at most 4096
// columns)
template <int LOGL1>
static constexpr int col_tile() {
    return (16384 >> LOGL1) > 4096 ? 4096 : (16384 >> LOGL1);
}

template <int LOGL1>
static hipError_t col_fwd_t(u32 *X, int cnt, int64_t stride, int logn2, const u32 *lv,
                            const u32 *olo, const u32 *ohi, const Family *fam, hipStream_t s) {
    constexpr int C = col_tile<LOGL1>();
    ProfScope ps(kProfColFwd, s);
    hipLaunchKernelGGL((k_col_fwd<LOGL1, C>), dim3((unsigned)(((int64_t)1 << logn2) / C), cnt),
                       dim3(Tile<LOGL1, C, true>::T), 0, s, X, stride, logn2, lv, olo, ohi,
                       mod_of(fam));
    return hipGetLastError();
}

template <int LOGL2>
static hipError_t row_out_t(const u32 *X, u32 *Y, int cnt, int64_t stride, int logn1,
                            const u32 *lv, u32 sc, const Family *fam, hipStream_t s) {
    constexpr int CR = LOGL2 >= 12 ? (1 << (14 - LOGL2)) : 4;   // 16384 words per tile
    using TL = Tile<LOGL2, CR, false>;
    const int nb = (int)(((int64_t)1 << logn1) / CR);
    ProfScope ps(kProfRowOut, s);
    hipLaunchKernelGGL((k_row_out<LOGL2, CR>), dim3(nb, cnt), dim3(TL::T), 0, s, X, Y, stride,
                       logn1, lv, mod_of(fam), sc);
    return hipGetLastError();
}

#define CM_K1_CASES(F, ...)                                                              \
    switch (k1) {                                                                        \
    case 1: return F<1>(__VA_ARGS__);   case 2: return F<2>(__VA_ARGS__);                \
    case 3: return F<3>(__VA_ARGS__);   case 4: return F<4>(__VA_ARGS__);                \
    case 5: return F<5>(__VA_ARGS__);   case 6: return F<6>(__VA_ARGS__);                \
    case 7: return F<7>(__VA_ARGS__);   case 8: return F<8>(__VA_ARGS__);                \
    case 9: return F<9>(__VA_ARGS__);   case 10: return F<10>(__VA_ARGS__);              \
    case 11: return F<11>(__VA_ARGS__); case 12: return F<12>(__VA_ARGS__);              \
    case 13: return F<13>(__VA_ARGS__);                                                  \
    }                                                                                    \
    return hipErrorInvalidValue;

static hipError_t col_fwd(int k1, u32 *X, int cnt, int64_t stride, int logn2, const u32 *lv,
                          const u32 *olo, const u32 *ohi, const Family *fam, hipStream_t s) {
    CM_K1_CASES(col_fwd_t, X, cnt, stride, logn2, lv, olo, ohi, fam, s)
}

hipError_t launch_mul_strided(int logn, const u32 *F, int64_t fs, int lf, const u32 *G,
                              int64_t gs, int lg, u32 *H, int64_t hs, int lh, int count,
                              const Family *fam, hipStream_t s) {
    if (count <= 0) return hipSuccess;
    if (logn < 4) logn = 4;
    // short operands, no wrap-around: the schoolbook kernel (same words)
    if (std::min(lf, lg) <= strided_plain_cutoff() && (int64_t)lf + lg - 1 <= ((int64_t)1 << logn) &&
        lh <= lf + lg - 1)
        return launch_plain_strided(F, fs, lf, G, gs, lg, H, hs, lh, count, fam->p, s);
    if (logn <= kMaxLdsLog) {
        const MulDesc sd{fs, gs, hs, lf, lg, lh, logn};
        return launch_mul_lds_strided(logn, F, G, H, sd, count, fam, s);
    }
    // four-step straight from the strided operands into the strided output,
    // in chunks whose two slabs stay within 1 GiB each
    const int64_t n = (int64_t)1 << logn;
    const int64_t chunk = std::max<int64_t>(1, ((int64_t)1 << 28) / n);
    for (int64_t c0 = 0; c0 < count; c0 += chunk) {
        const int cnt = (int)std::min<int64_t>(chunk, count - c0);
        u32 *sf = (u32 *)workspace(5, sizeof(u32) * (size_t)(n * cnt), s);
        u32 *sg = (u32 *)workspace(6, sizeof(u32) * (size_t)(n * cnt), s);
        if (!sf || !sg) return hipErrorOutOfMemory;
        FourStepIO io{F + c0 * fs, G + c0 * gs, lf, lg, fs, sf, sg, H + c0 * hs, lh, hs, cnt, gs};
        hipError_t e = launch_mul_four_step(logn, io, fam, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_rows_mul(int e, u32 *F, u32 *G, int rows, const Family *fam, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (e <= kMaxLdsLog) {
        const int L = 1 << e;
        const MulDesc sd{L, L, L, L, L, L, e};
        return launch_mul_lds_strided(e, F, G, F, sd, rows, fam, s);
    }
    const int64_t n = (int64_t)1 << e;
    FourStepIO io{F, G, n, n, n, F, G, F, n, n, rows};
    return launch_mul_four_step(e, io, fam, s);
}

hipError_t launch_ntt_four_step(int k, u32 *X, u32 *Y, int cnt, bool inverse, const Family *fam,
                                hipStream_t s) {
    if (k <= kMaxLdsLog || k > kMaxLog || k > fam->K) return hipErrorInvalidValue;
    const int k2 = nominal_split(k), k1 = k - k2;
    const Outer *o = outer_for(fam, k);
    if (!o) return hipErrorOutOfMemory;
    const int64_t n = (int64_t)1 << k;
    // the inverse transform is the forward transform with the inverse root
    const u32 *lv = inverse ? fam->lvi : fam->lv;
    const u32 *olo = inverse ? o->lo_i : o->lo_f, *ohi = inverse ? o->hi_i : o->hi_f;
    hipError_t e = col_fwd(k1, X, cnt, n, k2, lv, olo, ohi, fam, s);
    if (e != hipSuccess) return e;
    const u32 sc =
        inverse ? scale_mont(cm_host_inv(cm_host_pow(2, k, fam->p), fam->p), fam->p) : 0u;
    if (k2 == 12) e = row_out_t<12>(X, Y, cnt, n, k1, lv, sc, fam, s);
    else if (k2 == 13) e = row_out_t<13>(X, Y, cnt, n, k1, lv, sc, fam, s);
    else e = row_out_t<14>(X, Y, cnt, n, k1, lv, sc, fam, s);
    if (e != hipSuccess) return e;
    return hipMemcpyAsync(X, Y, sizeof(u32) * (size_t)(n * cnt), hipMemcpyDeviceToDevice, s);
}

template <int LOGM>
static hipError_t col_ntt_t(u32 *X, int64_t ncols, int nblk, int64_t bstride, u32 sc,
                            const Family *fam, hipStream_t s) {
    constexpr int C = col_tile<LOGM>();
    using TL = Tile<LOGM, C, true>;
    const int64_t nb = (ncols + C - 1) / C;
    ProfScope ps(kProfColNtt, s);
    hipLaunchKernelGGL((k_col_ntt<LOGM, C>), dim3((unsigned)nb, (unsigned)nblk), dim3(TL::T), 0,
                       s, X, ncols, bstride, fam->lv, mod_of(fam), sc);
    return hipGetLastError();
}

hipError_t launch_col_ntt(int em, u32 *X, int64_t ncols, u32 scale, const Family *fam,
                          hipStream_t s, int nblk, int64_t bstride) {
    if (nblk <= 0 || nblk > 65535) return hipErrorInvalidValue;
    const int k1 = em;
    const u32 sc = scale_mont(scale, fam->p);
    CM_K1_CASES(col_ntt_t, X, ncols, nblk, bstride, sc, fam, s)
}

hipError_t launch_pointwise(u32 *Y, const u32 *X, int64_t n, u32 p, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    u32 r1 = cm_host_r1(p);
    u32 r2 = cm_host_mul(r1, r1, p);
    hipLaunchKernelGGL(k_pointwise, dim3(ew_blocks(n)), dim3(256), 0, s, Y, X, n, p,
                       cm_host_pinv(p), r2);
    return hipGetLastError();
}

hipError_t launch_scale(u32 *X, int64_t n, u32 a, u32 p, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    a %= p;
    hipLaunchKernelGGL(k_scale, dim3(ew_blocks(n)), dim3(256), 0, s, X, n, a,
                       cm_host_shoup_q(a, p), p);
    return hipGetLastError();
}

hipError_t launch_powers(u32 *W, int64_t n, u32 w, u32 p, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    u32 one = cm_host_r1(p);
    hipLaunchKernelGGL(k_powers, dim3(ew_blocks(n)), dim3(256), 0, s, W, n,
                       cm_host_mul(w % p, one, p), one, p, cm_host_pinv(p));
    return hipGetLastError();
}

hipError_t launch_fill(u32 *X, int64_t n, u32 v, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill, dim3(ew_blocks(n)), dim3(256), 0, s, X, n, v);
    return hipGetLastError();
}

}  // namespace cm
