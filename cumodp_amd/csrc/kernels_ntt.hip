// kernels_ntt.hip -- column transforms of the bivariate DFT, elementwise
// kernels and the batched strided multiply.
//
// Replaces the reference's one-stage-per-launch radix-2 column passes and
// elementwise kernels (src/list_stockham.cu:108-576, src/fft_aux.cu:70-322).
// The multiplies are in mul_mx.hip, stand-alone transforms in ntt_nat.hip.
#include <algorithm>

#include "internal.h"
#include "ntt_core.h"

namespace cm {

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

// column tile width: C columns x 2^LOGL1 rows <= 16384 words (at most 4096
// columns)
template <int LOGL1>
static constexpr int col_tile() {
    return (16384 >> LOGL1) > 4096 ? 4096 : (16384 >> LOGL1);
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
