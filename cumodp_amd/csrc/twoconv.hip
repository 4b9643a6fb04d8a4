// twoconv.hip -- exact product of integer polynomials by two convolutions
// over 32-bit Fourier primes, CRT and carry recombination.
//
// Reference: two_convolution_poly_mul (src/two_convolution_poly_mul.cu:532-569)
// and its parts :58-428.  Each coefficient (sign + magnitude) is cut into K
// limbs of M bits, giving a bivariate A(x, y) with a(y) = A(2^M, y); a negative
// coefficient contributes (p - limb) mod p (:84-203).  The product C = A B has
// x-degree <= 2K-2, and
//     cyclic      C mod (x^K - 1) = C_lo + C_hi
//     negacyclic  C mod (x^K + 1) = C_lo - C_hi   (theta twist, :490-512)
// so c(y) = C_lo(2^M, y) + 2^(KM) C_hi(2^M, y)  (:407-423 recombine the
// CRT-reconstructed sum 2 C_lo and difference 2 C_hi the same way).
//
// Here both convolutions are evaluated at once: the length-2K DFT in x of the
// zero-padded limb vector has the cyclic convolution's points at even indices
// (w_2K^(2v) = w_K^v) and the theta-twisted negacyclic ones at odd indices
// (w_2K^(2v+1) = theta w_K^v, theta = w_2K).  Every x-point is an independent
// linear convolution in y (a row multiply), and the inverse length-2K DFT
// returns C_lo (j < K) and C_hi (j >= K) directly, i.e. the reference's
// (sum, diff)/2.  The reference pads x and y to one square power of two
// (:446-453) and therefore only recovers C_lo; its answers are exact while
// the limb product does not wrap.  Here x has exactly 2K points and y is
// padded to the product length, and (K, M, prime count) are chosen from the
// CRT bound  L * n_min * (2^M - 1)^2 < P / 2  (L = nonzero limb pairs), so the
// result is the exact integer product for every input size.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "internal.h"
#include "ntt_core.h"

namespace cm {

// CRT primes (p - 1 divisible by 2^25 or more) and the inverses Garner needs
static const u32 kTcPrimes[3] = {2013265921u, 2113929217u, 1811939329u};

struct TcPlan {
    int np;        // primes (2 or 3)
    int K, M;      // limbs per coefficient, bits per limb
    int lk2;       // log2(2K)
    int ey;        // y transform size 2^ey >= na + nb - 1
};

// (K, M, np) minimising np * K under the CRT bound; false if none fits.
static bool tc_choose(int bits, int64_t na, int64_t nb, TcPlan &pl) {
    const double lg_nmin = std::log2((double)std::min(na, nb));
    const double lgP[2] = {std::log2(2013265921.0) + std::log2(2113929217.0),
                           std::log2(2013265921.0) + std::log2(2113929217.0) +
                               std::log2(1811939329.0)};
    int best = 0;
    for (int np = 2; np <= 3; ++np) {
        for (int K = 2; K <= 512; K *= 2) {
            const int M = (bits + K - 1) / K;
            if (M > 30 || M < 1) continue;
            const int L = std::min(K, (bits + M - 1) / M);
            const double need = std::log2((double)L) + lg_nmin + 2.0 * M;
            if (need >= lgP[np - 2] - 1.01) continue;
            const int cost = np * K;
            if (!best || cost < best) {
                best = cost;
                pl.np = np; pl.K = K; pl.M = M;
            }
            break;   // larger K only costs more for this np
        }
    }
    if (!best) return false;
    pl.lk2 = 0;
    while ((1 << pl.lk2) < 2 * pl.K) ++pl.lk2;
    pl.ey = 0;
    while (((int64_t)1 << pl.ey) < na + nb - 1) ++pl.ey;
    if (pl.ey < 4) pl.ey = 4;
    return true;
}

// Plan shared by a class of batched products with y size 2^ey: the cheapest
// (np, K) whose widest admissible limb M_max (the CRT bound with every one of
// the K limbs nonzero and n_min = 2^(ey-1), the class's worst case) covers
// `bits`, with M = M_max.  Products of different bit widths then share a
// plan, and so a launch sequence, whenever one (np, K) serves them.
static bool tc_class_plan(int bits, int ey, TcPlan &pl) {
    const double lgP[2] = {std::log2(2013265921.0) + std::log2(2113929217.0),
                           std::log2(2013265921.0) + std::log2(2113929217.0) +
                               std::log2(1811939329.0)};
    int best = 0;
    for (int np = 2; np <= 3; ++np) {
        for (int K = 1; K <= 512; K *= 2) {
            int M = 30;
            while (M >= 1 && std::log2((double)K) + (ey - 1) + 2.0 * M >= lgP[np - 2] - 1.01) --M;
            if (M < 1 || (int64_t)K * M < bits) continue;
            const int cost = np * K;
            if (!best || cost < best) {
                best = cost;
                pl.np = np; pl.K = K; pl.M = M;
            }
            break;
        }
    }
    if (!best) return false;
    pl.lk2 = 0;
    while ((1 << pl.lk2) < 2 * pl.K) ++pl.lk2;
    pl.ey = ey;
    return true;
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
// One product of a batch (word offsets into A, B, C; coefficient counts;
// words per coefficient).
struct TcDesc {
    int64_t a_off, b_off, c_off, na, nb;
    int32_t wa, wb, wc, pad;
};

// Limb split of one operand of a batch: coefficient i of item r (w words,
// two's complement) -> out[(j R + r) Ly + i] for limb j < K: |a_i| bits
// [jM, jM+M) mod p, negated mod p when a_i < 0; limbs K .. 2K-1 and
// positions i >= n are zero.  grid.y: items (descriptor `one` when d is null).
__global__ void k_tc_split(const u64 *__restrict__ src, const TcDesc *__restrict__ d,
                           TcDesc one, int which, int K, int K2, int M, u32 p,
                           u32 *__restrict__ out, int64_t Ly, int R) {
    const int r = blockIdx.y;
    const TcDesc dd = d ? d[r] : one;
    const u64 *a = src + (which ? dd.b_off : dd.a_off);
    const int64_t n = which ? dd.nb : dd.na;
    const int w = which ? dd.wb : dd.wa;
    u32 *o = out + (int64_t)r * Ly;
    const int64_t js = (int64_t)R * Ly;           // stride between limb rows
    const u64 mask = (1ull << M) - 1;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < Ly;
         i += (int64_t)gridDim.x * blockDim.x) {
        int j = 0;
        if (i < n) {
            const u64 *x = a + i * w;
            const bool neg = (int64_t)x[w - 1] < 0;
            u64 carry = 1;                       // magnitude = ~x + 1 when negative
            unsigned __int128 buf = 0;           // holds `have` < M + 64 bits
            int have = 0;
            for (int q = 0; q < w && j < K; ++q) {
                u64 v = x[q];
                if (neg) {
                    v = ~v + carry;
                    carry = (carry && v == 0) ? 1u : 0u;
                }
                buf |= (unsigned __int128)v << have;
                have += 64;
                while (have >= M && j < K) {
                    const u32 limb = (u32)((u64)buf & mask);
                    o[j * js + i] = neg ? (limb ? p - limb : 0u) : limb;
                    buf >>= M;
                    have -= M;
                    ++j;
                }
            }
            for (; j < K; ++j) {                 // remaining bits, then zero limbs
                const u32 limb = (u32)((u64)buf & mask);
                o[j * js + i] = neg ? (limb ? p - limb : 0u) : limb;
                buf >>= M;
            }
        }
        for (; j < K2; ++j) o[j * js + i] = 0u;
    }
}

// One class of products in the fused form (one-word coefficients, 2K <= 8):
// rows of item r and x-point k at out[q][operand] + (k R + r) 2^ey, and per
// prime the tables of the x transforms.
struct TcCls {
    u32 *out[3][2];
    const u32 *lvf[3], *lvi[3];   // level tables of the x root and its inverse
    u32 p[3], np[3], ki[3];       // modulus, -p^-1 mod 2^32, Montgomery form of 1 / 2K
    int lk2, nprimes, M, ey, R, first;   // first: its first item among the descriptors
    int len[2];                   // words of a row that are written (longest operand)
};

// One block of work: positions from start of operand `which` (split) or of
// the product (CRT) of item `item` (counted within the class).
struct TcBlock {
    int cls, item, which, start;
};

// k_tc_split for one-word coefficients fused with the forward x transform:
// thread i forms the K limbs of coefficient i (upper K limbs zero) once, runs
// the natural-order length-2K DFT on them in registers for every prime (DIF
// stages, zero upper half) and writes the 2K words.  Positions from the item's
// length to the class's longest are zero rows.
template <int LK2>
CM_DEV void tc_split_block(const TcCls &c, const u64 *a, int n, int r, int which, int start,
                           int span) {
    constexpr int K2 = 1 << LK2, K = K2 / 2;
    const int64_t js = (int64_t)c.R << c.ey;
    const u64 mask = (1ull << c.M) - 1;
    const int end = min(start + span, c.len[which]);
    for (int i = start + threadIdx.x; i < end; i += blockDim.x) {
        const u64 x = i < n ? a[i] : 0;
        const bool neg = (int64_t)x < 0;
        const u64 mag = neg ? ~x + 1 : x;                // |x| (2^63 for the minimum)
        u32 limb[K];
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const int sh = j * c.M;
            limb[j] = sh < 64 ? (u32)((mag >> sh) & mask) : 0u;
        }
        for (int q = 0; q < c.nprimes; ++q) {
            const Mod md{c.p[q], c.np[q]};
            u32 v[1][K2];
#pragma unroll
            for (int j = 0; j < K; ++j) {
                v[0][j] = neg ? (limb[j] ? md.p - limb[j] : 0u) : limb[j];
                v[0][K + j] = 0u;
            }
            cm_dif_stages<LK2, LK2, 0, 0, 1, true>(v, 0, c.lvf[q], md);
            u32 *o = c.out[q][which] + ((int64_t)r << c.ey) + i;
#pragma unroll
            for (int m = 0; m < K2; ++m) o[(int64_t)cm_brev((u32)m, LK2) * js] = v[0][m];
        }
    }
}

// blocks: the work of each workgroup (null: class `one`, item 0, operand
// blockIdx.y, span positions per workgroup); d: descriptors (null: `od`).
__global__ __launch_bounds__(256) void k_tc_split_x(const u64 *__restrict__ A,
                                                    const u64 *__restrict__ B,
                                                    const TcDesc *__restrict__ d, TcDesc od,
                                                    const TcCls *__restrict__ cls, TcCls one,
                                                    const TcBlock *__restrict__ blocks, int span) {
    const TcBlock t = blocks ? blocks[blockIdx.x]
                             : TcBlock{0, 0, (int)blockIdx.y, (int)blockIdx.x * span};
    const TcCls &c = cls ? cls[t.cls] : one;
    const TcDesc dd = d ? d[c.first + t.item] : od;
    const u64 *a = t.which ? B + dd.b_off : A + dd.a_off;
    const int n = (int)(t.which ? dd.nb : dd.na);
    switch (c.lk2) {
    case 1: tc_split_block<1>(c, a, n, t.item, t.which, t.start, span); break;
    case 2: tc_split_block<2>(c, a, n, t.item, t.which, t.start, span); break;
    default: tc_split_block<3>(c, a, n, t.item, t.which, t.start, span); break;
    }
}

// Garner constants of the CRT over the first two or three primes
struct TcCrt {
    u32 p0, p1, p2, inv01, inv01q, inv012, inv012q, p0m2, p0m2q;
};

// The signed CRT value (in (-P/2, P/2]) of the residues r0, r1 (, r2).  Each
// prime exceeds half of every other, so one conditional subtraction takes a
// residue of one into the range of another (p0 < p1 needs none).
template <int NP>
__device__ __forceinline__ __int128 tc_crt_value(u32 r0, u32 r1, u32 r2, const TcCrt &k) {
    // Garner: t1 = (r1 - r0) p0^-1 mod p1;  z = r0 + p0 t1 (+ p0 p1 t2)
    const u32 t1 = cm_shoup(cm_sub(r1, r0, k.p1), k.inv01, k.inv01q, k.p1);
    const u64 z2 = (u64)k.p0 * t1 + r0, P2 = (u64)k.p0 * k.p1;
    if (NP == 2) return z2 > P2 / 2 ? (__int128)z2 - (__int128)P2 : (__int128)z2;
    // t2 = (r2 - (r0 + p0 t1)) (p0 p1)^-1 mod p2
    const u32 zm = cm_add(cm_reduce2p(r0, k.p2),
                          cm_shoup(cm_reduce2p(t1, k.p2), k.p0m2, k.p0m2q, k.p2), k.p2);
    const u32 t2 = cm_shoup(cm_sub(r2, zm, k.p2), k.inv012, k.inv012q, k.p2);
    const unsigned __int128 z = (unsigned __int128)P2 * t2 + z2, P = (unsigned __int128)P2 * k.p2;
    return z > P / 2 ? (__int128)z - (__int128)P : (__int128)z;
}

// Adds z 2^sh to the wc-word two's-complement accumulator o, where z is the
// CRT value of the residues r0, r1 (, r2).
template <int NP>
__device__ __forceinline__ void tc_crt_add(u64 *o, int wc, int sh, u32 r0, u32 r1, u32 r2,
                                           const TcCrt &k) {
    const __int128 sz = tc_crt_value<NP>(r0, r1, r2, k);
    if (sz == 0) return;
    // add sz << sh into the wc-word accumulator
    const int w0 = sh >> 6, b0 = sh & 63;
    const bool neg = sz < 0;
    unsigned __int128 mag = (unsigned __int128)(neg ? -sz : sz);
    u64 part[3];
    part[0] = (u64)(mag << b0);
    part[1] = (u64)((mag << b0) >> 64);
    part[2] = b0 ? (u64)(mag >> (128 - b0)) : 0;
    if (!neg) {
        u64 c = 0;
        for (int q = w0; q < wc; ++q) {
            const u64 s = (q - w0 < 3) ? part[q - w0] : 0;
            const u64 t = o[q] + s;
            const u64 c1 = t < s;
            const u64 t2 = t + c;
            c = c1 | (t2 < c);
            o[q] = t2;
            if (q - w0 >= 2 && !c) break;
        }
    } else {
        u64 b = 0;
        for (int q = w0; q < wc; ++q) {
            const u64 s = (q - w0 < 3) ? part[q - w0] : 0;
            const u64 v = o[q];
            const u64 t = v - s - b;
            b = (v < s) || (v - s < b);
            o[q] = t;
            if (q - w0 >= 2 && !b) break;
        }
    }
}

// CRT and recombination for a batch: output coefficient y of item r is
// sum_j z_j 2^(M j), where z_j (j < 2K-1) is the signed CRT value of the
// residues C_q[(j R + r) Ly + y].  grid.y: items.
template <int NP>
__global__ void k_tc_crt(const u32 *__restrict__ C0, const u32 *__restrict__ C1,
                         const u32 *__restrict__ C2, const TcDesc *__restrict__ d, TcDesc one,
                         int K2, int M, int64_t Ly, int R, u64 *__restrict__ out, TcCrt k) {
    const int r = blockIdx.y;
    const TcDesc dd = d ? d[r] : one;
    const int64_t ny = dd.na + dd.nb - 1;
    const int wc = dd.wc;
    const int64_t js = (int64_t)R * Ly, base = (int64_t)r * Ly;
    for (int64_t y = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; y < ny;
         y += (int64_t)gridDim.x * blockDim.x) {
        u64 *o = out + dd.c_off + y * wc;
        for (int q = 0; q < wc; ++q) o[q] = 0;
        for (int j = 0; j < K2 - 1; ++j) {
            const int64_t at = j * js + base + y;
            tc_crt_add<NP>(o, wc, M * j, C0[at], C1[at], NP == 3 ? C2[at] : 0u, k);
        }
    }
}

// Inverse x transforms of the residues of each prime (natural-order length-2K
// DFT with the inverse root's level table, times 1/2K) fused with the CRT and
// recombination of output coefficient y: sum_j z_j 2^(M j), j < 2K - 1, in four
// words of registers (one-word operands: the sum has at most 2 64 + 32 + 1
// bits), sign-extended to the wc words of the output.
template <int NP, int LK2>
CM_DEV void tc_crt_block(const TcCls &c, const TcDesc &dd, u64 *out, int r, int start, int span,
                         const TcCrt &k) {
    constexpr int K2 = 1 << LK2;
    const int64_t js = (int64_t)c.R << c.ey, base = (int64_t)r << c.ey;
    const int64_t ny = dd.na + dd.nb - 1;
    const int end = (int)(ny < start + span ? ny : start + span);
    const int wc = dd.wc;
    for (int y = start + threadIdx.x; y < end; y += blockDim.x) {
        u32 res[NP][K2];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const u32 *C = c.out[q][0] + base + y;
            u32 v[1][K2];
#pragma unroll
            for (int j = 0; j < K2; ++j) v[0][j] = C[j * js];
            const Mod md{c.p[q], c.np[q]};
            cm_dif_stages<LK2, LK2, 0, 0, 1>(v, 0, c.lvi[q], md);
#pragma unroll
            for (int j = 0; j < K2; ++j)
                res[q][j] = cm_mul_tw(v[0][cm_brev((u32)j, LK2)], c.ki[q], md.p, md.np);
        }
        u64 acc[4] = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < K2 - 1; ++j) {
            const __int128 z = tc_crt_value<NP>(res[0][j], res[1][j], NP == 3 ? res[2][j] : 0u, k);
            const int sh = c.M * j, w0 = sh >> 6, b0 = sh & 63;   // uniform
            const u64 sign = (u64)(int64_t)(z >> 127);
            const unsigned __int128 lo = (unsigned __int128)z << b0;
            const u64 part[3] = {(u64)lo, (u64)(lo >> 64),
                                 b0 ? (u64)((unsigned __int128)z >> 64) >> (64 - b0) | sign << b0
                                    : sign};
            u64 carry = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const u64 w = q < w0 ? 0 : (q == w0 ? part[0]
                                                    : (q == w0 + 1 ? part[1]
                                                                   : (q == w0 + 2 ? part[2] : sign)));
                const u64 t = acc[q] + w, u = t + carry;
                carry = (u64)(t < w) | (u64)(u < t);
                acc[q] = u;
            }
        }
        u64 *o = out + dd.c_off + (int64_t)y * wc;
        const u64 top = (u64)((int64_t)acc[3] >> 63);
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (q < wc) o[q] = acc[q];
        for (int q = 4; q < wc; ++q) o[q] = top;
    }
}

__global__ __launch_bounds__(256) void k_tc_crt_x(const TcDesc *__restrict__ d, TcDesc od,
                                                  const TcCls *__restrict__ cls, TcCls one,
                                                  const TcBlock *__restrict__ blocks, int span,
                                                  u64 *__restrict__ out, TcCrt k) {
    const TcBlock t = blocks ? blocks[blockIdx.x] : TcBlock{0, 0, 0, (int)blockIdx.x * span};
    const TcCls &c = cls ? cls[t.cls] : one;
    const TcDesc dd = d ? d[c.first + t.item] : od;
    switch (c.nprimes * 4 + c.lk2) {
    case 9: tc_crt_block<2, 1>(c, dd, out, t.item, t.start, span, k); break;
    case 10: tc_crt_block<2, 2>(c, dd, out, t.item, t.start, span, k); break;
    case 11: tc_crt_block<2, 3>(c, dd, out, t.item, t.start, span, k); break;
    case 13: tc_crt_block<3, 1>(c, dd, out, t.item, t.start, span, k); break;
    case 14: tc_crt_block<3, 2>(c, dd, out, t.item, t.start, span, k); break;
    default: tc_crt_block<3, 3>(c, dd, out, t.item, t.start, span, k); break;
    }
}

// theta scaling of the reference's scale_x_argument_dev
// (src/two_convolution_poly_mul.cu:207-245): A[i] *= theta^(i mod K)
__global__ void k_scale_x(u32 *__restrict__ A, int64_t len, int K, const uint2 *__restrict__ tp,
                          u32 p) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < len;
         i += (int64_t)gridDim.x * blockDim.x) {
        const uint2 t = tp[i % K];
        A[i] = cm_shoup(A[i] % p, t.x, t.y, p);
    }
}

static int blocks_for(int64_t n, int t = 256) {
    int64_t b = (n + t - 1) / t;
    return (int)std::max<int64_t>(1, std::min<int64_t>(b, 16384));
}

// ---------------------------------------------------------------------------
// host driver
// ---------------------------------------------------------------------------
int tc_bit_width(const u64 *a, int64_t n, int w) {
    int best = 1;
    std::vector<u64> mag((size_t)w);
    for (int64_t i = 0; i < n; ++i) {
        const u64 *x = a + i * w;
        const bool neg = (int64_t)x[w - 1] < 0;
        u64 carry = 1;
        for (int q = 0; q < w; ++q) {
            u64 v = x[q];
            if (neg) { v = ~v + carry; carry = (carry && v == 0); }
            mag[(size_t)q] = v;
        }
        int l = w;
        while (l > 0 && mag[(size_t)l - 1] == 0) --l;
        if (l) {
            int bits = 64 * (l - 1) + (64 - __builtin_clzll(mag[(size_t)l - 1]));
            best = std::max(best, bits);
        }
    }
    return best;
}

static TcCrt tc_crt_consts() {
    const u32 p0 = kTcPrimes[0], p1 = kTcPrimes[1], p2 = kTcPrimes[2];
    const u32 inv01 = cm_host_inv(p0 % p1, p1);
    const u32 p0m2 = p0 % p2;
    const u32 inv012 = cm_host_inv(cm_host_mul(p0 % p2, p1 % p2, p2), p2);
    return TcCrt{p0, p1, p2, inv01, cm_host_shoup_q(inv01, p1), inv012,
                 cm_host_shoup_q(inv012, p2), p0m2, cm_host_shoup_q(p0m2, p2)};
}

// The families of prime q's x transforms of 2^lk2 points (forward and inverse
// root).
static hipError_t tc_x_families(int q, int lk2, const Family *&fam, const Family *&fx,
                                const Family *&fxi) {
    const u32 p = kTcPrimes[q];
    fam = family_default(p);
    if (!fam) return hipErrorOutOfMemory;
    const u32 wx = cm_host_pow(fam->wN, (u64)1 << (fam->K - lk2), p);
    fx = family_for_root(p, wx, lk2);
    fxi = family_for_root(p, cm_host_inv(wx, p), lk2);
    return fx && fxi ? hipSuccess : hipErrorOutOfMemory;
}

// The products of one class (same plan and y size) over R items: per prime,
// A and B are 2K x R x Ly (limb row j of item r at (j R + r) Ly), so the x
// transforms are column transforms over R Ly columns and the y products are
// 2K R rows of Ly words.  d: device descriptors, or null with `one`.
static hipError_t tc_run_class(const TcPlan &pl, const u64 *A, const u64 *B, u64 *C,
                               const TcDesc *d, const TcDesc &one, int R, int64_t ymax, u32 *ws,
                               hipStream_t s) {
    const int K2 = 1 << pl.lk2;
    const int64_t Ly = (int64_t)1 << pl.ey;
    const size_t per = (size_t)2 * K2 * R * Ly;   // A and B rows of one prime
    const int bx = blocks_for(Ly);
    u32 *Cr[3] = {nullptr, nullptr, nullptr};
    for (int q = 0; q < pl.np; ++q) {
        const u32 p = kTcPrimes[q];
        const Family *fam, *fx, *fxi;
        hipError_t e = tc_x_families(q, pl.lk2, fam, fx, fxi);
        if (e != hipSuccess) return e;
        u32 *Aq = ws + per * q, *Bq = Aq + (size_t)K2 * R * Ly;
        Cr[q] = Aq;
        const u32 ki = cm_host_inv((u32)K2, p);
        {
            ProfScope ps(kProfTcSplit, s);
            hipLaunchKernelGGL(k_tc_split, dim3(bx, R), dim3(256), 0, s, A, d, one, 0, pl.K, K2,
                               pl.M, p, Aq, Ly, R);
            hipLaunchKernelGGL(k_tc_split, dim3(bx, R), dim3(256), 0, s, B, d, one, 1, pl.K, K2,
                               pl.M, p, Bq, Ly, R);
        }
        e = hipGetLastError();
        // x: length-2K DFT down the columns (cyclic points even, negacyclic odd)
        if (e == hipSuccess) e = launch_col_ntt(pl.lk2, Aq, (int64_t)R * Ly, 1u, fx, s);
        if (e == hipSuccess) e = launch_col_ntt(pl.lk2, Bq, (int64_t)R * Ly, 1u, fx, s);
        // y: 2K R independent cyclic products of length Ly (= linear: ny <= Ly)
        if (e == hipSuccess) e = launch_rows_mul(pl.ey, Aq, Bq, K2 * R, fam, s);
        // inverse x transform with the 1/(2K) scaling
        if (e == hipSuccess) e = launch_col_ntt(pl.lk2, Aq, (int64_t)R * Ly, ki, fxi, s);
        if (e != hipSuccess) return e;
    }
    ProfScope ps(kProfTcCrt, s);
    const dim3 g(blocks_for(ymax), R);
    const TcCrt kc = tc_crt_consts();
    const u32 *C2 = pl.np == 3 ? Cr[2] : Cr[1];
    if (pl.np == 2)
        hipLaunchKernelGGL((k_tc_crt<2>), g, dim3(256), 0, s, Cr[0], Cr[1], C2, d, one, K2, pl.M,
                           Ly, R, C, kc);
    else
        hipLaunchKernelGGL((k_tc_crt<3>), g, dim3(256), 0, s, Cr[0], Cr[1], C2, d, one, K2, pl.M,
                           Ly, R, C, kc);
    return hipGetLastError();
}

// The fused form serves one-word coefficients and 2K <= 8 (2K = 16 would
// spill in the CRT): x transforms in the split and CRT kernels, the y products
// of every class and prime as one list of row segments.
static bool tc_fused(const TcPlan &pl, int wa, int wb) {
    return wa == 1 && wb == 1 && pl.lk2 >= 1 && pl.lk2 <= 3;
}

static size_t tc_item_words(const TcPlan &pl) {
    return ((size_t)2 * pl.np << pl.lk2) << pl.ey;
}

// Fills one fused class over ws (R items, operands of at most la and lb
// coefficients) and appends its row segments.
static hipError_t tc_make_cls(const TcPlan &pl, int R, int la, int lb, int first, u32 *ws,
                              TcCls &c, std::vector<RowSeg> &segs) {
    c = TcCls{};
    c.lk2 = pl.lk2; c.nprimes = pl.np; c.M = pl.M; c.ey = pl.ey; c.R = R; c.first = first;
    c.len[0] = la; c.len[1] = lb;
    const size_t half = ((size_t)R << pl.lk2) << pl.ey;   // rows of one operand and prime
    for (int q = 0; q < pl.np; ++q) {
        const Family *fam, *fx, *fxi;
        hipError_t e = tc_x_families(q, pl.lk2, fam, fx, fxi);
        if (e != hipSuccess) return e;
        c.out[q][0] = ws + 2 * half * q;
        c.out[q][1] = c.out[q][0] + half;
        c.lvf[q] = fx->lv;
        c.lvi[q] = fxi->lv;
        c.p[q] = kTcPrimes[q];
        c.np[q] = fam->np;
        c.ki[q] = cm_host_mont(cm_host_inv(1u << pl.lk2, kTcPrimes[q]), kTcPrimes[q]);
        segs.push_back(RowSeg{c.out[q][0], c.out[q][1], R << pl.lk2, pl.ey, la, lb, fam});
    }
    return hipSuccess;
}

// Runs the whole product on device buffers.  bits: largest coefficient bit
// width of a and b (>= 1).
hipError_t launch_two_convolution(const u64 *a, int64_t na, int wa, const u64 *b, int64_t nb,
                                  int wb, u64 *c, int wc, int bits, hipStream_t s, int *err) {
    *err = 0;
    TcPlan pl;
    if (!tc_choose(bits, na, nb, pl) || pl.ey > kMaxLog || pl.lk2 > kMaxLdsLog) {
        *err = 1;
        return hipSuccess;
    }
    u32 *ws = (u32 *)workspace(10, sizeof(u32) * tc_item_words(pl), s);
    if (!ws) return hipErrorOutOfMemory;
    TcDesc one{0, 0, 0, na, nb, wa, wb, wc, 0};
    if (!tc_fused(pl, wa, wb))
        return tc_run_class(pl, a, b, c, nullptr, one, 1, na + nb - 1, ws, s);
    // one position per thread: a single product is bound by latency
    constexpr int span = 256;
    TcCls cls;
    std::vector<RowSeg> segs;
    hipError_t e = tc_make_cls(pl, 1, (int)na, (int)nb, 0, ws, cls, segs);
    if (e != hipSuccess) return e;
    {
        ProfScope ps(kProfTcSplit, s);
        const dim3 g((unsigned)((std::max(na, nb) + span - 1) / span), 2);
        hipLaunchKernelGGL(k_tc_split_x, g, dim3(256), 0, s, a, b, nullptr, one, nullptr, cls,
                           nullptr, span);
    }
    e = hipGetLastError();
    if (e == hipSuccess) e = launch_rows_batch(std::move(segs), s);
    if (e != hipSuccess) return e;
    ProfScope ps(kProfTcCrt, s);
    hipLaunchKernelGGL(k_tc_crt_x, dim3((unsigned)((na + nb - 1 + span - 1) / span)), dim3(256), 0,
                       s, nullptr, one, nullptr, cls, nullptr, span, c, tc_crt_consts());
    return hipGetLastError();
}

// Batch of products: items are grouped by class plan (tc_class_plan: one plan
// per y size and (np, K)), in chunks whose scratch stays under kTcChunkBytes.
static constexpr size_t kTcChunkBytes = (size_t)1 << 30;

// Class merging of the batched multiply: 0 keeps one class per exact plan;
// 1 gives every item of one y size the plan of the widest coefficients of
// that size (exact for all of them: K M covers every width and the bound
// depends on the y size only), trading transform work for fewer launches.
static int g_tc_merge = 0;

bool set_zmul_merge(int m) {
    if (m < 0 || m > 1) return false;
    g_tc_merge = m;
    return true;
}

int zmul_merge() { return g_tc_merge; }

namespace {
struct TcClass {
    TcPlan pl;
    bool fused;
    std::vector<int64_t> idx;
};
}  // namespace

// The fused classes of a batch: a split launch, the row products of all of
// them and a CRT launch per chunk.  Each workgroup takes `span` positions of
// one operand or product from a table.  (One launch sequence per class and
// prime, on four streams, took 198 launches and 1.16 ms for 96 requests of
// degrees 64 .. 65536; two uploads and 13 launches take 0.31 ms.)
static hipError_t tc_run_fused(const std::vector<const TcClass *> &classes, const TcItem *items,
                               const u64 *A, const u64 *B, u64 *C, hipStream_t s) {
    constexpr int span = 1024;
    size_t ci = 0, at = 0;   // next class, next item of it
    while (ci < classes.size()) {
        std::vector<TcCls> cls;
        std::vector<TcDesc> desc;
        std::vector<TcBlock> split, crt;
        std::vector<RowSeg> segs;
        std::vector<size_t> base;         // scratch offset of each class
        struct Part {
            const TcClass *c;
            size_t i0, i1;
        };
        std::vector<Part> parts;
        size_t words = 0;
        // parts of classes up to the chunk's scratch (at least one item)
        while (ci < classes.size()) {
            const TcClass &c = *classes[ci];
            const size_t per = tc_item_words(c.pl), room = kTcChunkBytes / sizeof(u32);
            size_t n = words < room ? (room - words) / per : 0;
            if (parts.empty() && n == 0) n = 1;
            n = std::min(n, c.idx.size() - at);
            if (n == 0) break;
            parts.push_back(Part{&c, at, at + n});
            base.push_back(words);
            words += per * n;
            at += n;
            if (at < c.idx.size()) break;
            ++ci;
            at = 0;
        }
        u32 *ws = (u32 *)workspace(10, sizeof(u32) * words, s);
        if (!ws) return hipErrorOutOfMemory;
        for (size_t k = 0; k < parts.size(); ++k) {
            const Part &q = parts[k];
            const int first = (int)desc.size(), R = (int)(q.i1 - q.i0);
            int64_t la = 0, lb = 0;
            for (size_t i = q.i0; i < q.i1; ++i) {
                const TcItem &it = items[q.c->idx[i]];
                desc.push_back(TcDesc{it.a_off, it.b_off, it.c_off, it.na, it.nb, it.wa, it.wb,
                                      it.wc, 0});
                la = std::max(la, it.na);
                lb = std::max(lb, it.nb);
            }
            TcCls c;
            hipError_t e =
                tc_make_cls(q.c->pl, R, (int)la, (int)lb, first, ws + base[k], c, segs);
            if (e != hipSuccess) return e;
            cls.push_back(c);
            for (int r = 0; r < R; ++r) {
                for (int w = 0; w < 2; ++w)
                    for (int x = 0; x < c.len[w]; x += span)
                        split.push_back(TcBlock{(int)k, r, w, x});
                const TcDesc &d = desc[(size_t)(first + r)];
                for (int64_t x = 0; x < d.na + d.nb - 1; x += span)
                    crt.push_back(TcBlock{(int)k, r, 0, (int)x});
            }
        }
        const size_t b0 = sizeof(TcCls) * cls.size(), b1 = sizeof(TcDesc) * desc.size(),
                     b2 = sizeof(TcBlock) * split.size(), b3 = sizeof(TcBlock) * crt.size();
        char *d = (char *)workspace(14, b0 + b1 + b2 + b3, s);
        if (!d) return hipErrorOutOfMemory;
        hipError_t e = stage_upload_fill(b0 + b1 + b2 + b3, d, s, [&](char *h) {
            memcpy(h, cls.data(), b0);
            memcpy(h + b0, desc.data(), b1);
            memcpy(h + b0 + b1, split.data(), b2);
            memcpy(h + b0 + b1 + b2, crt.data(), b3);
        });
        if (e != hipSuccess) return e;
        const TcCls *dc = (const TcCls *)d;
        const TcDesc *dd = (const TcDesc *)(d + b0);
        const TcBlock *ds = (const TcBlock *)(d + b0 + b1), *dr = (const TcBlock *)(d + b0 + b1 + b2);
        {
            ProfScope ps(kProfTcSplit, s);
            hipLaunchKernelGGL(k_tc_split_x, dim3((unsigned)split.size()), dim3(256), 0, s, A, B,
                               dd, TcDesc{}, dc, TcCls{}, ds, span);
        }
        e = hipGetLastError();
        if (e == hipSuccess) e = launch_rows_batch(std::move(segs), s);
        if (e != hipSuccess) return e;
        ProfScope ps(kProfTcCrt, s);
        hipLaunchKernelGGL(k_tc_crt_x, dim3((unsigned)crt.size()), dim3(256), 0, s, dd, TcDesc{},
                           dc, TcCls{}, dr, span, C, tc_crt_consts());
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_two_convolution_list(const TcItem *items, int64_t count, const u64 *A,
                                       const u64 *B, u64 *C, hipStream_t s, int *err) {
    *err = 0;
    std::vector<TcClass> classes;
    auto y_size = [](const TcItem &it) {
        int ey = 0;
        while (((int64_t)1 << ey) < it.na + it.nb - 1) ++ey;
        return ey < 4 ? 4 : ey;
    };
    int widest[64] = {0};   // merged classes: widest coefficients per y size
    if (g_tc_merge)
        for (int64_t i = 0; i < count; ++i) {
            const int ey = y_size(items[i]);
            if (ey < 64) widest[ey] = std::max(widest[ey], (int)items[i].bits);
        }
    for (int64_t i = 0; i < count; ++i) {
        const TcItem &it = items[i];
        const int ey = y_size(it);
        const int bits = (g_tc_merge && ey < 64) ? widest[ey] : it.bits;
        TcPlan pl;
        if (!tc_class_plan(bits, ey, pl) || pl.lk2 > kMaxLdsLog || pl.ey > kMaxLog) {
            *err = 1;
            return hipSuccess;
        }
        const bool fused = tc_fused(pl, it.wa, it.wb);
        TcClass *c = nullptr;
        for (auto &x : classes)
            if (x.fused == fused && x.pl.np == pl.np && x.pl.K == pl.K && x.pl.M == pl.M &&
                x.pl.ey == pl.ey)
                c = &x;
        if (!c) {
            classes.push_back(TcClass{pl, fused, {}});
            c = &classes.back();
        }
        c->idx.push_back(i);
    }
    std::vector<const TcClass *> fused, plain;
    for (const TcClass &c : classes) (c.fused ? fused : plain).push_back(&c);
    if (!fused.empty()) {
        const hipError_t e = tc_run_fused(fused, items, A, B, C, s);
        if (e != hipSuccess) return e;
    }
    if (plain.empty()) return hipSuccess;
    // descriptors of the other classes, in class order, uploaded once
    std::vector<TcDesc> hd;
    for (const TcClass *c : plain)
        for (int64_t i : c->idx) {
            const TcItem &it = items[i];
            hd.push_back(TcDesc{it.a_off, it.b_off, it.c_off, it.na, it.nb, it.wa, it.wb, it.wc, 0});
        }
    TcDesc *dd = (TcDesc *)workspace(22, sizeof(TcDesc) * hd.size(), s);
    if (!dd) return hipErrorOutOfMemory;
    hipError_t e = stage_upload(hd.data(), sizeof(TcDesc) * hd.size(), dd, s);
    if (e != hipSuccess) return e;
    // Classes are independent: with more than one they run on the caller
    // stream's auxiliary streams (forked after the descriptor upload, joined
    // back at the end), so one class's launch gaps overlap another's work.
    // Each auxiliary stream has its own scratch.
    const int nclass = (int)plain.size();
    AuxStreams *aux = nclass > 1 ? aux_streams(s) : nullptr;
    const int nuse = aux ? std::min(nclass, (int)kAuxStreams) : 0;
    if (aux) {
        e = hipEventRecord(aux->fork, s);
        for (int i = 0; i < nuse && e == hipSuccess; ++i)
            e = hipStreamWaitEvent(aux->s[i], aux->fork, 0);
        if (e != hipSuccess) return e;
    }
    size_t first = 0;
    for (int ci = 0; ci < nclass; ++ci) {
        const TcClass &c = *plain[(size_t)ci];
        const hipStream_t cs = aux ? aux->s[ci % nuse] : s;
        const size_t item_bytes = sizeof(u32) * tc_item_words(c.pl);
        const int64_t chunk = std::max<int64_t>(1, (int64_t)(kTcChunkBytes / item_bytes));
        const int64_t n = (int64_t)c.idx.size();
        for (int64_t k0 = 0; k0 < n; k0 += chunk) {
            const int R = (int)std::min<int64_t>(chunk, n - k0);
            u32 *ws = (u32 *)workspace(10, item_bytes * (size_t)R, cs);
            if (!ws) return hipErrorOutOfMemory;
            int64_t ymax = 1;
            for (int r = 0; r < R; ++r) {
                const TcItem &it = items[c.idx[(size_t)(k0 + r)]];
                ymax = std::max<int64_t>(ymax, it.na + it.nb - 1);
            }
            e = tc_run_class(c.pl, A, B, C, dd + first + k0, TcDesc{}, R, ymax, ws, cs);
            if (e != hipSuccess) return e;
        }
        first += (size_t)n;
    }
    for (int i = 0; i < nuse; ++i) {
        e = hipEventRecord(aux->join[i], aux->s[i]);
        if (e == hipSuccess) e = hipStreamWaitEvent(s, aux->join[i], 0);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_scale_x(u32 *A, int64_t len, int K, u32 theta, u32 p, hipStream_t s) {
    if (len <= 0 || K <= 0) return hipSuccess;
    std::vector<uint2> tp((size_t)K);
    u64 x = 1;
    for (int j = 0; j < K; ++j) {
        tp[(size_t)j] = make_uint2((u32)x, cm_host_shoup_q((u32)x, p));
        x = x * (theta % p) % p;
    }
    uint2 *d = (uint2 *)workspace(11, sizeof(uint2) * (size_t)K, s);
    if (!d) return hipErrorOutOfMemory;
    hipError_t e = hipMemcpy(d, tp.data(), sizeof(uint2) * (size_t)K, hipMemcpyHostToDevice);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_scale_x, dim3(blocks_for(len)), dim3(256), 0, s, A, len, K, d, p);
    return hipGetLastError();
}

int tc_plan_info(int bits, int64_t na, int64_t nb, int *np, int *K, int *M) {
    TcPlan pl;
    if (!tc_choose(bits, na, nb, pl)) return 0;
    *np = pl.np; *K = pl.K; *M = pl.M;
    return 1;
}

}  // namespace cm
