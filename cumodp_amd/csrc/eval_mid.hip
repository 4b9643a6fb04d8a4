// eval_mid.hip -- the values of F (degree < 2^k) at 2^k points by the transposed
// algorithm, k >= 9.
//
// Reference: fastEvaluation (src/fastPolyEvaluation.cu:1371-1400) descends a
// remainder tree with a power-series inverse per node (eval.hip does that when
// a caller keeps the remainders or the inverses).  For the values alone one
// inverse is enough: with M the root of the subproduct tree, n = 2^k,
//     Inv = rev(M)^-1 mod x^n,   b_root[v] = sum_s Inv[s] F[v+s],   v < n,
// and for the children of a node of 2h points, with S the SIBLING's polynomial,
//     b_child[v] = sum_u rev(S)[u] b[v+u] = (S b)[v+h],   v < h,
// until b of a leaf is the value at its point: F(x_j) = sum_i F[i] [z^i]
// 1/(1 - x_j z), and 1/(1 - x_j z) is Inv times the product of all other
// (1 - x_l z), which the descent multiplies in one sibling at a time.  Words h
// .. 2h-1 of S b are not touched by what wraps in a cyclic product on 2h
// points, so a level is one batch of products and no pass beside them; nothing
// is reversed, as the inverse is kept reversed (J[n-1-t] = Inv[t]).
//
// Bound by the serial chain of launches: 2^16 points take 7 products and a
// workgroup's chain of Newton steps for the inverse and 9 levels after the tree.
// The remainder tree has three products per level of inverses, and two products
// and two more passes per level on the way down.  2^16 points: 262 us, 74 of them
// the tree, against 493 us.
#include <algorithm>

#include "accum.h"
#include "internal.h"
#include "ntt_mx.h"

namespace cm {

constexpr int kMidBase = 8;      // levels below run in k_mid_descend
constexpr int kInvRootLog = 13;  // precision of k_inv_root

// Barriers of a transform with one exchange between the waves of a workgroup,
// after round 0.  All threads call this; those with act work.
template <int LOGL, int V, int NV>
CM_DEV void inv_forward(u32 (&x)[NV][V][4], u32 *const (&t)[NV], bool act, const MxCtx &cx) {
    using P = MxPlan<LOGL, 0, V>;
    static_assert(P::NR == 3 && P::words(0) > 4 + mx_log2(V) && P::words(1) <= 4 + mx_log2(V),
                  "one exchange");
    MxMat m;
    u32 tw[V][4];
    if (act) {
        mx_forward_begin<LOGL, 0, V>(m, tw, cx);
#pragma unroll
        for (int a = 0; a < NV; ++a) {
            mx_dft<V>(x[a], m, cx);
            mx_mul<V>(x[a], tw, cx);
            MxMap<P::words(0), V>::store(t[a], x[a]);
        }
        mx_load_tw<P::logs(1), 0, V>(tw, cx.tf);
    }
    __syncthreads();
    if (act) {
#pragma unroll
        for (int a = 0; a < NV; ++a) MxMap<P::words(1), V>::load(t[a], x[a]);
        mx_forward<LOGL, 0, V, 1, NV>(x, t, cx, m, tw);
    }
}

// x <- the product (canonical, natural order) of two transforms
template <int LOGL, int V>
CM_DEV void inv_product(u32 (&x)[V][4], const u32 (&y)[V][4], u32 *t, bool act, const MxCtx &cx) {
    using P = MxPlan<LOGL, 0, V>;
    MxMat m;
    u32 tw[V][4];
    if (act) {
        u32 w[4];
        m = mx_load_mat(cx, P::PAIR ? kMxInvPair : kMxInvFirst + P::T);
        if constexpr (P::PAIR) mx_pair_tw(w, cx.ti);
        mx_mul<V>(x, y, cx);
        if constexpr (P::PAIR) mx_pair_inv<V>(x, w, cx);
        mx_dft<V>(x, m, cx);
        MxMap<P::words(2), V>::store(t, x);
        m = mx_load_mat(cx, kMxInv);
        mx_load_tw<P::logs(1), 0, V>(tw, cx.ti);
        mx_sync<P::words(1), V>();
        MxMap<P::words(1), V>::load(t, x);
        mx_mul<V>(x, tw, cx);
        mx_dft<V>(x, m, cx);
        MxMap<P::words(1), V>::store(t, x);
        mx_load_tw<P::logs(0), 0, V>(tw, cx.ti);
    }
    __syncthreads();
    if (act) {
        MxMap<P::words(0), V>::load(t, x);
        mx_mul<V>(x, tw, cx);
        mx_dft<V>(x, m, cx);
#pragma unroll
        for (int s = 0; s < V; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) x[s][r] = mx_canon(x[s][r], cx);
    }
}

// Newton step of g in LDS from h = 2^(LOGL-1) to 2h words: f g = 1 + x^h E mod
// x^(2h), and g takes -(g E) mod x^h as its high half.  -E stays where the
// cyclic product on 2h points leaves it (words h .. 2h-1), and so does the new
// high half, so nothing moves between lanes.  f = rev(root).
template <int LOGL, int V>
CM_DEV void inv_step(u32 *A, u32 *B, u32 *g, const u32 *root_top, const MxCtx &cx) {
    constexpr int N = 1 << LOGL, H = N / 2;
    using Map = MxMap<MxPlan<LOGL, 0, V>::words(0), V>;
    const bool act = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < N / (256 * V);
    const int b = Map::base();
    u32 x[2][V][4];
    if (act) {
#pragma unroll
        for (int s = 0; s < V; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = b + Map::off(s, r);
                x[0][s][r] = root_top[-i];
                x[1][s][r] = i < H ? g[i] : 0u;
            }
    }
    u32 *const ab[2] = {A, B}, *const tb[1] = {B};
    inv_forward<LOGL, V, 2>(x, ab, act, cx);
    inv_product<LOGL, V>(x[0], x[1], A, act, cx);
    if (act) {
#pragma unroll
        for (int s = 0; s < V; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                x[0][s][r] = b + Map::off(s, r) >= H ? cm_sub(0u, x[0][s][r], cx.p) : 0u;
    }
    inv_forward<LOGL, V, 1>(reinterpret_cast<u32 (&)[1][V][4]>(x[0]), tb, act, cx);
    inv_product<LOGL, V>(x[0], x[1], A, act, cx);
    if (act) {
#pragma unroll
        for (int s = 0; s < V; ++s)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = b + Map::off(s, r);
                if (i >= H) g[i] = x[0][s][r];
            }
    }
    __syncthreads();
}

// J[-1-t] = [x^t] rev(root)^-1 for t < 2^prec (9 <= prec <= kInvRootLog), with
// root_top the address of the root's leading word and J one past the inverse's
// last.  One workgroup: a chain of prec - 4 Newton steps from 16 words (the
// recurrence, one thread), as sums of products up to 256 words and five
// transforms each from there.  11.8 us for 2^9 words, 15.7, 21.1, 29.0 and 45.1 us
// for 2^10 .. 2^13 (a step of 2^13 points as two four-step products: 21 us
// against the 16 us it takes here).
__global__ __launch_bounds__(1024) void k_inv_root(const u32 *__restrict__ root_top, int prec,
                                                   PlainMod pm, MxCtx cx, u32 *__restrict__ J) {
    constexpr int W = mx_lds_words(1 << kInvRootLog), H0 = 16, S = 256, PARTS = 8;
    __shared__ __align__(16) u32 A[W], B[W], g[1 << kInvRootLog];
    static_assert(W >= 1024 && W >= S + S / 2, "sums");
    u32 *const f = B, *const E = B + S, *const pp = A;
    const int tid = threadIdx.x, t = tid & (S / 2 - 1), part = tid / (S / 2);
    if (tid < S) f[tid] = root_top[-tid];
    __syncthreads();
    if (tid == 0) {
        u32 fl[H0], gl[H0];
#pragma unroll
        for (int i = 1; i < H0; ++i) fl[i] = f[i];
        gl[0] = 1u;
#pragma unroll
        for (int w = 1; w < H0; ++w) {
            u64 acc = 0;
#pragma unroll
            for (int i = 1; i <= w; ++i) {
                acc += (u64)fl[i] * gl[w - i];
                if ((i & 3) == 0) acc = plain_fold(acc, pm.c32);
            }
            gl[w] = cm_sub(0u, plain_reduce(acc, pm), pm.p);
        }
#pragma unroll
        for (int w = 0; w < H0; ++w) g[w] = gl[w];
    }
    __syncthreads();
    auto sum = [&]() {
        u32 v = 0;
#pragma unroll
        for (int q = 0; q < PARTS; ++q) v = cm_add(v, pp[q * (S / 2) + t], pm.p);
        return v;
    };
    for (int h = H0; h < S; h *= 2) {
        // -E_t = -sum_(k < h) f_(t+1+k) g_(h-1-k)
        if (t < h) {
            const int k0 = part * (h / PARTS);
            pp[tid] = plain_dot<1, -1>(f + t + 1 + k0, g + h - 1 - k0, h / PARTS, pm);
        }
        __syncthreads();
        if (tid < h) E[t] = cm_sub(0u, sum(), pm.p);
        __syncthreads();
        if (t < h) pp[tid] = plain_dot_part<1, -1, PARTS>(g, E + t, t + 1, part, pm);
        __syncthreads();
        if (tid < h) g[h + t] = sum();
        __syncthreads();
    }
    inv_step<9, 1>(A, B, g, root_top, cx);
    if (prec >= 10) inv_step<10, 1>(A, B, g, root_top, cx);
    if (prec >= 11) inv_step<11, 1>(A, B, g, root_top, cx);
    if (prec >= 12) inv_step<12, 1>(A, B, g, root_top, cx);
    if (prec >= 13) inv_step<13, 2>(A, B, g, root_top, cx);
    for (int i = tid; i < 1 << prec; i += 1024) J[-1 - i] = g[i];
}

// The last kMidBase levels: workgroup j takes node j of level kMidBase (256
// words of b) down to its 256 values in LDS.  Level i, thread t = c h + v (h =
// 2^i): b[v] + sum_(k < h) S_(h-1-k) b[v+1+k], the leading 1 of S apart; from
// 64 words up the sum is split over four threads, below that a node stays
// within a wave.  256 nodes take 7.3 us.
struct MidOffsets {
    int64_t off[kMidBase];   // word of level l in the tree
};

__global__ __launch_bounds__(4 << kMidBase) void k_mid_descend(const u32 *__restrict__ b,
                                                              const u32 *__restrict__ tree,
                                                              MidOffsets lo, PlainMod pm,
                                                              u32 *__restrict__ val) {
    constexpr int N = 1 << kMidBase, SPLIT = 6;
    __shared__ u32 cur[2][N], pp[4 * N], M[kMidBase * N + 2 * N];
    const int64_t j = blockIdx.x;
    const int tid = threadIdx.x, t = tid & (N - 1), part = tid / N;
    auto at = [](int l) { return l * N + 2 * N - ((2 * N) >> l); };   // level l in M
    if (part == 0) cur[0][t] = b[j * N + t];
#pragma unroll
    for (int l = 0; l < kMidBase; ++l) {
        const int words = N + (N >> l);
        const u32 *m = tree + lo.off[l] + j * words;
        if (tid < words) M[at(l) + tid] = m[tid];
    }
    __syncthreads();
#pragma unroll
    for (int i = kMidBase - 1; i >= 0; --i) {
        const int h = 1 << i, c = t >> i, v = t & (h - 1);
        const u32 *par = cur[(i + 1) & 1] + (c >> 1) * (2 * h);
        const u32 *S = M + at(i) + (c ^ 1) * (h + 1);
        u32 *out = cur[i & 1] + t;
        if (i >= SPLIT) {
            const int k0 = part * (h / 4);
            pp[tid] = plain_dot<-1, 1>(S + h - 1 - k0, par + v + 1 + k0, h / 4, pm);
            __syncthreads();
            if (part == 0)
                *out = cm_add(cm_add(cm_add(pp[t], pp[N + t], pm.p),
                                     cm_add(pp[2 * N + t], pp[3 * N + t], pm.p), pm.p),
                              par[v], pm.p);
            __syncthreads();
        } else {
            if (part) return;
            *out = cm_add(plain_dot<-1, 1>(S + h - 1, par + v + 1, h, pm), par[v], pm.p);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
    static_assert(kMidBase > SPLIT, "the values end in cur[0]");
    val[j * N + t] = cur[0][t];
}

// The product at the root is on 2^(k+1) points, which the modulus and the
// largest transform have to allow.  2^9 points: 39.8 us against 81.2 us by the
// remainder tree, 2^13: 142 against 343 us; at 2^8, one node of k_mid_descend, the
// remainder tree is a few launches (31.1 us).
bool evaluate_transposed_takes(int k, const Family *fam) {
    return k > kMidBase && k + 1 <= std::min(fam->K, kMaxLog);
}

hipError_t launch_evaluate_transposed(const u32 *F, int k, const u32 *tree, u32 *work, u32 *values,
                                      const Family *fam, hipStream_t s) {
    const int64_t n = (int64_t)1 << k;
    u32 *J = work, *E = J + n, *b = E + n, *next = b + n;
    const PlainMod pm = plain_mod(fam->p);
    const u32 *top = tree + tree_level_offset(k, k) + n;     // the root's leading word
    const int prec = std::min(k, kInvRootLog);
    hipLaunchKernelGGL(k_inv_root, dim3(1), dim3(1024), 0, s, top, prec, pm, mx_ctx(fam), J + n);
    hipError_t e = hipGetLastError();
    // Newton steps on reversed words: the last 2h words of the root times the
    // last h of J hold E at h-1 .. 2h-2, and so does -E times J the new words
    for (int q = prec; q < k && e == hipSuccess; ++q) {
        const int64_t h = (int64_t)1 << q;
        u32 *g = J + n - h;
        e = launch_mul_middle(q + 1, {top - 2 * h + 1, g, 0, 0, 0, 2 * h, h, E, h - 1, h, 1, 1}, fam,
                              s);
        if (e == hipSuccess)
            e = launch_mul_middle(q + 1, {E, g, 0, 0, 0, h, h, g - h, h - 1, h, 1, 0}, fam, s);
    }
    if (e == hipSuccess)
        e = launch_mul_middle(k + 1, {J, F, 0, 0, 0, n, n, b, n - 1, n, 1, 0}, fam, s);
    for (int i = k - 1; i >= kMidBase && e == hipSuccess; --i) {
        const int64_t h = (int64_t)1 << i;
        e = launch_mul_middle(i + 1,
                              {tree + tree_level_offset(k, i), b, h + 1, 2 * h, h, h + 1, 2 * h,
                               next, h, h, (int)(n >> i), 0},
                              fam, s);
        std::swap(b, next);
    }
    if (e != hipSuccess) return e;
    MidOffsets lo;
    for (int l = 0; l < kMidBase; ++l) lo.off[l] = tree_level_offset(k, l);
    hipLaunchKernelGGL(k_mid_descend, dim3((unsigned)(n >> kMidBase)), dim3(4 << kMidBase), 0, s, b,
                       tree, lo, pm, values);
    return hipGetLastError();
}

}  // namespace cm
