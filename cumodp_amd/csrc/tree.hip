// tree.hip -- subproduct tree over 2^k points, level by level.
//
// Reference: onlySubproductTree / subProductTree
// (src/fastPolyEvaluation.cu:512-656, :1411-1434).  The reference keeps two
// half-trees (Ml, Mr), leaves (-x_i, 1) with the raw negative, schoolbook
// products up to level 8 and FFT products with an implicit leading 1 above,
// and never forms the root.  Here one tree holds every level 0..k, each node
// the monic product of 2^i consecutive (x - x_j) stored with its leading
// coefficient (2^i + 1 canonical words), level i starting at word
//     off(i) = sum_{l < i} 2^(k-l) (2^l + 1).
// Level i is one batch of products on 2^i points of the whole monic nodes of
// level i-1 (leading 1 included): the product's x^(2^i) wraps onto its constant
// term, which the store takes back while it writes the leading 1, so a level
// is one launch up to 2^12 points and three above (of 2^13 points three for 2 to
// 32 nodes and one otherwise), with no pass that adds the leading terms.  (The reference multiplies without the leading terms and adds
// x^h (a + b) afterwards, :601-650.)  Levels 0 .. 8 are built before that in
// one launch, a 256-point subtree per workgroup (k_tree_bottom).
#include "accum.h"
#include "internal.h"

namespace cm {

int64_t tree_level_offset(int k, int i) {
    int64_t off = 0;
    for (int l = 0; l < i; ++l) off += ((int64_t)1 << (k - l)) * (((int64_t)1 << l) + 1);
    return off;
}

// Levels 0 .. pin of the tree in one launch: workgroup J (blockDim.x =
// kTreeParts 2^pin threads, 1 <= pin <= kTreeFuse) builds the subtree over points
// J 2^pin .. J 2^pin + 2^pin - 1 in LDS, level by level, and writes every
// level's nodes (a contiguous block of each level) to the tree.  LDS holds the
// nodes without their leading 1.  Word r of a node of 2h words (children a, b of
// h words) is sum_u a_u b_(r-u) and, from the children's leading terms,
// a_(r-h) + b_(r-h) for r >= h: a schoolbook sum in a 64-bit accumulator
// (accum.h).
//
// Bound by the chain of LDS loads and multiply-adds of a thread: 256 one after
// the other if a word has one thread.  The levels above 64 words split each sum
// over kTreeParts threads; up to 64 words a node stays within a wave, which
// needs no barrier.  Whole tree of 2^16 points: 84.6 us with one thread per
// word, 78.8 us so.
constexpr int kTreeFuse = 8;
constexpr int kTreeParts = 4;

__global__ __launch_bounds__(kTreeParts << kTreeFuse) void k_tree_bottom(
    const u32 *__restrict__ pts, int pin, PlainMod pm, u32 *__restrict__ tree, int64_t n) {
    constexpr int BMAX = 1 << kTreeFuse, WAVE = 6;
    __shared__ u32 buf[2][BMAX], pp[kTreeParts * BMAX];
    static_assert(kTreeParts == 4, "the partial sums are added as four terms");
    const int B = 1 << pin;
    const int64_t J = blockIdx.x;
    const int tid = threadIdx.x, t = tid & (B - 1), part = tid >> pin;
    const u32 p = pm.p;
    // word r of node c of level i, of 2h words, to the tree; then its leading 1
    auto put = [&](int i, int64_t off, u32 v) {
        const int H = 1 << i, c = t >> i, r = t & (H - 1);
        u32 *out = tree + off + ((J << (pin - i)) + c) * (H + 1) + r;
        buf[i & 1][t] = v;
        out[0] = v;
        if (r == H - 1) out[1] = 1u;
    };
    // part q of the sum of word t of level i, and what the leading terms add
    auto sum = [&](int i, int q, int parts) {
        const int h = 1 << (i - 1), r = t & (2 * h - 1);
        const u32 *a = buf[(i - 1) & 1] + (t - r), *b = a + h;
        const int lo = r < h ? 0 : r - h + 1, cnt = r < h ? r + 1 : 2 * h - 1 - r;
        const int k0 = cnt * q / parts, k1 = cnt * (q + 1) / parts;
        return plain_dot<1, -1>(a + lo + k0, b + (r - lo - k0), k1 - k0, pm);
    };
    auto lead = [&](int i) {
        const int h = 1 << (i - 1), r = t & (2 * h - 1);
        const u32 *a = buf[(i - 1) & 1] + (t - r);
        return r < h ? 0u : cm_add(a[r - h], a[r], p);
    };
    int64_t off = 0;                          // level i of the tree
    if (part == 0) {
        const u32 x = pts[J * B + t] % p;
        put(0, 0, x ? p - x : 0u);
    }
#pragma unroll
    for (int i = 1; i <= WAVE; ++i) {
        if (i > pin) return;
        off += (n >> (i - 1)) * ((1 << (i - 1)) + 1);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (part == 0) put(i, off, cm_add(sum(i, 0, 1), lead(i), p));
    }
#pragma unroll
    for (int i = WAVE + 1; i <= kTreeFuse; ++i) {
        if (i > pin) return;
        off += (n >> (i - 1)) * ((1 << (i - 1)) + 1);
        __syncthreads();
        pp[tid] = sum(i, part, kTreeParts);
        __syncthreads();
        if (part == 0)
            put(i, off, cm_add(cm_add(cm_add(pp[t], pp[B + t], p),
                                      cm_add(pp[2 * B + t], pp[3 * B + t], p), p),
                               lead(i), p));
    }
}

hipError_t launch_subproduct_tree(const u32 *pts, int k, u32 p, u32 *tree, const Family *fam,
                                  hipStream_t s) {
    const int64_t n = (int64_t)1 << k;
    // levels 0 .. pin in one launch, one workgroup per 2^pin points
    const int pin = k < kTreeFuse ? k : kTreeFuse;
    hipLaunchKernelGGL(k_tree_bottom, dim3((unsigned)(n >> pin)), dim3(kTreeParts << pin), 0, s, pts,
                       pin, plain_mod(p), tree, n);
    hipError_t e = hipGetLastError();
    for (int i = pin + 1; i <= k && e == hipSuccess; ++i) {
        e = launch_tree_level(i, tree + tree_level_offset(k, i - 1),
                              tree + tree_level_offset(k, i), n >> i, fam, s);
    }
    return e;
}

}  // namespace cm
