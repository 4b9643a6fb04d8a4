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
// is one launch up to 2^13 points and three above, with no pass that adds the
// leading terms.  (The reference multiplies without the leading terms and adds
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
// 2^pin threads, pin <= kTreeFuse) builds the subtree over points
// J 2^pin .. J 2^pin + 2^pin - 1 in LDS, level by level, and writes every
// level's nodes (a contiguous block of each level) to the tree.  Node
// coefficient r of level i (children a, b of level i-1, h + 1 words each,
// h = 2^(i-1)) is sum_u a_u b_(r-u), a schoolbook sum in a 64-bit
// accumulator (accum.h); the leading coefficients are 1 and come out of the
// same sum.
constexpr int kTreeFuse = 8;

__global__ __launch_bounds__(1 << kTreeFuse) void k_tree_bottom(const u32 *__restrict__ pts,
                                                               int pin, PlainMod pm,
                                                               u32 *__restrict__ tree,
                                                               int64_t n) {
    constexpr int BMAX = 1 << kTreeFuse;
    __shared__ u32 buf[2][2 * BMAX];
    const int B = 1 << pin;
    const int64_t J = blockIdx.x;
    const int t = threadIdx.x;
    {
        const u32 x = pts[J * B + t] % pm.p;
        const u32 lo = x ? pm.p - x : 0u;
        buf[0][2 * t] = lo;
        buf[0][2 * t + 1] = 1u;
        tree[2 * (J * B + t)] = lo;
        tree[2 * (J * B + t) + 1] = 1u;
    }
    int64_t off = 0;                          // word offset of level i - 1 in the tree
    for (int i = 1; i <= pin; ++i) {
        __syncthreads();
        const int h = 1 << (i - 1);
        const int len = 2 * h + 1, nodes = B >> i;
        off += (n >> (i - 1)) * (h + 1);      // level i
        const u32 *prev = buf[(i - 1) & 1];
        u32 *cur = buf[i & 1];
        u32 *out = tree + off + (J * nodes) * len;
        for (int x = t; x < nodes * len; x += B) {
            const int c = x / len, r = x - c * len;
            const u32 *a = prev + (2 * c) * (h + 1), *b = a + (h + 1);
            const int lo = r > h ? r - h : 0, hi = r < h ? r : h;
            const u32 v = plain_dot<1, -1>(a + lo, b + (r - lo), hi - lo + 1, pm);
            cur[x] = v;
            out[x] = v;
        }
    }
}

hipError_t launch_subproduct_tree(const u32 *pts, int k, u32 p, u32 *tree, const Family *fam,
                                  hipStream_t s) {
    const int64_t n = (int64_t)1 << k;
    // levels 0 .. pin in one launch, one workgroup per 2^pin points
    const int pin = k < kTreeFuse ? k : kTreeFuse;
    hipLaunchKernelGGL(k_tree_bottom, dim3((unsigned)(n >> pin)), dim3(1 << pin), 0, s, pts, pin,
                       plain_mod(p), tree, n);
    hipError_t e = hipGetLastError();
    for (int i = pin + 1; i <= k && e == hipSuccess; ++i) {
        e = launch_tree_level(i, tree + tree_level_offset(k, i - 1),
                              tree + tree_level_offset(k, i), n >> i, fam, s);
    }
    return e;
}

}  // namespace cm
