// internal.h -- shared declarations of the cumodp_amd runtime (not installed).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <functional>
#include <mutex>
#include <vector>

#include "modarith.h"

namespace cm {

constexpr int kMaxLdsLog = 13;     // largest multiply done inside one workgroup
constexpr int kMaxLevelLog = 15;   // largest level of the twiddle tables (in-LDS 2^15 products)
constexpr int kMaxLog = 26;        // largest transform supported (2^13 x 2^13)
constexpr int kNoAllocMaxLog = 22; // largest transform of the non-allocating multiply

// Scratch of the non-allocating multiply (noalloc.hip): a file-scope device
// array of noalloc_scratch_words() words, one copy per device.  noalloc_scratch
// returns its device address on the current device (looked up once per
// device; no allocation).
size_t noalloc_scratch_words();
hipError_t noalloc_scratch(u32 **out);

// A family of roots of unity: w_N of order N = 2^K and all its powers
// w_{2^k} = w_N^(2^(K-k)).  Tables live in device memory for the process
// lifetime (cached, never freed).
struct Family {
    u32 p, pinv, np;      // pinv = p^-1, np = -p^-1 (mod 2^32)
    int K;
    u32 wN;
    int LT;               // largest level of the twiddle tables (min(K, kMaxLevelLog))
    // level tables: for M = 2 .. 2^LT, w_M^q (q < M/2) at offset M/2 - 1,
    // in Montgomery form (w 2^32 mod p); lvi holds the inverse roots' powers
    u32 *lv, *lvi;
    // matrix-core transforms (ntt_mx.h; null when K < 4): the byte matrices,
    // and for M = 32 .. 2^LT the twiddles w_M^(k v) (k < 16, v < S = M / 16)
    // at M + k S + v, with their inverses
    void *mx_mat;
    u32 *mx_tf, *mx_ti;
};

// Four-step outer twiddles w_n^e for one transform size n = 2^k
// (n = 2^k1 rows x 2^k2 columns).
// For a row with frequency index k1 and T = 2^k2 / 16, element i = t + T m
// (m < 16): w_n^(k1 i) = rb[k1 T + t] * rc[16 k1 + m].
// The _f tables use w_n, the _i tables w_n^-1; all in Montgomery form.
struct Outer {
    int k, k1, k2;        // the split these tables were built for
    u32 *rb_f, *rc_f, *rb_i, *rc_i;
};

// Family lookup: the library's default root family for p (w from the
// smallest generator), or the family generated by a caller-supplied root w of
// order 2^k.  Returns nullptr on allocation failure.
const Family *family_default(u32 p);
const Family *family_for_root(u32 p, u32 w, int k);
const Outer *outer_for(const Family *f, int k);   // for the current split of k
const Outer *outer_for_split(const Family *f, int k, int k1, int k2);
// The same lookups that never build (and so never allocate): nullptr when the
// tables are not built yet.
const Family *family_default_cached(u32 p);
const Outer *outer_cached(const Family *f, int k);

// four-step split of a transform of size 2^k (kMaxLdsLog < k <= kMaxLog):
// columns of 2^k1 words, rows of 2^k2, as cumodp_tune_set_split or
// CUMODP_SPLIT_<k>=<k2> names them, else the library's own
void four_step_split(int k, int &k1, int &k2);
bool set_four_step_split(int k, int k2);

// Grow-only device scratch buffers owned by the library, one per (slot,
// stream): work queued on different streams never shares scratch, and work on
// one stream is ordered by the stream.  Entry points enqueue under
// api_mutex(), so two host threads never interleave their launches.
void *workspace(int slot, size_t bytes, hipStream_t s);
// frees the scratch buffers (and auxiliary streams) of a stream that is being
// destroyed (synchronised)
void release_workspace(hipStream_t s);

// Auxiliary streams of a caller stream, for running independent parts of one
// call concurrently (fork after `fork` is recorded on the caller stream, join
// through `join`).  Default priority; created on first use, destroyed with
// the caller stream's scratch.
constexpr int kAuxStreams = 4;
struct AuxStreams {
    hipStream_t s[kAuxStreams];
    hipEvent_t fork, join[kAuxStreams];
};
AuxStreams *aux_streams(hipStream_t s);
// host -> device copy of a small descriptor blob through pinned staging
// (stream ordered; the host buffer is reused once its previous copy is done).
// While s is being captured into a graph the copy reads a dedicated pinned
// buffer that the graph owns (take_captured_buffers).
hipError_t stage_upload(const void *src, size_t bytes, void *dst, hipStream_t s);
// the same with the bytes written by fill() straight into the pinned buffer
// (no intermediate copy)
hipError_t stage_upload_fill(size_t bytes, void *dst, hipStream_t s,
                             const std::function<void(char *)> &fill);
bool stream_capturing(hipStream_t s);
std::vector<void *> take_captured_buffers(hipStream_t s);
// A graph captured on s refers to the scratch buffers of s and of its
// auxiliary streams: hold_workspace_for_graph marks them held (returned for
// the graph to keep) so that neither a later, larger eager call on s nor the
// destruction of s frees them; release_graph_workspace (at graph
// destruction, after the device has finished its replays) frees those no
// stream uses any more.
std::vector<void *> hold_workspace_for_graph(hipStream_t s);
void release_graph_workspace(const std::vector<void *> &held);

// Serialises host-API calls that share workspace.
std::mutex &api_mutex();

// ---- optional per-kernel timing (prof.cpp) ----------------------------------
enum ProfId {
    kProfColFwd, kProfRowMul, kProfColInv, kProfMulLds, kProfMulMixed, kProfNttLds,
    kProfRowOut, kProfGatherScatter, kProfTcSplit, kProfTcCrt, kProfColNtt, kProfElementwise,
    kProfPlainMul, kProfListPersistent, kProfCount
};

// Records a HIP event pair around the launches in its scope when profiling is
// enabled; does nothing otherwise, nor while this thread has timing
// suspended (prof_suspend: calls that must not create events).
class ProfScope {
  public:
    ProfScope(int id, hipStream_t s);
    ~ProfScope();
    ProfScope(const ProfScope &) = delete;
    ProfScope &operator=(const ProfScope &) = delete;

  private:
    int id_;
    hipStream_t s_;
    void *ev_ = nullptr;
};

// Pointwise constant of a 2^logn-point multiply: the Montgomery form of
// 2^32 / 2^logn mod p (two lazy Montgomery products and the 1/N of the
// inverse transform folded into one factor).
u32 mul_scale(int logn, u32 p);

// Suspends (true) or resumes per-kernel timing on the calling thread.
void prof_suspend(bool on);

// ---- launchers (stream-ordered, no synchronisation) -----------------------
struct MulDesc {           // one product of a batch (word offsets)
    int64_t f, g, h;
    int32_t lf, lg, lh, logn;
};

// Schoolbook H[d] = F[d] * G[d] mod p (plain.hip) for any odd p < 2^31;
// descriptor logn != 0 marks an item whose G operand is the longer one.
hipError_t launch_plain_list(const MulDesc *descs, int64_t count, const u32 *F, const u32 *G,
                             u32 *H, u32 p, hipStream_t s);
// count items of one shape at strides fs, gs, hs: the first lh words of
// F[d fs ..] * G[d gs ..] (lh <= lf + lg - 1) to H + d hs
hipError_t launch_plain_strided(const u32 *F, int64_t fs, int lf, const u32 *G, int64_t gs,
                                int lg, u32 *H, int64_t hs, int lh, int count, u32 p,
                                hipStream_t s);

// H[d] = F[d] * G[d] mod p for descriptors with transform size 2^logn <= 2^13
hipError_t launch_mul_lds(int logn, const u32 *F, const u32 *G, u32 *H, const MulDesc *d_descs,
                          int ndesc, const Family *fam, hipStream_t s);
// same; with d_descs == nullptr the single descriptor `one` is passed by value
hipError_t launch_mul_lds_one(int logn, const u32 *F, const u32 *G, u32 *H,
                              const MulDesc *d_descs, int ndesc, const MulDesc &one,
                              const Family *fam, hipStream_t s);

// product d at d times the strides sd.f / sd.g / sd.h, lengths sd.lf / lg / lh
hipError_t launch_mul_lds_strided(int logn, const u32 *F, const u32 *G, u32 *H, const MulDesc &sd,
                                  int count, const Family *fam, hipStream_t s);

// In-place natural-order DFT of m rows of 2^k words (k <= 13); inverse uses
// the inverse root and scales by 2^-k.
hipError_t launch_ntt_lds(int k, u32 *X, int64_t m, bool inverse, const Family *fam,
                          hipStream_t s);

// Operands of a batch of four-step multiplies of size n = 2^k: pair a reads
// f_in[a*in_stride + i] for i < f_len (zero beyond; likewise g), works in
// f_ws/g_ws (n words per pair, stride n; in_* may equal ws_*) and writes
// h_out[a*out_stride + i] for i < h_len (cyclic product mod x^n - 1).
struct FourStepIO {
    const u32 *f_in, *g_in;
    int64_t f_len, g_len, in_stride;
    u32 *f_ws, *g_ws;
    u32 *h_out;
    int64_t h_len, out_stride;
    int cnt;
    int64_t g_stride = -1;   // stride of g_in when it differs from in_stride
    // pair a takes array a >> g_shift of g (g_ws has cnt >> g_shift arrays) and
    // writes output a ^ out_xor, words out_from .. h_len - 1; monic: operands
    // are monic of n/2 + 1 words, outputs monic of n + 1; neg: outputs negated
    int g_shift = 0, out_from = 0, out_xor = 0, monic = 0, neg = 0;
};
hipError_t launch_mul_four_step(int k, const FourStepIO &io, const Family *fam, hipStream_t s);
// the same with tables the caller looked up (no table is built here)
hipError_t launch_mul_four_step_with(const FourStepIO &io, const Family *fam, const Outer *o,
                                     hipStream_t s);

// Level i of the subproduct tree from level i - 1: node d of `cur` (2^i + 1
// words) is the product of nodes 2d and 2d + 1 of `prev` (2^(i-1) + 1 words).
hipError_t launch_tree_level(int i, const u32 *prev, u32 *cur, int64_t nodes, const Family *fam,
                             hipStream_t s);

// Middle products of one shape on 2^logn points (9 <= logn <= kMaxLog): product
// a reads lf words at f + a fs and lg words at g + (a >> 1) gs and writes words
// from .. from + len - 1 of the cyclic product to h + (a ^ 1) hs (a single
// product: fs, gs and hs 0).  neg: negated (logn > kMaxLdsLog only).
struct MidProduct {
    const u32 *f, *g;
    int64_t fs, gs, hs, lf, lg;
    u32 *h;
    int64_t from, len;
    int cnt, neg;
};
hipError_t launch_mul_middle(int logn, const MidProduct &q, const Family *fam, hipStream_t s);

// count products of one shape: product d reads lf words at F + d fs and lg
// words at G + d gs and writes the first lh words of the 2^logn-point cyclic
// product to H + d hs (no descriptors; outputs must not overlap the inputs
// when 2^logn > 2^13).
hipError_t launch_mul_strided(int logn, const u32 *F, int64_t fs, int lf, const u32 *G,
                              int64_t gs, int lg, u32 *H, int64_t hs, int lh, int count,
                              const Family *fam, hipStream_t s);

// Four-step natural-order DFT of cnt arrays of 2^k words (in place, using Y as
// cnt * 2^k words of temporary space); inverse as in launch_ntt_lds.
hipError_t launch_ntt_four_step(int k, u32 *X, u32 *Y, int cnt, bool inverse, const Family *fam,
                                hipStream_t s);

// Natural-order column DFTs of a row-major 2^em x ncols array (em <= 13),
// in place; outputs multiplied by the residue `scale` (1: none).  nblk
// arrays bstride words apart (nblk <= 65535).
hipError_t launch_col_ntt(int em, u32 *X, int64_t ncols, u32 scale, const Family *fam,
                          hipStream_t s, int nblk = 1, int64_t bstride = 0);

// Many products of uneven size (host descriptors with logn set; offsets into
// F, G, H).  Outputs must not overlap each other or the inputs.
hipError_t launch_list_mul(const MulDesc *descs, int64_t count, const u32 *F, const u32 *G,
                           u32 *H, const Family *fam, hipStream_t s);

// words per column tile of the four-step multiply's column passes (8192 or
// 16384)
bool set_col_tile_words(int words);
int col_tile_words();

// words per mixed-size tile of launch_list_mul (2048, 4096 or 8192)
bool set_list_tile_words(int words);
int list_tile_words();
bool set_list_plain_cutoff(int c);
int list_plain_cutoff();
// schoolbook cut-off of the strided (equal-shape) multiplies of tree and
// evaluation levels
int strided_plain_cutoff();
// 1: every product of a list call up to 2^15 points in one persistent launch
// (default); 0: one launch per size class
bool set_list_persistent(int on);
int list_persistent();

// F[r] <- F[r] * G[r] mod x^(2^e) - 1 for `rows` contiguous rows of 2^e words
// (G overwritten when 2^e > 2^13).
hipError_t launch_rows_mul(int e, u32 *F, u32 *G, int rows, const Family *fam, hipStream_t s);

// f[r] <- f[r] * g[r] mod x^(2^e) - 1 for the rows of several segments, each of
// one length and modulus (rows_batch.hip); only the first flen / glen words of
// a row of f / g are read, g is overwritten.
struct RowSeg {
    u32 *f, *g;
    int rows, e, flen, glen;
    const Family *fam;
};
hipError_t launch_rows_batch(std::vector<RowSeg> segs, hipStream_t s);

// two-convolution integer multiply on device buffers (twoconv.hip); *err is
// set when no (K, M, primes) satisfies the CRT bound
hipError_t launch_two_convolution(const u64 *a, int64_t na, int wa, const u64 *b, int64_t nb,
                                  int wb, u64 *c, int wc, int bits, hipStream_t s, int *err);
// batch of exact integer products (word offsets into A, B, C); *err is set
// when no plan fits an item
struct TcItem {
    int64_t a_off, b_off, c_off, na, nb;
    int32_t wa, wb, wc, bits;
};
hipError_t launch_two_convolution_list(const TcItem *items, int64_t count, const u64 *A,
                                       const u64 *B, u64 *C, hipStream_t s, int *err);
bool set_zmul_merge(int m);
int zmul_merge();
hipError_t launch_scale_x(u32 *A, int64_t len, int K, u32 theta, u32 p, hipStream_t s);
int tc_bit_width(const u64 *a, int64_t n, int w);
int tc_plan_info(int bits, int64_t na, int64_t nb, int *np, int *K, int *M);

// subproduct tree (tree.hip): levels 0..k of the monic products over 2^k
// points, level i at word tree_level_offset(k, i), nodes of 2^i + 1 words
int64_t tree_level_offset(int k, int i);
hipError_t launch_subproduct_tree(const u32 *pts, int k, u32 p, u32 *tree, const Family *fam,
                                  hipStream_t s);

// fast multipoint evaluation (eval.hip): values[x] = F(pts[x]) for 2^k points,
// F with 2^k coefficients (any 32-bit words, reduced mod p); scratch of
// eval_scratch_words(k) words.  The scratch begins with the subproduct tree
// (tree_level_offset layout) followed, at eval_inverse_offset(k), by the
// subinverse tree: level i (i >= min(k, 4)) at (i - min(k, 4)) 2^k words,
// node j at 2^i j, I_i(j) = rev(M_i(j))^-1 mod x^(2^i).
// keep (optional): trees_only stops after the two trees; rem != nullptr
// receives every remainder level, level i (0 <= i < k) at rem + i 2^k, node
// j at 2^i j holding F mod M_i(j) (level 0: the values).
struct EvalKeep {
    u32 *rem = nullptr;
    bool trees_only = false;
};
int64_t eval_scratch_words(int k);
int64_t eval_inverse_offset(int k);
// tree level 0 in the reference's layout: (-x, 1) per point, the first nh
// points to left, the next nh to right (2 nh words each)
hipError_t launch_ref_leaves(const u32 *pts, int64_t nh, u32 *left, u32 *right, hipStream_t s);
// the values alone, by the transposed algorithm (eval_mid.hip), from the
// subproduct tree at `tree` and 4 2^k further words at `work`, where
// evaluate_transposed_takes holds
bool evaluate_transposed_takes(int k, const Family *fam);
hipError_t launch_evaluate_transposed(const u32 *F, int k, const u32 *tree, u32 *work, u32 *values,
                                      const Family *fam, hipStream_t s);
hipError_t launch_fast_evaluation(const u32 *F, const u32 *pts, int k, u32 p, u32 *values,
                                  u32 *scratch, const Family *fam, hipStream_t s,
                                  const EvalKeep *keep = nullptr);

// elementwise helpers (src/fft_aux.cu:70-322 equivalents)
hipError_t launch_pointwise(u32 *Y, const u32 *X, int64_t n, u32 p, hipStream_t s);
hipError_t launch_scale(u32 *X, int64_t n, u32 a, u32 p, hipStream_t s);
hipError_t launch_powers(u32 *W, int64_t n, u32 w, u32 p, hipStream_t s);
hipError_t launch_fill(u32 *X, int64_t n, u32 v, hipStream_t s);

}  // namespace cm
