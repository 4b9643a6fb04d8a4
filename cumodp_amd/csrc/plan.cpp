// plan.cpp -- device-resident twiddle tables and scratch buffers.
//
// The reference rebuilds its twiddle table W[j] = w^j on every call
// (get_powers_binary, src/fft_aux.cu:87-132, one 4 KB host copy plus e-10
// doubling launches) and cudaMallocs every temporary.  Here each root family
// is built once per process, on the host, in Montgomery form, and kept in
// device memory; scratch space grows and is reused.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <tuple>
#include <vector>

#include "internal.h"
#include "ntt_mx.h"

namespace cm {

std::mutex &api_mutex() {
    static std::mutex m;
    return m;
}

namespace {

std::mutex g_plan_mutex;
std::map<std::tuple<u32, u32, int>, Family *> g_families;
std::map<std::tuple<const Family *, int, int>, Outer *> g_outer;
int g_split[kMaxLog + 1];   // named k2 per k (0: none)
std::map<u32, const Family *> g_default;

u32 *upload(const std::vector<u32> &h) {
    u32 *d = nullptr;
    if (hipMalloc((void **)&d, sizeof(u32) * h.size()) != hipSuccess) return nullptr;
    if (hipMemcpy(d, h.data(), sizeof(u32) * h.size(), hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(d);
        return nullptr;
    }
    return d;
}

// r^0 .. r^(2^log - 1) in Montgomery form, by doubling: t[h + j] = r^h t[j], so no
// entry waits for its neighbour.  The first 2^12-point product modulo a new prime
// takes 0.24 ms with the tables built this way, 0.82 with chains of 64-bit
// remainders; the first product of 2^22 points 1.20 against 2.75 ms.
void power_table(u32 *t, u32 r, int log, u32 p) {
    t[0] = cm_host_mont(1, p);
    u32 w = r;   // r^h
    for (size_t h = 1; h < (size_t)1 << log; h *= 2) {
        const u32 wq = cm_host_shoup_q(w, p);
        for (size_t j = 0; j < h; ++j) t[h + j] = cm_shoup(t[j], w, wq, p);
        w = cm_host_mul(w, w, p);
    }
}

// One byte matrix of ntt_mx.h: output k of 16 adjacent elements is
// scale * sum_d w^((d mod m)(k mod m)) x_d over the d in k's block of m = 2^t
// (t = 0: m = 16), w of order m, times 2^32.  Byte b of the constants is the
// signed digit of 256^b; the initial values of out_0 supply the part of the
// product that the bytes' offset of 128 leaves out.
void mx_matrix(int8_t *out, u32 w, int t, u32 scale, u32 p) {
    const int m = t ? 1 << t : 16;
    u32 *init = (u32 *)(out + 4 * 64 * 16);
    // the 16 digits, byte 4 b + a, of the entries at exponents (d mod m)(k mod m)
    u32 entry[226];
    int8_t digits[226][16];
    u32 e = cm_host_mul(scale, cm_host_r1(p), p);
    for (int x = 0; x <= (m - 1) * (m - 1); ++x, e = cm_host_mul(e, w, p)) {
        entry[x] = e;
        u32 y = e;
        for (int a = 0; a < 4; ++a, y = cm_host_mul(y, 256u, p)) {
            int64_t v = y > p / 2 ? (int64_t)y - p : (int64_t)y;
            for (int b = 0; b < 4; ++b) {
                const int8_t digit = (int8_t)(v & 255);
                v = (v - digit) / 256;
                digits[x][4 * b + a] = digit;
            }
        }
    }
    u32 sum[16];
    for (int k = 0; k < 16; ++k) {
        u64 acc = 0;
        for (int d = k / m * m; d < k / m * m + m; ++d) {
            const int x = (d % m) * (k % m);
            acc += entry[x];
            // lane (output k, group d / 4), bytes 4 (d mod 4) .. + 3; other blocks stay 0
            for (int b = 0; b < 4; ++b)
                memcpy(out + (b * 64 + (d / 4) * 16 + k) * 16 + 4 * (d % 4), digits[x] + 4 * b, 4);
        }
        sum[k] = (u32)(acc % p);
    }
    // out_0's initial value: the offset's share less the 2^32 kMxHigh that the
    // kernels add, a residue at or above kMxBias
    const u32 high = cm_host_mul(kMxHigh % p, cm_host_r1(p), p);
    for (int lane = 0; lane < 64; ++lane)
        for (int r = 0; r < 4; ++r) {
            const u32 sum_k = sum[4 * (lane >> 4) + r];
            const u32 c = cm_sub(cm_host_mul(0x80808080u % p, sum_k, p), high, p);
            init[lane * 4 + r] = c + (c < kMxBias ? (kMxBias - c + p - 1) / p * p : 0u);
        }
}

// matrices and twiddles of the matrix-core transforms; pw[dir]: the powers of the
// root of order 2^LT and of its inverse.  Every level's twiddles are among them.
bool make_mx(Family *f, const std::vector<u32> *pw) {
    const u32 p = f->p;
    std::vector<u32> mats((size_t)kMxMats * kMxMatWords * 4, 0u);
    auto mat = [&](int which) { return (int8_t *)(mats.data() + (size_t)which * kMxMatWords * 4); };
    for (int t = 0; t < 4; ++t) {
        const int lg = t ? t : 4;
        const u32 w = cm_host_pow(f->wN, (u64)1 << (f->K - lg), p), wi = cm_host_inv(w, p);
        const u32 sc = cm_host_inv((u32)(1 << lg) % p, p);
        mx_matrix(mat(kMxFwd + t), w, t, 1u, p);
        mx_matrix(mat(kMxInvFirst + t), wi, t, cm_host_mul(sc, cm_host_r1(p), p), p);
        mx_matrix(mat(kMxInv + t), wi, t, sc, p);
        if (t == 0)
            mx_matrix(mat(kMxInvPair), wi, 0,
                      cm_host_mul(cm_host_inv(32 % p, p), cm_host_r1(p), p), p);
    }
    f->mx_mat = upload(mats);
    for (int dir = 0; dir < 2; ++dir) {
        std::vector<u32> tab((size_t)2 << f->LT, 0u);
        for (int j = 5; j <= f->LT; ++j) {
            const size_t M = (size_t)1 << j, S = M / 16, step = (size_t)1 << (f->LT - j);
            for (size_t k = 0; k < 16; ++k)
                for (size_t v = 0; v < S; ++v) tab[M + k * S + v] = pw[dir][k * v * step];
        }
        (dir ? f->mx_ti : f->mx_tf) = upload(tab);
    }
    return f->mx_mat && f->mx_tf && f->mx_ti;
}

Family *make_family(u32 p, u32 wN, int K) {
    Family *f = new Family();
    f->p = p;
    f->pinv = cm_host_pinv(p);
    f->np = cm_host_npinv(p);
    f->K = K;
    f->wN = wN;
    f->LT = K < kMaxLevelLog ? K : kMaxLevelLog;
    // level tables: level M = 2^j (j = 1 .. LT) at offset 2^(j-1) - 1, each a part of
    // the largest level's powers
    std::vector<u32> pw[2];
    for (int dir = 0; dir < 2; ++dir) {
        const u32 w = cm_host_pow(wN, (u64)1 << (K - f->LT), p);   // order 2^LT
        pw[dir].resize((size_t)1 << f->LT);
        power_table(pw[dir].data(), dir ? cm_host_inv(w, p) : w, f->LT, p);
        std::vector<u32> lv;
        lv.reserve((size_t)1 << f->LT);
        for (int j = 1; j <= f->LT; ++j)
            for (size_t q = 0; q < (size_t)1 << (j - 1); ++q)
                lv.push_back(pw[dir][q << (f->LT - j)]);
        if (lv.empty()) lv.push_back(cm_host_mont(1, p));
        (dir ? f->lvi : f->lv) = upload(lv);
    }
    f->mx_mat = nullptr;
    f->mx_tf = f->mx_ti = nullptr;
    if (!f->lv || !f->lvi || (K >= 4 && !make_mx(f, pw))) {
        delete f;
        return nullptr;
    }
    return f;
}

}  // namespace

const Family *family_for_root(u32 p, u32 w, int k) {
    std::lock_guard<std::mutex> lk(g_plan_mutex);
    auto key = std::make_tuple(p, w, k);
    auto it = g_families.find(key);
    if (it != g_families.end()) return it->second;
    Family *f = make_family(p, w, k);
    if (f) g_families[key] = f;
    return f;
}

const Family *family_default(u32 p) {
    {
        std::lock_guard<std::mutex> lk(g_plan_mutex);
        auto it = g_default.find(p);
        if (it != g_default.end()) return it->second;
    }
    int K = cm_fourier_degree(p);
    if (K > 30) K = 30;
    u32 g = cm_host_generator(p);
    u32 wN = cm_host_pow(g, (u64)(p - 1) >> K, p);
    const Family *f = family_for_root(p, wN, K);
    if (f) {
        std::lock_guard<std::mutex> lk(g_plan_mutex);
        g_default[p] = f;
    }
    return f;
}

const Family *family_default_cached(u32 p) {
    std::lock_guard<std::mutex> lk(g_plan_mutex);
    auto it = g_default.find(p);
    return it != g_default.end() ? it->second : nullptr;
}

// The library's own columns: short enough that both passes fill the chip
// (measured over every split of 2^14 .. 2^24).
static int own_split(int k) {
    static const int k1[kMaxLog - kMaxLdsLog] = {6, 6, 6, 7, 8, 8, 8, 8, 10, 10, 11, 11, 12};
    return k - k1[k - kMaxLdsLog - 1];
}

// Row lengths that a caller may name: 2^12 to 2^14 with columns up to 2^13, and the
// library's own.
static bool named_split(int k, int k2) {
    if (k <= kMaxLdsLog || k > kMaxLog) return false;
    return k2 == own_split(k) || (k2 >= 12 && k2 <= 14 && k - k2 >= 1 && k - k2 <= kMaxLdsLog);
}

// 2^13 points (a few products of a tree level) have no choice.
void four_step_split(int k, int &k1, int &k2) {
    if (k <= kMaxLdsLog) {
        k1 = 5;
        k2 = k - k1;
        return;
    }
    k2 = g_split[k];
    if (!k2) {
        char name[32];
        snprintf(name, sizeof(name), "CUMODP_SPLIT_%d", k);
        const char *e = getenv(name);
        if (e) k2 = atoi(e);
    }
    if (!named_split(k, k2)) k2 = own_split(k);
    k1 = k - k2;
}

bool set_four_step_split(int k, int k2) {
    if (!named_split(k, k2)) return false;
    std::lock_guard<std::mutex> lk(g_plan_mutex);
    g_split[k] = k2;
    return true;
}

const Outer *outer_for(const Family *f, int k) {
    int k1, k2;
    four_step_split(k, k1, k2);
    return outer_for_split(f, k, k1, k2);
}

const Outer *outer_for_split(const Family *f, int k, int k1, int k2) {
    std::lock_guard<std::mutex> lk(g_plan_mutex);
    auto key = std::make_tuple(f, k, k2);
    auto it = g_outer.find(key);
    if (it != g_outer.end()) return it->second;
    if (k > f->K || k1 + k2 != k || k1 < 1 || k2 < 4) return nullptr;
    u32 p = f->p;
    u32 wn = cm_host_pow(f->wN, (u64)1 << (f->K - k), p);   // order 2^k
    u32 wni = cm_host_inv(wn, p);
    Outer *o = new Outer();
    o->k = k;
    o->k1 = k1;
    o->k2 = k2;
    // row-pass tables
    const size_t n1 = (size_t)1 << k1, T = ((size_t)1 << k2) / 16;
    for (int dir = 0; dir < 2; ++dir) {
        const u32 w = dir ? wni : wn, wT = cm_host_pow(w, T, p);
        std::vector<u32> rb(n1 * T), rc(n1 * 16);
        u32 wr = 1, wrT = 1;   // w^r, w^(r T)
        for (size_t r = 0; r < n1; ++r) {
            power_table(&rb[r * T], wr, k2 - 4, p);
            power_table(&rc[r * 16], wrT, 4, p);
            wr = cm_host_mul(wr, w, p);
            wrT = cm_host_mul(wrT, wT, p);
        }
        (dir ? o->rb_i : o->rb_f) = upload(rb);
        (dir ? o->rc_i : o->rc_f) = upload(rc);
    }
    if (!o->rb_f || !o->rc_f || !o->rb_i || !o->rc_i) {
        delete o;
        return nullptr;
    }
    g_outer[key] = o;
    return o;
}

const Outer *outer_cached(const Family *f, int k) {
    int k1, k2;
    four_step_split(k, k1, k2);
    std::lock_guard<std::mutex> lk(g_plan_mutex);
    auto it = g_outer.find(std::make_tuple(f, k, k2));
    return it != g_outer.end() ? it->second : nullptr;
}

namespace {
std::mutex g_ws_mutex;
std::map<std::pair<int, hipStream_t>, std::pair<void *, size_t>> g_ws;
// Scratch buffers that captured graphs refer to: buffer -> number of live
// graphs.  Such a buffer is never freed while a graph holds it; when its
// stream needs a larger one (or is destroyed) it is only detached
// (g_ws_detached) and freed when the last graph holding it is destroyed.
std::map<void *, int> g_ws_graph_refs;
std::map<void *, bool> g_ws_detached;

// drops buffer b from its (slot, stream) entry: freed at once unless a live
// graph refers to it (caller holds g_ws_mutex; work queued on the stream
// that may still use b has been synchronised)
void retire_buffer_locked(void *b) {
    if (!b) return;
    auto r = g_ws_graph_refs.find(b);
    if (r != g_ws_graph_refs.end() && r->second > 0) {
        g_ws_detached[b] = true;
        return;
    }
    (void)hipFree(b);
}
}  // namespace

bool stream_capturing(hipStream_t s) {
    if (!s) return false;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusActive;
}

void *workspace(int slot, size_t bytes, hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    auto &b = g_ws[std::make_pair(slot, s)];
    if (b.second >= bytes && b.first) return b.first;
    // a graph being captured cannot grow scratch (it would synchronise and
    // free memory the graph refers to): the same calls must run once eagerly
    // on this stream first
    if (stream_capturing(s)) return nullptr;
    if (b.first) {
        // work already queued on s may still use the old buffer
        (void)hipStreamSynchronize(s);
        retire_buffer_locked(b.first);
        b.first = nullptr;
        b.second = 0;
    }
    size_t sz = bytes < 4096 ? 4096 : bytes;
    void *d = nullptr;
    if (hipMalloc(&d, sz) != hipSuccess) return nullptr;
    b.first = d;
    b.second = sz;
    return d;
}

namespace {
// Pinned staging for descriptor uploads, one per stream; reused once the
// previous upload from it has finished.
struct Staging {
    void *host = nullptr;
    size_t cap = 0;
    hipEvent_t done = nullptr;
};
// A ring of staging buffers per stream: a buffer is rewritten only once the
// copy that last read it has run, so the host can queue several calls ahead
// of the device without waiting.
constexpr int kStagingRing = 8;
struct StagingRing {
    Staging b[kStagingRing];
    int next = 0;
};
std::map<hipStream_t, StagingRing> g_staging;   // guarded by g_ws_mutex
// pinned buffers whose copies were recorded into a graph being captured on a
// stream; they belong to that graph once the capture ends
std::map<hipStream_t, std::vector<void *>> g_captured;
}  // namespace

hipError_t stage_upload(const void *src, size_t bytes, void *dst, hipStream_t s) {
    return stage_upload_fill(bytes, dst, s, [&](char *h) { memcpy(h, src, bytes); });
}

hipError_t stage_upload_fill(size_t bytes, void *dst, hipStream_t s,
                             const std::function<void(char *)> &fill) {
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    hipError_t e;
    if (stream_capturing(s)) {
        // the recorded copy must keep reading these bytes at every replay
        void *h = nullptr;
        e = hipHostMalloc(&h, bytes ? bytes : 1);
        if (e != hipSuccess) return e;
        fill((char *)h);
        g_captured[s].push_back(h);
        return hipMemcpyAsync(dst, h, bytes, hipMemcpyHostToDevice, s);
    }
    // prefer a buffer that is already large enough and whose last copy has
    // run; else an unused slot; else wait for the oldest
    StagingRing &ring = g_staging[s];
    int pick = -1;
    for (int i = 0; i < kStagingRing && pick < 0; ++i) {
        const int j = (ring.next + i) % kStagingRing;
        Staging &b = ring.b[j];
        if (b.done && b.cap >= bytes && hipEventQuery(b.done) == hipSuccess) pick = j;
    }
    for (int i = 0; i < kStagingRing && pick < 0; ++i) {
        const int j = (ring.next + i) % kStagingRing;
        if (!ring.b[j].done) pick = j;
    }
    if (pick < 0) pick = ring.next;
    ring.next = (pick + 1) % kStagingRing;
    Staging &st = ring.b[pick];
    if (!st.done) {
        e = hipEventCreateWithFlags(&st.done, hipEventDisableTiming);
        if (e != hipSuccess) return e;
    } else {
        e = hipEventSynchronize(st.done);
        if (e != hipSuccess) return e;
    }
    if (st.cap < bytes) {
        if (st.host) (void)hipHostFree(st.host);
        st.host = nullptr;
        st.cap = 0;
        e = hipHostMalloc(&st.host, bytes);
        if (e != hipSuccess) return e;
        st.cap = bytes;
    }
    fill((char *)st.host);
    e = hipMemcpyAsync(dst, st.host, bytes, hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return e;
    return hipEventRecord(st.done, s);
}

namespace {
std::map<hipStream_t, AuxStreams *> g_aux;   // guarded by g_ws_mutex
}  // namespace

AuxStreams *aux_streams(hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    auto it = g_aux.find(s);
    if (it != g_aux.end()) return it->second;
    if (stream_capturing(s)) return nullptr;   // created eagerly, never inside a capture
    AuxStreams *a = new AuxStreams();
    bool ok = hipEventCreateWithFlags(&a->fork, hipEventDisableTiming) == hipSuccess;
    for (int i = 0; i < kAuxStreams && ok; ++i) {
        ok = hipStreamCreate(&a->s[i]) == hipSuccess &&
             hipEventCreateWithFlags(&a->join[i], hipEventDisableTiming) == hipSuccess;
    }
    if (!ok) return nullptr;   // leaks the partial set; the caller runs serially
    g_aux[s] = a;
    return a;
}

std::vector<void *> take_captured_buffers(hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    std::vector<void *> v;
    auto it = g_captured.find(s);
    if (it != g_captured.end()) {
        v.swap(it->second);
        g_captured.erase(it);
    }
    return v;
}

std::vector<void *> hold_workspace_for_graph(hipStream_t s) {
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    std::vector<hipStream_t> streams{s};
    auto a = g_aux.find(s);
    if (a != g_aux.end())
        for (int i = 0; i < kAuxStreams; ++i) streams.push_back(a->second->s[i]);
    std::vector<void *> held;
    for (auto &kv : g_ws) {
        if (!kv.second.first) continue;
        for (hipStream_t t : streams) {
            if (kv.first.second == t) {
                held.push_back(kv.second.first);
                ++g_ws_graph_refs[kv.second.first];
                break;
            }
        }
    }
    return held;
}

void release_graph_workspace(const std::vector<void *> &held) {
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    for (void *b : held) {
        auto r = g_ws_graph_refs.find(b);
        if (r == g_ws_graph_refs.end()) continue;
        if (--r->second > 0) continue;
        g_ws_graph_refs.erase(r);
        auto d = g_ws_detached.find(b);
        if (d != g_ws_detached.end()) {
            g_ws_detached.erase(d);
            (void)hipFree(b);
        }
    }
}

void release_workspace(hipStream_t s) {
    AuxStreams *a = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_ws_mutex);
        auto it = g_aux.find(s);
        if (it != g_aux.end()) {
            a = it->second;
            g_aux.erase(it);
        }
    }
    if (a) {
        for (int i = 0; i < kAuxStreams; ++i) {
            (void)hipStreamSynchronize(a->s[i]);
            release_workspace(a->s[i]);
            (void)hipStreamDestroy(a->s[i]);
            (void)hipEventDestroy(a->join[i]);
        }
        (void)hipEventDestroy(a->fork);
        delete a;
    }
    std::lock_guard<std::mutex> lk(g_ws_mutex);
    for (auto it = g_ws.begin(); it != g_ws.end();) {
        if (it->first.second == s) {
            retire_buffer_locked(it->second.first);
            it = g_ws.erase(it);
        } else {
            ++it;
        }
    }
    auto st = g_staging.find(s);
    if (st != g_staging.end()) {
        for (Staging &b : st->second.b) {
            if (b.done) (void)hipEventDestroy(b.done);
            if (b.host) (void)hipHostFree(b.host);
        }
        g_staging.erase(st);
    }
}

}  // namespace cm
