// C ABI of the GDN engine (declared in include/gdn_mi355x.h): argument checks, workspace layout, dispatch.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <mutex>
#include <algorithm>
#include <atomic>
#include <string>
#include <type_traits>
#include <vector>

#include "gdn_common.h"
#include "gdn_internal.h"
#include "../../include/gdn_mi355x.h"

namespace gdn {

static thread_local char g_err[512];

static int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof g_err, fmt, ap);
    va_end(ap);
    return code;
}

static bool debug_sync() {
    static const int on = [] {
        const char *s = getenv("GDN_DEBUG_SYNC");
        return s && s[0] == '1';
    }();
    return on != 0;
}

// After a launch: report launch errors, and in debug mode synchronise and report execution errors.
static int check_launch(hipStream_t st, const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(GDN_ERR_LAUNCH, "%s: launch failed: %s", what, hipGetErrorString(e));
    if (debug_sync()) {
        e = hipStreamSynchronize(st);
        if (e != hipSuccess) return fail(GDN_ERR_LAUNCH, "%s: execution failed: %s", what, hipGetErrorString(e));
    }
    return GDN_OK;
}

// Opt-in launch timing (gdn_profile_enable): each launch is bracketed by two HIP events recorded on the
// launch's own stream.  Off by default; the normal path records nothing.
struct ProfRec {
    const char *name;
    hipEvent_t start, stop;
};
static std::mutex g_prof_mu;
static std::vector<ProfRec> g_prof;
static std::atomic<bool> g_prof_on{false};  // read by every launch without the lock

struct Timed {
    const char *name;
    hipStream_t st;
    hipEvent_t start = nullptr, stop = nullptr;
    Timed(const char *n, hipStream_t s) : name(n), st(s) {
        if (!g_prof_on.load(std::memory_order_relaxed)) return;
        if (hipEventCreate(&start) != hipSuccess || hipEventCreate(&stop) != hipSuccess) {
            start = stop = nullptr;
            return;
        }
        (void)hipEventRecord(start, st);
    }
    ~Timed() {
        if (!start) return;
        (void)hipEventRecord(stop, st);
        std::lock_guard<std::mutex> lk(g_prof_mu);
        g_prof.push_back({name, start, stop});
    }
};

__global__ void copy_or_zero_kernel(float *dst, const float *src, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src ? src[i] : 0.f;
}

void launch_copy_or_zero(float *dst, const float *src, size_t n, hipStream_t st) {
    if (dst && n) hipLaunchKernelGGL(copy_or_zero_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                                     dst, src, n);
}

static bool dtype_ok(int dt) { return dt == DT_F32 || dt == DT_BF16 || dt == DT_F16; }

static int check_shape(int B, int T, int Hk, int Hv, int Dk, int Dv, int chunk, int gate, int form) {
    if (chunk <= 0) return fail(GDN_ERR_INVALID, "chunk must be a positive integer");
    if (B < 0 || T < 0) return fail(GDN_ERR_INVALID, "batch and timesteps must be non-negative");
    if (Hk <= 0 || Hv <= 0 || Dk <= 0 || Dv <= 0)
        return fail(GDN_ERR_INVALID, "head counts and head dims must be positive");
    if (Hv % Hk != 0) return fail(GDN_ERR_INVALID, "q/k head count must divide the value head count");
    if (gate != GATE_DECAY && gate != GATE_DECAY_VEC && gate != GATE_LOG && gate != GATE_LOG_VEC)
        return fail(GDN_ERR_INVALID, "Unsupported gating kind %d", gate);
    if (form != GDN_FORM_AUTO && form != GDN_FORM_RECURRENT && form != GDN_FORM_CHUNK)
        return fail(GDN_ERR_INVALID, "unknown form %d", form);
    if (pick_lane_width(Dk) == 0) return fail(GDN_ERR_UNSUPPORTED, "key_dim %d > 256 is not supported", Dk);
    if (Hv > 65535 || B > 65535) return fail(GDN_ERR_UNSUPPORTED, "batch and value heads must be <= 65535");
    return GDN_OK;
}

// Masked calls run on the chunked form (gdn_mask.hip) up to mask_max_heads() value heads.  Per-channel gates run on the
// chunked form with bf16 inputs and no mask (gdn_chunk_vg.hip).
static bool chunk_eligible(int Hv, int Dk, int Dv, int has_mask, int gate, int in_dt) {
    if (Dk != 128 || Dv != 128) return false;
    if (gate_vec(gate)) return !has_mask && chunk_vg_supported(in_dt);
    return !has_mask || Hv <= mask_max_heads();
}

// The form a (shape, mask, gate, requested form, input dtype) resolves to, or < 0 when a requested form cannot run.
static int resolve_form(int Hv, int Dk, int Dv, int has_mask, int gate, int form, int in_dt) {
    if (form == GDN_FORM_RECURRENT) return GDN_FORM_RECURRENT;
    const bool ok = chunk_eligible(Hv, Dk, Dv, has_mask, gate, in_dt);
    if (form == GDN_FORM_CHUNK) {
        if (ok) return GDN_FORM_CHUNK;
        if (Dk != 128 || Dv != 128) return fail(GDN_ERR_UNSUPPORTED, "the chunked form needs Dk = Dv = 128");
        if (gate_vec(gate))
            return fail(GDN_ERR_UNSUPPORTED, "the chunked form takes per-channel gates with bf16 inputs and no mask");
        return fail(GDN_ERR_UNSUPPORTED, "masked calls of the chunked form take Hv <= %d", mask_max_heads());
    }
    return ok ? GDN_FORM_CHUNK : GDN_FORM_RECURRENT;
}

static bool misaligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) != 0; }

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct BwdLayout {
    size_t sub, part_qk, part_gb, part_gv, total;
};

static BwdLayout bwd_layout(int B, int T, int Hv, int Dk, int Dv, int chunk, int gate) {
    const size_t nrb = (size_t)rec_bwd_row_blocks(B, Hv, Dk, Dv, gate);
    const size_t toks = (size_t)B * T * Hv;
    BwdLayout L;
    size_t off = 0;
    L.sub = off;
    off += align256(rec_sub_floats(B, Hv, Dk, Dv, T, chunk, gate) * sizeof(float));
    L.part_qk = off;
    off += align256(nrb * toks * 2 * Dk * sizeof(float));
    L.part_gb = off;
    off += align256(nrb * toks * 2 * sizeof(float));
    L.part_gv = off;
    if (gate_vec(gate)) off += align256(nrb * toks * Dk * sizeof(float));
    L.total = off;
    return L;
}

static size_t rec_saved_bytes(int B, int T, int Hv, int Dk, int Dv, int chunk) {
    const int64_t ns = T > 0 ? (int64_t)((T + chunk - 1) / chunk) - 1 : 0;
    return (size_t)(ns > 0 ? ns : 0) * B * Hv * Dv * Dk * sizeof(float);
}

// ---- chunked form: how a call is split
//
// chunk <= 64 keeps the whole tile set from forward to backward ("saved").  chunk > 64 checkpoints: the forward keeps
// only the states at every window of W = chunk rounded up to 64 tokens (ceil(T / W) - 1 fp32 snapshots, like the
// recurrent form's boundaries), and the backward rebuilds one group of windows at a time (prep, then the forward of
// every window of the group side by side from its snapshot) before running the backward stages over that group.
// A forward-only call (no saved buffer) runs group by group as well.  Groups live in the caller's workspace: the
// largest whole number of units (windows, or 64-token chunks when forward-only) that fits, capped at about
// kGroupChunkHeads chunk-heads.

constexpr int kGroupChunkHeads = 2048;

static int ck_window(int chunk) { return chunk <= kChunkC ? 0 : (chunk + kChunkC - 1) / kChunkC * kChunkC; }

static size_t ck_state_bytes(int B, int Hv) { return (size_t)B * Hv * kChunkD * kChunkD * sizeof(float); }

static size_t ck_snap_bytes(int B, int T, int Hv, int W) {
    const int nwin = (T + W - 1) / W;
    return nwin > 1 ? (size_t)(nwin - 1) * ck_state_bytes(B, Hv) : 0;
}

struct CkShape {
    int B, T, Hk, Hv;
    bool bf16;
    int vg;  // vg_kind of the gate: 0 one decay per head, 1 per-channel log decays, 2 per-channel decays
    bool masked;
};

static ChunkSizes ck_sizes(const CkShape &s, int T, bool bwd) {
    return chunk_sizes(s.B, T, s.Hk, s.Hv, s.bf16, bwd, s.vg, s.masked);
}

// Forward group workspace: the forward tile set of Tg tokens, plus two carried states between groups when no
// snapshots carry them.
static size_t ck_fwd_group_bytes(const CkShape &s, int Tg, bool ckpt) {
    return ck_sizes(s, Tg, false).saved + (ckpt ? 0 : 2 * align256(ck_state_bytes(s.B, s.Hv)));
}

// Backward group workspace: two carried state adjoints, the whole tile set and the backward buffers of Tg tokens.
static size_t ck_bwd_group_bytes(const CkShape &s, int Tg) {
    const ChunkSizes cs = ck_sizes(s, Tg, true);
    return 2 * align256(ck_state_bytes(s.B, s.Hv)) + align256(cs.saved) + cs.work;
}

// Units of u tokens per group: the target count, or fewer when the workspace is smaller; 0 when one unit does not fit.
template <class Bytes>
static int ck_group_units(const CkShape &s, int u, size_t avail, Bytes bytes) {
    const int total = (s.T + u - 1) / u;
    const size_t per_unit = (size_t)s.B * s.Hv * (u / kChunkC);
    int g = (int)std::max<size_t>(1, kGroupChunkHeads / per_unit);
    g = std::min(g, total);
    for (; g >= 1; --g)
        if (bytes(std::min(g * u, s.T)) <= avail) return g;
    return 0;
}

static size_t ck_fwd_target_bytes(const CkShape &s, int W, bool ckpt) {
    const int u = ckpt ? W : kChunkC;
    const int g = ck_group_units(s, u, SIZE_MAX, [](int) { return (size_t)0; });
    return ck_fwd_group_bytes(s, std::min(g * u, s.T), ckpt);
}

static size_t ck_bwd_target_bytes(const CkShape &s, int W) {
    const int g = ck_group_units(s, W, SIZE_MAX, [](int) { return (size_t)0; });
    return ck_bwd_group_bytes(s, std::min(g * W, s.T));
}

// ---- masked calls on the chunked form (gdn_mask.hip): what mask_query_kernel writes and the chunked kernels read, the
// effective gates g', beta', the masked tokens' queries (fp32, or bf16 hi and lo planes) and value factors, and the chunk
// flags.  A training call keeps them behind the tiles or snapshots, a forward-only call at the head of its workspace.
struct MaskBufs {
    size_t g2, b2, e, qm, cm, total;
};
static MaskBufs mask_bufs(const CkShape &s) {
    const size_t ng = (size_t)s.B * s.T * s.Hv * 4;
    MaskBufs m{};
    size_t off = 0;
    m.g2 = off; off += align256(ng);
    m.b2 = off; off += align256(ng);
    m.e = off; off += align256(ng);
    m.qm = off; off += align256(ng * kChunkD);
    m.cm = off; off += align256((size_t)s.B * ((s.T + kChunkC - 1) / kChunkC));
    m.total = off;
    return m;
}
static size_t mask_tiles_bytes(const CkShape &s, int chunk) {
    const int W = ck_window(chunk);
    return align256(W ? ck_snap_bytes(s.B, s.T, s.Hv, W) : ck_sizes(s, s.T, true).saved);
}
// Backward workspace of the chunked stages; a masked call puts dL/dq~ (fp32 [B][T][Hv][Dk]) behind it.
static size_t mask_stage_bytes(const CkShape &s, int chunk) {
    const int W = ck_window(chunk);
    return align256(W ? ck_bwd_target_bytes(s, W) : ck_sizes(s, s.T, true).work);
}
static size_t mask_work_bytes(const CkShape &s, int chunk) {
    return mask_stage_bytes(s, chunk) + align256((size_t)s.B * s.T * s.Hv * kChunkD * 4);
}

static size_t dt_size(int dt) { return dt == DT_F32 ? 4 : 2; }

// Gate values per (token, value head): one, or one per key channel.
static size_t gate_width(int gate) { return gate_vec(gate) ? kChunkD : 1; }

template <class P>
static P *tok_offset(P *p, size_t elems, int dt) {
    if (!p) return p;
    using C = typename std::conditional<std::is_const<P>::value, const char, char>::type;
    return reinterpret_cast<P *>(reinterpret_cast<C *>(p) + elems * dt_size(dt));
}

}  // namespace gdn

using namespace gdn;

extern "C" {

int gdn_version(void) { return (3 << 16) | 0; }

int gdn_profile_enable(int on) {
    g_prof_on.store(on != 0, std::memory_order_relaxed);
    return GDN_OK;
}

int gdn_profile_collect(int max_entries, char *names, int name_len, double *total_ms, int *counts) {
    std::vector<ProfRec> recs;
    {
        std::lock_guard<std::mutex> lk(g_prof_mu);
        recs.swap(g_prof);
    }
    std::map<std::string, std::pair<double, int>> agg;
    int rc = GDN_OK;
    for (auto &r : recs) {
        float ms = 0.f;
        if (hipEventSynchronize(r.stop) == hipSuccess && hipEventElapsedTime(&ms, r.start, r.stop) == hipSuccess) {
            auto &e = agg[r.name];
            e.first += ms;
            e.second += 1;
        } else {
            rc = fail(GDN_ERR_LAUNCH, "profiling event failed");
        }
        (void)hipEventDestroy(r.start);
        (void)hipEventDestroy(r.stop);
    }
    if (rc) return rc;
    int n = 0;
    for (auto &kv : agg) {
        if (n >= max_entries) break;
        snprintf(names + (size_t)n * name_len, name_len, "%s", kv.first.c_str());
        total_ms[n] = kv.second.first;
        counts[n] = kv.second.second;
        ++n;
    }
    return n;
}

const char *gdn_last_error(void) { return g_err; }

int64_t gdn_num_snapshots(int T, int chunk) {
    if (chunk <= 0 || T <= 0) return 0;
    return (int64_t)((T + chunk - 1) / chunk) - 1;
}

int gdn_select_form(int Hv, int Dk, int Dv, int has_mask, int gate_kind, int form, int in_dtype) {
    g_err[0] = 0;
    if (gate_kind != GATE_DECAY && gate_kind != GATE_DECAY_VEC && gate_kind != GATE_LOG && gate_kind != GATE_LOG_VEC)
        return fail(GDN_ERR_INVALID, "Unsupported gating kind %d", gate_kind);
    if (form != GDN_FORM_AUTO && form != GDN_FORM_RECURRENT && form != GDN_FORM_CHUNK)
        return fail(GDN_ERR_INVALID, "unknown form %d", form);
    return resolve_form(Hv, Dk, Dv, has_mask, gate_kind, form, in_dtype);
}

size_t gdn_saved_bytes(int B, int T, int Hk, int Hv, int Dk, int Dv, int chunk, int gate_kind, int has_mask,
                       int form, int in_dtype) {
    if (check_shape(B, T, Hk, Hv, Dk, Dv, chunk, gate_kind, form)) return 0;
    const int f = resolve_form(Hv, Dk, Dv, has_mask, gate_kind, form, in_dtype);
    if (f < 0 || B == 0 || T == 0) return 0;
    if (f == GDN_FORM_CHUNK) {
        const int W = ck_window(chunk);
        const CkShape shp{B, T, Hk, Hv, in_dtype == DT_BF16, vg_kind(gate_kind), has_mask != 0};
        if (has_mask) return mask_tiles_bytes(shp, chunk) + mask_bufs(shp).total;
        if (W) return ck_snap_bytes(B, T, Hv, W);
        return ck_sizes(shp, T, true).saved;
    }
    return rec_saved_bytes(B, T, Hv, Dk, Dv, chunk);
}

size_t gdn_fwd_workspace_bytes(int B, int T, int Hk, int Hv, int Dk, int Dv, int chunk, int gate_kind, int has_mask,
                               int form, int in_dtype, int with_saved) {
    if (check_shape(B, T, Hk, Hv, Dk, Dv, chunk, gate_kind, form)) return 0;
    const int f = resolve_form(Hv, Dk, Dv, has_mask, gate_kind, form, in_dtype);
    if (f != GDN_FORM_CHUNK || B == 0 || T == 0) return 0;
    const int W = ck_window(chunk);
    const CkShape shp{B, T, Hk, Hv, in_dtype == DT_BF16, vg_kind(gate_kind), has_mask != 0};
    if (with_saved && !W) return 0;
    return ck_fwd_target_bytes(shp, W, with_saved != 0) + (has_mask && !with_saved ? mask_bufs(shp).total : 0);
}

}  // extern "C"

namespace gdn {

// A masked call's pointers moved to token ts (a multiple of the chunk).
static void offset_mask(ChunkCall &cc, int ts) {
    if (!cc.mask) return;
    const size_t th = (size_t)ts * cc.Hv;
    cc.mask += ts;
    cc.cm += ts / kChunkC;
    cc.qm = tok_offset(cc.qm, th * kChunkD, cc.in_dt == DT_BF16 ? DT_BF16 : DT_F32);
    cc.e += th;
    if (cc.xm) cc.xm += th * kChunkD;
}

// Chunked forward (resolved form GDN_FORM_CHUNK, arguments checked).
static int ck_forward(const ChunkCall &base, int chunk, void *saved, size_t saved_bytes, void *ws, size_t ws_bytes,
                      hipStream_t st) {
    const int B = base.B, T = base.T, Hk = base.Hk, Hv = base.Hv;
    const CkShape shp{B, T, Hk, Hv, base.in_dt == DT_BF16, vg_kind(base.gate), base.mask != nullptr};
    const int W = ck_window(chunk);
    int rc;
    if (saved && !W) {  // the whole tile set, kept for the backward
        const size_t need = ck_sizes(shp, T, true).saved;
        if (saved_bytes < need)
            return fail(GDN_ERR_WORKSPACE, "saved buffer of %zu bytes is smaller than the %zu bytes required",
                        saved_bytes, need);
        ChunkCall cc = base;
        cc.tiles = saved;
        cc.Ts = T;
        {
            Timed tm("ck_prep", st);
            launch_chunk_stage(cc, "prep", st);
        }
        if ((rc = check_launch(st, "gdn_fwd(ck_prep)"))) return rc;
        {
            Timed tm("ck_fwd", st);
            launch_chunk_stage(cc, "fwd", st);
        }
        return check_launch(st, "gdn_fwd(ck_fwd)");
    }
    const bool ckpt = saved != nullptr;
    float *snap = static_cast<float *>(saved);
    if (ckpt && saved_bytes < ck_snap_bytes(B, T, Hv, W))
        return fail(GDN_ERR_WORKSPACE, "saved buffer of %zu bytes is smaller than the %zu bytes of snapshots",
                    saved_bytes, ck_snap_bytes(B, T, Hv, W));
    const int u = ckpt ? W : kChunkC;
    const int units = ck_group_units(shp, u, ws ? ws_bytes : 0,
                                     [&](int Tg) { return ck_fwd_group_bytes(shp, Tg, ckpt); });
    if (units == 0)
        return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes of one %d-token group",
                    ws ? ws_bytes : 0, ck_fwd_group_bytes(shp, std::min(u, T), ckpt), u);
    const int Gt = units * u;
    const size_t sb = align256(ck_state_bytes(B, Hv)), S = (size_t)B * Hv * kChunkD * kChunkD;
    char *w8 = static_cast<char *>(ws);
    float *carry[2] = {nullptr, nullptr};
    if (!ckpt) {
        carry[0] = reinterpret_cast<float *>(w8);
        carry[1] = reinterpret_cast<float *>(w8 + sb);
        w8 += 2 * sb;
    }
    for (int g = 0, ts = 0; ts < T; ++g, ts += Gt) {
        const int Tg = std::min(Gt, T - ts);
        const bool last = ts + Tg >= T;
        ChunkCall cc = base;
        cc.q = tok_offset(base.q, (size_t)ts * Hk * kChunkD, base.in_dt);
        cc.k = tok_offset(base.k, (size_t)ts * Hk * kChunkD, base.in_dt);
        cc.v = tok_offset(base.v, (size_t)ts * Hv * kChunkD, base.in_dt);
        cc.g = base.g + (size_t)ts * Hv * gate_width(base.gate);
        cc.beta = base.beta + (size_t)ts * Hv;
        cc.y = tok_offset(base.y, (size_t)ts * Hv * kChunkD, base.out_dt);
        offset_mask(cc, ts);
        cc.T = Tg;
        cc.Ts = T;
        cc.tiles = w8;
        cc.fwd_only = 1;
        if (ckpt) {
            const int win0 = ts / W;
            cc.snap = snap;
            cc.wc = W / kChunkC;
            cc.win0 = win0;
            cc.state0 = g == 0 ? base.state0 : snap + (size_t)(win0 - 1) * S;
            cc.state_T = last ? base.state_T : snap + (size_t)(win0 + Gt / W - 1) * S;
        } else {
            cc.state0 = g == 0 ? base.state0 : carry[g & 1];
            cc.state_T = last ? base.state_T : carry[(g + 1) & 1];
        }
        {
            Timed tm("ck_prep", st);
            launch_chunk_stage(cc, "prep", st);
        }
        if ((rc = check_launch(st, "gdn_fwd(ck_prep)"))) return rc;
        {
            Timed tm("ck_fwd", st);
            launch_chunk_stage(cc, "fwd", st);
        }
        if ((rc = check_launch(st, "gdn_fwd(ck_fwd)"))) return rc;
    }
    return GDN_OK;
}

// Chunked backward (resolved form GDN_FORM_CHUNK, arguments checked).
static int ck_backward(const ChunkCall &base, int chunk, const void *saved, size_t saved_bytes, void *ws,
                       size_t ws_bytes, hipStream_t st) {
    const int B = base.B, T = base.T, Hk = base.Hk, Hv = base.Hv;
    const CkShape shp{B, T, Hk, Hv, base.in_dt == DT_BF16, vg_kind(base.gate), base.mask != nullptr};
    const int W = ck_window(chunk);
    int rc;
    if (!W) {
        const ChunkSizes cs = ck_sizes(shp, T, true);
        if (!saved || saved_bytes < cs.saved)
            return fail(GDN_ERR_INVALID, "the saved buffer written by gdn_fwd (%zu bytes) is required", cs.saved);
        if (!ws || ws_bytes < cs.work)
            return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes required", ws_bytes,
                        cs.work);
        ChunkCall cc = base;
        cc.tiles = const_cast<void *>(saved);
        cc.work = ws;
        cc.Ts = T;
        {
            Timed tm("ck_bwd_seq", st);
            launch_chunk_stage(cc, "seq", st);
        }
        if ((rc = check_launch(st, "gdn_bwd(ck_bwd_seq)"))) return rc;
        {
            Timed tm("ck_bwd_local", st);
            launch_chunk_stage(cc, "local", st);
        }
        if ((rc = check_launch(st, "gdn_bwd(ck_bwd_local)"))) return rc;
        if (shp.vg == 2) {
            Timed tm("ck_vg_dg", st);
            launch_chunk_stage(cc, "dg", st);
        }
        return check_launch(st, "gdn_bwd(ck_vg_dg)");
    }
    const size_t need_snap = ck_snap_bytes(B, T, Hv, W);
    if (need_snap && (!saved || saved_bytes < need_snap))
        return fail(GDN_ERR_INVALID, "the snapshots written by gdn_fwd (%zu bytes) are required", need_snap);
    const int units = ck_group_units(shp, W, ws ? ws_bytes : 0, [&](int Tg) { return ck_bwd_group_bytes(shp, Tg); });
    if (units == 0)
        return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes of one %d-token group",
                    ws ? ws_bytes : 0, ck_bwd_group_bytes(shp, std::min(W, T)), W);
    const int Gt = units * W, ng = (T + Gt - 1) / Gt;
    const size_t sb = align256(ck_state_bytes(B, Hv));
    char *w8 = static_cast<char *>(ws);
    float *carry[2] = {reinterpret_cast<float *>(w8), reinterpret_cast<float *>(w8 + sb)};
    const ChunkSizes full = ck_sizes(shp, std::min(Gt, T), true);
    char *tiles = w8 + 2 * sb, *work = tiles + align256(full.saved);
    for (int g = ng - 1; g >= 0; --g) {
        const int ts = g * Gt, Tg = std::min(Gt, T - ts);
        const size_t qk = (size_t)ts * Hk * kChunkD, vv = (size_t)ts * Hv * kChunkD;
        ChunkCall cc = base;
        cc.q = tok_offset(base.q, qk, base.in_dt);
        cc.k = tok_offset(base.k, qk, base.in_dt);
        cc.v = tok_offset(base.v, vv, base.in_dt);
        cc.g = base.g + (size_t)ts * Hv * gate_width(base.gate);
        cc.beta = base.beta + (size_t)ts * Hv;
        cc.dy = tok_offset(base.dy, vv, base.dy_dt);
        cc.dq = tok_offset(base.dq, qk, base.grad_dt);
        cc.dk = tok_offset(base.dk, qk, base.grad_dt);
        cc.dv = tok_offset(base.dv, vv, base.grad_dt);
        cc.dg = base.dg + (size_t)ts * Hv * gate_width(base.gate);
        cc.dbeta = base.dbeta + (size_t)ts * Hv;
        offset_mask(cc, ts);
        cc.T = Tg;
        cc.Ts = T;
        cc.tiles = tiles;
        cc.work = work;
        {
            Timed tm("ck_prep", st);
            launch_chunk_stage(cc, "prep", st);
        }
        if ((rc = check_launch(st, "gdn_bwd(ck_prep)"))) return rc;
        {
            ChunkCall rf = cc;  // every window of the group from its entry state: H and Delta only
            rf.recompute = 1;
            rf.snap = static_cast<float *>(const_cast<void *>(saved));
            rf.wc = W / kChunkC;
            rf.win0 = ts / W;
            rf.state0 = base.state0;
            rf.y = nullptr;
            rf.state_T = nullptr;
            Timed tm("ck_fwd_recompute", st);
            launch_chunk_stage(rf, "fwd", st);
        }
        if ((rc = check_launch(st, "gdn_bwd(ck_fwd recompute)"))) return rc;
        cc.dstate_T = g == ng - 1 ? base.dstate_T : carry[(g + 1) & 1];
        cc.dstate0 = g == 0 ? base.dstate0 : carry[g & 1];
        {
            Timed tm("ck_bwd_seq", st);
            launch_chunk_stage(cc, "seq", st);
        }
        if ((rc = check_launch(st, "gdn_bwd(ck_bwd_seq)"))) return rc;
        {
            Timed tm("ck_bwd_local", st);
            launch_chunk_stage(cc, "local", st);
        }
        if ((rc = check_launch(st, "gdn_bwd(ck_bwd_local)"))) return rc;
        if (shp.vg == 2) {
            Timed tm("ck_vg_dg", st);
            launch_chunk_stage(cc, "dg", st);
            if ((rc = check_launch(st, "gdn_bwd(ck_vg_dg)"))) return rc;
        }
    }
    return GDN_OK;
}

static char *at_off(void *base, size_t off) { return static_cast<char *>(base) + off; }

static MaskArgs mask_args(const ChunkCall &base, const uint8_t *mask) {
    MaskArgs ma{};
    ma.q = base.q; ma.k = base.k; ma.v = base.v; ma.dy = base.dy; ma.g = base.g; ma.beta = base.beta; ma.mask = mask;
    ma.dq = base.dq; ma.dk = base.dk; ma.dv = base.dv; ma.dg = base.dg; ma.dbeta = base.dbeta;
    ma.B = base.B; ma.T = base.T; ma.Hk = base.Hk; ma.Hv = base.Hv; ma.Dk = kChunkD; ma.Dv = kChunkD;
    ma.in_dt = base.in_dt; ma.dy_dt = base.dy_dt; ma.grad_dt = base.grad_dt; ma.gate = base.gate;
    return ma;
}

// The chunked call over the effective gates and the masked tokens' queries in bufs (mask_bufs).
static ChunkCall masked_call(const ChunkCall &base, const uint8_t *mask, const MaskBufs &m, void *bufs) {
    ChunkCall c = base;
    c.g = reinterpret_cast<const float *>(at_off(bufs, m.g2));
    c.beta = reinterpret_cast<const float *>(at_off(bufs, m.b2));
    c.mask = mask;
    c.e = reinterpret_cast<const float *>(at_off(bufs, m.e));
    c.qm = at_off(bufs, m.qm);
    c.qm_lo = (size_t)base.B * base.T * base.Hv * kChunkD;
    c.cm = reinterpret_cast<const uint8_t *>(at_off(bufs, m.cm));
    c.cm_stride = (base.T + kChunkC - 1) / kChunkC;
    return c;
}

// Masked chunked forward (resolved form GDN_FORM_CHUNK, arguments checked).  base holds the caller's q, k, v, g,
// beta, state0, y, state_T and shapes.
static int ck_masked_forward(const ChunkCall &base, const uint8_t *mask, int chunk, void *saved, size_t saved_bytes,
                             void *ws, size_t ws_bytes, hipStream_t st) {
    const CkShape shp{base.B, base.T, base.Hk, base.Hv, base.in_dt == DT_BF16, vg_kind(base.gate), true};
    const MaskBufs m = mask_bufs(shp);
    size_t tiles_bytes = 0;
    void *bufs = ws;
    if (saved) {
        tiles_bytes = mask_tiles_bytes(shp, chunk);
        if (saved_bytes < tiles_bytes + m.total)
            return fail(GDN_ERR_WORKSPACE, "saved buffer of %zu bytes is smaller than the %zu bytes required",
                        saved_bytes, tiles_bytes + m.total);
        bufs = at_off(saved, tiles_bytes);
    } else {
        if (!ws || ws_bytes < m.total)
            return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes a masked call needs",
                        ws ? ws_bytes : 0, m.total);
        ws = at_off(ws, m.total);
        ws_bytes -= m.total;
    }
    const ChunkCall c = masked_call(base, mask, m, bufs);
    MaskArgs ma = mask_args(base, mask);
    ma.g2 = const_cast<float *>(c.g);
    ma.beta2 = const_cast<float *>(c.beta);
    ma.e = const_cast<float *>(c.e);
    ma.qm = const_cast<void *>(c.qm);
    ma.qm_lo = c.qm_lo;
    ma.cm = const_cast<uint8_t *>(c.cm);
    {
        Timed tm("mask_query", st);
        launch_mask_query(ma, st);
    }
    const int rc = check_launch(st, "gdn_fwd(mask queries)");
    if (rc) return rc;
    return ck_forward(c, chunk, saved, tiles_bytes, ws, ws ? ws_bytes : 0, st);
}

// Masked chunked backward (resolved form GDN_FORM_CHUNK, arguments checked).
static int ck_masked_backward(const ChunkCall &base, const uint8_t *mask, int chunk, const void *saved,
                              size_t saved_bytes, void *ws, size_t ws_bytes, hipStream_t st) {
    const CkShape shp{base.B, base.T, base.Hk, base.Hv, base.in_dt == DT_BF16, vg_kind(base.gate), true};
    const MaskBufs m = mask_bufs(shp);
    const size_t tiles_bytes = mask_tiles_bytes(shp, chunk);
    if (!saved || saved_bytes < tiles_bytes + m.total)
        return fail(GDN_ERR_INVALID, "the saved buffer written by gdn_fwd (%zu bytes) is required", tiles_bytes + m.total);
    const size_t stage_bytes = mask_stage_bytes(shp, chunk), need = mask_work_bytes(shp, chunk);
    if (!ws || ws_bytes < need)
        return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes required", ws_bytes, need);
    ChunkCall c = masked_call(base, mask, m, at_off(const_cast<void *>(saved), tiles_bytes));
    c.xm = reinterpret_cast<float *>(at_off(ws, stage_bytes));
    int rc = ck_backward(c, chunk, saved, tiles_bytes, ws, stage_bytes, st);
    if (rc) return rc;
    MaskArgs ma = mask_args(base, mask);
    ma.xm = c.xm;
    {
        Timed tm("mask_bwd_fix", st);
        launch_mask_bwd_fix(ma, st);
    }
    return check_launch(st, "gdn_bwd(masked tokens)");
}

// Fixed device scratch of gdn_fwd_noalloc: a file-scope device array, one copy per GPU, held until the process
// ends.  Host code never passes the array's name to a kernel (that is a host-side stand-in); it uses the address
// hipGetSymbolAddress returns for the current device.
constexpr size_t kNoAllocScratchBytes = 64u << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices];  // device ordinal -> that device's copy of `scratch` (NULL: not looked up)

// The current device's scratch address, looked up once per device with that device current; NULL (with the
// error set) on failure.
static void *device_scratch() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) {
        fail(GDN_ERR_LAUNCH, "gdn_fwd_noalloc: no current HIP device");
        return nullptr;
    }
    if (dev >= kMaxDevices) {
        fail(GDN_ERR_UNSUPPORTED, "gdn_fwd_noalloc: device ordinal %d >= %d", dev, kMaxDevices);
        return nullptr;
    }
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev]) return g_scratch_ptr[dev];
    void *ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        fail(GDN_ERR_LAUNCH, "gdn_fwd_noalloc: hipGetSymbolAddress of the scratch failed: %s", hipGetErrorString(e));
        return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
    return ptr;
}

}  // namespace gdn

extern "C" {

int gdn_fwd_noalloc(const void *q, const void *k, const void *v, const float *g, const float *beta,
                    const float *state0, const uint8_t *mask, void *y, float *state_T, int B, int T, int Hk, int Hv,
                    int Dk, int Dv, int in_dtype, int out_dtype, int gate_kind, int form, void *stream) {
    g_err[0] = 0;
    int rc = check_shape(B, T, Hk, Hv, Dk, Dv, kChunkC, gate_kind, form);
    if (rc) return rc;
    if (!dtype_ok(in_dtype) || !dtype_ok(out_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    // masked calls keep the recurrent form here: the chunked form's masked queries need buffers that grow with T
    if (mask && form == GDN_FORM_CHUNK)
        return fail(GDN_ERR_UNSUPPORTED, "gdn_fwd_noalloc runs masked calls in the recurrent form only");
    if (mask) form = GDN_FORM_RECURRENT;
    const int f = resolve_form(Hv, Dk, Dv, mask != nullptr, gate_kind, form, in_dtype);
    if (f < 0) return f;
    void *ws = nullptr;
    size_t ws_bytes = 0;
    if (f == GDN_FORM_CHUNK && B > 0 && T > 0) {
        const CkShape shp{B, T, Hk, Hv, in_dtype == DT_BF16, vg_kind(gate_kind), false};
        const size_t one = ck_fwd_group_bytes(shp, std::min(kChunkC, T), false);
        if (one > kNoAllocScratchBytes)
            return fail(GDN_ERR_UNSUPPORTED,
                        "gdn_fwd_noalloc: one 64-token group of %d x %d heads needs %zu bytes; the fixed scratch "
                        "holds %zu (use gdn_fwd with a workspace)", B, Hv, one, kNoAllocScratchBytes);
        ws = device_scratch();
        if (!ws) return GDN_ERR_LAUNCH;
        ws_bytes = kNoAllocScratchBytes;
    }
    // the forward-only call of gdn_fwd, with the fixed scratch as its workspace
    return gdn_fwd(q, k, v, g, beta, state0, mask, y, state_T, nullptr, 0, ws, ws_bytes, B, T, Hk, Hv, Dk, Dv,
                   kChunkC, in_dtype, out_dtype, gate_kind, form, stream);
}

int gdn_fwd(const void *q, const void *k, const void *v, const float *g, const float *beta,
            const float *state0, const uint8_t *mask, void *y, float *state_T, void *saved, size_t saved_bytes,
            void *workspace, size_t workspace_bytes, int B, int T, int Hk, int Hv, int Dk, int Dv, int chunk,
            int in_dtype, int out_dtype, int gate_kind, int form, void *stream) {
    g_err[0] = 0;
    int rc = check_shape(B, T, Hk, Hv, Dk, Dv, chunk, gate_kind, form);
    if (rc) return rc;
    if (!dtype_ok(in_dtype) || !dtype_ok(out_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    const int f = resolve_form(Hv, Dk, Dv, mask != nullptr, gate_kind, form, in_dtype);
    if (f < 0) return f;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (B == 0) return GDN_OK;
    if (T == 0) {
        launch_copy_or_zero(state_T, state0, (size_t)B * Hv * Dv * Dk, st);
        return check_launch(st, "gdn_fwd(T=0)");
    }
    if (!q || !k || !v || !g || !beta || !y) return fail(GDN_ERR_INVALID, "null input or output pointer");
    if (f == GDN_FORM_CHUNK) {
        if (misaligned16(q) || misaligned16(k) || misaligned16(v))
            return fail(GDN_ERR_INVALID, "the chunked form needs 16-byte aligned q, k and v");
        ChunkCall cc{};
        cc.q = q; cc.k = k; cc.v = v; cc.g = g; cc.beta = beta; cc.state0 = state0;
        cc.y = y; cc.state_T = state_T;
        cc.B = B; cc.T = T; cc.Ts = T; cc.Hk = Hk; cc.Hv = Hv; cc.in_dt = in_dtype; cc.out_dt = out_dtype;
        cc.gate = gate_kind;
        if (mask) return ck_masked_forward(cc, mask, chunk, saved, saved_bytes, workspace, workspace_bytes, st);
        return ck_forward(cc, chunk, saved, saved_bytes, workspace, workspace_bytes, st);
    }
    const size_t need = rec_saved_bytes(B, T, Hv, Dk, Dv, chunk);
    float *snaps = nullptr;
    if (saved) {
        if (saved_bytes < need)
            return fail(GDN_ERR_WORKSPACE, "saved buffer of %zu bytes is smaller than the %zu bytes required",
                        saved_bytes, need);
        snaps = static_cast<float *>(saved);
    }
    RecFwdArgs a{q, k, v, g, beta, state0, mask, y, state_T, snaps,
                 B, T, Hk, Hv, Dk, Dv, chunk, in_dtype, out_dtype, gate_kind};
    {
        Timed tm("rec_fwd", st);
        launch_rec_fwd(a, st);
    }
    return check_launch(st, "gdn_fwd");
}

int gdn_decode_step(const void *q, const void *k, const void *v, const float *g, const float *beta,
                    const float *state_in, float *state_out, void *y, int B, int Hk, int Hv, int Dk, int Dv,
                    int in_dtype, int out_dtype, int gate_kind, void *stream) {
    g_err[0] = 0;
    int rc = check_shape(B, 1, Hk, Hv, Dk, Dv, 1, gate_kind, GDN_FORM_RECURRENT);
    if (rc) return rc;
    if (!dtype_ok(in_dtype) || !dtype_ok(out_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (B == 0) return GDN_OK;
    if (!q || !k || !v || !g || !beta || !y || !state_out)
        return fail(GDN_ERR_INVALID, "null input or output pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    // one token of the recurrent form: every thread reads its state elements before writing the same ones, so
    // state_out may be state_in
    RecFwdArgs a{q, k, v, g, beta, state_in, nullptr, y, state_out, nullptr,
                 B, 1, Hk, Hv, Dk, Dv, 1, in_dtype, out_dtype, gate_kind};
    {
        Timed tm("rec_decode", st);
        launch_rec_decode(a, st);
    }
    return check_launch(st, "gdn_decode_step");
}

int gdn_small_linears(const void *x, const void *const *w, void *const *y, const int *n, int count, int tokens, int k,
                      int dtype, void *stream) {
    g_err[0] = 0;
    if (count < 1 || count > 4 || tokens < 0 || k < 1 || !w || !y || !n)
        return fail(GDN_ERR_INVALID, "one to four weights, tokens >= 0 and k > 0 are expected");
    if (!dtype_ok(dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (tokens > small_linears_max_tokens() || k % 8)
        return fail(GDN_ERR_UNSUPPORTED, "at most %d tokens and k a multiple of 8", small_linears_max_tokens());
    if (tokens == 0) return GDN_OK;
    SmallLinears a{};
    a.x = x;
    a.count = count;
    a.tokens = tokens;
    a.k = k;
    for (int i = 0; i < count; ++i) {
        if (n[i] < 1 || n[i] > (1 << 28)) return fail(GDN_ERR_INVALID, "rows of weight %d: %d", i, n[i]);
        if (!w[i] || !y[i]) return fail(GDN_ERR_INVALID, "null pointer");
        if (misaligned16(w[i])) return fail(GDN_ERR_INVALID, "weights must be 16-byte aligned");
        a.w[i] = w[i];
        a.y[i] = y[i];
        a.n[i] = n[i];
    }
    if (!x || misaligned16(x)) return fail(GDN_ERR_INVALID, "x must be a 16-byte aligned pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    {
        Timed tm("small_linears", st);
        launch_small_linears(a, dtype, st);
    }
    return check_launch(st, "gdn_small_linears");
}

int gdn_block_decode(const void *qkv, const void *z, const void *b, const void *a, const void *conv_w, const void *A_log,
                     const void *dt_bias, const void *norm_w, const float *conv_in, float *conv_out,
                     const float *state_in, float *state_out, void *out, int B, int Hk, int Hv, int Dk, int Dv, int K,
                     int dtype, int conv_dtype, int A_dtype, int dt_bias_dtype, int norm_dtype, float q_scale,
                     float eps_qk, float eps_norm, void *stream) {
    g_err[0] = 0;
    int rc = check_shape(B, 1, Hk, Hv, Dk, Dv, 1, GATE_DECAY, GDN_FORM_RECURRENT);
    if (rc) return rc;
    for (int dt : {dtype, conv_dtype, A_dtype, dt_bias_dtype, norm_dtype})
        if (!dtype_ok(dt)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (!block_decode_supported(Dk, Dv, K))
        return fail(GDN_ERR_UNSUPPORTED, "gdn_block_decode takes Dk = Dv = 128 and a conv of 4 taps");
    if (B == 0) return GDN_OK;
    if (!qkv || !z || !b || !a || !conv_w || !A_log || !dt_bias || !norm_w || !conv_out || !state_out || !out)
        return fail(GDN_ERR_INVALID, "null input or output pointer");
    if (conv_in == conv_out) return fail(GDN_ERR_INVALID, "conv_out may not be conv_in");
    if (misaligned16(state_in) || misaligned16(state_out))
        return fail(GDN_ERR_INVALID, "the states must be 16-byte aligned");
    BlockDecode d{qkv, z, b, a, conv_w, A_log, dt_bias, norm_w, conv_in, state_in, conv_out, state_out, out,
                  Hk, Hv, dtype, conv_dtype, A_dtype, dt_bias_dtype, norm_dtype, q_scale, eps_qk, eps_norm};
    hipStream_t st = static_cast<hipStream_t>(stream);
    {
        Timed tm("block_decode", st);
        launch_block_decode(d, B, st);
    }
    return check_launch(st, "gdn_block_decode");
}

size_t gdn_bwd_workspace_bytes(int B, int T, int Hk, int Hv, int Dk, int Dv, int chunk, int gate_kind,
                               int has_mask, int form, int in_dtype) {
    if (check_shape(B, T, Hk, Hv, Dk, Dv, chunk, gate_kind, form)) return 0;
    const int f = resolve_form(Hv, Dk, Dv, has_mask, gate_kind, form, in_dtype);
    if (f < 0) return 0;
    if (f == GDN_FORM_CHUNK) {
        if (B == 0 || T == 0) return 0;
        const int W = ck_window(chunk);
        const CkShape shp{B, T, Hk, Hv, in_dtype == DT_BF16, vg_kind(gate_kind), has_mask != 0};
        if (has_mask) return mask_work_bytes(shp, chunk);
        if (W) return ck_bwd_target_bytes(shp, W);
        return ck_sizes(shp, T, true).work;
    }
    return bwd_layout(B, T, Hv, Dk, Dv, chunk, gate_kind).total;
}

int gdn_bwd(const void *q, const void *k, const void *v, const float *g, const float *beta,
            const float *state0, const uint8_t *mask, const void *saved, size_t saved_bytes, const void *dy,
            const float *dstate_T, void *dq, void *dk, void *dv, float *dg, float *dbeta, float *dstate0,
            void *workspace, size_t workspace_bytes, int B, int T, int Hk, int Hv, int Dk, int Dv, int chunk,
            int in_dtype, int dy_dtype, int grad_dtype, int gate_kind, int form, void *stream) {
    g_err[0] = 0;
    int rc = check_shape(B, T, Hk, Hv, Dk, Dv, chunk, gate_kind, form);
    if (rc) return rc;
    if (!dtype_ok(in_dtype) || !dtype_ok(dy_dtype) || !dtype_ok(grad_dtype))
        return fail(GDN_ERR_INVALID, "unknown dtype code");
    const int f = resolve_form(Hv, Dk, Dv, mask != nullptr, gate_kind, form, in_dtype);
    if (f < 0) return f;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (B == 0) return GDN_OK;
    if (T == 0) {
        launch_copy_or_zero(dstate0, dstate_T, (size_t)B * Hv * Dv * Dk, st);
        return check_launch(st, "gdn_bwd(T=0)");
    }
    if (!q || !k || !v || !g || !beta || !dy || !dq || !dk || !dv || !dg || !dbeta)
        return fail(GDN_ERR_INVALID, "null input or output pointer");
    if (f == GDN_FORM_CHUNK) {
        if (in_dtype == DT_BF16 && dy_dtype == DT_F16)
            return fail(GDN_ERR_UNSUPPORTED, "the chunked form with bf16 inputs takes a bf16 or fp32 dy, not fp16");
        if (misaligned16(q) || misaligned16(k) || misaligned16(v) || misaligned16(dy))
            return fail(GDN_ERR_INVALID, "the chunked form needs 16-byte aligned q, k, v and dy");
        if (misaligned16(dq) || misaligned16(dk) || misaligned16(dv))
            return fail(GDN_ERR_INVALID, "the chunked form needs 16-byte aligned dq, dk and dv");
        ChunkCall cc{};
        cc.q = q; cc.k = k; cc.v = v; cc.g = g; cc.beta = beta; cc.state0 = state0;
        cc.dy = dy; cc.dstate_T = dstate_T; cc.dq = dq; cc.dk = dk; cc.dv = dv; cc.dg = dg; cc.dbeta = dbeta;
        cc.dstate0 = dstate0;
        cc.B = B; cc.T = T; cc.Ts = T; cc.Hk = Hk; cc.Hv = Hv; cc.in_dt = in_dtype; cc.dy_dt = dy_dtype;
        cc.grad_dt = grad_dtype; cc.gate = gate_kind;
        if (mask) return ck_masked_backward(cc, mask, chunk, saved, saved_bytes, workspace, workspace_bytes, st);
        return ck_backward(cc, chunk, saved, saved_bytes, workspace, workspace_bytes, st);
    }
    const size_t need_saved = rec_saved_bytes(B, T, Hv, Dk, Dv, chunk);
    if (need_saved && (!saved || saved_bytes < need_saved))
        return fail(GDN_ERR_INVALID, "the saved buffer written by gdn_fwd (%zu bytes) is required", need_saved);
    const size_t need_ws = bwd_layout(B, T, Hv, Dk, Dv, chunk, gate_kind).total;
    if (workspace_bytes < need_ws || (need_ws && !workspace))
        return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes required",
                    workspace_bytes, need_ws);
    RecBwdArgs a{};
    a.q = q; a.k = k; a.v = v; a.g = g; a.beta = beta; a.state0 = state0; a.mask = mask;
    a.snaps = static_cast<const float *>(saved); a.dy = dy; a.dstate_T = dstate_T;
    a.dq = dq; a.dk = dk; a.dv = dv; a.dg = dg; a.dbeta = dbeta; a.dstate0 = dstate0;
    a.B = B; a.T = T; a.Hk = Hk; a.Hv = Hv; a.Dk = Dk; a.Dv = Dv; a.chunk = chunk;
    a.in_dt = in_dtype; a.dy_dt = dy_dtype; a.grad_dt = grad_dtype; a.gate = gate_kind;
    const BwdLayout L = bwd_layout(B, T, Hv, Dk, Dv, chunk, gate_kind);
    char *ws = static_cast<char *>(workspace);
    a.ws_sub = reinterpret_cast<float *>(ws + L.sub);
    a.part_qk = reinterpret_cast<float *>(ws + L.part_qk);
    a.part_gb = reinterpret_cast<float *>(ws + L.part_gb);
    a.part_gv = reinterpret_cast<float *>(ws + L.part_gv);
    a.nrb = rec_bwd_row_blocks(B, Hv, Dk, Dv, gate_kind);
    a.max_sub = rec_max_sub(T, chunk);
    {
        Timed tm("rec_bwd", st);
        launch_rec_bwd(a, st);
    }
    rc = check_launch(st, "gdn_bwd");
    if (rc) return rc;
    {
        Timed tm("rec_bwd_reduce", st);
        launch_rec_bwd_reduce(a, st);
    }
    return check_launch(st, "gdn_bwd_reduce");
}

// ------------------------------------------------------------------------------------------- block ops

static bool all_aligned16(std::initializer_list<const void *> ps) {
    for (const void *p : ps)
        if (p && misaligned16(p)) return false;
    return true;
}

static size_t floats_bytes(size_t n) { return align256(n * sizeof(float)); }

int gdn_gates_fwd(const void *a, const void *b, const float *A_log, const float *dt_bias, float *g, float *beta,
                  int64_t tokens, int Hv, int in_dtype, int log_space, int allow_neg_eigval, void *stream) {
    g_err[0] = 0;
    if (tokens < 0 || Hv <= 0) return fail(GDN_ERR_INVALID, "tokens must be >= 0 and Hv > 0");
    if (Hv > gates_max_heads()) return fail(GDN_ERR_UNSUPPORTED, "Hv > %d is not supported", gates_max_heads());
    if (!dtype_ok(in_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (tokens == 0) return GDN_OK;
    if (!a || !b || !A_log || !dt_bias || !g || !beta) return fail(GDN_ERR_INVALID, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    {
        Timed tm("gates_fwd", st);
        launch_gates_fwd(a, b, A_log, dt_bias, g, beta, (size_t)tokens, Hv, in_dtype, log_space != 0,
                         allow_neg_eigval ? 2.f : 1.f, st);
    }
    return check_launch(st, "gdn_gates_fwd");
}

size_t gdn_gates_bwd_workspace_bytes(int64_t tokens, int Hv) {
    if (tokens < 0 || Hv <= 0) return 0;
    return floats_bytes(gates_bwd_work_floats((size_t)tokens, Hv));
}

int gdn_gates_bwd(const void *a, const void *b, const float *A_log, const float *dt_bias, const float *g,
                  const float *dg, const float *dbeta, void *da, void *db, float *dA_log, float *ddt_bias,
                  void *workspace, size_t workspace_bytes, int64_t tokens, int Hv, int in_dtype, int grad_dtype,
                  int log_space, int allow_neg_eigval, void *stream) {
    g_err[0] = 0;
    if (tokens < 0 || Hv <= 0) return fail(GDN_ERR_INVALID, "tokens must be >= 0 and Hv > 0");
    if (Hv > gates_max_heads()) return fail(GDN_ERR_UNSUPPORTED, "Hv > %d is not supported", gates_max_heads());
    if (!dtype_ok(in_dtype) || !dtype_ok(grad_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (!A_log || !dt_bias || !dA_log || !ddt_bias) return fail(GDN_ERR_INVALID, "null pointer");
    if (tokens > 0 && (!a || !b || !g || !dg || !dbeta || !da || !db)) return fail(GDN_ERR_INVALID, "null pointer");
    const size_t need = gdn_gates_bwd_workspace_bytes(tokens, Hv);
    if (need && (!workspace || workspace_bytes < need))
        return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes required",
                    workspace_bytes, need);
    hipStream_t st = static_cast<hipStream_t>(stream);
    {
        Timed tm("gates_bwd", st);
        launch_gates_bwd(a, b, A_log, dt_bias, g, dg, dbeta, da, db, dA_log, ddt_bias, static_cast<float *>(workspace),
                         (size_t)tokens, Hv, in_dtype, grad_dtype, log_space != 0, allow_neg_eigval ? 2.f : 1.f, st);
    }
    return check_launch(st, "gdn_gates_bwd");
}

int gdn_l2norm_fwd(const void *x, void *y, int64_t rows, int D, float eps, float scale, int dtype, void *stream) {
    g_err[0] = 0;
    if (rows < 0 || D <= 0) return fail(GDN_ERR_INVALID, "rows must be >= 0 and D > 0");
    if (!dtype_ok(dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (rows == 0) return GDN_OK;
    if (!x || !y) return fail(GDN_ERR_INVALID, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    {
        Timed tm("l2norm_fwd", st);
        launch_l2norm_fwd(x, y, (size_t)rows, D, eps, scale, dtype, all_aligned16({x, y}), st);
    }
    return check_launch(st, "gdn_l2norm_fwd");
}

int gdn_l2norm_bwd(const void *x, const void *dy, void *dx, int64_t rows, int D, float eps, float scale, int dtype,
                   int dy_dtype, void *stream) {
    g_err[0] = 0;
    if (rows < 0 || D <= 0) return fail(GDN_ERR_INVALID, "rows must be >= 0 and D > 0");
    if (!dtype_ok(dtype) || !dtype_ok(dy_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (rows == 0) return GDN_OK;
    if (!x || !dy || !dx) return fail(GDN_ERR_INVALID, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    {
        Timed tm("l2norm_bwd", st);
        launch_l2norm_bwd(x, dy, dx, (size_t)rows, D, eps, scale, dtype, dy_dtype, all_aligned16({x, dy, dx}), st);
    }
    return check_launch(st, "gdn_l2norm_bwd");
}

static int check_conv(int B, int T, int C, int K, int dtype) {
    if (B < 0 || T < 0 || C < 0) return fail(GDN_ERR_INVALID, "B, T and C must be >= 0");
    if (K < 2) return fail(GDN_ERR_INVALID, "the conv kernel size K must be >= 2");
    if (K > conv_kmax()) return fail(GDN_ERR_UNSUPPORTED, "conv kernel size K > %d is not supported", conv_kmax());
    if (!dtype_ok(dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    return GDN_OK;
}

int gdn_conv_silu_fwd(const void *x, const float *w, const float *state_in, void *out, float *state_out, int B,
                      int T, int C, int K, int dtype, void *stream) {
    g_err[0] = 0;
    int rc = check_conv(B, T, C, K, dtype);
    if (rc) return rc;
    if (B == 0 || C == 0) return GDN_OK;
    if (!w || (T > 0 && (!x || !out))) return fail(GDN_ERR_INVALID, "null pointer");
    if (state_out && state_out == state_in) return fail(GDN_ERR_INVALID, "state_out must not alias state_in");
    hipStream_t st = static_cast<hipStream_t>(stream);
    ConvCall c{};
    c.x = x; c.w = w; c.state_in = state_in; c.v = out; c.state_out = state_out;
    c.B = B; c.T = T; c.C = C; c.K = K; c.qk = 0; c.Dk = 0; c.dt = dtype; c.g_dt = dtype;
    c.vec = all_aligned16({x, out});
    {
        Timed tm("conv_fwd", st);
        launch_conv_fwd(c, st);
    }
    return check_launch(st, "gdn_conv_silu_fwd");
}

size_t gdn_conv_silu_bwd_workspace_bytes(int B, int T, int C, int K) {
    if (B < 0 || T < 0 || C < 0 || K < 2) return 0;
    return floats_bytes(conv_bwd_work_floats(B, T, C, K));
}

int gdn_conv_silu_bwd(const void *x, const float *w, const float *state_in, const void *dout, void *dx, float *dw,
                      void *workspace, size_t workspace_bytes, int B, int T, int C, int K, int dtype, int dout_dtype,
                      void *stream) {
    g_err[0] = 0;
    int rc = check_conv(B, T, C, K, dtype);
    if (rc) return rc;
    if (!dtype_ok(dout_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (C == 0) return GDN_OK;
    if (!w || !dw || (B > 0 && T > 0 && (!x || !dout || !dx))) return fail(GDN_ERR_INVALID, "null pointer");
    const size_t need = gdn_conv_silu_bwd_workspace_bytes(B, T, C, K);
    if (need && (!workspace || workspace_bytes < need))
        return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes required",
                    workspace_bytes, need);
    hipStream_t st = static_cast<hipStream_t>(stream);
    ConvCall c{};
    c.x = x; c.w = w; c.state_in = state_in; c.v = const_cast<void *>(dout); c.dx = dx; c.dw = dw;
    c.work = static_cast<float *>(workspace);
    c.B = B; c.T = T; c.C = C; c.K = K; c.qk = 0; c.Dk = 0; c.dt = dtype; c.g_dt = dout_dtype;
    c.vec = all_aligned16({x, dout, dx});
    {
        Timed tm("conv_bwd", st);
        launch_conv_bwd(c, st);
    }
    return check_launch(st, "gdn_conv_silu_bwd");
}

static int check_conv_qkv(int B, int T, int Hk, int Dk, int Hv, int Dv, int K, int dtype, int g_dtype, bool vec) {
    if (Hk <= 0 || Dk <= 0 || Hv <= 0 || Dv <= 0) return fail(GDN_ERR_INVALID, "head counts and dims must be > 0");
    const int64_t C = 2LL * Hk * Dk + (int64_t)Hv * Dv;
    if (C > (1 << 30)) return fail(GDN_ERR_INVALID, "too many channels");
    int rc = check_conv(B, T, (int)C, K, dtype);
    if (rc) return rc;
    if (!dtype_ok(g_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (!conv_qkv_supported(Dk, K, dtype, g_dtype, vec, (int)C))
        return fail(GDN_ERR_UNSUPPORTED,
                    "the fused conv + L2 norm needs K = 4, 16-byte aligned buffers, channels a multiple of 4 and "
                    "Dk / (channels per lane) a power of two in [4, 64]; use gdn_conv_silu_* and gdn_l2norm_*");
    return GDN_OK;
}

int gdn_conv_qkv_fwd(const void *x, const float *w, const float *state_in, void *q, void *k, void *v,
                     float *state_out, int B, int T, int Hk, int Dk, int Hv, int Dv, int K, float q_scale, float eps,
                     int dtype, void *stream) {
    g_err[0] = 0;
    int rc = check_conv_qkv(B, T, Hk, Dk, Hv, Dv, K, dtype, dtype, all_aligned16({x, q, k, v}));
    if (rc) return rc;
    if (B == 0) return GDN_OK;
    if (!w || (T > 0 && (!x || !q || !k || !v))) return fail(GDN_ERR_INVALID, "null pointer");
    if (state_out && state_out == state_in) return fail(GDN_ERR_INVALID, "state_out must not alias state_in");
    hipStream_t st = static_cast<hipStream_t>(stream);
    ConvCall c{};
    c.x = x; c.w = w; c.state_in = state_in; c.q = q; c.k = k; c.v = v; c.state_out = state_out;
    c.B = B; c.T = T; c.C = 2 * Hk * Dk + Hv * Dv; c.K = K; c.qk = Hk * Dk; c.Dk = Dk; c.dt = dtype; c.g_dt = dtype;
    c.scale_q = q_scale; c.eps = eps; c.vec = true;
    {
        Timed tm("conv_qkv_fwd", st);
        launch_conv_fwd(c, st);
    }
    return check_launch(st, "gdn_conv_qkv_fwd");
}

int gdn_conv_qkv_bwd(const void *x, const float *w, const float *state_in, const void *dq, const void *dk,
                     const void *dv, void *dx, float *dw, void *workspace, size_t workspace_bytes, int B, int T,
                     int Hk, int Dk, int Hv, int Dv, int K, float q_scale, float eps, int dtype, int g_dtype,
                     void *stream) {
    g_err[0] = 0;
    int rc = check_conv_qkv(B, T, Hk, Dk, Hv, Dv, K, dtype, g_dtype, all_aligned16({x, dq, dk, dv, dx}));
    if (rc) return rc;
    const int C = 2 * Hk * Dk + Hv * Dv;
    if (!w || !dw || (B > 0 && T > 0 && (!x || !dq || !dk || !dv || !dx))) return fail(GDN_ERR_INVALID, "null pointer");
    const size_t need = gdn_conv_silu_bwd_workspace_bytes(B, T, C, K);
    if (need && (!workspace || workspace_bytes < need))
        return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes required",
                    workspace_bytes, need);
    hipStream_t st = static_cast<hipStream_t>(stream);
    ConvCall c{};
    c.x = x; c.w = w; c.state_in = state_in;
    c.q = const_cast<void *>(dq); c.k = const_cast<void *>(dk); c.v = const_cast<void *>(dv);
    c.dx = dx; c.dw = dw; c.work = static_cast<float *>(workspace);
    c.B = B; c.T = T; c.C = C; c.K = K; c.qk = Hk * Dk; c.Dk = Dk; c.dt = dtype; c.g_dt = g_dtype;
    c.scale_q = q_scale; c.eps = eps; c.vec = true;
    {
        Timed tm("conv_qkv_bwd", st);
        launch_conv_bwd(c, st);
    }
    return check_launch(st, "gdn_conv_qkv_bwd");
}

static int check_grms(int64_t rows, int D, int dtype, int z_dtype, bool bwd) {
    if (rows < 0 || D <= 0) return fail(GDN_ERR_INVALID, "rows must be >= 0 and D > 0");
    if (bwd && D > grms_dmax())
        return fail(GDN_ERR_UNSUPPORTED, "gated RMSNorm backward of rows longer than %d", grms_dmax());
    if (!dtype_ok(dtype) || !dtype_ok(z_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    return GDN_OK;
}

int gdn_gated_rmsnorm_fwd(const void *y, const void *z, const float *w, void *out, int64_t rows, int D, float eps,
                          int dtype, int z_dtype, void *stream) {
    g_err[0] = 0;
    int rc = check_grms(rows, D, dtype, z_dtype, false);
    if (rc) return rc;
    if (rows == 0) return GDN_OK;
    if (!y || !z || !w || !out) return fail(GDN_ERR_INVALID, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    {
        Timed tm("grms_fwd", st);
        launch_grms_fwd(y, z, w, out, (size_t)rows, D, eps, dtype, z_dtype, all_aligned16({y, z, w, out}), st);
    }
    return check_launch(st, "gdn_gated_rmsnorm_fwd");
}

size_t gdn_gated_rmsnorm_bwd_workspace_bytes(int64_t rows, int D) {
    if (rows < 0 || D <= 0) return 0;
    return floats_bytes(grms_bwd_work_floats((size_t)rows, D));
}

int gdn_gated_rmsnorm_bwd(const void *y, const void *z, const float *w, const void *dout, void *dy, void *dz,
                          float *dw, void *workspace, size_t workspace_bytes, int64_t rows, int D, float eps,
                          int dtype, int z_dtype, int dout_dtype, void *stream) {
    g_err[0] = 0;
    int rc = check_grms(rows, D, dtype, z_dtype, true);
    if (rc) return rc;
    if (!dtype_ok(dout_dtype)) return fail(GDN_ERR_INVALID, "unknown dtype code");
    if (!w || !dw || (rows > 0 && (!y || !z || !dout || !dy || !dz))) return fail(GDN_ERR_INVALID, "null pointer");
    const size_t need = gdn_gated_rmsnorm_bwd_workspace_bytes(rows, D);
    if (need && (!workspace || workspace_bytes < need))
        return fail(GDN_ERR_WORKSPACE, "workspace of %zu bytes is smaller than the %zu bytes required",
                    workspace_bytes, need);
    hipStream_t st = static_cast<hipStream_t>(stream);
    {
        Timed tm("grms_bwd", st);
        launch_grms_bwd(y, z, w, dout, dy, dz, dw, static_cast<float *>(workspace), (size_t)rows, D, eps, dtype,
                        z_dtype, dout_dtype, all_aligned16({y, z, w, dout, dy, dz}), st);
    }
    return check_launch(st, "gdn_gated_rmsnorm_bwd");
}

}  // extern "C"
