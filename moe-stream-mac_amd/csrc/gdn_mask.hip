// Masked steps on the chunked form: what makes a masked call one chunked pass.
//
// A step with mask m_t = 0 keeps the state (S_t = S_{t-1}) but its output reads the candidate state
// (tools/gdn_vjp.py:3-6, _step_parts :238-256):
//   y_t = S~_t q_t = d_t S_{t-1} q_t + beta_t c_t (v_t - d_t S_{t-1} k_t),   c_t = k_t . q_t      (d_t the decay).
// The chunked form runs the effective recurrence with d'_t = m_t ? d_t : 1 and beta'_t = m_t beta_t, whose state
// equals the masked recurrence's state at every token.  y_t is linear in that state, so a masked token needs no pass of
// its own, only another query (one per value head, as d and beta are) and a term that the state does not enter:
//   y_t = S'_t q~_t + e_t v_t,   q~_t = d_t (q_t - beta_t c_t k_t),   e_t = beta_t c_t.
// mask_query_kernel writes the effective gates, q~ and e of the masked tokens and which 64-token chunks hold one; the
// chunked kernels read q~ in the place of q in those chunks (hi / lo planes in the bf16 set, whose q is exact where q~ is
// not) and add e v to y.  The backward's only special output is X_t = dL/dq~_t: a masked token's k
// and v enter nothing else (Delta_t = 0, beta'_t = 0), so all of its gradients follow from X_t and dy_t
// (mask_bwd_fix_kernel):
//   dv = e dy,   dc = beta (v . dy - d k . X),   dbeta = c (v . dy - d k . X),   dd = q . X - beta c k . X,
//   dq = sum over the key head's value heads of d X + dc k,   dk = ... of dc q - d beta c X.
// With no other use of the state behind them, dc, dbeta and dd are as exact as X: in the bf16 set a flagged chunk's dQ
// therefore takes in the lo parts of the entry state and of an fp32 dY too (ck_bwd_local_bf16), which costs 70 us below.
//
// The first form of this path ran the recurrence twice, the second time with k as the query, around fp32 copies of
// every output, cotangent and gradient: at B = 4, T = 4096, Hv = 32, bf16, a fifth of the tokens masked, 3.78 ms per
// forward + VJP, with the query rows 1.89 ms (1.42 ms without a mask).  Both kernels here are bound by the rows of the
// masked tokens: 43 us (forward) and 81 us (backward) of that.
#include "gdn_common.h"
#include "gdn_internal.h"

namespace gdn {

constexpr int MK_THREADS = 256;
constexpr int MK_MAX_HEADS = 256;
static_assert(MK_MAX_HEADS <= MK_THREADS, "one thread per value head's gates");

// Sum over the wave, the same bits in every lane: DPP row sums, then the lane swaps across rows and halves.
__device__ __forceinline__ float wave_sum(float x) {
    x = row16_allreduce(x);
    x += lane_xor16(x);
    return x + lane_xor32(x);
}

__device__ __forceinline__ float decay_of(const float *g, size_t gi, int gate) {
    return gate == GATE_LOG ? expf(g[gi]) : g[gi];
}

// A row of D <= 128 elements (even) over a wave: lane l holds elements 2 l and 2 l + 1.
__device__ __forceinline__ float2 load_row(const void *p, size_t base, int D, int l, int dt) {
    const size_t i = base + 2 * l;
    if (2 * l >= D) return make_float2(0.f, 0.f);
    if (dt == DT_F32) return *reinterpret_cast<const float2 *>(static_cast<const float *>(p) + i);
    const uint32_t w = *reinterpret_cast<const uint32_t *>(static_cast<const uint16_t *>(p) + i);
    if (dt == DT_BF16) return make_float2(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u));
    return make_float2(__half2float(__ushort_as_half((unsigned short)(w & 0xffffu))),
                       __half2float(__ushort_as_half((unsigned short)(w >> 16))));
}
__device__ __forceinline__ void store_row(void *p, size_t base, int D, int l, float2 x, int dt) {
    const size_t i = base + 2 * l;
    if (2 * l >= D) return;
    if (dt == DT_F32) {
        *reinterpret_cast<float2 *>(static_cast<float *>(p) + i) = x;
    } else if (dt == DT_BF16) {
        *reinterpret_cast<uint32_t *>(static_cast<uint16_t *>(p) + i) =
            f32_to_bf16_cvt(x.x) | ((uint32_t)f32_to_bf16_cvt(x.y) << 16);
    } else {
        store_from_f32(p, i, x.x, dt);
        store_from_f32(p, i + 1, x.y, dt);
    }
}
__device__ __forceinline__ float dot_row(float2 x, float2 y) { return wave_sum(fmaf(x.x, y.x, x.y * y.y)); }

// One workgroup per token, a wave per key head in turn: the effective gates, and in a chunk that holds a masked token the
// query rows of the value heads (an unmasked token's is q, so that the chunked kernels pick q or qm by the chunk alone)
// and e.  The workgroup of a chunk's first token writes the chunk's flag.
__global__ __launch_bounds__(MK_THREADS) void mask_query_kernel(MaskArgs a) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    const size_t tok = blockIdx.x;
    const int b = (int)(tok / a.T), t = (int)(tok - (size_t)b * a.T), t0 = t - t % kChunkC;
    const bool keep = a.mask[tok] != 0;
    const bool any = __ballot(t0 + l < a.T && a.mask[(size_t)b * a.T + min(t0 + l, a.T - 1)] == 0) != 0;
    if (t == t0 && threadIdx.x == 0) a.cm[(size_t)b * ((a.T + kChunkC - 1) / kChunkC) + t / kChunkC] = any;
    if ((int)threadIdx.x < a.Hv) {  // Hv <= MK_MAX_HEADS
        const size_t gi = tok * a.Hv + threadIdx.x;
        a.g2[gi] = keep ? a.g[gi] : (a.gate == GATE_LOG ? 0.f : 1.f);
        a.beta2[gi] = keep ? a.beta[gi] : 0.f;
    }
    if (!any) return;
    const int rep = a.Hv / a.Hk;
    if (w >= a.Hk) return;
    const size_t row0 = (tok * a.Hk + w) * a.Dk;
    float2 qn = load_row(a.q, row0, a.Dk, l, a.in_dt), kn = load_row(a.k, row0, a.Dk, l, a.in_dt);
    for (int hk = w; hk < a.Hk; hk += MK_THREADS / 64) {
        const float2 q = qn, k = kn;
        if (hk + MK_THREADS / 64 < a.Hk) {  // the wave's next key head, in flight during this one
            const size_t row = (tok * a.Hk + hk + MK_THREADS / 64) * a.Dk;
            qn = load_row(a.q, row, a.Dk, l, a.in_dt);
            kn = load_row(a.k, row, a.Dk, l, a.in_dt);
        }
        const float c = dot_row(q, k);
        for (int hv = hk * rep; hv < (hk + 1) * rep; ++hv) {
            const size_t gi = tok * a.Hv + hv, base = gi * a.Dk;
            float2 x = q;
            if (!keep) {
                const float d = decay_of(a.g, gi, a.gate), e = a.beta[gi] * c;
                if (l == 0) a.e[gi] = e;
                x = make_float2(d * (q.x - e * k.x), d * (q.y - e * k.y));
            }
            if (a.in_dt == DT_BF16) {
                store_row(a.qm, base, a.Dk, l, x, DT_BF16);
                const float2 lo = make_float2(x.x - bf16_to_f32(f32_to_bf16_cvt(x.x)), x.y - bf16_to_f32(f32_to_bf16_cvt(x.y)));
                store_row(a.qm, a.qm_lo + base, a.Dk, l, lo, DT_BF16);
            } else {
                store_row(a.qm, base, a.Dk, l, x, DT_F32);
            }
        }
    }
}

// Every gradient of the masked tokens from X = dL/dq~ and dy: one workgroup per token, a wave per key head in turn, the
// next value head's rows in flight.
__global__ __launch_bounds__(MK_THREADS) void mask_bwd_fix_kernel(MaskArgs a) {
    const size_t tok = blockIdx.x;
    if (a.mask[tok] != 0) return;
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63, rep = a.Hv / a.Hk;
    struct Rows {
        float2 X, v, dy;
        float g, beta;
    };
    auto load = [&](int hv) {
        const size_t gi = tok * a.Hv + hv;
        return Rows{load_row(a.xm, gi * a.Dk, a.Dk, l, DT_F32), load_row(a.v, gi * a.Dv, a.Dv, l, a.in_dt),
                    load_row(a.dy, gi * a.Dv, a.Dv, l, a.dy_dt), a.g[gi], a.beta[gi]};
    };
    if (w >= a.Hk) return;
    Rows nx = load(w * rep);
    for (int hk = w; hk < a.Hk; hk += MK_THREADS / 64) {
        const size_t qb = (tok * a.Hk + hk) * a.Dk;
        const float2 q = load_row(a.q, qb, a.Dk, l, a.in_dt), k = load_row(a.k, qb, a.Dk, l, a.in_dt);
        const float c = dot_row(q, k);
        float2 dq = make_float2(0.f, 0.f), dk = dq;
        for (int hv = hk * rep; hv < (hk + 1) * rep; ++hv) {
            const Rows r = nx;
            const int nhv = hv + 1 < (hk + 1) * rep ? hv + 1 : (hk + MK_THREADS / 64) * rep;
            if (nhv < a.Hv) nx = load(nhv);
            const size_t gi = tok * a.Hv + hv;
            const float d = a.gate == GATE_LOG ? expf(r.g) : r.g, e = r.beta * c;
            const float kx = dot_row(k, r.X), qx = dot_row(q, r.X), u = dot_row(r.v, r.dy) - d * kx;
            const float dc = r.beta * u, de = d * e;
            dq.x += d * r.X.x + dc * k.x;
            dq.y += d * r.X.y + dc * k.y;
            dk.x += dc * q.x - de * r.X.x;
            dk.y += dc * q.y - de * r.X.y;
            store_row(a.dv, gi * a.Dv, a.Dv, l, make_float2(e * r.dy.x, e * r.dy.y), a.grad_dt);
            if (l == 0) {
                const float dd = qx - e * kx;
                a.dg[gi] = a.gate == GATE_LOG ? d * dd : dd;
                a.dbeta[gi] = c * u;
            }
        }
        store_row(a.dq, qb, a.Dk, l, dq, a.grad_dt);
        store_row(a.dk, qb, a.Dk, l, dk, a.grad_dt);
    }
}

int mask_max_heads() { return MK_MAX_HEADS; }

void launch_mask_query(const MaskArgs &a, hipStream_t st) {
    const size_t tokens = (size_t)a.B * a.T;
    if (tokens) hipLaunchKernelGGL(mask_query_kernel, dim3((unsigned)tokens), dim3(MK_THREADS), 0, st, a);
}

void launch_mask_bwd_fix(const MaskArgs &a, hipStream_t st) {
    const size_t tokens = (size_t)a.B * a.T;
    if (tokens) hipLaunchKernelGGL(mask_bwd_fix_kernel, dim3((unsigned)tokens), dim3(MK_THREADS), 0, st, a);
}

}  // namespace gdn
