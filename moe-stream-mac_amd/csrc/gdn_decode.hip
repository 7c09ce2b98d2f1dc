// One decoded token of a whole GDN block (engine/src/gdn_layer.c:18-58 at one token) in three launches (five for 9 to 16
// sequences): the in-projections, everything between the projections, and the out-projection.
//
// As separate calls the token takes five library GEMMs, the conv, its state, the gates, the recurrence, the norm and the
// parameters' conversions to fp32, 16 launches that each cost more on the host than on the device: 248 us at B = 1,
// hidden 2048, Hk = 16, Hv = 32, D = 128, bf16, against the 14 us its 72 MB take at the copy rate.  In three launches 64
// us, 33 us of them on the device (the projections 23 us, 3.0 TB/s; the middle, one workgroup per head, 10 us).
#include "gdn_common.h"
#include "gdn_internal.h"

namespace gdn {

// Sum over the wave, the same bits in every lane.
__device__ __forceinline__ float wave_sum(float x) {
    x = row16_allreduce(x);
    x += lane_xor16(x);
    return x + lane_xor32(x);
}

// Eight consecutive elements from element i (16-byte aligned; fp32: two 16-byte loads) as fp32.
template <int DT>
struct Piece8 {
    uint4 a, b;
    __device__ __forceinline__ void load(const void *p, size_t i) {
        if constexpr (DT == DT_F32) {
            a = *reinterpret_cast<const uint4 *>(static_cast<const float *>(p) + i);
            b = *reinterpret_cast<const uint4 *>(static_cast<const float *>(p) + i + 4);
        } else {
            a = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(p) + i);
        }
    }
    __device__ __forceinline__ void get(float (&x)[8]) const {
        const uint32_t w[4] = {a.x, a.y, a.z, a.w};
        if constexpr (DT == DT_F32) {
            const uint32_t v[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = __uint_as_float(w[i]);
                x[4 + i] = __uint_as_float(v[i]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (DT == DT_BF16) {
                    x[2 * i] = __uint_as_float(w[i] << 16);
                    x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
                } else {
                    x[2 * i] = __half2float(__ushort_as_half((unsigned short)(w[i] & 0xffffu)));
                    x[2 * i + 1] = __half2float(__ushort_as_half((unsigned short)(w[i] >> 16)));
                }
            }
        }
    }
};

// y_i = x W_i^T for up to 8 tokens and up to four weights that share x.  A wave takes ROWS rows (of one weight) for all
// tokens, its lanes 8 consecutive inputs each: the weights are read once, in runs of 1 KiB (fp32: 2), and bound the
// kernel.  ROWS runs by an unroll of two are 8 KiB of weights in flight per wave at 4 rows, 16 at 8; more tokens take more
// rows, so that the inputs, re-read by every wave from L1, stay below the weights' bytes.
template <int DT, int NT, int ROWS>
__global__ __launch_bounds__(256) void small_linears_kernel(SmallLinears a) {
    const int l = threadIdx.x & 63;
    int row = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * ROWS, i = 0;
    while (i < a.count && row >= a.pad[i]) row -= a.pad[i++];  // every weight's rows rounded up to ROWS
    if (i == a.count) return;
    const int n = a.n[i];
    if (row >= n) return;
    const void *W = a.w[i];
    float acc[ROWS][NT];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[r][t] = 0.f;
#pragma unroll 2
    for (int k = 8 * l; k < a.k; k += 512) {
        Piece8<DT> w[ROWS], x[NT];
#pragma unroll
        for (int r = 0; r < ROWS; ++r) w[r].load(W, (size_t)min(row + r, n - 1) * a.k + k);
#pragma unroll
        for (int t = 0; t < NT; ++t) x[t].load(a.x, (size_t)min(t, a.tokens - 1) * a.k + k);
        float xv[NT][8];
#pragma unroll
        for (int t = 0; t < NT; ++t) x[t].get(xv[t]);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            float wv[8];
            w[r].get(wv);
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[r][t] = fmaf(wv[e], xv[t][e], acc[r][t]);
        }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float s = wave_sum(acc[r][t]);
            if (l == 0 && row + r < n && t < a.tokens) store_from_f32(a.y[i], (size_t)t * n + row + r, s, DT);
        }
}

constexpr int BD_D = 128, BD_K = 4, BD_THREADS = 512;

// Everything between the projections of one token: conv step + SiLU of a value head's q, k and v channels, their norms,
// the gates, the delta rule over the head's state and the gated RMSNorm, in fp32 throughout.  One workgroup per value
// head and sequence: a row of the state per 16 lanes, four rows per 16-lane group, the state loaded before anything else
// (it is the kernel's traffic: 128 KiB per workgroup).  The first value head of a key head moves on the conv state of the
// q and k channels.
__global__ __launch_bounds__(BD_THREADS) void block_decode_kernel(BlockDecode a) {
    __shared__ float sx[3 * BD_D];  // q, k, v after conv, SiLU and norm
    __shared__ float sy[BD_D], ssum[4], sred[2];
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, li = l & 15, row0 = 4 * (tid >> 4);
    const int hv = blockIdx.x, b = blockIdx.y, rep = a.Hv / a.Hk, hk = hv / rep;
    const size_t head = (size_t)b * a.Hv + hv;
    float4 S[4][2];
    if (a.state_in) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                S[r][i] = *reinterpret_cast<const float4 *>(a.state_in + (head * BD_D + row0 + r) * BD_D + 8 * li + 4 * i);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[r][0] = S[r][1] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const int kd = a.Hk * BD_D, C = 2 * kd + a.Hv * BD_D;
    if (tid < 3 * BD_D) {
        const int part = tid / BD_D, j = tid - part * BD_D;
        const int ch = part == 2 ? 2 * kd + hv * BD_D + j : part * kd + hk * BD_D + j;
        const float x = load_as_f32(a.qkv, (size_t)b * C + ch, a.dt);
        float s[BD_K - 1], acc = 0.f;
#pragma unroll
        for (int i = 0; i < BD_K - 1; ++i) {
            s[i] = a.conv_in ? a.conv_in[((size_t)b * (BD_K - 1) + i) * C + ch] : 0.f;
            acc = fmaf(load_as_f32(a.conv_w, (size_t)ch * BD_K + i, a.conv_dt), s[i], acc);
        }
        acc = fmaf(load_as_f32(a.conv_w, (size_t)ch * BD_K + BD_K - 1, a.conv_dt), x, acc);
        if (part == 2 || hv % rep == 0) {
#pragma unroll
            for (int i = 0; i < BD_K - 1; ++i)
                a.conv_out[((size_t)b * (BD_K - 1) + i) * C + ch] = i + 1 < BD_K - 1 ? s[i + 1 < BD_K - 1 ? i + 1 : 0] : x;
        }
        const float v = acc / (1.f + expf(-acc));
        sx[tid] = v;
        const float ss = wave_sum(v * v);
        if (l == 0 && w < 4) ssum[w] = ss;  // waves 0, 1: q; 2, 3: k
    }
    // the gates (every thread alike)
    const size_t gi = (size_t)b * a.Hv + hv;
    const float t = load_as_f32(a.a, gi, a.dt) + load_as_f32(a.dt_bias, hv, a.dtb_dt);
    const float sp = t > 20.f ? t : log1pf(expf(t));
    const float d = expf(-expf(load_as_f32(a.A_log, hv, a.A_dt)) * sp);
    const float beta = 1.f / (1.f + expf(-load_as_f32(a.b, gi, a.dt)));
    __syncthreads();
    const float qn = a.q_scale / sqrtf(ssum[0] + ssum[1] + a.eps_qk), kn = 1.f / sqrtf(ssum[2] + ssum[3] + a.eps_qk);
    float q[8], k[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        q[i] = sx[8 * li + i] * qn;
        k[i] = sx[BD_D + 8 * li + i] * kn;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float A[8] = {S[r][0].x, S[r][0].y, S[r][0].z, S[r][0].w, S[r][1].x, S[r][1].y, S[r][1].z, S[r][1].w};
        float kv = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            A[i] *= d;
            kv = fmaf(A[i], k[i], kv);
        }
        kv = row16_allreduce(kv);
        const float delta = beta * (sx[2 * BD_D + row0 + r] - kv);
        float y = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            A[i] = fmaf(delta, k[i], A[i]);
            y = fmaf(A[i], q[i], y);
        }
        y = row16_allreduce(y);
        if (li == 0) sy[row0 + r] = y;
        float *o = a.state_out + (head * BD_D + row0 + r) * BD_D + 8 * li;
        *reinterpret_cast<float4 *>(o) = make_float4(A[0], A[1], A[2], A[3]);
        *reinterpret_cast<float4 *>(o + 4) = make_float4(A[4], A[5], A[6], A[7]);
    }
    __syncthreads();
    if (tid < BD_D) {
        const float ss = wave_sum(sy[tid] * sy[tid]);
        if (l == 0) sred[w] = ss;
    }
    __syncthreads();
    if (tid < BD_D) {
        const float rms = 1.f / sqrtf((sred[0] + sred[1]) * (1.f / BD_D) + a.eps_norm);
        const float z = load_as_f32(a.z, head * BD_D + tid, a.dt);
        const float o = sy[tid] * rms * load_as_f32(a.norm_w, tid, a.norm_dt) * (z / (1.f + expf(-z)));
        store_from_f32(a.out, head * BD_D + tid, o, a.dt);
    }
}

// More tokens than a wave holds run in groups of 8, the weights then coming from the Infinity Cache.  Two groups are the
// most that pay: at hidden 2048 the whole block takes 92 us for a token of 16 sequences (140 us with the library's GEMMs in
// the place of this kernel) and would take 177 us for 32 (141 us).
int small_linears_max_tokens() { return 16; }

template <int DT, int NT, int ROWS>
static void small_linears_launch(SmallLinears a, hipStream_t st) {
    int rows = 0;
    for (int i = 0; i < a.count; ++i) rows += a.pad[i] = (a.n[i] + ROWS - 1) / ROWS * ROWS;
    const unsigned blocks = (unsigned)((rows / ROWS + 3) / 4);
    if (blocks) hipLaunchKernelGGL((small_linears_kernel<DT, NT, ROWS>), dim3(blocks), dim3(256), 0, st, a);
}
template <int DT>
static void small_linears_dt(const SmallLinears &a, hipStream_t st) {
    if (a.tokens <= 1) small_linears_launch<DT, 1, 4>(a, st);
    else if (a.tokens <= 2) small_linears_launch<DT, 2, 4>(a, st);
    else if (a.tokens <= 4) small_linears_launch<DT, 4, 4>(a, st);
    else small_linears_launch<DT, 8, 8>(a, st);
}
void launch_small_linears(const SmallLinears &call, int dt, hipStream_t st) {
    const size_t esz = dt == DT_F32 ? 4 : 2;
    for (int t = 0; t < call.tokens; t += 8) {
        SmallLinears a = call;
        a.tokens = call.tokens - t < 8 ? call.tokens - t : 8;
        a.x = static_cast<const char *>(call.x) + (size_t)t * call.k * esz;
        for (int i = 0; i < a.count; ++i) a.y[i] = static_cast<char *>(call.y[i]) + (size_t)t * call.n[i] * esz;
        if (dt == DT_F32) small_linears_dt<DT_F32>(a, st);
        else if (dt == DT_BF16) small_linears_dt<DT_BF16>(a, st);
        else small_linears_dt<DT_F16>(a, st);
    }
}

bool block_decode_supported(int Dk, int Dv, int K) { return Dk == BD_D && Dv == BD_D && K == BD_K; }
void launch_block_decode(const BlockDecode &a, int B, hipStream_t st) {
    hipLaunchKernelGGL(block_decode_kernel, dim3(a.Hv, B), dim3(BD_THREADS), 0, st, a);
}

}  // namespace gdn
