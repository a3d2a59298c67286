// Token mixers over a RAGGED step: the tokens of all rows of a step lie back to back, row b owning
// tokens [row_start[b], row_start[b] + row_len[b]) that continue its sequence at position row_ctx[b]
// (a prompt's portion of any length beside single decoded tokens).  What a sequence carries between
// steps lives either in pages of a key/value pool (block_table) or in its state slot (row_slot);
// a row with row_ctx == 0 starts from zero state whatever its slot held before.
//
//   conv_silu / conv_state_update  short causal convolution per channel with its tail kept per slot
//   conv_taps                      the same convolution without bias or activation, optionally added to its
//                                  input (y = u + conv(u)); output in fp32 and / or the activation type
//   conv_qkv_store                 the convolution over the q | k | v columns of one projection: queries to a
//                                  buffer, keys and values straight into their pages
//   softplus_decay                 step sizes and decays of a selective state-space head
//   scan_outer                     S_t = decay_t S_(t-1) + gain_t k_t v_t^T,  o_t = S_t^T q_t (+ skip_h v_t)
//                                  (state-space duality heads and fixed-decay retention heads alike)
//   scan_gated                     S_t = diag(f_t) S_(t-1) + (1 - f_t) v_t^T,  o_t = S_t^T q_t: a forget gate per
//                                  state row that also scales what is written (no key)
//   gate_lower_bound               q = silu(q), f = l + (1 - l) sigmoid(f + b) in place, ahead of scan_gated
//   rotary_pairs                   rotate-half rotation of the first `rot` dimensions of each head
//   gated_group_norm               unit-RMS per group with a SiLU gate before or after it
//   qk_unitnorm_store              per-head unit-RMS of queries and keys, keys/values into their pages
//   qk_rotary_store                biases on queries and keys, rotation of both over the first `rot` dimensions
//                                  of a head (adjacent pairs or halves); the rotated key into the key page and the
//                                  key as projected into the value page (attention whose values are its keys)
//   window_attn                    softmax attention over the last `window` positions (and, where asked for, the
//                                  sequence's first `keep_first` positions) with a per-head linear distance
//                                  penalty and / or a per-head sink in the denominator; optionally a sigmoid gate
//                                  on every output value.  `chunked`: over the positions of the token's own chunk
//                                  of `window` positions instead
//   qkv_headnorm_rotary_store      biases on q, k and v, an RMS norm with one weight for all heads on each head of q
//                                  and of k, rotation of both; keys and values into their pages; further columns of
//                                  the same projection cast to the activation type
//   qkv_norm_rotary_store          biases on q, k and v, RMS norms over ALL heads of q and of k at once, rotation of
//                                  both, values mixed with another layer's for the same token; keys and values into
//                                  their pages
// All of it in fp32; the activation type (bf16 or fp32) only concerns what goes to a projection or
// into the key/value pages.
#include "common.h"

namespace mv {

template <bool F32> struct ActS;
template <> struct ActS<true> {
    typedef float T;
    static __device__ __forceinline__ float ld(const float* p) { return *p; }
    static __device__ __forceinline__ void st(float* p, float v) { *p = v; }
};
template <> struct ActS<false> {
    typedef uint16_t T;
    static __device__ __forceinline__ float ld(const uint16_t* p) { return bf16_bits_to_f32(*p); }
    static __device__ __forceinline__ void st(uint16_t* p, float v) { *p = (uint16_t)f32_to_bf16_bits(v); }
};

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + expf(-v)); }
__device__ __forceinline__ float sigmoid_f(float v) { return 1.0f / (1.0f + expf(-v)); }

struct StepRows {
    const int* tok_row;    // [T] row of each token
    const int* tok_pos;    // [T] position of each token in its sequence
    const int* row_start;  // [B]
    const int* row_len;    // [B]
    const int* row_ctx;    // [B] tokens the sequence held before this step
    const int* row_slot;   // [B] state slot
};

constexpr int kMaxTaps = 16;

__global__ __launch_bounds__(256) void conv_silu_kernel(const float* in, int64_t ldi, const float* state,
                                                        const float* w, const float* bias, float* out, int64_t ldo,
                                                        StepRows r, int T, int C, int taps) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)T * C) return;
    const int t = (int)(i / C), c = (int)(i % C);
    const int b = r.tok_row[t];
    const int rel = t - r.row_start[b];
    const bool carried = r.row_ctx[b] > 0;
    const float* st = state + ((int64_t)r.row_slot[b] * (taps - 1)) * C + c;
    float acc = bias ? bias[c] : 0.f;
    for (int j = 0; j < taps; ++j) {
        const int src = rel - (taps - 1) + j;  // portion-relative index of the input under tap j
        float v;
        if (src >= 0) v = in[(int64_t)(t - (taps - 1) + j) * ldi + c];
        else v = carried ? st[(int64_t)(src + taps - 1) * C] : 0.f;
        acc = fmaf(w[(int64_t)c * taps + j], v, acc);
    }
    out[(int64_t)t * ldo + c] = silu_f(acc);
}

__global__ __launch_bounds__(256) void conv_state_update_kernel(const float* in, int64_t ldi, float* state,
                                                                StepRows r, int B, int C, int taps) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)B * C) return;
    const int b = (int)(i / C), c = (int)(i % C);
    const int keep = taps - 1, len = r.row_len[b], start = r.row_start[b];
    const bool carried = r.row_ctx[b] > 0;
    float* st = state + ((int64_t)r.row_slot[b] * keep) * C + c;
    float old[kMaxTaps];
    for (int s = 0; s < keep; ++s) old[s] = carried ? st[(int64_t)s * C] : 0.f;
    for (int s = 0; s < keep; ++s) {
        const int rel = len - keep + s;
        st[(int64_t)s * C] = rel >= 0 ? in[(int64_t)(start + rel) * ldi + c] : old[s + len];
    }
}

// The convolution four channels to a thread, for TAPS taps and 16-byte rows: a thread slides over kConvRun consecutive tokens,
// so an input is read once instead of once per tap, and nothing is divided per element.  Sums in the same order as above.
// 2048 tokens of 8448 channels (4 taps): 114 -> 36 us; 138 MB that have to move.
// Below kConvRunLeast outputs a thread's eight tokens are a longer chain than the launch of one thread per output: 64 tokens of
// 8448 channels 8.5 us that way and 10.2 here, 300 of 2304 9.2 and 10.1, 512 of 2304 11.6 and 10.3.
constexpr int kConvRun = 8;
constexpr int64_t kConvRunLeast = 5 << 18;

template <int TAPS>
__device__ __forceinline__ void load_taps(float (&wt)[4][TAPS], const float* w, int c) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < TAPS; ++j) wt[e][j] = w[(int64_t)(c + e) * TAPS + j];
}
template <int TAPS>
__device__ __forceinline__ f32x4_t conv_out(const float (&wt)[4][TAPS], const f32x4_t& bias, const f32x4_t (&x)[TAPS]) {
    f32x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float acc = bias[e];
#pragma unroll
        for (int j = 0; j < TAPS; ++j) acc = fmaf(wt[e][j], x[j][e], acc);
        o[e] = silu_f(acc);
    }
    return o;
}

template <int TAPS>
__global__ __launch_bounds__(256) void conv_silu_run_kernel(const float* in, int64_t ldi, const float* state, const float* w,
                                                            const float* bias, float* out, int64_t ldo, StepRows r, int T,
                                                            int C) {
    const int c = (blockIdx.x * 256 + threadIdx.x) * 4, t0 = blockIdx.y * kConvRun;
    if (c >= C) return;
    float wt[4][TAPS];
    load_taps<TAPS>(wt, w, c);
    const f32x4_t bs = bias ? *reinterpret_cast<const f32x4_t*>(bias + c) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    f32x4_t x[kConvRun + TAPS - 1];
#pragma unroll
    for (int i = 0; i < kConvRun + TAPS - 1; ++i)
        x[i] = *reinterpret_cast<const f32x4_t*>(in + (int64_t)min(max(t0 - (TAPS - 1) + i, 0), T - 1) * ldi + c);
#pragma unroll
    for (int i = 0; i < kConvRun; ++i) {
        const int t = t0 + i;
        if (t >= T) break;
        const int b = r.tok_row[t], rel = t - r.row_start[b];
        f32x4_t v[TAPS];
#pragma unroll
        for (int j = 0; j < TAPS; ++j) v[j] = x[i + j];
        if (rel < TAPS - 1) {       // the taps before the portion: what the row's slot keeps, or zero
            const bool carried = r.row_ctx[b] > 0;
            const float* st = state + ((int64_t)r.row_slot[b] * (TAPS - 1)) * C + c;
#pragma unroll
            for (int j = 0; j < TAPS - 1; ++j) {
                const int src = rel - (TAPS - 1) + j;
                if (src < 0)
                    v[j] = carried ? *reinterpret_cast<const f32x4_t*>(st + (int64_t)(src + TAPS - 1) * C) : f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        *reinterpret_cast<f32x4_t*>(out + (int64_t)t * ldo + c) = conv_out<TAPS>(wt, bs, v);
    }
}

// ... and, for steps of one token a row (decoding), a thread takes a row's tokens in turn and leaves the state behind
// them: one launch instead of two (one row of 8448 channels 5.2 + 4.7 -> 4.7 us).
template <int TAPS>
__device__ __forceinline__ void conv_silu_row(const float* in, int64_t ldi, float* state, const float* w, const float* bias,
                                              float* out, int64_t ldo, const StepRows& r, int C) {
    const int c = (blockIdx.x * 256 + threadIdx.x) * 4, b = blockIdx.y;
    if (c >= C) return;
    const int len = r.row_len[b], start = r.row_start[b];
    const bool carried = r.row_ctx[b] > 0;
    float* st = state + ((int64_t)r.row_slot[b] * (TAPS - 1)) * C + c;
    float wt[4][TAPS];
    load_taps<TAPS>(wt, w, c);
    const f32x4_t bs = bias ? *reinterpret_cast<const f32x4_t*>(bias + c) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    f32x4_t x[TAPS];
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j)
        x[j] = carried ? *reinterpret_cast<const f32x4_t*>(st + (int64_t)j * C) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int t = start; t < start + len; ++t) {
        x[TAPS - 1] = *reinterpret_cast<const f32x4_t*>(in + (int64_t)t * ldi + c);
        *reinterpret_cast<f32x4_t*>(out + (int64_t)t * ldo + c) = conv_out<TAPS>(wt, bs, x);
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) x[j] = x[j + 1];
    }
#pragma unroll
    for (int j = 0; j < TAPS - 1; ++j) *reinterpret_cast<f32x4_t*>(st + (int64_t)j * C) = x[j];
}
template <int TAPS>
__global__ __launch_bounds__(256) void conv_silu_row_kernel(const float* in, int64_t ldi, float* state, const float* w,
                                                            const float* bias, float* out, int64_t ldo, StepRows r, int C) {
    conv_silu_row<TAPS>(in, ldi, state, w, bias, out, ldo, r, C);
}

struct DecayArgs {     // raw step inputs [T, H] (rows ld apart) to gain = softplus, decay = e^(-e^a_log gain) and its logarithm
    const float *raw, *dt_bias, *a_log;
    int64_t ld;
    float *gain, *decay, *log_decay;
    int H;
};
__device__ __forceinline__ void step_decay(const DecayArgs& d, int64_t t, int h) {
    const float v = d.raw[t * d.ld + h] + d.dt_bias[h];
    const float dt = fmaxf(v, 0.f) + log1pf(expf(-fabsf(v)));  // log(1 + e^v), no clamp
    const int64_t i = t * d.H + h;
    d.gain[i] = dt;
    const float ld_ = -expf(d.a_log[h]) * dt;
    d.decay[i] = expf(ld_);
    if (d.log_decay) d.log_decay[i] = ld_;
}
__global__ __launch_bounds__(256) void softplus_decay_kernel(DecayArgs d, int T) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < T * d.H) step_decay(d, i / d.H, i % d.H);
}

// A decoding step's convolution and, in the workgroups behind the channels', the step gains and decays of the same projection:
// either is a launch of 4.6 us for what takes none, both 4.9 (one row, 8448 channels, 128 heads).
template <int TAPS>
__global__ __launch_bounds__(256) void conv_decay_row_kernel(const float* in, int64_t ldi, float* state, const float* w,
                                                             const float* bias, float* out, int64_t ldo, StepRows r, int C,
                                                             int conv_blocks, DecayArgs d) {
    if ((int)blockIdx.x < conv_blocks) {
        conv_silu_row<TAPS>(in, ldi, state, w, bias, out, ldo, r, C);
        return;
    }
    const int h = ((int)blockIdx.x - conv_blocks) * 256 + threadIdx.x, b = blockIdx.y;
    if (h >= d.H) return;
    const int len = r.row_len[b], start = r.row_start[b];
    for (int t = start; t < start + len; ++t) step_decay(d, t, h);
}

struct ScanArgs {
    const float *q, *k, *v, *decay, *gain, *skip;
    int64_t ldq, ldk, ldv, ld_decay, ld_gain, ldo;
    int q_div, k_div;
    float* state;
    float* out;
    StepRows r;
    int H, n, p, pt;
    int max_len;   // rows longer than this belong to the chunked form (0: every row is taken)
    // chunk mode (ch_start != NULL): blockIdx.z is a chunk of a long row, run from a zero state; what it
    // leaves goes to ds[chunk][head] instead of the slot
    const int *ch_start, *ch_len;
    float* ds;
};

// GATED: `decay` holds a forget gate per (token, head, state row) and the key is one minus it.
template <int MAXN, bool GATED = false>
__global__ __launch_bounds__(256) void scan_outer_kernel(ScanArgs a) {
    __shared__ float part[2][256];
    const int b = blockIdx.z, h = blockIdx.y, tid = threadIdx.x;
    const int PT = a.pt, NS = 256 / PT;
    const int cl = tid % PT, ng = tid / PT, c = blockIdx.x * PT + cl;
    const bool vc = c < a.p;
    const int npt = (a.n + NS - 1) / NS, n0 = ng * npt;
    const bool chunk = a.ch_start != nullptr;
    const int len = chunk ? a.ch_len[b] : a.r.row_len[b], start = chunk ? a.ch_start[b] : a.r.row_start[b];
    if (!chunk && a.max_len > 0 && len > a.max_len) return;   // the whole workgroup
    const bool carried = !chunk && a.r.row_ctx[b] > 0;
    float* sp = (chunk ? a.ds + (((int64_t)b * a.H + h) * a.n + n0) * a.p
                       : a.state + (((int64_t)a.r.row_slot[b] * a.H + h) * a.n + n0) * a.p) + c;
    float S[MAXN];
#pragma unroll
    for (int i = 0; i < MAXN; ++i) S[i] = (carried && vc && i < npt && n0 + i < a.n) ? sp[(int64_t)i * a.p] : 0.f;
    for (int t = 0; t < len; ++t) {
        const int64_t tok = start + t;
        const float vv = vc ? a.v[tok * a.ldv + (int64_t)h * a.p + c] : 0.f;
        const float* qp = a.q + tok * a.ldq + (int64_t)(h / a.q_div) * a.n + n0;
        float o = 0.f;
        if (GATED) {
            const float* fp = a.decay + tok * a.ld_decay + (int64_t)h * a.n + n0;
#pragma unroll
            for (int i = 0; i < MAXN; ++i) {
                if (i < npt && n0 + i < a.n) {
                    const float f = fp[i];
                    S[i] = fmaf(1.0f - f, vv, f * S[i]);
                    o = fmaf(S[i], qp[i], o);
                }
            }
        } else {
            const float dec = a.decay[tok * a.ld_decay + h];
            const float g = a.gain ? a.gain[tok * a.ld_gain + h] : 1.0f;
            const float gv = g * vv;
            const float* kp = a.k + tok * a.ldk + (int64_t)(h / a.k_div) * a.n + n0;
#pragma unroll
            for (int i = 0; i < MAXN; ++i) {
                if (i < npt && n0 + i < a.n) {
                    S[i] = fmaf(kp[i], gv, dec * S[i]);
                    o = fmaf(S[i], qp[i], o);
                }
            }
        }
        part[t & 1][tid] = o;
        __syncthreads();
        if (ng == 0 && vc) {
            float tot = 0.f;
            for (int j = 0; j < NS; ++j) tot += part[t & 1][j * PT + cl];
            if (a.skip) tot = fmaf(a.skip[h], vv, tot);
            a.out[tok * a.ldo + (int64_t)h * a.p + c] = tot;
        }
    }
    if (vc) {
#pragma unroll
        for (int i = 0; i < MAXN; ++i)
            if (i < npt && n0 + i < a.n) sp[(int64_t)i * a.p] = S[i];
    }
}

// The recurrence token by token for the usual shapes (n of 16 NR, p a multiple of 64, 16-byte rows): a workgroup takes 64
// columns of a (row, head), a thread four of them over NR state rows, all of whose loads are in flight together; the form
// above asks for its values one by one behind a test of every row.  A decoded token is one trip for the state, k, q and v
// and one write: 128 heads of 128 x 64, one row 15.5 -> 7.0 us, 8 MB that
// have to move; 32 rows 64.5 -> 25.1; 12 tokens of one row 50.7 -> 14.2.
template <int NR>
__global__ __launch_bounds__(256) void scan_outer_vec_kernel(ScanArgs a) {
    __shared__ __attribute__((aligned(16))) float part[2][4][64];
    const int b = blockIdx.z, h = blockIdx.y, tid = threadIdx.x, wv = tid >> 6;
    const int c = blockIdx.x * 64 + 4 * (tid & 15), n0 = NR * (tid >> 4);
    const int len = a.r.row_len[b], start = a.r.row_start[b];
    if (a.max_len > 0 && len > a.max_len) return;   // the whole workgroup
    float* sp = a.state + (((int64_t)a.r.row_slot[b] * a.H + h) * a.n + n0) * a.p + c;
    const bool carried = a.r.row_ctx[b] > 0;
    f32x4_t S[NR], kq[NR / 4], qq[NR / 4], v;
    float dec, gain = 1.f;
    auto fetch = [&](int64_t tok) {
        const float* kp = a.k + tok * a.ldk + (int64_t)(h / a.k_div) * a.n + n0;
        const float* qp = a.q + tok * a.ldq + (int64_t)(h / a.q_div) * a.n + n0;
#pragma unroll
        for (int i = 0; i < NR / 4; ++i) {
            kq[i] = *reinterpret_cast<const f32x4_t*>(kp + 4 * i);
            qq[i] = *reinterpret_cast<const f32x4_t*>(qp + 4 * i);
        }
        v = *reinterpret_cast<const f32x4_t*>(a.v + tok * a.ldv + (int64_t)h * a.p + c);
        dec = a.decay[tok * a.ld_decay + h];
        if (a.gain) gain = a.gain[tok * a.ld_gain + h];
    };
    if (len > 0) fetch(start);
#pragma unroll
    for (int i = 0; i < NR; ++i) S[i] = carried ? *reinterpret_cast<const f32x4_t*>(sp + (int64_t)i * a.p) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int t = 0; t < len; ++t) {
        const f32x4_t gv = gain * v, vt = v;
        f32x4_t o = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NR; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                S[i][e] = fmaf(kq[i / 4][i % 4], gv[e], dec * S[i][e]);
                o[e] = fmaf(S[i][e], qq[i / 4][i % 4], o[e]);
            }
        if (t + 1 < len) fetch(start + t + 1);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[e] += __shfl_xor(o[e], 16, 64);
            o[e] += __shfl_xor(o[e], 32, 64);
        }
        if ((tid & 63) < 16) *reinterpret_cast<f32x4_t*>(&part[t & 1][wv][4 * (tid & 15)]) = o;
        __syncthreads();
        if (tid < 16) {
            o = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < 4; ++w) o += *reinterpret_cast<const f32x4_t*>(&part[t & 1][w][4 * tid]);
            if (a.skip) {
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = fmaf(a.skip[h], vt[e], o[e]);
            }
            *reinterpret_cast<f32x4_t*>(a.out + (int64_t)(start + t) * a.ldo + (int64_t)h * a.p + c) = o;
        }
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) *reinterpret_cast<f32x4_t*>(sp + (int64_t)i * a.p) = S[i];
}

// ---- the same recurrence in chunks of 64 tokens, for rows long enough to pay for three launches ----
// Within a chunk that starts from state S0, with L_t the running sum of log decay over the chunk:
//   o_t = exp(L_t) S0^T q_t + sum_{s<=t} exp(L_t - L_s) gain_s (q_t . k_s) v_s
//   S_end = exp(L_end) S0 + sum_s exp(L_end - L_s) gain_s k_s v_s^T
// intra:  per (chunk, head)  the second term of o, the sum of S_end (dS) and exp(L_end), L_t kept
// carry:  per (row, head)    S0 of every chunk in turn (left where dS was), the row's final state
// inter:  per (chunk, head)  o_t += exp(L_t) S0^T q_t (+ skip_h v_t)
// fp32 throughout; differs from the token-by-token form by the order of the sums only.
constexpr int kCh = 64;

struct ChunkArgs {
    const float *q, *k, *v, *log_decay, *gain, *skip;
    int64_t ldq, ldk, ldv, ld_ld, ld_gain, ldo;
    int q_div, k_div;
    float* state;
    float* out;
    float* ds;     // [chunks, H, n, p]
    float* lsum;   // [tokens, H]  L_t
    float* atot;   // [chunks, H]  exp(L_end)
    const int *ch_start, *ch_len, *row_ch0, *row_nch;
    StepRows r;
    int H, n, p;
    int hb;   // heads of one group a workgroup takes in turn (they share q, k and the products q . k)
};

// All three products of a chunk run on v_mfma_f32_16x16x4_f32 (true fp32): operand A lane (r, g) = A[r][g],
// operand B lane (r, g) = B[g][r], result lane (r, g) = C[4 g + j][r] (r = lane % 16, g = lane / 16).
#define MV_MFMA4(acc, a_, b_) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a_, b_, acc, 0, 0, 0)

__global__ __launch_bounds__(256) void scan_chunk_intra_kernel(ChunkArgs a) {
    extern __shared__ float lds[];
    const int ch = blockIdx.x, tid = threadIdx.x;
    const int wv = tid >> 6, r = tid & 15, qd = (tid & 63) >> 4;
    const int n = a.n, p = a.p, n4 = (n + 3) & ~3, sn = n4 + 1, sp = p + 1;
    float* qs = lds;
    float* ks = qs + kCh * sn;
    float* vs = ks + kCh * sn;
    float* Ls = vs + kCh * sp;
    float* gs = Ls + kCh;
    float* ws = gs + kCh;
    const int start = a.ch_start[ch], len = a.ch_len[ch];
    // a.hb heads of one group per workgroup: they share q and k, staged once, and the products q_t . k_s
    const int h_first = blockIdx.y * a.hb;
    for (int i = tid; i < kCh * n4; i += 256) {
        const int t = i / n4, j = i % n4;
        const bool ok = t < len && j < n;
        qs[t * sn + j] = ok ? a.q[(int64_t)(start + t) * a.ldq + (int64_t)(h_first / a.q_div) * n + j] : 0.f;
        ks[t * sn + j] = ok ? a.k[(int64_t)(start + t) * a.ldk + (int64_t)(h_first / a.k_div) * n + j] : 0.f;
    }
    __syncthreads();
    // wave wv owns the tokens t = 16 wv + r.  P0[nt][j] = q_t . k_s, s = 16 nt + 4 qd + j, s-tiles above the
    // diagonal stay zero: A = k rows of the s-tile, B = q rows of the wave's tokens, summed over the state index
    const int t0 = 16 * wv, t = t0 + r;
    f32x4_t P0[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) P0[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int j0 = 0; j0 < n4; j0 += 4) {
        const float bq = qs[t * sn + j0 + qd];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
            if (nt <= wv) MV_MFMA4(P0[nt], ks[(16 * nt + r) * sn + j0 + qd], bq);
    }
    for (int hh = 0; hh < a.hb; ++hh) {
        const int h = h_first + hh;
        __syncthreads();   // the head before is done with vs, Ls, gs, ws
        for (int i = tid; i < kCh * p; i += 256) {
            const int tt = i / p, c = i % p;
            vs[tt * sp + c] = tt < len ? a.v[(int64_t)(start + tt) * a.ldv + (int64_t)h * p + c] : 0.f;
        }
        if (tid < kCh) {   // one wave: inclusive running sum of the log decays
            float l = 0.f, g = 0.f;
            if (tid < len) {
                l = fmaxf(a.log_decay[(int64_t)(start + tid) * a.ld_ld + h], -80.f);
                g = a.gain ? a.gain[(int64_t)(start + tid) * a.ld_gain + h] : 1.f;
            }
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const float up = __shfl_up(l, o, 64);
                if (tid >= o) l += up;
            }
            Ls[tid] = l;
            gs[tid] = g;
            if (tid < len) a.lsum[(int64_t)(start + tid) * a.H + h] = l;
            const float lend = __shfl(l, len - 1, 64);
            ws[tid] = expf(lend - l) * g;        // weight of token s in the state the chunk ends with
            if (tid == 0) a.atot[(int64_t)ch * a.H + h] = expf(lend);
        }
        __syncthreads();
        f32x4_t P[4];
        {
            const float Lt = Ls[t];
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int s_ = 16 * nt + 4 * qd + j;
                    P[nt][j] = (s_ <= t) ? P0[nt][j] * expf(Lt - Ls[s_]) * gs[s_] : 0.f;
                }
        }
        // o[t][c] = sum_s P[t][s] v[s][c]: A = v^T (columns c), B = P straight from the registers
        for (int c0 = 0; c0 < p; c0 += 64) {
            f32x4_t o[4];
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) o[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int nt = 0; nt < 4; ++nt) {
                if (nt > wv) continue;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float* vrow = vs + (16 * nt + 4 * qd + j) * sp;
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct) {
                        const int c = c0 + 16 * ct + r;
                        MV_MFMA4(o[ct], c < p ? vrow[c] : 0.f, P[nt][j]);
                    }
                }
            }
            if (t < len) {
#pragma unroll
                for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int c = c0 + 16 * ct + 4 * qd + j;
                        if (c < p) a.out[(int64_t)(start + t) * a.ldo + (int64_t)h * p + c] = o[ct][j];
                    }
            }
        }
        // dS[j][c] = sum_s (k[s][j] ws[s]) v[s][c]: A = k^T weighted as it is read, B = v, over the tokens
        float* dsp = a.ds + ((int64_t)ch * a.H + h) * n * p;
        for (int jt = wv; jt * 16 < n; jt += 4) {
            const int ja = 16 * jt + r;
            for (int c0 = 0; c0 < p; c0 += 64) {
                f32x4_t dd[4];
#pragma unroll
                for (int ct = 0; ct < 4; ++ct) dd[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                for (int s0 = 0; s0 < kCh; s0 += 4) {
                    const float ak = ja < n4 ? ks[(s0 + qd) * sn + ja] * ws[s0 + qd] : 0.f;
                    const float* vrow = vs + (s0 + qd) * sp;
#pragma unroll
                    for (int ct = 0; ct < 4; ++ct) {
                        const int c = c0 + 16 * ct + r;
                        MV_MFMA4(dd[ct], ak, c < p ? vrow[c] : 0.f);
                    }
                }
#pragma unroll
                for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int jj = 16 * jt + 4 * qd + j, c = c0 + 16 * ct + r;
                        if (jj < n && c < p) dsp[(int64_t)jj * p + c] = dd[ct][j];
                    }
            }
        }
    }
}

__global__ __launch_bounds__(256) void scan_chunk_carry_kernel(ChunkArgs a) {
    const int b = blockIdx.z, h = blockIdx.y;
    const int np = a.n * a.p, e = blockIdx.x * 256 + threadIdx.x;
    const int nch = a.row_nch[b];
    if (nch == 0 || e >= np) return;
    float* sp = a.state + ((int64_t)a.r.row_slot[b] * a.H + h) * np + e;
    float S = a.r.row_ctx[b] > 0 ? *sp : 0.f;
    const int c0 = a.row_ch0[b];
    for (int c = c0; c < c0 + nch; ++c) {
        float* d = a.ds + ((int64_t)c * a.H + h) * np + e;
        const float add = *d;
        *d = S;                                   // the state this chunk starts from
        S = fmaf(a.atot[(int64_t)c * a.H + h], S, add);
    }
    *sp = S;
}

__global__ __launch_bounds__(256) void scan_chunk_inter_kernel(ChunkArgs a) {
    extern __shared__ float lds[];
    const int ch = blockIdx.x, tid = threadIdx.x;
    const int wv = tid >> 6, r = tid & 15, qd = (tid & 63) >> 4;
    const int n = a.n, p = a.p, n4 = (n + 3) & ~3, sn = n4 + 1, sp = p + 1;
    float* qs = lds;
    float* Ss = qs + kCh * sn;
    const int start = a.ch_start[ch], len = a.ch_len[ch];
    const int h_first = blockIdx.y * a.hb;
    for (int i = tid; i < kCh * n4; i += 256) {
        const int t = i / n4, j = i % n4;
        qs[t * sn + j] =
            (t < len && j < n) ? a.q[(int64_t)(start + t) * a.ldq + (int64_t)(h_first / a.q_div) * n + j] : 0.f;
    }
    const int t = 16 * wv + r;
    for (int hh = 0; hh < a.hb; ++hh) {
        const int h = h_first + hh;
        __syncthreads();
        const float* dsp = a.ds + ((int64_t)ch * a.H + h) * n * p;
        for (int i = tid; i < n4 * p; i += 256) Ss[(i / p) * sp + i % p] = i < n * p ? dsp[i] : 0.f;
        __syncthreads();
        // o[t][c] += exp(L_t) sum_j q[t][j] S0[j][c]: A = S0^T (columns c), B = q rows of the wave's tokens
        const float sk = a.skip ? a.skip[h] : 0.f;
        const float w = t < len ? expf(a.lsum[(int64_t)(start + t) * a.H + h]) : 0.f;
        for (int c0 = 0; c0 < p; c0 += 64) {
            f32x4_t o[4];
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) o[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            for (int j0 = 0; j0 < n4; j0 += 4) {
                const float bq = qs[t * sn + j0 + qd];
                const float* srow = Ss + (j0 + qd) * sp;
#pragma unroll
                for (int ct = 0; ct < 4; ++ct) {
                    const int c = c0 + 16 * ct + r;
                    MV_MFMA4(o[ct], c < p ? srow[c] : 0.f, bq);
                }
            }
            if (t < len) {
#pragma unroll
                for (int ct = 0; ct < 4; ++ct)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int c = c0 + 16 * ct + 4 * qd + j;
                        if (c >= p) continue;
                        float* op = a.out + (int64_t)(start + t) * a.ldo + (int64_t)h * p + c;
                        float res = fmaf(w, o[ct][j], *op);
                        if (a.skip) res = fmaf(sk, a.v[(int64_t)(start + t) * a.ldv + (int64_t)h * p + c], res);
                        *op = res;
                    }
            }
        }
    }
}

// The same in two launches for the usual shapes (n of 64 or 128, p a multiple of 16, 16-byte rows), without the chunks'
// states in memory.  The columns of a state do not meet, so one workgroup takes a (row, head, 16 CT columns) through all of
// the row's chunks, its slice of S in registers:
//   scores  q_t . k_s of every chunk once per group of heads (they were formed once per four heads)
//   scan    waves 0 - 3 (one per 16 tokens): o_t = exp(L_t) S0^T q_t + sum_s P[t][s] v_s (+ skip v_t); waves 4 - 7: the n rows
//           of S = exp(L_end) S0 + k^T (w v).  The two kinds run side by side, one of each to a SIMD: S0 goes to the others
//           through LDS, two buffers, one barrier a chunk; the next chunk's q, k and scores are in flight to registers.
// The contraction index of a product is dealt out as 16 a + 4 g + e (e: step of the instruction), so a lane's operands of
// four steps are one 16-byte read.  What a chunk adds to the state, and its own part of an output, have accumulators of their own:
// rounded at the state's size sixteen times a chunk, states were three times as far from 64 bits.  A chunk takes a SIMD 160 of
// the fp32 instruction at 32 cycles (2.1 us at 32 columns) and measures 4.2: sums that wait for each other, exponentials, the
// barrier.  16 columns a workgroup, two workgroups to a unit, read q and k twice as often: 203 against 155 us when that was tried.
// Both launches, against the three above with the chunks' states written, carried and read back (us, n = 128, p = 64): 128 heads
// in one group, 2048 tokens 693 -> 136; 100 tokens 188 -> 18; 16 heads with q and k of their own, 2048 tokens 153 -> 111, 333
// tokens 71 -> 31; 24 heads, n = 64, 65 + 65 + 65 + 900 tokens 70 -> 55.
__global__ __launch_bounds__(256) void scan_scores_kernel(ChunkArgs a, float* scores) {
    const int ch = blockIdx.x, grp = blockIdx.y, tt = blockIdx.z;
    const int st = threadIdx.x >> 6, r = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    if (st > tt) return;
    const int start = a.ch_start[ch], last = a.ch_len[ch] - 1;
    const int tq = min(16 * tt + r, last), ts = min(16 * st + r, last);    // (tokens past the end: masked where they are read)
    const float* qp = a.q + (int64_t)(start + tq) * a.ldq + (int64_t)grp * a.n + 4 * g;
    const float* kp = a.k + (int64_t)(start + ts) * a.ldk + (int64_t)grp * a.n + 4 * g;
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < a.n; j += 64) {
        f32x4_t x[4], y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i] = *reinterpret_cast<const f32x4_t*>(qp + j + 16 * i);
            y[i] = *reinterpret_cast<const f32x4_t*>(kp + j + 16 * i);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) MV_MFMA4(acc, x[i][e], y[i][e]);
    }
    float* o = scores + ((int64_t)ch * gridDim.y + grp) * kCh * kCh + (16 * tt + 4 * g) * kCh + 16 * st + r;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j * kCh] = acc[j];
}

template <int NJ, int CT>   // n / 16, column tiles of 16
__global__ __launch_bounds__(512) void scan_rows_kernel(ChunkArgs a, const float* scores, int groups) {
    constexpr int n = 16 * NJ, BC = 16 * CT, SV = kCh + 4, SS = n + 4, JW = NJ / 4;
    __shared__ __attribute__((aligned(16))) float vt[2][BC * SV];       // [column][token]
    __shared__ __attribute__((aligned(16))) float s0[2][BC * SS];       // [column][state row]
    __shared__ __attribute__((aligned(16))) float Ls[2][kCh], gs[2][kCh], ws[2][kCh], el[2][kCh];
    __shared__ float at[2];
    const int blocks = a.p / BC, h = blockIdx.x / blocks, c0 = (blockIdx.x % blocks) * BC, b = blockIdx.y;
    const int nch = a.row_nch[b], ch0 = a.row_ch0[b];
    if (nch == 0) return;
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, g = lane >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);    // (a scalar: the two kinds of wave branch, they do not mask)
    const int grp = h / a.q_div, np = n * a.p;
    float* sp = a.state + ((int64_t)a.r.row_slot[b] * a.H + h) * np + c0;
    const float* qb = a.q + (int64_t)grp * n;
    const float* kb = a.k + (int64_t)grp * n;
    const float* vb = a.v + (int64_t)h * a.p + c0;

    // The workgroup's part of v and the decays of a chunk: requested two chunks ahead, staged one ahead.  (Loads stay plain
    // requests until they are used: arithmetic on them here would wait for them.)
    f32x4_t vn;
    float ldn = 0.f, gn = 1.f;
    const int vs_ = tid / (BC / 4), vc_ = 4 * (tid % (BC / 4));     // token and first column of this thread's piece of v
    auto fetch_v = [&](int start, int len) {
        vn = *reinterpret_cast<const f32x4_t*>(vb + (int64_t)(start + min(vs_, len - 1)) * a.ldv + vc_);
        if (wv == 0) {
            const int64_t t = start + min(lane, len - 1);
            ldn = a.log_decay[t * a.ld_ld + h];
            if (a.gain) gn = a.gain[t * a.ld_gain + h];
        }
    };
    auto stage = [&](int buf, int len) {
        if (vs_ < kCh)
#pragma unroll
            for (int i = 0; i < 4; ++i) vt[buf][(vc_ + i) * SV + vs_] = vs_ < len ? vn[i] : 0.f;
        if (wv == 0) {      // inclusive running sum of the log decays
            float l = lane < len ? fmaxf(ldn, -80.f) : 0.f;
            const float gain = lane < len ? gn : 0.f;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const float up = __shfl_up(l, o, 64);
                if (lane >= o) l += up;
            }
            const float lend = __shfl(l, len - 1, 64);
            Ls[buf][lane] = l;
            gs[buf][lane] = gain;
            ws[buf][lane] = expf(lend - l) * gain;    // weight of token s in the state the chunk ends with
            el[buf][lane] = expf(l);
            if (lane == 0) at[buf] = expf(lend);
        }
    };
    // chunk c of the row (past the end: the last)
    const int* cs = a.ch_start + ch0;
    const int* cl = a.ch_len + ch0;
    auto at_most = [&](int c) { return c < nch ? c : nch - 1; };
    int st0 = cs[0], ln0 = cl[0], st1 = cs[at_most(1)], ln1 = cl[at_most(1)];
    fetch_v(st0, ln0);
    if (wv < 4) {
        const int tt = wv;
        const float sk = a.skip ? a.skip[h] : 0.f;
        f32x4_t fr[NJ], pr[4];
        auto fetch = [&](int ch, int start, int len) {
            const float* qp = qb + (int64_t)(start + min(16 * tt + r, len - 1)) * a.ldq + 4 * g;
#pragma unroll
            for (int i = 0; i < NJ; ++i) fr[i] = *reinterpret_cast<const f32x4_t*>(qp + 16 * i);
            const float* pp = scores + ((int64_t)ch * groups + grp) * kCh * kCh + (16 * tt + r) * kCh + 4 * g;
#pragma unroll
            for (int i = 0; i < 4; ++i) pr[i] = *reinterpret_cast<const f32x4_t*>(pp + 16 * (i <= tt ? i : tt));
        };
        fetch(ch0, st0, ln0);
        stage(0, ln0);
        fetch_v(st1, ln1);
        __syncthreads();
        for (int c = 0; c < nch; ++c) {
            const int buf = c & 1, start = st0, len = ln0;
            f32x4_t now[NJ], sc[4];
#pragma unroll
            for (int i = 0; i < NJ; ++i) now[i] = fr[i];
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[i] = pr[i];
            st0 = st1, ln0 = ln1;
            st1 = cs[at_most(c + 2)], ln1 = cl[at_most(c + 2)];
            fetch(ch0 + at_most(c + 1), st0, ln0);
            f32x4_t o[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) o[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < NJ; ++i) {
                f32x4_t y[CT];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) y[ct] = *reinterpret_cast<const f32x4_t*>(&s0[buf][(16 * ct + r) * SS + 16 * i + 4 * g]);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) MV_MFMA4(o[ct], now[i][e], y[ct][e]);
            }
            f32x4_t in[CT];      // the chunk's own tokens, apart: their sums are rounded at their own size
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) in[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            const float Lt = Ls[buf][16 * tt + r];
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                if (st > tt) break;
                const f32x4_t L4 = *reinterpret_cast<const f32x4_t*>(&Ls[buf][16 * st + 4 * g]);
                const f32x4_t g4 = *reinterpret_cast<const f32x4_t*>(&gs[buf][16 * st + 4 * g]);
                f32x4_t P, y[CT];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool seen = st < tt || 4 * g + e <= r;
                    P[e] = seen ? sc[st][e] * expf(Lt - L4[e]) * g4[e] : 0.f;
                }
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) y[ct] = *reinterpret_cast<const f32x4_t*>(&vt[buf][(16 * ct + r) * SV + 16 * st + 4 * g]);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) MV_MFMA4(in[ct], P[e], y[ct][e]);
            }
            const f32x4_t w = *reinterpret_cast<const f32x4_t*>(&el[buf][16 * tt + 4 * g]);
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
#pragma unroll
                for (int j = 0; j < 4; ++j) o[ct][j] = fmaf(w[j], o[ct][j], in[ct][j]);
                const f32x4_t v4 = *reinterpret_cast<const f32x4_t*>(&vt[buf][(16 * ct + r) * SV + 16 * tt + 4 * g]);
                float* op = a.out + (int64_t)(start + 16 * tt + 4 * g) * a.ldo + (int64_t)h * a.p + c0 + 16 * ct + r;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (16 * tt + 4 * g + j < len) op[j * a.ldo] = a.skip ? fmaf(sk, v4[j], o[ct][j]) : o[ct][j];
            }
            stage(buf ^ 1, ln0);
            fetch_v(st1, ln1);
            __syncthreads();
        }
    } else {
        const int j0 = 16 * JW * (wv - 4);       // first of this wave's state rows
        f32x4_t S[JW][CT], fr[NJ];               // S: rows j0 + 16 i + 4 g .. + 3, column 16 ct + r
        auto fetch = [&](int start, int len) {
#pragma unroll
            for (int st = 0; st < 4; ++st)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float* kp = kb + (int64_t)(start + min(16 * st + 4 * g + e, len - 1)) * a.ldk + j0 + r;
#pragma unroll
                    for (int i = 0; i < JW; ++i) fr[4 * i + st][e] = kp[16 * i];
                }
        };
        auto publish = [&](int buf) {
#pragma unroll
            for (int i = 0; i < JW; ++i)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
                    *reinterpret_cast<f32x4_t*>(&s0[buf][(16 * ct + r) * SS + j0 + 16 * i + 4 * g]) = S[i][ct];
        };
        fetch(st0, ln0);
        const bool carried = a.r.row_ctx[b] > 0;
#pragma unroll
        for (int i = 0; i < JW; ++i)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    S[i][ct][j] = carried ? sp[(int64_t)(j0 + 16 * i + 4 * g + j) * a.p + 16 * ct + r] : 0.f;
        publish(0);
        stage(0, ln0);
        fetch_v(st1, ln1);
        __syncthreads();
        for (int c = 0; c < nch; ++c) {
            const int buf = c & 1, len = ln0;
            f32x4_t now[NJ];
#pragma unroll
            for (int i = 0; i < NJ; ++i) now[i] = fr[i];
            if (len < kCh) {     // (uniform) past the end the last token was read again: its weight is zero, but it may be infinite
#pragma unroll
                for (int st = 0; st < 4; ++st)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int i = 0; i < JW; ++i)
                            if (16 * st + 4 * g + e >= len) now[4 * i + st][e] = 0.f;
            }
            st0 = st1, ln0 = ln1;
            st1 = cs[at_most(c + 2)], ln1 = cl[at_most(c + 2)];
            fetch(st0, ln0);
            const float keep = at[buf];
            f32x4_t add[JW][CT];     // what the chunk adds, apart: summed into S one by one its parts would each be rounded at S's size
#pragma unroll
            for (int i = 0; i < JW; ++i)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) add[i][ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < 4; ++st) {
                const f32x4_t w4 = *reinterpret_cast<const f32x4_t*>(&ws[buf][16 * st + 4 * g]);
                f32x4_t y[CT];
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
                    y[ct] = *reinterpret_cast<const f32x4_t*>(&vt[buf][(16 * ct + r) * SV + 16 * st + 4 * g]) * w4;
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < JW; ++i)
#pragma unroll
                        for (int ct = 0; ct < CT; ++ct) MV_MFMA4(add[i][ct], now[4 * i + st][e], y[ct][e]);
            }
#pragma unroll
            for (int i = 0; i < JW; ++i)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int j = 0; j < 4; ++j) S[i][ct][j] = fmaf(keep, S[i][ct][j], add[i][ct][j]);
            publish(buf ^ 1);
            stage(buf ^ 1, ln0);
            fetch_v(st1, ln1);
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < JW; ++i)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int j = 0; j < 4; ++j) sp[(int64_t)(j0 + 16 * i + 4 * g + j) * a.p + 16 * ct + r] = S[i][ct][j];
    }
}

// ---- the gated recurrence in chunks of 64 tokens ----
// Within a chunk that starts from state S0, with P_t[i] the product of the gates f_s[i] over the chunk's tokens
// s <= t:  o_t = (local run from a zero state)_t + sum_i q_t[i] P_t[i] S0[i][:],  S_end = diag(P_end) S0 + local.
//   gate_cumprod   P_t for every token of every chunk
//   scan_outer_kernel in chunk mode: the local runs, all chunks side by side
//   gated_carry    per (row, head): the state each chunk starts from, in turn (left where the local sum was),
//                  and the row's final state
//   gated_inter    o_t += (q_t * P_t) S0, a [64 x n] . [n x p] product per (chunk, head) in fp32
// Products of gates, no logarithms: a gate of exactly zero or one is exact, long decays underflow to zero as
// the token-by-token run does.
__global__ __launch_bounds__(256) void gate_cumprod_kernel(const float* f, int64_t ldf, float* cum, int64_t ldc,
                                                           const int* ch_start, const int* ch_len, int width) {
    const int ch = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
    if (c >= width) return;
    const int start = ch_start[ch], len = ch_len[ch];
    float pr = 1.0f;
    for (int t = 0; t < len; ++t) {
        pr *= f[(int64_t)(start + t) * ldf + c];
        cum[(int64_t)(start + t) * ldc + c] = pr;
    }
}

struct GatedChunkArgs {
    const float* q;
    const float* cum;
    int64_t ldq, ldc, ldo;
    float* state;
    float* out;
    float* ds;
    const int *ch_start, *ch_len, *row_ch0, *row_nch, *row_ctx, *row_slot;
    int H, n, p;
};

__global__ __launch_bounds__(256) void gated_carry_kernel(GatedChunkArgs a) {
    const int b = blockIdx.z, h = blockIdx.y;
    const int np = a.n * a.p, e = blockIdx.x * 256 + threadIdx.x;
    const int nch = a.row_nch[b];
    if (nch == 0 || e >= np) return;
    const int i = e / a.p;
    float* sp = a.state + ((int64_t)a.row_slot[b] * a.H + h) * np + e;
    float S = a.row_ctx[b] > 0 ? *sp : 0.f;
    const int c0 = a.row_ch0[b];
    for (int c = c0; c < c0 + nch; ++c) {
        float* d = a.ds + ((int64_t)c * a.H + h) * np + e;
        const float add = *d;
        *d = S;                                   // the state this chunk starts from
        const int last = a.ch_start[c] + a.ch_len[c] - 1;
        S = fmaf(a.cum[(int64_t)last * a.ldc + (int64_t)h * a.n + i], S, add);
    }
    *sp = S;
}

// one workgroup per (chunk, head, 64 value columns): thread (ty, tx) owns 4 tokens x 4 columns
__global__ __launch_bounds__(256) void gated_inter_kernel(GatedChunkArgs a) {
    __shared__ float as[16][kCh + 4];
    __shared__ float ss[16][64 + 4];
    const int ch = blockIdx.x, h = blockIdx.y, c0 = blockIdx.z * 64;
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
    const int start = a.ch_start[ch], len = a.ch_len[ch];
    const float* S0 = a.ds + ((int64_t)ch * a.H + h) * a.n * a.p;
    const int lrow = tid >> 2, lcol = (tid & 3) * 4;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < a.n; k0 += 16) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int kk = k0 + lcol + i;
            const bool ok = lrow < len && kk < a.n;
            const int64_t tok = start + lrow;
            as[lcol + i][lrow] = ok ? a.q[tok * a.ldq + (int64_t)h * a.n + kk] * a.cum[tok * a.ldc + (int64_t)h * a.n + kk] : 0.f;
        }
        {   // the state tile: thread (k = tid / 16, four neighbouring columns)
            const int sk = k0 + (tid >> 4), sc = c0 + (tid & 15) * 4;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                ss[tid >> 4][(tid & 15) * 4 + i] = (sk < a.n && sc + i < a.p) ? S0[(int64_t)sk * a.p + sc + i] : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            float x[4], y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = as[kk][ty * 4 + i];
                y[i] = ss[kk][tx * 4 + i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(x[i], y[j], acc[i][j]);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int t = ty * 4 + i;
        if (t >= len) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int c = c0 + tx * 4 + j;
            if (c < a.p) a.out[(int64_t)(start + t) * a.ldo + (int64_t)h * a.p + c] += acc[i][j];
        }
    }
}

__global__ __launch_bounds__(256) void gate_lower_bound_kernel(float* q, int64_t ldq, float* f, int64_t ldf,
                                                               const float* bias, const float* lower, int T, int n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)T * n) return;
    const int t = (int)(i / n), c = (int)(i % n);
    float* qp = q + (int64_t)t * ldq + c;
    float* fp = f + (int64_t)t * ldf + c;
    *qp = silu_f(*qp);
    const float l = lower[c], z = *fp + (bias ? bias[c] : 0.f);
    *fp = fmaf(1.0f - l, 1.0f / (1.0f + expf(-z)), l);
}

__global__ __launch_bounds__(256) void rotary_pairs_kernel(float* x, int64_t ld, const double* inv_freq,
                                                           const int* tok_pos, int T, int heads, int dim, int rot,
                                                           float scale) {
    const int half = rot / 2, per = dim - half;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)T * heads * per) return;
    const int j = (int)(i % per), hh = (int)((i / per) % heads), t = (int)(i / ((int64_t)per * heads));
    float* p = x + (int64_t)t * ld + (int64_t)hh * dim;
    if (j < half) {
        const double ang = (double)tok_pos[t] * inv_freq[j];
        double sin_, cos_;
        sincos(ang, &sin_, &cos_);
        const float cs = (float)cos_, sn = (float)sin_;
        const float u = p[j], v = p[j + half];
        p[j] = (u * cs - v * sn) * scale;
        p[j + half] = (v * cs + u * sn) * scale;
    } else {
        p[j + half] *= scale;
    }
}

template <bool F32>
__global__ __launch_bounds__(256) void gated_group_norm_kernel(const float* y, int64_t ldy, const float* gate,
                                                               int64_t ldg, const float* w, void* out_, int64_t ldo,
                                                               int rows, int n, int groups, int mode,
                                                               int w_shared, float eps) {
    typedef typename ActS<F32>::T T;
    T* out = (T*)out_;
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (unit >= rows * groups) return;
    const int row = unit / groups, g = unit % groups, gs = n / groups;
    const float* yr = y + (int64_t)row * ldy + (int64_t)g * gs;
    const float* gr = gate + (int64_t)row * ldg + (int64_t)g * gs;
    float ss = 0.f;
    for (int c = lane; c < gs; c += 64) {
        const float u = mode == 1 ? yr[c] * silu_f(gr[c]) : yr[c];
        ss += u * u;
    }
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)gs + eps);
    for (int c = lane; c < gs; c += 64) {
        float u = mode == 1 ? (yr[c] * silu_f(gr[c])) * inv : (yr[c] * inv) * (mode == 2 ? sigmoid_f(gr[c]) : silu_f(gr[c]));
        if (w) u *= w[w_shared ? c : g * gs + c];
        ActS<F32>::st(out + (int64_t)row * ldo + (int64_t)g * gs + c, u);
    }
}

struct PagedRows {
    const int* tok_row;
    const int* tok_pos;
    const int* block_table;
    int bt_stride, page;
};

template <bool F32>
__global__ __launch_bounds__(256) void qk_unitnorm_store_kernel(float* qkv, int64_t ld, void* kc_, void* vc_,
                                                                PagedRows pr, int T, int H, int G, int d, int dv,
                                                                float eps) {
    typedef typename ActS<F32>::T T_;
    T_* kc = (T_*)kc_;
    T_* vc = (T_*)vc_;
    const int per = H + 2 * G;
    const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (unit >= (int64_t)T * per) return;
    const int t = (int)(unit / per), u = (int)(unit % per);
    float* row = qkv + (int64_t)t * ld;
    const int pos = pr.tok_pos[t];
    const int pg = pr.block_table[(int64_t)pr.tok_row[t] * pr.bt_stride + pos / pr.page];
    const int64_t slot = (int64_t)pg * pr.page + pos % pr.page;
    if (u < H + G) {
        float* p = row + (u < H ? (int64_t)u * d : (int64_t)H * d + (int64_t)(u - H) * d);
        float ss = 0.f;
        for (int c = lane; c < d; c += 64) ss += p[c] * p[c];
        ss = wave_sum(ss);
        const float inv = 1.0f / sqrtf(ss / (float)d + eps);
        if (u < H) {
            for (int c = lane; c < d; c += 64) p[c] = p[c] * inv;
        } else if (pg >= 0) {
            T_* dst = kc + (slot * G + (u - H)) * d;
            for (int c = lane; c < d; c += 64) ActS<F32>::st(dst + c, p[c] * inv);
        }
    } else if (pg >= 0) {
        const int g = u - H - G;
        const float* p = row + (int64_t)(H + G) * d + (int64_t)g * dv;
        T_* dst = vc + (slot * G + g) * dv;
        for (int c = lane; c < dv; c += 64) ActS<F32>::st(dst + c, p[c]);
    }
}

// One wave per (token, `hpw` consecutive query or key heads: the sines and cosines of a position are formed once for
// them).  q [T, ld]: heads * d query values then kv_heads * d key values, as one projection leaves them.  The query gets its bias and rotation in place; the key goes, with its bias, unrotated
// into the value page and rotated into the key page.  angle = position * inv_freq[i], formed in fp64.
template <bool F32>
__global__ __launch_bounds__(256) void qk_rotary_store_kernel(float* qk, int64_t ld, const float* qb, const float* kb,
                                                              void* kc_, void* vc_, const double* inv_freq,
                                                              PagedRows pr, int T, int H, int G, int d, int rot,
                                                              int adjacent, int hpw, unsigned rot_blocks, const float* act_in,
                                                              int64_t lda, void* act_out, int64_t ldao, int act_n,
                                                              int act_kind, float act_limit, float act_slope) {
    typedef typename ActS<F32>::T T_;
    if (blockIdx.x >= rot_blocks) {
        // the workgroups behind the rotation's: the gate of a feed-forward whose gate | up columns came out of the
        // same projection (a parallel layer), so that the step needs no launch of its own
        const unsigned b = blockIdx.x - rot_blocks, cb = (act_n + 255) / 256;
        const int64_t row = b / cb;
        const int c = (b % cb) * 256 + threadIdx.x;
        if (c < act_n)
            ActS<F32>::st((T_*)act_out + row * ldao + c,
                          gated_act_f(act_in[row * lda + c], act_in[row * lda + act_n + c], act_kind, act_limit, act_slope));
        return;
    }
    T_* kc = (T_*)kc_;
    T_* vc = (T_*)vc_;
    const int per = H + G, groups = (per + hpw - 1) / hpw;
    const int64_t unit = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (unit >= (int64_t)T * groups) return;
    const int t = (int)(unit / groups), u0 = (int)(unit % groups) * hpw, u1 = u0 + hpw < per ? u0 + hpw : per;
    const int pos = pr.tok_pos[t];
    float* row = qk + (int64_t)t * ld;
    int64_t slot = -1;            // the token's place in the pages (needed where the wave holds a key head)
    if (u1 > H) {
        const int pg = pr.block_table[(int64_t)pr.tok_row[t] * pr.bt_stride + pos / pr.page];
        if (pg >= 0) slot = ((int64_t)pg * pr.page + pos % pr.page) * G;
    }
    const int half = rot / 2;
    for (int i = lane; i < half; i += 64) {
        const int a = adjacent ? 2 * i : i, b = adjacent ? 2 * i + 1 : i + half;
        const double ang = (double)pos * inv_freq[i];
        double sin_, cos_;
        sincos(ang, &sin_, &cos_);          // once for all heads of the wave
        const float cs = (float)cos_, sn = (float)sin_;
        for (int u = u0; u < u1; ++u) {
            float* p = row + (int64_t)u * d;
            const float* bias = u < H ? (qb ? qb + (int64_t)u * d : nullptr) : (kb ? kb + (int64_t)(u - H) * d : nullptr);
            const float x0 = bias ? p[a] + bias[a] : p[a], x1 = bias ? p[b] + bias[b] : p[b];
            const float r0 = x0 * cs - x1 * sn, r1 = x1 * cs + x0 * sn;
            if (u < H) {
                p[a] = r0;
                p[b] = r1;
            } else if (slot >= 0) {
                T_* kdst = kc + (slot + (u - H)) * d;
                T_* vdst = vc + (slot + (u - H)) * d;
                ActS<F32>::st(kdst + a, r0);
                ActS<F32>::st(kdst + b, r1);
                ActS<F32>::st(vdst + a, x0);
                ActS<F32>::st(vdst + b, x1);
            }
        }
    }
    for (int u = u0; u < u1; ++u) {
        float* p = row + (int64_t)u * d;
        const float* bias = u < H ? (qb ? qb + (int64_t)u * d : nullptr) : (kb ? kb + (int64_t)(u - H) * d : nullptr);
        for (int c = rot + lane; c < d; c += 64) {
            const float x0 = bias ? p[c] + bias[c] : p[c];
            if (u < H) {
                p[c] = x0;
            } else if (slot >= 0) {
                ActS<F32>::st(kc + (slot + (u - H)) * d + c, x0);
                ActS<F32>::st(vc + (slot + (u - H)) * d + c, x0);
            }
        }
    }
}

// One workgroup per token.  qkv row: q [H * d] | k [G * d] | v [G * dv], as one projection leaves them.  Each of q and k gets
// its bias and an RMS norm over the WHOLE of it (plain weights; NULL: no norm), then the rotation of its heads' first
// `rot` dimensions (adjacent pairs or halves; the angle is formed in fp64, once per token for all heads); q stays in
// place, k goes to the key page.  v gets its bias; mix 1: v is kept in vfirst [T, G * dv]; mix 2: v = (1 - lam) v + lam
// vfirst; v goes to the value page.
template <bool F32>
__global__ __launch_bounds__(1024) void qkv_norm_rotary_store_kernel(float* qkv, int64_t ld, const float* qb,
                                                                    const float* kb, const float* vb, const float* qn,
                                                                    const float* kn, float eps, const double* inv_freq,
                                                                    float* vfirst, int mix, float lam, void* kc_,
                                                                    void* vc_, PagedRows pr, int H, int G, int d,
                                                                    int dv, int rot, int adjacent) {
    typedef typename ActS<F32>::T T_;
    extern __shared__ float ang[];     // [rot / 2] cosines, then sines
    __shared__ float red[32];
    T_* kc = (T_*)kc_;
    T_* vc = (T_*)vc_;
    const int t = blockIdx.x, tid = threadIdx.x, NT = blockDim.x, pos = pr.tok_pos[t];
    float* q = qkv + (int64_t)t * ld;
    float* k = q + (int64_t)H * d;
    const float* v = k + (int64_t)G * d;
    const int pg = pr.block_table[(int64_t)pr.tok_row[t] * pr.bt_stride + pos / pr.page];
    const int64_t slot = (int64_t)pg * pr.page + pos % pr.page;
    const int half = rot / 2;
    for (int i = tid; i < half; i += NT) {
        const double a = (double)pos * inv_freq[i];
        ang[i] = (float)cos(a);
        ang[half + i] = (float)sin(a);
    }
    float sq = 0.f, sk = 0.f;
    if (qn) {
#pragma unroll 4
        for (int c = tid; c < H * d; c += NT) {
            const float x = qb ? q[c] + qb[c] : q[c];
            sq += x * x;
        }
    }
    if (kn) {
#pragma unroll 4
        for (int c = tid; c < G * d; c += NT) {
            const float x = kb ? k[c] + kb[c] : k[c];
            sk += x * x;
        }
    }
    sq = wave_sum(sq);
    sk = wave_sum(sk);
    if ((tid & 63) == 0) {
        red[tid >> 6] = sq;
        red[16 + (tid >> 6)] = sk;
    }
    __syncthreads();
    sq = sk = 0.f;
    for (int i = 0; i < NT / 64; ++i) {
        sq += red[i];
        sk += red[16 + i];
    }
    const float iq = qn ? 1.0f / sqrtf(sq / (float)(H * d) + eps) : 1.f;
    const float ik = kn ? 1.0f / sqrtf(sk / (float)(G * d) + eps) : 1.f;
    const int per = d - half;         // a head's items: `half` rotated pairs, then the dimensions behind them
    for (int i = tid; i < (H + G) * per; i += NT) {
        const int u = i / per, j = i - u * per;
        const bool isq = u < H;
        const int base = isq ? u * d : (u - H) * d;
        float* src = isq ? q : k;
        const float* b = isq ? qb : kb;
        const float* w = isq ? qn : kn;
        const float inv = isq ? iq : ik;
        if (j < half) {
            const int a0 = base + (adjacent ? 2 * j : j), a1 = base + (adjacent ? 2 * j + 1 : j + half);
            float x0 = b ? src[a0] + b[a0] : src[a0], x1 = b ? src[a1] + b[a1] : src[a1];
            if (w) {
                x0 = (x0 * inv) * w[a0];
                x1 = (x1 * inv) * w[a1];
            }
            const float cs = ang[j], sn = ang[half + j];
            const float r0 = x0 * cs - x1 * sn, r1 = x1 * cs + x0 * sn;
            if (isq) {
                q[a0] = r0;
                q[a1] = r1;
            } else if (pg >= 0) {
                ActS<F32>::st(kc + slot * G * d + a0, r0);
                ActS<F32>::st(kc + slot * G * d + a1, r1);
            }
        } else {
            const int c = base + half + j;
            float x = b ? src[c] + b[c] : src[c];
            if (w) x = (x * inv) * w[c];
            if (isq) q[c] = x;
            else if (pg >= 0) ActS<F32>::st(kc + slot * G * d + c, x);
        }
    }
    for (int c = tid; c < G * dv; c += NT) {
        float x = vb ? v[c] + vb[c] : v[c];
        float* f = mix ? vfirst + (int64_t)t * G * dv + c : nullptr;
        if (mix == 1) *f = x;
        else if (mix == 2) x = (1.0f - lam) * x + lam * *f;
        if (pg >= 0) ActS<F32>::st(vc + slot * G * dv + c, x);
    }
}

// One wave per (token, `hpw` consecutive units): the H heads of q, the G heads of k, the G heads of v, then the cast columns.
// A head of q or k gets its bias, an RMS norm over itself (weights qn / kn [d], shared by the heads; NULL: no norm) and the
// rotation of its first `rot` dimensions (adjacent pairs or halves; the angle is formed in fp64 and brought into one turn
// there, once for the wave's heads); q stays in place, k goes to the key page.  v gets its bias and goes to the value page.
// A lane's items are the head's rotated pairs, then its other dimensions; NI: items per lane (d - rot / 2 <= 64 NI).
template <bool F32, int NI>
__global__ __launch_bounds__(256) void qkv_headnorm_rotary_store_kernel(float* qkv, int64_t ld, const float* qb,
                                                                        const float* kb, const float* vb,
                                                                        const float* qn, const float* kn, float eps,
                                                                        const double* inv_freq, void* kc_, void* vc_,
                                                                        PagedRows pr, int T, int H, int G, int d, int dv,
                                                                        int rot, int adjacent, int hpw, const float* low,
                                                                        int64_t ldl, void* low_out_, int low_n) {
    typedef typename ActS<F32>::T T_;
    T_* kc = (T_*)kc_;
    T_* vc = (T_*)vc_;
    const int units = H + 2 * G + (low_n > 0 ? 1 : 0), per = (units + hpw - 1) / hpw;
    const int64_t wave = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (wave >= (int64_t)T * per) return;
    const int t = (int)(wave / per), u0 = (int)(wave % per) * hpw, u1 = u0 + hpw < units ? u0 + hpw : units;
    float* row = qkv + (int64_t)t * ld;
    const int pos = pr.tok_pos[t];
    const int pg = pr.block_table[(int64_t)pr.tok_row[t] * pr.bt_stride + pos / pr.page];
    const int64_t slot = ((int64_t)pg * pr.page + pos % pr.page) * G;
    const int half = rot / 2, items = d - half;
    float cs[NI], sn[NI];
    if (u0 < H + G) {
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int j = lane + 64 * i;
            cs[i] = 1.f;
            sn[i] = 0.f;
            if (j < half) {
                const double turns = (double)pos * inv_freq[j] * 0.15915494309189533577;      // angle / 2 pi
                const float a = (float)((turns - rint(turns)) * 6.283185307179586477);
                sincosf(a, &sn[i], &cs[i]);
            }
        }
    }
    // a head's values and biases, requested while the head before it is worked on
    float n0[NI], n1[NI], m0[NI], m1[NI];
    auto fetch = [&](int u) {
        if (u >= u1 || u >= H + G) return;
        const float* x = row + (int64_t)u * d;       // q's heads, then k's
        const float* b = u < H ? (qb ? qb + (int64_t)u * d : nullptr) : (kb ? kb + (int64_t)(u - H) * d : nullptr);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int j = lane + 64 * i;
            n0[i] = n1[i] = m0[i] = m1[i] = 0.f;
            if (j >= items) continue;
            const int a0 = j < half ? (adjacent ? 2 * j : j) : half + j, a1 = adjacent ? 2 * j + 1 : j + half;
            n0[i] = x[a0];
            if (b) m0[i] = b[a0];
            if (j < half) {
                n1[i] = x[a1];
                if (b) m1[i] = b[a1];
            }
        }
    };
    fetch(u0);
    for (int u = u0; u < u1; ++u) {
        if (u < H + G) {
            const bool isq = u < H;
            float* x = row + (int64_t)u * d;
            const float* w = isq ? qn : kn;
            float x0[NI], x1[NI], ss = 0.f;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                x0[i] = n0[i] + m0[i];
                x1[i] = n1[i] + m1[i];
                ss += x0[i] * x0[i] + x1[i] * x1[i];
            }
            fetch(u + 1);
            float inv = 1.f;
            if (w) inv = 1.0f / sqrtf(wave_sum(ss) / (float)d + eps);
            T_* dst = kc + (slot + (u - H)) * d;
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int j = lane + 64 * i;
                if (j >= items) continue;
                const int a0 = j < half ? (adjacent ? 2 * j : j) : half + j;
                const int a1 = adjacent ? 2 * j + 1 : j + half;
                float y0 = w ? (x0[i] * inv) * w[a0] : x0[i], y1 = 0.f;
                if (j < half) {
                    y1 = w ? (x1[i] * inv) * w[a1] : x1[i];
                    const float r0 = y0 * cs[i] - y1 * sn[i];
                    y1 = y1 * cs[i] + y0 * sn[i];
                    y0 = r0;
                }
                if (isq) {
                    x[a0] = y0;
                    if (j < half) x[a1] = y1;
                } else if (pg >= 0) {
                    ActS<F32>::st(dst + a0, y0);
                    if (j < half) ActS<F32>::st(dst + a1, y1);
                }
            }
        } else if (u < H + 2 * G) {
            const int g = u - H - G;
            const float* x = row + (int64_t)(H + G) * d + (int64_t)g * dv;
            if (pg >= 0)
                for (int c = lane; c < dv; c += 64) ActS<F32>::st(vc + (slot + g) * dv + c, vb ? x[c] + vb[g * dv + c] : x[c]);
        } else {
            T_* lo = (T_*)low_out_ + (int64_t)t * low_n;
            for (int c = lane; c < low_n; c += 64) ActS<F32>::st(lo + c, low[(int64_t)t * ldl + c]);
        }
    }
}

// value of channel c at token t under a causal convolution of `taps` taps whose first inputs come from the slot
__device__ __forceinline__ float conv_at(const float* in, int64_t ldi, const float* state, const float* w,
                                         const StepRows& r, int t, int c, int C, int taps) {
    const int b = r.tok_row[t];
    const int rel = t - r.row_start[b];
    const bool carried = r.row_ctx[b] > 0;
    const float* st = state + ((int64_t)r.row_slot[b] * (taps - 1)) * C + c;
    float acc = 0.f;
    for (int j = 0; j < taps; ++j) {
        const int src = rel - (taps - 1) + j;
        float v;
        if (src >= 0) v = in[(int64_t)(t - (taps - 1) + j) * ldi + c];
        else v = carried ? st[(int64_t)(src + taps - 1) * C] : 0.f;
        acc = fmaf(w[(int64_t)c * taps + j], v, acc);
    }
    return acc;
}

template <bool F32>
__global__ __launch_bounds__(256) void conv_taps_kernel(const float* in, int64_t ldi, const float* state,
                                                        const float* w, float* o32, int64_t ld32, void* oact_,
                                                        int64_t ldoa, int add_input, StepRows r, int T, int C,
                                                        int taps) {
    typedef typename ActS<F32>::T T_;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)T * C) return;
    const int t = (int)(i / C), c = (int)(i % C);
    float v = conv_at(in, ldi, state, w, r, t, c, C, taps);
    if (add_input) v += in[(int64_t)t * ldi + c];
    if (o32) o32[(int64_t)t * ld32 + c] = v;
    if (oact_) ActS<F32>::st((T_*)oact_ + (int64_t)t * ldoa + c, v);
}

// columns [0, Cq) -> q (fp32), [Cq, Cq + Ck) -> the token's row of the key page, the last Cv -> the value page.
// w == NULL: no convolution, the columns go where they belong as they are
template <bool F32>
__global__ __launch_bounds__(256) void conv_qkv_store_kernel(const float* in, int64_t ldi, const float* state,
                                                             const float* w, float* q, int64_t ldq, void* kc_,
                                                             void* vc_, StepRows r, PagedRows pr, int T, int Cq,
                                                             int Ck, int Cv, int taps) {
    typedef typename ActS<F32>::T T_;
    const int C = Cq + Ck + Cv;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)T * C) return;
    const int t = (int)(i / C), c = (int)(i % C);
    const float v = w ? conv_at(in, ldi, state, w, r, t, c, C, taps) : in[(int64_t)t * ldi + c];
    if (c < Cq) {
        q[(int64_t)t * ldq + c] = v;
        return;
    }
    const int pos = pr.tok_pos[t];
    const int pg = pr.block_table[(int64_t)pr.tok_row[t] * pr.bt_stride + pos / pr.page];
    if (pg < 0) return;
    const int64_t slot = (int64_t)pg * pr.page + pos % pr.page;
    if (c < Cq + Ck) ActS<F32>::st((T_*)kc_ + slot * Ck + (c - Cq), v);
    else ActS<F32>::st((T_*)vc_ + slot * Cv + (c - Cq - Ck), v);
}

constexpr int kMaxVC = 4;  // value columns per lane: vdim <= 256

// the first position a query at `pos` sees: `size` positions back (a sliding window), or the start of its own chunk of
// `size` positions, counted from position 0 of the sequence
__device__ __forceinline__ int first_visible(int pos, int size, int chunked) {
    const int lo = chunked ? pos - pos % size : pos - size + 1;
    return lo > 0 ? lo : 0;
}

// What weights are taken against: the largest score so far.  Scores can all be -infinity (an infinite key); their weights
// are zero then, as they are beside a finite score, and not exp(-inf + inf).
__device__ __forceinline__ float finite_max(float m) { return m == -INFINITY ? 0.f : m; }

// One workgroup per (token, head).  Its NW waves (4, or 16 when a step has too few tokens to fill the
// chip otherwise: decoding) take the window's 64-key tiles in turn: a lane scores
// one key (q from LDS, the key row straight from its page), the wave forms max / sum of the tile and
// then, lanes now owning value columns, adds the tile's weighted values; the waves' partial softmaxes
// meet in LDS.  The same code serves a prompt's portion and a single decoded token.  Positions below
// `keep_first` stay visible after the window has passed them (a second run of tiles, at their true
// positions); sinks[h] joins the denominator as exp(sink) with no key and no value.
template <bool F32, int NW>
__global__ __launch_bounds__(64 * NW) void window_attn_kernel(const float* q, int64_t ldq, const void* kc_,
                                                          const void* vc_, void* out_, int64_t ldo, PagedRows pr,
                                                          const float* slopes, int T, int H, int G, int d, int dv,
                                                          float scale, int window, const int* row_len, int max_len,
                                                          int keep_first, const float* sinks, const float* gate,
                                                          int64_t ldg, int chunked) {
    typedef typename ActS<F32>::T T_;
    extern __shared__ float lds[];
    if (max_len > 0 && row_len[pr.tok_row[blockIdx.x / H]] > max_len) return;   // the tiled kernel's rows
    const T_* kc = (const T_*)kc_;
    const T_* vc = (const T_*)vc_;
    T_* out = (T_*)out_;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    float* qs = lds;
    float* ps = lds + d + wv * 64;
    float* mm = lds + d + 64 * NW;
    float* ll = mm + NW;
    float* aa = ll + NW;
    const int t = blockIdx.x / H, h = blockIdx.x % H, g = h / (H / G);
    const int pos = pr.tok_pos[t];
    const int* bt = pr.block_table + (int64_t)pr.tok_row[t] * pr.bt_stride;
    const int lo = first_visible(pos, window, chunked);
    const float slope = slopes ? slopes[h] : 0.f;
    for (int c = threadIdx.x; c < d; c += 64 * NW) qs[c] = q[(int64_t)t * ldq + (int64_t)h * d + c];
    __syncthreads();
    float m = -INFINITY, l = 0.f, acc[kMaxVC] = {0.f, 0.f, 0.f, 0.f};
    const int kept = keep_first < lo ? keep_first : lo;    // kept positions the window no longer covers: [0, kept)
    for (int run = kept > 0 ? 0 : 1; run < 2; ++run) {
    const int first = run ? lo : 0, last = run ? pos : kept - 1;
    for (int j0 = first + 64 * wv; j0 <= last; j0 += 64 * NW) {
        const int j = j0 + lane;
        float s = -INFINITY;
        if (j <= last) {
            const int pg = bt[j / pr.page];
            const T_* kr = kc + (((int64_t)pg * pr.page + j % pr.page) * G + g) * d;
            float dot = 0.f;
            if (!F32 && (d & 7) == 0) {
                for (int c = 0; c < d; c += 8) {
                    const uint4 kv = ld16(kr + c);
                    const uint32_t w[4] = {kv.x, kv.y, kv.z, kv.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        dot = fmaf(qs[c + 2 * e], bf16_lo(w[e]), dot);
                        dot = fmaf(qs[c + 2 * e + 1], bf16_hi(w[e]), dot);
                    }
                }
            } else {
                for (int c = 0; c < d; ++c) dot = fmaf(qs[c], ActS<F32>::ld(kr + c), dot);
            }
            s = dot * scale - slope * (float)(pos - j);
        }
        const float mn = fmaxf(m, wave_max(s)), at = finite_max(mn);
        const float pj_ = j <= last ? expf(s - at) : 0.f;
        const float corr = expf(m - at);   // m = -inf on the wave's first tile: exp(-inf) = 0
        l = l * corr + wave_sum(pj_);
        m = mn;
        __builtin_amdgcn_wave_barrier();
        ps[lane] = pj_;
        __builtin_amdgcn_wave_barrier();
        const int cnt = last - j0 + 1 < 64 ? last - j0 + 1 : 64;
#pragma unroll
        for (int ci = 0; ci < kMaxVC; ++ci) acc[ci] *= corr;
        // eight value rows at a time, their loads in flight together (a tile of 64 keys lies in two pages at
        // most when a page holds 64 tokens or more: their ids are looked up once)
        const int pA = j0 / pr.page;
        const bool two = pr.page >= 64;
        const int pgA = bt[pA], pgB = (two && (j0 + cnt - 1) / pr.page != pA) ? bt[pA + 1] : pgA;
        for (int jj = 0; jj < cnt; jj += 8) {
            float pj[8];
            const T_* vr[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const bool ok = jj + u < cnt;
                const int jk = ok ? j0 + jj + u : j0;
                const int pg = two ? (jk / pr.page == pA ? pgA : pgB) : bt[jk / pr.page];
                vr[u] = vc + (((int64_t)pg * pr.page + jk % pr.page) * G + g) * dv;
                pj[u] = ok ? ps[jj + u] : 0.f;
            }
#pragma unroll
            for (int ci = 0; ci < kMaxVC; ++ci) {
                const int c = lane + ci * 64;
                if (c < dv) {
                    float x[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) x[u] = ActS<F32>::ld(vr[u] + c);
#pragma unroll
                    for (int u = 0; u < 8; ++u) acc[ci] = fmaf(pj[u], x[u], acc[ci]);
                }
            }
        }
    }
    }
    if (lane == 0) {
        mm[wv] = m;
        ll[wv] = l;
    }
#pragma unroll
    for (int ci = 0; ci < kMaxVC; ++ci) {
        const int c = lane + ci * 64;
        if (c < dv) aa[wv * dv + c] = acc[ci];
    }
    __syncthreads();
    if (wv == 0) {
        float M = mm[0];
#pragma unroll
        for (int w = 1; w < NW; ++w) M = fmaxf(M, mm[w]);
        float L = 0.f;
        if (sinks) {
            M = fmaxf(M, sinks[h]);
            L = expf(sinks[h] - finite_max(M));
        }
        M = finite_max(M);
        float w4[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            w4[w] = expf(mm[w] - M);   // a wave without keys: exp(-inf) = 0
            L = fmaf(ll[w], w4[w], L);
        }
#pragma unroll
        for (int ci = 0; ci < kMaxVC; ++ci) {
            const int c = lane + ci * 64;
            if (c < dv) {
                float o = 0.f;
#pragma unroll
                for (int w = 0; w < NW; ++w) o = fmaf(aa[w * dv + c], w4[w], o);
                o /= L;
                if (gate) o *= sigmoid_f(gate[(int64_t)t * ldg + (int64_t)h * dv + c]);
                ActS<F32>::st(out + (int64_t)t * ldo + (int64_t)h * dv + c, o);
            }
        }
    }
}


// The same attention for steps of few tokens (decoding), where one workgroup per (token, head) leaves most of the chip
// idle and every query head of a key/value head reads the same pages again: one workgroup of four waves per (token,
// key/value head, group of up to eight of its query heads, split of the key tiles).  A wave takes 64-key tiles - those
// of the kept first positions, then the window's - in steps of 4 * splits; a lane scores ONE key for all heads of the
// group from one read of it, the heads' softmax pieces go through LDS, and the weighted values are gathered with
// 16-byte loads (dv / VEC lanes per value row, several rows per load; `vec` == 0: a lane per value column).  The
// waves' partial softmaxes meet in LDS; with splits > 1 the workgroup leaves (max, sum, weighted values) in `part`
// for window_attn_merge_kernel, which also adds the sink.
constexpr int kGrpMax = 8;

template <bool F32, int RT>
__global__ __launch_bounds__(256) void window_attn_group_kernel(const float* q, int64_t ldq, const void* kc_,
                                                                const void* vc_, void* out_, int64_t ldo, float* part,
                                                                PagedRows pr, const float* slopes, const float* sinks,
                                                                int H, int G, int d, int dv, float scale, int window,
                                                                int keep_first, const int* row_len, int max_len,
                                                                int splits, int vec, const float* gate, int64_t ldg,
                                                                int chunked) {
    typedef typename ActS<F32>::T T_;
    constexpr int VEC = F32 ? 4 : 8;
    extern __shared__ float lds[];
    const T_* kc = (const T_*)kc_;
    const T_* vc = (const T_*)vc_;
    const int R = H / G, ngrp = (R + kGrpMax - 1) / kGrpMax;
    const int unit = blockIdx.x, split = blockIdx.y;
    const int t = unit / (G * ngrp), g = (unit / ngrp) % G, grp = unit % ngrp;
    if (max_len > 0 && row_len[pr.tok_row[t]] > max_len) return;   // the tiled kernel's rows
    const int h0 = g * R + grp * kGrpMax;
    const int nh = R - grp * kGrpMax < kGrpMax ? R - grp * kGrpMax : kGrpMax;   // heads of this workgroup, <= RT
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    float* qs = lds;                    // [RT][d]
    float* ps = qs + RT * d;            // [4][RT][64]
    float* red = ps + 4 * RT * 64;      // [4][RT][dv]
    float* mm = red + 4 * RT * dv;      // [4][RT]
    float* ll = mm + 4 * RT;            // [4][RT]
    for (int i = tid; i < RT * d; i += 256) {
        const int r = i / d;
        qs[i] = r < nh ? q[(int64_t)t * ldq + (int64_t)(h0 + r) * d + (i - r * d)] : 0.f;
    }
    __syncthreads();
    const int pos = pr.tok_pos[t];
    const int* bt = pr.block_table + (int64_t)pr.tok_row[t] * pr.bt_stride;
    const int lo = first_visible(pos, window, chunked);
    const int kept = keep_first < lo ? keep_first : lo;
    const int nk = (kept + 63) / 64, nw = (pos - lo) / 64 + 1;
    float m[RT], l[RT], slope[RT], acc[RT][8];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        m[r] = -INFINITY;
        l[r] = 0.f;
        slope[r] = (slopes && r < nh) ? slopes[h0 + r] : 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r][e] = 0.f;
    }
    const int lpr = vec ? dv / VEC : 1, rp = vec ? 64 / lpr : 1;   // lanes per value row, rows per load
    const int sub = lane / lpr, cb = lane - sub * lpr;
    float* pw = ps + wv * RT * 64;
    for (int u = split * 4 + wv; u < nk + nw; u += 4 * splits) {
        const int first = u < nk ? 64 * u : lo + 64 * (u - nk);
        const int end = u < nk ? kept - 1 : pos;
        const int last = first + 63 < end ? first + 63 : end;
        const int j = first + lane;
        const bool valid = j <= last;
        float dot[RT];
#pragma unroll
        for (int r = 0; r < RT; ++r) dot[r] = 0.f;
        if (valid) {
            const T_* kr = kc + (((int64_t)bt[j / pr.page] * pr.page + j % pr.page) * G + g) * d;
            if (!F32 && (d & 7) == 0) {
                // four 16-byte pieces of the key row in flight at a time
                for (int c0 = 0; c0 < d; c0 += 32) {
                    uint4 kq[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) kq[u] = c0 + 8 * u < d ? ld16(kr + c0 + 8 * u) : make_uint4(0, 0, 0, 0);
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int c = c0 + 8 * u;
                        if (c >= d) break;
                        const uint4 kv = kq[u];
                        const float k8[8] = {bf16_lo(kv.x), bf16_hi(kv.x), bf16_lo(kv.y), bf16_hi(kv.y),
                                             bf16_lo(kv.z), bf16_hi(kv.z), bf16_lo(kv.w), bf16_hi(kv.w)};
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            const float4 qa = *reinterpret_cast<const float4*>(qs + r * d + c);
                            const float4 qb = *reinterpret_cast<const float4*>(qs + r * d + c + 4);
                            dot[r] = fmaf(qa.x, k8[0], dot[r]);
                            dot[r] = fmaf(qa.y, k8[1], dot[r]);
                            dot[r] = fmaf(qa.z, k8[2], dot[r]);
                            dot[r] = fmaf(qa.w, k8[3], dot[r]);
                            dot[r] = fmaf(qb.x, k8[4], dot[r]);
                            dot[r] = fmaf(qb.y, k8[5], dot[r]);
                            dot[r] = fmaf(qb.z, k8[6], dot[r]);
                            dot[r] = fmaf(qb.w, k8[7], dot[r]);
                        }
                    }
                }
            } else {
                for (int c = 0; c < d; ++c) {
                    const float kf = ActS<F32>::ld(kr + c);
#pragma unroll
                    for (int r = 0; r < RT; ++r) dot[r] = fmaf(qs[r * d + c], kf, dot[r]);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            const float sc = valid ? dot[r] * scale - slope[r] * (float)(pos - j) : -INFINITY;
            const float mn = fmaxf(m[r], wave_max(sc)), at = finite_max(mn);
            const float pj = valid ? expf(sc - at) : 0.f;
            const float corr = expf(m[r] - at);                // m = -inf on the wave's first tile: exp(-inf) = 0
            l[r] = l[r] * corr + wave_sum(pj);
            m[r] = mn;
            pw[r * 64 + lane] = pj;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[r][e] *= corr;
        }
        __builtin_amdgcn_wave_barrier();
        const int cnt = last - first + 1;
        if (vec) {
            if (sub < rp) {
                // a tile of 64 keys lies in two pages at most when a page holds 64 tokens or more: their ids are looked
                // up once; eight value rows in flight at a time
                const int pA = first / pr.page;
                const bool two = pr.page >= 64;
                const int pgA = bt[pA], pgB = (two && last / pr.page != pA) ? bt[pA + 1] : pgA;
                for (int row0 = sub; row0 < cnt; row0 += 8 * rp) {
                    uint4 vq[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int row = row0 + u * rp;
                        const int jk = first + (row < cnt ? row : 0);
                        const int pg = two ? (jk / pr.page == pA ? pgA : pgB) : bt[jk / pr.page];
                        vq[u] = ld16(vc + (((int64_t)pg * pr.page + jk % pr.page) * G + g) * dv + cb * VEC);
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int row = row0 + u * rp;
                        if (row >= cnt) break;
                        const uint4 vv = vq[u];
                        float v8[8];
                        if (F32) {
                            v8[0] = __uint_as_float(vv.x); v8[1] = __uint_as_float(vv.y);
                            v8[2] = __uint_as_float(vv.z); v8[3] = __uint_as_float(vv.w);
                            v8[4] = v8[5] = v8[6] = v8[7] = 0.f;
                        } else {
                            v8[0] = bf16_lo(vv.x); v8[1] = bf16_hi(vv.x); v8[2] = bf16_lo(vv.y); v8[3] = bf16_hi(vv.y);
                            v8[4] = bf16_lo(vv.z); v8[5] = bf16_hi(vv.z); v8[6] = bf16_lo(vv.w); v8[7] = bf16_hi(vv.w);
                        }
#pragma unroll
                        for (int r = 0; r < RT; ++r) {
                            const float w = pw[r * 64 + row];
#pragma unroll
                            for (int e = 0; e < VEC; ++e) acc[r][e] = fmaf(w, v8[e], acc[r][e]);
                        }
                    }
                }
            }
        } else {
            for (int row = 0; row < cnt; ++row) {
                const int jk = first + row;
                const T_* vr = vc + (((int64_t)bt[jk / pr.page] * pr.page + jk % pr.page) * G + g) * dv;
#pragma unroll
                for (int ci = 0; ci < kMaxVC; ++ci) {
                    const int c = lane + ci * 64;
                    if (c < dv) {
                        const float x = ActS<F32>::ld(vr + c);
#pragma unroll
                        for (int r = 0; r < RT; ++r) acc[r][ci] = fmaf(pw[r * 64 + row], x, acc[r][ci]);
                    }
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            mm[wv * RT + r] = m[r];
            ll[wv * RT + r] = l[r];
        }
    }
    float* rw = red + wv * RT * dv;
    if (vec) {
        // the row groups of a wave add their sums one after the other
        for (int s2 = 0; s2 < rp; ++s2) {
            if (sub == s2) {
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        const int i = r * dv + cb * VEC + e;
                        rw[i] = (s2 == 0 ? 0.f : rw[i]) + acc[r][e];
                    }
            }
            __builtin_amdgcn_wave_barrier();
        }
    } else {
#pragma unroll
        for (int ci = 0; ci < kMaxVC; ++ci) {
            const int c = lane + ci * 64;
            if (c < dv)
#pragma unroll
                for (int r = 0; r < RT; ++r) rw[r * dv + c] = acc[r][ci];
        }
    }
    __syncthreads();
    for (int i = tid; i < nh * dv; i += 256) {
        const int r = i / dv, c = i - r * dv;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) M = fmaxf(M, mm[w * RT + r]);
        float L = 0.f, o = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float mw = mm[w * RT + r];
            const float f = mw == -INFINITY ? 0.f : expf(mw - M);     // a wave (or a whole split) without keys
            L = fmaf(ll[w * RT + r], f, L);
            o = fmaf(red[(w * RT + r) * dv + c], f, o);
        }
        const int h = h0 + r;
        if (splits == 1) {
            if (sinks) {
                const float sk = sinks[h], mf = fmaxf(M, sk), f = expf(M - mf);
                L = L * f + expf(sk - mf);
                o *= f;
            }
            o /= L;
            if (gate) o *= sigmoid_f(gate[(int64_t)t * ldg + (int64_t)h * dv + c]);
            ActS<F32>::st((T_*)out_ + (int64_t)t * ldo + (int64_t)h * dv + c, o);
        } else {
            float* dst = part + (((int64_t)t * H + h) * splits + split) * (dv + 2);
            if (c == 0) {
                dst[0] = M;
                dst[1] = L;
            }
            dst[2 + c] = o;
        }
    }
}

// A single token's attention is a chain of trips to memory (token -> page table -> keys and values) and little else, so the
// head shapes of the tiled kernel below have a form of their own for it.  One workgroup of NW waves per (token, key/value
// head, group of up to HEADS of its query heads, split of the keys); a wave takes 16-key tiles - those of the kept first
// positions, then the window's - in steps of NW * splits and requests the whole tile, keys and values, at once.
//   q.k   bf16 keys: v_mfma_f32_16x16x32_bf16 with q split exactly into three bf16 numbers, a column each: column h + 4 s is
//         part s of head h, and two rotations within a row of lanes add the parts.  fp32 keys: v_mfma_f32_16x16x4_f32.  Either
//         way lane l ends with the scores of keys 4 (l / 16) .. + 3 for head l % 4.
//   P.V   v_mfma_f32_4x4x1_f32: the lanes that hold those four weights read the same four value rows, 16 lanes a row, so
//         weight j is the first operand where it lies and each element of value row j the second.  (HEADS = 1: plain products,
//         the instruction's other three rows would be idle.)
// The waves' partial softmaxes meet in LDS.  A token whose tiles are one to a wave is finished by its first split, and the
// other splits leave at once; else a split leaves (max, sum, weighted values) in `part` for window_attn_merge_kernel.
//
// Measured (us per call, 8 heads on 2 key/value heads, d = dv = 128, window 1024; kernel above with its 64-key tiles, five
// splits and their merge -> here): one token bf16 at 45 keys 19.5 -> 5.4, 300 21.8 -> 9.0, 1100 23.2 -> 17.2; fp32 19.8 -> 7.6,
// 23.6 -> 13.0, 25.1 -> 17.0; 64 tokens bf16 at 300 23.1 -> 10.0; a prompt of 333 in fp32 at 300 53.7 -> 40.
// 16 heads of 64 with keys of their own, one token 10.6 -> 4.7, 11.7 -> 7.0, 12.2 -> 11.8.
struct TileRun {
    int lo, kept, nk, n;      // n tiles: nk of the kept positions [0, kept), then those of [lo, pos]
};
__device__ __forceinline__ TileRun tile_run(int pos, int window, int keep_first, int chunked) {
    TileRun g;
    g.lo = first_visible(pos, window, chunked);
    g.kept = keep_first < g.lo ? keep_first : g.lo;
    g.nk = (g.kept + 15) / 16;
    g.n = g.nk + (pos - g.lo) / 16 + 1;
    return g;
}

__device__ __forceinline__ float swap_add16(float x, float y) {   // rows 0, 2: x summed over a pair of rows; 1, 3: y
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
__device__ __forceinline__ float swap_add32(float x, float y) {   // lower half: x summed over the halves; upper: y
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
__device__ __forceinline__ float rows_max(float x) {              // over the four rows of 16 lanes
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    const float y = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}

typedef __attribute__((ext_vector_type(8))) __bf16 wa_bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float wa_f32x4_t;

// What a step of single tokens does in front of its attention, in the same launch: qk_rotary_store_kernel's work, same arithmetic.
// Workgroups past the splits, in y, form the gate of a feed-forward, `act_blocks` pieces of 64 NW columns.  (Behind each split's in x they were
// left empty in all splits but one, and an empty workgroup, too, waits for room on a unit that the splits behind it could have: fp32, 24
// heads of 64 on 2, 4 tokens at 2000 keys in 16 splits, a gate of 4096 22.3 us, here 16.2, in two launches 19.8; bf16, 16 tokens at 1000 17.1,
// 12.9, 16.9.)
struct StepRotary {
    const float *q_bias, *k_new, *k_bias;      // k_new: the step's keys, rows as far apart as q's
    const double* inv_freq;
    int rot, adjacent;
    unsigned act_blocks;
    const float* act_in;
    void* act_out;
    int64_t lda, ldao;
    int act_n, act_kind;
    float act_limit, act_slope;
};

// ROT: q and the token's own key come as projected.  A wave each turns a query head or the key (the angles in fp64, as
// qk_rotary_store_kernel forms them) while the first tiles are on their way; the turned queries lie in LDS, and the tile that holds
// the token's own position takes key and value from there too: the page is written by the first split and read by later steps.
// What another split reads of that place meanwhile is not used.
// One launch against two (us, 8 heads of 128 on 2, a gate of 4096 beside them): one token bf16 at 45 keys 8.3 -> 6.0, 300 11.8 -> 10.4,
// 1100 19.0 -> 18.2; fp32 10.8 -> 8.1, 13.3 -> 11.6, 16.6 -> 15.2; 8 tokens of 16 heads on 4 at 500 keys 14.5 -> 13.1.
// OWN: bf16 queries are not shared (kShareQ below)
template <bool F32, int HEADS, int NW, int KS, int VE, bool ROT = false, bool OWN = false>
__global__ __launch_bounds__(64 * NW) void window_attn_few_kernel(const float* q, int64_t ldq, const void* kc_, const void* vc_,
                                                              void* out_, int64_t ldo, float* part, PagedRows pr,
                                                              const float* slopes, const float* sinks, int H, int G,
                                                              float scale, int window, int keep_first, const int* row_len,
                                                              int max_len, int splits, const float* gate, int64_t ldg,
                                                              int chunked, StepRotary ra) {
    typedef typename ActS<F32>::T T_;
    constexpr int d = 32 * KS, dv = 16 * VE, HB = HEADS == 8 ? 2 : 1, RT = HEADS;
    constexpr int NK = F32 ? 2 * KS : KS, VW = F32 ? VE : VE / 2;     // 16-byte pieces of a key, words of a value, per lane
    __shared__ __attribute__((aligned(16))) float red[NW * RT * dv];
    __shared__ float mm[NW * RT], ll[NW * RT];
    __shared__ __attribute__((aligned(16))) float qs[ROT ? RT * d : 4];          // ROT: turned queries, the token's own key
    __shared__ __attribute__((aligned(16))) T_ kn[ROT ? d : 8], vn[ROT ? dv : 8];   // and value
    // bf16 keys: the queries' three parts, formed once for the workgroup: a value's split is some eight instructions, and a wave has up to 32
    // values a lane to it, while what bounds a tile here is the issue slots of the waves that share a unit (one token of 8 heads on 2 of 128,
    // 45 keys, 7.35 -> 5.45 us, 1100 19.6 -> 17.2).  Not worth the barrier with a single head (4.7 -> 5.0 at 45 keys of a launch of its own) and with
    // 8 values a lane (each wave its own, shared: 16 heads of 32 on 4 at 45 keys 4.0, 4.6, at 1100 11.0 both); 16 are for four heads, which load twice
    // two heads' rows (16 of 64 on 4 at 45 and 1100 keys 5.2, 4.9 and 13.1, 12.7), and not for two or three (OWN; 4 of 64 on 2 4.4, 4.7 and 12.4, 12.5,
    // 12 on 4 5.1, 5.3 and 15.2 both).  The turned queries lie in LDS either way
    constexpr bool kShareQ = !F32 && (ROT || (HEADS > 1 && KS * HB > 1 && !OWN));
    __shared__ __attribute__((aligned(16))) uint16_t qp[kShareQ ? 3 * RT * d : 8];
    if constexpr (ROT) {
        if ((int)blockIdx.y >= splits) {
            const unsigned cb = (ra.act_n + 64 * NW - 1) / (64 * NW), i = (blockIdx.y - splits) * gridDim.x + blockIdx.x;
            const int64_t r = i / cb;
            const int c = (i % cb) * 64 * NW + threadIdx.x;
            if (i < ra.act_blocks && c < ra.act_n)
                ActS<F32>::st((T_*)ra.act_out + r * ra.ldao + c, gated_act_f(ra.act_in[r * ra.lda + c], ra.act_in[r * ra.lda + ra.act_n + c],
                                                                            ra.act_kind, ra.act_limit, ra.act_slope));
            return;
        }
    }
    const T_* kc = (const T_*)kc_;
    const T_* vc = (const T_*)vc_;
    const int R = H / G, ngrp = (R + kGrpMax - 1) / kGrpMax;
    const int unit = blockIdx.x, split = blockIdx.y;
    const int t = unit / (G * ngrp), g = (unit / ngrp) % G, grp = unit % ngrp;
    const int h0 = g * R + grp * kGrpMax;
    const int nh = R - grp * kGrpMax < kGrpMax ? R - grp * kGrpMax : kGrpMax;   // heads of this workgroup, <= RT
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, col = lane & 15, quad = lane >> 4;
    const int row = pr.tok_row[t], pos = pr.tok_pos[t];

    // q as the second operand: lane `col` holds head col % 4 (of bf16 keys: its part col / 4)
    wa_bf16x8_t qb[HB][F32 ? 1 : KS];
    wa_f32x4_t qf[HB][F32 ? NK : 1];
    float slope[HB];
    // three bf16 numbers whose sum is x: eight bits of the significand at a time
    auto part_query = [&](int at, float x) {
        const uint32_t a = __float_as_uint(x) & 0xffff0000u;
        const float r1 = x - __uint_as_float(a);
        const uint32_t b2 = __float_as_uint(r1) & 0xffff0000u;
        const float r2 = r1 - __uint_as_float(b2);
        qp[at] = (uint16_t)(a >> 16);
        qp[RT * d + at] = (uint16_t)(b2 >> 16);
        qp[2 * RT * d + at] = (uint16_t)(__float_as_uint(r2) >> 16);
    };
    auto take_queries = [&] {
#pragma unroll
        for (int b = 0; b < HB; ++b) {
            const int h = HEADS == 1 ? 0 : 4 * b + (lane & 3);
            const bool ok = h < nh;
            slope[b] = (slopes && ok) ? slopes[h0 + h] : 0.f;
            if constexpr (F32) {
                const float* qr = q + (int64_t)t * ldq + (int64_t)(h0 + (ok ? h : 0)) * d;
#pragma unroll
                for (int i = 0; i < NK; ++i) {
                    wa_f32x4_t x;
                    if constexpr (ROT) x = *reinterpret_cast<const wa_f32x4_t*>(&qs[(ok ? h : 0) * d + 16 * i + 4 * quad]);
                    else x = *reinterpret_cast<const wa_f32x4_t*>(qr + 16 * i + 4 * quad);
                    qf[b][i] = ok ? x : (wa_f32x4_t){0.f, 0.f, 0.f, 0.f};
                }
            } else if constexpr (kShareQ) {
                const int s = col >> 2;
                const bool has = ok && s < 3;
#pragma unroll
                for (int i = 0; i < KS; ++i) {
                    const uint4 x = *reinterpret_cast<const uint4*>(&qp[((has ? s * RT : 0) + (has ? h : 0)) * d + 32 * i + 8 * quad]);
                    qb[b][i] = __builtin_bit_cast(wa_bf16x8_t, has ? x : make_uint4(0, 0, 0, 0));
                }
            } else {
                const float* qr = q + (int64_t)t * ldq + (int64_t)(h0 + (ok ? h : 0)) * d;
                const int s = col >> 2;
#pragma unroll
                for (int i = 0; i < KS; ++i) {
                    const wa_f32x4_t x0 = *reinterpret_cast<const wa_f32x4_t*>(qr + 32 * i + 8 * quad);
                    const wa_f32x4_t x1 = *reinterpret_cast<const wa_f32x4_t*>(qr + 32 * i + 8 * quad + 4);
                    uint16_t p[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float x = e < 4 ? x0[e & 3] : x1[e & 3];
                        const uint32_t a = __float_as_uint(x) & 0xffff0000u;
                        const float r1 = x - __uint_as_float(a);
                        const uint32_t b2 = __float_as_uint(r1) & 0xffff0000u;
                        const float r2 = r1 - __uint_as_float(b2);
                        const uint32_t w = s == 0 ? a : s == 1 ? b2 : __float_as_uint(r2);
                        p[e] = ok && s < 3 ? (uint16_t)(w >> 16) : (uint16_t)0;
                    }
                    qb[b][i] = __builtin_bit_cast(wa_bf16x8_t, *reinterpret_cast<uint4*>(p));
                }
            }
        }
    };
    if constexpr (!ROT && kShareQ) {
        const float* qr = q + (int64_t)t * ldq + (int64_t)h0 * d;
        for (int i = tid; i < nh * d; i += 64 * NW) part_query(i, qr[i]);
    } else if constexpr (!ROT) {
        take_queries();
    }

    const TileRun gt = tile_run(pos, window, keep_first, chunked);
    const int* bt = pr.block_table + (int64_t)row * pr.bt_stride;
    float m[HB], l[HB];
    wa_f32x4_t acc[HB][VE];
#pragma unroll
    for (int b = 0; b < HB; ++b) {
        m[b] = -INFINITY;
        l[b] = 0.f;
#pragma unroll
        for (int e = 0; e < VE; ++e) acc[b][e] = (wa_f32x4_t){0.f, 0.f, 0.f, 0.f};
    }
    // the tile's keys, this lane's key (lane % 16; past the last key: the first) and the place of its row
    int first, cnt, j;
    int page_no;
    const bool pow2 = (pr.page & (pr.page - 1)) == 0;      // (uniform: a division by a number of the launch is some forty instructions)
    const int shift = 31 - __builtin_clz(pr.page);
    auto locate = [&](int u) {
        if (u >= gt.n) u = gt.n - 1;
        first = u < gt.nk ? 16 * u : gt.lo + 16 * (u - gt.nk);
        const int end = u < gt.nk ? gt.kept - 1 : pos;
        cnt = end - first + 1 < 16 ? end - first + 1 : 16;
        j = first + (col < cnt ? col : 0);
        page_no = bt[pow2 ? j >> shift : j / pr.page];
    };
    uint4 kq[NK];
    uint32_t vq[4][VW];
    unsigned vslot[4];
    auto fetch = [&] {
        const unsigned slot = pow2 ? ((unsigned)page_no << shift) + (unsigned)(j & (pr.page - 1))
                                   : (unsigned)page_no * (unsigned)pr.page + (unsigned)(j % pr.page);
        const T_* kr = kc + ((uint64_t)slot * G + g) * d;
#pragma unroll
        for (int i = 0; i < NK; ++i) kq[i] = ld16(kr + (F32 ? 16 * i + 4 * quad : 32 * i + 8 * quad));
#pragma unroll
        for (int k = 0; k < 4; ++k) vslot[k] = (unsigned)__shfl((int)slot, 4 * quad + k, 64);   // (lanes 0 - 15: keys in order)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t* vr = reinterpret_cast<const uint32_t*>(vc + ((uint64_t)vslot[k] * G + g) * dv) + col * VW;
            if constexpr (VW % 4 == 0) {
#pragma unroll
                for (int w = 0; w < VW; w += 4) {
                    const uint4 x = ld16(vr + w);
                    vq[k][w] = x.x; vq[k][w + 1] = x.y; vq[k][w + 2] = x.z; vq[k][w + 3] = x.w;
                }
            } else if constexpr (VW % 2 == 0) {
#pragma unroll
                for (int w = 0; w < VW; w += 2) {
                    const uint2 x = *reinterpret_cast<const uint2*>(vr + w);
                    vq[k][w] = x.x; vq[k][w + 1] = x.y;
                }
            } else {
#pragma unroll
                for (int w = 0; w < VW; ++w) vq[k][w] = vr[w];
            }
        }
    };
    locate(split * NW + wv);
    // (behind the page's request: the length in front of it would be one more trip to memory)
    if (!ROT && max_len > 0 && row_len[row] > max_len) return;   // the tiled kernel's rows
    if (split * NW >= gt.n) return;                      // no keys for this split
    if constexpr (ROT) {
        if (split * NW + wv < gt.n) fetch();
        // heads 0 .. nh - 1 of q, then the key
        for (int hh = wv; hh <= nh; hh += NW) {
            const bool key = hh == nh;
            const float* p = key ? ra.k_new + (int64_t)t * ldq + (int64_t)g * d : q + (int64_t)t * ldq + (int64_t)(h0 + hh) * d;
            const float* bias = key ? (ra.k_bias ? ra.k_bias + (int64_t)g * d : nullptr)
                                    : (ra.q_bias ? ra.q_bias + (int64_t)(h0 + hh) * d : nullptr);
            int64_t at = -1;                             // the key's place in the pages, for the one that stores it
            if (key && split == 0 && grp == 0) {
                const int pg = bt[pos / pr.page];
                if (pg >= 0) at = (((int64_t)pg * pr.page + pos % pr.page) * G + g) * d;
            }
            auto put = [&](int c, float turned, float plain) {
                if (!key) {
                    qs[hh * d + c] = turned;
                    if constexpr (!F32) part_query(hh * d + c, turned);
                    return;
                }
                ActS<F32>::st(kn + c, turned);
                ActS<F32>::st(vn + c, plain);
                if (at >= 0) {
                    ActS<F32>::st((T_*)kc_ + at + c, turned);
                    ActS<F32>::st((T_*)vc_ + at + c, plain);
                }
            };
            const int half = ra.rot / 2;
            for (int i = lane; i < half; i += 64) {
                const int a = ra.adjacent ? 2 * i : i, b = ra.adjacent ? 2 * i + 1 : i + half;
                const float x0 = bias ? p[a] + bias[a] : p[a], x1 = bias ? p[b] + bias[b] : p[b];
                const double ang = (double)pos * ra.inv_freq[i];
                double sin_, cos_;
                sincos(ang, &sin_, &cos_);
                const float cs = (float)cos_, sn = (float)sin_;
                put(a, x0 * cs - x1 * sn, x0);
                put(b, x1 * cs + x0 * sn, x1);
            }
            for (int c = ra.rot + lane; c < d; c += 64) {
                const float x0 = bias ? p[c] + bias[c] : p[c];
                put(c, x0, x0);
            }
        }
    }
    if constexpr (ROT || kShareQ) {
        __syncthreads();
        if (split * NW + wv < gt.n) take_queries();
    }
    for (int u = split * NW + wv; u < gt.n; u += NW * splits) {
        if constexpr (!ROT) {
            fetch();
        } else if (u == gt.n - 1) {      // (uniform) the tile of the token's own position
            if (j == pos) {
#pragma unroll
                for (int i = 0; i < NK; ++i) kq[i] = *reinterpret_cast<const uint4*>(kn + (F32 ? 16 * i + 4 * quad : 32 * i + 8 * quad));
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (first + 4 * quad + k == pos) {
#pragma unroll
                    for (int w = 0; w < VW; ++w) vq[k][w] = reinterpret_cast<const uint32_t*>(vn)[col * VW + w];
                }
        }
        wa_f32x4_t sc[HB];
#pragma unroll
        for (int b = 0; b < HB; ++b) {
            sc[b] = (wa_f32x4_t){0.f, 0.f, 0.f, 0.f};
            if constexpr (F32) {
#pragma unroll
                for (int i = 0; i < NK; ++i) {
                    const uint32_t kw[4] = {kq[i].x, kq[i].y, kq[i].z, kq[i].w};
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        sc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(kw[e]), qf[b][i][e], sc[b], 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int i = 0; i < KS; ++i)
                    sc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wa_bf16x8_t, kq[i]), qb[b][i], sc[b], 0, 0, 0);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    sc[b][k] += dpp<0x128>(sc[b][k]);      // row_ror:8, row_ror:4
                    sc[b][k] += dpp<0x124>(sc[b][k]);
                }
                // an infinite key or query times a part that is zero: the plain sum decides
                const int h = HEADS == 1 ? 0 : 4 * b + (lane & 3);
                const bool bad = h < nh && !(sc[b][0] == sc[b][0] && sc[b][1] == sc[b][1] &&
                                          sc[b][2] == sc[b][2] && sc[b][3] == sc[b][3]);
                if (__any(bad)) {
                    const float* qr = ROT ? qs + (h < nh ? h : 0) * d : q + (int64_t)t * ldq + (int64_t)(h0 + (h < nh ? h : 0)) * d;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const T_* kp = kc + ((uint64_t)vslot[k] * G + g) * d;
                        if (ROT && first + (4 * quad + k < cnt ? 4 * quad + k : 0) == pos) kp = kn;
                        float dot = 0.f;
#pragma unroll 1
                        for (int c = 0; c < d; ++c) dot = fmaf(qr[c], ActS<F32>::ld(kp + c), dot);
                        sc[b][k] = dot;
                    }
                }
            }
        }
        if (cnt < 16) {      // rows that repeat the first key: weight zero, and no value that could be infinite
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (4 * quad + k >= cnt)
#pragma unroll
                    for (int w = 0; w < VW; ++w) vq[k][w] = 0;
        }
#pragma unroll
        for (int b = 0; b < HB; ++b) {
            float p[4], mx = -INFINITY;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int key = 4 * quad + k;
                p[k] = key < cnt ? sc[b][k] * scale - slope[b] * (float)(pos - first - key) : -INFINITY;
                mx = fmaxf(mx, p[k]);
            }
            const float mn = fmaxf(m[b], rows_max(mx));
            const float at = finite_max(mn);
            const float corr = expf(m[b] - at);                // m = -inf on the wave's first tile: exp(-inf) = 0
            float sum = 0.f;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                p[k] = 4 * quad + k < cnt ? expf(p[k] - at) : 0.f;
                sum += p[k];
            }
            l[b] = l[b] * corr + sum;                          // this lane's four keys' share
            m[b] = mn;
            if (HEADS == 1) {
#pragma unroll
                for (int e = 0; e < VE; ++e) acc[b][e][0] *= corr;
            } else if (__any(corr != 1.f)) {
                const float c0 = dpp<0x00>(corr), c1 = dpp<0x55>(corr), c2 = dpp<0xAA>(corr), c3 = dpp<0xFF>(corr);
#pragma unroll
                for (int e = 0; e < VE; ++e) {
                    acc[b][e][0] *= c0;
                    acc[b][e][1] *= c1;
                    acc[b][e][2] *= c2;
                    acc[b][e][3] *= c3;
                }
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int e = 0; e < VE; ++e) {
                    const float v = F32 ? __uint_as_float(vq[k][F32 ? e : 0])
                                    : (e & 1) ? bf16_hi(vq[k][F32 ? 0 : e >> 1]) : bf16_lo(vq[k][F32 ? 0 : e >> 1]);
                    if (HEADS == 1) acc[b][e][0] = fmaf(p[k], v, acc[b][e][0]);
                    else acc[b][e] = __builtin_amdgcn_mfma_f32_4x4x1f32(p[k], v, acc[b][e], 0, 0, 0);
                }
        }
        locate(u + NW * splits);
        if constexpr (ROT) {
            if (u + NW * splits < gt.n) fetch();
        }
    }
    const int nact = gt.n - split * NW < NW ? gt.n - split * NW : NW;   // waves with a tile
    if (wv < nact) {
#pragma unroll
        for (int b = 0; b < HB; ++b) {
            l[b] = swap_add16(l[b], l[b]);
            l[b] = swap_add32(l[b], l[b]);
            if (lane < (HEADS == 1 ? 1 : 4)) {
                mm[wv * RT + 4 * b + lane] = m[b];
                ll[wv * RT + 4 * b + lane] = l[b];
            }
            // rows of lanes hold different keys: row h keeps the sum of head h
            float o[VE];
#pragma unroll
            for (int e = 0; e < VE; ++e)
                if (HEADS == 1) o[e] = swap_add16(swap_add32(acc[b][e][0], acc[b][e][0]), swap_add32(acc[b][e][0], acc[b][e][0]));
                else o[e] = swap_add16(swap_add32(acc[b][e][0], acc[b][e][2]), swap_add32(acc[b][e][1], acc[b][e][3]));
            float* rw = red + (wv * RT + (HEADS == 1 ? 0 : 4 * b + quad)) * dv + col * VE;
#pragma unroll
            for (int e = 0; e < VE; e += 2)
                if (HEADS > 1 || quad == 0) *reinterpret_cast<float2*>(rw + e) = make_float2(o[e], o[e + 1]);
        }
    }
    __syncthreads();
    const bool alone = gt.n <= NW || splits == 1;
    for (int i = tid; i < nh * dv; i += 64 * NW) {
        const int r = i / dv, c = i - r * dv;
        float M = -INFINITY;
        for (int w = 0; w < nact; ++w) M = fmaxf(M, mm[w * RT + r]);
        float L = 0.f, o = 0.f;
        const float at = finite_max(M);
        for (int w = 0; w < nact; ++w) {
            const float f = expf(mm[w * RT + r] - at);
            L = fmaf(ll[w * RT + r], f, L);
            o = fmaf(red[(w * RT + r) * dv + c], f, o);
        }
        const int h = h0 + r;
        if (alone) {
            if (sinks) {
                const float sk = sinks[h], mf = fmaxf(M, sk), f = expf(M - mf);
                L = L * f + expf(sk - mf);
                o *= f;
            }
            o /= L;
            if (gate) o *= sigmoid_f(gate[(int64_t)t * ldg + (int64_t)h * dv + c]);
            ActS<F32>::st((T_*)out_ + (int64_t)t * ldo + (int64_t)h * dv + c, o);
        } else {
            float* dst = part + (((int64_t)t * H + h) * splits + split) * (dv + 2);
            if (c == 0) {
                dst[0] = M;
                dst[1] = L;
            }
            dst[2 + c] = o;
        }
    }
}

// one wave per (token, head): the splits' pieces and the sink become the output row.  nw > 0: window_attn_few_kernel's splits
// of nw waves, of which those past the token's tiles left nothing and a single one is the finished row.
template <bool F32>
__global__ __launch_bounds__(64) void window_attn_merge_kernel(const float* part, void* out_, int64_t ldo,
                                                               const int* tok_row, const int* tok_pos, const float* sinks,
                                                               int H, int dv, int splits, int nw, int window, int keep_first,
                                                               int chunked, const int* row_len, int max_len,
                                                               const float* gate, int64_t ldg) {
    typedef typename ActS<F32>::T T_;
    const int t = blockIdx.x / H, h = blockIdx.x % H, lane = threadIdx.x;
    // The first pieces, their sums and what the row may be multiplied by are asked for before anything says how many there are
    // (what lies past those is not used): one trip to memory instead of one for every step below.  With the attention in front of it, fp32, 8
    // heads of 128 on 2 in four splits at 300 keys 13.4 -> 10.6 us, 1100 17.5 -> 13.1; bf16, 32 heads on 8, 2048 keys in eight 16.7 -> 11.3.
    constexpr int kAhead = 8;
    const float* src = part + (int64_t)blockIdx.x * splits * (dv + 2);
    float ahead[kAhead][2];
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
        if (s >= splits) break;   // uniform
#pragma unroll
        for (int k = 0; k < 2; ++k) ahead[s][k] = src[(int64_t)s * (dv + 2) + 2 + (lane + 64 * k < dv ? lane + 64 * k : 0)];
    }
    const float* mine = src + (int64_t)(lane < splits ? lane : 0) * (dv + 2);
    const float m0 = mine[0], l0 = mine[1];
    const float sink = sinks ? sinks[h] : 0.f;
    int n = splits;                            // pieces there are
    if (nw > 0) {
        const int tiles = tile_run(tok_pos[t], window, keep_first, chunked).n;
        if (tiles <= nw) return;
        if (tiles < splits * nw) n = (tiles + nw - 1) / nw;
    }
    if (max_len > 0 && row_len[tok_row[t]] > max_len) return;
    float M = lane < n ? m0 : -INFINITY, L = 0.f;
    for (int s = lane + 64; s < n; s += 64) M = fmaxf(M, src[(int64_t)s * (dv + 2)]);
    M = wave_max(M);
    if (sinks) M = fmaxf(M, sink);
    const float f0 = lane < n && m0 != -INFINITY ? expf(m0 - M) : 0.f;      // the weight of piece `lane`
    if (lane < n && m0 != -INFINITY) L = fmaf(l0, f0, L);
    for (int s = lane + 64; s < n; s += 64) {
        const float ms = src[(int64_t)s * (dv + 2)];
        if (ms != -INFINITY) L = fmaf(src[(int64_t)s * (dv + 2) + 1], expf(ms - M), L);
    }
    L = wave_sum(L);
    if (sinks) L += expf(sink - M);
    auto finish = [&](int c, float o) {
        o /= L;
        if (gate) o *= sigmoid_f(gate[(int64_t)t * ldg + (int64_t)h * dv + c]);
        ActS<F32>::st((T_*)out_ + (int64_t)t * ldo + (int64_t)h * dv + c, o);
    };
    if (n <= kAhead && dv <= 128) {
        float o[2] = {0.f, 0.f};
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
            if (s >= n) break;   // uniform
            const float f = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f0), s));
#pragma unroll
            for (int k = 0; k < 2; ++k) o[k] = fmaf(f != 0.f ? ahead[s][k] : 0.f, f, o[k]);
        }
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (lane + 64 * k < dv) finish(lane + 64 * k, o[k]);
        return;
    }
    for (int c = lane; c < dv; c += 64) {
        float o = 0.f;
#pragma unroll 4
        for (int s = 0; s < n; ++s) {
            const float ms = src[(int64_t)s * (dv + 2)], f = ms != -INFINITY ? expf(ms - M) : 0.f;
            o = fmaf(f != 0.f ? src[(int64_t)s * (dv + 2) + 2 + c] : 0.f, f, o);
        }
        finish(c, o);
    }
}

// The same attention for a prompt's portion, bf16 keys and values: one workgroup per (64 consecutive tokens
// of a row, head).  Key tiles are pages (64 tokens) staged once in LDS for all 64 queries; q.k on
// v_mfma_f32_16x16x32_bf16 (q rounded to bf16 as the keys are), scores, distance penalty, mask and softmax
// in fp32 per lane, and P.V with every fp32 weight split exactly into three bf16 numbers, on the same bf16
// instruction with fp32 accumulators: the score accumulators of a lane, S[key 16 nt + 4 (lane / 16) + j][query
// lane % 16], serve as its second operand where they lie, so P never leaves the registers.
template <int KS, int CT>
__global__ __launch_bounds__(256) void window_attn_tile_kernel(const float* q, int64_t ldq, const uint16_t* kc,
                                                               const uint16_t* vc, uint16_t* out, int64_t ldo,
                                                               PagedRows pr, const int* ch_start, const int* ch_len,
                                                               const float* slopes, int H, int G, float scale,
                                                               int window, int keep_first, const float* sinks,
                                                               const float* gate, int64_t ldg, int chunked) {
    constexpr int D = KS * 32, DV = CT * 16, SK = D + 8, SV = DV + 8;
    __shared__ __attribute__((aligned(16))) uint16_t Ks[64][SK];
    // values as pairs of neighbouring keys: dword [i][c] = V[2i][c] | V[2i+1][c] << 16, which is how the matrix
    // instruction wants them (two contraction slots per register)
    __shared__ __attribute__((aligned(16))) uint32_t Vp[32][SV];
    // Workgroups 256 apart share a compute unit; a chunk's place decides how many keys it reads.  The chunks of later heads
    // are taken in a rotated order, so that a unit gets chunks of unequal places.
    const int h = blockIdx.y, g = h / (H / G), nch = gridDim.x;
    const int rounds = (nch * (int)gridDim.y + 255) >> 8, turn = ((h * nch) >> 8) * (nch / rounds);
    const int ch = (int)((blockIdx.x + turn) % nch);
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, r = lane & 15, qd = lane >> 4;
    const int start = ch_start[ch], len = ch_len[ch];
    const int* bt = pr.block_table + (int64_t)pr.tok_row[start] * pr.bt_stride;
    const int p0 = pr.tok_pos[start];            // positions run on from here within the chunk
    const int myq = 16 * wv + r;
    const bool qok = myq < len;
    const int qpos = p0 + myq;
    wa_bf16x8_t qf[KS];
    {
        const float* qp = q + (int64_t)(start + (qok ? myq : 0)) * ldq + (int64_t)h * D + 8 * qd;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            const float4 a = *reinterpret_cast<const float4*>(qp + 32 * kk);
            const float4 b = *reinterpret_cast<const float4*>(qp + 32 * kk + 4);
            const uint4 pk = make_uint4(pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w), pack_bf16x2(b.x, b.y),
                                        pack_bf16x2(b.z, b.w));
            qf[kk] = __builtin_bit_cast(wa_bf16x8_t, pk);
        }
    }
    float m = -INFINITY, l = 0.f;
    f32x4_t o[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) o[ct] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const float slope = slopes ? slopes[h] : 0.f;
    const int klo = first_visible(p0, window, chunked), khi = p0 + len - 1;
    const int wq_lo = p0 + 16 * wv, wq_hi = wq_lo + 15;   // this wave's query positions
    const int wk_lo = first_visible(wq_lo, window, chunked), qlo = first_visible(qpos, window, chunked);
    // key tiles: those of the kept first positions that the window of the chunk's first query has left behind,
    // then the window's
    const int kt_lo = klo / 64, kt_keep = ((keep_first < klo ? keep_first : klo) + 63) / 64;
    // A tile's rows come in registers while the tile before is multiplied, its page's number a tile earlier: loaded where they
    // are stored, they were a third of a chunk's time (16 heads, one chunk behind 700 keys 50.8 -> 34.0 us; 32 heads of 2048 tokens 169 ->
    // 152, where several workgroups share a unit).
    auto next_tile = [&](int kt) { return (kt + 1 >= kt_keep && kt + 1 < kt_lo) ? kt_lo : kt + 1; };
    constexpr int NV = (CT + 3) / 4;
    uint4 kr[KS], va[NV], vb[NV];
    auto fetch = [&](int page) {
        const int64_t pgrow = (int64_t)page * 64;
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            const int i = tid + 256 * u, rr = i / (D / 8), cc = i % (D / 8);
            kr[u] = ld16(kc + ((pgrow + rr) * G + g) * D + cc * 8);
        }
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int i = min(tid + 256 * u, 32 * (DV / 8) - 1), rr = i / (DV / 8), cc = i % (DV / 8);
            va[u] = ld16(vc + ((pgrow + 2 * rr) * G + g) * DV + cc * 8);
            vb[u] = ld16(vc + ((pgrow + 2 * rr + 1) * G + g) * DV + cc * 8);
        }
    };
    const int last = khi / 64;
    int kt = kt_keep > 0 ? 0 : kt_lo, kn = next_tile(kt);      // (the first tile is one of the chunk's: kt <= last)
    int page_next = bt[min(kn, last)];
    fetch(bt[kt]);
    for (;;) {
        const int kbase = kt * 64;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            const int i = tid + 256 * u, rr = i / (D / 8), cc = i % (D / 8);
            st16(&Ks[rr][cc * 8], kr[u]);
        }
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int i = tid + 256 * u, rr = i / (DV / 8), cc = i % (DV / 8);
            if (CT % 4 && i >= 32 * (DV / 8)) continue;
            const uint4 a = va[u], b = vb[u];
            st16(&Vp[rr][cc * 8], make_uint4((a.x & 0xffffu) | (b.x << 16), (a.x >> 16) | (b.x & 0xffff0000u),
                                             (a.y & 0xffffu) | (b.y << 16), (a.y >> 16) | (b.y & 0xffff0000u)));
            st16(&Vp[rr][cc * 8 + 4], make_uint4((a.z & 0xffffu) | (b.z << 16), (a.z >> 16) | (b.z & 0xffff0000u),
                                                 (a.w & 0xffffu) | (b.w << 16), (a.w >> 16) | (b.w & 0xffff0000u)));
        }
        const bool more = kn <= last;      // uniform
        const int kn2 = next_tile(kn);
        if (more) {
            fetch(page_next);
            page_next = bt[min(kn2, last)];
        }
        __syncthreads();
        // nothing of a tile past the wave's queries, or between the kept keys and their windows, is visible to it
        if (!(kbase > wq_hi || (kbase + 63 < wk_lo && kbase >= keep_first))) {
        f32x4_t sc[4];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            sc[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < KS; ++kk) {
                const wa_bf16x8_t kf = __builtin_bit_cast(wa_bf16x8_t, ld16(&Ks[16 * nt + r][32 * kk + 8 * qd]));
                sc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[kk], sc[nt], 0, 0, 0);
            }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int kpos = kbase + 16 * nt + 4 * qd + j;
                const bool ok = qok && kpos <= qpos && (kpos >= qlo || kpos < keep_first);
                const float v = ok ? sc[nt][j] * scale - slope * (float)(qpos - kpos) : -INFINITY;
                sc[nt][j] = v;
                mx = fmaxf(mx, v);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mn = fmaxf(m, mx);
        constexpr float kLog2e = 1.4426950408889634f;      // e^x as 2^(x log2 e) on the hardware's exp2
        const float corr = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - mn) * kLog2e);
        float ps = 0.f;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float pv = sc[nt][j] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((sc[nt][j] - mn) * kLog2e);
                sc[nt][j] = pv;
                ps += pv;
            }
        ps += __shfl_xor(ps, 16, 64);
        ps += __shfl_xor(ps, 32, 64);
        l = l * corr + ps;
        m = mn;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) o[ct] *= corr;
        // P.V with P kept whole: an fp32 weight is the exact sum of three bf16 numbers (its leading 8, the next 8
        // and the last 8 bits of the mantissa, each cut off, not rounded), the values are bf16 as cached, so three
        // bf16 matrix instructions with fp32 accumulators form the same products as one in fp32 would - at three
        // eighths of its cost.  The contraction index of the instruction is only a label: slot (qd, e) of both
        // operands stands for key 32 kb + 16 (e / 4) + 4 qd + e % 4, which is where the lane's scores already lie.
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            uint32_t hi[4], mid[4], lo[4];
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2) {       // two weights per dword
                uint32_t h2[2], m2[2], l2[2];
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const int e = 2 * e2 + x;
                    const float pv = sc[2 * kb + e / 4][e % 4];
                    const uint32_t hb = __float_as_uint(pv) & 0xffff0000u;
                    const float r1 = pv - __uint_as_float(hb);
                    const uint32_t mb = __float_as_uint(r1) & 0xffff0000u;
                    const float r2 = r1 - __uint_as_float(mb);
                    h2[x] = hb;
                    m2[x] = mb;
                    l2[x] = __float_as_uint(r2) & 0xffff0000u;
                }
                hi[e2] = (h2[0] >> 16) | h2[1];
                mid[e2] = (m2[0] >> 16) | m2[1];
                lo[e2] = (l2[0] >> 16) | l2[1];
            }
            const wa_bf16x8_t ph = __builtin_bit_cast(wa_bf16x8_t, make_uint4(hi[0], hi[1], hi[2], hi[3]));
            const wa_bf16x8_t pm = __builtin_bit_cast(wa_bf16x8_t, make_uint4(mid[0], mid[1], mid[2], mid[3]));
            const wa_bf16x8_t pl = __builtin_bit_cast(wa_bf16x8_t, make_uint4(lo[0], lo[1], lo[2], lo[3]));
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                uint32_t vw[4];
#pragma unroll
                for (int e2 = 0; e2 < 4; ++e2)     // keys k0, k0 + 1 with k0 = 32 kb + 16 (e2 / 2) + 4 qd + 2 (e2 % 2)
                    vw[e2] = Vp[16 * kb + 8 * (e2 / 2) + 2 * qd + (e2 % 2)][16 * ct + r];
                const wa_bf16x8_t vf = __builtin_bit_cast(wa_bf16x8_t, make_uint4(vw[0], vw[1], vw[2], vw[3]));
                o[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, ph, o[ct], 0, 0, 0);
                o[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pm, o[ct], 0, 0, 0);
                o[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl, o[ct], 0, 0, 0);
            }
        }
        }
        if (!more) break;
        kt = kn;
        kn = kn2;
    }
    if (qok) {
        float inv = 1.0f / l;
        if (sinks) {   // one more term of the denominator, without a value (m is finite: a query sees itself)
            const float sk = sinks[h], mn = fmaxf(m, sk);
            inv = expf(m - mn) / (l * expf(m - mn) + expf(sk - mn));
        }
        uint16_t* op = out + (int64_t)(start + myq) * ldo + (int64_t)h * DV + 4 * qd;
        const float* gp = gate ? gate + (int64_t)(start + myq) * ldg + (int64_t)h * DV + 4 * qd : nullptr;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            if (gp) {
#pragma unroll
                for (int j = 0; j < 4; ++j) o[ct][j] *= sigmoid_f(gp[16 * ct + j]);
            }
            uint2 w;
            w.x = pack_bf16x2(o[ct][0] * inv, o[ct][1] * inv);
            w.y = pack_bf16x2(o[ct][2] * inv, o[ct][3] * inv);
            *reinterpret_cast<uint2*>(op + 16 * ct) = w;
        }
    }
}

// The same with a group's values in registers, V pieces of four a thread of NT: one pass over y and the gate where the loop
// below takes two.  NT = 1024 while the groups leave compute units idle (one row of 8192: 30.3 -> 4.9 us), else 256
// (2048 rows of 8192: 60 -> 30 us; 160 MB that have to move).
template <bool F32, int NT, int V>
__global__ __launch_bounds__(NT) void gated_group_norm_reg_kernel(const float* y, int64_t ldy, const float* gate, int64_t ldg,
                                                                  const float* w, void* out_, int64_t ldo, int n, int groups,
                                                                  int mode, int w_shared, float eps) {
    typedef typename ActS<F32>::T T;
    __shared__ float red[NT / 64];
    const int row = blockIdx.x / groups, g = blockIdx.x % groups, gs = n / groups;
    const float* yr = y + (int64_t)row * ldy + (int64_t)g * gs;
    const float* gr = gate + (int64_t)row * ldg + (int64_t)g * gs;
    const float* wr = w ? w + (w_shared ? 0 : (int64_t)g * gs) : nullptr;
    T* out = (T*)out_ + (int64_t)row * ldo + (int64_t)g * gs;
    f32x4_t u[V], z[V], wv[V];
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int c = min((i * NT + (int)threadIdx.x) * 4, gs - 4);     // (past the end: the last piece again, masked below)
        u[i] = *reinterpret_cast<const f32x4_t*>(yr + c);
        z[i] = *reinterpret_cast<const f32x4_t*>(gr + c);
        if (wr) wv[i] = *reinterpret_cast<const f32x4_t*>(wr + c);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const bool ok = (i * NT + (int)threadIdx.x) * 4 < gs;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (mode == 1) u[i][e] *= silu_f(z[i][e]);
            if (ok) ss += u[i][e] * u[i][e];
        }
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)gs + eps);
#pragma unroll
    for (int i = 0; i < V; ++i) {
        const int c = (i * NT + (int)threadIdx.x) * 4;
        if (c >= gs) break;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[e] = mode == 1 ? u[i][e] * inv : (u[i][e] * inv) * (mode == 2 ? sigmoid_f(z[i][e]) : silu_f(z[i][e]));
            if (wr) o[e] *= wv[i][e];
        }
        if constexpr (F32) *reinterpret_cast<float4*>(out + c) = make_float4(o[0], o[1], o[2], o[3]);
        else *reinterpret_cast<uint2*>(out + c) = make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
    }
}

// groups of a thousand values and more: one workgroup per (row, group)
template <bool F32>
__global__ __launch_bounds__(256) void gated_group_norm_wide_kernel(const float* y, int64_t ldy, const float* gate,
                                                                    int64_t ldg, const float* w, void* out_,
                                                                    int64_t ldo, int n, int groups, int mode,
                                                                    int w_shared, float eps) {
    typedef typename ActS<F32>::T T;
    __shared__ float red[4];
    T* out = (T*)out_;
    const int row = blockIdx.x / groups, g = blockIdx.x % groups, gs = n / groups;
    const float* yr = y + (int64_t)row * ldy + (int64_t)g * gs;
    const float* gr = gate + (int64_t)row * ldg + (int64_t)g * gs;
    float ss = 0.f;
    for (int c = threadIdx.x; c < gs; c += 256) {
        const float u = mode == 1 ? yr[c] * silu_f(gr[c]) : yr[c];
        ss += u * u;
    }
    ss = block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)gs + eps);
    for (int c = threadIdx.x; c < gs; c += 256) {
        float u = mode == 1 ? (yr[c] * silu_f(gr[c])) * inv : (yr[c] * inv) * (mode == 2 ? sigmoid_f(gr[c]) : silu_f(gr[c]));
        if (w) u *= w[w_shared ? c : g * gs + c];
        ActS<F32>::st(out + (int64_t)row * ldo + (int64_t)g * gs + c, u);
    }
}

}  // namespace mv

extern "C" {

using mv::StepRows;

int mv_conv_silu(const float* in, int64_t ldi, float* state, const float* w, const float* bias, float* out,
                 int64_t ldo, const int32_t* tok_row, const int32_t* row_start, const int32_t* row_len,
                 const int32_t* row_ctx, const int32_t* row_slot, int tokens, int rows, int channels, int taps,
                 mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || rows < 0 || channels <= 0 || taps < 1 || taps > kMaxTaps) return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!in || (!state && taps > 1) || !w || !out || ldi < channels || ldo < channels) return MV_ERR_INVALID_ARG;
    StepRows r{tok_row, nullptr, row_start, row_len, row_ctx, row_slot};
    hipStream_t s = (hipStream_t)stream;
    const int64_t work = (int64_t)tokens * channels;
    const bool by_row = tokens <= rows;     // one token a row (decoding)
    if (taps >= 2 && taps <= 4 && channels % 4 == 0 && ldi % 4 == 0 && ldo % 4 == 0 && aligned16(in) && aligned16(out) &&
        aligned16(state) && (!bias || aligned16(bias)) && (by_row ? rows : (tokens + kConvRun - 1) / kConvRun) <= 65535 &&
        (by_row || work >= kConvRunLeast)) {
        const unsigned gx = (unsigned)((channels / 4 + 255) / 256);
        const dim3 grid(gx, by_row ? rows : (tokens + kConvRun - 1) / kConvRun);
#define MV_CONV(T_)                                                                                                    \
    if (by_row) hipLaunchKernelGGL(conv_silu_row_kernel<T_>, grid, dim3(256), 0, s, in, ldi, state, w, bias, out, ldo, r, channels); \
    else hipLaunchKernelGGL(conv_silu_run_kernel<T_>, grid, dim3(256), 0, s, in, ldi, state, w, bias, out, ldo, r, tokens, channels)
        if (taps == 4) { MV_CONV(4); } else if (taps == 3) { MV_CONV(3); } else { MV_CONV(2); }
#undef MV_CONV
        if (by_row) return check_launch();
    } else {
        hipLaunchKernelGGL(conv_silu_kernel, dim3((unsigned)((work + 255) / 256)), dim3(256), 0, s, in, ldi, state, w, bias,
                           out, ldo, r, tokens, channels, taps);
    }
    if (taps > 1) {
        const int64_t w2 = (int64_t)rows * channels;
        hipLaunchKernelGGL(conv_state_update_kernel, dim3((unsigned)((w2 + 255) / 256)), dim3(256), 0, s, in, ldi, state,
                           r, rows, channels, taps);
    }
    return check_launch();
}

int mv_conv_taps(const float* in, int64_t ldi, float* state, const float* w, float* out32, int64_t ld32, void* out_act,
                 int64_t ldoa, int add_input, const int32_t* tok_row, const int32_t* row_start, const int32_t* row_len,
                 const int32_t* row_ctx, const int32_t* row_slot, int tokens, int rows, int channels, int taps, int f32,
                 mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || rows < 0 || channels <= 0 || taps < 1 || taps > kMaxTaps) return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!in || (!state && taps > 1) || !w || (!out32 && !out_act) || ldi < channels || (out32 && ld32 < channels) ||
        (out_act && ldoa < channels) || !tok_row || !row_start || !row_len || !row_ctx || !row_slot)
        return MV_ERR_INVALID_ARG;
    StepRows r{tok_row, nullptr, row_start, row_len, row_ctx, row_slot};
    hipStream_t s = (hipStream_t)stream;
    const int64_t work = (int64_t)tokens * channels;
    const dim3 grid((unsigned)((work + 255) / 256));
    if (f32) hipLaunchKernelGGL(conv_taps_kernel<true>, grid, dim3(256), 0, s, in, ldi, state, w, out32, ld32, out_act, ldoa, add_input, r, tokens, channels, taps);
    else hipLaunchKernelGGL(conv_taps_kernel<false>, grid, dim3(256), 0, s, in, ldi, state, w, out32, ld32, out_act, ldoa, add_input, r, tokens, channels, taps);
    if (taps > 1) {
        const int64_t w2 = (int64_t)rows * channels;
        hipLaunchKernelGGL(conv_state_update_kernel, dim3((unsigned)((w2 + 255) / 256)), dim3(256), 0, s, in, ldi, state,
                           r, rows, channels, taps);
    }
    return check_launch();
}

int mv_conv_qkv_store(const float* in, int64_t ldi, float* state, const float* w, float* q, int64_t ldq, void* k_cache,
                      void* v_cache, const int32_t* tok_row, const int32_t* tok_pos, const int32_t* row_start,
                      const int32_t* row_len, const int32_t* row_ctx, const int32_t* row_slot,
                      const int32_t* block_table, int bt_stride, int page, int tokens, int rows, int cq, int ck, int cv,
                      int taps, int f32, mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || rows < 0 || cq <= 0 || ck <= 0 || cv <= 0 || taps < 0 || taps > kMaxTaps || page <= 0)
        return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    const int C = cq + ck + cv;
    if (!in || ldi < C || (taps > 0 && !w) || (taps > 1 && !state) || !q || ldq < cq || !k_cache || !v_cache ||
        !tok_row || !tok_pos || !row_start || !row_len || !row_ctx || !row_slot || !block_table)
        return MV_ERR_INVALID_ARG;
    StepRows r{tok_row, tok_pos, row_start, row_len, row_ctx, row_slot};
    PagedRows pr{tok_row, tok_pos, block_table, bt_stride, page};
    hipStream_t s = (hipStream_t)stream;
    const int64_t work = (int64_t)tokens * C;
    const dim3 grid((unsigned)((work + 255) / 256));
    const float* wk = taps > 0 ? w : nullptr;
    if (f32) hipLaunchKernelGGL(conv_qkv_store_kernel<true>, grid, dim3(256), 0, s, in, ldi, state, wk, q, ldq, k_cache, v_cache, r, pr, tokens, cq, ck, cv, taps);
    else hipLaunchKernelGGL(conv_qkv_store_kernel<false>, grid, dim3(256), 0, s, in, ldi, state, wk, q, ldq, k_cache, v_cache, r, pr, tokens, cq, ck, cv, taps);
    if (taps > 1) {
        const int64_t w2 = (int64_t)rows * C;
        hipLaunchKernelGGL(conv_state_update_kernel, dim3((unsigned)((w2 + 255) / 256)), dim3(256), 0, s, in, ldi, state,
                           r, rows, C, taps);
    }
    return check_launch();
}

int mv_softplus_decay(const float* raw, int64_t ld, const float* dt_bias, const float* a_log, float* gain,
                      float* decay, float* log_decay, int tokens, int heads, mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || heads <= 0) return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!raw || !dt_bias || !a_log || !gain || !decay || ld < heads) return MV_ERR_INVALID_ARG;
    const DecayArgs d{raw, dt_bias, a_log, ld, gain, decay, log_decay, heads};
    hipLaunchKernelGGL(softplus_decay_kernel, dim3((tokens * heads + 255) / 256), dim3(256), 0, (hipStream_t)stream, d, tokens);
    return check_launch();
}

int mv_conv_silu_decay(const float* in, int64_t ldi, float* state, const float* w, const float* bias, float* out, int64_t ldo,
                       const int32_t* tok_row, const int32_t* row_start, const int32_t* row_len, const int32_t* row_ctx,
                       const int32_t* row_slot, int tokens, int rows, int channels, int taps, const float* raw, int64_t ld_raw,
                       const float* dt_bias, const float* a_log, float* gain, float* decay, float* log_decay, int heads,
                       mv_stream_t stream) {
    using namespace mv;
    const bool one = tokens > 0 && tokens <= rows && rows <= 65535 && taps >= 2 && taps <= 4 && channels > 0 && channels % 4 == 0 &&
                     ldi % 4 == 0 && ldo % 4 == 0 && aligned16(in) && aligned16(out) && aligned16(state) && (!bias || aligned16(bias));
    if (!one) {      // prompts, and what the vector form of the convolution does not take: two launches
        const int rc = mv_conv_silu(in, ldi, state, w, bias, out, ldo, tok_row, row_start, row_len, row_ctx, row_slot, tokens, rows,
                                    channels, taps, stream);
        return rc != MV_OK ? rc : mv_softplus_decay(raw, ld_raw, dt_bias, a_log, gain, decay, log_decay, tokens, heads, stream);
    }
    if (!in || !state || !w || !out || ldi < channels || ldo < channels) return MV_ERR_INVALID_ARG;
    if (heads <= 0 || !raw || !dt_bias || !a_log || !gain || !decay || ld_raw < heads) return MV_ERR_INVALID_ARG;
    const StepRows r{tok_row, nullptr, row_start, row_len, row_ctx, row_slot};
    const DecayArgs d{raw, dt_bias, a_log, ld_raw, gain, decay, log_decay, heads};
    const int conv = (channels / 4 + 255) / 256;
    const dim3 grid(conv + (heads + 255) / 256, rows);
    const auto kernel = taps == 4 ? conv_decay_row_kernel<4> : taps == 3 ? conv_decay_row_kernel<3> : conv_decay_row_kernel<2>;
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, in, ldi, state, w, bias, out, ldo, r, channels, conv, d);
    return check_launch();
}

int mv_scan_outer(const float* q, int64_t ldq, int q_div, const float* k, int64_t ldk, int k_div, const float* v,
                  int64_t ldv, const float* decay, int64_t ld_decay, const float* gain, int64_t ld_gain,
                  const float* skip, float* state, float* out, int64_t ldo, const int32_t* row_start,
                  const int32_t* row_len, const int32_t* row_ctx, const int32_t* row_slot, int rows, int heads, int n,
                  int p, int max_len, mv_stream_t stream) {
    using namespace mv;
    if (rows < 0 || heads <= 0 || n <= 0 || p <= 0 || q_div <= 0 || k_div <= 0) return MV_ERR_INVALID_ARG;
    if (rows == 0) return MV_OK;
    if (!q || !k || !v || !decay || !state || !out || rows > 65535 || heads > 65535) return MV_ERR_INVALID_ARG;
    ScanArgs a;
    a.q = q; a.k = k; a.v = v; a.decay = decay; a.gain = gain; a.skip = skip;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.ld_decay = ld_decay; a.ld_gain = ld_gain; a.ldo = ldo;
    a.q_div = q_div; a.k_div = k_div; a.state = state; a.out = out;
    a.r = StepRows{nullptr, nullptr, row_start, row_len, row_ctx, row_slot};
    a.H = heads; a.n = n; a.p = p; a.max_len = max_len;
    a.ch_start = nullptr; a.ch_len = nullptr; a.ds = nullptr;
    if ((n == 64 || n == 128 || n == 256) && p % 64 == 0 && ldq % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 && ldo % 4 == 0 &&
        aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out) && aligned16(state)) {
        const dim3 vgrid(p / 64, heads, rows);
        if (n == 64) hipLaunchKernelGGL(scan_outer_vec_kernel<4>, vgrid, dim3(256), 0, (hipStream_t)stream, a);
        else if (n == 128) hipLaunchKernelGGL(scan_outer_vec_kernel<8>, vgrid, dim3(256), 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL(scan_outer_vec_kernel<16>, vgrid, dim3(256), 0, (hipStream_t)stream, a);
        return check_launch();
    }
    a.pt = p % 64 == 0 ? 64 : (p % 32 == 0 ? 32 : 16);
    // a state too tall for 64 rows a thread: narrower column tiles leave more threads to share its rows
    while (a.pt > 16 && (n + 256 / a.pt - 1) / (256 / a.pt) > 64) a.pt /= 2;
    const int ns = 256 / a.pt, npt = (n + ns - 1) / ns;
    const dim3 grid((p + a.pt - 1) / a.pt, heads, rows);
    hipStream_t s = (hipStream_t)stream;
    if (npt <= 4) hipLaunchKernelGGL((scan_outer_kernel<4, false>), grid, dim3(256), 0, s, a);
    else if (npt <= 16) hipLaunchKernelGGL((scan_outer_kernel<16, false>), grid, dim3(256), 0, s, a);
    else if (npt <= 64) hipLaunchKernelGGL((scan_outer_kernel<64, false>), grid, dim3(256), 0, s, a);
    else return MV_ERR_UNSUPPORTED;
    return check_launch();
}

int mv_scan_gated(const float* q, int64_t ldq, const float* f, int64_t ldf, const float* v, int64_t ldv, float* state,
                  float* out, int64_t ldo, const int32_t* row_start, const int32_t* row_len, const int32_t* row_ctx,
                  const int32_t* row_slot, int rows, int heads, int n, int p, float* ds, float* cum,
                  const int32_t* ch_start, const int32_t* ch_len, const int32_t* row_ch0, const int32_t* row_nch,
                  int chunks, int max_len, mv_stream_t stream) {
    using namespace mv;
    if (rows < 0 || heads <= 0 || n <= 0 || p <= 0 || chunks < 0) return MV_ERR_INVALID_ARG;
    if (rows == 0) return MV_OK;
    if (!q || !f || !v || !state || !out || rows > 65535 || heads > 65535 || chunks > 65535) return MV_ERR_INVALID_ARG;
    if (ldq < (int64_t)heads * n || ldf < (int64_t)heads * n || ldv < (int64_t)heads * p || ldo < (int64_t)heads * p)
        return MV_ERR_INVALID_ARG;
    if (chunks > 0 && (!ds || !cum || !ch_start || !ch_len || !row_ch0 || !row_nch || max_len <= 0))
        return MV_ERR_INVALID_ARG;
    ScanArgs a;
    a.q = q; a.k = nullptr; a.v = v; a.decay = f; a.gain = nullptr; a.skip = nullptr;
    a.ldq = ldq; a.ldk = 0; a.ldv = ldv; a.ld_decay = ldf; a.ld_gain = 0; a.ldo = ldo;
    a.q_div = 1; a.k_div = 1; a.state = state; a.out = out;
    a.r = StepRows{nullptr, nullptr, row_start, row_len, row_ctx, row_slot};
    a.H = heads; a.n = n; a.p = p; a.max_len = chunks > 0 ? max_len : 0;
    a.ch_start = nullptr; a.ch_len = nullptr; a.ds = nullptr;
    hipStream_t s = (hipStream_t)stream;
    // rows of up to max_len tokens (all rows when nothing is cut into chunks): token by token from the slot's state
    for (int pass = 0; pass < (chunks > 0 ? 2 : 1); ++pass) {
        if (pass == 1) {
            a.ch_start = ch_start; a.ch_len = ch_len; a.ds = ds;
        }
        const int units = pass == 0 ? rows : chunks;
        a.pt = p % 64 == 0 ? 64 : (p % 32 == 0 ? 32 : 16);
        // a state too tall for 64 rows a thread: narrower column tiles leave more threads to share its rows; so do
        // launches that would not fill the chip otherwise (a few decoded tokens: the step is the state's traffic)
        while (a.pt > 16 && ((n + 256 / a.pt - 1) / (256 / a.pt) > 64 ||
                             (int64_t)((p + a.pt - 1) / a.pt) * heads * units < 2 * (int64_t)num_cus()))
            a.pt /= 2;
        const int ns = 256 / a.pt, npt = (n + ns - 1) / ns;
        if (npt > 64) return MV_ERR_UNSUPPORTED;
        const dim3 grid((p + a.pt - 1) / a.pt, heads, units);
        if (npt <= 4) hipLaunchKernelGGL((scan_outer_kernel<4, true>), grid, dim3(256), 0, s, a);
        else if (npt <= 16) hipLaunchKernelGGL((scan_outer_kernel<16, true>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((scan_outer_kernel<64, true>), grid, dim3(256), 0, s, a);
    }
    if (chunks > 0) {
        const int width = heads * n;
        hipLaunchKernelGGL(gate_cumprod_kernel, dim3(chunks, (width + 255) / 256), dim3(256), 0, s, f, ldf, cum,
                           (int64_t)width, ch_start, ch_len, width);
        GatedChunkArgs g;
        g.q = q; g.cum = cum; g.ldq = ldq; g.ldc = width; g.ldo = ldo; g.state = state; g.out = out; g.ds = ds;
        g.ch_start = ch_start; g.ch_len = ch_len; g.row_ch0 = row_ch0; g.row_nch = row_nch; g.row_ctx = row_ctx;
        g.row_slot = row_slot; g.H = heads; g.n = n; g.p = p;
        hipLaunchKernelGGL(gated_carry_kernel, dim3((n * p + 255) / 256, heads, rows), dim3(256), 0, s, g);
        hipLaunchKernelGGL(gated_inter_kernel, dim3(chunks, heads, (p + 63) / 64), dim3(256), 0, s, g);
    }
    return check_launch();
}

int mv_gate_lower_bound(float* q, int64_t ldq, float* f, int64_t ldf, const float* bias, const float* lower,
                        int tokens, int n, mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || n <= 0) return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!q || !f || !lower || ldq < n || ldf < n) return MV_ERR_INVALID_ARG;
    const int64_t total = (int64_t)tokens * n;
    hipLaunchKernelGGL(gate_lower_bound_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, q, ldq, f, ldf, bias, lower, tokens, n);
    return check_launch();
}

size_t mv_scan_chunked_lds_bytes(int n, int p) {
    const int n4 = (n + 3) & ~3;
    const size_t intra = (size_t)(2 * mv::kCh * (n4 + 1) + mv::kCh * (p + 1) + 3 * mv::kCh) * sizeof(float);
    const size_t inter = (size_t)(mv::kCh * (n4 + 1) + n4 * (p + 1)) * sizeof(float);
    return intra > inter ? intra : inter;
}

int mv_scan_chunked(const float* q, int64_t ldq, int q_div, const float* k, int64_t ldk, int k_div, const float* v,
                    int64_t ldv, const float* log_decay, int64_t ld_ld, const float* gain, int64_t ld_gain,
                    const float* skip, float* state, float* out, int64_t ldo, float* ds, float* lsum, float* atot,
                    const int32_t* ch_start, const int32_t* ch_len, const int32_t* row_ch0, const int32_t* row_nch,
                    const int32_t* row_ctx, const int32_t* row_slot, int chunks, int rows, int heads, int n, int p,
                    mv_stream_t stream) {
    using namespace mv;
    if (chunks < 0 || rows < 0 || heads <= 0 || n <= 0 || p <= 0 || q_div <= 0 || k_div <= 0) return MV_ERR_INVALID_ARG;
    if (chunks == 0) return MV_OK;
    if (!q || !k || !v || !log_decay || !state || !out || !ds || !lsum || !atot || !ch_start || !ch_len || !row_ch0 ||
        !row_nch || rows > 65535 || heads > 65535)
        return MV_ERR_INVALID_ARG;
    const int n4 = (n + 3) & ~3;
    const size_t lds = (size_t)(2 * kCh * (n4 + 1) + kCh * (p + 1) + 3 * kCh) * sizeof(float);
    const size_t lds2 = (size_t)(kCh * (n4 + 1) + n4 * (p + 1)) * sizeof(float);
    if (mv_scan_chunked_lds_bytes(n, p) > 150 * 1024) return MV_ERR_UNSUPPORTED;
    static LdsOptIn opt1, opt2;
    if (int rc = ensure_dynamic_lds((const void*)scan_chunk_intra_kernel, lds, opt1)) return rc;
    if (int rc = ensure_dynamic_lds((const void*)scan_chunk_inter_kernel, lds2, opt2)) return rc;
    ChunkArgs a;
    a.q = q; a.k = k; a.v = v; a.log_decay = log_decay; a.gain = gain; a.skip = skip;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.ld_ld = ld_ld; a.ld_gain = ld_gain; a.ldo = ldo;
    a.q_div = q_div; a.k_div = k_div; a.state = state; a.out = out; a.ds = ds; a.lsum = lsum; a.atot = atot;
    a.ch_start = ch_start; a.ch_len = ch_len; a.row_ch0 = row_ch0; a.row_nch = row_nch;
    a.r = StepRows{nullptr, nullptr, nullptr, nullptr, row_ctx, row_slot};
    a.H = heads; a.n = n; a.p = p;
    // Whole rows in two launches where the shapes allow it and there are sixteen heads: a row's chunks come one after the
    // other there (about 3.5 us each), the three launches below take them side by side (about 0.2 us per chunk and head).
    const int groups = heads / q_div;
    if ((n == 64 || n == 128) && p % 16 == 0 && q_div == k_div && heads % q_div == 0 && ldq % 4 == 0 && ldk % 4 == 0 &&
        ldv % 4 == 0 && aligned16(q) && aligned16(k) && aligned16(v) && aligned16(ds) &&
        (int64_t)groups * kCh * kCh <= (int64_t)heads * n * p && groups <= 65535 && heads >= 16 &&
        (int64_t)heads * (p / 16) <= 0x7fffffff) {
        hipStream_t s = (hipStream_t)stream;
        hipLaunchKernelGGL(scan_scores_kernel, dim3(chunks, groups, 4), dim3(256), 0, s, a, ds);
        const bool wide = p % 32 == 0 && (int64_t)heads * (p / 32) * rows >= num_cus();
        const dim3 grid((unsigned)(heads * (p / (wide ? 32 : 16))), rows);
        if (n == 64) {
            if (wide) hipLaunchKernelGGL((scan_rows_kernel<4, 2>), grid, dim3(512), 0, s, a, ds, groups);
            else hipLaunchKernelGGL((scan_rows_kernel<4, 1>), grid, dim3(512), 0, s, a, ds, groups);
        } else {
            if (wide) hipLaunchKernelGGL((scan_rows_kernel<8, 2>), grid, dim3(512), 0, s, a, ds, groups);
            else hipLaunchKernelGGL((scan_rows_kernel<8, 1>), grid, dim3(512), 0, s, a, ds, groups);
        }
        return check_launch();
    }
    // heads that read the same q and k (a group) go four or two to a workgroup
    a.hb = (q_div == k_div && heads % q_div == 0) ? (q_div % 4 == 0 ? 4 : (q_div % 2 == 0 ? 2 : 1)) : 1;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(scan_chunk_intra_kernel, dim3(chunks, heads / a.hb), dim3(256), lds, s, a);
    hipLaunchKernelGGL(scan_chunk_carry_kernel, dim3((n * p + 255) / 256, heads, rows), dim3(256), 0, s, a);
    hipLaunchKernelGGL(scan_chunk_inter_kernel, dim3(chunks, heads / a.hb), dim3(256), lds2, s, a);
    return check_launch();
}

int mv_rotary_pairs(float* x, int64_t ld, const double* inv_freq, const int32_t* tok_pos, int tokens, int heads,
                    int dim, int rot, float scale, mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || heads <= 0 || dim <= 0 || rot < 0 || rot > dim || rot % 2) return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!x || !tok_pos || (rot > 0 && !inv_freq) || ld < (int64_t)heads * dim) return MV_ERR_INVALID_ARG;
    const int64_t work = (int64_t)tokens * heads * (dim - rot / 2);
    hipLaunchKernelGGL(rotary_pairs_kernel, dim3((unsigned)((work + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x,
                       ld, inv_freq, tok_pos, tokens, heads, dim, rot, scale);
    return check_launch();
}

int mv_gated_group_norm(const float* y, int64_t ldy, const float* gate, int64_t ldg, const float* w, void* out,
                        int64_t ldo, int rows, int n, int groups, int mode, int w_shared, float eps, int f32,
                        mv_stream_t stream) {
    using namespace mv;
    if (rows < 0 || n <= 0 || groups <= 0 || n % groups || mode < 0 || mode > 2) return MV_ERR_INVALID_ARG;
    if (rows == 0) return MV_OK;
    if (!y || !gate || !out || ldy < n || ldg < n || ldo < n) return MV_ERR_INVALID_ARG;
    const int64_t units = (int64_t)rows * groups;
    hipStream_t s = (hipStream_t)stream;
    if (n / groups >= 1024) {
        const dim3 wide((unsigned)units);
        const int gs = n / groups;
        const bool few = units <= num_cus(), vec = gs % 4 == 0 && ldy % 4 == 0 && ldg % 4 == 0 && ldo % 4 == 0 && aligned16(y) &&
                                                   aligned16(gate) && aligned16(out) && (!w || aligned16(w));
        const int pieces = (gs + (few ? 4096 : 1024) - 1) / (few ? 4096 : 1024);     // of four values a thread
        if (vec && pieces <= 8) {
#define MV_GGN(F32_, NT_, V_)                                                                                          \
    hipLaunchKernelGGL((gated_group_norm_reg_kernel<F32_, NT_, V_>), wide, dim3(NT_), 0, s, y, ldy, gate, ldg, w, out, ldo, n, \
                       groups, mode, w_shared, eps)
#define MV_GGN_V(F32_, NT_)                                                                                            \
    do {                                                                                                               \
        if (pieces == 1) MV_GGN(F32_, NT_, 1);                                                                         \
        else if (pieces == 2) MV_GGN(F32_, NT_, 2);                                                                    \
        else if (pieces <= 4) MV_GGN(F32_, NT_, 4);                                                                    \
        else MV_GGN(F32_, NT_, 8);                                                                                     \
    } while (0)
            if (f32) { if (few) MV_GGN_V(true, 1024); else MV_GGN_V(true, 256); }
            else { if (few) MV_GGN_V(false, 1024); else MV_GGN_V(false, 256); }
#undef MV_GGN_V
#undef MV_GGN
            return check_launch();
        }
        if (f32) hipLaunchKernelGGL(gated_group_norm_wide_kernel<true>, wide, dim3(256), 0, s, y, ldy, gate, ldg, w, out, ldo, n, groups, mode, w_shared, eps);
        else hipLaunchKernelGGL(gated_group_norm_wide_kernel<false>, wide, dim3(256), 0, s, y, ldy, gate, ldg, w, out, ldo, n, groups, mode, w_shared, eps);
        return check_launch();
    }
    const dim3 grid((unsigned)((units + 3) / 4));
    if (f32) hipLaunchKernelGGL(gated_group_norm_kernel<true>, grid, dim3(256), 0, s, y, ldy, gate, ldg, w, out, ldo, rows, n, groups, mode, w_shared, eps);
    else hipLaunchKernelGGL(gated_group_norm_kernel<false>, grid, dim3(256), 0, s, y, ldy, gate, ldg, w, out, ldo, rows, n, groups, mode, w_shared, eps);
    return check_launch();
}

int mv_qk_unitnorm_store(float* qkv, int64_t ld, void* k_cache, void* v_cache, const int32_t* tok_row,
                         const int32_t* tok_pos, const int32_t* block_table, int bt_stride, int page, int tokens,
                         int heads, int kv_heads, int d, int dv, float eps, int f32, mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || heads <= 0 || kv_heads <= 0 || d <= 0 || dv <= 0 || page <= 0 || heads % kv_heads)
        return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!qkv || !k_cache || !v_cache || !tok_row || !tok_pos || !block_table ||
        ld < (int64_t)(heads + kv_heads) * d + (int64_t)kv_heads * dv)
        return MV_ERR_INVALID_ARG;
    PagedRows pr{tok_row, tok_pos, block_table, bt_stride, page};
    const int64_t units = (int64_t)tokens * (heads + 2 * kv_heads);
    const dim3 grid((unsigned)((units + 3) / 4));
    hipStream_t s = (hipStream_t)stream;
    if (f32) hipLaunchKernelGGL(qk_unitnorm_store_kernel<true>, grid, dim3(256), 0, s, qkv, ld, k_cache, v_cache, pr, tokens, heads, kv_heads, d, dv, eps);
    else hipLaunchKernelGGL(qk_unitnorm_store_kernel<false>, grid, dim3(256), 0, s, qkv, ld, k_cache, v_cache, pr, tokens, heads, kv_heads, d, dv, eps);
    return check_launch();
}

int mv_qk_rotary_store(float* qk, int64_t ld, const float* q_bias, const float* k_bias, void* k_cache, void* v_cache,
                       const double* inv_freq, const int32_t* tok_row, const int32_t* tok_pos,
                       const int32_t* block_table, int bt_stride, int page, int tokens, int heads, int kv_heads, int d,
                       int rot, int adjacent, const float* act_in, int64_t lda, void* act_out, int64_t ldao, int act_n,
                       int act_kind, float act_limit, float act_slope, int f32, mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || heads <= 0 || kv_heads <= 0 || d <= 0 || page <= 0 || rot < 0 || rot > d || rot % 2)
        return MV_ERR_INVALID_ARG;
    if (act_in && (!act_out || act_n <= 0 || lda < 2 * (int64_t)act_n || ldao < act_n || act_kind < 0 || act_kind > 2))
        return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!qk || !k_cache || !v_cache || (rot > 0 && !inv_freq) || !tok_row || !tok_pos || !block_table ||
        ld < (int64_t)(heads + kv_heads) * d)
        return MV_ERR_INVALID_ARG;
    PagedRows pr{tok_row, tok_pos, block_table, bt_stride, page};
    // steps of many tokens: a wave takes eight heads of a token and forms the angles' sines and cosines once for them
    const int hpw = (int64_t)tokens * (heads + kv_heads) >= 8 * 1024 ? 8 : 1;
    const int64_t units = (int64_t)tokens * ((heads + kv_heads + hpw - 1) / hpw);
    const int64_t rot_blocks = (units + 3) / 4, act_blocks = act_in ? (int64_t)tokens * ((act_n + 255) / 256) : 0;
    if (rot_blocks + act_blocks > 0x7fffffff) return MV_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)(rot_blocks + act_blocks));
    hipStream_t s = (hipStream_t)stream;
    if (f32) hipLaunchKernelGGL(qk_rotary_store_kernel<true>, grid, dim3(256), 0, s, qk, ld, q_bias, k_bias, k_cache, v_cache, inv_freq, pr, tokens, heads, kv_heads, d, rot, adjacent, hpw, (unsigned)rot_blocks, act_in, lda, act_out, ldao, act_n, act_kind, act_limit, act_slope);
    else hipLaunchKernelGGL(qk_rotary_store_kernel<false>, grid, dim3(256), 0, s, qk, ld, q_bias, k_bias, k_cache, v_cache, inv_freq, pr, tokens, heads, kv_heads, d, rot, adjacent, hpw, (unsigned)rot_blocks, act_in, lda, act_out, ldao, act_n, act_kind, act_limit, act_slope);
    return check_launch();
}

int mv_qkv_norm_rotary_store(float* qkv, int64_t ld, const float* q_bias, const float* k_bias, const float* v_bias,
                             const float* q_norm, const float* k_norm, float eps, const double* inv_freq,
                             float* v_first, int mix, float lam, void* k_cache, void* v_cache, const int32_t* tok_row,
                             const int32_t* tok_pos, const int32_t* block_table, int bt_stride, int page, int tokens,
                             int heads, int kv_heads, int d, int dv, int rot, int adjacent, int f32,
                             mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || d <= 0 || dv <= 0 || page <= 0 || rot < 0 ||
        rot > d || rot % 2 || rot > 8192 || mix < 0 || mix > 2)
        return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!qkv || ld < (int64_t)(heads + kv_heads) * d + (int64_t)kv_heads * dv || !k_cache || !v_cache || !tok_row ||
        !tok_pos || !block_table || (rot > 0 && !inv_freq) || (mix && !v_first))
        return MV_ERR_INVALID_ARG;
    PagedRows pr{tok_row, tok_pos, block_table, bt_stride, page};
    const size_t lds = (size_t)(rot > 0 ? rot : 1) * sizeof(float);
    const int nt = tokens <= 512 ? 1024 : 256;      // a token of a short step has its workgroup to itself on a compute unit
    hipStream_t s = (hipStream_t)stream;
    if (f32) hipLaunchKernelGGL(qkv_norm_rotary_store_kernel<true>, dim3(tokens), dim3(nt), lds, s, qkv, ld, q_bias, k_bias, v_bias, q_norm, k_norm, eps, inv_freq, v_first, mix, lam, k_cache, v_cache, pr, heads, kv_heads, d, dv, rot, adjacent);
    else hipLaunchKernelGGL(qkv_norm_rotary_store_kernel<false>, dim3(tokens), dim3(nt), lds, s, qkv, ld, q_bias, k_bias, v_bias, q_norm, k_norm, eps, inv_freq, v_first, mix, lam, k_cache, v_cache, pr, heads, kv_heads, d, dv, rot, adjacent);
    return check_launch();
}

int mv_qkv_headnorm_rotary_store(float* qkv, int64_t ld, const float* q_bias, const float* k_bias, const float* v_bias,
                                 const float* q_norm, const float* k_norm, float eps, const double* inv_freq,
                                 void* k_cache, void* v_cache, const int32_t* tok_row, const int32_t* tok_pos,
                                 const int32_t* block_table, int bt_stride, int page, int tokens, int heads,
                                 int kv_heads, int d, int dv, int rot, int adjacent, const float* low, int64_t ldl,
                                 void* low_out, int low_n, int f32, mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || d <= 0 || dv <= 0 || page <= 0 || rot < 0 ||
        rot > d || rot % 2 || low_n < 0)
        return MV_ERR_INVALID_ARG;
    if (d - rot / 2 > 512) return MV_ERR_UNSUPPORTED;
    if (tokens == 0) return MV_OK;
    if (!qkv || ld < (int64_t)(heads + kv_heads) * d + (int64_t)kv_heads * dv || !k_cache || !v_cache || !tok_row ||
        !tok_pos || !block_table || (rot > 0 && !inv_freq) || (low_n > 0 && (!low || !low_out || ldl < low_n)))
        return MV_ERR_INVALID_ARG;
    PagedRows pr{tok_row, tok_pos, block_table, bt_stride, page};
    const int units = heads + 2 * kv_heads + (low_n > 0 ? 1 : 0);
    // steps of many tokens: a wave takes eight heads of a token and forms the angles' sines and cosines once for them
    const int hpw = (int64_t)tokens * units >= 8 * 1024 ? 8 : 1;
    const int64_t blocks = ((int64_t)tokens * ((units + hpw - 1) / hpw) + 3) / 4;
    if (blocks > 0x7fffffff) return MV_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)blocks);
    hipStream_t s = (hipStream_t)stream;
    const int items = d - rot / 2;
#define MV_HEADNORM(F32_, NI_)                                                                                       \
    hipLaunchKernelGGL((qkv_headnorm_rotary_store_kernel<F32_, NI_>), grid, dim3(256), 0, s, qkv, ld, q_bias, k_bias,   \
                       v_bias, q_norm, k_norm, eps, inv_freq, k_cache, v_cache, pr, tokens, heads, kv_heads, d, dv, rot, \
                       adjacent, hpw, low, ldl, low_out, low_n)
#define MV_HEADNORM_N(F32_)                                                                                          \
    do {                                                                                                           \
        if (items <= 64) MV_HEADNORM(F32_, 1);                                                                       \
        else if (items <= 128) MV_HEADNORM(F32_, 2);                                                                 \
        else MV_HEADNORM(F32_, 8);                                                                                   \
    } while (0)
    if (f32) MV_HEADNORM_N(true);
    else MV_HEADNORM_N(false);
#undef MV_HEADNORM_N
#undef MV_HEADNORM
    return check_launch();
}

// Sixteen waves (eight where the registers of fp32 rows or of eight heads allow no more) while every workgroup has
// a compute unit to itself, else four.  One split while the window is up to 1280 keys, five tiles to a wave (640
// with fp32 rows, twice as long to read, and with eight waves): a merge is a launch more, 2 of 10 us at 45 keys.
// Past that one to 256 keys of the window, but no more workgroups than compute units, where a second round of
// them costs more than the splits give.  One token of bf16 at 2000 keys, window 2047, in one split and in eight
// (us): 8 heads of 128 on 2 29.6, 16.9; 16 on 2 51.8, 21.0; 8 heads of 64 on 8 18.6, 11.2 (in 64-key tiles 27.3, 34.8, 13.5);
// 32 tokens at 4000, 16 heads on 2, in one, four and eight splits 56.5, 28.3, 41.0; one fp32 token at 1100, window 1024, 8 heads on
// 2, in one, two and four splits 27.3, 21.8, 17.9.
struct FewPlan {
    int64_t groups;      // workgroups of a split
    int pieces, top;     // splits; query heads of a workgroup
    bool wide;
};
static FewPlan few_plan(int tokens, int heads, int kv_heads, int window, int keep_first, int f32, int splits) {
    const int R = heads / kv_heads, ngrp = (R + mv::kGrpMax - 1) / mv::kGrpMax, top = R < mv::kGrpMax ? R : mv::kGrpMax;
    const int64_t groups = (int64_t)tokens * kv_heads * ngrp;
    const int64_t keys = (int64_t)window + keep_first, room = mv::num_cus() / groups;
    int64_t want = keys <= (f32 || top > 4 ? 640 : 1280) ? 1 : (keys + 128) / 256;
    if (want > room) want = room;
    if (want > splits) want = splits;
    const int pieces = want < 1 ? 1 : (int)want;
    return FewPlan{groups, pieces, top, groups * pieces <= mv::num_cus()};
}

int mv_window_attn_splits(int tokens, int heads, int kv_heads, int window, int keep_first) {
    using namespace mv;
    if (tokens <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || window <= 0 || keep_first < 0) return 1;
    const int R = heads / kv_heads, ngrp = (R + kGrpMax - 1) / kGrpMax;
    const int64_t units = (int64_t)tokens * kv_heads * ngrp;
    const int64_t tiles = ((int64_t)window + keep_first) / 64 + 2;      // at most this many 64-key tiles a token
    int64_t want = (2 * (int64_t)num_cus() + units - 1) / units;         // about two workgroups a compute unit
    const int64_t most = (tiles + 3) / 4;                                // a wave should find a tile of its own
    if (want > most) want = most;
    if (want > 64) want = 64;
    return want < 1 ? 1 : (int)want;
}

int mv_window_attn(const float* q, int64_t ldq, const void* k_cache, const void* v_cache, void* out, int64_t ldo,
                   const int32_t* tok_row, const int32_t* tok_pos, const int32_t* block_table, int bt_stride,
                   int page, const float* slopes, int tokens, int heads, int kv_heads, int d, int dv, float scale,
                   int window, int f32, const int32_t* row_len, const int32_t* ch_start, const int32_t* ch_len,
                   int chunks, int max_len, int keep_first, const float* sinks, float* part, int splits,
                   int short_tokens, const float* gate, int64_t ldg, int chunked, mv_stream_t stream) {
    using namespace mv;
    if (gate && ldg < (int64_t)heads * dv) return MV_ERR_INVALID_ARG;
    if (tokens < 0 || heads <= 0 || kv_heads <= 0 || d <= 0 || dv <= 0 || page <= 0 || window <= 0 ||
        heads % kv_heads || keep_first < 0)
        return MV_ERR_INVALID_ARG;
    if (dv > 64 * kMaxVC || d > 4096) return MV_ERR_UNSUPPORTED;
    if (tokens == 0) return MV_OK;
    if (!q || !k_cache || !v_cache || !out || !tok_row || !tok_pos || !block_table) return MV_ERR_INVALID_ARG;
    PagedRows pr{tok_row, tok_pos, block_table, bt_stride, page};
    const int64_t units = (int64_t)tokens * heads;
    if (units > 0x7fffffff) return MV_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)units);
    hipStream_t s = (hipStream_t)stream;
    // rows of more than max_len tokens, cut into the chunks of the table: the tiled matrix-core kernel, where
    // the shapes are among those it is built for (bf16, 64-token pages, 16-byte rows)
    int skip_len = 0;
    if (!f32 && chunks > 0 && max_len > 0 && row_len && ch_start && ch_len && page == 64 && ldq % 4 == 0 &&
        ldo % 4 == 0 && aligned16(q) && aligned16(k_cache) && aligned16(v_cache) && (reinterpret_cast<uintptr_t>(out) & 7) == 0) {
        const dim3 tg(chunks, heads);
#define MV_WA_TILE(KS_, CT_)                                                                                         \
    hipLaunchKernelGGL((window_attn_tile_kernel<KS_, CT_>), tg, dim3(256), 0, s, q, ldq, (const uint16_t*)k_cache,      \
                       (const uint16_t*)v_cache, (uint16_t*)out, ldo, pr, ch_start, ch_len, slopes, heads, kv_heads, scale, \
                       window, keep_first, sinks, gate, ldg, chunked);                                                                \
    skip_len = max_len
        if (d == 64 && dv == 64) { MV_WA_TILE(2, 4); }
        else if (d == 96 && dv == 96) { MV_WA_TILE(3, 6); }
        else if (d == 128 && dv == 128) { MV_WA_TILE(4, 8); }
        else if (d == 128 && dv == 64) { MV_WA_TILE(4, 4); }
        else if (d == 64 && dv == 128) { MV_WA_TILE(2, 8); }
        else if (d == 32 && dv == 32) { MV_WA_TILE(1, 2); }
        else if (d == 64 && dv == 32) { MV_WA_TILE(2, 2); }
#undef MV_WA_TILE
        // every row of the step was long enough for the tiles: nothing is left for the per-token forms
        if (skip_len > 0 && short_tokens == 0) return check_launch();
    }
    // with a place for the splits' pieces: the kernel that shares every key among the query heads of its key/value
    // head and cuts the keys over several workgroups
    if (part && splits >= 1) {
        const int R = heads / kv_heads, ngrp = (R + kGrpMax - 1) / kGrpMax, top = R < kGrpMax ? R : kGrpMax;
        auto merge = [&](int pieces, int nw) {
#define MV_WA_MERGE(F32_)                                                                                              \
    hipLaunchKernelGGL(window_attn_merge_kernel<F32_>, grid, dim3(64), 0, s, part, out, ldo, tok_row, tok_pos, sinks, heads, \
                       dv, pieces, nw, window, keep_first, chunked, row_len, skip_len, gate, ldg)
            if (f32) MV_WA_MERGE(true);
            else MV_WA_MERGE(false);
#undef MV_WA_MERGE
        };
        if (aligned16(q) && ldq % 4 == 0 && aligned16(k_cache) && aligned16(v_cache)) {
            const FewPlan fp = few_plan(tokens, heads, kv_heads, window, keep_first, f32, splits);
            const int64_t groups = fp.groups;
            const int pieces = fp.pieces;
            const bool wide = fp.wide;
            int nw = 0;      // (0: a head shape without an instance)
#define MV_WA_FEW(F32_, HB_, NW_, KS_, VE_, OWN_)                                                                      \
    hipLaunchKernelGGL((window_attn_few_kernel<F32_, HB_, NW_, KS_, VE_, false, OWN_>), dim3((unsigned)groups, pieces), dim3(64 * NW_), 0, s, \
                       q, ldq, k_cache, v_cache, out, ldo, part, pr, slopes, sinks, heads, kv_heads, scale, window, keep_first, \
                       row_len, skip_len, pieces, gate, ldg, chunked, StepRotary{});                                   \
    nw = NW_
#define MV_WA_FEW_HB(F32_, KS_, VE_)                                                                                   \
    do {                                                                                                               \
        constexpr bool own = !F32_ && KS_ == 2;      /* of two or three heads to a key */                              \
        if (top > 4) { if (wide) { MV_WA_FEW(F32_, 8, 8, KS_, VE_, false); } else { MV_WA_FEW(F32_, 8, 4, KS_, VE_, false); } } \
        else if (top == 4) { if (wide) { MV_WA_FEW(F32_, 4, (F32_ ? 8 : 16), KS_, VE_, false); } else { MV_WA_FEW(F32_, 4, 4, KS_, VE_, false); } } \
        else if (top > 1) { if (wide) { MV_WA_FEW(F32_, 4, (F32_ ? 8 : 16), KS_, VE_, own); } else { MV_WA_FEW(F32_, 4, 4, KS_, VE_, own); } } \
        else if (wide) { MV_WA_FEW(F32_, 1, 16, KS_, VE_, false); }                                                    \
        else { MV_WA_FEW(F32_, 1, 4, KS_, VE_, false); }                                                               \
    } while (0)
#define MV_WA_FEW_D(F32_)                                                                                              \
    do {                                                                                                               \
        if (d == 128 && dv == 128) MV_WA_FEW_HB(F32_, 4, 8);                                                           \
        else if (d == 64 && dv == 64) MV_WA_FEW_HB(F32_, 2, 4);                                                        \
        else if (d == 96 && dv == 96) MV_WA_FEW_HB(F32_, 3, 6);                                                        \
        else if (d == 128 && dv == 64) MV_WA_FEW_HB(F32_, 4, 4);                                                       \
        else if (d == 64 && dv == 128) MV_WA_FEW_HB(F32_, 2, 8);                                                       \
        else if (d == 32 && dv == 32) MV_WA_FEW_HB(F32_, 1, 2);                                                        \
        else if (d == 64 && dv == 32) MV_WA_FEW_HB(F32_, 2, 2);                                                        \
    } while (0)
            if (f32) MV_WA_FEW_D(true);
            else MV_WA_FEW_D(false);
#undef MV_WA_FEW_D
#undef MV_WA_FEW_HB
#undef MV_WA_FEW
            if (nw) {
                if (pieces > 1) merge(pieces, nw);
                return check_launch();
            }
        }
        const int rt = top <= 1 ? 1 : top <= 2 ? 2 : top <= 4 ? 4 : 8;
        const int vecw = f32 ? 4 : 8;
        const int vec = dv % vecw == 0 && dv / vecw <= 64 && aligned16(v_cache);
        const size_t glds = ((size_t)rt * d + 4 * rt * 64 + 4 * (size_t)rt * dv + 8 * rt) * sizeof(float);
        if (glds <= 64 * 1024 && d % 4 == 0 && ldq % 4 == 0 && aligned16(q) && (f32 || d % 8 != 0 || aligned16(k_cache))) {
            const dim3 gg((unsigned)(tokens * kv_heads * ngrp), splits);
#define MV_WA_GROUP(F32_, RT_)                                                                                         \
    hipLaunchKernelGGL((window_attn_group_kernel<F32_, RT_>), gg, dim3(256), glds, s, q, ldq, k_cache, v_cache, out, ldo, \
                       part, pr, slopes, sinks, heads, kv_heads, d, dv, scale, window, keep_first, row_len, skip_len,   \
                       splits, vec, gate, ldg, chunked)
            if (f32) {
                if (rt == 1) MV_WA_GROUP(true, 1); else if (rt == 2) MV_WA_GROUP(true, 2);
                else if (rt == 4) MV_WA_GROUP(true, 4); else MV_WA_GROUP(true, 8);
            } else {
                if (rt == 1) MV_WA_GROUP(false, 1); else if (rt == 2) MV_WA_GROUP(false, 2);
                else if (rt == 4) MV_WA_GROUP(false, 4); else MV_WA_GROUP(false, 8);
            }
#undef MV_WA_GROUP
            if (splits > 1) merge(splits, 0);
            return check_launch();
        }
    }
    // few (token, head) pairs and a window of many tiles: sixteen waves share it
    const bool wide = units <= 2 * num_cus() && window > 256;
    const int nw = wide ? 16 : 4;
    const size_t lds = (size_t)(d + 64 * nw + 2 * nw + nw * dv) * sizeof(float);
    if (lds > 64 * 1024) return MV_ERR_UNSUPPORTED;
    if (wide) {
        if (f32) hipLaunchKernelGGL((window_attn_kernel<true, 16>), grid, dim3(1024), lds, s, q, ldq, k_cache, v_cache, out, ldo, pr, slopes, tokens, heads, kv_heads, d, dv, scale, window, row_len, skip_len, keep_first, sinks, gate, ldg, chunked);
        else hipLaunchKernelGGL((window_attn_kernel<false, 16>), grid, dim3(1024), lds, s, q, ldq, k_cache, v_cache, out, ldo, pr, slopes, tokens, heads, kv_heads, d, dv, scale, window, row_len, skip_len, keep_first, sinks, gate, ldg, chunked);
    } else {
        if (f32) hipLaunchKernelGGL((window_attn_kernel<true, 4>), grid, dim3(256), lds, s, q, ldq, k_cache, v_cache, out, ldo, pr, slopes, tokens, heads, kv_heads, d, dv, scale, window, row_len, skip_len, keep_first, sinks, gate, ldg, chunked);
        else hipLaunchKernelGGL((window_attn_kernel<false, 4>), grid, dim3(256), lds, s, q, ldq, k_cache, v_cache, out, ldo, pr, slopes, tokens, heads, kv_heads, d, dv, scale, window, row_len, skip_len, keep_first, sinks, gate, ldg, chunked);
    }
    return check_launch();
}

// The launches of a step of single tokens that mv_rotary_window_attn has a form for: head shapes with an instance, and few enough
// tokens that every workgroup has a compute unit to itself (the waves that turn the heads are the sixteen, or eight, of that form).
int mv_rotary_window_attn_ok(int tokens, int heads, int kv_heads, int d, int dv, int rot, int window, int keep_first, int splits,
                             int f32) {
    using namespace mv;
    if (tokens <= 0 || heads <= 0 || kv_heads <= 0 || heads % kv_heads || d != dv || (d != 128 && d != 64) || rot < 0 || rot > d ||
        rot % 2 || window <= 0 || keep_first < 0 || splits < 1)
        return 0;
    const FewPlan fp = few_plan(tokens, heads, kv_heads, window, keep_first, f32, splits);
    return fp.wide && !(f32 && fp.top == 1 && d == 128);   // sixteen waves of fp32 rows of 128: the registers of the turning spill
}

int mv_rotary_window_attn(const float* qk, int64_t ld, const float* q_bias, const float* k_bias, const double* inv_freq, int rot,
                          int adjacent, void* k_cache, void* v_cache, void* out, int64_t ldo, const int32_t* tok_row,
                          const int32_t* tok_pos, const int32_t* block_table, int bt_stride, int page, int tokens, int heads,
                          int kv_heads, int d, int dv, float scale, int window, int keep_first, const float* sinks, float* part,
                          int splits, const float* act_in, int64_t lda, void* act_out, int64_t ldao, int act_n, int act_kind,
                          float act_limit, float act_slope, int f32, mv_stream_t stream) {
    using namespace mv;
    if (tokens < 0 || page <= 0 || ld < (int64_t)(heads + kv_heads) * d) return MV_ERR_INVALID_ARG;
    if (act_in && (!act_out || act_n <= 0 || lda < 2 * (int64_t)act_n || ldao < act_n || act_kind < 0 || act_kind > 2))
        return MV_ERR_INVALID_ARG;
    if (tokens == 0) return MV_OK;
    if (!mv_rotary_window_attn_ok(tokens, heads, kv_heads, d, dv, rot, window, keep_first, splits, f32)) return MV_ERR_UNSUPPORTED;
    if (!qk || !k_cache || !v_cache || !out || !part || (rot > 0 && !inv_freq) || !tok_row || !tok_pos || !block_table)
        return MV_ERR_INVALID_ARG;
    if (!aligned16(k_cache) || !aligned16(v_cache)) return MV_ERR_UNSUPPORTED;
    const FewPlan fp = few_plan(tokens, heads, kv_heads, window, keep_first, f32, splits);
    const int nw = fp.top <= 1 ? 16 : fp.top <= 4 ? (f32 ? 8 : 16) : 8;
    int64_t act_blocks = act_in ? (int64_t)tokens * ((act_n + 64 * nw - 1) / (64 * nw)) : 0;
    if (act_blocks > (int64_t)(65535 - fp.pieces) * fp.groups) {      // more than the grid's rows hold: a launch of its own
        if (const int rc = mv_gated_act(act_in, lda, act_out, ldao, tokens, act_n, act_kind, act_limit, act_slope, f32, stream)) return rc;
        act_blocks = 0;
    }
    const int64_t act_rows = (act_blocks + fp.groups - 1) / fp.groups;
    PagedRows pr{tok_row, tok_pos, block_table, bt_stride, page};
    const StepRotary ra{q_bias, qk + (int64_t)heads * d, k_bias, inv_freq, rot, adjacent, (unsigned)act_blocks, act_in, act_out, lda,
                        ldao, act_n, act_kind, act_limit, act_slope};
    hipStream_t s = (hipStream_t)stream;
#define MV_RWA(F32_, HB_, NW_, KS_, VE_)                                                                               \
    hipLaunchKernelGGL((window_attn_few_kernel<F32_, HB_, NW_, KS_, VE_, true>), dim3((unsigned)fp.groups, (unsigned)(fp.pieces + act_rows)), \
                       dim3(64 * NW_), 0, s, qk, ld, k_cache, v_cache, out, ldo, part, pr, (const float*)nullptr, sinks, heads, kv_heads, \
                       scale, window, keep_first, (const int*)nullptr, 0, fp.pieces, (const float*)nullptr, (int64_t)0, 0, ra)
#define MV_RWA_HB(F32_, KS_, VE_)                                                                                      \
    do {                                                                                                               \
        if (fp.top > 4) MV_RWA(F32_, 8, 8, KS_, VE_);                                                                  \
        else if (fp.top > 1) MV_RWA(F32_, 4, (F32_ ? 8 : 16), KS_, VE_);                                               \
        else MV_RWA(F32_, 1, 16, KS_, VE_);                                                                            \
    } while (0)
    if (f32) {
        if (d == 128 && fp.top > 4) MV_RWA(true, 8, 8, 4, 8);
        else if (d == 128) MV_RWA(true, 4, 8, 4, 8);
        else MV_RWA_HB(true, 2, 4);
    } else {
        if (d == 128) MV_RWA_HB(false, 4, 8);
        else MV_RWA_HB(false, 2, 4);
    }
#undef MV_RWA_HB
#undef MV_RWA
    if (fp.pieces > 1) {
        const dim3 grid((unsigned)(tokens * heads));
        if (f32) hipLaunchKernelGGL(window_attn_merge_kernel<true>, grid, dim3(64), 0, s, part, out, ldo, tok_row, tok_pos, sinks, heads, dv, fp.pieces, nw, window, keep_first, 0, (const int*)nullptr, 0, (const float*)nullptr, (int64_t)0);
        else hipLaunchKernelGGL(window_attn_merge_kernel<false>, grid, dim3(64), 0, s, part, out, ldo, tok_row, tok_pos, sinks, heads, dv, fp.pieces, nw, window, keep_first, 0, (const int*)nullptr, 0, (const float*)nullptr, (int64_t)0);
    }
    return check_launch();
}

}  // extern "C"
