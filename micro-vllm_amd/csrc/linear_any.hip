// y[M,N] (fp32) = x[M,K] . W[N,K]^T for ANY M, N, K, row-major operands as a checkpoint stores them.
//
// The wave-tile projections (wgemm.hip, gemm_prefill.hip) want N % 16 == 0, K % 32 / 64 == 0 and a
// relaid-out weight image; layer stacks whose widths are whatever their configuration says (an
// input projection of 2*inner + 2*groups*state + heads rows, an inner width of heads * vdim) use
// this kernel for the shapes those cannot take.
//   bf16 operands: 64 x 64 output tile per workgroup of 4 waves, k in steps of 32 through LDS,
//                  v_mfma_f32_16x16x32_bf16, edges zero-filled in LDS; the sum over k in ascending order of those
//                  steps;
//   fp32 operands: products of 32-bit factors, every factor in three bf16 parts (no reduced-precision mode), on tiles of
//                  several sizes or, for a few rows, the weights streamed past them.  In all of these a sum over k is
//                  made of four quarters of k (in whole steps of 32) that are added up in ascending order, a quarter
//                  of the same sequence of matrix instructions.
// So in one product (mv_linear_any) a row's result does not depend on which other rows share the launch.  A launch of
// several products (heads, expert segments) has another form for up to kFewRows rows, linear_fewrows_kernel, whose lanes
// add every 64th piece of k and then each other: there a row's last bits differ from those of a larger launch.
#include "common.h"
#include <type_traits>

namespace mv {

typedef __attribute__((ext_vector_type(8))) __bf16 la_bf16x8_t;

// Rows in segments: with `seg` the launch's z-th product owns output rows seg[z] .. seg[z+1] (tokens sorted by
// the expert they go to) and reads, for output row i, operand row src[i] / src_div (src == NULL: row i).
struct RowSegments {
    const int* seg;
    const int* src;
    int src_div;
};

constexpr int kFewRows = 32;   // up to this many output rows a product takes the form without tiles
constexpr int kLaBM = 64, kLaBN = 64, kLaBK = 32, kLaPad = 40;  // LDS row = 40 bf16 = 80 bytes

__device__ __forceinline__ uint4 la_load8(const uint16_t* base, int64_t ld, int row, int nrows, int col, int k,
                                          bool vec) {
    if (row >= nrows || col >= k) return make_uint4(0, 0, 0, 0);
    const uint16_t* p = base + (int64_t)row * ld + col;
    if (vec && col + 8 <= k) return ld16(p);
    uint16_t e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = (col + i < k) ? p[i] : (uint16_t)0;
    return make_uint4(e[0] | ((uint32_t)e[1] << 16), e[2] | ((uint32_t)e[3] << 16), e[4] | ((uint32_t)e[5] << 16),
                      e[6] | ((uint32_t)e[7] << 16));
}

__global__ __launch_bounds__(256) void linear_any_bf16_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const uint16_t* __restrict__ w, int64_t ldw,
    float* __restrict__ y, int64_t ldy, int M, int N, int K, int vec_x, int vec_w, int64_t zx, int64_t zw,
    int64_t zy, RowSegments sg) {
    x += blockIdx.z * zx;   // blockIdx.z: one of several products that share a launch (per-head weights)
    w += blockIdx.z * zw;
    y += blockIdx.z * zy;
    __shared__ __attribute__((aligned(16))) uint16_t xs[kLaBM][kLaPad];
    __shared__ __attribute__((aligned(16))) uint16_t ws[kLaBN][kLaPad];
    const int m0 = blockIdx.y * kLaBM, n0 = blockIdx.x * kLaBN;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int lrow = tid >> 2, lcol = (tid & 3) * 8;
    int64_t y0 = 0;
    if (sg.seg) {   // blockIdx.z owns output rows seg[z] .. seg[z+1]
        y0 = sg.seg[blockIdx.z];
        M = sg.seg[blockIdx.z + 1] - (int)y0;
        if (m0 >= M) return;
        y += y0 * ldy;
    }
    // this thread's operand row: the output row itself, or the row the segment's list names for it
    {
        const int mr = m0 + lrow;
        const int64_t xrow = mr < M ? (sg.src ? sg.src[y0 + mr] / sg.src_div : y0 + mr) : 0;
        x += xrow * ldx - (int64_t)(m0 + lrow) * ldx;
    }
    f32x4_t acc[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
    uint4 xr = la_load8(x, ldx, m0 + lrow, M, lcol, K, vec_x);
    uint4 wr = la_load8(w, ldw, n0 + lrow, N, lcol, K, vec_w);
    for (int k0 = 0; k0 < K; k0 += kLaBK) {
        __syncthreads();
        st16(&xs[lrow][lcol], xr);
        st16(&ws[lrow][lcol], wr);
        __syncthreads();
        if (k0 + kLaBK < K) {
            xr = la_load8(x, ldx, m0 + lrow, M, k0 + kLaBK + lcol, K, vec_x);
            wr = la_load8(w, ldw, n0 + lrow, N, k0 + kLaBK + lcol, K, vec_w);
        }
        // first operand: 16 weight rows of this wave; second: 16 activation rows per m-tile
        const la_bf16x8_t wf = __builtin_bit_cast(la_bf16x8_t, ld16(&ws[wave * 16 + r][q * 8]));
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) {
            const la_bf16x8_t xf = __builtin_bit_cast(la_bf16x8_t, ld16(&xs[mt * 16 + r][q * 8]));
            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf, acc[mt], 0, 0, 0);
        }
    }
    // acc[mt][j] = C[n = n0 + 16 wave + 4 q + j][m = m0 + 16 mt + r]
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        const int m = m0 + mt * 16 + r;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + wave * 16 + q * 4 + j;
            if (n < N) y[(int64_t)m * ldy + n] = acc[mt][j];
        }
    }
}

// The same product on a 128 x 128 tile for launches with many rows: four waves as 2 x 2, each 64 x 64 (sixteen
// accumulator tiles), so that a k-step of 32 costs a wave eight LDS reads for sixteen matrix instructions
// instead of five for four.  Same order of the sums over k as the 64 x 64 form: the results are equal bit for bit.
constexpr int kLbBM = 128, kLbBN = 128, kLbBK = 64, kLbPad = 72;   // LDS row = 72 bf16 = 144 bytes

__global__ __launch_bounds__(256) void linear_any_bf16_big_kernel(
    const uint16_t* __restrict__ x, int64_t ldx, const uint16_t* __restrict__ w, int64_t ldw,
    float* __restrict__ y, int64_t ldy, int M, int N, int K, int vec_x, int vec_w, int64_t zx, int64_t zw,
    int64_t zy, RowSegments sg) {
    x += blockIdx.z * zx;
    w += blockIdx.z * zw;
    y += blockIdx.z * zy;
    __shared__ __attribute__((aligned(16))) uint16_t xs[kLbBM][kLbPad];
    __shared__ __attribute__((aligned(16))) uint16_t ws[kLbBN][kLbPad];
    const int m0 = blockIdx.y * kLbBM, n0 = blockIdx.x * kLbBN;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    const int lrow = tid >> 3, lcol = (tid & 7) * 8;   // a thread stages rows lrow + 32 u, eight values at lcol
    int64_t y0 = 0;
    if (sg.seg) {
        y0 = sg.seg[blockIdx.z];
        M = sg.seg[blockIdx.z + 1] - (int)y0;
        if (m0 >= M) return;
        y += y0 * ldy;
    }
    const uint16_t* xp[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int mr = m0 + lrow + 32 * u;
        const int64_t xrow = mr < M ? (sg.src ? sg.src[y0 + mr] / sg.src_div : y0 + mr) : 0;
        xp[u] = x + xrow * ldx;
    }
    f32x4_t acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = f32x4_t{0, 0, 0, 0};
    uint4 xr[4], wr[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        xr[u] = la_load8(xp[u], ldx, 0, m0 + lrow + 32 * u < M ? 1 : 0, lcol, K, vec_x);
        wr[u] = la_load8(w, ldw, n0 + lrow + 32 * u, N, lcol, K, vec_w);
    }
    for (int k0 = 0; k0 < K; k0 += kLbBK) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            st16(&xs[lrow + 32 * u][lcol], xr[u]);
            st16(&ws[lrow + 32 * u][lcol], wr[u]);
        }
        __syncthreads();
        if (k0 + kLbBK < K) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                xr[u] = la_load8(xp[u], ldx, 0, m0 + lrow + 32 * u < M ? 1 : 0, k0 + kLbBK + lcol, K, vec_x);
                wr[u] = la_load8(w, ldw, n0 + lrow + 32 * u, N, k0 + kLbBK + lcol, K, vec_w);
            }
        }
#pragma unroll
        for (int ks = 0; ks < kLbBK; ks += 32) {   // two steps of 32, in ascending k as the narrow tile takes them
            la_bf16x8_t wf[4], xf[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                wf[t] = __builtin_bit_cast(la_bf16x8_t, ld16(&ws[wn * 64 + t * 16 + r][ks + q * 8]));
                xf[t] = __builtin_bit_cast(la_bf16x8_t, ld16(&xs[wm * 64 + t * 16 + r][ks + q * 8]));
            }
#pragma unroll
            for (int nt = 0; nt < 4; ++nt)
#pragma unroll
                for (int mt = 0; mt < 4; ++mt)
                    acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[nt], xf[mt], acc[nt][mt], 0, 0, 0);
        }
    }
    // acc[nt][mt][j] = C[n = n0 + 64 wn + 16 nt + 4 q + j][m = m0 + 64 wm + 16 mt + r]
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
        const int m = m0 + wm * 64 + mt * 16 + r;
        if (m >= M) continue;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            const int n = n0 + wn * 64 + nt * 16 + q * 4;
            float* dst = y + (int64_t)m * ldy + n;
            if (n + 3 < N && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
                *reinterpret_cast<float4*>(dst) = make_float4(acc[nt][mt][0], acc[nt][mt][1], acc[nt][mt][2], acc[nt][mt][3]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (n + j < N) dst[j] = acc[nt][mt][j];
            }
        }
    }
}

// fp32 operands on the bf16 matrix instruction, every factor in three bf16 parts: x = hi + mid + lo exactly (8 bits each of the
// 24), of the nine products of parts the six that reach 2^-24 of x w, each of them exact in the instruction and added up in
// fp32.  v_mfma_f32_16x16x4_f32 does 256 FLOP a cycle and unit, v_mfma_f32_16x16x32_bf16 4096.  A weight whose low 16 bits are
// zero is its own hi: sixteen rows of weights that are so over a step of k (those of a bf16 checkpoint in a run of 32 bits)
// take three products, and the sum is the same bit for bit, for what is left out are zeros.
// Sums, in every form here: a step is 32 neighbouring k, its products go from the smallest parts to hi hi; steps in ascending
// order make a quarter of k, the quarters are added in ascending order.
// The parts are exact while their lowest bits are bf16 numbers: of a factor below about 2^-103 bits are lost, up to 2^-125 of it at
// the worst.  Times another factor of at most kLfHuge that is 2^-95, under 2^-35 of a sum that is not below kLfTiny.  Every other
// output is done by the fp32 instruction (lf_by_f32: the same quarters): where the largest magnitude of its row of x or of its row
// of W is past kLfHuge (an infinite factor among them, or one that the rounding of hi makes infinite), where the sum is not finite,
// below kLfTiny, or zero without a row of zeros.  NaN in a row is NaN in its sums either way.  Which form an output takes depends
// on its own row and column alone; the largest magnitudes cost half an instruction a value on its way into LDS.
constexpr int kLfBK = 32;
constexpr float kLfTiny = 0x1p-60f, kLfHuge = 0x1p30f;

__device__ __forceinline__ float lf_largest(float a, float b) { return __builtin_elementwise_maximum(a, b); }   // NaN stays
__device__ __forceinline__ float lf_largest(const f32x4_t& v, float so_far) {   // magnitudes
    // (assembly keeps it where it stands; moved about by the scheduler it holds the values longer: 16 to 30 registers, a workgroup a unit)
    asm volatile("v_maximum3_f32 %0, |%1|, |%2|, %0\n\tv_maximum3_f32 %0, |%3|, |%4|, %0" : "+v"(so_far) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]));
    return so_far;
}
__device__ __forceinline__ float lf_least(const f32x4_t& v, float so_far) {   // of magnitudes, NaN stays
    auto least = [](float a, float b) { return __builtin_elementwise_minimum(a, b); };
    return least(least(fabsf(v[2]), fabsf(v[3])), least(least(fabsf(v[0]), fabsf(v[1])), so_far));
}
// of a sum and the largest magnitudes of its two rows
__device__ __forceinline__ bool lf_outside(float v, float xmax, float wmax) {
    const float a = fabsf(v);
    const bool inside = a >= kLfTiny && a < INFINITY && xmax <= kLfHuge && wmax <= kLfHuge;
    const bool zeros = v == 0.f && (xmax == 0.f || wmax == 0.f);
    return !inside && !zeros && !(xmax != xmax || wmax != wmax);
}

// Four values.  A part is subtracted by v_dot2_f32_bf16, (-1, 0) or (0, -1) times the packed pair, where that is faster than to
// unpack it (streamed 16 rows 16384 x 4096 52.5 -> 50 us, 32 x 32 tiles 33 rows 1024 x 5120 28.8 -> 26.5; the wider tiles 0 to 3 % slower, x a
// step at a time in slices of 1024 x 5120 7.8 -> 8.2): every result is exact either way.
template <bool DOT>
__device__ __forceinline__ void lf_split4(const f32x4_t& v, uint2& hi, uint2& mid, uint2& lo) {
    uint32_t minus_lo = 0x0000bf80u, minus_hi = 0xbf800000u;
    asm("" : "+s"(minus_lo), "+s"(minus_hi));   // (in registers: as an inline constant the second is another pair)
    auto less = [&](const f32x4_t& x, const uint2& p) {
        if constexpr (DOT)
            return f32x4_t{dot2_bf16(p.x, minus_lo, x[0]), dot2_bf16(p.x, minus_hi, x[1]), dot2_bf16(p.y, minus_lo, x[2]),
                           dot2_bf16(p.y, minus_hi, x[3])};
        else
            return f32x4_t{x[0] - bf16_lo(p.x), x[1] - bf16_hi(p.x), x[2] - bf16_lo(p.y), x[3] - bf16_hi(p.y)};
    };
    auto pack = [](const f32x4_t& x) { return make_uint2(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])); };
    hi = pack(v);
    const f32x4_t rest = less(v, hi);
    mid = pack(rest);
    lo = pack(less(rest, mid));
}
struct LfParts {
    uint4 hi, mid, lo;   // eight values, two in each word
};
template <bool DOT>
__device__ __forceinline__ LfParts lf_split(const f32x4_t& v0, const f32x4_t& v1) {
    uint2 h[2], m[2], l[2];
    lf_split4<DOT>(v0, h[0], m[0], l[0]);
    lf_split4<DOT>(v1, h[1], m[1], l[1]);
    return {make_uint4(h[0].x, h[0].y, h[1].x, h[1].y), make_uint4(m[0].x, m[0].y, m[1].x, m[1].y),
            make_uint4(l[0].x, l[0].y, l[1].x, l[1].y)};
}
// whether any of eight values has bits beside those of bf16, and the values' upper halves
__device__ __forceinline__ uint32_t lf_low_bits(const f32x4_t& v0, const f32x4_t& v1) {
    uint32_t any = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) any |= __float_as_uint(v0[i]) | __float_as_uint(v1[i]);
    return any & 0xffffu;
}
__device__ __forceinline__ uint4 lf_upper(const f32x4_t& v0, const f32x4_t& v1) {
    auto two = [](float a, float b) { return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u); };
    return make_uint4(two(v0[0], v0[1]), two(v0[2], v0[3]), two(v1[0], v1[1]), two(v1[2], v1[3]));
}
__device__ __forceinline__ f32x4_t lf_mfma(uint4 w, uint4 x, f32x4_t acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(la_bf16x8_t, w), __builtin_bit_cast(la_bf16x8_t, x), acc, 0, 0, 0);
}

// VEC: rows at multiples of 16 bytes and K % 4 == 0.  Columns past the end of k are zeros and nothing is read there; rows
// past the last one were clamped by the caller (their outputs are not stored).
template <bool VEC>
__device__ __forceinline__ f32x4_t lf_load4_any(const float* p, int col, int k) {   // past the end: anything (lf_mask4)
    f32x4_t v;
    if (VEC) return *reinterpret_cast<const f32x4_t*>(p + (col < k ? col : 0));
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = p[col + i < k ? col + i : 0];
    return v;
}
__device__ __forceinline__ void lf_mask4(f32x4_t& v, int col, int k) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = col + i < k ? v[i] : 0.f;
}
template <bool VEC>
__device__ __forceinline__ f32x4_t lf_load4(const float* p, int col, int k) {
    f32x4_t v = lf_load4_any<VEC>(p, col, k);
    lf_mask4(v, col, k);
    return v;
}

// Sixteen outputs by sixteen on the fp32 instruction, straight from memory: lane (r, q)'s row of x and of W, the shares
// `share` .. `share + count` of `per` steps, added up in ascending order.  It is for few outputs: four steps are asked for together,
// for one by one it is a chain of latencies, but every block reads its operands for itself.  us with one row of activations below
// 2^-100 (a step at a time -> four; all on the fp32 instruction): 567 rows 9472 x 1024 138 -> 101 (114), 1024 x 5120 267 -> 185
// (95), 2048 rows 16384 x 4096 1500 -> 1250 (2155).
template <bool VEC>
__device__ __forceinline__ f32x4_t lf_by_f32(const float* x, const float* w, int q, int K, int per, int share, int count) {
    constexpr int kAhead = 4;   // steps asked for together
    f32x4_t sum = {0, 0, 0, 0}, acc = {0, 0, 0, 0};
    const int first = share * per, end = min(K, (share + count) * per * kLfBK);   // (zeros past it)
    int left = per;   // steps of the share that acc holds a part of
    for (int i = 0; i < count * per; i += kAhead) {
        f32x4_t xf[kAhead][2], wf[kAhead][2];
        const int k0 = (first + i) * kLfBK + q * 4;
#pragma unroll
        for (int n = 0; n < kAhead; ++n)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                xf[n][h] = lf_load4<VEC>(x, k0 + n * kLfBK + h * 16, end);
                wf[n][h] = lf_load4<VEC>(w, k0 + n * kLfBK + h * 16, end);
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < kAhead; ++n) {   // (no branch: it would take the loads with it)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[n][h][e], xf[n][h][e], acc, 0, 0, 0);
            const bool whole = --left == 0;   // uniform
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                sum[j] = whole ? sum[j] + acc[j] : sum[j];
                acc[j] = whole ? 0.f : acc[j];
            }
            left = whole ? per : left;
        }
    }
    return sum;
}

// Tiles of one column of outputs (one piece of W) go to one XCD, whose L2 then holds that piece: workgroups are dealt
// out over the eight XCDs in turn, so eight columns advance side by side.
__device__ __forceinline__ bool lf_place(int id, int cols, int rows, int& col, int& row) {
    col = (id / (8 * rows)) * 8 + (id & 7);
    row = (id >> 3) % rows;
    return col < cols;
}

// TM x TN accumulator tiles of 16 x 16 per wave, four waves as 2 x 2: (32 TM) x (32 TN) outputs.  KG groups of four waves take
// the quarters of k side by side, each its 4 / KG one after the other (a second set of accumulators holds the sum so far).  A
// step of 32 k: a wave splits sixteen rows at a time on their way into LDS, where a plane of parts of sixteen rows is 1 KB in the
// instruction's own lane order; the rows of lane group q are exchanged by xor with 2 q, so that neither the writes (four lanes a
// row, eight lanes a cycle) nor the reads (a lane a row) meet on a bank: no conflicts counted, without it in three of five cycles that LDS is busy.  PF
// steps are requested ahead.  DB: two buffers and one barrier a step, else one and two.
// What bounds it: no one unit - at 2048 rows 16384 x 4096 the matrix units are busy 42 % of the time, the vector units 30, LDS 28 - but
// the chain load, split, LDS, barrier, products of the two or three workgroups of a unit; splitting the next step in front of this
// one's products, into a second buffer, gained nothing, nor did requests of eight rows of 128 bytes.
// Against the fp32 matrix instruction (256 FLOP a cycle and unit) that was here, us, weights of bf16 values | of 32 bits, out of memory:
// 567 rows 9472 x 1024 114 -> 55 | 85, 1024 x 5120 95 -> 61 | 81, 1024 x 1024 22.5 -> 14.2 | 19.4; 2048 rows 16384 x 4096 2155 -> 905 (304
// TFLOP/s of fp32 products) | 1460; 33 rows 1024 x 5120 37 -> 26.5 | 33.6; 64 rows 9472 x 1024 25.4 -> 18.4 | 22.2; 1024 rows 4096 x 128 17.3 ->
// 15.1 | 17.6.  9 to 16 rows of 65536 x 64 take 12.9 | 14.0, 10.1 on it.
// Error against 64 bits (2-norm): 1024 x 5120 6.4e-7 -> 3.9e-7 | 5.6e-7, 9472 x 1024 2.9e-7 -> 1.7e-7 | 2.3e-7.
template <int TM, int TN, int KG, int PF, bool DB, bool VEC>
__global__ __launch_bounds__(256 * KG, KG == 1 ? 2 : 1) void linear_any_f32_kernel(
    const float* __restrict__ x, int64_t ldx, const float* __restrict__ w, int64_t ldw,
    float* __restrict__ y, int64_t ldy, int M, int N, int K, int64_t zx, int64_t zw, int64_t zy, RowSegments sg) {
    constexpr int BM = 32 * TM, BN = 32 * TN, RB = 2 * (TM + TN), U = RB / 4;   // row blocks; of them per wave
    constexpr int kPlane = RB * 64;                                            // 16-byte pieces of a plane
    constexpr bool kFold = KG < 4;
    static_assert(KG == 1 || KG == 2 || KG == 4, "a group has one quarter, two or all of them");
    static_assert(RB % 4 == 0 && (TM % 2 == 0 || (TM == 1 && TN == 1)), "a wave's row block is of x or of W");
    x += blockIdx.z * zx;
    w += blockIdx.z * zw;
    y += blockIdx.z * zy;
    extern __shared__ __attribute__((aligned(16))) float lf_lds[];
    __shared__ int more_parts[DB ? 2 : 1][KG][2 * TN];   // the step in which these rows of W last had low bits
    __shared__ float row_max[KG][RB * 16][4];   // largest magnitudes of the rows, x in front of W: of each staging lane
    __shared__ int far_rows;                 // whether any of them is NaN or past kLfHuge
    int nb, mb;
    if (!lf_place(blockIdx.x, (N + BN - 1) / BN, (M + BM - 1) / BM, nb, mb)) return;
    const int m0 = mb * BM, n0 = nb * BN;
    const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = threadIdx.x & 255;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane >> 2, lq = lane & 3;   // staging: row of the block, piece of the row
    int64_t y0 = 0;
    if (sg.seg) {
        y0 = sg.seg[blockIdx.z];
        M = sg.seg[blockIdx.z + 1] - (int)y0;
        if (m0 >= M) return;
        y += y0 * ldy;
    }
    auto x_row = [&](int i) { return x + (i < M ? (sg.src ? sg.src[y0 + i] / sg.src_div : y0 + i) : 0) * ldx; };
    auto w_row = [&](int i) { return w + (int64_t)min(i, N - 1) * ldw; };
    auto of_x = [&](int u) { return TM > 1 ? u < TM / 2 : wave < 2; };
    const float* p[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int row = (u * 4 + wave) * 16 + lr;
        p[u] = of_x(u) ? x_row(m0 + row) : w_row(n0 + row - BM);
    }
    uint4* buf = reinterpret_cast<uint4*>(lf_lds) + grp * (DB ? 2 : 1) * 3 * kPlane;
    if (threadIdx.x < (DB ? 2 : 1) * KG * 2 * TN) (&more_parts[0][0][0])[threadIdx.x] = -1;
    if (threadIdx.x == 0) far_rows = 0;
    f32x4_t acc[TN][TM], sum[TN][TM];
    const int per = ((K + kLfBK - 1) / kLfBK + 3) / 4;   // k-steps of a quarter
    auto clear = [&] {
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) acc[a][b] = f32x4_t{0, 0, 0, 0};
    };
    int fold = per;
    auto add_quarter = [&] {
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b)
#pragma unroll
                for (int j = 0; j < 4; ++j) sum[a][b][j] = fold == per ? acc[a][b][j] : sum[a][b][j] + acc[a][b][j];
        fold += per;
    };
    clear();
    f32x4_t v[PF][U][2];
    float largest[U];
#pragma unroll
    for (int u = 0; u < U; ++u) largest[u] = 0.f;
    const int first = grp * per * (4 / KG);   // this group's first step
#pragma unroll
    for (int u = 0; u < U; ++u) p[u] += first * kLfBK + lq * 4;
    auto request = [&](int set, int step) {   // steps are asked for in ascending order
        const int k0 = (first + step) * kLfBK;
        if (VEC && k0 + kLfBK <= K) {   // uniform
#pragma unroll
            for (int u = 0; u < U; ++u) {
                v[set][u][0] = *reinterpret_cast<const f32x4_t*>(p[u]);
                v[set][u][1] = *reinterpret_cast<const f32x4_t*>(p[u] + 16);
            }
        } else {   // the last step of k, or one past it
            const int col = k0 + lq * 4;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                v[set][u][0] = lf_load4_any<VEC>(p[u] - col, col, K);
                v[set][u][1] = lf_load4_any<VEC>(p[u] - col, col + 16, K);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) p[u] += kLfBK;
    };
    const int put = lq * 16 + (lr ^ (lq * 2)), get = q * 16 + (r ^ (q * 2));
    auto stage = [&](int set, int half, int step) {
        uint4* at = buf + (DB ? half * 3 * kPlane : 0);
        if ((first + step + 1) * kLfBK > K) {   // uniform, as above
            const int col = (first + step) * kLfBK + lq * 4;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                lf_mask4(v[set][u][0], col, K);
                lf_mask4(v[set][u][1], col + 16, K);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint4* to = at + (u * 4 + wave) * 64 + put;
            largest[u] = lf_largest(v[set][u][1], lf_largest(v[set][u][0], largest[u]));
            if (of_x(u) || __any(lf_low_bits(v[set][u][0], v[set][u][1]) != 0)) {   // uniform
                const LfParts s = lf_split<TM == 1>(v[set][u][0], v[set][u][1]);
                to[0] = s.hi;
                to[kPlane] = s.mid;
                to[2 * kPlane] = s.lo;
                if (!of_x(u) && lane == 0) more_parts[DB ? half : 0][grp][u * 4 + wave - 2 * TM] = step;
            } else {
                to[0] = lf_upper(v[set][u][0], v[set][u][1]);
            }
        }
        request(set, step + PF);
    };
    uint4 wf[TN], xf[TM][3];
    int tag[TN];
    auto fetch = [&](int half) {
        const uint4* at = buf + (DB ? half * 3 * kPlane : 0);
#pragma unroll
        for (int a = 0; a < TN; ++a) {
            wf[a] = at[(2 * TM + wn * TN + a) * 64 + get];
            tag[a] = more_parts[DB ? half : 0][grp][wn * TN + a];
        }
#pragma unroll
        for (int b = 0; b < TM; ++b)
#pragma unroll
            for (int part = 0; part < 3; ++part) xf[b][part] = at[part * kPlane + (wm * TM + b) * 64 + get];
    };
    auto multiply = [&](int half, int step) {
        if (kFold && step == fold) {
            add_quarter();
            clear();
        }
        bool more[TN], any = false;
#pragma unroll
        for (int a = 0; a < TN; ++a) {
            more[a] = __builtin_amdgcn_readfirstlane(tag[a]) == step;
            any = any || more[a];
        }
        if (any) {   // (rows without low bits beside rows with: their parts here are what an earlier step left)
            const uint4* ws = buf + (DB ? half * 3 * kPlane : 0) + (2 * TM + wn * TN) * 64 + get;
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                if (!more[a]) continue;
                const uint4 mid = ws[kPlane + a * 64], lo = ws[2 * kPlane + a * 64];
#pragma unroll
                for (int b = 0; b < TM; ++b) acc[a][b] = lf_mfma(lo, xf[b][0], acc[a][b]);
#pragma unroll
                for (int b = 0; b < TM; ++b) acc[a][b] = lf_mfma(mid, xf[b][1], acc[a][b]);
#pragma unroll
                for (int b = 0; b < TM; ++b) acc[a][b] = lf_mfma(mid, xf[b][0], acc[a][b]);
            }
        }
#pragma unroll
        for (int part = 2; part >= 0; --part)
#pragma unroll
            for (int b = 0; b < TM; ++b)
#pragma unroll
                for (int a = 0; a < TN; ++a) acc[a][b] = lf_mfma(wf[a], xf[b][part], acc[a][b]);
    };
    constexpr int TURN = PF > (DB ? 2 : 1) ? PF : (DB ? 2 : 1);   // steps after which register sets and buffers are where they were
    // Side by side the groups share the barriers, and a step past the end of k multiplies zeros.  One after the other the
    // quarters end with k, at a whole turn.
    const int steps = KG > 1 ? per * (4 / KG) : ((K + kLfBK - 1) / kLfBK + TURN - 1) / TURN * TURN;
    auto turn = [&](int set, int half, int step) {
        stage(set, half, step);
        __syncthreads();   // (DB: the other buffer was read a step ago, before this barrier by every wave)
        fetch(half);
        multiply(half, step);
        if (!DB && (KG > 1 || step + 1 < steps)) __syncthreads();
    };
#pragma unroll
    for (int i = 0; i < PF; ++i) request(i, i);
    __syncthreads();   // (more_parts)
    static_assert(!DB || TURN % 2 == 0, "a turn ends on the buffer it began with");
    int st = 0;
    for (; st + TURN <= steps; st += TURN)
#pragma unroll
        for (int i = 0; i < TURN; ++i) turn(i % PF, i & 1, st + i);
#pragma unroll
    for (int i = 0; i < TURN - 1; ++i)
        if (st + i < steps) turn(i % PF, i & 1, st + i);
    if (kFold && (KG == 1 || grp == 0)) {
        add_quarter();
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) acc[a][b] = sum[a][b];
    }
    bool far = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        row_max[grp][(u * 4 + wave) * 16 + lr][lq] = largest[u];
        far = far || !(largest[u] <= kLfHuge);
    }
    if (__any(far) && lane == 0) far_rows = 1;
    __syncthreads();
    if (KG > 1) {   // group 0 adds up the others' quarters, one by one
        constexpr int kAcc = TN * TM * 4, kQuarters = 4 / KG;
        float* part = lf_lds + ((grp - 1) * 256 + tid) * (kQuarters * kAcc + 1);
        if (grp > 0) {
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < TM; ++b)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int at = (a * TM + b) * 4 + j;
                        if (kFold) part[at] = sum[a][b][j];
                        part[(kQuarters - 1) * kAcc + at] = acc[a][b][j];
                    }
        }
        __syncthreads();
        if (grp > 0) return;
        for (int g = 0; g < KG - 1; ++g) {
            const float* o = lf_lds + (g * 256 + tid) * (kQuarters * kAcc + 1);
#pragma unroll
            for (int p = 0; p < kQuarters; ++p)
#pragma unroll
                for (int a = 0; a < TN; ++a)
#pragma unroll
                    for (int b = 0; b < TM; ++b)
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[a][b][j] += o[p * kAcc + (a * TM + b) * 4 + j];
        }
    }
    // acc[a][b][j] = C[n = n0 + 16 (TN wn + a) + 4 q + j][m = m0 + 16 (TM wm + b) + r]
#pragma unroll
    for (int b = 0; b < TM; ++b) {
        const int m = m0 + (wm * TM + b) * 16 + r;
        if (m >= M) continue;
#pragma unroll
        for (int a = 0; a < TN; ++a) {
            const int n = n0 + (wn * TN + a) * 16 + q * 4;
            float* dst = y + (int64_t)m * ldy + n;
            if (n + 3 < N && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
                *reinterpret_cast<float4*>(dst) = make_float4(acc[a][b][0], acc[a][b][1], acc[a][b][2], acc[a][b][3]);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (n + j < N) dst[j] = acc[a][b][j];
            }
        }
    }
    // which of them are not the parts' (over what was stored)
    float most = 0.f, least = INFINITY;
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) {
            most = lf_largest(acc[a][b], most);
            least = lf_least(acc[a][b], least);
        }
    if (!far_rows && !__any(!(most < INFINITY && least >= kLfTiny))) return;
    auto largest_at = [&](int row) {
        float m = 0.f;
#pragma unroll
        for (int g = 0; g < KG; ++g)
#pragma unroll
            for (int l = 0; l < 4; ++l) m = lf_largest(m, row_max[g][row][l]);
        return m;
    };
    uint64_t out = 0;   // a bit for j of a block
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = (wn * TN + a) * 16 + q * 4 + j;
            const float w_max = largest_at(BM + n);
#pragma unroll
            for (int b = 0; b < TM; ++b) {
                const int m = (wm * TM + b) * 16 + r;
                if (m0 + m < M && n0 + n < N && lf_outside(acc[a][b][j], largest_at(m), w_max)) out |= 1ull << ((a * TM + b) * 4 + j);
            }
        }
    for (int i = 0; i < TN * TM; ++i) {
        const unsigned mine = (unsigned)(out >> (i * 4)) & 15u;
        if (!__any(mine != 0)) continue;
        const int m = m0 + (wm * TM + i % TM) * 16, n = n0 + (wn * TN + i / TM) * 16;
        const f32x4_t o = lf_by_f32<VEC>(x_row(m + r), w_row(n + r), q, K, per, 0, 4);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (mine >> j & 1) y[(int64_t)(m + r) * ldy + n + q * 4 + j] = o[j];
    }
}

// fp32 operands, few rows: the weights are streamed past them.  A workgroup forms sixteen neighbouring outputs of up to
// sixteen rows, its four waves the four quarters of k, by the same matrix instructions in the same order as the tiles.  Rows
// past the last one repeat it: the matrix instruction takes sixteen either way, and a launch like this waits for memory.
// A wave takes 128 k of its sixteen weight rows at a time: half a wave reads 512 neighbouring bytes of a row, so that a
// request is four whole lines of two rows and not a piece of sixteen, and the rows meet the instruction's operand layout in
// the wave's own part of LDS (rows 528 bytes apart: the sixteen rows of a read are on different banks; no barrier, a wave's LDS
// operations are in order).  Two such pieces are in flight, 16 KB a wave.
// Measured against operands read straight into that layout, 64 bytes of sixteen rows to a request (outputs x k, 3 rows, us):
// 32000 x 1024 39.8 -> 22.8 (5.7 TB/s), 9472 x 1024 16.1 -> 10.1, 16384 x 4096 61.1 -> 43.3 (6.2 TB/s), 1024 x 5120 20.6 -> 12.3 (in four
// slices 10.8 -> 7.3), 65536 x 64 70 -> 16; 16 rows 1024 x 5120 28.7 -> 17.7, 1280 x 1024 8.4 -> 6.6.
// Against the fp32 instruction in this same form, us, it -> weights of bf16 values | of 32 bits.  Up to 8 rows: 32000 x 1024 22.9 ->
// 22.8 | 23.8, 16384 x 4096 44.2 -> 43.3 | 46.6 (8 rows 45 -> 44.4 | 48), 4096 x 2048 9.0 -> 8.5 | 9.8; few workgroups, each a chain of its own split:
// 1024 x 5120 12.6 -> 12.3 | 15.3 (8 rows 13.7 -> 13.4 | 16.1), 512 x 8192 17.4 -> 17.3 | 21.9.  16 rows split x behind LDS as well:
// 16384 x 4096 49.6 -> 50.1 | 56, 1024 x 5120 16.4 -> 17.7 | 20.7.  Rows of bf16 values are what a checkpoint in that type gives.
// Four steps' operands are read out of LDS before the first is used (1024 x 5120 13.8 -> 12.3 | 16.8 -> 15.3); one at a time leaves registers for a third
// workgroup on a unit, which is ahead where a wave has three pieces or fewer (3 rows 32000 x 1024 22.8 against 23.5, 65536 x 256
// 18.6 against 23.2, a slice of 1280 of 1024 x 5120 7.45 against 7.98; 32000 x 2048 42.0 against 40.8).
// From nine rows on the tiles are ahead where the output is wide and k is short (16 rows, 65536 x 256: 18.9 us against 25, 32000 x 448
// 16.3 against 22.5; 32000 x 512 28.6 against 18.9, 16384 x 4096 74 against 49), from 17 on everywhere; at k of up to 256 and
// 16384 outputs from five (8 rows 65536 x 256 19 against 25, 32000 x 256 10.4 against 13.7, 16384 x 256 7.8 against 8.3, 9472 x 256 7.2 against
// 6.8; 32000 x 448 15.8 each).
constexpr int kStreamRowsLess = 4, kStreamRows = 8, kStreamRowsMore = 16, kStreamNarrow = 8192, kStreamWide = 16384;
constexpr int kStreamShortK = 256, kStreamLongK = 512;
constexpr int kStreamSlice = 8, kStreamOneStep = 1536;   // (a slice's k up to which steps go one by one)
constexpr int kStreamK = 128, kStreamPad = kStreamK + 4;   // k of a piece, floats of a row in LDS
constexpr int kStreamParts = kStreamK * 2 + 16;            // bytes of a row's parts in LDS
// A wave's rows of x lie in LDS split (a lane of the instruction whose column is a row past MR reads a row again, so split behind
// LDS the work would be done 16 / MR times), up to eight of them; sixteen as they are.
constexpr int stream_x_bytes(int mr) { return mr == 16 ? mr * kStreamPad * 4 : 3 * mr * kStreamParts; }

// MR: rows of x that are read, 4, 8 or 16; STEPS of 32 k whose operands are read out of LDS together, for 4 rows also one
template <int MR, int STEPS>
__global__ __launch_bounds__(256, STEPS == 1 ? 3 : 2) void linear_stream_f32_kernel(const float* __restrict__ x, int64_t ldx,
                                                                const float* __restrict__ w, int64_t ldw,
                                                                float* __restrict__ y, int64_t ldy, int M, int N, int K) {
    // blockIdx.y: a slice of k of its own, [slice][M][N] in y (ldy = N); the wave's share is a quarter of the slice
    extern __shared__ __attribute__((aligned(16))) float ls_lds[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4, n0 = blockIdx.x * 16;
    const int half = lane >> 5, kl = (lane & 31) * 4;
    const int shares = 4 * gridDim.y, share = 4 * blockIdx.y + wave;
    const int per = ((K + kLfBK - 1) / kLfBK + shares - 1) / shares;
    y += (int64_t)blockIdx.y * M * ldy;
    // k of this wave, in pieces; past the share or the end of k a lane reads its row's start and puts zeros down
    const int first = share * per * kLfBK, end = min(K, first + per * kLfBK);
    const int pieces = (per * kLfBK + kStreamK - 1) / kStreamK;
    const float* wp[8];
    const float* xp[MR / 2];
#pragma unroll
    for (int i = 0; i < 8; ++i) wp[i] = w + (int64_t)min(n0 + 2 * i + half, N - 1) * ldw;
#pragma unroll
    for (int i = 0; i < MR / 2; ++i) xp[i] = x + (int64_t)min(2 * i + half, M - 1) * ldx;
    constexpr bool kSplitFirst = MR < 16;
    float* ws = ls_lds + wave * (16 * kStreamPad + stream_x_bytes(MR) / 4);
    float* xs = ws + 16 * kStreamPad;
    unsigned char* xb = reinterpret_cast<unsigned char*>(xs);
    f32x4_t acc = {0, 0, 0, 0};
    f32x4_t wv[2][8], xv[2][MR / 2];
    constexpr int kXMax = kSplitFirst ? MR / 2 : 1;
    float w_max = 0.f, x_max[kXMax];   // largest magnitudes: of row r of W, of rows 2 i + half of x (sixteen rows: of row r)
#pragma unroll
    for (int i = 0; i < kXMax; ++i) x_max[i] = 0.f;
    auto request = [&](int set, int piece) {
        const int col = first + piece * kStreamK + kl, at = col < end ? col : 0;
#pragma unroll
        for (int i = 0; i < MR / 2; ++i) xv[set][i] = *reinterpret_cast<const f32x4_t*>(xp[i] + at);
#pragma unroll
        for (int i = 0; i < 8; ++i) wv[set][i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(wp[i] + at));
    };
    auto put = [&](int set, int piece) {
        const bool in = first + piece * kStreamK + kl < end;
        const f32x4_t zero = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < MR / 2; ++i) {
            const f32x4_t v = in ? xv[set][i] : zero;
            if (kSplitFirst) {   // four values: a half of what lane (row, k / 4 % 4) of the instruction takes of their step
                x_max[i] = lf_largest(v, x_max[i]);
                uint2 hi, mid, lo;
                lf_split4<(STEPS > 1)>(v, hi, mid, lo);
                unsigned char* to = xb + (2 * i + half) * kStreamParts + (kl >> 5) * 64 + ((kl >> 2) & 3) * 16 + ((kl >> 4) & 1) * 8;
                *reinterpret_cast<uint2*>(to) = hi;
                *reinterpret_cast<uint2*>(to + MR * kStreamParts) = mid;
                *reinterpret_cast<uint2*>(to + 2 * MR * kStreamParts) = lo;
            } else {
                *reinterpret_cast<f32x4_t*>(xs + (2 * i + half) * kStreamPad + kl) = v;
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            *reinterpret_cast<f32x4_t*>(ws + (2 * i + half) * kStreamPad + kl) = in ? wv[set][i] : zero;
    };
    // `count` steps without a branch between them, so that one's split runs beside another's products (zeros past the share's end)
    auto multiply_steps = [&](auto count, int at) {
        constexpr int C = decltype(count)::value;
        f32x4_t wv0[C], wv1[C];
        uint32_t low = 0;
#pragma unroll
        for (int u = 0; u < C; ++u) {
            const float* wr = ws + r * kStreamPad + (at + u) * kLfBK + q * 4;
            wv0[u] = *reinterpret_cast<const f32x4_t*>(wr);
            wv1[u] = *reinterpret_cast<const f32x4_t*>(wr + 16);
        }
        auto parts_of_x = [&](int u) {
            LfParts p;
            if (kSplitFirst) {
                const unsigned char* xr = xb + min(r, MR - 1) * kStreamParts + (at + u) * 64 + q * 16;
                p.hi = *reinterpret_cast<const uint4*>(xr);
                p.mid = *reinterpret_cast<const uint4*>(xr + MR * kStreamParts);
                p.lo = *reinterpret_cast<const uint4*>(xr + 2 * MR * kStreamParts);
            } else {
                const float* xr = xs + r * kStreamPad + (at + u) * kLfBK + q * 4;
                const f32x4_t x0 = *reinterpret_cast<const f32x4_t*>(xr), x1 = *reinterpret_cast<const f32x4_t*>(xr + 16);
                x_max[0] = lf_largest(x1, lf_largest(x0, x_max[0]));
                p = lf_split<true>(x0, x1);
            }
            return p;
        };
        LfParts xs_of[C];
        if (kSplitFirst) {
#pragma unroll
            for (int u = 0; u < C; ++u) xs_of[u] = parts_of_x(u);
        }
        __builtin_amdgcn_sched_barrier(0);   // (all asked for before the first is used)
#pragma unroll
        for (int u = 0; u < C; ++u) {
            low |= lf_low_bits(wv0[u], wv1[u]);
            w_max = lf_largest(wv1[u], lf_largest(wv0[u], w_max));
        }
        if (__any(low != 0)) {   // uniform
#pragma unroll
            for (int u = 0; u < C; ++u) {
                const LfParts xp = kSplitFirst ? xs_of[u] : parts_of_x(u), wp = lf_split<true>(wv0[u], wv1[u]);
                acc = lf_mfma(wp.lo, xp.hi, acc);
                acc = lf_mfma(wp.mid, xp.mid, acc);
                acc = lf_mfma(wp.mid, xp.hi, acc);
                acc = lf_mfma(wp.hi, xp.lo, acc);
                acc = lf_mfma(wp.hi, xp.mid, acc);
                acc = lf_mfma(wp.hi, xp.hi, acc);
            }
        } else {
#pragma unroll
            for (int u = 0; u < C; ++u) {
                const LfParts xp = kSplitFirst ? xs_of[u] : parts_of_x(u);
                const uint4 hi = lf_upper(wv0[u], wv1[u]);
                acc = lf_mfma(hi, xp.lo, acc);
                acc = lf_mfma(hi, xp.mid, acc);
                acc = lf_mfma(hi, xp.hi, acc);
            }
        }
    };
    auto multiply = [&](int piece) {
#pragma unroll
        for (int at = 0; at < kStreamK / kLfBK; at += STEPS)
            if (per - piece * (kStreamK / kLfBK) > at) multiply_steps(std::integral_constant<int, STEPS>(), at);   // uniform
    };
    auto settle = [] {   // between a wave's own writes and reads of LDS: an order for the compiler, no instruction
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto turn = [&](int set, int piece, bool more) {
        put(set, piece);
        if (more) request(set, piece + 2);
        settle();
        multiply(piece);
        settle();
    };
    request(0, 0);
    if (pieces > 1) {
        request(1, 1);
        int p = 0;
        for (; p + 2 < pieces; p += 2) {
            turn(0, p, true);
            turn(1, p + 1, true);
        }
        turn(0, p, false);
        turn(1, p + 1, false);
    } else {
        turn(0, 0, false);
    }
    __shared__ int far_rows[4];
    {
        float most = w_max;
#pragma unroll
        for (int i = 0; i < kXMax; ++i) most = lf_largest(most, x_max[i]);
        const bool far = __any(!(most <= kLfHuge));
        if (lane == 0) far_rows[wave] = far;
    }
    __syncthreads();
    float(*part)[64][5] = reinterpret_cast<float(*)[64][5]>(ls_lds);
    float(*row_max)[64][1 + kXMax] = reinterpret_cast<float(*)[64][1 + kXMax]>(ls_lds + 3 * 64 * 5);   // of each wave's lanes
    row_max[wave][lane][0] = w_max;
#pragma unroll
    for (int i = 0; i < kXMax; ++i) row_max[wave][lane][1 + i] = x_max[i];
    if (wave > 0) {
#pragma unroll
        for (int j = 0; j < 4; ++j) part[wave - 1][lane][j] = acc[j];
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int g = 0; g < 3; ++g)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[j] += part[g][lane][j];
    // acc[j] = C[n = n0 + 4 q + j][m = r]
    if (r < M) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (n0 + q * 4 + j < N) y[(int64_t)r * ldy + n0 + q * 4 + j] = acc[j];
    }
    // which of them are not the parts' (over what was stored)
    if (!(far_rows[0] | far_rows[1] | far_rows[2] | far_rows[3]) &&
        !__any(!(lf_largest(acc, 0.f) < INFINITY && lf_least(acc, INFINITY) >= kLfTiny))) return;
    auto largest_of = [&](int first_lane, int step, int lanes, int i) {
        float m = 0.f;
        for (int g = 0; g < 4; ++g)
            for (int l = 0; l < lanes; ++l) m = lf_largest(m, row_max[g][first_lane + l * step][i]);
        return m;
    };
    const int row = min(r, MR - 1);
    float xm = 0.f;
    if (kSplitFirst) {
#pragma unroll
        for (int i = 0; i < kXMax; ++i)
            if (i == row >> 1) xm = largest_of((row & 1) * 32, 1, 32, 1 + i);
    } else {
        xm = largest_of(row, 16, 4, 1);
    }
    unsigned out = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (r < M && n0 + q * 4 + j < N && lf_outside(acc[j], xm, largest_of(q * 4 + j, 16, 4, 0))) out |= 1u << j;
    if (!__any(out != 0)) return;
    const f32x4_t o = lf_by_f32<true>(x + (int64_t)min(r, M - 1) * ldx, w + (int64_t)min(n0 + r, N - 1) * ldw, q, K, per, 4 * blockIdx.y, 4);
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (out >> j & 1) y[(int64_t)r * ldy + n0 + q * 4 + j] = o[j];
}

// Few output rows (decoding): a wave forms four neighbouring outputs of ONE row from 16-byte loads of the operand
// row and of four weight rows, no LDS, no barrier; grid = (column groups of 16, rows, products).  With segments
// the row's weight is found from the segment table.  Needs K % 8 == 0 (bf16) / K % 4 == 0 (fp32) and aligned rows.
template <bool F32>
__global__ __launch_bounds__(256) void linear_fewrows_kernel(const void* __restrict__ x_, int64_t ldx,
                                                             const void* __restrict__ w_, int64_t ldw,
                                                             float* __restrict__ y, int64_t ldy, int N, int K,
                                                             int64_t zx, int64_t zw, int64_t zy, RowSegments sg,
                                                             int segments) {
    typedef typename std::conditional<F32, float, uint16_t>::type T_;
    const T_* x = (const T_*)x_;
    const T_* w = (const T_*)w_;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int64_t row = blockIdx.y, xrow = row;
    if (sg.seg) {
        if (row >= sg.seg[segments]) return;
        int lo = 0, hi = segments;              // the segment that holds the row
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (sg.seg[mid] <= row) lo = mid; else hi = mid;
        }
        w += (int64_t)lo * zw;
        xrow = sg.src ? sg.src[row] / sg.src_div : row;
    } else {
        x += blockIdx.z * zx;
        w += blockIdx.z * zw;
        y += blockIdx.z * zy;
    }
    const int n0 = (blockIdx.x * 4 + wave) * 4;
    if (n0 >= N) return;
    const T_* xr = x + xrow * ldx;
    const T_* wr[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) wr[j] = w + (int64_t)(n0 + j < N ? n0 + j : n0) * ldw;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    constexpr int PER = F32 ? 4 : 8;
    for (int k = lane * PER; k < K; k += 64 * PER) {
        const uint4 xv = ld16(xr + k);
        uint4 wv[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) wv[j] = ld16_nt(wr[j] + k);
        if (F32) {
            const float xf[4] = {__uint_as_float(xv.x), __uint_as_float(xv.y), __uint_as_float(xv.z), __uint_as_float(xv.w)};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float wf[4] = {__uint_as_float(wv[j].x), __uint_as_float(wv[j].y), __uint_as_float(wv[j].z),
                                     __uint_as_float(wv[j].w)};
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[j] = fmaf(xf[e], wf[e], acc[j]);
            }
        } else {
            const uint32_t xp[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t wp[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[j] = fmaf(bf16_lo(xp[e]), bf16_lo(wp[e]), acc[j]);
                    acc[j] = fmaf(bf16_hi(xp[e]), bf16_hi(wp[e]), acc[j]);
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float tot = wave_sum(acc[j]);
        if (lane == 0 && n0 + j < N) y[row * ldy + n0 + j] = tot;
    }
}

}  // namespace mv

template <int TM, int TN, int KG, int PF, bool DB>
static int launch_linear_f32_tiles(const float* x, int64_t ldx, const float* w, int64_t ldw, float* y, int64_t ldy, int m,
                                   int n, int k, int batch, int64_t zx, int64_t zw, int64_t zy, hipStream_t s,
                                   mv::RowSegments sg) {
    using namespace mv;
    constexpr int BM = 32 * TM, BN = 32 * TN;
    const int64_t cols = (n + BN - 1) / BN, rows = (m + BM - 1) / BM, groups = (cols + 7) / 8 * 8 * rows;
    if (groups > 0x7fffffff) return MV_ERR_UNSUPPORTED;
    size_t lds = (size_t)KG * (DB ? 2 : 1) * 3 * (BM + BN) * kLfBK * 2;
    const size_t meet = (size_t)(KG - 1) * 256 * (4 / KG * TM * TN * 4 + 1) * 4;
    if (meet > lds) lds = meet;
    const bool vec = k % 4 == 0 && aligned16(x) && ldx % 4 == 0 && zx % 4 == 0 && aligned16(w) && ldw % 4 == 0 && zw % 4 == 0;
    static LdsOptIn done[2];
    const auto kernel = vec ? linear_any_f32_kernel<TM, TN, KG, PF, DB, true> : linear_any_f32_kernel<TM, TN, KG, PF, DB, false>;
    if (const int rc = ensure_dynamic_lds((const void*)kernel, lds, done[vec])) return rc;
    hipLaunchKernelGGL(kernel, dim3((unsigned)groups, 1, batch), dim3(256 * KG), lds, s, x, ldx, w, ldw, y, ldy, m, n, k,
                       zx, zw, zy, sg);
    return check_launch();
}

// whether the rows are few enough for the streamed form
static bool streams_f32(int m, int n, int k) {
    using namespace mv;
    if (n < kStreamNarrow || k >= kStreamLongK) return m <= kStreamRowsMore;
    return m <= (n < kStreamWide || k > kStreamShortK ? kStreamRows : kStreamRowsLess);
}

static int stream_form(int m, int k, int slices) { return m > 8 ? 3 : m > 4 ? 2 : k / slices > mv::kStreamOneStep ? 1 : 0; }

static int launch_linear_stream(const float* x, int64_t ldx, const float* w, int64_t ldw, float* y, int64_t ldy, int m, int n,
                                int k, int slices, hipStream_t s) {
    using namespace mv;
    const int form = stream_form(m, k, slices);
    const size_t lds = (size_t)4 * (16 * kStreamPad * 4 + stream_x_bytes(form == 3 ? 16 : form == 2 ? 8 : 4));
    static LdsOptIn done[4];
    const auto kernel = form == 0   ? linear_stream_f32_kernel<4, 1>
                        : form == 1 ? linear_stream_f32_kernel<4, 4>
                        : form == 2 ? linear_stream_f32_kernel<8, 4>
                                    : linear_stream_f32_kernel<16, 4>;
    if (const int rc = ensure_dynamic_lds((const void*)kernel, lds, done[form])) return rc;
    hipLaunchKernelGGL(kernel, dim3((n + 15) / 16, slices), dim3(256), lds, s, x, ldx, w, ldw, y, ldy, m, n, k);
    return check_launch();
}

// Which fp32 form.  Few rows of one product stream the weights (see kStreamRows).  Otherwise the tile by the time the launch
// takes in it, in hundredths of a us: with n = tiles over compute units, rounded up, a start, an end of every tile (its sums' way
// out), and a step in which the workgroups of a unit take turns at its matrix unit, vector unit and LDS (in four groups a quarter of the
// steps, one workgroup to a unit).  A launch of few tiles takes small ones and many groups, a large one the tile that reads
// and splits its operands least often; a short k is told by the tiles' ends.  Fitted to 1000 shapes of 17 to 2048 rows, 64 to 65536
// outputs and k of 64 to 8192: the tile it names takes 0.9 % more than the best of the six in the mean, 33 % at most (few rows of wide
// outputs, which wait for memory: 17 rows 48000 x 2048 108 us, 81 in 32 x 32; 65536 x 1024 69, 53 in 64 x 64 by two groups).  us in (outputs of the tile, groups), weights of bf16 values:
//   567 rows 9472 x 1024: 149 (32 x 32, 4), 82 (64 x 64, 4), 64 (64 x 64, 2), 61 (64 x 64), 49 (64 x 128), 62 (128 x 128)
//   567 rows 1024 x 5120:  78, 54, 61, 89, 129, 203        33 rows 1024 x 5120: 26, 49, 58, 88, 127, 200
//   2048 rows 16384 x 4096: 2724, 1632, 1273, 1208, 944, 873
//   1024 rows 32000 x 64: 350, 163, 103, 62.5, 61, 60.5 (70 on the fp32 instruction)    567 rows 9472 x 256: -, 37, 26.8, 23.7, 22, 27.5
// With segments `m` bounds a segment, not the launch: the rows are taken to be spread evenly.
static int f32_tiles(int64_t rows, int n, int k, int batch) {
    using namespace mv;
    const int64_t cus = num_cus();
    auto turns = [&](int bm, int bn) { return (((rows + bm - 1) / bm) * ((n + bn - 1) / bn) * batch + cus - 1) / cus; };
    const int64_t steps = (k + kLfBK - 1) / kLfBK, quarter = (steps + 3) / 4;
    const int64_t n32 = turns(32, 32), n64 = turns(64, 64), n128 = turns(64, 128), n256 = turns(128, 128);
    const int64_t cost[6] = {284 + n32 * (333 + 47 * quarter),
                             175 + n64 * (265 + 141 * quarter),
                             226 + 206 * n64 + 2 * quarter * (24 + 48 * n64),
                             294 + 133 * n64 + steps * (27 + 23 * n64),
                             340 + 267 * n128 + steps * (29 + 37 * n128),
                             114 + 744 * n256 + steps * (50 + 59 * n256)};
    int best = 0;
    for (int i = 1; i < 6; ++i)
        if (cost[i] < cost[best]) best = i;
    return best;
}

static int launch_linear_f32(const float* x, int64_t ldx, const float* w, int64_t ldw, float* y, int64_t ldy, int m, int n,
                             int k, int batch, int64_t zx, int64_t zw, int64_t zy, hipStream_t s, mv::RowSegments sg,
                             int total_rows) {
    using namespace mv;
    if (streams_f32(m, n, k) && !sg.seg && batch == 1 && k % 4 == 0 && ldx % 4 == 0 &&
        ldw % 4 == 0 && aligned16(x) && aligned16(w)) {
        return launch_linear_stream(x, ldx, w, ldw, y, ldy, m, n, k, 1, s);
    }
    switch (f32_tiles(sg.seg ? (total_rows + batch - 1) / batch : m, n, k, batch)) {
        case 0: return launch_linear_f32_tiles<1, 1, 4, 2, true>(x, ldx, w, ldw, y, ldy, m, n, k, batch, zx, zw, zy, s, sg);
        case 1: return launch_linear_f32_tiles<2, 2, 4, 1, false>(x, ldx, w, ldw, y, ldy, m, n, k, batch, zx, zw, zy, s, sg);
        case 2: return launch_linear_f32_tiles<2, 2, 2, 1, false>(x, ldx, w, ldw, y, ldy, m, n, k, batch, zx, zw, zy, s, sg);
        case 3: return launch_linear_f32_tiles<2, 2, 1, 1, false>(x, ldx, w, ldw, y, ldy, m, n, k, batch, zx, zw, zy, s, sg);
        case 4: return launch_linear_f32_tiles<2, 4, 1, 1, false>(x, ldx, w, ldw, y, ldy, m, n, k, batch, zx, zw, zy, s, sg);
        default: return launch_linear_f32_tiles<4, 4, 1, 1, false>(x, ldx, w, ldw, y, ldy, m, n, k, batch, zx, zw, zy, s, sg);
    }
}

extern "C" int mv_linear_any_form(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0) return -1;
    return streams_f32(m, n, k) && k % 4 == 0 ? stream_form(m, k, 1) : 4 + f32_tiles(m, n, k, 1);
}

static int launch_linear_any(const void* x, int64_t ldx, const void* w, int64_t ldw, float* y, int64_t ldy, int m, int n,
                             int k, int f32, int batch, int64_t zx, int64_t zw, int64_t zy, mv_stream_t stream,
                             mv::RowSegments sg = mv::RowSegments{nullptr, nullptr, 1}, int few_rows = 0,
                             bool big_tiles = false, int total_rows = 0) {
    using namespace mv;
    const dim3 grid((n + kLaBN - 1) / kLaBN, (m + kLaBM - 1) / kLaBM, batch);
    if (grid.y > 65535 || batch > 65535) return MV_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
    if (few_rows > 0) {
        const int per = f32 ? 4 : 8;
        const bool fits = k % per == 0 && ldx % per == 0 && ldw % per == 0 && zx % per == 0 && zw % per == 0 &&
                          aligned16(x) && aligned16(w);
        if (fits) {
            const dim3 g((n + 15) / 16, few_rows, sg.seg ? 1 : batch);
            if (f32) hipLaunchKernelGGL(linear_fewrows_kernel<true>, g, dim3(256), 0, s, x, ldx, w, ldw, y, ldy, n, k, zx, zw, zy, sg, batch);
            else hipLaunchKernelGGL(linear_fewrows_kernel<false>, g, dim3(256), 0, s, x, ldx, w, ldw, y, ldy, n, k, zx, zw, zy, sg, batch);
            return check_launch();
        }
    }
    if (f32) {
        return launch_linear_f32((const float*)x, ldx, (const float*)w, ldw, y, ldy, m, n, k, batch, zx, zw, zy, s, sg, total_rows);
    } else {
        const int vx = aligned16(x) && ldx % 8 == 0 && zx % 8 == 0, vw = aligned16(w) && ldw % 8 == 0 && zw % 8 == 0;
        if (big_tiles && n >= kLbBN) {
            const dim3 big((n + kLbBN - 1) / kLbBN, (m + kLbBM - 1) / kLbBM, batch);
            hipLaunchKernelGGL(linear_any_bf16_big_kernel, big, dim3(256), 0, s, (const uint16_t*)x, ldx,
                               (const uint16_t*)w, ldw, y, ldy, m, n, k, vx, vw, zx, zw, zy, sg);
            return check_launch();
        }
        hipLaunchKernelGGL(linear_any_bf16_kernel, grid, dim3(256), 0, s, (const uint16_t*)x, ldx, (const uint16_t*)w,
                           ldw, y, ldy, m, n, k, vx, vw, zx, zw, zy, sg);
    }
    return check_launch();
}

// k-slices of a streamed fp32 product whose next kernel adds them: where its strips of sixteen outputs leave compute units
// idle, as many as there are units for, each wave keeping kStreamSlice steps or more.  3 rows, us whole -> two -> four slices:
// 1024 x 5120 20.9 -> 14.3 -> 11.5, 1024 x 4096 15.4 -> 10.3 -> 7.6, 2048 x 4096 (128 strips) 16.5 -> 11.6 -> 12.4, 4096 x 16384 (256) 68.5 ->
// 72.6; 1024 x 1024 (two steps a wave in four) 6.9 -> 6.8 -> 6.6.  The error against 64 bits falls with the slices (6.4e-7 -> 3.2e-7).
extern "C" int mv_linear_any_slab_count(int m, int n, int k) {
    using namespace mv;
    if (m <= 0 || n <= 0 || k <= 0 || !streams_f32(m, n, k) || k % 4) return 1;
    const int strips = (n + 15) / 16, steps = (k + kLfBK - 1) / kLfBK;
    int ks = 1;
    while (2 * ks * strips <= num_cus() && steps >= 2 * ks * 4 * kStreamSlice) ks *= 2;
    return ks;
}

extern "C" int mv_linear_any_slabs(const float* x, int64_t ldx, const float* w, int64_t ldw, float* slabs, size_t slabs_bytes,
                                   int m, int n, int k, mv_stream_t stream) {
    using namespace mv;
    if (m < 0 || n <= 0 || k <= 0) return MV_ERR_INVALID_ARG;
    if (m == 0) return MV_OK;
    if (!x || !w || !slabs || ldx < k || ldw < k) return MV_ERR_INVALID_ARG;
    const int ks = mv_linear_any_slab_count(m, n, k);
    if (slabs_bytes < (size_t)ks * m * n * sizeof(float)) return MV_ERR_WORKSPACE;
    if (ks == 1) return mv_linear_any(x, ldx, w, ldw, slabs, n, m, n, k, 1, stream);
    if (ldx % 4 || ldw % 4 || !aligned16(x) || !aligned16(w)) return MV_ERR_UNSUPPORTED;
    return launch_linear_stream(x, ldx, w, ldw, slabs, n, m, n, k, ks, (hipStream_t)stream);
}

extern "C" int mv_linear_any(const void* x, int64_t ldx, const void* w, int64_t ldw, float* y, int64_t ldy,
                             int m, int n, int k, int f32, mv_stream_t stream) {
    if (m < 0 || n <= 0 || k <= 0) return MV_ERR_INVALID_ARG;
    if (m == 0) return MV_OK;
    if (!x || !w || !y || ldx < k || ldw < k || ldy < n) return MV_ERR_INVALID_ARG;
    return launch_linear_any(x, ldx, w, ldw, y, ldy, m, n, k, f32, 1, 0, 0, 0, stream,
                             mv::RowSegments{nullptr, nullptr, 1}, 0, m >= 256);
}

// `heads` products in one launch: y[:, h*zy + ..n] = x[:, h*zx + ..k] . W_h^T with W_h = w + h*zw ([n,k], row stride ldw)
extern "C" int mv_linear_heads(const void* x, int64_t ldx, int64_t zx, const void* w, int64_t ldw, int64_t zw, float* y,
                               int64_t ldy, int64_t zy, int m, int n, int k, int heads, int f32, mv_stream_t stream) {
    if (m < 0 || n <= 0 || k <= 0 || heads <= 0 || zx < 0 || zw < 0 || zy < 0) return MV_ERR_INVALID_ARG;
    if (m == 0) return MV_OK;
    if (!x || !w || !y || ldx < (heads - 1) * zx + k || ldw < k || ldy < (heads - 1) * zy + n) return MV_ERR_INVALID_ARG;
    return launch_linear_any(x, ldx, w, ldw, y, ldy, m, n, k, f32, heads, zx, zw, zy, stream,
                             mv::RowSegments{nullptr, nullptr, 1}, m <= mv::kFewRows ? m : 0, m >= 256);
}

// Products by segment: output rows seg[e] .. seg[e+1] (e < segments) use weight w + e*zw; `max_rows` bounds the
// rows of any one segment (the launch has that many row tiles per segment, the ones past a segment's end leave
// at once).  src: operand row of output row i is src[i] / src_div (NULL: i).  total_rows = seg[segments] as the host
// knows it (the rows of `y`): few of them take the form without tiles.
extern "C" int mv_linear_segments(const void* x, int64_t ldx, const void* w, int64_t ldw, int64_t zw, float* y,
                                  int64_t ldy, const int32_t* seg, const int32_t* src, int src_div, int segments,
                                  int max_rows, int total_rows, int n, int k, int f32, mv_stream_t stream) {
    if (max_rows < 0 || n <= 0 || k <= 0 || segments <= 0 || src_div <= 0 || zw < 0) return MV_ERR_INVALID_ARG;
    if (max_rows == 0) return MV_OK;
    if (!x || !w || !y || !seg || ldx < k || ldw < k || ldy < n) return MV_ERR_INVALID_ARG;
    return launch_linear_any(x, ldx, w, ldw, y, ldy, max_rows, n, k, f32, segments, 0, zw, 0, stream,
                             mv::RowSegments{seg, src, src_div}, total_rows <= mv::kFewRows ? total_rows : 0,
                             total_rows / segments >= 96, total_rows);
}
