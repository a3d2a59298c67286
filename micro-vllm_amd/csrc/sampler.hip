// Token selection on the device, one workgroup per row of bf16 logits, or several where that is the faster.
//   argmax_kernel : greedy pick (lowest index on ties); reads the row once with 16-byte loads.
//   sample_kernel : temperature -> top-k -> softmax -> top-p -> draw, the recipe of the reference's
//                   Sampler._sample_impl (core/layer/sampler.py:21-43), as one launch instead of
//                   topk + softmax + sort + cumsum + multinomial + two gathers.  The k largest
//                   logits are found by a two-pass radix select on the 16 bf16 bits (division by a
//                   positive temperature does not change the order), or for k up to 256 among the entries
//                   (up to 512) that reach the k-th largest of the threads' maxima, gathered into LDS (ties at
//                   the threshold by ascending index, so the result is deterministic), sorted there,
//                   and the draw is the inverse CDF of the caller's uniform number.
#include "common.h"

#include <algorithm>

namespace mv {

constexpr int kAmThreads = 1024;

__device__ __forceinline__ void amax_merge(float& v, int& i, float ov, int oi) {
    if (ov > v || (ov == v && oi < i)) {
        v = ov;
        i = oi;
    }
}

__global__ __launch_bounds__(kAmThreads) void argmax_kernel(const uint16_t* __restrict__ logits,
                                                          int64_t ld, int n,
                                                          int64_t* __restrict__ ids) {
    __shared__ float sv[kAmThreads / 64];
    __shared__ int si[kAmThreads / 64];
    const uint16_t* row = logits + (int64_t)blockIdx.x * ld;
    float best = -INFINITY;
    int bi = 0x7fffffff;
    const int nvec = n >> 3;
    for (int c = threadIdx.x; c < nvec; c += kAmThreads) {
        const uint4 v = ld16(row + c * 8);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            amax_merge(best, bi, bf16_lo(w[j]), c * 8 + 2 * j);
            amax_merge(best, bi, bf16_hi(w[j]), c * 8 + 2 * j + 1);
        }
    }
    for (int c = (nvec << 3) + threadIdx.x; c < n; c += kAmThreads)
        amax_merge(best, bi, bf16_bits_to_f32(row[c]), c);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        amax_merge(best, bi, __shfl_xor(best, o, 64), __shfl_xor(bi, o, 64));
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        sv[wid] = best;
        si[wid] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kAmThreads / 64; ++w) amax_merge(best, bi, sv[w], si[w]);
        ids[blockIdx.x] = bi == 0x7fffffff ? 0 : bi;  // all-NaN row: index 0
    }
}

// Few rows: one workgroup per row would leave the chip idle and read a 128k-entry row through a
// single CU (about 15 us).  The row is cut into parts, one workgroup each; partial results go to the
// caller's workspace (tickets | values | indices) with write-through stores, and the workgroup that
// draws the last arrival ticket of a row merges them.  The tickets are zero when the caller hands
// the workspace over for the first time and are returned to zero by every launch.  The merge is a maximum under a total order (value, then lowest
// index), so the result does not depend on arrival order.
constexpr int kAmPartThreads = 256;
constexpr int kAmMaxParts = 64;
constexpr int kAmMaxRows = 64;
constexpr size_t kAmTicketBytes = (size_t)kAmMaxRows * 64 * sizeof(unsigned int);  // 256 bytes apart
constexpr size_t kAmPartBytes = (size_t)kAmMaxRows * kAmMaxParts * 4;
constexpr size_t kAmWorkspaceBytes = kAmTicketBytes + 2 * kAmPartBytes;

struct AmScratch {
    float* val;
    int* idx;
    unsigned int* ticket;
};

template <int AHEAD>
__global__ __launch_bounds__(kAmPartThreads) void argmax_parts_kernel(const uint16_t* __restrict__ logits,
                                                                      int64_t ld, int n, int parts,
                                                                      int vec_per_part, AmScratch sc,
                                                                      int64_t* __restrict__ ids) {
    __shared__ float sv[kAmPartThreads / 64];
    __shared__ int si[kAmPartThreads / 64];
    __shared__ int is_last;
    const int rowi = blockIdx.x / parts, part = blockIdx.x - rowi * parts;
    const uint16_t* row = logits + (int64_t)rowi * ld;
    float best = -INFINITY;
    int bi = 0x7fffffff;
    const int nvec = n >> 3;
    const int c0 = part * vec_per_part, c1 = min(nvec, c0 + vec_per_part);
    for (int b = c0 + threadIdx.x; b < c1; b += AHEAD * kAmPartThreads) {
        uint4 v[AHEAD];   // requested together: a part is one trip to memory, not one per 16 bytes of a thread
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) v[u] = ld16(row + (int64_t)min(b + u * kAmPartThreads, c1 - 1) * 8);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int c = min(b + u * kAmPartThreads, c1 - 1);   // (the last one again: it changes nothing)
            const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                amax_merge(best, bi, bf16_lo(w[j]), c * 8 + 2 * j);
                amax_merge(best, bi, bf16_hi(w[j]), c * 8 + 2 * j + 1);
            }
        }
    }
    if (part == parts - 1)
        for (int c = (nvec << 3) + threadIdx.x; c < n; c += kAmPartThreads)
            amax_merge(best, bi, bf16_bits_to_f32(row[c]), c);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        amax_merge(best, bi, __shfl_xor(best, o, 64), __shfl_xor(bi, o, 64));
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        sv[wid] = best;
        si[wid] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kAmPartThreads / 64; ++w) amax_merge(best, bi, sv[w], si[w]);
        const int slot = rowi * kAmMaxParts + part;
        __hip_atomic_store(reinterpret_cast<unsigned int*>(sc.val + slot), __float_as_uint(best),
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(sc.idx + slot, bi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // both stores have left before the ticket
        const unsigned old = __hip_atomic_fetch_add(sc.ticket + rowi * 64, 1u, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        is_last = old == (unsigned)parts - 1u;
        if (is_last)  // back to zero for the next launch; nobody else touches it in this one
            __hip_atomic_store(sc.ticket + rowi * 64, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!is_last || threadIdx.x >= 64) return;
    best = -INFINITY;
    bi = 0x7fffffff;
    if (lane < parts) {
        const int slot = rowi * kAmMaxParts + lane;
        best = __uint_as_float(__hip_atomic_load(reinterpret_cast<unsigned int*>(sc.val + slot),
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        bi = __hip_atomic_load(sc.idx + slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        amax_merge(best, bi, __shfl_xor(best, o, 64), __shfl_xor(bi, o, 64));
    if (lane == 0) ids[rowi] = bi == 0x7fffffff ? 0 : bi;  // all-NaN row: index 0
}

static AmScratch am_scratch(void* workspace) {
    unsigned char* p = (unsigned char*)workspace;
    return AmScratch{(float*)(p + kAmTicketBytes), (int*)(p + kAmTicketBytes + kAmPartBytes),
                     (unsigned int*)p};
}

// ---------------------------------------------------------------- top-k / top-p sampling
constexpr int kSmThreads = 1024;
constexpr int kSmMaxK = 1024;
constexpr int kSmKeep = 16;   // 16-byte chunks of the row a thread keeps in registers
constexpr int kSmQuickK = 256;   // up to this k the candidates are found through the threads' maxima
constexpr int kSmQuickMost = 512;   // ... and there are at most this many of them

// Order-preserving signed keys of a pair of bf16 values, and (the same map again) the values of a pair of keys.  NaNs lie
// above +inf and below -inf.
typedef __attribute__((ext_vector_type(2))) short s16x2_t;
constexpr short kKeyLow = -32768, kKeyInf = 0x7f80, kKeyNegInf = (short)0x807f;
__device__ __forceinline__ s16x2_t pair_key(s16x2_t x) { return x ^ ((x >> 15) & (short)0x7fff); }

// order-preserving 16-bit key of a bf16 value (larger key = larger value); NaN sorts lowest
__device__ __forceinline__ unsigned bf16_key(unsigned bits) {
    if ((bits & 0x7f80u) == 0x7f80u && (bits & 0x7fu)) return 0u;
    return (bits & 0x8000u) ? (~bits & 0xffffu) : (bits | 0x8000u);
}

// inclusive scan over the workgroup (one value per thread); `ws` holds one slot per wave
template <typename T>
__device__ __forceinline__ T block_scan_incl(T v, T* ws, T& total) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T u = __shfl_up(v, o, 64);
        if (lane >= o) v += u;
    }
    __syncthreads();  // ws may still be read from a previous scan
    if (lane == 63) ws[wid] = v;
    __syncthreads();
    T base = 0, tot = 0;
    for (int w = 0; w < kSmThreads / 64; ++w) {
        const T x = ws[w];
        if (w < wid) base += x;
        tot += x;
    }
    total = tot;
    return v + base;
}

struct SampleShared {
    // Sixteen copies of the 256-bin histogram, one per lane group: logits share a handful of
    // exponents, so with a single copy nearly every lane of a wave adds to the same LDS word and the
    // adds are served one after the other.  A thread also counts runs of equal bins in a register
    // and adds a whole run at once.
    __attribute__((aligned(16))) unsigned hist[16][256];
    unsigned sh_u[8];
    float c_val[kSmMaxK];
    int c_idx[kSmMaxK];
    float ws_f[kSmThreads / 64];
    unsigned ws_u[kSmThreads / 64];
};

// A selection reads the row ONCE: the first kSmKeep chunks of every thread (rows up to 131 072 entries
// whole) stay in registers for all its passes, requested back to back so that the read costs
// one memory round trip instead of one per chunk and pass; longer rows stream the rest.
template <int KEEP>
__device__ __forceinline__ void load_row(uint4 (&v)[KEEP], const uint16_t* row, int nvec) {
#pragma unroll
    for (int i = 0; i < KEEP; ++i) v[i] = ld16(row + (int64_t)min((int)threadIdx.x + i * kSmThreads, nvec - 1) * 8);
}

__device__ __forceinline__ s16x2_t as_pair(uint32_t v) { return __builtin_bit_cast(s16x2_t, v); }
__device__ __forceinline__ uint4 to_keys(uint4 v) {
    v.x = __builtin_bit_cast(uint32_t, pair_key(as_pair(v.x)));
    v.y = __builtin_bit_cast(uint32_t, pair_key(as_pair(v.y)));
    v.z = __builtin_bit_cast(uint32_t, pair_key(as_pair(v.z)));
    v.w = __builtin_bit_cast(uint32_t, pair_key(as_pair(v.w)));
    return v;
}
// Largest of the values so far as signed and as unsigned 16-bit numbers, two instructions a pair where keys take five: bf16
// values of positive sign lie in the order of their keys, and the NaNs of negative sign are the largest unsigned numbers.
typedef __attribute__((ext_vector_type(2))) unsigned short u16x2_t;
struct Largest {
    s16x2_t s = {kKeyLow, kKeyLow};
    u16x2_t u = {0, 0};
    __device__ __forceinline__ void add(const uint4& v) {
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s = __builtin_elementwise_max(s, as_pair(w[j]));
            u = __builtin_elementwise_max(u, __builtin_bit_cast(u16x2_t, w[j]));
        }
    }
    __device__ __forceinline__ short top() const { return s.x > s.y ? s.x : s.y; }
    __device__ __forceinline__ bool nan() const { return top() > kKeyInf || max((int)u.x, (int)u.y) > 0xff80; }
};
// largest key of the eight of a chunk or of `top`
__device__ __forceinline__ short top_key(short top, const uint4& v) {
    const uint4 k = to_keys(v);
    const s16x2_t m = __builtin_elementwise_max(__builtin_elementwise_max(as_pair(k.x), as_pair(k.y)),
                                                __builtin_elementwise_max(as_pair(k.z), as_pair(k.w)));
    const short t = m.x > m.y ? m.x : m.y;
    return t > top ? t : top;
}
// what stands for the keys beside a bound: the values themselves where the bound is one of positive sign
__device__ __forceinline__ uint4 keys_beside(int thr, const uint4& v) { return thr >= 0 ? v : to_keys(v); }
// how many of eight entries reach the bound
__device__ __forceinline__ unsigned reaching(const uint4& keys, int thr) {
    const uint32_t w[4] = {keys.x, keys.y, keys.z, keys.w};
    const s16x2_t m = __builtin_elementwise_max(__builtin_elementwise_max(as_pair(w[0]), as_pair(w[1])),
                                                __builtin_elementwise_max(as_pair(w[2]), as_pair(w[3])));
    unsigned n = 0;
    if (m.x >= thr || m.y >= thr) {
#pragma unroll
        for (int j = 0; j < 4; ++j) n += (unsigned)(as_pair(w[j]).x >= thr) + (unsigned)(as_pair(w[j]).y >= thr);
    }
    return n;
}
// those entries of chunk c into cand from `slot` on, as key, then ~index: unsigned order is the row's order
__device__ __forceinline__ void list_entries(const uint4& keys, int c, int thr, unsigned& slot, uint64_t* cand, unsigned* zero_flag) {
    const uint32_t w[4] = {keys.x, keys.y, keys.z, keys.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const s16x2_t kk = as_pair(w[j >> 1]);
        const int key = j & 1 ? kk.y : kk.x;
        if (key < thr) continue;
        cand[slot++] = (uint64_t)(unsigned)(key + 32768) << 32 | (unsigned)~(c * 8 + j);
        if (key == -1) *zero_flag = 1;                  // -0.0
    }
}
// The k-th largest of N 16-bit maxima in LDS (offset by 32768: unsigned order), four bits a round: wave w counts who
// reaches digit w.  `reach`: two words per wave, in turn, so that a round is one barrier.
template <int N>
__device__ __forceinline__ unsigned kth_largest(const unsigned short* maxima, unsigned* reach, int k) {
    constexpr int PER = N / 64, WORDS = PER / 2;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    uint32_t mw[WORDS];
#pragma unroll
    for (int j = 0; j < WORDS; j += 4) {
        const uint4 m = *reinterpret_cast<const uint4*>(maxima + (j / 4 * 64 + lane) * 8);
        mw[j] = m.x; mw[j + 1] = m.y; mw[j + 2] = m.z; mw[j + 3] = m.w;
    }
    unsigned bound = 0;
    for (int shift = 12; shift >= 0; shift -= 4) {
        const unsigned digit_bound = bound | ((unsigned)wave << shift);
        unsigned cnt = 0;
#pragma unroll
        for (int j = 0; j < WORDS; ++j) {
            cnt += __popcll(__ballot((mw[j] & 0xffffu) >= digit_bound));
            cnt += __popcll(__ballot((mw[j] >> 16) >= digit_bound));
        }
        unsigned* turn = reach + (shift & 4 ? 16 : 0);
        if (lane == 0) turn[wave] = cnt;
        __syncthreads();
        int digit = 0;
#pragma unroll
        for (int w = 1; w < 16; ++w)
            if (turn[w] >= (unsigned)k) digit = w;    // fewer reach a larger digit
        bound |= (unsigned)digit << shift;
    }
    return bound;
}
// Up to kSmQuickMost candidates: the place of each by counting who comes before, F threads, one for each, for every part of
// the list (whole waves read the same entry); the first k go to c_val / c_idx.  `ranks` is zero.
__device__ __forceinline__ void place_candidates(SampleShared& sh, const uint64_t* cand, unsigned* ranks, unsigned found, int k) {
    const int tid = threadIdx.x;
    unsigned F = 64;
    while (F < found) F <<= 1;
    const unsigned parts = kSmThreads / F, span = (found + parts - 1) / parts;
    const unsigned i = tid & (F - 1), j0 = tid / F * span, j1 = min(found, j0 + span);
    const uint64_t me = i < found ? cand[i] : 0;
    unsigned before = 0;
    for (unsigned j = j0; j < j1; ++j) before += cand[j] > me;
    if (i < found && before) atomicAdd(&ranks[i], before);
    __syncthreads();
    const unsigned rank = tid < (int)found ? ranks[tid] : (unsigned)k;
    if (rank < (unsigned)k) {      // (threads below F hold entry tid)
        const int key = (int)(me >> 32) - 32768;
        sh.c_val[rank] = bf16_bits_to_f32((unsigned short)(key ^ ((key >> 15) & 0x7fff)));
        sh.c_idx[rank] = (int)~(unsigned)me;
    }
    __syncthreads();
}
// zeros of both signs are equal: among those the index decides
__device__ __forceinline__ void order_zeros(SampleShared& sh, int k) {
    const int tid = threadIdx.x;
    const bool mine = tid < k;
    const float my_val = mine ? sh.c_val[tid] : 0.f;
    const int my_idx = mine ? sh.c_idx[tid] : 0;
    unsigned place = 0;
    if (mine)
        for (int j = 0; j < k; ++j) place += sh.c_val[j] > my_val || (sh.c_val[j] == my_val && sh.c_idx[j] < my_idx);
    __syncthreads();
    if (mine) {
        sh.c_val[place] = my_val;
        sh.c_idx[place] = my_idx;
    }
    __syncthreads();
}

// The k largest entries of a row in order, by a radix selection over 16-bit keys in two passes: any k, rows with NaNs, equal
// entries without end.
__device__ __forceinline__ void radix_select(SampleShared& sh, const uint16_t* row, int nvec, int k) {
    auto& hist = sh.hist;
    auto& sh_u = sh.sh_u;
    auto& c_val = sh.c_val;
    auto& c_idx = sh.c_idx;
    auto& ws_u = sh.ws_u;
    const int tid = threadIdx.x;
    uint4 keep[kSmKeep];
    load_row(keep, row, nvec);
    auto for_each_chunk = [&](auto&& fn) {  // fn(chunk index, 8 values), every thread the same trip count
#pragma unroll
        for (int i = 0; i < kSmKeep; ++i) fn(tid + i * kSmThreads, keep[i]);
        for (int c0 = kSmKeep * kSmThreads; c0 < nvec; c0 += kSmThreads) {
            const int c = c0 + tid;
            fn(c, ld16(row + (int64_t)min(c, nvec - 1) * 8));
        }
    };
    auto for_each = [&](auto&& fn) {  // fn(key, index) over the row
        for_each_chunk([&](int c, const uint4& v) {
            if (c >= nvec) return;
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                fn(bf16_key(w[j] & 0xffffu), c * 8 + 2 * j);
                fn(bf16_key(w[j] >> 16), c * 8 + 2 * j + 1);
            }
        });
    };
    // the bin (scanning from the top) in which the running count reaches `want`
    auto pick_bin = [&](unsigned want, unsigned& bin, unsigned& above) {
        __syncthreads();
        if (tid < 256) {
            unsigned t = 0;
#pragma unroll
            for (int c = 0; c < 16; ++c) t += hist[c][tid];
            hist[0][tid] = t;
        }
        __syncthreads();
        // suffix sums from bin 255 down, all bins at once: thread t holds bin 255 - t; the first
        // thread whose running count reaches `want` names the bin (bin 0 if none does)
        const unsigned h = tid < 256 ? hist[0][255 - tid] : 0u;
        unsigned total;
        const unsigned incl = block_scan_incl(h, ws_u, total);
        if (tid == 0) sh_u[0] = 255u;
        __syncthreads();
        if (tid < 255 && incl >= want) atomicMin(&sh_u[0], (unsigned)tid);
        __syncthreads();
        if ((unsigned)tid == sh_u[0]) sh_u[1] = incl - h;
        __syncthreads();
        if (tid == 0) sh_u[0] = 255u - sh_u[0];
        __syncthreads();
        bin = sh_u[0];
        above = sh_u[1];
        __syncthreads();
    };

    // ---- radix select of the k-th largest key: high byte, then low byte
    unsigned* my_hist = hist[tid & 15];
    unsigned run_bin = 0, run_len = 0;
    auto count = [&](unsigned bin) {
        if (bin != run_bin) {
            if (run_len) atomicAdd(&my_hist[run_bin], run_len);
            run_bin = bin;
            run_len = 0;
        }
        ++run_len;
    };
    auto flush = [&]() {
        if (run_len) atomicAdd(&my_hist[run_bin], run_len);
        run_len = 0;
    };
    for (int i = tid; i < 16 * 256; i += kSmThreads) (&hist[0][0])[i] = 0;
    __syncthreads();
    for_each([&](unsigned key, int) { count(key >> 8); });
    flush();
    unsigned b1, above1;
    pick_bin((unsigned)k, b1, above1);
    for (int i = tid; i < 16 * 256; i += kSmThreads) (&hist[0][0])[i] = 0;
    __syncthreads();
    for_each([&](unsigned key, int) {
        if ((key >> 8) == b1) count(key & 255u);
    });
    flush();
    unsigned b2, above2;
    pick_bin((unsigned)k - above1, b2, above2);
    const unsigned thr = (b1 << 8) | b2;
    const unsigned n_gt = above1 + above2;           // keys strictly above the threshold (< k)
    const unsigned need_eq = (unsigned)k - n_gt;     // threshold-valued entries to take, lowest indices first

    // ---- gather: keys above the threshold in any order, threshold ties in index order
    if (tid == 0) sh_u[2] = 0;
    __syncthreads();
    unsigned eq_base = 0;
    for_each_chunk([&](int c, const uint4& v) {
        if (c - tid >= nvec) return;  // uniform: this pass of the workgroup lies past the row
        unsigned keys[8];
        unsigned my_eq = 0;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        if (c < nvec) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                keys[2 * j] = bf16_key(w[j] & 0xffffu);
                keys[2 * j + 1] = bf16_key(w[j] >> 16);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (keys[j] > thr) {
                    const unsigned slot = atomicAdd(&sh_u[2], 1u);
                    const uint32_t wj = w[j >> 1];
                    c_val[slot] = (j & 1) ? bf16_hi(wj) : bf16_lo(wj);
                    c_idx[slot] = c * 8 + j;
                }
                my_eq += (keys[j] == thr);
            }
        }
        if (eq_base < need_eq) {  // uniform: eq_base is the same in every thread
            unsigned total;
            const unsigned incl = block_scan_incl(my_eq, ws_u, total);
            unsigned rank = eq_base + incl - my_eq;
            if (c < nvec && my_eq) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    if (keys[j] == thr) {
                        if (rank < need_eq) {
                            const uint32_t wj = w[j >> 1];
                            c_val[n_gt + rank] = (j & 1) ? bf16_hi(wj) : bf16_lo(wj);
                            c_idx[n_gt + rank] = c * 8 + j;
                        }
                        ++rank;
                    }
                }
            }
            eq_base += total;
        }
    });
    // pad to a power of two for the sort
    int p2 = 1;
    while (p2 < k) p2 <<= 1;
    __syncthreads();
    if (tid >= k && tid < p2) {
        c_val[tid] = -INFINITY;
        c_idx[tid] = 0x7fffffff;
    }
    // ---- bitonic sort, descending by value, ascending index among equals
    for (int size = 2; size <= p2; size <<= 1) {
        for (int stride = size >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            const int i = tid, j = tid ^ stride;
            if (i < p2 && j > i) {
                const float vi = c_val[i], vj = c_val[j];
                const int ii = c_idx[i], ij = c_idx[j];
                const bool i_first = (vi > vj) || (vi == vj && ii < ij);  // i belongs before j
                const bool want_first = (i & size) == 0;
                if (i_first != want_first) {
                    c_val[i] = vj;
                    c_val[j] = vi;
                    c_idx[i] = ij;
                    c_idx[j] = ii;
                }
            }
        }
    }
    __syncthreads();
}

// ... out of line, for a kernel that takes it by exception: in line its eighteen thousand instructions and what lives across them
// cost the quick selection 0.1 to 0.3 us (a pick of 32 rows, with the greedy one in front, 19.1 -> 19.4); called it saves 60 registers a
// lane to memory (32 rows of equal logits 68.8 -> 70.5 us, 128 rows 70.3 -> 79.7).
__device__ __attribute__((noinline)) void radix_select_called(SampleShared& sh, const uint16_t* row, int nvec, int k) {
    radix_select(sh, row, nvec, k);
}

// Softmax over the first k of c_val / c_idx (in order), top-p prefix, inverse-CDF draw
__device__ __forceinline__ void draw_id(SampleShared& sh, int k, float temp, float top_p, float uniform, int64_t* id) {
    auto& c_val = sh.c_val;
    auto& c_idx = sh.c_idx;
    auto& ws_f = sh.ws_f;
    auto& ws_u = sh.ws_u;
    const int tid = threadIdx.x;
    if (!(temp > 0.f)) {  // uniform: greedy limit
        if (tid == 0) *id = c_idx[0];
        return;
    }
    if (k <= 64) {   // one wave holds the candidates: the same sums without the workgroup's barriers
        if (tid >= 64) return;
        const float smax = c_val[0] / temp;
        float cum = tid < k ? expf(c_val[tid] / temp - smax) : 0.f;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const float u = __shfl_up(cum, o, 64);
            if (tid >= o) cum += u;
        }
        const float cump = cum / __shfl(cum, 63, 64);
        const int m = __popcll(__ballot(tid < k && (cump < top_p || tid == 0)));
        const float target = uniform * __shfl(cump, m - 1, 64);
        const int nb = __popcll(__ballot(tid < m && cump <= target));
        if (tid == 0) *id = c_idx[min(nb, m - 1)];
        return;
    }
    const float smax = c_val[0] / temp;
    const float e = tid < k ? expf(c_val[tid] / temp - smax) : 0.f;
    float total;
    const float cum = block_scan_incl(e, ws_f, total);
    const float cump = cum / total;
    const unsigned valid = (tid < k) && (cump < top_p || tid == 0);
    unsigned m;
    block_scan_incl(valid, ws_u, m);               // the valid set is a prefix: m = its length
    if (tid == (int)m - 1) ws_f[0] = cump;           // mass kept
    __syncthreads();
    const float target = uniform * ws_f[0];
    __syncthreads();
    const unsigned below = (tid < (int)m) && (cump <= target);
    unsigned nb;
    block_scan_incl(below, ws_u, nb);
    if (tid == 0) *id = c_idx[min(nb, m - 1)];
}

// KEEP: chunks of the row a thread holds for the quick selection, 4 for rows of up to 32768 entries, whose threads would
// otherwise request the same chunk again and again (32 rows of 32000, top 50: 13.0 -> 8.7 us with what else changed there).
// QUICK: k up to kSmQuickK; beyond it the selection is all there is, in line (128 rows of 128256, top 1000: 106.5 us called, 96.1).
template <int KEEP, bool QUICK>
__global__ __launch_bounds__(kSmThreads) void sample_kernel(const uint16_t* __restrict__ logits,
                                                          int64_t ld, int n,
                                                          const float* __restrict__ temps,
                                                          const float* __restrict__ top_ps, int top_k,
                                                          const float* __restrict__ uniforms,
                                                          const int64_t* __restrict__ greedy_ids,
                                                          int64_t* __restrict__ ids) {
    // A row whose greedy pick is already known (temperature <= 0 and the caller has the argmax)
    // is done at once: the kernel can then sit in a captured decode step at no cost for greedy
    // batches.
    if (greedy_ids != nullptr && !(temps[blockIdx.x] > 0.f)) {  // uniform
        if (threadIdx.x == 0) ids[blockIdx.x] = greedy_ids[blockIdx.x];
        return;
    }
    __shared__ SampleShared sh;
    auto& sh_u = sh.sh_u;
    const int tid = threadIdx.x;
    const uint16_t* row = logits + (int64_t)blockIdx.x * ld;
    const int nvec = n >> 3;
    int k = min(min(top_k, n), kSmMaxK);
    // (asked for here: each would be a trip to memory behind the selection)
    const float temp = temps[blockIdx.x], top_p = top_ps[blockIdx.x], uniform = uniforms[blockIdx.x];
    // ---- The k largest through the threads' maxima.  The k-th largest of the 1024 maxima bounds the k-th largest entry
    // from below (k different entries reach it), and few others do: of 128256 random logits 52 reach the bound for k =
    // 50, 295 for 256.  Those are listed and ranked by counting.  Only where more than kSmQuickMost entries reach the
    // bound (rows of mostly equal logits), for larger k and for rows with a NaN or of -infinity alone the selection below
    // runs: for k = 512 ranking by counting took longer than it (98 against 90 us).  The maxima take two packed 16-bit instructions an
    // entry pair; the radix selection makes two LDS atomics an entry.  32 rows of 128256, top 50: 80 -> 11.9 us;
    // top 200: 85 -> 17.7; ten entries left of 128256 and the rest masked 57 -> 11.4.  A row that the selection has to take
    // after all reads its entries again (kept over both, they do not fit the registers) and saves registers around it: 32 rows of
    // equal logits, top 50, 70.5 us where the selection alone takes 63.4 (top 257), 128 rows 79.7 and 64.6.  What a call needs besides
    // the row - temperature, top-p, the uniform number - is requested in front: three trips to memory behind the selection were 1.5 us
    // of 15.6.
    auto in_row = [&](int i) { return tid + i * kSmThreads < nvec; };
    bool listed = false;
    if constexpr (QUICK) {
        uint4 keep[KEEP];
        load_row(keep, row, nvec);
        Largest most;
#pragma unroll
        for (int i = 0; i < KEEP; ++i)
            if (in_row(i)) most.add(keep[i]);
        for (int c = KEEP * kSmThreads + tid; c < nvec; c += kSmThreads) most.add(ld16(row + (int64_t)c * 8));
        short top = most.top();
        if (top < 0) {      // nothing of positive sign here: the order of the keys
            top = kKeyLow;
#pragma unroll
            for (int i = 0; i < KEEP; ++i)
                if (in_row(i)) top = top_key(top, keep[i]);
            for (int c = KEEP * kSmThreads + tid; c < nvec; c += kSmThreads) top = top_key(top, ld16(row + (int64_t)c * 8));
        }
        unsigned short* maxima = reinterpret_cast<unsigned short*>(&sh.hist[0][0]);   // offset by 32768: unsigned order
        uint64_t* cand = reinterpret_cast<uint64_t*>(&sh.hist[5][0]);
        unsigned* ranks = &sh.hist[9][0];
        if (tid == 0) sh_u[2] = sh_u[3] = sh_u[4] = 0;
        __syncthreads();
        maxima[tid] = (unsigned short)(top + 32768);
        if (tid < kSmQuickMost) ranks[tid] = 0;
        if (most.nan()) sh_u[3] = 1;
        __syncthreads();
        const unsigned bound = kth_largest<kSmThreads>(maxima, &sh.hist[4][0], k);
        // Entries of -infinity (masked out) have no weight beside any other: a row with fewer than k others has only those.
        const int thr = max((int)bound - 32768, kKeyNegInf + 1);
        if (!sh_u[3]) {   // uniform
            // Counted before anything is listed: a full list costs its rows no more than the count.  A chunk with an entry to
            // list is read again: one body for any chunk, where sixteen over `keep` are twelve KiB of code to fetch (32 rows of
            // 128256, top 50: 14.7 us with those, 11.9 without).
            unsigned hits = 0, mine_n = 0, slot = 0;
            auto count = [&](auto key) {
#pragma unroll
                for (int i = 0; i < KEEP; ++i)
                    if (in_row(i)) {
                        const unsigned c = reaching(key(keep[i]), thr);
                        hits |= c ? 1u << i : 0u;
                        mine_n += c;
                    }
            };
            if (top >= thr) {
                if (thr >= 0) count([](const uint4& v) { return v; });   // (values of positive sign are their keys)
                else count([](const uint4& v) { return to_keys(v); });
                for (int c = KEEP * kSmThreads + tid; c < nvec; c += kSmThreads) mine_n += reaching(to_keys(ld16(row + (int64_t)c * 8)), thr);
                if (mine_n) slot = atomicAdd(&sh_u[2], mine_n);
            }
            __syncthreads();
            const unsigned found = sh_u[2];
            if (found > 0 && found <= (unsigned)kSmQuickMost) {   // uniform
                listed = true;
                k = min(k, (int)found);
                auto list = [&](int c) {
                    const uint4 keys = to_keys(ld16(row + (int64_t)c * 8));
                    list_entries(keys, c, thr, slot, cand, &sh_u[4]);
                };
                if (mine_n) {
                    for (; hits; hits &= hits - 1) list(tid + (__ffs(hits) - 1) * kSmThreads);
                    for (int c = KEEP * kSmThreads + tid; c < nvec; c += kSmThreads) list(c);
                }
                __syncthreads();
                place_candidates(sh, cand, ranks, found, k);
                if (sh_u[4]) order_zeros(sh, k);   // uniform
            }
        }
        if (!listed) __syncthreads();
    }
    if constexpr (!QUICK) radix_select(sh, row, nvec, k);
    else if (!listed) radix_select_called(sh, row, nvec, k);
    draw_id(sh, k, temp, top_p, uniform, ids + blockIdx.x);
}

// The same with a row cut over kSmParts workgroups, for any k.  One workgroup a row is bound by what a compute unit reads and
// by the selection's passes over what it read; here each part only takes its threads' maxima (their 4 x 1024 bound the k-th
// largest entry closer than 1024 do: of 128256 random logits 50 reach it for k = 50, 1160 for 1000), and the workgroup
// that draws the row's last arrival ticket finds the bound and reads again only what lies behind the maxima that reach it.
// More than kSmQuickMost candidates are sorted in LDS.  Workspace: tickets | maxima, tickets as in the greedy pick above.
// For k up to kSmQuickK one workgroup is the faster one: handing the maxima over costs 4 us of its 8 to 18.  Top 1000 of 128256: 1 row
// 92.7 -> 36.9 us, 32 rows 94.7 -> 38.2, 64 rows 94.7 -> 40.7; 32 rows of 16384 36.0 -> 35.0, of 32000 45.2 -> 35.5; but 128 rows of
// 32000, whose parts come in several rounds, took 72 (in one workgroup each 45.8), so up to 64 rows.  Rows that are left to the selection after all come later by what the parts took: 32 rows of equal
// logits 67.8 -> 79.7, with a NaN in each 94.9 -> 98.5.
constexpr int kSmParts = 4;
constexpr int kSmMaxRows = 64;
constexpr int kSmSortMost = 2048;
constexpr int kSmMinVec = 2 * kSmThreads;   // chunks of a row that is worth cutting
constexpr size_t kSmTicketBytes = (size_t)kSmMaxRows * 64 * sizeof(unsigned int);
constexpr size_t kSmWorkspaceBytes = kSmTicketBytes + (size_t)kSmMaxRows * kSmParts * kSmThreads * sizeof(unsigned short);

__global__ __launch_bounds__(kSmThreads) void sample_parts_kernel(const uint16_t* __restrict__ logits, int64_t ld, int n,
                                                                const float* __restrict__ temps,
                                                                const float* __restrict__ top_ps, int top_k,
                                                                const float* __restrict__ uniforms,
                                                                const int64_t* __restrict__ greedy_ids,
                                                                int64_t* __restrict__ ids, unsigned int* tickets,
                                                                unsigned short* row_maxima) {
    constexpr int kGroups = kSmParts * kSmThreads;
    const int rowi = blockIdx.x / kSmParts, part = blockIdx.x % kSmParts, tid = threadIdx.x;
    if (greedy_ids != nullptr && !(temps[rowi] > 0.f)) {  // uniform over the row: nobody takes a ticket
        if (part == 0 && tid == 0) ids[rowi] = greedy_ids[rowi];
        return;
    }
    __shared__ SampleShared sh;
    __shared__ __attribute__((aligned(16))) unsigned short maxima[kGroups];
    __shared__ uint64_t cand[kSmSortMost];
    auto& sh_u = sh.sh_u;
    const uint16_t* row = logits + (int64_t)rowi * ld;
    const int nvec = n >> 3, span = (nvec + kSmParts - 1) / kSmParts;
    int k = min(min(top_k, n), kSmMaxK);
    // thread t of part p: chunks p * span + t, + 1024, .. of the part
    {
        const int c0 = part * span, c1 = min(nvec, c0 + span);
        short top = kKeyLow;
        bool nan = false;
        for (int b = c0 + tid; b < c1; b += 4 * kSmThreads) {
            uint4 v[4];
            Largest most;
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = ld16(row + (int64_t)min(b + i * kSmThreads, c1 - 1) * 8);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (b + i * kSmThreads < c1) most.add(v[i]);
            nan = nan || most.nan();
            if (most.top() >= 0) {
                top = most.top() > top ? most.top() : top;
            } else {      // nothing of positive sign here: the order of the keys
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (b + i * kSmThreads < c1) top = top_key(top, v[i]);
            }
        }
        // a NaN anywhere: the largest maximum there is
        const unsigned mine = nan ? 0xffffu : (unsigned)(top + 32768), next = __shfl_down(mine, 1, 64);
        if (!(tid & 1))
            __hip_atomic_store(reinterpret_cast<unsigned int*>(row_maxima) + ((size_t)rowi * kGroups + part * kSmThreads + tid) / 2,
                               mine | next << 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every storing wave's maxima have left before the ticket
    __syncthreads();
    if (tid == 0) {
        const unsigned old = __hip_atomic_fetch_add(tickets + rowi * 64, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sh_u[5] = old == (unsigned)kSmParts - 1u;
        if (sh_u[5])  // back to zero for the next launch; nobody else touches it in this one
            __hip_atomic_store(tickets + rowi * 64, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sh_u[2] = sh_u[3] = sh_u[4] = sh_u[6] = 0;
    }
    __syncthreads();
    if (!sh_u[5]) return;
    const float temp = temps[rowi], top_p = top_ps[rowi], uniform = uniforms[rowi];
    // the 4096 maxima of all parts, two words a thread
    bool nan = false;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const unsigned m = __hip_atomic_load(reinterpret_cast<unsigned int*>(row_maxima) + (size_t)rowi * kGroups / 2 + i * kSmThreads + tid,
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        reinterpret_cast<unsigned int*>(maxima)[i * kSmThreads + tid] = m;
        nan = nan || (int)(m & 0xffffu) - 32768 > kKeyInf || (int)(m >> 16) - 32768 > kKeyInf;
    }
    if (nan) sh_u[3] = 1;
    __syncthreads();
    bool listed = false;
    if (!sh_u[3]) {   // uniform
        const unsigned bound = kth_largest<kGroups>(maxima, &sh.hist[4][0], k);
        const int thr = max((int)bound - 32768, kKeyNegInf + 1);     // (-infinity has no weight beside any other, as above)
        // the threads whose maxima reach the bound
        unsigned short* groups = reinterpret_cast<unsigned short*>(&sh.hist[0][0]);
#pragma unroll
        for (int i = 0; i < kSmParts; ++i) {
            const int g = i * kSmThreads + tid;
            if ((int)maxima[g] - 32768 >= thr) {
                const unsigned at = atomicAdd(&sh_u[6], 1u);
                if (at < (unsigned)kSmSortMost) groups[at] = (unsigned short)g;
            }
        }
        __syncthreads();
        const int ngroups = sh_u[6];
        if (ngroups <= kSmSortMost) {   // uniform (each brings a candidate: more could not be held)
            for (int it = tid; it < ngroups; it += kSmThreads) {
                const int g = groups[it], c0 = g / kSmThreads * span, c1 = min(nvec, c0 + span);
                for (int b = c0 + g % kSmThreads; b < c1; b += 4 * kSmThreads) {
                    uint4 v[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = ld16(row + (int64_t)min(b + i * kSmThreads, c1 - 1) * 8);
                    unsigned cnt[4], all = 0;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        v[i] = keys_beside(thr, v[i]);
                        cnt[i] = b + i * kSmThreads < c1 ? reaching(v[i], thr) : 0;
                        all += cnt[i];
                    }
                    if (!all) continue;
                    unsigned slot = atomicAdd(&sh_u[2], all);
                    if (slot + all > (unsigned)kSmSortMost) continue;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (cnt[i]) list_entries(v[i], b + i * kSmThreads, thr, slot, cand, &sh_u[4]);
                    }
                }
            }
        }
        __syncthreads();
        const unsigned found = ngroups <= kSmSortMost ? sh_u[2] : 0;
        if (found > 0 && found <= (unsigned)kSmSortMost) {   // uniform
            listed = true;
            k = min(k, (int)found);
            if (found <= (unsigned)kSmQuickMost) {
                unsigned* ranks = &sh.hist[8][0];
                if (tid < kSmQuickMost) ranks[tid] = 0;
                __syncthreads();
                place_candidates(sh, cand, ranks, found, k);
            } else {      // bitonic, descending; a thread orders one pair a step
                unsigned size2 = kSmQuickMost;
                while (size2 < found) size2 <<= 1;
                for (unsigned i = found + tid; i < size2; i += kSmThreads) cand[i] = 0;
                // (a wave's threads hold 128 neighbouring entries: up to a stride of 64 the steps are its own)
                for (unsigned size = 2; size <= size2; size <<= 1)
                    for (unsigned stride = size >> 1; stride > 0; stride >>= 1) {
                        if (stride >= 64 || size == 2) __syncthreads();
                        else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                        const unsigned i = 2 * stride * (tid / stride) + tid % stride, j = i + stride;
                        if (j < size2) {
                            const uint64_t x = cand[i], y = cand[j];
                            if ((x < y) == ((i & size) == 0)) {
                                cand[i] = y;
                                cand[j] = x;
                            }
                        }
                    }
                __syncthreads();
                if (tid < k) {
                    const int key = (int)(cand[tid] >> 32) - 32768;
                    sh.c_val[tid] = bf16_bits_to_f32((unsigned short)(key ^ ((key >> 15) & 0x7fff)));
                    sh.c_idx[tid] = (int)~(unsigned)cand[tid];
                }
                __syncthreads();
            }
            if (sh_u[4]) order_zeros(sh, k);   // uniform
        }
    }
    if (!listed) {
        __syncthreads();
        radix_select(sh, row, nvec, k);
    }
    draw_id(sh, k, temp, top_p, uniform, ids + rowi);
}

}  // namespace mv

extern "C" int mv_sample_topk_topp(const void* logits, int64_t ld, int rows, int n,
                                   const float* temperatures, const float* top_ps, int top_k,
                                   const float* uniforms, int64_t* ids, mv_stream_t stream) {
    return mv_sample_or_greedy(logits, ld, rows, n, temperatures, top_ps, top_k, uniforms, nullptr, ids,
                               stream);
}

extern "C" int mv_sample_or_greedy(const void* logits, int64_t ld, int rows, int n,
                                   const float* temperatures, const float* top_ps, int top_k,
                                   const float* uniforms, const int64_t* greedy_ids, int64_t* ids,
                                   mv_stream_t stream) {
    return mv_sample_or_greedy_ws(logits, ld, rows, n, temperatures, top_ps, top_k, uniforms, greedy_ids, ids, nullptr, 0, stream);
}

extern "C" size_t mv_sample_workspace_bytes(void) { return mv::kSmWorkspaceBytes; }

// the one rule of which picks sample_parts_kernel takes (its comment has both sides)
extern "C" int mv_sample_parts(int rows, int n, int top_k) {
    return rows > 0 && rows <= mv::kSmMaxRows && top_k > mv::kSmQuickK && (n >> 3) >= mv::kSmMinVec;
}

extern "C" int mv_sample_or_greedy_ws(const void* logits, int64_t ld, int rows, int n,
                                      const float* temperatures, const float* top_ps, int top_k,
                                      const float* uniforms, const int64_t* greedy_ids, int64_t* ids,
                                      void* workspace, size_t workspace_bytes, mv_stream_t stream) {
    if (rows == 0 && n > 0) return MV_OK;
    if (!logits || !ids || !temperatures || !top_ps || !uniforms || rows < 0 || n <= 0 || ld < n ||
        top_k <= 0)
        return MV_ERR_INVALID_ARG;
    if (!mv::aligned16(logits) || (ld % 8) != 0) return MV_ERR_INVALID_ARG;
    if ((n % 8) != 0) return MV_ERR_UNSUPPORTED;
    if (workspace && workspace_bytes >= mv::kSmWorkspaceBytes && mv::aligned16(workspace) && mv_sample_parts(rows, n, top_k)) {
        hipLaunchKernelGGL(mv::sample_parts_kernel, dim3(rows * mv::kSmParts), dim3(mv::kSmThreads), 0, (hipStream_t)stream,
                           (const uint16_t*)logits, ld, n, temperatures, top_ps, top_k, uniforms, greedy_ids, ids,
                           (unsigned int*)workspace, (unsigned short*)((char*)workspace + mv::kSmTicketBytes));
        return mv::check_launch();
    }
    const auto kernel = std::min(top_k, n) > mv::kSmQuickK ? mv::sample_kernel<mv::kSmKeep, false>
                        : (n >> 3) <= 4 * mv::kSmThreads   ? mv::sample_kernel<4, true>
                                                           : mv::sample_kernel<mv::kSmKeep, true>;
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(mv::kSmThreads), 0, (hipStream_t)stream,
                       (const uint16_t*)logits, ld, n, temperatures, top_ps, top_k, uniforms, greedy_ids, ids);
    return mv::check_launch();
}

extern "C" size_t mv_argmax_workspace_bytes(void) { return mv::kAmWorkspaceBytes; }

extern "C" int mv_argmax(const void* logits, int64_t ld, int rows, int n, int64_t* ids, void* workspace,
                         size_t workspace_bytes, mv_stream_t stream) {
    if (rows == 0 && n > 0) return MV_OK;
    if (!logits || !ids || rows < 0 || n <= 0 || ld < n) return MV_ERR_INVALID_ARG;
    if (!mv::aligned16(logits) || (ld % 8) != 0) return MV_ERR_INVALID_ARG;
    // long rows: several workgroups per row, about two for every compute unit in all, meeting in the caller's
    // workspace (without one, or with too small a one, every row gets a single workgroup: same result, slower).
    // 32 rows of 128256 in four parts each with one load of a thread in flight: 12.0 us; in sixteen parts with four: 7.3.
    // (64 rows of 8192 take 5.1 us whole, 5.3 in parts.)
    const int nvec = n >> 3;
    if (workspace && workspace_bytes >= mv::kAmWorkspaceBytes && mv::aligned16(workspace) &&
        rows <= mv::kAmMaxRows && nvec >= (rows * 8 <= mv::num_cus() ? 4 : 8) * mv::kAmPartThreads) {
        const mv::AmScratch sc = mv::am_scratch(workspace);
        int parts = 2 * mv::num_cus() / rows;
        if (parts > mv::kAmMaxParts) parts = mv::kAmMaxParts;
        const int most = nvec / mv::kAmPartThreads;  // at least one 16-byte load per thread
        if (parts > most) parts = most;
        if (parts >= 2) {
            const int vec_per_part = (nvec + parts - 1) / parts;
            // as many loads of a thread in flight as its part has: one row of 8192 in single loads 5.0 us, in fours 6.0
            const auto kernel = vec_per_part <= mv::kAmPartThreads ? mv::argmax_parts_kernel<1>
                                : vec_per_part <= 2 * mv::kAmPartThreads ? mv::argmax_parts_kernel<2> : mv::argmax_parts_kernel<4>;
            hipLaunchKernelGGL(kernel, dim3(rows * parts), dim3(mv::kAmPartThreads), 0, (hipStream_t)stream,
                               (const uint16_t*)logits, ld, n, parts, vec_per_part, sc, ids);
            return mv::check_launch();
        }
    }
    hipLaunchKernelGGL(mv::argmax_kernel, dim3(rows), dim3(mv::kAmThreads), 0, (hipStream_t)stream,
                       (const uint16_t*)logits, ld, n, ids);
    return mv::check_launch();
}
