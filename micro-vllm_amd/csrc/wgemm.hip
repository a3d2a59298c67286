// Weight-streaming skinny GEMM for decode:  y[M,N] = x[M,K] @ W[N,K]^T,  1 <= M <= 64.
//
// The op is HBM-bound on W (2*N*K bytes read once; x and y are M/N-th of that), so
// the whole design serves one goal: every CU keeps >= 64 KiB of perfectly coalesced
// weight loads in flight, and every CU gets the same number of bytes.
//
//  * W is stored as wave tiles (mv_shuffle_weight): tile (nt,kt) = 16 output rows x
//    32 k = 1 KiB, lane l owning W[16nt + (l&15)][32kt + 8(l>>4) + 0..7].  One
//    global_load_dwordx4 per wave moves one tile and leaves it already laid out as
//    the A operand of v_mfma_f32_16x16x32_bf16 (rows on lanes&15, k on lanes>>4).
//    The tiles of one 16-row strip are contiguous along K.
//  * A unit of work is (strip nt, k-slice ks).  A 512-thread workgroup takes whole
//    units; its 8 waves interleave over the unit's tiles (wave w takes tile kt0+w,
//    kt0+w+8, ..., or pairs of tiles kt0+2w, kt0+2w+1, kt0+2w+16, ...) so the workgroup
//    reads one contiguous stream.  Partial sums of the 8 waves meet in LDS in a fixed
//    order: results are run-to-run identical.  Which tiles a wave adds up goes with the
//    form, so a row's last bits may change with the number of rows.  (Whole slices of k a
//    wave, for prompts: wgemm_mfma_kernel with KS > 0, four waves where there are four.)
//  * M <= 4: dot-product form (v_dot2c_f32_bf16), x staged once per workgroup in
//    LDS.  M > 4, or x too long for that: v_mfma_f32_16x16x32_bf16 with the x fragment (B operand) loaded
//    from L2, in the same lane layout or by lines of two k-tiles that are exchanged between lanes behind
//    the load.  Both read the same weight tiles.
//  * ksplit > 1 (picked when strips alone cannot balance the CUs) writes fp32
//    slabs; a small second kernel adds them in slab order and applies the epilogue.
//
// Epilogue rounding follows the reference's op boundaries: t = bf16(acc);
// t = bf16(t + bias); t = bf16(t + residual); SWIGLU: out = bf16(silu(gate_t) * up_t).
#include "common.h"

#include <algorithm>

#include <atomic>
#include <type_traits>

namespace mv {

constexpr int kGW = 8;           // waves per workgroup, MFMA form
constexpr int kGT = kGW * kWave;
constexpr int kMaxKsplit = 8;

// Experiment knobs (mv_wgemm_tune).  Atomics: a thread may set one while another is inside a call.
static std::atomic<int> g_tune_bpc{0};      // workgroups per CU the grid is sized for (0 = planner)
static std::atomic<int> g_tune_waves{0};    // waves per workgroup of the dot form: 8 or 16 (0 = planner)
static std::atomic<int> g_tune_sg{0};       // strips per workgroup of the MFMA form: 1, 2 or 4 (0 = planner)
static std::atomic<int> g_tune_ksplit{0};   // 0 = heuristic
static std::atomic<int> g_tune_contig{0};   // dot form: consecutive tiles per wave

enum { kProNone = 0, kProNorm = 1, kProAddNorm = 2 };

struct GemmArgs {
    const uint16_t* x;
    int64_t ldx;
    const uint4* w;
    const uint16_t* bias;
    const uint16_t* residual;
    int64_t ld_res;
    void* y;
    int64_t ldy;
    float* partial;  // [ksplit][M][N] fp32 when ksplit > 1
    int m, n, k;
    int nt, kt;      // strips, k-tiles per strip
    int ksplit, ktps;  // k-slices, k-tiles per slice
    int contig;        // dot form: a wave's tiles are consecutive (1) or interleaved with the other waves' (0)
    int nunits;
    int flags;
    // fused input transform (dot form only): x <- rmsnorm(x [+ add_r]) * ln_w
    int prologue;
    int var_from_rounded;       // kProAddNorm: variance from bf16(x + add_r) instead of the fp32 sum
    const uint16_t* add_r;
    int64_t ld_add_r;
    const uint16_t* ln_w;
    float eps;
    uint16_t* sum_out;          // kProAddNorm: bf16(x + add_r), written by workgroup 0
    int64_t ld_sum_out;
    // output transform of the slab reduction: normed = rmsnorm(y) * post_ln_w next to y itself
    const uint16_t* post_ln_w;
    uint16_t* post_out;
    int64_t ld_post;
    float post_eps;
    int post_var_from_rounded;  // variance from y as stored (bf16) instead of the unrounded t + residual
    GemmAct act;
#ifdef MV_WGEMM_STAMP
    int stamp_slot;             // which of the 32 stamp records this launch writes
#endif
};

#ifdef MV_WGEMM_STAMP
// Phase stamps (build variant for tools/stamp_wgemm.py): the constant 100 MHz counter at up to
// eight points of every workgroup of the last 32 launches, written by the workgroup's first thread.
static __device__ unsigned long long g_wstamp[32 * 256 * 8];
static int g_stamp_counter = 0;
#define MV_WSTAMP(slot)                                                                          \
    do {                                                                                         \
        __builtin_amdgcn_sched_barrier(0);                                                       \
        if (threadIdx.x == 0 && blockIdx.x < 256)                                                \
            g_wstamp[((a.stamp_slot & 31) * 256 + blockIdx.x) * 8 + (slot)] =                    \
                __builtin_amdgcn_s_memrealtime();                                                \
        __builtin_amdgcn_sched_barrier(0);                                                       \
    } while (0)
#else
#define MV_WSTAMP(slot) do {} while (0)
#endif

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;

// Final value of one output element from its fp32 accumulator.  ACT: an activation of the unrounded sum (GemmAct).  Kernels of their
// own: with the choice made at run time the plain ones carried 1.1 KiB of code more (28672 x 4096 at 32 rows 40.6 -> 41.2 us).
template <bool ACT = false>
__device__ __forceinline__ float epilogue_value(const GemmArgs& a, float acc, int m, int n) {
    if (ACT && a.act.kind == 1) {   // uniform
        const float v = fmaxf(acc, 0.f);
        return v * v;
    }
    float t = round_bf16(acc);
    if (a.bias) t = round_bf16(t + bf16_bits_to_f32(a.bias[n]));
    if (a.residual) t = round_bf16(t + bf16_bits_to_f32(a.residual[(int64_t)m * a.ld_res + n]));
    return t;
}

// ... and of a pair of rows, up and gate
template <bool ACT = false>
__device__ __forceinline__ float epilogue_gated(const GemmArgs& a, float gate, float up) {
    return ACT ? gated_act_f(gate, up, 2, a.act.limit, a.act.slope) : silu_mul_rounded(gate, up);
}

// ------------------------------------------------------------ M <= 4: dot form
struct UnitCtx {
    int nt, ks, kt0, ntile, nchunk, last, wfirst;
    const uint4* wbase;
};

// GW waves per workgroup, each keeping two stages of U weight tiles in flight; PRO = the
// input transform (kProNone / kProNorm / kProAddNorm).
template <int M, int GW, int U, int PRO, bool ACT = false>
__global__ __launch_bounds__(GW * kWave) void wgemm_dot_kernel(GemmArgs a) {
    constexpr int GT = GW * kWave;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // layout: x rows [M][K] bf16 | 16 zero bytes | red [GW][M][16] fp32
    uint16_t* xs = reinterpret_cast<uint16_t*>(smem);
    const int zero_off = M * a.k * 2;
    float* red = reinterpret_cast<float*>(smem + zero_off + 16);

    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    MV_WSTAMP(0);

    const int tstride = a.contig ? 1 : GW;   // tiles between two consecutive tiles of a wave
    const int wstride = tstride * 64;        // the same in 16-byte units
    auto setup = [&](int u) {
        UnitCtx c;
        c.nt = u / a.ksplit;
        c.ks = u - c.nt * a.ksplit;
        c.kt0 = c.ks * a.ktps;
        const int kt1 = min(a.kt, c.kt0 + a.ktps);
        if (a.contig) {  // wave w owns tiles [w * tpw, (w + 1) * tpw) of the slice
            const int tpw = (kt1 - c.kt0 + GW - 1) / GW;
            c.wfirst = wid * tpw;
            c.ntile = min(tpw, kt1 - c.kt0 - c.wfirst);
        } else {         // wave w owns tiles w, w + GW, w + 2 GW, ...
            c.wfirst = wid;
            c.ntile = (kt1 - c.kt0 - wid + GW - 1) / GW;  // tiles of this wave (may be <= 0)
        }
        c.nchunk = (c.ntile + U - 1) / U;
        c.last = max(c.ntile - 1, 0);
        // a wave without tiles still issues (clamped) loads: point it at the slice's first tile
        c.wbase = a.w + ((int64_t)c.nt * a.kt + c.kt0 + (c.ntile > 0 ? c.wfirst : 0)) * 64 + lane;
        return c;
    };
    auto load = [&](uint4(&buf)[U], const UnitCtx& c, int chunk) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int t = min(chunk * U + i, c.last);  // clamp: always a valid address (chunk < 2^24)
            buf[i] = ld16_nt(c.wbase + (int64_t)t * wstride);
        }
    };
    auto compute = [&](const uint4(&buf)[U], const UnitCtx& c, int chunk, float(&acc)[M]) {
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int t = chunk * U + i;
            // byte offset of this lane's 8 x values; out-of-range tiles read zeros
            const int xoff = (t < c.ntile) ? ((c.kt0 + c.wfirst + t * tstride) * 32 + q * 8) * 2 : -1;
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int off = (xoff < 0) ? zero_off : m * a.k * 2 + xoff;
                const uint4 xv = *reinterpret_cast<const uint4*>(smem + off);
                acc[m] = dot2_bf16(buf[i].x, xv.x, acc[m]);
                acc[m] = dot2_bf16(buf[i].y, xv.y, acc[m]);
                acc[m] = dot2_bf16(buf[i].z, xv.z, acc[m]);
                acc[m] = dot2_bf16(buf[i].w, xv.w, acc[m]);
            }
        }
    };

    // Memory requests of a wave return in issue order, and two stages of weight tiles per wave
    // are a couple of microseconds of HBM traffic: x (and the norm weight) are therefore
    // requested FIRST, into registers, the weight stream is started behind them, and only
    // then is x consumed.  Requested after the tiles, x would arrive behind them and the
    // stream would stall until the input transform is through.
    // Units go to workgroups by fixed stride.  Handing them out by ticket instead (an atomic
    // counter, drawn one unit ahead so that its round trip is hidden) was measured on MI355X to be
    // slower although workgroups on the odd XCDs finish a gate/up launch about 12 % later than
    // those on the even ones: 37.3 -> 41.1 us for N = 28672, 153 -> 166 us for N = 128256.
    int u = blockIdx.x;
    UnitCtx cur = setup(u);
    uint4 bufA[U], bufB[U];
    const int kvec = a.k >> 3;

    constexpr int kPT = 256;                              // threads of the input transform
    constexpr int XC = 2;                                 // early chunks per thread, plain staging
    constexpr int PC = (M == 1) ? 4 : (M == 2 ? 2 : 1);   // early chunks per thread and row, norm
    // Straight-line code with clamped addresses (no branches around the loads), so the compiler
    // can wait for exactly the x loads and leave the tile loads in flight.
    uint4 xe[XC];
    uint4 pxe[M][PC], pre[M][PC], pwe[PC];
    if (PRO == kProNone) {
#pragma unroll
        for (int j = 0; j < XC; ++j) {
            const int c = min((int)threadIdx.x + j * GT, M * kvec - 1);
            const int m = c / kvec, cv = c - m * kvec;
            xe[j] = ld16(a.x + (int64_t)m * a.ldx + cv * 8);
        }
    } else {
#pragma unroll
        for (int j = 0; j < PC; ++j) {
            if (j * kPT < kvec) {  // uniform
                const int c = min((int)(threadIdx.x & (kPT - 1)) + j * kPT, kvec - 1);
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    pxe[m][j] = ld16(a.x + (int64_t)m * a.ldx + c * 8);
                    if (PRO == kProAddNorm)
                        pre[m][j] = ld16(a.add_r + (int64_t)m * a.ld_add_r + c * 8);
                }
                pwe[j] = ld16(a.ln_w + c * 8);
            }
        }
    }
    // Keep the issue order x, A0..A3 (B0..B3 follow the transform): the loop below waits by
    // counting requests, and a first pass issued in any other order would make every later
    // wait conservative.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const int t = min(i, cur.last);  // indices past the end are clamped to the wave's last tile
        const uint4 v = ld16_nt(cur.wbase + (int64_t)t * wstride);
        bufA[i] = v;
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" ::: "memory");

    // ---- stage x into LDS, optionally as rmsnorm(x [+ add_r]) * ln_w ------------------
    if (PRO == kProNone) {
#pragma unroll
        for (int j = 0; j < XC; ++j) {
            const int c = threadIdx.x + j * GT;
            if (c < M * kvec) {
                const int m = c / kvec, cv = c - m * kvec;
                st16(xs + m * a.k + cv * 8, xe[j]);
            }
        }
        for (int c = threadIdx.x + XC * GT; c < M * kvec; c += GT) {
            const int m = c / kvec, cv = c - m * kvec;
            st16(xs + m * a.k + cv * 8, ld16(a.x + (int64_t)m * a.ldx + cv * 8));
        }
        if (threadIdx.x == 0) *reinterpret_cast<uint4*>(smem + zero_off) = make_uint4(0, 0, 0, 0);
    } else {
        // Same chunk assignment (256 threads, stride 256) and the same reduction order as the
        // stand-alone norm kernels, so fused and unfused paths agree bit for bit.
        float ss[M];
#pragma unroll
        for (int m = 0; m < M; ++m) ss[m] = 0.f;
        // one chunk of one row: (sum,) squares, LDS image, copy of the sum for the next block
        auto absorb = [&](int m, int c, const uint4& xv, const uint4& rv) {
            const uint32_t x4[4] = {xv.x, xv.y, xv.z, xv.w};
            if (PRO == kProAddNorm) {
                const uint32_t r4[4] = {rv.x, rv.y, rv.z, rv.w};
                uint32_t o[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float s0 = bf16_lo(x4[j]) + bf16_lo(r4[j]);
                    float s1 = bf16_hi(x4[j]) + bf16_hi(r4[j]);
                    o[j] = pack_bf16x2(s0, s1);
                    if (a.var_from_rounded) {
                        s0 = bf16_lo(o[j]);
                        s1 = bf16_hi(o[j]);
                    }
                    ss[m] += s0 * s0;
                    ss[m] += s1 * s1;
                }
                const uint4 ov = make_uint4(o[0], o[1], o[2], o[3]);
                st16(xs + m * a.k + c * 8, ov);
                if (blockIdx.x == 0) st16(a.sum_out + (int64_t)m * a.ld_sum_out + c * 8, ov);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float v0 = bf16_lo(x4[j]), v1 = bf16_hi(x4[j]);
                    ss[m] += v0 * v0;
                    ss[m] += v1 * v1;
                }
                st16(xs + m * a.k + c * 8, xv);
            }
        };
        if (threadIdx.x < kPT) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
#pragma unroll
                for (int j = 0; j < PC; ++j) {
                    const int c = threadIdx.x + j * kPT;
                    if (c < kvec) absorb(m, c, pxe[m][j], pre[m][j]);
                }
                for (int c = threadIdx.x + PC * kPT; c < kvec; c += kPT) {
                    const uint4 xv = ld16(a.x + (int64_t)m * a.ldx + c * 8);
                    uint4 rv = xv;
                    if (PRO == kProAddNorm) rv = ld16(a.add_r + (int64_t)m * a.ld_add_r + c * 8);
                    absorb(m, c, xv, rv);
                }
            }
        }
        if (threadIdx.x == 0) *reinterpret_cast<uint4*>(smem + zero_off) = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float v = wave_sum(ss[m]);
            if (lane == 0 && wid < kPT / 64) red[m * (kPT / 64) + wid] = v;
        }
        __syncthreads();
        float rrms[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float t = 0.f;
#pragma unroll
            for (int i = 0; i < kPT / 64; ++i) t += red[m * (kPT / 64) + i];
            rrms[m] = 1.0f / sqrtf(t / (float)a.k + a.eps);
        }
        auto scale = [&](int m, int c, const uint4& wv) {
            uint4* px = reinterpret_cast<uint4*>(xs + m * a.k + c * 8);
            const uint4 sv = *px;
            const uint32_t s4[4] = {sv.x, sv.y, sv.z, sv.w}, w4[4] = {wv.x, wv.y, wv.z, wv.w};
            uint32_t o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                o[j] = pack_bf16x2((bf16_lo(s4[j]) * rrms[m]) * bf16_lo(w4[j]),
                                   (bf16_hi(s4[j]) * rrms[m]) * bf16_hi(w4[j]));
            *px = make_uint4(o[0], o[1], o[2], o[3]);
        };
        if (threadIdx.x < kPT) {
#pragma unroll
            for (int j = 0; j < PC; ++j) {
                const int c = threadIdx.x + j * kPT;
                if (c < kvec) {
#pragma unroll
                    for (int m = 0; m < M; ++m) scale(m, c, pwe[j]);
                }
            }
            for (int c = threadIdx.x + PC * kPT; c < kvec; c += kPT) {
                const uint4 wv = ld16(a.ln_w + c * 8);
#pragma unroll
                for (int m = 0; m < M; ++m) scale(m, c, wv);
            }
        }
    }
    __syncthreads();
    MV_WSTAMP(1);

    // Stage B goes out only now.  Requesting both stages before the input transform measured
    // slower on MI355X for every decode projection (O: 8.0 vs 7.3 us).
#pragma unroll
    for (int i = U; i < 2 * U; ++i) {
        const int t = min(i, cur.last);
        bufB[i - U] = ld16_nt(cur.wbase + (int64_t)t * wstride);
        __builtin_amdgcn_sched_barrier(0);
    }
    // Chunks 0 and 1 of the current unit are in flight in bufA / bufB here and at the top of
    // every pass.  The stream is strictly A, B, A, B, ... with no branch around a load (a chunk
    // index past the end re-reads the wave's last tile, a cache hit; its product is masked to
    // zero), so every wait in the loop is for exactly one stage and the other stays in flight.
    constexpr int kPast = 1 << 24;
    for (;;) {
        const int un = u + gridDim.x;
        const bool more = un < a.nunits;
        UnitCtx nxt = cur;
        if (more) nxt = setup(un);

        float acc[M];
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = 0.f;

        const int npair = (cur.nchunk + 1) >> 1;
#ifdef MV_WGEMM_STAMP
        if (u == (int)blockIdx.x && npair > 1) {
            compute(bufA, cur, 0, acc);   // timing only: first stage landed (results are wrong)
            MV_WSTAMP(2);
        }
#endif
        for (int p = 0; p < npair - 1; ++p) {
            compute(bufA, cur, 2 * p, acc);
            load(bufA, cur, 2 * p + 2);
            compute(bufB, cur, 2 * p + 1, acc);
            load(bufB, cur, 2 * p + 3);
        }
        const int cl = npair > 0 ? 2 * (npair - 1) : kPast;  // nothing to add if the wave has no tiles
        if (more) {  // two copies so that each path keeps exact request counts
            compute(bufA, cur, cl, acc);
            load(bufA, nxt, 0);
            compute(bufB, cur, cl + 1, acc);
            load(bufB, nxt, 1);
        } else {
            compute(bufA, cur, cl, acc);
            compute(bufB, cur, cl + 1, acc);
        }
        if (!more) MV_WSTAMP(3);

        // lanes r, r+16, r+32, r+48 hold the four k-quarters of row r
#pragma unroll
        for (int m = 0; m < M; ++m) {
            acc[m] += __shfl_xor(acc[m], 16, 64);
            acc[m] += __shfl_xor(acc[m], 32, 64);
        }
        if (lane < 16) {
#pragma unroll
            for (int m = 0; m < M; ++m) red[(wid * M + m) * 16 + r] = acc[m];
        }
        __syncthreads();
        if (threadIdx.x < 16 * M) {
            const int m = threadIdx.x >> 4, rr = threadIdx.x & 15;
            float s = 0.f;
#pragma unroll
            for (int w8 = 0; w8 < GW; ++w8) s += red[(w8 * M + m) * 16 + rr];
            const int n = cur.nt * 16 + rr;
            if (a.partial) {
                a.partial[((int64_t)cur.ks * a.m + m) * a.n + n] = s;
            } else if (a.flags & MV_GEMM_OUT_F32) {
                reinterpret_cast<float*>(a.y)[(int64_t)m * a.ldy + n] = s;
            } else if (a.flags & MV_GEMM_SWIGLU) {
                if (rr < 8) {
                    float g = 0.f;
#pragma unroll
                    for (int w8 = 0; w8 < GW; ++w8) g += red[(w8 * M + m) * 16 + rr + 8];
                    reinterpret_cast<uint16_t*>(a.y)[(int64_t)m * a.ldy + cur.nt * 8 + rr] =
                        (uint16_t)f32_to_bf16_bits(epilogue_gated<ACT>(a, g, s));
                }
            } else {
                reinterpret_cast<uint16_t*>(a.y)[(int64_t)m * a.ldy + n] =
                    (uint16_t)f32_to_bf16_bits(epilogue_value<ACT>(a, s, m, n));
            }
        }
        if (!more) break;
        __syncthreads();
        u = un;
        cur = nxt;
    }
    MV_WSTAMP(4);
}

// ------------------------------------------------------------ M > 4: MFMA form
// HB = number of 8-row blocks of x (M <= 8*HB), MB of 16-row blocks; SG = strips a workgroup multiplies together.
// A wave loads the x fragments of a k-tile once and uses them against the SG weight tiles of
// that k-tile: x comes out of L2 for every workgroup, so without the sharing the x requests
// (MB per weight tile) outnumber the weight requests and the L2 path, not HBM, sets the pace.
//
// What a request of x costs is the compute unit's address path: neighbouring lanes in different lines are taken one after the
// other.  Sixteen rows of 64 bytes with a row to each lane - the operand's own layout - are 37 bytes a ns and unit, two lanes to
// a line 73, a weight tile's 1 KiB in one piece 120.  So a request is eight rows of two k-tiles, lane (r, q) taking 16 bytes q of
// row r / 2 and k-tile r % 2 (the odd 8-row block: k-tile 1 - r % 2), and the operands are made of two of them: the first k-tile's
// is the first block's even lanes and the second's odd ones, the second k-tile's the other lanes, exchanged with their neighbours
// (three vector instructions a register pair).  Column r of the product is then row r / 2 + 8 (r % 2) of its 16.  us, before ->
// after:
//   decoding (KS = 0)  64 rows 28672 x 4096 58.2 -> 50.8, 14336 wide down 28.0 -> 24.8, 2560 x 2048 8.2 -> 6.7; 24 rows 7168 x 8192 26.7 ->
//                      23.1; 16384 x 2048 at 8 rows 16.5 -> 13.5, at 32 17.6 -> 14.8
//   k in slices        37 rows 2560 x 2048 8.6 -> 6.9, 2048 x 2048 8.3 -> 6.8, 4096 x 4096 15.4 -> 11.6; 16 rows 4096 x 14336 28.7 -> 22.8
//
// KS = 0: the waves interleave over the unit's pairs of k-tiles.  KS = 4, 8, 16: k in KS whole slices, each added up by one wave
// and the slices in order - the sums of a prefill projection cut into KS slices (gemm_prefill.hip), bit for bit, without
// its slabs and their reduction launch.  Here every request is a scalar address and a 32-bit offset, three offsets for x and one for the
// weights: with a pair of registers for each the groups of four strips spilled from 49 rows on (<8, 4, 8> 20 registers, <7, 4, 8> 6,
// <8, 2, 16> 2; none so), 64 rows 16384 x 14336 102 -> 86 us, 12304 x 4096 30.9 -> 26.8, 56 rows 14336 x 14336 83 -> 77.  With four slices a workgroup has four waves, each with four stages in flight (a wave a
// SIMD has the registers; two halves of eight waves on strips of their own read x twice: 37 rows 11264 x 2048 14.0 us, 12.2 so, 8192 x
// 1024 7.7 -> 7.0, 4096 x 1024 6.9 -> 5.3); with sixteen a wave takes two slices one after the other.  Three or four stages elsewhere cost
// 0 to 35 %: a wave has few stages, and those past the end are asked for as well.
__device__ __forceinline__ int mfma_row(int b, int r) { return b * 16 + (r >> 1) + 8 * (r & 1); }

template <int HB, int SG, int KS = 0, bool ACT = false, bool PAIR = true>
__global__ __launch_bounds__(KS == 4 ? 4 * kWave : kGT) void wgemm_mfma_kernel(GemmArgs a) {
    constexpr int kWaves = KS == 4 ? 4 : kGW;
    constexpr int ST = KS == 4 ? 4 : 2;                      // stages in flight
    constexpr int MB = (HB + 1) / 2;
    constexpr int U = PAIR || SG + MB <= 6 ? 2 : 1;          // k-tiles per stage
    constexpr int kNext = PAIR ? 1 : kGW;                    // k-tiles between two of a stage
    constexpr int kStep = KS ? U : U * kGW;                  // ... and between a wave's stages
    static_assert(PAIR || KS == 0, "slices go by pairs");
    constexpr int kTurns = KS == 16 ? 2 : 1;
    constexpr int kSlots = KS == 0 ? kGW : KS;   // accumulator sets that meet in LDS
    // cross-wave reduction buffer [kSlots][SG][MB][64 lanes][4]: 4 KiB per (strip, row block) pair with four slices, 8, or 16 with
    // sixteen, up to 128 KiB (dynamic: past the 64 KiB a static array may have)
    extern __shared__ __attribute__((aligned(16))) float red[];

    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const bool odd = r & 1;
    // this lane's x rows, clamped into [0, M), at its 16 bytes of the first of two k-tiles; and which of the two it takes
    const uint16_t* xrow[HB];
    const int second = odd ? 32 : 0;
#pragma unroll
    for (int h = 0; h < HB; ++h) xrow[h] = a.x + (int64_t)min(PAIR ? h * 8 + (r >> 1) : h * 8 + r, a.m - 1) * a.ldx + q * 8;
    // KS > 0: bytes behind the scalar address of a block's first row - of the blocks that are whole, even and odd, and of the last
    const uint32_t row_bytes = 2 * (uint32_t)a.ldx, mine = 2 * (q * 8 + second), other = 2 * (q * 8 + 32 - second);
    const uint32_t x_even = (r >> 1) * row_bytes + mine, x_odd = (r >> 1) * row_bytes + other;
    const uint32_t x_last = min(r >> 1, a.m - 1 - (HB - 1) * 8) * row_bytes + (HB & 1 ? mine : other);

    for (int u = blockIdx.x; u < a.nunits; u += gridDim.x) {
        const int g = KS ? u : u / a.ksplit, ks = KS ? 0 : u - g * a.ksplit;
#pragma unroll
        for (int turn = 0; turn < kTurns; ++turn) {
        const int slice = wid + turn * kGW;   // (KS > 0)
        const int slot = KS == 16 ? slice : wid;
        const int strip0 = g * SG;
        const int kt0 = KS ? slice * a.ktps : ks * a.ktps;
        const int kt1 = min(a.kt, kt0 + a.ktps);
        // this wave's stages, and the first k-tile; a wave without tiles still loads (clamped)
        const int ntile = PAIR ? (kt1 - kt0 + 1) >> 1 : kt1 - kt0;   // (PAIR: of two)
        const int mine = KS ? ntile : (ntile - wid + kGW - 1) / kGW;
        const int nchunk = PAIR ? mine : (mine + U - 1) / U;
        const int last = max(nchunk - 1, 0);
        const int ktw = KS ? kt0 : kt0 + (mine > 0 ? (PAIR ? 2 : 1) * wid : 0);
        const uint4* wbase[SG];
#pragma unroll
        for (int sI = 0; sI < SG; ++sI)
            wbase[sI] = a.w + ((int64_t)min(strip0 + sI, a.nt - 1) * a.kt) * 64;   // uniform, in scalar registers

        f32x4_t acc[SG][MB];
#pragma unroll
        for (int sI = 0; sI < SG; ++sI)
#pragma unroll
            for (int b = 0; b < MB; ++b) acc[sI][b] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

        constexpr int XR = PAIR ? HB : U * MB;   // requests of x in a stage
        uint4 wr[ST][U][SG], xr[ST][XR];
        auto load = [&](uint4(&wb)[U][SG], uint4(&xb)[XR], int c) {
            const int t = ktw + min(c, last) * kStep;
            const bool whole = t + kNext < kt1;   // uniform: half a stage at the end is asked for twice
            if constexpr (PAIR) {
                if constexpr (KS > 0) {
                    const uint32_t even_back = whole ? 0 : 2 * second, odd_back = whole ? 0 : 2 * (32 - second);
                    const uint32_t e = x_even - even_back, o = x_odd - odd_back, l = x_last - (HB & 1 ? even_back : odd_back);
#pragma unroll
                    for (int h = 0; h < HB; ++h)
                        xb[h] = ld16(reinterpret_cast<const char*>(a.x + h * 8 * a.ldx + t * 32) + (h == HB - 1 ? l : h & 1 ? o : e));
                } else {
                    const int even_block = t * 32 + (whole ? second : 0), odd_block = t * 32 + (whole ? 32 - second : 0);
#pragma unroll
                    for (int h = 0; h < HB; ++h) xb[h] = ld16(xrow[h] + (h & 1 ? odd_block : even_block));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const int ti = whole ? t + i * kNext : t;
                uint32_t lane_bytes = lane * 16u;
                asm("" : "+v"(lane_bytes));   // (the address stays a scalar one and an offset: summed outside the loop it is SG pairs of registers)
#pragma unroll
                for (int sI = 0; sI < SG; ++sI) wb[i][sI] = ld16_nt(reinterpret_cast<const char*>(wbase[sI] + (int64_t)ti * 64) + lane_bytes);
                if constexpr (!PAIR) {
#pragma unroll
                    for (int b = 0; b < MB; ++b) xb[i * MB + b] = ld16(xrow[2 * b] + ti * 32);
                }
            }
        };
        auto compute = [&](const uint4(&wb)[U][SG], const uint4(&xb)[XR], int c, bool all) {
            if (!all && c >= nchunk) return;   // wave-uniform
            auto swap = [](uint32_t v) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, true); };   // lanes 1 0 3 2
            auto one = [&](uint32_t e, uint32_t o) { return odd ? o : e; };
            auto operand = [&](int i, int b) {
                if constexpr (!PAIR) return __builtin_bit_cast(bf16x8_t, xb[i * MB + b]);
                const uint4 e = xb[2 * b], o = xb[2 * b + 1 < HB ? 2 * b + 1 : 2 * b];
                const uint4 v = i == 0 ? make_uint4(one(e.x, o.x), one(e.y, o.y), one(e.z, o.z), one(e.w, o.w))
                                       : make_uint4(swap(one(o.x, e.x)), swap(one(o.y, e.y)), swap(one(o.z, e.z)), swap(one(o.w, e.w)));
                return __builtin_bit_cast(bf16x8_t, v);
            };
            auto multiply = [&](int i, int b, bf16x8_t xf) {
#pragma unroll
                for (int sI = 0; sI < SG; ++sI)
                    acc[sI][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wb[i][sI]), xf, acc[sI][b], 0, 0, 0);
            };
            const bool whole = U == 2 && (all || ktw + c * kStep + kNext < kt1);   // wave-uniform (only the last stage may be half of one)
            if constexpr (SG * MB >= 8) {   // (a row block at a time: the operands of all of them do not fit)
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    __builtin_amdgcn_sched_barrier(0);
                    multiply(0, b, operand(0, b));
                    if (whole) multiply(U - 1, b, operand(U - 1, b));
                }
            } else {
                bf16x8_t f[U][MB];
#pragma unroll
                for (int b = 0; b < MB; ++b)
#pragma unroll
                    for (int i = 0; i < U; ++i) f[i][b] = operand(i, b);
#pragma unroll
                for (int b = 0; b < MB; ++b) multiply(0, b, f[0][b]);
                if (whole) {
#pragma unroll
                    for (int b = 0; b < MB; ++b) multiply(U - 1, b, f[U - 1][b]);
                }
            }
        };

        // The first stages go out unconditionally (indices past the end are clamped) and the steady
        // state has no branch around a request, so the compiler's wait counts are exact: with a
        // request under an `if` anywhere before or inside the loop every wait covers all stages
        // and only one is ever in flight.  The last 2 ST - 1 chunks at most are handled after it.
        // (The fences keep the first stages in the order the loop issues them: interleaved by
        // the scheduler they would make the loop's first wait, and through the back edge all of
        // them, cover them all.)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < ST; ++i) {
            load(wr[i], xr[i], i);
            __builtin_amdgcn_sched_barrier(0);
        }
        int c = 0;
        for (; c + 2 * ST <= nchunk; c += ST) {
#pragma unroll
            for (int i = 0; i < ST; ++i) {
                compute(wr[i], xr[i], c + i, true);
                __builtin_amdgcn_sched_barrier(0);
                load(wr[i], xr[i], c + i + ST);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int i = 0; i < ST; ++i) {
            compute(wr[i], xr[i], c + i, false);
            if (i < ST - 1 && c + i + ST < nchunk) load(wr[i], xr[i], c + i + ST);
        }
#pragma unroll
        for (int i = 0; i < ST - 1; ++i) compute(wr[i], xr[i], c + i + ST, false);

        // acc[s][b][j] = C[n = 16 (g SG + s) + 4q + j][m = 16 b + r, PAIR: mfma_row(b, r)]
#pragma unroll
        for (int sI = 0; sI < SG; ++sI)
#pragma unroll
            for (int b = 0; b < MB; ++b)
                *reinterpret_cast<f32x4_t*>(&red[(((slot * SG + sI) * MB + b) * 64 + lane) * 4]) = acc[sI][b];
        }
        __syncthreads();
        // one wave per (strip, row block) pair; more pairs than waves take a second turn
        for (int sb = wid; sb < MB * SG; sb += kWaves) {
            const int l = lane;
            const int sI = sb / MB, b = sb - sI * MB;
            const int rr = l & 15, qq = l >> 4;
            const int m = PAIR ? mfma_row(b, rr) : b * 16 + rr;
            const int nt = g * SG + sI;
            auto sum_at = [&](int ll) {
                f32x4_t s = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int w8 = 0; w8 < kSlots; ++w8)
                    s += *reinterpret_cast<const f32x4_t*>(
                        &red[(((w8 * SG + sI) * MB + b) * 64 + ll) * 4]);
                return s;
            };
            if (m < a.m && nt < a.nt) {
                const f32x4_t s = sum_at(l);
                const int n0 = nt * 16 + qq * 4;
                if (a.partial) {
                    *reinterpret_cast<f32x4_t*>(&a.partial[((int64_t)ks * a.m + m) * a.n + n0]) = s;
                } else if (a.flags & MV_GEMM_OUT_F32) {
                    *reinterpret_cast<f32x4_t*>(
                        &reinterpret_cast<float*>(a.y)[(int64_t)m * a.ldy + n0]) = s;
                } else if (a.flags & MV_GEMM_SWIGLU) {
                    if (qq < 2) {  // rows 0..7 = up; their gates sit 8 rows (32 lanes) further
                        const f32x4_t gt = sum_at(l + 32);
                        uint2 o;
                        o.x = pack_bf16x2(epilogue_gated<ACT>(a, gt[0], s[0]), epilogue_gated<ACT>(a, gt[1], s[1]));
                        o.y = pack_bf16x2(epilogue_gated<ACT>(a, gt[2], s[2]), epilogue_gated<ACT>(a, gt[3], s[3]));
                        *reinterpret_cast<uint2*>(&reinterpret_cast<uint16_t*>(
                            a.y)[(int64_t)m * a.ldy + nt * 8 + qq * 4]) = o;
                    }
                } else {
                    uint2 o;
                    o.x = pack_bf16x2(epilogue_value<ACT>(a, s[0], m, n0), epilogue_value<ACT>(a, s[1], m, n0 + 1));
                    o.y = pack_bf16x2(epilogue_value<ACT>(a, s[2], m, n0 + 2), epilogue_value<ACT>(a, s[3], m, n0 + 3));
                    *reinterpret_cast<uint2*>(
                        &reinterpret_cast<uint16_t*>(a.y)[(int64_t)m * a.ldy + n0]) = o;
                }
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------ slab reduction
// Eight consecutive outputs of a row per thread, for bf16 outputs with bias / residual epilogues on
// 16-byte-aligned rows: the slabs of many-token products are tens of megabytes (the down projection
// at 2048 tokens in two k-slices: 67 MB of slabs, 17 of residual in, 17 out), and one element per
// thread read them at 2.3 TB/s (43 us).  Same sums in the same order, same rounding points.
__global__ __launch_bounds__(256) void wgemm_finalize_vec8_kernel(GemmArgs a) {
    const int nvec = a.n >> 3;
    const int64_t total = (int64_t)a.m * nvec;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int m = (int)(i / nvec), n0 = (int)(i - (int64_t)m * nvec) * 8;
        f32x4_t lo[kMaxKsplit], hi[kMaxKsplit];
#pragma unroll
        for (int ks = 0; ks < kMaxKsplit; ++ks) {
            if (ks >= a.ksplit) break;   // uniform
            const float* p = a.partial + ((int64_t)ks * a.m + m) * a.n + n0;
            lo[ks] = *reinterpret_cast<const f32x4_t*>(p);
            hi[ks] = *reinterpret_cast<const f32x4_t*>(p + 4);
        }
        const uint4 bv = a.bias ? ld16(a.bias + n0) : make_uint4(0, 0, 0, 0);
        const uint4 rv = a.residual ? ld16(a.residual + (int64_t)m * a.ld_res + n0) : make_uint4(0, 0, 0, 0);
        f32x4_t slo = (f32x4_t){0.f, 0.f, 0.f, 0.f}, shi = slo;
#pragma unroll
        for (int ks = 0; ks < kMaxKsplit; ++ks)
            if (ks < a.ksplit) {
                slo += lo[ks];
                shi += hi[ks];
            }
        const float acc[8] = {slo[0], slo[1], slo[2], slo[3], shi[0], shi[1], shi[2], shi[3]};
        const uint32_t b4[4] = {bv.x, bv.y, bv.z, bv.w}, r4[4] = {rv.x, rv.y, rv.z, rv.w};
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float t0 = round_bf16(acc[2 * e]), t1 = round_bf16(acc[2 * e + 1]);
            if (a.bias) {
                t0 = round_bf16(t0 + bf16_lo(b4[e]));
                t1 = round_bf16(t1 + bf16_hi(b4[e]));
            }
            if (a.residual) {
                t0 = round_bf16(t0 + bf16_lo(r4[e]));
                t1 = round_bf16(t1 + bf16_hi(r4[e]));
            }
            o[e] = pack_bf16x2(t0, t1);
        }
        st16(reinterpret_cast<uint16_t*>(a.y) + (int64_t)m * a.ldy + n0, make_uint4(o[0], o[1], o[2], o[3]));
    }
}

// One thread per output element (per up/gate pair for SWIGLU); slabs added in order.
template <bool ACT>
__global__ __launch_bounds__(256) void wgemm_finalize_kernel(GemmArgs a) {
    const bool sw = (a.flags & MV_GEMM_SWIGLU) != 0;
    const int ncols = sw ? a.n / 2 : a.n;
    const int64_t total = (int64_t)a.m * ncols;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * 256) {
        const int m = (int)(i / ncols), c = (int)(i - (int64_t)m * ncols);
        // all slabs of the element requested before the first is added (they are added in order)
        auto slab_sum = [&](int n) {
            float v[kMaxKsplit];
#pragma unroll
            for (int ks = 0; ks < kMaxKsplit; ++ks) {
                if (ks >= a.ksplit) break;   // uniform
                v[ks] = a.partial[((int64_t)ks * a.m + m) * a.n + n];
            }
            float s = 0.f;
#pragma unroll
            for (int ks = 0; ks < kMaxKsplit; ++ks)
                if (ks < a.ksplit) s += v[ks];
            for (int ks = kMaxKsplit; ks < a.ksplit; ++ks) s += a.partial[((int64_t)ks * a.m + m) * a.n + n];
            return s;
        };
        if (sw) {
            const int nu = (c >> 3) * 16 + (c & 7);
            const float up = slab_sum(nu), gate = slab_sum(nu + 8);
            reinterpret_cast<uint16_t*>(a.y)[(int64_t)m * a.ldy + c] =
                (uint16_t)f32_to_bf16_bits(epilogue_gated<ACT>(a, gate, up));
        } else if (a.flags & MV_GEMM_OUT_F32) {
            reinterpret_cast<float*>(a.y)[(int64_t)m * a.ldy + c] = slab_sum(c);
        } else {
            reinterpret_cast<uint16_t*>(a.y)[(int64_t)m * a.ldy + c] =
                (uint16_t)f32_to_bf16_bits(epilogue_value<ACT>(a, slab_sum(c), m, c));
        }
    }
}

// Slab reduction + output epilogue + RMSNorm of the result, one workgroup per row:
//   t = bf16(sum of slabs); t = bf16(t + bias); s = t + residual (fp32); y = bf16(s);
//   normed = bf16((float(y) * rrms) * ln_w),  rrms = 1 / sqrt(mean(s^2) + eps)
// with the mean over the unrounded s (what add+RMSNorm after a projection computes) or, with
// post_var_from_rounded, over y as stored (what RMSNorm of a stored hidden state computes).
// Chunk assignment and summation order are those of the stand-alone norm kernels (256 threads,
// stride 256, block_sum), so the fused and the separate path agree bit for bit.
constexpr int kPostChunks = 4;  // 16-byte chunks of y a thread keeps: rows up to 8192 wide
// NT = 256 holds up to four chunks a thread; NT = 512 and 1024, for a few rows, one: a row's slabs then come in through more
// requests at a time, and the first 256 threads add the squares out of LDS in the order of NT = 256, so the norm is the same
// bit for bit.  8 rows of 8192 6.5 -> 4.9 us, 32 rows of 4096 5.2 -> 4.8; more rows than compute units keep 256.
template <int NT>
__global__ __launch_bounds__(NT) void wgemm_finalize_norm_kernel(GemmArgs a) {
    constexpr int CH = NT == 256 ? kPostChunks : 1;
    __shared__ float red[NT / 64];
    __shared__ __attribute__((aligned(16))) float sq[NT == 256 ? 4 : NT * 8];
    const int m = blockIdx.x;
    const int nvec = a.n >> 3;
    uint4 keep[CH];
    float ss = 0.f;
    // Every operand of every chunk is requested before the first is used - the first kPostAhead slabs
    // included (the usual splits are 2 and 4): the slabs were written by another kernel, so each
    // dependent round of loads is a trip to memory, and this kernel is nothing but such trips.
    // (Chunk rows and slabs that do not exist are skipped: both conditions are uniform.)
    constexpr int kPostAhead = 4;
    f32x4_t p_lo[CH][kPostAhead], p_hi[CH][kPostAhead];
    uint4 b_in[CH], r_in[CH], w_in[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        if (j * NT >= nvec) break;
        const int n0 = min(threadIdx.x + j * NT, nvec - 1) * 8;
#pragma unroll
        for (int ks = 0; ks < kPostAhead; ++ks) {
            if (ks >= a.ksplit) break;
            const float* p = a.partial + ((int64_t)ks * a.m + m) * a.n + n0;
            p_lo[j][ks] = *reinterpret_cast<const f32x4_t*>(p);
            p_hi[j][ks] = *reinterpret_cast<const f32x4_t*>(p + 4);
        }
        b_in[j] = a.bias ? ld16(a.bias + n0) : make_uint4(0, 0, 0, 0);
        r_in[j] = a.residual ? ld16(a.residual + (int64_t)m * a.ld_res + n0) : make_uint4(0, 0, 0, 0);
        w_in[j] = ld16(a.post_ln_w + n0);
    }
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const int c = threadIdx.x + j * NT;
        if (c < nvec) {
            const int n0 = c * 8;
            f32x4_t lo = (f32x4_t){0.f, 0.f, 0.f, 0.f}, hi = lo;
#pragma unroll
            for (int ks = 0; ks < kPostAhead; ++ks) {
                if (ks < a.ksplit) {   // slabs are added in order, whichever way they were fetched
                    lo += p_lo[j][ks];
                    hi += p_hi[j][ks];
                }
            }
            for (int ks = kPostAhead; ks < a.ksplit; ++ks) {
                const float* p = a.partial + ((int64_t)ks * a.m + m) * a.n + n0;
                lo += *reinterpret_cast<const f32x4_t*>(p);
                hi += *reinterpret_cast<const f32x4_t*>(p + 4);
            }
            const float acc[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            const uint4 bv = b_in[j], rv = r_in[j];
            const uint32_t b4[4] = {bv.x, bv.y, bv.z, bv.w}, r4[4] = {rv.x, rv.y, rv.z, rv.w};
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float t0 = round_bf16(acc[2 * e]), t1 = round_bf16(acc[2 * e + 1]);
                if (a.bias) {
                    t0 = round_bf16(t0 + bf16_lo(b4[e]));
                    t1 = round_bf16(t1 + bf16_hi(b4[e]));
                }
                float s0 = t0, s1 = t1;
                if (a.residual) {
                    s0 = t0 + bf16_lo(r4[e]);
                    s1 = t1 + bf16_hi(r4[e]);
                }
                o[e] = pack_bf16x2(s0, s1);
                if (a.post_var_from_rounded) {
                    s0 = bf16_lo(o[e]);
                    s1 = bf16_hi(o[e]);
                }
                if (NT == 256) {
                    ss += s0 * s0;
                    ss += s1 * s1;
                } else {
                    *reinterpret_cast<float2*>(&sq[c * 8 + 2 * e]) = make_float2(s0 * s0, s1 * s1);
                }
            }
            keep[j] = make_uint4(o[0], o[1], o[2], o[3]);
            st16(reinterpret_cast<uint16_t*>(a.y) + (int64_t)m * a.ldy + n0, keep[j]);
        }
    }
    if (NT > 256) {
        __syncthreads();
        if (threadIdx.x < 256)
            for (int c = threadIdx.x; c < nvec; c += 256) {
                const float4 x = *reinterpret_cast<const float4*>(&sq[c * 8]), y = *reinterpret_cast<const float4*>(&sq[c * 8 + 4]);
                ss += x.x;
                ss += x.y;
                ss += x.z;
                ss += x.w;
                ss += y.x;
                ss += y.y;
                ss += y.z;
                ss += y.w;
            }
    }
    const float total = block_sum(ss, red);     // (waves past the fourth add zero)
    const float rrms = 1.0f / sqrtf(total / (float)a.n + a.post_eps);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        const int c = threadIdx.x + j * NT;
        if (c < nvec) {
            const uint4 wv = w_in[j];
            const uint32_t s4[4] = {keep[j].x, keep[j].y, keep[j].z, keep[j].w};
            const uint32_t w4[4] = {wv.x, wv.y, wv.z, wv.w};
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                o[e] = pack_bf16x2((bf16_lo(s4[e]) * rrms) * bf16_lo(w4[e]),
                                   (bf16_hi(s4[e]) * rrms) * bf16_hi(w4[e]));
            st16(a.post_out + (int64_t)m * a.ld_post + c * 8, make_uint4(o[0], o[1], o[2], o[3]));
        }
    }
}

static int launch_finalize_norm(const GemmArgs& a, hipStream_t s) {
    const int nvec = a.n / 8;
    if (nvec > 512 && a.m <= num_cus()) hipLaunchKernelGGL(wgemm_finalize_norm_kernel<1024>, dim3(a.m), dim3(1024), 0, s, a);
    else if (nvec > 256 && a.m <= num_cus()) hipLaunchKernelGGL(wgemm_finalize_norm_kernel<512>, dim3(a.m), dim3(512), 0, s, a);
    else hipLaunchKernelGGL(wgemm_finalize_norm_kernel<256>, dim3(a.m), dim3(256), 0, s, a);
    return check_launch();
}

// The slab reduction for other kernels of the library that split k (the prefill GEMM): same
// layout partial[ks][m][n], same epilogues.
int launch_wgemm_finalize(float* partial, int ksplit, int m, int n, int flags, const uint16_t* bias,
                          const uint16_t* residual, int64_t ld_res, void* y, int64_t ldy, hipStream_t s, GemmAct act) {
    GemmArgs a = {};
    a.act = act;
    a.partial = partial;
    a.ksplit = ksplit;
    a.m = m;
    a.n = n;
    a.flags = flags;
    a.bias = bias;
    a.residual = residual;
    a.ld_res = ld_res;
    a.y = y;
    a.ldy = ldy;
    const int ncols = (flags & MV_GEMM_SWIGLU) ? n / 2 : n;
    const int most = num_cus() * 8;
    const bool vec8 = !act.kind && !(flags & (MV_GEMM_SWIGLU | MV_GEMM_OUT_F32)) && ksplit <= kMaxKsplit && (n % 8) == 0 &&
                      (ldy % 8) == 0 && aligned16(y) && aligned16(partial) && (!bias || aligned16(bias)) &&
                      (!residual || (aligned16(residual) && (ld_res % 8) == 0)) && (int64_t)m * n >= (1 << 16);
    if (vec8) {
        int64_t blocks = ((int64_t)m * (n / 8) + 255) / 256;
        if (blocks > most) blocks = most;
        hipLaunchKernelGGL(wgemm_finalize_vec8_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a);
        return check_launch();
    }
    const int64_t total = (int64_t)m * ncols;
    int64_t blocks = (total + 255) / 256;
    if (blocks > most) blocks = most;
    hipLaunchKernelGGL(a.act.kind ? wgemm_finalize_kernel<true> : wgemm_finalize_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, s, a);
    return check_launch();
}

// ------------------------------------------------------------ host planning
// Which form takes m rows: up to four the dot form while their x lies in LDS beside what its waves meet in (four rows up to
// k = 20128, three up to 26944, two up to 40544), the matrix form otherwise: it streams x.
static size_t dot_form_lds(int m, int k, int waves) { return (size_t)m * k * 2 + 16 + (size_t)waves * m * 16 * 4; }
static bool dot_form_fits(int m, int k, int waves) { return dot_form_lds(m, k, waves) + 512 <= 160 * 1024; }
static bool dot_form_takes(int m, int k) { return m <= 4 && dot_form_fits(m, k, 8); }

// k-slices per strip: balance whole units over the CUs.  Cost in tiles per CU,
// with a split paying roughly one extra kernel boundary.
static int mfma_strip_group(int m, int nt, int kt, bool free_reduce);

// k-slices for `units` whole-k work items: split while fewer than half the CUs would have one and
// every wave keeps at least 4 tiles
static int ksplit_for_units(int units, int kt) {
    const int cus = num_cus();
    int best = 1;
    for (int ks = 2; ks <= kMaxKsplit; ks *= 2) {
        if (kt % ks) break;
        if (kt / ks < 4 * kGW) break;             // keep >= 4 tiles per wave
        if ((long)units * best * 2 > cus) break;  // already at least half the CUs busy
        best = ks;
    }
    return best;
}

// `nt` = work items along N: strips for the dot form, strip groups for the MFMA form.
// `free_reduce`: the slabs are added by a launch that runs anyway (the caller's next kernel for
// MV_GEMM_SLABS, the norm kernel of mv_wgemm_postnorm), so a k-split costs no launch of its own.
static int pick_ksplit(int m, int nt, int kt, bool free_reduce = false) {
    const bool dot = dot_form_takes(m, kt * 32);
    if (!dot) {
        const int sg = mfma_strip_group(m, nt, kt, free_reduce);
        nt = (nt + sg - 1) / sg;
    }
    if (const int forced = g_tune_ksplit; forced > 0) {
        int ks = forced;
        while (ks > 1 && (kt % ks) != 0) --ks;
        return ks;
    }
    // Measured on MI355X (tools/bench_wgemm.py, M=1): whole strips beat every k-split for all
    // four decode projections (QKV 11.8 vs 14.8 us, O 8.0 vs 11.4, gate/up 38.8 vs 48.5, down
    // 20.8 vs 23.7): the second launch that adds the slabs costs more than the imbalance of
    // 1.5 strips per CU.  Splitting only pays when there are far fewer strips than CUs.
    // ... and for the dot form not even then: shards of tensor-parallel runs (tools/sweep_small_gemv.py,
    // M=1) run 5.4 us unsplit against 6.5-8.7 us split at 48 strips (N=768, K=4096), 5.8 against
    // 7.2-10.0 at 96 strips.
    if (dot && nt >= 32) return 1;
    return ksplit_for_units(nt, kt);
}

// Waves per workgroup of the dot form for a projection of `nunits` units of `kt` k-tiles each (the
// rule above wgemm_impl's launch explains the numbers).  qkv_attn.hip runs the QKV projection in
// the same shape, so that its sums are formed in the same order.
static int dot_form_waves_for_units(int nunits, int kt) {
    const int cus = num_cus();
    const bool one_long_strip_per_cu = nunits <= cus && nunits * 8 >= cus * 7 && kt >= 128;
    const int forced = g_tune_waves;
    return forced ? forced : (one_long_strip_per_cu ? 16 : 8);
}
int dot_form_ksplit(int m, int nt, int kt) { return g_tune_contig ? 0 : pick_ksplit(m, nt, kt); }
int dot_form_waves(int m, int nt, int kt) { return dot_form_waves_for_units(nt * pick_ksplit(m, nt, kt), kt); }

template <int M, int GW, int U, int PRO, bool ACT>
static int launch_dot_stage(const GemmArgs& a, int grid, hipStream_t s) {
    const size_t lds = dot_form_lds(M, a.k, GW);
    if (lds > 160 * 1024) return MV_ERR_UNSUPPORTED;
    static LdsOptIn opted;  // per instantiation
    if (int rc = ensure_dynamic_lds((const void*)wgemm_dot_kernel<M, GW, U, PRO, ACT>,
                                    lds > 64 * 1024 ? 160 * 1024 : lds, opted))
        return rc;
#ifdef MV_WGEMM_STAMP
    GemmArgs as = a;
    as.stamp_slot = g_stamp_counter++;
    hipLaunchKernelGGL((wgemm_dot_kernel<M, GW, U, PRO, ACT>), dim3(grid), dim3(GW * kWave), lds, s, as);
    return check_launch();
#endif
    hipLaunchKernelGGL((wgemm_dot_kernel<M, GW, U, PRO, ACT>), dim3(grid), dim3(GW * kWave), lds, s, a);
    return check_launch();
}

// Tiles per stage: four for one and two rows, two for three and four (register budget: 128 VGPRs at 16 waves per CU).  Where a wave
// has no more than four tiles of a strip (k <= 1024 on eight waves) two as well: a stage of four would hold them all, and the second
// one ask for its last tile four times over (one row, us, four -> two a stage: 32000 x 1024 15.2 -> 11.5, 9472 x 1024 6.9 -> 5.3, 1024 x
// 1024 3.5 -> 3.3, 8192 x 512 5.0 -> 4.3; two rows 32000 x 1024 15.0 -> 11.5, 1024 x 1024 4.0 -> 3.4, with a norm in front 15.5 -> 12.5, 4.6 -> 4.2;
// slices of a longer k, 256 x 4096 5.5 -> 5.3; no slower over 22 shapes of plain, gated and normed forms).  The sums are the same bits.
template <int M, int GW, int PRO, bool ACT = false>
static int launch_dot(const GemmArgs& a, int grid, hipStream_t s) {
    if constexpr (M <= 2 && GW == 8) {
        if (std::min(a.kt, a.ktps) <= 4 * GW) return launch_dot_stage<M, GW, 2, PRO, ACT>(a, grid, s);
    }
    return launch_dot_stage<M, GW, M <= 2 ? 4 : 2, PRO, ACT>(a, grid, s);
}

template <int M, int GW>
static int launch_dot_pro(const GemmArgs& a, int grid, hipStream_t s) {
    switch (a.prologue) {
        case kProNone: return a.act.kind ? launch_dot<M, GW, kProNone, true>(a, grid, s) : launch_dot<M, GW, kProNone>(a, grid, s);
        case kProNorm: return launch_dot<M, GW, kProNorm>(a, grid, s);
        default: return launch_dot<M, GW, kProAddNorm>(a, grid, s);
    }
}

template <int M>
static int launch_dot_waves(const GemmArgs& a, int waves, int grid, hipStream_t s) {
    return waves == 16 ? launch_dot_pro<M, 16>(a, grid, s) : launch_dot_pro<M, 8>(a, grid, s);
}

template <int HB, int SG, bool ACT, bool PAIR>
static int launch_mfma_act(const GemmArgs& a, int grid, hipStream_t s) {
    constexpr size_t lds = (size_t)kGW * SG * ((HB + 1) / 2) * 64 * 4 * sizeof(float);
    static_assert(lds <= 128 * 1024, "reduction buffer fits LDS");
    static LdsOptIn opted;  // per instantiation
    if (int rc = ensure_dynamic_lds((const void*)wgemm_mfma_kernel<HB, SG, 0, ACT, PAIR>, lds, opted)) return rc;
    hipLaunchKernelGGL((wgemm_mfma_kernel<HB, SG, 0, ACT, PAIR>), dim3(grid), dim3(kGT), lds, s, a);
    return check_launch();
}

// Pairs of k-tiles, or a k-tile a request (PAIR = false).  By pairs the waves read their weights two tiles at a time, which a long
// stream takes 3 to 7 % slower (128256 x 8192 at 8 rows 317 -> 339 us, 128256 x 4096 169 -> 175: the eight waves' 1 KiB pieces no longer
// lie side by side), so it is for where x is what costs.  A k-tile a request instead:
//   groups of seven strips (32 rows, 28672 x 1024 13.3 us, 13.9 by pairs, 28672 x 2048 21.9, 22.7, 28672 x 4096 47.5, 49.5);
//   one 8-row block, whose operand repeats its rows, in groups narrower than four;
//   up to 16 rows of k past 2048 in groups;
//   groups of four strips, 128 KB of each, up to 48 rows: their requests by pairs meet on memory channels (24 rows 16384 x 4096 25.0, 28.8 by
//   pairs, 128256 x 4096 175, 190, 8192 x 8192 in two slices 24.6, 28.9; 48 rows 32000 x 4096 52.9, 55.7; of 64, 96 or 160 KB pairs are
//   ahead: 8192 x 4096 in two slices 20.2, 14.1, 32000 x 5120 55, 51).
template <int HB>
static int launch_mfma(const GemmArgs& a, int sg, int grid, hipStream_t s) {
    auto strips = [&](auto count) {
        constexpr int SG = decltype(count)::value;
        constexpr bool kNever = SG == 7 || (HB == 1 && SG < 4);
        constexpr bool kLong = HB <= 2 && SG > 1, kMeet = SG == 4 && HB > 2 && HB <= 6;
        if constexpr (kNever || kLong || kMeet) {
            constexpr int rows = (HB + 1) / 2 * 2;
            if (kNever || (kLong && a.k > 2048) || (kMeet && a.ktps == 128))
                return a.act.kind ? launch_mfma_act<rows, SG, true, false>(a, grid, s) : launch_mfma_act<rows, SG, false, false>(a, grid, s);
        }
        if constexpr (!kNever)
            return a.act.kind ? launch_mfma_act<HB, SG, true, true>(a, grid, s) : launch_mfma_act<HB, SG, false, true>(a, grid, s);
    };
    if constexpr (HB <= 4) {
        if (sg == 7) return strips(std::integral_constant<int, 7>());
    }
    return sg == 4   ? strips(std::integral_constant<int, 4>())
           : sg == 3 ? strips(std::integral_constant<int, 3>())
           : sg == 2 ? strips(std::integral_constant<int, 2>())
                     : strips(std::integral_constant<int, 1>());
}
// `launch` with the 8-row blocks of `m` rows
template <class F>
static int with_row_blocks(int m, F launch) {
    switch ((m + 7) / 8) {
        case 1: return launch(std::integral_constant<int, 1>());
        case 2: return launch(std::integral_constant<int, 2>());
        case 3: return launch(std::integral_constant<int, 3>());
        case 4: return launch(std::integral_constant<int, 4>());
        case 5: return launch(std::integral_constant<int, 5>());
        case 6: return launch(std::integral_constant<int, 6>());
        case 7: return launch(std::integral_constant<int, 7>());
        default: return launch(std::integral_constant<int, 8>());
    }
}

// strips per workgroup of the MFMA form: the cross-wave reduction buffer is 8 KiB per
// (strip, row block) pair, 128 KiB for four strips of four row blocks
static int mfma_strip_group(int m, int nt, int kt, bool free_reduce) {
    const int mb = (m + 15) / 16;
    const int most = 4;
    if (const int forced = g_tune_sg; (forced >= 1 && forced <= 4) || (forced == 7 && mb <= 2)) return forced;
    // Seven strips per workgroup where that deals the strips out to the CUs exactly (Llama-3-8B
    // gate/up: 1792 strips = 7 x 256): in groups of four 448 units fall on 256 CUs as two rounds, the
    // second three quarters full, and every workgroup re-reads x for four strips instead of seven.
    if (mb <= 2 && nt % 7 == 0 && (nt / 7) % num_cus() == 0) return 7;
    // A small model of the three costs, fitted to the Llama-3-8B
    // projections at 8, 16 and 32 rows (tools/bench_mfma_gemv.py, tools/bench_slabs.py): weights
    // stream at 6.45 MB/us over the CUs that have a unit, every unit re-reads its k-slice of x out of
    // L2 at about 12.9 MB/us, and a k-split pays a slab-reduction launch of 3.6 us (QKV at 32 rows:
    // groups of three in two k-slices, one unit per CU, 11.8 + 3.0 us against 16.2 for pairs without
    // a split, which leave a quarter of the CUs idle).  (Down projection, 14336 wide: single
    // strips win at 8 rows, 21.6 against 22.8 us, and lose at 16, 27.3 against 22.9, because x is
    // then as many bytes as the weights; the 4096-wide O projection keeps single strips at both,
    // 9.1 against 11.2 us, its split costing more than its x.)
    // With a free slab reduction the same model decides with that term dropped.
    // At 33-64 rows it picks the widest group wherever that fills the chip, because x is then most of what moves, and
    // narrower ones for small projections (37 rows, 2560 x 2048 10.4 -> 8.4 us, 2048 x 2048 9.8 -> 8.0, 11264 x 2048 in
    // threes 14.6 -> 13.5, 6144 x 4096 18.7 -> 16.1; 28672 x 4096 stays with fours, 54).
    const int cus = num_cus();
    int best = 1;
    double best_us = 1e30;
    for (int sg = most; sg >= 1; --sg) {
        const int groups = (nt + sg - 1) / sg;
        const int ks = ksplit_for_units(groups, kt);
        const long units = (long)groups * ks;
        const double fill = (double)units / (double)(((units + cus - 1) / cus) * cus);
        const double w_mb = (double)nt * kt * 1024e-6, x_mb = (double)units * m * (kt / ks) * 64e-6;
        const double us = w_mb / (6.45 * fill) + x_mb / 12.9 + (ks > 1 && !free_reduce ? 3.6 : 0.0);
        if (us < best_us) {
            best_us = us;
            best = sg;
        }
    }
    return best;
}

// Strips of a workgroup of the ordered form: the model above, x out of L2 at 17 MB/us, in 8-row blocks (requests of two k-tiles; the
// groups that measured fastest at 31 of 33 shapes, 29 at 12.9).  Groups of three where those deal the strips out (two -> four -> three):
// 64 rows 8208 x 4096 29.2 -> 25.7 -> 20.2 us, 37 rows 11264 x 4096 27.0 -> 23.1 -> 19.8, but 12304 x 4096 27.4 -> 24.2 -> 29.4.
int wgemm_ordered_group(int m, int nt, int kt, int ks) {
    const int mb = (m + 15) / 16, rows = (m + 7) / 8 * 8;
    const int cus = num_cus();
    int best = 1;
    double best_us = 1e30;
    for (int sg = 4; sg >= 1; --sg) {
        if (ks == 16 && sg > 2) continue;   // 128 KiB of LDS
        const long units = (nt + sg - 1) / sg;
        const double fill = (double)units / (double)(((units + cus - 1) / cus) * cus);
        const double us = (double)nt * kt * 1024e-6 / (6.45 * fill) + (double)units * rows * kt * 64e-6 / 17.0;
        if (us < best_us) {
            best_us = us;
            best = sg;
        }
    }
    return best;
}

template <int HB, int SG, int KS>
static int launch_ordered(const GemmArgs& a, int grid, hipStream_t s) {
    constexpr size_t lds = (size_t)KS * SG * ((HB + 1) / 2) * 64 * 4 * sizeof(float);
    static_assert(lds <= 128 * 1024, "reduction buffer fits LDS");
    static LdsOptIn opted;  // per instantiation
    if (int rc = ensure_dynamic_lds((const void*)wgemm_mfma_kernel<HB, SG, KS>, lds, opted)) return rc;
    hipLaunchKernelGGL((wgemm_mfma_kernel<HB, SG, KS>), dim3(grid), dim3(KS == 4 ? 4 * kWave : kGT), lds, s, a);
    return check_launch();
}
template <int HB>
static int launch_ordered_rows(const GemmArgs& a, int sg, int ks, int grid, hipStream_t s) {
    switch (ks * 8 + sg) {
        case 4 * 8 + 1: return launch_ordered<HB, 1, 4>(a, grid, s);
        case 4 * 8 + 2: return launch_ordered<HB, 2, 4>(a, grid, s);
        case 4 * 8 + 3: return launch_ordered<HB, 3, 4>(a, grid, s);
        case 4 * 8 + 4: return launch_ordered<HB, 4, 4>(a, grid, s);
        case 8 * 8 + 1: return launch_ordered<HB, 1, 8>(a, grid, s);
        case 8 * 8 + 2: return launch_ordered<HB, 2, 8>(a, grid, s);
        case 8 * 8 + 3: return launch_ordered<HB, 3, 8>(a, grid, s);
        case 8 * 8 + 4: return launch_ordered<HB, 4, 8>(a, grid, s);
        case 16 * 8 + 1: return launch_ordered<HB, 1, 16>(a, grid, s);
        case 16 * 8 + 2: return launch_ordered<HB, 2, 16>(a, grid, s);
        default: return MV_ERR_UNSUPPORTED;
    }
}

// Up to a limit on rows x k-tiles: a workgroup reads all of x for the strips it has, whatever their number, where the sliced tiles
// read a piece and pay for slabs and their reduction.  Sixty a strip and no fewer than 4096 (n x k, us, sliced
// tiles and their reduction -> here): 37 rows 2048 x 2048 8.8 -> 6.9, 11264 x 2048 17.3 -> 12.2, 6144 x 4096 18.3 -> 14.4, 7168 x 8192 35.2 ->
// 26.3, 8192 x 3584 19.8 -> 13.7, 4096 x 3584 12.8 -> 10.4; 64 rows 2048 x 2048 9.7 -> 8.3, 8192 x 1024 13.6 -> 8.2, 8208 x 4096 30 -> 20,
// 14336 x 14336 91 -> 83, 6144 x 11264 (22528) 42.1 -> 43.3, 5120 x 14336 (28672, out) 46 -> 52; 256 strips of 448 k-tiles 32 rows 31.2 ->
// 29.4, 40 rows (17920) 32.0 -> 32.9.
// Tiles narrow enough to give every unit a slice are ahead sooner.  One strip a wave and a long k: eight rows, and of those 512 x 14336
// (3584) 12.3 -> 12.8, 768 x 11264 (2816) 11.7 -> 11.8.  Two: 65536 over the slices - in sixteen 1536 x 5120 at 24 rows (3840) 12.3 ->
// 11.3, 2048 x 8192 at 16 (4096) 13.9 -> 13.0, but 2048 x 5120 at 24 10.9 -> 11.5, at 40 (6400) 11.1 -> 14.5, 2048 x 6144 at 24 (4608) 11.2 ->
// 12.2, 1536 x 11264 at 16 (5632) 15.2 -> 16.6; in eight 4096 x 4096 at 64 (8192) 14.4 -> 13.9, 4096 x 5120 at 64 (10240) 16.0 -> 18.2.
bool wgemm_ordered_takes(int m, int nt, int kt, int ks, int strips) {
    if ((ks != 4 && ks != 8 && ks != 16) || m > 64) return false;
    const int rows = (m + 7) / 8 * 8;
    if (strips == 1 && kt > 128) return rows * kt <= 3072 && rows <= 8;
    if (strips == 2) return rows * kt <= 65536 / ks;
    return (int64_t)rows * kt <= std::max(60 * nt, 4096);
}

// x [m, k] . W^T with the sums of `ks` slices of k added in order, epilogue as mv_gemm_prefill_ws, or the norm's.
// Arguments as the callers have checked them.
int launch_wgemm_ordered(const void* x, int64_t ldx, const void* w_tiles, const void* bias, const void* residual,
                         int64_t ld_res, void* y, int64_t ldy, int m, int n, int k, int ks, int flags, PostNorm* norm,
                         hipStream_t s) {
    if (norm && ((flags & (MV_GEMM_SWIGLU | MV_GEMM_OUT_F32)) || !wgemm_finalize_norm_takes(n))) norm = nullptr;
    GemmArgs a = {};
    a.x = (const uint16_t*)x;
    a.ldx = ldx;
    a.w = (const uint4*)w_tiles;
    a.bias = (const uint16_t*)bias;
    a.residual = (const uint16_t*)residual;
    a.ld_res = ld_res;
    a.y = y;
    a.ldy = ldy;
    a.m = m;
    a.n = n;
    a.k = k;
    a.nt = n / 16;
    a.kt = k / 32;
    a.flags = flags;
    a.ksplit = 1;
    a.ktps = a.kt / ks;
    a.partial = norm ? norm->slab : nullptr;
    const int sg = wgemm_ordered_group(m, a.nt, a.kt, ks);
    a.nunits = (a.nt + sg - 1) / sg;
    const int mb = (m + 15) / 16;
    // more workgroups a CU where their registers allow it (four waves of four slices) or their reduction buffers do
    const int per_cu = ks == 4 ? 4 : ks * sg * mb <= 64 ? 2 : 1;
    const int grid = a.nunits < num_cus() * per_cu ? a.nunits : num_cus() * per_cu;
    const int rc = with_row_blocks(m, [&](auto hb) { return launch_ordered_rows<decltype(hb)::value>(a, sg, ks, grid, s); });
    if (rc != MV_OK || !norm) return rc;
    return launch_wgemm_finalize_norm(norm->slab, 1, m, n, bias, norm, s);
}

bool wgemm_finalize_norm_takes(int n) { return n % 8 == 0 && n <= 8 * 256 * kPostChunks; }

// Rows and the norm's weight 16-byte aligned (the callers' checks)
int launch_wgemm_finalize_norm(float* partial, int ksplit, int m, int n, const void* bias, PostNorm* norm, hipStream_t s) {
    GemmArgs a = {};
    a.partial = partial;
    a.ksplit = ksplit;
    a.m = m;
    a.n = n;
    a.bias = (const uint16_t*)bias;
    a.residual = (const uint16_t*)norm->residual;
    a.ld_res = norm->ld;
    a.y = norm->y;
    a.ldy = norm->ld;
    a.post_ln_w = (const uint16_t*)norm->ln_w;
    a.post_out = (uint16_t*)norm->out;
    a.ld_post = norm->ld;
    a.post_eps = norm->eps;
    a.post_var_from_rounded = norm->var_from_rounded;
    norm->done = true;
    return launch_finalize_norm(a, s);
}

// k-slices of a projection whose next kernel adds them.  Past four rows as everywhere; up to four (the dot form) two, where the
// strips are few and long: half the compute units or fewer have one, and they would walk it longer than the chip takes for
// the whole.  One row, us whole -> two slices: 1024 x 5120 6.2 -> 5.0, 1024 x 4096 5.0 -> 4.1, 512 x 4096 4.8 -> 3.8, 2048 x 8192
// 9.0 -> 7.6; but 2048 x 4096 5.8 -> 6.3, 2048 x 2048 4.1 -> 4.3, 1024 x 1024 3.5 -> 3.5.  Four slices: 1024 x 5120 5.3, 2048 x
// 8192 7.0 and of two rows 8.1 where two take 7.7.
int wgemm_slices(int m, int n, int k) {
    const int nt = n / 16, kt = k / 32;
    if (!dot_form_takes(m, k) || g_tune_ksplit) return pick_ksplit(m, nt, kt, true);
    return nt <= num_cus() / 2 && kt >= 128 && kt >= 2 * nt ? 2 : 1;
}

static int wgemm_impl(const void* x, int64_t ldx, const void* add_r, int64_t ld_add_r,
                      const void* ln_w, float eps, void* sum_out, int64_t ld_sum_out, int prologue,
                      int var_from_rounded, const void* w_tiles, const void* bias,
                      const void* residual, int64_t ld_res, void* y, int64_t ldy, int m, int n,
                      int k, void* workspace, size_t workspace_bytes, int flags,
                      mv_stream_t stream, const void* post_ln_w = nullptr, float post_eps = 0.f,
                      void* post_out = nullptr, int64_t ld_post = 0, int post_var_from_rounded = 0,
                      int slices = 0, GemmAct act = {0, 0.f, 0.f}) {
    const bool slabs_only = (flags & MV_GEMM_SLABS) != 0;
    if (!x || !w_tiles || (!y && !slabs_only) || m <= 0 || n <= 0 || k <= 0) return MV_ERR_INVALID_ARG;
    if (m > 64 || (n % 16) != 0 || (k % 32) != 0) return MV_ERR_UNSUPPORTED;
    if (!aligned16(x) || !aligned16(w_tiles) || (ldx % 8) != 0 || ldx < k) return MV_ERR_INVALID_ARG;
    const bool sw = (flags & MV_GEMM_SWIGLU) != 0, of32 = (flags & MV_GEMM_OUT_F32) != 0;
    if (sw && (bias || residual || of32)) return MV_ERR_UNSUPPORTED;
    if (of32 && (bias || residual)) return MV_ERR_UNSUPPORTED;
    if (slabs_only && (sw || of32 || bias || residual || post_ln_w)) return MV_ERR_UNSUPPORTED;
    const int ncols = sw ? n / 2 : n;
    if (!slabs_only) {
        if (ldy < ncols) return MV_ERR_INVALID_ARG;
        if (!of32 && ((reinterpret_cast<uintptr_t>(y) & 7) != 0 || (ldy % 4) != 0))
            return MV_ERR_INVALID_ARG;
        if (of32 && (!aligned16(y) || (ldy % 4) != 0)) return MV_ERR_INVALID_ARG;
    }
    if (residual && ld_res < n) return MV_ERR_INVALID_ARG;
    if (prologue != kProNone) {
        if (!aligned16(ln_w)) return MV_ERR_INVALID_ARG;
        if (prologue == kProAddNorm &&
            (!aligned16(add_r) || !aligned16(sum_out) || (ld_add_r % 8) || (ld_sum_out % 8) ||
             ld_add_r < k || ld_sum_out < k))
            return MV_ERR_INVALID_ARG;
    }
    const bool dot = dot_form_takes(m, k);
    if (prologue != kProNone && !dot) return MV_ERR_UNSUPPORTED;   // the matrix form reads x as it is

    GemmArgs a = {};
    a.x = (const uint16_t*)x;
    a.ldx = ldx;
    a.w = (const uint4*)w_tiles;
    a.bias = (const uint16_t*)bias;
    a.residual = (const uint16_t*)residual;
    a.ld_res = ld_res;
    a.y = y;
    a.ldy = ldy;
    a.m = m;
    a.n = n;
    a.k = k;
    a.nt = n / 16;
    a.kt = k / 32;
    a.act = act;
    a.prologue = prologue;
    a.var_from_rounded = var_from_rounded;
    a.add_r = (const uint16_t*)add_r;
    a.ld_add_r = ld_add_r;
    a.ln_w = (const uint16_t*)ln_w;
    a.eps = eps;
    a.sum_out = (uint16_t*)sum_out;
    a.ld_sum_out = ld_sum_out;
    const bool free_reduce = slabs_only || post_ln_w != nullptr || (flags & MV_GEMM_PLAN_SLABS) != 0;
    a.ksplit = slices ? slices : pick_ksplit(m, a.nt, a.kt, free_reduce);
    a.partial = nullptr;
    a.post_ln_w = (const uint16_t*)post_ln_w;
    a.post_out = (uint16_t*)post_out;
    a.ld_post = ld_post;
    a.post_eps = post_eps;
    a.post_var_from_rounded = post_var_from_rounded;
    if (slabs_only) {
        // the caller's next kernel adds the slabs (one slab when the planner would not split)
        const size_t need = (size_t)a.ksplit * m * n * sizeof(float);
        if (!workspace || workspace_bytes < need || !aligned16(workspace)) return MV_ERR_WORKSPACE;
        a.partial = (float*)workspace;
    } else if (post_ln_w) {
        // the norm lives in the slab reduction, so the product always goes through slabs (one
        // slab when the planner would not split)
        if (sw || of32 || (n % 8) != 0 || n > 8 * 256 * kPostChunks) return MV_ERR_UNSUPPORTED;
        if (!post_out || !aligned16(post_ln_w) || !aligned16(post_out) || !aligned16(y) ||
            (ld_post % 8) != 0 || ld_post < n || (ldy % 8) != 0)
            return MV_ERR_INVALID_ARG;
        if ((bias && !aligned16(bias)) || (residual && (!aligned16(residual) || (ld_res % 8) != 0)))
            return MV_ERR_INVALID_ARG;
        const size_t need = (size_t)a.ksplit * m * n * sizeof(float);
        if (!workspace || workspace_bytes < need || !aligned16(workspace)) return MV_ERR_WORKSPACE;
        a.partial = (float*)workspace;
    } else if (a.ksplit > 1) {
        const size_t need = (size_t)a.ksplit * m * n * sizeof(float);
        if (!workspace || workspace_bytes < need || !aligned16(workspace)) {
            a.ksplit = 1;  // no room for slabs: fall back to whole strips (slower, same result class)
        } else {
            a.partial = (float*)workspace;
        }
    }
    a.ktps = a.kt / a.ksplit;
    a.contig = g_tune_contig;
    const int sg = dot ? 1 : mfma_strip_group(m, a.nt, a.kt, free_reduce);
    a.nunits = ((a.nt + sg - 1) / sg) * a.ksplit;
    a.flags = flags;

    const int cus = num_cus();
    // Dot-form shape, from sweeps on MI355X (tools/sweep_wgemm.py, M=1, 4 tiles per stage):
    // with at most one strip per CU a single 16-wave workgroup hides HBM latency best
    // (O 8.0 -> 7.4 us, down 20.6 -> 20.4); with more strips than CUs two 8-wave workgroups
    // per CU even out the tail (QKV 12.8 -> 11.3 us, gate/up 39.1 -> 37.6).
    // Sixteen waves only pay when nearly every CU has a strip and the strip is long: shards with
    // short k (K=1792: 4.8 vs 5.8 us) or few strips (48: 5.4 vs 5.8) are faster with eight.
    const int forced_bpc = g_tune_bpc;
    int waves = dot_form_waves_for_units(a.nunits, a.kt);
    if (dot && !dot_form_fits(m, k, waves)) waves = 8;
    int bpc = forced_bpc ? forced_bpc : (dot && waves == 8 ? 2 : 1);
    if (dot) {
        // LDS limits co-residency; never size the grid past what fits
        const int fit = (int)((160 * 1024) / (dot_form_lds(m, k, waves) + 512));
        if (bpc > fit) bpc = fit;
    }
    if (bpc > 4) bpc = 4;  // 4 x 512 threads = 32 waves per CU
    int grid = a.nunits < cus * bpc ? a.nunits : cus * bpc;
    hipStream_t s = (hipStream_t)stream;

    int rc;
    switch (dot ? m : 0) {
        case 1: rc = launch_dot_waves<1>(a, waves, grid, s); break;
        case 2: rc = launch_dot_waves<2>(a, waves, grid, s); break;
        case 3: rc = launch_dot_waves<3>(a, waves, grid, s); break;
        case 4: rc = launch_dot_waves<4>(a, waves, grid, s); break;
        default: {
            rc = with_row_blocks(m, [&](auto hb) { return launch_mfma<decltype(hb)::value>(a, sg, grid, s); });
        }
    }
    if (rc != MV_OK || slabs_only) return rc;
    if (post_ln_w) {
        rc = launch_finalize_norm(a, s);
    } else if (a.ksplit > 1) {
        const int64_t total = (int64_t)m * ncols;
        int blocks = (int)((total + 255) / 256);
        if (blocks > cus * 4) blocks = cus * 4;
        hipLaunchKernelGGL(a.act.kind ? wgemm_finalize_kernel<true> : wgemm_finalize_kernel<false>, dim3(blocks), dim3(256), 0, s, a);
        rc = check_launch();
    }
    return rc;
}

int launch_wgemm_slices(const void* x, int64_t ldx, const void* w_tiles, float* slabs, size_t slabs_bytes, int m, int n, int k,
                        mv_stream_t stream) {
    return wgemm_impl(x, ldx, nullptr, 0, nullptr, 0.f, nullptr, 0, kProNone, 0, w_tiles, nullptr, nullptr, 0, nullptr, 0, m, n,
                      k, slabs, slabs_bytes, MV_GEMM_SLABS, stream, nullptr, 0.f, nullptr, 0, 0, wgemm_slices(m, n, k));
}

int launch_wgemm_act(const void* x, int64_t ldx, const void* w_tiles, void* y, int64_t ldy, int m, int n, int k, void* workspace,
                     size_t workspace_bytes, GemmAct act, mv_stream_t stream) {
    return wgemm_impl(x, ldx, nullptr, 0, nullptr, 0.f, nullptr, 0, kProNone, 0, w_tiles, nullptr, nullptr, 0, y, ldy, m, n, k,
                      workspace, workspace_bytes, act.kind == 2 ? MV_GEMM_SWIGLU : 0, stream, nullptr, 0.f, nullptr, 0, 0, 0, act);
}

}  // namespace mv

extern "C" {

// Tuning hook for experiments: key 0 = workgroups per CU, key 1 = forced ksplit,
// key 2 = waves per workgroup of the dot form (8 or 16), key 3 = strips per workgroup of the
// MFMA form (1, 2, 3, 4, 7); 0 = let the planner choose.
int mv_wgemm_tune(int key, int value) {
    if (key == 2 && (value == 0 || value == 8 || value == 16)) {
        mv::g_tune_waves = value;
        return MV_OK;
    }
    if (key == 3 && (value == 0 || value == 1 || value == 2 || value == 3 || value == 4 || value == 7)) {
        mv::g_tune_sg = value;
        return MV_OK;
    }
    if (key == 0 && value >= 0 && value <= 8) {
        mv::g_tune_bpc = value;
        return MV_OK;
    }
    if (key == 1 && value >= 0 && value <= mv::kMaxKsplit) {
        mv::g_tune_ksplit = value;
        return MV_OK;
    }
    if (key == 4 && (value == 0 || value == 1)) {
        mv::g_tune_contig = value;
        return MV_OK;
    }
    return MV_ERR_INVALID_ARG;
}

size_t mv_wgemm_workspace_bytes(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0 || (n % 16) || (k % 32)) return 0;
    // slabs for the split the planner picks now; a call that later finds the
    // workspace too small (tuning changed) runs unsplit instead of failing
    // (the larger of the plain plan and the MV_GEMM_PLAN_SLABS one: the flag is not known here)
    const int ks = std::max(mv::pick_ksplit(m, n / 16, k / 32), mv::pick_ksplit(m, n / 16, k / 32, true));
    return ks > 1 ? (size_t)ks * (size_t)m * (size_t)n * sizeof(float) : 0;
}

int mv_wgemm(const void* x, int64_t ldx, const void* w_tiles, const void* bias,
             const void* residual, int64_t ld_res, void* y, int64_t ldy, int m, int n, int k,
             void* workspace, size_t workspace_bytes, int flags, mv_stream_t stream) {
    return mv::wgemm_impl(x, ldx, nullptr, 0, nullptr, 0.f, nullptr, 0, mv::kProNone, 0, w_tiles, bias,
                          residual, ld_res, y, ldy, m, n, k, workspace, workspace_bytes, flags,
                          stream);
}

int mv_wgemm_slab_count(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0 || (n % 16) || (k % 32)) return 0;
    return mv::pick_ksplit(m, n / 16, k / 32, true);
}

size_t mv_wgemm_postnorm_workspace_bytes(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0 || (n % 16) || (k % 32)) return 0;
    const int ks = mv::pick_ksplit(m, n / 16, k / 32, true);
    return (size_t)(ks > 1 ? ks : 1) * (size_t)m * (size_t)n * sizeof(float);
}

int mv_wgemm_postnorm(const void* x, int64_t ldx, const void* w_tiles, const void* bias,
                      const void* residual, int64_t ld_res, void* y, int64_t ldy, const void* ln_w,
                      float eps, void* normed, int64_t ld_normed, int norm_flags, int m, int n, int k,
                      void* workspace, size_t workspace_bytes, mv_stream_t stream) {
    if (!ln_w || !normed) return MV_ERR_INVALID_ARG;
    return mv::wgemm_impl(x, ldx, nullptr, 0, nullptr, 0.f, nullptr, 0, mv::kProNone, 0, w_tiles, bias,
                          residual, ld_res, y, ldy, m, n, k, workspace, workspace_bytes, 0, stream,
                          ln_w, eps, normed, ld_normed,
                          (norm_flags & MV_NORM_VAR_FROM_ROUNDED) ? 1 : 0);
}

int mv_wgemm_norm(const void* x, int64_t ldx, const void* add_r, int64_t ld_add_r,
                  const void* ln_w, float eps, void* sum_out, int64_t ld_sum_out, int norm_flags,
                  const void* w_tiles, const void* bias, const void* residual, int64_t ld_res,
                  void* y, int64_t ldy, int m, int n, int k, void* workspace,
                  size_t workspace_bytes, int flags, mv_stream_t stream) {
    if (!ln_w) return MV_ERR_INVALID_ARG;
    if ((add_r == nullptr) != (sum_out == nullptr)) return MV_ERR_INVALID_ARG;
    if (m > 4) return MV_ERR_UNSUPPORTED;  // the fused input transform lives in the dot form
    return mv::wgemm_impl(x, ldx, add_r, ld_add_r, ln_w, eps, sum_out, ld_sum_out,
                          add_r ? mv::kProAddNorm : mv::kProNorm,
                          (norm_flags & MV_NORM_VAR_FROM_ROUNDED) ? 1 : 0, w_tiles, bias, residual,
                          ld_res, y, ldy, m, n, k, workspace, workspace_bytes, flags, stream);
}

}  // extern "C"

#ifdef MV_WGEMM_STAMP
extern "C" int mv_debug_read_wgemm_stamps(void* dst, size_t bytes) {
    return hipMemcpyFromSymbol(dst, HIP_SYMBOL(mv::g_wstamp), bytes) == hipSuccess ? 0 : -3;
}
#endif
