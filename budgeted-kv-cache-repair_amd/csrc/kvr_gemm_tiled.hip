// Projection GEMMs of more packed refresh rows than the streaming kernel of
// kvr_gemm.hip serves (gfx950 MFMA):
//   y[m, r] = sum_k x[m, k] * w[r, k]      bf16 / fp16, fp32 accumulation
// i.e. the q/k/v/o and MLP projections of the decoder layers (transformers
// 5.15.0 models/llama/modeling_llama.py:165-175, 243-252) for 65 rows up to a
// whole suffix. As in the streaming kernel one launch takes up to three weights
// (rows concatenated) or a gate/up pair with the SiLU-gated product in its
// epilogue, a residual can be added, and K can be split, the fp32 partials
// being summed by the consumer (fresh-row epilogue, residual + RMSNorm) or by
// tiled_reduce_kernel.
//
// What bounds it: reading the weights below ~200 rows (0.44 GB per layer of an
// 8B model), the matrix cores above. So the block tile follows the row count:
// every weight byte is read from HBM by as few blocks as LDS allows (the tile
// covers all rows up to 288), and the tile and the K split are chosen together
// so that the grid fills the 256 CUs in whole rounds (choose()).
//
// A stage of 64 k (128-byte rows, whole cache lines) of both operands goes
// straight from global memory to LDS (global_load_lds_dwordx4, no registers),
// 2 to 4 stages deep; LDS is full, so a CU runs one block (two of the smallest
// tile). Fragments of the next 32 k are read while the current ones are
// multiplied; at the turn of a stage every wave holds its last fragments, so
// after the barrier the stage's buffer is refilled at once, its loads and the
// next reads issued one by one between the MFMAs (in a burst before them
// 256 x 256 ran 5% slower; spread over the whole half step the last loads came
// too late, 3-5%: three quarters is best). 16-byte pieces are swizzled by row
// (SQ_LDS_BANK_CONFLICT counts none).
//
// Measured in the refreshes (us for the four projections of one 8B layer, from their
// kernel traces): 71 rows 100, 141 rows (fp16) 123, 282 rows 182, 1383 rows (Qwen3
// shape) 537, 15104 rows 5120 = 1.29 PFLOP/s; hipBLASLt's separate q, k, v, o, gate,
// up, down, SiLU and residual launches, timed alone, took 210, 230, 270 and 560 for
// the first four. Gate/up at 71 rows 44.6 us = 5.3 TB/s of weights, at 15104 rows
// 1.31 PFLOP/s: the matrix cores are busy 69% of the cycles of an engine clock that
// falls to 1.7 GHz; the rest are the turns of the stages and their LDS reads.
#include "kvr_internal.h"

#include <math.h>
#include <string.h>

#include <type_traits>
#include <utility>

namespace kvr {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct tile_t;
template <> struct tile_t<bf16_t> {
    typedef __bf16 v8 __attribute__((ext_vector_type(8)));
    __device__ static inline f32x4 mma(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <> struct tile_t<f16_t> {
    typedef _Float16 v8 __attribute__((ext_vector_type(8)));
    __device__ static inline f32x4 mma(v8 a, v8 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

constexpr int kStageK = 64;       // k of one LDS stage
constexpr int kRowBytes = 128;
constexpr int kGroupRows = 8;     // rows of one wave-wide 1 KB load
constexpr int kXcds = 8;
constexpr int kCusPerXcd = 32;
constexpr int kStreamRows = 192;  // STREAM tiles
constexpr int kPanelGroup = 4;    // weight panels that consecutive blocks of an XCD walk together

struct TiledArgs {
    const char* x;                // [M][ldx]
    const char* w0;               // weights: [rows_i][ldw_i]
    const char* w1;
    const char* w2;
    char* y;                      // [M][ldy]
    const char* res;              // residual [M][ldr] added to y, or null
    float* partial;               // splits > 1: fp32 [ceil(rows / 64)][splits][m][64]
    int64_t ldx, ldy, ldr, ldw0, ldw1, ldw2;
    int32_t end0, end1;           // concatenated row boundaries of w0 | w1 | w2
    int32_t rows;                 // streamed weight rows in total (multiple of 8)
    int32_t gated;                // 1: y = silu(x w0^T) * (x w1^T)
    int32_t m;
    int32_t steps;                // k / 64
    int32_t split_steps;          // steps per split
    int32_t splits;
    int32_t tiles_m, tiles_n;
};

// 16 bytes per lane from `base` (wave-uniform) + off into LDS at dst
// (wave-uniform) + 16 * lane; the second form with the nontemporal hint.
__device__ inline void load_lds(const char* base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off),
                 "s"(reinterpret_cast<uint64_t>(base)), "s"(dst)
                 : "memory", "m0");
}

__device__ inline void load_lds_once(const char* base, uint32_t off, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(off),
                 "s"(reinterpret_cast<uint64_t>(base)), "s"(dst)
                 : "memory", "m0");
}

template <int N>
__device__ inline void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt is six bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ inline const char* uniform(const char* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return reinterpret_cast<const char*>((static_cast<uint64_t>(hi) << 32) | lo);
}

template <typename F, int... I>
__device__ inline __attribute__((always_inline)) void static_for_each(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>): unrolled whatever the body's size.
template <int N, typename F>
__device__ inline __attribute__((always_inline)) void static_for(F&& f) {
    static_for_each(f, std::make_integer_sequence<int, (N > 0 ? N : 0)>{});
}

// `items` spread evenly over `slots`: the first item of slot t (item i goes to slot i * slots / items).
constexpr int first_slot(int t, int slots, int items) {
    return t >= slots ? items : (t * items + slots - 1) / slots;
}

// Block tile: BM rows of x by BN streamed weight rows; WM x WN waves of TM x TN
// MFMA tiles (16 x 16); NST LDS stages.
template <int TM_, int TN_, int WM_, int WN_, int NST_>
struct TileCfg {
    static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, NST = NST_;
    static constexpr int kWaves = WM * WN;
    static constexpr int kThreads = 64 * kWaves;
    static constexpr int BM = 16 * TM * WM;
    static constexpr int BN = 16 * TN * WN;
    static constexpr int kGroups = (BM + BN) / kGroupRows;            // loads per stage
    static constexpr int kLoads = (kGroups + kWaves - 1) / kWaves;    // per wave
    static constexpr int kStage = (BM + BN) * kRowBytes;
    static constexpr int kLds = NST * kStage;
    static_assert(kThreads <= 1024 && kLds <= 163840 && NST >= 2, "one CU");
    static_assert((NST - 1) * kLoads < 64, "vmcnt");
};

// 16-byte piece p of row r lies at piece p ^ swz(r): the 16 rows of a fragment
// read (one piece column) then cover all 64 banks.
__device__ constexpr int swz(int r) { return (r >> 1) & 7; }

// STREAM (one x tile of at most 192 rows: every weight byte is read once, and
// reading them is what bounds the launch): weights load nontemporally, and
// weight panel p starts at stage p of its k range and wraps around, so that
// concurrent blocks are not all at the same offset of their 8 KB and longer
// rows. Gate/up of an 8B model, 71 rows: 53.7 us, 49.4 nontemporal, 42.6 with
// the staggered start too (5.5 TB/s); 160 rows: 61.7, 58.8, 57.2. With more rows
// per panel or several x tiles, which read a panel together, both lose.
template <typename T, typename C, bool STREAM>
__global__ void __launch_bounds__(C::kThreads) tiled_gemm_kernel(TiledArgs a) {
    using G = tile_t<T>;
    using E = elem<T>;
    using v8 = typename G::v8;
    constexpr int TM = C::TM, TN = C::TN, BM = C::BM, BN = C::BN, NST = C::NST, L = C::kLoads;
    extern __shared__ __align__(16) char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lq = lane & 15;
    const int lj = lane >> 4;

    // blocks are dealt round-robin over the XCDs: give each XCD a run of
    // consecutive (weight panel, x tile) pairs, x tiles innermost
    const int total = a.tiles_m * a.tiles_n * a.splits;
    const int per = (total + kXcds - 1) / kXcds;
    const int item = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
    if (item >= total) return;
    const int panels = a.tiles_n * a.splits;
    const int first = item / (kPanelGroup * a.tiles_m) * kPanelGroup;
    const int wide = min(kPanelGroup, panels - first);
    const int at = item - first * a.tiles_m;
    const int mt = at / wide;
    const int panel = first + at % wide;
    const int nt = panel % a.tiles_n;
    const int split = panel / a.tiles_n;
    const int s0 = split * a.split_steps;
    const int steps = min(a.steps - s0, a.split_steps);
    const int m0 = mt * BM;

    // ---- this wave's loads of a stage: group g = rows 8g .. 8g + 7 of [BN weight rows | BM x rows] ----
    const char* base[L];
    uint32_t off[L];
    uint32_t dst[L];
#pragma unroll
    for (int j = 0; j < L; ++j) {
        int g = wave + j * C::kWaves;
        if (C::kGroups % C::kWaves != 0 && g >= C::kGroups) g -= C::kGroups;  // the same bytes again
        const int lr = lane >> 3;
        const int piece = (lane & 7) ^ swz((g * kGroupRows + lr) & 15);
        if (g < BN / kGroupRows) {
            // the group's rows belong to one weight, so its base is the wave's
            int r = nt * BN + g * kGroupRows;
            const char* wb = a.w0;
            int64_t ld = a.ldw0;
            if (r >= a.rows) r = 0;  // never written
            if (a.gated) {  // groups alternate: gate features, then the same of up
                const bool up = (r / kGroupRows) & 1;
                r = r / (2 * kGroupRows) * kGroupRows;
                wb = up ? a.w1 : a.w0;
                ld = up ? a.ldw1 : a.ldw0;
            } else if (r >= a.end1) {
                wb = a.w2;
                ld = a.ldw2;
                r -= a.end1;
            } else if (r >= a.end0) {
                wb = a.w1;
                ld = a.ldw1;
                r -= a.end0;
            }
            base[j] = uniform(wb + (static_cast<int64_t>(r) * ld + static_cast<int64_t>(s0) * kStageK) * 2);
            off[j] = static_cast<uint32_t>(lr * ld * 2) + piece * 16;
        } else {
            const int r = m0 + (g - BN / kGroupRows) * kGroupRows + lr;
            base[j] = uniform(a.x + (static_cast<int64_t>(m0) * a.ldx + static_cast<int64_t>(s0) * kStageK) * 2);
            off[j] = static_cast<uint32_t>((min(r, a.m - 1) - m0) * a.ldx * 2) + piece * 16;
        }
        dst[j] = __builtin_amdgcn_readfirstlane(
            static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
                reinterpret_cast<__attribute__((address_space(3))) char*>(
                    (__attribute__((address_space(3))) char*)smem)) + g * 1024));
    }
    // ---- fragments ----
    const int wm = wave % C::WM;
    const int wn = wave / C::WM;
    const char* wfrag[2];
    const char* xfrag[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
        const int at = lq * kRowBytes + (((kk * 4 + lj) ^ swz(lq)) * 16);
        wfrag[kk] = smem + wn * (16 * TN) * kRowBytes + at;
        xfrag[kk] = smem + (BN + wm * (16 * TM)) * kRowBytes + at;
    }
    u32x4 fw[2][TN], fx[2][TM];
    // fragment f of half kk: the weight fragments, then x's
    auto read = [&](int kk, int at, int f) __attribute__((always_inline)) {
        if (f < TN)
            fw[kk][f] = *reinterpret_cast<const u32x4*>(wfrag[kk] + at + f * 16 * kRowBytes);
        else
            fx[kk][f - TN] = *reinterpret_cast<const u32x4*>(xfrag[kk] + at + (f - TN) * 16 * kRowBytes);
    };
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // load l of the stage that comes next (`next_k` its byte offset in the k range) to LDS offset `at`
    const int64_t k_bytes = static_cast<int64_t>(steps) * kRowBytes;
    int64_t next_k = STREAM ? static_cast<int64_t>(panel % steps) * kRowBytes : 0;
    auto load = [&](int l, uint32_t at) __attribute__((always_inline)) {
        if constexpr (STREAM) {
            if (wave + l * C::kWaves < BN / kGroupRows)
                load_lds_once(base[l] + next_k, off[l], dst[l] + at);
            else
                load_lds(base[l] + next_k, off[l], dst[l] + at);
        } else {
            load_lds(base[l], off[l], dst[l] + at);
            base[l] += kRowBytes;
        }
    };
    auto loaded = [&]() __attribute__((always_inline)) {
        if constexpr (STREAM) {
            next_k += kRowBytes;
            if (next_k == k_bytes) next_k = 0;
        }
    };
    // The MFMAs of half kk, with the reads of the other half's next fragments
    // (and, with_load, the loads of a stage) issued between the first three
    // quarters of them.
    constexpr int kMul = TM * TN, kReads = TM + TN;
    constexpr int kSpan = kMul * 3 / 4 > 0 ? kMul * 3 / 4 : 1;
    auto multiply = [&](int kk, auto with_load, int read_at, uint32_t load_at) __attribute__((always_inline)) {
        static_for<kMul>([&](auto tc) __attribute__((always_inline)) {
            constexpr int t = decltype(tc)::value, i = t / TN, j = t % TN;
            acc[i][j] = G::mma(__builtin_bit_cast(v8, fw[kk][j]), __builtin_bit_cast(v8, fx[kk][i]), acc[i][j]);
            constexpr int l0 = first_slot(t, kSpan, L), l1 = first_slot(t + 1, kSpan, L);
            constexpr int f0 = first_slot(t, kSpan, kReads), f1 = first_slot(t + 1, kSpan, kReads);
            if constexpr (decltype(with_load)::value)
                static_for<l1 - l0>([&](auto lc) __attribute__((always_inline)) {
                    constexpr int l = l0 + decltype(lc)::value;
                    load(l, load_at);
                });
            static_for<f1 - f0>([&](auto fc) __attribute__((always_inline)) {
                read(kk ^ 1, read_at, f0 + decltype(fc)::value);
            });
            if constexpr (f1 > f0 || (decltype(with_load)::value && l1 > l0)) __builtin_amdgcn_sched_barrier(0);
        });
    };

    static_for<NST>([&](auto sc) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
        if (s < steps) {
#pragma unroll
            for (int l = 0; l < L; ++l) load(l, s * C::kStage);
            loaded();
        }
    });
    if (steps >= NST)
        wait_vm<(NST - 1) * L>();
    else
        wait_vm<0>();
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int f = 0; f < kReads; ++f) read(0, 0, f);
    const std::integral_constant<bool, true> yes{};
    const std::integral_constant<bool, false> no{};
    int stage = 0;
    // Every wave holds the last fragments of stage `stage` once all pass the
    // barrier, so its buffer takes stage s + NST (with_load) while the next
    // stage's first half is read. `ahead`: stages that may still be in flight
    // once the next one has landed. Past the last stage the reads are in bounds
    // and unused.
    auto turn = [&](auto with_load, auto ahead) __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        const int next = stage + C::kStage == C::kLds ? 0 : stage + C::kStage;
        wait_vm<decltype(ahead)::value * L>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, with_load, next, static_cast<uint32_t>(stage));
        if constexpr (decltype(with_load)::value) loaded();
        stage = next;
    };
    int s = 0;
    for (; s + NST < steps; ++s) {
        __builtin_amdgcn_sched_barrier(0);
        multiply(0, no, stage, 0);
        turn(yes, std::integral_constant<int, NST - 2>{});
    }
    for (; s < steps; ++s) {  // the last min(NST, steps) stages: nothing left to load
        __builtin_amdgcn_sched_barrier(0);
        multiply(0, no, stage, 0);
        turn(no, std::integral_constant<int, 0>{});
    }

    // ---- lane: x row 16 i + lq, weight rows 16 j + 4 lj .. + 3 ----
    const int mrow = m0 + wm * (16 * TM) + lq;
    const int n0 = nt * BN + wn * (16 * TN) + 4 * lj;
    if (a.splits > 1) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int m = mrow + 16 * i;
            if (m >= a.m) continue;
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = n0 + 16 * j;
                if (n < a.rows)
                    *reinterpret_cast<f32x4*>(a.partial +
                                              ((static_cast<int64_t>(n >> 6) * a.splits + split) * a.m + m) * 64 +
                                              (n & 63)) = acc[i][j];
            }
        }
        return;
    }
    uint16_t* y = reinterpret_cast<uint16_t*>(a.y);
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    if (a.gated) {
        // Lanes 0-31 hold gate features, lanes 32-63 the same features of up:
        // swapping the upper half of tile i with the lower half of tile i + 1
        // puts gate and up of tile i in the lower lanes, of tile i + 1 in the upper.
#pragma unroll
        for (int i = 0; i < TM; i += 2) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                u16x4 out;
                const bool pair = i + 1 < TM;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t g = __float_as_uint(acc[i][j][e]);
                    uint32_t u = pair ? __float_as_uint(acc[pair ? i + 1 : i][j][e]) : 0u;
                    const auto sw2 = __builtin_amdgcn_permlane32_swap(g, u, false, false);
                    g = sw2[0];
                    u = sw2[1];
                    out[e] = E::from_float(silu_gate<T>(round_through<T>(__uint_as_float(g)),
                                                        round_through<T>(__uint_as_float(u))));
                }
                const int m = mrow + 16 * (i + (lj >> 1));
                const int n = nt * BN + wn * (16 * TN) + 16 * j;  // streamed row of the tile
                const int f = (n >> 1) + 4 * (lj & 1);
                if (m < a.m && n < a.rows && (pair || lj < 2))
                    *reinterpret_cast<u16x4*>(y + static_cast<int64_t>(m) * a.ldy + f) = out;
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = mrow + 16 * i;
        if (m >= a.m) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + 16 * j;
            if (n >= a.rows) continue;
            u16x4 out;
            if (a.res) {
                const u16x4 r = *reinterpret_cast<const u16x4*>(reinterpret_cast<const uint16_t*>(a.res) +
                                                                static_cast<int64_t>(m) * a.ldr + n);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    out[e] = E::from_float(round_through<T>(acc[i][j][e]) + E::to_float(r[e]));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) out[e] = E::from_float(acc[i][j][e]);
            }
            *reinterpret_cast<u16x4*>(y + static_cast<int64_t>(m) * a.ldy + n) = out;
        }
    }
}

// Sum of the split-K partials in split order (+ residual), four columns per thread.
constexpr int kReduceThreads = 256;

template <typename T>
__global__ void __launch_bounds__(kReduceThreads) tiled_reduce_kernel(TiledArgs a) {
    using E = elem<T>;
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    const int quads = a.rows / 4;
    const int64_t e = static_cast<int64_t>(blockIdx.x) * kReduceThreads + threadIdx.x;
    if (e >= static_cast<int64_t>(a.m) * quads) return;
    const int64_t m = e / quads;
    const int n = static_cast<int>(e - m * quads) * 4;
    const int64_t step = static_cast<int64_t>(a.m) * 64;
    const float* at = a.partial + (static_cast<int64_t>(n >> 6) * a.splits * a.m + m) * 64 + (n & 63);
    f32x4 sum = *reinterpret_cast<const f32x4*>(at);
    for (int s = 1; s < a.splits; ++s) sum += *reinterpret_cast<const f32x4*>(at + s * step);
    u16x4 out;
    if (a.res) {
        const u16x4 r = *reinterpret_cast<const u16x4*>(reinterpret_cast<const uint16_t*>(a.res) + m * a.ldr + n);
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = E::from_float(round_through<T>(sum[i]) + E::to_float(r[i]));
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = E::from_float(sum[i]);
    }
    *reinterpret_cast<u16x4*>(reinterpret_cast<uint16_t*>(a.y) + m * a.ldy + n) = out;
}

// The tiles, each with the measured time of one stage (us, every CU busy). They
// differ in how many rows they cover with the weights read once and in how
// they divide a projection's grid into whole rounds of 256 CUs.
#define KVR_TILES(X) \
    X(8, 4, 2, 4, 2, 1.23f) /* 256 x 256 */ \
    X(7, 4, 2, 4, 2, 1.23f) /* 224 x 256 */ \
    X(6, 4, 2, 4, 2, 1.16f) /* 192 x 256 */ \
    X(5, 4, 2, 4, 3, 0.90f) /* 160 x 256 */ \
    X(4, 4, 2, 4, 3, 0.81f) /* 128 x 256 */ \
    X(6, 3, 3, 4, 2, 1.19f) /* 288 x 192 */ \
    X(9, 2, 2, 4, 3, 0.86f) /* 288 x 128 */ \
    X(8, 2, 2, 4, 3, 0.77f) /* 256 x 128 */ \
    X(7, 2, 2, 4, 3, 0.75f) /* 224 x 128 */ \
    X(6, 2, 2, 4, 3, 0.60f) /* 192 x 128 */ \
    X(5, 2, 2, 4, 4, 0.60f) /* 160 x 128 */ \
    X(3, 2, 3, 4, 4, 0.52f) /* 144 x 128 */ \
    X(4, 2, 2, 4, 4, 0.46f) /* 128 x 128 */ \
    X(3, 2, 2, 4, 4, 0.43f) /* 96 x 128 */ \
    X(5, 1, 1, 8, 4, 0.37f) /* 80 x 128 */ \
    X(5, 1, 1, 7, 4, 0.31f) /* 80 x 112 */ \
    X(6, 1, 1, 7, 4, 0.36f) /* 96 x 112 */ \
    X(9, 1, 1, 7, 4, 0.51f) /* 144 x 112 */ \
    X(5, 1, 1, 4, 4, 0.27f) /* 80 x 64 */ \
    X(8, 1, 1, 4, 4, 0.41f) /* 128 x 64 */ \
    X(5, 1, 1, 6, 4, 0.29f) /* 80 x 96 */ \
    X(8, 1, 1, 6, 4, 0.43f) /* 128 x 96 */

struct Tile {
    int32_t bm, bn;
    float step_us;
};
constexpr Tile kTiles[] = {
#define X(TM, TN, WM, WN, NST, US) \
    {TileCfg<TM, TN, WM, WN, NST>::BM, TileCfg<TM, TN, WM, WN, NST>::BN, US},
    KVR_TILES(X)
#undef X
};
constexpr int kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int32_t kMaxSplits = 8;
constexpr int32_t kMinSplitSteps = 4;  // k of a split at least: four stages

// The smallest tile, two blocks of which share a CU.
constexpr bool smallest_tile(int bm, int bn) { return bm == 80 && bn == 64; }

struct Choice {
    int32_t tile;
    int32_t splits;
    int32_t split_steps;
};

// The tile and K split with the least modelled time, of a model fitted to 260
// measured projections (q/k/v, o, gate/up, down of 8B shapes, 65 to 8192 rows;
// the choice is 0.7% slower than the fastest tile on average, 19% at most):
// blocks run in rounds of 32 CUs per XCD, a round costs its stages plus 2.1 us
// (2.3 us more for the gated epilogue); against it stands the weight stream,
// 5.9 TB/s with every CU loading, 7.0 nontemporal; both overlap as a 2-norm.
// Split partials cost 0.16 us/MB to write and 0.2 in their consumer. The
// smallest tile has no place beside other x tiles: two of its blocks share a CU.
Choice model_choice(int32_t m, int32_t rows, int32_t k, bool gated) {
    const int32_t steps = k / kStageK;
    Choice best{0, 1, steps};
    double least = 1e30;
    for (int t = 0; t < kTileCount; ++t) {
        const Tile& tile = kTiles[t];
        const int64_t tiles_m = ceil_div(m, tile.bm);
        if (smallest_tile(tile.bm, tile.bn) && tiles_m > 1) continue;
        const int64_t tiles = tiles_m * ceil_div(rows, tile.bn);
        const bool once = tiles_m == 1 && tile.bm <= kStreamRows;
        for (int32_t want = 1; want <= kMaxSplits; want *= 2) {
            if (want > 1 && (gated || steps / want < kMinSplitSteps)) break;
            const int32_t split_steps = static_cast<int32_t>(ceil_div(steps, want));
            const int32_t splits = static_cast<int32_t>(ceil_div(steps, split_steps));
            const int64_t blocks = tiles * splits;
            const int64_t rounds = ceil_div(ceil_div(blocks, kXcds), kCusPerXcd);
            const double work = rounds * (split_steps * static_cast<double>(tile.step_us) + (gated ? 4.4 : 2.1));
            const double busy = blocks < 256 ? static_cast<double>(blocks) / 256 : 1.0;
            const double stream = static_cast<double>(rows) * k * 2 / (once ? 7.0e6 : 5.9e6) / sqrt(busy);
            double us = sqrt(work * work + stream * stream);
            if (splits > 1) us += static_cast<double>(m) * rows * 4 * splits * 0.36e-6;
            if (us < least) {
                least = us;
                best = Choice{t, splits, split_steps};
            }
            if (blocks >= 1024) break;  // more splits only add partials
        }
    }
    return best;
}

// model_choice (~1 us of host time), remembered per thread for the few
// projections that a forward runs layer after layer.
Choice choose(int32_t m, int32_t rows, int32_t k, bool gated) {
    struct Entry {
        int32_t m, rows, k, gated;
        Choice choice;
    };
    constexpr int kEntries = 8;
    static thread_local Entry memo[kEntries] = {};
    static thread_local int next = 0;
    for (const Entry& e : memo)
        if (e.m == m && e.rows == rows && e.k == k && e.gated == (gated ? 1 : 0)) return e.choice;
    const Choice c = model_choice(m, rows, k, gated);
    memo[next] = Entry{m, rows, k, gated ? 1 : 0, c};
    next = (next + 1) % kEntries;
    return c;
}

template <typename T, typename C, bool STREAM>
int launch_tile(const TiledArgs& a, hipStream_t s) {
    static const bool ok = C::kLds <= 65536 ||
                           hipFuncSetAttribute(reinterpret_cast<const void*>(tiled_gemm_kernel<T, C, STREAM>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, C::kLds) == hipSuccess;
    if (!ok) return KVR_E_LAUNCH_FAILED;
    const int64_t total = static_cast<int64_t>(a.tiles_m) * a.tiles_n * a.splits;
    tiled_gemm_kernel<T, C, STREAM>
        <<<static_cast<unsigned>(ceil_div(total, kXcds) * kXcds), C::kThreads, C::kLds, s>>>(a);
    return launch_status();
}

template <typename T, typename C>
int launch_tile(const TiledArgs& a, hipStream_t s) {
    if constexpr (C::BM <= kStreamRows) {
        if (a.tiles_m == 1) return launch_tile<T, C, true>(a, s);
    }
    if constexpr (smallest_tile(C::BM, C::BN))
        return KVR_E_INVALID_ARGUMENT;  // never chosen for more x tiles
    else
        return launch_tile<T, C, false>(a, s);
}

template <typename T>
int launch_tiled(TiledArgs a, int32_t tile, bool reduce, hipStream_t s) {
    a.tiles_m = static_cast<int32_t>(ceil_div(a.m, kTiles[tile].bm));
    a.tiles_n = static_cast<int32_t>(ceil_div(a.rows, kTiles[tile].bn));
    int st = KVR_E_INVALID_ARGUMENT;
    int t = 0;
#define X(TM, TN, WM, WN, NST, US) \
    if (t++ == tile) st = launch_tile<T, TileCfg<TM, TN, WM, WN, NST>>(a, s);
    KVR_TILES(X)
#undef X
    if (st != KVR_OK || a.splits == 1 || !reduce) return st;
    const int64_t quads = static_cast<int64_t>(a.m) * (a.rows / 4);
    tiled_reduce_kernel<T><<<static_cast<unsigned>(ceil_div(quads, kReduceThreads)), kReduceThreads, 0, s>>>(a);
    return launch_status();
}

bool aligned(const void* p, uintptr_t to) { return (reinterpret_cast<uintptr_t>(p) & (to - 1)) == 0; }

// Rows of the weights of one call in total, or a negative status.
int64_t total_rows(int32_t n_weights, const int32_t* rows, bool gated) {
    if (n_weights < 1 || n_weights > 3 || !rows) return KVR_E_INVALID_ARGUMENT;
    if (gated && (n_weights != 2 || rows[0] != rows[1])) return KVR_E_UNSUPPORTED_SHAPE;
    int64_t total = 0;
    for (int i = 0; i < n_weights; ++i) {
        if (rows[i] <= 0 || rows[i] % kGroupRows) return KVR_E_UNSUPPORTED_SHAPE;
        total += rows[i];
    }
    return total > (1 << 24) ? KVR_E_UNSUPPORTED_SHAPE : total;
}

}  // namespace

bool tiled_linear_ok(int32_t m, int32_t rows, int32_t k) {
    return m > 0 && m <= kTiledMaxRows && rows > 0 && rows % kGroupRows == 0 && rows <= (1 << 24) && k > 0 &&
           k % kStageK == 0 && k <= (1 << 24);
}

int64_t tiled_workspace_bytes(int32_t m, int32_t rows, int32_t k) {
    if (!tiled_linear_ok(m, rows, k)) return KVR_E_UNSUPPORTED_SHAPE;
    const Choice c = choose(m, rows, k, false);
    return c.splits == 1 ? 0 : ceil_div(rows, kPartialTileCols) * kPartialTileCols * c.splits * m * 4;
}

int tiled_linear(const void* x, int32_t n_weights, const void* const* w, const int32_t* rows, const int64_t* ldw,
                 void* y, int32_t m, int32_t k, int64_t ldx, int64_t ldy, int32_t epilogue, const void* residual,
                 int64_t ldr, void* workspace, int64_t workspace_bytes, int32_t dtype, void* stream, bool reduce,
                 int32_t* splits_out) {
    if (dtype != KVR_DTYPE_BF16 && dtype != KVR_DTYPE_F16) return KVR_E_UNSUPPORTED_DTYPE;
    if (epilogue != KVR_LINEAR_CONCAT && epilogue != KVR_LINEAR_SILU_GATE && epilogue != KVR_LINEAR_RESIDUAL)
        return KVR_E_INVALID_ARGUMENT;
    const bool gated = epilogue == KVR_LINEAR_SILU_GATE;
    const int64_t total = total_rows(n_weights, rows, gated);
    if (total < 0) return static_cast<int>(total);
    if (!tiled_linear_ok(m, static_cast<int32_t>(total), k)) return KVR_E_UNSUPPORTED_SHAPE;
    if (!w || !ldw) return KVR_E_INVALID_ARGUMENT;
    const int64_t n_out = gated ? rows[0] : total;
    constexpr int64_t kMaxLd = int64_t(1) << 21;  // a tile's byte offsets fit 32 bits
    if (ldx < k || ldx % 8 || ldx > kMaxLd || ldy < n_out || ldy % 4) return KVR_E_BAD_STRIDE;
    for (int i = 0; i < n_weights; ++i)
        if (ldw[i] < k || ldw[i] % 8 || ldw[i] > kMaxLd) return KVR_E_BAD_STRIDE;
    if (epilogue == KVR_LINEAR_RESIDUAL) {
        if (!residual) return KVR_E_NULL_POINTER;
        if (ldr < n_out || ldr % 4 || !aligned(residual, 8)) return KVR_E_BAD_STRIDE;
        if (!reduce) return KVR_E_INVALID_ARGUMENT;  // partial consumers take plain sums
    }
    if (!x || !y) return KVR_E_NULL_POINTER;
    if (!aligned(x, 16) || !aligned(y, 8)) return KVR_E_BAD_STRIDE;
    for (int i = 0; i < n_weights; ++i) {
        if (!w[i]) return KVR_E_NULL_POINTER;
        if (!aligned(w[i], 16)) return KVR_E_BAD_STRIDE;
    }
    const Choice c = choose(m, static_cast<int32_t>(total), k, gated);
    if (c.splits > 1 && (!workspace || !aligned(workspace, 16) ||
                         workspace_bytes < tiled_workspace_bytes(m, static_cast<int32_t>(total), k)))
        return KVR_E_WORKSPACE_TOO_SMALL;
    TiledArgs a;
    memset(&a, 0, sizeof(a));
    a.x = static_cast<const char*>(x);
    a.w0 = static_cast<const char*>(w[0]);
    a.w1 = static_cast<const char*>(n_weights > 1 ? w[1] : w[0]);
    a.w2 = static_cast<const char*>(n_weights > 2 ? w[2] : w[0]);
    a.ldw0 = ldw[0];
    a.ldw1 = n_weights > 1 ? ldw[1] : ldw[0];
    a.ldw2 = n_weights > 2 ? ldw[2] : ldw[0];
    a.end0 = rows[0];
    a.end1 = n_weights > 1 ? rows[0] + rows[1] : rows[0];
    a.rows = static_cast<int32_t>(total);
    a.gated = gated ? 1 : 0;
    a.y = static_cast<char*>(y);
    a.res = epilogue == KVR_LINEAR_RESIDUAL ? static_cast<const char*>(residual) : nullptr;
    a.partial = static_cast<float*>(workspace);
    a.ldx = ldx;
    a.ldy = ldy;
    a.ldr = ldr;
    a.m = m;
    a.steps = k / kStageK;
    a.split_steps = c.split_steps;
    a.splits = c.splits;
    if (splits_out) *splits_out = c.splits;
    hipStream_t s = as_stream(stream);
    return dtype == KVR_DTYPE_BF16 ? launch_tiled<bf16_t>(a, c.tile, reduce, s)
                                   : launch_tiled<f16_t>(a, c.tile, reduce, s);
}

}  // namespace kvr

using namespace kvr;

extern "C" int kvr_internal_tiled_choice(int32_t m, int32_t rows, int32_t k, int32_t gated, int32_t out[4]) {
    if (!out || !tiled_linear_ok(m, rows, k)) return KVR_E_UNSUPPORTED_SHAPE;
    const Choice c = model_choice(m, rows, k, gated != 0);
    out[0] = kTiles[c.tile].bm;
    out[1] = kTiles[c.tile].bn;
    out[2] = m <= kTiles[c.tile].bm && kTiles[c.tile].bm <= kStreamRows;
    out[3] = c.splits;
    return KVR_OK;
}

extern "C" int64_t kvr_tiled_linear_workspace_bytes(int32_t m, int32_t rows, int32_t k) {
    return tiled_workspace_bytes(m, rows, k);
}

extern "C" int kvr_tiled_linear_multi(const void* x, int32_t n_weights, const void* const* w, const int32_t* rows,
                                      const int64_t* ldw, void* y, int32_t m, int32_t k, int64_t ldx, int64_t ldy,
                                      int32_t epilogue, const void* residual, int64_t ldr, void* workspace,
                                      int64_t workspace_bytes, int32_t dtype, void* stream) {
    return tiled_linear(x, n_weights, w, rows, ldw, y, m, k, ldx, ldy, epilogue, residual, ldr, workspace,
                        workspace_bytes, dtype, stream, true, nullptr);
}
