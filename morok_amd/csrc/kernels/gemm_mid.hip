// 16-bit products on output tiles of 64 and 128 rows and columns: shapes whose 128 x 256 tiles (gemm_bf16.hip) would leave
// compute units without work, and operands whose rows start on any element, read as they are.
//
// What bounds it: the path from the caches into the LDS.  A K step of a 128 x 128 tile brings 32 KB and takes 0.50 us
// with one workgroup per compute unit (66 GB/s), one of a 64 x 64 tile 16 KB and 0.18 us with two or three (93 GB/s; 24 TB/s over the
// chip, as 128 x 64 tiles reach with two), where the matrix instructions of either would take half of that; a 128 x 256 tile does
// twice the work of the former in 0.68 us (73 GB/s), so it stays where enough such tiles exist (profiles/gemm_mid_steps.txt).  Hence smaller tiles for fewer rows and columns, K split over
// workgroups where even those are few, and the choice by an estimate of the time (plan_mid).
//
// us before (128 x 256 tiles, split along K where that paid, padded copies of odd operands) and now: 1024 x 1024 x 1024 12.3 / 7.3,
// 198 x 3072 x 1024 12.2 / 7.5, [N, K] weights: 219 x 4288 x 3232 43.1 / 19.1, 700 x 700 x 4096 53.1 / 15.6,
// 75 x 1536 x 4576 18.7 / 11.5, 1000 x 3000 x 2048 22.9 / 19.8, 2791 x 96 x 13584 30.0 / 25.0, 487 x 4920 x 13416 171 / 98; odd: 300 x 3001 x 777 23.4 / 8.5, 5 x 7152 x 1638 27.8 / 9.0.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "gemm_elem.h"
#include "gemm_mid.h"
#include "kernels.h"

namespace mrk::dev {

// The elements of a chunk moved `by` places towards its start, zeros behind them (by <= 0: as it is).
__device__ __forceinline__ u32x4 shift_elems(u32x4 v, int by) {
    unsigned long long lo = ((unsigned long long)v[1] << 32) | v[0], hi = ((unsigned long long)v[3] << 32) | v[2];
    const int s = by * 16;
    if (s >= 64) {
        lo = s < 128 ? hi >> (s - 64) : 0;
        hi = 0;
    } else if (s > 0) {
        lo = (lo >> s) | (hi << (64 - s));
        hi >>= s;
    }
    return u32x4{(unsigned)lo, (unsigned)(lo >> 32), (unsigned)hi, (unsigned)(hi >> 32)};
}

// kTM x kTN output tile per workgroup of 4 waves (2 x 2), K step 64.  B is [K, N] or (kBT) [N, K].
// kDirect: operand rows are whole 16-byte chunks (K, and N of a [K, N] operand, multiples of 8) on 16-byte bases: tiles go
// global -> LDS directly, a ring of kAhead stages.  Otherwise (rows that start on any element, K and N at least 8) they pass
// through registers: kAhead register sets in flight and two stages.
// kSplit: blockIdx.z selects a range of kt_per_split K steps, f32 partial tiles go to W[z][batch][M][N].
// kEpilogue: kGate and kRotate put columns that belong together (a gate column and its up column F further on; the two of a rotated
// pair, 64 apart in a head of 128) into the two halves of a column pair, so that a lane holds both: the arithmetic of the
// 256-row tile's epilogues (gemm_bf16.hip), the same bits.
// The products, their order per accumulator and the roundings are those of the tiled kernels of gemm_bf16.hip: the same bits.
// The columns of a pair of 16-column matrix tiles are dealt to the two so that a lane ends up with eight consecutive ones.
enum MidEpilogue { kPlain, kGate, kRotate };
template <int kTM, int kTN, int kAhead, bool kBT, bool kF16, bool kDirect, bool kSplit, MidEpilogue kEpilogue = kPlain>
__global__ __launch_bounds__(256, 2) void gemm_mid(
    const __bf16* __restrict__ A, const __bf16* __restrict__ B, __bf16* __restrict__ C, float* __restrict__ W, const __bf16* __restrict__ R,
    int r_pitch, int M, int N, int K, int tiles_m, int tiles_n, int kt_per_split, MidRope rope) {
    static_assert(kEpilogue == kPlain || (kDirect && !kSplit && !kF16), "the gated and the rotary epilogue: bf16, whole chunks, one range of K");
    constexpr int kWM = kTM / 2, kWN = kTN / 2, kI = kWM / 16, kP = kWN / 32;  // a wave's tile, its 16-row blocks and 32-column pairs
    constexpr int kAq = kTM / 32, kBq = kTN / 32;                             // 16-byte chunks per work-item and K step
    constexpr int kAStage = kTM * 128, kBStage = kTN * 128, kStage = kAStage + kBStage;
    constexpr int kStages = kDirect ? kAhead : 2;
    __shared__ __attribute__((aligned(1024))) char smem[kStages * kStage];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    A += (size_t)blockIdx.y * M * K;
    B += (size_t)blockIdx.y * N * K;
    int tile_m, tile_n;
    tile_of_block(blockIdx.x, tiles_m, tiles_n, &tile_m, &tile_n);
    const int m0 = tile_m * kTM;
    const int n0 = tile_n * (kEpilogue == kGate ? kTN / 2 : kTN);  // (gated: of the F columns; rotary: the first in the order below)
    // Where column `c` of half `h` of the tile's column pair `p` lies: gated, F = N / 2 between gate and up; rotary, heads of 128
    auto paired_col = [&](int p, int h, int c) {
        if constexpr (kEpilogue == kGate) {
            const int F = N >> 1, col = n0 + p * 16 + c;
            return (col < F ? col : F - 1) + h * F;
        } else {
            const int col = (n0 & ~127) + (((n0 & 127) >> 1) + p * 16) + c + h * 64;
            return col < N ? col : N - 1;
        }
    };
    const int KT_all = (K + 63) >> 6;
    const int kt0 = kSplit ? (int)blockIdx.z * kt_per_split : 0;
    const int KT = kSplit ? (KT_all - kt0 < kt_per_split ? KT_all - kt0 : kt_per_split) : KT_all;
    const int k_left = K - kt0 * 64;  // depth from this range's first step to the end of K
    // the last step of the range is the partial last one of K
    const bool ragged = (K & 63) && kt0 + KT == KT_all;

    // Sources.  A and B^T chunk q of a wave: eight rows of 128 bytes, LDS chunk lane % 8 of row lane / 8 holds the logical chunk of
    // the row's swizzle.  Rows beyond the edge are the last valid one (their products are not stored).
    const char* a_base = reinterpret_cast<const char*>(A + (size_t)m0 * K + (size_t)kt0 * 64);
    // (paired columns are addressed from the first of B)
    const int b_first = kEpilogue == kPlain ? n0 : 0;
    const char* b_base = kBT ? reinterpret_cast<const char*>(B + (size_t)b_first * K + (size_t)kt0 * 64)
                             : reinterpret_cast<const char*>(B + (size_t)kt0 * 64 * N + b_first);
    const size_t b_step = kBT ? 128 : (size_t)N * 128;
    // first k of a lane's chunk q of A and of B inside a step (its k-row, [K, N] form)
    auto a_chunk = [&](int l, int q) { return ((l & 7) ^ (((wave * (kTM / 4) + q * 8 + (l >> 3)) >> 1) & 7)) * 8; };
    auto b_chunk = [&](int l, int q) {
        const int r = wave * (kTN / 4) + q * 8 + (l >> 3);
        return kBT ? ((l & 7) ^ (((r >> 1) & 1) | (((r >> 3) & 3) << 1))) * 8 : (wave * kBq + q) * (512 / kTN) + l / (kTN / 8);
    };
    unsigned a_off[kAq], b_off[kBq];  // byte offsets of the chunks from the bases of a step
    int b_back[kBq];                  // [K, N] form at the edge of N: elements by which a chunk was moved back to end at N
#pragma unroll
    for (int q = 0; q < kAq; q++) {
        const int r = wave * (kTM / 4) + q * 8 + (lane >> 3), row = m0 + r < M ? r : M - 1 - m0;
        a_off[q] = (unsigned)row * (unsigned)K * 2u + (kDirect ? a_chunk(lane, q) * 2 : 0);
    }
#pragma unroll
    for (int q = 0; q < kBq; q++) {
        b_back[q] = 0;
        if constexpr (kBT) {
            const int r = wave * (kTN / 4) + q * 8 + (lane >> 3);
            const int row = kEpilogue != kPlain ? paired_col(r >> 5, (r >> 2) & 1, 4 * ((r & 31) >> 3) + (r & 3)) : n0 + r < N ? r : N - 1 - n0;
            b_off[q] = (unsigned)row * (unsigned)K * 2u + (kDirect ? b_chunk(lane, q) * 2 : 0);
        } else {
            // k-rows of kTN * 2 bytes, 64-byte granules swizzled by the k-row
            const int kr = b_chunk(lane, q), ch = lane % (kTN / 8), f = kTN == 128 ? kr & 3 : (kr >> 1) & 1;
            const int col = (((ch >> 2) ^ f) * 4 + (ch & 3)) * 8;
            // (paired: a granule holds 16 columns of one half, then the 16 of the other)
            const int c = kEpilogue != kPlain ? paired_col((ch >> 2) ^ f, (ch >> 1) & 1, (ch & 1) * 8) / 8 * 8 : n0 + col + 8 <= N ? col : N - 8 - n0;
            b_off[q] = (unsigned)(kr * N + c) * 2u;
            b_back[q] = col - c;
        }
    }
    const int lds_w = wave * (kAq * 1024);
    const int lds_wb = kAStage + wave * (kBq * 1024);

    // fragment addresses
    int a_fr[2], b_fr[2][2];  // per 32-deep sub-step; [half of the pair] for B^T
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
        const int r = lane & 15;
        a_fr[ks] = (wm * kWM + r) * 128 + (((ks * 4 + (lane >> 4)) ^ ((r >> 1) & 7)) << 4);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int br = 8 * (r >> 2) + 4 * h + (r & 3);  // column of the pair this operand row stands for
            b_fr[ks][h] = kAStage + (wn * kWN + br) * 128 + (((ks * 4 + (lane >> 4)) ^ (((br >> 1) & 1) | (((br >> 3) & 3) << 1))) << 4);
        }
    }
    f32x4 acc[kI][kP][2];
#pragma unroll
    for (int i = 0; i < kI; i++)
#pragma unroll
        for (int p = 0; p < kP; p++)
#pragma unroll
            for (int h = 0; h < 2; h++) acc[i][p][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // Fragments are read a 32-deep sub-step ahead of their matrix instructions, into two register slots.
    bf16x8 fa[2][kI], fb[2][kP][2];
    bf16x4 lo[2][kP][2];  // ([K, N] form: the first four k of a fragment, until the other four are read)
    constexpr int kReads = kI + kP * (kBT ? 2 : 4), kMul = kI * kP * 2;
    auto read_one = [&](auto ks_c, int n, const char* st) {  // read n of sub-step ks
        constexpr int ks = decltype(ks_c)::value;
        if (n < kI) {
            fa[ks][n] = *LDS_PTR(const bf16x8, st + a_fr[ks] + n * 2048);
            return;
        }
        if constexpr (kBT) {
            const int p = (n - kI) >> 1, h = (n - kI) & 1;
            fb[ks][p][h] = *LDS_PTR(const bf16x8, st + b_fr[ks][h] + p * 4096);
        } else {
            const int p = (n - kI) >> 2, h = ((n - kI) >> 1) & 1, second = (n - kI) & 1;
            const int kr = ks * 32 + 8 * (lane >> 4) + ((lane & 15) >> 2) + 4 * second;
            const int g = wn * kP + p, f = kTN == 128 ? kr & 3 : (kr >> 1) & 1;
            const char* at = st + kAStage + (kEpilogue == kPlain ? 16 * (lane & 3) + 8 * h : 8 * (lane & 3) + 32 * h) + kr * (kTN * 2) + ((g ^ f) << 6);
            const bf16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, (char*)at));
            if (!second) lo[ks][p][h] = v;
            else fb[ks][p][h] = __builtin_shufflevector(lo[ks][p][h], v, 0, 1, 2, 3, 4, 5, 6, 7);
        }
    };
    // The matrix instruction written out, so that the accumulator stays in place.
    auto mfma = [&](f32x4& c, const bf16x8& a, const bf16x8& b) {
        if constexpr (kF16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
        else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    };
    auto touch_acc = [&]() {
#pragma unroll
        for (int i = 0; i < kI; i++)
#pragma unroll
            for (int p = 0; p < kP; p++)
#pragma unroll
                for (int h = 0; h < 2; h++) asm volatile("" : "+a"(acc[i][p][h]));
    };
    // Half a step: the matrix instructions of sub-step ks with, between them, the reads of the other slot from `st` (first, if
    // at all) and the copies of the half, evenly spread (a burst of copies holds up the instruction stream
    // behind it: the vector-memory path takes one of 1 KB about every 16 cycles).
    auto half = [&](auto ks_c, auto read_c, const char* st, auto&& copy, auto copies_c) {
        constexpr int ks = decltype(ks_c)::value, kCopies = decltype(copies_c)::value;
        constexpr int kPerSlot = (kReads + kMul - 1) / kMul;
#pragma unroll
        for (int n = 0; n < kMul; n++) {
            const int i = n / (2 * kP), r = n % (2 * kP), j = (i & 1) ? 2 * kP - 1 - r : r;  // back and forth: neighbours share an operand
            mfma(acc[i][j >> 1][j & 1], fb[ks][j >> 1][j & 1], fa[ks][i]);
            if constexpr (decltype(read_c)::value) {
#pragma unroll
                for (int q = n * kPerSlot; q < (n + 1) * kPerSlot; q++)
                    if (q < kReads) read_one(std::integral_constant<int, ks ^ 1>{}, q, st);
            }
#pragma unroll
            for (int c = 0; c < kCopies; c++)
                if ((c * kMul + kMul / 2) / (kCopies ? kCopies : 1) == n) copy(c);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using K0 = std::integral_constant<int, 0>;
    using K1 = std::integral_constant<int, 1>;
    auto none = [](int) {};
    touch_acc();
    asm volatile("s_nop 7" ::: "memory");

    if constexpr (kDirect) {
        const unsigned lds0 = (unsigned)(uintptr_t)LDS_PTR(char, smem);
        const char* zero16 = reinterpret_cast<const char*>(g_zero16);
        constexpr int kCopies = kAq + kBq;
        // copy c of the tile at as / bs into the stage at LDS address `stage`, skipped unless live > 0
        auto copy_at = [&](int c, unsigned stage, const char* as, const char* bs, int live) {
            const unsigned dst = stage + (c < kAq ? lds_w + c * 1024 : lds_wb + (c - kAq) * 1024);
            const unsigned off = c < kAq ? a_off[c < kAq ? c : 0] : b_off[c < kAq ? 0 : c - kAq];
            asm volatile("s_cmp_lt_i32 %3, 1\n\ts_cbranch_scc1 .Lskip%=\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n.Lskip%=:"
                         :
                         : "s"(dst), "v"(off), "s"(c < kAq ? as : bs), "s"(live)
                         : "m0", "scc");
        };
        // the partial last step: chunks whose k lies beyond K come from zeros (the lane hidden from the compiler: what only this
        // step needs is not kept)
        auto copy_ragged = [&](int kt, unsigned stage) {
            const char* as = a_base + (size_t)kt * 128;
            const char* bs = b_base + (size_t)kt * b_step;
            const int left = k_left - kt * 64;
            int l = lane;
            asm volatile("" : "+v"(l));
#pragma unroll
            for (int q = 0; q < kAq; q++) {
                const char* at = a_chunk(l, q) < left ? as + a_off[q] : zero16;
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(stage + lds_w + q * 1024), "v"(at) : "m0");
            }
#pragma unroll
            for (int q = 0; q < kBq; q++) {
                const char* at = b_chunk(l, q) < left ? bs + b_off[q] : zero16;
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(stage + lds_wb + q * 1024), "v"(at) : "m0");
            }
        };
#pragma unroll
        for (int t = 0; t < kStages; t++)
            if (t < KT) {
                if (ragged && t == KT - 1) copy_ragged(t, lds0 + t * kStage);
                else {
#pragma unroll
                    for (int c = 0; c < kCopies; c++) copy_at(c, lds0 + t * kStage, a_base + (size_t)t * 128, b_base + (size_t)t * b_step, 1);
                }
            }
        if (KT >= kStages) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((kStages - 1) * kCopies) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int n = 0; n < kReads; n++) read_one(K0{}, n, smem);
        // Step kt: its first half carries the second half of the copies of tile kt - 1 + kStages, which the barrier in the
        // middle of step kt - 1 made room for, its second half the first of those of tile kt + kStages.
        int slot = 0, prev = 0;
        int live = 0;  // > 0: there is such a tile
        const char *as = a_base + (size_t)kStages * 128, *bs = b_base + (size_t)kStages * b_step;  // tile kt + kStages
        const char *as_p = as, *bs_p = bs;                                                        // the one whose copies are under way
        for (int kt = 0; kt < KT; kt++) {
            const char* st = smem + slot * kStage;
            half(K0{}, std::true_type{}, st, [&](int c) { copy_at(kCopies / 2 + c, lds0 + prev * kStage, as_p, bs_p, live); }, std::integral_constant<int, kCopies / 2>{});
            if (kt + 1 == KT) break;
            // stage kt + 1 has landed (the copies of the kStages - 2 behind it may be in flight), and everyone has read stage kt
            if (kt + kStages <= KT) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((kStages - 2) * kCopies) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            live = __builtin_amdgcn_readfirstlane(KT - kStages - kt);
            if (ragged && kt + kStages == KT - 1) {
                copy_ragged(kt + kStages, lds0 + slot * kStage);
                live = 0;
            }
            prev = slot;
            as_p = as;
            bs_p = bs;
            slot = slot == kStages - 1 ? 0 : slot + 1;
            half(K1{}, std::true_type{}, smem + slot * kStage, [&](int c) { copy_at(c, lds0 + prev * kStage, as_p, bs_p, live); }, std::integral_constant<int, kCopies / 2>{});
            as += 128;
            bs += b_step;
        }
        half(K1{}, std::false_type{}, nullptr, none, std::integral_constant<int, 0>{});
    } else {
        // Through registers: chunks of 2-byte alignment.  In the partial last step a chunk that reaches past K is read where it ends at
        // K and moved down, so nothing behind a row is read; likewise the column chunks of a [K, N] operand at the edge of N.
        u32x4 ra[kAhead][kAq], rb[kAhead][kBq];
        auto load = [&](int set, int kt) {
            const char* as = a_base + (size_t)kt * 128;
            const char* bs = b_base + (size_t)kt * b_step;
            const int end = k_left - kt * 64 - 8;  // the last k at which a whole chunk begins: 56 and more but in the partial last step
#pragma unroll
            for (int q = 0; q < kAq; q++) {
                const int k = a_chunk(lane, q);
                ra[set][q] = *reinterpret_cast<const u32x4_any*>(as + a_off[q] + (k < end ? k : end) * 2);
            }
#pragma unroll
            for (int q = 0; q < kBq; q++) {
                const int k = b_chunk(lane, q);
                if constexpr (kBT) rb[set][q] = *reinterpret_cast<const u32x4_any*>(bs + b_off[q] + (k < end ? k : end) * 2);
                else rb[set][q] = *reinterpret_cast<const u32x4_any*>(bs + (int)b_off[q] - (k < end + 8 ? 0 : (long)(k - end - 7) * N * 2));
            }
        };
        const bool n_edge = !kBT && n0 + kTN > N;
        auto put = [&](int set, int kt, char* st) {
            if (ragged && kt == KT - 1) {
                const int end = k_left - kt * 64 - 8;
#pragma unroll
                for (int q = 0; q < kAq; q++) ra[set][q] = shift_elems(ra[set][q], a_chunk(lane, q) - end);
#pragma unroll
                for (int q = 0; q < kBq; q++) {
                    if constexpr (kBT) rb[set][q] = shift_elems(rb[set][q], b_chunk(lane, q) - end);
                    else if (b_chunk(lane, q) >= end + 8) rb[set][q] = u32x4{0u, 0u, 0u, 0u};
                }
            }
            if (n_edge) {
#pragma unroll
                for (int q = 0; q < kBq; q++) rb[set][q] = shift_elems(rb[set][q], b_back[q]);
            }
#pragma unroll
            for (int q = 0; q < kAq; q++) *LDS_PTR(u32x4, st + lds_w + q * 1024 + lane * 16) = ra[set][q];
#pragma unroll
            for (int q = 0; q < kBq; q++) *LDS_PTR(u32x4, st + lds_wb + q * 1024 + lane * 16) = rb[set][q];
        };
#pragma unroll
        for (int t = 0; t < kAhead; t++) load(t, t < KT ? t : KT - 1);
        put(0, 0, smem);
        load(0, kAhead < KT ? kAhead : KT - 1);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int n = 0; n < kReads; n++) read_one(K0{}, n, smem);
        for (int kt = 0; kt < KT; kt += kAhead) {
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                if (kt + u >= KT) break;
                const int cur = (kt + u) & 1;
                if (kt + u + 1 < KT) {
                    // (everyone has read the stage tile kt + u - 1 was in)
                    put((u + 1) % kAhead, kt + u + 1, smem + (cur ^ 1) * kStage);
                    const int t = kt + u + 1 + kAhead;
                    load((u + 1) % kAhead, t < KT ? t : KT - 1);
                }
                half(K0{}, std::true_type{}, smem + cur * kStage, none, std::integral_constant<int, 0>{});
                asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                half(K1{}, std::true_type{}, smem + (cur ^ 1) * kStage, none, std::integral_constant<int, 0>{});  // (behind the last tile: read and not used)
            }
        }
    }
    // the last matrix instructions' results have to have left the matrix pipe before the vector unit reads them
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    touch_acc();

    if constexpr (kEpilogue != kPlain) {
        // lane l: C[m = i * 16 + l % 16], columns 4 * (l / 16) + 0..3 of either half of a pair
        const int row_p = wm * kWM + (lane & 15), c4 = 4 * (lane >> 4);
        const bool rotated = kEpilogue == kRotate && n0 < rope.split;
#pragma unroll
        for (int i = 0; i < kI; i++) {
            const int row = m0 + row_p + i * 16;
            if (row >= M) continue;
            const size_t pos = rotated ? (size_t)(row % rope.seq) * 64 : 0;
#pragma unroll
            for (int p = 0; p < kP; p++) {
                const int pair = wn * kP + p;
                const f32x4 x = __builtin_convertvector(round_to_elem<false>(acc[i][p][0]), f32x4);
                const f32x4 y = __builtin_convertvector(round_to_elem<false>(acc[i][p][1]), f32x4);
                if constexpr (kEpilogue == kGate) {
                    const int F = N >> 1, col = n0 + pair * 16 + c4;
                    f32x4 o;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        // x * sigmoid(x) * y with sigmoid(x) = 1 / (1 + exp2(x * (-1 / ln 2)))
                        const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(x[e] * -1.4426950408889634f));
                        o[e] = x[e] * sg * y[e];
                    }
                    if (col < F) *reinterpret_cast<bf16x4*>(C + (size_t)row * F + col) = __builtin_convertvector(o, bf16x4);
                } else {
                    const int in_head = ((n0 & 127) >> 1) + pair * 16 + c4, col = (n0 & ~127) + in_head;
                    f32x4 first = x, second = y;
                    if (rotated) {
                        const f32x4 cs = *reinterpret_cast<const f32x4*>(rope.cos + pos + in_head), sn = *reinterpret_cast<const f32x4*>(rope.sin + pos + in_head);
                        first = x * cs + y * -sn;
                        second = y * cs + x * sn;
                    }
                    // rotated columns: row pitch `split`; those behind: a matrix of their own
                    const size_t ldc = rotated ? (size_t)rope.split : (size_t)(N - rope.split);
                    __bf16* at = (rotated ? C : static_cast<__bf16*>(rope.rest) - rope.split) + (size_t)row * ldc + col;
                    if (col < N) *reinterpret_cast<bf16x4*>(at) = __builtin_convertvector(first, bf16x4);
                    if (col + 64 < N) *reinterpret_cast<bf16x4*>(at + 64) = __builtin_convertvector(second, bf16x4);
                }
            }
        }
        return;
    }
    // With swapped operands lane l holds, in the eight registers of a pair, C[m = i * 16 + l % 16][n = pair * 32 + 8 * (l / 16) + 0..7].
    const int row_l = wm * kWM + (lane & 15), col_l = wn * kWN + 8 * (lane >> 4);
    if constexpr (kSplit) {
        float* Wt = W + ((size_t)blockIdx.z * gridDim.y + blockIdx.y) * (size_t)M * N;
#pragma unroll
        for (int i = 0; i < kI; i++)
#pragma unroll
            for (int p = 0; p < kP; p++) {
                const int row = m0 + row_l + i * 16, col = n0 + col_l + p * 32;
                if (row >= M) continue;
                float* at = Wt + (size_t)row * N + col;
                if (col + 8 <= N) {
                    *reinterpret_cast<f32x4_any*>(at) = acc[i][p][0];
                    *reinterpret_cast<f32x4_any*>(at + 4) = acc[i][p][1];
                } else {
#pragma unroll
                    for (int e = 0; e < 7; e++)
                        if (col + e < N) at[e] = acc[i][p][e >> 2][e & 3];
                }
            }
        return;
    }
    C += (size_t)blockIdx.y * M * N;
    if (R) R += (size_t)blockIdx.y * M * r_pitch;
#pragma unroll
    for (int i = 0; i < kI; i++)
#pragma unroll
        for (int p = 0; p < kP; p++) {
            const int row = m0 + row_l + i * 16, col = n0 + col_l + p * 32;
            if (row >= M) continue;
            const bf16x4 lo = round_to_elem<kF16>(acc[i][p][0]), hi = round_to_elem<kF16>(acc[i][p][1]);
            u32x4 v = __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            __bf16* at = C + (size_t)row * N + col;
            const __bf16* r = R + (size_t)row * r_pitch + col;
            if (col + 8 <= N) {
                if (R) {
                    const u32x4 add = *reinterpret_cast<const u32x4_any*>(r);
                    v = add_elems<kF16>(v, add);
                }
                *reinterpret_cast<u32x4_any*>(at) = v;
            } else if (col < N) {
                if (R) {
                    bf16x8 e8 = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
#pragma unroll
                    for (int e = 0; e < 7; e++)
                        if (col + e < N) e8[e] = r[e];
                    v = add_elems<kF16>(v, __builtin_bit_cast(u32x4, e8));
                }
                const bf16x8 e8 = __builtin_bit_cast(bf16x8, v);
#pragma unroll
                for (int e = 0; e < 7; e++)
                    if (col + e < N) at[e] = e8[e];
            }
        }
}

}  // namespace mrk::dev

namespace mrk {

namespace {
// The tiles and what one costs in us, fitted to 25000 timings of every tile and number of ranges over 950 shapes (10 to 12 % off,
// root mean square): start of a launch, step of K that waits for its data (any number of workgroups resident at
// once), step of one workgroup more on the same compute unit, start and end of a workgroup, TB/s of the operands, TB/s of what all
// tiles bring into the LDS.
struct Tile {
    int tm, tn, resident;  // resident: workgroups a compute unit holds
    double start, wait, step, edge, tbps, staged;
};
constexpr Tile kTiles[] = {
    {128, 128, 2, 0.63, 0.69, 0.45, 4.3, 4.9, 15.1},  // two stages: two workgroups share a compute unit
    {128, 128, 1, 1.3, 0.40, 0.41, 4.75, 5.0, 13.0},  // three stages
    {128, 64, 2, 2.7, 0.0, 0.31, 1.6, 5.5, 64.0},
    {64, 64, 3, 3.0, 0.24, 0.20, 0.64, 5.6, 21.5},
    {64, 64, 4, 2.4, 0.40, 0.27, 1.27, 50.0, 11.5},  // through registers
};
// The same with the gated or the rotary epilogue, where neither the depth nor the unevenness below is told apart: the choice against tiles of
// 256 x 256 (tiles256_us) is as good without (over the widths of decoder blocks; 0.46 of the time of those tiles alone, none
// slower by more than 12 % of 320).
constexpr Tile kPairedTiles[] = {
    {128, 128, 2, 2.7, 0.71, 0.50, 1.6, 5.7, 1e3},
    {128, 128, 1, 2.7, 0.31, 0.46, 1.6, 6.1, 1e3},
    {128, 64, 2, 3.0, 0.33, 0.29, 1.0, 6.0, 1e3},
    {64, 64, 3, 3.3, 0.26, 0.19, 0.4, 7.0, 1e3},
};
// The second launch of a split, in us: its start, per range, per MB of partial sums.  A split has to promise 4 % to be taken.
constexpr double kReduce = 2.5, kReduceRange = 0.25, kReduceMb = 0.06, kSplitGain = 1.04;
}  // namespace

MidPlan plan_mid(long M, long N, long K, long batch, bool whole_chunks, bool paired) {
    MidPlan best;
    if (M <= 0 || N < 8 || K < 8 || batch <= 0 || batch > 65535 || M > 0x7fffffffL || K > (1L << 23) || N > (1L << 24)) return best;
    const long kt = (K + 63) / 64;
    const double operands = 2.0 * batch * ((double)M * K + (double)N * K + (double)M * N) * 1e-6;
    // Long rows: each of a tile's is a page of its own, and workgroups that share an operand drift apart over many steps.  A step takes 10 %
    // longer per doubling of K, and the compute unit that holds the most workgroups ends last instead of the chip evening out
    // (376 tiles of 128 x 64: 1000 x 3000 x 2048 0.47 us a step; 308: 487 x 4920 x 13416 0.88).
    const double deep = paired || K <= 2048 ? 0.0 : K >= 11585 ? 2.5 : std::log2(K / 2048.0);
    for (int i = 0; i < (paired ? 4 : 5); i++) {
        if ((i == kMidUnaligned) == whole_chunks) continue;
        const Tile& t = paired ? kPairedTiles[i] : kTiles[i];
        const long tm = (M + t.tm - 1) / t.tm, tn = (N + t.tn - 1) / t.tn;
        // fewer than 2^32 work-items, 256 a tile, in the grid's first dimension (rotary: whole heads)
        if ((double)tm * (paired ? ((N + 127) / 128 * 128 + t.tn - 1) / t.tn : tn) > 0xffffff) continue;
        for (long want : {1L, 2L, 3L, 4L, 6L, 8L, 12L, 16L}) {
            if (want > 1 && (paired || kt < 10)) break;  // few steps are not split
            const long per = (kt + want - 1) / want, splits = (kt + per - 1) / per, groups = tm * tn * batch * splits;
            const double partial = 4.0 * splits * batch * M * N;
            // at least two steps a range; partial sums within the scratch of a call that must not allocate
            if (want > 1 && (splits != want || per < 2 || groups > 1024 || partial > (32 << 20))) continue;
            const long rounds = (groups + 255) / 256, waits = (groups + 256 * t.resident - 1) / (256 * t.resident);
            const double even = groups > 256 ? groups / 256.0 : 1.0, uneven = t.resident == 1 || deep > 2.16 ? 1.0 : paired ? 0.0 : 0.35 + 0.3 * deep;
            const double share = even + uneven * (rounds - even);
            double us = (t.wait * waits > t.step * share ? t.wait * waits : t.step * share) * per * (1.0 + 0.1 * deep) + t.edge * rounds;
            if (operands / t.tbps > us) us = operands / t.tbps;
            const double staged = 1e-6 * groups * per * (t.tm + t.tn) * 128;
            if (staged / t.staged > us) us = staged / t.staged;
            // operands that come from memory rather than from the L2s keep the two register sets waiting for longer (2 x 22088 x 3134 33 us
            // in one range of K, 26 in two)
            if (i == kMidUnaligned && operands > 32.0 && 0.49 * per * waits > us) us = 0.49 * per * waits;
            us += t.start;
            if (splits > 1) us = (us + kReduce + kReduceRange * splits + kReduceMb * partial * 1e-6) * kSplitGain;
            if (best.tile < 0 || us < best.us) best = MidPlan{i, splits, per, us};
        }
    }
    return best;
}

namespace {
// f(tile rows, tile columns, stages) of a tile as constants
template <class F>
void with_tile(int tile, F&& f) {
    using std::integral_constant;
    using I64 = integral_constant<int, 64>;
    using I128 = integral_constant<int, 128>;
    switch (tile) {
        case 0: f(I128{}, I128{}, integral_constant<int, 2>{}); break;
        case 1: f(I128{}, I128{}, integral_constant<int, 3>{}); break;
        case 2: f(I128{}, I64{}, integral_constant<int, 3>{}); break;
        default: f(I64{}, I64{}, integral_constant<int, 3>{}); break;
    }
}
}  // namespace

void mid_tile_shape(int tile, int* rows, int* cols, int* stages) {
    *rows = kTiles[tile].tm, *cols = kTiles[tile].tn;
    *stages = tile == kMidUnaligned || tile == 0 ? 2 : 3;
}

int launch_gemm_mid(hipStream_t s, const MidPlan& p, const void* A, const void* B, void* C, float* W, const void* add, long add_pitch, long M, long N, long K,
                    long batch, bool b_transposed, bool f16) {
    using namespace mrk::dev;
    if (p.tile < 0 || p.tile >= 5) return (int)hipErrorInvalidValue;
    const bool split = p.splits > 1;
    if (split && (!W || batch * p.splits > 65535)) return (int)hipErrorInvalidValue;
    const long tm = (M + kTiles[p.tile].tm - 1) / kTiles[p.tile].tm, tn = (N + kTiles[p.tile].tn - 1) / kTiles[p.tile].tn;
    const dim3 grid((unsigned)(tm * tn), (unsigned)batch, (unsigned)(split ? p.splits : 1));
    auto go = [&](auto tile_m, auto tile_n, auto ahead, auto direct) {
        constexpr int kTM = decltype(tile_m)::value, kTN = decltype(tile_n)::value, kAhead = decltype(ahead)::value;
        constexpr bool kDirect = decltype(direct)::value;
        auto pick = [&](auto bt, auto half) {
            constexpr bool kBT = decltype(bt)::value, kF16 = decltype(half)::value;
            auto kernel = split ? gemm_mid<kTM, kTN, kAhead, kBT, kF16, kDirect, true> : gemm_mid<kTM, kTN, kAhead, kBT, kF16, kDirect, false>;
            kernel<<<grid, 256, 0, s>>>(static_cast<const __bf16*>(A), static_cast<const __bf16*>(B), static_cast<__bf16*>(C), W,
                                        static_cast<const __bf16*>(add), (int)add_pitch, (int)M, (int)N, (int)K, (int)tm, (int)tn, (int)p.kt_per_split,
                                        MidRope{});
        };
        using T = std::true_type;
        using F = std::false_type;
        if (b_transposed) f16 ? pick(T{}, T{}) : pick(T{}, F{});
        else f16 ? pick(F{}, T{}) : pick(F{}, F{});
    };
    if (p.tile == kMidUnaligned) go(std::integral_constant<int, 64>{}, std::integral_constant<int, 64>{}, std::integral_constant<int, 2>{}, std::false_type{});
    else with_tile(p.tile, [&](auto tile_m, auto tile_n, auto stages) { go(tile_m, tile_n, stages, std::true_type{}); });
    return (int)hipGetLastError();
}

// The gated product C[M, N / 2] (rope null) or the rotated one C[M, rope->split].
int launch_gemm_mid_paired(hipStream_t s, int tile, const void* A, const void* B, void* C, long M, long N, long K, bool b_transposed,
                           const MidRope* rope) {
    using namespace mrk::dev;
    if (tile < 0 || tile >= kMidUnaligned || (rope && (rope->split % 128 || rope->seq <= 0))) return (int)hipErrorInvalidValue;
    const long tm = (M + kTiles[tile].tm - 1) / kTiles[tile].tm;
    // (a tile of 64 columns takes half of a head's pairs: the last head is covered whole)
    const long cols = rope ? (N + 127) / 128 * 128 : N, tn = (cols + kTiles[tile].tn - 1) / kTiles[tile].tn;
    with_tile(tile, [&](auto tile_m, auto tile_n, auto stages) {
        constexpr int kTM = decltype(tile_m)::value, kTN = decltype(tile_n)::value, kStages = decltype(stages)::value;
        auto kernel = rope ? (b_transposed ? gemm_mid<kTM, kTN, kStages, true, false, true, false, kRotate> : gemm_mid<kTM, kTN, kStages, false, false, true, false, kRotate>)
                           : (b_transposed ? gemm_mid<kTM, kTN, kStages, true, false, true, false, kGate> : gemm_mid<kTM, kTN, kStages, false, false, true, false, kGate>);
        kernel<<<dim3((unsigned)(tm * tn)), 256, 0, s>>>(static_cast<const __bf16*>(A), static_cast<const __bf16*>(B), static_cast<__bf16*>(C), nullptr, nullptr, 0,
                                                         (int)M, (int)N, (int)K, (int)tm, (int)tn, 0, rope ? *rope : MidRope{});
    });
    return (int)hipGetLastError();
}

}  // namespace mrk
