// 16-bit products on output tiles of 64 and 128 rows and columns: shapes whose 128 x 256 tiles (gemm_bf16.hip) would leave
// compute units without work, and operands whose rows start on any element, read as they are.
//
// What bounds it: with one workgroup on a compute unit, the instruction stream of its four waves.  A copy of 1 KB into the LDS waits for its
// turn on the vector-memory path (one takes 16 cycles, four waves ask at once), and the matrix instructions behind it wait as well: a K step
// of a 128 x 128 tile, 512 cycles of matrix instructions, 512 of copies and 512 of LDS reads, took 0.49 us (1170 cycles).  Above four steps of
// K (copies_apart), four more waves make the copies, two waves to a SIMD, and the four that multiply issue nothing else but their LDS reads: 0.38 to 0.42 us, and a
// launch starts 1 to 2 us sooner.  A ring of four or five stages changes neither (0.49 / 0.46 without such waves, 0.38 to 0.41 with them).  With several
// workgroups on a compute unit the path from the caches into the LDS bounds it (90 to 94 GB/s, 24 TB/s over the chip; profiles/gemm_mid_steps.txt), with
// or without them.  Tiles of 128 x 128 and more leave room for one workgroup: it takes its tiles in turn, and the next one's copies run under the stores
// of the last (against a workgroup to each tile, us: 1639 x 10368 x 416 on 128 x 128 31.2 -> 25.4, 791 x 9248 x 384 12.0 -> 10.7; on 256 x 128
// 1627 x 9296 x 320 19.9 -> 17.0, 4096 x 5632 x 512 35.3 -> 28.2).  A lane of 256 x 128 tiles has no registers left: 2 to 8 of its values, all of them
// of the stores and of what is set up before the first step, lie in scratch (up to 5 in the plain and the gated product); the K loop touches none.
// Hence smaller tiles for fewer rows and columns, K split over workgroups where even those are few, and the choice by an estimate of the
// time (plan_mid).
//
// us in a prepared plan against an [N, K] weight, two inputs in turn, without copying waves (large tiles in the last two) and now: 1024 x 1024 x 1024
// 7.2 / 6.3, 198 x 3072 x 1024 7.0 / 6.1, 1000 x 3000 x 2048 19.2 / 15.9, 3076 x 1024 x 1024 11.8 / 10.6, 512 x 8192 x 8192 76 to 79 / 73 to 74,
// 1639 x 10368 x 416 34.4 / 25.4, 1627 x 9296 x 320 24.2 / 17.3.
// On 128 x 256 tiles, split along K where that paid, padded copies of odd operands, and on these: 219 x 4288 x 3232 43.1 / 17.7, 700 x 700 x 4096
// 53.1 / 13.4, 75 x 1536 x 4576 18.7 / 10.7; odd: 300 x 3001 x 777 23.4 / 9.2, 5 x 7152 x 1638 27.8 / 10.3.
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
// kCopyWaves: eight waves, of which the last four make all copies; workgroups take tiles blockIdx.x, + gridDim.x, ... in turn (else one each).
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
template <int kTM, int kTN, int kAhead, bool kBT, bool kF16, bool kDirect, bool kSplit, MidEpilogue kEpilogue = kPlain, bool kCopyWaves = false>
__global__ __launch_bounds__(kCopyWaves ? 512 : 256, !kCopyWaves || kTM * kTN >= 128 * 128 ? 2 : kTM * kTN == 128 * 64 ? 4 : 6) void gemm_mid(
    const __bf16* __restrict__ A, const __bf16* __restrict__ B, __bf16* __restrict__ C, float* __restrict__ W, const __bf16* __restrict__ R,
    int r_pitch, int M, int N, int K, int tiles_m, int tiles_n, int kt_per_split, MidRope rope) {
    static_assert(kEpilogue == kPlain || (kDirect && !kSplit && !kF16), "the gated and the rotary epilogue: bf16, whole chunks, one range of K");
    constexpr int kWM = kTM / 2, kWN = kTN / 2, kI = kWM / 16, kP = kWN / 32;  // a wave's tile, its 16-row blocks and 32-column pairs
    constexpr int kAq = kTM / 32, kBq = kTN / 32;                             // 16-byte chunks per work-item and K step
    constexpr int kAStage = kTM * 128, kBStage = kTN * 128, kStage = kAStage + kBStage;
    constexpr int kStages = kDirect ? kAhead : 2;
    __shared__ __attribute__((aligned(1024))) char smem[kStages * kStage];
    const int tid = threadIdx.x, lane = tid & 63, wave_of_8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = kCopyWaves ? wave_of_8 & 3 : wave_of_8;
    const int wm = wave >> 1, wn = wave & 1;
    A += (size_t)blockIdx.y * M * K;
    B += (size_t)blockIdx.y * N * K;
    int m0, n0;  // (gated: n0 of the F columns; rotary: the first in the order below)
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

    auto at_tile = [&](int t) {
        int tile_m, tile_n;
        tile_of_block(t, tiles_m, tiles_n, &tile_m, &tile_n);
        m0 = tile_m * kTM;
        n0 = tile_n * (kEpilogue == kGate ? kTN / 2 : kTN);
    };

    // Sources.  A and B^T chunk q of a wave: eight rows of 128 bytes, LDS chunk lane % 8 of row lane / 8 holds the logical chunk of
    // the row's swizzle.  Rows beyond the edge are the last valid one (their products are not stored).
    const char *a_base, *b_base;
    const size_t b_step = kBT ? 128 : (size_t)N * 128;
    // first k of a lane's chunk q of A and of B inside a step (its k-row, [K, N] form)
    auto a_chunk = [&](int l, int q) { return ((l & 7) ^ (((wave * (kTM / 4) + q * 8 + (l >> 3)) >> 1) & 7)) * 8; };
    auto b_chunk = [&](int l, int q) {
        const int r = wave * (kTN / 4) + q * 8 + (l >> 3);
        return kBT ? ((l & 7) ^ (((r >> 1) & 1) | (((r >> 3) & 3) << 1))) * 8 : (wave * kBq + q) * (512 / kTN) + l / (kTN / 8);
    };
    unsigned a_off[kAq], b_off[kBq];  // byte offsets of the chunks from the bases of a step
    int b_back[kBq];                  // [K, N] form at the edge of N: elements by which a chunk was moved back to end at N
    auto sources = [&]() {
        a_base = reinterpret_cast<const char*>(A + (size_t)m0 * K + (size_t)kt0 * 64);
        // (paired columns are addressed from the first of B)
        const int b_first = kEpilogue == kPlain ? n0 : 0;
        b_base = kBT ? reinterpret_cast<const char*>(B + (size_t)b_first * K + (size_t)kt0 * 64)
                     : reinterpret_cast<const char*>(B + (size_t)kt0 * 64 * N + b_first);
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
    };
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
    auto clear_acc = [&]() {
#pragma unroll
        for (int i = 0; i < kI; i++)
#pragma unroll
            for (int p = 0; p < kP; p++)
#pragma unroll
                for (int h = 0; h < 2; h++) acc[i][p][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
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
    auto start_acc = [&]() {
        clear_acc();
        touch_acc();
        asm volatile("s_nop 7" ::: "memory");
    };
    // stores the tile at m0, n0
    auto finish = [&]() {
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
                            // (the product that is rounded is the sine's; on tiles of 256 x 256 it is in a quarter of the rows, and some 12 of a
                            // million results lie an ulp from these)
                            first = __builtin_elementwise_fma(x, cs, y * -sn);
                            second = __builtin_elementwise_fma(y, cs, x * sn);
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
        __bf16* Cb = C + (size_t)blockIdx.y * M * N;
        const __bf16* Rb = R + (size_t)blockIdx.y * M * r_pitch;
#pragma unroll
        for (int i = 0; i < kI; i++)
#pragma unroll
            for (int p = 0; p < kP; p++) {
                const int row = m0 + row_l + i * 16, col = n0 + col_l + p * 32;
                if (row >= M) continue;
                const bf16x4 lo = round_to_elem<kF16>(acc[i][p][0]), hi = round_to_elem<kF16>(acc[i][p][1]);
                u32x4 v = __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                __bf16* at = Cb + (size_t)row * N + col;
                const __bf16* r = Rb + (size_t)row * r_pitch + col;
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
    };
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
        if constexpr (kCopyWaves) {
            const int tiles = tiles_m * tiles_n;
            const int rounds = ((tiles - (int)blockIdx.x - 1) / (int)gridDim.x) + 1;
            if (wave_of_8 >= 4) {
                // The copying waves: one sequence of steps over all of the workgroup's tiles, up to kStages ahead of the multiplying waves.  Both
                // meet at one barrier a step.  (A copy that waits for an issue slot holds up all waves one step on: priority.)
                __builtin_amdgcn_s_setprio(1);
                const int total = rounds * KT;
                int t = blockIdx.x, kt = 0, slot = 0;
                const char *as, *bs;
                auto aim = [&]() {
                    at_tile(t);
                    sources();
                    as = a_base;
                    bs = b_base;
                };
                auto copy_step = [&]() {  // the step at (t, kt) into `slot`
                    if (ragged && kt == KT - 1) copy_ragged(kt, lds0 + slot * kStage);
                    else {
#pragma unroll
                        for (int c = 0; c < kCopies; c++) copy_at(c, lds0 + slot * kStage, as, bs, 1);
                    }
                    as += 128;
                    bs += b_step;
                    slot = slot == kStages - 1 ? 0 : slot + 1;
                    if (++kt == KT) {
                        kt = 0;
                        t += gridDim.x;
                        if (t < tiles) aim();
                    }
                };
                aim();
#pragma clang loop unroll(disable)
                for (int g = 0; g < kStages && g < total; g++) copy_step();
                if (total >= kStages) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((kStages - 1) * kCopies) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
                for (int g = 0; g + 1 < total; g++) {
                    // step g + 1 has landed (those behind it may be in flight), and everyone has read step g
                    if (g + kStages <= total) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"((kStages - 2) * kCopies) : "memory");
                    else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
                    if (g + kStages < total) copy_step();
                }
                return;
            }
            asm volatile("s_barrier" ::: "memory");
#pragma unroll
            for (int n = 0; n < kReads; n++) read_one(K0{}, n, smem);
            int slot = 0, left = rounds * KT;
            for (int r = 0; r < rounds; r++) {
                at_tile(blockIdx.x + r * gridDim.x);
                start_acc();
                for (int kt = 0; kt < KT; kt++) {
                    half(K0{}, std::true_type{}, smem + slot * kStage, none, std::integral_constant<int, 0>{});
                    // everyone has read this step, and the next one has landed (there is none behind the last: what is read then is not used)
                    if (--left) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    slot = slot == kStages - 1 ? 0 : slot + 1;
                    half(K1{}, std::true_type{}, smem + slot * kStage, none, std::integral_constant<int, 0>{});
                }
                finish();
            }
            return;
        }
        at_tile(blockIdx.x);
        sources();
        start_acc();
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
        int steps = KT;
        asm volatile("" : "+s"(steps));  // (kept from being tied to the tests above: the loop would be split up and its accumulators copied)
        int slot = 0, prev = 0;
        int live = 0;  // > 0: there is such a tile
        const char *as = a_base + (size_t)kStages * 128, *bs = b_base + (size_t)kStages * b_step;  // tile kt + kStages
        const char *as_p = as, *bs_p = bs;                                                        // the one whose copies are under way
        for (int kt = 0; kt + 1 < steps; kt++) {
            half(K0{}, std::true_type{}, smem + slot * kStage, [&](int c) { copy_at(kCopies / 2 + c, lds0 + prev * kStage, as_p, bs_p, live); }, std::integral_constant<int, kCopies / 2>{});
            // stage kt + 1 has landed (the copies of the kStages - 2 behind it may be in flight), and everyone has read stage kt
            if (kt + kStages <= steps) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((kStages - 2) * kCopies) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            live = __builtin_amdgcn_readfirstlane(steps - kStages - kt);
            if (ragged && kt + kStages == steps - 1) {
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
        half(K0{}, std::true_type{}, smem + slot * kStage, none, std::integral_constant<int, 0>{});
        half(K1{}, std::false_type{}, nullptr, none, std::integral_constant<int, 0>{});
    } else {
        // Through registers: chunks of 2-byte alignment.  In the partial last step a chunk that reaches past K is read where it ends at
        // K and moved down, so nothing behind a row is read; likewise the column chunks of a [K, N] operand at the edge of N.
        at_tile(blockIdx.x);
        sources();
        start_acc();
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
    if constexpr (!kCopyWaves) finish();
}

}  // namespace mrk::dev

namespace mrk {

namespace {
// Up to four steps of K the multiplying waves copy as well: 1.5 to 2.5 us of copies in flight hide nothing, and starting four more waves costs 0.15 to
// 0.25 us (541 x 1216 x 192 3.47 us / 3.73 with them, 567 x 512 x 256 3.65 / 3.81; 384 deep and more is faster with them).
constexpr long kFewSteps = 4;
// So they do up to eight steps on tiles of 64 x 64, and on more of those than compute units, which take the copies of one workgroup beside the steps of
// another anyway (without / with copying waves, us: 266 x 80 x 384 3.82 / 4.05, 806 x 984 x 384 4.26 / 4.44, 273 x 200 x 752 5.28 / 5.13, 2045 x 304 x 1384
// 7.6 / 7.1; 145 x 8392 x 384 4.85 / 5.20, 144 x 9392 x 2368 18.2 / 18.7; 21 such products 1.4 % faster without), and in ranges of K, whose
// workgroups are as many (23 products 1 to 4 % faster without: 1163 x 680 x 4512 19.7 / 20.2, 826 x 240 x 2080 8.7 / 8.9).
constexpr long kFewSteps64 = 8;
bool copies_apart(long rows, long cols, long groups, long kt, bool split) {
    if (rows == 256) return true;  // (built in this form alone)
    if (split || kt <= kFewSteps) return false;
    return rows * cols > 64 * 64 || (kt > kFewSteps64 && groups <= 256);
}
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
// 256 x 256 is as good without (over the widths of decoder blocks; 0.46 of the time of those tiles alone, none
// slower by more than 12 % of 320).  Of gated products up to four steps of K; of rotary products against 256 x 256 at any K (ranges_us).
constexpr Tile kPairedTiles[] = {
    {128, 128, 2, 2.7, 0.71, 0.50, 1.6, 5.7, 1e3},
    {128, 128, 1, 2.7, 0.31, 0.46, 1.6, 6.1, 1e3},
    {128, 64, 2, 3.0, 0.33, 0.29, 1.0, 6.0, 1e3},
    {64, 64, 3, 3.3, 0.26, 0.19, 0.4, 7.0, 1e3},
};
// The second launch of a split, in us: its start, per range, per MB of partial sums.  A split has to promise 4 % to be taken.
constexpr double kReduce = 2.5, kReduceRange = 0.25, kReduceMb = 0.06, kSplitGain = 1.04;

// Products in one range of K of more than four steps, whole chunks: what a pass of tiles takes, in us, fitted to 2800 timings over 1400 shapes
// of 17 to 8192 rows and 256 to 52000 columns (11 % off, root mean square; the tile chosen by it costs 0.5 % over the best of them, and 0.55
// of tiles of 128 x 256 alone).
// Start of a launch; a step of K on an empty chip, what a chip with a workgroup on each compute unit adds, and one more on
// the same compute unit (that one in parts: `whole` of it as soon as any compute unit has one); start and end of one more; the share a step
// grows by per doubling of K beyond 2048; TB/s of the operands behind the first 64 MB (40 x 33792 x 2112 on 64 x 64: 30.4 us, 25.7 on 128 x 256).
struct Timed {
    int tile, tm, tn;
    double start, step, full, layer, whole, edge, deep, tbps;
};
constexpr Timed kTimed[] = {
    {1, 128, 128, 4.0, 0.265, 0.178, 0.334, 0.7, 3.3, 0.055, 4.7},
    {2, 128, 64, 3.2, 0.202, 0.123, 0.259, 0.51, 1.0, 0.078, 4.7},
    {kMidSmallest, 64, 64, 2.9, 0.167, 0.070, 0.176, 0.35, 0.46, 0.092, 4.7},
    {kMidTall, 256, 128, 5.5, 0.449, 0.241, 0.0, 0.0, 0.0, 0.009, 4.7},  // (in one round)
};
constexpr Timed kTimed128x256 = {-1, 128, 256, 4.6, 0.508, 0.203, 0.0, 0.0, 0.0, 0.019, 7.0};  // (in one round)
double timed_us(const Timed& t, double groups, double kt, double K, double operands) {
    const double x = groups / 256, layers = std::ceil(x) - 1;
    const double step = t.step + t.full * (x < 1.0 ? x : 1.0) + t.layer * (layers * t.whole + (x > 1.0 ? x - 1.0 : 0.0) * (1.0 - t.whole));
    const double multiply = step * kt * (K > 2048 ? 1.0 + t.deep * std::log2(K / 2048) : 1.0), read = operands < 64.0 ? operands / 7.0 : 64.0 / 7.0 + (operands - 64.0) / t.tbps;
    return t.start + t.edge * layers + (multiply > read ? multiply : read);
}
// The same where more than 256 tiles of 128 x 256 exist: start of a launch, per round of 256 tiles its start and end and a step of K, what a
// step of the last round is shorter by where that is not full; TB/s of the operands.  Fitted to the 262 of those timings (10 % off): 0.967
// of the time of tiles of 256 x 256 alone (1639 x 10368 x 416 34.4 / 23.5 us), which win where K is long.
struct Rounds {
    int tile, tm, tn;
    double start, round, step, spare, tbps;
};
constexpr Rounds kRounds[] = {{1, 128, 128, 2.5, 1.6, 0.462, 0.276, 19.0}, {kMidTall, 256, 128, 2.3, 3.6, 0.721, 0.264, 14.9}};
constexpr Rounds kRounds256 = {-1, 256, 256, 0.0, 8.4, 1.268, 0.558, 6.2};
double rounds_us(const Rounds& t, double groups, double kt, double operands) {
    const double layers = std::ceil(groups / 256);
    const double us = t.start + layers * (t.round + kt * t.step) - t.spare * kt * (layers - groups / 256);
    return us > t.start + operands / t.tbps ? us : t.start + operands / t.tbps;
}
double operand_mb(long M, long N, long K, long batch) { return 2e-6 * batch * ((double)M * K + (double)N * K + (double)M * N); }
}  // namespace

double large_pass_us(long M, long N, long K, long batch) {
    if (mid_many_tiles(M, N, batch))
        return rounds_us(kRounds256, (double)(((M + 255) / 256) * ((N + 255) / 256) * batch), (double)((K + 63) / 64), operand_mb(M, N, K, batch));
    return timed_us(kTimed128x256, (double)(((M + 127) / 128) * ((N + 255) / 256) * batch), (double)((K + 63) / 64), (double)K, operand_mb(M, N, K, batch));
}

MidPlan plan_mid(long M, long N, long K, long batch, bool whole_chunks, bool paired) {
    MidPlan best;
    if (M <= 0 || N < 8 || K < 8 || batch <= 0 || batch > 65535 || M > 0x7fffffffL || K > (1L << 23) || N > (1L << 24)) return best;
    const long kt = (K + 63) / 64;
    const double operands = operand_mb(M, N, K, batch);
    // Long rows: each of a tile's is a page of its own, and workgroups that share an operand drift apart over many steps.  A step takes 10 %
    // longer per doubling of K, and the compute unit that holds the most workgroups ends last instead of the chip evening out
    // (376 tiles of 128 x 64: 1000 x 3000 x 2048 0.47 us a step; 308: 487 x 4920 x 13416 0.88).
    const double deep = paired || K <= 2048 ? 0.0 : K >= 11585 ? 2.5 : std::log2(K / 2048.0);
    for (int i = 0; i < (paired ? 4 : 5); i++) {
        if ((i == kMidUnaligned) == whole_chunks) continue;
        const Tile& t = paired ? kPairedTiles[i] : kTiles[i];
        const long tm = (M + t.tm - 1) / t.tm, tn = (N + t.tn - 1) / t.tn;
        // fewer than 2^32 work-items, up to 512 a tile, in the grid's first dimension (rotary: whole heads)
        if ((double)tm * (paired ? ((N + 127) / 128 * 128 + t.tn - 1) / t.tn : tn) > 0x7fffff) continue;
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
            if (best.tile < 0 || us < best.us) best = MidPlan{i, splits, per, us, us};
        }
    }
    // How many ranges K is summed in is a matter of the estimates above alone: it decides the bits.
    if (best.tile < 0 || best.splits > 1 || !whole_chunks || !mid_pipelined(N, K)) return best;
    const double ranges_us = best.us;
    best = MidPlan();
    const bool many = mid_many_tiles(M, N, batch);
    auto consider = [&](const auto& t, auto&& estimate) {
        const long cols = paired ? (N + 127) / 128 * 128 : N, groups = ((M + t.tm - 1) / t.tm) * ((cols + t.tn - 1) / t.tn);
        if ((double)groups > 0x7fffff || (!many && t.tile == kMidTall && (!paired || groups * batch > 256))) return;  // (the plain product has tiles of 128 x 256)
        const double us = estimate(t, (double)groups * batch);
        if (best.tile < 0 || us < best.us) best = MidPlan{t.tile, 1, kt, us, ranges_us};
    };
    if (many) for (const Rounds& t : kRounds) consider(t, [&](const Rounds& r, double groups) { return rounds_us(r, groups, (double)kt, operands); });
    else for (const Timed& t : kTimed) consider(t, [&](const Timed& r, double groups) { return timed_us(r, groups, (double)kt, (double)K, operands); });
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
        case kMidTwoStages: f(I128{}, I128{}, integral_constant<int, 2>{}); break;
        case kMidThreeStages: f(I128{}, I128{}, integral_constant<int, 3>{}); break;
        case 2: f(I128{}, I64{}, integral_constant<int, 3>{}); break;
        case kMidTall: f(integral_constant<int, 256>{}, I128{}, integral_constant<int, 3>{}); break;
        default: f(I64{}, I64{}, integral_constant<int, 3>{}); break;
    }
}
}  // namespace

void mid_tile_shape(int tile, int* rows, int* cols, int* stages) {
    if (tile == kMidTall) {
        *rows = 256, *cols = 128, *stages = 3;
        return;
    }
    *rows = kTiles[tile].tm, *cols = kTiles[tile].tn;
    *stages = tile == kMidUnaligned || tile == 0 ? 2 : 3;
}

int launch_gemm_mid(hipStream_t s, const MidPlan& p, const void* A, const void* B, void* C, float* W, const void* add, long add_pitch, long M, long N, long K,
                    long batch, bool b_transposed, bool f16) {
    using namespace mrk::dev;
    if (p.tile < 0 || p.tile > kMidTall) return (int)hipErrorInvalidValue;
    const bool split = p.splits > 1;
    if (split && (!W || batch * p.splits > 65535 || p.tile == kMidTall)) return (int)hipErrorInvalidValue;  // (256 x 128: one range of K)
    int rows = 0, cols = 0, stages = 0;
    mid_tile_shape(p.tile, &rows, &cols, &stages);
    const long tm = (M + rows - 1) / rows, tn = (N + cols - 1) / cols;
    const dim3 grid((unsigned)(tm * tn), (unsigned)batch, (unsigned)(split ? p.splits : 1));
    auto go = [&](auto tile_m, auto tile_n, auto ahead, auto direct) {
        constexpr int kTM = decltype(tile_m)::value, kTN = decltype(tile_n)::value, kAhead = decltype(ahead)::value;
        constexpr bool kDirect = decltype(direct)::value;
        auto pick = [&](auto bt, auto half) {
            constexpr bool kBT = decltype(bt)::value, kF16 = decltype(half)::value;
            // (tiles of 128 x 128 and more, one workgroup to a compute unit, are taken in turn)
            constexpr bool kMay = kDirect && kAhead == 3, kAlways = kTM == 256;
            const bool copy_waves = kMay && copies_apart(kTM, kTN, tm * tn * batch, (K + 63) / 64, split);
            auto of = [&](auto waves) {
                constexpr bool kWaves = decltype(waves)::value;
                auto whole = gemm_mid<kTM, kTN, kAhead, kBT, kF16, kDirect, false, kPlain, kWaves>;
                if constexpr (kWaves) return whole;
                else return split ? gemm_mid<kTM, kTN, kAhead, kBT, kF16, kDirect, true> : whole;
            };
            auto kernel = copy_waves ? of(std::integral_constant<bool, kMay>{}) : of(std::integral_constant<bool, kAlways>{});
            const bool in_turn = copy_waves && kTM * kTN >= 128 * 128 && !split && batch == 1 && tm * tn > 256;
            kernel<<<in_turn ? dim3(256) : grid, copy_waves ? 512 : 256, 0, s>>>(static_cast<const __bf16*>(A), static_cast<const __bf16*>(B), static_cast<__bf16*>(C), W,
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
    if (tile < 0 || tile > kMidTall || tile == kMidUnaligned || (rope && (rope->split % 128 || rope->seq <= 0))) return (int)hipErrorInvalidValue;
    int rows = 0, width = 0, stages = 0;
    mid_tile_shape(tile, &rows, &width, &stages);
    const long tm = (M + rows - 1) / rows;
    // (a tile of 64 columns takes half of a head's pairs: the last head is covered whole)
    const long cols = rope ? (N + 127) / 128 * 128 : N, tn = (cols + width - 1) / width;
    with_tile(tile, [&](auto tile_m, auto tile_n, auto stages) {
        constexpr int kTM = decltype(tile_m)::value, kTN = decltype(tile_n)::value, kStages = decltype(stages)::value;
        constexpr bool kMay = kStages == 3, kAlways = kTM == 256;
        const bool copy_waves = kMay && copies_apart(kTM, kTN, tm * tn, (K + 63) / 64, false), in_turn = copy_waves && kTM * kTN >= 128 * 128 && tm * tn > 256;
        auto of = [&](auto waves) {
            constexpr bool kWaves = decltype(waves)::value;
            return rope ? (b_transposed ? gemm_mid<kTM, kTN, kStages, true, false, true, false, kRotate, kWaves> : gemm_mid<kTM, kTN, kStages, false, false, true, false, kRotate, kWaves>)
                        : (b_transposed ? gemm_mid<kTM, kTN, kStages, true, false, true, false, kGate, kWaves> : gemm_mid<kTM, kTN, kStages, false, false, true, false, kGate, kWaves>);
        };
        auto kernel = copy_waves ? of(std::integral_constant<bool, kMay>{}) : of(std::integral_constant<bool, kAlways>{});
        kernel<<<dim3(in_turn ? 256u : (unsigned)(tm * tn)), copy_waves ? 512 : 256, 0, s>>>(static_cast<const __bf16*>(A), static_cast<const __bf16*>(B), static_cast<__bf16*>(C), nullptr, nullptr, 0,
                                                         (int)M, (int)N, (int)K, (int)tm, (int)tn, 0, rope ? *rope : MidRope{});
    });
    return (int)hipGetLastError();
}

}  // namespace mrk
