// bf16 GEMM for gfx950: C[M,N] = A[M,K] * B[K,N], row-major bf16 in, f32 accumulate on
// MFMA, one round-to-nearest-even to bf16 at the end.
//
// Stands for the lazy graph of Tensor::matmul on bf16 operands
// (tensor/src/matmul.rs:82-110: broadcast multiply then sum(-1) with the accumulator
// promoted to f32, tensor/src/reduce.rs:101-117, cast back 665-691) after the tensor-core
// rewrite (schedule/src/optimizer/tc.rs:36-94 strips the CAST around the product, so
// exact bf16*bf16 products are accumulated in f32).  The instruction is the 16x16x32 shape the
// reference names in its CDNA table (schedule/src/optimizer/renderer.rs:549-558,724-733): of
// the two bf16 shapes of gfx950 it is the one the part sustains the higher clock on (it moves
// less accumulator data per product than 32x32x16; 1.96 against 1.72 PFLOP/s from registers).
//
// Main kernel: 256x256 output tile per workgroup of 4 waves (2x2), each wave 128x128 =
// 8x8 MFMA tiles (256 accumulator registers), K step 64 = two 32-deep sub-steps.  Tiles travel
// global -> LDS directly (global_load_lds, 16 B per lane, no register staging).  A is kept in LDS
// row-major with an XOR swizzle of its 16-byte chunks, B row-major (n contiguous) with
// an XOR swizzle of its 32-byte granules and read through the transposing LDS load,
// which hands each lane the 4 consecutive-k values of its column.  The MFMA is issued with
// swapped operands (D' = B^T A^T) so each lane ends up with 4 consecutive n of one row,
// which makes the epilogue 8-byte LDS writes and 16-byte coalesced global stores.  A second
// operand stored as B^T [N, K] (k contiguous: a Linear layer's weight) is staged and read
// exactly like A instead.
//
// Pipeline.  The vector-memory path takes a 1 KB copy every ~16 cycles, so the 64 copies a
// workgroup issues per K step need about half of the step's MFMA time; issued in one burst
// they stall the waves' instruction streams behind them.  They are therefore spread evenly,
// four per 32-MFMA phase and wave: the LDS holds two A stages and three B stages (160 KB, all
// of it), the copies of B tile kt+2 go out during the first two phases of tile kt into the
// stage tile kt-1 left, the one barrier of the step sits in the middle of it, and the copies
// of A tile kt+2 follow in the last two phases into the stage tile kt has just left.  For the
// barrier to sit there every fragment of tile kt must have been read by then: fragments are
// read a sub-step ahead of their MFMAs into two register slots (one per 32-deep sub-step).
//
// Shapes.  Any M, N and K: edge tiles redirect out-of-range rows and column chunks to the last
// valid one and mask their stores; a partial last K step is copied from zeros beyond K.  The
// 16-byte copies need operand rows that start on 16 bytes: an operand whose row length is no
// multiple of 8 elements is first written out with padded rows (gemm_repitch), and C, whose rows
// cannot be padded, is stored with 16-byte stores of 2-byte alignment.  A second instance of the
// same body with a 128x256 workgroup tile serves shapes that would otherwise leave most compute
// units idle; a leading batch dimension runs as grid.y.  The kernel at the end of this file, one
// wave per 32x32 tile straight from global memory, is left for fewer than eight columns or a K below eight, and for sums in several
// ranges of K without scratch.  Shapes of up to 256 tiles of 128x256 mostly run on smaller tiles (gemm_mid.hip, route_16bit).
#include <hip/hip_runtime.h>
#include <atomic>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "gemm_elem.h"
#include "gemm_mid.h"
#include "kernels.h"

namespace mrk::dev {

constexpr int kBM = 256, kBN = 256, kBK = 64;
constexpr int kBStageSw = kBK * kBN * 2;       // 32768 B per B stage, row pitch 512 B, granule-swizzled
// (an A stage is rows x 128 B, chunk-swizzled: 32768 B for the 256-row tile, which with two A
// and three B stages fills all 160 KB of the LDS)

// kAny: K is not a multiple of 64, or N not of 8.  The copies of a partial last K step use
// per-lane 64-bit addresses so that chunks beyond K can be redirected to g_zero16: zero
// operands on both sides contribute nothing.  Every other step is copied as in the full case.
// The operands have row pitches of their own (lda, ldb elements, multiples of 8, zeros from K on
// inside a row's padding), and C and R rows may start on any element: they are accessed in
// 16-byte pieces of 2-byte alignment, the last piece of a row element by element.
//
// kJ: 32-column blocks (two MFMA tile columns each) per wave.  kJ = 4: 256x256 workgroup tile, waves 2x2, each 128x128.
// kJ = 2: 128x256 workgroup tile, waves 1x4, each 128x64 (half the accumulators, an A stage of
// half the size, the same B stages and pipeline) for shapes whose 256x256 tiles would leave
// most compute units without work.
//
// kSplitK: blockIdx.z selects a range of `kt_per_split` K steps; the workgroup writes its f32
// partial tile to W[z][batch][M][N] instead of C and gemm_splitk_reduce adds the partials up in
// a fixed order.  For shapes with so few tiles that the K loop itself has to be spread over
// the chip (a handful of rows against a large weight matrix).
//
// kResidual: the epilogue adds a bf16 matrix R of C's shape to the rounded product,
// C = bf16(float(bf16(A B)) + float(R)): the bits of the product kernel followed by an
// elementwise add, without writing and re-reading the product.
//
// kBT: the second operand is stored as B^T [N, K] (k contiguous).  Its stage holds 256 n-rows of
// 128 B, chunk-swizzled, copied and read like an A stage: one 16-byte read per fragment instead of
// two transposing 8-byte reads.  Same products in the same order: the same bits as the [K, N] form.
//
// kSwiGLU (256-row tile only): B is [K, 2F] holding a gate matrix in its columns [0, F) and an up
// matrix in [F, 2F) (N = 2F is B's row pitch); the workgroup's 256 tile columns are 128 gate
// columns followed by the 128 up columns at the same offset, and the epilogue writes
// C[M, F] = bf16(silu(float(bf16(A gate))) * float(bf16(A up))): the two products rounded to bf16
// as separate kernels would leave them, then x * sigmoid(x) * y in f32 with one rounding, without
// the 2F-wide product ever reaching memory.
//
// kF16: the operands and the result are IEEE half precision instead of bf16
// (v_mfma_f32_16x16x32_f16: the f16 entry of the reference's CDNA4 table,
// schedule/src/optimizer/renderer.rs:724-733).  Both are 16-bit elements, so copies, LDS layout,
// fragment reads and stores are the same bytes; only the matrix instruction and the conversion of
// the f32 accumulators differ.  The element pointers stay typed as 16-bit carriers.
//
// kRope (256-row tile only): the product of a packed projection whose first `split` columns are
// attention heads of 128 columns each (q | k of a fused QKV product).  The epilogue applies the
// rotary embedding (non-interleaved form, tensor/src/transformer.rs:32-69) to those heads on the
// bf16-rounded product, as the separate kernel would: with x1 = columns 0..63 and x2 = columns
// 64..127 of a head, out = [x1 cos - x2 sin | x1 sin + x2 cos] in f32 and one rounding, cos / sin
// [seq, 64] f32 indexed by the row's position (row % seq).  A wave's 128 columns are exactly one
// head, so both halves of a pair sit in the tile row the wave has just staged.  The rotated
// columns go to C with a row pitch of `split`; the columns behind them (v) go, unrotated, to a
// second matrix of their own with a row pitch of N - split.
struct RopeEpilogue {
    const float* cos;
    const float* sin;
    __bf16* rest;  // [M, N - split]: the columns from `split` on
    int seq, split;
};
template <bool kAny, int kJ, bool kSplitK = false, bool kResidual = false, bool kSwiGLU = false, bool kBT = false, bool kF16 = false,
          bool kRope = false>
__device__ __forceinline__ void gemm_tile_body(const __bf16* __restrict__ A, const __bf16* __restrict__ B,
                                               __bf16* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n,
                                               float* __restrict__ W = nullptr, int kt_per_split = 0,
                                               const __bf16* __restrict__ R = nullptr, const RopeEpilogue& rope = RopeEpilogue{},
                                               int ldr = -1, int lda = 0, int ldb = 0) {
    static_assert(!kF16 || (!kSwiGLU && !kRope), "the gated and the rotary epilogue exist for bf16 only");
    static_assert(!kRope || (kJ == 4 && !kSplitK && !kResidual && !kSwiGLU), "the rotary epilogue exists for the plain 256-row tile only");
    constexpr int kTM = kJ == 4 ? 256 : 128;      // rows of the workgroup tile
    constexpr int kAq = kTM / 32;                 // 1 KB A chunks (8 rows) each wave copies per K step
    constexpr int kAStageT = kTM * kBK * 2;       // bytes of an A stage
    constexpr int kCPitchT = kJ * 64 + 16;        // epilogue staging pitch per wave
    constexpr int kCWaveT = 128 * kCPitchT;
    constexpr int kSmemMainT = 2 * kAStageT + 3 * kBStageSw;
    constexpr int kSmemT = 4 * kCWaveT > kSmemMainT ? 4 * kCWaveT : kSmemMainT;
    constexpr int kI16 = 8, kJ16 = 2 * kJ;        // 16x16 MFMA tiles per wave: rows, columns
    constexpr int kSlots = 4 * kJ16;              // MFMAs per phase (four tile rows x all tile columns)
    // A stage: kTM rows x 128 B, 16 B chunks XOR-swizzled by ((row >> 1) & 7);
    // B stage: 64 k-rows x 512 B, 32 B granules XOR-swizzled by (k & 3).
    __shared__ __attribute__((aligned(1024))) char smem[kSmemT];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = kJ == 4 ? wave >> 1 : 0, wn = kJ == 4 ? (wave & 1) : wave;
    // row pitches of the operands in elements
    const size_t a_pitch = kAny ? (size_t)lda : (size_t)K;
    const size_t b_pitch = kAny ? (size_t)ldb : kBT ? (size_t)K : (size_t)N;
    // blockIdx.y: which of the back-to-back stored products
    A += (size_t)blockIdx.y * M * a_pitch;
    B += (size_t)blockIdx.y * (kBT ? N : K) * b_pitch;
    if (!kSplitK) C += (size_t)blockIdx.y * M * N;
    // row pitch of R in elements: N for a matrix of C's shape, 0 for one row added to every row of C (a bias)
    const size_t r_pitch = ldr < 0 ? (size_t)N : (size_t)ldr;
    if (kResidual) R += (size_t)blockIdx.y * M * r_pitch;
    int tile_m, tile_n;
    tile_of_block(blockIdx.x, tiles_m, tiles_n, &tile_m, &tile_n);
    static_assert(!kSwiGLU || (kJ == 4 && !kSplitK && !kResidual), "the gated epilogue exists for the 256-row tile only");
    const size_t m0 = (size_t)tile_m * kTM, n0 = (size_t)tile_n * (kSwiGLU ? kBN / 2 : kBN);
    char* sA0 = smem;                 // two A stages
    char* sB0 = smem + 2 * kAStageT;  // three B stages

    // ---- direct global -> LDS copies: each wave moves kAq KB of A and 8 KB of B per tile,
    // one instruction = 64 lanes x 16 B = 1 KB of contiguous LDS.
    // A chunk q (1 KB = 8 rows): lane -> row q*8 + lane/8, LDS chunk lane%8 holds logical
    // chunk (lane%8) ^ ((row >> 1) & 7).  The LDS serves 16 lanes x 16 B per cycle over 64
    // banks; with 128 B rows this swizzle puts 16 consecutive rows of one logical chunk
    // into 16 different 16 B slots.  ((row >> 1) & 7 depends on the parity of q: two variants.)
    // B chunk q (1 KB = 2 k-rows): lane -> k-row q*2 + lane/32, LDS 16 B chunk lane%32 ->
    // granule (lane%32)/2 ^ (krow & 3).
    // Ragged edges: a tile may reach past row M or column N.  Source rows / column chunks
    // beyond the edge are redirected to the last valid one (the duplicates only feed outputs
    // the epilogue does not store), which costs nothing per K step: the redirected offsets do
    // not depend on it.  N % 8 == 0 keeps the redirected chunk 16-byte aligned.
    unsigned a_voff[kAq];
#pragma unroll
    for (int q = 0; q < kAq; q++) {
        size_t row = m0 + wave * (kAq * 8) + q * 8 + (lane >> 3);
        row = row < (size_t)M ? row : (size_t)M - 1;
        const int chunk = (lane & 7) ^ ((q & 1) * 4 + (lane >> 4));
        a_voff[q] = (unsigned)(((row - m0) * a_pitch + (chunk << 3)) * 2);
    }
    const int b_h = lane & 1, b_g = (lane & 31) >> 1, b_r = lane >> 5;
    // kBT: B^T chunk q (1 KB = 8 n-rows of 128 B), copied and swizzled exactly like an A chunk;
    // each wave moves the 64 rows wave*64 .. wave*64+63 of the stage.
    unsigned bt_voff[kBT ? 8 : 1];
    if constexpr (kBT) {
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const size_t lr = wave * 64 + q * 8 + (lane >> 3);  // row inside the 256-row stage
            size_t row;
            if (kSwiGLU) {
                // stage rows 0..127 are gate rows of B^T, 128..255 the up rows at the same offset
                const size_t F = (size_t)N / 2, half = lr >> 7;
                row = n0 + (lr & 127);
                row = (row < F ? row : F - 1) + half * F;
            } else {
                row = n0 + lr;
                row = row < (size_t)N ? row : (size_t)N - 1;
            }
            const int chunk = (lane & 7) ^ ((q & 1) * 4 + (lane >> 4));
            bt_voff[q] = (unsigned)(((row - n0) * b_pitch + (chunk << 3)) * 2);
        }
    }
    unsigned b_voff[2];
#pragma unroll
    for (int par = 0; par < 2; par++) {
        size_t col = n0 + ((((b_g ^ (par * 2 + b_r)) << 1) | b_h) << 3);
        if (kSwiGLU) {
            // tile columns 0..127 come from the gate half of B, 128..255 from the up half
            const size_t F = (size_t)N / 2, lc = col - n0, half = lc >> 7;
            col = n0 + (lc & 127);
            col = (col + 8 <= F ? col : F - 8) + half * F;
        } else {
            col = col + 8 <= b_pitch ? col : b_pitch - 8;
        }
        b_voff[par] = (unsigned)(((size_t)(wave * 16 + b_r) * b_pitch + (col - n0)) * 2);
    }
    const int KT_all = (K + kBK - 1) / kBK;
    const int kt0 = kSplitK ? (int)blockIdx.z * kt_per_split : 0;  // first K step of this workgroup
    const int KT = kSplitK ? (KT_all - kt0 < kt_per_split ? KT_all - kt0 : kt_per_split) : KT_all;
    const bool has_last = kt0 + KT == KT_all;  // the (possibly partial) last K step is in this range
    const char* a_tile = reinterpret_cast<const char*>(A + m0 * a_pitch) + (size_t)kt0 * kBK * 2;
    const char* b_tile = kBT ? reinterpret_cast<const char*>(B + n0 * b_pitch) + (size_t)kt0 * kBK * 2
                             : reinterpret_cast<const char*>(B + n0) + (size_t)kt0 * kBK * b_pitch * 2;
    const unsigned lds_a = (unsigned)(uintptr_t)LDS_PTR(char, sA0) + wave * (kAq * 1024);
    const unsigned lds_b = (unsigned)(uintptr_t)LDS_PTR(char, sB0) + wave * 8192;
    // One direct copy: 64 lanes x 16 B land at LDS [m0, m0 + 1 KB); the compiler is not told
    // about it (it would otherwise wait for the copy before every later LDS read), so the
    // waits are explicit in the barriers below.
    auto dma = [&](unsigned lds_addr, unsigned voff, const char* sbase) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(lds_addr), "v"(voff), "s"(sbase)
                     : "m0");
    };
    auto dma_from = [&](unsigned lds_addr, const char* addr) {  // per-lane 64-bit source address
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_addr), "v"(addr) : "m0");
    };
    const int k_last = K - (KT_all - 1) * kBK;  // depth of the last K step: 64, or 1..63
    const char* zero16 = reinterpret_cast<const char*>(g_zero16);
    // (stage_off: byte offset of the stage inside the A or B part of the LDS)
    auto dma_a = [&](int q, int kt, unsigned stage_off) {
        if (kAny && has_last && kt == KT - 1) {
            const int chunk = (lane & 7) ^ ((q & 1) * 4 + (lane >> 4));  // logical 8-deep k chunk of this lane
            dma_from(lds_a + stage_off + q * 1024,
                     chunk * 8 < k_last ? a_tile + (size_t)kt * kBK * 2 + a_voff[q] : zero16);
        } else {
            dma(lds_a + stage_off + q * 1024, a_voff[q], a_tile + (size_t)kt * kBK * 2);
        }
    };
    auto dma_b = [&](int q, int kt, unsigned stage_off) {
        if constexpr (kBT) {
            if (kAny && has_last && kt == KT - 1) {
                const int chunk = (lane & 7) ^ ((q & 1) * 4 + (lane >> 4));
                dma_from(lds_b + stage_off + q * 1024,
                         chunk * 8 < k_last ? b_tile + (size_t)kt * kBK * 2 + bt_voff[q] : zero16);
            } else {
                dma(lds_b + stage_off + q * 1024, bt_voff[q], b_tile + (size_t)kt * kBK * 2);
            }
            return;
        }
        if (kAny && has_last && kt == KT - 1) {
            dma_from(lds_b + stage_off + q * 1024,
                     wave * 16 + q * 2 + b_r < k_last ? b_tile + ((size_t)kt * kBK + q * 2) * b_pitch * 2 + b_voff[q & 1] : zero16);
            return;
        }
        dma(lds_b + stage_off + q * 1024, b_voff[q & 1], b_tile + ((size_t)kt * kBK + q * 2) * b_pitch * 2);
    };

    f32x4 acc[kI16][kJ16];
#pragma unroll
    for (int i = 0; i < kI16; i++)
#pragma unroll
        for (int j = 0; j < kJ16; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][j][e] = 0.0f;

    // lane-constant parts of the fragment addresses.  An operand fragment of the 16x16x32 MFMA is
    // row (lane % 16) of a 16-row tile, k = 8 * (lane / 16) .. +7 of the 32-deep sub-step.
    const int a_base_l = (wm * 128 + (lane & 15)) * 128;  // + i*2048
    int a_xo[2];
#pragma unroll
    for (int ks = 0; ks < 2; ks++) a_xo[ks] = ((ks * 4 + (lane >> 4)) ^ ((lane >> 1) & 7)) << 4;
    // B through the transposing read: 16-lane block b = lane / 16 covers k-rows 8b .. 8b+7 (two
    // reads of four rows), lane j' of the block points at k-row j'/4, 8-byte unit j'%4 of the
    // 32-byte granule (16 columns) of its tile column
    const int b_rr = (lane & 15) >> 2;
    const int b_row_l = (8 * (lane >> 4) + b_rr) * 512 + 8 * (lane & 3) + ((wn * kJ16) << 5);  // + ks*32*512 (+ 4*512: second read)
    int b_p[4];  // tile column j: b_p[j & 3] + (j >> 2) * 128
#pragma unroll
    for (int q = 0; q < 4; q++) b_p[q] = b_row_l + ((q ^ b_rr) << 5);
    const int bt_base_l = (wn * (kJ * 32) + (lane & 15)) * 128;  // kBT: + j*2048, chunk offset a_xo[ks]

    bf16x8 fa[2][kI16], fb[2][kJ16];  // fragment slot = 32-deep sub-step
    // all but this wave's newest 8 copies (the B chunks issued since the last barrier) have
    // landed, its LDS reads are complete; then all waves meet
    auto tile_barrier = [&]() { asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    auto full_barrier = [&]() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

#pragma unroll
    for (int q = 0; q < kAq; q++) dma_a(q, 0, 0);
#pragma unroll
    for (int q = 0; q < 8; q++) dma_b(q, 0, 0);
#pragma unroll
    for (int q = 0; q < kAq; q++) dma_a(q, KT > 1 ? 1 : 0, kAStageT);
#pragma unroll
    for (int q = 0; q < 8; q++) dma_b(q, KT > 1 ? 1 : 0, kBStageSw);
    // tile 0 has landed (the kAq + 8 copies of tile 1 may still be in flight; the first
    // tile_barrier() covers them)
    if (kAq == 8) asm volatile("s_waitcnt vmcnt(16) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(12) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // B fragment of tile column j, sub-step base sB (a stage plus ks * 32 rows)
    auto read_b = [&](const char* sB, int j, bf16x4* lo, bf16x4* hi) {
        const int off = b_p[j & 3] + (j >> 2) * 128;
        *lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, sB + off));
        *hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, sB + off + 4 * 512));
    };
    {  // the fragments of sub-step 0 of tile 0
        const char* sA = sA0 + a_base_l + a_xo[0];
#pragma unroll
        for (int i = 0; i < kI16; i++) fa[0][i] = *LDS_PTR(bf16x8, sA + i * 2048);
#pragma unroll
        for (int j = 0; j < kJ16; j++) {
            if constexpr (kBT) {
                fb[0][j] = *LDS_PTR(bf16x8, sB0 + bt_base_l + a_xo[0] + j * 2048);
            } else {
                bf16x4 lo, hi;
                read_b(sB0, j, &lo, &hi);
                fb[0][j] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        }
    }

    // The accumulators as the matrix instructions below see them: initialised, and the writes of
    // the initial zeros a few wait states back.
    auto touch_acc = [&]() {
#pragma unroll
        for (int i = 0; i < kI16; i++)
#pragma unroll
            for (int j = 0; j < kJ16; j++) asm volatile("" : "+a"(acc[i][j]));
    };
    touch_acc();
    asm volatile("s_nop 7" ::: "memory");

    // Scalars carried from one K step to the next: the tile the copies of this step fetch
    // (kt2 = min(kt + 2, KT - 1)), its source addresses, and the three B stages' byte offsets
    // (tile kt, tile kt + 1, the stage being filled).  They are advanced at the end of a step, in
    // issue slots nothing else uses, instead of being recomputed from kt at the top of the next.
    struct Carried {
        int kt2;
        const char* a_src;  // A tile kt2 (row 0 of the workgroup tile)
        const char* b_src;  // B tile kt2: k-row 0 of it ([K, N] form) or n-row 0 (B^T form)
        unsigned sb_cur, sb_nxt, sb_fill;
    } ls;
    const unsigned b_step32 = kBT ? (unsigned)(kBK * 2) : (unsigned)kBK * (unsigned)b_pitch * 2u;  // bytes from one B tile to the next (b_pitch < 2^25)
    unsigned adv = 0;
    const size_t b_row2 = b_pitch * 4;                                  // [K, N] form: bytes from one 1 KB chunk (2 k-rows) to the next
    ls.kt2 = KT > 2 ? 2 : KT - 1;
    ls.a_src = a_tile + (size_t)ls.kt2 * kBK * 2;
    ls.b_src = b_tile + (size_t)ls.kt2 * b_step32;
    ls.sb_cur = 0, ls.sb_nxt = kBStageSw, ls.sb_fill = 2 * kBStageSw;

    // The matrix instruction, written out so that the accumulator stays in place in the
    // accumulation registers (through the builtin the compiler leaves this shape untied and copies
    // tiles around) ...
    auto mfma = [&](f32x4& c, const bf16x8& a, const bf16x8& b) {
        if constexpr (kF16) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
        else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    };
    // One direct copy with the LDS address formed in the instruction that writes M0 ...
    auto dma_at = [&](unsigned lds_base, auto q_c, unsigned voff, const char* sbase) {
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3"
                     :
                     : "s"(lds_base), "n"(decltype(q_c)::value * 1024), "v"(voff), "s"(sbase)
                     : "m0", "scc");
    };
    // ... and the matrix instruction with one such copy behind it in one statement (the LDS address is formed
    // in the instruction that writes M0), so that nothing else lands between them.
    auto mfma_dma = [&](f32x4& c, const bf16x8& a, const bf16x8& b, unsigned lds_base, auto q_c, unsigned voff, const char* sbase) {
        if constexpr (kF16)
            asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0\n\ts_add_u32 m0, %3, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %6"
                         : "+a"(c)
                         : "v"(a), "v"(b), "s"(lds_base), "n"(decltype(q_c)::value * 1024), "v"(voff), "s"(sbase)
                         : "m0", "scc");
        else
            asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\ts_add_u32 m0, %3, %4\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %5, %6"
                         : "+a"(c)
                         : "v"(a), "v"(b), "s"(lds_base), "n"(decltype(q_c)::value * 1024), "v"(voff), "s"(sbase)
                         : "m0", "scc");
    };

    // One phase = half of a 32-deep sub-step: phase p covers sub-step p / 2 (fragment slot p / 2)
    // and tile rows 4 * (p % 2) .. +3 against every tile column, 4 * kJ16 MFMAs, with the other
    // pipes' work slotted between them: the LDS reads of the other slot's fragments (the next
    // sub-step; from sAn / sBn) for the same four tile rows and half of the tile columns, and
    // chunk copies of tile kt2: phases 0-1 four of its B chunks each into the B stage being
    // filled, phases 2-3 (after the barrier) kAq / 2 of its A chunks each into A stage `cur`.
    // The columns loaded during the second phase of a sub-step are the ones the next sub-step
    // multiplies last.  A wave issues one instruction every four cycles and an MFMA of this shape
    // occupies the pipe for sixteen, so at most three other instructions fit behind an MFMA
    // without delaying the next one: the reads take the first slots of a phase one by one, every
    // copy (M0, the wait state, the load) a later slot of its own, its source address the slot
    // before, and the carried scalars the tail of the last phase.
    auto phase = [&](auto p_c, auto cur_c, auto last_c, const char* sAn, const char* sBn) {
        constexpr int p = decltype(p_c)::value, cur = decltype(cur_c)::value;
        constexpr int slot = p >> 1, nslot = slot ^ 1, h = p & 1;
        constexpr int kHalfJ = kJ16 / 2;  // tile columns per half
        bf16x4 lo[kHalfJ], hi[kHalfJ];
        constexpr int kCopies = p < 2 ? 4 : kAq / 2;                 // copies of this phase
        constexpr int kFirst = 4 + kJ16;                             // first slot without a fragment read
        constexpr int kTail = p == 3 ? 3 : p == 2 ? 1 : 0;           // last slots, kept for the carried scalars
        constexpr int kEvery = (kSlots - kFirst - kTail) / kCopies;  // slots per copy (address, then copy)
        static_assert(kEvery >= 2, "a copy needs two slots");
        const unsigned lds_dst = p < 2 ? lds_b + ls.sb_fill : lds_a + cur * kAStageT;
        constexpr bool kMaybe = kAny && decltype(last_c)::value;         // one of the last steps, which copy the last tile
        const bool ragged_now = kMaybe && has_last && ls.kt2 == KT - 1;  // this step copies the partial last tile
        const char* src = p < 2 ? ls.b_src : ls.a_src;
        if (p == 1 && !kBT) src += 4 * b_row2;
#pragma unroll
        for (int n = 0; n < kSlots; n++) {
            // first the columns whose fragments arrived a sub-step ago, then the other half; back
            // and forth over the columns and the rows, so that consecutive instructions share one
            // operand register set (fewer operand bits toggle: about 1 % on the clock the part
            // sustains)
            const int jh = n / (kSlots / 2), r = n % (kSlots / 2), rr = r / kHalfJ, jj = r % kHalfJ;
            const int mi = 4 * h + (jh ? 3 - rr : rr);
            const int mj = jh * kHalfJ + ((rr & 1) ? kHalfJ - 1 - jj : jj);
            const bool copy_range = n >= kFirst && (n - kFirst) / kEvery < kCopies;
            const int c = copy_range ? (n - kFirst) / kEvery : 0, part = copy_range ? (n - kFirst) % kEvery : -1;
            const int q = (p & 1) * kCopies + c;  // chunk of the tile
            // a copy slot: the MFMA and the copy as one statement; where a step may have to copy
            // the partial last tile instead (kMaybe) the choice is made at run time, and the MFMA
            // stays outside that branch: an accumulator that flows through a branch would be moved
            // by the compiler, which does not know that it has to wait for the matrix pipe first
            auto with_q = [&](auto&& f) {
                switch (q) {  // q is a constant of the unrolled loop
                    case 0: f(std::integral_constant<int, 0>{}); break;
                    case 1: f(std::integral_constant<int, 1>{}); break;
                    case 2: f(std::integral_constant<int, 2>{}); break;
                    case 3: f(std::integral_constant<int, 3>{}); break;
                    case 4: f(std::integral_constant<int, 4>{}); break;
                    case 5: f(std::integral_constant<int, 5>{}); break;
                    case 6: f(std::integral_constant<int, 6>{}); break;
                    default: f(std::integral_constant<int, 7>{}); break;
                }
            };
            auto voff_of = [&](auto q_c) {
                constexpr int qq = decltype(q_c)::value;
                return p >= 2 ? a_voff[qq < kAq ? qq : 0] : kBT ? bt_voff[kBT ? qq : 0] : b_voff[qq & 1];
            };
            if (part == 1 && !kMaybe) {
                with_q([&](auto q_c) { mfma_dma(acc[mi][mj], fb[slot][mj], fa[slot][mi], lds_dst, q_c, voff_of(q_c), src); });
            } else {
                mfma(acc[mi][mj], fb[slot][mj], fa[slot][mi]);
                if (part == 1) {
                    if (ragged_now) {
                        if (p < 2) dma_b(q, ls.kt2, ls.sb_fill);
                        else dma_a(q, ls.kt2, cur * kAStageT);
                    } else {
                        with_q([&](auto q_c) { dma_at(lds_dst, q_c, voff_of(q_c), src); });
                    }
                }
            }
            if (n < 4) fa[nslot][4 * h + n] = *LDS_PTR(bf16x8, sAn + (4 * h + n) * 2048);
            else if constexpr (kBT) {
                if (n < 4 + kHalfJ) fb[nslot][h * kHalfJ + n - 4] = *LDS_PTR(bf16x8, sBn + (h * kHalfJ + n - 4) * 2048);
            } else if (n < 4 + 2 * kHalfJ) {
                const int jl = (n - 4) >> 1, j = h * kHalfJ + jl;
                const int off = b_p[j & 3] + (j >> 2) * 128;
                if ((n & 1) == 0) lo[jl] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, sBn + off));
                else hi[jl] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(LDS_PTR(bf16x4, sBn + off + 4 * 512));
            }
            if (part == 0) {
                // the chunk's source address, one slot ahead of the copy
                if (p < 2 && !kBT && c > 0) src += b_row2;
                asm volatile("" : "+s"(src));
            }
            // the scalars of the next K step, in the slots left over at the end
            if (p == 2 && n == kSlots - 1) {
                // (the copies of this step into the stage being filled went out in phases 0-1)
                const unsigned t = ls.sb_cur;
                ls.sb_cur = ls.sb_nxt;
                ls.sb_nxt = ls.sb_fill;
                ls.sb_fill = t;
            }
            if (p == 3 && n == kSlots - 3) {
                // 1 while the copies have not reached the last tile (as a minimum: a comparison's
                // result would take a detour through the vector unit to become a number)
                adv = (unsigned)__builtin_elementwise_min(KT - 1 - ls.kt2, 1);
                ls.kt2 += (int)adv;
                asm volatile("" : "+s"(adv));
            }
            if (p == 3 && n == kSlots - 2) {
                ls.a_src += adv * (unsigned)(kBK * 2);
                asm volatile("" : "+s"(ls.a_src));
            }
            if (p == 3 && n == kSlots - 1) {
                ls.b_src += adv * b_step32;  // (a tile-to-tile step stays below 4 GiB: b_pitch < 2^25)
                asm volatile("" : "+s"(ls.b_src));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!kBT) {
#pragma unroll
            for (int jl = 0; jl < kHalfJ; jl++)
                fb[nslot][h * kHalfJ + jl] = __builtin_shufflevector(lo[jl], hi[jl], 0, 1, 2, 3, 4, 5, 6, 7);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    using C0 = std::integral_constant<int, 0>;
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    // tile kt: A in stage cur = kt & 1, B in the stage at ls.sb_cur (next tile's B at ls.sb_nxt, the one after goes to ls.sb_fill)
    auto iteration = [&](auto cur_c, auto last_c) {
        constexpr int cur = decltype(cur_c)::value;
        using C = std::integral_constant<int, cur>;
        const char* sAc = sA0 + cur * kAStageT + a_base_l;
        const char* sBc = sB0 + ls.sb_cur + (kBT ? bt_base_l : 0);
        const char* sAx = sA0 + (cur ^ 1) * kAStageT + a_base_l;
        const char* sBx = sB0 + ls.sb_nxt + (kBT ? bt_base_l : 0);
        // sub-step ks of a B stage: 32 k-rows of 512 B further, or (kBT) the same chunk offset as A's
        auto b_ks = [&](int ks) { return kBT ? a_xo[ks] : ks * 32 * 512; };
        phase(C0{}, C{}, last_c, sAc + a_xo[1], sBc + b_ks(1));
        phase(C1{}, C{}, last_c, sAc + a_xo[1], sBc + b_ks(1));
        // tile kt+1 has landed; nobody reads A stage cur any more
        tile_barrier();
        phase(C2{}, C{}, last_c, sAx + a_xo[0], sBx + b_ks(0));
        phase(C3{}, C{}, last_c, sAx + a_xo[0], sBx + b_ks(0));
    };
    // What the epilogue of the plain and the residual product needs, ahead of the loop's end: lane l
    // stores (and fetches from R) 16-byte chunk l % kChunks of row it * kRowsPerIt + l / kChunks of
    // the wave's 128-row tile, for it = 0 .. kIts-1.
    const size_t row0 = m0 + wm * 128, col0 = n0 + wn * (kJ * 32);
    constexpr int kChunks = kJ * 4;          // 16-byte chunks per row of the wave's tile
    constexpr int kRowsPerIt = 64 / kChunks;  // rows one store instruction covers
    constexpr int kIts = 128 / kRowsPerIt;
    const int lr = lane / kChunks, lc = lane % kChunks;
    const int rows_here = row0 >= (size_t)M ? 0 : (size_t)M - row0 < 128 ? (int)((size_t)M - row0) : 128;  // rows of the wave's tile inside C
    const bool col_ok = col0 + lc * 8 + 8 <= (size_t)N;
    // columns of this lane's chunk inside C when the chunk is the partial last one of a row (kAny: N % 8 of them), else 0
    const int col_tail = kAny && !col_ok && col0 + lc * 8 < (size_t)N ? (int)((size_t)N - (col0 + lc * 8)) : 0;
    auto store_any = [&](__bf16* dst, const u32x4& v, bool row_ok) {
        if (col_ok && row_ok) *reinterpret_cast<u32x4_any*>(dst) = v;
        else if (row_ok) {
            const bf16x8 e8 = __builtin_bit_cast(bf16x8, v);
#pragma unroll
            for (int e = 0; e < 7; e++)
                if (e < col_tail) dst[e] = e8[e];
        }
    };
    u32x4 res[kResidual ? kIts : 1];
    auto fetch_residual = [&](int first, int last) {
        const __bf16* Rl = R + (row0 + lr) * r_pitch + col0 + lc * 8;
#pragma unroll
        for (int it = first; it < last; it++) {
            res[it] = u32x4{0u, 0u, 0u, 0u};
            const __bf16* src = Rl + (size_t)(it * kRowsPerIt) * r_pitch;
            if constexpr (kAny) {
                const bool row_ok = it * kRowsPerIt + lr < rows_here;
                if (col_ok && row_ok) res[it] = *reinterpret_cast<const u32x4_any*>(src);
                else if (row_ok) {
                    bf16x8 e8 = __builtin_bit_cast(bf16x8, res[it]);
#pragma unroll
                    for (int e = 0; e < 7; e++)
                        if (e < col_tail) e8[e] = src[e];
                    res[it] = __builtin_bit_cast(u32x4, e8);
                }
            } else {
                if (col_ok && it * kRowsPerIt + lr < rows_here) res[it] = *reinterpret_cast<const u32x4*>(src);
            }
        }
    };
    {
        using Last = std::true_type;
        int kt = 0;
        // (us with the choice of the source in every step / so: 512 x 50264 x 776 52.6 / 49.6, 4096 x 4096 x 4088 107.6 / 94.4; odd columns, which have
        // no partial step, 512 x 50257 x 768 47.2 / 44.1, 1000 x 30001 x 2048 107 / 97.  Stores of whole tiles without a test beside them are not worth
        // the longer code: 2600 x 4127 x 256 17.6, 16.9 without; 3000 x 8193 x 264 44.3 / 42.7, 1322 x 6672 x 72 13.8 / 12.9; level in long K.)
        if constexpr (kAny) {
            const int whole = has_last ? KT - 3 : KT;  // the first step that copies tile KT - 1, clamped to which those behind it do as well
            for (; kt + 1 < whole; kt += 2) {
                iteration(C0{}, std::false_type{});
                iteration(C1{}, std::false_type{});
            }
        }
        for (; kt + 1 < KT; kt += 2) {
            iteration(C0{}, Last{});
            iteration(C1{}, Last{});
        }
        if (kt < KT) iteration(C0{}, Last{});
    }
    // The residual rows are on their way while the accumulators are converted and staged: the
    // fragment registers of the loop are free from here on.  (Fetching half of them before the
    // last two K steps instead measured the same: the loop's waits on its own copies count
    // vector-memory operations in order, so they wait for the residual rows as well.)
    if constexpr (kResidual) fetch_residual(0, kIts);
    full_barrier();
    // the last MFMAs' results must have left the matrix pipe before the vector ALUs read them (the
    // compiler does not see the instructions above as matrix operations); the empty statements
    // behind the wait keep every later use of an accumulator behind it
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    touch_acc();

    // Epilogue.  With swapped operands lane l of tile (i, j) holds, in its four registers,
    // C[m = i*16 + l%16][n = j*16 + 4*(l/16) + 0..3].
    if (kSplitK) {
        // f32 partials straight from the registers: 16 bytes per lane, rows and columns masked
        float* Wt = W + ((size_t)blockIdx.z * gridDim.y + blockIdx.y) * (size_t)M * N;
#pragma unroll
        for (int i = 0; i < kI16; i++)
#pragma unroll
            for (int j = 0; j < kJ16; j++) {
                const size_t row = row0 + i * 16 + (lane & 15), col = col0 + j * 16 + 4 * (lane >> 4);
                if constexpr (kAny) {
                    if (row < (size_t)M && col + 4 <= (size_t)N) *reinterpret_cast<f32x4_any*>(Wt + row * N + col) = acc[i][j];
                    else if (row < (size_t)M) {
#pragma unroll
                        for (int e = 0; e < 3; e++)
                            if (col + e < (size_t)N) Wt[row * N + col + e] = acc[i][j][e];
                    }
                } else {
                    if (row < (size_t)M && col + 4 <= (size_t)N) *reinterpret_cast<f32x4*>(Wt + row * N + col) = acc[i][j];
                }
            }
        return;
    }
    char* sC = smem + wave * kCWaveT;
    if constexpr (!kSwiGLU) {
        // The plain and the residual product: 16 rows at a time.  A wave reads back only what it
        // staged itself, and the LDS serves a wave's requests in order, so the rows of tile row i
        // are read back and stored while tile row i + 1 is being converted and staged: the stores
        // start one tile row after the loop ends instead of after the whole staging.
        constexpr int kPerRow = 16 / kRowsPerIt;  // store instructions per tile row
        // (rotary epilogue: the tile's columns lie either all in front of `split` or all behind it)
        const bool rotate = kRope && n0 < (size_t)rope.split;
        const size_t ldc = !kRope ? (size_t)N : rotate ? (size_t)rope.split : (size_t)(N - rope.split);
        __bf16* Cl = (!kRope || rotate ? C + col0 : rope.rest + (col0 - rope.split)) + (row0 + lr) * ldc + lc * 8;
        const char* sCl = sC + lr * kCPitchT + lc * 16;
        auto stage_row = [&](int i) {
#pragma unroll
            for (int j = 0; j < kJ16; j++) {
                bf16x4 h = round_to_elem<kF16>(acc[i][j]);
                *LDS_PTR(bf16x4, sC + (i * 16 + (lane & 15)) * kCPitchT + (j * 16 + 4 * (lane >> 4)) * 2) = h;
            }
        };
        // Rotary epilogue: the angles of a tile row (four store steps: eight cos and eight sin values each)
        // are requested one tile row ahead; the row's position advances by the rows of a store step,
        // wrapping at seq, so the only division is the one that finds the first position.
        f32x8 cs_nxt[kRope ? kPerRow : 1], sn_nxt[kRope ? kPerRow : 1], cs_cur[kRope ? kPerRow : 1], sn_cur[kRope ? kPerRow : 1];
        unsigned rope_pos = 0;
        auto fetch_angles = [&]() {
            if constexpr (kRope) {
                const unsigned seq = (unsigned)rope.seq;
#pragma unroll
                for (int t = 0; t < kPerRow; t++) {
                    cs_nxt[t] = *reinterpret_cast<const f32x8*>(rope.cos + (size_t)rope_pos * 64 + (lc & 7) * 8);
                    sn_nxt[t] = *reinterpret_cast<const f32x8*>(rope.sin + (size_t)rope_pos * 64 + (lc & 7) * 8);
                    rope_pos += kRowsPerIt;
                    if (seq < (unsigned)kRowsPerIt) rope_pos %= seq;
                    else if (rope_pos >= seq) rope_pos -= seq;
                }
            }
        };
        if constexpr (kRope) {
            if (rotate) {
                rope_pos = (unsigned)((row0 + lr) % (size_t)rope.seq);
                fetch_angles();
            }
        }
        stage_row(0);
#pragma unroll
        for (int i = 0; i < kI16; i++) {
            u32x4 v[kPerRow], pv[kRope ? kPerRow : 1];
#pragma unroll
            for (int t = 0; t < kPerRow; t++) v[t] = *LDS_PTR(u32x4, sCl + (i * 16 + t * kRowsPerIt) * kCPitchT);
            if constexpr (kRope) {
                if (rotate) {
                    // the partners 64 columns away: chunk lc ^ 8 of the same staged rows
#pragma unroll
                    for (int t = 0; t < kPerRow; t++) {
                        pv[t] = *LDS_PTR(u32x4, sC + (i * 16 + t * kRowsPerIt + lr) * kCPitchT + (lc ^ 8) * 16);
                        cs_cur[t] = cs_nxt[t];
                        sn_cur[t] = sn_nxt[t];
                    }
                    if (i + 1 < kI16) fetch_angles();
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (i + 1 < kI16) stage_row(i + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < kPerRow; t++) {
                const int r = i * 16 + t * kRowsPerIt;
                if constexpr (kResidual) {
                    v[t] = add_elems<kF16>(v[t], res[i * kPerRow + t]);
                }
                if constexpr (kRope) {
                    if (rotate) {
                        // this lane's 8 columns of a head, their partners, and the 8 angles of the row's position
                        const f32x8 x = __builtin_convertvector(__builtin_bit_cast(bf16x8, v[t]), f32x8);
                        const f32x8 y = __builtin_convertvector(__builtin_bit_cast(bf16x8, pv[t]), f32x8);
                        const f32x8 sn = lc < 8 ? -sn_cur[t] : sn_cur[t];  // first half: x1 cos - x2 sin; second half: x2 cos + x1 sin
                        // (which of the two products is rounded decides the last bit: the sine's in rows 0..3 of sixteen, the cosine's below)
                        const f32x8 o = t == 0 ? __builtin_elementwise_fma(x, cs_cur[t], y * sn) : __builtin_elementwise_fma(y, sn, x * cs_cur[t]);
                        v[t] = __builtin_bit_cast(u32x4, __builtin_convertvector(o, bf16x8));
                    }
                }
                if constexpr (kAny) store_any(Cl + (size_t)r * ldc, v[t], r + lr < rows_here);
                else if (col_ok && r + lr < rows_here) *reinterpret_cast<u32x4*>(Cl + (size_t)r * ldc) = v[t];
            }
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < kI16; i++)
#pragma unroll
        for (int j = 0; j < kJ16; j++) {
            bf16x4 h = __builtin_convertvector(acc[i][j], bf16x4);
            const int ml = i * 16 + (lane & 15);
            const int nl = j * 16 + 4 * (lane >> 4);
            *LDS_PTR(bf16x4, sC + ml * kCPitchT + nl * 2) = h;
        }
    // The gated epilogue: waves (wm, 0) and (wm, 1) staged the gate and the up block of the same
    // 128 rows x 128 columns; each of the two now combines 64 of those rows: 16 chunks of 8 columns
    // per row.
    if constexpr (kSwiGLU) {
        __syncthreads();
        const size_t F = (size_t)N / 2;
        const char* sG = smem + (wm * 2 + 0) * kCWaveT;
        const char* sU = smem + (wm * 2 + 1) * kCWaveT;
#pragma unroll 4
        for (int it = 0; it < 16; it++) {
            const int r = wn * 64 + it * 4 + (lane >> 4);
            const int ch = lane & 15;
            const f32x8 gf = __builtin_convertvector(__builtin_bit_cast(bf16x8, *LDS_PTR(u32x4, sG + r * kCPitchT + ch * 16)), f32x8);
            const f32x8 uf = __builtin_convertvector(__builtin_bit_cast(bf16x8, *LDS_PTR(u32x4, sU + r * kCPitchT + ch * 16)), f32x8);
            f32x8 y;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                // x * sigmoid(x) * y with sigmoid(x) = 1 / (1 + exp2(x * (-1 / ln 2)))
                const float sg = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gf[e] * -1.4426950408889634f));
                y[e] = gf[e] * sg * uf[e];
            }
            const u32x4 v = __builtin_bit_cast(u32x4, __builtin_convertvector(y, bf16x8));
            if (row0 + r < (size_t)M && n0 + ch * 8 + 8 <= F) *reinterpret_cast<u32x4*>(C + (row0 + r) * F + n0 + ch * 8) = v;
        }
    }
}

// Instantiations.  B is [K, N], or ("_nt") Bt [N, K] row-major (k contiguous, the layout of a Linear layer's weight),
// C = A Bt^T; for the gated epilogue B is [K, 2F] or Bt [2F, K], gate first.  lda / ldb are read by the "_any" kernels.
#define MRK_GEMM_KERNEL(name, ...)                                                                                                    \
    __global__ __launch_bounds__(256) void name(const __bf16* __restrict__ A, const __bf16* __restrict__ B, __bf16* __restrict__ C,   \
                                                int M, int N, int K, int tiles_m, int tiles_n, int lda, int ldb) {                    \
        gemm_tile_body<__VA_ARGS__>(A, B, C, M, N, K, tiles_m, tiles_n, nullptr, 0, nullptr, RopeEpilogue{}, -1, lda, ldb);            \
    }
#define MRK_GEMM_RESIDUAL_KERNEL(name, ...)                                                                                           \
    __global__ __launch_bounds__(256) void name(const __bf16* __restrict__ A, const __bf16* __restrict__ B,                           \
                                                const __bf16* __restrict__ R, __bf16* __restrict__ C, int M, int N, int K,            \
                                                int tiles_m, int tiles_n, int ldr, int lda, int ldb) {                                \
        gemm_tile_body<__VA_ARGS__>(A, B, C, M, N, K, tiles_m, tiles_n, nullptr, 0, R, RopeEpilogue{}, ldr, lda, ldb);                 \
    }
#define MRK_GEMM_SPLITK_KERNEL(name, ...)                                                                                             \
    __global__ __launch_bounds__(256) void name(const __bf16* __restrict__ A, const __bf16* __restrict__ B, float* __restrict__ W,    \
                                                int M, int N, int K, int tiles_m, int tiles_n, int kt_per_split, int lda, int ldb) {  \
        gemm_tile_body<__VA_ARGS__>(A, B, nullptr, M, N, K, tiles_m, tiles_n, W, kt_per_split, nullptr, RopeEpilogue{}, -1, lda, ldb); \
    }
MRK_GEMM_KERNEL(gemm_bf16_tile256, false, 4, false, false, false, false, false)
MRK_GEMM_KERNEL(gemm_bf16_tile256_any, true, 4, false, false, false, false, false)
MRK_GEMM_KERNEL(gemm_bf16_tile128, false, 2, false, false, false, false, false)
MRK_GEMM_KERNEL(gemm_bf16_tile128_any, true, 2, false, false, false, false, false)
MRK_GEMM_RESIDUAL_KERNEL(gemm_bf16_tile256_residual, false, 4, false, true, false, false, false)
MRK_GEMM_RESIDUAL_KERNEL(gemm_bf16_tile256_residual_any, true, 4, false, true, false, false, false)
MRK_GEMM_RESIDUAL_KERNEL(gemm_bf16_tile128_residual, false, 2, false, true, false, false, false)
MRK_GEMM_RESIDUAL_KERNEL(gemm_bf16_tile128_residual_any, true, 2, false, true, false, false, false)
MRK_GEMM_SPLITK_KERNEL(gemm_bf16_tile128_splitk, false, 2, true, false, false, false, false)
MRK_GEMM_SPLITK_KERNEL(gemm_bf16_tile128_splitk_any, true, 2, true, false, false, false, false)
MRK_GEMM_KERNEL(gemm_bf16_nt_tile256, false, 4, false, false, false, true, false)
MRK_GEMM_KERNEL(gemm_bf16_nt_tile256_any, true, 4, false, false, false, true, false)
MRK_GEMM_KERNEL(gemm_bf16_nt_tile128, false, 2, false, false, false, true, false)
MRK_GEMM_KERNEL(gemm_bf16_nt_tile128_any, true, 2, false, false, false, true, false)
MRK_GEMM_RESIDUAL_KERNEL(gemm_bf16_nt_tile256_residual, false, 4, false, true, false, true, false)
MRK_GEMM_RESIDUAL_KERNEL(gemm_bf16_nt_tile256_residual_any, true, 4, false, true, false, true, false)
MRK_GEMM_RESIDUAL_KERNEL(gemm_bf16_nt_tile128_residual, false, 2, false, true, false, true, false)
MRK_GEMM_RESIDUAL_KERNEL(gemm_bf16_nt_tile128_residual_any, true, 2, false, true, false, true, false)
MRK_GEMM_SPLITK_KERNEL(gemm_bf16_nt_tile128_splitk, false, 2, true, false, false, true, false)
MRK_GEMM_SPLITK_KERNEL(gemm_bf16_nt_tile128_splitk_any, true, 2, true, false, false, true, false)
MRK_GEMM_KERNEL(gemm_f16_tile256, false, 4, false, false, false, false, true)
MRK_GEMM_KERNEL(gemm_f16_tile256_any, true, 4, false, false, false, false, true)
MRK_GEMM_KERNEL(gemm_f16_tile128, false, 2, false, false, false, false, true)
MRK_GEMM_KERNEL(gemm_f16_tile128_any, true, 2, false, false, false, false, true)
MRK_GEMM_RESIDUAL_KERNEL(gemm_f16_tile256_residual, false, 4, false, true, false, false, true)
MRK_GEMM_RESIDUAL_KERNEL(gemm_f16_tile256_residual_any, true, 4, false, true, false, false, true)
MRK_GEMM_RESIDUAL_KERNEL(gemm_f16_tile128_residual, false, 2, false, true, false, false, true)
MRK_GEMM_RESIDUAL_KERNEL(gemm_f16_tile128_residual_any, true, 2, false, true, false, false, true)
MRK_GEMM_SPLITK_KERNEL(gemm_f16_tile128_splitk, false, 2, true, false, false, false, true)
MRK_GEMM_SPLITK_KERNEL(gemm_f16_tile128_splitk_any, true, 2, true, false, false, false, true)
MRK_GEMM_KERNEL(gemm_f16_nt_tile256, false, 4, false, false, false, true, true)
MRK_GEMM_KERNEL(gemm_f16_nt_tile256_any, true, 4, false, false, false, true, true)
MRK_GEMM_KERNEL(gemm_f16_nt_tile128, false, 2, false, false, false, true, true)
MRK_GEMM_KERNEL(gemm_f16_nt_tile128_any, true, 2, false, false, false, true, true)
MRK_GEMM_RESIDUAL_KERNEL(gemm_f16_nt_tile256_residual, false, 4, false, true, false, true, true)
MRK_GEMM_RESIDUAL_KERNEL(gemm_f16_nt_tile256_residual_any, true, 4, false, true, false, true, true)
MRK_GEMM_RESIDUAL_KERNEL(gemm_f16_nt_tile128_residual, false, 2, false, true, false, true, true)
MRK_GEMM_RESIDUAL_KERNEL(gemm_f16_nt_tile128_residual_any, true, 2, false, true, false, true, true)
MRK_GEMM_SPLITK_KERNEL(gemm_f16_nt_tile128_splitk, false, 2, true, false, false, true, true)
MRK_GEMM_SPLITK_KERNEL(gemm_f16_nt_tile128_splitk_any, true, 2, true, false, false, true, true)
MRK_GEMM_KERNEL(gemm_bf16_tile256_swiglu, false, 4, false, false, true, false)
MRK_GEMM_KERNEL(gemm_bf16_tile256_swiglu_any, true, 4, false, false, true, false)
MRK_GEMM_KERNEL(gemm_bf16_nt_tile256_swiglu, false, 4, false, false, true, true)
MRK_GEMM_KERNEL(gemm_bf16_nt_tile256_swiglu_any, true, 4, false, false, true, true)
#undef MRK_GEMM_KERNEL
#undef MRK_GEMM_RESIDUAL_KERNEL
#undef MRK_GEMM_SPLITK_KERNEL
__global__ __launch_bounds__(256) void gemm_bf16_tile256_rope(const __bf16* __restrict__ A, const __bf16* __restrict__ B,
                                                              __bf16* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n,
                                                              RopeEpilogue rope) {
    gemm_tile_body<false, 4, false, false, false, false, false, true>(A, B, C, M, N, K, tiles_m, tiles_n, nullptr, 0, nullptr, rope);
}
__global__ __launch_bounds__(256) void gemm_bf16_nt_tile256_rope(const __bf16* __restrict__ A, const __bf16* __restrict__ B,
                                                              __bf16* __restrict__ C, int M, int N, int K, int tiles_m, int tiles_n,
                                                              RopeEpilogue rope) {
    gemm_tile_body<false, 4, false, false, false, true, false, true>(A, B, C, M, N, K, tiles_m, tiles_n, nullptr, 0, nullptr, rope);
}

// dst[rows][pitch] = src[rows][cols] with zeros from cols to pitch (a multiple of 8): an operand whose rows start on odd
// elements, laid out for the 16-byte copies of the tiled kernels.  A wave moves up to 128 consecutive 16-byte pieces of a row
// (the loads aligned to 2 bytes only); grid y counts such runs of long rows, so that few long
// rows fill the chip too.
constexpr int kRepitchRun = 128;
__global__ __launch_bounds__(256) void gemm_repitch(const unsigned short* __restrict__ src, unsigned short* __restrict__ dst, long rows,
                                                    int cols, int pitch) {
    const int first = (int)blockIdx.y * kRepitchRun + (int)(threadIdx.x & 63);
    for (long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6); row < rows; row += (long)gridDim.x * 4) {
        const unsigned short* s = src + (size_t)row * cols;
        u32x4* d = reinterpret_cast<u32x4*>(dst + (size_t)row * pitch);
        u32x4 v[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int c = (first + 64 * i) * 8;
            v[i] = u32x4{0u, 0u, 0u, 0u};
            if (c + 8 <= cols) v[i] = *reinterpret_cast<const u32x4_any*>(s + c);
            else if (c < cols) {
#pragma unroll
                for (int e = 0; e < 8; e++)
                    if (c + e < cols) v[i][e >> 1] |= (unsigned)s[c + e] << (16 * (e & 1));
            }
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
            if (first + 64 * i < pitch / 8) d[first + 64 * i] = v[i];
    }
}
// C[i] = bf16(W[0][i] + W[1][i] + ... + W[splits-1][i]), 8 elements per work-item, partials added
// in the order of their K ranges so the result does not depend on timing.  R, when given, is added to the rounded
// sum and the result rounded again (the bits of the product followed by an elementwise add): a matrix of C's shape
// (r_period 0) or one row repeated every r_period elements (a bias).
// kAny: total (or r_period) is no multiple of 8: one element per work-item and the row of R element by element.
template <bool kF16, bool kAny>
__global__ __launch_bounds__(256) void gemm_splitk_reduce(const float* __restrict__ W, __bf16* __restrict__ C, long total,
                                                          int splits, const __bf16* __restrict__ R, long r_period) {
    if constexpr (kAny) {
        const long i = (long)blockIdx.x * 256 + threadIdx.x;
        if (i >= total) return;
        float s = 0.0f;
        for (int k = 0; k < splits; k++) s += W[(size_t)k * total + i];
        const __bf16* r = R ? R + (r_period ? i % r_period : i) : nullptr;
        if constexpr (kF16) {
            _Float16 h = (_Float16)s;
            if (r) h = (_Float16)((float)h + (float)__builtin_bit_cast(_Float16, *r));
            C[i] = __builtin_bit_cast(__bf16, h);
        } else {
            __bf16 h = (__bf16)s;
            if (r) h = (__bf16)((float)h + (float)*r);
            C[i] = h;
        }
        return;
    }
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= total) return;
    f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
    for (int s = 0; s < splits; s++) {
        const f32x4* p = reinterpret_cast<const f32x4*>(W + (size_t)s * total + i);
        lo += p[0];
        hi += p[1];
    }
    bf16x4 l = round_to_elem<kF16>(lo), h = round_to_elem<kF16>(hi);
    if (R) {
        const bf16x8 r = *reinterpret_cast<const bf16x8*>(R + (r_period ? i % r_period : i));
        auto widen = [](const bf16x4& v) {
            if constexpr (kF16) return __builtin_convertvector(__builtin_bit_cast(f16x4, v), f32x4);
            else return __builtin_convertvector(v, f32x4);
        };
        l = round_to_elem<kF16>(widen(l) + widen(__builtin_shufflevector(r, r, 0, 1, 2, 3)));
        h = round_to_elem<kF16>(widen(h) + widen(__builtin_shufflevector(r, r, 4, 5, 6, 7)));
    }
    *reinterpret_cast<bf16x8*>(C + i) = __builtin_shufflevector(l, h, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Any shape: one wave per 32x32 output tile, operands fetched straight from global memory
// with bounds checks (zero fill), no LDS.  Correct for every M, N, K; used when the shape
// does not fit the tiled kernel.  The same instructions on the same k in the same order as the tiled
// kernels', and sums of `k_range` deep ranges of K added up in order as the split-K reduction adds its partial
// results: the same bits, whether or not there is scratch for padded operands and partial results.
// kBT: B is stored [N, K].  add (may be null): a matrix of C's shape or (add_pitch 0) one row, added to the rounded sums.
template <bool kF16, bool kBT>
__global__ __launch_bounds__(256) void gemm_bf16_generic(const __bf16* __restrict__ A, const __bf16* __restrict__ B,
                                                         __bf16* __restrict__ C, int M, int N, int K, int tiles_n,
                                                         long total_tiles, int k_range, const __bf16* __restrict__ add, long add_pitch) {
    const int lane = threadIdx.x & 63;
    const long tile = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (tile >= total_tiles) return;
    A += (size_t)blockIdx.y * M * K;
    B += (size_t)blockIdx.y * K * N;
    C += (size_t)blockIdx.y * M * N;
    const long m0 = (tile / tiles_n) * 32, n0 = (tile % tiles_n) * 32;
    const int lr = lane & 15, kg = 8 * (lane >> 4);
    f32x4 sum[2][2] = {};
    for (long first = 0; first < K; first += k_range) {
        const long end = first + k_range < K ? first + k_range : K;
        f32x4 acc[2][2] = {};
        for (long k0 = first; k0 < end; k0 += 32) {
            bf16x8 a[2], b[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const long m = m0 + t * 16 + lr, n = n0 + t * 16 + lr;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const long k = k0 + kg + e;
                    a[t][e] = (m < M && k < K) ? A[m * K + k] : (__bf16)0.0f;
                    b[t][e] = (n < N && k < K) ? B[kBT ? n * K + k : k * N + n] : (__bf16)0.0f;
                }
            }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    if constexpr (kF16)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[i]), __builtin_bit_cast(f16x8, b[j]), acc[i][j], 0, 0, 0);
                    else acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
                }
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) sum[i][j] += acc[i][j];
    }
    // lane l register e of tile (i, j): row 4*(l/16) + e, column l%16
    auto store = [&](auto with_add) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const long r = m0 + i * 16 + 4 * (lane >> 4) + e, n = n0 + j * 16 + lr;
                    if (r >= M || n >= N) continue;
                    using T = std::conditional_t<kF16, _Float16, __bf16>;
                    T h = (T)sum[i][j][e];
                    if constexpr (decltype(with_add)::value) h = (T)((float)h + (float)__builtin_bit_cast(T, add[r * add_pitch + n]));
                    C[r * N + n] = __builtin_bit_cast(__bf16, h);
                }
    };
    if (add) {
        add += (size_t)blockIdx.y * M * add_pitch;
        store(std::true_type{});
    } else {
        store(std::false_type{});
    }
}

}  // namespace mrk::dev

// Split-K partials for callers that cannot allocate: 32 MiB per device, held until the process
// ends.  That is the most plan_split_k ever asks for (at most 256 workgroups in flight, each
// with one 128 x 256 f32 partial tile).  In host code the name is only a handle for
// hipGetSymbolAddress; kernels receive the resolved per-device address as an argument.
static constexpr size_t kStaticWsBytes = size_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kStaticWsBytes];

namespace mrk {

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_static_ws[kMaxDevices];  // resolved address of `scratch` on each device

// Split-K plan for a shape: how many K ranges and how many 64-deep steps each, or splits = 1
// when the plain tiled kernel already has enough workgroups (or the K loop is too short).
struct SplitPlan {
    long splits = 1, kt_per_split = 0;
};
SplitPlan plan_split_k(long M, long N, long K, long batch) {
    SplitPlan p;
    const long tiles = ((M + 127) / 128) * ((N + 255) / 256) * batch;
    const long kt_all = (K + 63) / 64;
    // at most a quarter of the CUs busy; with up to 64 rows (the weight is streamed once, the partial results are
    // small) up to half of them, and then two or three ranges already pay (16 x 22016 x 4096: 86 tiles)
    const bool few_rows = M <= 64;
    if (tiles > (few_rows ? 128 : 64) || kt_all < 8) return p;
    long want = 256 / tiles;                 // ranges that would put one workgroup on every CU
    if (want > kt_all / 2) want = kt_all / 2;  // at least two K steps per range
    // the partial results are written and read back once per range: worth it only while that
    // traffic stays below what the operands themselves move
    const double operand_bytes = 2.0 * batch * ((double)M * K + (double)K * N);
    const long least = few_rows ? 2 : 4;
    while (want >= least && 2.0 * want * batch * M * N * 4.0 > operand_bytes) want--;
    if (want < least) return p;
    p.kt_per_split = (kt_all + want - 1) / want;
    p.splits = (kt_all + p.kt_per_split - 1) / p.kt_per_split;
    if (p.splits < 2) p.splits = 1;
    return p;
}
// shapes the tiled kernels address (32-bit offsets inside a tile, and from one tile of B to the next 64 rows on: the limits
// hold for the row pitches, which round N and K up to 8); without scratch the operands' rows have to be whole
// 16-byte chunks, see operand_padding
bool tile_addressable(long M, long N, long K, long batch) {
    if (M <= 0 || N <= 0 || K <= 0 || batch <= 0 || batch > 65535) return false;
    if (M > 0x7fffffffL || K > (1L << 23) || N > (1L << 25) - 8) return false;
    const long tn = (N + mrk::dev::kBN - 1) / mrk::dev::kBN, tm128 = (M + 127) / 128;
    return tm128 * tn <= 0x7fffffffL;
}
// The operands whose rows are no whole 16-byte chunks, and the scratch their padded copies take (in front of the
// split-K partials).  Copying costs twice the operand's bytes on top of the product's own traffic; what it replaces (one
// wave per 32x32 tile, 2-byte loads straight from global memory) ran at 0.036 PFLOP/s on every shape: a projection of 512
// rows onto 50257 columns at K = 768, weight [N, K], took 1560 us with the transposed copy that kernel needs and takes 50
// (only C's rows are odd there: nothing is padded).
struct OperandPadding {
    bool a = false, b = false;
    long lda = 0, ldb = 0;            // row pitches in elements as the kernel reads the operands
    size_t a_bytes = 0, b_bytes = 0;  // scratch for the padded copies, multiples of 256
};
OperandPadding operand_padding(long M, long N, long K, long batch, bool b_transposed) {
    OperandPadding o;
    // A small [K, N] product asks for no scratch: it is one launch of a few steps of K on kernels that need no padding
    // (4.6-6.9 us from 33 x 7 x 19 to 256 x 255 x 63), two or three launches here (12-13 us).
    if (!b_transposed && (K % 8 || N % 8) && K <= 128 && ((M + 31) / 32) * ((N + 31) / 32) * batch <= 1024) return o;
    const long row_b = b_transposed ? K : N, rows_b = batch * (b_transposed ? N : K);
    o.a = K % 8 != 0;
    o.b = row_b % 8 != 0;
    o.lda = (K + 7) / 8 * 8;
    o.ldb = (row_b + 7) / 8 * 8;
    if (o.a) o.a_bytes = ((size_t)batch * M * o.lda * 2 + 255) / 256 * 256;
    if (o.b) o.b_bytes = ((size_t)rows_b * o.ldb * 2 + 255) / 256 * 256;
    return o;
}
// Which kernels a product of more rows than the streaming kernels take runs on: small tiles (gemm_mid.hip), several to a
// compute unit and odd rows read as they are, or the 128- and 256-row tiles of this file.  A matter of the shape alone (not of the
// layout of B, of scratch or of bases), and either way with the sums in ranges of kt_per_split steps of K: the same bits on every kernel.
struct Route {
    bool mid = false;
    MidPlan plan;  // (mid: which tile)
    long splits = 1, kt_per_split = 0;
};
// One pass of 128-row tiles, up to 256 of them, or one split along K, in us (fitted to 2000 products, 15 % off).
double large_tiles_us(long M, long N, long K, long batch, long splits, long kt_per_split) {
    const double deep = K <= 2048 ? 0.0 : K >= 11585 ? 2.5 : std::log2(K / 2048.0);
    const double operands = 2e-6 * batch * ((double)M * K + (double)N * K + (double)M * N);
    const double staged = 1e-6 * ((M + 127) / 128) * ((N + 255) / 256) * batch * splits * kt_per_split * (128 + 256) * 128;
    double us = 0.67 * kt_per_split * (1.0 + 0.05 * deep);
    if (operands / 6.5 > us) us = operands / 6.5;
    if (staged / 13.3 > us) us = staged / 13.3;
    return us + 6.5 + (splits > 1 ? 4.2 + 0.25 * splits + 0.06 * 4e-6 * splits * batch * M * N : 0.0);
}
// One pass of 256-row tiles, in us (tiles of 256 x 256: fitted to 39 shapes, 8 % off)
double rounds256_us(long M, long N, long K) {
    const double rounds = (double)((((M + 255) / 256) * ((N + 255) / 256) + 255) / 256), mb = 2e-6 * ((double)M * K + (double)N * K + (double)M * N);
    const double us = rounds * (1.02 * ((K + 63) / 64) + 5.8);
    return 4.8 + (us > mb / 4.0 ? us : mb / 4.0);
}
double tiles256_us(long M, long N, long K) { return mid_pipelined(N, K) && mid_many_tiles(M, N, 1) ? large_pass_us(M, N, K, 1) : rounds256_us(M, N, K); }
// Where more than 256 tiles of 128 x 256 exist the large tiles win (2222 x 6144 x 2048 44 us against 66); below, the estimates of both
// decide, with a margin for their errors: against the large tiles alone 0.71 of the time over 1400 shapes (geometric mean), 2 of them
// slower by more than 5 % (8 at most).  Above 256 the estimates of rounds decide for a single product whose pipeline is long enough; those count
// on tiles taken in turn, which those of a batch are not (us on large tiles / as estimated: 8 x 1000 x 3000 x 384 31.1 / 38.5, 20 x 640 x 768 x 320
// 16.0 / 20.5, 14 x 1627 x 384 x 512 18.7 / 25.0; 64 x 128 x 2048 x 320 34.1 / 32.1).  Odd operands cost the large tiles a padded copy each (3.5 us
// and its traffic).
Route choose_route(long M, long N, long K, long batch) {
    Route r;
    const SplitPlan sp = tile_addressable(M, N, K, batch) ? plan_split_k(M, N, K, batch) : SplitPlan();
    r.splits = sp.splits, r.kt_per_split = sp.kt_per_split;
    const long tiles = ((M + 127) / 128) * ((N + 255) / 256) * batch, kt = (K + 63) / 64;
    const bool pipelined = sp.splits == 1 && mid_pipelined(N, K);
    if (tiles > 256 && (batch > 1 || !pipelined)) return r;
    const bool whole = N % 8 == 0 && K % 8 == 0;
    r.plan = plan_mid(M, N, K, batch, whole);
    if (r.plan.tile < 0) return r;
    if (pipelined && r.plan.splits == 1) {
        r.mid = r.plan.us < 0.97 * large_pass_us(M, N, K, batch);
        if (r.mid) r.splits = 1, r.kt_per_split = r.plan.kt_per_split;
        return r;
    }
    if (tiles > 256) return r;
    const double us = large_tiles_us(M, N, K, batch, sp.splits, sp.splits > 1 ? sp.kt_per_split : kt);
    const double copies = (K % 8 ? 7.0 : 3.5) + 0.7e-6 * batch * ((K % 8 ? (double)M * K : 0.0) + (double)K * N);
    // (where N alone is odd an [N, K] operand needs no copy: the small tiles have to win there as well)
    if (whole) r.mid = r.plan.ranges_us < 0.95 * us;
    else r.mid = r.plan.ranges_us < 0.85 * (us + copies) && (K % 8 || r.plan.ranges_us < us);
    if (r.mid) r.splits = r.plan.splits, r.kt_per_split = r.plan.kt_per_split;
    return r;
}
// What the estimates of paired products do not know is their epilogue.  On 256 x 128, a lane gates or rotates twice as many values as on 128 x 128, with
// nothing beside it on the compute unit, and so it is where workgroups take two tiles of 128 x 128 in turn.  Up to `tall_from` of K, and 2048 in the second
// case, such products (up to 256 tiles of 128 x 256) run on 128 x 128 with two stages, two workgroups to a compute unit, one's epilogue beside the other's
// steps (us as estimated / so, [K, N] and [N, K] weights).  Gated: 438 x 11904 x 288 10.8 / 8.9 and 10.9 / 8.4, 751 x 9200 x 408 13.5 / 11.8 and 13.1 / 11.4,
// 664 deep 15.7 / 15.3 and 15.7 / 13.5, but 824 deep 16.7 / 17.4 and 16.7 / 17.1; in turn 348 x 19264 x 504 13.7 / 12.4, 1589 x 4672 x 1440 31.2 / 28.7.
// Rotary: 1708 x 3072 x 1024 22.9 / 22.1 and 22.5 / 20.6, 1054 x 6144 x 640 20.3 / 17.8 and 20.0 / 16.5, 1817 x 3072 x 1152 23.7 / 24.3 and 23.8 / 22.1,
// 964 x 6144 x 1280 25.9 / 25.6 and 25.7 / 23.9, but 793 x 6144 x 1408 25.5 / 26.9 and 25.8 / 24.7; in turn 815 x 9216 x 1600 33.2 / 31.4 and 31.2 / 29.8.
constexpr long kGatedTall = 11 * 64, kRotatedTall = 20 * 64;
int paired_beside(int tile, long M, long N, long K, long tall_from) {
    if (!mid_pipelined(N, K) || mid_many_tiles(M, N, 1)) return tile;
    const bool in_turn = tile == kMidThreeStages && ((M + 127) / 128) * ((N + 127) / 128) > 256;
    return (tile == kMidTall && K <= tall_from) || (in_turn && K <= 2048) ? kMidTwoStages : tile;
}
// The gated product (N = 2 F): small tiles where they are faster by estimate (557 x 22016 x 4096: 258 tiles of 256 x 256,
// two rounds of 256, against 860 of 128 x 128).  A negative answer: tiles of 256 x 256.
int gated_tile(const MidPlan& p, long M, long N, long K) {
    // (the kernel addresses B's columns from its first with 32-bit offsets)
    return p.tile >= 0 && (double)N * K < 1e9 && p.us < 0.95 * tiles256_us(M, N, K) ? paired_beside(p.tile, M, N, K, kGatedTall) : -1;
}
// The rotary product.  Tiles of 256 x 256 round the products of a rotation as they always have, small tiles as they do: which of the two a shape
// runs on decides the last bit of a few results (16 of a million), so that is a matter of the estimates the number of K ranges follows from, and
// those of gemm_mid.hip choose among the small tiles alone.  Where more than 256 tiles of 128 x 256 exist that is 128 x 128, taken in turn where
// the pipeline is long enough for it, with two stages and two workgroups to a compute unit where it is not (us on 256 x 256 / on the one that
// small tiles then run on: 2568 x 6144 x 2048 95.5 / 76.4, 5384 x 3072 x 1024 55.1 / 54.7, 2440 x 3112 x 384 22.3 / 16.8, 6531 x 2344 x 2432 100 / 78;
// 4000 x 4608 x 256 35.9 / 29.6, 9149 x 5680 x 64 50.1 / 44.7 (60.9 with three stages); 80 shapes 0.84 in the geometric mean).  Up to 256 rows
// tiles of 256 x 256 come out in as many or fewer rounds: 156 x 61680 x 1984 59.2 / 82.9, 230 x 59600 x 64 16.9 / 18.4, 183 x 35008 x 768 28.2 / 28.8.
int rotary_tile(const MidPlan& p, long M, long N, long K) {
    const bool many = mid_many_tiles(M, N, 1);
    if (p.tile < 0 || (double)N * K >= 1e9 || (many && M <= 256) || p.ranges_us >= 0.95 * rounds256_us(M, N, K)) return -1;
    if (!many) return paired_beside(p.tile, M, N, K, kRotatedTall);
    return mid_pipelined(N, K) ? kMidThreeStages : kMidTwoStages;
}
// Whether the product alone, on the tiles of its route, and a kernel for the gate or the rotation are faster than the fused form: against the
// faster of its tiles by estimate, for the rotation too where it runs on the other ones.  (Against those, 3 of 1000 shapes more would be separate,
// and 7 of 8 of them measured slower so: fused / product + rotation in us, 9053 x 2464 x 12928 498 / 553, 10868 x 4408 x 7680 595 / 601.)
bool choose_separate(const Route& r, long M, long N, long K) {
    if (!r.mid) return r.splits > 1;  // (as large tiles: the fused forms are theirs)
    const MidPlan fused = plan_mid(M, N, K, 1, true, true);
    const double large = tiles256_us(M, N, K), best = fused.tile >= 0 && fused.us < large ? fused.us : large;
    return r.plan.us + 2.7 + 4e-6 * M * N / 5.0 < best;
}
// The estimates take about 2 us, a launch 3, and a realization matches a product several times: each thread keeps what it chose for the
// last shapes it met (pure functions of the shape).
struct Chosen {
    long M = 0, N = 0, K = 0, batch = 0;
    bool has_route = false, has_paired[2] = {}, has_separate = false, separate = false;
    Route route;
    int paired[2] = {-1, -1};  // gated, rotary
};
Chosen& chosen(long M, long N, long K, long batch) {
    static thread_local Chosen kept[32];
    const unsigned long long h = (unsigned long long)M * 0x9e3779b97f4a7c15ull ^ (unsigned long long)N * 0xc2b2ae3d27d4eb4full ^
                                 (unsigned long long)K * 0x165667b19e3779f9ull ^ (unsigned long long)batch * 0x27d4eb2f165667c5ull;
    Chosen& e = kept[(h >> 40) % 32];
    if (e.M != M || e.N != N || e.K != K || e.batch != batch) {
        e = Chosen();
        e.M = M, e.N = N, e.K = K, e.batch = batch;
    }
    return e;
}
Route route_16bit(long M, long N, long K, long batch) {
    Chosen& e = chosen(M, N, K, batch);
    if (!e.has_route) e.route = choose_route(M, N, K, batch), e.has_route = true;
    return e.route;
}
// f32 partial results of a product whose K is split
size_t partial_bytes(const Route& r, long M, long N, long batch) { return r.splits > 1 ? (size_t)r.splits * batch * M * N * sizeof(float) : 0; }
// Scratch a route takes: padded operands in front of the partial results (small tiles read odd operands as they are, but what a caller
// has to bring for them is a matter of the shape: no less than the copies).
size_t route_bytes(long M, long N, long K, long batch, bool b_transposed) {
    const OperandPadding pad = operand_padding(M, N, K, batch, b_transposed);
    const Route r = route_16bit(M, N, K, batch);
    const size_t copies = pad.a_bytes + pad.b_bytes, partial = partial_bytes(r, M, N, batch);
    return r.mid ? (copies > partial ? copies : partial) : copies + partial;
}
}  // namespace

size_t gemm_bf16_workspace_bytes(long M, long N, long K, long batch) {
    if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return 0;
    long ks = 0, kr = 0;
    // a handful of rows: streamed (one row on the vector ALUs where that kernel's plan takes the shape, more on the matrix pipes)
    if (gemm_kn_skinny_plan(M, N, K, batch, &ks, &kr)) return (size_t)ks * M * N * sizeof(float);
    if (gemm_kn_rows_plan(M, N, K, batch, &ks, &kr)) return ks > 1 ? (size_t)ks * M * N * sizeof(float) : 0;
    if (!tile_addressable(M, N, K, batch)) return 0;
    return operand_padding(M, N, K, batch, false).lda ? route_bytes(M, N, K, batch, false) : 0;
}

int gemm_bf16_static_workspace_init(int device_id) {
    if (device_id < 0 || device_id >= kMaxDevices) return (int)hipErrorInvalidDevice;
    if (g_static_ws[device_id].load(std::memory_order_acquire)) return 0;
    void* p = nullptr;  // the array's address on the current device (every device has its own copy)
    hipError_t rc = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (rc != hipSuccess) return (int)rc;
    if (!p || reinterpret_cast<uintptr_t>(p) % 256) return (int)hipErrorInvalidSymbol;
    g_static_ws[device_id].store(p, std::memory_order_release);
    return 0;
}

size_t gemm_bf16_static_workspace_capacity() { return kStaticWsBytes; }

size_t gemm_bf16_static_workspace_need(long M, long N, long K) {
    const size_t need = gemm_bf16_workspace_bytes(M, N, K, 1);
    // padded operands and partial results that do not fit: the kernel that needs no scratch and gives the same bits
    return need > kStaticWsBytes && (N % 8 || K % 8) ? 0 : need;
}

int launch_gemm_bf16_static_ws(void* stream, int device_id, const void* A, const void* B, void* C, long M, long N, long K) {
    if (device_id < 0 || device_id >= kMaxDevices) return (int)hipErrorInvalidDevice;
    const size_t need = gemm_bf16_static_workspace_need(M, N, K);
    if (need > kStaticWsBytes) return (int)hipErrorInvalidValue;
    void* ws = g_static_ws[device_id].load(std::memory_order_acquire);
    if (!ws) return (int)hipErrorNotInitialized;
    // every element of a partial tile that the reduce kernel reads is written by the split
    // kernel of the same call, so nothing has to be cleared between calls
    return launch_gemm_bf16(stream, A, B, C, M, N, K, 0, 1, need ? ws : nullptr, need);
}

bool gemm_bf16_residual_supported(long M, long N, long K, long batch);  // (defined behind tiled_shape)

namespace {
// shapes the tiled kernels take without scratch for padded operands (any M; N and K in whole 16-byte chunks)
bool tiled_shape(long M, long N, long K, long batch) { return tile_addressable(M, N, K, batch) && N % 8 == 0 && K % 8 == 0; }
}  // namespace

bool gemm_bf16_residual_supported(long M, long N, long K, long batch) { return tiled_shape(M, N, K, batch); }

bool gemm_bf16_nt_supported(long M, long N, long K, long batch) {
    // the tiled kernels (no any-shape kernel for this operand layout), or the streaming kernels for a
    // handful of rows
    return tiled_shape(M, N, K, batch) || gemm_nt_skinny_supported(M, N, K, batch) || gemm_nt_rows_supported(M, N, K, batch);
}

bool gemm_bf16_nt_padded_supported(long M, long N, long K, long batch) {
    return gemm_bf16_nt_supported(M, N, K, batch) || tile_addressable(M, N, K, batch);
}

size_t gemm_bf16_nt_workspace_bytes(long M, long N, long K, long batch) {
    if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return 0;
    if (gemm_nt_skinny_supported(M, N, K, batch) || gemm_nt_rows_supported(M, N, K, batch)) return 0;  // streamed in one launch
    if (!tile_addressable(M, N, K, batch)) return 0;
    return route_bytes(M, N, K, batch, true);
}

ProductTile gemm_16bit_tile(long M, long N, long K, long batch, bool b_transposed, int paired) {
    using namespace mrk::dev;
    ProductTile t;
    if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return t;
    if (paired) {
        const int tile = gemm_bf16_paired_tile(M, N, K, paired == 2);
        t.rows = kBM, t.cols = kBN;
        if (tile >= 0) mid_tile_shape(tile, &t.rows, &t.cols, &t.stages);
        return t;
    }
    long splits = 0, per = 0;
    if (b_transposed ? gemm_nt_skinny_supported(M, N, K, batch) || gemm_nt_rows_supported(M, N, K, batch)
                     : gemm_kn_skinny_plan(M, N, K, batch, &splits, &per) || gemm_kn_rows_plan(M, N, K, batch, &splits, &per))
        return t;
    const Route r = route_16bit(M, N, K, batch);
    const bool large = tile_addressable(M, N, K, batch) && operand_padding(M, N, K, batch, b_transposed).lda;
    const MidPlan p = r.mid ? r.plan : plan_mid(M, N, K, batch, false);
    t.k_ranges = r.splits;
    if (r.mid || (!large && p.tile >= 0)) {
        // (launch_mid's choice between the two tiles of 64 x 64)
        const bool chunks = K % 8 == 0 && (b_transposed || N % 8 == 0);
        const int tile = !r.mid ? kMidUnaligned : chunks && p.tile == kMidUnaligned ? kMidSmallest : p.tile;
        mid_tile_shape(tile, &t.rows, &t.cols, &t.stages);
    } else {
        t.rows = !large ? 32 : r.splits > 1 || ((M + 127) / 128) * ((N + kBN - 1) / kBN) * batch <= 256 ? 128 : kBM;
        t.cols = large ? kBN : 32;
    }
    return t;
}

int launch_gemm_16bit(void* stream, const void* A, const void* B, void* C, long M, long N, long K, int variant, long batch, void* workspace,
                      size_t workspace_bytes, bool b_transposed, bool f16, const void* add, bool add_is_row);

int launch_gemm_bf16_residual(void* stream, const void* A, const void* B, const void* R, void* C, long M, long N, long K, long batch,
                              bool b_transposed, bool r_is_row, void* workspace, size_t workspace_bytes, bool f16) {
    if (!R) return (int)hipErrorInvalidValue;
    return launch_gemm_16bit(stream, A, B, C, M, N, K, 0, batch, workspace, workspace_bytes, b_transposed, f16, R, r_is_row);
}

bool gemm_bf16_bias_supported(long M, long N, long K, long batch, bool b_transposed) {
    if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return false;
    return (b_transposed && gemm_nt_bias_streamed(M, N, K, batch)) || (tile_addressable(M, N, K, batch) && operand_padding(M, N, K, batch, b_transposed).lda);
}

bool gemm_bf16_bias_launchable(long M, long N, long K, long batch, bool b_transposed) { return gemm_bf16_bias_supported(M, N, K, batch, b_transposed); }

int launch_gemm_bf16_bias(void* stream, const void* a, const void* b, const void* bias, void* c, long M, long N, long K, long batch,
                          bool b_transposed, void* workspace, size_t workspace_bytes) {
    return launch_gemm_bf16_residual(stream, a, b, bias, c, M, N, K, batch, b_transposed, true, workspace, workspace_bytes);
}

bool gemm_bf16_swiglu_supported(long M, long F, long K, bool b_transposed) {
    if (M <= 0 || F <= 0 || K <= 0) return false;
    // [2F, K] form: the up rows are addressed F rows behind the gate rows with 32-bit byte offsets
    if (b_transposed && (F + 256) * K * 2 >= (1L << 32)) return false;
    if (M > 0x7fffffffL || F % 8 || K % 8 || K > (1L << 23) || 2 * F >= (1L << 25)) return false;
    const long tn = (F + 127) / 128, tm = (M + mrk::dev::kBM - 1) / mrk::dev::kBM;
    return tm * tn <= 0x7fffffffL;
}

bool gemm_bf16_separate_preferred(long M, long N, long K) {
    if (M <= 64 && K >= 512) return true;  // (the programs a block over a few tokens consists of stay as they are)
    const Route r = route_16bit(M, N, K, 1);
    Chosen& e = chosen(M, N, K, 1);
    if (!e.has_separate) e.separate = choose_separate(r, M, N, K), e.has_separate = true;
    return e.separate;
}

int gemm_bf16_paired_tile(long M, long N, long K, bool rotary) {
    if (M <= 0 || N <= 0 || K <= 0) return -1;
    Chosen& e = chosen(M, N, K, 1);
    if (!e.has_paired[rotary]) {
        const MidPlan p = plan_mid(M, N, K, 1, true, true);
        e.paired[rotary] = rotary ? rotary_tile(p, M, N, K) : gated_tile(p, M, N, K), e.has_paired[rotary] = true;
    }
    return e.paired[rotary];
}

int launch_gemm_bf16_swiglu(void* stream, const void* A, const void* B, void* C, long M, long F, long K, bool b_transposed, int tile) {
    using namespace mrk::dev;
    if (M <= 0 || F <= 0) return 0;
    if (!gemm_bf16_swiglu_supported(M, F, K, b_transposed)) return (int)hipErrorInvalidValue;
    if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C)) % 16) return (int)hipErrorInvalidValue;
    // a handful of rows against a [2F, K] weight: the gated form of the streaming kernel
    if (b_transposed && gemm_nt_swiglu_streamed(M, F, K)) return launch_gemm_nt_swiglu_streamed(stream, A, B, C, M, F, K);
    hipStream_t s = static_cast<hipStream_t>(stream);
    (void)hipGetLastError();
    if (tile == kChooseTile) tile = gemm_bf16_paired_tile(M, 2 * F, K, false);
    if (tile >= 0) return launch_gemm_mid_paired(s, tile, A, B, C, M, 2 * F, K, b_transposed, nullptr);
    const long tn = (F + 127) / 128, tm = (M + kBM - 1) / kBM;
    const dim3 grid((unsigned)(tm * tn), 1);
    const __bf16* a = static_cast<const __bf16*>(A);
    const __bf16* b = static_cast<const __bf16*>(B);
    __bf16* c = static_cast<__bf16*>(C);
    const bool any = K % kBK != 0;
    auto kernel = b_transposed ? (any ? gemm_bf16_nt_tile256_swiglu_any : gemm_bf16_nt_tile256_swiglu)
                               : (any ? gemm_bf16_tile256_swiglu_any : gemm_bf16_tile256_swiglu);
    kernel<<<grid, 256, 0, s>>>(a, b, c, (int)M, (int)(2 * F), (int)K, (int)tm, (int)tn, (int)K, b_transposed ? (int)K : (int)(2 * F));
    return (int)hipGetLastError();
}

bool gemm_bf16_rope_supported(long M, long N, long K, long split, long seq) {
    using namespace mrk::dev;
    return M > 0 && N > 0 && K > 0 && seq > 0 && K % kBK == 0 && N % 8 == 0 && split > 0 && split <= N && split % kBN == 0 &&
           M <= 0x7fffffffL && N < (1L << 25) && K <= (1L << 23) && ((M + kBM - 1) / kBM) * ((N + kBN - 1) / kBN) <= 0x7fffffffL;
}

int launch_gemm_bf16_rope(void* stream, const void* A, const void* B, void* C_rot, void* C_rest, long M, long N, long K, long split,
                          const void* cos, const void* sin, long seq, bool b_transposed, int tile) {
    using namespace mrk::dev;
    if (!gemm_bf16_rope_supported(M, N, K, split, seq) || !A || !B || !C_rot || !cos || !sin || (split < N && !C_rest))
        return (int)hipErrorInvalidValue;
    const uintptr_t all = reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C_rot) |
                          reinterpret_cast<uintptr_t>(C_rest) | reinterpret_cast<uintptr_t>(cos) | reinterpret_cast<uintptr_t>(sin);
    if (all % 16 || reinterpret_cast<uintptr_t>(cos) % 32 || reinterpret_cast<uintptr_t>(sin) % 32) return (int)hipErrorInvalidValue;
    (void)hipGetLastError();
    if (tile == kChooseTile) tile = gemm_bf16_paired_tile(M, N, K, true);
    if (tile >= 0) {
        const MidRope angles{static_cast<const float*>(cos), static_cast<const float*>(sin), C_rest, (int)seq, (int)split};
        return launch_gemm_mid_paired(static_cast<hipStream_t>(stream), tile, A, B, C_rot, M, N, K, b_transposed, &angles);
    }
    const long tm = (M + kBM - 1) / kBM, tn = (N + kBN - 1) / kBN;
    RopeEpilogue rope{static_cast<const float*>(cos), static_cast<const float*>(sin), static_cast<__bf16*>(C_rest), (int)seq, (int)split};
    auto kernel = b_transposed ? gemm_bf16_nt_tile256_rope : gemm_bf16_tile256_rope;
    kernel<<<dim3((unsigned)(tm * tn)), 256, 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<const __bf16*>(A), static_cast<const __bf16*>(B), static_cast<__bf16*>(C_rot), (int)M, (int)N, (int)K, (int)tm, (int)tn, rope);
    return (int)hipGetLastError();
}

namespace {
// C = the sums over `splits` partial results W[splits][batch][M][N], with the addend
void reduce_partials(hipStream_t s, const float* w, __bf16* c, long M, long N, long batch, long splits, bool f16, const __bf16* add, bool add_is_row) {
    using namespace mrk::dev;
    const long total = batch * M * N;
    const bool each = total % 8 != 0 || (add_is_row && N % 8 != 0) || (reinterpret_cast<uintptr_t>(c) | reinterpret_cast<uintptr_t>(add)) % 16;
    auto reduce_kernel = f16 ? (each ? gemm_splitk_reduce<true, true> : gemm_splitk_reduce<true, false>)
                             : (each ? gemm_splitk_reduce<false, true> : gemm_splitk_reduce<false, false>);
    reduce_kernel<<<(unsigned)(((each ? total : total / 8) + 255) / 256), 256, 0, s>>>(w, c, total, (int)splits, add, add_is_row ? N : 0);
}

// Output tiles over the chip: the K loop spread over ranges when the shape has a split plan and the caller brought the
// scratch for the partial results, else one pass of 256-row or 128-row tiles.  Operands aligned to 16 bytes; those whose
// rows are no whole 16-byte chunks are padded into the scratch first.  False when the scratch for that is missing.
bool launch_tiles(hipStream_t s, const void* A, const void* B, void* C, long M, long N, long K, int variant, long batch, void* workspace,
                  size_t workspace_bytes, bool b_transposed, bool f16, const __bf16* add, bool add_is_row, const Route& route) {
    using namespace mrk::dev;
    const OperandPadding pad = operand_padding(M, N, K, batch, b_transposed);
    const __bf16 *a = static_cast<const __bf16*>(A), *b = static_cast<const __bf16*>(B);
    __bf16* c = static_cast<__bf16*>(C);
    char* ws = static_cast<char*>(workspace);
    size_t ws_left = reinterpret_cast<uintptr_t>(workspace) % 16 == 0 && workspace ? workspace_bytes : 0;
    if (pad.a_bytes + pad.b_bytes > ws_left || !pad.lda) return false;
    auto padded = [&](const __bf16* src, long rows, long cols, long pitch, size_t bytes) {
        const long groups = (rows + 3) / 4;
        const dim3 grid((unsigned)(groups < (1L << 20) ? groups : (1L << 20)), (unsigned)((pitch / 8 + kRepitchRun - 1) / kRepitchRun));
        gemm_repitch<<<grid, 256, 0, s>>>(
            reinterpret_cast<const unsigned short*>(src), reinterpret_cast<unsigned short*>(ws), rows, (int)cols, (int)pitch);
        const __bf16* at = reinterpret_cast<const __bf16*>(ws);
        ws += bytes;
        ws_left -= bytes;
        return at;
    };
    if (pad.a) a = padded(a, batch * M, K, pad.lda, pad.a_bytes);
    if (pad.b) b = padded(b, batch * (b_transposed ? N : K), b_transposed ? K : N, pad.ldb, pad.b_bytes);
    const bool any = K % kBK != 0 || N % 8 != 0;
    const int pitch_a = (int)pad.lda, pitch_b = (int)pad.ldb;
    const long tn = (N + kBN - 1) / kBN, tm128 = (M + 127) / 128;
#define MRK_PICK(stem) (f16 ? (b_transposed ? (any ? gemm_f16_nt_##stem##_any : gemm_f16_nt_##stem) : (any ? gemm_f16_##stem##_any : gemm_f16_##stem)) \
                            : (b_transposed ? (any ? gemm_bf16_nt_##stem##_any : gemm_bf16_nt_##stem) : (any ? gemm_bf16_##stem##_any : gemm_bf16_##stem)))
    const size_t partial = variant == 0 || variant == 5 ? partial_bytes(route, M, N, batch) : 0;
    if (partial && ws_left >= partial && batch * route.splits <= 65535) {
        float* w = reinterpret_cast<float*>(ws);
        MRK_PICK(tile128_splitk)<<<dim3((unsigned)(tm128 * tn), (unsigned)batch, (unsigned)route.splits), 256, 0, s>>>(
            a, b, w, (int)M, (int)N, (int)K, (int)tm128, (int)tn, (int)route.kt_per_split, pitch_a, pitch_b);
        reduce_partials(s, w, c, M, N, batch, route.splits, f16, add, add_is_row);
        return true;
    }
    // the 128-row tile when all its workgroups are resident at once (at most one per compute unit): twice the
    // workgroups of the 256-row tile for the same work.  3 / 4 force one.
    const bool small = variant == 4 || (variant != 3 && tm128 * tn * batch <= 256);
    const long tm = small ? tm128 : (M + kBM - 1) / kBM;
    const dim3 grid((unsigned)(tm * tn), (unsigned)batch);
    if (add) {
        auto kernel = small ? MRK_PICK(tile128_residual) : MRK_PICK(tile256_residual);
        kernel<<<grid, 256, 0, s>>>(a, b, add, c, (int)M, (int)N, (int)K, (int)tm, (int)tn, add_is_row ? 0 : -1, pitch_a, pitch_b);
    } else {
        auto kernel = small ? MRK_PICK(tile128) : MRK_PICK(tile256);
        kernel<<<grid, 256, 0, s>>>(a, b, c, (int)M, (int)N, (int)K, (int)tm, (int)tn, pitch_a, pitch_b);
    }
#undef MRK_PICK
    return true;
}
}  // namespace

namespace {
// Small tiles, in the route's ranges of K: odd rows and bases are read as they are (`chunks`: rows of whole 16-byte chunks on 16-byte
// bases, in this layout).  A negative answer: not covered (K or N below one chunk, or no scratch for the partial results).
int launch_mid(hipStream_t s, const void* A, const void* B, void* C, long M, long N, long K, long batch, void* workspace, size_t workspace_bytes,
               bool b_transposed, bool f16, const __bf16* add, bool add_is_row, const Route& route, bool chunks) {
    MidPlan p = route.mid ? route.plan : plan_mid(M, N, K, batch, false);
    if (p.tile < 0) return -1;
    if (!route.mid || (!chunks && N % 8 == 0 && K % 8 == 0)) p.tile = kMidUnaligned;
    else if (chunks && p.tile == kMidUnaligned) p.tile = kMidSmallest;  // (odd rows of C alone)
    p.splits = route.splits, p.kt_per_split = route.kt_per_split;
    const size_t partial = partial_bytes(route, M, N, batch);
    if (partial && (!workspace || workspace_bytes < partial || reinterpret_cast<uintptr_t>(workspace) % 16 || batch * p.splits > 65535)) return -1;
    int rc = launch_gemm_mid(s, p, A, B, C, static_cast<float*>(workspace), add, add_is_row ? 0 : N, M, N, K, batch, b_transposed, f16);
    if (rc == 0 && partial) {
        reduce_partials(s, static_cast<float*>(workspace), static_cast<__bf16*>(C), M, N, batch, p.splits, f16, add, add_is_row);
        rc = (int)hipGetLastError();
    }
    return rc;
}

// One wave per 32 x 32 tile, any shape, no scratch.
int launch_generic(hipStream_t s, const void* A, const void* B, void* C, long M, long N, long K, long batch, bool b_transposed, bool f16,
                   const __bf16* add, bool add_is_row, const Route& route) {
    using namespace mrk::dev;
    const long tn = (N + 31) / 32, total = ((M + 31) / 32) * tn, blocks = (total + 3) / 4;
    if (blocks > 0x7fffffffL) return (int)hipErrorInvalidValue;
    // (the K ranges the other kernels take: the result does not depend on whether there was scratch for them)
    const int k_range = route.splits > 1 ? (int)route.kt_per_split * kBK : 0x7fffffff;
    auto kernel = f16 ? (b_transposed ? gemm_bf16_generic<true, true> : gemm_bf16_generic<true, false>)
                      : (b_transposed ? gemm_bf16_generic<false, true> : gemm_bf16_generic<false, false>);
    kernel<<<dim3((unsigned)blocks, (unsigned)batch), 256, 0, s>>>(static_cast<const __bf16*>(A), static_cast<const __bf16*>(B),
                                                                  static_cast<__bf16*>(C), (int)M, (int)N, (int)K, (int)tn, total, k_range, add,
                                                                  add_is_row ? 0 : N);
    return (int)hipGetLastError();
}
}  // namespace

// The product, with `add` (a matrix of C's shape or, add_is_row, one row [N]; of C's type) added to the rounded result by
// whichever kernel writes it: the streaming kernels, the split-K reduction or the tiled kernels' residual epilogue.
int launch_gemm_16bit(void* stream, const void* A, const void* B, void* C, long M, long N, long K, int variant, long batch, void* workspace,
                      size_t workspace_bytes, bool b_transposed, bool f16, const void* add, bool add_is_row) {
    using namespace mrk::dev;
    if (M <= 0 || N <= 0 || batch <= 0) return 0;
    if (add && reinterpret_cast<uintptr_t>(add) % 16) return (int)hipErrorInvalidValue;
    const __bf16* addp = static_cast<const __bf16*>(add);
    if (batch > 65535) return (int)hipErrorInvalidValue;  // grid y extent
    if (M > 0x7fffffffL || N > 0x7fffffffL || K > 0x7fffffffL || K < 0) return (int)hipErrorInvalidValue;
    hipStream_t s = static_cast<hipStream_t>(stream);
    (void)hipGetLastError();
    const bool aligned = ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C)) % 16) == 0;
    const bool choose = variant == 0 || variant == 5;  // (3 / 4 force a tile size, 2 the any-shape kernel)
    if (b_transposed) {
        // B given as Bt[N, K]: the streaming or the tiled kernels, or nothing
        if (!aligned || !gemm_bf16_nt_padded_supported(M, N, K, batch)) return (int)hipErrorInvalidValue;
        // up to 64 rows: one pass over the weight streams it faster than any tile (one or two rows on the
        // vector ALUs, more on the matrix pipes with 16-row blocks staged through LDS)
        if (choose || !tiled_shape(M, N, K, batch)) {
            if (add) {
                if (gemm_nt_bias_streamed(M, N, K, batch)) return launch_gemm_nt_bias_streamed(stream, A, B, add, C, M, N, K, f16, add_is_row);
            } else {
                if (gemm_nt_skinny_supported(M, N, K, batch)) return launch_gemm_nt_skinny(stream, A, B, C, M, N, K, batch, f16);
                if (gemm_nt_rows_supported(M, N, K, batch)) return launch_gemm_nt_rows(stream, A, B, C, M, N, K, batch, f16);
            }
        }
        if (!tile_addressable(M, N, K, batch)) return (int)hipErrorInvalidValue;
        const OperandPadding pad = operand_padding(M, N, K, batch, true);
        const Route route = route_16bit(M, N, K, batch);
        // (odd operands want scratch for their copies, whichever kernel runs)
        if (pad.a_bytes + pad.b_bytes > (workspace && reinterpret_cast<uintptr_t>(workspace) % 16 == 0 ? workspace_bytes : 0)) return (int)hipErrorInvalidValue;
        if (choose && route.mid) {
            const int rc = launch_mid(s, A, B, C, M, N, K, batch, workspace, workspace_bytes, true, f16, addp, add_is_row, route, K % 8 == 0);
            if (rc >= 0) return rc;
        }
        if (!launch_tiles(s, A, B, C, M, N, K, variant, batch, workspace, workspace_bytes, true, f16, addp, add_is_row, route))
            return (int)hipErrorInvalidValue;
        return (int)hipGetLastError();
    }
    // up to 16 rows: one streaming pass over the weight into f32 partial sums, then their sum
    {
        long ks = 0, kr = 0;
        if (choose && aligned && gemm_kn_skinny_plan(M, N, K, batch, &ks, &kr) && workspace &&
            workspace_bytes >= (size_t)ks * M * N * sizeof(float) && reinterpret_cast<uintptr_t>(workspace) % 16 == 0) {
            return launch_gemm_kn_skinny(stream, A, B, C, workspace, M, N, K, ks, kr, f16, add, add_is_row);
        }
        if (choose && aligned && gemm_kn_rows_plan(M, N, K, batch, &ks, &kr) &&
            (ks == 1 || (workspace && workspace_bytes >= (size_t)ks * M * N * sizeof(float) && reinterpret_cast<uintptr_t>(workspace) % 16 == 0))) {
            return launch_gemm_kn_rows(stream, A, B, C, workspace, M, N, K, ks, kr, f16, add, add_is_row);
        }
    }
    OperandPadding pad;
    Route route;
    if (K > 0) {
        pad = operand_padding(M, N, K, batch, false);
        route = route_16bit(M, N, K, batch);
    }
    // (an addend is taken where there is scratch for the tiles, whichever kernel runs)
    if (add && (!aligned || variant == 2 || !tile_addressable(M, N, K, batch) || !pad.lda ||
                pad.a_bytes + pad.b_bytes > (workspace && reinterpret_cast<uintptr_t>(workspace) % 16 == 0 ? workspace_bytes : 0)))
        return (int)hipErrorInvalidValue;
    const bool whole = N % 8 == 0 && K % 8 == 0;
    if (choose && K > 0 && route.mid) {
        const int rc = launch_mid(s, A, B, C, M, N, K, batch, workspace, workspace_bytes, false, f16, addp, add_is_row, route, aligned && whole);
        if (rc >= 0) return rc;
    }
    if (variant != 2 && aligned && tile_addressable(M, N, K, batch) &&
        launch_tiles(s, A, B, C, M, N, K, variant, batch, workspace, workspace_bytes, false, f16, addp, add_is_row, route))
        return (int)hipGetLastError();
    // no scratch for padded operands, or unaligned bases
    if (choose && K > 0) {
        const int rc = launch_mid(s, A, B, C, M, N, K, batch, workspace, workspace_bytes, false, f16, addp, add_is_row, route, false);
        if (rc >= 0) return rc;
    }
    return launch_generic(s, A, B, C, M, N, K, batch, false, f16, addp, add_is_row, route);
}

int launch_gemm_bf16(void* stream, const void* A, const void* B, void* C, long M, long N, long K, int variant, long batch, void* workspace,
                     size_t workspace_bytes, bool b_transposed, bool f16) {
    return launch_gemm_16bit(stream, A, B, C, M, N, K, variant, batch, workspace, workspace_bytes, b_transposed, f16, nullptr, false);
}

}  // namespace mrk

