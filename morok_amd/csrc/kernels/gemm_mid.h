// The 16-bit product kernel on small tiles (gemm_mid.hip), as the dispatch in gemm_bf16.hip uses it.
#pragma once
#include <hip/hip_runtime.h>

namespace mrk {

// Which tile, how many ranges of K of how many 64-deep steps, and the time estimated for it; tile < 0: not covered.
struct MidPlan {
    int tile = -1;
    long splits = 1, kt_per_split = 0;
    double us = 0.0;
    double ranges_us = 0.0;  // what the number of ranges follows from (us, where that is more than one), and the rounding of a rotation
};
constexpr int kMidTwoStages = 0, kMidThreeStages = 1;  // tiles of 128 x 128
constexpr int kMidSmallest = 3, kMidUnaligned = 4;  // tiles of 64 x 64: rows of whole chunks; rows that start on any element
constexpr int kMidTall = 5;                         // tiles of 256 x 128
// The fastest by estimate.  whole_chunks: rows of both operands are whole 16-byte chunks on 16-byte bases, whichever way B is stored; else
// (N and K at least 8) they are read element-aligned.  paired: for the gated or the rotary epilogue, K in one range.
MidPlan plan_mid(long M, long N, long K, long batch, bool whole_chunks, bool paired = false);
// Whether a product of these extents in one range of K is a matter of the estimates below: long enough for a pipeline, whole chunks.
inline bool mid_pipelined(long N, long K) { return N % 8 == 0 && K % 8 == 0 && K > 256; }
inline bool mid_many_tiles(long M, long N, long batch) { return ((M + 127) / 128) * ((N + 255) / 256) * batch > 256; }
// One pass of the tiles of gemm_bf16.hip (256 x 256, up to 256 tiles of 128 x 256 those) over such a product, in us
double large_pass_us(long M, long N, long K, long batch);
// rows, columns and stages of a tile
void mid_tile_shape(int tile, int* rows, int* cols, int* stages);
// C = A B (B [K, N] or, b_transposed, [N, K]); with p.splits > 1 the partial sums W[splits][batch][M][N] instead, without
// the addend.  add (may be null): rows add_pitch elements apart (0: one row) of C's type.
int launch_gemm_mid(hipStream_t s, const MidPlan& p, const void* A, const void* B, void* C, float* W, const void* add, long add_pitch, long M, long N, long K,
                    long batch, bool b_transposed, bool f16);

// Rotary epilogue: angles [seq, 64] of a row's position (row % seq); columns from `split` (a multiple of 128) on go to rest [M, N - split].
struct MidRope {
    const float* cos = nullptr;
    const float* sin = nullptr;
    void* rest = nullptr;
    int seq = 1, split = 0;
};
// bf16 products of whole chunks with an epilogue that pairs columns: the gated one (rope null; B holds F = N / 2 gate columns, then F up
// columns: C [M, F]) and the rotary one (C [M, rope->split]).  K in one range.
int launch_gemm_mid_paired(hipStream_t s, int tile, const void* A, const void* B, void* C, long M, long N, long K, bool b_transposed,
                           const MidRope* rope);

}  // namespace mrk
