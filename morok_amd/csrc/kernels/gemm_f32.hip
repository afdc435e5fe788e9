// f32 products on the matrix pipes: C[M, N] = A[M, K] B (+ a row or a matrix), every operand and every sum in f32
// (v_mfma_f32_32x32x2_f32: 64 flops per cycle and SIMD, twice the vector ALUs' rate without packed arithmetic).  B is
// [K, N], or (kNT) [N, K] as a Linear layer stores its weight.  Any M, N, K.
//
// Which k a matrix instruction multiplies is free as long as both operands agree: lane half g = lane / 32 holds the four
// consecutive k = 8 c + 4 g .. + 3 of chunk c, so that one 16-byte read feeds four instructions, the i-th of them
// adding the products of k = 8 c + i and 8 c + 4 + i.
//
// Two kernels:
//  - f32_tiled: a workgroup of eight waves owns a 64 x 64 (128 x 128) tile of C; four waves (2 x 2) share the tile, and two
//    such groups halve every K step and add their sums at the end: two waves per SIMD, so that one's reads of the
//    local memory run under the other's matrix instructions, and two shorter chains of additions.  Global ->
//    registers -> local memory, one step ahead, two stages, one barrier per step.
//  - f32_direct: few output tiles.  A workgroup owns one 32 x 32 tile and its 4 (16) waves split K; a wave's operands
//    go from memory straight to registers, a batch of loads ahead of the matrix instructions, and the waves' sums
//    meet in local memory, added in the waves' order.  No barrier until then: a small product is one trip to memory.
// Both add in an order that depends on the shape alone.  Error against 64 bits (2-norm, uniform operands, K = 1024): tiled
// 4.0e-7, direct 1.6e-7; one chain of K fused multiply-adds, as the generated kernel has, 5.8e-7.
// Bound by the f32 matrix rate (157 TFLOP/s nominal).  Measured: 1024^3 25.9 us (83 TFLOP/s; generated kernel on the vector
// ALUs 55.3), 4096^3 1.20 ms (114 TFLOP/s), 64 x 256 x 784 against a [N, K] weight 4.3 us (36.8 and a transposing copy before).
// What is left at 1024^3, one workgroup per CU: the fill and drain of sixteen steps, and the barrier in each.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kernels.h"

namespace mrk::dev {

typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace {

// Four elements of one row: p points at the row, k .. k + 3 of `n` elements; past the end zeros (kZero), or whatever
// the last elements hold (columns that are not stored).  kVec: rows are whole 16-byte chunks, so a group is
// inside or outside as a whole.
template <bool kVec, bool kZero>
__device__ __forceinline__ f32x4v load4(const float* p, long k, long n) {
    f32x4v v = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (kVec) {
        if (k < n) v = *reinterpret_cast<const f32x4v*>(p + k);
        else if (!kZero) v = *reinterpret_cast<const f32x4v*>(p + n - 4);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const long c = k + i < n ? k + i : n - 1;
            const float x = p[c];
            v[i] = kZero && k + i >= n ? 0.0f : x;
        }
    }
    return v;
}

// kAdd: 0 nothing, 1 one row [N], 2 a matrix of C's shape
template <int kAdd>
__device__ __forceinline__ void store_c(float* __restrict__ C, const float* __restrict__ add, long M, long N, long row, long col, float v) {
    if (row < M && col < N) {
        if constexpr (kAdd == 1) v += add[col];
        if constexpr (kAdd == 2) v += add[row * N + col];
        C[row * N + col] = v;
    }
}

// row of C inside a 32 x 32 block that register e of lane l holds (its column is l % 32)
__device__ __forceinline__ int c_row(int e, int lane) { return 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); }

}  // namespace

template <int kT, bool kNT, bool kVec, int kAdd>
__device__ __forceinline__ void f32_tiled_body(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                                               const float* __restrict__ add, long M, long N, long K, int tiles_m, int tiles_n) {
    constexpr int kBM = 64 * kT, kBN = 64 * kT;
    constexpr int kBK = kT == 1 ? 64 : 32;   // K step of the workgroup; each group of four waves takes half of it
    constexpr int kChunks = kBK / 16;        // 8-deep chunks per step and group
    constexpr int kSlots = kBK / 4;          // 16-byte slots of a row of either tile in local memory, k contiguous
    constexpr int kAF = kBM * kBK, kBF = kBN * kBK;
    constexpr int kStage = kAF + kBF;
    __shared__ __attribute__((aligned(16))) float smem[2 * kStage];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
    const int lr = lane & 31, lg = lane >> 5;
    // Workgroups congruent mod 8 share an L2: each such set takes a run of consecutive tiles, walked in bands of four
    // rows of tiles, so that it reads a few rows of A and of B many times instead of all of both.
    int tm, tn;
    {
        const int n = tiles_m * tiles_n;
        int t = blockIdx.x;
        if ((n & 7) == 0) t = (t & 7) * (n >> 3) + (t >> 3);
        const int band = t / (4 * tiles_n), first = band * 4;
        const int rows = tiles_m - first < 4 ? tiles_m - first : 4;
        const int in = t - band * 4 * tiles_n;
        tm = first + in % rows;
        tn = in / rows;
    }
    const long m0 = (long)tm * kBM, n0 = (long)tn * kBN;

    // Slot c of row r lies at c ^ swizzle(r).  The local memory serves 16 lanes of 16 bytes from its 64 banks at a time: 16
    // consecutive rows (a fragment read) and 16 rows four apart (the stores of a transposed block) fall into
    // different banks (rows of 128 bytes: two of the latter share one).
    auto swizzle = [](int r) { return kT == 1 ? ((r >> 2) & 3) | (((r ^ (r >> 4)) & 3) << 2) : ((r >> 1) & 7) ^ ((r >> 4) & 1); };
    // staging: waves 4-7 move A, waves 0-3 move B, four 16-byte groups per thread and step; of a [K, N] matrix a block of
    // four rows by four columns, which goes to local memory transposed, so that both fragments are read alike
    const bool moves_a = wave >= 4;
    const int tq = tid & 255;
    // Group i of a step that starts at k0 lies at pr[i] + min(at + kr[i] * pitch, last * pitch) with at = k0 * pitch: the address
    // of a group past the end of K is pulled back inside, and what it brought is cleared on the way to local memory.  No branch
    // around the loads: the compiler can only count how many are in flight in straight code.
    const bool transpose = !kNT && !moves_a;
    const float* pr[4];
    int kr[4], to[4];
    const long bn = n0 + 4 * (tq % (kBN / 4));
    const long pitch = transpose ? N : 1, last = (transpose || !kVec ? K - 1 : K - 4) * pitch;
    const long step_pitch = kBK * pitch;
    long at = 0, ofs[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (!transpose) {
            const float* base = moves_a ? A : B;
            const long first = moves_a ? m0 : n0, end = moves_a ? M : N;
            const int r = tq / kSlots + i * (256 / kSlots);
            pr[i] = base + (first + r < end ? first + r : end - 1) * K;
            kr[i] = 4 * (tq % kSlots);
            ofs[i] = kr[i];
            to[i] = (moves_a ? 0 : kAF) + r * kBK + (((tq % kSlots) ^ swizzle(r)) << 2);
        } else {
            const int r = 4 * (tq % (kBN / 4)) + i, k = 4 * (tq / (kBN / 4));
            pr[i] = B + (bn + 4 <= N || !kVec ? bn : N - 4);
            kr[i] = k + i;
            ofs[i] = kr[i] * N;
            to[i] = kAF + r * kBK + (((k >> 2) ^ swizzle(r)) << 2);
        }
    }
    auto fetch = [&](f32x4v(&v)[4]) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const long o = at + ofs[i];
            if constexpr (kVec) {
                v[i] = *reinterpret_cast<const f32x4v*>(pr[i] + (o < last ? o : last));
            } else {
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    const long c = bn + x < N ? x : N - 1 - bn, ox = transpose ? o : o + x;
                    v[i][x] = pr[i][(ox < last ? ox : last) + (transpose ? c : 0)];
                }
            }
        }
        at += step_pitch;
        __builtin_amdgcn_sched_barrier(0);  // the loads set out before the step's matrix instructions, not after them
    };
    auto stash = [&](float* st, long k0, const f32x4v(&v)[4]) {
        f32x4v z[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int x = 0; x < 4; x++) z[i][x] = k0 + kr[i] + (transpose || kVec ? 0 : x) < K ? v[i][x] : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++)
            *reinterpret_cast<f32x4v*>(st + to[i]) = transpose ? f32x4v{z[0][i], z[1][i], z[2][i], z[3][i]} : z[i];
    };

    f32x16 acc[kT][kT];
#pragma unroll
    for (int i = 0; i < kT; i++)
#pragma unroll
        for (int j = 0; j < kT; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0.0f;

    const long steps = (K + kBK - 1) / kBK;
    // Step s multiplies stage s & 1 while step s + 1's operands are on their way to registers since step s - 1 (an L2 miss
    // takes longer than a step) and step s + 2's set out.
    f32x4v in0[4], in1[4];
    auto step = [&](long s, f32x4v(&arriving)[4], f32x4v(&leaving)[4]) {
        const float* st = smem + (s & 1) * kStage;
        fetch(leaving);
        const int slot = group * (kSlots / 2) + lg;
        f32x4v fa[2][kT], fb[2][kT];
        auto fragments = [&](int c) {
#pragma unroll
            for (int i = 0; i < kT; i++) {
                const int ra = (wm * kT + i) * 32 + lr, rb = (wn * kT + i) * 32 + lr;
                fa[c & 1][i] = *reinterpret_cast<const f32x4v*>(st + ra * kBK + (((slot + 2 * c) ^ swizzle(ra)) << 2));
                fb[c & 1][i] = *reinterpret_cast<const f32x4v*>(st + kAF + rb * kBK + (((slot + 2 * c) ^ swizzle(rb)) << 2));
            }
        };
        fragments(0);
#pragma unroll
        for (int c = 0; c < kChunks; c++) {
            if (c + 1 < kChunks) fragments(c + 1);
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int i = 0; i < kT; i++)
#pragma unroll
                    for (int j = 0; j < kT; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[c & 1][i][x], fb[c & 1][j][x], acc[i][j], 0, 0, 0);
            // (a chunk's fragments are read under the matrix instructions of the chunk before)
            if (c + 1 < kChunks) {
                if (c == 0) __builtin_amdgcn_sched_group_barrier(0x100, 2 * kT, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2 * kT, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x8, 4 * kT * kT, 0);
        }
        // (the other stage was last read in step s - 1, which every wave has left at the barrier before this step)
        stash(smem + ((s + 1) & 1) * kStage, (s + 1) * kBK, arriving);
        __syncthreads();
    };
    fetch(in0);
    fetch(in1);
    stash(smem, 0, in0);
    __syncthreads();
    for (long s = 0; s + 1 < steps; s += 2) {
        step(s, in1, in0);
        step(s + 1, in0, in1);
    }
    if (steps & 1) step(steps - 1, in1, in0);
    // the second group hands its sums over through local memory (all reads of the stages are behind the last barrier)
    static_assert(4 * kT * kT * 16 * 64 <= 2 * kStage, "the second group's sums fit into the stages");
    float* x = smem + (wave & 3) * (kT * kT * 16 * 64) + lane;
    if (group == 1) {
#pragma unroll
        for (int i = 0; i < kT; i++)
#pragma unroll
            for (int j = 0; j < kT; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) x[((i * kT + j) * 16 + e) * 64] = acc[i][j][e];
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
        for (int i = 0; i < kT; i++)
#pragma unroll
            for (int j = 0; j < kT; j++)
#pragma unroll
                for (int e = 0; e < 16; e++)
                    store_c<kAdd>(C, add, M, N, m0 + (wm * kT + i) * 32 + c_row(e, lane), n0 + (wn * kT + j) * 32 + lr,
                                  acc[i][j][e] + x[((i * kT + j) * 16 + e) * 64]);
    }
}

template <int kT, bool kNT, bool kVec, int kAdd>
__global__ void __launch_bounds__(512, kT == 1 && kVec ? 4 : 2) f32_tiled(const float* A, const float* B, float* C, const float* add, long M, long N, long K, int tiles_m,
                                                 int tiles_n) {
    f32_tiled_body<kT, kNT, kVec, kAdd>(A, B, C, add, M, N, K, tiles_m, tiles_n);
}

// kWaves waves split K into runs of whole chunks (of eight for tiles of 32, of sixteen for tiles of 16, whose lane groups
// are four)
template <int kTile, int kWaves, bool kNT, bool kVec, int kAdd>
__global__ void __launch_bounds__(kWaves * 64) f32_direct(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                                                          const float* __restrict__ add, long M, long N, long K, int tiles_n) {
    constexpr int kBatch = 4;  // chunks whose loads are in flight together
    constexpr int kDeep = 4 * (64 / kTile), kOut = kTile * kTile;
    using Acc = std::conditional_t<kTile == 32, f32x16, f32x4v>;
    __shared__ float sums[kWaves * kOut];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane % kTile, lg = lane / kTile;
    const int tm = blockIdx.x / tiles_n, tn = blockIdx.x - tm * tiles_n;
    const long m0 = (long)tm * kTile, n0 = (long)tn * kTile;
    const long row = m0 + lr < M ? m0 + lr : M - 1, col = n0 + lr < N ? n0 + lr : N - 1;
    const float* pa = A + row * K;
    const float* pb = kNT ? B + col * K : B + col;
    const long chunks = (K + kDeep - 1) / kDeep, per = (chunks + kWaves - 1) / kWaves;
    const long c0 = wave * per, c1 = c0 + per < chunks ? c0 + per : chunks;
    Acc acc;
#pragma unroll
    for (int e = 0; e < kOut / 64; e++) acc[e] = 0.0f;
    f32x4v fa[2][kBatch], fb[2][kBatch];
    auto fetch = [&](long c, f32x4v(&a)[kBatch], f32x4v(&b)[kBatch]) {
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
            // chunks past this wave's run multiply zeros
            const long k = c + i < c1 ? (c + i) * kDeep + 4 * lg : K;
            a[i] = load4<kVec, true>(pa, k, K);
            if constexpr (kNT) {
                b[i] = load4<kVec, true>(pb, k, K);
            } else {
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    const float v = pb[(k + x < K ? k + x : K - 1) * N];
                    b[i][x] = k + x < K ? v : 0.0f;
                }
            }
        }
    };
    auto multiply = [&](f32x4v(&a)[kBatch], f32x4v(&b)[kBatch]) {
#pragma unroll
        for (int i = 0; i < kBatch; i++)
#pragma unroll
            for (int x = 0; x < 4; x++) {
                if constexpr (kTile == 32) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][x], b[i][x], acc, 0, 0, 0);
                else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][x], b[i][x], acc, 0, 0, 0);
            }
    };
    if (c0 < c1) {
        fetch(c0, fa[0], fb[0]);
        for (long c = c0; c < c1; c += 2 * kBatch) {
            if (c + kBatch < c1) fetch(c + kBatch, fa[1], fb[1]);
            multiply(fa[0], fb[0]);
            if (c + kBatch < c1) {
                if (c + 2 * kBatch < c1) fetch(c + 2 * kBatch, fa[0], fb[0]);
                multiply(fa[1], fb[1]);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < kOut / 64; e++) sums[wave * kOut + e * 64 + lane] = acc[e];
    __syncthreads();
#pragma unroll
    for (int q = tid; q < kOut; q += kWaves * 64) {
        float v = sums[q];
#pragma unroll
        for (int w = 1; w < kWaves; w++) v += sums[w * kOut + q];
        const int r = kTile == 32 ? c_row(q >> 6, q & 63) : 4 * ((q & 63) >> 4) + (q >> 6);
        store_c<kAdd>(C, add, M, N, m0 + r, n0 + q % kTile, v);
    }
}

}  // namespace mrk::dev

namespace mrk {

namespace {
template <bool kNT, bool kVec, int kAdd>
int launch(hipStream_t s, const float* a, const float* b, float* c, const float* add, long M, long N, long K, int variant) {
    const long t16 = ((M + 15) / 16) * ((N + 15) / 16), t32 = ((M + 31) / 32) * ((N + 31) / 32);
    const long t64 = ((M + 63) / 64) * ((N + 63) / 64), t128 = ((M + 127) / 128) * ((N + 127) / 128);
    // Measured (us, [K, N] weight): up to two 16 x 16 tiles per CU they win (256 x 256 x 1536: 8.6, tiles of 32 16.4, of 64 35;
    // 64 x 256 x 784: 5.1 / 9.8 / 20; 8192 x 10 x 784: 16.3 / 20.8 / 32), then 32 x 32 while they make one round
    // (512^3: 6.8 against 17.8 and 14.7), at two rounds 64 x 64 draws level (512 x 1000 x 1024: 25.1 / 26.4) and
    // ahead from there (768^3: 30.2 / 21.0); 128 x 128 from one tile per CU (1536^3, 144 tiles: 118 against 104;
    // 2048^3, 256 tiles: 169 against 196).  Element-wise loads need too many registers for 128 x 128.
    if (variant == 0) variant = t16 <= 512 ? 4 : t32 <= 384 ? 1 : kVec && t128 >= 256 ? 3 : 2;
    if (!kVec && variant == 3) variant = 2;
    if (t16 > 0x7fffffffL) return hipErrorInvalidValue;
    if (variant == 1) {
        const dim3 grid((unsigned)t32);
        const int tn = (int)((N + 31) / 32);
        if (K <= 256) dev::f32_direct<32, 4, kNT, kVec, kAdd><<<grid, 256, 0, s>>>(a, b, c, add, M, N, K, tn);
        else dev::f32_direct<32, 16, kNT, kVec, kAdd><<<grid, 1024, 0, s>>>(a, b, c, add, M, N, K, tn);
    } else if (variant == 4) {
        const dim3 grid((unsigned)t16);
        const int tn = (int)((N + 15) / 16);
        if (K <= 256) dev::f32_direct<16, 4, kNT, kVec, kAdd><<<grid, 256, 0, s>>>(a, b, c, add, M, N, K, tn);
        else dev::f32_direct<16, 16, kNT, kVec, kAdd><<<grid, 1024, 0, s>>>(a, b, c, add, M, N, K, tn);
    } else if (variant == 2) {
        dev::f32_tiled<1, kNT, kVec, kAdd><<<dim3((unsigned)t64), 512, 0, s>>>(a, b, c, add, M, N, K, (int)((M + 63) / 64), (int)((N + 63) / 64));
    } else if constexpr (kVec) {
        dev::f32_tiled<2, kNT, kVec, kAdd><<<dim3((unsigned)t128), 512, 0, s>>>(a, b, c, add, M, N, K, (int)((M + 127) / 128), (int)((N + 127) / 128));
    }
    return hipGetLastError();
}
}  // namespace

bool gemm_f32_supported(long M, long N, long K) {
    return M > 0 && N > 0 && K >= 64 && M * N >= ((1L << 18) + K - 1) / K && ((M + 15) / 16) * ((N + 15) / 16) <= 0x7fffffffL &&
           (K <= 8192 || ((M + 63) / 64) * ((N + 63) / 64) >= 256);
}

int launch_gemm_f32(void* stream, const void* a, const void* b, void* c, const void* add, bool add_is_row, long M, long N, long K,
                    bool b_transposed, int variant) {
    if (M <= 0 || N <= 0 || K <= 0 || variant < 0 || variant > 4) return hipErrorInvalidValue;
    auto misaligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) != 0; };
    const bool vec = K % 4 == 0 && (b_transposed || N % 4 == 0) && !misaligned(a) && !misaligned(b);
    const auto s = static_cast<hipStream_t>(stream);
    const float *pa = static_cast<const float*>(a), *pb = static_cast<const float*>(b), *pr = static_cast<const float*>(add);
    float* pc = static_cast<float*>(c);
    auto with_add = [&](auto nt, auto v) {
        if (!pr) return launch<decltype(nt)::value, decltype(v)::value, 0>(s, pa, pb, pc, pr, M, N, K, variant);
        if (add_is_row) return launch<decltype(nt)::value, decltype(v)::value, 1>(s, pa, pb, pc, pr, M, N, K, variant);
        return launch<decltype(nt)::value, decltype(v)::value, 2>(s, pa, pb, pc, pr, M, N, K, variant);
    };
    const std::true_type yes;
    const std::false_type no;
    if (b_transposed) return vec ? with_add(yes, yes) : with_add(yes, no);
    return vec ? with_add(no, yes) : with_add(no, no);
}

}  // namespace mrk
