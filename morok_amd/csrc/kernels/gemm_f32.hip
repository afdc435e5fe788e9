// f32 products on the matrix pipes: C[M, N] = A[M, K] B (+ a row or a matrix), every operand in f32
// (v_mfma_f32_32x32x2_f32: 64 flops per cycle and SIMD, twice the vector ALUs' rate without packed arithmetic).  B is
// [K, N], or (kNT) [N, K] as a Linear layer stores its weight.  Any M, N, K.
//
// Which k a matrix instruction multiplies is free as long as both operands agree: lane half g = lane / 32 holds the four
// consecutive k = 8 c + 4 g .. + 3 of chunk c, so that one 16-byte read feeds four instructions, the i-th of them
// adding the products of k = 8 c + i and 8 c + 4 + i.
//
// Two kernels:
//  - f32_tiled: a workgroup of eight waves owns a 64 x 64 (128 x 128) tile of C; four waves (2 x 2) share the tile (two of four: 64 x 32), and two
//    such groups halve every K step and add their sums at the end: two waves per SIMD, so that one's reads of the
//    local memory run under the other's matrix instructions, and two shorter chains of additions.  Global ->
//    registers -> local memory, one step ahead, two stages, one barrier per step.
//  - f32_direct: few output tiles.  A workgroup owns one 16 x 16 (32 x 32) tile and its 4 (16) waves split K; a wave's operands
//    go from memory straight to registers, a batch of loads ahead of the matrix instructions, and the waves' sums
//    meet in local memory.  No barrier until then: a small product is one trip to memory.
//
// The order of the additions depends on the shape and the layout of B and on nothing else.  How far a sum is off grows with the root of the longest chain of additions.  The kernels these
// took over from added 64 partial sums of K / 64 products for ragged sizes, and one chain of K for sizes of whole 64 x 64
// tiles; neither loses precision here.  f32_direct chains 8 products, adds those sums up per wave, and the waves' in
// 64 bits.  f32_tiled leaves whole tiles (and K < 128, where ragged sizes were one chain too) with a chain of K / 2 per
// group; for ragged sizes a chain ends after 16 products (8 up to K of 192, and in 64 x 32 tiles that stand in for two rounds of 32 x 32,
// whole ones too) and goes on in 64 bits, in registers: the vector
// instructions for that do not run under f32 matrix instructions and cost 10 to 18 %.  (f32 totals cost as much:
// short of the old error they need two levels of them.)  Error against 64 bits, 2-norm, uniform operands, in 1e-7, before and
// now: 1000 x 1000 x K 0.77 / 0.59 at K = 130, 0.82 / 0.78 at 257, 1.04 / 0.78 at 1000, 1.62 / 0.78 at 4000; 130 x 200 x K
// 0.77 / 0.74, 0.82 / 0.71, 1.04 / 0.77, 1.60 / 1.00; 1024 x 1024 x K 2.05 / 1.48, 2.88 / 2.06, 5.67 / 4.02, 11.3 / 8.0.
// Bound by the f32 matrix rate (157 TFLOP/s nominal).  Measured: 1024^3 22.7 us (95 TFLOP/s; generated kernel on the vector
// ALUs 55.3); 4096^3 1.06 ms (129 TFLOP/s); 1000^3 28.7 us (reduction 3500); 64 x 256 x 784 against
// a [N, K] weight 4.3 us (36.8 and a transposing copy before).
// Rows that are no whole groups of four are read in 16-byte loads of 4-byte alignment, the last group of a row where it ends with the
// row; element by element before: 368 x 932 x 1342 59.9 -> 39.0 us, 602 x 640 x 1031 45.3 -> 31.0, 896 x 958 x 768 31.6 -> 24.4 (22.5 now), same bits.
// What is left at 1024^3, one workgroup per CU: the launch and the fill and drain of sixteen steps.  Not the barrier in each: a third stage, with
// the next step's fragments read before this step's last matrix instructions, measured 23.1 us against 22.7.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kernels.h"

namespace mrk::dev {

typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef f32x4v f32x4_any __attribute__((aligned(4)));  // (a row may start on any float)
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace {

// v's elements `by` places further down (by 0 .. 3; what comes from behind the last is not used)
__device__ __forceinline__ f32x4v move_down(const f32x4v& v, int by) {
    f32x4v r = (by & 1) ? f32x4v{v[1], v[2], v[3], v[3]} : v;
    return (by & 2) ? f32x4v{r[2], r[3], r[3], r[3]} : r;
}

// Four elements k .. k + 3 of a row of n >= 4 elements at p, zeros past the end.
enum Rows {
    kGroups4,   // n is a multiple of four: a group is inside or outside as a whole
    kAnyLength,  // one load of 4-byte alignment, moved back where it would reach past the row
    kShort,     // element by element: 0.2 us faster where K ends a few groups on (434 x 540 x 94 4.5 us against 4.8)
};
template <Rows kRows>
__device__ __forceinline__ f32x4v load4(const float* p, long k, long n) {
    f32x4v v = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (kRows == kGroups4) {
        if (k < n) v = *reinterpret_cast<const f32x4_any*>(p + k);
    } else if constexpr (kRows == kAnyLength) {
        const int left = n - k < 4 ? (int)(n - k) : 4;
        if (left > 0) {
            const f32x4v at = *reinterpret_cast<const f32x4_any*>(p + (left < 4 ? n - 4 : k));
            v = move_down(at, 4 - left);
#pragma unroll
            for (int x = 1; x < 4; x++) v[x] = x < left ? v[x] : 0.0f;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float x = p[k + i < n ? k + i : n - 1];
            v[i] = k + i >= n ? 0.0f : x;
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

// kRun: products one accumulator chains before its sum goes on into 64 bits, 8 or 16; 0: all of a wave's share of K.
template <int kT, bool kNT, bool kVec, int kAdd, int kRun>
__device__ __forceinline__ void f32_tiled_body(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                                               const float* __restrict__ add, long M, long N, long K, int tiles_m, int tiles_n) {
    constexpr int kBM = kT ? 64 * kT : 64, kBN = kT ? 64 * kT : 32;
    // Groups of four waves that share the tile and split every K step, and a wave's 32 x 32 blocks of C.  (The 128 tile with
    // 64-bit totals is shared out over all eight waves instead: 128 x 128 totals twice do not fit the registers.)
    constexpr int kGroups = kT == 2 && kRun ? 1 : 2, kMi = kT ? kT : 1, kNj = kT == 2 && kRun ? 1 : kMi;
    constexpr int kBK = kT == 2 ? 32 : 64;        // K step of the workgroup
    constexpr int kChunks = kBK / (8 * kGroups);  // 8-deep chunks per step and wave
    constexpr int kSlots = kBK / 4;           // 16-byte slots of a row of either tile in local memory, k contiguous
    constexpr int kAF = kBM * kBK, kBF = kBN * kBK;
    constexpr int kStage = kAF + kBF;
    __shared__ __attribute__((aligned(16))) float smem[2 * kStage];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = kGroups == 1 ? 0 : kT ? wave >> 2 : wave >> 1;
    const int wm = kGroups == 1 ? wave >> 2 : kT ? (wave >> 1) & 1 : wave & 1, wn = kGroups == 1 ? wave & 3 : kT ? wave & 1 : 0;
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
    auto swizzle = [](int r) { return kT != 2 ? ((r >> 2) & 3) | (((r ^ (r >> 4)) & 3) << 2) : ((r >> 1) & 7) ^ ((r >> 4) & 1); };
    // staging: waves 4-7 move A, waves 0-3 move B, four 16-byte groups per thread and step; of a [K, N] matrix a block of
    // four rows by four columns, which goes to local memory transposed, so that both fragments are read alike
    const bool moves_a = wave >= 4;
    const int tq = tid & 255;
    // Addresses are a wave's own 64-bit base, advanced with the step, and 32-bit byte offsets from it (the launcher keeps the
    // larger extents out).  Offset of group i: fixed[i] + k * pitch with k counted from the base's; k past the end of K is
    // pulled back inside, and what it brought is cleared on the way to local memory.  No branch
    // around the loads: the compiler can only count how many are in flight in straight code.
    const bool transpose = !kNT && !moves_a;
    const long first = moves_a ? m0 : n0, end = moves_a ? M : N;
    // kVec: rows are whole groups of four.  Otherwise a group that reaches past the end of its row (of K, or of the columns of a
    // [K, N] operand) is read where it ends with the row and moved down on the way to local memory.  The loads need no more than
    // 4-byte alignment either way.
    const int past = (int)(N - 1 - n0 < kBN ? N - 1 - n0 : kBN);
    const int before = !kVec && past < 3 ? 3 - past : 0;  // columns in front of the tile that are read with its last group
    const char* base = reinterpret_cast<const char*>(transpose ? B + n0 - before : (moves_a ? A : B) + first * K);
    const unsigned pitch = transpose ? (unsigned)N * 4u : 4u;
    unsigned fixed[4];
    int kr, to[4];  // a group's first k in the step (transpose: + i)
    int moved = 0;  // transpose: columns the group was read too far in front
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (!transpose) {
            const int r = tq / kSlots + i * (256 / kSlots);
            fixed[i] = (unsigned)(first + r < end ? r : end - 1 - first) * (unsigned)K * 4u;
            kr = 4 * (tq % kSlots);
            to[i] = (moves_a ? 0 : kAF) + r * kBK + (((tq % kSlots) ^ swizzle(r)) << 2);
        } else {
            const int r = 4 * (tq % (kBN / 4));
            fixed[i] = 4u * (unsigned)((r + 3 <= past ? r : past - 3) + before);
            moved = r + 3 <= past ? 0 : r - (past - 3);
            kr = 4 * (tq / (kBN / 4));
            to[i] = kAF + (r + i) * kBK + (((kr >> 2) ^ swizzle(r + i)) << 2);
        }
    }
    // Tiles of 64 x 32 are staged by four waves that all move both operands: per work-item four groups of A, and of B two groups or (transposed)
    // two k-rows by four columns.
    unsigned a_fixed[4], b_fixed[2];
    int a_to[4], b_to[4], b_kr = 0;
    const char *a_base = nullptr, *b_base = nullptr;
    constexpr bool kFlip = !kNT;
    if constexpr (kT == 0) {
        kr = 4 * (tq % kSlots);
        a_base = reinterpret_cast<const char*>(A + m0 * K);
        b_base = reinterpret_cast<const char*>(kFlip ? B + n0 - before : B + n0 * K);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = tq / kSlots + i * 16;
            a_fixed[i] = (unsigned)(m0 + r < M ? r : M - 1 - m0) * (unsigned)K * 4u;
            a_to[i] = r * kBK + (((tq % kSlots) ^ swizzle(r)) << 2);
        }
        if constexpr (kFlip) {
            const int r = 4 * (tq % 8);
            b_kr = 2 * (tq / 8);
            b_fixed[0] = b_fixed[1] = 4u * (unsigned)((r + 3 <= past ? r : past - 3) + before);
            moved = r + 3 <= past ? 0 : r - (past - 3);
#pragma unroll
            for (int x = 0; x < 4; x++) b_to[x] = kAF + (r + x) * kBK + (((b_kr >> 2) ^ swizzle(r + x)) << 2) + (b_kr & 3);
        } else {
            b_kr = kr;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int r = tq / kSlots + i * 16;
                b_fixed[i] = (unsigned)(n0 + r < N ? r : N - 1 - n0) * (unsigned)K * 4u;
                b_to[i] = kAF + r * kBK + (((tq % kSlots) ^ swizzle(r)) << 2);
            }
        }
    }
    constexpr int kLoads = kT ? 4 : 6;
    int k_next = 0;  // first k of the step to be fetched
    // Steps that end before K does (`inside`) need neither a clamped k nor zeros: their offsets are worked out here, once.
    unsigned inside_at[kLoads];
    if constexpr (kT == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++) inside_at[i] = a_fixed[i] + (unsigned)kr * 4u;
#pragma unroll
        for (int i = 0; i < 2; i++) inside_at[4 + i] = b_fixed[i] + (kFlip ? (unsigned)(b_kr + i) * (unsigned)N * 4u : (unsigned)b_kr * 4u);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) inside_at[i] = fixed[i] + (unsigned)(transpose ? kr + i : kr) * pitch;
    }
    auto fetch = [&](auto inside, f32x4v(&v)[kLoads]) {
        if constexpr (decltype(inside)::value) {
            const char* a_at = (kT ? base : a_base) + (long)k_next * (kT ? pitch : 4u);
            const char* b_at = kT ? a_at : b_base + (long)k_next * (kFlip ? (long)N * 4 : 4);
#pragma unroll
            for (int i = 0; i < kLoads; i++) v[i] = *reinterpret_cast<const f32x4_any*>((i < 4 ? a_at : b_at) + inside_at[i]);
            k_next += kBK;
            __builtin_amdgcn_sched_barrier(0);
            return;
        }
        if constexpr (kT == 0) {
            const int kb = k_next <= (int)K - kBK ? k_next : (int)K > kBK ? (int)K - kBK : 0;
            const int k = kr + (k_next - kb), bk = b_kr + (k_next - kb), last = (int)K - 1 - kb;
            const char* aa = a_base + (long)kb * 4;
            const char* bb = b_base + (long)kb * (kFlip ? (long)N * 4 : 4);
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const f32x4_any*>(aa + (a_fixed[i] + (unsigned)(k < last - 3 ? k : last - 3) * 4u));
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int ki = kFlip ? (bk + i < last ? bk + i : last) : (bk < last - 3 ? bk : last - 3);
                v[4 + i] = *reinterpret_cast<const f32x4_any*>(bb + (b_fixed[i] + (unsigned)ki * (kFlip ? (unsigned)N * 4u : 4u)));
            }
            k_next += kBK;
            __builtin_amdgcn_sched_barrier(0);
            return;
        }
        // (the base stays inside K: the steps fetched past the end read the last one again)
        const int kb = k_next <= (int)K - kBK ? k_next : (int)K > kBK ? (int)K - kBK : 0;
        const char* at = base + (long)kb * pitch;
        const int k = kr + (k_next - kb), last = (int)K - 1 - kb;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int ki = transpose ? (k + i < last ? k + i : last) : (k < last - 3 ? k : last - 3);
            v[i] = *reinterpret_cast<const f32x4_any*>(at + (fixed[i] + (unsigned)ki * pitch));
        }
        k_next += kBK;
        __builtin_amdgcn_sched_barrier(0);  // the loads set out before the step's matrix instructions, not after them
    };
    const bool columns_end = !kVec && transpose && past < kBN && (N & 3), rows_end = !kVec && !transpose && (K & 3);
    auto stash = [&](auto inside, float* st, int k0, const f32x4v(&v)[kLoads]) {
        constexpr bool kInside = decltype(inside)::value;
        const int left = (int)K - k0 - kr;
        if constexpr (kT == 0) {
            f32x4v z[6];
#pragma unroll
            for (int i = 0; i < 6; i++) z[i] = v[i];
            if constexpr (!kVec) {
                if (!kInside && (K & 3) && k0 + kBK > (int)K) {
                    const int by = left < 4 ? 4 - left : 0;
#pragma unroll
                    for (int i = 0; i < (kFlip ? 4 : 6); i++) z[i] = move_down(z[i], by);
                }
                if (kFlip && past < kBN && (N & 3)) {
                    z[4] = move_down(z[4], moved);
                    z[5] = move_down(z[5], moved);
                }
            }
#pragma unroll
            for (int i = 0; i < (kFlip ? 4 : 6); i++)
#pragma unroll
                for (int x = 0; x < 4; x++) z[i][x] = kInside || (kVec ? 0 : x) < left ? z[i][x] : 0.0f;
#pragma unroll
            for (int i = 0; i < 4; i++) *reinterpret_cast<f32x4v*>(st + a_to[i]) = z[i];
            if constexpr (kFlip) {
                const int b_left = (int)K - k0 - b_kr;
#pragma unroll
                for (int x = 0; x < 4; x++)
                    *reinterpret_cast<f32x2*>(st + b_to[x]) = f32x2{kInside || 0 < b_left ? z[4][x] : 0.0f, kInside || 1 < b_left ? z[5][x] : 0.0f};
            } else {
#pragma unroll
                for (int i = 0; i < 2; i++) *reinterpret_cast<f32x4v*>(st + b_to[i]) = z[4 + i];
            }
            return;
        }
        f32x4v z[4];
#pragma unroll
        for (int i = 0; i < 4; i++) z[i] = v[i];
        if (!kVec && (columns_end || (!kInside && rows_end && k0 + kBK > (int)K))) {
            const int by = transpose ? moved : left < 4 ? 4 - left : 0;
#pragma unroll
            for (int i = 0; i < 4; i++) z[i] = move_down(z[i], by);
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int x = 0; x < 4; x++) z[i][x] = kInside || (transpose ? i : kVec ? 0 : x) < left ? z[i][x] : 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++)
            *reinterpret_cast<f32x4v*>(st + to[i]) = transpose ? f32x4v{z[0][i], z[1][i], z[2][i], z[3][i]} : z[i];
    };

    f32x16 acc[kMi][kNj];
    using Total = std::conditional_t<kRun == 0, float, double>;
    Total total[kRun ? kMi : 1][kRun ? kNj : 1][16];
    auto each = [&](auto&& f) {
#pragma unroll
        for (int i = 0; i < kMi; i++)
#pragma unroll
            for (int j = 0; j < kNj; j++)
#pragma unroll
                for (int e = 0; e < 16; e++) f(i, j, e);
    };
    each([&](int i, int j, int e) {
        acc[i][j][e] = 0.0f;
        if constexpr (kRun != 0) total[i][j][e] = 0.0;
    });

    const int steps = (int)((K + kBK - 1) / kBK);
    // Step s multiplies stage s & 1 while step s + 1's operands are on their way to registers since step s - 1 (an L2 miss
    // takes longer than a step) and step s + 2's set out.  `inside`: step s + 2 ends before K does.  Those steps' offsets and zeros
    // are not worked out again and again: f32 matrix instructions leave the vector ALUs no time of their own (us before / now: 1024^3
    // 24.0 / 22.7, 512 x 1024 x 1024 16.1 / 14.4, 1408 x 320 x 1408 20.7 / 18.4, 896 x 958 x 768 24.1 / 22.5, 4096^3 1084 / 1062).
    // A second form of the step spills where 64-bit totals fill the registers (700 x 500 x 777 17.7 / 23.1): not there.
    constexpr bool kTwoForms = kRun == 0 || (kT == 1 && !kVec);
    f32x4v in0[kLoads], in1[kLoads];
    auto step = [&](auto inside, int s, f32x4v(&arriving)[kLoads], f32x4v(&leaving)[kLoads]) {
        constexpr bool kAll = decltype(inside)::value || !kTwoForms;  // nothing is left out of the last steps
        const float* st = smem + (s & 1) * kStage;
        if (kAll || s + 2 < steps) fetch(inside, leaving);
        const int slot = group * (kSlots / kGroups) + lg;
        f32x4v fa[2][kMi], fb[2][kNj];
        auto fragments = [&](int c) {
#pragma unroll
            for (int i = 0; i < kMi; i++) {
                const int ra = (wm * kMi + i) * 32 + lr;
                fa[c & 1][i] = *reinterpret_cast<const f32x4v*>(st + ra * kBK + (((slot + 2 * c) ^ swizzle(ra)) << 2));
            }
#pragma unroll
            for (int j = 0; j < kNj; j++) {
                const int rb = (wn * kNj + j) * 32 + lr;
                fb[c & 1][j] = *reinterpret_cast<const f32x4v*>(st + kAF + rb * kBK + (((slot + 2 * c) ^ swizzle(rb)) << 2));
            }
        };
        fragments(0);
#pragma unroll
        for (int c = 0; c < kChunks; c++) {
            if (c + 1 < kChunks) fragments(c + 1);
            const bool opens = kRun == 8 || (kRun == 16 && c % 2 == 0), closes = kRun == 8 || (kRun == 16 && c % 2 == 1);
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int i = 0; i < kMi; i++)
#pragma unroll
                    for (int j = 0; j < kNj; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[c & 1][i][x], fb[c & 1][j][x], opens && x == 0 ? f32x16{} : acc[i][j], 0, 0, 0);
            if constexpr (kRun == 0) {
                // (a chunk's fragments are read under the matrix instructions of the chunk before)
                if (c + 1 < kChunks) {
                    if (c == 0) __builtin_amdgcn_sched_group_barrier(0x100, 2 * kMi, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 2 * kMi, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x8, 4 * kMi * kMi, 0);
            } else if (closes) {
                each([&](int i, int j, int e) { total[i][j][e] += (double)acc[i][j][e]; });
                __builtin_amdgcn_sched_barrier(0);  // (one set of accumulators at a time: there are no registers for two)
            }
        }
        // (the other stage was last read in step s - 1, which every wave has left at the barrier before this step)
        if (kAll || s + 1 < steps) stash(inside, smem + ((s + 1) & 1) * kStage, (s + 1) * kBK, arriving);
        __syncthreads();
    };
    constexpr std::true_type kInside{};
    constexpr std::false_type kEdge{};
    fetch(kEdge, in0);
    fetch(kEdge, in1);
    stash(kEdge, smem, 0, in0);
    __syncthreads();
    int s = 0;
    if constexpr (kTwoForms) {
        const int full = (int)(K / kBK);
        for (; s + 3 < full; s += 2) {
            step(kInside, s, in1, in0);
            step(kInside, s + 1, in0, in1);
        }
    }
    for (; s + 1 < steps; s += 2) {
        step(kEdge, s, in1, in0);
        step(kEdge, s + 1, in0, in1);
    }
    if (s < steps) step(kEdge, s, in1, in0);
    auto sum = [&](int i, int j, int e) -> Total {
        if constexpr (kRun == 0) return acc[i][j][e];
        else return total[i][j][e];
    };
    auto store = [&](int i, int j, int e, Total other) {
        store_c<kAdd>(C, add, M, N, m0 + (wm * kMi + i) * 32 + c_row(e, lane), n0 + (wn * kNj + j) * 32 + lr, (float)(sum(i, j, e) + other));
    };
    if constexpr (kGroups == 2) {
        // the second group hands its sums over through local memory (all reads of the stages are behind the last barrier)
        constexpr int kWave = kMi * kNj * 16 * 64;
        constexpr int kShare = kT ? 4 : 2;  // waves of a group
        static_assert(kShare * kWave * sizeof(Total) <= sizeof smem, "the second group's sums fit into the stages");
        Total* x = reinterpret_cast<Total*>(smem) + (wave & (kShare - 1)) * kWave + lane;
        if (group == 1) each([&](int i, int j, int e) { x[((i * kNj + j) * 16 + e) * 64] = sum(i, j, e); });
        __syncthreads();
        if (group == 0) each([&](int i, int j, int e) { store(i, j, e, x[((i * kNj + j) * 16 + e) * 64]); });
    } else {
        each([&](int i, int j, int e) { store(i, j, e, 0); });
    }
}

template <int kT, bool kNT, bool kVec, int kAdd, int kRun>
__global__ void __launch_bounds__(kT ? 512 : 256, kT == 1 && kVec ? 4 : 2) f32_tiled(const float* A, const float* B, float* C, const float* add, long M, long N, long K, int tiles_m,
                                                 int tiles_n) {
    f32_tiled_body<kT, kNT, kVec, kAdd, kRun>(A, B, C, add, M, N, K, tiles_m, tiles_n);
}

// kWaves waves split K into runs of whole chunks (of eight for tiles of 32, of sixteen for tiles of 16, whose lane groups
// are four)
template <int kTile, int kWaves, bool kNT, Rows kRows, int kAdd>
__global__ void __launch_bounds__(kWaves * 64) f32_direct(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C,
                                                          const float* __restrict__ add, long M, long N, long K, int tiles_n) {
    constexpr int kBatch = 4;  // chunks whose loads are in flight together
    constexpr int kDeep = 4 * (64 / kTile), kOut = kTile * kTile;
    constexpr int kRun = kTile == 32 ? 4 : 2;  // matrix instructions in a row on one accumulator: 8 products
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
    float total[kOut / 64];
#pragma unroll
    for (int e = 0; e < kOut / 64; e++) total[e] = 0.0f;
    f32x4v fa[2][kBatch], fb[2][kBatch];
    auto fetch = [&](long c, f32x4v(&a)[kBatch], f32x4v(&b)[kBatch]) {
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
            // chunks past this wave's run multiply zeros
            const long k = c + i < c1 ? (c + i) * kDeep + 4 * lg : K;
            a[i] = load4<kRows>(pa, k, K);
            if constexpr (kNT) {
                b[i] = load4<kRows>(pb, k, K);
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
        for (int i = 0; i < kBatch; i++) {
            Acc run[4 / kRun];
#pragma unroll
            for (int x = 0; x < 4; x++) {
                Acc& acc = run[x / kRun];
                if (x % kRun == 0) acc = Acc{};
                if constexpr (kTile == 32) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][x], b[i][x], acc, 0, 0, 0);
                else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][x], b[i][x], acc, 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < kOut / 64; e++) total[e] += kRun == 4 ? run[0][e] : run[0][e] + run[4 / kRun - 1][e];
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
    for (int e = 0; e < kOut / 64; e++) sums[wave * kOut + e * 64 + lane] = total[e];
    __syncthreads();
#pragma unroll
    for (int q = tid; q < kOut; q += kWaves * 64) {
        double v = sums[q];
#pragma unroll
        for (int w = 1; w < kWaves; w++) v += (double)sums[w * kOut + q];
        const int r = kTile == 32 ? c_row(q >> 6, q & 63) : 4 * ((q & 63) >> 4) + (q >> 6);
        store_c<kAdd>(C, add, M, N, m0 + r, n0 + q % kTile, (float)v);
    }
}

}  // namespace mrk::dev

namespace mrk {

namespace {
struct F32Call {
    hipStream_t s;
    const float *a, *b, *add;
    float* c;
    long M, N, K;
};

long tiles(long M, long N, long t) { return ((M + t - 1) / t) * ((N + t - 1) / t); }
// What tiles of a size compute, whether it is stored or not: a product with a side of 1 to 32 in tiles of 128 is mostly
// padding (65536 x 1 x 1024 144 us in tiles of 128, 62 in tiles of 16).
double padded(long M, long N, long t) { return (double)tiles(M, N, t) * t * t; }

// 16 and 32: f32_direct; 64: f32_tiled, which takes 128 where launch() says.
// Measured (us, [K, N] weight): up to two 16 x 16 tiles per CU they win (256 x 256 x 1536: 8.6, tiles of 32 16.4, of 64 35;
// 64 x 256 x 784: 5.1 / 9.8 / 20; 8192 x 10 x 784: 16.3 / 20.8 / 32), then 32 x 32 while they make one round
// (512^3: 6.8 against 17.8 and 14.7), at two rounds 64 x 64 draws level (512 x 1000 x 1024: 25.1 / 26.4) and
// ahead from there (768^3: 30.2 / 21.0).  A larger tile may pad as much more as it is faster: 1.4 from 32 to 64; tiles of
// 16 read the longer operand's lines in halves and pay on long K only (65536 x 5 x 1024 68 us against 77 in tiles of 32,
// 65536 x 8 x 500 47 / 41).  The tiled kernels' offsets inside a step are 32-bit: up to 128 rows of K floats, or 64 of N.
int tile_size(long M, long N, long K, bool b_transposed) {
    const bool narrow = padded(M, N, 64) > 1.4 * padded(M, N, 32), far = K > (1L << 22) || (!b_transposed && N > (1L << 22));
    if (tiles(M, N, 16) <= 512 || far || (narrow && K >= 768 && padded(M, N, 32) > 1.4 * padded(M, N, 16))) return 16;
    return tiles(M, N, 32) <= (K > 256 ? 256 : 384) || narrow ? 32 : 64;
}
// Products that tiles of 32 would take in two rounds (257 to 384 of them) run on tiles of 64 x 32 in one, above K = 256: 602 x 640 x 1031
// 31.0 us there, 22.2 here, 700 x 500 x 777 30.9 / 18.0, 1472 x 256 x 704 20.7 / 15.8, 576 x 640 x 256 7.6 / 7.9.  They keep sums of eight
// products: 0.59e-7 off (2-norm) at every K measured, f32_direct 0.69 to 0.90.
bool two_rounds_of_32(long M, long N, long K) { return K > 256 && tiles(M, N, 32) > 256 && tiles(M, N, 32) <= 384; }

// Times in us of f32_direct, and of the generated reduction that a product is without these kernels (K >= 128: one wave
// per output; below: one work-item), fitted to 890 products with a side of 1 to 24 against 300 to 10^6, and of 17 to 600,
// K from 64 to 4096.  Either is within a quarter of the measured time for most of them.
double direct_us(double M, double N, double K, bool b_transposed, int tile, double area, long count) {
    const double columns = b_transposed ? 0.0 : 0.2 + 3e-4 * K;
    if (tile == 16) return columns + (count <= 512 ? 3.4 + 1.8e-3 * K + 2.2e-8 * area * K + 1.9e-7 * (M + N) * K : 6.2e-8 * area * K + 1.4e-5 * M * N);
    return columns + (count <= 384 ? 3.0 + 7.4e-3 * K + 1.3e-6 * M * N : 2.8 + 3.7e-8 * area * K + 1.2e-6 * area);
}
double reduction_us(double M, double N, double K, bool b_transposed) {
    const double x = M * N * K, edges = (M + N) * K;
    if (K < 128) return 0.8 + 0.026 * K + (b_transposed ? 5e-7 : 2.5e-7) * x + (M < N ? 4e-7 : 3e-7) * edges;
    // (a wide [N, K] operand is read again for every row)
    if (b_transposed && M < N && N * K > (2 << 20)) return 8e-4 * K + 2.6e-7 * x + 6e-5 * M * N + 2e-7 * edges;
    if (b_transposed) return 2.3 + 2e-4 * K + 1.9e-7 * x + 4.3e-5 * M * N + 1.2e-7 * edges;
    // (a wave's lanes walk a column of a [K, N] operand, a line each)
    if (N == 1) return 2.0 + 2e-4 * K + 4.5e-5 * M + 3.6e-7 * edges;
    if (N <= 3) return 2.4 + 5e-7 * x + 2.4e-5 * M * N;
    if (N <= 12) return 2.4 + (N >= 8 && K >= 1024 ? 2e-6 : 9e-7) * x + 1.5e-5 * M * N;
    return N * K < (1 << 18) ? 1.8 + 1.5e-3 * K + 1.5e-6 * x : 1.8 + 1.5e-3 * K + 3.5e-6 * x + 2.5e-6 * edges;
}

// Tiles of 64 x 32 instead of 64 x 64: half the work each, where they come out in fewer rounds of one workgroup per CU (us, 64 x 64 / 64 x 32:
// 512 x 1024 x 1024, 128 tiles 23.7 / 16.2; 1100^3, 324 tiles 55.0 / 45.8; 1536^3 87 / 76; but 1280^3, 400 tiles 50 / 54, 768^3, 144
// tiles 18.9 / 19.0).
bool half_tiles(long M, long N) {
    const long whole = (tiles(M, N, 64) + 255) / 256, half = ((M + 63) / 64 * ((N + 31) / 32) + 255) / 256;
    return half * 0.53 < (double)whole;
}

template <int kTile, bool kNT, dev::Rows kRows, int kAdd>
void launch_direct_rows(const F32Call& p) {
    const int tn = (int)((p.N + kTile - 1) / kTile);
    const dim3 grid((unsigned)((p.M + kTile - 1) / kTile * tn));
    if (kRows == dev::kShort || p.K <= 256) dev::f32_direct<kTile, 4, kNT, kRows, kAdd><<<grid, 256, 0, p.s>>>(p.a, p.b, p.c, p.add, p.M, p.N, p.K, tn);
    else if constexpr (kRows != dev::kShort) dev::f32_direct<kTile, 16, kNT, kRows, kAdd><<<grid, 1024, 0, p.s>>>(p.a, p.b, p.c, p.add, p.M, p.N, p.K, tn);
}

template <int kTile, bool kNT, int kAdd>
void launch_direct(const F32Call& p) {
    if (p.K % 4 == 0) launch_direct_rows<kTile, kNT, dev::kGroups4, kAdd>(p);
    else if (p.K >= 128) launch_direct_rows<kTile, kNT, dev::kAnyLength, kAdd>(p);
    else launch_direct_rows<kTile, kNT, dev::kShort, kAdd>(p);
}

template <int kT, bool kNT, bool kVec, int kAdd, int kRun>
void launch_tiled(const F32Call& p) {
    constexpr int kBM = kT ? 64 * kT : 64, kBN = kT ? 64 * kT : 32;
    const long tm = (p.M + kBM - 1) / kBM, tn = (p.N + kBN - 1) / kBN;
    dev::f32_tiled<kT, kNT, kVec, kAdd, kRun><<<dim3((unsigned)(tm * tn)), kT ? 512 : 256, 0, p.s>>>(p.a, p.b, p.c, p.add, p.M, p.N, p.K, (int)tm, (int)tn);
}

template <bool kNT, int kAdd>
int launch(const F32Call& p) {
    const long M = p.M, N = p.N, K = p.K;
    if (tiles(M, N, 16) > 0x7fffffffL) return hipErrorInvalidValue;
    (void)hipGetLastError();  // (an error that an earlier call left behind is not this launch's)
    const bool vec = K % 4 == 0 && (kNT || N % 4 == 0);  // rows of whole groups of four
    const int tile = tile_size(M, N, K, kNT);
    if (tile == 16) {
        launch_direct<16, kNT, kAdd>(p);
    } else if (tile == 32) {
        launch_direct<32, kNT, kAdd>(p);
    } else {
        // 128 x 128 from one tile per CU (1536^3, 144 tiles: 118 us against 104; 2048^3, 256 tiles: 169 against 196) and where they
        // pad no more than they gain.
        // Products of whole 64 x 64 tiles, and short ones, keep one chain per wave, see the head of the file.
        const bool chain = (M % 64 == 0 && N % 64 == 0) || K < 128;
        if (vec && tiles(M, N, 128) >= 256 && padded(M, N, 128) <= 1.14 * padded(M, N, 64) && (chain || K >= 192))
            chain ? launch_tiled<2, kNT, true, kAdd, 0>(p) : launch_tiled<2, kNT, true, kAdd, 16>(p);
        else if (two_rounds_of_32(M, N, K)) vec ? launch_tiled<0, kNT, true, kAdd, 8>(p) : launch_tiled<0, kNT, false, kAdd, 8>(p);
        else if (half_tiles(M, N)) {
            if (chain) vec ? launch_tiled<0, kNT, true, kAdd, 0>(p) : launch_tiled<0, kNT, false, kAdd, 0>(p);
            else if (K < 192) vec ? launch_tiled<0, kNT, true, kAdd, 8>(p) : launch_tiled<0, kNT, false, kAdd, 8>(p);
            else vec ? launch_tiled<0, kNT, true, kAdd, 16>(p) : launch_tiled<0, kNT, false, kAdd, 16>(p);
        } else if (chain) vec ? launch_tiled<1, kNT, true, kAdd, 0>(p) : launch_tiled<1, kNT, false, kAdd, 0>(p);
        else if (K < 192) vec ? launch_tiled<1, kNT, true, kAdd, 8>(p) : launch_tiled<1, kNT, false, kAdd, 8>(p);
        else vec ? launch_tiled<1, kNT, true, kAdd, 16>(p) : launch_tiled<1, kNT, false, kAdd, 16>(p);
    }
    return hipGetLastError();
}
}  // namespace

bool gemm_f32_supported(long M, long N, long K) {
    return M > 0 && N > 0 && K >= 64 && M * N >= ((1L << 18) + K - 1) / K && tiles(M, N, 16) <= 0x7fffffffL &&
           (K <= 8192 || tiles(M, N, 64) >= 256);
}

// Whole 64 x 64 tiles are a generated kernel of register tiles otherwise, whose work-items walk all of K, and lose to these
// at every size (64 x 256 x 784: 36 us against 5).  Of the others the narrow ones are faster as reductions, the
// more so the more K there is per output: 1000000 x 1 x 64 65 us against 128 in tiles of 32, 300 x 3 x 4096 4.2 / 13.7,
// 64 x 10 x 784 3.1 / 4.9; but 65536 x 5 x 1024 91 / 68, 8192 x 10 x 784 69 / 9.  They go where the estimates are further apart
// than they are off (1 us on the smallest), inside the sizes they were fitted to.  An addend is a kernel of its own (2.6 us) there.
// The smallest stay here although a reduction is 0.3 to 0.7 us shorter (up to some 0.9 M multiply-adds, 3 M against a [N, K]
// operand: 65 x 192 x 64 3.5 us against 3.0, 100 x 29 x 192 3.5 / 2.9): with an addend, where these win, the sums would
// come in another order than without.
bool gemm_f32_preferred(long M, long N, long K, bool b_transposed, bool added) {
    if (!gemm_f32_supported(M, N, K)) return false;
    const int tile = tile_size(M, N, K, b_transposed);
    if (tile == 64 || (M % 64 == 0 && N % 64 == 0) || ((M < N ? M : N) > 24 && K > 1024)) return true;
    const double direct = direct_us((double)M, (double)N, (double)K, b_transposed, tile, padded(M, N, tile), tiles(M, N, tile));
    const double reduction = reduction_us((double)M, (double)N, (double)K, b_transposed) + (added ? 2.6 : 0.0);
    return direct < 1.05 * reduction || direct < reduction + 1.3;
}

int launch_gemm_f32(void* stream, const void* a, const void* b, void* c, const void* add, bool add_is_row, long M, long N, long K,
                    bool b_transposed) {
    if (M <= 0 || N <= 0 || K <= 0) return hipErrorInvalidValue;
    const F32Call p{static_cast<hipStream_t>(stream), static_cast<const float*>(a), static_cast<const float*>(b), static_cast<const float*>(add),
                    static_cast<float*>(c), M, N, K};
    if (b_transposed) return !add ? launch<true, 0>(p) : add_is_row ? launch<true, 1>(p) : launch<true, 2>(p);
    return !add ? launch<false, 0>(p) : add_is_row ? launch<false, 1>(p) : launch<false, 2>(p);
}

}  // namespace mrk
