// Attention for a handful of queries against a long key sequence (a decode step over a key/value cache,
// tensor/src/transformer.rs:78-137 with Sq of 1 to 32): O = softmax(Q K^T * scale) V is a stream over K and V,
// 4 * Sk * D bytes per (batch, head) against a few flops per byte, and with few (batch, head) pairs the kernel that
// gives every pair one workgroup leaves most of the chip without work.  Here the key sequence is split as well:
// grid = (splits, pairs), a workgroup owns a contiguous range of keys, its waves take the range's 32-key
// chunks in turn.  A wave copies its chunk of K and of V (32 rows each) with direct global -> LDS loads into a
// region of its own (1 KB per instruction, non-temporal: every byte is read once), so the loop has no barrier,
// and what streams is bounded by the bytes in flight per CU, i.e. by what the LDS holds: the next chunk's keys are
// requested as soon as this one's are in registers, its values likewise, so that half of a wave's region is always
// under way (32 pairs of 4096 keys, D = 128: 16.9 us with a launch for the merge, 18.1 where both were requested after the
// products; 5 x 8 pairs of 3703, D = 256: 29.1 and 32.1).  Under an additive mask, and where the caches grow, a lane has other
// loads or stores in the queue that the waits count: there a chunk is requested and awaited as a whole.  A Bool mask's bytes are copied
// to LDS in a fixed number of instructions a chunk, [slot][32 keys], for that reason (loaded per lane, with a chunk awaited as a whole / copied:
// 32 pairs of 4096 keys 17.4 / 15.4 us, 64 x 22360 118 / 111, 128 x 2000, D = 256 48.4 / 44.6; 22 shapes 1.07 of the speed).
// S^T = K Q^T on v_mfma_f32_16x16x32_bf16 (operand A: 16 keys x 32 d read back from LDS, rows swizzled by the key
// so that the 16 rows of a read fall into different banks; operand B: the queries, 16 columns, loaded once;
// queries beyond Sq repeat the last one and are not written; from 17 on a second block of 16 takes the same K and V
// fragments): a lane then holds, for query l % 16, the keys
// 4 * (l / 16) + 0..3 of each of the chunk's two 16-key blocks.  Those eight values, exponentiated against the
// running maximum and rounded to bf16, are directly the lane's operand of O^T += V^T P^T if the instruction's
// eight k-slots of lane group g are taken to be exactly those keys; V's side follows through the transposing
// LDS read (ds_read_b64_tr_b16: lane j of a 16-lane group receives column j of the four rows the group's lanes
// point at), pointed at rows 4 g + 0..3 of either block.  Running maximum and sum per query as in any online
// softmax; a query's maximum sits in four lanes (l % 16 equal), two exchanges per chunk.
// At the end the waves' (maximum, sum, O) meet in LDS and are merged in a fixed order; with one split the
// workgroup writes O, otherwise f32 partial results W[split][pair][16][D + 2] (the unnormalised O, then
// maximum and sum), which the pair's last workgroup to arrive or, without counters for that, flash_decode_merge folds the same way.  Results do not depend on scheduling.
// A pair is a (batch, head), or a (batch, run of consecutive heads) when those heads share their K and V (zero
// head strides: multi-query / grouped-query attention): the run's heads then occupy the query slots together
// and K and V are read once for all of them.  attn_mask (Bool bytes or additive bf16, any broadcast layout) and
// softcap of the reference (transformer.rs:112-132) are template options: a lane has the mask of its eight keys
// with the chunk's copies and applies it, then the cap, to its scores before the maximum.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.h"

namespace mrk::dev {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

#define MRK_FD_LDS(T, p) ((__attribute__((address_space(3))) T*)(p))

constexpr int kChunkKeys = 32;  // keys a wave handles per step
constexpr int kMaxQueries = 32;  // query slots of a pair: one or two blocks of 16

struct DecodeLayout {
    long long q_batch, q_head, k_batch, k_head, v_batch, v_head, o_batch, o_head;  // element strides
    unsigned q_row, k_row, v_row, o_row;                                           // byte strides of a row
    int heads;  // pairs per batch: the head count divided by `group`
    int group;  // consecutive heads folded into one pair's query slots (they share K and V: zero head strides), 1 = none
};

// attn_mask of the reference (transformer.rs:112-125) as a [batch, head, query, key] view with contiguous keys:
// element strides per batch, head and query row (0 broadcasts).  Kind 1: Bool bytes, nonzero = attend; 2: additive bf16.
struct DecodeMask {
    const void* mask;
    long long batch, head, row;
    float cap;  // softcap in score units (transformer.rs:128-132), used by the kCap instantiations
};

// A cache grown by one key in passing (kAppend): K and V hold the Sk - 1 keys before it, the last key of every pair lies in k_new /
// v_new (element strides per batch and head), and all Sk are written to k_out / v_out [pair, Sk, D] from where the copies left them in
// LDS, so that the grown cache is neither copied beforehand nor read back.  Bound by memory: the caches are read once and
// written once, 2 x 268 MB for 8 sequences of 2048 keys of 4096 columns, where copies before the attention read them twice.  That
// decoder step: 218 us with the copies, 187 in this form.
struct DecodeAppend {
    const unsigned short *k_new, *v_new;
    long long kn_batch, kn_head, vn_batch, vn_head;
    unsigned short *k_out, *v_out;
};

// The fold of a query's key ranges in their order, four columns at d: part(s) points at range s's unnormalised O [kD], maximum and sum.
template <int kD, class Part>
__device__ __forceinline__ void fold_ranges(Part part, int splits, unsigned short* __restrict__ O, int bh, int q, int d, int Sq, const DecodeLayout& lay) {
    // (both loops unrolled by four: the loads of four ranges are in flight together, the sums keep their order)
    float m_tot = -INFINITY;
#pragma unroll 4
    for (int s = 0; s < splits; s++) m_tot = fmaxf(m_tot, part(s)[kD]);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
    float l_tot = 0.0f;
#pragma unroll 4
    for (int s = 0; s < splits; s++) {
        const float* p = part(s);
        const float wgt = __builtin_amdgcn_exp2f(p[kD] - m_tot);
        const float2 a = *reinterpret_cast<const float2*>(p + d), c = *reinterpret_cast<const float2*>(p + d + 2);
        o += f32x4{a.x, a.y, c.x, c.y} * wgt;
        l_tot += p[kD + 1] * wgt;
    }
    const float inv = 1.0f / l_tot;
    const f32x4 v = {o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv};
    const int b = bh / lay.heads, h = (bh % lay.heads) * lay.group, og = q / Sq, orw = q - og * Sq;
    char* orow = reinterpret_cast<char*>(O + b * lay.o_batch + (h + og) * lay.o_head) + (size_t)orw * lay.o_row;
    *reinterpret_cast<bf16x4*>(orow + d * 2) = __builtin_convertvector(v, bf16x4);
}

template <int kD>
constexpr int decode_waves() {
    return kD == 256 ? 4 : 8;  // a wave's region is 4 * 32 * kD bytes: 128 KB of LDS for 128 and 256, 64 KB for 64
}

// kQB: 16-slot query blocks a workgroup carries (1 or 2: up to 32 query slots per pair); the K and V fragments a wave
// reads from LDS serve every block.
// kCounted: the pair's last workgroup to arrive folds its ranges.
template <int kD, int kMask, bool kCap, int kQB, bool kAppend = false, bool kCounted = false>
__global__ __launch_bounds__(decode_waves<kD>() * 64) void flash_decode_split(
    const unsigned short* __restrict__ Q, const unsigned short* __restrict__ K, const unsigned short* __restrict__ V,
    unsigned short* __restrict__ O, float* __restrict__ W, int Sq, int Sk, int keys_per_split, float scale_log2e, DecodeLayout lay,
    DecodeMask dm, DecodeAppend ap, unsigned* __restrict__ arrivals) {
    constexpr int kWaves = decode_waves<kD>();
    constexpr int kRowBytes = kD * 2;
    constexpr int kPieces = kD / 8;                      // 16-byte pieces of a row
    constexpr int kRowsPerCopy = 1024 / kRowBytes;       // 8, 4, 2
    constexpr int kCopies = kChunkKeys / kRowsPerCopy;   // per operand and chunk
    constexpr int kOperandBytes = kChunkKeys * kRowBytes;
    constexpr int kWaveBytes = 2 * kOperandBytes;
    constexpr int kSteps = kD / 32;                      // matrix steps of a score block
    constexpr int kColBlocks = kD / 16;                  // 16-column blocks of O
    constexpr int kSlots = 16 * kQB;                     // query slots of a pair
    constexpr int kPartBytes = kQB * (kColBlocks * 1024 + 128);  // a wave's O blocks, then maximum and sum, per query block
    constexpr int kLds = kWaves * kWaveBytes > kWaves * kPartBytes ? kWaves * kWaveBytes : kWaves * kPartBytes;
    // A Bool mask's bytes of a chunk, [query slot][32 keys], are copied like the keys, so that the next chunk can be under way here too
    constexpr bool kPipe = kMask != 2 && !kAppend;
    constexpr int kMaskCopies = kMask == 1 ? 2 * kQB : 0;  // of 64 words
    constexpr int kMaskBytes = kMaskCopies * 256;
    static_assert(kLds + kWaves * kMaskBytes <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) char smem[kLds + kWaves * kMaskBytes];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int jl = lane & 15, blk = lane >> 4;
    const int bh = blockIdx.y, b = bh / lay.heads, h = (bh % lay.heads) * lay.group;  // h: the pair's first head
    const int k_begin = blockIdx.x * keys_per_split;
    const int k_end = k_begin + keys_per_split < Sk ? k_begin + keys_per_split : Sk;
    const unsigned lds_k = (unsigned)(uintptr_t)MRK_FD_LDS(char, smem) + wave * kWaveBytes;
    const unsigned lds_v = lds_k + kOperandBytes;
    const char* k_head = reinterpret_cast<const char*>(K + b * lay.k_batch + h * lay.k_head);
    const char* v_head = reinterpret_cast<const char*>(V + b * lay.v_batch + h * lay.v_head);

    // copy side: copy i covers rows i * kRowsPerCopy ..; lane -> row rsub of them, position pos of the row in LDS.
    // K: position p holds piece p ^ key(row), key = row & 15 (rows of 256 bytes and more) or (row >> 1) & 7
    // (128-byte rows, two to a bank period).  V: 32-byte granule G at granule G ^ key(row), key = row & 7
    // or (row >> 1) & 3.
    const int pos = lane % kPieces, rsub = lane / kPieces;
    unsigned k_piece[kCopies], v_piece[kCopies];
#pragma unroll
    for (int i = 0; i < kCopies; i++) {
        const int r = i * kRowsPerCopy + rsub;
        const int kk = kD >= 128 ? (r & 15) : ((r >> 1) & 7);
        const int vk = kD >= 128 ? (r & 7) : ((r >> 1) & 3);
        k_piece[i] = (unsigned)(pos ^ kk) * 16u;
        v_piece[i] = (unsigned)((((pos >> 1) ^ vk) << 1) | (pos & 1)) * 16u;
    }
    // read side, K: row jl of a 16-key block, piece 4 s + blk of it
    const unsigned kx = (unsigned)(kD >= 128 ? jl : ((jl >> 1) & 7));
    const unsigned rd_k = lds_k + jl * kRowBytes;
    // read side, V: rows 4 blk + (jl >> 2) of either block, 8-byte unit jl & 3 of column block c's granule
    const int vr = 4 * blk + (jl >> 2);
    const unsigned vx = (unsigned)(kD >= 128 ? (vr & 7) : ((vr >> 1) & 3));
    const unsigned rd_v = lds_v + vr * kRowBytes + (jl & 3) * 8;

    f32x4 acc[kQB][kColBlocks];
    float m_run[kQB], l_run[kQB];  // l_run: this lane's share of the sum (its eight keys per chunk)
#pragma unroll
    for (int qb = 0; qb < kQB; qb++) {
#pragma unroll
        for (int c = 0; c < kColBlocks; c++) acc[qb][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        m_run[qb] = -INFINITY;
        l_run[qb] = 0.0f;
    }

    const char *kn = nullptr, *vn = nullptr;
    char *k_out = nullptr, *v_out = nullptr;
    if constexpr (kAppend) {
        kn = reinterpret_cast<const char*>(ap.k_new + b * ap.kn_batch + h * ap.kn_head);
        vn = reinterpret_cast<const char*>(ap.v_new + b * ap.vn_batch + h * ap.vn_head);
        k_out = reinterpret_cast<char*>(ap.k_out + (size_t)bh * Sk * kD);
        v_out = reinterpret_cast<char*>(ap.v_out + (size_t)bh * Sk * kD);
    }

    const int chunks = (k_end - k_begin + kChunkKeys - 1) / kChunkKeys;
    // (rows past the end repeat the last one, masked below)
    auto copy = [&](int ci, unsigned lds, const char* head, unsigned row, const unsigned* piece) {
        const int k0 = k_begin + ci * kChunkKeys, last = k_end - 1 - k0;
        const char* base = head + (size_t)k0 * row;
#pragma unroll
        for (int i = 0; i < kCopies; i++) {
            int r = i * kRowsPerCopy + rsub;
            r = r < last ? r : last;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                         :
                         : "s"(lds + i * 1024), "v"((unsigned)r * row + piece[i]), "s"(base)
                         : "m0", "memory");
        }
    };
    const unsigned lds_m = (unsigned)(uintptr_t)MRK_FD_LDS(char, smem) + kLds + wave * kMaskBytes;
    const char* mask_of[kMaskCopies ? kMaskCopies : 1];  // the mask row of the slot that a lane copies words of: slot 8 i + lane / 8, word lane % 8
    auto copy_mask = [&](int ci) {
        const int k0 = k_begin + ci * kChunkKeys, words = (k_end - k0) >> 2;  // (words past the end repeat the last one: those keys do not exist)
        const int word = (lane & 7) < words ? lane & 7 : words - 1;
#pragma unroll
        for (int i = 0; i < kMaskCopies; i++) {
            const char* at = mask_of[i] + k0 + 4 * word;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(lds_m + i * 256), "v"(at) : "m0", "memory");
        }
    };
    if (kPipe && wave < chunks) copy(wave, lds_k, k_head, lay.k_row, k_piece);
    if constexpr (kMask == 1) {
#pragma unroll
        for (int i = 0; i < kMaskCopies; i++) {
            const int nq = Sq * lay.group, want = 8 * i + (lane >> 3), slot = want < nq ? want : nq - 1, qg = slot / Sq, qi = slot - qg * Sq;
            mask_of[i] = static_cast<const char*>(dm.mask) + (b * dm.batch + (h + qg) * dm.head + qi * dm.row);
        }
    }
    if (kPipe && wave < chunks) {
        if constexpr (kMask == 1) copy_mask(wave);
        copy(wave, lds_v, v_head, lay.v_row, v_piece);
    }
    // the queries: operand B, query slot 16 qb + jl (the last one again beyond the pair's slots), eight d at 32 s + 8 blk
    // (query slots: head g of a folded run, row r of its Sq rows, slot g * Sq + r)
    u32x4 qf[kQB][kSteps];
    const int nq = Sq * lay.group;
    // the mask row of a lane's query: a lane needs the mask of its eight keys per chunk, two groups of four
    // consecutive ones (the key count is a multiple of 4 under a mask, so a group is inside the sequence or outside)
    const char* mrow[kQB];
#pragma unroll
    for (int qb = 0; qb < kQB; qb++) {
        const int want = 16 * qb + jl;
        const int slot = want < nq ? want : nq - 1;
        const int qg = slot / Sq, qi = slot - qg * Sq;
        mrow[qb] = nullptr;
        if constexpr (kMask == 2) mrow[qb] = static_cast<const char*>(dm.mask) + (b * dm.batch + (h + qg) * dm.head + qi * dm.row) * 2;
        const char* qrow = reinterpret_cast<const char*>(Q + b * lay.q_batch + (h + qg) * lay.q_head) + (size_t)qi * lay.q_row;
#pragma unroll
        for (int s = 0; s < kSteps; s++) qf[qb][s] = *reinterpret_cast<const u32x4*>(qrow + 64 * s + 16 * blk);
    }
    if constexpr (kPipe) {  // here, so that the loop's waits are those for the copies alone
#pragma unroll
        for (int qb = 0; qb < kQB; qb++)
#pragma unroll
            for (int st = 0; st < kSteps; st++) asm volatile("" : "+v"(qf[qb][st]));
    }
    for (int ci = wave; ci < chunks; ci += kWaves) {
        const int k0 = k_begin + ci * kChunkKeys;
        const bool full = k0 + kChunkKeys <= k_end;
        const int last = k_end - 1 - k0;  // the chunk's last valid row
        const char* kb = k_head + (size_t)k0 * lay.k_row;
        const char* vb = v_head + (size_t)k0 * lay.v_row;
        if (!kPipe) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the previous chunk's fragment reads are done
        const bool newest = kAppend && k0 + kChunkKeys >= Sk;  // the chunk with the key that is not in the cache yet, its row Sk - 1 - k0
        if (newest) {
#pragma unroll
            for (int i = 0; i < kCopies; i++) {
                int r = i * kRowsPerCopy + rsub;
                r = r < last ? r : last;
                const char* ka = r == last ? kn + k_piece[i] : kb + ((unsigned)r * lay.k_row + k_piece[i]);
                const char* va = r == last ? vn + v_piece[i] : vb + ((unsigned)r * lay.v_row + v_piece[i]);
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_k + i * 1024), "v"(ka) : "m0", "memory");
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(lds_v + i * 1024), "v"(va) : "m0", "memory");
            }
        } else if (!kPipe) {
            copy(ci, lds_k, k_head, lay.k_row, k_piece);
            copy(ci, lds_v, v_head, lay.v_row, v_piece);
        }
        // the mask of this lane's keys, requested together with the copies
        unsigned mb0[kQB], mb1[kQB];  // Bool: four bytes per group
        u32x2 ma0[kQB], ma1[kQB];     // additive: four bf16 per group
#pragma unroll
        for (int qb = 0; qb < kQB; qb++) {
            mb0[qb] = mb1[qb] = 0u;
            ma0[qb] = ma1[qb] = u32x2{0u, 0u};
            if constexpr (kMask == 2) {
                const int g0 = k0 + 4 * blk, g1 = g0 + 16;
                if (g0 < k_end) ma0[qb] = *reinterpret_cast<const u32x2*>(mrow[qb] + 2 * (size_t)g0);
                if (g1 < k_end) ma1[qb] = *reinterpret_cast<const u32x2*>(mrow[qb] + 2 * (size_t)g1);
            }
        }
        const bool more = ci + kWaves < chunks;
        if constexpr (kPipe)
            asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kCopies) : "memory");  // the keys (and their mask); the values may still be on their way
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if constexpr (kMask == 1) {
#pragma unroll
            for (int qb = 0; qb < kQB; qb++) {
                mb0[qb] = *MRK_FD_LDS(unsigned, lds_m + (16 * qb + jl) * 32 + 4 * blk);
                mb1[qb] = *MRK_FD_LDS(unsigned, lds_m + (16 * qb + jl) * 32 + 4 * blk + 16);
            }
        }
        if constexpr (kAppend) {
            // what this lane copied, to its place in the grown cache
#pragma unroll
            for (int i = 0; i < kCopies; i++) {
                const int r = i * kRowsPerCopy + rsub;
                const u32x4 kv = *MRK_FD_LDS(u32x4, lds_k + i * 1024 + lane * 16), vv = *MRK_FD_LDS(u32x4, lds_v + i * 1024 + lane * 16);
                if (full || r <= last) {
                    __builtin_nontemporal_store(kv, reinterpret_cast<u32x4*>(k_out + (size_t)(k0 + r) * kRowBytes + k_piece[i]));
                    __builtin_nontemporal_store(vv, reinterpret_cast<u32x4*>(v_out + (size_t)(k0 + r) * kRowBytes + v_piece[i]));
                }
            }
        }
        // scores of the two 16-key blocks, per query block
        f32x4 s0[kQB], s1[kQB];
#pragma unroll
        for (int qb = 0; qb < kQB; qb++) s0[qb] = s1[qb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < kSteps; s++) {
            const unsigned po = (((unsigned)(4 * s + blk)) ^ kx) * 16u;
            const u32x4 f0 = *MRK_FD_LDS(u32x4, rd_k + po);
            const u32x4 f1 = *MRK_FD_LDS(u32x4, rd_k + 16 * kRowBytes + po);
#pragma unroll
            for (int qb = 0; qb < kQB; qb++) {
                s0[qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f0), __builtin_bit_cast(bf16x8, qf[qb][s]), s0[qb], 0, 0, 0);
                s1[qb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f1), __builtin_bit_cast(bf16x8, qf[qb][s]), s1[qb], 0, 0, 0);
            }
        }
        if (kPipe && more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this chunk's keys are in registers
            if constexpr (kMask == 1) copy_mask(ci + kWaves);
            copy(ci + kWaves, lds_k, k_head, lay.k_row, k_piece);
        }
        bf16x8 pb[kQB];
        float alpha[kQB];
#pragma unroll
        for (int qb = 0; qb < kQB; qb++) {
            float x[8];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                x[r] = s0[qb][r] * scale_log2e;
                x[4 + r] = s1[qb][r] * scale_log2e;
            }
            if constexpr (kMask == 1) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (((mb0[qb] >> (8 * r)) & 0xffu) == 0u) x[r] = -INFINITY;
                    if (((mb1[qb] >> (8 * r)) & 0xffu) == 0u) x[4 + r] = -INFINITY;
                }
            }
            if constexpr (kMask == 2) {
                // scale, then the mask (transformer.rs:96-125), both in exp2 units here
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const unsigned w0 = ma0[qb][r >> 1], w1 = ma1[qb][r >> 1];
                    x[r] += __builtin_bit_cast(float, (r & 1) ? (w0 & 0xffff0000u) : (w0 << 16)) * 1.4426950408889634f;
                    x[4 + r] += __builtin_bit_cast(float, (r & 1) ? (w1 & 0xffff0000u) : (w1 << 16)) * 1.4426950408889634f;
                }
            }
            if constexpr (kCap) {
                // cap * tanh(x / cap) after the mask, with tanh(y) = 1 - 2 / (exp(2 y) + 1); x in exp2 units, so
                // exp(2 x / cap) = exp2(2 t / cap); a masked score (-inf) becomes -cap and still takes part, as in
                // the reference's graph
                const float cap_out = dm.cap * 1.4426950408889634f, cap_in = 2.0f / dm.cap;
#pragma unroll
                for (int r = 0; r < 8; r++) {
                    const float z = __builtin_amdgcn_exp2f(x[r] * cap_in);
                    x[r] = cap_out * (1.0f - 2.0f * __builtin_amdgcn_rcpf(z + 1.0f));
                }
            }
            if (!full) {  // keys that do not exist
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (4 * blk + r > last) x[r] = -INFINITY;
                    if (16 + 4 * blk + r > last) x[4 + r] = -INFINITY;
                }
            }
            float mx = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float m_new = fmaxf(m_run[qb], mx);  // without a mask finite: the chunk's first key is valid
            // under a mask every key so far may be masked out (maximum -inf): such keys weigh nothing, and nothing has
            // been summed yet; the differences below must not become -inf - -inf
            const float m_ref = kMask != 0 && !kCap && m_new == -INFINITY ? 0.0f : m_new;
            alpha[qb] = __builtin_amdgcn_exp2f(m_run[qb] - m_ref);
            m_run[qb] = m_new;
            f32x8 p;
            float psum = 0.0f;
#pragma unroll
            for (int r = 0; r < 8; r++) {
                p[r] = __builtin_amdgcn_exp2f(x[r] - m_ref);
                psum += p[r];
            }
            l_run[qb] = l_run[qb] * alpha[qb] + psum;
            pb[qb] = __builtin_convertvector(p, bf16x8);
        }
        if constexpr (kPipe) {  // the values
            if (more) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kCopies + kMaskCopies) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
#pragma unroll
        for (int c = 0; c < kColBlocks; c++) {
            const unsigned off = rd_v + (((unsigned)c ^ vx) << 5);
            bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(MRK_FD_LDS(bf16x4, off));
            bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(MRK_FD_LDS(bf16x4, off + 16 * kRowBytes));
            if (!full) {
                // the rows past the end hold copies of the last row; their weights are zero, but a zero times an
                // infinity or a NaN of that row must not reach the sum
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (4 * blk + r > last) lo[r] = (__bf16)0.0f;
                    if (16 + 4 * blk + r > last) hi[r] = (__bf16)0.0f;
                }
            }
            const bf16x8 vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int qb = 0; qb < kQB; qb++) acc[qb][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pb[qb], acc[qb][c] * alpha[qb], 0, 0, 0);
        }
        if (kPipe && more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // its values too
            copy(ci + kWaves, lds_v, v_head, lay.v_row, v_piece);
        }
    }
    // a query's sum over the four lanes that share it
#pragma unroll
    for (int qb = 0; qb < kQB; qb++) {
        l_run[qb] += __shfl_xor(l_run[qb], 16);
        l_run[qb] += __shfl_xor(l_run[qb], 32);
    }

    // the waves' results meet in LDS, over the copy regions: per wave and query block, the O blocks, then maxima and sums
    __syncthreads();
    char* part = smem;  // [kWaves][kQB][kColBlocks * 1024 + 128]
    constexpr int kBlockPart = kColBlocks * 1024 + 128;
#pragma unroll
    for (int qb = 0; qb < kQB; qb++) {
        f32x4* po = reinterpret_cast<f32x4*>(part + wave * kPartBytes + qb * kBlockPart);
#pragma unroll
        for (int c = 0; c < kColBlocks; c++) po[c * 64 + lane] = acc[qb][c];
        if (blk == 0) {
            float* ml = reinterpret_cast<float*>(part + wave * kPartBytes + qb * kBlockPart + kColBlocks * 1024);
            ml[jl] = m_run[qb];
            ml[16 + jl] = l_run[qb];
        }
    }
    __syncthreads();
    // (to be read by a workgroup that another XCD may run: written through, past this one's L2)
    auto put = [&](float* to, float x, float y) {
        const float2 v = make_float2(x, y);
        if constexpr (kCounted) __hip_atomic_store(reinterpret_cast<unsigned long long*>(to), __builtin_bit_cast(unsigned long long, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *reinterpret_cast<float2*>(to) = v;
    };
    // element e: query block, column block c, lane l of it: slot 16 qb + l % 16, columns 16 c + 4 (l / 16) + 0..3
    for (int e = threadIdx.x; e < kQB * kColBlocks * 64; e += kWaves * 64) {
        const int qb = e / (kColBlocks * 64), c = (e >> 6) % kColBlocks, l = e & 63, ql = l & 15, q = 16 * qb + ql;
        if (q >= nq) continue;
        const char* mine = part + qb * kBlockPart;
        float m_tot = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; w++) m_tot = fmaxf(m_tot, reinterpret_cast<const float*>(mine + w * kPartBytes + kColBlocks * 1024)[ql]);
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
        float l_tot = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const float* ml = reinterpret_cast<const float*>(mine + w * kPartBytes + kColBlocks * 1024);
            // a wave without a chunk, or whose keys are all masked out: maximum -inf, weight 0; a workgroup of such waves
            // only leaves (0, -inf, 0), which weighs nothing among other ranges and ends as 0 / 0 = NaN without them
            // (the softmax over -inf only of the reference)
            const float wgt = m_tot == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml[ql] - m_tot);
            o += reinterpret_cast<const f32x4*>(mine + w * kPartBytes)[c * 64 + l] * wgt;
            l_tot += ml[16 + ql] * wgt;
        }
        const int d = 16 * c + 4 * (l >> 4);
        if (W) {
            float* dst = W + (((size_t)blockIdx.x * gridDim.y + bh) * kSlots + q) * (kD + 2);
            put(dst + d, o[0], o[1]);
            put(dst + d + 2, o[2], o[3]);
            if (d == 0) put(dst + kD, m_tot, l_tot);
        } else {
            const float inv = 1.0f / l_tot;
            const f32x4 v = {o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv};
            const int og = q / Sq, orw = q - og * Sq;
            char* orow = reinterpret_cast<char*>(O + b * lay.o_batch + (h + og) * lay.o_head) + (size_t)orw * lay.o_row;
            *reinterpret_cast<bf16x4*>(orow + d * 2) = __builtin_convertvector(v, bf16x4);
        }
    }
    if constexpr (!kCounted) return;
    // The pair's workgroup that arrives last folds its ranges: all partial results of the others have left their compute units (each wave waits
    // for its own before the barrier, one work-item counts the workgroup behind it).  The counter wraps to zero with the last arrival, ready
    // for the next launch.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    unsigned* told = reinterpret_cast<unsigned*>(smem);
    if (threadIdx.x == 0) *told = atomicInc(arrivals + bh, gridDim.x - 1);
    __syncthreads();
    const bool last_in = *told == gridDim.x - 1;
    __syncthreads();
    if (!last_in) return;
    // (all of them into LDS first: one trip to memory instead of one per four ranges)
    const int row = nq * (kD + 2), splits = (int)gridDim.x;
    float* all = reinterpret_cast<float*>(smem);
    constexpr int kInFlight = 8;
    const int pieces = splits * (row / 2);
    for (int i = threadIdx.x; i < pieces; i += kInFlight * kWaves * 64) {
        unsigned long long v[kInFlight];
#pragma unroll
        for (int u = 0; u < kInFlight; u++) {
            const int at = i + u * kWaves * 64;
            if (at >= pieces) break;
            const int s = at / (row / 2), x = 2 * (at - s * (row / 2));
            const float* src = W + ((size_t)s * gridDim.y + bh) * kSlots * (kD + 2) + x;
            v[u] = __hip_atomic_load(reinterpret_cast<const unsigned long long*>(src), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int u = 0; u < kInFlight; u++)
            if (i + u * kWaves * 64 < pieces) *reinterpret_cast<unsigned long long*>(all + 2 * (i + u * kWaves * 64)) = v[u];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nq * (kD / 4); e += kWaves * 64) {
        const int q = e / (kD / 4), d = 4 * (e % (kD / 4));
        fold_ranges<kD>([&](int s) { return all + s * row + q * (kD + 2); }, splits, O, bh, q, d, Sq, lay);
    }
}

// O[bh][q][d] from the splits' partial results: the same merge as inside a workgroup, splits in order.
// One work-item per four columns; grid = ceil(pairs * slots * D / 4 / 256) with slots = Sq * group query slots per pair.
template <int kD>
__global__ __launch_bounds__(256) void flash_decode_merge(const float* __restrict__ W, unsigned short* __restrict__ O, int BH, int Sq, int splits,
                                                          int slot_cap, DecodeLayout lay) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    constexpr int kQuads = kD / 4;
    const int nq = Sq * lay.group;
    if (e >= (long)BH * nq * kQuads) return;
    const int d = (int)(e % kQuads) * 4;
    const int q = (int)((e / kQuads) % nq);
    const int bh = (int)(e / ((long)kQuads * nq));
    const size_t slice = (size_t)BH * slot_cap * (kD + 2);  // slot_cap: 16 or 32 slots per pair, as the split kernel laid them out
    const float* src = W + ((size_t)bh * slot_cap + q) * (kD + 2);
    fold_ranges<kD>([&](int s) { return src + s * slice; }, splits, O, bh, q, d, Sq, lay);
}

__global__ __launch_bounds__(256) void clear_words(unsigned* words, long n) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) words[i] = 0u;
}

}  // namespace mrk::dev

namespace mrk {
using namespace mrk::dev;

int launch_clear_words(void* stream, void* words, long n) {
    if (n <= 0) return 0;
    if (n > 0x7fffffffL || !words) return (int)hipErrorInvalidValue;
    (void)hipGetLastError();
    clear_words<<<(unsigned)((n + 255) / 256), 256, 0, static_cast<hipStream_t>(stream)>>>(static_cast<unsigned*>(words), n);
    return (int)hipGetLastError();
}

// Shapes the split kernel takes and the number of key ranges it uses: up to 32 query slots of a pair (two blocks
// of 16: 17 and more cost a second set of matrix instructions per chunk, still far from what the stream of K and V
// leaves room for), no causal rule, at least 256 keys.  Measured against one workgroup per 128 queries of a (batch, head) pair it streams K and V
// faster at every count of pairs (7.0 against 6.1 TB/s with 1024 and more), so the count does not limit it.
// Ranges are multiples of 32 keys and at least 512 keys long (two chunks per wave and more); about 192
// workgroups measured best where the pairs alone are fewer (4096 keys, 32 pairs: 41 us in one range, 20 in
// four to eight, 27 in sixteen: the second kernel and the ranges' fixed cost grow with the count).
bool flash_decode_plan(long BH, long Sq, long Sk, long D, int causal, long* splits, long* keys_per_split) {
    if (causal || Sq < 1 || Sq > kMaxQueries || Sk < 256 || Sk > (1L << 24) || BH < 1 || BH > 65535) return false;
    if (D != 256 && D != 128 && D != 64) return false;
    // (two chunks per wave and range at least: 512 keys with eight waves, 256 with the four of head dim 256, whose
    // workgroups, one per CU, measured best at one per CU: 21 against 24 us at [1, 16, 1, 4096], 30 against 33 with 32 pairs)
    const long min_keys = D == 256 ? 256 : 512, target = D == 256 ? 256 : 192;
    const long max_splits = Sk / min_keys > 0 ? Sk / min_keys : 1;
    // Rows of 256: no more workgroups than compute units, each of which holds one (rounded to the nearest count of ranges, us before / now: 96 pairs of
    // 1500 40.7 / 28.4, 72 x 2500 47.2 / 34.3, 160 x 700 33.4 / 23.5, 20 x 4000 30.4 / 23.0).
    long want = D == 256 ? target / BH : (target + BH / 2) / BH;
    // A few pairs more than compute units, each of which holds one workgroup of these: three shorter ranges a pair instead of a second round for
    // those few, from where the rounds are longer than three sets of partial results, which grow with the slots (us in one / three: one slot of 288 x 4000
    // 114 / 98, 257 x 1600 46.1 / 44.3; 16 of 320 x 1500 47.9 / 52.8, x 2500 76.2 / 78.2, x 5000 147 / 141; 8 of 288 x 1500 46.4 / 47.8, x 2500 74.2 / 70.4;
    // D = 256 one of 257 x 1500 87.6 / 79.8, 8 of 320 x 1500 92.9 / 91.6, 16 of 320 x 1500 93.7 / 97.6, x 2500 150.5 / 149; 384 x 2500 78 / 82).  One slot
    // of fewer than 1536 keys of 128 has room for two ranges (in one / two: 257 x 1500 44.5 / 43.1, 320 x 1530 49.1 / 48.1).
    if (D != 64 && Sq <= 16 && BH > 256 && BH <= 320 && Sk >= (D == 128 ? 1400 + 100 * Sq : Sq <= 8 ? 1500 : 2500)) want = 3;
    want = want < max_splits ? want : max_splits;
    want = want < 1 ? 1 : want;
    const long per = ((Sk + want - 1) / want + kChunkKeys - 1) / kChunkKeys * kChunkKeys;
    *keys_per_split = per;
    *splits = (Sk + per - 1) / per;
    return true;
}

// Query slots the partial results of a pair are laid out for: 16, or 32 from 17 slots on.
long flash_decode_slot_capacity(long slots) { return slots <= 16 ? 16 : 32; }

// The workspace a caller provides for (batch * heads) pairs: enough for the plan over those pairs and for the plans
// over fewer pairs that folding heads which share their keys gives (the launchers see the strides, the caller of this
// function need not).
size_t flash_fwd_workspace_bytes(long BH, long Sq, long Sk, long D, int causal) {
    size_t most = 0;
    for (long g = 1; g * Sq <= kMaxQueries && g <= BH; g++) {
        if (BH % g) continue;
        long splits = 0, per = 0;
        if (!flash_decode_plan(BH / g, Sq * g, Sk, D, causal, &splits, &per) || splits <= 1) continue;
        const size_t need = (size_t)splits * (BH / g) * flash_decode_slot_capacity(Sq * g) * (D + 2) * sizeof(float);
        most = need > most ? need : most;
    }
    return most;
}

// The last workgroup of a pair folds its ranges where its three trips to memory in a row (results out, the count, results in) take less than a second
// launch, which folds a query's ranges one behind the other in as many threads as there are results.  By what a pair's ranges leave (us with the
// launch / without): 32 pairs of 4096 keys, 3 KB 16.6 / 14.8, 16 slots of 64 x 4096, 24 KB 25.9 / 25.2, 8 of 16 x 4096, 32 KB 12.5 / 12.7, 16 of 16 x
// 12000, 98 KB 21.7 / 23.9, 24 of 8 x 4096, 98 KB 14.1 / 16.7; many ranges of few slots are a long chain for the launch: 8 of 4 x 12000, 23 ranges,
// 93 KB 15.3 / 14.8, D = 64 13.3 / 10.9.  Rows of 256, which four waves fold: 2 of 32 x 4096, 16 KB 28.3 / 27.8, 3 of 32 x 4096, 24 KB level, 2 of
// 8 x 12000, 64 KB 25.7 / 26.3, 4 of 8 x 4096, 64 KB 15.5 / 17.8; one slot of 4 x 12000, 42 KB 21.9 / 19.2.
bool flash_decode_folds(long splits, long slots, long D) {
    const long bytes = splits * slots * (D + 2) * (long)sizeof(float);
    if (splits <= 1 || bytes > (D == 64 ? 64 : 128) * 1024) return false;  // (the local memory a workgroup has anyway)
    if (D == 256) return slots == 1 || (slots <= 4 && bytes <= 17 * 1024);
    return bytes <= 25 * 1024 || (splits >= 20 && slots <= 8);
}

// (rows of 256 in 17 and more slots are never folded by counting)
template <int kD, int kMask, bool kCap, int kQB>
static auto split_kernel(bool counted) {
    auto kernel = flash_decode_split<kD, kMask, kCap, kQB>;
    if constexpr (kD == 256 && kQB == 2) return kernel;
    else return counted ? flash_decode_split<kD, kMask, kCap, kQB, false, true> : kernel;
}

// strides: (batch, head, row) element strides of q, k, v and o (validated by the caller: multiples of 8, rows
// addressable in 32 bits, pointers 16-byte aligned); W: splits * pairs * flash_decode_slot_capacity(group * Sq) * (D + 2)
// floats, needed with several splits (pairs = B * H / group).
// arrivals (may be null): one counter per pair, zero before the first launch that uses them and after every one, for launches that follow each other
// (one plan's): the ranges are folded by the split kernel itself, without a second launch.
// mask_kind 0: none; 1: Bool bytes, 2: additive bf16, with (batch, head, query row) element strides that are multiples
// of 4, a mask pointer aligned to four elements and Sk a multiple of 4 (validated by the caller as well).  softcap 0: none.
int launch_flash_decode(void* stream, const void* q, const void* k, const void* v, void* o, long B, long H, long Sq, long Sk, long D,
                        float scale, const long* strides, long splits, long keys_per_split, void* W, const void* mask, int mask_kind,
                        const long* mask_strides, float softcap, long group, unsigned* arrivals) {
    // group > 1: runs of `group` consecutive heads share K and V (zero head strides) and become query slots of one pair
    if (B <= 0 || H <= 0 || group < 1 || H % group || !strides || !q || !k || !v || !o) return (int)hipErrorInvalidValue;
    const long pairs = B * (H / group), slots = group * Sq;
    if (Sq < 1 || slots > kMaxQueries || Sk < 1 || splits < 1 || pairs > 65535) return (int)hipErrorInvalidValue;
    if (group > 1 && (strides[4] != 0 || strides[7] != 0)) return (int)hipErrorInvalidValue;
    if (keys_per_split < kChunkKeys || keys_per_split % kChunkKeys || splits * keys_per_split < Sk || (splits - 1) * keys_per_split >= Sk)
        return (int)hipErrorInvalidValue;
    if (splits > 1 && !W) return (int)hipErrorInvalidValue;
    DecodeLayout lay;
    lay.q_batch = strides[0], lay.q_head = strides[1], lay.q_row = (unsigned)(strides[2] * 2);
    lay.k_batch = strides[3], lay.k_head = strides[4], lay.k_row = (unsigned)(strides[5] * 2);
    lay.v_batch = strides[6], lay.v_head = strides[7], lay.v_row = (unsigned)(strides[8] * 2);
    lay.o_batch = strides[9], lay.o_head = strides[10], lay.o_row = (unsigned)(strides[11] * 2);
    lay.heads = (int)(H / group);
    lay.group = (int)group;
    if (mask_kind < 0 || mask_kind > 2 || (mask_kind != 0 && (!mask || !mask_strides || Sk % 4)) || !(softcap >= 0.0f)) return (int)hipErrorInvalidValue;
    DecodeMask dm{};
    dm.cap = softcap;
    const bool cap = softcap > 0.0f;
    if (mask_kind != 0) {
        dm.mask = mask;
        dm.batch = mask_strides[0], dm.head = mask_strides[1], dm.row = mask_strides[2];
    }
    const float scale_log2e = scale * 1.4426950408889634f;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid((unsigned)splits, (unsigned)pairs);
    float* w = splits > 1 ? static_cast<float*>(W) : nullptr;
    auto qp = static_cast<const unsigned short*>(q);
    auto kp = static_cast<const unsigned short*>(k);
    auto vp = static_cast<const unsigned short*>(v);
    auto op = static_cast<unsigned short*>(o);
    (void)hipGetLastError();
    const long quads = pairs * slots * (D / 4);
    const unsigned merge_blocks = (unsigned)((quads + 255) / 256);
    const int slot_cap = (int)flash_decode_slot_capacity(slots);
    unsigned* counted = w && flash_decode_folds(splits, slots, D) ? arrivals : nullptr;
#define MRK_DECODE_QB(DIM, MASK, CAP, QB) \
    split_kernel<DIM, MASK, CAP, QB>(counted != nullptr)<<<grid, decode_waves<DIM>() * 64, 0, s>>>(qp, kp, vp, op, w, (int)Sq, (int)Sk, (int)keys_per_split, scale_log2e, lay, dm, DecodeAppend{}, counted)
#define MRK_DECODE(DIM, MASK)                              \
    do {                                                   \
        if (cap) {                                         \
            if (slot_cap == 16) MRK_DECODE_QB(DIM, MASK, true, 1);  \
            else MRK_DECODE_QB(DIM, MASK, true, 2);        \
        } else {                                           \
            if (slot_cap == 16) MRK_DECODE_QB(DIM, MASK, false, 1); \
            else MRK_DECODE_QB(DIM, MASK, false, 2);       \
        }                                                  \
    } while (0)
#define MRK_DECODE_DIM(DIM)                                                                                         \
    do {                                                                                                            \
        if (mask_kind == 0) MRK_DECODE(DIM, 0);                                                                     \
        else if (mask_kind == 1) MRK_DECODE(DIM, 1);                                                                \
        else MRK_DECODE(DIM, 2);                                                                                    \
        if (w && !counted) flash_decode_merge<DIM><<<merge_blocks, 256, 0, s>>>(w, op, (int)pairs, (int)Sq, (int)splits, slot_cap, lay); \
    } while (0)
    if (D == 128) MRK_DECODE_DIM(128);
    else if (D == 64) MRK_DECODE_DIM(64);
    else if (D == 256) MRK_DECODE_DIM(256);
    else return (int)hipErrorInvalidValue;
#undef MRK_DECODE_DIM
#undef MRK_DECODE
#undef MRK_DECODE_QB
    return (int)hipGetLastError();
}

bool flash_decode_append_supported(long B, long H, long Sk, long D) {
    long splits = 0, per = 0;
    return B > 0 && H > 0 && B * H <= 65535 && flash_fwd_rows_addressable(Sk, D * 2, D) && flash_decode_plan(B * H, 1, Sk, D, 0, &splits, &per);
}

// strides, in elements and multiples of 8: q batch, head; new key batch, head; new value batch, head; o batch, head.
int launch_flash_decode_append(void* stream, const void* q, const void* past_k, const void* past_v, const void* new_k, const void* new_v, void* o,
                               void* k_out, void* v_out, long B, long H, long Sk, long D, float scale, const long* strides, void* W, size_t W_bytes) {
    if (!flash_decode_append_supported(B, H, Sk, D) || !strides || !(scale > 0.0f)) return (int)hipErrorInvalidValue;
    const void* ptrs[8] = {q, past_k, past_v, new_k, new_v, o, k_out, v_out};
    for (const void* p : ptrs)
        if (!p || reinterpret_cast<uintptr_t>(p) % 16) return (int)hipErrorInvalidValue;
    for (int i = 0; i < 8; i++)
        if (strides[i] < 0 || strides[i] % 8) return (int)hipErrorInvalidValue;
    long splits = 0, per = 0;
    flash_decode_plan(B * H, 1, Sk, D, 0, &splits, &per);
    const size_t slice = (size_t)B * H * flash_decode_slot_capacity(1) * (D + 2) * sizeof(float);
    if (splits > 1) {  // as many key ranges as the workspace holds
        const long fit = W ? (long)(W_bytes / slice) : 0;
        if (fit < splits) {
            const long want = fit < 2 ? 1 : fit;
            per = ((Sk + want - 1) / want + kChunkKeys - 1) / kChunkKeys * kChunkKeys;
            splits = (Sk + per - 1) / per;
        }
    }
    DecodeLayout lay{};
    lay.q_batch = strides[0], lay.q_head = strides[1], lay.q_row = 0;
    lay.k_batch = lay.v_batch = H * (Sk - 1) * D, lay.k_head = lay.v_head = (Sk - 1) * D, lay.k_row = lay.v_row = (unsigned)(D * 2);
    lay.o_batch = strides[6], lay.o_head = strides[7], lay.o_row = 0;
    lay.heads = (int)H;
    lay.group = 1;
    const auto as = [](const void* p) { return static_cast<const unsigned short*>(p); };
    const DecodeAppend ap{as(new_k), as(new_v), strides[2], strides[3], strides[4], strides[5], static_cast<unsigned short*>(k_out),
                          static_cast<unsigned short*>(v_out)};
    float* w = splits > 1 ? static_cast<float*>(W) : nullptr;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid((unsigned)splits, (unsigned)(B * H));
    const unsigned merge_blocks = (unsigned)((B * H * (D / 4) + 255) / 256);
    (void)hipGetLastError();
    auto go = [&](auto dim) {
        constexpr int kD = decltype(dim)::value;
        flash_decode_split<kD, 0, false, 1, true><<<grid, decode_waves<kD>() * 64, 0, s>>>(
            as(q), as(past_k), as(past_v), static_cast<unsigned short*>(o), w, 1, (int)Sk, (int)per, scale * 1.4426950408889634f, lay, DecodeMask{}, ap, nullptr);
        if (w) flash_decode_merge<kD><<<merge_blocks, 256, 0, s>>>(w, static_cast<unsigned short*>(o), (int)(B * H), 1, (int)splits, 16, lay);
    };
    if (D == 128) go(std::integral_constant<int, 128>{});
    else if (D == 64) go(std::integral_constant<int, 64>{});
    else go(std::integral_constant<int, 256>{});
    return (int)hipGetLastError();
}

}  // namespace mrk
