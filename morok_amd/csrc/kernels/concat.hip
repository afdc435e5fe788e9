// Concatenation of tensors in memory along one axis: a key/value cache grown by the tokens of a step.
//
// Bound by HBM: every byte is read once and written once.  The extents are launch arguments: the generated kernel it stands
// in for holds them as literals, so that a cache that grows by one token was two new kernels to compile on every step (a decode
// step of 8 sequences at a position not seen before: 200 ms, 1.0 ms so; 0.4 since the attention grows the caches itself).  A work-item copies one sixteen-byte piece (7.0 TB/s over 8 x 32 rows of
// 2047 tokens of 256 bytes, 38 us, as the generated kernel; two pieces 6.9, four 6.7); only at the seams are the piece's part
// and, in parts whose runs lie apart, its run looked up.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

namespace mrk::dev {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_any __attribute__((aligned(1)));  // (a view may start on any byte)

__device__ __forceinline__ u32x4 piece_at(const char* p) { return *reinterpret_cast<const u32x4_any*>(p); }

__global__ __launch_bounds__(256) void concat_copy(char* __restrict__ out, ConcatShape s) {
    const long long start = (long long)blockIdx.x * 256, first = start + threadIdx.x;
    for (long long row = blockIdx.y; row < s.outer0 * s.outer1; row += gridDim.y) {
        const unsigned o0 = s.outer0 == 1 ? 0 : (unsigned)row / (unsigned)s.outer1, o1 = (unsigned)row - o0 * (unsigned)s.outer1;
        char* o = out + (row * s.row_pieces + first) * 16;
        // workgroups inside the first part, one run per row: all but the few at the seams
        if (s.part[0].run == s.part[0].pieces && start + 256 <= s.part[0].pieces) {
            *reinterpret_cast<u32x4_any*>(o) = piece_at(s.part[0].src + o0 * s.part[0].stride0 + o1 * s.part[0].stride1 + first * 16);
            continue;
        }
        if (first >= s.row_pieces) continue;
        long long c = first;
        int p = 0;
        while (p + 1 < s.parts && c >= s.part[p].pieces) c -= s.part[p++].pieces;
        const ConcatPart& part = s.part[p];
        const char* at = part.src + o0 * part.stride0 + o1 * part.stride1;
        if (part.run == part.pieces) at += c * 16;
        else {
            const unsigned l = (unsigned)c / (unsigned)part.run;
            at += l * part.stride + (c - (long long)l * part.run) * 16;
        }
        *reinterpret_cast<u32x4_any*>(o) = piece_at(at);
    }
}

}  // namespace mrk::dev

namespace mrk {

int launch_concat(void* stream, void* out, const ConcatShape& s) {
    if (s.parts < 1 || s.parts > kConcatParts || s.outer0 < 0 || s.outer1 < 0 || !out) return (int)hipErrorInvalidValue;
    long long pieces = 0;
    for (int p = 0; p < s.parts; p++) {
        const ConcatPart& c = s.part[p];
        if (!c.src || c.pieces <= 0 || c.run <= 0 || c.pieces % c.run || c.pieces > 0x7fffffffLL) return (int)hipErrorInvalidValue;
        pieces += c.pieces;
    }
    if (pieces != s.row_pieces || pieces > kConcatRowPieces) return (int)hipErrorInvalidValue;
    if (s.outer0 > 0x7fffffffLL || s.outer1 > 0x7fffffffLL || s.outer0 * s.outer1 > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    const long long rows = s.outer0 * s.outer1, groups = (s.row_pieces + 255) / 256;
    if (rows == 0) return 0;
    (void)hipGetLastError();
    mrk::dev::concat_copy<<<dim3((unsigned)groups, (unsigned)(rows < 65535 ? rows : 65535)), 256, 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<char*>(out), s);
    return (int)hipGetLastError();
}

}  // namespace mrk
