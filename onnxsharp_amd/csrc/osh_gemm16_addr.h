// osh_gemm16_addr.h -- where gemm16_kernel's operand loads go, the same on the
// device and on the host (which checks that no load leaves its operand).
//
// A buffer load reads zeros, without an access, for each word that fails the
// range check against its descriptor's size.  gfx950 checks the vector plus the
// scalar offset (180 pairs of them inside one buffer); the offsets here are also
// right for a check of the vector offset alone.  A k offset sits in the scalar
// offset, which costs nothing, where every word of the load exists, and in the
// vector offset in the chunk that K ends in.
#pragma once

#if defined(__HIP__)
#define OSH_G16_FN __host__ __device__ __forceinline__
#else
#define OSH_G16_FN inline
#endif

namespace osh {

struct G16Off {
    int vec, scalar;
};

template <bool TAIL>
OSH_G16_FN G16Off g16_off(int lane, int k_bytes) {
    return TAIL ? G16Off{lane + k_bytes, 0} : G16Off{lane, k_bytes};
}

// Bytes of the operands, which their descriptors hold.
OSH_G16_FN int g16_bytes_a(int M, int K, int lda) { return (int)(((long long)(M - 1) * lda + K) * 4); }
OSH_G16_FN int g16_bytes_b(int K, int N, int ldb) { return (int)(((long long)(K - 1) * ldb + N) * 4); }

// A: 16 bytes at k = 4 kq of a chunk of row `row` (at most M - 1).  In the tail
// chunk (K % KC) the k past K are the next row's, and past row M - 1 nothing.
OSH_G16_FN int g16_lane_a(int row, int kq, int lda) { return (row * lda + 4 * kq) * 4; }
template <bool TAIL>
OSH_G16_FN G16Off g16_off_a(int lane, int k0) {
    return g16_off<TAIL>(lane, k0 * 4);
}

// B: row g of a k4 step, BV <= N columns from g16_col(col) on: a vector that
// would cross N starts at N - BV instead, so that every word of it exists.  In
// the tail chunk the rows from K on do not exist.
template <int BV>
OSH_G16_FN int g16_col(int col, int N) {
    return col < N - BV ? col : N - BV;
}
OSH_G16_FN int g16_lane_b(int g, int col, int ldb) { return (g * ldb + col) * 4; }
template <bool TAIL>
OSH_G16_FN G16Off g16_off_b(int lane, int k0, int ldb) {
    return g16_off<TAIL>(lane, k0 * ldb * 4);
}

}  // namespace osh
