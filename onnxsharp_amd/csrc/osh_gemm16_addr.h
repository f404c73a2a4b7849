// osh_gemm16_addr.h -- byte offsets of gemm16_kernel's operand loads, the same
// on the device and on the host (which checks that no load leaves its operand).
//
// A buffer load's range check compares the vector offset (and not the scalar
// one) with the descriptor's size, word by word.  So a k offset may sit in a
// scalar register, which costs no instruction per load, only where every word
// of the load exists; where some may not, it goes into the vector offset and
// the words past the operand read as zero without an access.
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

// A lane's offset and a uniform one, `ranged` when the sum may lie past the operand.
template <bool ranged>
OSH_G16_FN G16Off g16_off(int lane, int uniform) {
    return ranged ? G16Off{lane + uniform, 0} : G16Off{lane, uniform};
}

// A: 16 bytes at k = 4 kq of a chunk of row `row` (at most M - 1).  In the tail
// chunk (K % KC) the k past K are the next row's, and past row M - 1 nothing.
OSH_G16_FN int g16_lane_a(int row, int kq, int lda) { return (row * lda + 4 * kq) * 4; }
template <bool TAIL>
OSH_G16_FN G16Off g16_off_a(int lane, int k0) {
    return g16_off<TAIL>(lane, k0 * 4);
}

// B: row g of a k4 step, BV columns from `col` on; a vector that starts past N
// reads column 0 instead and is not stored.  In the tail chunk the rows from K
// on do not exist; with N % BV (RAG) a vector that crosses N reads on into the
// next rows, past row K - 1 nothing.
OSH_G16_FN int g16_lane_b(int g, int col, int N, int ldb) { return (g * ldb + (col < N ? col : 0)) * 4; }
template <bool TAIL, bool RAG>
OSH_G16_FN G16Off g16_off_b(int lane, int k0, int ldb) {
    return g16_off<TAIL || RAG>(lane, k0 * ldb * 4);
}

// Bytes of the operands, which their descriptors hold.
OSH_G16_FN int g16_bytes_a(int M, int K, int lda) { return (int)(((long long)(M - 1) * lda + K) * 4); }
OSH_G16_FN int g16_bytes_b(int K, int N, int ldb) { return (int)(((long long)(K - 1) * ldb + N) * 4); }

}  // namespace osh
