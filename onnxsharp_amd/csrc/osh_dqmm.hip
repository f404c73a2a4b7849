// osh_dqmm.hip -- DynamicQuantizeMatMul and DynamicQuantizeLinear on gfx950.
//
// Reference: DynamicQuantizeMatMulLayer.Forward (src/OnnxSharp/Ops/QuantizedMatMulOps.cs:115-201),
// Quantizer.MinMax (src/OnnxSharp/Tensors/Quantization.cs:109-181), QuantizeAndWiden
// (QuantizedMatMulOps.cs:280-335) and the zero-point identity of PackedInt8Weights
// (src/OnnxSharp/Kernels/Int8Gemm.cs:66-70).
//
// Pipeline (three launches, all on the caller's stream; smaller products run 2
// and 3 as one launch, dqmm_fused*_kernel or, up to 16 rows, dqmm_skinny_kernel):
//   1. dqmm_minmax_kernel   grid-stride min/max of A (0 included, NaN skipped) into per-block
//                           partials.
//   2. dqmm_quantize_kernel every block reduces the partials to scale = (max-min)/255 (1 if
//                           not > 0), zp = clamp(rne(-min/scale)), inv = 1/scale -- single IEEE
//                           ops, no contraction -- then q = clamp(rne(x*inv) + zp, 0, 255); stores
//                           a'' = q - 128 as s8 in the MFMA operand layout and a per-row flag
//                           for x*inv = NaN (the reference's q is then NaN and its whole
//                           output row is NaN).
//   3. dqmm_gemm_kernel     v_mfma_i32_32x32x32_i8 over a'' x w'' (both s8), then the exact
//                           integer correction
//                             acc = sum a''w'' + off_j*rowsum_i + alpha*colsum_j + K*alpha*off_j
//                           with alpha = 128 - zp and w' = w'' + off_j (w'' is the raw s8
//                           weight, or w - 128 for u8 weights; off_j = (u8 ? 128 : 0) - w_zp_j),
//                           which equals sum (q - zp)(w - w_zp) exactly; then
//                           out = fmaf((float)acc, scale * w_scale[j], bias[j]).
//
// Operand layout (both operands): fragment f = (tile, kstep) holds 64 lanes x 16 bytes;
// lane l carries row/column (l & 31) of the tile and k = kstep*32 + 16*(l >> 5) + byte.
// A and B use the same k assignment, so the MFMA pairs matching k regardless of the
// hardware's internal k order.
#include <type_traits>
#include "osh_common.h"

using namespace osh;

namespace osh {

constexpr int DQ_MINMAX_BLOCKS = 256;
constexpr int DQ_THREADS = 256;
constexpr int DQ_MMU = 4;  // 16-byte loads a thread of the min/max launch has in flight

struct DqScratch {  // layout of the caller's scratch buffer
    float partial_min[DQ_MINMAX_BLOCKS];
    float partial_max[DQ_MINMAX_BLOCKS];
    int zp;
    float scale;
    float inv;
    int alpha;  // a - a_zp = a'' + alpha for the packed a'' (128 - zp for quantized u8)
    int pad[60];
    // followed by: int rownan[mpad]; int spare[mpad]; int8 a_packed[mpad * kpad]
};

__host__ __device__ static inline int pad32(int v) { return (v + 31) & ~31; }

static size_t scratch_bytes(int m, int k) {
    return sizeof(DqScratch) + (size_t)pad32(m) * 8 + (size_t)pad32(m) * pad32(k);
}

__device__ __forceinline__ float wave_min(float v) {
    for (int o = 32; o > 0; o >>= 1) v = __builtin_fminf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int o = 32; o > 0; o >>= 1) v = __builtin_fmaxf(v, __shfl_xor(v, o));
    return v;
}

// Block-level min/max of (lo, hi) into thread 0's return values (NW waves).
template <int NW = DQ_THREADS / 64>
__device__ void block_minmax(float &lo, float &hi) {
    __shared__ float smin[NW], smax[NW];
    lo = wave_min(lo);
    hi = wave_max(hi);
    int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        smin[w] = lo;
        smax[w] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < NW; i++) {
            lo = __builtin_fminf(lo, smin[i]);
            hi = __builtin_fmaxf(hi, smax[i]);
        }
    }
}

// `zero` (zero_n ints, may be none): the NaN flags the quantize launch raises,
// cleared here so that the scratch needs no initialisation.
__global__ __launch_bounds__(DQ_THREADS) void dqmm_minmax_kernel(const float *__restrict__ a, long long n,
                                                                  DqScratch *__restrict__ sc, int *__restrict__ zero,
                                                                  int zero_n) {
    float lo = 0.f, hi = 0.f;  // 0 is always inside the range (Quantization.cs:115-116)
    const long long stride = (long long)gridDim.x * blockDim.x;
    // XCD-banded block ids: the workgroups of one XCD read one contiguous band
    // of A, which the fused kernel's workgroups on the same XCD (banded the
    // same way, row tiles first) then find in that XCD's L2.  Min and max are
    // exact in any order, so the partials' assignment does not matter.
    const long long i = (long long)xcd_band(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
    for (long long z = (long long)blockIdx.x * blockDim.x + threadIdx.x; z < zero_n; z += stride) zero[z] = 0;
    // 16-byte loads when the base is aligned (all callers pass tensor bases)
    const long long n4 = (reinterpret_cast<uintptr_t>(a) & 15) == 0 ? n / 4 : 0;
    const float4 *a4 = reinterpret_cast<const float4 *>(a);
    // NaN lanes are skipped (compare-false keeps the running value)
    auto take = [&](const float4 &v) {
        lo = v.x < lo ? v.x : lo; hi = v.x > hi ? v.x : hi;
        lo = v.y < lo ? v.y : lo; hi = v.y > hi ? v.y : hi;
        lo = v.z < lo ? v.z : lo; hi = v.z > hi ? v.z : hi;
        lo = v.w < lo ? v.w : lo; hi = v.w > hi ? v.w : hi;
    };
    // DQ_MMU loads in flight a pass: the partials allow no more than 256
    // workgroups, so a large A is many passes (2048 x 2048: 5.5 -> 4.0 us)
    long long j = i;
    for (; j + (DQ_MMU - 1) * stride < n4; j += DQ_MMU * stride) {
        float4 v[DQ_MMU];
#pragma unroll
        for (int u = 0; u < DQ_MMU; u++) v[u] = a4[j + u * stride];
#pragma unroll
        for (int u = 0; u < DQ_MMU; u++) take(v[u]);
    }
    for (; j < n4; j += stride) take(a4[j]);
    for (j = n4 * 4 + i; j < n; j += stride) {
        float v = a[j];
        lo = v < lo ? v : lo;
        hi = v > hi ? v : hi;
    }
    block_minmax(lo, hi);
    if (threadIdx.x == 0) {
        sc->partial_min[blockIdx.x] = lo;
        sc->partial_max[blockIdx.x] = hi;
    }
}

// scale = (max-min)/255 (1 if not > 0), zp = clamp(rne(-min/scale)),
// inv = 1/scale: single IEEE ops, no contraction (QuantizedMatMulOps.cs:151-155;
// QuantizeAndWiden multiplies by the reciprocal, :282).
__device__ __forceinline__ void dq_param_values(float lo, float hi, float &scale, int &zp, float &inv) {
    scale = (hi - lo) / 255.0f;
    if (!(scale > 0.0f)) scale = 1.0f;
    const float zf = __builtin_rintf(-lo / scale);
    zp = (int)zf;
    zp = zp < 0 ? 0 : (zp > 255 ? 255 : zp);
    inv = 1.0f / scale;
}

// The parameters for later launches and the caller.
__device__ __forceinline__ void dq_publish_params(DqScratch *__restrict__ sc, int *__restrict__ qparams, float scale,
                                                  int zp, float inv) {
    sc->scale = scale;
    sc->zp = zp;
    sc->inv = inv;
    sc->alpha = 128 - zp;
    if (qparams) {
        qparams[0] = __float_as_int(scale);
        qparams[1] = zp;
    }
}

// Every consumer block reduces the per-block partials itself (a few hundred
// floats from L2), so no grid-wide counter is needed and the scratch needs no
// initialisation.  One block (`publish`) stores the parameters for later
// launches and the caller.
template <int NW = DQ_THREADS / 64>
__device__ void dq_finish(DqScratch *__restrict__ sc, float lo, float hi, int *__restrict__ qparams,
                          bool publish, float &inv_out, int &zp_out, float *scale_out) {
    __shared__ float s_inv, s_scale;
    __shared__ int s_zp;
    block_minmax<NW>(lo, hi);
    if (threadIdx.x == 0) {
        float scale, inv;
        int zp;
        dq_param_values(lo, hi, scale, zp, inv);
        s_inv = inv;
        s_scale = scale;
        s_zp = zp;
        if (publish) dq_publish_params(sc, qparams, scale, zp, inv);
    }
    __syncthreads();
    inv_out = s_inv;
    zp_out = s_zp;
    if (scale_out) *scale_out = s_scale;
}

__device__ void dq_params(DqScratch *__restrict__ sc, int nparts, int *__restrict__ qparams, bool publish,
                          float &inv_out, int &zp_out) {
    float lo = 0.f, hi = 0.f;
    for (int b = threadIdx.x; b < nparts; b += blockDim.x) {
        lo = __builtin_fminf(lo, sc->partial_min[b]);
        hi = __builtin_fmaxf(hi, sc->partial_max[b]);
    }
    dq_finish(sc, lo, hi, qparams, publish, inv_out, zp_out, nullptr);
}

// q = clamp(rne(x * inv) + zp, 0, 255) as QuantizeAndWiden computes it in float.
// A NaN product yields 0 here; callers flag it (the reference's q is NaN then).
__device__ __forceinline__ int quantize_one(float x, float inv, float zpf) {
    float q = __builtin_rintf(x * inv) + zpf;
    q = __builtin_fminf(255.0f, __builtin_fmaxf(0.0f, q));
    return (int)q;
}

// Four consecutive k of one row.
struct Quad {
    float v[4];
};

// MatMulInteger's activations: u8 (a - 128) or s8 (a) into the s8 a'' of the
// MFMA layout.  A wave takes one fragment (32 rows x 32 k; four a wave were
// slower at every size: 1000 x 1000 x 64, both launches, 8.4 us against 7.5, 8192 x
// 2048 x 64 18.8 against 17.6).
// VEC, every row 16-byte aligned: lane l loads 16 consecutive bytes of row l &
// 31, k half l >> 5, and stores them at l * 16.  Else lane l takes the four
// bytes at k = 4 (l % 8) of row l / 8 + 8 i, with one 4-byte load at whatever
// address; one that would pass the end of A starts earlier and is shifted.  No
// load waits for another (16 guarded bytes a lane, in four fragments: 318 x 115 x
// 519 11.6 us, so 5.7; 9 x 121 x 16 10.1, so 4.6).
// Block 0 publishes alpha = (u8 ? 128 : 0) - a_zp so that a - a_zp = a'' +
// alpha; no row is NaN.
template <bool VEC>
__global__ __launch_bounds__(DQ_THREADS) void mmi_pack_a_kernel(const uint8_t *__restrict__ a, int m, int k,
                                                                 int a_signed, int a_zp, DqScratch *__restrict__ sc,
                                                                 int *__restrict__ rownan, int8_t *__restrict__ apk) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ks = pad32(k) / 32;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        sc->alpha = (a_signed ? 0 : 128) - a_zp;
        sc->scale = 1.0f;
        sc->zp = a_zp;
    }
    const long long w = (long long)blockIdx.x * (DQ_THREADS / 64) + wave;
    const int mt = (int)(w / ks), s = (int)(w % ks);
    if ((long long)mt * 32 >= m) return;
    if (s == 0 && lane < 32) rownan[mt * 32 + lane] = 0;
    const unsigned flip = a_signed ? 0u : 0x80808080u;  // u8 - 128, byte by byte
    int8_t *dst = apk + w * 1024;
    if constexpr (VEC) {
        const int row = mt * 32 + (lane & 31), kk = s * 32 + 16 * (lane >> 5);
        const bool live = row < m && kk < k;
        i32x4 v = *reinterpret_cast<const i32x4 *>(a + (live ? (long long)row * k + kk : 0));
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = live ? v[e] ^ (int)flip : 0;  // padding rows and columns carry a'' = 0
        *reinterpret_cast<i32x4 *>(dst + lane * 16) = v;
    } else {
        const int r8 = lane >> 3, c8 = lane & 7, kk = s * 32 + 4 * c8;
        const long long total = (long long)m * k, last = total < 4 ? 0 : total - 4;
        unsigned v[4];
        int past[4];
        auto each = [&](auto load) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const long long at = (long long)(mt * 32 + 8 * i + r8) * k + kk;
                const long long from = at < last ? at : last;
                past[i] = at - from < 3 ? (int)(at - from) : 3;  // more only past the row
                v[i] = load(a + from);
            }
        };
        if (total >= 4) {
            each([](const uint8_t *src) {
                unsigned u;
                __builtin_memcpy(&u, src, 4);
                return u;
            });
        } else {  // all of an A of 1 to 3 bytes
            unsigned u = 0;
            for (int e = 0; e < total; e++) u |= (unsigned)a[e] << (8 * e);
            each([&](const uint8_t *) { return u; });
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int row = mt * 32 + 8 * i + r8, left = row < m ? k - kk : 0;
            const unsigned mask = left >= 4 ? ~0u : (left > 0 ? (1u << (8 * left)) - 1 : 0u);
            // lane slot (row & 31) + 32 * (c8 >> 2); byte 4 (c8 & 3)
            reinterpret_cast<unsigned *>(dst)[(8 * i + r8 + 32 * (c8 >> 2)) * 4 + (c8 & 3)] =
                ((v[i] >> (8 * past[i])) ^ flip) & mask;
        }
    }
}

// DynamicQuantizeLinear output: u8 q in the input's own layout.
__global__ __launch_bounds__(DQ_THREADS) void dql_quantize_kernel(const float *__restrict__ x, long long n,
                                                                   DqScratch *__restrict__ sc, int nparts,
                                                                   int *__restrict__ qparams,
                                                                   uint8_t *__restrict__ q) {
    float inv;
    int zp;
    dq_params(sc, nparts, qparams, blockIdx.x == 0, inv, zp);
    const float zpf = (float)zp;
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    long long stride = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += stride) q[i] = (uint8_t)quantize_one(x[i], inv, zpf);
}

// Packed weight buffer: int8 fragments [npad/32][kpad/32][64][16], then int colsum[npad],
// then int off[npad].
static size_t packed_w_bytes(int k, int n) { return (size_t)pad32(n) * pad32(k) + (size_t)pad32(n) * 8; }

__global__ void dqmm_pack_kernel(int k, int n, const void *__restrict__ w, int w_signed,
                                 const int *__restrict__ wzp, int n_wzp, int8_t *__restrict__ out,
                                 int *__restrict__ colsum, int *__restrict__ off) {
    // one thread per column
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    int npad = pad32(n), kpad = pad32(k);
    if (j >= npad) return;
    int zp = (j < n && n_wzp > 0) ? (n_wzp == 1 ? wzp[0] : wzp[j]) : 0;
    int o = (w_signed ? 0 : 128) - zp;
    int s = 0;
    for (int kk = 0; kk < kpad; kk++) {
        int v = 0;
        if (j < n && kk < k) {
            long long idx = (long long)kk * n + j;
            v = w_signed ? (int)reinterpret_cast<const int8_t *>(w)[idx]
                         : (int)reinterpret_cast<const uint8_t *>(w)[idx] - 128;
            s += v;
        }
        long long frag = (long long)(j >> 5) * (kpad / 32) + (kk >> 5);
        int lane = (j & 31) + 32 * ((kk >> 4) & 1);
        out[(frag * 64 + lane) * 16 + (kk & 15)] = (int8_t)v;
    }
    colsum[j] = s;
    off[j] = j < n ? o : 0;
}

// What the epilogue needs of output column j: loaded without a condition (a
// lane past the last column reads the last one's and stores nothing), so that
// nothing waits before the operand loads that follow.
struct ColOperands {
    int off, csum;
    float ws, bias;
};
__device__ __forceinline__ ColOperands load_column(int j, int n, const int *__restrict__ colsum,
                                                   const int *__restrict__ off, const float *__restrict__ wscale,
                                                   int n_wscale, const float *__restrict__ bias) {
    const int jc = j < n ? j : n - 1;
    ColOperands c;
    c.off = off[jc];
    c.csum = colsum[jc];
    c.ws = wscale ? wscale[n_wscale == 1 ? 0 : jc] : 0.0f;
    c.bias = bias ? bias[jc] : 0.0f;
    return c;
}

// The int8 GEMM over packed operands.  A workgroup owns 32 TM rows x 128
// columns; each of its four waves one 32-column tile and all TM row tiles, on
// v_mfma_i32_32x32x32_i8.
//
// Fragments are 1 KB (one 32-row or 32-column tile x 32 k, already in the
// MFMA's lane order).  A wave's W fragments are its own, so they come straight
// into registers; the A fragments, which all four waves read, go through LDS,
// four k-steps a stage: wave w loads k-step w of every row tile, one barrier a
// stage, two buffers, lane l at l * 16 (no bank conflicts).  SETS stages
// are in flight in registers.
//
// Each tile has its own buffer descriptor of exactly its k-steps (none for a
// tile past the last): loads past it return zeros and fetch nothing, which
// ends the prefetch and pads the last stage without a branch.  Row sums of a''
// come from the staged registers (v_dot4).
//
// Bound by what the L2s deliver and, at the ends, the first loads and the output
// stores: 1028 x 1280 x 5120 takes 15.7 us here (13.5 G int-ops, 858 TOP/s), in
// which the workgroups read 167 MB of fragments from L2 (10.6 TB/s) while LDS is
// active 15% of the time and the int8 units 18%; 512 x 512 x 2048 4.8.
constexpr int DQG_KS = 4;
enum { DQG_FLOAT = 1, DQG_ACC = 2 };  // which outputs a launch writes

template <int TM, int SETS, int OUT>
__global__ __launch_bounds__(256, 2) void dqmm_gemm_kernel(int m, int k, int n, const int8_t *__restrict__ apk,
                                                           const int8_t *__restrict__ wpk,
                                                           const int *__restrict__ colsum,
                                                           const int *__restrict__ off,
                                                           const int *__restrict__ rownan,
                                                           const DqScratch *__restrict__ sc,
                                                           const float *__restrict__ wscale, int n_wscale,
                                                           const float *__restrict__ bias, float *__restrict__ out,
                                                           int *__restrict__ acc_out) {
    static_assert(DQG_KS == 4 && SETS % 2 == 0, "a wave loads one k-step of a stage; buffers alternate");
    static_assert(32 * TM <= 256, "one row sum a thread");
    __shared__ __align__(16) i32x4 frag[2][TM * DQG_KS * 64];
    __shared__ __align__(16) int lds_rs[32 * TM], lds_rn[32 * TM];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = pad32(k) / 32, nmt = pad32(m) / 32, nnt = pad32(n) / 32, mpad = pad32(m);
    // XCD-banded ids, rows first: an XCD's workgroups share a band of W's
    // columns and all of A's rows
    const int nmb = (nmt + TM - 1) / TM;
    const int id = xcd_band(blockIdx.x, gridDim.x);
    const int mt0 = (id % nmb) * TM, nt = (id / nmb) * 4 + wave;

    struct Set {
        i32x4 a[TM], b[DQG_KS];
    };
    auto load_tile = [&](const int8_t *base, int tile, int ntiles, int voff) {
        const bool live = tile < ntiles;
        __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(base + (live ? (long long)tile * ks * 1024 : 0)), (short)0, live ? ks * 1024 : 0, 0x00020000);
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff, 0, 0);
        return i32x4{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
    };
    auto load = [&](Set &r, int st) {
        const int voff = lane * 16 + st * DQG_KS * 1024;
#pragma unroll
        for (int t = 0; t < TM; t++) r.a[t] = load_tile(apk, mt0 + t, nmt, voff + wave * 1024);
#pragma unroll
        for (int kk = 0; kk < DQG_KS; kk++) r.b[kk] = load_tile(wpk, nt, nnt, voff + kk * 1024);
    };
    auto stage = [&](const Set &r, int buf) {
#pragma unroll
        for (int t = 0; t < TM; t++) frag[buf][(t * DQG_KS + wave) * 64 + lane] = r.a[t];
    };
    const int nst = (ks + DQG_KS - 1) / DQG_KS;
    Set r[SETS];
#pragma unroll
    for (int u = 0; u < SETS; u++) load(r[u], u);
    // the epilogue's operands: NaN flags (and, after the loop, the row sums)
    // through LDS, columns in registers
    if (tid < 32 * TM) {
        lds_rs[tid] = 0;
        lds_rn[tid] = rownan[mt0 * 32 + tid < mpad ? mt0 * 32 + tid : 0];
    }
    const int j = nt * 32 + (lane & 31);
    const bool jlive = j < n;
    const ColOperands col = load_column(j, n, colsum, off, wscale, n_wscale, bias);
    const unsigned alpha = (unsigned)sc->alpha;
    const float ascale = sc->scale;

    i32x16 acc[TM] = {};
    int rsum[TM] = {};  // sum of a'' over this wave's k-steps of row lane & 31 (and k half lane >> 5)
    auto add_rows = [&](const Set &r) {
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int e = 0; e < 4; e++) rsum[t] = __builtin_amdgcn_sdot4(r.a[t][e], 0x01010101, rsum[t], false);
    };
    stage(r[0], 0);
    add_rows(r[0]);
    __syncthreads();
    for (int st = 0; st < nst; st += SETS) {
#pragma unroll
        for (int u = 0; u < SETS; u++) {
            // LDS buffer u & 1 holds stage st + u's A, r[u] its W; the other
            // sets the stages after it; stages past the last are zeros
            const i32x4 *fa = frag[u & 1] + lane;
#pragma unroll
            for (int kk = 0; kk < DQG_KS; kk++)
#pragma unroll
                for (int t = 0; t < TM; t++)
                    acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[(t * DQG_KS + kk) * 64], r[u].b[kk], acc[t], 0,
                                                                   0, 0);
            if (st + u + 1 >= nst) break;
            load(r[u], st + u + SETS);
            stage(r[(u + 1) % SETS], (u + 1) & 1);
            add_rows(r[(u + 1) % SETS]);
            __syncthreads();
        }
    }
#pragma unroll
    for (int t = 0; t < TM; t++) atomicAdd(lds_rs + t * 32 + (lane & 31), rsum[t]);
    __syncthreads();
    if (!jlive) return;
    // Epilogue.  two's-complement wrap-around is exact as long as the final sum
    // fits in int32.  A zero point and a row sum fit 24 bits (|sum a''| <=
    // 128 * 33025), so the row term is one full-rate mad.
    const int half = lane >> 5;
    const int offj = col.off;
    const float bj = col.bias;
    const int colterm = (int)(alpha * (unsigned)col.csum + (unsigned)k * alpha * (unsigned)offj);
    const float comb = ascale * col.ws;  // CombinedScale, QuantizedMatMulOps.cs:203-221
    auto epilogue = [&](auto full) {  // full: every row is inside the matrix
#pragma unroll
        for (int t = 0; t < TM; t++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int il = t * 32 + 8 * q + 4 * half;
                const int4 s4 = *reinterpret_cast<const int4 *>(lds_rs + il);
                const int4 n4 = *reinterpret_cast<const int4 *>(lds_rn + il);
                const long long at = (long long)(mt0 * 32 + il) * n + j;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int rs = e == 0 ? s4.x : e == 1 ? s4.y : e == 2 ? s4.z : s4.w;
                    const int rnan = e == 0 ? n4.x : e == 1 ? n4.y : e == 2 ? n4.z : n4.w;
                    if (full || mt0 * 32 + il + e < m) {
                        const int v = (int)((unsigned)acc[t][4 * q + e] + (unsigned)(__mul24(offj, rs) + colterm));
                        if constexpr (OUT & DQG_ACC) acc_out[at + (long long)e * n] = v;
                        if constexpr (OUT & DQG_FLOAT) {
                            const float o = __builtin_fmaf((float)v, comb, bj);
                            out[at + (long long)e * n] = rnan ? __builtin_nanf("") : o;
                        }
                    }
                }
            }
    };
    if ((mt0 + TM) * 32 <= m) epilogue(std::true_type{});
    else epilogue(std::false_type{});
}

// Quantize + GEMM in one launch, after dqmm_minmax_kernel.  A workgroup owns
// 32 rows of A and DQF_WAVES column tiles of 32.  Its 256 threads load the
// rows' floats (thread -> row tid/8, four consecutive k at 32*i + 4*(tid%8))
// and each wave its column tile's B fragments for a pass of DQF_KS k-steps,
// all issued at once behind the min/max partials and the epilogue's column
// operands.  The threads quantize with the parameters every workgroup reduces
// from the partials and store a'' = q - 128 in the MFMA A-operand order in
// LDS; after one barrier each wave runs its v_mfma_i32_32x32x32_i8 chain.  The
// row sums of a'' (v_dot4 over the packed bytes) and the NaN flags come from
// the same registers; nothing but the parameters goes through global scratch.
// Arithmetic (quantization, zero-point correction, epilogue) is the
// three-launch pipeline's, so both give identical bits.
//
// Time line of one launch at C5's size (512 x 512 x 2048; per-workgroup
// s_memrealtime stamps in a copy of the kernel, medians): workgroups start
// over 0.7 us; the first loads return after ~2 us (a cold first load takes
// that long even with nothing else in flight); quantization 0.9 us; the MFMA
// chain 1.0 us; the output stores 1.2 us, near the HBM write rate for 4 MB.
constexpr int DQF_WAVES = 4;
constexpr int DQF_KS = 16;  // k-steps of 32 per pass: K = 512 in one pass
constexpr int DQF_GM = 4;   // row tiles per group of the tile order
static_assert(DQ_MINMAX_BLOCKS <= 256, "one min/max partial per thread of a 256-thread workgroup");

// Four elements of one row, quantized: returns the packed a'' bytes
// (q - 128 as s8) and adds their sum and NaN flag.  `live_mask` bit e says
// whether element e is a real element (else its a'' is 0).  v_cvt_pk_u8_f32
// converts with round-to-nearest-even and saturates to [0, 255] (a NaN gives
// 0), so on the integer-valued q = rne(x * inv) + zp it is the clamp of
// QuantizeAndWiden; both facts were checked on the device for every integer
// from -1000 to 1300, the .25/.5/.75 fractions, +-inf and NaN, and the
// pipelines' bit equality is tested.
__device__ __forceinline__ unsigned quantize4(const Quad &x, float inv, float zpf, unsigned live_mask, int &sum,
                                              bool &nan) {
    unsigned packed = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float p = x.v[e] * inv;
        const float q = __builtin_rintf(p) + zpf;
        if (live_mask & (1u << e)) {
            nan |= !(p == p);
            packed = __builtin_amdgcn_cvt_pk_u8_f32(q, e, packed);
        } else {
            packed |= 128u << (8 * e);  // q = 128 <-> a'' = 0
        }
    }
    packed ^= 0x80808080u;  // q -> q - 128, byte by byte
    sum = __builtin_amdgcn_sdot4((int)packed, 0x01010101, sum, false);
    return packed;
}

// The quantize launch: a wave takes DQ_QF fragments (32 rows x 32 k) of one row
// tile.  Lane l loads four consecutive k of row l / 8 + 8 i -- a row's 8 lanes
// one whole 128-byte line -- all before the parameter reduction, and stores the
// packed four bytes into the fragment, 128 contiguous bytes per eight rows.
// A row with a NaN raises its flag, which the min/max launch cleared; the
// GEMM sums the rows itself.
constexpr int DQ_QF = 2;

__global__ __launch_bounds__(DQ_THREADS) void dqmm_quantize_kernel(const float *__restrict__ a, int m, int k,
                                                                    DqScratch *__restrict__ sc, int nparts,
                                                                    int *__restrict__ qparams,
                                                                    int *__restrict__ rownan,
                                                                    int8_t *__restrict__ apk) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ks = pad32(k) / 32;
    const int nch = (ks + DQ_QF - 1) / DQ_QF;
    const int w = blockIdx.x * (DQ_THREADS / 64) + wave;
    const int mt = w / nch, s0 = w % nch * DQ_QF;
    const bool any = mt * 32 < m;
    const int r8 = lane >> 3, c8 = lane & 7;
    // Unconditional loads: a descriptor of the row tile's rows, an offset past
    // it for rows and columns that do not exist (zeros, nothing fetched).  A
    // quad that crosses k reads into the next row, masked below; 4-byte
    // alignment is all a buffer load needs.
    const int rows = any ? (m - mt * 32 < 32 ? m - mt * 32 : 32) : 0;
    __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)(a + (any ? (long long)mt * 32 * k : 0)),
                                                                  (short)0, rows * k * 4, 0x00020000);
    Quad x[DQ_QF][4];
#pragma unroll
    for (int f = 0; f < DQ_QF; f++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int kk = (s0 + f) * 32 + 4 * c8;
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(ra, kk < k ? ((8 * i + r8) * k + kk) * 4 : -1, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; e++) x[f][i].v[e] = __uint_as_float(v[e]);
        }
    __builtin_amdgcn_sched_barrier(0);
    float inv;
    int zp;
    dq_params(sc, nparts, qparams, blockIdx.x == 0, inv, zp);
    if (!any) return;
    const float zpf = (float)zp;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int row = mt * 32 + 8 * i + r8;
        int sum = 0;
        bool nan = false;
#pragma unroll
        for (int f = 0; f < DQ_QF; f++) {
            const int s = s0 + f, kk = s * 32 + 4 * c8;
            unsigned lm = 0;  // padding rows and columns carry a'' = 0
#pragma unroll
            for (int e = 0; e < 4; e++) lm |= (row < m && kk + e < k) ? (1u << e) : 0u;
            // fragment (mt, s); lane slot (row & 31) + 32 * (c8 >> 2); byte 4 (c8 & 3)
            const unsigned q = quantize4(x[f][i], inv, zpf, lm, sum, nan);
            if (s < ks)
                reinterpret_cast<unsigned *>(
                    apk)[((long long)mt * ks + s) * 256 + (8 * i + r8 + 32 * (c8 >> 2)) * 4 + (c8 & 3)] = q;
        }
        if (nan) atomicOr(rownan + row, 1);
    }
}

// The same with every element live and the sum left to the caller.
__device__ __forceinline__ unsigned quantize4(const Quad &x, float inv, float zpf, bool &nan) {
    unsigned packed = 0;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float p = x.v[e] * inv;
        nan |= !(p == p);
        packed = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_rintf(p) + zpf, e, packed);
    }
    return packed ^ 0x80808080u;  // q -> q - 128, byte by byte
}

// FULL: m % 32 == 0, n % 128 == 0, k % 512 == 0 and A 16-byte aligned, so
// every row, column and k-step is live and no load or store needs a check.
// The host picks it whenever it applies; the kernel then has no divergent
// paths, so the compiler issues all operand loads before the first wait
// (with the checks, the registers of the two load paths are merged by copies
// that wait for every A load before any B load is issued).
//
// KS: k-steps a pass.  All of them are loaded, quantized and staged whatever K
// is, so a K of at most 4 or 8 steps takes a pass of 4 or 8, with fewer
// registers and less LDS (16 for every K, then by K): 1352 x 78 x 6499 40.9 ->
// 21.9 us, 489 x 118 x 212 11.0 -> 8.2, 417 x 96 x 2432 10.8 -> 8.5, 130 x 206 x
// 3094 11.2 -> 9.7.
//
// A and W are not declared __restrict__: the operand loads must stay ahead of
// the barriers that follow them (the compiler may otherwise sink loads of
// restrict read-only memory to their first use).
template <bool FULL, int KS>
__global__ __launch_bounds__(64 * DQF_WAVES) void dqmm_fused_kernel(
    int m, int k, int n, const float *a, DqScratch *__restrict__ sc, int nparts, int *__restrict__ qparams,
    const int8_t *wpk, const int *__restrict__ colsum, const int *__restrict__ off,
    const float *__restrict__ wscale, int n_wscale, const float *__restrict__ bias, float *__restrict__ out,
    int *__restrict__ acc_out) {
    __shared__ __attribute__((aligned(16))) int lds_a[KS * 256];  // [kstep][64 lanes][16 bytes]
    __shared__ int lds_rs[32], lds_rn[32];
    const int tid = threadIdx.x, lane = tid & 63, wt = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kpad = pad32(k), ks = kpad / 32, npad = pad32(n);
    // Tiles: XCD-banded ids, then groups of DQF_GM row tiles x all column
    // blocks, so one XCD's L2 holds a few row tiles of A and part of W.
    const int ncb = (npad / 32 + DQF_WAVES - 1) / DQF_WAVES, nmt = pad32(m) / 32;
    const int id = xcd_band(blockIdx.x, gridDim.x);
    const int grp = id / (DQF_GM * ncb), gl = id % (DQF_GM * ncb);
    const int mt0 = grp * DQF_GM;
    const int gm = nmt - mt0 < DQF_GM ? nmt - mt0 : DQF_GM;
    const int mt = mt0 + gl % gm;
    const int nt = (gl / gm) * DQF_WAVES + wt;
    const bool col_live = FULL || nt * 32 < npad;
    const int r = tid >> 3, c8 = tid & 7;
    const int row = mt * 32 + r;
    const bool live = FULL || row < m;
    const float *src = a + (long long)(live ? row : 0) * k;
    const int npass = (ks + KS - 1) / KS;
    const i32x4 *B = reinterpret_cast<const i32x4 *>(wpk) + (long long)(col_live ? nt : 0) * ks * 64 + lane;

    // nparts <= 256: one partial per thread (threads past nparts repeat
    // partial 0), consumed after the operand loads are issued
    const int pidx = tid < nparts ? tid : 0;
    const float pmin = sc->partial_min[pidx], pmax = sc->partial_max[pidx];
    // the epilogue's column operands, loaded now so their latency hides under the pass
    const int j = nt * 32 + (lane & 31);
    const bool jlive = col_live && (FULL || j < n);
    const ColOperands col = load_column(j, n, colsum, off, wscale, n_wscale, bias);

    Quad x[KS];
    i32x4 b[KS];
    // Without FULL the loads go through buffer descriptors (of the row tile's
    // rows, of the column tile's k-steps): rows, columns and k-steps that do
    // not exist return zeros and fetch nothing, so every load is unconditional
    // and in flight at once; a quad that crosses k reads into the next row and
    // is masked when quantized.  (Guarded loads merged their registers by
    // copies that waited for each other: 70 x 96 x 300 9.5 us.)
    const int rows = m - mt * 32 < 32 ? m - mt * 32 : 32;
    __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)(a + (long long)mt * 32 * k), (short)0,
                                                                  rows * k * 4, 0x00020000);
    __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(wpk + (col_live ? (long long)nt * ks * 1024 : 0)), (short)0, col_live ? ks * 1024 : 0, 0x00020000);
    auto load_pass = [&](int s0) {
        if constexpr (FULL) {
#pragma unroll
            for (int i = 0; i < KS; i++) {
                const float4 v = *reinterpret_cast<const float4 *>(src + (s0 + i) * 32 + 4 * c8);
                x[i].v[0] = v.x; x[i].v[1] = v.y; x[i].v[2] = v.z; x[i].v[3] = v.w;
            }
#pragma unroll
            for (int t = 0; t < KS; t++) b[t] = B[(s0 + t) * 64];
        } else {
#pragma unroll
            for (int i = 0; i < KS; i++) {
                const int kk = (s0 + i) * 32 + 4 * c8;
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(ra, kk < k ? (r * k + kk) * 4 : -1, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) x[i].v[e] = __uint_as_float(v[e]);
            }
#pragma unroll
            for (int t = 0; t < KS; t++) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b128(rb, lane * 16 + (s0 + t) * 1024, 0, 0);
                b[t] = i32x4{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
            }
        }
    };
    load_pass(0);
    // nothing below moves above this point: every load is out before the
    // first wait
    __builtin_amdgcn_sched_barrier(0);

    float inv, scale;
    int zp;
    dq_finish(sc, __builtin_fminf(0.f, pmin), __builtin_fmaxf(0.f, pmax), qparams, blockIdx.x == 0, inv, zp,
              &scale);
    const float zpf = (float)zp;

    // The MFMA chain runs as two interleaved chains (even and odd k-steps)
    // summed at the end; int32 sums are exact in any order.
    int sum = 0;
    bool nan = false;
    i32x16 acc0 = {}, acc1 = {};
    int *dst = lds_a + (r + 32 * (c8 >> 2)) * 4 + (c8 & 3);
    for (int ps = 0; ps < npass; ps++) {
        const int s0 = ps * KS;
        if constexpr (FULL) {
#pragma unroll
            for (int i = 0; i < KS; i++) dst[i * 256] = (int)quantize4(x[i], inv, zpf, 0xfu, sum, nan);
        } else {
            // k % 4 == 0: a quad is all inside its row or not there at all, so
            // one select masks it, and one its NaN flag (it loaded zeros, but
            // 0 * inv is a NaN where a tiny range makes inv infinite)
            if ((k & 3) == 0) {
#pragma unroll
                for (int i = 0; i < KS; i++) {
                    const bool in = live && (s0 + i) * 32 + 4 * c8 < k;
                    bool qnan = false;
                    const unsigned q = quantize4(x[i], inv, zpf, qnan);
                    nan |= in && qnan;
                    const int v = in ? (int)q : 0;
                    sum = __builtin_amdgcn_sdot4(v, 0x01010101, sum, false);
                    dst[i * 256] = v;
                }
            } else {  // element by element, and no more than 8 k-steps where that is all
#pragma unroll
                for (int i = 0; i < KS; i++) {
                    if (i == 8 && s0 + i >= ks) break;
                    const int kk = (s0 + i) * 32 + 4 * c8;
                    unsigned lm = 0;
#pragma unroll
                    for (int e = 0; e < 4; e++) lm |= (live && kk + e < k) ? (1u << e) : 0u;
                    dst[i * 256] = (int)quantize4(x[i], inv, zpf, lm, sum, nan);
                }
            }
        }
        __syncthreads();
        {
            const int *srcl = lds_a + lane * 4;
            if (FULL || s0 + KS <= ks) {  // k-steps past the last are zeros
                i32x4 av[KS];
#pragma unroll
                for (int t = 0; t < KS; t++) av[t] = *reinterpret_cast<const i32x4 *>(srcl + t * 256);
#pragma unroll
                for (int t = 0; t < KS; t += 2) {
                    acc0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[t], b[t], acc0, 0, 0, 0);
                    acc1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(av[t + 1], b[t + 1], acc1, 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int t = 0; t < KS; t++) {
                    if (s0 + t < ks) {
                        const i32x4 av = *reinterpret_cast<const i32x4 *>(srcl + t * 256);
                        if (t & 1) acc1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, b[t], acc1, 0, 0, 0);
                        else acc0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, b[t], acc0, 0, 0, 0);
                    }
                }
            }
        }
        if (ps + 1 < npass) {
            // the next pass's loads go out after this pass's MFMAs, whose b
            // registers they reuse
            __builtin_amdgcn_sched_barrier(0);
            load_pass(s0 + KS);  // x and b are free: the pass is quantized and multiplied
            __syncthreads();         // every wave's MFMAs have read the pass before it is rewritten
        }
    }
    const i32x16 acc = acc0 + acc1;
    // a row's 8 threads are consecutive lanes of one wave
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        sum += __shfl_xor(sum, o);
        const int other = __shfl_xor(nan ? 1 : 0, o);
        nan = nan || other != 0;
    }
    if (c8 == 0) {
        lds_rs[r] = sum;
        lds_rn[r] = nan ? 1 : 0;
    }
    __syncthreads();
    if (!jlive) return;
    const unsigned offj = (unsigned)col.off;
    const float bj = col.bias;
    const unsigned alpha = (unsigned)(128 - zp);
    const unsigned colterm = alpha * (unsigned)col.csum + (unsigned)k * alpha * offj;
    const float comb = scale * col.ws;  // CombinedScale, QuantizedMatMulOps.cs:203-221
    if constexpr (FULL) {
        // Float output only, 16-byte aligned: the wave's 32 x 32 tile goes
        // through its own 4 KB of lds_a (every wave's A reads ended before
        // the barrier above) so that each lane stores four 16-byte vectors
        // -- eight lanes a 128-byte row -- instead of 16 single words.  The
        // values are the ones the loop below computes.
        if (out && !acc_out && (reinterpret_cast<uintptr_t>(out) & 15) == 0) {  // uniform
            float *tl = reinterpret_cast<float *>(lds_a) + wt * 1024;
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const int il = 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
                const int v = (int)((unsigned)acc[q] + offj * (unsigned)lds_rs[il] + colterm);
                float o = __builtin_fmaf((float)v, comb, bj);
                if (lds_rn[il]) o = __builtin_nanf("");
                tl[il * 32 + (lane & 31)] = o;
            }
            // the lanes of this wave read what the others wrote (LDS accesses
            // of a wave are in order; this keeps the compiler from moving them)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int pass = 0; pass < 4; pass++) {
                const int rr = pass * 8 + (lane >> 3), c4 = (lane & 7) * 4;
                const float4 v4 = *reinterpret_cast<const float4 *>(tl + rr * 32 + c4);
                *reinterpret_cast<float4 *>(out + (long long)(mt * 32 + rr) * n + nt * 32 + c4) = v4;
            }
            return;
        }
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int il = 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
        const int i = mt * 32 + il;
        if (FULL || i < m) {
            const int rs = lds_rs[il], rn = lds_rn[il];
            const int v = (int)((unsigned)acc[q] + offj * (unsigned)rs + colterm);
            if (acc_out) acc_out[(long long)i * n + j] = v;
            if (out) {
                float o = __builtin_fmaf((float)v, comb, bj);
                if (rn) o = __builtin_nanf("");
                out[(long long)i * n + j] = o;
            }
        }
    }
}

// The fused kernel on 16 x 16 output tiles (v_mfma_i32_16x16x64_i8), for
// the full-tile case (m % 32 == 0, n % 128 == 0, k % 512 == 0, A 16-byte
// aligned).  Same workgroup tile (32 rows x 128 columns), same quantization
// and arithmetic as dqmm_fused_kernel, so the same bits; what differs is the
// schedule after the quantization barrier.  A wave's 32 x 32 block is four
// 16 x 16 tiles, each an 8-step chain over K = 512, run one after another:
// the integer correction, dequantization and stores of one tile are issued
// between the next tile's MFMAs, so the epilogue's VALU work and the output
// writes overlap the matrix core instead of following it.  The row sums and
// NaN flags are reduced before the barrier, so every tile's epilogue can run
// as soon as its chain ends.
//
// Operands: A (16 rows x 64 k per step) lane l holds row l & 15 and k =
// 64 s + 16 (l >> 4) + byte.  B is read straight from the 32 x 32 x 32
// packing: lane l of 16-column subtile c takes packed lane
// 16 c + (l & 15) + 32 ((l >> 4) & 1) of fragment 2 s + (l >> 5), whose k
// is the same 64 s + 16 (l >> 4) + byte, so A and B pair matching k.  The
// output tile's lane l holds column l & 15 and rows 4 (l >> 4) + v,
// v = 0..3.  ACC: the int32 accumulators are stored too.
//
// Tried and slower: the second half of K quantized between the first half's
// MFMAs, behind one more barrier (7.33 -> 7.65 us per op).
template <bool ACC>
__global__ __launch_bounds__(64 * DQF_WAVES) void dqmm_fused16_kernel(
    int m, int k, int n, const float *a, DqScratch *__restrict__ sc, int nparts, int *__restrict__ qparams,
    const int8_t *wpk, const int *__restrict__ colsum, const int *__restrict__ off,
    const float *__restrict__ wscale, int n_wscale, const float *__restrict__ bias, float *__restrict__ out,
    int *__restrict__ acc_out) {
    __shared__ __attribute__((aligned(16))) int lds_a[DQF_KS * 256];  // [kstep64 8][row tile 2][64 lanes][16 bytes]
    __shared__ __attribute__((aligned(16))) int lds_rs[32];
    __shared__ __attribute__((aligned(16))) int lds_rn[32];
    const int tid = threadIdx.x, lane = tid & 63, wt = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = k / 32;
    const int ncb = n / 32 / DQF_WAVES, nmt = m / 32;
    const int id = xcd_band(blockIdx.x, gridDim.x);
    const int grp = id / (DQF_GM * ncb), gl = id % (DQF_GM * ncb);
    const int mt0 = grp * DQF_GM;
    const int gm = nmt - mt0 < DQF_GM ? nmt - mt0 : DQF_GM;
    const int mt = mt0 + gl % gm;
    const int nt = (gl / gm) * DQF_WAVES + wt;
    const int r = tid >> 3, c8 = tid & 7;
    const float *src = a + (long long)(mt * 32 + r) * k;
    const int npass = ks / DQF_KS;
    // B: this lane's 16 bytes of packed lane 16 c + (lane & 15) + 32 ((lane >> 4) & 1)
    // of fragment (nt, 2 s + (lane >> 5)); subtile c adds 16 lanes (256 bytes)
    const int8_t *bl = wpk + ((long long)nt * ks + (lane >> 5)) * 1024 + ((lane & 15) + 32 * ((lane >> 4) & 1)) * 16;

    const int pidx = tid < nparts ? tid : 0;
    const float pmin = sc->partial_min[pidx], pmax = sc->partial_max[pidx];
    // the epilogue's column operands of both 16-column subtiles
    int offj_raw[2], csum[2];
    float ws[2], bj[2];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int j = nt * 32 + 16 * c + (lane & 15);
        offj_raw[c] = off[j];
        csum[c] = colsum[j];
        ws[c] = n_wscale == 1 ? wscale[0] : wscale[j];
        bj[c] = bias ? bias[j] : 0.0f;
    }

    Quad x[DQF_KS];
    i32x4 b[2][DQF_KS / 2];
    auto load_pass = [&](int s0) {
#pragma unroll
        for (int i = 0; i < DQF_KS; i++) {
            const float4 v = *reinterpret_cast<const float4 *>(src + (s0 + i) * 32 + 4 * c8);
            x[i].v[0] = v.x; x[i].v[1] = v.y; x[i].v[2] = v.z; x[i].v[3] = v.w;
        }
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int s = 0; s < DQF_KS / 2; s++)
                b[c][s] = *reinterpret_cast<const i32x4 *>(bl + (long long)(s0 + 2 * s) * 1024 + c * 256);
    };
    load_pass(0);
    __builtin_amdgcn_sched_barrier(0);

    float inv, scale;
    int zp;
    dq_finish(sc, __builtin_fminf(0.f, pmin), __builtin_fmaxf(0.f, pmax), qparams, blockIdx.x == 0, inv, zp,
              &scale);
    const float zpf = (float)zp;
    const unsigned alpha = (unsigned)(128 - zp);

    int sum = 0;
    bool nan = false;
    i32x4 acc[2][2] = {};
    i32x4 av[2][DQF_KS / 2];
    // quad i of this thread: k = 32 i + 4 c8 -> step i / 2, lane group 2 (i & 1) + c8 / 4
    int *dst = lds_a + ((r >> 4) * 64 + (r & 15) + 16 * (c8 >> 2)) * 4 + (c8 & 3);
    auto quantize_pass = [&]() {
#pragma unroll
        for (int i = 0; i < DQF_KS; i++)
            dst[(i >> 1) * 512 + (i & 1) * 128] = (int)quantize4(x[i], inv, zpf, 0xfu, sum, nan);
    };
    auto read_a = [&]() {
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
#pragma unroll
            for (int s = 0; s < DQF_KS / 2; s++)
                av[rt][s] = *reinterpret_cast<const i32x4 *>(lds_a + ((s * 2 + rt) * 64 + lane) * 4);
    };
    auto chain = [&](int t) {
#pragma unroll
        for (int s = 0; s < DQF_KS / 2; s++)
            acc[t >> 1][t & 1] =
                __builtin_amdgcn_mfma_i32_16x16x64_i8(av[t >> 1][s], b[t & 1][s], acc[t >> 1][t & 1], 0, 0, 0);
    };
    for (int ps = 0; ps + 1 < npass; ps++) {  // passes before the last (K > 512)
        quantize_pass();
        __syncthreads();
        read_a();
#pragma unroll
        for (int t = 0; t < 4; t++) chain(t);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();  // every wave has read this pass's a'' before it is rewritten
        load_pass((ps + 1) * DQF_KS);
    }
    quantize_pass();
    // row sums and NaN flags: a row's 8 threads are consecutive lanes
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
        sum += __shfl_xor(sum, o);
        const int other = __shfl_xor(nan ? 1 : 0, o);
        nan = nan || other != 0;
    }
    if (c8 == 0) {
        lds_rs[r] = sum;
        lds_rn[r] = nan ? 1 : 0;
    }
    __syncthreads();
    read_a();
    // the lane's row sums and NaN flags (rows 16 rt + 4 (lane >> 4) + v)
    int4 rs4[2], rn4[2];
#pragma unroll
    for (int rt = 0; rt < 2; rt++) {
        rs4[rt] = *reinterpret_cast<const int4 *>(lds_rs + 16 * rt + 4 * (lane >> 4));
        rn4[rt] = *reinterpret_cast<const int4 *>(lds_rn + 16 * rt + 4 * (lane >> 4));
    }
    auto epilogue = [&](int t) {
        const int rt = t >> 1, c = t & 1;
        const int j = nt * 32 + 16 * c + (lane & 15);
        const unsigned offj = (unsigned)offj_raw[c];
        const unsigned colterm = alpha * (unsigned)csum[c] + (unsigned)k * alpha * offj;
        const float comb = scale * ws[c];  // CombinedScale, QuantizedMatMulOps.cs:203-221
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int il = 16 * rt + 4 * (lane >> 4) + v;
            const int rsv = v == 0 ? rs4[rt].x : v == 1 ? rs4[rt].y : v == 2 ? rs4[rt].z : rs4[rt].w;
            const int rnv = v == 0 ? rn4[rt].x : v == 1 ? rn4[rt].y : v == 2 ? rn4[rt].z : rn4[rt].w;
            const int val = (int)((unsigned)acc[rt][c][v] + offj * (unsigned)rsv + colterm);
            const long long o_idx = (long long)(mt * 32 + il) * n + j;
            if constexpr (ACC) acc_out[o_idx] = val;
            const float o = __builtin_fmaf((float)val, comb, bj[c]);
            out[o_idx] = rnv ? __builtin_nanf("") : o;
        }
    };
    // tile t's chain, with tile t - 1's epilogue issued between its MFMAs:
    // the epilogue's VALU work and stores overlap the matrix core
    chain(0);
#pragma unroll
    for (int t = 1; t < 4; t++) {
        chain(t);
        epilogue(t - 1);
#pragma unroll
        for (int q = 0; q < DQF_KS / 2; q++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);  // five VALU
            __builtin_amdgcn_sched_group_barrier(0x040, 1, 0);  // one global store
        }
    }
    epilogue(3);
}

// Quantize + GEMM for at most RT <= 16 rows (a token, a few beams), after
// dqmm_minmax_kernel.  A 32-row tile would leave most threads without a row to
// quantize and a 128-column workgroup most CUs without work (3 x 1912 x 168 ran
// on two workgroups, 28 us), so here a workgroup owns 32 columns and its four
// waves split K, k-step s to wave s % 4; the sums meet in LDS, exact in int32.
// 256 / RT threads quantize each row, DQS_KS k-steps a pass; every wave's W
// fragments of two passes (K = 2048) are in flight before the parameter
// reduction.  Rows of the A tile past m, and k-steps past the last that are not
// quantized, are whatever LDS held: the ones reach only output rows that do not
// exist, the others meet zero W.
constexpr int DQS_KS = 32;  // k-steps a pass
constexpr int DQS_WS = DQS_KS / 4;

template <int RT>
__global__ __launch_bounds__(256) void dqmm_skinny_kernel(
    int m, int k, int n, const float *a, DqScratch *__restrict__ sc, int nparts, int *__restrict__ qparams,
    const int8_t *wpk, const int *__restrict__ colsum, const int *__restrict__ off,
    const float *__restrict__ wscale, int n_wscale, const float *__restrict__ bias, float *__restrict__ out,
    int *__restrict__ acc_out) {
    static_assert(RT <= 16, "two row quads of the accumulator");
    constexpr int TPR = 256 / RT;  // threads a row
    __shared__ __attribute__((aligned(16))) int lds_a[DQS_KS * 256];  // [kstep][64 lanes][16 bytes]
    __shared__ int lds_acc[4][8][64];
    __shared__ int lds_rs[RT], lds_rn[RT];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = pad32(k) / 32, nt = blockIdx.x;
    const int r = tid / TPR, c = tid % TPR;
    const int pidx = tid < nparts ? tid : 0;
    const float pmin = sc->partial_min[pidx], pmax = sc->partial_max[pidx];
    const int oc = tid & 31, j = nt * 32 + oc;  // the output column this thread ends with
    const ColOperands col = load_column(j, n, colsum, off, wscale, n_wscale, bias);
    __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void *)a, (short)0, m * k * 4, 0x00020000);
    __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)(wpk + (long long)nt * ks * 1024), (short)0,
                                                                  ks * 1024, 0x00020000);
    Quad x[RT];  // quad i of this thread: k = 32 s0 + 4 (c + TPR i)
    auto load_a = [&](int s0) {
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const int kk = s0 * 32 + 4 * (c + TPR * i);
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(ra, kk < k ? (r * k + kk) * 4 : -1, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; e++) x[i].v[e] = __uint_as_float(v[e]);
        }
    };
    i32x4 b[2][DQS_WS];
    auto load_b = [&](i32x4 (&bb)[DQS_WS], int s0) {
#pragma unroll
        for (int t = 0; t < DQS_WS; t++) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(rb, lane * 16 + (s0 + 4 * t + wave) * 1024, 0, 0);
            bb[t] = i32x4{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
        }
    };
    load_a(0);
    load_b(b[0], 0);
    load_b(b[1], DQS_KS);
    if (tid < RT) lds_rs[tid] = lds_rn[tid] = 0;
    __builtin_amdgcn_sched_barrier(0);
    float inv, scale;
    int zp;
    dq_finish(sc, __builtin_fminf(0.f, pmin), __builtin_fmaxf(0.f, pmax), qparams, blockIdx.x == 0, inv, zp,
              &scale);
    const float zpf = (float)zp;
    int sum = 0;
    bool nan = false;
    i32x16 acc0 = {}, acc1 = {};
    auto pass = [&](i32x4 (&bb)[DQS_WS], int s0) {
#pragma unroll
        for (int i = 0; i < RT; i++) {
            // every 256 k: no more of them (9 x 90 x 88 8.6 us, so 7.0)
            if (i && TPR * 4 * i % 256 == 0 && s0 * 32 + TPR * 4 * i >= k) break;
            const int kl = 4 * (c + TPR * i), kk = s0 * 32 + kl;
            unsigned lm = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) lm |= (r < m && kk + e < k) ? (1u << e) : 0u;
            lds_a[(kl >> 5) * 256 + (r + 32 * ((kl >> 4) & 1)) * 4 + ((kl & 15) >> 2)] =
                (int)quantize4(x[i], inv, zpf, lm, sum, nan);
        }
        __syncthreads();
        const int *src = lds_a + lane * 4;
#pragma unroll
        for (int t = 0; t < DQS_WS; t += 2) {
            acc0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                *reinterpret_cast<const i32x4 *>(src + (4 * t + wave) * 256), bb[t], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(
                *reinterpret_cast<const i32x4 *>(src + (4 * t + 4 + wave) * 256), bb[t + 1], acc1, 0, 0, 0);
        }
        if (s0 + DQS_KS < ks) {
            load_a(s0 + DQS_KS);
            load_b(bb, s0 + 2 * DQS_KS);
            __syncthreads();  // every wave has read the pass before it is rewritten
        }
    };
    for (int s0 = 0; s0 < ks; s0 += 2 * DQS_KS) {
        pass(b[0], s0);
        if (s0 + DQS_KS < ks) pass(b[1], s0 + DQS_KS);
    }
    // a row's threads: whole waves, or consecutive lanes of one
#pragma unroll
    for (int o = 1; o < (TPR < 64 ? TPR : 64); o <<= 1) {
        sum += __shfl_xor(sum, o);
        const int other = __shfl_xor(nan ? 1 : 0, o);
        nan = nan || other != 0;
    }
    if ((tid & ((TPR < 64 ? TPR : 64) - 1)) == 0) {
        atomicAdd(lds_rs + r, sum);
        if (nan) lds_rn[r] = 1;
    }
#pragma unroll
    for (int v = 0; v < 8; v++) lds_acc[wave][v][lane] = acc0[v] + acc1[v];
    __syncthreads();
    if (j >= n) return;
    const unsigned alpha = (unsigned)(128 - zp), offj = (unsigned)col.off;
    const unsigned colterm = alpha * (unsigned)col.csum + (unsigned)k * alpha * offj;
    const float comb = scale * col.ws;  // CombinedScale, QuantizedMatMulOps.cs:203-221
    for (int row = tid >> 5; row < m; row += 8) {
        // the accumulator's row 8 q + 4 half + e: register 4 q + e of lane column + 32 half
        const int reg = 4 * (row >> 3) + (row & 3), l = oc + 32 * ((row >> 2) & 1);
        unsigned v = 0;
#pragma unroll
        for (int w = 0; w < 4; w++) v += (unsigned)lds_acc[w][reg][l];
        const int val = (int)(v + offj * (unsigned)lds_rs[row] + colterm);
        if (acc_out) acc_out[(long long)row * n + j] = val;
        if (out) {
            const float o = __builtin_fmaf((float)val, comb, col.bias);
            out[(long long)row * n + j] = lds_rn[row] ? __builtin_nanf("") : o;
        }
    }
}

static osh_status run_minmax(const float *a, long long count, DqScratch *sc, int *nparts, hipStream_t st,
                             int *zero = nullptr, int zero_n = 0) {
    long long blocks = (count / 4 + DQ_THREADS - 1) / DQ_THREADS;
    if (blocks < 1) blocks = 1;
    if (blocks > DQ_MINMAX_BLOCKS) blocks = DQ_MINMAX_BLOCKS;
    OSH_LAUNCH(dqmm_minmax_kernel, dim3((unsigned)blocks), dim3(DQ_THREADS), 0, st, a, count, sc, zero,
               zero_n);
    *nparts = (int)blocks;
    OSH_LAUNCH_CHECK("dqmm_minmax_kernel");
    return OSH_OK;
}

static osh_status launch_int8_gemm(int m, int k, int n, const int8_t *apk, const int8_t *wpk, const int *colsum,
                                   const int *off, const int *rownan, const DqScratch *sc, const float *wscale,
                                   int n_wscale, const float *bias, float *out, int *acc_out, hipStream_t st) {
    const int mt = pad32(m) / 32, nb = (pad32(n) / 32 + 3) / 4;
    if ((long long)mt * nb > 0x7fffffffLL) return fail(OSH_E_UNSUPPORTED, "int8 GEMM grid too large");
#define OSH_I8_GEMM_OUT(TM, SETS, OUT)                                                                       \
    OSH_LAUNCH((dqmm_gemm_kernel<TM, SETS, OUT>), dim3((unsigned)((long long)((mt + TM - 1) / TM) * nb)),    \
               dim3(256), 0, st, m, k, n, apk, wpk, colsum, off, rownan, sc, wscale, n_wscale, bias, out, acc_out)
#define OSH_I8_GEMM(TM, SETS)                                         \
    do {                                                              \
        if (!acc_out) OSH_I8_GEMM_OUT(TM, SETS, DQG_FLOAT);           \
        else if (!out) OSH_I8_GEMM_OUT(TM, SETS, DQG_ACC);            \
        else OSH_I8_GEMM_OUT(TM, SETS, DQG_FLOAT | DQG_ACC);          \
    } while (0)
    // 64-row tiles (half the W traffic) where they still give 3 workgroups for
    // every 2 CUs, with two stages in flight so that more workgroups share a CU:
    // 1028 x 1280 x 5120 25.2 us (32-row tiles 30.0); 669 x 352 x 2368 13.6 (13.3).
    if ((long long)((mt + 1) / 2) * nb >= 3LL * device_cus() / 2) OSH_I8_GEMM(2, 2);
    // of which no more in flight than there are (1 x 18 x 3094 5.05 us, with four 5.24)
    else if (k <= 2 * 32 * DQG_KS) OSH_I8_GEMM(1, 2);
    else OSH_I8_GEMM(1, 4);
#undef OSH_I8_GEMM
#undef OSH_I8_GEMM_OUT
    OSH_LAUNCH_CHECK("dqmm_gemm_kernel");
    return OSH_OK;
}

static thread_local int t_dqmm_launches = 0;
int dqmm_last_launches() { return t_dqmm_launches; }

static osh_status dqmm_run(int m, int k, int n, const float *d_a, const void *d_wpacked, const float *d_wscale,
                           int n_wscale, const float *d_bias, float *d_out, int32_t *d_acc, int32_t *d_qparams,
                           void *d_scratch, hipStream_t st) {
    DqScratch *sc = static_cast<DqScratch *>(d_scratch);
    int *rownan = reinterpret_cast<int *>(sc + 1);  // the second mpad ints of the layout are spare
    int8_t *apk = reinterpret_cast<int8_t *>(rownan + 2 * pad32(m));
    const int8_t *frag = static_cast<const int8_t *>(d_wpacked);
    const int *colsum = reinterpret_cast<const int *>(frag + (size_t)pad32(n) * pad32(k));
    const int *off = colsum + pad32(n);
    const long long fblocks = (long long)((pad32(n) / 32 + DQF_WAVES - 1) / DQF_WAVES) * (pad32(m) / 32);
    const long long total = (long long)m * k;
    int nparts = 0;
    const bool full = m % 32 == 0 && n % 128 == 0 && k % (32 * DQF_KS) == 0 &&
                      (reinterpret_cast<uintptr_t>(d_a) & 15) == 0;
    const int variant = dqmm_variant();
    // Every 128-column block of the fused launch quantizes its rows again, which
    // a separate quantize launch (about 4.3 us) ends.  The two cross at 4e9
    // products on full tiles (2048 x 512 x 2048 15.1 us in two launches, 18.3 in
    // three; 1024 x 1024 x 4096 22.1 and 20.3) and between 0.5e9 and 2e9 on ragged
    // ones: later with K % 4 == 0 (669 x 352 x 2368 11.7 and 13.3; 1256 x 812 x
    // 1242 14.9 and 16.6; 777 x 700 x 3000 21.7 and 17.8; 1028 x 1280 x 5120 42.1
    // and 25.2) than without, where the fused launch masks each element (268 x
    // 1946 x 1907, just below the line, 25.1 and 15.5).  At most 16 rows take the
    // skinny kernel instead (16 x 2048 x 8192 14.1 us, 14.2 in three).
    const double macs = (double)m * n * k;
    const bool three = variant == 1 || fblocks > 0x7fffffffLL || (m > 16 && macs > (full ? 4e9 : 1e9));
    osh_status r = run_minmax(d_a, total, sc, &nparts, st, three ? rownan : nullptr, three ? pad32(m) : 0);
    if (r != OSH_OK) return r;
    if (!three) {
        if (m <= 16) {
            const dim3 grid((unsigned)(pad32(n) / 32));
#define OSH_SKINNY(RT)                                                                                               \
    OSH_LAUNCH(dqmm_skinny_kernel<RT>, grid, dim3(256), 0, st, m, k, n, d_a, sc, nparts, (int *)d_qparams, frag, colsum, \
               off, d_wscale, n_wscale, d_bias, d_out, (int *)d_acc)
            if (m == 1) OSH_SKINNY(1);
            else if (m == 2) OSH_SKINNY(2);
            else if (m <= 4) OSH_SKINNY(4);
            else if (m <= 8) OSH_SKINNY(8);
            else OSH_SKINNY(16);
#undef OSH_SKINNY
        } else if (full && variant == 0 && d_acc)
            OSH_LAUNCH(dqmm_fused16_kernel<true>, dim3((unsigned)fblocks), dim3(64 * DQF_WAVES), 0, st, m, k, n,
                       d_a, sc, nparts, (int *)d_qparams, frag, colsum, off, d_wscale, n_wscale, d_bias, d_out,
                       (int *)d_acc);
        else if (full && variant == 0)
            OSH_LAUNCH(dqmm_fused16_kernel<false>, dim3((unsigned)fblocks), dim3(64 * DQF_WAVES), 0, st, m, k, n,
                       d_a, sc, nparts, (int *)d_qparams, frag, colsum, off, d_wscale, n_wscale, d_bias, d_out,
                       (int *)d_acc);
        else if (full)
            OSH_LAUNCH((dqmm_fused_kernel<true, DQF_KS>), dim3((unsigned)fblocks), dim3(64 * DQF_WAVES), 0, st, m, k, n,
                               d_a, sc, nparts, (int *)d_qparams, frag, colsum, off, d_wscale, n_wscale, d_bias, d_out,
                               (int *)d_acc);
        else {
#define OSH_RAGGED(KS)                                                                                               \
    OSH_LAUNCH((dqmm_fused_kernel<false, KS>), dim3((unsigned)fblocks), dim3(64 * DQF_WAVES), 0, st, m, k, n, d_a, sc, \
               nparts, (int *)d_qparams, frag, colsum, off, d_wscale, n_wscale, d_bias, d_out, (int *)d_acc)
            if (k <= 4 * 32) OSH_RAGGED(4);
            else if (k <= 8 * 32) OSH_RAGGED(8);
            else OSH_RAGGED(DQF_KS);
#undef OSH_RAGGED
        }
        OSH_LAUNCH_CHECK("dqmm_fused_kernel");
        t_dqmm_launches = 2;
        return OSH_OK;
    }
    const long long waves = (long long)(pad32(m) / 32) * ((pad32(k) / 32 + DQ_QF - 1) / DQ_QF);
    const long long qblocks = (waves + DQ_THREADS / 64 - 1) / (DQ_THREADS / 64);
    if (qblocks > 0x7fffffffLL) return fail(OSH_E_UNSUPPORTED, "DQM: m too large");
    OSH_LAUNCH(dqmm_quantize_kernel, dim3((unsigned)qblocks), dim3(DQ_THREADS), 0, st, d_a, m, k, sc, nparts,
               (int *)d_qparams, rownan, apk);
    OSH_LAUNCH_CHECK("dqmm_quantize_kernel");
    r = launch_int8_gemm(m, k, n, apk, frag, colsum, off, rownan, sc, d_wscale, n_wscale, d_bias, d_out, (int *)d_acc,
                         st);
    if (r != OSH_OK) return r;
    t_dqmm_launches = 3;
    return OSH_OK;
}

static osh_status dqmm_check(int m, int k, int n, const float *d_a, const void *d_wpacked, const float *d_wscale,
                             int n_wscale, float *d_out) {
    if (m < 0 || k <= 0 || n <= 0) return fail(OSH_E_INVALID, "DQM: bad size m=%d k=%d n=%d", m, k, n);
    if (m == 0) return OSH_OK;
    if (!d_a || !d_wpacked || !d_wscale || !d_out) return fail(OSH_E_INVALID, "DQM: NULL pointer");
    if (n_wscale != 1 && n_wscale != n) return fail(OSH_E_INVALID, "DQM: w_scale has %d entries", n_wscale);
    if ((long long)k * 255 * 255 > 2147483647LL)
        return fail(OSH_E_UNSUPPORTED, "DQM: K=%d can overflow the int32 accumulator", k);
    if (pad32(m) / 32 > 2 * 65535) return fail(OSH_E_UNSUPPORTED, "DQM: m too large");
    return OSH_OK;
}

// The no-allocation variant's scratch: one array per GPU, held until the
// process ends.  `scratch` names the host-side stand-in; kernels take the
// device address hipGetSymbolAddress returns for the current device.
constexpr size_t kNoAllocScratchBytes = (size_t)4 << 20;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kNoAllocMaxDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kNoAllocMaxDevices];

// Resolves (once per device, with that device current) the device address of
// `scratch`; osh_init calls it, and the entry point calls it on its first
// call on a device that osh_init did not set up.
osh_status noalloc_scratch_setup(int dev) {
    if (dev < 0 || dev >= kNoAllocMaxDevices)
        return fail(OSH_E_UNSUPPORTED, "DQM (no allocation): device %d beyond %d devices", dev, kNoAllocMaxDevices);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev]) return OSH_OK;
    void *ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        (void)hipGetLastError();
        return fail(OSH_E_DEVICE, "DQM (no allocation): hipGetSymbolAddress(scratch) on device %d failed: %s", dev,
                    hipGetErrorString(e));
    }
    g_scratch_ptr[dev] = ptr;
    return OSH_OK;
}

}  // namespace osh

extern "C" {

OSH_API osh_status osh_dqmm_packed_weight_bytes(int k, int n, size_t *bytes) {
    if (k <= 0 || n <= 0 || !bytes) return fail(OSH_E_INVALID, "DQM: bad size");
    *bytes = packed_w_bytes(k, n);
    return OSH_OK;
}

OSH_API osh_status osh_dqmm_scratch_bytes(int m, int k, size_t *bytes) {
    if (m < 0 || k <= 0 || !bytes) return fail(OSH_E_INVALID, "DQM: bad size");
    *bytes = scratch_bytes(m, k);
    return OSH_OK;
}

OSH_API osh_status osh_dqmm_pack_weights(int k, int n, const void *d_w, int w_signed, const int32_t *h_wzp,
                                         int n_wzp, void *d_packed, osh_stream s) {
    if (k <= 0 || n <= 0 || !d_w || !d_packed) return fail(OSH_E_INVALID, "DQM pack: bad argument");
    if (n_wzp != 0 && n_wzp != 1 && n_wzp != n)
        return fail(OSH_E_INVALID, "DQM pack: w_zero_point has %d entries (need 1 or %d)", n_wzp, n);
    if (n_wzp > 0 && !h_wzp) return fail(OSH_E_INVALID, "DQM pack: w_zero_point is NULL");
    if ((long long)k * 255 * 255 > 2147483647LL)
        return fail(OSH_E_UNSUPPORTED, "DQM: K=%d can overflow the int32 accumulator", k);
    // a zero point has the weights' element type (ONNX MatMulInteger /
    // DynamicQuantizeMatMul), so |w - w_zp| <= 255 and K * 255 * 255 bounds
    // the accumulator (checked above)
    const int zlo = w_signed ? -128 : 0, zhi = w_signed ? 127 : 255;
    for (int i = 0; i < n_wzp; i++)
        if (h_wzp[i] < zlo || h_wzp[i] > zhi)
            return fail(OSH_E_INVALID, "DQM pack: weight zero point %d outside the %s range [%d, %d]", h_wzp[i],
                        w_signed ? "int8" : "uint8", zlo, zhi);
    hipStream_t st = to_stream(s);
    int *d_zp = nullptr;
    if (n_wzp > 0) {
        OSH_HIP_CHECK(hipMalloc((void **)&d_zp, sizeof(int) * n_wzp));
        hipError_t e = hipMemcpyAsync(d_zp, h_wzp, sizeof(int) * n_wzp, hipMemcpyHostToDevice, st);
        if (e != hipSuccess) {
            (void)hipFree(d_zp);
            return fail(OSH_E_DEVICE, "DQM pack: copy of zero points failed: %s", hipGetErrorString(e));
        }
    }
    int8_t *frag = static_cast<int8_t *>(d_packed);
    int *colsum = reinterpret_cast<int *>(frag + (size_t)pad32(n) * pad32(k));
    int *off = colsum + pad32(n);
    OSH_LAUNCH(dqmm_pack_kernel, dim3((pad32(n) + 63) / 64), dim3(64), 0, st, k, n, d_w, w_signed, d_zp,
                       n_wzp, frag, colsum, off);
    hipError_t le = hipGetLastError();
    hipError_t se = hipStreamSynchronize(st);
    if (d_zp) (void)hipFree(d_zp);
    if (le != hipSuccess) return fail(OSH_E_DEVICE, "dqmm_pack_kernel launch failed: %s", hipGetErrorString(le));
    if (se != hipSuccess) return fail(OSH_E_DEVICE, "DQM pack failed: %s", hipGetErrorString(se));
    return OSH_OK;
}

OSH_API osh_status osh_dqmm_u8s8(int m, int k, int n, const float *d_a, const void *d_wpacked,
                                 const float *d_wscale, int n_wscale, const float *d_bias, float *d_out,
                                 int32_t *d_acc, int32_t *d_qparams, void *d_scratch, osh_stream s) {
    osh_status st = dqmm_check(m, k, n, d_a, d_wpacked, d_wscale, n_wscale, d_out);
    if (st != OSH_OK || m == 0) return st;
    if (!d_scratch) return fail(OSH_E_INVALID, "DQM: NULL pointer");
    return dqmm_run(m, k, n, d_a, d_wpacked, d_wscale, n_wscale, d_bias, d_out, d_acc, d_qparams, d_scratch,
                    to_stream(s));
}

OSH_API osh_status osh_dqmm_u8s8_noalloc(int m, int k, int n, const float *d_a, const void *d_wpacked,
                                         const float *d_wscale, int n_wscale, const float *d_bias, float *d_out,
                                         int32_t *d_acc, int32_t *d_qparams, osh_stream s) {
    osh_status st = dqmm_check(m, k, n, d_a, d_wpacked, d_wscale, n_wscale, d_out);
    if (st != OSH_OK || m == 0) return st;
    if (scratch_bytes(m, k) > kNoAllocScratchBytes)
        return fail(OSH_E_UNSUPPORTED,
                    "DQM (no allocation): m=%d, k=%d need %zu scratch bytes; the static scratch holds %zu", m, k,
                    scratch_bytes(m, k), kNoAllocScratchBytes);
    int dev = 0;
    OSH_HIP_CHECK(hipGetDevice(&dev));
    void *ptr = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        if (dev >= 0 && dev < kNoAllocMaxDevices) ptr = g_scratch_ptr[dev];
    }
    if (!ptr) {
        st = noalloc_scratch_setup(dev);
        if (st != OSH_OK) return st;
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        ptr = g_scratch_ptr[dev];
    }
    return dqmm_run(m, k, n, d_a, d_wpacked, d_wscale, n_wscale, d_bias, d_out, d_acc, d_qparams, ptr,
                    to_stream(s));
}

OSH_API osh_status osh_matmul_integer(int m, int k, int n, const void *d_a, int a_signed, int a_zp,
                                      const void *d_wpacked, int32_t *d_c, void *d_scratch, osh_stream s) {
    if (m < 0 || k <= 0 || n <= 0) return fail(OSH_E_INVALID, "MatMulInteger: bad size m=%d k=%d n=%d", m, k, n);
    if (m == 0) return OSH_OK;
    if (!d_a || !d_wpacked || !d_c || !d_scratch) return fail(OSH_E_INVALID, "MatMulInteger: NULL pointer");
    if (a_zp < (a_signed ? -128 : 0) || a_zp > (a_signed ? 127 : 255))
        return fail(OSH_E_INVALID, "MatMulInteger: a_zero_point %d outside the %s range", a_zp,
                    a_signed ? "int8" : "uint8");
    if ((long long)k * 255 * 255 > 2147483647LL)
        return fail(OSH_E_UNSUPPORTED, "MatMulInteger: K=%d can overflow the int32 accumulator", k);
    if (pad32(m) / 32 > 2 * 65535) return fail(OSH_E_UNSUPPORTED, "MatMulInteger: m too large");
    hipStream_t st = to_stream(s);
    DqScratch *sc = static_cast<DqScratch *>(d_scratch);
    int *rownan = reinterpret_cast<int *>(sc + 1);  // the second mpad ints of the layout are spare
    int8_t *apk = reinterpret_cast<int8_t *>(rownan + 2 * pad32(m));
    const uint8_t *a = static_cast<const uint8_t *>(d_a);
    const bool vec = k % 16 == 0 && (reinterpret_cast<uintptr_t>(a) & 15) == 0;
    const long long frags = (long long)(pad32(m) / 32) * (pad32(k) / 32);
    const long long pblocks = (frags + DQ_THREADS / 64 - 1) / (DQ_THREADS / 64);
    if (pblocks > 0x7fffffffLL) return fail(OSH_E_UNSUPPORTED, "MatMulInteger: m too large");
#define OSH_MMI_PACK(VEC)                                                                                      \
    OSH_LAUNCH(mmi_pack_a_kernel<VEC>, dim3((unsigned)pblocks), dim3(DQ_THREADS), 0, st, a, m, k, a_signed, \
               a_zp, sc, rownan, apk)
    if (vec) OSH_MMI_PACK(true);
    else OSH_MMI_PACK(false);
#undef OSH_MMI_PACK
    OSH_LAUNCH_CHECK("mmi_pack_a_kernel");
    const int8_t *frag = static_cast<const int8_t *>(d_wpacked);
    const int *colsum = reinterpret_cast<const int *>(frag + (size_t)pad32(n) * pad32(k));
    const int *off = colsum + pad32(n);
    return launch_int8_gemm(m, k, n, apk, frag, colsum, off, rownan, sc, nullptr, 1, nullptr, nullptr, (int *)d_c, st);
}

OSH_API osh_status osh_dynamic_quantize_linear(int64_t n, const float *d_x, uint8_t *d_q, int32_t *d_qparams,
                                               void *d_scratch, osh_stream s) {
    if (n <= 0 || !d_x || !d_q || !d_scratch) return fail(OSH_E_INVALID, "DQL: bad argument");
    hipStream_t st = to_stream(s);
    DqScratch *sc = static_cast<DqScratch *>(d_scratch);
    int nparts = 0;
    osh_status r = run_minmax(d_x, n, sc, &nparts, st);
    if (r != OSH_OK) return r;
    long long blocks = (n + DQ_THREADS - 1) / DQ_THREADS;
    if (blocks > 4096) blocks = 4096;
    OSH_LAUNCH(dql_quantize_kernel, dim3((unsigned)blocks), dim3(DQ_THREADS), 0, st, d_x, n, sc, nparts,
                       (int *)d_qparams, d_q);
    OSH_LAUNCH_CHECK("dql_quantize_kernel");
    return OSH_OK;
}

}  // extern "C"
