// osh_winograd.h -- Winograd F(2x2, 3x3) convolution (stride 1, pad 1) on
// v_mfma_f32_16x16x4f32, in the arithmetic of the reference's Winograd.cs:
//
//   weights  u = G g G^T with the 1/2 factors          (Winograd.cs:125-166)
//   input    v = B^T d B of each 4x4 patch (pad = 0)   (Winograd.cs:260-357)
//   product  M[comp][oc][tile] = sum over ic, ascending, of U[comp][oc][ic] * V[comp][ic][tile],
//            one fmaf chain from 0                       (Winograd.cs:234-258 -> GemmKernel.Multiply)
//   output   y = A^T M A, bias added last               (Winograd.cs:444-536)
//
// then the fused activation and an optional residual, as the other conv
// kernels apply them.  Every transform is the reference's sequence of single
// IEEE additions (this file is built with -ffp-contract=off), and the MFMA
// adds its four lane-group products one after another like fmaf, with ic in
// ascending order, so the result is the reference's Winograd path bit for
// bit (the GEMM's scalar tail columns aside: GemmKernel.MultiplyRow sums
// columns past the last full 8-column vector of a partial 16-column panel
// with separate multiply and add).
//
// One workgroup owns 16 tiles (a tile is a 2x2 output block; tiles run over
// batch, tile row, tile column) x 16 OB output channels for all 16 components,
// four waves an output block.  Per chunk of 16 input channels the first four
// waves transform one (ic, tile) patch a thread into LDS as [comp][ic][tile];
// wave w runs the MFMA chains of components 4 (w % 4) .. + 3 of output block
// w / 4.  Patches and weights are loaded a chunk ahead of their use, all
// without a condition (what does not exist lies outside the buffer descriptors
// and loads as zero), a patch row as one value and three; the component planes
// are double-buffered.  At the end the accumulators go through LDS as
// [comp][oc][tile] and each thread transforms one (oc, tile) to its 2x2
// outputs, stored two at a time.
//
// Bound by waiting: at 8 x 64 x 56 x 56 -> 64 with a residual (21.3 us; 33.5 with
// patch loads and stores one guarded value at a time) the waves wait for 48% of
// their cycles, at each chunk's barrier and for the loads behind it, with the MFMAs
// 24% busy, vector issue 19%, LDS 14%, L2 reads 8 TB/s.  One output block a
// workgroup reads a third more through L1 and takes the same time.  Slower:
// workgroups of 32 tiles, weights shared through L1 (5-10%); all 16 components x 32
// x 32 in four waves (40%: registers); patches two chunks ahead, no change.
#pragma once

#include "osh_common.h"

namespace osh {

// Winograd.TryConv3x3's gate (Winograd.cs:58-122) on a resolved conv.
inline bool winograd_eligible(const osh_conv_params *p, long long max_pixels) {
    return p->group == 1 && p->kh == 3 && p->kw == 3 && p->sh == 1 && p->sw == 1 && p->dh == 1 && p->dw == 1 &&
           p->pt == 1 && p->pl == 1 && p->c >= 8 && p->m >= 8 && p->oh == p->h && p->ow == p->w && p->h >= 6 &&
           p->w >= 6 && (long long)p->h * p->w <= max_pixels && (long long)p->m * p->c * 16 <= (1LL << 24) &&
           (long long)p->n * p->c * p->h * p->w < (1LL << 31) && (long long)p->n * p->m * p->h * p->w < (1LL << 31) &&
           (long long)p->n * ((p->h + 1) / 2) * ((p->w + 1) / 2) <= 16LL * 65535;  // grid y
}

// Packed U: [16 comps][ceil(M/16)][ceil(C/16)][64 lanes][4]; lane (j, g) =
// (lane & 15, lane >> 4) holds U[comp][16*ob + j][16*cb + 4*s + g] in slot s,
// zero for padding channels.
inline size_t winograd_packed_bytes(const osh_conv_params *p) {
    return (size_t)16 * ((p->m + 15) / 16) * ((p->c + 15) / 16) * 256 * sizeof(float);
}

__global__ void wino_pack_kernel(int M, int C, const float *__restrict__ w, float *__restrict__ out) {
    const int ocbs = (M + 15) / 16, cbs = (C + 15) / 16;
    const long long total = (long long)ocbs * 16 * cbs * 16;
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int oc = (int)(idx / (cbs * 16)), ic = (int)(idx % (cbs * 16));
    float u[16];
    if (oc < M && ic < C) {
        const float *g = w + ((long long)oc * C + ic) * 9;
        float s[12];
        for (int j = 0; j < 3; j++) {  // s = G g (4x3)
            const float g0 = g[j], g1 = g[3 + j], g2 = g[6 + j];
            s[j] = g0;
            s[3 + j] = (g0 + g1 + g2) * 0.5f;
            s[6 + j] = (g0 - g1 + g2) * 0.5f;
            s[9 + j] = g2;
        }
        for (int i = 0; i < 4; i++) {  // u = s G^T (4x4)
            const float a = s[i * 3], b = s[i * 3 + 1], c = s[i * 3 + 2];
            u[i * 4] = a;
            u[i * 4 + 1] = (a + b + c) * 0.5f;
            u[i * 4 + 2] = (a - b + c) * 0.5f;
            u[i * 4 + 3] = c;
        }
    } else {
        for (int i = 0; i < 16; i++) u[i] = 0.0f;
    }
    const int ob = oc >> 4, j = oc & 15, cb = ic >> 4, icl = ic & 15;
    const int lane = (icl & 3) * 16 + j, slot = icl >> 2;
    for (int comp = 0; comp < 16; comp++)
        out[((((long long)comp * ocbs + ob) * cbs + cb) * 64 + lane) * 4 + slot] = u[comp];
}

typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

// Buffer records end at least 64 bytes below this offset: a load there is zero.
constexpr int kWinoNowhere = 0x7fffff80;

template <int ACT, int OB>
__global__ __launch_bounds__(256 * OB, 4) void wino_f23_kernel(osh_conv_params p, const float *__restrict__ x,
                                                                   const float4 *__restrict__ up,
                                                                   const float *__restrict__ bias,
                                                                   const float *__restrict__ res,
                                                                   float *__restrict__ y) {
    static_assert(OB <= 2, "the accumulators take the two buffers of planes");
    constexpr int NT = 16;                // tiles
    constexpr int PLANE = 16 * NT;        // floats of one component's [ic 16][tile]
    constexpr int MPLANE = 16 * OB * NT;  // floats of one component's [oc][tile]
    __shared__ __attribute__((aligned(16))) float lds[2][16 * PLANE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int C = p.c, H = p.h, W = p.w, M = p.m, HW = H * W;
    const int tilesX = (W + 1) >> 1, tilesY = (H + 1) >> 1, T = tilesX * tilesY;
    const int ocbs = (M + 15) >> 4, cbs = (C + 15) >> 4;
    const int ob = blockIdx.x * OB + (wave >> 2);
    const bool transforms = wave < 4;  // the waves that transform patches (uniform)
    // thread role: tile tid % NT, channel (of a chunk, then of the outputs) tid / NT
    const int row = tid / NT, tl = tid % NT;
    const unsigned tg = blockIdx.y * (unsigned)NT + tl;  // n * T fits 31 bits (winograd_eligible)
    const unsigned imgb = blockIdx.y * (unsigned)NT / (unsigned)T;  // the workgroup's first image
    const unsigned img = tg / (unsigned)T, tr = tg - img * (unsigned)T;
    const int ty = (int)(tr / (unsigned)tilesX), tx = (int)tr - ty * tilesX;
    const bool tile_ok = img < (unsigned)p.n;
    // byte offsets of the patch rows at column 2 tx, from channel 0 of the
    // chunk in the workgroup's first image (the host keeps the images of one
    // workgroup within 31 bits)
    int off[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int yy = 2 * ty - 1 + i;
        off[i] = tile_ok && (unsigned)yy < (unsigned)H
                     ? ((((int)(img - imgb) * C + row) * H + yy) * W + 2 * tx) * 4
                     : kWinoNowhere;
    }
    const bool in0 = tx > 0, in2 = 2 * tx + 1 < W, in3 = 2 * tx + 2 < W;
    const long long xtotal = (long long)p.n * C * HW;

    struct Patch {
        float d[16];
    };
    auto load_patch = [&](Patch &q, int ch) {
        const int c0 = ch * 16;
        const long long at = ((long long)imgb * C + c0) * HW;
        const long long rest = c0 < C ? (xtotal - at) * 4 : 0;
        __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(x + (c0 < C ? at : 0)), (short)0, rest > kWinoNowhere - 64 ? kWinoNowhere - 64 : (int)rest,
            0x00020000);
        const bool ok = c0 + row < C;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int o = ok ? off[i] : kWinoNowhere;
            q.d[4 * i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, o - 4, 0, 0));
            const auto v = __builtin_amdgcn_raw_buffer_load_b96(rx, o, 0, 0);
#pragma unroll
            for (int e = 0; e < 3; e++) q.d[4 * i + 1 + e] = __uint_as_float(v[e]);
        }
    };
    // V = B^T d B (columns off the map zero), stored at [comp][row][tl]
    auto transform_store = [&](const Patch &q, float *vb) {
        float d[16], t[16];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            d[4 * i] = in0 ? q.d[4 * i] : 0.0f;
            d[4 * i + 1] = q.d[4 * i + 1];
            d[4 * i + 2] = in2 ? q.d[4 * i + 2] : 0.0f;
            d[4 * i + 3] = in3 ? q.d[4 * i + 3] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float d0 = d[j], d1 = d[4 + j], d2 = d[8 + j], d3 = d[12 + j];
            t[j] = d0 - d2;
            t[4 + j] = d1 + d2;
            t[8 + j] = d2 - d1;
            t[12 + j] = d1 - d3;
        }
        float *dst = vb + tid;  // row * NT + tl
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float e0 = t[i * 4], e1 = t[i * 4 + 1], e2 = t[i * 4 + 2], e3 = t[i * 4 + 3];
            dst[(i * 4) * PLANE] = e0 - e2;
            dst[(i * 4 + 1) * PLANE] = e1 + e2;
            dst[(i * 4 + 2) * PLANE] = e2 - e1;
            dst[(i * 4 + 3) * PLANE] = e1 - e3;
        }
    };
    // weight fragments of this wave's four components and output block; an
    // output block past the last has no descriptor and chunks past it lie
    // outside: zeros
    struct Weights {
        f32x4 u[4];
    };
    __amdgpu_buffer_rsrc_t ru[4];
#pragma unroll
    for (int q = 0; q < 4; q++)
        ru[q] = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(up + ((long long)(4 * (wave & 3) + q) * ocbs + (ob < ocbs ? ob : 0)) * cbs * 64), (short)0,
            ob < ocbs ? cbs * 1024 : 0, 0x00020000);
    auto load_u = [&](Weights &w, int ch) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(ru[q], lane * 16 + ch * 1024, 0, 0);
            w.u[q] = f32x4{__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3])};
        }
    };

    f32x4 acc[4];
#pragma unroll
    for (int q = 0; q < 4; q++) acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto multiply = [&](const Weights &w, const float *vs) {
        const float *vb = vs + 4 * (wave & 3) * PLANE + lane;  // B operand: V[k = 4 s + lane >> 4][tile lane & 15]
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                acc[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(w.u[q][s], vb[q * PLANE + 4 * s * NT], acc[q], 0, 0, 0);
    };
    Patch pa;
    Weights w0, w1;
    if (transforms) load_patch(pa, 0);
    load_u(w0, 0);
    if (transforms) {
        transform_store(pa, lds[0]);
        load_patch(pa, 1);
    }
    load_u(w1, 1);
    __syncthreads();
    int ch = 0;
    for (; ch + 2 < cbs; ch += 2) {
        // planes of chunk ch in buffer 0; pa and w1 hold chunk ch + 1
        multiply(w0, lds[0]);
        load_u(w0, ch + 2);
        if (transforms) {
            transform_store(pa, lds[1]);
            load_patch(pa, ch + 2);
        }
        __syncthreads();
        multiply(w1, lds[1]);
        load_u(w1, ch + 3);
        if (transforms) {
            transform_store(pa, lds[0]);
            load_patch(pa, ch + 3);
        }
        __syncthreads();
    }
    // the last one or two chunks, with nothing left to load or, after them, to
    // transform (a chunk too many, of zeros, cost 4 x 8 x 33 x 28 -> 168 6.9 us;
    // 6.0 so)
    multiply(w0, lds[0]);
    if (ch + 1 < cbs) {
        if (transforms) transform_store(pa, lds[1]);
        __syncthreads();
        multiply(w1, lds[1]);
    }
    __syncthreads();
    // accumulators -> [comp][oc][tile]; D[row 4g + r][col j]
    float *ms = lds[0];
    {
        float *d = ms + 4 * (wave & 3) * MPLANE + (16 * (wave >> 2) + 4 * (lane >> 4)) * NT + (lane & 15);
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int r = 0; r < 4; r++) d[q * MPLANE + r * NT] = acc[q][r];
    }
    // the outputs of this thread: two rows of two neighbours (8-byte accesses
    // at any 4-byte address), the residual on its way while the others arrive
    const int oc = blockIdx.x * 16 * OB + row;
    const int oy = 2 * ty, ox = 2 * tx;
    const bool live = tile_ok && oc < M;
    const long long base = live ? ((long long)img * M + oc) * HW + (long long)oy * W + ox : 0;
    const int row1 = oy + 1 < H ? W : 0;  // the second row, or the first again
    float rv[4] = {0.f, 0.f, 0.f, 0.f};
    if (res && live) {
        const float *src = res + base;
        if (in2) {
            const f32x2u a = *reinterpret_cast<const f32x2u *>(src), b = *reinterpret_cast<const f32x2u *>(src + row1);
            rv[0] = a[0], rv[1] = a[1], rv[2] = b[0], rv[3] = b[1];
        } else {
            rv[0] = src[0], rv[2] = src[row1];
        }
    }
    __syncthreads();
    if (!live) return;
    float m[16];
#pragma unroll
    for (int comp = 0; comp < 16; comp++) m[comp] = ms[comp * MPLANE + tid];
    float t[8];
#pragma unroll
    for (int j = 0; j < 4; j++) {  // A^T M
        const float m0 = m[j], m1 = m[4 + j], m2 = m[8 + j], m3 = m[12 + j];
        t[j] = m0 + m1 + m2;
        t[4 + j] = m1 - m2 - m3;
    }
    const float b = bias ? bias[oc] : 0.0f;
    float o[4];
    o[0] = t[0] + t[1] + t[2] + b;  // (A^T M) A, bias last
    o[1] = t[1] - t[2] - t[3] + b;
    o[2] = t[4] + t[5] + t[6] + b;
    o[3] = t[5] - t[6] - t[7] + b;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        o[e] = activate<ACT>(o[e]);
        if (res) o[e] = o[e] + rv[e];
    }
    float *dst = y + base;
    if (in2) {
        *reinterpret_cast<f32x2u *>(dst) = f32x2u{o[0], o[1]};
        if (row1) *reinterpret_cast<f32x2u *>(dst + row1) = f32x2u{o[2], o[3]};
    } else {
        dst[0] = o[0];
        if (row1) dst[row1] = o[2];
    }
}

inline osh_status winograd_pack(const osh_conv_params *p, const float *w, void *out, hipStream_t st) {
    const long long total = (long long)((p->m + 15) / 16) * 16 * ((p->c + 15) / 16) * 16;
    OSH_LAUNCH(wino_pack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, p->m, p->c, w,
                       static_cast<float *>(out));
    OSH_LAUNCH_CHECK("wino_pack_kernel");
    return OSH_OK;
}

}  // namespace osh
