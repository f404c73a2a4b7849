// osh_conv_gen.h -- convolutions no other kernel takes (any kernel size,
// stride, dilation, pads, groups; 3x3 with C % 16 != 0), as an implicit GEMM
// on v_mfma_f32_16x16x4f32 over an input patch in LDS.
//
//   y[m, pixel] = act( bias[m] + sum_k W[m, k] * patch[k, pixel] ) (+ res)
//
// k = ic * KH * KW + ky * KW + kx ascending: the reference's im2col chain
// (ConvKernels.cs:554-563), and the MFMA adds its four lane-group products one
// after another like fmaf, so every output is that chain from the bias, bit
// for bit.
//
// Structure.  A workgroup (4 waves) owns a tile of TH x TW output pixels (TW a
// power of two) and WM 16-channel output blocks: WM waves along the channels,
// 4 / WM along the pixels, each wave BV blocks of 16 pixels.  Per chunk of CC
// input channels the receptive field of the whole tile goes to LDS, zeros where
// it leaves the map (the padding terms of the im2col matrix); a gather straight
// from memory reads every input value once per tap that covers it and pays two
// integer divisions for each (4 x 3 x 224 x 224 -> 64, 7x7 stride 2: 37 us).
// The patch is copied in flat order, at most NE values a thread, whose places
// in the map are found once; a chunk's loads go out a chunk ahead and are
// written to the second of two buffers.  A table in LDS holds the patch offset
// of each k, so a B operand is one ds_read_b32 at (the lane's pixel) + (the
// k's offset), the table four k-steps a ds_read_b128.  Weights are packed so
// that 16 bytes give a lane its A operands of four k-steps, read three such
// groups ahead; the reads of a group are pinned between the MFMAs of the one
// before (left alone the compiler sinks each to just before its use).
//
// Measured: the 7x7 stem above 19.6 us (48 TFLOP/s; the loop 12 us of it, whose
// 160 MFMAs a wave on CUs with four workgroups take 8.5, the rest the first
// loads and 12.8 MB of output, which the workgroups reach together); 200 x 40 x
// 40 -> 64 3x3 stride 2 137 -> 21.9; 512 x 14 x 14 -> 512 5x5 1628 -> 109.  Without
// the operand reads the loop takes the same time.
//
// k past the last: W is -0 and the patch value +0 (a plane of zeros behind the
// channels), and their product -0 leaves every accumulator as it is.
#pragma once

#include "osh_common.h"

namespace osh {

struct GenConvArgs {
    osh_conv_params p;
    const float *x;
    const float *w;  // gen_conv_pack's layout
    const float *bias, *res;
    float *y;
    int cc, chunks;        // channels a chunk, chunks
    int planes;            // planes staged (cc, or cc + 1 with the plane of zeros)
    int ph, pw;            // patch rows and columns (odd: stride-2 reads of two rows meet in no bank)
    int twl;               // log2 of the tile's columns
    int th;                // the tile's rows
    int tiles_x, tiles_y;
    int kgc, kgt;          // groups of 16 k: a chunk's, all
    unsigned rplane, rpw, rkhw, rkw;  // gen_recip of ph * pw, pw, kh * kw, kw
};

// ceil(2^32 / d): e / d = the high word of e * gen_recip(d) for e < 2^16, 1 < d <=
// 2^16 (a division per patch value and table entry costs more than the entry);
// 0 stands for d = 1.
inline unsigned gen_recip(unsigned d) { return d == 1 ? 0u : (unsigned)(((1ULL << 32) + d - 1) / d); }
__device__ __forceinline__ int gen_div(int e, unsigned recip) {
    return recip ? (int)__umulhi((unsigned)e, recip) : e;
}

constexpr int kGenLdsBytes = 60 * 1024;

// [group][ceil(opg / 16)][kgt][64 lanes][4]: lane (j, g) holds W[16 mb + j][16
// kb + 4 s + g] in slot s; k past the last -0, rows past the last 0.
inline size_t gen_conv_packed_bytes(const osh_conv_params *p) {
    const int opg = p->m / p->group;
    const long long K = (long long)(p->c / p->group) * p->kh * p->kw;
    return (size_t)p->group * ((opg + 15) / 16) * ((K + 15) / 16) * 256 * sizeof(float);
}

static __global__ void gen_conv_pack_kernel(int opg, int K, int mbs, int kgt, long long total, const float *__restrict__ w,
                                     float *__restrict__ out) {
    const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int s = (int)(idx & 3), lane = (int)((idx >> 2) & 63);
    long long r = idx >> 8;
    const int kb = (int)(r % kgt);
    r /= kgt;
    const int mb = (int)(r % mbs), g = (int)(r / mbs);
    const int m = 16 * mb + (lane & 15), k = 16 * kb + 4 * s + (lane >> 4);
    float v = k < K ? 0.0f : -0.0f;
    if (m < opg && k < K) v = w[((long long)g * opg + m) * K + k];
    out[idx] = v;
}

template <int WM, int BV, int NE, int ACT>
__global__ __launch_bounds__(256) void gen_conv_kernel(GenConvArgs a) {
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    const osh_conv_params &p = a.p;
    int *tab = reinterpret_cast<int *>(lds_raw);             // [kgc][g 4][s 4] byte offsets into the patch
    float *patch = reinterpret_cast<float *>(tab + a.kgc * 16);  // [2][256 NE], flat [planes][ph][pw]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g4 = lane >> 4;
    const int wm = wave % WM, wn = wave / WM;
    const int grp = blockIdx.z, cpg = p.c / p.group, opg = p.m / p.group;
    const int mb = blockIdx.y * WM + wm, mbs = (opg + 15) / 16;
    unsigned t = blockIdx.x;
    const int txi = (int)(t % (unsigned)a.tiles_x);
    t /= (unsigned)a.tiles_x;
    const int tyi = (int)(t % (unsigned)a.tiles_y), n = (int)(t / (unsigned)a.tiles_y);
    const int tw = 1 << a.twl;
    const int oy0 = tyi * a.th, ox0 = txi * tw;
    const int iy0 = oy0 * p.sh - p.pt, ix0 = ox0 * p.sw - p.pl;
    const int khw = p.kh * p.kw, HW = p.h * p.w, plane = a.ph * a.pw;

    // A: this wave's output block (no descriptor past the last), group kb at kb * 1 KB
    const bool mlive = mb < mbs;
    __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.w + (((long long)grp * mbs + (mlive ? mb : 0)) * a.kgt) * 256), (short)0, mlive ? a.kgt * 1024 : 0,
        0x00020000);
    auto load_a = [&](int kb) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(ra, lane * 16 + kb * 1024, 0, 0);
        return f32x4{__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3])};
    };
    f32x4 av[4];
#pragma unroll
    for (int i = 0; i < 3; i++) av[i] = load_a(i);

    // accumulators start at the bias
    f32x4 acc[BV];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int m = 16 * mb + 4 * g4 + r;
        const float b = a.bias && m < opg ? a.bias[grp * opg + m] : 0.f;
#pragma unroll
        for (int v = 0; v < BV; v++) acc[v][r] = b;
    }
    // the table: two divisions a k, once per workgroup
    for (int e = tid; e < a.kgc * 16; e += 256) {
        const int k = (e >> 4) * 16 + 4 * (e & 3) + ((e >> 2) & 3);
        int off = a.cc * plane;  // the plane of zeros
        if (k < a.cc * khw) {
            const int ic = gen_div(k, a.rkhw), rem = k - ic * khw, ky = gen_div(rem, a.rkw), kx = rem - ky * p.kw;
            off = ic * plane + ky * p.dh * a.pw + kx * p.dw;
        }
        tab[e] = off * 4;
    }
    // this lane's pixels: byte offset of their first tap
    int pb[BV];
#pragma unroll
    for (int v = 0; v < BV; v++) {
        const int px = (wn * BV + v) * 16 + j;
        pb[v] = ((px >> a.twl) * p.sh * a.pw + (px & (tw - 1)) * p.sw) * 4;
    }
    // this thread's patch values e = tid + 256 i: byte offsets from the chunk's
    // first channel (outside the map: past every descriptor, which reads zero,
    // as do channels past the last)
    int goff[NE];
    {
        int c = gen_div(tid, a.rplane), q = tid - c * plane, r = gen_div(q, a.rpw), col = q - r * a.pw;
        const int sc = gen_div(256, a.rplane), sq = 256 - sc * plane, sr = gen_div(sq, a.rpw), scol = sq - sr * a.pw;
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int iy = iy0 + r, ix = ix0 + col;
            const bool ok = (unsigned)iy < (unsigned)p.h && (unsigned)ix < (unsigned)p.w && c < a.cc;
            goff[i] = ok ? (c * HW + iy * p.w + ix) * 4 : -1;
            col += scol;
            r += sr;
            c += sc;
            if (col >= a.pw) col -= a.pw, r++;
            if (r >= a.ph) r -= a.ph, c++;
        }
    }
    float xv[NE];
    auto load_x = [&](int ch) {
        const int c0 = ch * a.cc, left = cpg - c0;
        const int live = left < 0 ? 0 : (left < a.cc ? left : a.cc);
        __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(a.x + ((long long)n * p.c + grp * cpg + (live ? c0 : 0)) * HW), (short)0, live * HW * 4,
            0x00020000);
#pragma unroll
        for (int i = 0; i < NE; i++) xv[i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, goff[i], 0, 0));
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NE; i++) patch[buf * 256 * NE + tid + 256 * i] = xv[i];
    };
    struct BGroup {
        float v[4][BV];
    };
    load_x(0);
    store_x(0);
    load_x(1);
    __syncthreads();
    for (int ch = 0; ch < a.chunks; ch++) {
        const char *pbytes = reinterpret_cast<const char *>(patch + (ch & 1) * 256 * NE);
        // groups of 16 k: offsets two groups ahead, B one, A three
        const int kb0 = ch * a.kgc;
        const int kgc = ch + 1 < a.chunks ? a.kgc : a.kgt - kb0;
        auto read_tab = [&](int kb) {
            return *reinterpret_cast<const i32x4 *>(tab + (kb < a.kgc ? kb : a.kgc - 1) * 16 + 4 * g4);
        };
        auto read_b = [&](BGroup &b, const i32x4 &o) {
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int v = 0; v < BV; v++) b.v[s][v] = *reinterpret_cast<const float *>(pbytes + (o[s] + pb[v]));
        };
        auto mul = [&](const f32x4 &w, const BGroup &b) {
#pragma unroll
            for (int s = 0; s < 4; s++)
#pragma unroll
                for (int v = 0; v < BV; v++)
                    acc[v] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[s], b.v[s][v], acc[v], 0, 0, 0);
        };
        BGroup b0, b1;
        i32x4 o0 = read_tab(0), o1 = read_tab(1);
        read_b(b0, o0);
        int kb = 0;
        for (; kb + 4 <= kgc; kb += 4) {
            // av[u] holds group kb + u, b0 / b1 the B of the even / odd ones
#define OSH_GEN_STEP(U, BC, BN, OC, ON)                              \
    __builtin_amdgcn_sched_barrier(0);                               \
    OC = read_tab(kb + U + 2);                                       \
    read_b(BN, ON);                                                  \
    av[(U + 3) & 3] = load_a(kb0 + kb + U + 3);                      \
    mul(av[U], BC);                                                  \
    _Pragma("unroll") for (int i = 0; i < 4 * BV; i++) {             \
        __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);           \
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);           \
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);           \
    }
            OSH_GEN_STEP(0, b0, b1, o0, o1)
            OSH_GEN_STEP(1, b1, b0, o1, o0)
            OSH_GEN_STEP(2, b0, b1, o0, o1)
            OSH_GEN_STEP(3, b1, b0, o1, o0)
#undef OSH_GEN_STEP
            __builtin_amdgcn_sched_barrier(0);
        }
        // up to three groups more: av[0 .. 2] hold them
        if (kb < kgc) {
            read_b(b1, o1);
            mul(av[0], b0);
            if (kb + 1 < kgc) {
                o0 = read_tab(kb + 2);
                mul(av[1], b1);
                if (kb + 2 < kgc) {
                    read_b(b0, o0);
                    mul(av[2], b0);
                }
            }
        }
        if (ch + 1 < a.chunks) {
            if (kgc & 3) {
#pragma unroll
                for (int i = 0; i < 3; i++) av[i] = load_a(kb0 + kgc + i);
            }
            store_x((ch + 1) & 1);
            load_x(ch + 2);
            __syncthreads();
        }
    }
    // epilogue: acc[v][r] is row 4 g + r, pixel j of block v
    const long long OHW = (long long)p.oh * p.ow;
#pragma unroll
    for (int v = 0; v < BV; v++) {
        const int px = (wn * BV + v) * 16 + j;
        const int oy = oy0 + (px >> a.twl), ox = ox0 + (px & (tw - 1));
        if (oy >= p.oh || ox >= p.ow) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int m = 16 * mb + 4 * g4 + r;
            if (m < opg) {
                const long long at = ((long long)n * p.m + grp * opg + m) * OHW + (long long)oy * p.ow + ox;
                float o = activate<ACT>(acc[v][r]);
                if (a.res) o += a.res[at];
                a.y[at] = o;
            }
        }
    }
}

constexpr int kGenMaxNE = 24;  // patch values a thread

// The tile for a conv: columns, rows, channels a chunk, patch values a thread;
// false when no patch fits (or a chunk's bytes pass a 31-bit offset).
inline bool gen_conv_plan(const osh_conv_params *p, int wm, int bv, GenConvArgs *a, int *ne) {
    const int cpg = p->c / p->group, khw = p->kh * p->kw;
    if ((long long)cpg * khw > (1 << 22) || khw > 1024) return false;
    const int wn = 4 / wm;
    int twl = 4;
    while (twl > 0 && (1 << (twl - 1)) >= p->ow) twl--;
    const int px = 16 * bv * wn, tw = 1 << twl, th = px / tw;
    const long long ph = (long long)(th - 1) * p->sh + (long long)(p->kh - 1) * p->dh + 1;
    const long long pw = ((long long)(tw - 1) * p->sw + (long long)(p->kw - 1) * p->dw + 1) | 1;
    if (ph > 4096 || pw > 4096) return false;
    const long long plane = ph * pw;
    const int K = cpg * khw;
    // a chunk is whole groups of 16 k (cc * khw a multiple of 16) or all
    // channels, with a plane of zeros behind them for the k past the last
    int unit = 16;
    while (unit > 1 && (unit / 2) * khw % 16 == 0) unit /= 2;
    auto lds = [&](long long cc, int n) { return (cc * khw + 15) / 16 * 64 + 2LL * 256 * n * 4; };
    auto values = [&](long long planes) { return (int)((planes * plane + 255) / 256); };
    int cc = cpg, planes = cpg + (K % 16 != 0), n = planes * plane > 256 * kGenMaxNE ? kGenMaxNE + 1 : values(planes);
    if (n > 8 && unit < cpg) {  // as many channels as fit, so that a chunk's work covers the next one's loads
        const long long fit = 256LL * kGenMaxNE / plane / unit * unit;
        if (fit >= unit) {
            cc = (int)(fit < cpg ? fit : (cpg + unit - 1) / unit * unit);
            planes = cc;
            n = values(planes);
        }
    }
    if (n > kGenMaxNE) return false;
    n = n <= 8 ? 8 : (n <= 16 ? 16 : 24);
    if (lds(cc, n) > kGenLdsBytes || (long long)cc * p->h * p->w * 4 >= (1LL << 31) - 64) return false;
    a->cc = cc;
    a->chunks = (cpg + cc - 1) / cc;
    a->planes = planes;
    a->ph = (int)ph;
    a->pw = (int)pw;
    a->twl = twl;
    a->th = th;
    a->tiles_x = (p->ow + tw - 1) / tw;
    a->tiles_y = (p->oh + th - 1) / th;
    a->kgc = (cc * khw + 15) / 16;
    a->kgt = (K + 15) / 16;
    a->rplane = gen_recip((unsigned)plane);
    a->rpw = gen_recip((unsigned)pw);
    a->rkhw = gen_recip((unsigned)khw);
    a->rkw = gen_recip((unsigned)p->kw);
    *ne = n;
    return true;
}

inline bool gen_conv_eligible(const osh_conv_params *p) {
    GenConvArgs a;
    int ne;
    return gen_conv_plan(p, 4, 1, &a, &ne);
}

inline osh_status gen_conv_pack(const osh_conv_params *p, const float *w, void *out, hipStream_t st) {
    const int opg = p->m / p->group, K = p->c / p->group * p->kh * p->kw;
    const long long total = (long long)(gen_conv_packed_bytes(p) / sizeof(float));
    OSH_LAUNCH(gen_conv_pack_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, opg, K, (opg + 15) / 16,
               (K + 15) / 16, total, w, static_cast<float *>(out));
    OSH_LAUNCH_CHECK("gen_conv_pack_kernel");
    return OSH_OK;
}

osh_status gen_conv_launch(const osh_conv_params *p, const float *x, const float *w, const float *bias,
                           const float *res, int act, float *y, hipStream_t st);

}  // namespace osh
