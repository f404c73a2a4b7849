// osh_conv_gen.hip -- launches of the general conv kernel (osh_conv_gen.h).
#include "osh_conv_gen.h"

namespace osh {

template <int WM, int BV>
static osh_status gen_launch(const GenConvArgs &a, int ne, int act, hipStream_t st) {
    const osh_conv_params &p = a.p;
    const int opg = p.m / p.group, mbs = (opg + 15) / 16;
    const long long tiles = (long long)a.tiles_x * a.tiles_y * p.n;
    if (tiles > 0x7fffffffLL) return fail(OSH_E_UNSUPPORTED, "Conv: grid too large");
    const dim3 grid((unsigned)tiles, (unsigned)((mbs + WM - 1) / WM), (unsigned)p.group);
    const size_t lds = (size_t)a.kgc * 64 + (size_t)2 * 256 * ne * 4;
#define OSH_GEN_NE(NE) \
    OSH_DISPATCH_ACT(act, ACT, OSH_LAUNCH((gen_conv_kernel<WM, BV, NE, ACT>), grid, dim3(256), lds, st, a))
    if (ne == 8) {
        OSH_GEN_NE(8);
    } else if (ne == 16) {
        OSH_GEN_NE(16);
    } else {
        OSH_GEN_NE(24);
    }
#undef OSH_GEN_NE
    OSH_LAUNCH_CHECK("gen_conv_kernel");
    return OSH_OK;
}

osh_status gen_conv_launch(const osh_conv_params *p, const float *x, const float *w, const float *bias,
                           const float *res, int act, float *y, hipStream_t st) {
    const int mbs = (p->m / p->group + 15) / 16;
    GenConvArgs a{};
    int ne = 0, bv = 0;
    const long long cus = device_cus();
    auto plan = [&](int wm) {
        return gen_conv_plan(p, wm, bv, &a, &ne)
                   ? (long long)a.tiles_x * a.tiles_y * p->n * ((mbs + wm - 1) / wm) * p->group
                   : 0;
    };
    // Waves along the channels: all four share a patch, but the ones past the
    // last block idle.  Three blocks of a large conv go one after another over
    // wider tiles instead: 2 x 88 x 90 x 90 -> 48 (12.8e6 pixels x k) 34.1 -> 27.8
    // us; 120 x 80 x 80 -> 40 (6.9e6) 19.9 against 20.8, 8 x 3 x 231 x 152 -> 48 5x5
    // stride 2 (5.3e6) 18.1 against 20.0.  A last workgroup of one block is spared
    // where the grid is large: 2 x 40 x 80 x 80 -> 144 29.9 -> 25.1 (24 x 100 x 100
    // -> 80, a small one, 8.0 against 9.3).
    int wm = mbs >= 3 ? 4 : mbs;
    bv = 4;
    const double terms = (double)p->n * p->oh * p->ow * (p->c / p->group) * p->kh * p->kw;
    if (mbs == 3 && terms >= 10e6) wm = 1;
    else if (mbs > 4 && mbs % 4 == 1 && plan(4) >= 2 * cus) wm = 2;
    // The largest tile that still gives three workgroups for every two CUs:
    // 200 x 40 x 40 -> 64 stride 2 takes 61, 36, 22 us with 4, 2, 1 blocks of
    // pixels a wave, 4 x 3 x 300 x 300 -> 48 16.2, 17.7, 23.8.
    while (bv > 1 && plan(wm) < 3 * cus / 2) bv /= 2;
    if (!plan(wm)) {
        wm = 4, bv = 1;  // the plan eligibility asks for
        if (!plan(wm)) return fail(OSH_E_UNSUPPORTED, "Conv: no patch fits");
    }
    a.p = *p;
    a.x = x;
    a.w = w;
    a.bias = bias;
    a.res = res;
    a.y = y;
#define OSH_GEN(WM)                                                  \
    do {                                                             \
        if (bv == 4) return gen_launch<WM, 4>(a, ne, act, st);       \
        if (bv == 2) return gen_launch<WM, 2>(a, ne, act, st);       \
        return gen_launch<WM, 1>(a, ne, act, st);                    \
    } while (0)
    if (wm == 4) OSH_GEN(4);
    if (wm == 2) OSH_GEN(2);
    OSH_GEN(1);
#undef OSH_GEN
}

}  // namespace osh
