// divmod_host.cpp -- TEST INFRASTRUCTURE: the long division of dec_device.h
// (divmod) built for the host CPU at several widths, so the CPU suite checks
// the digit estimate, its saturated form and the add-back against exact
// integer division before any GPU run.
#define __HIPCC_RTC__ 1
#define __device__
#define __forceinline__ inline
#define __global__
#include <cstdint>
#include <cstring>
static inline unsigned upd_alignbyte(unsigned hi, unsigned lo, unsigned s)
{
    return (unsigned)((((unsigned long long)hi << 32) | lo) >> (8 * (s & 3)));
}
#define __builtin_amdgcn_alignbyte(a, b, c) upd_alignbyte((a), (b), (c))
#define __builtin_nontemporal_load(p) (*(p))
static inline int __shfl_xor(int v, int, int) { return v; }
#include "dec_device.h"
using namespace updec;

template <int NX, int NB> static void run(const uint32_t* X, const uint32_t* B, int n, uint32_t* q, uint32_t* r)
{
    for (int i = 0; i < n; i++) {
        Mag<NX> x;
        Mag<NB> b, R;
        Mag<NX + 1> Q;
        memcpy(x.w, X + i * NX, sizeof x.w);
        memcpy(b.w, B + i * NB, sizeof b.w);
        divmod<NX, NB>(x, b, Q, R);
        memcpy(q + i * (NX + 1), Q.w, sizeof Q.w);
        memcpy(r + i * NB, R.w, sizeof R.w);
    }
}

extern "C" int divmod_run(int nx, int nb, const uint32_t* X, const uint32_t* B, int n, uint32_t* q, uint32_t* r)
{
#define CASE(x, b) \
    if (nx == x && nb == b) return run<x, b>(X, B, n, q, r), 0
    CASE(1, 1);
    CASE(3, 1);
    CASE(2, 2);
    CASE(5, 2);
    CASE(4, 3);
    CASE(2, 3);
    CASE(9, 5);
    CASE(12, 8);
    CASE(20, 17);
#undef CASE
    return 1;
}

extern "C" uint32_t recip2_run(uint32_t d1, uint32_t d0) { return recip_2word(d1, d0); }

// x / y with the reference's path quirks at S = 24, one row
extern "C" void ddiv_run(uint32_t a, uint32_t aneg, const uint32_t* b, uint32_t bneg, uint32_t* out)
{
    Dec<1> x;
    Dec<3> y;
    x.m.w[0] = a;
    x.neg = aneg;
    memcpy(y.m.w, b, sizeof y.m.w);
    y.neg = bneg;
    const Dec<4> r = ddiv<4, 1, 3, 24, 1>(x, y);
    memcpy(out, r.m.w, sizeof r.m.w);
    out[4] = r.neg;
}
