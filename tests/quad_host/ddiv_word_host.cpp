// ddiv_word_host.cpp -- TEST INFRASTRUCTURE: the faithful division of
// dec_device.h by one-word divisors, built for the host CPU, so the CPU suite
// checks its shortcuts against the reference's rules before any GPU run.
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

// a: two words a row (WA = 1 reads the low one); out: three words and the sign
template <int WA, int S, int LIT> static void run(const uint32_t* A, const uint32_t* B, const uint32_t* neg, int n, uint32_t* out)
{
    for (int i = 0; i < n; i++) {
        Dec<WA> a;
        Dec<1> b;
        for (int w = 0; w < WA; w++) a.m.w[w] = A[2 * i + w];
        b.m.w[0] = B[i];
        a.neg = neg[2 * i];
        b.neg = neg[2 * i + 1];
        const Dec<3> r = ddiv<3, WA, 1, S, 1, LIT>(a, b);
        memcpy(out + 4 * i, r.m.w, sizeof r.m.w);
        out[4 * i + 3] = r.neg;
    }
}

extern "C" int ddiv_word_run(int wa, int s, const uint32_t* A, const uint32_t* B, const uint32_t* neg, int n, uint32_t* out)
{
#define CASE(S_) \
    if (s == S_) return wa == 1 ? run<1, S_, 0>(A, B, neg, n, out) : run<2, S_, 1>(A, B, neg, n, out), 0
    CASE(4);
    CASE(5);
    CASE(6);
    CASE(7);
    CASE(8);
    CASE(9);
    CASE(10);
#undef CASE
    return 1;
}
