// vm_wide.h -- the interpreter's evaluation of wide programs and of those
// that spend their time in divisions (vm.h, runs_wide): one lane per row,
// values in memory.
//
// A program's register width is the worst case of its widest intermediate;
// the values themselves are mostly far shorter (a quotient has its scale's
// digits, a difference may vanish).  So every value here has the number of
// limbs that the longest of the wave's 64 rows needs, found when it is
// computed, and each operation runs over exactly those: loops with
// wave-uniform trip counts over limbs that lie in a workspace of the wave,
// [limb][lane], so that a limb of all rows is one 256-byte line.  Inner
// blocks are held in registers: 16 limbs of a product's shorter factor, and
// a division's divisor and running remainder up to 32 limbs.
//
// Compiled for the device by vm.hip and for the host (one lane) by the CPU
// tests.
#ifndef UPDEC_VM_WIDE_H
#define UPDEC_VM_WIDE_H
#include "dec_device.h"
#include "vm.h"

namespace updec_vm {
namespace wide {

using namespace updec;

#if defined(__HIP_DEVICE_COMPILE__)
constexpr u32 kLanes = 64;
UPD_DEV u32 lane_id() { return threadIdx.x & 63u; }
UPD_DEV u64 ballot(bool x) { return __builtin_amdgcn_ballot_w64(x); }
UPD_DEV u32 uni(u32 x) { return (u32)__builtin_amdgcn_readfirstlane((int)x); }
UPD_DEV u32 wave_max(u32 x)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const u32 y = (u32)__shfl_xor((int)x, o, 64);
        x = y > x ? y : x;
    }
    return uni(x);
}
// words that the kernel only reads: scalar loads
UPD_DEV u32 kword(const u32* p, u32 i) { return ((const __attribute__((address_space(4))) u32*)p)[i]; }
#else
constexpr u32 kLanes = 1;
UPD_DEV u32 lane_id() { return 0u; }
UPD_DEV u64 ballot(bool x) { return x ? 1u : 0u; }
UPD_DEV u32 uni(u32 x) { return x; }
UPD_DEV u32 wave_max(u32 x) { return x; }
UPD_DEV u32 kword(const u32* p, u32 i) { return p[i]; }
#endif

// Workspace and columns are addressed as device memory by type: their pointers
// come from memory, and through plain ones every access would be a flat one,
// which may go to LDS too and end in any order, so that each wait is for all
// that are in flight.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(1))) u8 gu8;
typedef __attribute__((address_space(1))) u32 gu32;
typedef __attribute__((address_space(1))) u32x4u gu32x4;
#else
typedef u8 gu8;
typedef u32 gu32;
typedef u32x4u gu32x4;
#endif

constexpr u32 kRow = 4u * kLanes;  // bytes of one limb of every lane

// A magnitude of n limbs (n the same for all lanes): limb i of this lane is
// the word at b + i * st + off.  In the workspace st is kRow and off the
// lane's; a constant has st = 4 and off = 0.
struct Src {
    const gu8* b;
    u32 st, off, n;
    UPD_DEV u32 at(u32 i) const { return *(const gu32*)(b + (i * st + off)); }
    UPD_DEV u32 get(u32 i) const { return i < n ? at(i) : 0u; }
    // limb i of this lane, i its own (any value): zero outside
    UPD_DEV u32 sel(i32 i) const
    {
        const u32 j = i < 0 ? 0u : ((u32)i < n ? (u32)i : n - 1u);
        const u32 x = at(j);
        return i >= 0 && (u32)i < n ? x : 0u;
    }
};

struct Dst {
    gu8* b;
    u32 off;
    UPD_DEV void put(u32 i, u32 x) const { *(gu32*)(b + (i * kRow + off)) = x; }
    UPD_DEV u32 at(u32 i) const { return *(const gu32*)(b + (i * kRow + off)); }
    UPD_DEV Src src(u32 n) const { return Src{b, kRow, off, n}; }
};

// Limbs are loaded a group ahead of their use.  A wave's loads and stores
// complete in the order they were issued, so a load that comes after a
// store waits for it too: the next group is asked for before this one's
// results are stored.  Sums and scalings take 16 limbs a group (8: one query of
// 1.2 M rows at 64 limbs, a product and three sums of DECIMAL(300,100), 1472
// instead of 1330 us; 16-limb programs of five divisions 426 instead of 452,
// for their values are short), and a group ends at the value's last limb at
// once: with a test for each of its limbs the two took 1520 and 561.
template <int G> struct Group {
    u32 w[G];
};
template <int G> UPD_DEV Group<G> fetch(const Src& s, u32 i)
{
    Group<G> g;
    if (i + (u32)G <= s.n) {
#pragma unroll
        for (int k = 0; k < G; k++) g.w[k] = s.at(i + (u32)k);
    } else {
#pragma unroll
        for (int k = 0; k < G; k++) g.w[k] = 0u;
#pragma unroll
        for (int k = 0; k < G; k++) {
            if (i + (u32)k >= s.n) break;
            g.w[k] = s.at(i + (u32)k);
        }
    }
    return g;
}

// ---------------------------------------------------------------- scaling

// d = s * first * 10^(9 (NP - 1)): NP one-word products in one pass over the
// limbs, each with its own carry; returns the limbs
template <int NP> UPD_DEV u32 mul_sweep(const Dst& d, const Src& s, u32 first)
{
    u32 c[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) c[p] = 0u;
    auto step = [&](u32 x) {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const u64 t = (u64)x * (p == 0 ? first : 1000000000u) + c[p];
            x = (u32)t;
            c[p] = (u32)(t >> 32);
        }
        return x;
    };
    constexpr int G = 16;
    Group<G> x = fetch<G>(s, 0u);
    u32 i = 0;
    for (; i < s.n; i += (u32)G) {
        const Group<G> y = fetch<G>(s, i + (u32)G);
#pragma unroll
        for (int k = 0; k < G; k++) {
            if (i + (u32)k >= s.n) break;
            d.put(i + (u32)k, step(x.w[k]));
        }
        x = y;
    }
    i = s.n;
    for (;;) {
        u32 any = 0;
#pragma unroll
        for (int p = 0; p < NP; p++) any |= c[p];
        if (!any_lane(any != 0u)) break;
        d.put(i++, step(0u));
    }
    return i;
}

// d = s * 10^e (d may be s); returns the limbs
UPD_DEV u32 mul_pow10(const Dst& d, Src s, u32 e)
{
    u32 passes = (e + 8u) / 9u;
    u32 first = e % 9u ? pow10_word(e % 9u) : 1000000000u;
    while (passes) {
        u32 n;
        if (passes >= 16u) {
            n = mul_sweep<16>(d, s, first);
            passes -= 16u;
        } else if (passes >= 12u) {
            n = mul_sweep<12>(d, s, first);
            passes -= 12u;
        } else if (passes >= 8u) {
            n = mul_sweep<8>(d, s, first);
            passes -= 8u;
        } else if (passes >= 4u) {
            n = mul_sweep<4>(d, s, first);
            passes -= 4u;
        } else if (passes >= 2u) {
            n = mul_sweep<2>(d, s, first);
            passes -= 2u;
        } else {
            n = mul_sweep<1>(d, s, first);
            passes -= 1u;
        }
        first = 1000000000u;
        s = d.src(n);
    }
    return s.n;
}

// d = floor(s / 10^e); returns the limbs
UPD_DEV u32 div_pow10(const Dst& d, Src s, u32 e)
{
    u32 top = 0;
    while (e) {
        const u32 k = e < 9u ? e : 9u;
        const u32 dv = pow10_word(k);
        const int sh = __builtin_clz(dv);
        const u32 dn = dv << sh, v = recip_word(dn);
        // two divisions a pass while there are two
        const bool two = e >= 18u;
        u32 r0 = 0, r1 = 0;
        top = 0;
        for (u32 i = s.n; i-- > 0u;) {
            u32 x = s.at(i), rr;
            u32 u1 = (r0 << sh) | (x >> ((32 - sh) & 31));
            x = div_2by1(u1, x << sh, dn, v, rr);
            r0 = rr >> sh;
            if (two) x = div_word_const<1000000000u>(r1, x);
            d.put(i, x);
            top = x && !top ? i + 1u : top;
        }
        top = wave_max(top);
        s = d.src(top);
        e -= two ? 18u : k;
    }
    return s.n;
}

// ---------------------------------------------------------------- sum and product

// d = a + b with signs (dadd's rules; d may be a or b); neg receives the
// result's sign, returns the limbs
UPD_DEV u32 add(const Dst& d, const Src& a, u32 aneg, const Src& b, u32 bneg, u32& neg)
{
    const bool same = aneg == bneg;
    const u32 m = same ? 0u : 0xffffffffu;
    u32 c = same ? 0u : 1u;
    u32 n = a.n > b.n ? a.n : b.n;
    u32 top = 0;
    constexpr int G = 16;
    Group<G> x = fetch<G>(a, 0u), y = fetch<G>(b, 0u);
    for (u32 i = 0; i < n; i += (u32)G) {
        const Group<G> x1 = fetch<G>(a, i + (u32)G), y1 = fetch<G>(b, i + (u32)G);
#pragma unroll
        for (int k = 0; k < G; k++) {
            if (i + (u32)k >= n) break;
            const u32 t = addc(x.w[k], y.w[k] ^ m, c);
            d.put(i + (u32)k, t);
            top = t ? i + (u32)k + 1u : top;
        }
        x = x1;
        y = y1;
    }
    // different signs and no carry: |a| < |b|, the difference is negated
    const bool flip = !same && c == 0u;
    if (any_lane(flip)) {
        const u32 fm = flip ? 0xffffffffu : 0u;
        u32 cc = flip ? 1u : 0u;
        const Src r = d.src(n);
        top = 0u;
        x = fetch<G>(r, 0u);
        for (u32 i = 0; i < n; i += (u32)G) {
            const Group<G> x1 = fetch<G>(r, i + (u32)G);
#pragma unroll
            for (int k = 0; k < G; k++) {
                if (i + (u32)k >= n) break;
                const u32 t = addc(x.w[k] ^ fm, 0u, cc);
                d.put(i + (u32)k, t);
                top = t ? i + (u32)k + 1u : top;
            }
            x = x1;
        }
    }
    neg = same ? aneg : (flip ? bneg : (top ? aneg : 0u));
    if (any_lane(same && c != 0u)) {
        d.put(n, same ? c : 0u);
        return n + 1u;
    }
    return wave_max(top);
}

// limbs i0 .. i0 + K - 1 of a (zero past its end) times b, added to d from
// limb i0 on (FIRST: d is empty); returns the last limb written
template <int K, bool FIRST> UPD_DEV u32 mul_block(const Dst& d, const Src& a, u32 i0, const Src& b)
{
    u32 A[K], w[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        A[k] = a.get(i0 + (u32)k);
        w[k] = 0u;
    }
    u32 rc = 0u, out = 0u;
    auto column = [&](u32 j, u32 bj, u32 r) {
        u32 hi = 0u, c = 0u;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const u64 t = (u64)A[k] * bj + hi;
            hi = (u32)(t >> 32);
            w[k] = addc(w[k], (u32)t, c);
        }
        out = FIRST ? w[0] : addc(w[0], r, rc);
        d.put(i0 + j, out);
#pragma unroll
        for (int k = 0; k + 1 < K; k++) w[k] = w[k + 1];
        w[K - 1] = hi + c;
    };
    constexpr int G = 4;
    // what the earlier blocks left at limbs i0 .. i0 + b.n - 1
    const Src old{d.b + i0 * kRow, kRow, d.off, FIRST ? 0u : b.n};
    Group<G> y = fetch<G>(b, 0u), r = fetch<G>(old, 0u);
    for (u32 j = 0; j < b.n; j += (u32)G) {
        const Group<G> y1 = fetch<G>(b, j + (u32)G), r1 = fetch<G>(old, j + (u32)G);
#pragma unroll
        for (int k = 0; k < G; k++)
            if (j + (u32)k < b.n) column(j + (u32)k, y.w[k], r.w[k]);
        y = y1;
        r = r1;
    }
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (i0 + (u32)k < a.n) {
            out = FIRST ? w[k] : addc(w[k], 0u, rc);
            d.put(i0 + b.n + (u32)k, out);
        }
    }
    return out;
}

template <int K> UPD_DEV u32 mul_blocks(const Dst& d, const Src& a, const Src& b)
{
    u32 out = mul_block<K, true>(d, a, 0u, b);
    for (u32 i = K; i < a.n; i += K) out = mul_block<K, false>(d, a, i, b);
    return out;
}

// d = a * b; returns the limbs
UPD_DEV u32 mul(const Dst& d, const Src& x, const Src& y)
{
    if (x.n == 0u || y.n == 0u) return 0u;
    const Src& a = x.n <= y.n ? x : y;
    const Src& b = x.n <= y.n ? y : x;
    const u32 last = a.n <= 4u ? mul_blocks<4>(d, a, b) : a.n <= 8u ? mul_blocks<8>(d, a, b) : mul_blocks<16>(d, a, b);
    return a.n + b.n - (any_lane(last != 0u) ? 0u : 1u);
}

// ---------------------------------------------------------------- quotient

// quotient digit, and what it leaves of the top two words, of the three
// words (u2, u1, u0) by (d1, d0): see divmod_digit.  r2: the third word of
// what is left when the top words are equal and the digit saturates.
UPD_DEV u32 digit3by2(u32 u2, u32 u1, u32 u0, u32 d1, u32 d0, u32 v, u64& r, u32& r2)
{
    const u64 D = ((u64)d1 << 32) | d0;
    const u64 qe = (u64)v * u2 + (((u64)u2 << 32) | u1);
    u32 q = (u32)(qe >> 32);
    r = ((((u64)u1 << 32) | u0) - D) - (u64)q * d0 - ((u64)(q * d1) << 32);
    q += 1u;
    if ((u32)(r >> 32) >= (u32)qe) {
        q -= 1u;
        r += D;
    }
    if (r >= D) {
        q += 1u;
        r -= D;
    }
    r2 = 0u;
    if (u2 == d1 && u1 == d0) {
        q = 0xffffffffu;
        r = D + u0;
        r2 = r < D ? 1u : 0u;
    }
    return q;
}

// q = floor(X / B) for divisors of up to NB limbs, held with the running
// remainder in registers: B is shifted (per lane) to fill NB limbs, and the
// limbs of the equally shifted X are taken in from the top, one quotient
// digit each.  X lies in q's rows: digit j is written when only limbs below
// j are still to be read.  bl: the lane's bit length of B (not 0).  Returns
// the limbs of q; rnd = 1 where twice the remainder is at least B; rtop: the
// shifted remainder's top limb.
template <int NB> UPD_DEV u32 div_reg(const Dst& q, const Src& X, const Src& B, u32 bl, u32& rnd, u32& rtop)
{
    const u32 k = 32u * NB - bl, bs = k & 31u;
    const i32 ws = (i32)(k >> 5);
    Mag<NB> V, win;
    {
        u32 lo = 0u;
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const u32 hi = B.sel(i - ws);
            V.w[i] = funnel_l(hi, lo, bs);
            lo = hi;
        }
    }
    const u32 d1 = V.w[NB - 1], d0 = V.w[NB - 2], v = recip_2word(d1, d0);
    // X 2^k has limbs 0 .. X.n + ws: above digit J its first NB - 1 limbs
    // are less than V, so the digits from J + 1 on are zero
    const i32 J = (i32)X.n + (i32)wave_max((u32)ws) + 1 - NB;
    i32 p = J < 0 ? 0 : J + 1;  // lowest limb of the first window
    u32 hi = X.sel(p + NB - 1 - ws);
#pragma unroll
    for (int i = NB - 1; i >= 0; i--) {
        const u32 lo = X.sel(p + i - 1 - ws);
        win.w[i] = funnel_l(hi, lo, bs);
        hi = lo;
    }
    u32 top = 0;
    u32 next = X.sel(J - 1 - ws);
    for (i32 j = J; j >= 0; j--) {
        const u32 u = funnel_l(hi, next, bs);
        hi = next;
        next = X.sel(j - 2 - ws);
        const u32 u2 = win.w[NB - 1], u1 = win.w[NB - 2], u0 = win.w[NB - 3];
        u32 qd = 0u;
        if (!any_lane(u2 != 0u || u1 >= d1)) {
#pragma unroll
            for (int i = NB - 1; i >= 1; i--) win.w[i] = win.w[i - 1];
            win.w[0] = u;
        } else {
            u64 r;
            u32 r2;
            qd = digit3by2(u2, u1, u0, d1, d0, v, r, r2);
            u32 cy = 0u, br = 0u, prev = u;
#pragma unroll
            for (int i = 0; i < NB - 2; i++) {
                const u64 t = (u64)qd * V.w[i] + cy;
                cy = (u32)(t >> 32);
                const u32 cur = win.w[i];
                win.w[i] = subb(prev, (u32)t, br);
                prev = cur;
            }
            win.w[NB - 2] = subb((u32)r, cy, br);
            win.w[NB - 1] = subb((u32)(r >> 32), 0u, br);
            const bool back = br > r2;  // rare: the digit was one too large
            if (any_lane(back)) {
                qd -= back ? 1u : 0u;
                const u32 mask = back ? 0xffffffffu : 0u;
                u32 c = 0u;
#pragma unroll
                for (int i = 0; i < NB; i++) win.w[i] = addc(win.w[i], V.w[i] & mask, c);
            }
        }
        q.put((u32)j, qd);
        top = qd && !top ? (u32)j + 1u : top;
    }
    Mag<NB> T;
    sub_to<NB>(T, V, win);
    rnd = ge(win, T) ? 1u : 0u;
    rtop = win.w[NB - 1];
    return wave_max(top);
}

// The same for a divisor of any length, divisor and dividend shifted in
// memory: U holds X on entry and has room for X.n + B.n + 2 limbs, V for B.n.
UPD_DEV u32 div_mem(const Dst& q, const Dst& U, u32 nx, const Src& B, u32 bl, const Dst& V, u32& rnd)
{
    const u32 nb = B.n;
    const u32 k = 32u * nb - bl, bs = k & 31u;
    const i32 ws = (i32)(k >> 5);
    {
        // from the top down: B may lie in V
        u32 hi = B.sel((i32)nb - 1 - ws);
        for (u32 i = nb; i-- > 0u;) {
            const u32 lo = B.sel((i32)i - 1 - ws);
            V.put(i, funnel_l(hi, lo, bs));
            hi = lo;
        }
    }
    const u32 d1 = V.at(nb - 1u), d0 = V.at(nb - 2u), v = recip_2word(d1, d0);
    const Src X = U.src(nx);
    const u32 wm = wave_max((u32)ws);
    const i32 J = (i32)nx + (i32)wm + 1 - (i32)nb;
    const u32 len = nx + wm + 2u > nb ? nx + wm + 2u : nb;
    // from the top down, each limb is written where nothing is read any more
    u32 hi = X.sel((i32)len - 1 - ws);
    for (u32 i = len; i-- > 0u;) {
        const u32 lo = X.sel((i32)i - 1 - ws);
        U.put(i, funnel_l(hi, lo, bs));
        hi = lo;
    }
    u32 top = 0;
    for (i32 j = J; j >= 0; j--) {
        const u32 base = (u32)j;
        const u32 u2 = U.at(base + nb), u1 = U.at(base + nb - 1u), u0 = U.at(base + nb - 2u);
        u32 qd = 0u;
        if (any_lane(u2 != 0u || u1 >= d1)) {
            u64 r;
            u32 r2;
            qd = digit3by2(u2, u1, u0, d1, d0, v, r, r2);
            u32 cy = 0u, br = 0u;
            constexpr int G = 8;
            const Src win{U.b + base * kRow, kRow, U.off, nb - 2u}, vs = V.src(nb - 2u);
            Group<G> x = fetch<G>(win, 0u), y = fetch<G>(vs, 0u);
            for (u32 i = 0; i < nb - 2u; i += (u32)G) {
                const Group<G> x1 = fetch<G>(win, i + (u32)G), y1 = fetch<G>(vs, i + (u32)G);
#pragma unroll
                for (int t = 0; t < G; t++) {
                    if (i + (u32)t < nb - 2u) {
                        const u64 p = (u64)qd * y.w[t] + cy;
                        cy = (u32)(p >> 32);
                        U.put(base + i + (u32)t, subb(x.w[t], (u32)p, br));
                    }
                }
                x = x1;
                y = y1;
            }
            U.put(base + nb - 2u, subb((u32)r, cy, br));
            U.put(base + nb - 1u, subb((u32)(r >> 32), 0u, br));
            U.put(base + nb, 0u);
            const bool back = br > r2;
            if (any_lane(back)) {
                qd -= back ? 1u : 0u;
                u32 c = 0u;
                for (u32 t = 0; t < nb; t++) U.put(base + t, addc(U.at(base + t), back ? V.at(t) : 0u, c));
            }
        }
        q.put(base, qd);
        top = qd && !top ? base + 1u : top;
    }
    u32 br = 0u, bit = 0u;
    for (u32 i = 0; i < nb; i++) {
        const u32 r = U.at(i);
        (void)subb((r << 1) | bit, V.at(i), br);
        bit = r >> 31;
    }
    rnd = bit != 0u || br == 0u ? 1u : 0u;
    return wave_max(top);
}

// the lane's bit length of s, from the top
UPD_DEV u32 bits_of(const Src& s)
{
    u32 bl = 0;
    for (u32 i = s.n; i-- > 0u;) {
        const u32 x = s.at(i);
        bl = !bl && x ? 32u * i + 32u - (u32)__builtin_clz(x) : bl;
        if (!any_lane(bl == 0u)) break;
    }
    return bl;
}

// Where ddiv's faithful rules differ from the exact quotient, by lane:
// q64 replaces it (own: the uint64 division, where the scaled dividend or
// twice the remainder passes 64 bits), it is one (one: the bisection on a
// dividend up to 64 bits shorter than the divisor), or a remainder with bit
// 31 set rounds down (half: 32-bit doubling, divisors of 32 bits).
struct Quirks {
    bool own, one, half;
    u64 q64;
};
UPD_DEV Quirks quirks(const Src& a, const Src& X, const Src& B, u32 bl, bool zero, u32 S)
{
    const u32 bla = bits_of(a), blx = bits_of(X);
    const bool in64 = !zero && bla + (u32)est_shift_bits((int)S) - 1u <= 64u && bl <= 64u;
    Quirks k;
    k.half = !in64 && bl == 32u;
    k.one = !in64 && bl > 32u && bla != 0u && blx < bl && bl - blx <= 64u;
    k.own = in64 && (blx > 64u || bl == 64u);
    k.q64 = 0u;
    if (any_lane(k.own)) {
        Mag<2> x, y, r;
        Mag<3> q;
        x.w[0] = a.get(0u);
        x.w[1] = a.get(1u);
        y.w[0] = k.own ? B.get(0u) : 1u;
        y.w[1] = k.own ? B.get(1u) : 0u;
        x = mul_p10_rt<2>(x, S);
        divmod<2, 2>(x, y, q, r);
        const u64 b64 = ((u64)y.w[1] << 32) | y.w[0], r64 = ((u64)r.w[1] << 32) | r.w[0];
        k.q64 = (((u64)q.w[1] << 32) | q.w[0]) + (r64 << 1 >= b64 ? 1u : 0u);
    }
    return k;
}

// q = round-half-up(|a| 10^S / |b|), x / 0 = |x| (ddiv's rules; faith: its
// faithful ones); q has room for the scaled dividend, U and V as div_mem
// says; returns the limbs
UPD_DEV u32 div(const Dst& q, const Src& a, const Src& b, u32 S, const Dst& U, const Dst& V, bool faith)
{
    // bit length of the lane's divisor, from the top
    u32 bl = 0, nb = 0;
    for (u32 i = b.n; i-- > 0u;) {
        const u32 x = b.at(i);
        if (!nb && any_lane(x != 0u)) nb = i + 1u;
        bl = !bl && x ? 32u * i + 32u - (u32)__builtin_clz(x) : bl;
        if (!any_lane(bl == 0u)) break;
    }
    const bool zero = bl == 0u, some = any_lane(zero);
    if (nb == 0u) nb = 1u;
    Src B = b;
    B.n = nb;
    const Dst X = nb <= 32u ? q : U;
    const u32 nx = mul_pow10(X, a, S);
    if (nx == 0u) return 0u;
    if (some) {
        // those lanes divide the unscaled dividend by one
        for (u32 i = 0; i < nx; i++) X.put(i, zero ? a.get(i) : X.at(i));
        for (u32 i = 0; i < nb; i++) V.put(i, zero ? (i == 0u ? 1u : 0u) : b.get(i));
        B = V.src(nb);
        bl = zero ? 1u : bl;
    }
    Quirks k{false, false, false, 0u};
    if (faith) k = quirks(a, X.src(nx), B, bl, zero, S);
    u32 rnd, n, rtop = 0u;
    if (nb <= 4u) n = div_reg<4>(q, X.src(nx), B, bl, rnd, rtop);
    else if (nb <= 8u) n = div_reg<8>(q, X.src(nx), B, bl, rnd, rtop);
    else if (nb <= 16u) n = div_reg<16>(q, X.src(nx), B, bl, rnd, rtop);
    else if (nb <= 32u) n = div_reg<32>(q, X.src(nx), B, bl, rnd, rtop);
    else n = div_mem(q, U, nx, B, bl, V, rnd);
    if (any_lane(k.own || k.one || k.half)) {
        // a divisor of 32 bits is shifted by whole limbs: rtop is the remainder
        if (k.half && rtop >> 31) rnd = 0u;
        if (k.own || k.one) rnd = 0u;
        const u32 lo = k.one ? 1u : (u32)k.q64, hi = k.one ? 0u : (u32)(k.q64 >> 32);
        const bool put = k.own || k.one;
        const u32 m = wave_max(put ? (hi ? 2u : lo ? 1u : 0u) : 0u);
        const u32 n1 = m > n ? m : n;
        for (u32 i = 0; i < n1; i++) {
            const u32 x = i < n ? q.at(i) : 0u;
            q.put(i, put ? (i == 0u ? lo : i == 1u ? hi : 0u) : x);
        }
        n = n1;
    }
    for (u32 i = 0; any_lane(rnd != 0u); i++) {
        const u32 x = i < n ? q.at(i) : 0u;
        q.put(i, addc(x, 0u, rnd));
        n = i + 1u > n ? i + 1u : n;
    }
    return n;
}

// ---------------------------------------------------------------- columns

// the compact row of B bytes into d; neg receives its sign, returns the limbs
UPD_DEV u32 load_column(const Dst& d, const gu8* col, usize row, u32 B, usize colbytes, u32& neg)
{
    const u32 nl = (B + 3u) / 4u;
    const usize off = row * (usize)B;
    const usize d0 = off >> 2;
    const u32 sh = (u32)(off & 3u);
    const gu32* p = (const gu32*)col + d0;
    const u32 tail = B & 3u ? (1u << (8u * (B & 3u))) - 1u : 0xffffffffu;
    const u32 sb = (8u * B - 1u) & 31u;
    u32 top = 0;
    neg = 0u;
    auto put = [&](u32 i, u32 x) {
        if (i + 1u == nl) {
            x &= tail;
            neg = (x >> sb) & 1u;
            x &= ~(1u << sb);
        }
        d.put(i, x);
        top = x ? i + 1u : top;
    };
    if (!any_lane((d0 + ((nl + 3u) & ~3u) + 1u) * 4u > colbytes)) {
        // sixteen bytes a load, four loads ahead
        constexpr u32 N = 16u;
        u32 w[2u * N];
        auto ask = [&](u32 g, u32* to) {
#pragma unroll
            for (u32 t = 0; t < N; t += 4u)
                if (g + t < nl) {
                    const u32x4u x = *(const gu32x4*)(p + g + t);
#pragma unroll
                    for (u32 j = 0; j < 4u; j++) to[t + j] = x[j];
                }
        };
        const u32 past = p[nl];
        ask(0u, w);
        for (u32 g = 0; g < nl; g += N) {
            ask(g + N, w + N);
#pragma unroll
            for (u32 t = 0; t < N; t++) {
                if (g + t >= nl) break;
                put(g + t, __builtin_amdgcn_alignbyte(g + t + 1u < ((nl + 3u) & ~3u) ? w[t + 1u] : past, w[t], sh));
            }
#pragma unroll
            for (u32 t = 0; t < N; t++) w[t] = w[t + N];
        }
    } else {
        for (u32 i = 0; i < nl; i++) {
            u32 x = 0;
            for (u32 t = 0; t < 4u; t++)
                if (4u * i + t < B) x |= (u32)col[off + 4u * i + t] << (8u * t);
            put(i, x);
        }
    }
    return wave_max(top);
}

// ---------------------------------------------------------------- programs

// where the values live: columns are slots 0 .. 7, results the others
struct Slots {
    u32 row[kSlots];
    u32 n[kSlots];
    u64 neg[kSlots];   // bit l: lane l's sign
};

// operand word: slot or constant | constant? << 8 | shift << 16
UPD_DEV Src operand(u32 ow, const gu8* ws, const Slots* sl, const u32* cst, u32 W, u32 off, u32& neg)
{
    const u32 idx = ow & 0xffu;
    if (ow & 0x100u) {
        const u32* c = cst + idx * (W + 1u);
        const u32 h = kword(c, 0u);
        neg = h & 1u;
        return Src{(const gu8*)(c + 1), 4u, 0u, h >> 8};
    }
    neg = bit64(sl->neg[idx], lane_id());
    return Src{ws + (usize)uni(sl->row[idx]) * kRow, kRow, off, uni(sl->n[idx])};
}

// the program for this wave's rows (`row`: the lane's); neg receives the
// result's sign, returns the result
UPD_DEV Src eval(const Query* q, const u32* prog, const u32* cst, u32 W, gu8* ws, Slots* sl, usize row, u32& neg)
{
    const u32 off = 4u * lane_id();
    auto at = [&](u32 r) { return Dst{ws + (usize)r * kRow, off}; };
    const u32 cols = kword(prog, kHeadCols);
    for (u32 c = 0; c < (u32)kMaxCols; c++) {
        if (!((cols >> c) & 1u)) continue;
        const u32 r = kword(prog, kHeadCol + c);
        const u32 B = q->colbytes[c];
        u32 s;
        const u32 n = load_column(at(r), (const gu8*)q->col[c], row, B, (usize)q->rows * B, s);
        sl->row[c] = r;
        sl->n[c] = n;
        sl->neg[c] = ballot(s != 0u);
    }
    const Dst U = at(kword(prog, kHeadU)), V = at(kword(prog, kHeadV));
    Src res{ws, kRow, off, 0u};
    const u32 nins = q->nins;
    for (u32 pc = 0; pc < nins; pc++) {
        const u32* ip = prog + kHead + kIns * pc;
        const u32 w0 = kword(ip, 0u), w1 = kword(ip, 1u), w2 = kword(ip, 2u);
        const u32 op = w0 & 0xfu, slot = (w0 >> 4) & 0xffu, r = w0 >> 12;
        const Dst d = at(r);
        u32 an, bn = 0u;
        Src a = operand(w1, ws, sl, cst, W, off, an);
        const u32 sa = w1 >> 16, arg = w2 >> 16;
        u32 n;
        neg = an;
        if (op == OP_MOV || op == OP_NEG) {
            for (u32 i = 0; i < a.n; i++) d.put(i, a.at(i));
            n = a.n;
            neg ^= op == OP_NEG ? 1u : 0u;
        } else if (op == OP_UP || op == OP_DOWN) {
            if (arg == 0u) {
                for (u32 i = 0; i < a.n; i++) d.put(i, a.at(i));
                n = a.n;
            } else {
                n = op == OP_UP ? mul_pow10(d, a, arg) : div_pow10(d, a, arg);
            }
        } else {
            Src b = operand(w2, ws, sl, cst, W, off, bn);
            if (op == OP_ADD || op == OP_SUB) {
                // at most one operand is aligned, in the result's rows
                if (sa) a = d.src(mul_pow10(d, a, sa));
                else if (arg) b = d.src(mul_pow10(d, b, arg));
                n = add(d, a, an, b, bn ^ (op == OP_SUB ? 1u : 0u), neg);
            } else if (op == OP_MUL) {
                n = mul(d, a, b);
                neg = an ^ bn;
            } else {
                // 0 / x = +0
                u32 any = 0;
                for (u32 i = 0; i < a.n; i++) any |= a.at(i);
                n = div(d, a, b, sa, U, V, q->faithful != 0u);
                neg = any ? an ^ bn : 0u;
            }
        }
        sl->row[slot] = r;
        sl->n[slot] = n;
        sl->neg[slot] = ballot(neg != 0u);
        res = d.src(n);
    }
    return res;
}

// pos or neg += the row's materialized value (stored_rt's rules at outB
// bytes): magnitudes by sign, so that carries end where they end
UPD_DEV void accumulate(const Src& v, u32 neg, bool active, u32 outB, const Dst& pos, const Dst& negd)
{
    const u32 topbit = 8u * outB - 1u, tl = topbit >> 5, tb = topbit & 31u;
    u32 n = v.n;
    u32 last = 0;
    const bool cut = n > tl;
    if (cut) {
        last = v.at(tl);
        neg |= (last >> tb) & 1u;
        last &= (1u << tb) - 1u;
        n = tl;
    }
    const u32 keep = active ? 0xffffffffu : 0u;
    // the two accumulators lie in one workspace: the lane's sign picks its own
    const Dst acc{pos.b, pos.off + (neg ? (u32)(negd.b - pos.b) : 0u)};
    u32 c = 0u;
    constexpr int G = 16;
    Src vs = v;
    vs.n = n;
    const Src old = acc.src(n);
    Group<G> x = fetch<G>(vs, 0u), y = fetch<G>(old, 0u);
    for (u32 i = 0; i < n; i += (u32)G) {
        const Group<G> x1 = fetch<G>(vs, i + (u32)G), y1 = fetch<G>(old, i + (u32)G);
#pragma unroll
        for (int k = 0; k < G; k++) {
            if (i + (u32)k >= n) break;
            acc.put(i + (u32)k, addc(y.w[k], x.w[k] & keep, c));
        }
        x = x1;
        y = y1;
    }
    u32 i = n;
    if (cut) {
        acc.put(i, addc(acc.at(i), last & keep, c));
        i++;
    }
    for (; any_lane(c != 0u); i++) acc.put(i, addc(acc.at(i), 0u, c));
}

}  // namespace wide
}  // namespace updec_vm
#endif
