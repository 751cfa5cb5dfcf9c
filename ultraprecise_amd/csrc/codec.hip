// codec.hip -- the compact codec at the edges of the path: bulk ingest of
// decimal text into compact columns, and bulk output formatting of compact
// columns (include/updec.h, "codec").
//
// Ingest, one lane per row, reproduces Decimal(P, S, text)
// (src/datatypes/decimal.cu:154-165) followed by ToCompactDecimal
// (decimal.cu:337-341), the per-value step of the CSV import
// (src/server/mysql/importCsvFile.cpp:640-660):
//   StringToDecimal (decimal.cu:2980-3025): after an optional leading '-',
//   every character c is accumulated as v = v*10 + (c - '0') modulo 2^1024,
//   (c - '0') signed, so a character that is not a digit still shifts and
//   offsets the value; a '.' sets the fraction flag and the character after
//   it is taken as a digit whatever it is; every character after the first
//   '.' counts one fractional digit.  A row ends at its length or at its
//   first NUL; a '.' that ends the row ends it (the reference goes on to
//   read its terminator as a digit and past it).
//   cast (decimal.cu:471-533): scale up multiplies by 10^(S - frac) modulo
//   2^1024; scale down is floor division by 10^(frac - S); the sign is kept.
//   ToCompactDecimal: the low B(P) bytes of the magnitude with the sign
//   OR-ed into bit 7 of the last one.
// Multiplication and addition modulo 2^(32 W) give the low 32 W bits of the
// reference's 32-limb result exactly, so a row whose cast only scales up is
// parsed at the output's width.  A row that is cast down divides the whole
// value.
//
// Output, one lane per row, formats Decimal(compact, P, S)
// (decimal.cu:167-176) either as GetDecimal (decimal.cu:362-397, the form
// AriesDataBuffer::GetCompactDecimalAsString returns,
// src/CudaAcc/AriesEngineDef.cu:817-829): '+' or '-', eight upper-case hex
// digits per limb from the top nonzero limb down, "(" three digits of the
// scale ")"; or as decimal text with exactly `scale` fractional digits
// ("-123.4500"), the form the reference's decimal tests print.  Each row
// goes to a fixed stride-byte slot, NUL-terminated and zero-filled; rows are
// assembled in LDS and written out with coalesced dword stores.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "../../include/updec.h"
#include "api_internal.h"
#include "dec_device.h"
#include "planner.h"

using namespace updec;

namespace {

#define CODECCHK(expr)                                                                                       \
    do {                                                                                                     \
        hipError_t e_ = (expr);                                                                              \
        if (e_ != hipSuccess) return api_fail(UPDEC_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

inline hipStream_t st_of(updec_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

// the reference's Decimal holds 32 limbs; B(P) above 128 bytes would not fit it
constexpr int kMaxParseBytes = 128;

// limb class (2, 4, 8, 16, 32) that holds B bytes
int limb_class(int B)
{
    const int w = (B + 3) / 4;
    return w <= 2 ? 2 : w <= 4 ? 4 : w <= 8 ? 8 : w <= 16 ? 16 : 32;
}

// ---------------------------------------------------------------- ingest

// Rows cast down from more than 16 characters, or from any that are not plain
// (below), are held in memory, in as many limbs as they need: rolled loops over
// a run-time limb count keep this code's registers out of the kernel's, which
// the plain rows need for eight waves per SIMD.
struct WideRow {
    u32 w[32];
    u32 n;  // limbs held; the value is modulo 2^1024 once there are 32
};

// v = v * m + add
__device__ __forceinline__ void wide_mul_add(WideRow& v, u32 m, u32 add)
{
    u32 c = add;
#pragma unroll 1
    for (u32 i = 0; i < v.n; i++) {
        const u64 t = (u64)v.w[i] * m + c;
        v.w[i] = (u32)t;
        c = (u32)(t >> 32);
    }
    if (c != 0u && v.n < 32u) v.w[v.n++] = c;
}

// v = floor(v / d), d normalized to dn = d << s with reciprocal r
__device__ __forceinline__ void wide_div_word(WideRow& v, u32 dn, u32 s, u32 r)
{
    u32 rem = 0;
#pragma unroll 1
    for (u32 i = v.n; i-- > 0;) {
        const u32 x = v.w[i];
        const u32 u1 = s ? (rem << s) | (x >> (32u - s)) : rem;
        u32 rr;
        v.w[i] = div_2by1(u1, x << s, dn, r, rr);
        rem = rr >> s;
    }
}

// to scale S: floor of the division by 10^(frac - S)
__device__ void wide_cast(WideRow& v, u32 frac, u32 S)
{
    u32 k = frac - S;
    while (k != 0u) {
        const u32 step = k < 9u ? k : 9u;
        const u32 d = pow10_word(step);
        const u32 s = (u32)__builtin_clz(d);
        wide_div_word(v, d << s, s, recip_word(d << s));
        k -= step;
    }
}

// ---- plain rows
//
// A plain row is an optional '-', then decimal digits with at most one '.'
// among or after them: every row that a database writes.  It is parsed sixteen characters at a time in registers, without a
// branch per character: the dwords covering them are realigned, the '.' is
// found and closed up, the digits are moved to the end of the sixteen bytes
// (so that the front fills with zeros) and checked, and each four become a
// number by one byte dot product.  Any other row takes the walk over
// characters above.

// The sixteen characters from s on (a byte address): the dwords that hold
// one of them and begin before `end`, the last offset, realigned; or before
// the row's own end, `left` characters on, where the offsets go down after it.
// Characters past both come out as anything.
__device__ __forceinline__ void load_chars16(uintptr_t s, uintptr_t end, u32 left, u64& x0, u64& x1)
{
    const u32* p = reinterpret_cast<const u32*>(s & ~(uintptr_t)3);
    const u32 sh = (u32)(s & 3u);
    u32 w[5];
    if (reinterpret_cast<uintptr_t>(p + 5) <= end) {
        load_dwords<5, false>(p, w);
    } else {
        const uintptr_t stop = s + left > end ? s + left : end;
#pragma unroll
        for (int k = 0; k < 5; k++) w[k] = reinterpret_cast<uintptr_t>(p + k) < stop ? p[k] : 0u;
    }
    u32 t[4];
#pragma unroll
    for (int j = 0; j < 4; j++) t[j] = __builtin_amdgcn_alignbyte(w[j + 1], w[j], sh);
    x0 = ((u64)t[1] << 32) | t[0];
    x1 = ((u64)t[3] << 32) | t[2];
}

// index of the first C in eight characters, 8 when there is none
template <char C> __device__ __forceinline__ u32 first_char(u64 x)
{
    const u64 z = x ^ (0x0101010101010101ull * (u64)(u8)C);
    const u64 m = (z - 0x0101010101010101ull) & ~z & 0x8080808080808080ull;
    return m ? (u32)__builtin_ctzll(m) >> 3 : 8u;
}

// four digits (most significant in the lowest byte) as a number
__device__ __forceinline__ u32 digits4(u32 d) { return __builtin_amdgcn_udot4(d, 0x00010A64u, 0u, false) * 10u + (d >> 24); }

// `cnt` <= 16 characters: the digits among them as hi * 10^8 + lo, their
// number, the place of the '.' (16: none), and whether all of them but the
// '.' are digits
struct Piece {
    u32 hi, lo, n, dot;
    bool plain;
};

__device__ __forceinline__ Piece piece16(u64 x0, u64 x1, u32 cnt)
{
    Piece r;
    const u32 p0 = first_char<'.'>(x0), p1 = first_char<'.'>(x1);
    u32 p = p0 < 8u ? p0 : 8u + p1;
    if (p >= cnt) p = 16u;
    r.dot = p;
    // close the '.' up: bytes past it move down by one
    const u64 y0 = (x0 >> 8) | (x1 << 56), y1 = x1 >> 8;
    const u64 m0 = p < 8u ? ~0ull << (8u * p) : 0ull;
    const u64 m1 = p < 8u ? ~0ull : (p < 16u ? ~0ull << (8u * (p - 8u)) : 0ull);
    const u64 d0 = (x0 ^ ((x0 ^ y0) & m0)) ^ 0x3030303030303030ull;
    const u64 d1 = (x1 ^ ((x1 ^ y1) & m1)) ^ 0x3030303030303030ull;
    r.n = cnt - (p < 16u ? 1u : 0u);
    // the digits to the end of the sixteen bytes
    const u32 sb = 8u * (16u - r.n);  // 0 .. 128
    u64 z0, z1;
    if (sb >= 64u) {
        z0 = 0;
        z1 = sb < 128u ? d0 << (sb - 64u) : 0ull;
    } else {
        z0 = d0 << sb;
        z1 = (d1 << sb) | ((d0 >> 1) >> (63u - sb));
    }
    const u64 bad = (z0 | (z0 + 0x0606060606060606ull) | z1 | (z1 + 0x0606060606060606ull)) & 0xf0f0f0f0f0f0f0f0ull;
    r.plain = bad == 0;
    r.hi = digits4((u32)z0) * 10000u + digits4((u32)(z0 >> 32));
    r.lo = digits4((u32)z1) * 10000u + digits4((u32)(z1 >> 32));
    return r;
}

// v = v * m + add modulo 2^(32 W)
template <int W> __device__ __forceinline__ void mul_add_word(Mag<W>& v, u32 m, u32 add)
{
    u32 c = add;
#pragma unroll
    for (int i = 0; i < W; i++) {
        const u64 t = (u64)v.w[i] * m + c;
        v.w[i] = (u32)t;
        c = (u32)(t >> 32);
    }
}

// A plain row of up to 16 characters: its value (below 10^16) and sign
__device__ __forceinline__ bool plain_short(uintptr_t s, uintptr_t end, u32 len, u64& v, u32& frac, u32& neg)
{
    u64 x0, x1;
    load_chars16(s, end, len, x0, x1);
    neg = len > 0u && (x0 & 255u) == (u64)'-' ? 1u : 0u;
    if (neg) {
        x0 = (x0 >> 8) | (x1 << 56);
        x1 >>= 8;
    }
    const Piece q = piece16(x0, x1, len - neg);
    v = (u64)q.hi * 100000000u + q.lo;
    frac = q.dot < 16u ? len - neg - q.dot - 1u : 0u;
    return q.plain;
}

// A plain row of any length: its value modulo 2^(32 W)
template <int W> __device__ bool plain_long(uintptr_t s, uintptr_t end, u32 len, Mag<W>& v, u32& frac)
{
    v = mzero<W>();
    frac = 0u;
    bool dot = false, ok = true;
    for (u32 i = 0; i < len && ok; i += 16u) {
        u64 x0, x1;
        load_chars16(s + i, end, len - i, x0, x1);
        const u32 cnt = len - i < 16u ? len - i : 16u;
        const Piece q = piece16(x0, x1, cnt);
        ok = ok && q.plain;
        if (q.dot < 16u) {
            ok = ok && !dot;  // a second '.' is a character like any other
            dot = true;
            frac = len - (i + q.dot) - 1u;
        }
        if (q.n > 8u) mul_add_word<W>(v, q.n == 16u ? 100000000u : pow10_word(q.n - 8u), q.hi);
        mul_add_word<W>(v, q.n >= 8u ? 100000000u : pow10_word(q.n), q.lo);
    }
    return ok;
}

// Any row behind its sign by the rules above: fold(k, x) is v = v 10^k + x for
// each sixteen characters, k of them digits, |x| < 2^59.  One character a step
// where they are not plain, also when cut at the row's first NUL.  (Rows with a
// NUL or a foreign character took a walk over single characters loaded one by
// one, twice, and folds over all limbs of the output in memory: 98,000 rows of
// DECIMAL(300,100) NUL-padded 473 -> 85 us, beginning with a space 474 -> 63;
// 2 M of DECIMAL(15,2), one in 64 ending in a space, 222 -> 72.)
template <class Fold> __device__ __forceinline__ void walk_any(uintptr_t s, uintptr_t end, u32 len, u32& frac, const Fold& fold)
{
    frac = 0u;
    bool dot = false, force = false;   // force: the character behind a '.', a digit whatever it is
#pragma unroll 1
    for (u32 i = 0; i < len; i += 16u) {
        u64 x0, x1;
        load_chars16(s + i, end, len - i, x0, x1);
        u32 cnt = len - i < 16u ? len - i : 16u;
        u32 stop = first_char<'\0'>(x0);
        if (stop == 8u) stop += first_char<'\0'>(x1);
        if (stop < cnt) {
            cnt = stop;
            len = i + stop;
        }
        const Piece q = piece16(x0, x1, cnt);
        if (q.plain && !force) {
            frac += dot ? q.n : q.dot < 16u ? cnt - q.dot - 1u : 0u;
            dot = dot || q.dot < 16u;
            force = q.dot < 16u && q.dot == cnt - 1u;
            fold(q.n, (i64)((u64)q.hi * 100000000u + q.lo));
            continue;
        }
        i64 x = 0;
        u32 k = 0;
#pragma unroll 1
        for (u32 j = 0; j < cnt; j++) {
            const u32 c = (u32)x0 & 255u;
            x0 = (x0 >> 8) | (x1 << 56);
            x1 >>= 8;
            if (!force && c == (u32)'.') {
                dot = force = true;
                continue;
            }
            force = false;
            frac += dot ? 1u : 0u;
            x = x * 10 + ((i32)(signed char)(char)c - '0');
            k++;
        }
        fold(k, x);
    }
}

// to any width, modulo 2^(32 W)
template <int W> __device__ __forceinline__ void any_row(uintptr_t s, uintptr_t end, u32 len, Mag<W>& v, u32& frac)
{
    v = mzero<W>();
    walk_any(s, end, len, frac, [&](u32 k, i64 x) {
        if (k > 8u) mul_add_word<W>(v, pow10_word(k - 8u), 0u);
        mul_add_word<W>(v, pow10_word(k < 8u ? k : 8u), 0u);
        const u32 ext = x < 0 ? 0xffffffffu : 0u;
        u32 c = 0u;
#pragma unroll
        for (int i = 0; i < W; i++) v.w[i] = addc(v.w[i], i == 0 ? (u32)x : (i == 1 ? (u32)((u64)x >> 32) : ext), c);
    });
}

// to be cast down: two's complement of v.n limbs, modulo 2^1024 from 32 on
__device__ __forceinline__ void signed_mul_add(WideRow& v, u32 m, i64 add)
{
    const u32 ext = v.n != 0u && (i32)v.w[v.n - 1u] < 0 ? 0xffffffffu : 0u;
    const u32 n = v.n == 0u ? 2u : v.n < 32u ? v.n + 1u : 32u;
    u64 c = 0;
#pragma unroll 1
    for (u32 i = 0; i < n; i++) {
        const u32 a = i == 0u ? (u32)add : (i == 1u ? (u32)((u64)add >> 32) : (add < 0 ? 0xffffffffu : 0u));
        const u64 t = (u64)(i < v.n ? v.w[i] : ext) * m;
        const u64 lo = (t & 0xffffffffull) + a + (c & 0xffffffffull);
        v.w[i] = (u32)lo;
        c = (t >> 32) + (lo >> 32) + (c >> 32);
    }
    v.n = n;
}

__device__ void wide_any(uintptr_t s, uintptr_t end, u32 len, u32 S, WideRow& v)
{
    v.n = 0u;
    u32 frac;
    walk_any(s, end, len, frac, [&](u32 k, i64 x) {
        if (k > 8u && v.n != 0u) signed_mul_add(v, pow10_word(k - 8u), 0);
        signed_mul_add(v, pow10_word(k < 8u ? k : 8u), x);
    });
    // the division is of the 1024-bit number
    if (v.n != 0u && (i32)v.w[v.n - 1u] < 0)
        while (v.n < 32u) v.w[v.n++] = 0xffffffffu;
    wide_cast(v, frac, S);
}

// A plain row cast down: the division needs the whole value (modulo 2^1024,
// as the reference holds it)
__device__ void wide_plain(uintptr_t s, uintptr_t end, u32 len, u32 frac, u32 S, WideRow& v)
{
    v.n = 0u;
    for (u32 i = 0; i < len; i += 16u) {
        u64 x0, x1;
        load_chars16(s + i, end, len - i, x0, x1);
        const Piece q = piece16(x0, x1, len - i < 16u ? len - i : 16u);
        if (q.n > 8u) wide_mul_add(v, pow10_word(q.n - 8u), q.hi);
        wide_mul_add(v, pow10_word(q.n < 8u ? q.n : 8u), q.lo);
    }
    wide_cast(v, frac, S);
}

// rows per block of the ingest kernel, and of the two format kernels
constexpr int kParseBlock = 256;
constexpr int kCodecBlock = 64;
constexpr int kShortBlock = 256;

// One lane per row; the block's compact rows are assembled in LDS and leave
// as dwords.
//
// What bounds it: integer issue, then HBM.  Walking the characters of a row
// cost about 600 instructions a wave, two thirds of them the scalar
// bookkeeping of its branches; sixteen at a time it is about
// 200.  10 M rows of DECIMAL(15,2) text: 147 -> 60 us; 2 M of DECIMAL(38,10):
// 226 -> 35, cast down from four more digits 227 -> 93; 200,000 of
// DECIMAL(300,100): 601 -> 52.  Eight waves per SIMD are worth a third of it
// (94 us at four), which is why the wide rows are kept out of registers.
template <int WO>
__global__ void __launch_bounds__(kParseBlock, WO <= 16 ? 8 : 1) k_parse_compact(const char* __restrict__ chars,
                                                               const int64_t* __restrict__ offsets, int64_t rows,
                                                               u32 B, u32 S, u8* __restrict__ out)
{
    extern __shared__ u32 tile[];  // kParseBlock * B bytes, rounded up to dwords
    u8* t8 = reinterpret_cast<u8*>(tile);
    const int64_t base = (int64_t)blockIdx.x * kParseBlock;
    const int64_t row = base + threadIdx.x;
    const uintptr_t end = reinterpret_cast<uintptr_t>(chars + offsets[rows]);
    if (row < rows) {
        const int64_t o0 = offsets[row], o1 = offsets[row + 1];
        const char* s = chars + o0;
        u32 len = o1 > o0 ? (u32)(o1 - o0) : 0u;
        Mag<WO> m;
        u32 neg = 0u, frac = 0u;
        bool done = false;
        const uintptr_t a = reinterpret_cast<uintptr_t>(s);
        bool plain;
        if (len <= 16u) {
            u64 u;
            plain = plain_short(a, end, len, u, frac, neg);
            if (plain) {
                if (S < frac) {
                    // floor(v / 10^(frac - S)), frac - S <= 15
                    u64 d = 1;
                    for (u32 k = 0; k < frac - S; k++) d *= 10u;
                    u /= d;
                    frac = S;
                }
#pragma unroll
                for (int i = 0; i < WO; i++) m.w[i] = i == 0 ? (u32)u : (i == 1 ? (u32)(u >> 32) : 0u);
                done = true;
            }
        } else {
            neg = s[0] == '-' ? 1u : 0u;
            plain = done = plain_long<WO>(a + neg, end, len - neg, m, frac);
        }
        if (!plain) {
            neg = len != 0u && s[0] == '-' ? 1u : 0u;
            any_row<WO>(a + neg, end, len - neg, m, frac);
            done = S >= frac;
        } else if (S < frac) {
            done = false;
        }
        if (done) {
            if (S > frac) m = mul_p10_rt<WO>(m, S - frac);
        } else {
            WideRow v;
            if (plain) wide_plain(a + neg, end, len - neg, frac, S, v);
            else wide_any(a + neg, end, len - neg, S, v);
#pragma unroll
            for (int i = 0; i < WO; i++) m.w[i] = (u32)i < v.n ? v.w[i] : 0u;
        }
        // B bytes at byte offset tid * B: whole dwords (unaligned), then bytes
        u8* dst = t8 + (u32)threadIdx.x * B;
        const u32 sign = neg << 7;
#pragma unroll
        for (int i = 0; i < WO; i++) {
            if (4u * (u32)i + 4u < B) {
                __builtin_memcpy(dst + 4 * i, &m.w[i], 4);
            } else {
#pragma unroll
                for (int b = 4 * i; b < 4 * i + 4; b++) {
                    const u32 x = (m.w[i] >> (8 * (b & 3))) & 255u;
                    if ((u32)b + 1u < B) dst[b] = (u8)x;
                    else if ((u32)b + 1u == B) dst[b] = (u8)(x | sign);
                }
            }
        }
    }
    __syncthreads();
    const int64_t nrows = rows - base < kParseBlock ? rows - base : kParseBlock;
    const u32 n = (u32)nrows * B;
    u8* d = out + base * (int64_t)B;
    // the block's span starts at base * B: dword stores when that is aligned
    if (((uintptr_t)d & 3u) == 0) {
        for (u32 i = threadIdx.x; i < n / 4; i += kParseBlock) reinterpret_cast<u32*>(d)[i] = tile[i];
        for (u32 i = (n / 4) * 4 + threadIdx.x; i < n; i += kParseBlock) d[i] = t8[i];
    } else {
        for (u32 i = threadIdx.x; i < n; i += kParseBlock) d[i] = t8[i];
    }
}

// ---------------------------------------------------------------- output

// x = floor(x / 10^8), the remainder returned; `n` limbs of x can be nonzero
template <int W> __device__ __forceinline__ u32 div_1e8_rem(Mag<W>& x, u32 n)
{
    u32 r = 0;
#pragma unroll
    for (int i = W - 1; i >= 0; i--)
        if ((u32)i < n) x.w[i] = div_word_const<100000000u>(r, x.w[i]);
    return r;
}

// the four digits of v < 10^4, most significant in the lowest byte, as
// characters
__device__ __forceinline__ u32 chars4(u32 v)
{
    const u32 q = (v * 5243u) >> 19;               // v / 100
    const u32 pair = q | ((v - 100u * q) << 16);   // two numbers below 100
    const u32 tens = ((pair * 103u) >> 10) & 0x000f000fu;
    return (tens | ((pair - 10u * tens) << 8)) + 0x30303030u;
}

// the four hex digits of v < 2^16, most significant in the lowest byte
__device__ __forceinline__ u32 hex4(u32 v)
{
    u32 x = (v | (v << 8)) & 0x00ff00ffu;
    x = (x | (x << 4)) & 0x0f0f0f0fu;
    x = __builtin_bswap32(x);
    return x + 0x30303030u + ((x + 0x06060606u) >> 4 & 0x01010101u) * 7u;
}

struct FormatArgs {
    const u8* col;
    char* out;
    i64 rows;
    u32 B, S, hex;
    u32 end;        // bytes of a row's LDS area up to the end of its text
    u32 area;       // bytes of a row's LDS area
    u32 groups;     // text: groups of four digits that a row can have
    u32 slot;       // bytes of the longest form, rounded to dwords
    u32 stride;     // bytes from row to row in the output
    u32 magic;      // ceil(2^32 / (stride / 4)), 0: divide
};

// One lane per row, one wave per block.  A row's text is written from its
// last character back, so that every digit has its place before the length
// is known: four at a time as a dword at the fixed distance from the end
// that the scale gives (the '.' too).  The copy to the slots then starts
// each row where its text starts.  Divisions and digits end with the longest
// row of the wave: with those of the column's precision, values of 3 digits in
// DECIMAL(300,100), 200,000 rows, took 156 us instead of 51.
//
// What bounds it: integer issue (the divisions by 10^8 and the characters),
// then the stores.  It had divided by 10^9, written and read every character
// twice through LDS, and divided by the stride for every dword stored:
// 1 M rows of DECIMAL(76,20) as text 90 -> 75 us, 200,000 of DECIMAL(300,100)
// 333 -> 157, as hex 65 -> 44.
template <int W> __global__ void __launch_bounds__(kCodecBlock) k_format_compact(FormatArgs a)
{
    extern __shared__ u32 tile[];
    __shared__ u32 start[kCodecBlock];
    u8* t8 = reinterpret_cast<u8*>(tile);
    const i64 base = (i64)blockIdx.x * kCodecBlock;
    const i64 row = base + threadIdx.x;
    u8* const o = t8 + (u32)threadIdx.x * a.area;
    auto put4 = [](u8* p, u32 x) { __builtin_memcpy(p, &x, 4); };
    if (row < a.rows) {
        const Dec<W> v = load_compact_rt<W>(a.col, (usize)row, a.B, (usize)a.rows * a.B);
        u32 p;  // where the text starts
        // limbs that any row of the wave has
        u32 most = 0;
#pragma unroll
        for (int i = 0; i < W; i++) most = any_lane(v.m.w[i] != 0u) ? (u32)i + 1u : most;
        if (a.hex) {
            // eight digits a limb from the top nonzero limb down, "(SSS)"
            u32 top = 0;
#pragma unroll
            for (int i = 0; i < W; i++) {
                if ((u32)i < most) {
                    u8* d = o + a.end - 13u - 8u * (u32)i;
                    put4(d, hex4(v.m.w[i] >> 16));
                    put4(d + 4, hex4(v.m.w[i] & 0xffffu));
                    top = v.m.w[i] ? (u32)i + 1u : top;
                }
            }
            put4(o + a.end - 5u, (u32)'(' | ((u32)'0' + a.S / 100u) << 8 | ((u32)'0' + a.S / 10u % 10u) << 16 |
                                     ((u32)'0' + a.S % 10u) << 24);
            o[a.end - 1u] = ')';
            p = a.end - 6u - 8u * top;
            o[p] = v.neg ? '-' : '+';
        } else {
            Mag<W> x = v.m;
            const u32 point = a.S > 0u ? 1u : 0u;
            u32 n = 0;     // digits up to the highest nonzero one
            u32 bits = 32u * most < 8u * a.B ? 32u * most : 8u * a.B;
            // the group of four whose last is digit k
            auto put_group = [&](u32 k, u32 c) {
                if (k + 4u <= a.S || point == 0u) {
                    put4(o + a.end - k - 4u, c);
                } else if (k >= a.S) {
                    put4(o + a.end - k - 5u, c);
                } else {
                    // the '.' falls inside the group
#pragma unroll
                    for (u32 b = 0; b < 4u; b++)
                        o[a.end - k - 1u - b - (k + b >= a.S ? 1u : 0u)] = (u8)(c >> (8u * (3u - b)));
                }
            };
            u32 j = 0;
            for (; j < a.groups && bits != 0u; j += 2u) {
                const u32 r = div_1e8_rem<W>(x, (bits + 31u) / 32u);
                bits = bits > 26u ? bits - 26u : 0u;   // 10^8 > 2^26
                const u32 hi = r / 10000u;
#pragma unroll
                for (u32 h = 0; h < 2u; h++) {
                    const u32 g = h ? hi : r - 10000u * hi;
                    const u32 k = 4u * (j + h);
                    if (g) n = k + (g >= 1000u ? 4u : g >= 100u ? 3u : g >= 10u ? 2u : 1u);
                    put_group(k, chars4(g));
                }
            }
            // zeros up to the digit before the '.'
            for (; j < a.groups && 4u * j <= a.S; j++) put_group(4u * j, 0x30303030u);
            if (point) o[a.end - 1u - a.S] = '.';
            n = n > a.S ? n : a.S + 1u;
            p = a.end - n - point - v.neg;
            if (v.neg) o[p] = '-';
        }
        start[threadIdx.x] = (u32)threadIdx.x * a.area + p;
    }
    __syncthreads();
    // the block's rows are consecutive stride-byte slots: dword stores,
    // zeros past each row's text
    const u32 nrows = (u32)(a.rows - base < kCodecBlock ? a.rows - base : kCodecBlock);
    const u32 sw = a.stride / 4;
    const u32 nw = nrows * sw;
    u32* d = reinterpret_cast<u32*>(a.out + base * (i64)a.stride);
    for (u32 i = threadIdx.x; i < nw; i += kCodecBlock) {
        const u32 r = a.magic ? (u32)(((u64)i * a.magic) >> 32) : i / sw, w = i - r * sw;
        const u32 at = start[r] + 4u * w, stop = r * a.area + a.end;
        u32 x = 0;
        if (at < stop) {
            __builtin_memcpy(&x, t8 + at, 4);
            const u32 left = stop - at;
            if (left < 4u) x &= (1u << (8u * left)) - 1u;
        }
        d[i] = x;
    }
}

// ---- rows of up to 16 bytes
//
// One lane per row, all in registers.  The text is assembled at the end of
// ND dwords, where every character's place is known but for the scale, which
// is the same for all rows (so the masks that part the digits at the '.' are
// scalar); then it is moved to the front by the row's own number of leading
// places.  42 characters of text, or 38 of hex, is the longest.  The block's
// slots leave through LDS as 16-byte stores.
//
// What bounds it: the stores as hex (5.2 TB/s read and written), integer
// issue as text.  10 M rows of DECIMAL(15,2): text 117 -> 73 us, hex 77 -> 59;
// 3 M rows of DECIMAL(38,10): text 93 -> 43, hex 45 -> 31.
template <int W> struct ShortText {
    static constexpr int G = W == 2 ? 5 : 10;       // groups of four decimal digits: 2^63 has 19, 2^127 39
    static constexpr int ND = W == 2 ? 6 : 11;      // dwords: digits, '.' and sign; or 8 W hex digits and 6 more
};

// the bytes of t moved to the front by `by`, zeros behind them
template <int ND> __device__ __forceinline__ Mag<ND> move_front(Mag<ND> t, u32 by)
{
    const u32 ws = by >> 2;
#pragma unroll
    for (int st = 1; st < ND; st <<= 1) {
        const bool on = (ws & (u32)st) != 0u;
        if (!any_lane(on)) continue;
        Mag<ND> u;
#pragma unroll
        for (int k = 0; k < ND; k++) u.w[k] = k + st < ND ? t.w[k + st] : 0u;
#pragma unroll
        for (int k = 0; k < ND; k++) t.w[k] = on ? u.w[k] : t.w[k];
    }
    Mag<ND> r;
#pragma unroll
    for (int k = 0; k < ND; k++) r.w[k] = __builtin_amdgcn_alignbyte(k + 1 < ND ? t.w[k + 1] : 0u, t.w[k], by & 3u);
    return r;
}

template <int W, bool HEX> __global__ void __launch_bounds__(kShortBlock) k_format_short(FormatArgs a)
{
    constexpr int ND = ShortText<W>::ND, G = ShortText<W>::G;
    __shared__ u32 tile[kShortBlock * ND];
    const i64 base = (i64)blockIdx.x * kShortBlock;
    const i64 row = base + threadIdx.x;
    // lanes past the last row format it again; what they write is not stored
    const Dec<W> v = load_compact_rt<W>(a.col, (usize)(row < a.rows ? row : a.rows - 1), a.B, (usize)a.rows * a.B);
    Mag<ND> t;
    u32 from;  // where the text starts
    if constexpr (HEX) {
        // eight digits a limb from the top nonzero limb down, then "(SSS)":
        // one character of it stands before the last dword
        u32 h[ND];
        u32 top = 0;
#pragma unroll
        for (int k = 0; k < ND; k++) h[k] = 0u;
#pragma unroll
        for (int i = 0; i < W; i++) {
            h[ND - 2 - 2 * i] = hex4(v.m.w[i] & 0xffffu);
            h[ND - 3 - 2 * i] = hex4(v.m.w[i] >> 16);
            top = v.m.w[i] ? (u32)i + 1u : top;
        }
        h[ND - 1] = (u32)'(';
#pragma unroll
        for (int k = 0; k < ND - 1; k++) t.w[k] = __builtin_amdgcn_alignbyte(h[k + 1], h[k], 1u);
        t.w[ND - 1] = ((u32)'0' + a.S / 100u) | ((u32)'0' + a.S / 10u % 10u) << 8 | ((u32)'0' + a.S % 10u) << 16 |
                    (u32)')' << 24;
        from = 4u * ND - 6u - 8u * top;
    } else {
        // digits: group g (four, the lowest first) in dword ND - 1 - g
        Mag<ND> d;
#pragma unroll
        for (int k = 0; k < ND; k++) d.w[k] = 0x30303030u;
        if constexpr (W == 2) {
            const u64 x = ((u64)v.m.w[1] << 32) | v.m.w[0];
            const u64 q = x / 100000000u;                      // below 2^37
            const u32 r0 = (u32)x - (u32)q * 100000000u;
            const u32 h = (u32)(q >> 8) / 390625u;             // q / 10^8
            const u32 r1 = (u32)q - h * 100000000u;
            const u32 q0 = r0 / 10000u, q1 = r1 / 10000u;
            d.w[ND - 1] = chars4(r0 - 10000u * q0);
            d.w[ND - 2] = chars4(q0);
            d.w[ND - 3] = chars4(r1 - 10000u * q1);
            d.w[ND - 4] = chars4(q1);
            d.w[ND - 5] = chars4(h);
        } else {
            Mag<W> x = v.m;
#pragma unroll
            for (int j = 0; j < G; j += 2) {
                if ((u32)j >= a.groups) continue;
                // 10^8 > 2^26: what is left after j / 2 divisions fits these limbs
                const int left = 32 * W - 1 - 13 * j;
                const u32 r = left > 27 ? div_1e8_rem<W>(x, (u32)(left + 31) / 32u) : x.w[0];
                const u32 hi = r / 10000u;
                d.w[ND - 1 - j] = chars4(r - 10000u * hi);
                d.w[ND - 2 - j] = chars4(hi);
            }
        }
        // digits from the first nonzero one on
        u32 lead = 4u * ND;
#pragma unroll
        for (int k = ND - 1; k >= 0; k--) {
            const u32 z = d.w[k] ^ 0x30303030u;
            lead = z ? 4u * (u32)k + ((u32)__builtin_ctz(z) >> 3) : lead;
        }
        u32 n = 4u * ND - lead;
        n = n > a.S ? n : a.S + 1u;
        const u32 point = a.S > 0u ? 1u : 0u;
#pragma unroll
        for (int k = 0; k < ND; k++) {
            // of this dword's characters the last m stand behind the '.',
            // which is character 3 - m when it falls inside
            const i32 m = (i32)a.S - 4 * (ND - 1 - k);
            const u32 after = !point || m >= 4 ? 0xffffffffu : (m <= 0 ? 0u : 0xffffffffu << (32 - 8 * m));
            const u32 before = !point || m >= 4 ? 0u : (m < 0 ? 0xffffffffu : (1u << (8 * (3 - m))) - 1u);
            const u32 dot = point && m >= 0 && m < 4 ? (u32)'.' << (8 * (3 - m)) : 0u;
            const u32 up = __builtin_amdgcn_alignbyte(k + 1 < ND ? d.w[k + 1] : 0u, d.w[k], 1u);
            t.w[k] = (d.w[k] & after) | (up & before) | dot;
        }
        from = 4u * ND - n - point - v.neg;
    }
    t = move_front<ND>(t, from);
    if (HEX || v.neg) t.w[0] = (t.w[0] & ~255u) | (v.neg ? (u32)'-' : (u32)'+');
    const u32 sw = a.stride / 4, lw = a.slot / 4;
    const u32 nrows = (u32)(a.rows - base < kShortBlock ? a.rows - base : kShortBlock);
#pragma unroll
    for (int k = 0; k < ND; k++)
        if ((u32)k < lw) tile[threadIdx.x * lw + k] = t.w[k];
    __syncthreads();
    u32* o = reinterpret_cast<u32*>(a.out + base * (i64)a.stride);
    if (sw == lw) {
        // the block's slots are one span: 16 bytes a lane, then the rest
        const u32 n = nrows * lw, quads = n / 4u;
        for (u32 i = threadIdx.x; i < quads; i += kShortBlock) {
            u32x4u q;
            q[0] = tile[4u * i];
            q[1] = tile[4u * i + 1u];
            q[2] = tile[4u * i + 2u];
            q[3] = tile[4u * i + 3u];
            *reinterpret_cast<u32x4u*>(o + 4u * i) = q;
        }
        for (u32 i = 4u * quads + threadIdx.x; i < n; i += kShortBlock) o[i] = tile[i];
    } else {
        for (u32 i = threadIdx.x; i < nrows * sw; i += kShortBlock) {
            const u32 r = i / sw, w = i - r * sw;
            o[i] = w < lw ? tile[r * lw + w] : 0u;
        }
    }
}

// characters of the longest decimal text of DECIMAL(P, S): sign, the
// digits of 2^(8B - 1) - 1 (or S + 1 when more), the point, NUL
int64_t text_slot(int P, int S)
{
    const int B = compact_bytes(P);
    const int bits = 8 * B - 1;
    const int digits = (int)std::floor(bits * 0.30102999566398119521) + 1;
    const int body = digits > S + 1 ? digits : S + 1;
    return 1 + body + (S > 0 ? 1 : 0) + 1;
}

// GetDecimal's longest form: sign, 8 hex digits per limb of a magnitude
// below 2^(8B - 1), "(SSS)", NUL
int64_t hex_slot(int P)
{
    const int B = compact_bytes(P);
    const int limbs = (8 * B - 1 + 31) / 32;
    return 1 + 8 * (int64_t)limbs + 5 + 1;
}

}  // namespace

extern "C" {

int updec_parse_compact(const char* d_chars, const int64_t* d_offsets, int64_t rows, int32_t precision,
                        int32_t scale, uint8_t* d_out, updec_stream_t stream)
{
    if (rows < 0 || (rows && (!d_chars || !d_offsets || !d_out))) return api_fail(UPDEC_EINVAL, "bad argument");
    if (precision < 1 || scale < 0 || scale > precision) return api_fail(UPDEC_EINVAL, "bad precision or scale");
    const int B = compact_bytes(precision);
    if (B > kMaxParseBytes)
        return api_fail(UPDEC_EUNSUPPORTED, "B(P) above 128 bytes: the reference's 32-limb Decimal cannot hold it");
    if (rows == 0) return UPDEC_OK;
    const unsigned grid = (unsigned)((rows + kParseBlock - 1) / kParseBlock);
    const size_t lds = ((size_t)kParseBlock * B + 3) / 4 * 4;
    hipStream_t st = st_of(stream);
    switch (limb_class(B)) {
    case 2: hipLaunchKernelGGL(k_parse_compact<2>, dim3(grid), dim3(kParseBlock), lds, st, d_chars, d_offsets, rows, (u32)B, (u32)scale, d_out); break;
    case 4: hipLaunchKernelGGL(k_parse_compact<4>, dim3(grid), dim3(kParseBlock), lds, st, d_chars, d_offsets, rows, (u32)B, (u32)scale, d_out); break;
    case 8: hipLaunchKernelGGL(k_parse_compact<8>, dim3(grid), dim3(kParseBlock), lds, st, d_chars, d_offsets, rows, (u32)B, (u32)scale, d_out); break;
    case 16: hipLaunchKernelGGL(k_parse_compact<16>, dim3(grid), dim3(kParseBlock), lds, st, d_chars, d_offsets, rows, (u32)B, (u32)scale, d_out); break;
    default: hipLaunchKernelGGL(k_parse_compact<32>, dim3(grid), dim3(kParseBlock), lds, st, d_chars, d_offsets, rows, (u32)B, (u32)scale, d_out); break;
    }
    CODECCHK(hipGetLastError());
    return UPDEC_OK;
}

int updec_format_stride(int32_t precision, int32_t scale, int32_t form, int64_t* stride)
{
    if (!stride || precision < 1 || scale < 0 || scale > precision) return api_fail(UPDEC_EINVAL, "bad argument");
    if (form != UPDEC_FORMAT_HEX && form != UPDEC_FORMAT_TEXT) return api_fail(UPDEC_EINVAL, "unknown format");
    if (compact_bytes(precision) > kMaxParseBytes) return api_fail(UPDEC_EUNSUPPORTED, "B(P) above 128 bytes");
    const int64_t n = form == UPDEC_FORMAT_HEX ? hex_slot(precision) : text_slot(precision, scale);
    *stride = (n + 3) / 4 * 4;
    return UPDEC_OK;
}

int updec_format_compact(const uint8_t* d_col, int64_t rows, int32_t precision, int32_t scale, int32_t form,
                         char* d_out, int64_t stride, updec_stream_t stream)
{
    int64_t need = 0;
    const int rc = updec_format_stride(precision, scale, form, &need);
    if (rc != UPDEC_OK) return rc;
    if (rows < 0 || (rows && (!d_col || !d_out))) return api_fail(UPDEC_EINVAL, "bad argument");
    if (stride < need || (stride & 3) || stride > (1 << 20))
        return api_fail(UPDEC_EINVAL, "stride below updec_format_stride, not a multiple of 4, or above 1 MiB");
    if (reinterpret_cast<uintptr_t>(d_out) & 3u) return api_fail(UPDEC_EINVAL, "output must be 4-byte aligned");
    if (rows == 0) return UPDEC_OK;
    const int B = compact_bytes(precision);
    const unsigned grid = (unsigned)((rows + kCodecBlock - 1) / kCodecBlock);
    FormatArgs f{};
    f.col = d_col;
    f.out = d_out;
    f.rows = rows;
    f.B = (u32)B;
    f.S = (u32)scale;
    f.hex = form == UPDEC_FORMAT_HEX ? 1u : 0u;
    f.slot = (u32)need;
    f.stride = (u32)stride;
    const u32 sw = f.stride / 4;
    // floor(i magic / 2^32) = floor(i / sw) while i (magic sw - 2^32) < 2^32,
    // so for every i < 64 sw when 64 sw^2 < 2^32
    f.magic = sw > 1 && sw < 8192 ? (u32)((((u64)1 << 32) + sw - 1) / sw) : 0u;
    if (f.hex) {
        f.end = 8u * (((u32)B + 3u) / 4u) + 6u;
    } else {
        // digits of 2^(8B - 1) - 1, or S + 1 when more, in groups of eight
        const u32 digits = std::max((u32)std::floor((8 * B - 1) * 0.30102999566398119521) + 1u, (u32)scale + 1u);
        f.groups = 2u * ((digits + 7u) / 8u);
        f.end = 4u * f.groups + 2u;  // sign and '.'
    }
    // an odd number of dwords a row: the lanes' areas start in different banks
    f.area = 4u * ((f.end + 3u) / 4u | 1u);
    const size_t lds = (size_t)kCodecBlock * f.area + 4u;
    hipStream_t st = st_of(stream);
    // Rows of up to 16 bytes are formatted in registers, wider ones through
    // LDS, where 8-byte rows take 129 us per 10 M rows of text and 16-byte
    // rows 99 us per 3 M, against 73 and 43 in registers
    const unsigned sgrid = (unsigned)((rows + kShortBlock - 1) / kShortBlock);
    switch (limb_class(B)) {
    case 2:
        if (f.hex) hipLaunchKernelGGL((k_format_short<2, true>), dim3(sgrid), dim3(kShortBlock), 0, st, f);
        else hipLaunchKernelGGL((k_format_short<2, false>), dim3(sgrid), dim3(kShortBlock), 0, st, f);
        break;
    case 4:
        if (f.hex) hipLaunchKernelGGL((k_format_short<4, true>), dim3(sgrid), dim3(kShortBlock), 0, st, f);
        else hipLaunchKernelGGL((k_format_short<4, false>), dim3(sgrid), dim3(kShortBlock), 0, st, f);
        break;
    case 8: hipLaunchKernelGGL(k_format_compact<8>, dim3(grid), dim3(kCodecBlock), lds, st, f); break;
    case 16: hipLaunchKernelGGL(k_format_compact<16>, dim3(grid), dim3(kCodecBlock), lds, st, f); break;
    default: hipLaunchKernelGGL(k_format_compact<32>, dim3(grid), dim3(kCodecBlock), lds, st, f); break;
    }
    CODECCHK(hipGetLastError());
    return UPDEC_OK;
}

}  // extern "C"
