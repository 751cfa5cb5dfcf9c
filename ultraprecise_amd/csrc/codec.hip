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

// scan of one row: fractional digits and sign
struct RowScan {
    u32 frac, neg;
};

__device__ RowScan scan_row(const char* s, u32 len)
{
    RowScan r{0u, 0u};
    u32 i = 0;
    if (len > 0 && s[0] == '-') {
        r.neg = 1u;
        i = 1;
    }
    bool dot = false;
    for (; i < len; i++) {
        char c = s[i];
        if (c == 0) break;
        if (c == '.') {
            dot = true;
            i++;
            if (i >= len || s[i] == 0) break;
            c = s[i];
        }
        if (dot) r.frac++;
    }
    return r;
}

// Rows of the long way round -- not plain (below), or cast down -- are held
// in memory, in as many limbs as they need: rolled loops over a run-time
// limb count keep this code's registers out of the kernel's, which the plain
// rows need for eight waves per SIMD.
struct WideRow {
    u32 w[32];
    u32 n;  // limbs held; the value is modulo 2^(32 n) once n has reached `most`
};

// v = v * m + add, up to `most` limbs
__device__ __forceinline__ void wide_mul_add(WideRow& v, u32 m, u32 add, u32 most)
{
    u32 c = add;
#pragma unroll 1
    for (u32 i = 0; i < v.n; i++) {
        const u64 t = (u64)v.w[i] * m + c;
        v.w[i] = (u32)t;
        c = (u32)(t >> 32);
    }
    if (c != 0u && v.n < most) v.w[v.n++] = c;
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

// to scale S: times 10^(S - frac), or floor of the division by 10^(frac - S)
__device__ void wide_cast(WideRow& v, u32 frac, u32 S, u32 most)
{
    const bool down = frac > S;
    u32 k = down ? frac - S : S - frac;
    while (k != 0u) {
        const u32 step = k < 9u ? k : 9u;
        const u32 d = pow10_word(step);
        if (down) {
            const u32 s = (u32)__builtin_clz(d);
            wide_div_word(v, d << s, s, recip_word(d << s));
        } else {
            wide_mul_add(v, d, 0u, most);
        }
        k -= step;
    }
}

// StringToDecimal and the cast, modulo 2^(32 most), nine characters a fold;
// the value is all `most` limbs of w
__device__ void wide_any(const char* s, u32 len, u32 frac, u32 S, u32 most, WideRow& v)
{
    v.n = most;
#pragma unroll 1
    for (u32 i = 0; i < most; i++) v.w[i] = 0u;
    auto fold = [&](u32 k, i64 chunk) {
        const u32 m = pow10_word(k);
        u64 c = 0;
#pragma unroll 1
        for (u32 i = 0; i < most; i++) {
            const u32 a = i == 0u ? (u32)chunk : (i == 1u ? (u32)((u64)chunk >> 32) : (chunk < 0 ? 0xffffffffu : 0u));
            const u64 t = (u64)v.w[i] * m;
            const u64 lo = (t & 0xffffffffull) + a + (c & 0xffffffffull);
            v.w[i] = (u32)lo;
            c = (t >> 32) + (lo >> 32) + (c >> 32);
        }
    };
    u32 i = (len > 0 && s[0] == '-') ? 1u : 0u;
    i64 chunk = 0;
    u32 k = 0;
    for (; i < len; i++) {
        char c = s[i];
        if (c == 0) break;
        if (c == '.') {
            i++;
            if (i >= len || s[i] == 0) break;
            c = s[i];
        }
        chunk = chunk * 10 + ((i64)(signed char)c - '0');
        if (++k == 9u) {
            fold(k, chunk);
            chunk = 0;
            k = 0;
        }
    }
    if (k) fold(k, chunk);
    wide_cast(v, frac, S, most);
}

// ---- plain rows
//
// A plain row is an optional '-', then decimal digits with at most one '.'
// among them, which is not its last character: every row that a database
// writes.  It is parsed sixteen characters at a time in registers, without a
// branch per character: the dwords covering them are realigned, the '.' is
// found and closed up, the digits are moved to the end of the sixteen bytes
// (so that the front fills with zeros) and checked, and each four become a
// number by one byte dot product.  Any other row takes the walk over
// characters above.

// The sixteen characters from s on (a byte address): the dwords that hold
// one of them and begin before `end`, the end of the text, realigned.
// Characters at and past `end` come out as anything.
__device__ __forceinline__ void load_chars16(uintptr_t s, uintptr_t end, u64& x0, u64& x1)
{
    const u32* p = reinterpret_cast<const u32*>(s & ~(uintptr_t)3);
    const u32 sh = (u32)(s & 3u);
    u32 w[5];
    if (reinterpret_cast<uintptr_t>(p + 5) <= end) {
        load_dwords<5, false>(p, w);
    } else {
#pragma unroll
        for (int k = 0; k < 5; k++) w[k] = reinterpret_cast<uintptr_t>(p + k) < end ? p[k] : 0u;
    }
    u32 t[4];
#pragma unroll
    for (int j = 0; j < 4; j++) t[j] = __builtin_amdgcn_alignbyte(w[j + 1], w[j], sh);
    x0 = ((u64)t[1] << 32) | t[0];
    x1 = ((u64)t[3] << 32) | t[2];
}

// index of the first '.' in eight characters, 8 when there is none
__device__ __forceinline__ u32 first_dot(u64 x)
{
    const u64 z = x ^ 0x2e2e2e2e2e2e2e2eull;
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
    const u32 p0 = first_dot(x0), p1 = first_dot(x1);
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
    load_chars16(s, end, x0, x1);
    neg = len > 0u && (x0 & 255u) == (u64)'-' ? 1u : 0u;
    if (neg) {
        x0 = (x0 >> 8) | (x1 << 56);
        x1 >>= 8;
    }
    const Piece q = piece16(x0, x1, len - neg);
    v = (u64)q.hi * 100000000u + q.lo;
    frac = q.dot < 16u ? len - neg - q.dot - 1u : 0u;
    return q.plain && !(q.dot < 16u && frac == 0u);
}

// A plain row of any length: its value modulo 2^(32 W)
template <int W> __device__ bool plain_long(uintptr_t s, uintptr_t end, u32 len, Mag<W>& v, u32& frac)
{
    v = mzero<W>();
    frac = 0u;
    bool dot = false, ok = true;
    for (u32 i = 0; i < len && ok; i += 16u) {
        u64 x0, x1;
        load_chars16(s + i, end, x0, x1);
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
    return ok && !(dot && frac == 0u);
}

// Any row of up to 16 characters by the rules above, one character a step;
// the value fits an int64 (|v| < 208 * 10^16 / 9)
__device__ __forceinline__ i64 short_any(uintptr_t s, uintptr_t end, u32 len, u32& frac, u32& neg)
{
    u64 x0, x1;
    load_chars16(s, end, x0, x1);
    i64 v = 0;
    bool dot = false, force = false;
    frac = neg = 0u;
#pragma unroll 1
    for (u32 i = 0; i < len; i++) {
        const u32 c = (u32)x0 & 255u;
        x0 = (x0 >> 8) | (x1 << 56);
        x1 >>= 8;
        if (i == 0u && c == (u32)'-') {
            neg = 1u;
            continue;
        }
        if (c == 0u) break;  // the row ends at its first NUL, also right after a '.'
        if (!force && c == (u32)'.') {
            dot = force = true;  // the next character is taken as a digit whatever it is
            continue;
        }
        force = false;
        frac += dot ? 1u : 0u;
        v = v * 10 + ((i32)(signed char)(char)c - '0');
    }
    return v;
}

// A plain row cast down: the division needs the whole value (modulo 2^1024,
// as the reference holds it)
__device__ void wide_plain(uintptr_t s, uintptr_t end, u32 len, u32 frac, u32 S, WideRow& v)
{
    v.n = 0u;
    for (u32 i = 0; i < len; i += 16u) {
        u64 x0, x1;
        load_chars16(s + i, end, x0, x1);
        const Piece q = piece16(x0, x1, len - i < 16u ? len - i : 16u);
        if (q.n > 8u) wide_mul_add(v, pow10_word(q.n - 8u), q.hi, 32u);
        wide_mul_add(v, pow10_word(q.n < 8u ? q.n : 8u), q.lo, 32u);
    }
    wide_cast(v, frac, S, 32u);
}

// rows per block of the ingest kernel, and of the format kernel (one wave)
constexpr int kParseBlock = 256;
constexpr int kCodecBlock = 64;

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
        const u32 len = o1 > o0 ? (u32)(o1 - o0) : 0u;
        Mag<WO> m;
        u32 neg = 0u, frac = 0u;
        bool done = false;
        const uintptr_t a = reinterpret_cast<uintptr_t>(s);
        if (len <= 16u) {
            u64 u;
            if (plain_short(a, end, len, u, frac, neg)) {
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
            } else {
                const i64 x = short_any(a, end, len, frac, neg);
                const u32 ext = x < 0 ? 0xffffffffu : 0u;
#pragma unroll
                for (int i = 0; i < WO; i++) m.w[i] = i == 0 ? (u32)(u64)x : (i == 1 ? (u32)((u64)x >> 32) : ext);
                done = S >= frac;
            }
        } else {
            neg = s[0] == '-' ? 1u : 0u;
            const u32 n = len - neg;
            done = plain_long<WO>(a + neg, end, n, m, frac);
            if (done && S < frac) {
                WideRow v;
                wide_plain(a + neg, end, n, frac, S, v);
#pragma unroll
                for (int i = 0; i < WO; i++) m.w[i] = (u32)i < v.n ? v.w[i] : 0u;
                frac = S;
            }
        }
        if (done) {
            if (S > frac) m = mul_p10_rt<WO>(m, S - frac);
        } else {
            const RowScan sc = scan_row(s, len);
            neg = sc.neg;
            WideRow v;
            wide_any(s, len, sc.frac, S, S < sc.frac ? 32u : (u32)WO, v);
#pragma unroll
            for (int i = 0; i < WO; i++) m.w[i] = v.w[i];
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

template <int W> __device__ u32 div_1e9_rem(Mag<W>& x)
{
    u32 r = 0;
#pragma unroll
    for (int i = W - 1; i >= 0; i--) x.w[i] = div_word_const<1000000000u>(r, x.w[i]);
    return r;
}

// LDS per row: the formatted slot (`slot` bytes, the longest form rounded
// to dwords) and, for text, a digit area of slot + 12 bytes (digits come in
// groups of nine, up to eight past the longest form)
template <int W>
__global__ void __launch_bounds__(kCodecBlock) k_format_compact(const u8* __restrict__ col, int64_t rows, u32 B,
                                                                u32 S, u32 hex, u32 slot, u32 stride,
                                                                char* __restrict__ out)
{
    extern __shared__ u32 tile[];
    u8* t8 = reinterpret_cast<u8*>(tile);
    const int64_t base = (int64_t)blockIdx.x * kCodecBlock;
    const int64_t row = base + threadIdx.x;
    u8* o = t8 + (u32)threadIdx.x * slot;
    for (u32 i = 0; i < slot; i++) o[i] = 0;
    if (row < rows) {
        const Dec<W> v = load_compact_rt<W>(col, (usize)row, B, (usize)rows * B);
        u32 p = 0;
        if (hex) {
            o[p++] = v.neg ? '-' : '+';
            bool lead = false;
#pragma unroll
            for (int i = W - 1; i >= 0; i--) {
                lead = lead || v.m.w[i] != 0u;
                if (lead) {
#pragma unroll
                    for (int j = 7; j >= 0; j--) {
                        const u32 nib = (v.m.w[i] >> (4 * j)) & 0xFu;
                        o[p++] = (u8)(nib < 10u ? '0' + nib : 'A' + nib - 10u);
                    }
                }
            }
            o[p++] = '(';
            o[p++] = (u8)('0' + S / 100u);
            o[p++] = (u8)('0' + S / 10u % 10u);
            o[p++] = (u8)('0' + S % 10u);
            o[p++] = ')';
        } else {
            // decimal digits, least significant first, into the digit area
            u8* dig = t8 + (u32)kCodecBlock * slot + (u32)threadIdx.x * (slot + 12u);
            Mag<W> x = v.m;
            u32 n = 0;
            while (!is_zero(x)) {
                u32 r = div_1e9_rem<W>(x);
                for (int k = 0; k < 9; k++) {
                    dig[n++] = (u8)('0' + r % 10u);
                    r /= 10u;
                }
            }
            while (n > 1 && dig[n - 1] == '0') n--;
            if (n == 0) dig[n++] = '0';
            while (n <= S) dig[n++] = '0';
            if (v.neg) o[p++] = '-';
            for (int i = (int)n - 1; i >= 0; i--) {
                o[p++] = dig[i];
                if ((u32)i == S && S > 0) o[p++] = '.';
            }
        }
    }
    __syncthreads();
    // the block's rows are consecutive stride-byte slots: dword stores,
    // zeros past each row's formatted slot
    const int64_t nrows = rows - base < kCodecBlock ? rows - base : kCodecBlock;
    const u32 sw = stride / 4, lw = slot / 4;
    const u32 nw = (u32)nrows * sw;
    u32* d = reinterpret_cast<u32*>(out + base * (int64_t)stride);
    for (u32 i = threadIdx.x; i < nw; i += kCodecBlock) {
        const u32 r = i / sw, w = i - r * sw;
        d[i] = w < lw ? tile[r * lw + w] : 0u;
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
    const u32 hex = form == UPDEC_FORMAT_HEX ? 1u : 0u;
    const u32 slot = (u32)need;
    const size_t lds = (size_t)kCodecBlock * slot + (hex ? 0 : (size_t)kCodecBlock * (slot + 12u));
    hipStream_t st = st_of(stream);
    const u32 sb = (u32)B, ss = (u32)scale, sd = (u32)stride;
    switch (limb_class(B)) {
    case 2: hipLaunchKernelGGL(k_format_compact<2>, dim3(grid), dim3(kCodecBlock), lds, st, d_col, rows, sb, ss, hex, slot, sd, d_out); break;
    case 4: hipLaunchKernelGGL(k_format_compact<4>, dim3(grid), dim3(kCodecBlock), lds, st, d_col, rows, sb, ss, hex, slot, sd, d_out); break;
    case 8: hipLaunchKernelGGL(k_format_compact<8>, dim3(grid), dim3(kCodecBlock), lds, st, d_col, rows, sb, ss, hex, slot, sd, d_out); break;
    case 16: hipLaunchKernelGGL(k_format_compact<16>, dim3(grid), dim3(kCodecBlock), lds, st, d_col, rows, sb, ss, hex, slot, sd, d_out); break;
    default: hipLaunchKernelGGL(k_format_compact<32>, dim3(grid), dim3(kCodecBlock), lds, st, d_col, rows, sb, ss, hex, slot, sd, d_out); break;
    }
    CODECCHK(hipGetLastError());
    return UPDEC_OK;
}

}  // extern "C"
