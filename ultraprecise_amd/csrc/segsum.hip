// segsum.hip -- segmented SUM of a compact decimal column
// (updec_segsum_compact, updec_segsum_compact_noalloc in include/updec.h).
//
// The reference sums a compact column per group with aggregate_column
// (src/CudaAcc/AriesEngineAlgorithm.h:832-857): rows are visited in
// `associated` order and segment s covers positions [groups[s], groups[s+1])
// (the last one up to `rows`); segreduce (kernel_segreduce.hxx:535-612)
// reduces each segment into a 133-byte nullable_type<Decimal>.
//
// Here the whole operation is two stream-ordered launches of kernels
// compiled with the library, with nothing read back to the host:
//   k_seg_main   a block takes one chunk of consecutive positions and walks
//                it in tiles.  A tile inside one segment (large groups) is
//                added to every lane's running sum.  In a tile with segment
//                starts the block sums each segment in an LDS slot, and
//                writes the images of the segments that end there, through
//                LDS, as one span of consecutive bytes.  What a chunk knows
//                only in part it leaves behind: the sum before its first
//                start (head) and the sum since its last one (tail).
//   k_seg_join   one wave per chunk boundary: the segment that is open
//                there, if it began in the chunk before, is that chunk's
//                tail and the heads of the chunks it goes on into; and the
//                +0 images of segments that start past the last position.
// No segment has an accumulator in memory, so nothing is cleared, no atomic
// leaves the CU, and the time does not depend on how many blocks meet in one
// segment.
//
// What bounds it: the loads (positions in row order are row quads, see
// dec_device.h; gathered rows cost a cache line or part of one each), and in
// tiles with starts the LDS additions and the barriers around them.  It
// replaced a form that cleared an accumulator per segment, added to it with
// 64-bit atomics (16 consecutive positions a lane, so every load touched 64
// cache lines), and wrote each image byte by byte from one lane:
//   20 M rows of DECIMAL(15,2), 6 segments, gathered   327 -> 138 us
//   12 M rows of DECIMAL(38,10), 300,000 segments      580 -> 107 us (2.2 TB/s)
//   20 M rows of DECIMAL(9,2), one segment             255 ->  30 us
//   1 M rows of DECIMAL(300,75), 10 segments           361 -> 137 us
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "../../include/updec.h"
#include "api_internal.h"
#include "dec_device.h"
#include "planner.h"

using namespace updec;

namespace {

#define SEGCHK(expr)                                                                                          \
    do {                                                                                                      \
        hipError_t e_ = (expr);                                                                               \
        if (e_ != hipSuccess) return api_fail(UPDEC_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

constexpr int kSegThreads = 256;
// segments summed in LDS at a time
constexpr int kSegSlots = 64;

struct SegArgs {
    const u8* col;
    usize colbytes;
    u32 B;
    u32 P, S;
    i32 ngroups;
    const i32* assoc;   // positions gathered through it, or null: position i is row i
    const i32* groups;  // segment starts
    i64 rows;
    i64 chunk;          // positions of a block
    u32* head;          // per chunk, AW limbs: the sum before its first start
    u32* tail;          // per chunk, AW limbs: the sum since its last start
    u8* out;
};

// Sums are two's complement of AW = W + 1 limbs: at most 2^31 magnitudes
// below 2^(32 W - 1).  In an LDS slot a sum is K words of 64 bits holding 48
// bits each, the last one all the bits above: a word takes 2^15 additions,
// more than a tile has positions and lanes, before it would overflow.
template <int W> struct SegSum {
    static constexpr int AW = W + 1;
    static constexpr int K = (32 * AW - 64 + 47) / 48 + 1;
    // positions a lane takes of a tile
    static constexpr int R = W <= 4 ? 4 : W == 8 ? 2 : 1;
};

// the 48-bit words of a two's complement sum
template <int W> __device__ __forceinline__ u64 seg_word(const Mag<SegSum<W>::AW>& m, int k)
{
    constexpr int AW = SegSum<W>::AW;
    const u32 ext = (u32)((i32)m.w[AW - 1] >> 31);
    const int b = 48 * k / 32;
    auto limb = [&](int i) { return i < AW ? m.w[i] : ext; };
    const u64 two = ((u64)limb(b + 1) << 32) | limb(b);
    if (k == SegSum<W>::K - 1) return (k & 1) ? (two >> 16) | ((u64)limb(b + 2) << 48) : two;
    return (k & 1) ? two >> 16 : two & 0xffffffffffffull;
}

template <int W> __device__ __forceinline__ void seg_slot_add(u64* slot, const Mag<SegSum<W>::AW>& m)
{
#pragma unroll
    for (int k = 0; k < SegSum<W>::K; k++)
        atomicAdd(reinterpret_cast<unsigned long long*>(slot + k), (unsigned long long)seg_word<W>(m, k));
}

template <int W> __device__ __forceinline__ Mag<SegSum<W>::AW> seg_slot_value(const u64* slot)
{
    constexpr int AW = SegSum<W>::AW, K = SegSum<W>::K;
    u64 piece[K + 1];
    i64 c = 0;
#pragma unroll
    for (int k = 0; k < K; k++) {
        const i64 t = (i64)slot[k] + c;
        piece[k] = k < K - 1 ? (u64)t & 0xffffffffffffull : (u64)t;
        c = t >> 48;
    }
    piece[K] = 0;
    Mag<AW> m;
#pragma unroll
    for (int i = 0; i < AW; i++) {
        const int k = 32 * i / 48, sh = 32 * i % 48;  // sh: 0, 32, 16
        if (k >= K - 1) m.w[i] = (u32)(piece[K - 1] >> (32 * i - 48 * (K - 1)));
        else m.w[i] = (u32)(piece[k] >> sh) | (sh == 32 ? (u32)(piece[k + 1] << 16) : 0u);
    }
    return m;
}

// starts at or before position p, of n ascending ones; the whole wave takes
// part, 64 probes a step, and gets the result
__device__ __forceinline__ i32 seg_upper_bound(const i32* g, i32 n, i64 p)
{
    const i32 lane = (i32)(threadIdx.x & 63u);
    i32 lo = 0, len = n;
    while (len > 0) {
        const i32 step = (len + 63) >> 6;
        const i64 i = (i64)lane * step;
        const bool le = i < len && (i64)g[lo + (i32)i] <= p;
        const i32 c = __popcll(__ballot(le));
        if (c == 0) break;
        lo += (c - 1) * step + 1;
        const i32 rest = len - ((c - 1) * step + 1);
        len = rest < step - 1 ? rest : step - 1;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

template <int AW> __device__ __forceinline__ void seg_store(u32* p, const Mag<AW>& m)
{
#pragma unroll
    for (int w = 0; w < AW; w++) p[w] = m.w[w];
}

// CB: the row bytes when they are a compile-time constant (positions in row
// order, row quads), 0 for a run-time width
template <int W, int CB, bool GATHER> __global__ void __launch_bounds__(kSegThreads) k_seg_main(SegArgs a)
{
    constexpr int AW = SegSum<W>::AW, K = SegSum<W>::K, R = SegSum<W>::R;
    constexpr i64 TILE = (i64)kSegThreads * R;
    constexpr int IMG = (kSegSlots * 133 + 3) / 4;
    __shared__ u64 slots[(kSegSlots + 1) * K];
    __shared__ u32 img[IMG];
    __shared__ i64 st[kSegSlots];
    __shared__ i32 s_n;
    const i32 tid = (i32)threadIdx.x;
    const i64 c0 = (i64)blockIdx.x * a.chunk;
    const i64 c1 = c0 + a.chunk < a.rows ? c0 + a.chunk : a.rows;
    // the segment open before the chunk (-1: none)
    i32 s = seg_upper_bound(a.groups, a.ngroups, c0 - 1) - 1;
    bool first = true;  // no start seen yet: the open segment began before the chunk
    Mag<AW> acc = mzero<AW>();
    for (i64 p0 = c0; p0 < c1; p0 += TILE) {
        const i64 p1 = p0 + TILE < c1 ? p0 + TILE : c1;
        // Rows in order: R consecutive positions a lane.  Gathered: positions
        // kSegThreads apart, so that the lanes of one load read neighbouring
        // indices, whose rows share cache lines where the indices ascend, as a
        // stable sort's permutation does within a segment (20 M rows, 6
        // segments: 138 us against 380 with four consecutive indices a lane)
        constexpr int STEP = GATHER ? kSegThreads : 1;
        const i64 mine = p0 + (GATHER ? (i64)tid : (i64)tid * R);
        const i64 next = s + 1 < a.ngroups ? (i64)a.groups[s + 1] : a.rows;
        Dec<W> v[R];
#pragma unroll
        for (int r = 0; r < R; r++) v[r].m = mzero<W>(), v[r].neg = 0u;
        if (mine < p1) {
            if constexpr (GATHER) {
                u32 row[R];
#pragma unroll
                for (int r = 0; r < R; r++) row[r] = mine + r * STEP < p1 ? (u32)a.assoc[mine + r * STEP] : 0u;
#pragma unroll
                for (int r = 0; r < R; r++)
                    if (mine + r * STEP < p1) v[r] = load_compact_rt<W, false>(a.col, (usize)row[r], a.B, a.colbytes);
            } else if constexpr (CB != 0) {
                static_assert(R == 4 && (CB + 3) / 4 <= W, "row quads");
                const Quad<CB> q = load_quad<CB>(a.col, (usize)mine >> 2, a.colbytes);
#pragma unroll
                for (int r = 0; r < R; r++)
                    if (mine + r < p1) v[r] = dresize<W>(quad_row<CB>(q, (u32)r));
            } else {
#pragma unroll
                for (int r = 0; r < R; r++)
                    if (mine + r < p1) v[r] = load_compact_rt<W>(a.col, (usize)(mine + r), a.B, a.colbytes);
            }
        }
        if (next >= p1) {
            // inside one segment
            if (s >= 0) {
#pragma unroll
                for (int r = 0; r < R; r++) acc_add<AW, W>(acc, v[r]);
            }
            continue;
        }
        i64 lo = p0;
        for (;;) {
            __syncthreads();
            // a window of the starts after s: slot 0 is segment s, slot j
            // the segment of the j-th start
            if (tid < kSegSlots) {
                const i64 x = (i64)s + 1 + tid < a.ngroups ? (i64)a.groups[s + 1 + tid] : a.rows;
                const i32 m = __popcll(__ballot(x < p1));
                st[tid] = x;
                if (tid == 0) s_n = m;
            }
            for (int i = tid; i < (kSegSlots + 1) * K; i += kSegThreads) slots[i] = 0;
            for (int i = tid; i < IMG; i += kSegThreads) img[i] = 0;
            __syncthreads();
            const i32 n = s_n;
            const bool whole = n < kSegSlots;  // the window holds every start of the tile
            const i64 hi = whole ? p1 : st[kSegSlots - 1];
            u32 any = 0;
#pragma unroll
            for (int w = 0; w < AW; w++) any |= acc.w[w];
            if (any && s >= 0) seg_slot_add<W>(slots, acc);
            acc = mzero<AW>();
            // the lane's rows, one addition per segment they lie in
            i32 cur = -1;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const i64 p = mine + r * STEP;
                if (p < lo || p >= hi) continue;
                i32 j = cur;
                if (j < 0) {
                    i32 x = 0, y = n;
                    while (x < y) {
                        const i32 mid = (x + y) >> 1;
                        if (st[mid] <= p) x = mid + 1;
                        else y = mid;
                    }
                    j = x;
                } else {
                    while (j < n && st[j] <= p) j++;
                }
                if (j != cur) {
                    if (cur > 0 || (cur == 0 && s >= 0)) seg_slot_add<W>(slots + cur * K, acc);
                    acc = mzero<AW>();
                    cur = j;
                }
                acc_add<AW, W>(acc, v[r]);
            }
            if (cur > 0 || (cur == 0 && s >= 0)) seg_slot_add<W>(slots + cur * K, acc);
            acc = mzero<AW>();
            __syncthreads();
            // slots 0 .. n-1 have ended: their images, and the head in
            // place of slot 0's where that segment began before the chunk
            const bool skip0 = s < 0 || first;
            if (tid < n) {
                const Mag<AW> m = seg_slot_value<W>(slots + tid * K);
                if (tid > 0 || !skip0) {
                    const Dec<AW> d = sum_value<AW>(m);
                    u8* o = reinterpret_cast<u8*>(img) + tid * 133;
                    o[0] = 1;
                    o[1] = (u8)d.neg;
                    o[2] = (u8)a.P;
                    o[3] = (u8)a.S;
#pragma unroll
                    for (int w = 0; w < (AW < 32 ? AW : 32); w++) {
                        o[5 + 4 * w] = (u8)d.m.w[w];
                        o[6 + 4 * w] = (u8)(d.m.w[w] >> 8);
                        o[7 + 4 * w] = (u8)(d.m.w[w] >> 16);
                        o[8 + 4 * w] = (u8)(d.m.w[w] >> 24);
                    }
                } else if (s >= 0) {
                    seg_store<AW>(a.head + (usize)blockIdx.x * AW, m);
                }
            }
            if (whole && tid == 0) acc = seg_slot_value<W>(slots + n * K);  // the open segment
            __syncthreads();
            const i32 f = skip0 ? 1 : 0;
            if (n > f) {
                // bytes [f 133, n 133) of img to consecutive images
                const u8* src = reinterpret_cast<const u8*>(img) + f * 133;
                u8* dst = a.out + ((usize)s + (usize)f) * 133u;
                const u32 len = (u32)(n - f) * 133u;
                const u32 pre = (u32)(-(usize)dst & 3u);
                const u32 words = (len - pre) >> 2;
                for (u32 i = (u32)tid; i < words; i += kSegThreads) {
                    u32 x;
                    __builtin_memcpy(&x, src + pre + 4u * i, 4);
                    reinterpret_cast<u32*>(dst + pre)[i] = x;
                }
                const u32 rest = len - pre - 4u * words;
                if ((u32)tid < pre) dst[tid] = src[tid];
                if ((u32)tid < rest) dst[pre + 4u * words + (u32)tid] = src[pre + 4u * words + (u32)tid];
            }
            if (n > 0) first = false;
            s += n;
            if (whole) break;
            lo = hi;
        }
    }
    // what is open at the end
    __syncthreads();
    u32* red = img;
    wave_reduce<AW>(acc);
    if ((tid & 63) == 0) seg_store<AW>(red + (tid >> 6) * AW, acc);
    __syncthreads();
    if (tid == 0) {
        for (int wv = 1; wv < kSegThreads / 64; wv++) {
            Mag<AW> o;
#pragma unroll
            for (int w = 0; w < AW; w++) o.w[w] = red[wv * AW + w];
            add_to<AW>(acc, acc, o);
        }
        seg_store<AW>((first ? a.head : a.tail) + (usize)blockIdx.x * AW, acc);
    }
}

template <int W> __global__ void __launch_bounds__(64) k_seg_join(SegArgs a, i32 nchunks)
{
    constexpr int AW = SegSum<W>::AW;
    const i32 lane = (i32)threadIdx.x;
    const i32 b = (i32)blockIdx.x + 1;  // the boundary after chunk b - 1
    if (b <= nchunks) {
        const i64 at = (i64)b * a.chunk < a.rows ? (i64)b * a.chunk : a.rows;
        const i32 s = seg_upper_bound(a.groups, a.ngroups, at - 1) - 1;
        if (s >= 0 && (i64)a.groups[s] >= (i64)(b - 1) * a.chunk) {
            const i64 end = s + 1 < a.ngroups ? (i64)a.groups[s + 1] : a.rows;
            Mag<AW> acc = mzero<AW>();
            if (lane == 0)
#pragma unroll
                for (int w = 0; w < AW; w++) acc.w[w] = a.tail[(usize)(b - 1) * AW + w];
#pragma unroll 4
            for (i32 k = b + lane; k < nchunks; k += 64) {
                if ((i64)k * a.chunk >= end) break;
                Mag<AW> o;
#pragma unroll
                for (int w = 0; w < AW; w++) o.w[w] = a.head[(usize)k * AW + w];
                add_to<AW>(acc, acc, o);
            }
            wave_reduce<AW>(acc);
            if (lane == 0) write_sum_image<AW>(a.out + (usize)s * 133u, acc, a.P, a.S, 0u);
        }
    }
    // segments that start past the last position are +0
    const i32 s0 = seg_upper_bound(a.groups, a.ngroups, a.rows - 1);
    for (i64 s = (i64)s0 + (i64)blockIdx.x * 64 + lane; s < a.ngroups; s += (i64)gridDim.x * 64)
        write_sum_image<AW>(a.out + (usize)s * 133u, mzero<AW>(), a.P, a.S, 0u);
}

// width class of a compact row of B bytes: limbs W >= ceil(B / 4)
int seg_class_words(int B)
{
    return B <= 8 ? 2 : B <= 16 ? 4 : B <= 32 ? 8 : B <= 64 ? 16 : B <= 128 ? 32 : 0;
}

int seg_check(const uint8_t* d_col, int precision, int64_t rows, const int32_t* d_groups, int32_t ngroups,
              uint8_t* d_out, int* B, int* W)
{
    if (rows < 0 || ngroups < 0 || (ngroups && (!d_groups || !d_out)) || (rows && !d_col) || precision <= 0)
        return api_fail(UPDEC_EINVAL, "bad argument");
    if (rows > (int64_t)INT32_MAX + 1)
        return api_fail(UPDEC_EINVAL, "positions are int32 (associated, groups): at most 2^31 rows");
    *B = compact_bytes(precision);
    *W = seg_class_words(*B);
    if (!*W) return api_fail(UPDEC_EUNSUPPORTED, "rows wider than 128 bytes (the 32-limb Decimal) are not summed");
    return UPDEC_OK;
}

// positions of a block: about eight blocks a CU (what the LDS slots and
// registers of the narrow widths allow to be resident), in whole tiles
i64 seg_chunk(i64 rows)
{
    const i64 per = (rows + (i64)api_device_cus() * 8 - 1) / ((i64)api_device_cus() * 8);
    return std::max<i64>(1024, (per + 1023) / 1024 * 1024);
}

i64 seg_chunks(i64 rows) { return rows > 0 ? (rows + seg_chunk(rows) - 1) / seg_chunk(rows) : 0; }

// 64-bit words of scratch: a head and a tail of W + 1 limbs per chunk
usize seg_scratch_words(i64 rows, int W) { return (usize)seg_chunks(rows) * (usize)(W + 1) + 1; }

template <int W> void seg_main_launch(const SegArgs& a, i64 n, hipStream_t st)
{
#define UPD_SEG(CB, G) hipLaunchKernelGGL((k_seg_main<W, CB, G>), dim3((unsigned)n), dim3(kSegThreads), 0, st, a)
    // Gathered rows are loaded one by one at their run-time width.  Rows in
    // order are loaded as quads, whose decoding needs the width at compile
    // time, up to 16 bytes; wider ones row by row.
    if (a.assoc) {
        UPD_SEG(0, true);
        return;
    }
    if constexpr (W == 2) {
        switch (a.B) {
        case 1: UPD_SEG(1, false); return;
        case 2: UPD_SEG(2, false); return;
        case 3: UPD_SEG(3, false); return;
        case 4: UPD_SEG(4, false); return;
        case 5: UPD_SEG(5, false); return;
        case 6: UPD_SEG(6, false); return;
        case 7: UPD_SEG(7, false); return;
        default: UPD_SEG(8, false); return;
        }
    } else if constexpr (W == 4) {
        switch (a.B) {
        case 9: UPD_SEG(9, false); return;
        case 10: UPD_SEG(10, false); return;
        case 11: UPD_SEG(11, false); return;
        case 12: UPD_SEG(12, false); return;
        case 13: UPD_SEG(13, false); return;
        case 14: UPD_SEG(14, false); return;
        case 15: UPD_SEG(15, false); return;
        default: UPD_SEG(16, false); return;
        }
    } else {
        UPD_SEG(0, false);
    }
#undef UPD_SEG
}

template <int W> int seg_launch_w(SegArgs a, u32* scratch, hipStream_t st)
{
    constexpr int AW = SegSum<W>::AW;
    const i64 n = seg_chunks(a.rows);
    a.chunk = seg_chunk(a.rows);
    a.head = scratch;
    a.tail = scratch + (usize)n * AW;
    if (n > 0) {
        seg_main_launch<W>(a, n, st);
        SEGCHK(hipGetLastError());
    }
    const i64 grid = std::max<i64>(n, std::min<i64>(((i64)a.ngroups + 63) / 64, 512));
    hipLaunchKernelGGL(k_seg_join<W>, dim3((unsigned)grid), dim3(64), 0, st, a, (i32)n);
    SEGCHK(hipGetLastError());
    return UPDEC_OK;
}

int seg_launch(const uint8_t* d_col, int P, int S_, int B, int W, int64_t rows, const int32_t* d_assoc,
               const int32_t* d_groups, int32_t ngroups, uint8_t* d_out, u64* scratch, hipStream_t st)
{
    SegArgs a{};
    a.col = d_col;
    a.colbytes = (usize)rows * (usize)B;
    a.B = (u32)B;
    a.P = (u32)P & 0xffu;
    a.S = (u32)S_ & 0xffu;
    a.ngroups = ngroups;
    a.assoc = d_assoc;
    a.groups = d_groups;
    a.rows = rows;
    a.out = d_out;
    u32* sc = reinterpret_cast<u32*>(scratch);
    switch (W) {
    case 2: return seg_launch_w<2>(a, sc, st);
    case 4: return seg_launch_w<4>(a, sc, st);
    case 8: return seg_launch_w<8>(a, sc, st);
    case 16: return seg_launch_w<16>(a, sc, st);
    default: return seg_launch_w<32>(a, sc, st);
    }
}

// ------------------------------------------------------------------ fixed scratch of the no-alloc entry point

// Scratch of updec_segsum_compact_noalloc: 8 MiB on every device the library
// runs on, held until the process ends.  A call needs a head and a tail per
// chunk (at most 8 chunks a CU while rows < 2^31, so 0.6 MB at 32 limbs); the
// entry point's limit on segments is what the array held when every segment
// had an accumulator of W + 2 words, and stays.  The array's name is a host
// stand-in; kernels get the device address from hipGetSymbolAddress.
constexpr usize kSegScratchWords = (usize)1 << 20;
__device__ __align__(256) u64 scratch[kSegScratchWords];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
u64* g_scratch_ptr[kMaxDevices] = {};

int scratch_for_current_device(u64** out)
{
    int dev = 0;
    SEGCHK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return api_fail(UPDEC_EUNSUPPORTED, "device index beyond the scratch table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        SEGCHK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        g_scratch_ptr[dev] = static_cast<u64*>(p);
    }
    *out = g_scratch_ptr[dev];
    return UPDEC_OK;
}

}  // namespace

namespace updec {
// set-up of the no-alloc entry point's scratch on the current device (called
// by updec_init)
int segsum_scratch_setup()
{
    u64* p = nullptr;
    return scratch_for_current_device(&p);
}
}  // namespace updec

extern "C" {

int updec_segsum_compact(const uint8_t* d_col, int precision, int scale, int64_t rows, const int32_t* d_associated,
                         const int32_t* d_groups, int32_t ngroups, uint8_t* d_out, int mode, updec_stream_t stream)
{
    (void)mode;  // a sum is the same in both modes: the image keeps 32 limbs
    int B = 0, W = 0;
    int rc = seg_check(d_col, precision, rows, d_groups, ngroups, d_out, &B, &W);
    if (rc != UPDEC_OK || ngroups == 0) return rc;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    u64* acc = nullptr;
    SEGCHK(hipMallocAsync(reinterpret_cast<void**>(&acc), seg_scratch_words(rows, W) * sizeof(u64), st));
    rc = seg_launch(d_col, precision, scale, B, W, rows, d_associated, d_groups, ngroups, d_out, acc, st);
    const hipError_t fe = hipFreeAsync(acc, st);
    if (rc != UPDEC_OK) return rc;
    if (fe != hipSuccess) return api_fail(UPDEC_EHIP, std::string("hipFreeAsync: ") + hipGetErrorString(fe));
    return UPDEC_OK;
}

int updec_segsum_compact_noalloc(const uint8_t* d_col, int precision, int scale, int64_t rows,
                                 const int32_t* d_associated, const int32_t* d_groups, int32_t ngroups, uint8_t* d_out,
                                 int mode, updec_stream_t stream)
{
    (void)mode;
    int B = 0, W = 0;
    int rc = seg_check(d_col, precision, rows, d_groups, ngroups, d_out, &B, &W);
    if (rc != UPDEC_OK || ngroups == 0) return rc;
    const usize need = (usize)ngroups * (W + 2);
    if (need > kSegScratchWords)
        return api_fail(UPDEC_EINVAL, "too many segments for the fixed scratch: at most " +
                                          std::to_string(kSegScratchWords / (W + 2)) + " at this precision");
    u64* acc = nullptr;
    rc = scratch_for_current_device(&acc);
    if (rc != UPDEC_OK) return rc;
    return seg_launch(d_col, precision, scale, B, W, rows, d_associated, d_groups, ngroups, d_out, acc,
                      reinterpret_cast<hipStream_t>(stream));
}

int updec_segsum_noalloc_max_segments(int precision, int32_t* max_segments)
{
    if (precision <= 0 || !max_segments) return api_fail(UPDEC_EINVAL, "bad argument");
    const int W = seg_class_words(compact_bytes(precision));
    if (!W) return api_fail(UPDEC_EUNSUPPORTED, "rows wider than 128 bytes (the 32-limb Decimal) are not summed");
    *max_segments = (int32_t)(kSegScratchWords / (W + 2));
    return UPDEC_OK;
}

}  // extern "C"
