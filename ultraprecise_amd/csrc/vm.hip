// vm.hip -- the precompiled decimal interpreter and its batch launcher
// (include/updec.h, "interpreter and batches").
//
// Kernels: one persistent k_vm_sum<W> per register width class.  Its
// blocks take work items (a row range of one query) from a per-class
// counter, evaluate the query's register program for every row, fold the
// materialized result into a per-lane two's complement accumulator and
// write one partial per item; k_vm_final adds a query's partials in item
// order and writes the SUM image and COUNT.  A batch of many queries is one
// set of launches (captured once into a HIP graph, the classes on parallel
// branches), a single query is the same launches with one query.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <set>
#include <string>
#include <vector>

#include "../../include/updec.h"
#include "api_internal.h"
#include "dec_device.h"
#include "planner.h"
#include "vm.h"
#include "vm_device.h"
#include "vm_wide.h"

using namespace updec;
using namespace updec_vm;

namespace {

#define VMCHK(expr)                                                                                          \
    do {                                                                                                     \
        hipError_t e_ = (expr);                                                                              \
        if (e_ != hipSuccess) return api_fail(UPDEC_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

constexpr int kBlock[kFirstMultiLane] = {256, 256, 128, 64, 64};

template <int W> constexpr int class_of()
{
    return W == 2 ? 0 : W == 4 ? 1 : W == 8 ? 2 : W == 16 ? 3 : 4;
}

template <int W, int T>
__global__ void __launch_bounds__(T)
    k_vm_sum(Header* h, const Query* qs, const u32* prog, const u32* cst, const Item* items, u32* partials)
{
    constexpr int CLS = class_of<W>();
    constexpr int AW = W + 2;
    constexpr int NWAVE = T / 64;
    __shared__ u32 s_item;
    __shared__ u32 red[NWAVE * AW];
    __shared__ u32 regs[kClassRegs[CLS] * (W + 1) * T];
    const u32 tid = threadIdx.x;
    RegFile<W, T> R{regs + tid};
    const u32 n = h->class_nitems[CLS];
    const u32 i0 = h->class_item0[CLS];
    for (;;) {
        // The barrier first: the thread-0 work that ends one iteration (the
        // partial) and the thread-0 atomic that starts the next must stay
        // separated by a barrier.  Without one the compiler may merge the
        // two thread-0 regions into a divergent exit of the item loop, and
        // the other lanes of wave 0 re-enter the loop (and its barriers)
        // ahead of thread 0, re-reading an item number only thread 0 can
        // advance.  It also orders the reads of s_item and red of the last
        // iteration before they are written again.
        __syncthreads();
        if (tid == 0) s_item = atomicAdd(&h->counter[CLS], 1u);
        __syncthreads();
        const u32 it = __builtin_amdgcn_readfirstlane(s_item);
        if (it >= n) break;
        const Item I = items[i0 + it];
        const Query* q = qs + I.query;
        const u32* qp = prog + 3u * q->ins_off;
        const u32* qc = cst + q->const_off;
        const u32 ob = q->outB;
        Mag<AW> acc = mzero<AW>();
        for (usize row = I.row0 + tid; row < I.row1; row += T) {
            const Dec<W> v = vm_eval<W>(q, qp, qc, row, R);
            acc_add<AW, W>(acc, stored_rt<W>(v, ob));
        }
        wave_reduce<AW>(acc);
        if ((tid & 63u) == 0) {
#pragma unroll
            for (int w = 0; w < AW; w++) red[(tid >> 6) * AW + w] = acc.w[w];
        }
        __syncthreads();
        if (tid == 0) {
            Mag<AW> t = mzero<AW>();
            for (int wv = 0; wv < NWAVE; wv++) {
                Mag<AW> o;
#pragma unroll
                for (int w = 0; w < AW; w++) o.w[w] = red[wv * AW + w];
                add_to<AW>(t, t, o);
            }
            u32* dst = partials + (usize)(i0 + it) * kMaxAccWords;
#pragma unroll
            for (int w = 0; w < AW; w++) dst[w] = t.w[w];
        }
    }
}

// ---------------------------------------------------------------- wide classes

// Persistent kernel of the classes of 64 limbs and more (vm_wide.h): a block
// is one wave, an item's rows are taken 64 at a time, one lane each, with
// every value in the block's workspace.
//
// What bounds it: the workspace, whose lines mostly do not stay in L2 (a wave's
// live values are some 64 KB; counters at DECIMAL(300,100): 4 TB/s read and
// written past L2, 80 % of the wave time waiting).  The form it replaced spread
// every value over 16 to 64 lanes at the program's worst-case width: a batch
// of 32 queries of the serving stream, 50 M rows, 470 -> 41 ms.  1.2 M rows of
// "((((c-c)*a)*((a/c)*(c/a)))+(b+((b/(a-a))/c)))" at DECIMAL(300,100), a
// 256-limb program, at two waves a CU 7.1 ms, at four 4.3, at eight 3.0, at
// ten and twelve 2.6.
constexpr u32 kSumLimbs = 512;   // of the accumulators at a time
__global__ void __launch_bounds__(64, 3)
    k_vm_sum_wide(Header* h, const Query* qs, const u32* prog, const u32* cst, const Item* items, u32* partials)
{
    __shared__ u32 s_item;
    __shared__ wide::Slots slots;
    __shared__ i64 csum[kSumLimbs];
    const u32 lane = threadIdx.x;
    if (blockIdx.x >= h->wide_blocks) return;
    wide::gu8* const ws = (wide::gu8*)h->workspace + (usize)blockIdx.x * (usize)h->stride;
    u32 n = 0;
    for (int c = kFirstMultiLane; c < kNumClasses; c++) n += h->class_nitems[c];
    const u32 i0 = h->class_item0[kFirstMultiLane];
    for (;;) {
        // as in k_vm_sum: the barrier keeps thread 0's item fetch apart from
        // its partial write of the previous iteration
        __syncthreads();
        if (lane == 0) s_item = atomicAdd(&h->counter[kFirstMultiLane], 1u);
        __syncthreads();
        const u32 it = __builtin_amdgcn_readfirstlane(s_item);
        if (it >= n) break;
        const Item I = items[i0 + it];
        const Query* q = qs + I.query;
        const u32* qp = prog + 3u * q->ins_off;
        const u32* qc = cst + q->const_off;
        const u32 W = (u32)kClassW[0] << q->wclass;
        const u32 na = wide::kword(qp, wide::kHeadAcc);
        const u32 off = 4u * lane;
        const wide::Dst pos{ws + (usize)wide::kword(qp, wide::kHeadPos) * wide::kRow, off};
        const wide::Dst neg{ws + (usize)wide::kword(qp, wide::kHeadNeg) * wide::kRow, off};
        for (u32 i = 0; i < na; i++) {
            pos.put(i, 0u);
            neg.put(i, 0u);
        }
        for (usize r0 = I.row0; r0 < I.row1; r0 += 64u) {
            // lanes past the item's end repeat its last row, uncounted
            const bool active = r0 + lane < I.row1;
            u32 sign;
            const wide::Src v = wide::eval(q, qp, qc, W, ws, &slots, active ? r0 + lane : I.row1 - 1u, sign);
            wide::accumulate(v, sign, active, q->outB, pos, neg);
        }
        __syncthreads();
        // limb by limb over the lanes, then a carry pass
        u32* dst = partials + (usize)(i0 + it) * kMaxAccWords;
        i64 c = 0;
        for (u32 w0 = 0; w0 < na; w0 += kSumLimbs) {
            const u32 m = na - w0 < kSumLimbs ? na - w0 : kSumLimbs;
            for (u32 w = lane; w < m; w += 64u) {
                const u32* a = (const u32*)(pos.b + (usize)(w0 + w) * wide::kRow);
                const u32* b = (const u32*)(neg.b + (usize)(w0 + w) * wide::kRow);
                i64 s = 0;
                for (u32 k = 0; k < 64u; k += 4u) {
                    u32 x[4], y[4];
                    load_dwords<4, false>(a + k, x);
                    load_dwords<4, false>(b + k, y);
#pragma unroll
                    for (int t = 0; t < 4; t++) s += (i64)x[t] - (i64)y[t];
                }
                csum[w] = s;
            }
            __syncthreads();
            // every lane follows the carries, lane 0 writes
            for (u32 w = 0; w < m; w++) {
                const i64 t = csum[w] + c;
                if (lane == 0 && w0 + w < W + 2u) dst[w0 + w] = (u32)t;
                c = t >> 32;
            }
            __syncthreads();
        }
        for (u32 w = na + lane; w < W + 2u; w += 64u) dst[w] = (u32)c;
    }
}

// SUM image and COUNT of every query.  Lanes take the words of the items'
// partials (consecutive words of an item, as many items at once as fit a
// wave), waves take items in turn; the words are added without carries as
// 64-bit sums, then one carry pass, and the image gets the low 32 limbs of
// the magnitude.  A query of many items has several blocks, each for a
// contiguous part of them; the one that ends last adds their sums, which the
// others left in their first two items' places.
//
// What bounds it: latency of the partials' loads.  With one wave per query,
// walking the items one after the other, 7,800 partials of a 256-limb query
// took 6 ms; the 12,000 partials of such a query at 9 M rows took one block of
// 16 waves 1.6 ms, several 0.19.  Up to
// 1,000 items a query stays with one block: two that share 391 items take 7 us
// longer for handing over.
constexpr int kFinalThreads = 1024, kFinalAhead = 4;
constexpr u32 kFinalSlices = 16, kSliceItems = 512;   // blocks a query at most, items a block at least
constexpr u32 kFinalBlocks = 2048;                    // of all queries, where one a query are fewer
UPD_DEV u64* slice_sums(u32* partials, const Query* q, u32 y, u32 n)
{
    return reinterpret_cast<u64*>(partials + (usize)(q->item0 + (u32)((u64)q->nitems * y / n)) * kMaxAccWords);
}
__global__ void __launch_bounds__(kFinalThreads) k_vm_final(const Header* h, Query* qs, u32* partials)
{
    __shared__ u64 cs[kMaxAccWords];
    __shared__ u32 s_last;
    const u32 qi = blockIdx.x, tid = threadIdx.x, y = blockIdx.y;
    if (qi >= h->nqueries) return;
    Query* q = qs + qi;
    const u32 parts = q->nitems / kSliceItems, n = parts < 1u ? 1u : parts < gridDim.y ? parts : gridDim.y;
    if (y >= n) return;
    const u32 aw = ((u32)kClassW[0] << q->wclass) + 2u;
    for (u32 w = tid; w < aw; w += kFinalThreads) cs[w] = 0;
    __syncthreads();
    // words a row of lanes takes of one item, and the rows of the block
    u32 wide = 4;
    while (wide < aw && wide < 64u) wide <<= 1;
    const u32 rows = kFinalThreads / wide, row = tid / wide;
    const u32 k0 = (u32)((u64)q->nitems * y / n), k1 = (u32)((u64)q->nitems * (y + 1u) / n);
    const u32* base = partials + (usize)q->item0 * kMaxAccWords;
    for (u32 w = tid % wide; w < aw; w += wide) {
        u64 s = 0;
        for (u32 k = k0 + row; k < k1; k += rows * kFinalAhead) {
#pragma unroll
            for (u32 t = 0; t < (u32)kFinalAhead; t++)
                if (k + t * rows < k1) s += base[(usize)(k + t * rows) * kMaxAccWords + w];
        }
        if (s) atomicAdd(reinterpret_cast<unsigned long long*>(&cs[w]), (unsigned long long)s);
    }
    __syncthreads();
    if (n > 1u) {
        u64* mine = slice_sums(partials, q, y, n);
        for (u32 w = tid; w < aw; w += kFinalThreads) __hip_atomic_store(mine + w, cs[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __threadfence();
        __syncthreads();
        if (tid == 0) s_last = __hip_atomic_fetch_add(&q->done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1u == n ? 1u : 0u;
        __syncthreads();
        if (!s_last) return;
        __threadfence();
        for (u32 w = tid; w < aw; w += kFinalThreads) {
            u64 s = 0;
            for (u32 k = 0; k < n; k++) s += __hip_atomic_load(slice_sums(partials, q, k, n) + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            cs[w] = s;
        }
        __syncthreads();
    }
    if (tid == 0) {
        u64 c = 0;
        for (u32 w = 0; w < aw; w++) {
            const u64 t = cs[w] + c;
            cs[w] = (u32)t;
            c = t >> 32;
        }
        const bool neg = ((u32)cs[aw - 1u] >> 31) != 0u;
        // magnitude of the two's complement value
        u64 cc = neg ? 1u : 0u;
        const u32 fm = neg ? 0xffffffffu : 0u;
        u8* o = q->image;
        o[0] = 1;
        o[1] = neg ? 1 : 0;
        o[2] = (u8)(q->outP & 0xffu);
        o[3] = (u8)(q->outS & 0xffu);
        o[4] = 0;
        for (u32 w = 0; w < 32u; w++) {
            const u64 t = (u64)(w < aw ? (u32)cs[w] ^ fm : 0u) + (w < aw ? cc : 0u);
            const u32 x = (u32)t;
            cc = t >> 32;
            o[5 + 4 * w + 0] = (u8)x;
            o[5 + 4 * w + 1] = (u8)(x >> 8);
            o[5 + 4 * w + 2] = (u8)(x >> 16);
            o[5 + 4 * w + 3] = (u8)(x >> 24);
        }
        *q->count = (int64_t)q->rows;
    }
}

// ---------------------------------------------------------------- staging

// A batch's tables (header, queries, items, programs, constants) from pinned
// host memory to the device in one launch, 16 bytes a thread.  As five copies
// of a few KB they took 55 us before the first kernel started, most of it
// between the copies: with this and without the graph's empty branches one
// query of 700 rows at 8 limbs went from 121 to 30 us, ten queries on four
// kernels from 1666 to 1606.
constexpr int kTables = 5;
struct Staging {
    const uint4* src[kTables];
    uint4* dst[kTables];
    u32 end[kTables];   // of each table, in the 16-byte words of all
};
__global__ void __launch_bounds__(256) k_vm_stage(Staging t)
{
    const u32 i = blockIdx.x * 256u + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kTables; k++) {
        const u32 b = k ? t.end[k - 1] : 0u;
        if (i >= b && i < t.end[k]) t.dst[k][i - b] = t.src[k][i - b];
    }
}

// ---------------------------------------------------------------- host

// one kernel per register class, one for all wide ones
constexpr int kNumKernels = kFirstMultiLane + 1;
constexpr size_t kMaxWorkspace = (size_t)1 << 30;
constexpr size_t kWideRow = 64 * sizeof(uint32_t);   // bytes of one limb of a wave's 64 values

// words of a program as the kernels read it
uint32_t program_words(const VmProgram& p, bool wide)
{
    return !wide ? 3u * (uint32_t)p.ins.size() : (uint32_t)p.wide.size();
}

struct Pending {
    std::shared_ptr<const VmProgram> prog;
    const uint8_t* cols[kMaxCols];
    uint32_t colbytes[kMaxCols];
    int64_t rows;
    int64_t chunk;  // rows per work item of this query
    bool wide;      // runs on the kernel of vm_wide.h
    uint8_t* image;
    int64_t* count;
};

// (whole 16-byte words, which k_vm_stage copies)
template <typename T> int host_alloc(T** p, size_t n)
{
    VMCHK(hipHostMalloc(reinterpret_cast<void**>(p), (sizeof(T) * std::max<size_t>(1, n) + 15) / 16 * 16, hipHostMallocMapped));
    return UPDEC_OK;
}
template <typename T> int dev_alloc(T** p, size_t n)
{
    VMCHK(hipMalloc(reinterpret_cast<void**>(p), (sizeof(T) * std::max<size_t>(1, n) + 15) / 16 * 16));
    return UPDEC_OK;
}

}  // namespace

struct updec_vm_s {
    std::shared_ptr<const VmProgram> prog;
    std::vector<uint32_t> colbytes;
};

// rows per work item unless updec_batch_tuning says otherwise, so that one
// 10^7-row query alone makes >= 4 items per CU
constexpr int64_t kItemRows[kNumClasses] = {8192, 8192, 4096, 2048, 1024, 512, 256, 128, 64};

struct updec_batch_s {
    int device = 0;   // the one that was current when the batch was made
    int max_queries = 0, max_items = 0, max_prog_words = 0, max_const_words = 0;
    int64_t rows_per_item[kNumClasses];
    // (a block of the wide classes is one wave)
    int blocks_per_cu[kNumClasses] = {4, 4, 4, 4, 4, 12, 12, 12, 12};
    // workspace of the wide kernel, grown by updec_batch_add to what the
    // largest wide program met so far needs, at most kMaxWorkspace
    uint8_t* d_work = nullptr;
    size_t work_bytes = 0;
    std::vector<uint8_t*> old_work;
    bool work_short = false;  // the last allocation got less than it asked for
    size_t pend_stride = 0;   // bytes per block of the pending queries' largest
    Header* h_hdr = nullptr;
    Query* h_q = nullptr;
    Item* h_items = nullptr;
    uint32_t* h_prog = nullptr;
    uint32_t* h_cst = nullptr;
    Header* d_hdr = nullptr;
    Query* d_q = nullptr;
    Item* d_items = nullptr;
    uint32_t* d_prog = nullptr;
    uint32_t* d_cst = nullptr;
    uint32_t* d_partials = nullptr;
    hipEvent_t staged = nullptr;  // the last launch's host-to-device copies are done
    bool staged_pending = false;
    hipStream_t side[kNumKernels] = {};
    hipEvent_t fork = nullptr, join[kNumKernels] = {};
    hipGraphExec_t graph = nullptr;
    std::vector<Pending> pending;
    // space the pending queries take at launch
    uint32_t pend_items = 0, pend_prog_words = 0, pend_const_words = 0;
    std::set<std::pair<const VmProgram*, bool>> pend_programs;
    std::mutex mu;

    updec_batch_s() { std::copy(kItemRows, kItemRows + kNumClasses, rows_per_item); }
    ~updec_batch_s()
    {
        if (staged_pending && staged) (void)hipEventSynchronize(staged);
        if (graph) (void)hipGraphExecDestroy(graph);
        for (auto& s : side)
            if (s) (void)hipStreamDestroy(s);
        for (auto& e : join)
            if (e) (void)hipEventDestroy(e);
        if (fork) (void)hipEventDestroy(fork);
        if (staged) (void)hipEventDestroy(staged);
        (void)hipHostFree(h_hdr);
        (void)hipHostFree(h_q);
        (void)hipHostFree(h_items);
        (void)hipHostFree(h_prog);
        (void)hipHostFree(h_cst);
        (void)hipFree(d_hdr);
        (void)hipFree(d_q);
        (void)hipFree(d_items);
        (void)hipFree(d_prog);
        (void)hipFree(d_cst);
        (void)hipFree(d_partials);
        (void)hipFree(d_work);
        for (uint8_t* p : old_work) (void)hipFree(p);
    }

    void clear_pending()
    {
        pending.clear();
        pend_items = pend_prog_words = pend_const_words = 0;
        pend_stride = 0;
        pend_programs.clear();
    }

    // blocks of the wide kernel on a full device
    int wide_grid() const
    {
        int bpc = 1;
        for (int c = kFirstMultiLane; c < kNumClasses; c++) bpc = std::max(bpc, blocks_per_cu[c]);
        return api_device_cus() * bpc;
    }

    // workspace for blocks of `stride` bytes: for every block of a full
    // device up to kMaxWorkspace, and where that much memory is not free, for
    // as many as there is.  One that is too small is kept until the batch
    // ends, not freed: launches may be running on it, which hipFree would wait
    // for with every stream of the device, and a caller's captured launch may
    // be replayed with it.  Each is twice as large as the last (half as large
    // again where memory is short), so those kept are at most as much again
    // (twice as much).
    int reserve(size_t stride)
    {
        const size_t most = std::max(kMaxWorkspace, 64 * stride);
        size_t want = std::min(most, (size_t)wide_grid() * stride);
        if (want <= work_bytes) return UPDEC_OK;
        const bool serves = work_bytes >= stride;
        // what there is has to do until the next batch, which asks again
        if (serves && work_short && !pending.empty()) return UPDEC_OK;
        const OnDevice on(device);   // queries are staged by any thread
        const AllocWhileCapturing allowed;
        want = std::min(most, std::max(want, 2 * work_bytes));
        const size_t least = serves ? work_bytes + work_bytes / 2 : stride;
        work_short = false;
        uint8_t* p = nullptr;
        while (want < least || hipMalloc(reinterpret_cast<void**>(&p), want) != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
            work_short = true;
            if (want <= least)
                return serves ? UPDEC_OK : api_fail(UPDEC_EHIP, "no device memory for the wide kernel's workspace");
            want = std::max(want / 2, least);
        }
        if (d_work) old_work.push_back(d_work);
        d_work = p;
        work_bytes = want;
        return UPDEC_OK;
    }

    // launch the class kernels (on `s` or on the side streams) and the final kernel
    int launch_kernels(hipStream_t s, bool fork_join, const uint32_t* nitems_per_class)
    {
        // kernel k: class k of the register classes, or all the wide ones
        auto items_of = [&](int k) {
            uint32_t n = 0;
            for (int c = k; c < (k < kFirstMultiLane ? k + 1 : kNumClasses); c++) n += nitems_per_class[c];
            return n;
        };
        auto launch_kernel = [&](int k, hipStream_t st) -> int {
            int g = k < kFirstMultiLane ? api_device_cus() * blocks_per_cu[k] : wide_grid();
            if (nitems_per_class) g = std::max(1, std::min<int>(g, (int)items_of(k)));
            switch (k) {
            case 0: hipLaunchKernelGGL((k_vm_sum<2, kBlock[0]>), dim3(g), dim3(kBlock[0]), 0, st, d_hdr, d_q, d_prog, d_cst, d_items, d_partials); break;
            case 1: hipLaunchKernelGGL((k_vm_sum<4, kBlock[1]>), dim3(g), dim3(kBlock[1]), 0, st, d_hdr, d_q, d_prog, d_cst, d_items, d_partials); break;
            case 2: hipLaunchKernelGGL((k_vm_sum<8, kBlock[2]>), dim3(g), dim3(kBlock[2]), 0, st, d_hdr, d_q, d_prog, d_cst, d_items, d_partials); break;
            case 3: hipLaunchKernelGGL((k_vm_sum<16, kBlock[3]>), dim3(g), dim3(kBlock[3]), 0, st, d_hdr, d_q, d_prog, d_cst, d_items, d_partials); break;
            case 4: hipLaunchKernelGGL((k_vm_sum<32, kBlock[4]>), dim3(g), dim3(kBlock[4]), 0, st, d_hdr, d_q, d_prog, d_cst, d_items, d_partials); break;
            default: hipLaunchKernelGGL(k_vm_sum_wide, dim3(g), dim3(64), 0, st, d_hdr, d_q, d_prog, d_cst, d_items, d_partials); break;
            }
            VMCHK(hipGetLastError());
            return UPDEC_OK;
        };
        if (fork_join) {
            VMCHK(hipEventRecord(fork, s));
            for (int k = 0; k < kNumKernels; k++) {
                VMCHK(hipStreamWaitEvent(side[k], fork, 0));
                int rc = launch_kernel(k, side[k]);
                if (rc) return rc;
                VMCHK(hipEventRecord(join[k], side[k]));
                VMCHK(hipStreamWaitEvent(s, join[k], 0));
            }
        } else {
            for (int k = 0; k < kNumKernels; k++) {
                if (nitems_per_class && items_of(k) == 0) continue;
                int rc = launch_kernel(k, s);
                if (rc) return rc;
            }
        }
        const uint32_t nq = fork_join ? (uint32_t)max_queries : h_hdr->nqueries;
        if (nq) {
            const u32 slices = std::min(kFinalSlices, std::max(1u, kFinalBlocks / nq));
            hipLaunchKernelGGL(k_vm_final, dim3(nq, slices), dim3(kFinalThreads), 0, s, d_hdr, d_q, d_partials);
            VMCHK(hipGetLastError());
        }
        return UPDEC_OK;
    }
};

// ---------------------------------------------------------------- C ABI

int updec_vm_compile(const char* text, const updec_column_desc* cols, int ncols, int mode, updec_vm_t* out)
{
    if (!text || !out || ncols < 0 || ncols > kMaxCols || (ncols && !cols)) return api_fail(UPDEC_EINVAL, "bad argument");
    std::vector<std::string> names;
    auto types = api_types(cols, ncols, &names);
    Plan plan;
    std::string err;
    if (!api_make_plan(text, names, types, mode, &plan, &err)) return api_fail(UPDEC_ECOMPILE, err);
    auto prog = std::make_shared<VmProgram>();
    if (!build_vm_program(plan, types, prog.get(), &err)) return api_fail(UPDEC_EUNSUPPORTED, err);
    std::unique_ptr<updec_vm_s> v(new updec_vm_s());
    v->prog = prog;
    for (auto& t : types) v->colbytes.push_back((uint32_t)compact_bytes(t.P));
    *out = v.release();
    return UPDEC_OK;
}

int updec_vm_info(updec_vm_t v, int32_t* width, int32_t* nins, int32_t* nregs, int32_t* precision, int32_t* scale,
                  int32_t* faithful)
{
    if (!v) return api_fail(UPDEC_EINVAL, "null program");
    const VmProgram& p = *v->prog;
    if (width) *width = p.W;
    if (nins) *nins = (int32_t)p.ins.size();
    if (nregs) *nregs = p.nregs;
    if (precision) *precision = p.outP;
    if (scale) *scale = p.outS;
    if (faithful) *faithful = p.faithful ? 1 : 0;
    return UPDEC_OK;
}

int updec_vm_workspace(updec_vm_t v, int64_t* bytes)
{
    if (!v || !bytes) return api_fail(UPDEC_EINVAL, "bad argument");
    *bytes = (int64_t)(v->prog->wide.empty() ? 0 : (size_t)v->prog->wide_rows * kWideRow);
    return UPDEC_OK;
}

int updec_vm_listing(updec_vm_t v, char* buf, size_t cap, size_t* needed)
{
    if (!v) return api_fail(UPDEC_EINVAL, "null program");
    std::string s = v->prog->text();
    if (needed) *needed = s.size() + 1;
    if (buf && cap) {
        size_t n = std::min(cap - 1, s.size());
        memcpy(buf, s.data(), n);
        buf[n] = 0;
    }
    return UPDEC_OK;
}

void updec_vm_free(updec_vm_t v) { delete v; }

int updec_batch_create(int32_t max_queries, int32_t max_items, updec_batch_t* out)
{
    if (!out || max_queries <= 0 || max_items < max_queries) return api_fail(UPDEC_EINVAL, "bad argument");
    std::unique_ptr<updec_batch_s> b(new updec_batch_s());
    VMCHK(hipGetDevice(&b->device));
    b->max_queries = max_queries;
    b->max_items = max_items;
    b->max_prog_words = max_queries * (3 * 64 + (int)wide::kHead);
    b->max_const_words = max_queries * 8 * (512 + 1);
    int rc;
    if ((rc = host_alloc(&b->h_hdr, 1)) || (rc = host_alloc(&b->h_q, max_queries)) || (rc = host_alloc(&b->h_items, max_items)) ||
        (rc = host_alloc(&b->h_prog, b->max_prog_words)) || (rc = host_alloc(&b->h_cst, b->max_const_words)) ||
        (rc = dev_alloc(&b->d_hdr, 1)) || (rc = dev_alloc(&b->d_q, max_queries)) || (rc = dev_alloc(&b->d_items, max_items)) ||
        (rc = dev_alloc(&b->d_prog, b->max_prog_words)) || (rc = dev_alloc(&b->d_cst, b->max_const_words)) ||
        (rc = dev_alloc(&b->d_partials, (size_t)max_items * kMaxAccWords)))
        return rc;
    memset(b->h_hdr, 0, sizeof(Header));
    VMCHK(hipEventCreateWithFlags(&b->staged, hipEventDisableTiming));
    VMCHK(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
    for (int c = 0; c < kNumKernels; c++) {
        VMCHK(hipStreamCreateWithFlags(&b->side[c], hipStreamNonBlocking));
        VMCHK(hipEventCreateWithFlags(&b->join[c], hipEventDisableTiming));
    }
    *out = b.release();
    return UPDEC_OK;
}

int updec_batch_tuning(updec_batch_t b, int32_t width_class, int64_t rows_per_item, int32_t blocks_per_cu)
{
    if (!b || width_class < 0 || width_class >= kNumClasses || rows_per_item < 64 || blocks_per_cu < 1 ||
        blocks_per_cu > 64)
        return api_fail(UPDEC_EINVAL, "bad argument");
    std::lock_guard<std::mutex> g(b->mu);
    if (!b->pending.empty()) return api_fail(UPDEC_EINVAL, "tuning changes while queries are staged");
    b->rows_per_item[width_class] = rows_per_item;
    b->blocks_per_cu[width_class] = blocks_per_cu;
    if (b->graph) {
        (void)hipGraphExecDestroy(b->graph);
        b->graph = nullptr;
    }
    return UPDEC_OK;
}

int updec_batch_lanes(updec_batch_t b, int32_t width_class, int32_t lanes)
{
    if (!b || width_class < kFirstMultiLane || width_class >= kNumClasses)
        return api_fail(UPDEC_EINVAL, "lanes per value apply to the wide classes (W = 64 .. 512)");
    const int W = kClassW[width_class];
    if ((lanes != W / 4 && lanes != W / 8) || lanes > 64)
        return api_fail(UPDEC_EINVAL, "lanes per value must be W / 4 or W / 8, at most 64");
    std::lock_guard<std::mutex> g(b->mu);
    if (!b->pending.empty()) return api_fail(UPDEC_EINVAL, "tuning changes while queries are staged");
    return UPDEC_OK;   // a value lies in one lane's memory whatever is asked
}

int updec_batch_add(updec_batch_t b, updec_vm_t v, const uint8_t* const* d_cols, int64_t rows, uint8_t* d_image,
                    int64_t* d_count, int32_t* index_out)
{
    if (!b || !v || rows < 0 || !d_image || !d_count || (!d_cols && !v->colbytes.empty()))
        return api_fail(UPDEC_EINVAL, "bad argument");
    std::lock_guard<std::mutex> g(b->mu);
    const VmProgram& pr = *v->prog;
    const size_t stride = (size_t)pr.wide_rows * kWideRow;
    bool wide = !pr.wide.empty();
    if (wide) {
        const size_t block = std::max(stride, b->pend_stride);
        const int rc = b->reserve(block);
        // what the register kernels have a class for needs no workspace
        if (pr.wclass < kFirstMultiLane) wide = rc == UPDEC_OK && b->work_bytes >= 64 * block;
        else if (rc) return rc;
    }
    // the class's tuned rows per item, raised (in steps of 64 rows) for a
    // query that would otherwise need more items than the whole batch holds
    int64_t ch = b->rows_per_item[pr.wclass];
    // a large query takes items of at least rows / (4 x the class's resident
    // blocks): four items per block keep the load balanced while the
    // per-item work (fetch, block reduction, partial write) stays small next
    // to the item's rows
    const int64_t slots = 4 * (int64_t)api_device_cus() * b->blocks_per_cu[item_class(pr.wclass, wide)];
    const int64_t big = (rows + slots - 1) / slots;
    if (big > ch) ch = (big + 63) / 64 * 64;
    if ((rows + ch - 1) / ch > b->max_items) ch = ((rows + b->max_items - 1) / b->max_items + 63) / 64 * 64;
    const uint32_t items = (uint32_t)std::max<int64_t>(1, (rows + ch - 1) / ch);
    const bool new_prog = b->pend_programs.find({&pr, wide}) == b->pend_programs.end();
    const uint32_t pw = new_prog ? program_words(pr, wide) : 0u, cw = new_prog ? (uint32_t)pr.consts.size() : 0u;
    if ((int)b->pending.size() >= b->max_queries || b->pend_items + items > (uint32_t)b->max_items ||
        b->pend_prog_words + pw > (uint32_t)b->max_prog_words || b->pend_const_words + cw > (uint32_t)b->max_const_words) {
        if (b->pending.empty()) return api_fail(UPDEC_EINVAL, "query does not fit an empty batch");
        return api_fail(UPDEC_EFULL, "batch is full");
    }
    Pending p{};
    p.prog = v->prog;
    for (size_t c = 0; c < v->colbytes.size(); c++) {
        if (!d_cols[c] && rows > 0) return api_fail(UPDEC_EINVAL, "null column");
        p.cols[c] = d_cols[c];
        p.colbytes[c] = v->colbytes[c];
    }
    p.rows = rows;
    p.chunk = ch;
    p.image = d_image;
    p.count = d_count;
    p.wide = wide;
    if (wide) b->pend_stride = std::max(stride, b->pend_stride);
    b->pending.push_back(p);
    b->pend_items += items;
    b->pend_prog_words += pw;
    b->pend_const_words += cw;
    b->pend_programs.insert({&pr, wide});
    if (index_out) *index_out = (int32_t)b->pending.size() - 1;
    return UPDEC_OK;
}

int updec_batch_pending(updec_batch_t b, int32_t* n)
{
    if (!b || !n) return api_fail(UPDEC_EINVAL, "bad argument");
    std::lock_guard<std::mutex> g(b->mu);
    *n = (int32_t)b->pending.size();
    return UPDEC_OK;
}

int updec_batch_launch(updec_batch_t b, int use_graph, updec_stream_t stream)
{
    if (!b) return api_fail(UPDEC_EINVAL, "null batch");
    std::lock_guard<std::mutex> g(b->mu);
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (b->pending.empty()) return UPDEC_OK;
    // the staging buffers are rewritten below: the previous copies must be done
    if (b->staged_pending) {
        VMCHK(hipEventSynchronize(b->staged));
        b->staged_pending = false;
    }
    // items per class, in class order; programs and constants deduplicated
    uint32_t nitems[kNumClasses] = {};
    // The rows per item of updec_batch_add suit queries that fill the device;
    // one of 50,000 rows had 7 to 49 of its blocks.  Where a kernel's rows
    // would leave it with fewer than two items for each resident block, its
    // queries are cut finer, down to one row a thread, as far as the items
    // that the batch has to spare go (dealt out evenly): one query of 50,000
    // rows 714 -> 151 us at 16 limbs, 274 -> 127 at 2; 1.2 M rows at 16 limbs
    // 783 -> 550.
    const int64_t spare = (b->max_items - (int64_t)b->pend_items) / (int64_t)b->pending.size();
    int64_t rows_of[kNumKernels] = {};
    for (const Pending& p : b->pending) rows_of[std::min(item_class(p.prog->wclass, p.wide), kFirstMultiLane)] += p.rows;
    for (Pending& p : b->pending) {
        const int c = item_class(p.prog->wclass, p.wide);
        const int64_t T = p.wide ? 64 : kBlock[c];
        const int64_t most = std::max<int64_t>(1, (p.rows + p.chunk - 1) / p.chunk) + spare;
        int64_t even = rows_of[std::min(c, kFirstMultiLane)] / (2 * (int64_t)api_device_cus() * b->blocks_per_cu[c]);
        // What a register class is tuned to suits its own kernel's blocks, not
        // the wide kernel's waves: items of 8,000 rows of 16 limbs took one of
        // those some 10 ms, a quarter of a batch of 50 M rows.
        if (p.wide && p.prog->wclass < kFirstMultiLane)
            even = std::min(even, std::max(kItemRows[p.prog->wclass], p.rows / (4 * (int64_t)b->wide_grid())));
        p.chunk = std::min(p.chunk, std::max(T, (std::max(even, (p.rows + most - 1) / most) + T - 1) / T * T));
        nitems[c] += (uint32_t)std::max<int64_t>(1, (p.rows + p.chunk - 1) / p.chunk);
    }
    uint32_t total = 0, first[kNumClasses];
    for (int c = 0; c < kNumClasses; c++) {
        first[c] = total;
        total += nitems[c];
    }
    if (total > (uint32_t)b->max_items) {
        b->clear_pending();
        return api_fail(UPDEC_EINVAL, "batch needs more work items than it was created for");
    }
    std::map<std::pair<const VmProgram*, bool>, std::pair<uint32_t, uint32_t>> placed;  // program -> (ins_off, const_off)
    uint32_t prog_words = 0, const_words = 0, fill[kNumClasses];
    memcpy(fill, first, sizeof fill);
    Header& H = *b->h_hdr;
    memset(&H, 0, sizeof H);
    H.nqueries = (uint32_t)b->pending.size();
    H.workspace = b->d_work;
    H.stride = b->pend_stride;
    H.wide_blocks = b->pend_stride ? (uint32_t)std::min<size_t>(b->work_bytes / b->pend_stride, (size_t)INT32_MAX) : 0u;
    for (int c = 0; c < kNumClasses; c++) {
        H.class_item0[c] = first[c];
        H.class_nitems[c] = nitems[c];
    }
    for (size_t qi = 0; qi < b->pending.size(); qi++) {
        const Pending& p = b->pending[qi];
        const VmProgram& pr = *p.prog;
        auto it = placed.find({&pr, p.wide});
        if (it == placed.end()) {
            const uint32_t pw = program_words(pr, p.wide), cw = (uint32_t)pr.consts.size();
            if (prog_words + pw > (uint32_t)b->max_prog_words || const_words + cw > (uint32_t)b->max_const_words) {
                b->clear_pending();
                return api_fail(UPDEC_EINVAL, "batch programs exceed the staging space");
            }
            if (p.wide) memcpy(b->h_prog + prog_words, pr.wide.data(), 4u * pw);
            for (size_t k = 0; !p.wide && k < pr.ins.size(); k++) {
                const Ins& I = pr.ins[k];
                uint32_t* w = b->h_prog + prog_words + 3 * k;
                w[0] = (uint32_t)I.op | ((uint32_t)I.dst << 8) | ((uint32_t)I.arg << 16);
                w[1] = (uint32_t)I.a.kind | ((uint32_t)I.a.idx << 8) | ((uint32_t)I.a.shift << 16);
                w[2] = (uint32_t)I.b.kind | ((uint32_t)I.b.idx << 8) | ((uint32_t)I.b.shift << 16);
            }
            if (cw) memcpy(b->h_cst + const_words, pr.consts.data(), 4u * cw);
            if (p.wide)
                // a constant's sign word also tells its limbs
                for (uint32_t* k = b->h_cst + const_words; k < b->h_cst + const_words + cw; k += pr.W + 1) {
                    uint32_t n = (uint32_t)pr.W;
                    while (n > 0 && k[n] == 0u) n--;
                    *k = (*k & 1u) | (n << 8);
                }
            it = placed.emplace(std::make_pair(&pr, p.wide), std::make_pair(prog_words / 3u, const_words)).first;
            prog_words += pw;
            const_words += cw;
        }
        Query& Q = b->h_q[qi];
        memset(&Q, 0, sizeof Q);
        for (int c = 0; c < kMaxCols; c++) {
            Q.col[c] = p.cols[c];
            Q.colbytes[c] = p.colbytes[c];
        }
        Q.rows = (uint64_t)p.rows;
        Q.ins_off = it->second.first;
        Q.nins = (uint32_t)pr.ins.size();
        Q.const_off = it->second.second;
        Q.root = (uint32_t)pr.root;
        Q.outB = (uint32_t)pr.outB;
        Q.outP = (uint32_t)pr.outP;
        Q.outS = (uint32_t)pr.outS;
        Q.faithful = pr.faithful ? 1u : 0u;
        Q.wclass = (uint32_t)pr.wclass;
        Q.image = p.image;
        Q.count = p.count;
        const int c = item_class(pr.wclass, p.wide);
        const int64_t ch = p.chunk;
        const uint32_t n = (uint32_t)std::max<int64_t>(1, (p.rows + ch - 1) / ch);
        Q.item0 = fill[c];
        Q.nitems = n;
        for (uint32_t k = 0; k < n; k++) {
            Item& I = b->h_items[fill[c] + k];
            I.query = (uint32_t)qi;
            I.pad = 0;
            I.row0 = (uint64_t)std::min<int64_t>(p.rows, (int64_t)k * ch);
            I.row1 = (uint64_t)std::min<int64_t>(p.rows, (int64_t)(k + 1) * ch);
        }
        fill[c] += n;
    }
    const size_t nq = b->pending.size();
    b->clear_pending();
    Staging t;
    const void* src[kTables] = {b->h_hdr, b->h_q, b->h_items, b->h_prog, b->h_cst};
    void* dst[kTables] = {b->d_hdr, b->d_q, b->d_items, b->d_prog, b->d_cst};
    const size_t bytes[kTables] = {sizeof(Header), sizeof(Query) * nq, sizeof(Item) * total, 4u * prog_words, 4u * const_words};
    for (int k = 0; k < kTables; k++) {
        void* p = nullptr;
        VMCHK(hipHostGetDevicePointer(&p, const_cast<void*>(src[k]), 0));
        t.src[k] = static_cast<const uint4*>(p);
        t.dst[k] = static_cast<uint4*>(dst[k]);
        t.end[k] = (k ? t.end[k - 1] : 0u) + (uint32_t)((bytes[k] + 15) / 16);
    }
    hipLaunchKernelGGL(k_vm_stage, dim3((t.end[kTables - 1] + 255u) / 256u), dim3(256), 0, s, t);
    VMCHK(hipGetLastError());
    VMCHK(hipEventRecord(b->staged, s));
    b->staged_pending = true;
    // one kernel's work needs no branches: the graph's fork, its other five
    // kernels (empty) and the join take about as long as a small query
    int kernels = 0;
    for (int c = 0; c < kNumClasses; c++) kernels += (c < kFirstMultiLane ? nitems[c] : 0u) != 0u;
    for (int c = kFirstMultiLane; c < kNumClasses; c++)
        if (nitems[c]) { kernels++; break; }
    if (!use_graph || kernels == 1) return b->launch_kernels(s, false, nitems);
    if (!b->graph) {
        // capture once: every class kernel on its own branch, sized for a
        // full device; kernels with no items exit at once
        hipStream_t cap;
        VMCHK(hipStreamCreateWithFlags(&cap, hipStreamNonBlocking));
        hipGraph_t graph = nullptr;
        int rc = UPDEC_OK;
        hipError_t e = hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
            rc = b->launch_kernels(cap, true, nullptr);
            hipError_t e2 = hipStreamEndCapture(cap, &graph);
            if (rc == UPDEC_OK && e2 != hipSuccess) rc = api_fail(UPDEC_EHIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e2));
        } else {
            rc = api_fail(UPDEC_EHIP, std::string("hipStreamBeginCapture: ") + hipGetErrorString(e));
        }
        if (rc == UPDEC_OK) {
            e = hipGraphInstantiate(&b->graph, graph, nullptr, nullptr, 0);
            if (e != hipSuccess) rc = api_fail(UPDEC_EHIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
        }
        if (graph) (void)hipGraphDestroy(graph);
        (void)hipStreamDestroy(cap);
        if (rc) return rc;
    }
    VMCHK(hipGraphLaunch(b->graph, s));
    return UPDEC_OK;
}

void updec_batch_free(updec_batch_t b) { delete b; }
