// vm_wide_host.cpp -- TEST INFRASTRUCTURE: the interpreter's wide evaluation
// (vm_wide.h) built for the host CPU with one lane, so the CPU suite checks
// its programs row by row before any GPU run.  Every program is put into the
// wide form, whatever its class, and its workspace is checked for writes
// past its end.
#define __HIPCC_RTC__ 1
#define __device__
#define __forceinline__ inline
#define __global__
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>
#include <string>
static inline unsigned upd_alignbyte(unsigned hi, unsigned lo, unsigned s) { return (unsigned)((((unsigned long long)hi << 32) | lo) >> (8 * (s & 3))); }
#define __builtin_amdgcn_alignbyte(a, b, c) upd_alignbyte((a), (b), (c))
#define __builtin_nontemporal_load(p) (*(p))
static inline int __shfl_xor(int v, int, int) { return v; }
#include "dec_device.h"
#include "vm_wide.h"
#include "planner.h"
using namespace updec;
using namespace updec_vm;

// out: the 1024-limb two's complement sum of the materialized rows
extern "C" int vmw_sum(const char* text, const char** names, const int* P, const int* S, int ncols,
                       const uint8_t* const* data, int64_t rows, uint32_t* out, int* width, char* err, int cap, int mode)
{
    std::vector<std::string> nm;
    std::vector<ColumnType> ty(ncols);
    for (int i = 0; i < ncols; i++) { nm.push_back(names[i]); ty[i].P = P[i]; ty[i].S = S[i]; ty[i].bits = 0; }
    Plan plan;
    std::string e;
    if (!plan_expression(text, nm, ty, mode, &plan, &e)) { snprintf(err, cap, "%s", e.c_str()); return 1; }
    VmProgram pr;
    if (!build_vm_program(plan, ty, &pr, &e)) { snprintf(err, cap, "%s", e.c_str()); return 2; }
    *width = pr.W;
    if (pr.wide.empty()) { snprintf(err, cap, "no wide form"); return 3; }
    Query Q{};
    for (int c = 0; c < ncols; c++) { Q.col[c] = data[c]; Q.colbytes[c] = compact_bytes(P[c]); }
    Q.rows = rows; Q.nins = pr.ins.size(); Q.outB = pr.outB; Q.faithful = pr.faithful;
    std::vector<uint32_t> cst = pr.consts;
    for (size_t k = 0; k + pr.W < cst.size(); k += pr.W + 1) {
        uint32_t n = 0;
        for (int w = 0; w < pr.W; w++) if (cst[k + 1 + w]) n = w + 1;
        cst[k] = (cst[k] & 1u) | (n << 8);
    }
    constexpr uint32_t kGuard = 64, kMark = 0xdeadbeefu;
    std::vector<uint32_t> ws(pr.wide_rows + kGuard, kMark);
    uint8_t* base = reinterpret_cast<uint8_t*>(ws.data());
    auto at = [&](uint32_t h) { return wide::Dst{base + 4 * pr.wide[h], 0u}; };
    const wide::Dst pos = at(wide::kHeadPos), neg = at(wide::kHeadNeg);
    const uint32_t na = pr.wide[wide::kHeadAcc];
    for (uint32_t i = 0; i < na; i++) { pos.put(i, 0); neg.put(i, 0); }
    wide::Slots sl;
    for (int64_t r = 0; r < rows; r++) {
        uint32_t s;
        const wide::Src v = wide::eval(&Q, pr.wide.data(), cst.data(), (uint32_t)pr.W, base, &sl, (usize)r, s);
        wide::accumulate(v, s, true, Q.outB, pos, neg);
    }
    for (uint32_t i = 0; i < kGuard; i++)
        if (ws[pr.wide_rows + i] != kMark) { snprintf(err, cap, "wrote past the workspace"); return 4; }
    int64_t c = 0;
    for (uint32_t i = 0; i < 1024; i++) {
        const int64_t t = (i < na ? (int64_t)pos.at(i) - (int64_t)neg.at(i) : 0) + c;
        out[i] = (uint32_t)t;
        c = t >> 32;
    }
    return 0;
}
