// lgca_force.hip -- the count-mode body force, apply_body_force(int forcing)
// (src/omp_lattice.cpp:254-346): candidate cells from the hash, each visited
// cell forced if its flip rule allows, until `forcing` particles are reverted
// or 2N tries are spent (always after at least one try).
//
// The sequential loop's result depends on the order of its tries only through
// where it stops: a cell that has been visited never flips again (its visit
// makes its flip rules infeasible, or they were so already), so after M tries
// exactly the feasible rules of the distinct cells among them have been
// applied.  Four kernels use that:
//   list    over the whole GPU, the first `tries` tries against the state as
//           it is; the feasible ones (a tenth, as a rule) are listed in order;
//   bulk    over the whole GPU, as many entries as cannot reach the amount even
//           if none repeats a cell are applied at once, a repeated cell going
//           to whichever lane clears its bit first;
//   commit  one workgroup takes the entries around the stop in order, 1024 at
//           a time (repeats dropped through a hash table in LDS, a prefix sum
//           finds the first try whose running total reaches the amount);
//   finish  one workgroup continues with unlisted tries, 4096 at a time in
//           the same manner, where the list did not reach the amount.
// What bounds it: the launches and the commit's round trips to the L2.  Finding
// 10,952 reverts on a 1480 x 740 lattice (some 90,000 tries): 8.2 ms with one
// wave and 64 tries at a time, 0.47 ms with the finish kernel alone, 81 us with
// the bulk in the commit's one workgroup (3 ns an atomic), 51 us so (list 6, bulk
// 21, commit 17, finish 7).
#include "lgca_dev.hpp"
#include "lgca_kernels.hpp"

#include <algorithm>

namespace lgca {

namespace {

constexpr uint32_t kForceThreads = 1024, kForceTries = 4;
constexpr uint32_t kListThreads = 256;                    // tries of one segment of the list
constexpr uint32_t kMaxSegments = kForceThreads;          // the commit scans one count per lane
constexpr uint32_t kHashSlots = 2 * kForceThreads;
constexpr long long kUnlisted = 64;                       // largest amount that no tries are listed for

// Workspace: this header, the segments' counts, then kListThreads entries per
// segment (cell | feasible rules << 62).
struct ForceList {
    long long reverted;  // by the listed tries
    uint64_t next;       // first try after them
    uint32_t stopped, pad;
    uint32_t counts[kMaxSegments];
};

__device__ __forceinline__ uint64_t* list_entries(void* ws) { return (uint64_t*)((char*)ws + sizeof(ForceList)); }

// The call's amount (-1: none) and number.
__device__ __forceinline__ long long force_amount(const CountForceArgs& a) { return a.ctrl ? a.ctrl->amount : a.amount; }
__device__ __forceinline__ uint32_t force_call(const CountForceArgs& a) { return a.ctrl ? a.ctrl->calls : a.call; }

// floor(a / n) and a - n * floor(a / n) from m = floor((2^64 - 1) / n): the
// product's high half is the quotient or one less.
__device__ __forceinline__ uint64_t divmod_magic(uint64_t a, uint64_t n, uint64_t m, uint64_t& rem)
{
    uint64_t q = __umul64hi(a, m);
    rem = a - q * n;
    if (rem >= n) {
        rem -= n;
        ++q;
    }
    return q;
}

// The flip rules (src/omp_lattice.cpp:293-337): a particle moves from plane
// `from` to plane `to` where `to` is empty.
template <int KIND>
struct ForceRules {
    static constexpr int Q = num_dir_of_kind(KIND);
    const CountForceArgs& a;
    uint32_t rules, from[2], to[2];

    __device__ __forceinline__ explicit ForceRules(const CountForceArgs& args) : a(args)
    {
        const bool x = a.dir == 1;
        rules = KIND != kHPP && !x ? 2u : 1u;
        from[0] = KIND == kHPP ? (x ? 2u : 1u) : (x ? 3u : 1u);
        to[0] = KIND == kHPP ? (x ? 0u : 3u) : (x ? 0u : 5u);
        from[1] = 2u;
        to[1] = 4u;
    }

    struct Try {
        uint64_t cell;
        uint32_t* word;  // word of the cell's row and column in plane 0
        uint32_t bit;    // 0: not a FLUID cell, or past the last try
    };
    __device__ __forceinline__ Try at_cell(uint64_t cell, bool mask) const
    {
        Try t;
        uint64_t x;
        const uint32_t y = (uint32_t)divmod_magic(cell, a.g.dim_x, a.row_magic, x);
        const uint32_t w = (uint32_t)x >> 5;
        t.cell = cell;
        t.word = a.planes + (size_t)y * Q * a.g.P + w;
        t.bit = 1u << ((uint32_t)x & 31u);
        if (mask && a.mask)
            t.bit &= ~(a.mask[((size_t)y * 2 + 0) * a.g.P + w] | a.mask[((size_t)y * 2 + 1) * a.g.P + w]);
        return t;
    }
    __device__ __forceinline__ Try at(uint64_t i, uint32_t call) const
    {
        const uint64_t n = (uint64_t)a.g.dim_x * a.g.dim_y;
        const U4 r = philox4x32_10((uint32_t)i, (uint32_t)(i >> 32), call, 3u, a.key0, a.key1);
        uint64_t cell;
        divmod_magic(((uint64_t)r.y << 32) | r.x, n, a.cells_magic, cell);
        Try t = at_cell(cell, true);
        if (i >= 2 * n) t.bit = 0;
        return t;
    }
    // the planes change under the commit and finish kernels: read past the L1
    __device__ __forceinline__ uint32_t plane(const Try& t, uint32_t d) const
    {
        return __hip_atomic_load(t.word + (size_t)d * a.g.P, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // feasible rules of a try, bit r for rule r (every cell is on the lattice,
    // so the loads need no test)
    __device__ __forceinline__ uint32_t feasible(const Try& t) const
    {
        uint32_t f = (plane(t, from[0]) & ~plane(t, to[0]) & t.bit) ? 1u : 0u;
        if (rules == 2) f |= (plane(t, from[1]) & ~plane(t, to[1]) & t.bit) ? 2u : 0u;
        return f;
    }
    // applies rules f of a try, feasible unless a repeat of its cell came
    // first; the number that this lane applied
    __device__ __forceinline__ uint32_t flip(const Try& t, uint32_t f) const
    {
        uint32_t k = 0;
        for (uint32_t r = 0; r < rules; ++r) {
            if (!((f >> r) & 1u)) continue;
            if (atomicAnd(t.word + (size_t)from[r] * a.g.P, ~t.bit) & t.bit) {
                atomicOr(t.word + (size_t)to[r] * a.g.P, t.bit);
                ++k;
            }
        }
        return k;
    }
};

// Sums and orders over the one workgroup of the commit and finish kernels.
struct ForceShared {
    uint32_t part[2][kForceThreads / 64];
    uint32_t first_hit, at_hit;
    uint64_t key[kHashSlots];
    uint32_t first[kHashSlots];
};

// Sum of v over the workgroup; every lane gets it.  Flips made before it are
// in the L2 after it.  Calls alternate the slot.
__device__ __forceinline__ uint32_t force_sum(ForceShared& sh, uint32_t v, uint32_t slot)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63u) == 0) sh.part[slot][threadIdx.x >> 6] = v;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint32_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < kForceThreads / 64; ++k) s += sh.part[slot][k];
    return s;
}

// One try per lane, in the order of the lanes: applies them up to the first
// whose running total from `reverted` on reaches `amount`, adds what they
// reverted and returns whether one did.  counts: the lane holds a try (one
// past the last, or past the list's end, cannot be the stop).
template <int KIND>
__device__ __forceinline__ bool force_in_order(ForceShared& sh, const ForceRules<KIND>& R,
                                               const typename ForceRules<KIND>::Try& t, bool counts, long long amount,
                                               long long& reverted)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    for (uint32_t s = tid; s < kHashSlots; s += kForceThreads) {
        sh.key[s] = ~0ull;
        sh.first[s] = ~0u;
    }
    if (tid == 0) sh.first_hit = kForceThreads;
    uint32_t f = counts ? R.feasible(t) : 0u, slot = 0;
    __syncthreads();
    // of the feasible tries of a cell only the first counts
    if (f) {
        slot = (uint32_t)((t.cell * 0x9E3779B97F4A7C15ull) >> 53) & (kHashSlots - 1u);
        for (;;) {
            const unsigned long long was = atomicCAS((unsigned long long*)&sh.key[slot], ~0ull, (unsigned long long)t.cell);
            if (was == ~0ull || was == t.cell) break;
            slot = (slot + 1u) & (kHashSlots - 1u);
        }
        atomicMin(&sh.first[slot], tid);
    }
    __syncthreads();
    if (f && sh.first[slot] != tid) f = 0;
    uint32_t incl = __popc(f);
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off, 64);
        if ((int)lane >= off) incl += v;
    }
    const uint32_t total = force_sum(sh, __popc(f), 1);
    for (uint32_t k = 0; k < wave; ++k) incl += sh.part[1][k];
    if (counts && reverted + (long long)incl >= amount) atomicMin(&sh.first_hit, tid);
    __syncthreads();
    const uint32_t limit = sh.first_hit;
    if (f && tid <= limit) R.flip(t, f);
    if (tid == limit) sh.at_hit = incl;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    const bool stop = limit < kForceThreads;
    reverted += stop ? (long long)sh.at_hit : (long long)total;
    return stop;
}

template <int KIND>
__global__ __launch_bounds__(kListThreads) void count_force_list_kernel(CountForceArgs a)
{
    if (force_amount(a) <= 0) return;  // (at amount 0 the first try alone counts: the finish kernel's)
    const ForceRules<KIND> R(a);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    __shared__ uint32_t part[kListThreads / 64];
    const auto t = R.at((uint64_t)blockIdx.x * kListThreads + threadIdx.x, force_call(a));
    const uint32_t f = R.feasible(t);
    const unsigned long long any = __ballot(f != 0);
    if (lane == 0) part[wave] = (uint32_t)__popcll(any);
    __syncthreads();
    uint32_t pos = (uint32_t)__popcll(any & ((1ull << lane) - 1ull)), n = 0;
    for (uint32_t w = 0; w < kListThreads / 64; ++w) {
        if (w < wave) pos += part[w];
        n += part[w];
    }
    if (f) list_entries(a.ws)[(uint64_t)blockIdx.x * kListThreads + pos] = t.cell | ((uint64_t)f << 62);
    ForceList& ws = *(ForceList*)a.ws;
    if (threadIdx.x == 0) ws.counts[blockIdx.x] = n;
    if (threadIdx.x == 0 && blockIdx.x == 0) ws.reverted = 0;
}

// Entries that the bulk applies: those that cannot reach the amount even if
// none repeats a cell, unless the commit can order them all at once.
__device__ __forceinline__ uint32_t bulk_entries(uint32_t entries, long long amount, uint32_t rules)
{
    const uint32_t n = (uint32_t)min((uint64_t)entries, (uint64_t)(amount - 1) / rules);
    return n >= kForceThreads || n == entries ? n : 0u;
}

template <int KIND>
__global__ __launch_bounds__(kListThreads) void count_force_bulk_kernel(CountForceArgs a)
{
    const long long amount = force_amount(a);
    if (amount <= 0) return;
    const ForceRules<KIND> R(a);
    ForceList& ws = *(ForceList*)a.ws;
    __shared__ uint32_t part[2][kListThreads / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6, segments = a.tries / kListThreads;
    // entries before this segment, and in all
    uint32_t before = 0, all = 0;
    for (uint32_t s = tid; s < segments; s += kListThreads) {
        const uint32_t c = ws.counts[s];
        all += c;
        before += s < blockIdx.x ? c : 0u;
    }
    for (int off = 32; off > 0; off >>= 1) {
        all += __shfl_xor(all, off, 64);
        before += __shfl_xor(before, off, 64);
    }
    if (lane == 0) {
        part[0][wave] = all;
        part[1][wave] = before;
    }
    __syncthreads();
    all = before = 0;
    for (uint32_t w = 0; w < kListThreads / 64; ++w) {
        all += part[0][w];
        before += part[1][w];
    }
    const uint32_t n = bulk_entries(all, amount, R.rules);
    if (before >= n) return;
    uint32_t k = 0;
    if (tid < min(ws.counts[blockIdx.x], n - before)) {
        const uint64_t c = list_entries(a.ws)[(uint64_t)blockIdx.x * kListThreads + tid];
        k = R.flip(R.at_cell(c & ((1ull << 62) - 1ull), false), (uint32_t)(c >> 62));
    }
    // one addition per workgroup (they serialise)
    const unsigned long long won = __ballot((k & 1u) != 0), two = __ballot((k & 2u) != 0);
    __syncthreads();
    if (lane == 0) part[0][wave] = (uint32_t)__popcll(won) + 2u * (uint32_t)__popcll(two);
    __syncthreads();
    if (tid == 0) {
        for (uint32_t w = 1; w < kListThreads / 64; ++w) part[0][0] += part[0][w];
        atomicAdd((unsigned long long*)&ws.reverted, (unsigned long long)part[0][0]);
    }
}

template <int KIND>
__global__ __launch_bounds__(kForceThreads) void count_force_commit_kernel(CountForceArgs a)
{
    __shared__ ForceShared sh;
    __shared__ uint32_t before[kMaxSegments + 1];  // entries before each segment
    const long long amount = force_amount(a);
    ForceList& ws = *(ForceList*)a.ws;
    if (amount <= 0) {
        if (threadIdx.x == 0) {
            ws.reverted = 0;
            ws.next = 0;
            ws.stopped = 0;
        }
        return;
    }
    const ForceRules<KIND> R(a);
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t segments = a.tries / kListThreads;
    const uint32_t mine = tid < segments ? ws.counts[tid] : 0u;
    uint32_t incl = mine;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(incl, off, 64);
        if ((int)lane >= off) incl += v;
    }
    const uint32_t entries = force_sum(sh, mine, 0);
    for (uint32_t k = 0; k < wave; ++k) incl += sh.part[0][k];
    before[tid] = incl - mine;
    if (tid == 0) before[kMaxSegments] = entries;
    __syncthreads();
    const uint64_t* list = list_entries(a.ws);
    auto entry = [&](uint32_t e) {  // the segment holding entry e: the last with before[] <= e
        uint32_t s = 0;
#pragma unroll
        for (uint32_t step = kMaxSegments / 2; step; step >>= 1)
            if (before[s + step] <= e) s += step;
        return list[(uint64_t)s * kListThreads + (e - before[s])];
    };
    long long reverted = ws.reverted;
    uint32_t pos = bulk_entries(entries, amount, R.rules);
    bool stop = false;
    while (pos < entries && !stop) {
        const bool counts = pos + tid < entries;
        const uint64_t c = counts ? entry(pos + tid) : 0ull;
        // (listed tries are on FLUID cells)
        stop = force_in_order<KIND>(sh, R, R.at_cell(c & ((1ull << 62) - 1ull), false), counts, amount, reverted);
        pos += min(entries - pos, kForceThreads);
    }
    if (tid == 0) {
        ws.reverted = reverted;
        ws.next = a.tries;
        ws.stopped = stop ? 1u : 0u;
    }
}

template <int KIND>
__global__ __launch_bounds__(kForceThreads) void count_force_finish_kernel(CountForceArgs a)
{
    __shared__ ForceShared sh;
    const long long amount = force_amount(a);
    if (a.ctrl && amount < 0) return;
    const uint32_t call = force_call(a);
    const ForceRules<KIND> R(a);
    const uint32_t tid = threadIdx.x;
    const uint64_t it_max = 2 * (uint64_t)a.g.dim_x * a.g.dim_y;
    long long reverted = 0;
    uint64_t base = 0;
    bool stop = false;
    if (a.tries) {
        const ForceList& ws = *(const ForceList*)a.ws;
        reverted = ws.reverted;
        base = ws.next;
        stop = ws.stopped != 0;
    }
    __syncthreads();  // every lane has read the call's number
    // a small amount is reached within 1024 tries as a rule, so they are not
    // weighed 4096 at a time first
    if (!stop && base < it_max && amount - reverted <= kUnlisted) {
        stop = force_in_order<KIND>(sh, R, R.at(base + tid, call), base + tid < it_max, amount, reverted);
        base += kForceThreads;
    }
    for (; base < it_max && !stop; base += kForceThreads * kForceTries) {
        typename ForceRules<KIND>::Try t[kForceTries];
        uint32_t f[kForceTries], most = 0;
#pragma unroll
        for (uint32_t u = 0; u < kForceTries; ++u) t[u] = R.at(base + u * kForceThreads + tid, call);
#pragma unroll
        for (uint32_t u = 0; u < kForceTries; ++u) f[u] = R.feasible(t[u]);
#pragma unroll
        for (uint32_t u = 0; u < kForceTries; ++u) most += __popc(f[u]);
        if (reverted + (long long)force_sum(sh, most, 0) < amount) {
            uint32_t k = 0;
#pragma unroll
            for (uint32_t u = 0; u < kForceTries; ++u) k += R.flip(t[u], f[u]);
            reverted += force_sum(sh, k, 1);
            continue;
        }
        // the sequence may stop here
#pragma unroll 1
        for (uint32_t u = 0; u < kForceTries && !stop; ++u) {
            const uint64_t i = base + u * kForceThreads + tid;
            stop = force_in_order<KIND>(sh, R, R.at(i, call), i < it_max, amount, reverted);
        }
    }
    if (tid == 0) {
        if (a.ctrl) {
            a.ctrl->reverted = reverted;
            a.ctrl->calls = call + 1;
        } else {
            *a.result = reverted;
        }
    }
}

template <int KIND>
hipError_t launch_count_force_k(const CountForceArgs& a, hipStream_t s)
{
    if (a.tries) {
        hipLaunchKernelGGL(count_force_list_kernel<KIND>, dim3(a.tries / kListThreads), dim3(kListThreads), 0, s, a);
        hipLaunchKernelGGL(count_force_bulk_kernel<KIND>, dim3(a.tries / kListThreads), dim3(kListThreads), 0, s, a);
        hipLaunchKernelGGL(count_force_commit_kernel<KIND>, dim3(1), dim3(kForceThreads), 0, s, a);
    }
    hipLaunchKernelGGL(count_force_finish_kernel<KIND>, dim3(1), dim3(kForceThreads), 0, s, a);
    return hipGetLastError();
}

}  // namespace

// A try is feasible with probability about d (1 - d), 0.12 at the density
// the viewers fill with: 16 tries per particle reach the amount as a rule.  The
// smallest amounts, the viewers' in their steady flow, are the finish kernel's
// alone, whose one launch costs less than four: us a call in four kernels / in
// one, 1480 x 740, amount 4 42.5 / 29.6, 64 42.6 / 28.7, 128 42.7 / 45.4, 1000 51.7 / 72.
uint32_t count_force_tries(uint64_t n, int64_t most)
{
    if (most <= kUnlisted) return 0;
    const uint64_t want = std::min<uint64_t>(16 * (uint64_t)most, kMaxSegments * kListThreads);
    const uint64_t tries = std::min<uint64_t>(std::max<uint64_t>(want, 4096), 2 * n);
    return (uint32_t)(tries / kListThreads * kListThreads);
}

size_t count_force_bytes(uint32_t tries) { return sizeof(ForceList) + (size_t)tries * 8; }

hipError_t launch_count_force(int kind, const CountForceArgs& a, hipStream_t s)
{
    if (a.tries % kListThreads || a.tries > kMaxSegments * kListThreads) return hipErrorInvalidValue;
    switch (kind) {
    case kHPP: return launch_count_force_k<kHPP>(a, s);
    case kFHP1: return launch_count_force_k<kFHP1>(a, s);
    default: return launch_count_force_k<kFHP2>(a, s);
    }
}

}  // namespace lgca
