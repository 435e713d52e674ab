// lgca_kernels.hip -- hand-written gfx950 kernels of the lattice-gas engine.
//
// The hot kernel is step_kernel: one fused pass per time step that pulls the
// hexagonal (or square) neighbourhood out of the bit-planes, collides, applies
// the solid-cell rules and the body force, and stores the next state.  Every
// (row, plane) word is read exactly once per step: a thread owns one 16-byte
// quad (128 cells) of one output row, loads the planes it pulls from rows
// y-1, y, y+1, and gets the one word of x-halo each shifted plane needs from
// the neighbouring lane (ds_bpermute), falling back to a global load only at
// workgroup-row edges.  The rest are small helper kernels (codec, masks, hash
// fill, force draws, post-processing, reductions).
#include "lgca_dev.hpp"
#include "lgca_kernels.hpp"

#include <algorithm>

namespace lgca {

static inline uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

__device__ __forceinline__ uint32_t valid_mask(const Geometry& g, uint32_t w)
{
    if (w + 1 < g.W) return 0xFFFFFFFFu;
    if (w + 1 == g.W) return g.nb == 32 ? 0xFFFFFFFFu : ((1u << g.nb) - 1u);
    return 0u;
}

__device__ __forceinline__ u32x4 ldq(const uint32_t* p) { return *(const u32x4*)p; }

__device__ __forceinline__ u32x4 valid_quad(const Geometry& g, uint32_t q)
{
    return u32x4{valid_mask(g, 4 * q), valid_mask(g, 4 * q + 1), valid_mask(g, 4 * q + 2),
                 valid_mask(g, 4 * q + 3)};
}

// ------------------------------------------------------------------ step

// Shifts one plane-row quad by one cell along x, cyclically over dim_x cells.
//   m1: out cell x = in cell x-1 (particles arriving from the west side)
//   p1: out cell x = in cell x+1
// `row` points at word 0 of the plane-row (for the halo fallback loads).
struct ShiftCtx {
    uint32_t lane, q, W, nb;
    bool has_left, has_right, has_last;  // has_last: quad holds word W-1
};

__device__ __forceinline__ u32x4 shift_quad(const u32x4 v, bool m1, const uint32_t* row,
                                            const ShiftCtx& c)
{
    const uint32_t send = m1 ? v.w : v.x;
    const int src = m1 ? (int)c.lane - 1 : (int)c.lane + 1;
    const uint32_t nbw = (uint32_t)__builtin_amdgcn_ds_bpermute(src << 2, (int)send);
    u32x4 o;
    if (m1) {
        uint32_t L;
        if (c.has_left) L = nbw;
        else if (c.q == 0) L = row[c.W - 1] << (32u - c.nb);  // cell dim_x-1 wraps to x = 0
        else L = row[4 * c.q - 1];
        o.x = __builtin_amdgcn_alignbit(v.x, L, 31);
        o.y = __builtin_amdgcn_alignbit(v.y, v.x, 31);
        o.z = __builtin_amdgcn_alignbit(v.z, v.y, 31);
        o.w = __builtin_amdgcn_alignbit(v.w, v.z, 31);
    } else {
        uint32_t R = 0;
        if (c.has_right) R = nbw;
        else if (4 * c.q + 4 < c.W) R = row[4 * c.q + 4];
        o.x = __builtin_amdgcn_alignbit(v.y, v.x, 1);
        o.y = __builtin_amdgcn_alignbit(v.z, v.y, 1);
        o.z = __builtin_amdgcn_alignbit(v.w, v.z, 1);
        o.w = __builtin_amdgcn_alignbit(R, v.w, 1);
        if (c.has_last) {
            // cell 0 wraps to x = dim_x - 1, bit nb-1 of word W-1
            const uint32_t k = c.W - 1 - 4 * c.q;
            const uint32_t carry = (row[0] & 1u) << (c.nb - 1u);
            if (k == 0) o.x = (v.x >> 1) | carry;
            else if (k == 1) o.y = (v.y >> 1) | carry;
            else if (k == 2) o.z = (v.z >> 1) | carry;
            else o.w = (v.w >> 1) | carry;
        }
    }
    return o;
}

template <int KIND>
__global__ __launch_bounds__(256) void step_kernel(StepArgs a)
{
    constexpr int Q = num_dir_of_kind(KIND);
    const Geometry& g = a.g;
    const uint32_t qb = 1u << g.qb_log;
    const uint32_t lane_row = threadIdx.x & (qb - 1u);
    const uint32_t q = (blockIdx.x << g.qb_log) | lane_row;
    const uint32_t y = blockIdx.y * (256u >> g.qb_log) + (threadIdx.x >> g.qb_log);
    if (q >= g.Wq || y >= g.dim_y) return;

    ShiftCtx c;
    c.lane = threadIdx.x & 63u;
    c.q = q;
    c.W = g.W;
    c.nb = g.nb;
    c.has_left = lane_row != 0;
    c.has_right = lane_row != qb - 1u && q + 1 < g.Wq;
    c.has_last = 4 * q <= g.W - 1 && g.W - 1 < 4 * q + 4;

    const uint32_t ym = y ? y - 1 : g.dim_y - 1;
    const uint32_t yp = (y + 1 == g.dim_y) ? 0 : y + 1;
    const bool odd = (y & 1u) != 0;
    const uint32_t* src = a.src;
    auto rowp = [&](uint32_t row, int d) { return src + ((size_t)row * Q + d) * g.P; };

    // Pull stream (src/omp_lattice.cpp:141-180; sources per direction as
    // the torus neighbours of the reference's offset tables).
    u32x4 in[7];
    if (KIND == kHPP) {
        in[0] = shift_quad(ldq(rowp(y, 0) + 4 * q), true, rowp(y, 0), c);   // from (x-1, y)
        in[1] = ldq(rowp(ym, 1) + 4 * q);                                    // from (x, y-1)
        in[2] = shift_quad(ldq(rowp(y, 2) + 4 * q), false, rowp(y, 2), c);  // from (x+1, y)
        in[3] = ldq(rowp(yp, 3) + 4 * q);                                    // from (x, y+1)
    } else {
        // dir 0 from (x-1, y), dir 3 from (x+1, y), rest in place.
        // even rows: 1 from (x-1, y-1), 2 from (x, y-1), 4 from (x, y+1), 5 from (x-1, y+1)
        // odd rows:  1 from (x, y-1),   2 from (x+1, y-1), 4 from (x+1, y+1), 5 from (x, y+1)
        const u32x4 a0 = ldq(rowp(y, 0) + 4 * q), a3 = ldq(rowp(y, 3) + 4 * q);
        const u32x4 b1 = ldq(rowp(ym, 1) + 4 * q), b2 = ldq(rowp(ym, 2) + 4 * q);
        const u32x4 c4 = ldq(rowp(yp, 4) + 4 * q), c5 = ldq(rowp(yp, 5) + 4 * q);
        if (Q == 7) in[6] = ldq(rowp(y, 6) + 4 * q);
        in[0] = shift_quad(a0, true, rowp(y, 0), c);
        in[3] = shift_quad(a3, false, rowp(y, 3), c);
        const u32x4 sb = shift_quad(odd ? b2 : b1, !odd, rowp(ym, odd ? 2 : 1), c);
        const u32x4 sc = shift_quad(odd ? c4 : c5, !odd, rowp(yp, odd ? 4 : 5), c);
        in[1] = odd ? b1 : sb;
        in[2] = odd ? sb : b2;
        in[4] = odd ? sc : c4;
        in[5] = odd ? c5 : sc;
    }

    u32x4 s[7];
#pragma unroll
    for (int d = 0; d < Q; ++d) s[d] = in[d];

    // Chirality word of word w: philox({w, y, step >> 2, 0})[step & 3].
    u32x4 p = {0, 0, 0, 0};
    if (KIND != kHPP) {
        const uint32_t sel = a.step & 3u;
        uint32_t pw[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const U4 ch = philox4x32_10(4 * q + k, y, a.step >> 2, 0u, a.key0, a.key1);
            pw[k] = sel == 0 ? ch.x : (sel == 1 ? ch.y : (sel == 2 ? ch.z : ch.w));
        }
        p = u32x4{pw[0], pw[1], pw[2], pw[3]};
    }
    collide<KIND, u32x4>(s, p);

    // Solid cells (rows without non-fluid cells skip the mask load).
    u32x4 fluid = {~0u, ~0u, ~0u, ~0u};
    if (a.mask) {
        const int lo = a.row_range[y], hi = a.row_range[g.dim_y + y];
        if ((int)(4 * q) < hi && (int)(4 * q + 4) > lo) {
            const u32x4 ns = ldq(a.mask + ((size_t)y * 2 + 0) * g.P + 4 * q);
            const u32x4 sl = ldq(a.mask + ((size_t)y * 2 + 1) * g.P + 4 * q);
            u32x4 edge = {q == 0 ? 1u : 0u, 0u, 0u, 0u};
            if (c.has_last) {
                const uint32_t k = g.W - 1 - 4 * q, b = 1u << (g.nb - 1u);
                edge.x |= k == 0 ? b : 0u;
                edge.y |= k == 1 ? b : 0u;
                edge.z |= k == 2 ? b : 0u;
                edge.w |= k == 3 ? b : 0u;
            }
            apply_solids<KIND, u32x4>(s, in, ns, sl, edge, y == 0 || y + 1 == g.dim_y);
            fluid = ~(ns | sl);
        }
    }

    // Body force on this quad's FLUID cells (decisions drawn ahead of time).
    if (a.fdec && y >= a.fy0 && y < a.fy1 && 4 * q < a.fw0 + a.fwn && 4 * q + 4 > a.fw0) {
        const uint32_t* drow = a.fdec + (size_t)(y - a.fy0) * a.fwn;
        u32x4 fd;
        fd.x = (4 * q + 0 >= a.fw0 && 4 * q + 0 < a.fw0 + a.fwn) ? drow[4 * q + 0 - a.fw0] : 0u;
        fd.y = (4 * q + 1 >= a.fw0 && 4 * q + 1 < a.fw0 + a.fwn) ? drow[4 * q + 1 - a.fw0] : 0u;
        fd.z = (4 * q + 2 >= a.fw0 && 4 * q + 2 < a.fw0 + a.fwn) ? drow[4 * q + 2 - a.fw0] : 0u;
        fd.w = (4 * q + 3 >= a.fw0 && 4 * q + 3 < a.fw0 + a.fwn) ? drow[4 * q + 3 - a.fw0] : 0u;
        apply_force<KIND, u32x4>(s, fd & fluid, a.force_dir);
    }

    const u32x4 vm = valid_quad(g, q);
    uint32_t* dst = a.dst;
#pragma unroll
    for (int d = 0; d < Q; ++d) *(u32x4*)(dst + ((size_t)y * Q + d) * g.P + 4 * q) = s[d] & vm;
}

hipError_t launch_step(int kind, const StepArgs& a, hipStream_t s)
{
    const uint32_t qb = 1u << a.g.qb_log;
    const dim3 grid(div_up(a.g.Wq, qb), div_up(a.g.dim_y, 256u / qb));
    switch (kind) {
    case kHPP: hipLaunchKernelGGL(step_kernel<kHPP>, grid, dim3(256), 0, s, a); break;
    case kFHP1: hipLaunchKernelGGL(step_kernel<kFHP1>, grid, dim3(256), 0, s, a); break;
    default: hipLaunchKernelGGL(step_kernel<kFHP2>, grid, dim3(256), 0, s, a); break;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------ force draws
// Decision words of steps [step0, step0 + nsteps) of the forced rows and
// words: bit b of word (step, y, w) forces cell 32w + b (see draw_chunk).
// Groups of four steps follow step >> 2 (steps mod 2^32).

__global__ __launch_bounds__(kDrawThreads) void force_draw_kernel(ForceDrawArgs a)
{
    // grid: x over chunks of (row, word) pairs of the force region, y over groups
    __shared__ DrawShared sh;
    force_table(sh.nQ, a.q);
    DrawRegion r{};
    r.dec = a.dec;
    r.plane = (uint64_t)(a.fy1 - a.fy0) * a.fwn;
    r.nsteps = a.nsteps;
    r.step0 = a.step0;
    r.key0 = a.key0;
    r.key1 = a.key1;
    r.fx0 = a.fx0;
    r.fx1 = a.fx1;
    r.fy0 = a.fy0;
    r.fw0 = a.fw0;
    r.fwn = a.fwn;
    r.dim_x = a.dim_x;
    r.words = a.words;
    draw_chunk(r, (uint64_t)blockIdx.x * a.words, blockIdx.y, sh);
}

hipError_t launch_force_draw(const ForceDrawArgs& args, hipStream_t s)
{
    ForceDrawArgs a = args;
    const uint32_t groups = ((a.step0 & 3u) + a.nsteps + 3u) / 4u;
    const uint64_t n = (uint64_t)(a.fy1 - a.fy0) * a.fwn;
    a.words = draw_words((n + kDrawWords - 1) / kDrawWords * groups < kDrawFew, a.q);
    if ((n + a.words - 1) / a.words >= ((uint64_t)1 << 31) || groups > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(force_draw_kernel, dim3(div_up(n, a.words), groups), dim3(kDrawThreads), 0, s, a);
    return hipGetLastError();
}

// ------------------------------------------------------------------ codec
// One byte per cell to and from planes.  Bytes and planes cross memory once
// each, which is the bound; a lane therefore moves 16 bytes at a time.  A row
// starts at any byte (y * dim_x): loads are unaligned, as global memory takes
// them on this target, stores are aligned to the memory, and only the cells at a
// row's ends are moved byte by byte.  4100 x 2050, one byte at a time -> so:
// unpack 12.5 -> 8.0 us (6000 x 3000 23 -> 8.9), cell types 24 -> 5.4 us; pack of 8192 x 4096 71 -> 14 us.
// Workgroups are qx lanes wide (row_lanes) by 256 / qx rows.

constexpr uint32_t kCodecCells = 16;

// Lanes along x for rows of n items: as many, up to a wave, as leave at most
// an eighth of the lanes without work, and at least 8.
static uint32_t row_lanes(uint32_t n)
{
    uint32_t qx = 64;
    while (qx > 8 && div_up(n, qx) * qx > n + n / 8) qx >>= 1;
    return qx;
}

static dim3 row_grid(const Geometry& g, uint32_t n, uint32_t qx) { return dim3(div_up(n, qx), div_up(g.dim_y, 256u / qx)); }

struct Bytes16 {
    uint32_t v[4];
};

__device__ __forceinline__ Bytes16 load_bytes16(const uint8_t* p)
{
    Bytes16 r;
    __builtin_memcpy(&r, p, 16);
    return r;
}

// Bit d of 16 bytes, the byte of cell 0 first.
__device__ __forceinline__ uint32_t gather_bits(const Bytes16& c, int d)
{
    const uint32_t m = 0x01010101u;
    const uint32_t lo = __builtin_amdgcn_udot4((c.v[1] >> d) & m, 0x80402010u,
                                               __builtin_amdgcn_udot4((c.v[0] >> d) & m, 0x08040201u, 0u, false), false);
    const uint32_t hi = __builtin_amdgcn_udot4((c.v[3] >> d) & m, 0x80402010u,
                                               __builtin_amdgcn_udot4((c.v[2] >> d) & m, 0x08040201u, 0u, false), false);
    return lo | (hi << 8);
}

// Transpose of an 8 x 8 bit matrix, row r in byte r of hi:lo (the three swaps of
// Hacker's Delight, section 7-3).
__device__ __forceinline__ void transpose8(uint32_t& lo, uint32_t& hi)
{
    uint32_t t = (lo ^ (lo >> 7)) & 0x00AA00AAu, u = (hi ^ (hi >> 7)) & 0x00AA00AAu;
    lo ^= t ^ (t << 7);
    hi ^= u ^ (u << 7);
    t = (lo ^ (lo >> 14)) & 0x0000CCCCu;
    u = (hi ^ (hi >> 14)) & 0x0000CCCCu;
    lo ^= t ^ (t << 14);
    hi ^= u ^ (u << 14);
    t = (lo ^ (hi << 4)) & 0xF0F0F0F0u;
    lo ^= t;
    hi ^= t >> 4;
}

template <int Q>
__global__ __launch_bounds__(256) void pack_kernel(const uint8_t* __restrict__ st, uint32_t* __restrict__ planes,
                                                   Geometry g, uint32_t* err)
{
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    if (w >= g.P || y >= g.dim_y) return;
    uint32_t acc[Q] = {}, bad = 0;
    const uint8_t* row = st + (size_t)y * g.dim_x;
#pragma unroll
    for (uint32_t half = 0; half < 2; ++half) {
        const uint32_t x = 32 * w + kCodecCells * half;
        Bytes16 c = {};
        if (x + kCodecCells <= g.dim_x) c = load_bytes16(row + x);
        else
            for (uint32_t b = 0; x + b < g.dim_x; ++b) {
                const uint32_t v = (uint32_t)row[x + b] << (8 * (b & 3u));
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) c.v[k] |= b >> 2 == k ? v : 0u;
            }
        bad |= (c.v[0] | c.v[1] | c.v[2] | c.v[3]) & ((0xFFu << Q & 0xFFu) * 0x01010101u);
#pragma unroll
        for (int d = 0; d < Q; ++d) acc[d] |= gather_bits(c, d) << (16 * half);
    }
#pragma unroll
    for (int d = 0; d < Q; ++d) planes[((size_t)y * Q + d) * g.P + w] = acc[d];
    if (bad) atomicOr(err, 1u);
}

hipError_t launch_pack(const uint8_t* state, uint32_t* planes, const Geometry& g, uint32_t* err,
                       hipStream_t s)
{
    const uint32_t qx = row_lanes(g.P);
    const dim3 grid = row_grid(g, g.P, qx), block(qx, 256u / qx);
    switch (g.Q) {
    case 4: hipLaunchKernelGGL(pack_kernel<4>, grid, block, 0, s, state, planes, g, err); break;
    case 6: hipLaunchKernelGGL(pack_kernel<6>, grid, block, 0, s, state, planes, g, err); break;
    default: hipLaunchKernelGGL(pack_kernel<7>, grid, block, 0, s, state, planes, g, err); break;
    }
    return hipGetLastError();
}

// Q planes per lattice row (a state's, or the two of a type mask) to bytes; null
// planes are empty.  A lane writes 16 bytes that start at a multiple of 16 in
// memory (at cells x..x + 15, from up to two words of a plane) in each of
// kUnpackRows rows, all of whose words are in flight together.  Neighbouring
// lanes, through the workgroup and on to the next one, take neighbouring
// chunks: narrow workgroups over many rows read each 128-byte line of a plane
// several times.
constexpr uint32_t kUnpackRows = 4;

template <int Q>
__global__ __launch_bounds__(256) void unpack_kernel(const uint32_t* __restrict__ planes, uint8_t* __restrict__ st,
                                                     Geometry g, uint32_t chunks, uint32_t slab)
{
    // blockIdx.y picks a slab of row groups
    const uint32_t id = blockIdx.x * 256 + threadIdx.x;
    const uint32_t group = id / chunks, i = id - group * chunks;
    const uint32_t y0 = (blockIdx.y * slab + group) * kUnpackRows;
    if (group >= slab || y0 >= g.dim_y) return;
    uint32_t w[kUnpackRows][Q] = {}, n[kUnpackRows][Q] = {};
    int32_t x[kUnpackRows];  // the lattice is narrower than 2^30 cells
#pragma unroll
    for (uint32_t k = 0; k < kUnpackRows; ++k)
        x[k] = (int32_t)(kCodecCells * i) - (int32_t)((uintptr_t)(st + (size_t)min(y0 + k, g.dim_y - 1) * g.dim_x) & 15u);
    if (planes) {
#pragma unroll
        for (uint32_t k = 0; k < kUnpackRows; ++k) {
            const uint32_t at = min((uint32_t)max(x[k], 0) >> 5, g.W - 1);
            const uint32_t up = min((uint32_t)(x[k] + (int32_t)kCodecCells - 1) >> 5, g.W - 1);
            const uint32_t* row = planes + (size_t)min(y0 + k, g.dim_y - 1) * Q * g.P;
#pragma unroll
            for (int d = 0; d < Q; ++d, row += g.P) {
                w[k][d] = row[at];
                n[k][d] = row[up];
            }
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kUnpackRows; ++k) {
        const uint32_t y = y0 + k;
        if (y >= g.dim_y || x[k] >= (int32_t)g.dim_x) continue;
        // sixteen cells of each plane in the low half; a chunk that starts
        // before the row has its first cells at the top of it
        uint32_t pl[8] = {};
#pragma unroll
        for (int d = 0; d < Q; ++d)
            pl[d] = x[k] < 0 ? w[k][d] << (uint32_t)-x[k] : __builtin_amdgcn_alignbit(n[k][d], w[k][d], (uint32_t)x[k]);
        uint32_t c[4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            // byte h of every plane
            const uint32_t two = h ? 0x0c0c0501u : 0x0c0c0400u;
            c[2 * h] = __builtin_amdgcn_perm(pl[1], pl[0], two) | (__builtin_amdgcn_perm(pl[3], pl[2], two) << 16);
            c[2 * h + 1] = __builtin_amdgcn_perm(pl[5], pl[4], two) | (__builtin_amdgcn_perm(pl[7], pl[6], two) << 16);
            transpose8(c[2 * h], c[2 * h + 1]);
        }
        uint8_t* out = st + (size_t)y * g.dim_x;
        if (x[k] >= 0 && x[k] + (int32_t)kCodecCells <= (int32_t)g.dim_x) {
            *(u32x4*)(out + x[k]) = u32x4{c[0], c[1], c[2], c[3]};
        } else {
            const int32_t first = max(-x[k], 0), end = min((int32_t)kCodecCells, (int32_t)g.dim_x - x[k]);
#pragma unroll 1
            for (int32_t b = first; b < end; ++b) {
                const uint32_t v = b < 8 ? (b < 4 ? c[0] : c[1]) : (b < 12 ? c[2] : c[3]);
                out[x[k] + b] = (uint8_t)(v >> (8 * (b & 3)));
            }
        }
    }
}

template <int Q>
static hipError_t unpack_planes(const uint32_t* planes, uint8_t* out, const Geometry& g, hipStream_t s)
{
    const uint32_t chunks = div_up(g.dim_x + kCodecCells - 1, kCodecCells), groups = div_up(g.dim_y, kUnpackRows);
    const uint32_t slab = std::min(groups, std::max(1u, (1u << 30) / chunks));
    hipLaunchKernelGGL(unpack_kernel<Q>, dim3(div_up((uint64_t)chunks * slab, 256), div_up(groups, slab)), dim3(256), 0,
                       s, planes, out, g, chunks, slab);
    return hipGetLastError();
}

hipError_t launch_unpack(const uint32_t* planes, uint8_t* state, const Geometry& g, hipStream_t s)
{
    switch (g.Q) {
    case 4: return unpack_planes<4>(planes, state, g, s);
    case 6: return unpack_planes<6>(planes, state, g, s);
    default: return unpack_planes<7>(planes, state, g, s);
    }
}

// ------------------------------------------------------------- cell types

__global__ __launch_bounds__(256) void types_kernel(const uint8_t* __restrict__ types,
                                                    uint32_t* __restrict__ mask,
                                                    int32_t* __restrict__ row_range, Geometry g,
                                                    uint32_t* err)
{
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    if (w >= g.P || y >= g.dim_y) return;
    uint32_t ns = 0, sl = 0, bad = 0;
    const uint8_t* row = types + (size_t)y * g.dim_x;
#pragma unroll
    for (uint32_t half = 0; half < 2; ++half) {
        const uint32_t x = 32 * w + kCodecCells * half;
        if (x + kCodecCells <= g.dim_x) {
            const Bytes16 c = load_bytes16(row + x);
            const uint32_t any = c.v[0] | c.v[1] | c.v[2] | c.v[3];
            if (!any) continue;  // FLUID, as nearly all cells are
            const uint32_t t1 = gather_bits(c, 0), t2 = gather_bits(c, 1);
            if (!(any & 0xFCFCFCFCu) && !(t1 & t2)) {
                ns |= t1 << (16 * half);
                sl |= t2 << (16 * half);
                continue;
            }
        }
        for (uint32_t b = 0; b < kCodecCells && x + b < g.dim_x; ++b) {
            const uint32_t t = row[x + b];
            ns |= (uint32_t)(t == 1) << (16 * half + b);
            sl |= (uint32_t)(t == 2) << (16 * half + b);
            bad |= t > 2;
        }
    }
    mask[((size_t)y * 2 + 0) * g.P + w] = ns;
    mask[((size_t)y * 2 + 1) * g.P + w] = sl;
    if (ns | sl) {
        // one of a run of words with solid cells speaks for it at each end
        const unsigned long long some = __ballot(true);
        const uint32_t lane = (threadIdx.y * blockDim.x + threadIdx.x) & 63u, at = threadIdx.x & 63u;
        const bool before = at && ((some >> (lane - 1u)) & 1ull), after = at + 1u < blockDim.x && lane < 63u && ((some >> (lane + 1u)) & 1ull);
        if (!before) atomicMin(row_range + y, (int32_t)w);
        if (!after) atomicMax(row_range + g.dim_y + y, (int32_t)w + 1);
    }
    if (bad) atomicOr(err, 1u);
}

hipError_t launch_types(const uint8_t* types, uint32_t* mask, int32_t* row_range,
                        const Geometry& g, uint32_t* err, hipStream_t s)
{
    const uint32_t qx = row_lanes(g.P);
    hipLaunchKernelGGL(types_kernel, row_grid(g, g.P, qx), dim3(qx, 256u / qx), 0, s, types, mask, row_range, g, err);
    return hipGetLastError();
}

hipError_t launch_types_unpack(const uint32_t* mask, uint8_t* types, const Geometry& g,
                               hipStream_t s)
{
    return unpack_planes<2>(mask, types, g, s);
}

// ------------------------------------------------------------ hash fill
// init_random (src/lattice.cpp:198-217) with the draw of cell (x, y),
// direction d = philox({x>>2, y, d, 2})[x & 3] < thr, on FLUID cells only.
// Bound by the hash, one call per four bits: 4100 x 2050, 38 -> 31 us with the
// eight calls of a word in flight together and 32-bit comparisons.

__global__ __launch_bounds__(256) void init_fill_kernel(uint32_t* __restrict__ planes,
                                                        const uint32_t* __restrict__ mask,
                                                        const uint8_t* __restrict__ region,
                                                        Geometry g, uint32_t key0, uint32_t key1,
                                                        uint64_t thr, uint32_t planes_each)
{
    const uint32_t w = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    if (w >= g.W || y >= g.dim_y) return;
    uint32_t fluid = valid_mask(g, w);
    if (mask)
        fluid &= ~(mask[((size_t)y * 2 + 0) * g.P + w] | mask[((size_t)y * 2 + 1) * g.P + w]);
    if (region) {
        uint32_t sel = 0;
        for (uint32_t b = 0; b < 32; ++b) {
            const uint32_t x = 32 * w + b;
            if (x >= g.dim_x) break;
            sel |= (uint32_t)(region[(size_t)y * g.dim_x + x] != 0) << b;
        }
        fluid &= sel;
    }
    for (uint32_t d = blockIdx.z * planes_each; d < min(g.Q, (blockIdx.z + 1) * planes_each); ++d) {
        const uint32_t word = fill_word(w, y, d, key0, key1, thr);
        uint32_t* p = planes + ((size_t)y * g.Q + d) * g.P + w;
        *p = (word & fluid) | (*p & ~fluid);
    }
}

hipError_t launch_init_fill(uint32_t* planes, const uint32_t* mask, const uint8_t* region,
                            const Geometry& g, uint32_t key0, uint32_t key1, uint64_t thr,
                            hipStream_t s)
{
    const uint32_t qx = row_lanes(g.W);
    dim3 grid = row_grid(g, g.W, qx);
    // A lane fills one plane's word while the lattice has few words, so that the
    // last workgroups do not run alone (4100 x 2050: 31 us, 34 with a lane per
    // word), and all planes' words above, reading the masks once (32768 x 8192:
    // 650 us, 732 with a lane per plane).
    const bool split = (uint64_t)grid.x * grid.y < 4096;
    if (split) grid.z = g.Q;
    hipLaunchKernelGGL(init_fill_kernel, grid, dim3(qx, 256u / qx), 0, s, planes, mask, region, g, key0, key1, thr,
                       split ? 1u : g.Q);
    return hipGetLastError();
}

// ---------------------------------------------------------- post-process
// Lattice vectors (src/lgca_models.h:51-52, 246-247, 453-454): per cell the
// momentum is an exact multiple of (1/2, sin(pi/3)) for FHP and of 1 for HPP,
// so the reference's running FP32 sums over directions are reproduced by
// integer weights times one FP32 constant.
__device__ constexpr float kSin60 = 0.866025388240814208984375f;  // (float)sin(pi/3)

template <int KIND>
__device__ __forceinline__ void cell_values(const uint32_t* s, int& rho, float& mx, float& my)
{
    if (KIND == kHPP) {
        rho = (int)(s[0] + s[1] + s[2] + s[3]);
        mx = (float)((int)s[0] - (int)s[2]);
        my = (float)((int)s[1] - (int)s[3]);
    } else {
        rho = (int)(s[0] + s[1] + s[2] + s[3] + s[4] + s[5]);
        if (KIND == kFHP2) rho += (int)s[6];
        const int kx = 2 * (int)s[0] + (int)s[1] - (int)s[2] - 2 * (int)s[3] - (int)s[4] + (int)s[5];
        const int ky = (int)s[1] + (int)s[2] - (int)s[4] - (int)s[5];
        mx = 0.5f * (float)kx;
        my = (float)ky * kSin60;
    }
}

// A wave owns kFieldCells cells of a row, lane l the cells l and l + 64: the
// planes' words are the same for the whole wave, so they are scalar loads whose
// 64 bits select a lane's value, and each store covers 64 neighbouring cells.
// Bound by the 12 bytes a cell that it writes: 4400 x 2200, 109 us with a lane
// per word (stores 128 and 256 bytes apart), 21 us so.
constexpr uint32_t kFieldCells = 128;

template <int KIND>
__global__ __launch_bounds__(256) void cell_fields_kernel(const uint32_t* __restrict__ planes,
                                                          Geometry g, float* __restrict__ dens,
                                                          float* __restrict__ mom)
{
    constexpr int Q = num_dir_of_kind(KIND);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t x0 = kFieldCells * (4 * blockIdx.x + wave), y = blockIdx.y;
    if (x0 >= g.dim_x) return;
    uint64_t pl[Q][2];  // four words of every plane: the pitch is a multiple of four words
#pragma unroll
    for (int d = 0; d < Q; ++d) {
        const u32x4 v = ldq(planes + ((size_t)y * Q + d) * g.P + (x0 >> 5));
        pl[d][0] = v.x | (uint64_t)v.y << 32;
        pl[d][1] = v.z | (uint64_t)v.w << 32;
    }
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
        uint32_t s[Q];
#pragma unroll
        for (int d = 0; d < Q; ++d) s[d] = __builtin_amdgcn_inverse_ballot_w64(pl[d][k]) ? 1u : 0u;
        int rho;
        float mx, my;
        cell_values<KIND>(s, rho, mx, my);
        const uint32_t x = x0 + 64 * k + lane;
        if (x >= g.dim_x) return;
        const size_t cell = (size_t)y * g.dim_x + x;
        if (dens) dens[cell] = (float)rho;
        if (mom) ((float2*)mom)[cell] = make_float2(mx, my);
    }
}

hipError_t launch_cell_fields(int kind, const uint32_t* planes, const Geometry& g, float* density,
                              float* momentum, hipStream_t s)
{
    const dim3 grid(div_up(g.dim_x, 4 * kFieldCells), g.dim_y);
    switch (kind) {
    case kHPP: hipLaunchKernelGGL(cell_fields_kernel<kHPP>, grid, dim3(256), 0, s, planes, g, density, momentum); break;
    case kFHP1: hipLaunchKernelGGL(cell_fields_kernel<kFHP1>, grid, dim3(256), 0, s, planes, g, density, momentum); break;
    default: hipLaunchKernelGGL(cell_fields_kernel<kFHP2>, grid, dim3(256), 0, s, planes, g, density, momentum); break;
    }
    return hipGetLastError();
}

// Coarse graining (src/omp_lattice.cpp:397-454).  Coarse cell c has its corner
// at (2r * (c % cdx), 2r * (c / cdx)); it sums, y-outer and x-inner, the cells
// of columns x0..x0+r on rows y0..y0+2r that exist, plus -- only when
// dim_x == 2r -- the candidate x = 2r of each row, which wraps to column 0 of
// the next row.  Sums are sequential FP32 in that order; one divide by the
// count.
//
// Density and x momentum (and HPP's y momentum) are sums of multiples of 1/2
// that FP32 holds exactly for r up to kCoarseExactRadius, so any order gives
// their bits and popcounts give the sums.  The y momentum of FHP rounds at
// every cell: its chain of (2r + 1)(r + 1) dependent adds is the kernel's
// bound (2145 adds at r = 32).  So one wave of a workgroup does nothing else,
// one chain per lane for 64 coarse cells, with the addends already in LDS in
// the order it needs; the other kCoarseProducers waves read the planes, up
// to kCoarseColumns columns of a row at a time (a unit), turn them into addends
// and keep the popcounts.  An 8192 x 4096 lattice at r = 32: 242 us with one
// thread per coarse cell doing all of it, waiting out a memory latency per
// word, 52 us with units of 16 columns (twice the stages, whose barriers and
// loads' latency count), 26 us so (4400 x 2200 at r = 20: 113, 25 and 15 us;
// 1480 x 740 at r = 10: 36, 9.9 and 7.8 us).  The producers' arithmetic bounds
// it: loads two stages ahead in place of one make no difference.

// Addends of the y-momentum chain for the cells of one unit, zeros past its
// end: bit j of the four planes is cell j; out[j] = ky * sin(pi/3), ky = a1 + a2 - a4 - a5,
// exact.  The float's bits are put together from three planes: zero or not,
// |ky| == 2 (exponent one up), sign.
__device__ __forceinline__ void y_addends(uint32_t a1, uint32_t a2, uint32_t a4, uint32_t a5, uint32_t quads,
                                          float4* out)
{
    const uint32_t p1 = a1 ^ a2, p2 = a1 & a2, n1 = a4 ^ a5, n2 = a4 & a5;
    uint32_t nz = (p1 ^ n1) | (p2 ^ n2);
    uint32_t two = (p2 & ~(n1 | n2)) | (n2 & ~(p1 | p2));
    uint32_t neg = (n2 & ~p2) | (n1 & ~(p1 | p2));
    const uint32_t one = __float_as_uint(kSin60);
    for (uint32_t k = 0; k < quads; ++k) {
        float f[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t v = ((neg << (31 - j)) & 0x80000000u) | ((two << (23 - j)) & 0x00800000u) | one;
            f[j] = __uint_as_float(v & (uint32_t)__builtin_amdgcn_sbfe((int)nz, j, 1));
        }
        out[k * 64] = make_float4(f[0], f[1], f[2], f[3]);
        nz >>= 4;
        two >>= 4;
        neg >>= 4;
    }
}

template <int KIND>
__global__ __launch_bounds__(64 * (1 + kCoarseProducers))
void coarse_kernel(const uint32_t* __restrict__ planes, Geometry g, uint32_t r, uint32_t chunks, uint32_t chunk,
                   float* __restrict__ md, float* __restrict__ mm, float* __restrict__ vel,
                   float* __restrict__ host)
{
    constexpr int Q = num_dir_of_kind(KIND);
    constexpr bool kChain = KIND != kHPP;
    // [2 stages][producer][chunk / 4 quads][64 coarse cells] addends
    extern __shared__ float4 addends[];
    __shared__ int sums[kCoarseProducers][3][64];
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t cdx = g.dim_x / (2 * r), cdy = g.dim_y / (2 * r), nc = cdx * cdy;
    const uint32_t c = blockIdx.x * 64 + lane;
    const bool live = c < nc;
    const uint32_t x0 = live ? (c % cdx) * 2 * r : 0u, y0 = live ? (c / cdx) * 2 * r : 0u;
    const bool wrap_col = g.dim_x == 2 * r;
    const uint32_t per_row = chunks + (wrap_col ? 1u : 0u), units = (2 * r + 1) * per_row;
    const uint32_t stages = (units + kCoarseProducers - 1) / kCoarseProducers;
    const uint32_t slot = chunk / 4 * 64;  // float4s of one unit
    // cells of a unit: `chunk` columns of the row, the rest of the r + 1 in
    // the last chunk, and the wrapped cell
    auto unit_cells = [&](uint32_t i) {
        return i >= chunks ? 1u : i + 1 == chunks ? r + 1 - (chunks - 1) * chunk : chunk;
    };

    int rho = 0, kx = 0, ky = 0;  // producers: density, x momentum in halves (HPP: ones), HPP y momentum
    float sy = 0.0f;              // wave 0: the chain
    uint32_t word[3][Q];          // producers: the unit's plane words, loaded a stage ahead
    auto load_unit = [&](uint32_t u) {
        const uint32_t i = u % per_row, n = unit_cells(i);
        const uint32_t y = y0 + u / per_row + (i >= chunks ? 1u : 0u), x = i >= chunks ? 0u : x0 + i * chunk;
        const bool ok = live && u < units && y < g.dim_y;
        const uint32_t* p = planes + (size_t)y * Q * g.P + (x >> 5);
        const bool two = ok && (x & 31u) + n > 32, three = ok && (x & 31u) + n > 64;
#pragma unroll
        for (int d = 0; d < Q; ++d) {
            word[0][d] = ok ? p[(size_t)d * g.P] : 0u;
            word[1][d] = two ? p[(size_t)d * g.P + 1] : 0u;
            word[2][d] = three ? p[(size_t)d * g.P + 2] : 0u;
        }
    };
    if (wave) load_unit(wave - 1);
    else __builtin_amdgcn_s_setprio(3);  // every add of the chain waits for the last one
    for (uint32_t st = 0; st <= stages; ++st) {
        if (wave && st < stages) {
            const uint32_t u = st * kCoarseProducers + wave - 1, i = u % per_row, n = unit_cells(i);
            const uint32_t sh = i >= chunks ? 0u : (x0 + i * chunk) & 31u;
            // the unit's first 32 cells and the rest
            const uint32_t valid = n >= 32 ? 0xFFFFFFFFu : (1u << n) - 1u, rest = n > 32 ? (1u << (n - 32u)) - 1u : 0u;
            uint32_t a[Q], e[Q];
#pragma unroll
            for (int d = 0; d < Q; ++d) {
                a[d] = __builtin_amdgcn_alignbit(word[1][d], word[0][d], sh) & valid;
                e[d] = __builtin_amdgcn_alignbit(word[2][d], word[1][d], sh) & rest;
            }
            if (st + 1 < stages) load_unit(u + kCoarseProducers);
            auto count = [&](const uint32_t* v) {
#pragma unroll
                for (int d = 0; d < Q; ++d) rho += __popc(v[d]);
                if (KIND == kHPP) {
                    kx += __popc(v[0]) - __popc(v[2]);
                    ky += __popc(v[1]) - __popc(v[3]);
                } else {
                    kx += 2 * (__popc(v[0]) - __popc(v[3])) + __popc(v[1]) - __popc(v[2]) - __popc(v[4]) + __popc(v[5]);
                }
            };
            count(a);
            if (n > 32) count(e);
            if (kChain) {
                float4* out = addends + ((st & 1u) * kCoarseProducers + wave - 1) * slot + lane;
                y_addends(a[1], a[2], a[4], a[5], min(chunk, 32u) / 4, out);
                if (chunk > 32) y_addends(e[1], e[2], e[4], e[5], (chunk - 32) / 4, out + 8 * 64);
            }
        }
        if (kChain && !wave && st) {
            // the stage's addends are one stream: the next kChainAhead quads
            // are on their way from LDS while the chain takes the last ones
            const uint32_t quads = min(kCoarseProducers, units - (st - 1) * kCoarseProducers) * (chunk / 4);
            const float4* a = addends + ((st - 1) & 1u) * kCoarseProducers * slot + lane;
            float4 even[kChainAhead], odd[kChainAhead];
            auto fetch = [&](float4 (&v)[kChainAhead], uint32_t q) {
#pragma unroll
                for (uint32_t k = 0; k < kChainAhead; ++k) v[k] = a[(q + k) * 64];
            };
            auto take = [&](const float4 (&v)[kChainAhead], uint32_t q) {
#pragma unroll
                for (uint32_t k = 0; k < kChainAhead; ++k) {
                    if (q + k >= quads) return;
                    sy += v[k].x;
                    sy += v[k].y;
                    sy += v[k].z;
                    sy += v[k].w;
                }
            };
            fetch(even, 0);
            for (uint32_t q = 0; q < quads; q += 2 * kChainAhead) {
                fetch(odd, q + kChainAhead);
                take(even, q);
                fetch(even, q + 2 * kChainAhead);
                take(odd, q + kChainAhead);
            }
        }
        if (kChain) __syncthreads();
    }
    if (wave) {
        sums[wave - 1][0][lane] = rho;
        sums[wave - 1][1][lane] = kx;
        sums[wave - 1][2][lane] = ky;
    }
    __syncthreads();
    if (wave || !live) return;
    for (uint32_t p = 0; p < kCoarseProducers; ++p) {
        rho += sums[p][0][lane];
        kx += sums[p][1][lane];
        ky += sums[p][2][lane];
    }
    const uint32_t rows = min(2 * r + 1, g.dim_y - y0);
    const uint32_t wrapped = wrap_col ? min(rows, g.dim_y - 1 - y0) : 0u;
    const float fc = (float)(int)(rows * (r + 1) + wrapped);
    const float sd = (float)rho, sx = KIND == kHPP ? (float)kx : 0.5f * (float)kx;
    if (KIND == kHPP) sy = (float)ky;
    const float den = sd / fc, ux = sx / fc, uy = sy / fc;
    md[c] = den;
    mm[2 * c] = ux;
    mm[2 * c + 1] = uy;
    if (host) {
        host[c] = den;
        host[nc + 2 * c] = ux;
        host[nc + 2 * c + 1] = uy;
    }
    if (vel) {
        vel[2 * c] = den > 0.0f ? ux / den : 0.0f;
        vel[2 * c + 1] = den > 0.0f ? uy / den : 0.0f;
    }
}

// The same one cell at a time, one thread per coarse cell: for radii whose
// density sums FP32 may round (more than 2^24 particles in a window), and where
// many small cells fill the GPU with lanes (coarse_in_units).
template <int KIND>
__global__ __launch_bounds__(64) void coarse_lane_kernel(const uint32_t* __restrict__ planes,
                                                          Geometry g, uint32_t r,
                                                          float* __restrict__ md, float* __restrict__ mm,
                                                          float* __restrict__ vel, float* __restrict__ host)
{
    constexpr int Q = num_dir_of_kind(KIND);
    const uint32_t cdx = g.dim_x / (2 * r), cdy = g.dim_y / (2 * r);
    const uint32_t c = blockIdx.x * 64 + threadIdx.x;
    if (c >= cdx * cdy) return;
    const uint32_t x0 = (c % cdx) * 2 * r, y0 = (c / cdx) * 2 * r;
    const bool wrap_col = g.dim_x == 2 * r;
    float sd = 0.0f, sx = 0.0f, sy = 0.0f;
    int cnt = 0;
    uint32_t pl[7];
    auto visit = [&](uint32_t x, uint32_t y) {
        int rho;
        float mx, my;
        uint32_t b[7];
#pragma unroll
        for (int d = 0; d < Q; ++d) b[d] = (pl[d] >> (x & 31u)) & 1u;
        cell_values<KIND>(b, rho, mx, my);
        sd += (float)rho;
        sx += mx;
        sy += my;
        ++cnt;
    };
    for (uint32_t yy = 0; yy <= 2 * r; ++yy) {
        const uint32_t y = y0 + yy;
        if (y >= g.dim_y) break;
        uint32_t cur_w = 0xFFFFFFFFu;
        for (uint32_t x = x0; x <= x0 + r; ++x) {
            if ((x >> 5) != cur_w) {
                cur_w = x >> 5;
#pragma unroll
                for (int d = 0; d < Q; ++d) pl[d] = planes[((size_t)y * Q + d) * g.P + cur_w];
            }
            visit(x, y);
        }
        if (wrap_col && y + 1 < g.dim_y) {
#pragma unroll
            for (int d = 0; d < Q; ++d) pl[d] = planes[((size_t)(y + 1) * Q + d) * g.P];
            visit(0, y + 1);
        }
    }
    const float fc = (float)cnt;
    const float rho = sd / fc, ux = sx / fc, uy = sy / fc;
    md[c] = rho;
    mm[2 * c] = ux;
    mm[2 * c + 1] = uy;
    if (host) {
        host[c] = rho;
        host[cdx * cdy + 2 * c] = ux;
        host[cdx * cdy + 2 * c + 1] = uy;
    }
    if (vel) {
        vel[2 * c] = rho > 0.0f ? ux / rho : 0.0f;
        vel[2 * c + 1] = rho > 0.0f ? uy / rho : 0.0f;
    }
}

hipError_t launch_coarse(int kind, const uint32_t* planes, const Geometry& g, uint32_t r, uint32_t ncu,
                         float* mean_density, float* mean_momentum, float* velocity, float* host, hipStream_t s)
{
    const uint32_t n = (g.dim_x / (2 * r)) * (g.dim_y / (2 * r));
    const dim3 grid(div_up(n, 64));
    if (!coarse_in_units(kind, r, n, ncu)) {
        switch (kind) {
        case kHPP: hipLaunchKernelGGL(coarse_lane_kernel<kHPP>, grid, dim3(64), 0, s, planes, g, r, mean_density, mean_momentum, velocity, host); break;
        case kFHP1: hipLaunchKernelGGL(coarse_lane_kernel<kFHP1>, grid, dim3(64), 0, s, planes, g, r, mean_density, mean_momentum, velocity, host); break;
        default: hipLaunchKernelGGL(coarse_lane_kernel<kFHP2>, grid, dim3(64), 0, s, planes, g, r, mean_density, mean_momentum, velocity, host); break;
        }
        return hipGetLastError();
    }
    const CoarseUnits u = coarse_units(kind, r);
    const dim3 block(64 * (1 + kCoarseProducers));
    switch (kind) {
    case kHPP: hipLaunchKernelGGL(coarse_kernel<kHPP>, grid, block, u.lds, s, planes, g, r, u.chunks, u.chunk, mean_density, mean_momentum, velocity, host); break;
    case kFHP1: hipLaunchKernelGGL(coarse_kernel<kFHP1>, grid, block, u.lds, s, planes, g, r, u.chunks, u.chunk, mean_density, mean_momentum, velocity, host); break;
    default: hipLaunchKernelGGL(coarse_kernel<kFHP2>, grid, block, u.lds, s, planes, g, r, u.chunks, u.chunk, mean_density, mean_momentum, velocity, host); break;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------ reductions
// Sums over a whole lattice.  What bounds them is one pass over the planes; an
// atomic on one address takes about 11 ns however many waves make it, so
// every workgroup adds its waves up first and makes one atomic per sum, and
// the grid is at most one workgroup of kReduceThreads per CU.  With one atomic
// per wave (16,384 and 49,152 of them on an 8192 x 4096 FHP-II lattice, 29 MB)
// the count took 177 us and the mean velocity 597 us; so they take 8.6 and
// 13.7 us.
constexpr uint32_t kReduceThreads = 1024, kReduceBlocks = 256;

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Adds v of every thread of the workgroup to *out (n sums side by side).
template <int N>
__device__ __forceinline__ void block_add_u64(unsigned long long (&v)[N], unsigned long long* out)
{
    __shared__ unsigned long long part[kReduceThreads / 64][N];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        v[k] = wave_sum_u64(v[k]);
        if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6][k] = v[k];
    }
    __syncthreads();
    if (threadIdx.x < N) {
        unsigned long long t = 0;
        for (uint32_t w = 0; w < blockDim.x / 64; ++w) t += part[w][threadIdx.x];
        atomicAdd(out + threadIdx.x, t);
    }
}

__global__ __launch_bounds__(kReduceThreads) void count_kernel(const u32x4* __restrict__ quads, uint64_t n,
                                                               unsigned long long* out)
{
    unsigned long long acc[1] = {0};
    const uint64_t stride = (uint64_t)gridDim.x * kReduceThreads;
    for (uint64_t i = (uint64_t)blockIdx.x * kReduceThreads + threadIdx.x; i < n; i += 4 * stride) {
        u32x4 q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) q[k] = i + k * stride < n ? quads[i + k * stride] : u32x4{0, 0, 0, 0};
        uint32_t c = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) c += __popc(q[k].x) + __popc(q[k].y) + __popc(q[k].z) + __popc(q[k].w);
        acc[0] += c;
    }
    block_add_u64(acc, out);
}

// nwords is a state buffer's: rows are whole quads, and buffers 16-byte aligned.
hipError_t launch_count(const uint32_t* words, uint64_t nwords, unsigned long long* out,
                        hipStream_t s)
{
    const uint64_t n = nwords / 4;
    if (nwords % 4) return hipErrorInvalidValue;
    const uint32_t blocks = std::min(std::max(div_up(n, kReduceThreads), 1u), kReduceBlocks);
    hipLaunchKernelGGL(count_kernel, dim3(blocks), dim3(kReduceThreads), 0, s, (const u32x4*)words, n, out);
    return hipGetLastError();
}

// get_mean_velocity (src/omp_lattice.cpp:508-557), summed exactly: with
// density rho in 1..7, 840 * (momentum / rho) is an integer multiple of the
// unit (1 for HPP x and y, 1/2 for FHP x, sin(pi/3) for FHP y), so three
// 64-bit integer sums (x, y, FLUID count) give an order-independent result.
// A word of 32 cells is summed at once: the density's three bits come from a
// chain of full adders, and for every density the momentum of its cells is a
// few popcounts (about 100 operations a word, against 30 for each cell taken
// one by one).  A workgroup covers 1 << tw_log words of 1024 >> tw_log rows at a time.
template <int KIND>
__global__ __launch_bounds__(kReduceThreads) void mean_velocity_kernel(const uint32_t* __restrict__ planes,
                                                                       const uint32_t* __restrict__ mask,
                                                                       Geometry g, uint32_t tw_log,
                                                                       unsigned long long* acc)
{
    constexpr int Q = num_dir_of_kind(KIND);
    const uint32_t tw = 1u << tw_log, rows = kReduceThreads >> tw_log;
    unsigned long long sum[3] = {0, 0, 0};
    for (uint32_t y = blockIdx.x * rows + (threadIdx.x >> tw_log); y < g.dim_y; y += gridDim.x * rows) {
        for (uint32_t w = blockIdx.y * tw + (threadIdx.x & (tw - 1u)); w < g.W; w += gridDim.y * tw) {
            uint32_t fluid = valid_mask(g, w);
            if (mask)
                fluid &= ~(mask[((size_t)y * 2 + 0) * g.P + w] | mask[((size_t)y * 2 + 1) * g.P + w]);
            uint32_t s[7];
#pragma unroll
            for (int d = 0; d < Q; ++d) s[d] = planes[((size_t)y * Q + d) * g.P + w];
            // density bits of every cell
            uint32_t b0, b1, b2 = 0;
            if (KIND == kHPP) {
                const uint32_t x1 = bit3<kXor3>(s[0], s[1], s[2]), c1 = bit3<kMaj>(s[0], s[1], s[2]);
                b0 = x1 ^ s[3];
                const uint32_t c2 = x1 & s[3];
                b1 = c1 ^ c2;
                b2 = c1 & c2;
            } else {
                const uint32_t x1 = bit3<kXor3>(s[0], s[1], s[2]), c1 = bit3<kMaj>(s[0], s[1], s[2]);
                const uint32_t x2 = bit3<kXor3>(s[3], s[4], s[5]), c2 = bit3<kMaj>(s[3], s[4], s[5]);
                const uint32_t r = Q == 7 ? s[6] : 0u;
                b0 = bit3<kXor3>(x1, x2, r);
                const uint32_t c3 = bit3<kMaj>(x1, x2, r);
                b1 = bit3<kXor3>(c1, c2, c3);
                b2 = bit3<kMaj>(c1, c2, c3);
            }
            int sx = 0, sy = 0;
#pragma unroll
            for (int rho = 1; rho <= Q; ++rho) {
                const uint32_t m = fluid & (rho & 1 ? b0 : ~b0) & (rho & 2 ? b1 : ~b1) & (rho & 4 ? b2 : ~b2);
                int nx, ny;
                if (KIND == kHPP) {
                    nx = 2 * (__popc(m & s[0]) - __popc(m & s[2]));
                    ny = __popc(m & s[1]) - __popc(m & s[3]);
                } else {
                    const int n1 = __popc(m & s[1]), n2 = __popc(m & s[2]);
                    const int n4 = __popc(m & s[4]), n5 = __popc(m & s[5]);
                    nx = 2 * (__popc(m & s[0]) - __popc(m & s[3])) + n1 + n5 - n2 - n4;
                    ny = n1 + n2 - n4 - n5;
                }
                sx += nx * (420 / rho);  // 840 / rho is even for every rho
                sy += ny * (840 / rho);
            }
            sum[0] += (unsigned long long)(long long)sx;
            sum[1] += (unsigned long long)(long long)sy;
            sum[2] += __popc(fluid);
        }
    }
    block_add_u64(sum, acc);
}

hipError_t launch_mean_velocity(int kind, const uint32_t* planes, const uint32_t* mask,
                                const Geometry& g, long long* acc3, hipStream_t s)
{
    uint32_t tw_log = 0;
    while ((1u << tw_log) < g.W && (1u << tw_log) < kReduceThreads) ++tw_log;
    // a workgroup per row (or rows); flat lattices share long rows out too (20000000 x
    // 2 FHP-II 936 us a call with a workgroup per row, 28 so)
    dim3 grid(std::min(div_up(g.dim_y, kReduceThreads >> tw_log), kReduceBlocks)), block(kReduceThreads);
    grid.y = std::max(1u, std::min(div_up(g.W, 1u << tw_log), kReduceBlocks / grid.x));
    unsigned long long* acc = (unsigned long long*)acc3;
    switch (kind) {
    case kHPP: hipLaunchKernelGGL(mean_velocity_kernel<kHPP>, grid, block, 0, s, planes, mask, g, tw_log, acc); break;
    case kFHP1: hipLaunchKernelGGL(mean_velocity_kernel<kFHP1>, grid, block, 0, s, planes, mask, g, tw_log, acc); break;
    default: hipLaunchKernelGGL(mean_velocity_kernel<kFHP2>, grid, block, 0, s, planes, mask, g, tw_log, acc); break;
    }
    return hipGetLastError();
}

// Counters to pinned memory, and zero for their next use.
__global__ __launch_bounds__(64) void publish_kernel(unsigned long long* counters, unsigned long long* page, uint32_t n)
{
    if (threadIdx.x >= n) return;
    page[threadIdx.x] = counters[threadIdx.x];
    counters[threadIdx.x] = 0;
}

hipError_t launch_publish(unsigned long long* counters, unsigned long long* page, uint32_t n, hipStream_t s)
{
    hipLaunchKernelGGL(publish_kernel, dim3(1), dim3(64), 0, s, counters, page, n);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void copy_u32_kernel(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src,
                                                       uint64_t n)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

hipError_t launch_copy_u32(uint32_t* dst, const uint32_t* src, uint64_t n, hipStream_t s)
{
    if (n) hipLaunchKernelGGL(copy_u32_kernel, dim3(div_up(n, 256)), dim3(256), 0, s, dst, src, n);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* p, uint32_t v, uint64_t n)
{
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256)
        p[i] = v;
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t value, uint64_t n, hipStream_t s)
{
    uint32_t blocks = div_up(n, 256);
    if (blocks > 65535) blocks = 65535;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks), dim3(256), 0, s, p, value, n);
    return hipGetLastError();
}

}  // namespace lgca
