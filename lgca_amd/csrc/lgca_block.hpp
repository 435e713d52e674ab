// lgca_block.hpp -- temporally blocked collide-and-propagate for lattices
// whose passes the row walk of lgca_tile.hpp cannot fill the GPU with.
//
// A walk turns th + 2K rows into th stored ones one after the other, K
// dependent levels a row: on a lattice of a few thousand waves that chain is
// the whole pass.  Here a workgroup holds a block of rows in registers
// instead, M consecutive rows per wave (and per segment of a wave, where rows
// are short), one 32-cell word per lane, and all its waves advance them one
// step at a time.  A step needs two planes of the row above a wave's rows and
// two of the row below (the rest it holds itself): they pass through LDS, with
// one barrier per step.  The state crosses HBM once per pass.  us per step
// walked -> in blocks as they came -> now (packed lanes, 32-step collision):
// 256 x 256 HPP 0.78 -> 0.24, 1001 x 754 FHP-I slip box 3.06 -> 0.82 -> 0.80,
// 2048 x 512 FHP-II pipe 3.05 -> 1.13 -> 1.06, 4400 x 2200 FHP-III cylinder 5.2
// -> 2.4 -> 1.85, 6000 x 3000 FHP-II forced channel 8.0 -> 5.4 -> 4.1 (1.2 of it
// the force draws).
//
// What bounds it: on the small ones the launch and the first loads (3 us a
// pass) and each step's chain of dependent instructions through one barrier;
// on the larger ones VALU issue (51 instructions per wave-row and step, as the
// walk) with the halo rows' share of it.
//
// y-halo: the block reads hk >= K extra rows on either side of its th stored
// rows (hk even where M is, so that the hexagonal row parity is known at
// compile time).  The rows that the stored ones still depend on shrink by one on
// either side per step; waves with none of them left only keep the barrier.
// x-halo: as in lgca_tile.hpp (strips of 64 words with `halo` words either
// side that are not stored; whole rows in segment mode), or packed: the row
// tiles' words, `halo` either side of each tile's row included, form one
// sequence, and a wave takes 64 of it, so that the end of one tile's rows
// shares a wave with the start of the next one's.  Neighbours in the sequence
// are neighbours in the row except at the halos' outer ends, where strips have
// the same garbage.  A 188-word row takes 3.06 waves so, and 4 strips: 6000 x
// 3000 FHP-II 3.2 -> 2.5 us a step, 4400 x 2200 (138 words) 2.4 -> 2.0 (both
// with a 43-step collision; 2.2 and 1.85 now).
//
// Chirality: a row's Philox call serves its word for a group of four steps;
// the words wait in LDS (read once a step), which costs no registers and no
// selects.
#pragma once

#include "lgca_tile.hpp"

namespace lgca {

// A further segment mode, of blocks only: packed strips.
constexpr int kPacked = 3;

// One workgroup's block: strip `strip` of row tile `tile` (packed: `strip`
// counts the waves' shares of the sequence, and `tile` is unused), k steps with
// hk halo rows.  FEAT: 0 no solids and no forcing on the lattice, 1 either.  Every
// wave of the workgroup makes k + 1 barriers.
template <int KIND, int M, bool RAGGED, int SEG, int FEAT>
__device__ __forceinline__ void block_body(const TileArgs& a, uint32_t k, uint32_t hk, uint32_t strip, uint32_t tile,
                                           uint32_t* lds)
{
    constexpr int Q = num_dir_of_kind(KIND);
    constexpr uint32_t NX = KIND == kHPP ? 1 : 2;  // planes exchanged per direction
    constexpr bool kRows = SEG != kStrips;                    // rows differ from lane to lane
    constexpr bool kStacked = kRows && SEG != kPacked;        // segments hold one above the other
    constexpr int SHIFT = SEG == kPacked ? kStrips : SEG;     // where neighbouring words are
    const Geometry& g = a.g;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwave = blockDim.x >> 6;
    uint32_t y0 = tile * a.th, rows = min(a.th, g.dim_y - y0);  // packed: this lane's

    // this lane's word and the group of M rows it works on
    const uint32_t S = kStacked ? 64u / g.W : 1u;
    uint32_t group = wave;
    int wabs;
    bool writer;
    LaneCtx c;
    if (SEG == kPacked) {
        const uint32_t stride = 64u - 2u * a.halo, span = g.W + 2u * a.halo;
        const uint32_t total = (g.dim_y + a.th - 1) / a.th * span;
        const int f = (int)(strip * stride) - (int)a.halo + (int)lane;
        const uint32_t at = (uint32_t)min(max(f, 0), (int)total - 1), t = at / span;
        y0 = t * a.th;
        rows = min(a.th, g.dim_y - y0);
        wabs = (int)(at - t * span) - (int)a.halo;
        writer = lane >= a.halo && lane < 64u - a.halo && f < (int)total && wabs >= 0 && wabs < (int)g.W;
        c.lsrc = c.rsrc = 0;
    } else if (SEG) {
        const uint32_t seg = lane / g.W, base = seg * g.W;
        group = wave * S + min(seg, S - 1u);
        wabs = (int)(lane - base);
        writer = seg < S;
        c.lsrc = 4u * ((wabs == 0 ? base + g.W - 1u : lane - 1u) & 63u);
        c.rsrc = 4u * (((uint32_t)wabs + 1u == g.W ? base : lane + 1u) & 63u);
    } else {
        const uint32_t stride = 64u - 2u * a.halo;
        wabs = (int)(strip * stride) - (int)a.halo + (int)lane;
        writer = lane >= a.halo && lane < 64u - a.halo && wabs < (int)g.W;
        c.lsrc = c.rsrc = 0;
    }
    c.w = (uint32_t)((wabs + (int)g.W) % (int)g.W);
    c.wb = 4u * c.w;
    c.nb = g.nb;
    c.first_shl = c.w == 0 ? 32u - g.nb : 0u;
    const uint32_t last_bit = c.w + 1 == g.W ? 1u << (g.nb - 1u) : 0u;
    c.last_bit = last_bit;
    c.vmask = (last_bit && g.nb < 32) ? ((1u << g.nb) - 1u) : 0xFFFFFFFFu;
    const uint32_t edge = (c.w == 0 ? 1u : 0u) | last_bit;  // this lane's cells on the east / west columns

    // rows of the lattice behind the lane's M rows
    const int dy = (int)g.dim_y;
    uint32_t j[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        int r = (int)y0 - (int)hk + (int)(group * M + m);
        if (r < 0) r += dy;
        else if (r >= dy) r -= dy;
        if (r < 0 || r >= dy) r = (r % dy + dy) % dy;  // (blocks taller than the lattice)
        j[m] = (uint32_t)r;
        if (!kRows) j[m] = __builtin_amdgcn_readfirstlane(j[m]);
    }
    // The stored rows depend on rows [hk - left, hk + rows + left) of the block
    // with `left` steps to go: the wave works on its rows [wave_lo, wave_hi)
    // for the pass's first `act` steps.
    const int wave_lo = (int)(wave * S * M), wave_hi = wave_lo + (int)(S * M);
    const uint32_t most = SEG == kPacked ? a.th : rows;
    const int idle = max(0, max(wave_lo - (int)(hk + most) + 1, (int)hk - wave_hi + 1));
    const int act = (int)k - idle;
    const bool work = act >= 0;  // (at 0 its initial planes are still read)

    const uint32_t plane_b = g.P * 4u, row_b = (uint32_t)Q * plane_b;
    constexpr uint32_t kOutside = 0x80000000u;  // past any descriptor: reads 0, stores nothing
    uint32_t s[M][Q];
    uint32_t ns[M], sl[M], fd[M];
    uint32_t solid_rows = 0;   // bit m: some lane's row m holds solids,
    uint32_t slip_rows = 0;    // SLIP cells,
    uint32_t inner_slip = 0;   // SLIP cells off the east and west columns
    bool forced = false;       // the wave holds forced words
    // Force decisions: [step][row][word], one descriptor over the pass's steps.
    // Strip mode keeps the lane's part of the offset and adds the (uniform)
    // row's; in segment mode rows differ per lane.
    const uint32_t fplane_b = (a.fy1 - a.fy0) * a.fwn * 4u;
    const bool fcol = c.w >= a.fw0 && c.w < a.fw0 + a.fwn;
    uint32_t foff[kRows ? M : 1];
    if (!kRows) foff[0] = fcol ? (c.w - a.fw0) * 4u : kOutside;
    auto frow = [&](int m) { return j[m] >= a.fy0 && j[m] < a.fy1; };
    auto load_force = [&](int m, uint32_t step) {
        const uint32_t off = kRows ? foff[kRows ? m : 0] : (frow(m) ? foff[0] : kOutside);
        const uint32_t row = !kRows && frow(m) ? (j[m] - a.fy0) * a.fwn * 4u : 0u;
        return bload(make_rsrc(a.fdec, k * fplane_b), off, step * fplane_b + row);
    };
    if (work) {
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int d = 0; d < Q; ++d)
                s[m][d] = kRows ? bload(make_rsrc(a.src, g.dim_y * row_b), j[m] * row_b + c.wb, (uint32_t)d * plane_b)
                              : bload(make_rsrc(a.src + (size_t)j[m] * Q * g.P, row_b), c.wb, (uint32_t)d * plane_b);
        if (FEAT) {
            if (a.fdec) {
                bool any = false;
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    if (kRows) foff[kRows ? m : 0] = fcol && frow(m) ? ((j[m] - a.fy0) * a.fwn + (c.w - a.fw0)) * 4u : kOutside;
                    any |= fcol && frow(m);
                }
                forced = __builtin_amdgcn_ballot_w64(any) != 0;
                if (forced)
#pragma unroll
                    for (int m = 0; m < M; ++m) fd[m] = load_force(m, 0);
            }
#pragma unroll
            for (int m = 0; m < M; ++m) ns[m] = sl[m] = 0;
            if (a.mask) {
                const uint32_t mrow_b = 2u * plane_b;
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const uint32_t* row = a.mask + (kRows ? (size_t)0 : (size_t)j[m] * 2 * g.P);
                    const __amdgpu_buffer_rsrc_t r = make_rsrc(row, kRows ? g.dim_y * mrow_b : mrow_b);
                    const uint32_t off = (kRows ? j[m] * mrow_b : 0u) + c.wb;
                    ns[m] = bload(r, off, 0);
                    sl[m] = bload(r, off, plane_b);
                }
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    if (__builtin_amdgcn_ballot_w64((ns[m] | sl[m]) != 0)) solid_rows |= 1u << m;
                    if (__builtin_amdgcn_ballot_w64(sl[m] != 0)) slip_rows |= 1u << m;
                    if (__builtin_amdgcn_ballot_w64((sl[m] & ~edge) != 0)) inner_slip |= 1u << m;
                }
            }
        }
    }

    // LDS: exchanged planes [2][wave][down NX, up NX][64], then chirality
    // words [wave][row][4][64]
    const uint32_t xbuf = nwave * 2u * NX * 64u;
    uint32_t* xch = lds;
    uint32_t* chir = lds + 2u * xbuf + wave * (uint32_t)(M * 4 * 64) + lane;
    const uint32_t mine = wave * 2u * NX * 64u + lane;
    // where the groups above and below left their planes: the next wave, or
    // the next segment of this one; past the block's ends the own wave's slot
    // (those rows are not needed)
    uint32_t above = wave > 0 ? wave - 1u : 0u, below = wave + 1u < nwave ? wave + 1u : wave;
    uint32_t alane = lane, blane = lane;
    if (kStacked) {
        const uint32_t seg = min(lane / g.W, S - 1u);
        if (seg > 0) { above = wave; alane = lane - g.W; }
        else alane = lane + (S - 1u) * g.W;
        if (seg + 1u < S) { below = wave; blane = lane + g.W; }
        else blane = lane - (S - 1u) * g.W;
        alane &= 63u;  // (idle lanes)
        blane &= 63u;
    }
    const uint32_t from_above = above * 2u * NX * 64u + alane, from_below = below * 2u * NX * 64u + NX * 64u + blane;
    auto publish = [&](uint32_t buf) {
        uint32_t* x = xch + buf * xbuf + mine;
        if (KIND == kHPP) {
            x[0] = s[M - 1][1];
            x[64] = s[0][3];
        } else {
            x[0] = s[M - 1][1];
            x[64] = s[M - 1][2];
            x[128] = s[0][4];
            x[192] = s[0][5];
        }
    };
    if (work) publish(0);
    __syncthreads();

    // One step of the wave's rows.  SOL: 0 no solids, 1 NO_SLIP only, 2 any;
    // FRC: 0 not forced, 1 along x, 2 any (both 2 together only).
    auto advance = [&](auto sol_tag, auto frc_tag, uint32_t step) {
        constexpr int SOL = decltype(sol_tag)::value, FRC = decltype(frc_tag)::value;
        const uint32_t t = a.t0 + step, word = t & 3u;
        if (KIND != kHPP && (step == 0 || word == 0)) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const U4 r = philox4x32_10(c.w, j[m], t >> 2, 0u, a.key0, a.key1);
                uint32_t* q = chir + m * 256;
                q[0] = r.x;
                q[64] = r.y;
                q[128] = r.z;
                q[192] = r.w;
            }
        }
        const uint32_t* xa = xch + (step & 1u) * xbuf + from_above;
        const uint32_t* xb = xch + (step & 1u) * xbuf + from_below;
        uint32_t p1 = xa[0], p2 = NX == 2 ? xa[64] : 0u;         // planes 1, 2 of the row above
        const uint32_t n4 = xb[0], n5 = NX == 2 ? xb[64] : 0u;   // planes 4, 5 (HPP: 3) of the row below
#pragma unroll
        for (int m = 0; m < M; ++m) {
            uint32_t in[7], st[7];
            if (KIND == kHPP) {
                in[0] = shift_m1<RAGGED, SHIFT>(s[m][0], c);
                in[1] = p1;
                in[2] = shift_p1<RAGGED, SHIFT>(s[m][2], c);
                in[3] = m + 1 < M ? s[m + 1 < M ? m + 1 : 0][3] : n4;
                p1 = s[m][1];
            } else {
                const uint32_t r4 = m + 1 < M ? s[m + 1 < M ? m + 1 : 0][4] : n4;
                const uint32_t r5 = m + 1 < M ? s[m + 1 < M ? m + 1 : 0][5] : n5;
                in[0] = shift_m1<RAGGED, SHIFT>(s[m][0], c);
                in[3] = shift_p1<RAGGED, SHIFT>(s[m][3], c);
                if (Q == 7) in[6] = s[m][Q - 1];
                auto odd_row = [&] {
                    in[1] = p1;
                    in[2] = shift_p1<RAGGED, SHIFT>(p2, c);
                    in[4] = shift_p1<RAGGED, SHIFT>(r4, c);
                    in[5] = r5;
                };
                auto even_row = [&] {
                    in[1] = shift_m1<RAGGED, SHIFT>(p1, c);
                    in[2] = p2;
                    in[4] = r4;
                    in[5] = shift_m1<RAGGED, SHIFT>(r5, c);
                };
                if (M % 2 == 0) {  // blocks start on even rows
                    if (m & 1) odd_row();
                    else even_row();
                } else if (SEG != kSegments) {  // one row per wave: wave-uniform
                    if ((wave + hk) & 1u) odd_row();
                    else even_row();
                } else {
                    // one row per segment: each lane shifts the way its row does
                    const bool odd = ((group + hk) & 1u) != 0;
                    auto shifted = [&](uint32_t even_v, uint32_t odd_v) {
                        const uint32_t v = odd ? odd_v : even_v;
                        uint32_t n = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(odd ? c.rsrc : c.lsrc), (int)v);
                        if (RAGGED && !odd) n <<= c.first_shl;
                        uint32_t o = __builtin_amdgcn_alignbit(odd ? n : v, odd ? v : n, odd ? 1u : 31u);
                        if (RAGGED) o = bit3<kMux>(odd ? last_bit : 0u, n << (c.nb - 1u), o);
                        return o;
                    };
                    const uint32_t u = shifted(p1, p2), v = shifted(r5, r4);
                    in[1] = odd ? p1 : u;
                    in[2] = odd ? u : p2;
                    in[4] = odd ? v : r4;
                    in[5] = odd ? r5 : v;
                }
                p1 = s[m][1];
                p2 = s[m][2];
            }
#pragma unroll
            for (int d = 0; d < Q; ++d) st[d] = in[d];
            collide<KIND, uint32_t>(st, KIND == kHPP ? 0u : chir[m * 256 + word * 64]);
            if (SOL == 1) apply_no_slip<KIND, uint32_t>(st, in, ns[m]);
            if (SOL == 2) {
                // apply_solids' dispatch as selects: SLIP cells on the east and
                // west columns mirror in y, the others in x on the north and
                // south rows, and pass through elsewhere
                uint32_t o[7], rim = edge;
                asm("" : "+v"(rim));  // keeps sl & rim out of registers held across steps
#pragma unroll
                for (int d = 0; d < Q; ++d) {
                    o[d] = bit3<kMux>(ns[m], in[inv_dir<KIND>(d)], st[d]);
                    o[d] = bit3<kMux>(sl[m] & rim, in[miry_dir<KIND>(d)], o[d]);
                }
                if ((inner_slip >> m) & 1u) {
                    const bool ns_row = j[m] == 0 || j[m] + 1 == g.dim_y;
#pragma unroll
                    for (int d = 0; d < Q; ++d)
                        o[d] = bit3<kMux>(sl[m] & ~rim, ns_row ? in[mirx_dir<KIND>(d)] : in[d], o[d]);
                }
#pragma unroll
                for (int d = 0; d < Q; ++d) st[d] = o[d];
            }
            if (FRC) {
                const uint32_t f = SOL == 2 ? bit3<kX & ~(kY | kZ)>(fd[m], ns[m], sl[m])
                                   : SOL == 1 ? bit3<kX & ~kY>(fd[m], ns[m], 0u) : fd[m];
                if (FRC == 1) apply_force<KIND, uint32_t>(st, f, 1);
                else if (forced) apply_force<KIND, uint32_t>(st, f, a.force_dir);
                // the next step's decisions (the last step's again after it: a
                // test would wait for the load at its join)
                if (FRC == 1 || forced) fd[m] = load_force(m, min(step + 1u, k - 1u));
            }
#pragma unroll
            for (int d = 0; d < Q; ++d) s[m][d] = st[d];
        }
        publish((step + 1u) & 1u);
    };
    // A loop per mode, so that the force decisions of the next step stay in
    // flight across the barrier (with one loop and tests in it, the paths
    // without loads made every step wait for them).  The mode and the steps
    // that a wave works on are wave-uniform, and every wave makes k barriers.
    auto pass = [&](auto sol_tag, auto frc_tag) {
        for (int step = 0; step < act; ++step) {
            advance(sol_tag, frc_tag, (uint32_t)step);
            __syncthreads();
        }
        for (int step = max(act, 0); step < (int)k; ++step) __syncthreads();
        if (idle) return;  // the wave holds no stored row
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const uint32_t l = group * M + m;
            const bool wr = writer && l >= hk && l < hk + rows;
            if (!kStacked && !(l >= hk && l < hk + most)) continue;  // wave-uniform
#pragma unroll
            for (int d = 0; d < Q; ++d) {
                if (RAGGED) s[m][d] &= c.vmask;
                if (kRows) bstore(s[m][d], make_rsrc(a.dst, g.dim_y * row_b), wr ? j[m] * row_b + c.wb : kOutside, (uint32_t)d * plane_b);
                else bstore(s[m][d], make_rsrc(a.dst + (size_t)j[m] * Q * g.P, row_b), wr ? c.wb : kOutside, (uint32_t)d * plane_b);
            }
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    if (!FEAT || (!solid_rows && !forced)) pass(I0{}, I0{});
    else if (slip_rows || (forced && a.force_dir != 1)) pass(I2{}, I2{});
    else if (!solid_rows) pass(I0{}, I1{});
    else if (!forced) pass(I1{}, I0{});
    else pass(I1{}, I1{});
}

template <int KIND, int M, bool RAGGED, int SEG, int FEAT>
__global__ __launch_bounds__(kBlockMaxWaves * 64) __attribute__((amdgpu_waves_per_eu(4, 8)))
void block_kernel(BlockArgs b)
{
    extern __shared__ uint32_t block_lds[];
    // Workgroups go to the 8 XCDs round-robin; each XCD takes a contiguous
    // run of blocks, whose halo rows meet in its L2.
    const uint32_t xcd = blockIdx.x & 7u, xq = gridDim.x >> 3, xr = gridDim.x & 7u;
    const uint32_t item = xcd * xq + min(xcd, xr) + (blockIdx.x >> 3);
    const uint32_t tile = item / b.nstrips, strip = item - tile * b.nstrips;
    block_body<KIND, M, RAGGED, SEG, FEAT>(b.a, b.k, b.hk, strip, tile, block_lds);
}

// Batched form (tile_batch_kernel's): every workgroup takes one work item.  A
// job's steps in the round are in its items (block_shape_bits), so jobs at
// their last steps share the launch, and a pass may start at any step.
template <int M, bool RAGGED>
__global__ __launch_bounds__(kBlockMaxWaves * 64) __attribute__((amdgpu_waves_per_eu(4, 8)))
void block_batch_kernel(const BatchJob* __restrict__ jobs, BatchState* state, const WorkItem* __restrict__ items,
                        uint32_t n_heavy)
{
    extern __shared__ uint32_t block_lds[];
    // the leading (heavy) items and the rest each map to contiguous runs per XCD
    const bool in_heavy = blockIdx.x < n_heavy;
    const uint32_t i = in_heavy ? blockIdx.x : blockIdx.x - n_heavy, n = in_heavy ? n_heavy : gridDim.x - n_heavy;
    const uint32_t xcd = i & 7u, q = n >> 3, r = n & 7u;
    const uint32_t wi = __builtin_amdgcn_readfirstlane((in_heavy ? 0u : n_heavy) + xcd * q + min(xcd, r) + (i >> 3));
    const WorkItem it = items[wi];
    const BatchState bs = state[it.job];
    TileArgs a = jobs[it.job].a;
    a.t0 = bs.step;
    a.th = it.shape & 0xFFFFu;
    a.halo = (it.shape >> 16) & 0x7Fu;
    a.src = bs.cur ? jobs[it.job].buf1 : jobs[it.job].buf0;
    a.dst = bs.cur ? jobs[it.job].buf0 : jobs[it.job].buf1;
    if (a.fdec) a.fdec += (size_t)(bs.step - bs.fdec_step0) * a.fdec_stride;
    const uint32_t k = (it.shape >> 24) & 0x7Fu, hk = block_halo(M, k);
    const bool seg = (it.shape >> 31) != 0, packed = ((it.shape >> 23) & 1u) != 0;
    const uint32_t Q = __builtin_amdgcn_readfirstlane(a.g.Q);
    if (Q == 4) {
        if (seg) block_body<kHPP, M, RAGGED, kSegments, 1>(a, k, hk, it.strip, it.tile, block_lds);
        else if (packed) block_body<kHPP, M, RAGGED, kPacked, 1>(a, k, hk, it.strip, it.tile, block_lds);
        else block_body<kHPP, M, RAGGED, kStrips, 1>(a, k, hk, it.strip, it.tile, block_lds);
    } else if (Q == 6) {
        if (seg) block_body<kFHP1, M, RAGGED, kSegments, 1>(a, k, hk, it.strip, it.tile, block_lds);
        else if (packed) block_body<kFHP1, M, RAGGED, kPacked, 1>(a, k, hk, it.strip, it.tile, block_lds);
        else block_body<kFHP1, M, RAGGED, kStrips, 1>(a, k, hk, it.strip, it.tile, block_lds);
    } else {
        if (seg) block_body<kFHP2, M, RAGGED, kSegments, 1>(a, k, hk, it.strip, it.tile, block_lds);
        else if (packed) block_body<kFHP2, M, RAGGED, kPacked, 1>(a, k, hk, it.strip, it.tile, block_lds);
        else block_body<kFHP2, M, RAGGED, kStrips, 1>(a, k, hk, it.strip, it.tile, block_lds);
    }
    // The job's last workgroup of the round advances it.  Every wave of every
    // other one has read the state by now: a wave comes here after the body's
    // barriers, which its workgroup's waves pass with the state read.
    if (threadIdx.x == 0) {
        BatchState& st = state[it.job];
        if (atomicAdd(&st.done, 1u) + 1u == it.job_items) {
            st.done = 0;
            st.step = bs.step + k;
            st.cur = bs.cur ^ 1u;
        }
    }
}

template <int KIND, int M>
hipError_t launch_block_km(const BlockArgs& b, uint32_t waves, uint32_t blocks, bool ragged, int seg, hipStream_t s)
{
    const dim3 grid(blocks), block(64 * waves);
    const size_t lds = block_lds_bytes(KIND, M, waves);
    const bool feat = b.a.mask || b.a.fdec;
#define LGCA_BLOCK_LAUNCH(RG, SG)                                                                        \
    do {                                                                                                 \
        if (feat) hipLaunchKernelGGL((block_kernel<KIND, M, RG, SG, 1>), grid, block, lds, s, b);        \
        else hipLaunchKernelGGL((block_kernel<KIND, M, RG, SG, 0>), grid, block, lds, s, b);             \
    } while (0)
    if (ragged) {
        if (seg == kPacked) LGCA_BLOCK_LAUNCH(true, kPacked);
        else if (seg) LGCA_BLOCK_LAUNCH(true, kSegments);
        else LGCA_BLOCK_LAUNCH(true, kStrips);
    } else {
        if (seg == kPacked) LGCA_BLOCK_LAUNCH(false, kPacked);
        else if (seg == kWholeRow) LGCA_BLOCK_LAUNCH(false, kWholeRow);
        else if (seg) LGCA_BLOCK_LAUNCH(false, kSegments);
        else LGCA_BLOCK_LAUNCH(false, kStrips);
    }
#undef LGCA_BLOCK_LAUNCH
    return hipGetLastError();
}

template <int M>
hipError_t launch_block_batch_m(const BatchJob* jobs, BatchState* state, const WorkItem* items, uint32_t n_items,
                                uint32_t n_heavy, uint32_t waves, bool ragged, hipStream_t s)
{
    const dim3 grid(n_items), block(64 * waves);
    const size_t lds = block_lds_bytes(kFHP2, M, waves);
    if (ragged) hipLaunchKernelGGL((block_batch_kernel<M, true>), grid, block, lds, s, jobs, state, items, n_heavy);
    else hipLaunchKernelGGL((block_batch_kernel<M, false>), grid, block, lds, s, jobs, state, items, n_heavy);
    return hipGetLastError();
}

}  // namespace lgca
