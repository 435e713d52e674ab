// lgca_plan.cpp -- host-only launch planning: lattice geometry, the tiled
// step's halo and strip counts, the strip-mode wave dispatch order, the band
// plan of multi-pass launches, and the shapes of block passes and rounds.  Plain C++ (no device code), so that test
// programs can build it with the host compiler and check the plans without a
// GPU.
#include "lgca_kernels.hpp"

#include <algorithm>
#include <climits>
#include <cstdint>
#include <utility>

namespace lgca {

Geometry make_geometry(uint32_t dim_x, uint32_t dim_y, uint32_t Q)
{
    Geometry g{};
    g.dim_x = dim_x;
    g.dim_y = dim_y;
    g.W = (dim_x + 31) / 32;
    g.P = (g.W + 3) & ~3u;
    g.Wq = g.P / 4;
    g.nb = dim_x - 32 * (g.W - 1);
    g.Q = Q;
    uint32_t l = 0;
    while ((1u << l) < g.Wq && l < 6) ++l;
    g.qb_log = l;
    return g;
}

uint32_t tile_halo(const Geometry& g, int k)
{
    if (g.W == 1) return (uint32_t)((k + (int)g.nb - 1) / (int)g.nb);
    return (int)g.nb < k ? 2u : 1u;
}

uint32_t tile_strips(const Geometry& g, int k)
{
    const uint32_t stride = 64u - 2u * tile_halo(g, k);
    return (g.W + stride - 1) / stride;
}

bool tile_segments(const Geometry& g, int k)
{
    return g.W <= 64 && (64 / g.W >= 2 || tile_strips(g, k) >= 2);
}

// Does strip st (words [st * stride - halo, + 64) modulo W) touch words
// [lo, hi) of its rows?
bool tile_strip_hits(const Geometry& g, uint32_t stride, uint32_t halo, uint32_t st, int64_t lo, int64_t hi)
{
    if (lo >= hi) return false;
    const int64_t W = g.W;
    if (W <= 64) return true;  // the strip wraps the whole row
    const int64_t a0 = (((int64_t)st * stride - halo) % W + W) % W;
    for (int64_t k = -1; k <= 1; ++k)
        if (a0 < hi + k * W && a0 + 64 > lo + k * W) return true;
    return false;
}

namespace {

// Appends v in the order that hands each XCD a contiguous run of it:
// workgroups go to the 8 XCDs round-robin, so entry b of the appended range
// runs on XCD (start + b) mod 8.
void append_xcd_runs(std::vector<uint32_t>& order, const std::vector<uint32_t>& v)
{
    const uint32_t n = (uint32_t)v.size(), q = n >> 3, r = n & 7u;
    for (uint32_t b = 0; b < n; ++b) {
        const uint32_t xcd = b & 7u;
        order.push_back(v[xcd * q + std::min(xcd, r) + (b >> 3)]);
    }
}

// The cost class of every strip-mode wave of a pass (tile * nstrips + strip):
// 2 when its walk crosses solids (about twice a plain walk), 1 when it crosses
// forced words (about a sixth longer), else 0.  False when the pass is not in
// strip mode or has too many waves to list.
bool wave_classes(const TileArgs& a, int k, const int32_t* row_lo, const int32_t* row_hi,
                  uint32_t& nstrips, uint32_t& ntiles, std::vector<uint8_t>& cls)
{
    if (tile_segments(a.g, k) || a.th < 2) return false;
    const uint32_t stride = 64u - 2u * a.halo;
    nstrips = (a.g.W + stride - 1) / stride;
    ntiles = (a.g.dim_y + a.th - 1) / a.th;
    if ((uint64_t)nstrips * ntiles > ((uint64_t)1 << 24)) return false;
    const bool forced = a.fdec && a.fwn;
    std::vector<uint8_t> fstrip(nstrips, 0);
    if (forced)
        for (uint32_t st = 0; st < nstrips; ++st)
            fstrip[st] = tile_strip_hits(a.g, stride, a.halo, st, a.fw0, (int64_t)a.fw0 + a.fwn);
    cls.assign((size_t)nstrips * ntiles, 0);
    const int64_t dy = a.g.dim_y;
    for (uint32_t t = 0; t < ntiles; ++t) {
        const int64_t y0 = (int64_t)t * a.th, rows = std::min<int64_t>(a.th, dy - y0);
        int64_t lo = INT64_MAX, hi = INT64_MIN;  // hull of the walk rows' solid words
        bool frow = false;
        for (int64_t y = y0 - k; y < y0 + rows + k; ++y) {
            const int64_t r = ((y % dy) + dy) % dy;
            if (row_lo && row_lo[r] < row_hi[r]) {
                lo = std::min<int64_t>(lo, row_lo[r]);
                hi = std::max<int64_t>(hi, row_hi[r]);
            }
            frow |= r >= (int64_t)a.fy0 && r < (int64_t)a.fy1;
        }
        for (uint32_t st = 0; st < nstrips; ++st) {
            uint8_t c = 0;
            if (lo < hi && tile_strip_hits(a.g, stride, a.halo, st, lo, hi)) c = 2;
            else if (forced && frow && fstrip[st]) c = 1;
            cls[(size_t)t * nstrips + st] = c;
        }
    }
    return true;
}

}  // namespace

bool tile_wave_order(const TileArgs& a, int k, const int32_t* row_lo, const int32_t* row_hi,
                     std::vector<uint32_t>& order)
{
    order.clear();
    uint32_t nstrips = 0, ntiles = 0;
    std::vector<uint8_t> cls;
    if (!wave_classes(a, k, row_lo, row_hi, nstrips, ntiles, cls)) return false;
    std::vector<uint32_t> solid, force, plain;
    for (uint32_t it = 0; it < (uint32_t)cls.size(); ++it) {
        const uint32_t e = it << kPartBits;  // whole tile
        if (cls[it] != 2) {
            (cls[it] == 1 ? force : plain).push_back(e);
            continue;
        }
        // A walk over solids runs up to 2.5 times as long as a plain one,
        // long enough to outlast the pass: it is cut into quarters of the
        // tile (halves on short tiles), each walking its rows plus the
        // K-row halo, which costs more in all but ends sooner.
        const uint32_t t = it / nstrips, rows = std::min(a.th, a.g.dim_y - t * a.th);
        if (rows >= 16)
            for (uint32_t p = 3; p <= 6; ++p) solid.push_back(e | p);
        else if (rows >= 8)
            for (uint32_t p = 1; p <= 2; ++p) solid.push_back(e | p);
        else
            solid.push_back(e);
    }
    // The solid walks go first, spread over the XCDs; then the forced and
    // the plain ones, each in contiguous runs per XCD, so that the tiles an
    // XCD holds are vertical neighbours whose halo rows meet in its L2.
    order.reserve(solid.size() + force.size() + plain.size());
    order.insert(order.end(), solid.begin(), solid.end());
    append_xcd_runs(order, force);
    append_xcd_runs(order, plain);
    return true;
}

bool tile_pipe_plan(const TileArgs& a, int k, uint32_t nband, const int32_t* row_lo, const int32_t* row_hi,
                    PipePlan& plan)
{
    plan = PipePlan{};
    if ((k != 4 && k != 8) || nband < 1 || nband > kMaxBands) return false;
    if (a.g.nb != 32 || a.th < (uint32_t)k || (a.th & 1u)) return false;
    uint32_t nstrips = 0, ntiles = 0;
    std::vector<uint8_t> cls;
    if (!wave_classes(a, k, row_lo, row_hi, nstrips, ntiles, cls)) return false;
    if (ntiles < 2 * nband) return false;
    // bands of whole tiles with about equal work, at least two tiles each
    std::vector<double> cost(ntiles + 1, 0.0);  // prefix sums
    for (uint32_t t = 0; t < ntiles; ++t) {
        double c = 0.0;
        for (uint32_t st = 0; st < nstrips; ++st) c += 1.0 + (double)cls[(size_t)t * nstrips + st] * 0.5;
        cost[t + 1] = cost[t] + c;
    }
    std::vector<uint32_t> cut(nband + 1, 0);
    cut[nband] = ntiles;
    for (uint32_t b = 1; b < nband; ++b) {
        const double target = cost[ntiles] * b / nband;
        uint32_t t = cut[b - 1] + 2;
        while (t < ntiles && cost[t] + 0.5 * (cost[t + 1] - cost[t]) < target) ++t;
        cut[b] = std::min(std::max(t, cut[b - 1] + 2), ntiles - 2 * (nband - b));
    }
    for (uint32_t b = 0; b < nband; ++b) {
        const uint32_t y0 = cut[b] * a.th, y1 = std::min<uint64_t>((uint64_t)cut[b + 1] * a.th, a.g.dim_y);
        if (y1 - y0 < 2u * (uint32_t)k) return false;
        plan.band_y0[b] = y0;
        plan.band_y1[b] = y1;
        plan.band_first[b] = (uint32_t)plan.order.size();
        for (uint32_t t = cut[b]; t < cut[b + 1]; ++t)
            for (uint32_t st = 0; st < nstrips; ++st) plan.order.push_back(t * nstrips + st);
        plan.band_items[b] = (uint32_t)plan.order.size() - plan.band_first[b];
    }
    plan.nband = nband;
    plan.nstrips = nstrips;
    plan.ntiles = ntiles;
    return true;
}

size_t tile_pipe_exch_words(const Geometry& g, int k, uint32_t nband)
{
    return (size_t)2 * nband * 2 * (size_t)k * g.Q * g.P;
}

// ------------------------------------------------- block passes (lgca_block.hpp)

uint32_t block_lds_bytes(int kind, uint32_t m, uint32_t waves)
{
    // two buffers of the exchanged planes, and the chirality words of every row
    return waves * 64u * 4u * (kind == 0 ? 4u : 8u + 4u * m);
}

// Packed strips where rows of more than half a wave leave lanes of their
// strips idle: their rows differ per lane, which costs three instructions a
// Philox call, so from 3 % fewer waves on.  (Their row offsets are lane
// offsets, below 2 GiB.)  Shorter rows stack 64 / W segments, whose blocks are
// that much taller.
BlockLanes block_lanes(const Geometry& g, int k)
{
    if (tile_segments(g, k)) return kLanesRows;
    const uint64_t h = tile_halo(g, k), span = g.W + 2 * h, stride = 64 - 2 * h;
    const bool fits = (uint64_t)g.dim_y * g.Q * g.P * 4 < ((uint64_t)1 << 31);
    return fits && g.W > 32 && span * 100 <= 97 * stride * tile_strips(g, k) ? kLanesPacked : kLanesStrips;
}

uint64_t block_count(const Geometry& g, int k, uint32_t tiles)
{
    switch (block_lanes(g, k)) {
    case kLanesRows: return tiles;
    case kLanesStrips: return (uint64_t)tiles * tile_strips(g, k);
    default: break;
    }
    const uint64_t h = tile_halo(g, k), stride = 64 - 2 * h;
    return ((uint64_t)tiles * (g.W + 2 * h) + stride - 1) / stride;
}

// Rows of 64 words (or the whole rows that a wave holds), packed as the blocks
// have them.
static uint64_t block_wave_rows(const Geometry& g)
{
    return tile_segments(g, 8) ? (uint64_t)g.dim_y / (64 / g.W) : block_count(g, 8, g.dim_y);
}

// Lattices of up to 36 wave-rows per SIMD.  us per step in blocks / walked, FHP-II: 4400 x 2200 1.7 /
// 2.9, 8192 x 4096 (17,045 wave-rows) 3.2 / 4.8, 12000 x 4000 (24,323) 4.7 /
// 5.2, 32768 x 2048 (33,891) 5.8 / 6.0, 12000 x 6000 (36,484) 6.0 / 6.4, 13001 x
// 6000 (39,581) 8.3 / 8.0 with walls and forced columns, 16384 x
// 8192 (67,914) 11.2 / 9.5: the larger ones fill the GPU with walks, which read
// and compute fewer halo rows.
// Nor do flat ones whose strips alone do, without solids: 4000000 x 2 FHP-II 3.3
// us a step in blocks and 2.3 walked, x 4 3.8 / 2.9, x 6 4.3 / 4.8, 2000000 x 2 1.97 /
// 1.82, x 4 2.2 / 2.3, 4000000 x 4 with walls 4.2 / 4.7.
bool block_lattice(const Geometry& g, bool solids)
{
    if (g.dim_y <= 4 && !solids && !tile_segments(g, 8) && tile_strips(g, 8) >= 500 * g.dim_y) return false;
    return block_wave_rows(g) < 36864;
}

// A call of 1, 2 or 4 steps is one pass either way.  A block pass starts all its
// loads at once and stores only when its steps are done, so on many rows, for few
// steps, walks over tiles of 4 or 8 rows, whose loads and stores overlap, are
// faster; other counts take a walk two launches or more.  us per call in
// blocks / walked: 4096 x 2048 FHP-II (4,295 wave-rows) 1 step 6.7 / 6.0, 2 steps
// 7.4 / 7.2, 4 steps 9.2 / 10.9; 6000 x 3000 (9,194) 11.0 / 8.6, 11.7 / 10.1, 13.5 /
// 14.9; 7000 x 3500 with walls (12,476) 14.9 / 10.2, 16.6 / 11.2, 18.2 / 16.3;
// 8192 x 4096 (17,045) 16.1 / 11.7, 17.1 / 12.6, 22.1 / 18.6, HPP 8.8 / 7.6, 9.1 / 8.3,
// 11.7 / 9.2; 12000 x 5800 forced everywhere (35,268) 41.3 / 36.3, 54 / 40, 53 /
// 51.  Blocks keep flat lattices (1000000 x 16, 1 step 5.5 / 6.7) and HPP rows that
// a wave holds whole (2048 x 16384, 4 steps 8.7 / 10.0).
uint32_t short_walk_rows(const Geometry& g, int kind, uint64_t steps)
{
    if (steps != 1 && steps != 2 && steps != 4) return 0;
    if (g.dim_y < 256 || (kind == 0 && tile_segments(g, (int)steps))) return 0;
    const uint64_t wave_rows = block_wave_rows(g);
    if (wave_rows < (steps == 4 ? 12288 : 4096 * steps)) return 0;
    return wave_rows < 8192 ? 4 : 8;
}

std::vector<BlockShape> block_shapes(const Geometry& g, int kind, uint32_t k)
{
    std::vector<BlockShape> out;
    const uint32_t S = tile_segments(g, (int)k) ? 64 / g.W : 1;
    for (uint32_t m : {1u, 2u, 4u, 6u})
        for (uint32_t waves : {4u, 8u, 12u, 16u}) {
            const uint32_t held = m * waves * S, halo = 2 * block_halo(m, k);
            if (held < halo + 2 || block_lds_bytes(kind, m, waves) > 160u * 1024u) continue;
            const uint32_t most = (held - halo) & ~1u;
            const uint32_t tiles = (g.dim_y + most - 1) / most;
            uint32_t th = (g.dim_y + tiles - 1) / tiles;
            th += th & 1u;
            out.push_back(BlockShape{m, waves, th});
        }
    return out;
}

// A pass takes its launch, loads and stores (3.2 us, 1.3 more where masks and
// decisions are read), then per step a barrier with the exchange through LDS
// and the rows' work: at least one wave's chain of m rows, at most the VALU
// time of the rows a SIMD still works on.  Constants from passes of 5 to 28
// steps on 256 x 256 HPP (0.12 us a step), the 2048 x 512 FHP-II pipe (0.45)
// and 4400 x 2200 FHP-II (1.6); the best predicted shape was within 10 % of
// the best measured one on each, and is with the shorter collision (constants
// a sixth smaller pick no better shapes).  Forced lattices past 8192 x 4096 are
// the exception: the model does not know that six rows a wave spill with solids
// or forcing (10000 x 4000 FHP-II forced everywhere 7.9 us a step, 6.3 in the
// four-row shape that lgca_tune finds; 8192 x 4096 6.0 and 5.5).
float block_pass_us(const Geometry& g, int kind, bool feat, uint32_t ncu, uint32_t k, const BlockShape& s)
{
    const bool seg = tile_segments(g, (int)k);
    const uint32_t S = seg ? 64 / g.W : 1, held = s.m * s.waves * S, hk = block_halo(s.m, k);
    if (!k || !s.th || held < s.th + 2 * hk || (!seg && k > 32)) return -1.0f;
    const uint64_t blocks = block_count(g, (int)k, (g.dim_y + s.th - 1) / s.th);
    // workgroups a CU holds: 128 registers allow 16 waves, half of them 32
    const uint32_t waves_cu = feat && s.m > 2 ? 16 : 32;
    const uint32_t fit = std::max(1u, std::min(waves_cu / s.waves, 160u * 1024u / block_lds_bytes(kind, s.m, s.waves)));
    const uint32_t cus = std::max(ncu, 1u);
    const uint32_t per_cu = (uint32_t)std::min<uint64_t>(fit, (blocks + cus - 1) / cus);
    const uint64_t rounds = (blocks + (uint64_t)cus * per_cu - 1) / ((uint64_t)cus * per_cu);
    float row = kind == 0 ? 0.045f : kind == 1 ? 0.090f : 0.119f;  // us of a SIMD per wave-row
    if (feat) row *= 1.15f;
    if (g.nb != 32) row *= 1.1f;
    const float chain = (kind == 0 ? 0.04f : 0.16f) * (float)s.m;
    float us = 0.0f;
    for (uint32_t left = 0; left < k; ++left) {
        const uint32_t rows = std::min(held, s.th + 2 * left);
        const float work = (float)per_cu * (float)((rows + S * s.m - 1) / (S * s.m) * s.m) / 4.0f * row;
        us += 0.08f * (float)per_cu + std::max(work, chain);
    }
    // reads of the held rows and writes of the stored ones, at 4.5 TB/s: half of
    // them overlap other blocks' steps
    const float bytes = (float)blocks * (float)((s.m * s.waves) + (s.th + S - 1) / S) * 256.0f * (float)g.Q;
    return 3.2f + (feat ? 1.3f : 0.0f) + (float)rounds * us + 0.5f * bytes / 4.5e6f;
}

// ------------------------------------------------- rounds of a batch in blocks

JobBlocks job_blocks(const Geometry& g, const RoundShape& s, int k)
{
    const bool seg = tile_segments(g, k);
    const uint32_t held = s.m * s.waves * (seg ? 64 / g.W : 1);
    const uint32_t most = (held - 2 * block_halo(s.m, (uint32_t)k)) & ~1u;
    JobBlocks b;
    b.tiles = (g.dim_y + most - 1) / most;
    b.th = (g.dim_y + b.tiles - 1) / b.tiles;
    b.th += b.th & 1u;
    b.tiles = (g.dim_y + b.th - 1) / b.th;
    b.blocks = (uint32_t)block_count(g, k, b.tiles);
    return b;
}

// A shape chosen before a job with a large force region came may have more
// steps than that job's decisions allow.  Jobs are accepted with 8 or more, and
// a multiple of 4 keeps the job's step one, as walks need it.
int round_steps(const RoundShape& s, uint64_t left, uint64_t force_words)
{
    uint64_t k = (uint64_t)s.k;
    if (force_pass_steps(force_words) < k) k = force_pass_steps(force_words) & ~(uint64_t)3;
    return (int)std::min(k, left);
}

namespace {

// The block shapes that rounds may take.  Steps are multiples of 4, so that a
// round of walks may follow.
struct RoundShapeList {
    RoundShape shape[kRoundShapes]{};
    uint32_t n = 0;
    constexpr RoundShapeList()
    {
        for (int k = 4; k <= 24; k += 4)
            for (uint32_t m = 2; m <= 4; m += 2)
                for (uint32_t waves = 4; waves <= 16; waves += 4)
                    if (m * waves >= 2 * (uint32_t)k + 2) shape[n++] = RoundShape{k, waves, m};
    }
};
constexpr RoundShapeList kShapes;
static_assert(kShapes.n == kRoundShapes, "shapes of a round");

// A job's part of block_pass_us for a round of k steps of it in shape i.
void set_terms(RoundTerms& t, uint32_t i, const RoundJob& j, int k)
{
    const RoundShape& s = kShapes.shape[i];
    const Geometry& g = j.g;
    const JobBlocks n = job_blocks(g, s, k);
    const uint32_t S = tile_segments(g, k) ? 64 / g.W : 1, group = S * s.m, held = group * s.waves;
    float row = j.kind == 0 ? 0.045f : j.kind == 1 ? 0.090f : 0.119f;
    if (j.feat) row *= 1.1f;
    const float chain = (j.kind == 0 ? 0.04f : 0.16f) * (float)s.m;
    float bw = 0.0f, bl = 0.0f;  // one block's VALU time, and its time alone on a CU
    uint32_t groups = (n.th + group - 1) / group;  // that hold rows still worked on
    for (int left = 0; left < k; ++left) {
        while (groups * group < std::min(held, n.th + 2 * (uint32_t)left)) ++groups;
        const float w = (float)(groups * s.m) / 4.0f * row;
        bw += w;
        bl += 0.08f + std::max(w, chain);
    }
    const float blocks = (float)n.blocks;
    t.work[i] = blocks * bw;
    t.wait[i] = blocks * (bl - bw + 1.5f);
    t.most[i] = bl;
    t.bytes[i] = blocks * (float)(held + n.th) / (float)S * 256.0f * (float)g.Q;
}

}  // namespace

void round_terms(const RoundJob& job, RoundTerms& terms)
{
    for (uint32_t i = 0; i < kRoundShapes; ++i)
        set_terms(terms, i, job, round_steps(kShapes.shape[i], UINT64_MAX, job.force_words));
}

// block_pass_us over a mix, whose blocks share the CUs.  A job's terms do not
// change until its last steps, and the worker keeps them: it predicts anew
// whenever a job comes or ends, with the GPU at most a few rounds behind.  A
// prediction from the start / from the terms: 1000 jobs of 128 x 128 1.1 ms / 10 us
// (rounds of 37 us), 4000 of 64 x 64 4.6 ms / 44 us (rounds of 122).
std::vector<RoundShape> round_shapes(const std::vector<RoundJob>& jobs, uint32_t window, uint32_t ncu)
{
    constexpr uint64_t kMostSteps = kShapes.shape[kRoundShapes - 1].k;
    RoundTerms sum{};
    uint64_t most_words = 0;
    for (const RoundJob& j : jobs) {
        most_words = std::max(most_words, j.force_words);
        RoundTerms own;
        const RoundTerms* t = j.terms;
        if (!t || j.left < kMostSteps) {
            for (uint32_t i = 0; i < kRoundShapes; ++i) set_terms(own, i, j, round_steps(kShapes.shape[i], j.left, j.force_words));
            t = &own;
        }
        for (uint32_t i = 0; i < kRoundShapes; ++i) {
            sum.work[i] += t->work[i];
            sum.wait[i] += t->wait[i];
            sum.most[i] = std::max(sum.most[i], t->most[i]);
            sum.bytes[i] += t->bytes[i];
        }
    }
    const float cus = (float)std::max(ncu, 1u);
    std::vector<std::pair<float, RoundShape>> v;
    for (uint32_t i = 0; i < kRoundShapes; ++i) {
        const RoundShape& s = kShapes.shape[i];
        // with a forced job the steps divide the window and keep its decisions in bounds
        if (most_words && (window % (uint32_t)s.k || (uint64_t)s.k > force_pass_steps(most_words))) continue;
        const uint32_t fit = std::max(1u, std::min(16u / s.waves, 160u * 1024u / block_lds_bytes(2, s.m, s.waves)));
        const float us = 4.5f + std::max(sum.most[i], sum.work[i] / cus + sum.wait[i] / (cus * (float)fit)) +
                         0.5f * sum.bytes[i] / 4.5e6f;
        v.emplace_back(us / (float)s.k, s);
    }
    std::sort(v.begin(), v.end(), [](const auto& x, const auto& y) { return x.first < y.first; });
    std::vector<RoundShape> out;
    for (const auto& x : v) out.push_back(x.second);
    return out;
}

// ------------------------------------------------------------- coarse fields

CoarseUnits coarse_units(int kind, uint32_t r)
{
    // the r + 1 columns in units of at most kCoarseColumns, of about equal size,
    // whole quads of addends: two stages of them take 126 KiB of LDS at most
    const uint32_t chunks = (r + kCoarseColumns) / kCoarseColumns;
    CoarseUnits u;
    u.chunk = ((r + 1 + chunks - 1) / chunks + 3) & ~3u;
    u.chunks = (r + u.chunk) / u.chunk;  // those that hold a column
    // (the chain reads up to three times kChainAhead quads past the last one)
    u.lds = kind == 0 ? 0 : (2 * kCoarseProducers * u.chunk + 3 * 4 * kChainAhead) * 64 * 4;
    return u;
}

// Predicted times of the two kernels.  In units a workgroup's stages follow each
// other, so the time goes by rounds of workgroups on the CUs; a lane per
// coarse cell waits for its chain, or, with enough of them, for the cells'
// arithmetic.  FHP-II, us in units / a lane each: 4096 x 2048 at r = 1 137.5 / 22.2,
// r = 4 18.3 / 10.5, r = 6 11.4 / 16.0, r = 16 11.6 / 63; 8192 x 4096 at r = 2
// 140 / 36.8, r = 5 41.1 / 31.8, r = 8 29.3 / 25.6, r = 16 21.4 / 69; 32768 x
// 8192 at r = 16 154 / 125, r = 32 98 / 247.  On none of 248 sizes (HPP, FHP-I and
// FHP-II, 512 x 256 to 32768 x 8192, r 1 to 32) does it take a kernel that is
// more than a twentieth slower than the other.
bool coarse_in_units(int kind, uint32_t r, uint64_t cells, uint32_t ncu)
{
    if (r > kCoarseExactRadius) return false;
    const float wgs = (float)((cells + 63) / 64), cus = (float)std::max(ncu, 1u);
    if (wgs <= cus) return true;
    const CoarseUnits u = coarse_units(kind, r);
    const uint32_t stages = ((2 * r + 1) * u.chunks + kCoarseProducers - 1) / kCoarseProducers;
    const uint32_t fit = std::min(4u, 160u * 1024u / (u.lds + 6u * 1024u));
    const float wg = kind == 0 ? 2.8f + 1.1f * (float)stages : 4.2f + 0.06f * (float)(stages * u.chunk);
    const float units = 1.8f + wg * std::max(1.0f, wgs / (cus * (float)fit));
    const float visits = (float)(2 * r + 1) * (float)(r + 1);
    const float latency = 4.5f + (kind == 0 ? 0.075f : 0.1f) * visits;
    const float flow = wgs * (0.077f + 0.013f * visits) / cus;
    return units * units <= latency * latency + flow * flow;
}

}  // namespace lgca
