// The mapping of block passes (block_body in lgca_amd/csrc/lgca_block.hpp, with
// the shapes of lgca_plan.cpp), checked without a GPU by going through every
// workgroup, wave, lane and row of a pass as the kernel does:
//   * every (row, word) of the lattice is stored exactly once;
//   * the words `halo` lanes either side of a stored one are its neighbours in
//     the row (modulo the row), and hold at least k cells a side;
//   * a block holds hk >= k rows either side of the stored ones, on even rows
//     where the row parity is taken from the place in the block, and its waves
//     work as long as a stored row depends on theirs;
//   * offsets stay below the 2 GiB that mean "none", and an item's shape bits
//     come back as they went in.
// Prints "BLOCKS PASSED" and exits 0 when every check holds.
#include "lgca_kernels.hpp"

#include <algorithm>
#include <cstdio>
#include <vector>

using namespace lgca;

static int failures = 0;
static long passes = 0;

#define CHECK(cond, ...)                         \
    do {                                         \
        if (!(cond) && ++failures < 40) {        \
            std::printf("FAILED: " __VA_ARGS__); \
            std::printf("\n");                   \
        }                                        \
    } while (0)

struct Lane {
    int wabs;          // word before the wrap
    uint32_t w;        // word of the row
    uint32_t group;    // group of m rows
    uint32_t y0, rows; // its row tile
    bool writer;
    uint32_t left, right;  // lanes that hold words w - 1 and w + 1
};

static void check_pass(const Geometry& g, uint32_t k, const BlockShape& s)
{
    ++passes;
    const uint32_t hk = block_halo(s.m, k), halo = tile_halo(g, (int)k);
    const BlockLanes lanes = block_lanes(g, (int)k);
    const uint32_t tiles = (g.dim_y + s.th - 1) / s.th;
    const uint64_t blocks = block_count(g, (int)k, tiles);
    const uint32_t nstrips = (uint32_t)(lanes == kLanesPacked ? blocks : blocks / tiles);
    const uint32_t S = lanes == kLanesRows ? 64 / g.W : 1;
#define WHERE "%u x %u, %u steps, m %u, waves %u, th %u", g.dim_x, g.dim_y, k, s.m, s.waves, s.th
    CHECK(s.th % 2 == 0 && hk >= k && (s.m == 1 || hk % 2 == 0), "halo and tile: " WHERE);
    CHECK(s.m * s.waves * S >= s.th + 2 * hk, "rows held: " WHERE);
    CHECK(blocks % nstrips == 0 && (lanes == kLanesRows || halo <= 16), "strips: " WHERE);
    CHECK(lanes == kLanesRows ? g.W <= 64 : (k <= 32 && halo < g.W + 64), "lanes: " WHERE);
    if (lanes != kLanesStrips) CHECK((uint64_t)g.dim_y * g.Q * g.P * 4 < (1ull << 31), "offsets: " WHERE);
    if (lanes != kLanesRows) {
        uint32_t west = 0, east = 0;  // cells of the halo words beside word 0 and beside word W - 1
        for (uint32_t i = 1; i <= halo; ++i) {
            west += (g.W * 64 - i) % g.W + 1 == g.W ? g.nb : 32;
            east += (g.W - 1 + i) % g.W + 1 == g.W ? g.nb : 32;
        }
        CHECK(west >= k && east >= k, "cells of the halo: " WHERE);
    }
    std::vector<uint8_t> stored((size_t)g.dim_y * g.W, 0);
    for (uint64_t item = 0; item < blocks; ++item) {
        const uint32_t tile = (uint32_t)(item / nstrips), strip = (uint32_t)(item - (uint64_t)tile * nstrips);
        for (uint32_t wave = 0; wave < s.waves; ++wave) {
            Lane L[64];
            for (uint32_t lane = 0; lane < 64; ++lane) {
                Lane& c = L[lane];
                c.y0 = tile * s.th;
                c.rows = lanes == kLanesPacked ? 0 : std::min(s.th, g.dim_y - c.y0);
                c.group = wave;
                c.left = lane - 1;
                c.right = lane + 1;
                if (lanes == kLanesPacked) {
                    const uint32_t stride = 64u - 2u * halo, span = g.W + 2u * halo, total = tiles * span;
                    const int f = (int)(strip * stride) - (int)halo + (int)lane;
                    const uint32_t at = (uint32_t)std::min(std::max(f, 0), (int)total - 1), t = at / span;
                    c.y0 = t * s.th;
                    c.rows = std::min(s.th, g.dim_y - c.y0);
                    c.wabs = (int)(at - t * span) - (int)halo;
                    c.writer = lane >= halo && lane < 64u - halo && f < (int)total && c.wabs >= 0 && c.wabs < (int)g.W;
                } else if (lanes == kLanesRows) {
                    const uint32_t seg = lane / g.W, base = seg * g.W;
                    c.group = wave * S + std::min(seg, S - 1u);
                    c.wabs = (int)(lane - base);
                    c.writer = seg < S;
                    c.left = (c.wabs == 0 ? base + g.W - 1u : lane - 1u) & 63u;
                    c.right = ((uint32_t)c.wabs + 1u == g.W ? base : lane + 1u) & 63u;
                } else {
                    c.wabs = (int)(strip * (64u - 2u * halo)) - (int)halo + (int)lane;
                    c.writer = lane >= halo && lane < 64u - halo && c.wabs < (int)g.W;
                }
                CHECK(c.wabs + (int)g.W >= 0, "word below the row: " WHERE);
                c.w = (uint32_t)((c.wabs + (int)g.W) % (int)g.W);
            }
            const uint32_t most = lanes == kLanesPacked ? s.th : L[0].rows;
            const int lo = (int)(wave * S * s.m), hi = lo + (int)(S * s.m);
            const int idle = std::max(0, std::max(lo - (int)(hk + most) + 1, (int)hk - hi + 1)), act = (int)k - idle;
            for (int step = 0; step < (int)k; ++step) {
                const int left = (int)k - 1 - step;  // steps after this one
                const bool needed = lo < (int)hk + (int)most + left && hi > (int)hk - left;
                CHECK(!needed || step < act, "a wave idle too early: " WHERE);
            }
            for (uint32_t lane = 0; lane < 64; ++lane) {
                const Lane& c = L[lane];
                if (!c.writer) continue;
                uint32_t l = lane, r = lane;
                for (uint32_t i = 1; i <= (lanes == kLanesRows ? g.W : halo); ++i) {
                    l = L[l].left;
                    r = L[r].right;
                    const bool in = l < 64 && r < 64;
                    CHECK(in, "neighbours in the wave: " WHERE);
                    if (!in) break;
                    CHECK(L[l].w == (c.w + (uint64_t)g.W * 64 - i) % g.W && L[r].w == (c.w + i) % g.W && L[l].y0 == c.y0 &&
                              L[r].y0 == c.y0 && L[l].group == c.group && L[r].group == c.group,
                          "neighbours in the row: " WHERE);
                }
                for (uint32_t m = 0; m < s.m; ++m) {
                    const uint32_t row = c.group * s.m + m;  // of the block
                    if (row < hk || row >= hk + c.rows) continue;
                    CHECK(idle == 0, "stored rows of an idle wave: " WHERE);
                    const int64_t y = (int64_t)c.y0 - hk + row;
                    CHECK(y >= 0 && y < (int64_t)g.dim_y, "stored row: " WHERE);
                    // parity as the kernel has it: m (even m), or the row's place in the block
                    CHECK(((s.m % 2 == 0 ? m : row + hk) & 1u) == ((uint64_t)y & 1u), "row parity: " WHERE);
                    if (y >= 0 && y < (int64_t)g.dim_y) ++stored[(size_t)y * g.W + c.w];
                }
            }
        }
    }
    CHECK(std::count(stored.begin(), stored.end(), (uint8_t)1) == (long)stored.size(), "stored once: " WHERE);
    const uint32_t bits = block_shape_bits(s.th, lanes == kLanesRows ? 0 : halo, k, lanes);
    CHECK((bits & 0xFFFFu) == s.th && ((bits >> 16) & 0x7Fu) == (lanes == kLanesRows ? 0 : halo) && ((bits >> 24) & 0x7Fu) == k &&
              (bits >> 31) == (lanes == kLanesRows) && ((bits >> 23) & 1u) == (lanes == kLanesPacked),
          "shape bits: " WHERE);
#undef WHERE
}

int main()
{
    // rows of one word, of several a wave, of just a wave, of a little more, packed and in strips
    for (uint32_t dim_x : {1u, 7u, 32u, 33u, 100u, 512u, 1024u, 1056u, 1100u, 1984u, 1985u, 2016u, 2017u, 2048u, 2049u, 2100u, 3000u,
                           3970u, 4400u, 6000u})
        for (uint32_t dim_y : {2u, 6u, 14u, 90u, 256u})
            for (int kind : {2}) {
                const Geometry g = make_geometry(dim_x, dim_y, kind ? 7 : 4);
                for (uint32_t k : {1u, 2u, 3u, 7u, 8u, 13u, 16u, 24u, 27u, 28u}) {
                    const std::vector<BlockShape> shapes = block_shapes(g, kind, k);
                    // (the smallest shape of all holds 4 rows)
                    CHECK(!shapes.empty(), "a shape for %u x %u, %u steps", dim_x, dim_y, k);
                    for (const BlockShape& s : shapes)
                        if (block_pass_us(g, kind, true, 256, k, s) > 0.0f && (k < 8 || s.waves >= 8)) check_pass(g, k, s);
                    // a batch's
                    for (uint32_t m : {2u, 4u})
                        for (uint32_t waves : {4u, 16u})
                            if (m * waves >= 2 * block_halo(m, k) + 2 && k <= 24) {
                                const RoundShape r{(int)k, waves, m};
                                const JobBlocks b = job_blocks(g, r, (int)k);
                                CHECK(b.blocks == block_count(g, (int)k, b.tiles), "a job's blocks");
                                check_pass(g, k, BlockShape{m, waves, b.th});
                            }
                }
            }
    if (failures) {
        std::printf("%d checks failed\n", failures);
        return 1;
    }
    std::printf("%ld passes\nBLOCKS PASSED\n", passes);
    return 0;
}
