// Rules that choose between kernels (lgca_amd/csrc/lgca_plan.cpp), checked
// without a GPU at sizes where both sides were measured (the faster one by a
// tenth or more is expected; 256 CUs).
// Prints "RULES PASSED" and exits 0 when every check holds.
#include "lgca_kernels.hpp"

#include <cstdio>

using namespace lgca;

static int failures = 0;

#define CHECK(cond, ...)                         \
    do {                                         \
        if (!(cond)) {                           \
            std::printf("FAILED: " __VA_ARGS__); \
            std::printf("\n");                   \
            ++failures;                          \
        }                                        \
    } while (0)

static void check_coarse()
{
    struct {
        int kind;
        uint32_t dim_x, dim_y, r;
        bool units;
    } cases[] = {
        // many small coarse cells: a lane each
        {2, 1480, 740, 1, false}, {0, 1480, 740, 1, false}, {2, 1480, 740, 2, false}, {2, 4096, 2048, 1, false},
        {0, 4096, 2048, 2, false}, {2, 4096, 2048, 4, false}, {0, 4096, 2048, 4, false}, {2, 8192, 4096, 4, false},
        {1, 8192, 4096, 8, false}, {2, 8192, 4096, 8, false}, {2, 16384, 8192, 8, false}, {2, 32768, 8192, 16, false},
        // few or large ones: in units
        {2, 256, 256, 1, true}, {2, 1480, 740, 4, true}, {2, 1480, 740, 10, true}, {0, 4096, 2048, 6, true},
        {2, 4096, 2048, 6, true}, {1, 4096, 2048, 8, true}, {0, 8192, 4096, 7, true}, {2, 8192, 4096, 16, true},
        {2, 4400, 2200, 20, true}, {2, 8192, 4096, 32, true}, {2, 32768, 8192, 32, true}, {0, 32768, 8192, 16, true},
        {2, 2046, 2046, 1023, true},
        // sums that FP32 may round
        {0, 2048, 2050, 1024, false}, {2, 100000, 50000, 2000, false}};
    for (const auto& c : cases)
        CHECK(coarse_in_units(c.kind, c.r, (uint64_t)(c.dim_x / (2 * c.r)) * (c.dim_y / (2 * c.r)), 256) == c.units,
              "coarse fields of kind %d, %u x %u at r = %u %s", c.kind, c.dim_x, c.dim_y, c.r, c.units ? "in units" : "by lanes");
    for (uint32_t r = 1; r <= kCoarseExactRadius; ++r) {
        const CoarseUnits u = coarse_units(2, r);
        CHECK(u.chunk % 4 == 0 && u.chunk <= kCoarseColumns && (u.chunks - 1) * u.chunk < r + 1 && u.chunks * u.chunk >= r + 1,
              "units at r = %u", r);
        CHECK(u.lds <= 142 * 1024 && coarse_units(0, r).lds == 0, "LDS at r = %u", r);
    }
}

static void check_short_calls()
{
    struct {
        int kind;
        uint32_t dim_x, dim_y;
        bool walk[3];  // 1, 2, 4 steps
    } cases[] = {
        {2, 2048, 2048, {false, false, false}}, {0, 2048, 512, {false, false, false}}, {2, 4096, 2048, {true, false, false}},
        {2, 6000, 3000, {true, true, false}},   {2, 7000, 3500, {true, true, true}},   {0, 8192, 4096, {true, true, true}},
        {1, 8192, 4096, {true, true, true}},    {2, 12000, 5800, {true, true, true}},  {2, 512, 65534, {true, true, true}},
        {0, 2048, 16384, {false, false, false}}, {2, 1000000, 16, {false, false, false}}, {0, 1000000, 64, {false, false, false}}};
    for (const auto& c : cases) {
        const Geometry g = make_geometry(c.dim_x, c.dim_y, c.kind == 0 ? 4 : c.kind == 1 ? 6 : 7);
        CHECK(block_lattice(g, false) && block_lattice(g, true), "%u x %u runs in blocks", c.dim_x, c.dim_y);
        for (uint32_t i = 0; i < 3; ++i) {
            const uint32_t th = short_walk_rows(g, c.kind, 1u << i);
            CHECK((th != 0) == c.walk[i] && th % 2 == 0 && th <= g.dim_y, "kind %d, %u x %u, %u steps", c.kind, c.dim_x, c.dim_y, 1u << i);
        }
        for (uint64_t n : {0u, 3u, 5u, 6u, 7u, 8u, 12u, 100u}) CHECK(!short_walk_rows(g, c.kind, n), "a walk of %u steps", (uint32_t)n);
    }
}

static void check_block_lattices()
{
    struct {
        uint32_t dim_x, dim_y;
        bool open, solids;  // in blocks without and with solids
    } cases[] = {
        {256, 256, true, true}, {1480, 740, true, true}, {12000, 6000, true, true}, {16384, 8192, false, false},
        {32768, 8192, false, false}, {300000, 40, true, true}, {1000000, 2, true, true}, {2000000, 2, false, true},
        {2000000, 4, true, true}, {4000000, 2, false, true}, {4000000, 4, false, true}, {4000000, 6, true, true},
        {8000000, 4, false, true}, {20, 2, true, true}};
    for (const auto& c : cases) {
        const Geometry g = make_geometry(c.dim_x, c.dim_y, 7);
        CHECK(block_lattice(g, false) == c.open && block_lattice(g, true) == c.solids, "%u x %u in blocks", c.dim_x, c.dim_y);
    }
}

int main()
{
    check_block_lattices();
    check_coarse();
    check_short_calls();
    if (failures) {
        std::printf("%d checks failed\n", failures);
        return 1;
    }
    std::printf("RULES PASSED\n");
    return 0;
}
