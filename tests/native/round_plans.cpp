// Shapes of a batch's rounds in blocks (lgca_amd/csrc/lgca_plan.cpp), checked
// without a GPU: a round reads a forced job's decisions of all its steps
// through one buffer descriptor, in which offset 2^31 and up must mean "no
// decision" (kOutside in lgca_block.hpp), so the decisions of any pass stay
// below 2 GiB, whatever was running when the shape was chosen.
// Prints "ROUNDS PASSED" and exits 0 when every check holds.
#include "lgca_kernels.hpp"

#include <cstdio>
#include <vector>

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

constexpr uint32_t kWindow = 32;

static RoundJob job(int kind, uint32_t dim_x, uint32_t dim_y, uint64_t force_words, uint64_t left)
{
    return RoundJob{make_geometry(dim_x, dim_y, kind == 0 ? 4 : kind == 1 ? 6 : 7), kind, force_words != 0, force_words, left};
}

static void check_force_bound()
{
    // regions of 0.5 to 2.147 G cells, the largest that 8-step passes can read
    struct {
        uint32_t dim_x, dim_y, words, rows;  // region: words x rows from the origin
    } regions[] = {{32768, 32768, 512, 32766}, {32768, 32768, 1024, 30518}, {32768, 32768, 1024, 32766},
                   {32768, 32768, 1024, 32768}, {65536, 32768, 1049, 32768}, {65536, 32768, 2048, 16500},
                   {65536, 32768, 1500, 32768}, {40000000, 34, 1250000, 32}, {40000000, 64, 1250000, 53},
                   {32768, 65534, 1024, 65534}, {65536, 32768, 2047, 32768}};
    for (int kind : {0, 1, 2})
        for (const auto& r : regions) {
            const uint64_t words = (uint64_t)r.words * r.rows;
            const RoundJob forced = job(kind, r.dim_x, r.dim_y, words, 1000);
            CHECK(words * 8 * 4 < (1ull << 31) && force_pass_steps(words) >= 8, "an accepted region (%u x %u words)", r.words, r.rows);
            std::vector<std::vector<RoundJob>> mixes = {{forced}, {job(2, 512, 512, 0, 100), forced, job(0, 64, 64, 128, 7)}};
            for (const auto& mix : mixes) {
                const std::vector<RoundShape> shapes = round_shapes(mix, kWindow);
                CHECK(!shapes.empty(), "a shape for every mix");
                for (const RoundShape& s : shapes) {
                    CHECK(s.k * words * 4 < (1ull << 31), "%d steps of %u x %u words", s.k, r.words, r.rows);
                    CHECK(kWindow % (uint32_t)s.k == 0, "%d steps divide the window", s.k);
                }
            }
            // shapes chosen before the job was admitted
            for (const RoundShape& s : round_shapes({job(kind, 2048, 1024, 0, 1000)}, kWindow))
                for (uint64_t left : {1ull, 3ull, 7ull, 8ull, 15ull, 16ull, 1000ull}) {
                    const int k = round_steps(s, left, words);
                    CHECK(k >= 1 && (uint64_t)k <= left && k <= s.k, "%d of %d steps", k, s.k);
                    CHECK(k * words * 4 < (1ull << 31), "%d steps (of %d) of %u x %u words", k, s.k, r.words, r.rows);
                    CHECK((uint64_t)k == left || k % 4 == 0, "%d steps keep a multiple of 4", k);
                }
        }
    // small regions change nothing
    for (const RoundShape& s : round_shapes({job(2, 2048, 1024, 0, 1000)}, kWindow))
        CHECK(round_steps(s, 1000, 64 * 1024) == s.k, "steps of an ordinary job");
}

int main()
{
    check_force_bound();
    if (failures) {
        std::printf("%d checks failed\n", failures);
        return 1;
    }
    std::printf("ROUNDS PASSED\n");
    return 0;
}
