// Shapes of a batch's rounds in blocks (lgca_amd/csrc/lgca_plan.cpp), checked
// without a GPU: a round reads a forced job's decisions of all its steps
// through one buffer descriptor, in which offset 2^31 and up must mean "no
// decision" (kOutside in lgca_block.hpp), so the decisions of any pass stay
// below 2 GiB, whatever was running when the shape was chosen.
// A prediction from the jobs' kept terms chooses what one from the start does, at
// a small part of its cost, which the worker pays whenever a job comes or ends.
// Prints "ROUNDS PASSED" and exits 0 when every check holds.
#include "lgca_kernels.hpp"

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <memory>
#include <random>
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

constexpr uint32_t kWindow = 32, kCus = 256;

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
                const std::vector<RoundShape> shapes = round_shapes(mix, kWindow, kCus);
                CHECK(!shapes.empty(), "a shape for every mix");
                for (const RoundShape& s : shapes) {
                    CHECK(s.k * words * 4 < (1ull << 31), "%d steps of %u x %u words", s.k, r.words, r.rows);
                    CHECK(kWindow % (uint32_t)s.k == 0, "%d steps divide the window", s.k);
                }
            }
            // shapes chosen before the job was admitted
            for (const RoundShape& s : round_shapes({job(kind, 2048, 1024, 0, 1000)}, kWindow, kCus))
                for (uint64_t left : {1ull, 3ull, 7ull, 8ull, 15ull, 16ull, 1000ull}) {
                    const int k = round_steps(s, left, words);
                    CHECK(k >= 1 && (uint64_t)k <= left && k <= s.k, "%d of %d steps", k, s.k);
                    CHECK(k * words * 4 < (1ull << 31), "%d steps (of %d) of %u x %u words", k, s.k, r.words, r.rows);
                    CHECK((uint64_t)k == left || k % 4 == 0, "%d steps keep a multiple of 4", k);
                }
        }
    // small regions change nothing
    for (const RoundShape& s : round_shapes({job(2, 2048, 1024, 0, 1000)}, kWindow, kCus))
        CHECK(round_steps(s, 1000, 64 * 1024) == s.k, "steps of an ordinary job");
}

static void check_kept_terms()
{
    std::mt19937 rng(7);
    for (int mix = 0; mix < 60; ++mix) {
        std::vector<RoundJob> fresh, kept;
        std::vector<std::unique_ptr<RoundTerms>> terms;
        const uint32_t n = 1 + rng() % 40;
        for (uint32_t i = 0; i < n; ++i) {
            const uint32_t dim_x = 20 + rng() % (mix % 3 ? 400 : 9000), dim_y = 2 + 2 * (rng() % 800);
            RoundJob j = job((int)(rng() % 3), dim_x, dim_y, mix % 4 == 3 && rng() % 2 ? rng() % 100000 + 1 : 0, 1000);
            if (mix == 59 && !i) j = job(2, 65536, 32768, 2000ull * 32768, 1000);  // cut to 8 steps
            terms.push_back(std::make_unique<RoundTerms>());
            round_terms(j, *terms.back());
            j.left = rng() % 4 ? 24 + rng() % 500 : 1 + rng() % 30;
            fresh.push_back(j);
            j.terms = terms.back().get();
            kept.push_back(j);
        }
        const std::vector<RoundShape> a = round_shapes(fresh, kWindow, kCus), b = round_shapes(kept, kWindow, kCus);
        CHECK(a.size() == b.size() && !a.empty(), "shapes of mix %d", mix);
        for (size_t i = 0; i < std::min(a.size(), b.size()); ++i)
            CHECK(a[i].k == b[i].k && a[i].m == b[i].m && a[i].waves == b[i].waves, "mix %d, shape %zu", mix, i);
    }
    std::vector<RoundJob> jobs(4000, job(2, 64, 64, 0, 1000));
    auto seconds = [&] {
        double best = 1e9;
        for (int rep = 0; rep < 10; ++rep) {
            const auto t0 = std::chrono::steady_clock::now();
            (void)round_shapes(jobs, kWindow, kCus);
            best = std::min(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
        }
        return best;
    };
    const double anew = seconds();
    RoundTerms terms;
    round_terms(jobs[0], terms);
    for (RoundJob& j : jobs) j.terms = &terms;
    const double kept = seconds();
    CHECK(kept * 5 < anew, "4000 jobs: %.0f us with kept terms, %.0f anew", kept * 1e6, anew * 1e6);
}

// A device with fewer CUs takes longer over the same work: a mix that leaves
// 256 of them half idle takes tall blocks of few redundant rows on 16.
static void check_cus()
{
    const std::vector<RoundJob> mix = {job(2, 2048, 512, 0, 1000), job(2, 1024, 1024, 0, 1000)};
    const RoundShape wide = round_shapes(mix, kWindow, 256).front(), narrow = round_shapes(mix, kWindow, 16).front();
    const JobBlocks a = job_blocks(mix[0].g, wide, wide.k), b = job_blocks(mix[0].g, narrow, narrow.k);
    const double da = (double)(wide.m * wide.waves) / a.th, db = (double)(narrow.m * narrow.waves) / b.th;  // rows held per stored one
    CHECK(db < da, "16 CUs: %.2f rows held per stored one, 256: %.2f", db, da);
}

int main()
{
    check_cus();
    check_force_bound();
    check_kept_terms();
    if (failures) {
        std::printf("%d checks failed\n", failures);
        return 1;
    }
    std::printf("ROUNDS PASSED\n");
    return 0;
}
