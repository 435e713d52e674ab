// lgca_dev.hpp -- device building blocks of the lattice-gas engine (gfx950).
//
// Cells are multi-spin coded: one bit per cell in 32-bit words, one word per
// direction ("plane") per 32 consecutive cells of a row.  Bit b of word w of a
// row is cell x = 32*w + b.  Every rule below is pure bitwise logic on such
// words, so one VALU op advances 32 cells; gfx950 fuses most 3-input
// expressions into a single v_bitop3_b32.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lgca {

// Models (src/lgca_common.h:49-54).  FHP-III collides exactly like FHP-II in the
// reference (every FHP-III-only term of src/lgca_models.h:816-839 is
// identically zero), so kernels are instantiated for kinds 0..2 only.
enum : int { kHPP = 0, kFHP1 = 1, kFHP2 = 2 };

// Four consecutive words of one plane-row (128 cells).  Bitwise operators act
// element-wise, so every rule below is written once for T = uint32_t (one
// word) and T = u32x4 (a quad); the compiler emits one VALU op per element.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int num_dir_of_kind(int kind) { return kind == kHPP ? 4 : (kind == kFHP1 ? 6 : 7); }

// ------------------------------------------------------- three-input logic
// Any bitwise function of three words is one v_bitop3_b32 on gfx950.  Its
// truth table LUT holds f(x, y, z) at bit 4x + 2y + z, so writing f on the
// operand masks kX, kY, kZ gives the table: bit3<kX & ~kY & kZ>(x, y, z) is
// x & ~y & z.  Left to itself the compiler splits many such expressions into
// two-input ops; the rules below are written directly as three-input steps.
constexpr uint32_t kX = 0xF0u, kY = 0xCCu, kZ = 0xAAu;

template <uint32_t LUT>
__host__ __device__ __forceinline__ uint32_t bit3(uint32_t x, uint32_t y, uint32_t z)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_bitop3_b32(x, y, z, (unsigned char)(LUT & 0xFFu));
#else
    uint32_t r = 0;
    for (int i = 0; i < 8; ++i)
        if ((LUT >> i) & 1u) r |= ((i & 4) ? x : ~x) & ((i & 2) ? y : ~y) & ((i & 1) ? z : ~z);
    return r;
#endif
}

template <uint32_t LUT>
__host__ __device__ __forceinline__ u32x4 bit3(u32x4 x, u32x4 y, u32x4 z)
{
    u32x4 r;
    r.x = bit3<LUT>(x.x, y.x, z.x);
    r.y = bit3<LUT>(x.y, y.y, z.y);
    r.z = bit3<LUT>(x.z, y.z, z.z);
    r.w = bit3<LUT>(x.w, y.w, z.w);
    return r;
}

constexpr uint32_t kXor3 = kX ^ kY ^ kZ;
constexpr uint32_t kMaj = (kX & kY) | (kZ & (kX | kY));
constexpr uint32_t kAnd3 = kX & kY & kZ;
constexpr uint32_t kOr3 = kX | kY | kZ;
constexpr uint32_t kMux = (kX & kY) | (~kX & kZ);  // x ? y : z

// --------------------------------------------------------------- Philox4x32-10
// Salmon, Moraes, Dror, Shaw, SC'11.  The key schedule is wave-uniform, so the
// per-round Weyl increments stay in scalar registers.
struct U4 { uint32_t x, y, z, w; };

__host__ __device__ __forceinline__ U4 philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                            uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) { k0 += 0x9E3779B9u; k1 += 0xBB67AE85u; }
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        // the first two rounds often work on wave-uniform counter words,
        // which the compiler keeps in scalar registers; later rounds use
        // one three-input xor each
        const uint32_t n0 = r < 2 ? ((uint32_t)(p1 >> 32) ^ c1 ^ k0) : bit3<kXor3>((uint32_t)(p1 >> 32), c1, k0);
        const uint32_t n2 = r < 2 ? ((uint32_t)(p0 >> 32) ^ c3 ^ k1) : bit3<kXor3>((uint32_t)(p0 >> 32), c3, k1);
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
    }
    return U4{c0, c1, c2, c3};
}

// ------------------------------------------------------------------- collision
// HPP (src/lgca_models.h:134-152): an isolated head-on pair along one axis
// turns into a pair along the other, which happens exactly when s0 == s2,
// s1 == s3 and s0 != s1.
template <typename T>
__host__ __device__ __forceinline__ void collide_hpp(T s[4])
{
    const T k = bit3<~(kX ^ kY) & (kX ^ kZ)>(s[0], s[2], s[1]);  // s0 == s2 != s1
    const T h = bit3<kX & ~(kY ^ kZ)>(k, s[1], s[3]);             // and s1 == s3
    s[0] ^= h; s[1] ^= h; s[2] ^= h; s[3] ^= h;
}

// FHP-I / FHP-II (src/lgca_models.h:367-395, 568-613), restated by occupancy.
// s[0..5] moving directions, s[6] rest (FHP-II), p chirality (1 = clockwise).
//   * exactly two moving particles, head-on {k, k+3}: rotate by +60 degrees
//     (p = 0) or -60 degrees (p = 1), rest untouched;
//   * exactly three, {0,2,4} or {1,3,5}: swap, rest untouched;
//   * FHP-II: rest + exactly one moving particle i -> particles i-1 and i+1;
//     exactly two moving at i-1 and i+1 without rest -> rest + particle i.
// Every step is one three-input operation (32 for FHP-II, 21 for FHP-I).  The
// sums are those of the triples {0,2,4} and {1,3,5}: a head-on pair has one
// particle in each, a pair i-1, i+1 both in one, and a symmetric triple is one
// triple full and the other empty, so each class of events is a function of
// the two sums.  (With the triples {0,1,2} and {3,4,5} and occupancy counts it
// took 43 and 25: 32768 x 8192 FHP-III 20.1 us a step, 18.5 so; 128 ensemble
// FHP-II jobs 47.7 ms, 41.9 so.)
template <bool WITH_REST, typename T>
__host__ __device__ __forceinline__ void collide_fhp(T s[7], T p)
{
    const T a0 = s[0], a1 = s[1], a2 = s[2], a3 = s[3], a4 = s[4], a5 = s[5];
    // particles in the triples: x1 + 2 c1 and x2 + 2 c2
    const T x1 = bit3<kXor3>(a0, a2, a4), c1 = bit3<kMaj>(a0, a2, a4);
    const T x2 = bit3<kXor3>(a1, a3, a5), c2 = bit3<kMaj>(a1, a3, a5);
    // symmetric triples: both sums 0 or 3 (x == c), and not the same
    const T f = bit3<~(kX ^ kY) & (kX ^ kZ)>(x1, c1, x2);
    const T t = bit3<kX & ~(kY ^ kZ)>(f, x2, c2);
    // head-on pairs with nothing else moving: at most one particle a triple
    const T q = bit3<~(kX | kY)>(c1, c2, c2);
    const T h0 = bit3<kAnd3>(q, a0, a3), h1 = bit3<kAnd3>(q, a1, a4), h2 = bit3<kAnd3>(q, a2, a5);
    // class m = d mod 3 flips when its own pair leaves or a pair rotates in:
    // p = 0 moves pair k to class k+1, p = 1 to class k+2.  A pair flips two
    // classes, a symmetric triple all three.
    const T A0 = bit3<kOr3>(t, h0, bit3<kMux>(p, h1, h2));
    const T A1 = bit3<kOr3>(t, h1, bit3<kMux>(p, h2, h0));
    const T A2 = bit3<kXor3>(t, A0, A1);
    if (WITH_REST) {
        const T r = s[6];
        // A rest-rule event: with rest, a lone particle i moves to i-1 and
        // i+1; without, two particles i-1, i+1 merge into i; the rest bit
        // flips.  Either way one triple is empty before and the other after,
        // and the directions d that are set are those opposite an unset d+3:
        // a lone i leaves unset the two others of its triple, opposite i-1 and
        // i+1, and the pair i-1, i+1 leaves unset the direction opposite i.
        // E: the particles are in {0,2,4}; O: in {1,3,5}.
        constexpr uint32_t kOne = (kX & kY & ~kZ) | (~kX & ~kY & kZ);  // (r, x, c): 1 with rest, 2 without
        const T E = bit3<kX & ~(kY | kZ)>(bit3<kOne>(r, x1, c1), x2, c2);
        const T O = bit3<kX & ~(kY | kZ)>(bit3<kOne>(r, x2, c2), x1, c1);
        constexpr uint32_t kKeep = (kX ^ kY) & ~kZ, kSet = kX | (kY & ~kZ);
        s[0] = bit3<kSet>(bit3<kKeep>(a0, A0, E), O, a3);
        s[1] = bit3<kSet>(bit3<kKeep>(a1, A1, O), E, a4);
        s[2] = bit3<kSet>(bit3<kKeep>(a2, A2, E), O, a5);
        s[3] = bit3<kSet>(bit3<kKeep>(a3, A0, O), E, a0);
        s[4] = bit3<kSet>(bit3<kKeep>(a4, A1, E), O, a1);
        s[5] = bit3<kSet>(bit3<kKeep>(a5, A2, O), E, a2);
        s[6] = bit3<kXor3>(r, E, O);
    } else {
        s[0] = a0 ^ A0; s[1] = a1 ^ A1; s[2] = a2 ^ A2;
        s[3] = a3 ^ A0; s[4] = a4 ^ A1; s[5] = a5 ^ A2;
    }
}

template <int KIND, typename T>
__host__ __device__ __forceinline__ void collide(T s[7], T p)
{
    if (KIND == kHPP) collide_hpp<T>(s);
    else collide_fhp<KIND == kFHP2, T>(s, p);
}

// ---------------------------------------------------------- solid-cell rules
// Direction permutations (src/lgca_models.h:44-48, 239-243, 446-450):
//   inverse: HPP d+2, FHP d+3; mirror in x: -d; mirror in y: HPP 2-d, FHP 3-d
//   (mod 4 or 6; the rest direction maps to itself).
template <int KIND> __host__ __device__ constexpr int inv_dir(int d)
{ return KIND == kHPP ? ((d + 2) & 3) : (d == 6 ? 6 : (d + 3) % 6); }
template <int KIND> __host__ __device__ constexpr int mirx_dir(int d)
{ return KIND == kHPP ? ((4 - d) & 3) : (d == 6 ? 6 : (6 - d) % 6); }
template <int KIND> __host__ __device__ constexpr int miry_dir(int d)
{ return KIND == kHPP ? ((6 - d) & 3) : (d == 6 ? 6 : (9 - d) % 6); }

// Applies the destination-cell dispatch of src/omp_lattice.cpp:193-231 to one
// word: fluid bits keep the collided value c, NO_SLIP bits take the bounce-back
// of the pulled value in, SLIP bits take the x-mirror on the north/south rows,
// the y-mirror on the east/west columns (y wins at corners), and pass through
// elsewhere.  ns, sl: NO_SLIP and SLIP masks; edge: cells on x = 0 or
// x = dim_x - 1; ns_row: the word lies on row 0 or dim_y - 1.
template <int KIND, typename T>
__host__ __device__ __forceinline__ void apply_solids(T c[7], const T in[7], T ns, T sl, T edge,
                                                      bool ns_row)
{
    constexpr int Q = num_dir_of_kind(KIND);
    const T fl = ~(ns | sl);
    T o[7];
#pragma unroll
    for (int d = 0; d < Q; ++d) {
        T sp = ns_row ? in[mirx_dir<KIND>(d)] : in[d];
        sp = (edge & in[miry_dir<KIND>(d)]) | (~edge & sp);
        o[d] = (fl & c[d]) | (ns & in[inv_dir<KIND>(d)]) | (sl & sp);
    }
#pragma unroll
    for (int d = 0; d < Q; ++d) c[d] = o[d];
}

// apply_solids where no cell of the word is SLIP (sl == 0): a NO_SLIP bit
// takes the bounce-back of the pulled value, a fluid bit the collided value,
// one three-input select per plane.
template <int KIND, typename T>
__host__ __device__ __forceinline__ void apply_no_slip(T c[7], const T in[7], T ns)
{
    constexpr int Q = num_dir_of_kind(KIND);
    T o[7];
#pragma unroll
    for (int d = 0; d < Q; ++d) o[d] = bit3<kMux>(ns, in[inv_dir<KIND>(d)], c[d]);
#pragma unroll
    for (int d = 0; d < Q; ++d) c[d] = o[d];
}

// Body-force flip rules of apply_body_force (src/omp_lattice.cpp:293-337) on
// the cells selected by f (already restricted to FLUID cells).
template <int KIND, typename T>
__host__ __device__ __forceinline__ void apply_force(T s[7], T f, int dir)
{
    if (KIND == kHPP) {
        if (dir == 1) { const T m = f & ~s[0] & s[2]; s[0] ^= m; s[2] ^= m; }
        else          { const T m = f & s[1] & ~s[3]; s[1] ^= m; s[3] ^= m; }
    } else {
        if (dir == 1) { const T m = f & ~s[0] & s[3]; s[0] ^= m; s[3] ^= m; }
        else {
            const T m1 = f & s[1] & ~s[5];
            const T m2 = f & s[2] & ~s[4];
            s[1] ^= m1; s[5] ^= m1;
            s[2] ^= m2; s[4] ^= m2;
        }
    }
}

// Initial fill of plane d of word w of row y (hash stream 2): bit b is set
// when philox({x >> 2, y, d, 2})[x & 3] < thr for x = 32w + b, also past the end
// of the row: the caller masks.
__device__ __forceinline__ uint32_t fill_word(uint32_t w, uint32_t y, uint32_t d, uint32_t key0, uint32_t key1,
                                              uint64_t thr)
{
    const uint32_t t = (uint32_t)thr, all = (uint32_t)(thr >> 32);  // thr = 2^32 fills every cell
    uint32_t word = 0;
#pragma unroll
    for (uint32_t gi = 0; gi < 8; ++gi) {
        const U4 r = philox4x32_10(8 * w + gi, y, d, 2u, key0, key1);
        word |= ((uint32_t)(r.x < t) | (uint32_t)(r.y < t) << 1 | (uint32_t)(r.z < t) << 2 | (uint32_t)(r.w < t) << 3)
                << (4 * gi);
    }
    return all ? ~0u : word;
}

// Per-cell force decisions of word w of row y at one step of the four-step
// group G = step >> 2: 32 independent Bernoulli(thr / 2^32) bits by
// first-fire sampling.  u0 is the word's first uniform for this step,
// philox({w, y, G, 1})[step & 3] (one call serves the group).  Further
// uniforms, needed only after a fire, are the group's extras
// E_e = philox({w, y, G, 5 + 4 (e >> 2)})[e & 3], e = 0, 1, ..., shared by the
// group's steps in step order, each step starting after the extras that the
// group's earlier steps took.  With Q_1 = q = 2^32 - thr and
// Q_{k+1} = floor(Q_k q / 2^32), the first of the next n cells to fire is the
// smallest m < n with u + Q_{m+1} < 2^32, and there is none when
// u + Q_n >= 2^32.  The table holds the complements ~Q_1..~Q_32 (force_table):
// u + Q >= 2^32 exactly when u > ~Q.
__device__ __forceinline__ bool force_fires(uint32_t u0, const uint32_t* nQ) { return u0 <= nQ[31]; }

// Offset of the first fire among 32 cells for uniform u, 32 when none fires:
// the number of k in [0, 32) with u > nQ[k], a prefix because Q decreases.
// Five fixed lifting steps find it up to 31, and nQ[31] adds the last; no
// branches, so the lanes of a wave stay in step.  For the next n cells of a
// word the first fire is this offset when it is < n, else there is none (the
// prefix covers the first n cells).
__device__ __forceinline__ uint32_t force_first(uint32_t u, const uint32_t* nQ)
{
    uint32_t m = 0;
#pragma unroll
    for (uint32_t step = 16; step; step >>= 1) m += u > nQ[m + step - 1] ? step : 0u;
    return m + (u > nQ[31] ? 1u : 0u);
}

// Fills nQ[0..31] = ~Q_1..~Q_32 for q = 2^32 - thr (exact integer steps, the
// same on every platform) and makes it visible to the whole workgroup.
__device__ __forceinline__ void force_table(uint32_t* nQ, uint32_t q)
{
    if (threadIdx.x == 0) {
        uint32_t Qk = q;
        for (int k = 0; k < 32; ++k) {
            nQ[k] = ~Qk;
            Qk = __umulhi(Qk, q);
        }
    }
    __syncthreads();
}

// Bits of word w inside the forced columns [fx0, fx1) and the lattice.
__device__ __forceinline__ uint32_t force_columns(uint32_t w, uint32_t fx0, uint32_t fx1, uint32_t dim_x)
{
    const uint32_t x0 = 32 * w;
    const uint32_t hi = min(min(fx1, dim_x), x0 + 32);
    const uint32_t lo = max(fx0, x0);
    if (lo >= hi) return 0;
    const uint32_t nbits = hi - lo, sh = lo - x0;
    return (nbits == 32 ? 0xFFFFFFFFu : ((1u << nbits) - 1u)) << sh;
}

// Force draws.  A workgroup of kDrawThreads threads draws the decision words of
// kDrawWords consecutive (row, word) pairs of a force region for one group of
// four steps.  At p <= 5e-3 a word fires in at most 15 % of its steps, but of
// the 64 words of a wave one almost always does, so a thread per word had
// every wave make the second Philox call and walk every step for a few lanes:
// about 500 instructions a wave.  So the first pass only makes the first call,
// stores zeros for the words that never fire in the group and lists the
// others in LDS; the second takes the listed words, 64 to a wave again, each
// lane stepping through its own fires, one search of the table each.
// 6000 x 3000 cells forced at p = 5e-3, 28 steps: 59 -> 32 us (searching the
// table by a logarithm and two reads: 41 for 39 at the time; results through
// LDS to whole-line stores: 42).
//
// 1024 words leave the second pass few idle lanes where few words fire.  Where
// most do (p >= 0.05, by q), or chunks of 1024 are fewer than two a CU (`few`), a
// lane would walk four words' fires one after the other, and takes one.  64 steps
// of FHP-II, us with chunks of 1024 / 256: 512 x 256 at p = 5e-3 65 / 59, p = 0.5
// 305 / 123; 2048 x 512 at p = 1e-3 83 / 86, p = 0.5 343 / 201; 6000 x 3000 at p =
// 5e-3 259 / 291, p = 0.5 1550 / 1435; 8192 x 4096 at p = 0.02 610 / 651, p = 0.1
// 1101 / 1079.
constexpr uint32_t kDrawThreads = 256, kDrawWords = 1024;
constexpr uint64_t kDrawFew = 512;  // chunks
__host__ __device__ inline bool draw_dense(uint32_t q) { return q <= 4080218932u; }
__host__ __device__ inline uint32_t draw_words(bool few, uint32_t q)
{
    return few || draw_dense(q) ? kDrawThreads : kDrawWords;
}

struct DrawShared {
    uint32_t nQ[32];
    uint32_t count;
    uint32_t idx[kDrawWords];   // of the region's (row, word) pairs, from the chunk's first
    uint32_t u[4][kDrawWords];  // the group's first uniforms
};
struct DrawRegion {
    uint32_t* dec;              // decision word of step step0 + k and pair i at dec[k * plane + i]
    uint64_t plane;             // (row, word) pairs
    uint32_t nsteps, step0, key0, key1;
    uint32_t fx0, fx1, fy0, fw0, fwn, dim_x;
    uint32_t words;             // words of a chunk (draw_words)
};

// force_table has filled sh.nQ.  Group `group` is counted from step0 & ~3;
// steps of the group before step0 are walked too: they take extras before
// the later steps do.
__device__ __forceinline__ void draw_chunk(const DrawRegion& a, uint64_t first_pair, uint32_t group, DrawShared& sh)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t skip = a.step0 & 3u;
    const uint32_t G = ((a.step0 & ~3u) + 4u * group) >> 2;  // of the group's steps mod 2^32
    const uint32_t i0 = group == 0 ? skip : 0u;                   // the group's steps in the window
    const uint32_t i1 = min(4u, skip + a.nsteps - 4u * group);
    // (i0 may lie past the first steps, so the pointer arithmetic is signed)
    uint32_t* dec = a.dec + (int64_t)(4 * (int64_t)group - (int64_t)skip) * (int64_t)a.plane;
    const uint32_t magic = 0xFFFFFFFFu / a.fwn;  // at * magic >> 32 is at / fwn or one less
    auto pair = [&](uint64_t at, uint32_t& w, uint32_t& y) {
        if (a.plane < ((uint64_t)1 << 32)) {  // the usual case
            y = __umulhi((uint32_t)at, magic);
            w = (uint32_t)at - y * a.fwn;
            if (w >= a.fwn) {
                w -= a.fwn;
                ++y;
            }
        } else {
            y = (uint32_t)(at / a.fwn);
            w = (uint32_t)(at - (uint64_t)y * a.fwn);
        }
        w += a.fw0;
        y += a.fy0;
    };
    if (tid == 0) sh.count = 0;
    __syncthreads();
    for (uint32_t k = 0; k < a.words; k += kDrawThreads) {
        const uint64_t at = first_pair + k + tid;
        bool fires = false;
        U4 r{0, 0, 0, 0};
        if (at < a.plane) {
            uint32_t w, y;
            pair(at, w, y);
            r = philox4x32_10(w, y, G, 1u, a.key0, a.key1);
            fires = force_fires(min(min(r.x, r.y), min(r.z, r.w)), sh.nQ);
            if (!fires)
                for (uint32_t i = i0; i < i1; ++i) dec[i * a.plane + at] = 0u;
        }
        const unsigned long long any = __ballot(fires);
        uint32_t base = 0;
        if (lane == 0 && any) base = atomicAdd(&sh.count, (uint32_t)__popcll(any));
        base = __builtin_amdgcn_readfirstlane(base);
        if (fires) {
            const uint32_t e = base + (uint32_t)__popcll(any & ((1ull << lane) - 1ull));
            sh.idx[e] = k + tid;
            sh.u[0][e] = r.x;
            sh.u[1][e] = r.y;
            sh.u[2][e] = r.z;
            sh.u[3][e] = r.w;
        }
    }
    __syncthreads();
    const uint32_t n = sh.count;
    for (uint32_t e = tid; e < n; e += kDrawThreads) {
        const uint64_t at = first_pair + sh.idx[e];
        uint32_t w, y, left = 0;  // left: steps still to walk, those that fire
        pair(at, w, y);
        const uint32_t cols = force_columns(w, a.fx0, a.fx1, a.dim_x);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const bool f = force_fires(sh.u[i][e], sh.nQ);
            left |= f ? 1u << i : 0u;
            if (!f && i >= i0 && i < i1) dec[i * a.plane + at] = 0u;
        }
        U4 ext = philox4x32_10(w, y, G, 5u, a.key0, a.key1);
        uint32_t used = 0, pos = 0, word = 0, i = __ffs(left) - 1;
        uint32_t u = sh.u[i][e];
        for (;;) {
            // u fires among the step's remaining 32 - pos cells
            const uint32_t m = force_first(u, sh.nQ);
            word |= 1u << (pos + m);
            pos += m + 1u;
            bool again = false;
            if (pos < 32u) {
                if ((used & 3u) == 0 && used) ext = philox4x32_10(w, y, G, 5u + used, a.key0, a.key1);
                const uint32_t j = used & 3u;
                u = j == 0 ? ext.x : (j == 1 ? ext.y : (j == 2 ? ext.z : ext.w));
                ++used;
                again = u <= sh.nQ[31u - pos];
            }
            if (again) continue;
            if (i >= i0 && i < i1) dec[i * a.plane + at] = word & cols;
            left &= left - 1u;
            if (!left) break;
            i = __ffs(left) - 1;
            u = sh.u[i][e];
            pos = word = 0;
        }
    }
    __syncthreads();  // the list is free for the next chunk
}

}  // namespace lgca
