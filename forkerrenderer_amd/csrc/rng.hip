// rng.hip -- the reference's random stream on gfx950.
//
// The reference draws every random float from one function-static
// std::mt19937 (default seed 5489) through uniform_real_distribution<float>
// (src/utility.h:90-103), and builds its random vectors by rejection
// (src/geometry.h:947-990).  Its consumers (Render::DoSSAO, the PCF / PCSS
// shadow filters) take the stream strictly in pixel (or fragment) order, so
// the device replays it in parallel chunks reached by jumping ahead, each
// chunk writing its accepted vectors in stream order into its own region;
// the per-pixel kernels then read the vectors of their pixel at a known
// offset (StreamVectors, fgl_device.hpp).
//
// Arithmetic, fixed by the C++ library the reference is built with:
//  * MT19937: the standard twist and tempering on 624 words;
//  * generate_canonical<float, 24>: one 32-bit draw u, float(u) * 2^-32
//    (float(u) rounded to nearest), a result of 1 replaced by the largest
//    float below 1;
//  * Random(-1, 1) = -1 + 2 * r in float;
//  * Vector3f(Random(..), Random(..), Random(..)) evaluates its arguments
//    right to left (the g++ that builds the reference), so a unit-sphere try
//    takes z, y, x from three consecutive draws, a unit-disk try y, x from
//    two; a try is kept when (x*x + y*y) + z*z < 1.
#include "fgl_kernels.hpp"
#include "mt_jump.hpp"

namespace fgl {

constexpr uint32_t kMtN = 624, kMtM = 397;
constexpr uint32_t kMtUpper = 0x80000000u, kMtLower = 0x7fffffffu, kMtMatrix = 0x9908b0dfu;

void mt_seed_state(uint32_t seed, MtState &st)
{
    st.mt[0] = seed;
    for (uint32_t i = 1; i < kMtN; ++i) st.mt[i] = 1812433253u * (st.mt[i - 1] ^ (st.mt[i - 1] >> 30)) + i;
    st.idx = kMtN;
    st.pad = 0;
    st.draws = 0;
}

__device__ __forceinline__ uint32_t mt_twist_word(uint32_t cur, uint32_t next, uint32_t far)
{
    const uint32_t y = (cur & kMtUpper) | (next & kMtLower);
    return far ^ (y >> 1) ^ ((y & 1u) ? kMtMatrix : 0u);
}

__device__ __forceinline__ uint32_t mt_temper(uint32_t z)
{
    z ^= z >> 11;
    z ^= (z << 7) & 0x9d2c5680u;
    z ^= (z << 15) & 0xefc60000u;
    z ^= z >> 18;
    return z;
}

// Random(-1, 1) from one draw: float(u) 2^-32, at most the float below 1, then
// -1 + 2 r -- the scalings are exact, so one fused operation rounds as the sum.
__device__ __forceinline__ float random_pm1(uint32_t u)
{
    return __builtin_fmaf(fminf((float)u, 4294967040.f), 4.6566128730773926e-10f, -1.f);
}

// The generator as one sequence: x_{n+624} = twist(x_n, x_{n+1}, x_{n+397})
// (a block's twist is this recurrence, new words used as they appear).  227
// consecutive words read only words at least 227 back, so a workgroup makes
// them together, a thread each -- and the next 227 as well before anyone has
// to wait: thread t's second word reads x_{j+227} and x_{j+228}, at least 396
// back, and its own first word.  So a pair of steps, 454 words, takes one
// barrier.  The words lie in an LDS array in sequence order, so an interval's
// accesses are one address and constant offsets; a long run copies its last
// 624 words to the front every kMtLap intervals.
//
// The barrier orders LDS alone (a __syncthreads() made a step of 227 words 860
// cycles).
constexpr uint32_t kMtLag = kMtN - kMtM, kMtPair = 2 * kMtLag;

// A running generator: `made` words in, the array holds x_made ..
// x_{made+623} from at - threadIdx.x on.  The first 227 threads make words;
// `far` is x_{made + 397 + t}, the thread's own last one.
struct MtRun {
    uint32_t *at, far;
    __device__ __forceinline__ explicit MtRun(uint32_t *words) : at(words + threadIdx.x), far(0)
    {
        if (threadIdx.x < kMtLag) far = at[kMtM];
    }
    // 454 more words (w0, w1: this thread's), ready after the next barrier.
    __device__ __forceinline__ void pair(uint32_t &w0, uint32_t &w1)
    {
        if (threadIdx.x < kMtLag) {
            const uint32_t c0 = at[0], n0 = at[1], c1 = at[kMtLag], n1 = at[kMtLag + 1];
            w0 = mt_twist_word(c0, n0, far);
            w1 = mt_twist_word(c1, n1, w0);
            at[kMtN] = w0;
            at[kMtN + kMtLag] = w1;
            far = w1;
        }
        at += kMtPair;
    }
};

// The vector that a try of the draws w makes.
template <int D>
__device__ __forceinline__ void mt_vector(const uint32_t (&w)[D], float &x, float &y, float &z)
{
    float r[D];
#pragma unroll
    for (int e = 0; e < D; ++e) r[e] = random_pm1(mt_temper(w[e]));
    z = D == 3 ? r[0] : 0.f;
    y = r[D - 2];
    x = r[D - 1];
}

template <int D>
__device__ __forceinline__ void mt_words(const uint32_t *p, uint32_t (&w)[D])
{
#pragma unroll
    for (int e = 0; e < D; ++e) w[e] = p[e];
}

// ---- the stream in parallel: jump ahead, generate, keep ----
//
// A fill takes the stream's next draws in chunks of L = 624 K draws, L a
// multiple of D, so that no try crosses chunks.  The base sequence x_0, x_1 ..
// starts at the context's next draw; chunk c starts from the 624 words c L
// words into it, which the jump gives (mt_jump.hpp): the XOR of the windows
// x_i .. x_{i+623} over the set bits i of t^(c L) mod phi.  A chunk makes its
// words in LDS, tests its tries there and writes the kept vectors
// only; its draws never reach memory.  Checkpoints -- the generator's words
// and the vectors kept so far, every kMtCkEvery intervals -- let a commit find
// the try that kept the m-th vector without the draws.  Every window of a
// jump, x_{19967 + 623} at most, lies in the base sequence.
static_assert(kMtBaseWords >= 64 * kMtPolyWords + 623, "the jump's windows stay in the base sequence");

// One workgroup: the base sequence's first n words, untempered.
__global__ __launch_bounds__(256) void k_mt_base(const MtState *__restrict__ st, uint32_t n, uint32_t *__restrict__ base)
{
    __shared__ uint32_t words[kMtN + kMtBaseWords + kMtPair];
    const uint32_t tid = threadIdx.x, idx = st->idx;
    for (uint32_t i = tid; i < kMtN; i += 256) {
        const uint32_t v = st->mt[i];
        words[i] = v;
        if (i >= idx && i - idx < n) base[i - idx] = v;
    }
    __syncthreads();
    MtRun run(words);
    for (uint32_t at = kMtN - idx; at < n; at += kMtPair) {
        uint32_t w0, w1;
        run.pair(w0, w1);
        if (tid < kMtLag) {
            if (at + tid < n) base[at + tid] = w0;
            if (at + kMtLag + tid < n) base[at + kMtLag + tid] = w1;
        }
        lds_barrier();
    }
}

// A jump is the XOR of the base sequence's windows x_i .. x_{i+623} over the
// set bits i of a polynomial.  It is bound by LDS reads, so up to three bits
// i, i + 1, i + 2 (i set) are taken by one read: beside x itself the LDS holds
// x_j ^ x_{j+1}, x_j ^ x_{j+2} and x_j ^ x_{j+1} ^ x_{j+2} -- a read per four
// bits of the polynomial on average instead of one per two.  The four arrays
// of the whole base sequence do not fit: a jump is cut into kJumpSegs segments
// of the polynomial, a workgroup each, which also keeps the last round over
// the CUs short.  For the reads at i = 4 q + r thread t gathers the 16-byte
// group q + t, words k + r of the result for k + r in [4 t, 4 t + 4); three
// wavefronts per class r, and the classes' partial arrays are combined at the
// end (word k = XOR over r of partial r at k + r).  269 jumps 180 -> 71 us, 593
// and 505 jumps 234 -> 117 on average.
//
// Which groups are read depends on the polynomial alone: k_mt_lists writes
// them once per polynomial, per segment and class, padded to sixteen with a
// group whose reads are zero, and a jump's wavefronts get them through scalar
// loads.
constexpr int kJumpGroups = ((int)kMtN + 3 + 3) / 4;            // 157: k + r < 627
constexpr int kJumpClassThreads = 192;                          // three wavefronts per class
constexpr int kJumpThreads = 4 * kJumpClassThreads;
static_assert(kJumpGroups <= kJumpClassThreads, "a thread per 16-byte group of a class");
constexpr int kJumpSegs = 3;
static_assert(kMtStateWords == kJumpSegs * (int)kMtN, "a chunk's parts");
constexpr int kSegWords64 = kMtPolyWords / kJumpSegs;           // the polynomial's words of a segment
constexpr int kSegGroups = kSegWords64 * 16 + kJumpGroups;      // groups a segment's reads reach
constexpr int kJumpZero = 4 * kSegGroups;                       // first zero group
constexpr int kJumpLists = 4 * kJumpSegs;
static_assert(kMtDegree + 2 + 623 <= kMtBaseWords, "every word a result takes lies in the base");
static_assert(kJumpLists + 1 == kMtListStarts && kMtPolyWords % kJumpSegs == 0 && kMtBaseWords % 4 == 0, "whole words and groups");
static_assert(kJumpZero + kJumpGroups < 65536 && (kJumpZero + kJumpGroups) * 16 <= 128 * 1024, "16-bit entries; the LDS");

// The reads of a word of the polynomial, ascending: f(bit, array).
template <typename F>
__device__ __forceinline__ void jump_reads(uint64_t v, F f)
{
    while (v) {
        const int b = __builtin_ctzll(v);
        const uint32_t next = (uint32_t)(v >> b) >> 1 & 3u;   // bits b + 1, b + 2 of the word
        f(b, next);
        v = b >= 61 ? 0ull : v & ~0ull << (b + 3);
    }
}

// Workgroup c: polynomial c's lists.  start[13 c + 4 s + r] .. [.. + 1]: the
// list of segment s, class r, in sixteens.
__global__ __launch_bounds__(320) void k_mt_lists(const uint64_t *__restrict__ polys, uint16_t *__restrict__ entries,
                                                  uint32_t *__restrict__ start)
{
    __shared__ uint16_t n[4][kMtPolyWords];
    __shared__ uint32_t sum[kJumpLists], at[kJumpLists + 1];
    const int w = threadIdx.x;
    const uint64_t v = w < kMtPolyWords ? polys[(size_t)blockIdx.x * kMtPolyWords + w] : 0ull;
    uint32_t k[4] = {0, 0, 0, 0};
    jump_reads(v, [&](int b, uint32_t) { ++k[b & 3]; });
    if (w < kMtPolyWords)
        for (int r = 0; r < 4; ++r) n[r][w] = (uint16_t)k[r];
    __syncthreads();
    if (w < kJumpLists) {
        uint32_t run = 0;
        for (int e = 0; e < kSegWords64; ++e) {
            uint16_t &x = n[w & 3][(w >> 2) * kSegWords64 + e];
            const uint32_t m = x;
            x = (uint16_t)run;
            run += m;
        }
        sum[w] = run;
    }
    __syncthreads();
    if (w == 0) {
        uint32_t a = 0;
        for (int l = 0; l < kJumpLists; ++l) {
            at[l] = a;
            a += (sum[l] + 15u) / 16u;
        }
        at[kJumpLists] = a;
    }
    __syncthreads();
    uint16_t *e = entries + (size_t)blockIdx.x * kMtListMax;
    if (w <= kJumpLists) start[(size_t)blockIdx.x * (kJumpLists + 1) + w] = at[w];
    if (w < kJumpLists)
        for (uint32_t i = at[w] * 16u + sum[w]; i < at[w + 1] * 16u; ++i) e[i] = (uint16_t)kJumpZero;
    if (w < kMtPolyWords) {
        const int s = w / kSegWords64;
        for (int r = 0; r < 4; ++r) k[r] = at[4 * s + r] * 16u + n[r][w];
        jump_reads(v, [&](int b, uint32_t p) {
            e[k[b & 3]++] = (uint16_t)(p * kSegGroups + (uint32_t)((w - s * kSegWords64) * 16 + (b >> 2)));
        });
    }
}
static_assert(kMtListMax >= kMtPolyWords * 22 + kJumpLists * 15 && kMtListMax % 16 == 0, "every list fits");

// Workgroup (c - 1, s) makes segment s's part of chunk c's array.
__global__ __launch_bounds__(kJumpThreads) void k_mt_jump(const uint32_t *__restrict__ base, const uint16_t *__restrict__ entries,
                                                          const uint32_t *__restrict__ start, uint32_t *__restrict__ states)
{
    typedef const __attribute__((address_space(4))) uint32_t *ScalarWords;   // scalar loads
    __shared__ uint4 x[kJumpZero + kJumpGroups];
    const int tid = threadIdx.x;
    const int r = __builtin_amdgcn_readfirstlane(tid / kJumpClassThreads), t = tid - r * kJumpClassThreads;
    const ScalarWords first = (ScalarWords)(uintptr_t)(start + (size_t)blockIdx.x * (kJumpLists + 1));
    const ScalarWords list = (ScalarWords)(uintptr_t)(entries + (size_t)blockIdx.x * kMtListMax);
    constexpr int kBaseGroups = kMtBaseWords / 4;
    for (int g = tid; g < kJumpGroups; g += kJumpThreads) x[kJumpZero + g] = make_uint4(0u, 0u, 0u, 0u);
    uint4 acc = make_uint4(0u, 0u, 0u, 0u);
    const int s = blockIdx.y;
    for (int g = tid; g < kSegGroups; g += kJumpThreads) {
        // (past the base: words no result takes)
        const int b = imin(s * kSegWords64 * 16 + g, kBaseGroups - 1);
        const uint4 a = ((const uint4 *)base)[b], n = ((const uint4 *)base)[imin(b + 1, kBaseGroups - 1)];
        const uint4 p = make_uint4(a.x ^ a.y, a.y ^ a.z, a.z ^ a.w, a.w ^ n.x);
        x[g] = a;
        x[kSegGroups + g] = p;
        x[2 * kSegGroups + g] = make_uint4(a.x ^ a.z, a.y ^ a.w, a.z ^ n.x, a.w ^ n.y);
        x[3 * kSegGroups + g] = make_uint4(p.x ^ a.z, p.y ^ a.w, p.z ^ n.x, p.w ^ n.y);
    }
    __syncthreads();
    if (t < kJumpGroups) {
        const uint4 *mine = x + t;
        const uint32_t end = first[4 * s + r + 1];
        for (uint32_t e = first[4 * s + r]; e < end; ++e) {
            uint32_t v[8];
#pragma unroll
            for (int h = 0; h < 8; ++h) v[h] = list[8 * e + h];
#pragma unroll
            for (int h = 0; h < 8; ++h) {
                const uint4 a = mine[v[h] & 0xffffu], b = mine[v[h] >> 16];
                acc.x ^= a.x ^ b.x;
                acc.y ^= a.y ^ b.y;
                acc.z ^= a.z ^ b.z;
                acc.w ^= a.w ^ b.w;
            }
        }
    }
    __syncthreads();
    if (t < kJumpGroups) x[r * kJumpGroups + t] = acc;
    __syncthreads();
    const uint32_t *part = (const uint32_t *)x;
    for (int k = tid; k < (int)kMtN; k += kJumpThreads)
        states[((size_t)(blockIdx.x + 1) * kJumpSegs + s) * kMtN + k] =
            part[k] ^ part[4 * kJumpGroups + k + 1] ^ part[8 * kJumpGroups + k + 2] ^ part[12 * kJumpGroups + k + 3];
}

// The tries of interval q (the words of one pair): [mt_first(q), mt_first(q +
// 1)), at most 227, all of whose words are there when the interval starts.
template <int D>
__host__ __device__ constexpr uint32_t mt_first(uint32_t q) { return q * kMtPair / (uint32_t)D; }

// A thread's try of one interval.
struct MtTry {
    uint32_t rank;                // its vector among its wavefront's kept ones
    unsigned long long kept;      // the wavefront's
    float x, y, z;
    __device__ __forceinline__ MtTry() : rank(0), kept(0), x(0.f), y(0.f), z(0.f) {}
    __device__ __forceinline__ bool ok() const { return __builtin_amdgcn_inverse_ballot_w64(kept); }
    // Which of the wavefront's tries are kept, n in the interval; its count
    // is byte `wave` of cnt (227 at most in all).
    template <int D>
    __device__ __forceinline__ void test(uint32_t &cnt, uint32_t wave, uint32_t n)
    {
        const float r = D == 3 ? (x * x + y * y) + z * z : x * x + y * y;
        const int in = (int)n - 64 * (int)wave;
        kept = __ballot(r < 1.f) & (in >= 64 ? ~0ull : in <= 0 ? 0ull : (1ull << in) - 1ull);
        rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(kept >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)kept, 0u));
        if ((threadIdx.x & 63) == 0) ((uint8_t *)&cnt)[wave] = (uint8_t)__popcll(kept);
    }
};

// Kept before wavefront `wave` (uniform) of an interval with counts k, and in
// the whole interval.
__device__ __forceinline__ uint32_t mt_before(uint32_t k, uint32_t wave) { return (k & ((1u << 8 * wave) - 1u)) * 0x01010101u >> 24; }
__device__ __forceinline__ uint32_t mt_all(uint32_t k) { return k * 0x01010101u >> 24; }

// Workgroup c runs chunk c, T tries: four wavefronts make words, four (D = 2)
// or three (D = 3) test tries and write the kept vectors.  With a workgroup or
// two a CU a slot takes as long as its longest chain of instructions, so the
// testers take two intervals at a time, two neighbouring tries a thread, with
// twice the independent operations between barriers: in slot 2 j + 1 they read
// the tries of intervals 2 j and 2 j + 1 and write what they kept of the two
// before, whose counts are known by then; in slot 2 j + 2 they test them.
// 86 M draws (D = 2) 292 -> 229 us, 190 M (D = 3) 422 -> 331.
constexpr uint32_t kMtLap = 18;                // intervals before the words move to the front, a multiple of 6: whole tries
constexpr uint32_t kMtCkEvery = 2 * kMtLap;    // intervals between checkpoints
template <int D>
constexpr uint32_t kMtFillThreads = 256 + (D == 2 ? 256 : 192);

template <int D>
__global__ __launch_bounds__(kMtFillThreads<D>) void k_mt_fill(const uint32_t *__restrict__ base,
                                                               const uint32_t *__restrict__ states, uint32_t T,
                                                               uint32_t stride, uint32_t n_ck, float *__restrict__ out,
                                                               uint32_t *__restrict__ kept, uint32_t *__restrict__ ck_words,
                                                               uint32_t *__restrict__ ck_kept)
{
    constexpr uint32_t kLapWords = kMtLap * kMtPair;
    static_assert(kLapWords % D == 0 && kMtLap % 2 == 0, "whole tries and pairs of intervals a lap");
    static_assert(D * (mt_first<D>(kMtLap - 2) + 2 * (kMtFillThreads<D> - 256)) <= kMtN + kLapWords, "reads stay in the words");
    __shared__ __align__(16) uint32_t words[kMtN + kLapWords];
    __shared__ __align__(8) uint16_t cnt[2][4];
    const uint32_t tid = threadIdx.x, c = blockIdx.x;
    const uint32_t *src = c == 0 ? base : states + (size_t)c * kMtStateWords;
    for (uint32_t i = tid; i < kMtN; i += kMtFillThreads<D>) {
        uint32_t v = src[i];
        for (int s = 1; s < kJumpSegs && c > 0; ++s) v ^= src[s * kMtN + i];
        words[i] = v;
    }
    if (tid < 8) cnt[tid >> 2][tid & 3] = 0;
    __syncthreads();
    const uint32_t Q = (T * D + kMtPair - 1) / kMtPair;
    if (tid < 256) {
        MtRun run(words);
        for (uint32_t q = 0, iq = 0; q < Q; ++q, ++iq) {
            if (iq == kMtLap) {
                iq = 0;
                run.at = words + tid;
                for (uint32_t i = tid; i < kMtN; i += 256) words[i] = words[kLapWords + i];
                lds_barrier();
            }
            if (iq == 0 && q % kMtCkEvery == 0) {
                uint32_t *ck = ck_words + ((size_t)c * n_ck + q / kMtCkEvery) * kMtN;
                for (uint32_t i = tid; i < kMtN; i += 256) ck[i] = words[i];
            }
            uint32_t w0, w1;
            run.pair(w0, w1);
            lds_barrier();
        }
    } else {
        const uint32_t i = tid - 256, wave = __builtin_amdgcn_readfirstlane(i >> 6);
        const uint32_t lo_mask = wave >= 2 ? ~0u : wave == 1 ? 0xffffu : 0u, hi_mask = wave == 3 ? 0xffffu : 0u;
        char *o = (char *)(out + (size_t)c * stride * D);
        auto put = [&](uint32_t at, const float (&v)[3]) {
            if (D == 2) {
                *(float2 *)(o + at * 8u) = make_float2(v[0], v[1]);
            } else {
                float *p = (float *)(o + at * 12u);
                p[0] = v[0];
                p[1] = v[1];
                p[2] = v[2];
            }
        };
        const uint32_t J = (Q + 1) / 2;
        uint32_t total = 0, rank = 0, ck = 0, ck_at = 1;   // the j that settles checkpoint ck's interval
        unsigned long long k0 = 0, k1 = 0;                 // the wavefront's kept tries, first and second of each thread
        float v0[3] = {0.f, 0.f, 0.f}, v1[3] = {0.f, 0.f, 0.f};
        for (uint32_t j = 0, ij = 0; j <= J; ++j, ++ij) {
            if (ij == kMtLap / 2 && 2 * j < Q) {
                ij = 0;
                lds_barrier();
            }
            {   // slot 2 j: test the tries of intervals 2 j - 2 and 2 j - 1
                const uint32_t first = mt_first<D>(2 * j - 2), end = mt_first<D>(2 * j);
                const int n = j == 0 ? 0 : (int)((end < T ? end : T) - first) - 128 * (int)wave;
                auto lanes = [](int m) { return m >= 64 ? ~0ull : m <= 0 ? 0ull : (1ull << m) - 1ull; };
                const float r0 = D == 3 ? (v0[0] * v0[0] + v0[1] * v0[1]) + v0[2] * v0[2] : v0[0] * v0[0] + v0[1] * v0[1];
                const float r1 = D == 3 ? (v1[0] * v1[0] + v1[1] * v1[1]) + v1[2] * v1[2] : v1[0] * v1[0] + v1[1] * v1[1];
                k0 = __ballot(r0 < 1.f) & lanes((n + 1) >> 1);
                k1 = __ballot(r1 < 1.f) & lanes(n >> 1);
                rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(k0 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)k0, 0u));
                rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(k1 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)k1, rank));
                if ((i & 63) == 0) cnt[j & 1][wave] = (uint16_t)(__popcll(k0) + __popcll(k1));
                lds_barrier();
            }
            // slot 2 j + 1: write what was kept of them, read the next ones
            const uint32_t *k = (const uint32_t *)cnt[j & 1];
            uint32_t w[2 * D];
            mt_words<2 * D>(words + D * (mt_first<D>(2 * (ij < kMtLap / 2 ? ij : 0)) + 2 * i), w);
            const uint32_t lo = __builtin_amdgcn_readfirstlane(k[0]), hi = __builtin_amdgcn_readfirstlane(k[1]);
            const uint32_t before = (lo & lo_mask) + (hi & hi_mask), all = lo + hi;
            if (j == ck_at) {
                if (i == 0) ck_kept[(size_t)c * n_ck + ck] = total;
                ++ck;
                ck_at += kMtCkEvery / 2;
            }
            const uint32_t at = total + (before & 0xffffu) + (before >> 16) + rank;
            const bool ok0 = __builtin_amdgcn_inverse_ballot_w64(k0);
            if (ok0) put(at, v0);
            if (__builtin_amdgcn_inverse_ballot_w64(k1)) put(at + (ok0 ? 1u : 0u), v1);
            total += (all & 0xffffu) + (all >> 16);
            uint32_t a[D], b[D];
#pragma unroll
            for (int e = 0; e < D; ++e) {
                a[e] = w[e];
                b[e] = w[D + e];
            }
            mt_vector<D>(a, v0[0], v0[1], v0[2]);
            mt_vector<D>(b, v1[0], v1[1], v1[2]);
            lds_barrier();
        }
        if (i == 0) kept[c] = total;
    }
}

// One workgroup: prefix[c] = vectors kept before chunk c, prefix[n] the total.
__global__ __launch_bounds__(256) void k_mt_prefix(const uint32_t *__restrict__ kept, uint32_t n,
                                                   uint32_t *__restrict__ prefix)
{
    __shared__ uint32_t part[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t carry = 0;
    for (uint32_t c0 = 0; c0 < n; c0 += 256) {
        const uint32_t v = c0 + tid < n ? kept[c0 + tid] : 0u;
        uint32_t inc = v;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(inc, d, 64);
            if (lane >= (uint32_t)d) inc += o;
        }
        if (lane == 63) part[wave] = inc;
        __syncthreads();
        uint32_t at = carry + inc - v;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            const uint32_t k = part[w];
            if (w < wave) at += k;
            carry += k;
        }
        if (c0 + tid < n) prefix[c0 + tid] = at;
        __syncthreads();
    }
    if (tid == 0) prefix[n] = carry;
}

// The first kStreamRun vectors of chunk c + 1 behind chunk c's own, so that
// a reader's run of that many never leaves the region it starts in.
template <int D>
__global__ __launch_bounds__(128) void k_mt_join(const uint32_t *__restrict__ kept, uint32_t stride, float *__restrict__ out)
{
    const size_t c = blockIdx.x;
    float *dst = out + (c * stride + kept[c]) * D;
    const float *src = out + (c + 1) * stride * D;
    for (int i = threadIdx.x; i < kStreamRun * D; i += 128) dst[i] = src[i];
}

// The fill's first n vectors as one array.
template <int D>
__global__ __launch_bounds__(256) void k_mt_gather(StreamVectors sv, uint32_t n, float *__restrict__ out)
{
    const uint32_t j = blockIdx.x * 256 + threadIdx.x;
    if (j >= n) return;
    const float *v = stream_at<D>(sv, j);
#pragma unroll
    for (int e = 0; e < D; ++e) out[(size_t)j * D + e] = v[e];
}

// The stream moves past the try that kept the m-th vector (m >= 1, at most
// the total): the chunk and the checkpoint before it are found by every
// thread at once, its intervals run again to the try, and the context's array
// becomes the 624 words from the next draw on (idx 0).
template <int D>
__global__ __launch_bounds__(512) void k_mt_commit(MtState *__restrict__ st, const uint32_t *__restrict__ prefix, uint32_t n,
                                                   uint32_t T, uint32_t n_ck, const uint32_t *__restrict__ ck_words,
                                                   const uint32_t *__restrict__ ck_kept, uint32_t m)
{
    // a checkpoint's intervals, one more the loop may start, one for the window
    __shared__ __align__(8) uint32_t words[kMtN + (kMtCkEvery + 2) * kMtPair];
    __shared__ uint32_t cnt[2];
    __shared__ uint32_t s_c, s_k, s_t;
    const uint32_t tid = threadIdx.x;
    if (tid < 2) cnt[tid] = 0u;
    for (uint32_t c = tid; c < n; c += 512)
        if (prefix[c] < m && m <= prefix[c + 1]) s_c = c;
    __syncthreads();
    const uint32_t c = s_c, want = m - prefix[c];   // the want-th kept of chunk c
    const uint32_t *ck = ck_kept + (size_t)c * n_ck;
    for (uint32_t k = tid; k < n_ck; k += 512)
        if (ck[k] < want && (k + 1 == n_ck || want <= ck[k + 1])) s_k = k;
    __syncthreads();
    const uint32_t ck_k = s_k, before = ck[ck_k];
    for (uint32_t i = tid; i < kMtN; i += 512) words[i] = ck_words[((size_t)c * n_ck + ck_k) * kMtN + i];
    __syncthreads();
    const uint32_t first = mt_first<D>(ck_k * kMtCkEvery);   // the checkpoint's try
    const bool maker = tid < 256;
    const uint32_t i = tid & 255, wave = __builtin_amdgcn_readfirstlane(i >> 6);
    MtRun run(words);
    MtTry tried;
    uint32_t w0, w1, total = before;
    // The vector lies in the checkpoint's kMtCkEvery intervals; every thread
    // follows the counts and stops at the same one.
    for (uint32_t q = 0; q <= kMtCkEvery; ++q) {
        const uint32_t k = __builtin_amdgcn_readfirstlane(cnt[(q + 1) & 1]);
        if (!maker && tried.ok() && total + mt_before(k, wave) + tried.rank + 1 == want) s_t = mt_first<D>(q - 1) + i;
        total += mt_all(k);
        if (total >= want) break;
        if (maker) {
            run.pair(w0, w1);
        } else {
            const uint32_t a = mt_first<D>(q), b = mt_first<D>(q + 1), e = T - first;
            uint32_t w[D];
            mt_words<D>(words + D * (a + i), w);
            mt_vector<D>(w, tried.x, tried.y, tried.z);
            tried.test<D>(cnt[q & 1], wave, a < e ? (b < e ? b : e) - a : 0u);
        }
        lds_barrier();
    }
    // the window after a try at the end of its interval reaches into the
    // next pair's words
    if (maker) run.pair(w0, w1);
    __syncthreads();
    const uint32_t w = D * (s_t + 1);   // the next draw, in words past the checkpoint
    for (uint32_t j = tid; j < kMtN; j += 512) st->mt[j] = words[w + j];
    if (tid == 0) {
        st->idx = 0;
        st->draws += (unsigned long long)D * ((unsigned long long)c * T + first + s_t + 1ull);
    }
}

void launch_mt_base(const MtState *st, uint32_t n, uint32_t *base, hipStream_t s)
{
    hipLaunchKernelGGL(k_mt_base, dim3(1), dim3(256), 0, s, st, n, base);
}

void launch_mt_lists(const uint64_t *polys, int n, uint16_t *entries, uint32_t *start, hipStream_t s)
{
    if (n > 0) hipLaunchKernelGGL(k_mt_lists, dim3(n), dim3(320), 0, s, polys, entries, start);
}

void launch_mt_jump(const uint32_t *base, const uint16_t *entries, const uint32_t *start, int n_jumps, uint32_t *states,
                    hipStream_t s)
{
    if (n_jumps <= 0) return;
    hipLaunchKernelGGL(k_mt_jump, dim3(n_jumps, kJumpSegs), dim3(kJumpThreads), 0, s, base, entries, start, states);
}

uint32_t mt_checkpoints(uint32_t words) { return (words + kMtPair * kMtCkEvery - 1) / (kMtPair * kMtCkEvery); }

template <int D>
static void launch_mt_fill_t(const uint32_t *base, const uint32_t *states, const MtFill &f, hipStream_t s)
{
    hipLaunchKernelGGL(k_mt_fill<D>, dim3(f.chunks), dim3(kMtFillThreads<D>), 0, s, base, states, f.T, f.stride, f.n_ck, f.out, f.kept,
                       f.ck_words, f.ck_kept);
    hipLaunchKernelGGL(k_mt_prefix, dim3(1), dim3(256), 0, s, f.kept, f.chunks, f.prefix);
    if (f.chunks > 1) hipLaunchKernelGGL(k_mt_join<D>, dim3(f.chunks - 1), dim3(128), 0, s, f.kept, f.stride, f.out);
}

void launch_mt_fill(const uint32_t *base, const uint32_t *states, const MtFill &f, hipStream_t s)
{
    if (f.D == 3) launch_mt_fill_t<3>(base, states, f, s);
    else launch_mt_fill_t<2>(base, states, f, s);
}

void launch_mt_commit(MtState *st, const MtFill &f, uint32_t m, hipStream_t s)
{
    if (m == 0) return;
    if (f.D == 3)
        hipLaunchKernelGGL(k_mt_commit<3>, dim3(1), dim3(512), 0, s, st, f.prefix, f.chunks, f.T, f.n_ck, f.ck_words,
                           f.ck_kept, m);
    else
        hipLaunchKernelGGL(k_mt_commit<2>, dim3(1), dim3(512), 0, s, st, f.prefix, f.chunks, f.T, f.n_ck, f.ck_words,
                           f.ck_kept, m);
}

void launch_mt_gather(const MtFill &f, uint32_t n, float *out, hipStream_t s)
{
    if (n == 0) return;
    const unsigned b = (unsigned)(((size_t)n + 255) / 256);
    if (f.D == 3) hipLaunchKernelGGL(k_mt_gather<3>, dim3(b), dim3(256), 0, s, f.vectors(), n, out);
    else hipLaunchKernelGGL(k_mt_gather<2>, dim3(b), dim3(256), 0, s, f.vectors(), n, out);
}

}  // namespace fgl
