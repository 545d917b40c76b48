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

// Random(-1, 1) from one draw.
__device__ __forceinline__ float random_pm1(uint32_t u)
{
    float r = (float)u * 2.3283064365386963e-10f;   // 2^-32, exact scaling
    if (r >= 1.f) r = __uint_as_float(0x3f7fffffu);
    return -1.f + 2.f * r;
}

// The generator as one sequence: x_{n+624} = twist(x_n, x_{n+1}, x_{n+397})
// (a block's twist is this recurrence, new words used as they appear).  227
// consecutive words read only words at least 227 back, so a workgroup makes
// them together, a thread each -- and the next 227 as well before anyone has
// to wait: thread t's second word reads x_{j+227} and x_{j+228}, at least 396
// back, and its own first word.  So a pair of steps, 454 words, takes one
// barrier.  The last 2048 words are kept in an LDS ring (word n in slot n %
// 2048).
//
// The barrier orders LDS alone: a __syncthreads() also waits for the
// interval's global stores, which made a step of 227 words 860 cycles.
constexpr uint32_t kMtRing = 2048, kMtLag = kMtN - kMtM, kMtPair = 2 * kMtLag;

__device__ __forceinline__ void mt_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A running generator: the ring holds x_0 .. x_{623 + made}.  The first 227
// threads make words; `far` is x_{made + 397 + t}, the thread's own last one.
struct MtRun {
    uint32_t *ring;
    uint32_t made, far;
    __device__ __forceinline__ explicit MtRun(uint32_t *r) : ring(r), made(0), far(0)
    {
        if (threadIdx.x < kMtLag) far = ring[threadIdx.x + kMtM];
    }
    // 454 more words (w0, w1: this thread's), ready after the next barrier.
    __device__ __forceinline__ void pair(uint32_t &w0, uint32_t &w1)
    {
        constexpr uint32_t R = kMtRing - 1;
        if (threadIdx.x < kMtLag) {
            const uint32_t j = made + threadIdx.x;
            const uint32_t c0 = ring[j & R], n0 = ring[(j + 1) & R];
            const uint32_t c1 = ring[(j + kMtLag) & R], n1 = ring[(j + kMtLag + 1) & R];
            w0 = mt_twist_word(c0, n0, far);
            w1 = mt_twist_word(c1, n1, w0);
            ring[(j + kMtN) & R] = w0;
            ring[(j + kMtN + kMtLag) & R] = w1;
            far = w1;
        }
        made += kMtPair;
    }
};

// The try of D draws at word p of the sequence in the ring: the vector (x, y,
// z) and whether it is kept.
template <int D>
__device__ __forceinline__ bool mt_try(const uint32_t *ring, uint32_t p, float &x, float &y, float &z)
{
    constexpr uint32_t R = kMtRing - 1;
    float r[D];
#pragma unroll
    for (int e = 0; e < D; ++e) r[e] = random_pm1(mt_temper(ring[(p + e) & R]));
    z = D == 3 ? r[0] : 0.f;
    y = r[D - 2];
    x = r[D - 1];
    return (x * x + y * y) + z * z < 1.f;
}

// ---- the stream in parallel: jump ahead, generate, keep ----
//
// A fill takes the stream's next draws in chunks of L = 624 K draws, L a
// multiple of D, so that no try crosses chunks.  The base sequence x_0, x_1 ..
// starts at the context's next draw; chunk c starts from the 624 words c L
// words into it, which the jump gives (mt_jump.hpp): the XOR of the windows
// x_i .. x_{i+623} over the set bits i of t^(c L) mod phi.  A chunk makes its
// words in an LDS ring, tests its tries there and writes the kept vectors
// only; its draws never reach memory.  Checkpoints -- the generator's words
// and the vectors kept so far, every kMtCkEvery intervals -- let a commit find
// the try that kept the m-th vector without the draws.  Every window of a
// jump, x_{19967 + 623} at most, lies in the base sequence.
static_assert(kMtBaseWords >= 64 * kMtPolyWords + 623, "the jump's windows stay in the base sequence");

// One workgroup: the base sequence's first n words, untempered.
__global__ __launch_bounds__(256) void k_mt_base(const MtState *__restrict__ st, uint32_t n, uint32_t *__restrict__ base)
{
    __shared__ uint32_t ring[kMtRing];
    const uint32_t tid = threadIdx.x, idx = st->idx;
    for (uint32_t i = tid; i < kMtN; i += 256) {
        const uint32_t v = st->mt[i];
        ring[i] = v;
        if (i >= idx && i - idx < n) base[i - idx] = v;
    }
    __syncthreads();
    MtRun run(ring);
    for (uint32_t at = kMtN - idx; at < n; at += kMtPair) {
        uint32_t w0, w1;
        run.pair(w0, w1);
        if (tid < kMtLag) {
            if (at + tid < n) base[at + tid] = w0;
            if (at + kMtLag + tid < n) base[at + kMtLag + tid] = w1;
        }
        mt_barrier();
    }
}

// Workgroup c - 1 jumps to chunk c's array: states[c][k] = XOR of base[i + k]
// over the set bits i of polynomial c, the base sequence in LDS.  The set
// bits are split by i mod 4: for the bits i = 4 q + r, thread t gathers the
// 16-byte group base[4 (q + t) .. 4 (q + t) + 3], words k + r of the result
// for k + r in [4 t, 4 t + 4), so each bit costs a thread one 16-byte LDS
// read; three wavefronts per class, so each class's chain of dependent LDS
// reads runs beside the others; the four partial arrays are combined at the
// end (word k = XOR over r of partial r at k + r).  Each class's q values are listed in LDS (per-word
// counts scanned by one wavefront per class), padded to a multiple of eight
// with a q whose groups are zero, so every wavefront reads eight q values
// with one broadcast load.
constexpr int kJumpGroups = ((int)kMtN + 3 + 3) / 4;                       // 157: k + r < 627
constexpr int kJumpClassThreads = 192;                                     // three wavefronts per class
constexpr int kJumpThreads = 4 * kJumpClassThreads;
static_assert(kJumpGroups <= kJumpClassThreads, "a thread per 16-byte group of a class");
constexpr int kJumpZeroQ = kMtBaseWords / 4;                               // groups past the base: zero
constexpr int kJumpLdsWords = kMtBaseWords + 4 * kJumpGroups;              // base, then the zero groups
constexpr int kJumpListMax = kMtPolyWords * 64 + 4 * 7 + 8;                // every bit, padding, one read ahead
static_assert(kMtBaseWords % 4 == 0 && kJumpZeroQ < 65536, "16-bit q values; aligned zero groups");
static_assert(4 * (kMtDegree / 4 + kJumpGroups - 1) + 3 < kMtBaseWords, "the groups a bit reads lie in the base");

__global__ __launch_bounds__(kJumpThreads) void k_mt_jump(const uint32_t *__restrict__ base, const uint64_t *__restrict__ polys,
                                                 uint32_t *__restrict__ states)
{
    __shared__ __align__(16) uint32_t b[kJumpLdsWords];
    __shared__ __align__(16) uint16_t qs[kJumpListMax];
    __shared__ uint32_t off[4][kMtPolyWords];
    __shared__ uint32_t ncls[4], cls[5];                // class sizes; starts (multiples of 8), cls[4] = the end
    __shared__ uint32_t part[4][4 * kJumpGroups];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = blockIdx.x + 1;
    const uint64_t *g = polys + (size_t)(c - 1) * kMtPolyWords;
    constexpr uint64_t kRes = 0x1111111111111111ull;   // bits i with i mod 4 = 0
    for (int i = tid; i < kMtBaseWords / 4; i += kJumpThreads) ((uint4 *)b)[i] = ((const uint4 *)base)[i];
    for (int i = tid; i < kJumpGroups; i += kJumpThreads) ((uint4 *)b)[kJumpZeroQ + i] = make_uint4(0u, 0u, 0u, 0u);
    for (int w = tid; w < kMtPolyWords; w += kJumpThreads) {
        const uint64_t v = g[w];
#pragma unroll
        for (int r = 0; r < 4; ++r) off[r][w] = (uint32_t)__popcll(v & (kRes << r));
    }
    __syncthreads();
    if (wave < 4) {
        // wavefront r: exclusive scan of class r's 312 counts, 5 words a lane
        constexpr int kPer = (kMtPolyWords + 63) / 64;
        const int r = wave;
        uint32_t v[kPer], sum = 0;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            const int q = lane * kPer + e;
            v[e] = q < kMtPolyWords ? off[r][q] : 0u;
            sum += v[e];
        }
        uint32_t incl = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d);
            if (lane >= d) incl += o;
        }
        uint32_t run = incl - sum;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            const int q = lane * kPer + e;
            if (q < kMtPolyWords) off[r][q] = run;
            run += v[e];
        }
        if (lane == 63) ncls[r] = incl;
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t at = 0;
        for (int r = 0; r < 4; ++r) {
            cls[r] = at;
            at += (ncls[r] + 7u) & ~7u;
        }
        cls[4] = at;
    }
    __syncthreads();
    for (int w = tid; w < kMtPolyWords; w += kJumpThreads) {
        const uint64_t v = g[w];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            uint32_t pos = cls[r] + off[r][w];
            uint64_t bits = v & (kRes << r);
            while (bits) {
                qs[pos++] = (uint16_t)((w * 64 + __builtin_ctzll(bits)) >> 2);
                bits &= bits - 1;
            }
        }
    }
    if (tid < 4)   // pad class tid to its rounded length with the zero groups
        for (uint32_t e = cls[tid] + ncls[tid]; e < cls[tid + 1]; ++e) qs[e] = (uint16_t)kJumpZeroQ;
    __syncthreads();
    const int r = tid / kJumpClassThreads, t = tid - r * kJumpClassThreads;
    if (t < kJumpGroups) {
        const uint4 *b4 = (const uint4 *)b + t;
        {
            uint4 acc = make_uint4(0u, 0u, 0u, 0u);
            const uint4 *q8 = (const uint4 *)(qs + cls[r]);
            const uint32_t n8 = (cls[r + 1] - cls[r]) / 8;
            uint4 v = q8[0];
            for (uint32_t e = 0; e < n8; ++e) {
                const uint4 next = q8[e + 1];   // read ahead (past the class: unused)
                const uint4 a0 = b4[v.x & 0xffffu], a1 = b4[v.x >> 16];
                const uint4 a2 = b4[v.y & 0xffffu], a3 = b4[v.y >> 16];
                const uint4 a4 = b4[v.z & 0xffffu], a5 = b4[v.z >> 16];
                const uint4 a6 = b4[v.w & 0xffffu], a7 = b4[v.w >> 16];
                acc.x ^= ((a0.x ^ a1.x) ^ (a2.x ^ a3.x)) ^ ((a4.x ^ a5.x) ^ (a6.x ^ a7.x));
                acc.y ^= ((a0.y ^ a1.y) ^ (a2.y ^ a3.y)) ^ ((a4.y ^ a5.y) ^ (a6.y ^ a7.y));
                acc.z ^= ((a0.z ^ a1.z) ^ (a2.z ^ a3.z)) ^ ((a4.z ^ a5.z) ^ (a6.z ^ a7.z));
                acc.w ^= ((a0.w ^ a1.w) ^ (a2.w ^ a3.w)) ^ ((a4.w ^ a5.w) ^ (a6.w ^ a7.w));
                v = next;
            }
            ((uint4 *)part[r])[t] = acc;
        }
    }
    __syncthreads();
    for (int k = tid; k < (int)kMtN; k += kJumpThreads)
        states[(size_t)c * kMtN + k] = part[0][k] ^ part[1][k + 1] ^ part[2][k + 2] ^ part[3][k + 3];
}

// The tries of interval q (the words of one pair): [mt_first(q), mt_first(q +
// 1)), at most 227, all of whose words the ring holds when the interval
// starts.
template <int D>
__device__ __forceinline__ uint32_t mt_first(uint32_t q) { return q * kMtPair / (uint32_t)D; }

// Half a workgroup's tries over the generator's intervals: in an interval a
// thread tests one try of it and writes the vector it kept in the one
// before, whose wavefronts' counts the barrier between has published.
template <int D>
struct MtTries {
    uint32_t total;       // kept before the interval being tested
    uint32_t rank;        // this thread's vector among its wavefront's
    bool ok;
    float x, y, z;
    __device__ __forceinline__ MtTries() : total(0), rank(0), ok(false), x(0.f), y(0.f), z(0.f) {}
    // The interval before, counted: where this thread's vector goes (valid
    // when ok).
    __device__ __forceinline__ uint32_t settle(const uint32_t *cnt, uint32_t wave)
    {
        uint32_t at = total + rank;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            const uint32_t k = cnt[w];
            if (w < wave) at += k;
            total += k;
        }
        return at;
    }
    __device__ __forceinline__ void test(const uint32_t *ring, uint32_t *cnt, uint32_t q, uint32_t T, uint32_t i)
    {
        const uint32_t t = mt_first<D>(q) + i, end = mt_first<D>(q + 1);
        ok = mt_try<D>(ring, D * t, x, y, z) && t < end && t < T;
        const unsigned long long m = __ballot(ok);
        rank = (uint32_t)__popcll(m & ((1ull << (i & 63)) - 1));
        if ((i & 63) == 0) cnt[i >> 6] = (uint32_t)__popcll(m);
    }
};

// Workgroup c runs chunk c, T tries: four wavefronts make words, four test
// tries and write the kept vectors.  An interval is bound by either half's
// chain (LDS reads, some 60 operations, barrier); written as tempered draws,
// counted, scanned and read back by two more kernels, 187 M draws (D = 3) took
// 890 us.
constexpr uint32_t kMtCkEvery = 33;   // intervals between checkpoints, a multiple of 3: whole tries

template <int D>
__global__ __launch_bounds__(512) void k_mt_fill(const uint32_t *__restrict__ base, const uint32_t *__restrict__ states,
                                                 uint32_t T, uint32_t stride, uint32_t n_ck, float *__restrict__ out,
                                                 uint32_t *__restrict__ kept, uint32_t *__restrict__ ck_words,
                                                 uint32_t *__restrict__ ck_kept)
{
    constexpr uint32_t R = kMtRing - 1;
    __shared__ uint32_t ring[kMtRing];
    __shared__ uint32_t cnt[2][4];
    const uint32_t tid = threadIdx.x, c = blockIdx.x;
    const uint32_t *src = c == 0 ? base : states + (size_t)c * kMtN;
    for (uint32_t i = tid; i < kMtN; i += 512) ring[i] = src[i];
    if (tid < 8) cnt[tid >> 2][tid & 3] = 0u;
    __syncthreads();
    const uint32_t Q = (T * D + kMtPair - 1) / kMtPair;
    if (tid < 256) {
        MtRun run(ring);
        for (uint32_t q = 0; q < Q; ++q) {
            uint32_t w0, w1;
            if (q % kMtCkEvery == 0) {
                const size_t k = (size_t)c * n_ck + q / kMtCkEvery;
                for (uint32_t i = tid; i < kMtN; i += 256) ck_words[k * kMtN + i] = ring[(kMtPair * q + i) & R];
            }
            run.pair(w0, w1);
            mt_barrier();
        }
    } else {
        const uint32_t i = tid - 256, wave = i >> 6;
        float *o = out + (size_t)c * stride * D;
        MtTries<D> tries;
        auto write = [&](uint32_t q) {
            const uint32_t at = tries.settle(cnt[(q + 1) & 1], wave);
            if (!tries.ok) return;
            float *v = o + (size_t)at * D;
            if (D == 2) {
                *(float2 *)v = make_float2(tries.x, tries.y);
            } else {
                v[0] = tries.x;
                v[1] = tries.y;
                v[2] = tries.z;
            }
        };
        for (uint32_t q = 0; q < Q; ++q) {
            write(q);
            if (q % kMtCkEvery == 0 && i == 0) ck_kept[(size_t)c * n_ck + q / kMtCkEvery] = tries.total;
            tries.test(ring, cnt[q & 1], q, T, i);
            mt_barrier();
        }
        write(Q);
        if (i == 0) kept[c] = tries.total;
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
    constexpr uint32_t R = kMtRing - 1;
    __shared__ uint32_t ring[kMtRing];
    __shared__ uint32_t cnt[2][4];
    __shared__ uint32_t s_c, s_k, s_t;
    const uint32_t tid = threadIdx.x;
    if (tid < 8) cnt[tid >> 2][tid & 3] = 0u;
    for (uint32_t c = tid; c < n; c += 512)
        if (prefix[c] < m && m <= prefix[c + 1]) s_c = c;
    __syncthreads();
    const uint32_t c = s_c, want = m - prefix[c];   // the want-th kept of chunk c
    const uint32_t *ck = ck_kept + (size_t)c * n_ck;
    for (uint32_t k = tid; k < n_ck; k += 512)
        if (ck[k] < want && (k + 1 == n_ck || want <= ck[k + 1])) s_k = k;
    __syncthreads();
    const uint32_t k = s_k;
    for (uint32_t i = tid; i < kMtN; i += 512) ring[i] = ck_words[((size_t)c * n_ck + k) * kMtN + i];
    __syncthreads();
    const uint32_t first = mt_first<D>(k * kMtCkEvery);   // the checkpoint's try
    const bool maker = tid < 256;
    const uint32_t i = tid & 255, wave = i >> 6;
    MtRun run(ring);
    MtTries<D> tries;
    uint32_t w0, w1;
    // The vector lies in the checkpoint's kMtCkEvery intervals; every thread
    // follows the counts and stops at the same one.
    for (uint32_t q = 0; q <= kMtCkEvery; ++q) {
        const uint32_t at = tries.settle(cnt[(q + 1) & 1], wave);
        if (!maker && tries.ok && at + 1 + ck[k] == want) s_t = mt_first<D>(q - 1) + i;
        if (tries.total + ck[k] >= want) break;
        if (maker) run.pair(w0, w1);
        else tries.test(ring, cnt[q & 1], q, T - first, i);
        mt_barrier();
    }
    // the window after a try at the end of its interval reaches into the
    // next pair's words
    if (maker) run.pair(w0, w1);
    __syncthreads();
    const uint32_t w = D * (s_t + 1);   // the next draw, in words past the checkpoint
    for (uint32_t j = tid; j < kMtN; j += 512) st->mt[j] = ring[(w + j) & R];
    if (tid == 0) {
        st->idx = 0;
        st->draws += (unsigned long long)D * ((unsigned long long)c * T + first + s_t + 1ull);
    }
}

void launch_mt_base(const MtState *st, uint32_t n, uint32_t *base, hipStream_t s)
{
    hipLaunchKernelGGL(k_mt_base, dim3(1), dim3(256), 0, s, st, n, base);
}

void launch_mt_jump(const uint32_t *base, const uint64_t *polys, int n_jumps, uint32_t *states, hipStream_t s)
{
    if (n_jumps <= 0) return;
    hipLaunchKernelGGL(k_mt_jump, dim3(n_jumps), dim3(kJumpThreads), 0, s, base, polys, states);
}

uint32_t mt_checkpoints(uint32_t words) { return (words + kMtPair * kMtCkEvery - 1) / (kMtPair * kMtCkEvery); }

template <int D>
static void launch_mt_fill_t(const uint32_t *base, const uint32_t *states, const MtFill &f, hipStream_t s)
{
    hipLaunchKernelGGL(k_mt_fill<D>, dim3(f.chunks), dim3(512), 0, s, base, states, f.T, f.stride, f.n_ck, f.out, f.kept,
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
