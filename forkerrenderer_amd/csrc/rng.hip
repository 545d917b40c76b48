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
// (a block's twist is this recurrence, new words used as they appear).  The
// 227 words x_n .. x_{n+226} read only words at least 227 back, so a
// workgroup makes them together, one barrier per step, keeping the last 2048
// words in an LDS ring (word n in slot n % 2048).  In step s thread t makes
// x_{624+j}, j = 227 s + t, from x_j and x_{j+1} (made two steps back or
// earlier, so read during the step before, while it computes) and x_{j+397}
// (the word the thread made in the step before).
//
// The barrier orders LDS alone: a __syncthreads() also waits for the step's
// global stores, which made a step 860 cycles.
constexpr uint32_t kMtRing = 2048, kMtLag = kMtN - kMtM;

__device__ __forceinline__ void mt_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A running generator: the ring holds x_0 .. x_{623 + made}.  Needs at least
// 227 threads; every thread of the workgroup calls it.
struct MtRun {
    uint32_t *ring;
    uint32_t made, cur, nxt, far;
    __device__ __forceinline__ explicit MtRun(uint32_t *r) : ring(r), made(0), cur(0), nxt(0), far(0)
    {
        if (threadIdx.x < kMtLag) {
            cur = ring[threadIdx.x];
            nxt = ring[threadIdx.x + 1];
            far = ring[threadIdx.x + kMtM];
        }
    }
    // 227 more words; this thread's (the first 227 threads) is returned.
    __device__ __forceinline__ uint32_t step()
    {
        constexpr uint32_t R = kMtRing - 1;
        uint32_t v = 0;
        if (threadIdx.x < kMtLag) {
            const uint32_t j = made + threadIdx.x;
            const uint32_t ncur = ring[(j + kMtLag) & R], nnxt = ring[(j + kMtLag + 1) & R];
            v = mt_twist_word(cur, nxt, far);
            ring[(j + kMtN) & R] = v;
            cur = ncur;
            nxt = nnxt;
            far = v;
        }
        made += kMtLag;
        mt_barrier();
        return v;
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
// and the vectors kept so far, every kMtCkRounds rounds -- let a commit find
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
    for (uint32_t at = kMtN - idx; at < n; at += kMtLag) {
        const uint32_t v = run.step();
        if (tid < kMtLag && at + tid < n) base[at + tid] = v;
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

// Workgroup c runs chunk c: rounds of D steps, 227 tries a round (a thread
// each), T tries in all.  A round's tries are read, tempered and tested in
// the interval before its last steps' barrier and written after it, when
// every wavefront's count is known.  The step is bound by its LDS latency and
// barrier; written as tempered draws, counted, scanned and read back by two
// more kernels, the same fill took 1,390 us for 187 M draws (D = 3).
constexpr uint32_t kMtCkRounds = 32;

template <int D>
__global__ __launch_bounds__(256) void k_mt_fill(const uint32_t *__restrict__ base, const uint32_t *__restrict__ states,
                                                 uint32_t T, uint32_t stride, uint32_t n_ck, float *__restrict__ out,
                                                 uint32_t *__restrict__ kept, uint32_t *__restrict__ ck_words,
                                                 uint32_t *__restrict__ ck_kept)
{
    constexpr uint32_t R = kMtRing - 1;
    __shared__ uint32_t ring[kMtRing];
    __shared__ uint32_t cnt[4];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = blockIdx.x;
    const uint32_t *src = c == 0 ? base : states + (size_t)c * kMtN;
    for (uint32_t i = tid; i < kMtN; i += 256) ring[i] = src[i];
    __syncthreads();
    MtRun run(ring);
    float *o = out + (size_t)c * stride * D;
    uint32_t total = 0;
    for (uint32_t t0 = 0, r = 0; t0 < T; t0 += kMtLag, ++r) {
        if (r % kMtCkRounds == 0) {
            const size_t k = (size_t)c * n_ck + r / kMtCkRounds;
            for (uint32_t i = tid; i < kMtN; i += 256) ck_words[k * kMtN + i] = ring[(D * t0 + i) & R];
            if (tid == 0) ck_kept[k] = total;
        }
        run.step();
        float x, y, z;
        const bool ok = mt_try<D>(ring, D * (t0 + tid), x, y, z) && tid < kMtLag && t0 + tid < T;
        const unsigned long long m = __ballot(ok);
        if (lane == 0) cnt[wave] = (uint32_t)__popcll(m);
        run.step();
        uint32_t at = total + (uint32_t)__popcll(m & ((1ull << lane) - 1));
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            const uint32_t k = cnt[w];
            if (w < wave) at += k;
            total += k;
        }
        if (ok) {
            float *v = o + (size_t)at * D;
            if (D == 2) {
                *(float2 *)v = make_float2(x, y);
            } else {
                v[0] = x;
                v[1] = y;
                v[2] = z;
            }
        }
        if (D == 3) run.step();
    }
    if (tid == 0) kept[c] = total;
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
// thread at once, its rounds run again to the try, and the context's array
// becomes the 624 words from the next draw on (idx 0).
template <int D>
__global__ __launch_bounds__(256) void k_mt_commit(MtState *__restrict__ st, const uint32_t *__restrict__ prefix, uint32_t n,
                                                   uint32_t T, uint32_t n_ck, const uint32_t *__restrict__ ck_words,
                                                   const uint32_t *__restrict__ ck_kept, uint32_t m)
{
    constexpr uint32_t R = kMtRing - 1;
    __shared__ uint32_t ring[kMtRing];
    __shared__ uint32_t cnt[4];
    __shared__ uint32_t s_c, s_k, s_t;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (uint32_t c = tid; c < n; c += 256)
        if (prefix[c] < m && m <= prefix[c + 1]) s_c = c;
    __syncthreads();
    const uint32_t c = s_c, want = m - prefix[c];   // the want-th kept of chunk c
    const uint32_t *ck = ck_kept + (size_t)c * n_ck;
    for (uint32_t k = tid; k < n_ck; k += 256)
        if (ck[k] < want && (k + 1 == n_ck || want <= ck[k + 1])) s_k = k;
    __syncthreads();
    const uint32_t k = s_k;
    for (uint32_t i = tid; i < kMtN; i += 256) ring[i] = ck_words[((size_t)c * n_ck + k) * kMtN + i];
    __syncthreads();
    MtRun run(ring);
    uint32_t total = ck[k], t0 = 0;
    const uint32_t first = k * kMtCkRounds * kMtLag;   // the checkpoint's try
    for (; first + t0 < T; t0 += kMtLag) {
        run.step();
        float x, y, z;
        const bool ok = mt_try<D>(ring, D * (t0 + tid), x, y, z) && tid < kMtLag && first + t0 + tid < T;
        const unsigned long long b = __ballot(ok);
        if (lane == 0) cnt[wave] = (uint32_t)__popcll(b);
        run.step();
        uint32_t at = total + (uint32_t)__popcll(b & ((1ull << lane) - 1));
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            const uint32_t q = cnt[w];
            if (w < wave) at += q;
            total += q;
        }
        if (ok && at + 1 == want) s_t = t0 + tid;
        if (D == 3) run.step();
        if (total >= want) break;
    }
    __syncthreads();
    const uint32_t w = D * (s_t + 1);   // the next draw, in words past the checkpoint
    for (uint32_t i = tid; i < kMtN; i += 256) st->mt[i] = ring[(w + i) & R];
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

uint32_t mt_checkpoints(uint32_t T) { return (T + kMtLag * kMtCkRounds - 1) / (kMtLag * kMtCkRounds); }

template <int D>
static void launch_mt_fill_t(const uint32_t *base, const uint32_t *states, const MtFill &f, hipStream_t s)
{
    hipLaunchKernelGGL(k_mt_fill<D>, dim3(f.chunks), dim3(256), 0, s, base, states, f.T, f.stride, f.n_ck, f.out, f.kept,
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
        hipLaunchKernelGGL(k_mt_commit<3>, dim3(1), dim3(256), 0, s, st, f.prefix, f.chunks, f.T, f.n_ck, f.ck_words,
                           f.ck_kept, m);
    else
        hipLaunchKernelGGL(k_mt_commit<2>, dim3(1), dim3(256), 0, s, st, f.prefix, f.chunks, f.T, f.n_ck, f.ck_words,
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
