// shade.hip -- screen-space passes for gfx950: deferred lighting, kernel SSAO,
// AO blurs and the quantise + SSAA resolve.  All read/write SoA float planes
// in HBM with 64-wide rows per wavefront.
#include "shade_core.hpp"

#include <cmath>

namespace fgl {

template <bool STREAM, int MODE>
__global__ __launch_bounds__(256) void k_lighting(FrameUniforms u, const float *__restrict__ g,
                                                  const float *__restrict__ ao, int ao_is_one, NetAo net,
                                                  const float *__restrict__ smap, ShadowSamples ss,
                                                  float *__restrict__ fb)
{
    int x, y;
    grid_px<16>(x, y);
    if (x >= u.W || y >= u.H) return;
    lighting_px<STREAM, MODE>(u, g, ao, ao_is_one, smap, ss, fb, x, y, net);
}

__global__ __launch_bounds__(256) void k_ssao_ref(FrameUniforms u, StreamVectors samples,
                                                  const float *__restrict__ pow3,
                                                  const float *__restrict__ depth,
                                                  const float *__restrict__ g, float *__restrict__ ao)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= u.W || y >= u.H) return;
    ssao_ref_px(u, samples, pow3, depth, g, ao, x, y);
}

// ---- PCSS sample offsets for the stochastic filter (FGL_SHADOW_REF_PCSS) ----
//
// The lighting pass visits pixels in row order (the forward pass its passing
// fragments in raster order) and each shading point draws n_blocker
// unit-disk samples, plus n_pcf more when its blocker search finds a blocker
// (PCSS, shadow.cpp:93-106), so a point's offset into the stream depends on
// the outcome of every search before it.  Most searches are decided by the
// shadow map alone: k_pcss_classify checks every texel a sample of the point
// could reach (the square around the disk) and marks the point "no blocker
// for any sample set", "a blocker for any sample set" or "depends on the
// samples".  Only the last kind is walked in order (k_pcss_points,
// k_pcss_guess, k_pcss_band, k_pcss_walk_blocks, k_pcss_chain below), at
// offsets that count the decided points before it.  The points' inputs are planes of stride P:
// normal, world position, light NDC.

// Light 0's shadow coordinate and bias at point i, as shade_point computes them.
__device__ __forceinline__ void pcss_pixel(const FrameUniforms &u, const float *__restrict__ g, size_t P, size_t i,
                                           Vec3 &sc, float &bias)
{
    const Vec3 N = vec3(g[i], g[P + i], g[2 * P + i]);
    const Vec3 Pw = vec3(g[3 * P + i], g[4 * P + i], g[5 * P + i]);
    const Vec3 lndc = vec3(g[6 * P + i], g[7 * P + i], g[8 * P + i]);
    sc = shadow_coord(lndc);
    bias = shadow_bias(N, light_dir(u.lights[0], Pw));
}

// The texel's depth as the blocker search sees it.
__device__ __forceinline__ float pcss_texel(float d) { return ((double)d < 0.001) ? 1.f : d; }

// mm[x + y SW] = (least, largest) pcss_texel over the bx x by texels from (x,
// y) on, a NaN counting as +infinity in both; written where those lie in the
// map.  A workgroup makes 64 x 32 of them from LDS: bx texels of a row, then
// by rows of the results.
constexpr int kMmW = 64, kMmH = 32, kMmMax = 16;
__global__ __launch_bounds__(256) void k_pcss_minmax(const float *__restrict__ smap, int SW, int SH, int bx, int by,
                                                     float2 *__restrict__ mm)
{
    __shared__ float t[(kMmH + kMmMax) * (kMmW + kMmMax)];
    __shared__ float2 row[(kMmH + kMmMax) * kMmW];
    const int x0 = blockIdx.x * kMmW, y0 = blockIdx.y * kMmH, w = kMmW + bx - 1, h = kMmH + by - 1;
    for (int k = threadIdx.x; k < w * h; k += 256) {
        const int x = x0 + k % w, y = y0 + k / w;
        float s = __builtin_inff();
        if (x < SW && y < SH) {
            s = pcss_texel(smap[(size_t)x + (size_t)y * SW]);
            if (!(s == s)) s = __builtin_inff();
        }
        t[k] = s;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kMmW * h; k += 256) {
        const float *p = t + (k / kMmW) * w + k % kMmW;
        float lo = p[0], hi = p[0];
        for (int e = 1; e < bx; ++e) {
            lo = fminf(lo, p[e]);
            hi = fmaxf(hi, p[e]);
        }
        row[k] = make_float2(lo, hi);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kMmW * kMmH; k += 256) {
        const int x = x0 + k % kMmW, y = y0 + k / kMmW;
        if (x + bx > SW || y + by > SH) continue;
        float2 m = row[k];
        for (int e = 1; e < by; ++e) {
            const float2 n = row[k + e * kMmW];
            m.x = fminf(m.x, n.x);
            m.y = fmaxf(m.y, n.y);
        }
        mm[(size_t)x + (size_t)y * SW] = m;
    }
}

// cnt[i] = n_blocker + n_pcf for "a blocker for any sample set", n_blocker
// otherwise; unc[i] = 1 for "depends on the samples".  Nothing is drawn with
// shadows off or without a light.  Whether any or every texel of the square
// blocks is whether its least or largest depth does (float addition is
// monotone), so with mm (k_pcss_minmax; may be null) squares that hold a bx x
// by window are covered by windows: a 14 x 9 square at 1280 x 800 takes 4 reads
// instead of 126 (220 -> 16 us, and 15 for the windows).
__global__ __launch_bounds__(256) void k_pcss_classify(FrameUniforms u, const float *__restrict__ g, size_t P,
                                                       const float *__restrict__ smap, const float2 *__restrict__ mm,
                                                       int bx, int by, uint32_t *__restrict__ cnt,
                                                       uint32_t *__restrict__ unc)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P) return;
    const DevShadowCfg &c = u.shadow;
    if (!(u.shadow_on && u.n_lights > 0)) {
        cnt[i] = 0;
        unc[i] = 0;
        return;
    }
    Vec3 sc;
    float bias;
    pcss_pixel(u, g, P, i, sc, bias);
    // every sample coordinate lies in [sc - F, sc + F], F = (float)blocker_filter
    // (|(float)(d * filter)| <= (float)filter for |d| < 1; float add and the
    // texel index are monotone)
    const float F = (float)c.blocker_filter;
    const float u0 = sc.x + (-F), u1 = sc.x + F, v0 = sc.y + (-F), v1 = sc.y + F;
    int cls = 2;
    if (u0 == u0 && u1 == u1 && v0 == v0 && v1 == v1 && sc.z == sc.z && bias == bias) {
        const bool inside = u0 >= 0.f && u1 <= 1.f && v0 >= 0.f && v1 <= 1.f;
        bool any_blk = false, any_clear = !inside;   // samples off the map never block
        if (u1 >= 0.f && u0 <= 1.f && v1 >= 0.f && v0 <= 1.f) {
            const int w = (int)((float)u.SW - 0.001f), h = (int)((float)u.SH - 0.001f);
            const int x0 = (int)((float)w * (u0 < 0.f ? 0.f : u0)), x1 = (int)((float)w * (u1 > 1.f ? 1.f : u1));
            const int y0 = (int)((float)h * (v0 < 0.f ? 0.f : v0)), y1 = (int)((float)h * (v1 > 1.f ? 1.f : v1));
            // a depth s: blocks or not; a blocker depth within reach of 0.001
            // could average below it: not decided
            auto take = [&](float lo, float hi) {
                const bool blk = sc.z > lo + bias;
                any_blk |= blk;
                any_clear |= !(sc.z > hi + bias) || (blk && !((double)lo > 0.0011));
            };
            if (mm && x1 - x0 + 1 >= bx && y1 - y0 + 1 >= by) {
                const int xe = x1 - bx + 1, ye = y1 - by + 1;   // the last window ends the square
                for (int y = y0;; y = imin(y + by, ye)) {
                    for (int x = x0;; x = imin(x + bx, xe)) {
                        const float2 m = mm[(size_t)x + (size_t)y * u.SW];
                        take(m.x, m.y);
                        if (x == xe) break;
                    }
                    if (y == ye || (any_blk && any_clear)) break;
                }
            } else {
                for (int y = y0; y <= y1 && !(any_blk && any_clear); ++y)
                    for (int x = x0; x <= x1; ++x) {
                        const float s = pcss_texel(smap[(size_t)x + (size_t)y * u.SW]);
                        take(s, s);
                    }
            }
        }
        if (!any_blk) cls = 0;
        else if (!any_clear) cls = 1;
    }
    cnt[i] = (uint32_t)c.n_blocker + (cls == 1 ? (uint32_t)c.n_pcf : 0u);
    unc[i] = cls == 2 ? 1u : 0u;
}

// list[upos[i]] = i for the undecided pixels (upos = exclusive scan of the
// undecided flags, total at upos[P]; a flag is upos[i + 1] - upos[i]).
__global__ __launch_bounds__(256) void k_pcss_compact(const uint32_t *__restrict__ upos, size_t P,
                                                      uint32_t *__restrict__ list)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < P && upos[i + 1] != upos[i]) list[upos[i]] = (uint32_t)i;
}

// The undecided points' inputs that do not depend on the stream: light 0's
// shadow coordinate and bias, and the offset of their samples were no earlier
// undecided point to find a blocker (base of the point).
__global__ __launch_bounds__(256) void k_pcss_points(FrameUniforms u, const float *__restrict__ g, size_t P,
                                                     const uint32_t *__restrict__ base,
                                                     const uint32_t *__restrict__ list, uint32_t n,
                                                     float4 *__restrict__ pt, uint32_t *__restrict__ pbase)
{
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const size_t i = list[k];
    Vec3 sc;
    float bias;
    pcss_pixel(u, g, P, i, sc, bias);
    pt[k] = make_float4(sc.x, sc.y, sc.z, bias);
    pbase[k] = base[i];
}

// The undecided points in order: point k draws from
// pbase[k] + n_pcf * (k - M_k), M_k the undecided points before it that find
// no blocker, so each outcome moves every later point's samples.  They are
// settled a segment [s0, s0 + L) at a time, M_{s0} = M0 known:
//  * a prediction of M_k: every point evaluated once at the current
//    prediction (k_pcss_guess), its misses scanned (kGuesses times, from a
//    straight line at the miss rate so far) -- exact wherever the outcomes
//    do not depend on the samples' offset, which is most points;
//  * k_pcss_band evaluates every point at the 63 values of M_k around its
//    prediction, a wavefront per point, eight of them at a time, the outcomes
//    as a bit mask;
//  * k_pcss_walk_blocks and k_pcss_chain follow the actual M_k through the
//    masks in order, write found[k] (1: a blocker) and stop where M_k
//    leaves the band or the segment ends; the host starts the next segment
//    there.
// Every evaluation is the blocker search exactly as FindAverageBlockDepth
// runs it (shadow.cpp:65-91: the samples in order, blocker depths summed in
// that order).  Every segment settles its first point (its prediction is
// exact).
constexpr int kBandHalf = 31;   // M_k in [prediction - 31, prediction + 31]: a wavefront per point
constexpr int kGuesses = 2;     // prediction rounds per segment (more do not pay)

// The blocker search of an undecided point by the kSearchLanes lanes whose
// lowest is a multiple of that, with its samples from offset o of the stream:
// lane j takes the samples j, j + kSearchLanes ..., so a load of the group's is
// one run of the stream and a guess's chain of loads a quarter as long (all 32
// of a point in one lane, a line per lane and load: segments of 8,192 to 32,768
// points 10.3 -> 4.9 us a guess, 48.5 -> 44.8 a band).  Found is whether a
// blocker's depth lies beyond 0.0011: no depth is below 0.001f, and the average
// of up to 64 of them with that one does not round below 0.001; where the only
// blockers are within reach of 0.001 the search is run as it is.
constexpr int kSearchLanes = 8;   // also the rounds of a band's 64 candidates
template <bool INSIDE>
__device__ __forceinline__ void pcss_samples(const FrameUniforms &u, const float *__restrict__ smap, const float2 *d, float4 q,
                                             int n, int sub, bool &any, bool &sure)
{
    const double filter = u.shadow.blocker_filter;
    const int w = (int)((float)u.SW - 0.001f), h = (int)((float)u.SH - 0.001f);
    constexpr int G = 4;   // 32 samples: one group
    for (int s0 = sub; s0 < n; s0 += G * kSearchLanes) {
        float2 ds[G];
#pragma unroll
        for (int e = 0; e < G; ++e) ds[e] = d[imin(s0 + e * kSearchLanes, n - 1)];   // (the last again: nothing new)
        float dd[G];
        bool in[G];
#pragma unroll
        for (int e = 0; e < G; ++e) {
            const float su = q.x + (float)((double)ds[e].x * filter);
            const float sv = q.y + (float)((double)ds[e].y * filter);
            in[e] = true;
            if (INSIDE) dd[e] = smap[(uint32_t)((int)((float)w * su) + (int)((float)h * sv) * u.SW)];
            else dd[e] = smap[shadow_texel(u.SW, w, h, su, sv, in[e])];
        }
#pragma unroll
        for (int e = 0; e < G; ++e) {
            const float v = shadow_value(in[e], dd[e]);
            const bool blk = q.z > v + q.w;
            any = any || blk;
            sure = sure || (blk && v > 0.0011f);
        }
    }
}

// Every sample of the point q on the map (true of its whole search area).
__device__ __forceinline__ bool pcss_inside(const FrameUniforms &u, float4 q)
{
    const float F = fabsf((float)u.shadow.blocker_filter);
    return q.x - F >= 0.f && q.x + F <= 1.f && q.y - F >= 0.f && q.y + F <= 1.f && (size_t)u.SW * u.SH < 0x80000000ull;
}

// OR over a group's lanes.
__device__ __forceinline__ uint32_t search_or(uint32_t v)
{
#pragma unroll
    for (int d = 1; d < kSearchLanes; d <<= 1) v |= __shfl_xor(v, d, 64);
    return v;
}

__device__ __forceinline__ bool pcss_search_exact(const FrameUniforms &u, const float *__restrict__ smap, const float *d, float4 q)
{
    return !((double)pcss_blocker_stream(u, smap, vec3(q.x, q.y, q.z), q.w, d, u.shadow.n_blocker) < 0.001);
}

// pred == nullptr: the prediction M0 + round(i * rate); else M0 + pred[i]
// (the scanned misses of the previous guess).  Clamped to the possible
// [M0, M0 + i].
__device__ __forceinline__ uint32_t pcss_predict(const uint32_t *__restrict__ pred, uint32_t M0, float rate,
                                                 uint32_t i)
{
    const uint32_t e = pred ? pred[i] : (uint32_t)((float)i * rate + 0.5f);
    return M0 + (e < i ? e : i);
}

__global__ __launch_bounds__(256) void k_pcss_guess(FrameUniforms u, const float *__restrict__ smap,
                                                    StreamVectors pairs, const float4 *__restrict__ pt,
                                                    const uint32_t *__restrict__ pbase, uint32_t s0, uint32_t L,
                                                    uint32_t M0, float rate, const uint32_t *__restrict__ pred,
                                                    uint32_t *__restrict__ miss)
{
    const uint32_t i = (blockIdx.x * 256 + threadIdx.x) / kSearchLanes;
    if (i >= L) return;
    const uint32_t k = s0 + i, M = pcss_predict(pred, M0, rate, i);
    const float4 q = pt[k];
    const float *d = stream_at<2>(pairs, pbase[k] + (uint32_t)u.shadow.n_pcf * (k - M));
    const int sub = (int)(threadIdx.x & (kSearchLanes - 1)), n = u.shadow.n_blocker;
    bool any = false, sure = false;
    if (__all(pcss_inside(u, q))) pcss_samples<true>(u, smap, (const float2 *)d, q, n, sub, any, sure);
    else pcss_samples<false>(u, smap, (const float2 *)d, q, n, sub, any, sure);
    const uint32_t got = search_or((any ? 1u : 0u) | (sure ? 2u : 0u));
    const bool f = got == 1u ? pcss_search_exact(u, smap, d, q) : got != 0u;
    if ((threadIdx.x & (kSearchLanes - 1)) == 0) miss[i] = f ? 0u : 1u;
}

__global__ __launch_bounds__(256) void k_pcss_band(FrameUniforms u, const float *__restrict__ smap,
                                                   StreamVectors pairs, const float4 *__restrict__ pt,
                                                   const uint32_t *__restrict__ pbase, uint32_t s0, uint32_t L,
                                                   uint32_t M0, const uint32_t *__restrict__ pred,
                                                   unsigned long long *__restrict__ masks)
{
    const uint32_t i = __builtin_amdgcn_readfirstlane((blockIdx.x * 256 + threadIdx.x) >> 6), lane = threadIdx.x & 63;
    if (i >= L) return;   // whole wavefronts
    const uint32_t k = s0 + i, n = (uint32_t)u.shadow.n_blocker, np = (uint32_t)u.shadow.n_pcf;
    const float4 q = pt[k];
    const uint32_t base = pbase[k];
    // candidate c: M = first + c, of those in [M0, M0 + i]; the samples of the
    // highest come first in the stream
    const long long first = (long long)pcss_predict(pred, M0, 0.f, i) - kBandHalf;
    const int lo = first < (long long)M0 ? (int)((long long)M0 - first) : 0;
    const long long top = (long long)M0 + i - first;
    const int hi = top < 2 * kBandHalf ? (int)top : 2 * kBandHalf;
    const uint32_t o_hi = base + np * (k - (uint32_t)(first + hi)), span = np * (uint32_t)(hi - lo);
    const StreamRun run = stream_run(pairs, o_hi);
    const bool one = span + n <= run.left, inside = pcss_inside(u, q);
    const int group = (int)(lane / kSearchLanes), sub = (int)(lane & (kSearchLanes - 1));
    uint32_t any_bits = 0, sure_bits = 0;   // of candidates group, group + 8, ...
#pragma unroll 2
    for (int t = 0; t < kSearchLanes; ++t) {
        const int c = t * (64 / kSearchLanes) + group;
        const int at = c < lo ? lo : c > hi ? hi : c;   // outside: masked below
        const uint32_t o = np * (uint32_t)(hi - at);
        const float *d = one ? run.v + 2 * (size_t)o : stream_at<2>(pairs, o_hi + o);
        bool any = false, sure = false;
        if (inside) pcss_samples<true>(u, smap, (const float2 *)d, q, (int)n, sub, any, sure);
        else pcss_samples<false>(u, smap, (const float2 *)d, q, (int)n, sub, any, sure);
        any_bits |= any ? 1u << t : 0u;
        sure_bits |= sure ? 1u << t : 0u;
    }
    uint32_t got = search_or(any_bits | sure_bits << 16);
    uint32_t found = got >> 16;
    for (uint32_t left = got & 0xffffu & ~found; left; left &= left - 1) {   // rare
        const int t = __builtin_ctz(left), c = t * (64 / kSearchLanes) + group;
        if (c < lo || c > hi) continue;
        if (pcss_search_exact(u, smap, stream_at<2>(pairs, o_hi + np * (uint32_t)(hi - c)), q)) found |= 1u << t;
    }
    unsigned long long m = 0ull;
#pragma unroll
    for (int t = 0; t < kSearchLanes; ++t) {
        const int c = t * (64 / kSearchLanes) + group;
        // bit j of the 8 candidates': lane 8 j's
        const unsigned long long b = __ballot((found >> t & 1u) && c >= lo && c <= hi) & 0x0101010101010101ull;
        m |= (b * 0x0102040810204080ull >> 56) << 8 * t;
    }
    if (lane == 0) masks[i] = m;
}

// Following the actual M_k through the masks.  With P_i the prediction
// (misses before point i in the segment, pred[i]) and D_i = 31 + M_i - M0 -
// P_i the actual M_i's place in point i's band, D_{i+1} = D_i + (miss_i(D_i)
// - (P_{i+1} - P_i)): D stays put while the prediction holds.  So a
// wavefront walking 64 points tests them all at one D; a ballot finds the
// first point whose outcome breaks the prediction (equals the predicted
// step), the points up to it settle (every one before it with the opposite
// outcome), and D moves by one from there.
//
// The segment is cut into blocks of kPcssChainBlock points, and every block is walked
// from each of the 63 places D can enter it with (k_pcss_walk_blocks: a
// workgroup per block and 16 places, a wavefront per place; block 0 only
// from 31), each walk writing its outcomes, the points it settled and the D
// it left with.  k_pcss_chain then follows the actual D from block to block
// through those results and copies the chosen walks' outcomes.  A walk stops
// where D leaves the band; so does the chain, at the first block whose walk
// stopped or which D enters from outside the band.
constexpr int kBandWidth = 2 * kBandHalf + 1;
constexpr int kChainWaves = 16;   // start places per workgroup
static_assert(kPcssChainBlock % 64 == 0 && kPcssBandWidth == kBandWidth, "chain layout");

__global__ __launch_bounds__(64 * kChainWaves) void k_pcss_walk_blocks(const unsigned long long *__restrict__ masks,
                                                                      const uint32_t *__restrict__ pred, uint32_t L,
                                                                      unsigned long long *__restrict__ fbits,
                                                                      uint32_t *__restrict__ res)
{
    __shared__ unsigned long long sm[kPcssChainBlock];
    __shared__ int sdl[kPcssChainBlock];
    const uint32_t b = blockIdx.x, at = b * kPcssChainBlock;
    const uint32_t nb = L - at < kPcssChainBlock ? L - at : kPcssChainBlock;
    for (uint32_t j = threadIdx.x; j < nb; j += 64 * kChainWaves) {
        sm[j] = masks[at + j];
        sdl[j] = (int)(pred[at + j + 1] - pred[at + j]);   // pred[L]: the segment's predicted total
    }
    __syncthreads();
    const int lane = (int)(threadIdx.x & 63), d0 = (int)blockIdx.y * kChainWaves + (int)(threadIdx.x >> 6);
    if (d0 >= kBandWidth || (b == 0 && d0 != kBandHalf)) return;   // whole wavefronts, after the only barrier
    unsigned long long *fo = fbits + ((size_t)b * kBandWidth + d0) * (kPcssChainBlock / 64);
    int D = d0;
    uint32_t settled = 0;
    for (uint32_t g = 0; g < nb; g += 64) {
        const uint32_t cnt = nb - g < 64 ? nb - g : 64;
        const unsigned long long valid = cnt == 64 ? ~0ull : ((1ull << cnt) - 1ull);
        // (slots past the block are never settled: valid masks them out)
        const unsigned long long m = sm[g + lane];
        const int dl = sdl[g + lane];
        const unsigned long long bm = dl ? m : ~m;
        const unsigned long long dlm = __ballot(dl != 0);
        uint32_t start = 0;
        unsigned long long brks = 0;
        bool stop = false;
        while (start < cnt) {
            if (D < 0 || D > 2 * kBandHalf) {
                stop = true;
                break;
            }
            const unsigned long long hit = __ballot((uint32_t)(bm >> D) & 1u) & valid & (~0ull << start);
            if (!hit) {
                start = cnt;
                break;
            }
            const uint32_t j = (uint32_t)__builtin_ctzll(hit);
            brks |= 1ull << j;
            D += ((dlm >> j) & 1ull) ? -1 : 1;
            start = j + 1;
        }
        if (lane == 0) fo[g / 64] = ~(dlm ^ brks);   // outcomes of the settled points
        settled += start;
        if (stop) break;
    }
    if (lane == 0) {
        uint32_t *r = res + 2 * ((size_t)b * kBandWidth + d0);
        r[0] = settled;
        r[1] = (uint32_t)D;
    }
}

// One workgroup: the chain through the blocks' walks (their results staged
// in LDS), then found[] for the settled points.  out = (first unsettled
// point, M there).
constexpr uint32_t kChainThreads = 1024;
__global__ __launch_bounds__(kChainThreads) void k_pcss_chain(const unsigned long long *__restrict__ fbits,
                                                    const uint32_t *__restrict__ res, const uint32_t *__restrict__ pred,
                                                    uint32_t s0, uint32_t L, uint32_t M0, uint32_t *__restrict__ found,
                                                    uint32_t *__restrict__ out)
{
    constexpr uint32_t kMaxBlocks = kPcssSegmentMax / kPcssChainBlock;
    __shared__ __align__(8) uint32_t sres[2 * kBandWidth * kMaxBlocks];
    __shared__ int pick[kMaxBlocks];
    __shared__ uint32_t s_settled;
    __shared__ int s_D;
    const uint32_t tid = threadIdx.x;
    const uint32_t nblk = (L + kPcssChainBlock - 1) / kPcssChainBlock;
    for (uint32_t i = tid; i < 2 * kBandWidth * nblk; i += kChainThreads) sres[i] = res[i];
    __syncthreads();
    if (tid == 0) {
        int D = kBandHalf;
        uint32_t settled = 0;
        for (uint32_t b = 0; b < nblk; ++b) {
            if (D < 0 || D > 2 * kBandHalf) break;
            const uint32_t len = L - b * kPcssChainBlock < kPcssChainBlock ? L - b * kPcssChainBlock : kPcssChainBlock;
            const uint2 r = *(const uint2 *)(sres + 2 * (b * kBandWidth + (uint32_t)D));
            pick[b] = D;
            D = (int)r.y;
            settled += r.x;
            if (r.x < len) break;
        }
        s_settled = settled;
        s_D = D;
    }
    __syncthreads();
    const uint32_t settled = s_settled;
#pragma unroll 4
    for (uint32_t k = tid; k < settled; k += kChainThreads) {
        const uint32_t b = k / kPcssChainBlock, kk = k - b * kPcssChainBlock;
        const unsigned long long w = fbits[((size_t)b * kBandWidth + (uint32_t)pick[b]) * (kPcssChainBlock / 64) + kk / 64];
        found[s0 + k] = (uint32_t)(w >> (kk & 63)) & 1u;
    }
    if (tid == 0) {
        out[0] = s0 + settled;
        out[1] = (uint32_t)((int)M0 + (int)pred[settled] + s_D - kBandHalf);
    }
}

// offs[i] = base[i] + n_pcf * fpos[upos[i]] for i = 0..P (offs[P] = total).
__global__ __launch_bounds__(256) void k_pcss_offsets(const uint32_t *__restrict__ base,
                                                      const uint32_t *__restrict__ upos,
                                                      const uint32_t *__restrict__ fpos, uint32_t n_pcf, size_t P,
                                                      uint32_t *__restrict__ offs)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i <= P) offs[i] = base[i] + n_pcf * fpos[upos[i]];
}

// Kernel SSAO over 64 x 16-pixel tiles (1024 threads, a wavefront per row):
// the workgroup first copies the depth plane around its tile, 32 pixels
// each side, into LDS (coalesced 16-byte loads), and taps that land there
// read LDS; the others read the plane.  Per tap it issues about 42 vector
// ALU operations (projection, reciprocal, bounds, address, compare).  A
// workgroup none of whose pixels can be occluded (nothing drawn there) is
// done before the copy, a wavefront of a mixed one before its taps.
constexpr int kSsaoTW = 64, kSsaoTH = 16, kSsaoHalo = 32;
static_assert(kSsaoTW * kSsaoTH == 1024 && kSsaoHalo % 4 == 0, "one thread per pixel; 16-byte staging");
constexpr int kSsaoLW = kSsaoTW + 2 * kSsaoHalo, kSsaoLH = kSsaoTH + 2 * kSsaoHalo;

__global__ __launch_bounds__(1024) void k_ssao_tiled(FrameUniforms u, SsaoArgs sa,
                                                     const float *__restrict__ depth,
                                                     const float *__restrict__ g,
                                                     float *__restrict__ ao)
{
    __shared__ float tile[kSsaoLH * kSsaoLW];
    const int x0 = blockIdx.x * kSsaoTW, y0 = blockIdx.y * kSsaoTH;
    const int lx0 = x0 - kSsaoHalo, ly0 = y0 - kSsaoHalo;
    const int x = x0 + (int)(threadIdx.x % kSsaoTW), y = y0 + (int)(threadIdx.x / kSsaoTW);
    const bool on = x < u.W && y < u.H;
    SsaoPx px;
    px.none = true;
    if (on) px = ssao_setup(u, sa, depth, g, x, y);
    float *out = ao + (size_t)x + (size_t)y * u.W;
    if (__syncthreads_and(px.none)) {
        if (on) *out = 1.f;
        return;
    }
    const bool vec = (u.W & 3) == 0;   // rows start 16-byte aligned
    for (int k = threadIdx.x; k < kSsaoLH * kSsaoLW / 4; k += 1024) {
        const int row = k / (kSsaoLW / 4), c4 = k - row * (kSsaoLW / 4);
        const int gy = ly0 + row, gx = lx0 + 4 * c4;
        float v[4] = {0.f, 0.f, 0.f, 0.f};   // outside the plane: never read
        if (gy >= 0 && gy < u.H) {
            const float *src = depth + (size_t)gy * u.W;
            if (vec && gx >= 0 && gx + 3 < u.W) {
                const float4 q = *(const float4 *)(src + gx);
                v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (gx + e >= 0 && gx + e < u.W) v[e] = src[gx + e];
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) tile[row * kSsaoLW + 4 * c4 + e] = v[e];
    }
    __syncthreads();
    if (!on) return;
    if (__all(px.none)) {
        *out = 1.f;
        return;
    }
    const uint32_t W = (uint32_t)u.W;
    // The plane is read through a global-address-space pointer: with two
    // generic pointers the compiler merges both reads into one flat load,
    // which sends the LDS taps down the vector-memory path as well.
    const __attribute__((address_space(1))) float *gdepth =
        (const __attribute__((address_space(1))) float *)depth;
    *out = ssao_taps(u, sa, px, [&](int sx, int sy) {
        const uint32_t tx = (uint32_t)(sx - lx0), ty = (uint32_t)(sy - ly0);
        const bool near = tx < (uint32_t)kSsaoLW && ty < (uint32_t)kSsaoLH;
        // Every lane reads LDS (a far lane at the tile's first word) and far
        // lanes also read the plane, into another register: the LDS read
        // does not wait for the plane's.
        const float dl = tile[near ? ty * kSsaoLW + tx : 0u];
        float dg = 0.f;
        if (!near) dg = gdepth[(uint32_t)sx + (uint32_t)sy * W];
        return near ? dl : dg;
    });
}

// Buffer1f::TwoPassGaussianBlurDenoised (src/buffer.cpp:59-98) is in place and
// order dependent: the taps left of (or below) a pixel read values already
// blurred.  One thread owns a whole row (then a whole column) and walks it in
// the reference's order, so every read sees exactly what the reference sees.
__constant__ float c_ref_blur_w[5] = {(float)0.227027, (float)0.1945946, (float)0.1216216,
                                      (float)0.054054, (float)0.016216};

// Buffer1f::TwoPassGaussianBlurDenoised (src/buffer.cpp:59-98) along lines of
// n samples, in place: each output is the reference's sum in its order -- the
// centre, then for i = 1..4 the sample i ahead (not yet blurred) and the
// sample i behind (already blurred), indices clamped to the line.
//
// A line is a chain: a step needs the output before it, and a frame has fewer
// lines than the chip has lanes, so the kernel is bound by the instructions of
// one step.  One wavefront takes the steps of 64 lines and is left only the
// sums in order and the products of its outputs (8 additions, 4 products); four
// others make what does not depend on outputs -- centre plus first sample
// ahead, the other products ahead -- a chunk of samples before it, and carry
// its results out a chunk after it.  Every step done by its line's thread with
// its loads and stores: 1280 x 800 rows 128 -> 53 us, columns 64 -> 36.
constexpr int kRecChunk = 32, kRecWaves = 4, kRecPer = kRecChunk / kRecWaves;

// ROWS: line l is row l (n = W), else column l (n = H).  vec: rows start
// 16-byte aligned and hold whole quads.
template <bool ROWS>
__global__ __launch_bounds__(64 * (kRecWaves + 1)) void k_blur_rec(float *p, int W, int H, bool vec)
{
    __shared__ float4 ahead[2][kRecChunk][64];
    __shared__ float done[2][kRecChunk][65];
    const float w0 = c_ref_blur_w[0], w1 = c_ref_blur_w[1], w2 = c_ref_blur_w[2], w3 = c_ref_blur_w[3],
                w4 = c_ref_blur_w[4];
    const int lines = ROWS ? H : W, n = ROWS ? W : H, l0 = blockIdx.x * 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int line = imin(l0 + lane, lines - 1);   // past the last: computed, not written
    const size_t step = ROWS ? 1 : W;
    float *mine = p + (ROWS ? (size_t)line * W : (size_t)line);
    const int chunks = (n + kRecChunk - 1) / kRecChunk;
    // slot t: chunk t is prepared, chunk t - 1 stepped through, chunk t - 2 written
    if (wave == 0) {
        const float first = mine[0];   // x = 0: every sample behind clamps to sample 0, not yet blurred
        float p1 = first * w1, p2[2] = {first * w2, 0.f}, p3[3] = {first * w3, 0.f, 0.f}, p4[4] = {first * w4, 0.f, 0.f, 0.f};
        lds_barrier();
        for (int c = 0; c < chunks; ++c) {
            const int buf = c & 1;
#pragma unroll 1
            for (int e0 = 0; e0 < kRecChunk; e0 += 8) {
                float4 v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = ahead[buf][e0 + e][lane];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    float q = v[e].x + p1;
                    q += v[e].y;
                    q += p2[0];
                    q += v[e].z;
                    q += p3[0];
                    q += v[e].w;
                    q += p4[0];
                    done[buf][e0 + e][lane] = q;
                    const float r2 = q * w2, r3 = q * w3, r4 = q * w4;
                    p1 = q * w1;
                    p2[0] = p2[1]; p2[1] = r2;
                    p3[0] = p3[1]; p3[1] = p3[2]; p3[2] = r3;
                    p4[0] = p4[1]; p4[1] = p4[2]; p4[2] = p4[3]; p4[3] = r4;
                    if (e == 0 && e0 == 0 && c == 0) {   // from here on they clamp to the blurred sample 0
                        p2[0] = r2;
                        p3[0] = p3[1] = r3;
                        p4[0] = p4[1] = p4[2] = r4;
                    }
                }
            }
            lds_barrier();
        }
        return;
    }
    const int w = wave - 1, tid = threadIdx.x - 64;
    float a[kRecPer + 4];   // the samples of this thread's part of the next chunk, and four ahead
    auto load = [&](int c) {
        const int x0 = c * kRecChunk + w * kRecPer;
        if (ROWS && vec) {
#pragma unroll
            for (int e = 0; e < kRecPer + 4; e += 4) {
                if (x0 + e < n) {
                    const float4 v = *(const float4 *)(mine + x0 + e);
                    a[e] = v.x; a[e + 1] = v.y; a[e + 2] = v.z; a[e + 3] = v.w;
                } else {
                    a[e] = a[e + 1] = a[e + 2] = a[e + 3] = mine[n - 1];
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < kRecPer + 4; ++e) a[e] = mine[(size_t)imin(x0 + e, n - 1) * step];
        }
    };
    load(0);
    for (int t = 0; t < chunks + 2; ++t) {
        if (t < chunks) {
#pragma unroll
            for (int e = 0; e < kRecPer; ++e)
                ahead[t & 1][w * kRecPer + e][lane] = make_float4(a[e] * w0 + a[e + 1] * w1, a[e + 2] * w2, a[e + 3] * w3,
                                                                  a[e + 4] * w4);
            if (t + 1 < chunks) load(t + 1);
        }
        if (t >= 2) {
            const int c = t - 2;
            if (ROWS) {
                const int x = tid & 31, at = c * kRecChunk + x;
#pragma unroll
                for (int r = 0; r < 64; r += 2 * kRecWaves) {
                    const int row = r + (tid >> 5);
                    if (at < n && l0 + row < lines) p[(size_t)(l0 + row) * W + at] = done[c & 1][x][row];
                }
            } else {
#pragma unroll
                for (int e = 0; e < kRecPer; ++e) {
                    const int x = c * kRecChunk + w * kRecPer + e;
                    if (x < n && l0 + lane < lines) p[(size_t)x * W + l0 + lane] = done[c & 1][w * kRecPer + e][lane];
                }
            }
        }
        lds_barrier();
    }
}

struct BlurWeights {
    float w[9];
    int R;
};

// Separable Gaussian in one pass: a workgroup stages a (16 + 2R) x (64 + 2R)
// block of the source in LDS (coordinates clamped to the image, as the taps
// are), runs the horizontal taps for its 16 + 2R rows (the rows the vertical
// taps of its 64 x 16 outputs read, clamped likewise) into a second LDS
// block, then the vertical taps; each tap sum in the reference loop's order
// (centre, then +i and -i for i = 1..R), so the result is the
// horizontal-then-vertical two-pass filter bit for bit, without an
// intermediate plane in HBM.  Writes dst (not src: neighbouring workgroups
// read src).
constexpr int kBlurTW = 64, kBlurTH = 16, kBlurMaxR = 8;

template <int R>
__global__ __launch_bounds__(256) void k_blur_fused(const float *__restrict__ src, float *__restrict__ dst,
                                                    int W, int H, BlurWeights bw)
{
    __shared__ float s[kBlurTH + 2 * kBlurMaxR][kBlurTW + 2 * kBlurMaxR];
    __shared__ float t[kBlurTH + 2 * kBlurMaxR][kBlurTW];
    constexpr int rows = kBlurTH + 2 * R, cols = kBlurTW + 2 * R;
    const int x0 = blockIdx.x * kBlurTW, y0 = blockIdx.y * kBlurTH;
    for (int k = threadIdx.x; k < rows * cols; k += 256) {
        const int j = k / cols, i = k - j * cols;
        const int gy = clampi(y0 - R + j, 0, H - 1), gx = clampi(x0 - R + i, 0, W - 1);
        s[j][i] = src[(size_t)gx + (size_t)gy * W];
    }
    __syncthreads();
    for (int k = threadIdx.x; k < rows * kBlurTW; k += 256) {
        const int j = k / kBlurTW, x = k - j * kBlurTW;
        float r = s[j][x + R] * bw.w[0];
#pragma unroll
        for (int i = 1; i <= R; ++i) {
            r += s[j][x + R + i] * bw.w[i];
            r += s[j][x + R - i] * bw.w[i];
        }
        t[j][x] = r;
    }
    __syncthreads();
    for (int k = threadIdx.x; k < kBlurTH * kBlurTW; k += 256) {
        const int yy = k / kBlurTW, x = k - yy * kBlurTW;
        const int gx = x0 + x, gy = y0 + yy;
        if (gx >= W || gy >= H) continue;
        float r = t[yy + R][x] * bw.w[0];
#pragma unroll
        for (int i = 1; i <= R; ++i) {
            r += t[yy + R + i][x] * bw.w[i];
            r += t[yy + R - i][x] * bw.w[i];
        }
        dst[(size_t)gx + (size_t)gy * W] = r;
    }
}

__global__ __launch_bounds__(256) void k_resolve(const float *__restrict__ fb, int W, int H, int k,
                                                 uint8_t *__restrict__ img)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= W / k || y >= H / k) return;
    resolve_px(fb, W, H, k, img, x, y);
}

// Plain 16-byte copy: the reference point for HBM byte counters.
__global__ __launch_bounds__(256) void k_copy(const float4 *__restrict__ src, float4 *__restrict__ dst,
                                              size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

void launch_copy(const void *src, void *dst, size_t bytes, hipStream_t s)
{
    size_t n = bytes / 16;
    if (n == 0) return;
    hipLaunchKernelGGL(k_copy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (const float4 *)src,
                       (float4 *)dst, n);
}

static inline dim3 grid2(int W, int H) { return dim3((W + 63) / 64, (H + 3) / 4); }

void launch_lighting(const FrameUniforms &u, const float *gbuf, const float *ao, int ao_is_one, const NetAo &net,
                     const float *shadow_map, const ShadowSamples &ss, float *fb, hipStream_t s)
{
    if (u.W <= 0 || u.H <= 0) return;
    const dim3 grid = grid2(u.W, u.H);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, u, gbuf, ao, ao_is_one, net, shadow_map, ss, fb);
    };
    if (ss.sv.v) return go(k_lighting<true, -1>);
    switch (u.shadow_on ? u.shadow.mode : 0) {
    case 0: return go(k_lighting<false, 0>);
    case 1: return go(k_lighting<false, 1>);
    case 2: return go(k_lighting<false, 2>);
    case 3: return go(k_lighting<false, 3>);
    default: return go(k_lighting<false, -1>);
    }
}

void launch_ssao_reference(const FrameUniforms &u, const StreamVectors &samples, const float *pow3,
                           const float *depth, const float *gbuf, float *ao, hipStream_t s)
{
    if (u.W <= 0 || u.H <= 0) return;
    hipLaunchKernelGGL(k_ssao_ref, grid2(u.W, u.H), dim3(256), 0, s, u, samples, pow3, depth, gbuf, ao);
}

// Windows of a power of two up to 16 texels a side that the square of most
// points holds; none where making them reads the map more than they save.
bool pcss_windows(const FrameUniforms &u, size_t P, int &bx, int &by)
{
    const double f = 2.0 * (float)u.shadow.blocker_filter;
    if (!(f > 0.0) || u.SW <= 0 || u.SH <= 0) return false;
    const double nx = std::fmin(f * u.SW, u.SW - 1.0) + 1.0, ny = std::fmin(f * u.SH, u.SH - 1.0) + 1.0;
    bx = by = 1;
    while (2 * bx <= nx && bx < kMmMax) bx *= 2;
    while (2 * by <= ny && by < kMmMax) by *= 2;
    return bx * by >= 4 && (double)P * nx * ny > 4.0 * u.SW * u.SH;
}

void launch_pcss_minmax(const FrameUniforms &u, const float *shadow_map, int bx, int by, float2 *mm, hipStream_t s)
{
    hipLaunchKernelGGL(k_pcss_minmax, dim3((u.SW + kMmW - 1) / kMmW, (u.SH + kMmH - 1) / kMmH), dim3(256), 0, s, shadow_map,
                       u.SW, u.SH, bx, by, mm);
}

void launch_pcss_classify(const FrameUniforms &u, const float *g, size_t P, const float *shadow_map, const float2 *mm,
                          int bx, int by, uint32_t *cnt, uint32_t *unc, hipStream_t s)
{
    if (P == 0) return;
    hipLaunchKernelGGL(k_pcss_classify, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, s, u, g, P, shadow_map, mm, bx, by,
                       cnt, unc);
}

void launch_pcss_compact(const uint32_t *upos, size_t P, uint32_t *list, hipStream_t s)
{
    if (P == 0) return;
    hipLaunchKernelGGL(k_pcss_compact, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, s, upos, P, list);
}

void launch_pcss_points(const FrameUniforms &u, const float *g, size_t P, const uint32_t *base, const uint32_t *list,
                        uint32_t n, float4 *pt, uint32_t *pbase, hipStream_t s)
{
    if (n == 0) return;
    hipLaunchKernelGGL(k_pcss_points, dim3((n + 255) / 256), dim3(256), 0, s, u, g, P, base, list, n, pt, pbase);
}

void launch_pcss_segment(const FrameUniforms &u, const float *shadow_map, const StreamVectors &pairs, const float4 *pt,
                         const uint32_t *pbase, uint32_t s0, uint32_t L, uint32_t M0, float rate, uint32_t *pred,
                         uint32_t *scan_tmp, unsigned long long *masks, unsigned long long *fbits, uint32_t *res,
                         uint32_t *found, uint32_t *out, hipStream_t s)
{
    if (L == 0 || L > kPcssSegmentMax) return;
    // kGuesses guesses: from the straight line, then each from the misses of
    // the one before; the last lands in pred + (L + 1)
    uint32_t *bufs[2] = {pred + (L + 1), pred};
    const uint32_t *prev = nullptr;
    for (int q = 0; q < kGuesses; ++q) {
        uint32_t *dst = bufs[(kGuesses - 1 - q) & 1];
        hipLaunchKernelGGL(k_pcss_guess, dim3((L + 256 / kSearchLanes - 1) / (256 / kSearchLanes)), dim3(256), 0, s, u, shadow_map, pairs, pt, pbase, s0, L,
                           M0, rate, prev, dst);
        launch_exclusive_scan(dst, dst, L, scan_tmp, s);
        prev = dst;
    }
    const uint32_t *pred2 = prev;
    hipLaunchKernelGGL(k_pcss_band, dim3((L + 3) / 4), dim3(256), 0, s, u, shadow_map, pairs, pt, pbase, s0, L, M0,
                       (const uint32_t *)pred2, masks);
    const uint32_t nblk = (L + kPcssChainBlock - 1) / kPcssChainBlock;
    hipLaunchKernelGGL(k_pcss_walk_blocks, dim3(nblk, (kBandWidth + kChainWaves - 1) / kChainWaves),
                       dim3(64 * kChainWaves), 0, s, masks, pred2, L, fbits, res);
    hipLaunchKernelGGL(k_pcss_chain, dim3(1), dim3(kChainThreads), 0, s, fbits, res, pred2, s0, L, M0, found, out);
}

void launch_pcss_offsets(const uint32_t *base, const uint32_t *upos, const uint32_t *fpos, uint32_t n_pcf, size_t P,
                         uint32_t *offs, hipStream_t s)
{
    hipLaunchKernelGGL(k_pcss_offsets, dim3((unsigned)((P + 1 + 255) / 256)), dim3(256), 0, s, base, upos, fpos, n_pcf,
                       P, offs);
}

void launch_ssao(const FrameUniforms &u, const SsaoArgs &sa, const float *depth,
                 const float *gbuf, float *ao, hipStream_t s)
{
    if (u.W <= 0 || u.H <= 0) return;
    hipLaunchKernelGGL(k_ssao_tiled, dim3((u.W + kSsaoTW - 1) / kSsaoTW, (u.H + kSsaoTH - 1) / kSsaoTH), dim3(1024),
                       0, s, u, sa, depth, gbuf, ao);
}

void launch_blur_recursive(float *ao, int W, int H, hipStream_t s)
{
    if (W <= 0 || H <= 0) return;
    const bool vec = (W & 3) == 0 && ((uintptr_t)ao & 15) == 0;
    const dim3 block(64 * (kRecWaves + 1));
    hipLaunchKernelGGL(k_blur_rec<true>, dim3((H + 63) / 64), block, 0, s, ao, W, H, vec);
    hipLaunchKernelGGL(k_blur_rec<false>, dim3((W + 63) / 64), block, 0, s, ao, W, H, vec);
}

void launch_blur_separable(const float *src, float *dst, int W, int H, const float *w, int R, hipStream_t s)
{
    if (W <= 0 || H <= 0) return;
    BlurWeights bw;
    for (int i = 0; i < 9; ++i) bw.w[i] = i <= R ? w[i] : 0.f;
    bw.R = R;
    const dim3 grid((W + kBlurTW - 1) / kBlurTW, (H + kBlurTH - 1) / kBlurTH);
    switch (R) {
#define FGL_BLUR_CASE(r) \
    case r: hipLaunchKernelGGL(k_blur_fused<r>, grid, dim3(256), 0, s, src, dst, W, H, bw); break;
        FGL_BLUR_CASE(1) FGL_BLUR_CASE(2) FGL_BLUR_CASE(3) FGL_BLUR_CASE(4)
        FGL_BLUR_CASE(5) FGL_BLUR_CASE(6) FGL_BLUR_CASE(7) FGL_BLUR_CASE(8)
#undef FGL_BLUR_CASE
    default: break;
    }
}

// recip(w) against the IEEE quotient 1.f / w for every non-NaN float w:
// counts[0] += floats compared, counts[1] += those that differ, counts[2] +=
// those that took the reciprocal-and-Newton path.
__global__ __launch_bounds__(256) void k_check_recip(unsigned long long *__restrict__ counts)
{
    __shared__ unsigned long long part[3][4];
    unsigned long long n = 0, bad = 0, fast = 0;
    const uint64_t stride = (uint64_t)gridDim.x * 256;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < (1ull << 32); i += stride) {
        const float w = __uint_as_float((uint32_t)i);
        if (w != w) continue;
        ++n;
        const float a = fabsf(w);
        fast += (a >= 0x1p-125f && a <= 0x1p125f) ? 1u : 0u;
        bad += __float_as_uint(recip(w)) != __float_as_uint(1.f / w) ? 1u : 0u;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        n += __shfl_xor(n, o, 64);
        bad += __shfl_xor(bad, o, 64);
        fast += __shfl_xor(fast, o, 64);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        part[0][wave] = n;
        part[1][wave] = bad;
        part[2][wave] = fast;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        const unsigned long long v = part[threadIdx.x][0] + part[threadIdx.x][1] + part[threadIdx.x][2] +
                                     part[threadIdx.x][3];
        atomicAdd(&counts[threadIdx.x], v);
    }
}

void launch_check_recip(unsigned long long *counts, hipStream_t s)
{
    hipLaunchKernelGGL(k_check_recip, dim3(4096), dim3(256), 0, s, counts);
}

void launch_resolve(const float *fb, int W, int H, int k, uint8_t *img, hipStream_t s)
{
    int ow = W / k, oh = H / k;
    if (ow <= 0 || oh <= 0) return;
    hipLaunchKernelGGL(k_resolve, grid2(ow, oh), dim3(256), 0, s, fb, W, H, k, img);
}

}  // namespace fgl
