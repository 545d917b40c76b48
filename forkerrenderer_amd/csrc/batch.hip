// batch.hip -- batched-view kernels for gfx950.  Each pass covers every view
// of a batch in one launch; per-view parameters come from the DevView table
// (indexed by the draw's view, by a (view, tile) queue item, or by the view
// of a 64 x 4 pixel block).  The per-vertex, per-triangle, per-tile and
// per-pixel bodies are the single-view ones (raster_core.hpp,
// shade_core.hpp), so a view's results are those of its single-view render.
//
// A batch is rendered through the tile lists while its (tile, triangle) pairs
// are being counted or may not fit their capacity, and through the direct
// rasteriser (raster_core.hpp) once they are known to fit.  24 views of 75,516
// to 1,701,780 pixels (14.1 M), 25 M shadow-map pixels: the tile rasteriser's
// two launches alone 760 us, all direct kernels 670 us; a render 3,715 -> 3,311
// us, of which copying the images out takes 820.
//
// The pair count of a pass is known only on the device: the emit kernels
// drop pairs beyond the capacity, the sort and tile-range kernels read the
// count from device memory, and an overflow flag tells the host to re-render
// with more room.  Nothing here needs the host mid-pass, so the whole
// sequence can be captured in a HIP graph.
#include "batch.hpp"
#include "raster_core.hpp"
#include "shade_core.hpp"

namespace fgl {

// Vertex and setup grids are flat lists of 256-item blocks: block b covers
// items blocks[b].y .. + 255 of draw blocks[b].x (draws differ in size by
// orders of magnitude in a batch, so a draws x largest-draw grid would be
// mostly empty).
template <int PASS>
__global__ __launch_bounds__(256) void k_bv_vertex(const DevDraw *__restrict__ draws,
                                                   const DevView *__restrict__ views,
                                                   const uint2 *__restrict__ blocks,
                                                   int4 *__restrict__ out, float *__restrict__ ndc_z,
                                                   float4 *__restrict__ vary)
{
    const uint2 bk = blocks[blockIdx.x];
    const DevDraw &dr = draws[bk.x];
    const int vi = (int)bk.y + threadIdx.x;
    if (vi >= dr.n_pos) return;
    const FrameUniforms &u = views[dr.view].u;
    if (PASS == kBvShadow) {
        const Vec4 n = depth_ndc(dr, vi);
        out[dr.vert_base + vi] = to_screen(u.shadow_viewport, n);
        ndc_z[dr.vert_base + vi] = n.z;
    } else {
        out[dr.vert_base + vi] = to_screen(u.viewport, main_vertex_pass(dr, u, vi, vary));
    }
}

template <int PASS>
__global__ __launch_bounds__(256) void k_bv_setup(const DevDraw *__restrict__ draws,
                                                  const DevView *__restrict__ views,
                                                  const uint2 *__restrict__ blocks,
                                                  const int4 *__restrict__ screen, int TS,
                                                  uint2 *__restrict__ rect,
                                                  uint32_t *__restrict__ count,
                                                  int4 *__restrict__ tri_v,
                                                  uint32_t *__restrict__ big_list,
                                                  uint32_t *__restrict__ big_count)
{
    const uint2 bk = blocks[blockIdx.x];
    const int d = (int)bk.x;
    const DevDraw &dr = draws[d];
    const int f = (int)bk.y + threadIdx.x;
    if (f >= dr.n_faces) return;
    const DevView &v = views[dr.view];
    const int W = PASS == kBvShadow ? v.S : v.W, H = PASS == kBvShadow ? v.S : v.H;
    setup_tri(dr, d, f, screen, W, H, TS, rect, count, tri_v, big_list, big_count);
}

template <int PASS>
__global__ __launch_bounds__(256) void k_bv_emit_small(BvBinArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.n_tri) return;
    const uint32_t o = a.off[t], n = a.off[t + 1] - o;
    if (n == 0 || n > (uint32_t)kSmallTriTiles) return;
    const DevView &v = a.views[a.draws[a.tri_v[t].w].view];
    const uint2 r = a.rect[t];
    for (uint32_t j = 0; j < n; ++j) {
        if (o + j >= a.cap) break;
        a.keys[o + j] = pair_key(r, j, v.tiles_x[PASS], v.tile_base[PASS]);
        a.vals[o + j] = (uint32_t)t;
    }
}

// Persistent: workgroups stride over the device-side big-triangle list.
template <int PASS>
__global__ __launch_bounds__(256) void k_bv_emit_big(BvBinArgs a)
{
    const uint32_t nbig = *a.big_count;
    for (uint32_t b = blockIdx.x; b < nbig; b += gridDim.x) {
        const uint32_t t = a.big_list[b];
        const uint32_t o = a.off[t], n = a.off[t + 1] - o;
        const DevView &v = a.views[a.draws[a.tri_v[t].w].view];
        const uint2 r = a.rect[t];
        for (uint32_t j = threadIdx.x; j < n; j += blockDim.x) {
            if (o + j >= a.cap) break;
            a.keys[o + j] = pair_key(r, j, v.tiles_x[PASS], v.tile_base[PASS]);
            a.vals[o + j] = t;
        }
    }
}

__global__ void k_bv_overflow(const uint32_t *__restrict__ total, uint32_t cap, uint32_t *__restrict__ flag)
{
    if (threadIdx.x == 0) flag[0] = *total > cap ? 1u : 0u;
}

// Persistent rasteriser: each workgroup pulls (view, tile) items from the
// queue until it runs dry, and rasterises each as the single-view kernel
// rasterises that view's tile.
template <int TS, int BLOCK, bool SHADOW>
__global__ __launch_bounds__(BLOCK) void k_bv_raster(BvRasterArgs b)
{
    __shared__ RasterLds<TS, BLOCK> lds;
    __shared__ uint32_t s_item;
    constexpr int P = SHADOW ? kBvShadow : kBvMain;
    for (;;) {
        if (threadIdx.x == 0) s_item = atomicAdd(b.queue, 1u);
        __syncthreads();
        const uint32_t it = s_item;
        __syncthreads();
        if (it >= b.n_items) return;
        const uint32_t code = b.items[it];
        const DevView &v = b.views[code >> 24];
        const int tile = (int)(code & 0xffffffu);
        RasterArgs a;
        a.draws = b.draws;
        a.n_draws = 0;
        a.screen = b.screen;
        a.tri_v = b.tri_v;
        a.vals = b.vals;
        a.tile_start = b.tile_start + v.tile_base[P];
        a.tile_end = b.tile_end + v.tile_base[P];
        a.W = SHADOW ? v.S : v.W;
        a.H = SHADOW ? v.S : v.H;
        a.tiles_x = v.tiles_x[P];
        a.tiles_y = v.tiles_y[P];
        a.fresh = 1;
        a.depth = SHADOW ? b.shadow_depth + v.spx_off : b.depth + v.px_off;
        a.vis = b.vis + v.px_off;
        a.shadow_out = b.shadow + v.spx_off;
        a.ndc_z = b.ndc_z;
        raster_tile<TS, BLOCK, SHADOW>(a, tile, lds);
    }
}

// ---- the direct rasteriser over all views ----

// The vertex records, the key plane cleared (8 keys a thread) by the
// workgroups past the vertices', the overflow flags zeroed (views do not
// change, so a batch whose pairs were counted has none).
template <int PASS>
__global__ __launch_bounds__(256) void k_bv_direct_vertex(BvDirectArgs a, const uint2 *__restrict__ blocks, int n_blocks,
                                                          int4 *__restrict__ out, float *__restrict__ ndc_z,
                                                          float4 *__restrict__ vary, size_t n_keys,
                                                          uint32_t *__restrict__ flags)
{
    const int b = blockIdx.x;
    if (b >= n_blocks) {
        if (b == n_blocks && threadIdx.x < 2) flags[threadIdx.x] = 0u;
        const size_t k0 = (size_t)(b - n_blocks) * (256 * kClearKeys);
        ulonglong2 c;
        c.x = c.y = kDirectClear;
#pragma unroll
        for (int e = 0; e < kClearKeys / 2; ++e) {
            const size_t k = k0 + 2 * ((size_t)e * 256 + threadIdx.x);
            if (k + 1 < n_keys) *(ulonglong2 *)(a.key + k) = c;
            else if (k < n_keys) a.key[k] = kDirectClear;
        }
        return;
    }
    const uint2 bk = blocks[b];
    const DevDraw &dr = a.draws[bk.x];
    const int vi = (int)bk.y + threadIdx.x;
    if (vi >= dr.n_pos) return;
    const FrameUniforms &u = a.views[dr.view].u;
    if (PASS == kBvShadow) {
        const Vec4 n = depth_ndc(dr, vi);
        out[dr.vert_base + vi] = to_screen(u.shadow_viewport, n);
        ndc_z[dr.vert_base + vi] = n.z;
    } else {
        out[dr.vert_base + vi] = to_screen(u.viewport, main_vertex_pass(dr, u, vi, a.views[dr.view].corner ? nullptr : vary));
    }
}

template <int PASS>
__device__ __forceinline__ DirectArgs bv_direct_args(const BvDirectArgs &b, const DevView &v)
{
    DirectArgs a;
    a.draws = b.draws;
    a.n_draws = b.n_draws;
    a.screen = b.screen;
    a.key = b.key + (PASS == kBvShadow ? v.spx_off : v.px_off);
    a.fix = nullptr;
    a.deep_from = b.deep_from;
    a.big_start = b.big_start;
    a.big_tri = b.big_tri;
    a.ctr = b.ctr;
    a.W = PASS == kBvShadow ? v.S : v.W;
    a.H = PASS == kBvShadow ? v.S : v.H;
    return a;
}

template <int PASS>
__global__ __launch_bounds__(256) void k_bv_direct(BvDirectArgs b, const uint2 *__restrict__ blocks)
{
    __shared__ DirectLds lds;
    const uint2 bk = blocks[xcd_remap(blockIdx.x, gridDim.x)];
    const DevDraw &dr = b.draws[bk.x];
    const DirectArgs a = bv_direct_args<PASS>(b, b.views[dr.view]);
    const int first = (int)(bk.y & 0x3fffffffu);
    const uint32_t code = bk.y >> 30;
    if (code == 0) direct_group<1>(a, dr, first, lds);
    else if (code == 1) direct_group<4>(a, dr, first, lds);
    else direct_group<16>(a, dr, first, lds);
}

template <int PASS>
__global__ __launch_bounds__(256) void k_bv_direct_big(BvDirectArgs b)
{
    direct_big<FoldPlane>(b, [&](int d) { return bv_direct_args<PASS>(b, b.views[b.draws[d].view]); });
}

// The shadow targets of every view, and the pass's counters zeroed.
__global__ __launch_bounds__(256) void k_bv_direct_shadow(BvDirectArgs b, const uint8_t *__restrict__ sblk_view,
                                                          const float *__restrict__ ndc_z, float *__restrict__ depth,
                                                          float *__restrict__ shadow)
{
    const int blk = chunk_remap(blockIdx.x, gridDim.x);
    const DevView &v = b.views[__builtin_amdgcn_readfirstlane(sblk_view[blk])];
    int x, y;
    block_px<32>((int)(blk - v.sblk_base), (v.S + 3) / 4, x, y);
    if (x >= v.S || y >= v.S) return;
    const size_t i = (size_t)x + (size_t)y * v.S;
    const Winner w = direct_winner(b.draws + v.draw_base[kBvShadow], v.n_draws, b.key + v.spx_off, nullptr, b.screen, v.S, v.S,
                                   i, x, y);
    float z = 0.f;
    if (w.g >= 0) z = dot3(vec3(ndc_z[w.tv.x], ndc_z[w.tv.y], ndc_z[w.tv.z]), w.b) * 0.5f + 0.5f;
    depth[v.spx_off + i] = w.depth;
    shadow[v.spx_off + i] = z;
    if (blockIdx.x == 0 && threadIdx.x == 0) *b.ctr = DirectCtr{0ull, 0u, 0u};
}

// Pixel (x, y) of this thread in the view that owns its 64 x 4 block; false when it is
// outside the view.
template <int WT>
__device__ __forceinline__ bool bv_pixel(const BvPixelArgs &a, int &vi, int &x, int &y)
{
    const int blk = chunk_remap(blockIdx.x, gridDim.x);
    vi = __builtin_amdgcn_readfirstlane(a.blk_view[blk]);
    const DevView &v = a.views[vi];
    block_px<WT>((int)(blk - v.blk_base), (v.H + 3) / 4, x, y);
    return x < v.W && y < v.H;
}

template <bool DIRECT>
__global__ __launch_bounds__(256) void k_bv_gbuffer(BvPixelArgs b)
{
    int vi, x, y;
    if (!bv_pixel<32>(b, vi, x, y)) return;
    const DevView &v = b.views[vi];
    ResolveArgs a;
    a.draws = DIRECT ? b.draws + v.draw_base[kBvMain] : b.draws;
    a.n_draws = v.n_draws;
    a.screen = b.screen;
    a.tri_v = b.tri_v;
    a.vary = b.vary;
    a.vis = b.vis + v.px_off;
    a.key = DIRECT ? const_cast<unsigned long long *>(b.key) + v.px_off : nullptr;
    a.fix = nullptr;
    a.depth = DIRECT ? b.depth + v.px_off : nullptr;
    a.W = v.W;
    a.H = v.H;
    a.fresh = 1;
    a.clear[0] = a.clear[1] = a.clear[2] = 0.f;
    a.gbuf = b.gbuf + kGbufPlanes * v.px_off;
    a.fb = nullptr;
    a.materials = b.materials;
    a.textures = b.textures;
    a.shadow_map = nullptr;
    a.ss = ShadowSamples{};
    if (DIRECT && v.corner) gbuffer_px<DIRECT, DIRECT>(a, v.u, x, y);
    else gbuffer_px<DIRECT, false>(a, v.u, x, y);
    // last: a store before them would keep the loads above from their scalar form
    if (DIRECT && blockIdx.x == 0 && threadIdx.x == 0) *b.ctr = DirectCtr{0ull, 0u, 0u};
}

// MODE: the shadow filter of every view, or -1.
template <int MODE>
__global__ __launch_bounds__(256) void k_bv_lighting(BvPixelArgs b)
{
    int vi, x, y;
    if (!bv_pixel<16>(b, vi, x, y)) return;
    const DevView &v = b.views[vi];
    const ShadowSamples none = {};
    lighting_px<false, MODE>(v.u, b.gbuf + kGbufPlanes * v.px_off, b.ao + v.px_off, b.ao_is_one, b.shadow + v.spx_off, none,
                b.fb + 3 * v.px_off, x, y);
}

__global__ __launch_bounds__(256) void k_bv_resolve(BvPixelArgs b)
{
    int vi, x, y;
    if (!bv_pixel<32>(b, vi, x, y)) return;
    const DevView &v = b.views[vi];
    resolve_px(b.fb + 3 * v.px_off, v.W, v.H, 1, b.img + 3 * v.px_off, x, y);
}

// ---------------- launch wrappers ----------------

static inline unsigned nblk(size_t n, unsigned b) { return (unsigned)((n + b - 1) / b); }

void launch_bv_vertex(int pass, const DevDraw *draws, const DevView *views, const uint2 *blocks, int n_blocks,
                      int4 *screen, float *ndc_z, float4 *vary, hipStream_t s)
{
    if (n_blocks <= 0) return;
    if (pass == kBvShadow)
        hipLaunchKernelGGL(k_bv_vertex<kBvShadow>, dim3(n_blocks), dim3(256), 0, s, draws, views, blocks, screen,
                           ndc_z, vary);
    else
        hipLaunchKernelGGL(k_bv_vertex<kBvMain>, dim3(n_blocks), dim3(256), 0, s, draws, views, blocks, screen,
                           ndc_z, vary);
}

void launch_bv_setup(int pass, const DevDraw *draws, const DevView *views, const uint2 *blocks, int n_blocks,
                     const int4 *screen, int TS, uint2 *rect, uint32_t *count, int4 *tri_v,
                     uint32_t *big_list, uint32_t *big_count, hipStream_t s)
{
    if (n_blocks <= 0) return;
    if (pass == kBvShadow)
        hipLaunchKernelGGL(k_bv_setup<kBvShadow>, dim3(n_blocks), dim3(256), 0, s, draws, views, blocks, screen, TS,
                           rect, count, tri_v, big_list, big_count);
    else
        hipLaunchKernelGGL(k_bv_setup<kBvMain>, dim3(n_blocks), dim3(256), 0, s, draws, views, blocks, screen, TS,
                           rect, count, tri_v, big_list, big_count);
}

void launch_bv_emit(int pass, const BvBinArgs &a, hipStream_t s)
{
    if (a.n_tri <= 0) return;
    // big triangles: a fixed grid strides over the device-side list
    const unsigned big_grid = 1024;
    if (pass == kBvShadow) {
        hipLaunchKernelGGL(k_bv_emit_small<kBvShadow>, dim3(nblk(a.n_tri, 256)), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k_bv_emit_big<kBvShadow>, dim3(big_grid), dim3(256), 0, s, a);
    } else {
        hipLaunchKernelGGL(k_bv_emit_small<kBvMain>, dim3(nblk(a.n_tri, 256)), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k_bv_emit_big<kBvMain>, dim3(big_grid), dim3(256), 0, s, a);
    }
}

void launch_bv_overflow(const uint32_t *total, uint32_t cap, uint32_t *flag, hipStream_t s)
{
    hipLaunchKernelGGL(k_bv_overflow, dim3(1), dim3(64), 0, s, total, cap, flag);
}

template <bool SHADOW>
static void bv_raster_t(int TS, unsigned n_wg, const BvRasterArgs &a, hipStream_t s)
{
    if (TS == 8) hipLaunchKernelGGL((k_bv_raster<8, 64, SHADOW>), dim3(n_wg), dim3(64), 0, s, a);
    else if (TS == 16) hipLaunchKernelGGL((k_bv_raster<16, 256, SHADOW>), dim3(n_wg), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_bv_raster<32, 256, SHADOW>), dim3(n_wg), dim3(256), 0, s, a);
}

void launch_bv_raster(int pass, int TS, unsigned n_wg, const BvRasterArgs &a, hipStream_t s)
{
    if (a.n_items == 0 || n_wg == 0) return;
    if (pass == kBvShadow) bv_raster_t<true>(TS, n_wg, a, s);
    else bv_raster_t<false>(TS, n_wg, a, s);
}

void launch_bv_direct_vertex(int pass, const BvDirectArgs &a, const uint2 *vblocks, int n_vblocks, int4 *screen,
                             float *ndc_z, float4 *vary, size_t n_keys, uint32_t *flags, hipStream_t s)
{
    const unsigned grid = (unsigned)(n_vblocks + clear_blocks((long long)n_keys));
    if (grid == 0) return;
    if (pass == kBvShadow)
        hipLaunchKernelGGL(k_bv_direct_vertex<kBvShadow>, dim3(grid), dim3(256), 0, s, a, vblocks, n_vblocks, screen, ndc_z,
                           vary, n_keys, flags);
    else
        hipLaunchKernelGGL(k_bv_direct_vertex<kBvMain>, dim3(grid), dim3(256), 0, s, a, vblocks, n_vblocks, screen, ndc_z,
                           vary, n_keys, flags);
}

void launch_bv_direct(int pass, const BvDirectArgs &a, const uint2 *fblocks, int n_fblocks, hipStream_t s)
{
    if (n_fblocks <= 0) return;
    const unsigned big_grid = 1024;
    if (pass == kBvShadow) {
        hipLaunchKernelGGL(k_bv_direct<kBvShadow>, dim3(n_fblocks), dim3(256), 0, s, a, fblocks);
        hipLaunchKernelGGL(k_bv_direct_big<kBvShadow>, dim3(big_grid), dim3(256), 0, s, a);
    } else {
        hipLaunchKernelGGL(k_bv_direct<kBvMain>, dim3(n_fblocks), dim3(256), 0, s, a, fblocks);
        hipLaunchKernelGGL(k_bv_direct_big<kBvMain>, dim3(big_grid), dim3(256), 0, s, a);
    }
}

void launch_bv_direct_shadow(const BvDirectArgs &a, const uint8_t *sblk_view, uint32_t n_sblocks, const float *ndc_z,
                             float *depth, float *shadow, hipStream_t s)
{
    if (n_sblocks) hipLaunchKernelGGL(k_bv_direct_shadow, dim3(n_sblocks), dim3(256), 0, s, a, sblk_view, ndc_z, depth, shadow);
}

void launch_bv_gbuffer(const BvPixelArgs &a, hipStream_t s)
{
    if (!a.n_blocks) return;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(a.n_blocks), dim3(256), 0, s, a); };
    if (a.key) go(k_bv_gbuffer<true>);
    else go(k_bv_gbuffer<false>);
}

void launch_bv_lighting(const BvPixelArgs &a, int mode, hipStream_t s)
{
    if (!a.n_blocks) return;
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(a.n_blocks), dim3(256), 0, s, a); };
    switch (mode) {
    case 0: return go(k_bv_lighting<0>);
    case 1: return go(k_bv_lighting<1>);
    case 2: return go(k_bv_lighting<2>);
    case 3: return go(k_bv_lighting<3>);
    default: return go(k_bv_lighting<-1>);
    }
}

void launch_bv_resolve(const BvPixelArgs &a, hipStream_t s)
{
    if (a.n_blocks) hipLaunchKernelGGL(k_bv_resolve, dim3(a.n_blocks), dim3(256), 0, s, a);
}

}  // namespace fgl
