// raster_core.hpp -- per-vertex, per-triangle, per-tile and per-pixel bodies
// of the raster pipeline, shared by the single-view kernels (raster.hip) and
// the batched multi-view kernels (batch.hip), so both run the same
// arithmetic.
//
// Exactness: coverage is the reference's Barycentric (src/geometry.cpp:20-56).
// When every window coordinate satisfies |X|,|Y| <= 8191 the FP32 differences
// and FP64 cross products are exact integers, so they are computed in int32
// and only u = cx*inv, v = cy*inv, 1-(u+v) run in FP64 -- the same doubles.
// Otherwise the literal FP32/FP64 sequence runs.
#pragma once

#include "fgl_kernels.hpp"

namespace fgl {

constexpr int kExactLimit = 8191;

// Window coordinates of one vertex: Viewport * NDC with all four terms of
// each row, truncated like x86 cvttss2si (src/forkergl.cpp:244-249).
__device__ __forceinline__ int4 to_screen(const float *vp, Vec4 ndc)
{
    Vec4 c = mv4(vp, ndc);
    int X = trunc_int(c.x), Y = trunc_int(c.y);
    int exact = (X >= -kExactLimit && X <= kExactLimit && Y >= -kExactLimit && Y <= kExactLimit);
    return make_int4(X, Y, __float_as_int(c.z), exact);
}

// BoundBox::GenerateBoundBox (src/forkergl.cpp:145-163)
__device__ __forceinline__ void clamped_bbox(int4 a, int4 b, int4 c, int W, int H, int &minx,
                                             int &miny, int &maxx, int &maxy)
{
    minx = clampi(imin(a.x, imin(b.x, c.x)), 0, W - 1);
    miny = clampi(imin(a.y, imin(b.y, c.y)), 0, H - 1);
    maxx = clampi(imax(a.x, imax(b.x, c.x)), 0, W - 1);
    maxy = clampi(imax(a.y, imax(b.y, c.y)), 0, H - 1);
}

// Cross-product z of Barycentric, which does not depend on the pixel:
// |cz| > 1e-2 decides whether the triangle can cover anything.
__device__ __forceinline__ bool nondegenerate_general(int4 a, int4 b, int4 c)
{
    float Ax = (float)a.x, Ay = (float)a.y, Bx = (float)b.x, By = (float)b.y;
    float Cx = (float)c.x, Cy = (float)c.y;
    double s0x = (double)(Bx - Ax), s0y = (double)(Cx - Ax);
    double s1x = (double)(By - Ay), s1y = (double)(Cy - Ay);
    double uz = s0x * s1y - s0y * s1x;
    return fabs(uz) > 1e-2;
}

// Whether a triangle can cover a pixel of the W x H screen: not degenerate
// and, in the exact regime, not off the screen.
__device__ __forceinline__ bool keep_tri(int4 a, int4 b, int4 c, int W, int H)
{
    if (a.w && b.w && c.w && W <= 8192 && H <= 8192) {
        int cz = (b.x - a.x) * (c.y - a.y) - (c.x - a.x) * (b.y - a.y);
        int ux0 = imin(a.x, imin(b.x, c.x)), ux1 = imax(a.x, imax(b.x, c.x));
        int uy0 = imin(a.y, imin(b.y, c.y)), uy1 = imax(a.y, imax(b.y, c.y));
        // Every clamped-bbox pixel of an off-screen triangle lies strictly
        // outside it, and in the exact regime one computed weight is then
        // strictly negative: nothing can be covered.
        return cz != 0 && !(ux1 < 0 || ux0 > W - 1 || uy1 < 0 || uy0 > H - 1);
    }
    return nondegenerate_general(a, b, c);
}

// Triangle setup of face f of draw d (pass-wide triangle id g): clamped
// bbox, degenerate / off-screen cull, screen-tile rectangle and count.
__device__ __forceinline__ void setup_tri(const DevDraw &dr, int d, int f,
                                          const int4 *__restrict__ screen, int W, int H, int TS,
                                          uint2 *__restrict__ rect, uint32_t *__restrict__ count,
                                          int4 *__restrict__ tri_v,
                                          uint32_t *__restrict__ big_list,
                                          uint32_t *__restrict__ big_count)
{
    const int g = dr.tri_base + f;
    const int v0 = dr.vert_base + dr.vi[3 * f], v1 = dr.vert_base + dr.vi[3 * f + 1];
    const int v2 = dr.vert_base + dr.vi[3 * f + 2];
    const int4 a = screen[v0], b = screen[v1], c = screen[v2];
    int minx, miny, maxx, maxy;
    clamped_bbox(a, b, c, W, H, minx, miny, maxx, maxy);
    const bool keep = keep_tri(a, b, c, W, H);
    const uint32_t tx0 = minx / TS, tx1 = maxx / TS, ty0 = miny / TS, ty1 = maxy / TS;
    const uint32_t n = keep ? (tx1 - tx0 + 1) * (ty1 - ty0 + 1) : 0u;
    rect[g] = make_uint2(tx0 | (tx1 << 16), ty0 | (ty1 << 16));
    count[g] = n;
    tri_v[g] = make_int4(v0, v1, v2, d);
    // The big-triangle list only decides which workgroup writes a triangle's
    // pairs; their positions come from the scan, so its order is irrelevant.
    if (n > (uint32_t)kSmallTriTiles) big_list[atomicAdd(big_count, 1u)] = (uint32_t)g;
}

// Pair j of triangle t: key = tile_base + tile index, row-major over the
// triangle's tile rectangle.
__device__ __forceinline__ uint32_t pair_key(uint2 r, uint32_t j, int tiles_x, uint32_t tile_base)
{
    const uint32_t tx0 = r.x & 0xffff, tx1 = r.x >> 16, ty0 = r.y & 0xffff;
    const uint32_t wx = tx1 - tx0 + 1;
    return tile_base + (ty0 + j / wx) * (uint32_t)tiles_x + tx0 + j % wx;
}

// Per-triangle record of the rasteriser (registers; staged in LDS as TriSoA).
struct TriL {
    int X0, Y0;
    // exact: B-A, C-A as s0x = Bx-Ax, s0y = Cx-Ax, s1x = By-Ay, s1y = Cy-Ay;
    // otherwise the other two vertices X1, Y1, X2, Y2
    int q0, q1, q2, q3;
    float z0, z1, z2;
    int bb0, bb1;            // minx | miny << 16, maxx | maxy << 16
    int cz;                  // exact cross product z
    int exact;
    int g;
    double inv;              // 1.0 / cz (exact regime)
};

__device__ __forceinline__ void stage_tri(TriL &t, int g, int4 a, int4 b, int4 c, int W, int H)
{
    t.X0 = a.x; t.Y0 = a.y;
    t.z0 = __int_as_float(a.z); t.z1 = __int_as_float(b.z); t.z2 = __int_as_float(c.z);
    int minx, miny, maxx, maxy;
    clamped_bbox(a, b, c, W, H, minx, miny, maxx, maxy);
    t.bb0 = minx | (miny << 16);
    t.bb1 = maxx | (maxy << 16);
    t.exact = a.w && b.w && c.w && W <= 8192 && H <= 8192;
    t.g = g;
    if (t.exact) {
        t.q0 = b.x - a.x; t.q1 = c.x - a.x; t.q2 = b.y - a.y; t.q3 = c.y - a.y;
        t.cz = t.q0 * t.q3 - t.q1 * t.q2;
        t.inv = 1.0 / (double)t.cz;
    } else {
        t.q0 = b.x; t.q1 = b.y; t.q2 = c.x; t.q3 = c.y;
        t.cz = 0;
        t.inv = 0.0;
    }
}

// Coverage of pixel (px,py) by a staged triangle; on success the three
// barycentric weights exactly as Barycentric returns them.
__device__ __forceinline__ bool cover(const TriL &t, int px, int py, float &b0, float &b1, float &b2)
{
    if (t.exact) {
        int s0z = t.X0 - px, s1z = t.Y0 - py;
        int cx = t.q1 * s1z - s0z * t.q3;    // s0y * s1z - s0z * s1y
        int cy = s0z * t.q2 - t.q0 * s1z;    // s0z * s1x - s0x * s1z
        // exact sign pre-test: weights cx/cz, cy/cz and (cz-cx-cy)/cz
        if (t.cz > 0) {
            if (cx < 0 || cy < 0 || cx + cy > t.cz) return false;
        } else {
            if (cx > 0 || cy > 0 || cx + cy < t.cz) return false;
        }
        double u = (double)cx * t.inv, v = (double)cy * t.inv;
        float r0 = (float)(1.0 - (u + v)), r1 = (float)u, r2 = (float)v;
        if (r0 < 0.f || r1 < 0.f || r2 < 0.f) return false;
        b0 = r0; b1 = r1; b2 = r2;
        return true;
    }
    return barycentric_ref(t.X0, t.Y0, t.q0, t.q1, t.q2, t.q3, px, py, &b0, &b1, &b2);
}

// XCD-aware tile order: workgroups are dealt round-robin to the 8 XCDs, so
// give each XCD a contiguous run of tiles (neighbouring tiles share
// triangles and vertex data in that XCD's L2).
__device__ __forceinline__ int xcd_remap(int bid, int n)
{
    const int X = 8;
    int per = n / X, rem = n % X;
    int xcd = bid % X, local = bid / X;
    int start = xcd * per + imin(xcd, rem);
    return start + local;
}

// ---------------- order-independent tile rasteriser ----------------
//
// The submission-order depth fold of src/forkergl.cpp:180-199 -- replace when
// !(d >= best), fragments in increasing pass-wide id g -- is reproduced
// without any order:
//  * no NaN involved: the winner is the lowest g among fragments of minimum
//    depth (-0 == +0), or the initial value if it is not beaten: a minimum
//    over 64-bit keys (order(depth) << 32 | g + 1), initial value g + 1 = 0;
//  * a NaN fragment always replaces, and whatever follows a NaN replaces it:
//    with J the highest g of a NaN fragment at the pixel, the winner is the
//    key minimum over the fragments with g > J (the initial value excluded),
//    or J itself when there are none;
//  * a NaN initial depth with no NaN fragment: the key minimum over all
//    fragments (the initial value excluded), or the initial value.
// So any lane can fold any triangle into any pixel with LDS atomics, and the
// tile's triangle list needs no particular order.  Triangles whose bbox
// covers at most kSmallTriArea pixels of the tile are rasterised one per lane
// (the common case for dense meshes, where a wave-per-triangle walk would
// leave most lanes idle); larger ones one per wave, a lane per pixel.  Tiles
// with a NaN run the fragment walk a second time for the affected pixels.

constexpr int kSmallTriArea = 16;

// Monotone map of float depth to uint32 with -0 == +0.
__device__ __forceinline__ uint32_t depth_order(float d)
{
    const uint32_t u = __float_as_uint(d == 0.f ? 0.f : d);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float depth_from_order(uint32_t k)
{
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// The staged triangles of a chunk, one array per field: lanes reading
// consecutive triangles hit consecutive banks (an array of 64- or 80-byte
// records puts 8 to 32 lanes on one bank).
template <int BLOCK>
struct TriSoA {
    int X0[BLOCK], Y0[BLOCK], q0[BLOCK], q1[BLOCK], q2[BLOCK], q3[BLOCK];
    float z0[BLOCK], z1[BLOCK], z2[BLOCK];
    int bb0[BLOCK], bb1[BLOCK], cz[BLOCK], exact[BLOCK], g[BLOCK];
    double inv[BLOCK];
    __device__ __forceinline__ void put(int i, const TriL &t)
    {
        X0[i] = t.X0; Y0[i] = t.Y0; q0[i] = t.q0; q1[i] = t.q1; q2[i] = t.q2; q3[i] = t.q3;
        z0[i] = t.z0; z1[i] = t.z1; z2[i] = t.z2;
        bb0[i] = t.bb0; bb1[i] = t.bb1; cz[i] = t.cz; exact[i] = t.exact; g[i] = t.g;
        inv[i] = t.inv;
    }
    __device__ __forceinline__ TriL get(int i) const
    {
        TriL t;
        t.X0 = X0[i]; t.Y0 = Y0[i]; t.q0 = q0[i]; t.q1 = q1[i]; t.q2 = q2[i]; t.q3 = q3[i];
        t.z0 = z0[i]; t.z1 = z1[i]; t.z2 = z2[i];
        t.bb0 = bb0[i]; t.bb1 = bb1[i]; t.cz = cz[i]; t.exact = exact[i]; t.g = g[i];
        t.inv = inv[i];
        return t;
    }
};

template <int TS, int BLOCK>
struct RasterLds {
    TriSoA<BLOCK> tri;
    unsigned long long key[TS * TS];
    int nan_g[TS * TS];       // highest id of a NaN fragment, -1 if none
    uint8_t nan_init[TS * TS];
    int nan_seen;
};

// Depth of staged triangle t at a covered pixel: Dot(bary, depths) in the
// reference's order.
__device__ __forceinline__ float tri_depth(const TriL &t, float b0, float b1, float b2)
{
    float dd = 0.f;
    dd += b0 * t.z0;
    dd += b1 * t.z1;
    dd += b2 * t.z2;
    return dd;
}

// One walk over the tile's triangles.  PASS 0: every fragment; PASS 1 (NaN
// tiles): only pixels touched by a NaN, only fragments after their last NaN.
template <int TS, int BLOCK, int PASS>
__device__ __forceinline__ void raster_walk(const RasterArgs &a, int tile, RasterLds<TS, BLOCK> &L)
{
    constexpr int NW = BLOCK / 64;
    constexpr int QS = (NW == 1) ? TS : TS / 2;
    constexpr int NPX = QS * QS / 64;
    const int tx = tile % a.tiles_x, ty = tile / a.tiles_x;
    const int x0 = tx * TS, y0 = ty * TS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int qx0 = x0 + (NW == 1 ? 0 : (wave & 1) * QS);
    const int qy0 = y0 + (NW == 1 ? 0 : (wave >> 1) * QS);
    const int rx1 = qx0 + QS - 1, ry1 = qy0 + QS - 1;
    const uint32_t start = a.tile_start[tile], end = a.tile_end[tile];
    auto fold = [&](const TriL &t, int px, int py, float dd) {
        const int p = (py - y0) * TS + (px - x0);
        if (PASS == 0) {
            if (dd != dd) {
                atomicMax(&L.nan_g[p], t.g);
                L.nan_seen = 1;
                return;
            }
        } else {
            const int j = L.nan_g[p];
            if (!(j >= 0 || L.nan_init[p]) || t.g <= j || dd != dd) return;
        }
        atomicMin(&L.key[p], ((unsigned long long)depth_order(dd) << 32) | (unsigned long long)(uint32_t)(t.g + 1));
    };
    for (uint32_t base = start; base < end; base += BLOCK) {
        const int n = imin(BLOCK, (int)(end - base));
        __syncthreads();   // previous chunk's triangles fully consumed
        if (tid < n) {
            const int g = (int)a.vals[base + tid];
            const int4 tv = a.tri_v[g];
            TriL t;
            stage_tri(t, g, a.screen[tv.x], a.screen[tv.y], a.screen[tv.z], a.W, a.H);
            L.tri.put(tid, t);
        }
        __syncthreads();
        // small triangles: one per lane
        if (tid < n) {
            const TriL t = L.tri.get(tid);
            const int bx0 = imax(t.bb0 & 0xffff, x0), bx1 = imin(t.bb1 & 0xffff, x0 + TS - 1);
            const int by0 = imax(t.bb0 >> 16, y0), by1 = imin(t.bb1 >> 16, y0 + TS - 1);
            const int area = (bx1 >= bx0 && by1 >= by0) ? (bx1 - bx0 + 1) * (by1 - by0 + 1) : 0;
            if (area > 0 && area <= kSmallTriArea) {
                for (int py = by0; py <= by1; ++py)
                    for (int px = bx0; px <= bx1; ++px) {
                        float b0, b1, b2;
                        if (cover(t, px, py, b0, b1, b2)) fold(t, px, py, tri_depth(t, b0, b1, b2));
                    }
            }
        }
        // large triangles: one per wave over its quadrant, a lane per pixel
        unsigned long long mask[NW];
#pragma unroll
        for (int jj = 0; jj < NW; ++jj) {
            const int si = jj * 64 + lane;
            bool hit = false;
            if (si < n) {
                const int bb0 = L.tri.bb0[si], bb1 = L.tri.bb1[si];
                const int minx = bb0 & 0xffff, miny = bb0 >> 16;
                const int maxx = bb1 & 0xffff, maxy = bb1 >> 16;
                const int bx0 = imax(minx, x0), bx1 = imin(maxx, x0 + TS - 1);
                const int by0 = imax(miny, y0), by1 = imin(maxy, y0 + TS - 1);
                const int area = (bx1 >= bx0 && by1 >= by0) ? (bx1 - bx0 + 1) * (by1 - by0 + 1) : 0;
                hit = area > kSmallTriArea && !(maxx < qx0 || minx > rx1 || maxy < qy0 || miny > ry1);
            }
            mask[jj] = __ballot(hit);
        }
#pragma unroll
        for (int jj = 0; jj < NW; ++jj) {
            unsigned long long m = mask[jj];
            while (m) {
                const int i = jj * 64 + __builtin_ctzll(m);
                m &= m - 1;
                const TriL t = L.tri.get(i);
                const int minx = t.bb0 & 0xffff, miny = t.bb0 >> 16;
                const int maxx = t.bb1 & 0xffff, maxy = t.bb1 >> 16;
#pragma unroll
                for (int k = 0; k < NPX; ++k) {
                    const int lin = lane + 64 * k;
                    const int px = qx0 + lin % QS, py = qy0 + lin / QS;
                    if (px < a.W && py < a.H && px >= minx && px <= maxx && py >= miny && py <= maxy) {
                        float b0, b1, b2;
                        if (cover(t, px, py, b0, b1, b2)) fold(t, px, py, tri_depth(t, b0, b1, b2));
                    }
                }
            }
        }
    }
    __syncthreads();
}

template <int TS, int BLOCK, bool SHADOW>
__device__ __forceinline__ void raster_tile(const RasterArgs &a, int tile, RasterLds<TS, BLOCK> &L)
{
    const int tx = tile % a.tiles_x, ty = tile / a.tiles_x;
    const int x0 = tx * TS, y0 = ty * TS;
    const int tid = threadIdx.x;
    if (tid == 0) L.nan_seen = 0;
    __syncthreads();
    for (int p = tid; p < TS * TS; p += BLOCK) {
        const int px = x0 + p % TS, py = y0 + p / TS;
        float init = 3.40282347e+38f;
        if (!a.fresh && px < a.W && py < a.H) init = a.depth[(size_t)px + (size_t)py * a.W];
        const bool ni = init != init;
        if (ni) L.nan_seen = 1;
        L.nan_init[p] = ni ? 1 : 0;
        L.nan_g[p] = -1;
        L.key[p] = ni ? ~0ull : (unsigned long long)depth_order(init) << 32;
    }
    raster_walk<TS, BLOCK, 0>(a, tile, L);   // ends with a barrier
    if (L.nan_seen) {
        for (int p = tid; p < TS * TS; p += BLOCK)
            if (L.nan_g[p] >= 0 || L.nan_init[p]) L.key[p] = ~0ull;
        raster_walk<TS, BLOCK, 1>(a, tile, L);
    }
    for (int p = tid; p < TS * TS; p += BLOCK) {
        const int px = x0 + p % TS, py = y0 + p / TS;
        if (px >= a.W || py >= a.H) continue;
        const size_t i = (size_t)px + (size_t)py * a.W;
        const unsigned long long key = L.key[p];
        int win = key == ~0ull ? -1 : (int)(uint32_t)(key & 0xffffffffu) - 1;
        bool from_key = win >= 0;
        if (!from_key && L.nan_g[p] >= 0) win = L.nan_g[p];   // nothing after the last NaN fragment
        if (win >= 0) {
            float dd = from_key ? depth_from_order((uint32_t)(key >> 32)) : 0.f;
            TriL t;
            float b0 = 0.f, b1 = 0.f, b2 = 0.f;
            const int4 tv = a.tri_v[win];
            if (!from_key || dd == 0.f || SHADOW) {
                stage_tri(t, win, a.screen[tv.x], a.screen[tv.y], a.screen[tv.z], a.W, a.H);
                cover(t, px, py, b0, b1, b2);
                if (!from_key || dd == 0.f) dd = tri_depth(t, b0, b1, b2);   // NaN, or a zero with its sign
            }
            a.depth[i] = dd;
            if (!SHADOW) {
                a.vis[i] = win;
            } else {
                // DepthShader::ProcessFragment (depthshader.h:30-36), with
                // the vertices' NDC z as the vertex pass computed them
                float z = dot3(vec3(a.ndc_z[tv.x], a.ndc_z[tv.y], a.ndc_z[tv.z]), vec3(b0, b1, b2));
                a.shadow_out[i] = z * 0.5f + 0.5f;
            }
        } else {
            if (a.fresh) a.depth[i] = 3.40282347e+38f;
            if (!SHADOW) a.vis[i] = -1;
            else if (a.fresh) a.shadow_out[i] = 0.f;
        }
    }
}

// ---------------- direct rasteriser ----------------
//
// A pass that starts from cleared targets needs no tile lists: the depth
// fold is a minimum over keys, so workgroups fold their triangles' fragments
// into a plane of 64-bit keys in HBM with device-scope atomic minima, and the
// resolve reads each pixel's key.
//
// A workgroup takes 256 / G neighbouring triangles (the model's faces in
// spatial order, fgl_upload_model) and folds them in LDS over the box of
// pixels they share, then folds the box's pixels into the plane, neighbouring
// lanes neighbouring pixels.  What bounds the fold is the atomics' memory
// traffic -- one by one, in the faces' own order, each fetched and wrote back
// a cache line (5.2 M triangles at 3840 x 2160: 668 us for the main pass, 137
// without the atomics) -- and a box touches each of its lines once (205 us,
// of which the items below take a quarter; the tile lists' own setup, scan,
// emit, sort, ranges and rasteriser took 515).  A box of more than kDirectBox pixels folds straight into the plane: its
// triangles are large, their own rows of pixels neighbours.
//
// kDirectBig bounds what one triangle costs the lanes that own it: a larger
// one goes to a list, and the wavefronts of k_direct_big share out its items of
// 64 x 16 pixels.  The list has room for every triangle of the pass: what does
// not go there is never more than kDirectBig pixels of one wavefront.
//
// NaN depths (a vertex on the camera plane) follow the rule above in two
// more steps: the first walk marks the pixel with the NaN fragment's id --
// high word 0, below every real depth's -- and the mark with the highest id
// is the minimum; k_direct_nan, which returns at once unless a mark was made,
// walks the triangles and the items again and folds the fragments after the mark into a
// second plane (all ones between passes: the resolve puts back what it
// read).  A pass whose vertices the host has shown to have finite depths
// (context.cpp, bound_pass) has neither that plane nor that walk.
constexpr unsigned long long kDirectClear = 0xff7fffffull << 32;   // depth_order(FLT_MAX), no fragment
constexpr int kDirectItemW = 64, kDirectItemH = 16;
constexpr int kDirectBig = 4096;      // pixels of the bounding box
constexpr int kDirectBox = 2048;      // pixels of a workgroup's LDS box: 16 KiB; a CU's 32 wavefronts are eight workgroups

// The last of n ascending starts (start[0] is 0) that is at most i, by whole
// wavefronts, 64 probes a step.  Of owners with nothing of their own the last
// one of equal starts, which owns i, is found.
template <typename T>
__device__ __forceinline__ uint32_t owner_of(const T *start, uint32_t n, T i)
{
    const uint32_t lane = threadIdx.x & 63;
    uint32_t lo = 0, len = n;
    while (len > 1) {
        const uint32_t step = (len + 63) / 64, at = lane * step;
        const unsigned long long le = __ballot(at < len && start[lo + (at < len ? at : 0u)] <= i);
        const uint32_t k = (uint32_t)__popcll(le) - 1u;
        lo += k * step;
        len = len - k * step < step ? len - k * step : step;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// The draw of workgroup b and the workgroups before the draw's.
__device__ __forceinline__ int draw_of_group(const DrawStarts &s, int n_draws, int b, int &before)
{
    if (n_draws > kFewDraws) {
        const int d = (int)owner_of(s.table, (uint32_t)n_draws, b);
        before = s.table[d];
        return d;
    }
    int d = 0;
    before = 0;
#pragma unroll
    for (int k = 1; k < kFewDraws; ++k)
        if (s.few[k] <= b) {
            d = k;
            before = s.few[k];
        }
    return d;
}

// The draw of pass-wide triangle g (their tri_base ascend).
__device__ __forceinline__ int draw_of(const DevDraw *draws, int n_draws, int g)
{
    int lo = 0, hi = n_draws - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (draws[mid].tri_base <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

struct DirectLds {
    unsigned long long key[kDirectBox];
    uint32_t lo[4], hi[4];            // per wavefront: (min x | min y << 16), the complement of the maxima
};

// A fragment's key; a NaN depth's is its mark.
__device__ __forceinline__ unsigned long long direct_key(const DirectArgs &a, const TriL &t, float dd)
{
    if (dd != dd) {
        a.ctr->nan = 1u;
        return (unsigned long long)(uint32_t)~(uint32_t)t.g;
    }
    return ((unsigned long long)depth_order(dd) << 32) | (unsigned long long)(uint32_t)(t.g + 1);
}

__device__ __forceinline__ void direct_min(unsigned long long *key, unsigned long long k)
{
    (void)__hip_atomic_fetch_min(key, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Where a walk's fragments go (wants: whether any fragment of an item's column
// px, rows py to y1, can change it): the key plane,
struct FoldPlane {
    const DirectArgs &a;
    __device__ __forceinline__ bool wants(int, int, int) const { return true; }
    __device__ __forceinline__ void operator()(const TriL &t, int px, int py, float dd) const
    {
        direct_min(a.key + (size_t)px + (size_t)py * a.W, direct_key(a, t, dd));
    }
    // of an item: not where the plane held a smaller key already (keys only fall)
    __device__ __forceinline__ unsigned long long held(int px, int py) const { return a.key[(size_t)px + (size_t)py * a.W]; }
    __device__ __forceinline__ void operator()(const TriL &t, int px, int py, float dd, unsigned long long held) const
    {
        const unsigned long long k = direct_key(a, t, dd);
        if (k < held) direct_min(a.key + (size_t)px + (size_t)py * a.W, k);
    }
};

// the workgroup's box in LDS (w pixels wide, its corner at (x0, y0)),
struct FoldBox {
    const DirectArgs &a;
    DirectLds &L;
    int x0, y0, w;
    __device__ __forceinline__ void operator()(const TriL &t, int px, int py, float dd) const
    {
        atomicMin(&L.key[(px - x0) + (py - y0) * w], direct_key(a, t, dd));
    }
};

// or, in the second walk of a pass with NaN marks, the second plane: the
// fragments after the pixel's mark.
struct FoldAfterNan {
    const DirectArgs &a;
    // few pixels are marked, and the keys of a column load together
    __device__ __forceinline__ bool wants(int px, int py, int y1) const
    {
        bool any = false;
#pragma unroll
        for (int e = 0; e < kDirectItemH; ++e) {
            const int y = py + e < y1 ? py + e : y1 - 1;
            any = any || (a.key[(size_t)px + (size_t)y * a.W] >> 32) == 0ull;
        }
        return any;
    }
    __device__ __forceinline__ void operator()(const TriL &t, int px, int py, float dd) const
    {
        const size_t i = (size_t)px + (size_t)py * a.W;
        const unsigned long long m = a.key[i];
        if ((m >> 32) != 0ull || dd != dd || t.g <= (int)~(uint32_t)m) return;
        direct_min(a.fix + i, ((unsigned long long)depth_order(dd) << 32) | (unsigned long long)(uint32_t)(t.g + 1));
    }
    __device__ __forceinline__ unsigned long long held(int, int) const { return 0ull; }
    __device__ __forceinline__ void operator()(const TriL &t, int px, int py, float dd, unsigned long long) const
    {
        (*this)(t, px, py, dd);
    }
};

// Pixels first, first + step, ... of t's box, row by row: its fragments
// among them to fold.  first < step <= 64.
template <typename Fold>
__device__ __forceinline__ void direct_box(const TriL &t, int first, int step, const Fold &fold)
{
    const int x0 = t.bb0 & 0xffff, y0 = t.bb0 >> 16;
    const int w = (t.bb1 & 0xffff) - x0 + 1, h = (t.bb1 >> 16) - y0 + 1;
    int y = 0, x = 0, sy = 0, sx = 1;
    if (step > 1) {
        // first / w and step / w: at most 64 and off an integer by 0.5 / w or
        // more after the half is added, so the product truncates exactly
        const float inv = __builtin_amdgcn_rcpf((float)w);
        y = (int)(((float)first + 0.5f) * inv);
        x = first - y * w;
        sy = (int)(((float)step + 0.5f) * inv);
        sx = step - sy * w;
    }
    while (y < h) {
        float b0, b1, b2;
        if (cover(t, x0 + x, y0 + y, b0, b1, b2)) fold(t, x0 + x, y0 + y, tri_depth(t, b0, b1, b2));
        x += sx;
        y += sy;
        if (x >= w) {
            x -= w;
            ++y;
        }
    }
}

__device__ __forceinline__ int direct_area(const TriL &t)
{
    return ((t.bb1 & 0xffff) - (t.bb0 & 0xffff) + 1) * ((t.bb1 >> 16) - (t.bb0 >> 16) + 1);
}

// Face number n of draw dr in the model's spatial order, staged; false when
// it covers nothing (degenerate, or off the screen in the exact regime).
__device__ __forceinline__ bool direct_stage(const DirectArgs &a, const DevDraw &dr, int n, TriL &t)
{
    const int4 v = dr.tri[n];
    const int4 p = a.screen[dr.vert_base + v.x], q = a.screen[dr.vert_base + v.y], r = a.screen[dr.vert_base + v.z];
    if (!keep_tri(p, q, r, a.W, a.H)) return false;
    stage_tri(t, dr.tri_base + v.w, p, q, r, a.W, a.H);
    return true;
}

__device__ __forceinline__ TriL direct_lane(const TriL &t, int l)
{
    TriL o;
    o.X0 = __builtin_amdgcn_readlane(t.X0, l);
    o.Y0 = __builtin_amdgcn_readlane(t.Y0, l);
    o.q0 = __builtin_amdgcn_readlane(t.q0, l);
    o.q1 = __builtin_amdgcn_readlane(t.q1, l);
    o.q2 = __builtin_amdgcn_readlane(t.q2, l);
    o.q3 = __builtin_amdgcn_readlane(t.q3, l);
    o.z0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.z0), l));
    o.z1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.z1), l));
    o.z2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.z2), l));
    o.bb0 = __builtin_amdgcn_readlane(t.bb0, l);
    o.bb1 = __builtin_amdgcn_readlane(t.bb1, l);
    o.cz = __builtin_amdgcn_readlane(t.cz, l);
    o.exact = __builtin_amdgcn_readlane(t.exact, l);
    o.g = __builtin_amdgcn_readlane(t.g, l);
    const long long iv = __double_as_longlong(t.inv);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)iv, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(iv >> 32), l);
    o.inv = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    return o;
}

// The wavefront's triangles, G lanes each: a box of up to kSmallTriArea
// pixels a lane stays with its group, the whole wavefront takes a larger one.
template <int G, typename Fold>
__device__ __forceinline__ void direct_walk(const TriL &t, bool keep, int area, const Fold &fold)
{
    const int lane = threadIdx.x & 63, sub = lane % G;
    const bool small = area <= kSmallTriArea * G;
    if (keep && small) direct_box(t, sub, G, fold);
    unsigned long long m = __ballot(keep && !small && sub == 0);
    while (m) {
        const int l = __builtin_ctzll(m);
        m &= m - 1;
        direct_box(direct_lane(t, l), lane, 64, fold);
    }
}

__device__ __forceinline__ unsigned long long lane_u64(unsigned long long v, int l)
{
    return (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l) << 32 |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
}

// Triangles of more than kDirectBig pixels to the list, one claim a wavefront
// (n: the items of this lane's triangle, 0 if it is no such triangle).
__device__ __forceinline__ void direct_claim(const DirectArgs &a, int g, uint32_t n)
{
    const unsigned long long m = __ballot(n != 0u);
    if (!m) return;
    const int lane = threadIdx.x & 63;
    uint32_t inc = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
    unsigned long long at = 0;
    if (lane == 63) at = atomicAdd(&a.ctr->claims, ((unsigned long long)__popcll(m) << kBigShift) | total);
    at = __shfl(at, 63, 64);
    if (n) {
        const size_t p = (size_t)(at >> kBigShift) + __popcll(m & ((1ull << lane) - 1ull));
        a.big_start[p] = (at & ((1ull << kBigShift) - 1ull)) + (inc - n);
        a.big_tri[p] = (uint32_t)g;
    }
}

// A workgroup's 256 / G triangles of draw dr, from number first of its
// spatial order on.
template <int G>
__device__ __forceinline__ void direct_group(const DirectArgs &a, const DevDraw &dr, int first, DirectLds &L)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = first + tid / G;
    TriL t;
    bool keep = n < dr.n_faces && direct_stage(a, dr, n, t);
    int area = keep ? direct_area(t) : 0;
    {
        const int w = keep ? (t.bb1 & 0xffff) - (t.bb0 & 0xffff) + 1 : 0, h = keep ? (t.bb1 >> 16) - (t.bb0 >> 16) + 1 : 0;
        const bool big = area > kDirectBig;
        const uint32_t k = big && lane % G == 0 ? (uint32_t)((w + kDirectItemW - 1) / kDirectItemW) *
                                                      (uint32_t)((h + kDirectItemH - 1) / kDirectItemH) : 0u;
        direct_claim(a, keep ? t.g : 0, k);
        keep = keep && !big;
    }
    // the box of what is left
    typedef unsigned short v2u __attribute__((ext_vector_type(2)));
    v2u lo = {0xffff, 0xffff}, hi = {0xffff, 0xffff};
    if (keep) {
        lo = __builtin_bit_cast(v2u, t.bb0);
        hi = __builtin_bit_cast(v2u, ~t.bb1);
    }
#pragma unroll
    for (int o = G; o < 64; o <<= 1) {
        lo = __builtin_elementwise_min(lo, __builtin_bit_cast(v2u, __shfl_xor(__builtin_bit_cast(int, lo), o, 64)));
        hi = __builtin_elementwise_min(hi, __builtin_bit_cast(v2u, __shfl_xor(__builtin_bit_cast(int, hi), o, 64)));
    }
    if (lane == 0) {
        L.lo[wave] = __builtin_bit_cast(uint32_t, lo);
        L.hi[wave] = __builtin_bit_cast(uint32_t, hi);
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        lo = __builtin_elementwise_min(lo, __builtin_bit_cast(v2u, L.lo[v]));
        hi = __builtin_elementwise_min(hi, __builtin_bit_cast(v2u, L.hi[v]));
    }
    const int x0 = lo.x, y0 = lo.y, w = (int)(uint16_t)~hi.x - x0 + 1, h = (int)(uint16_t)~hi.y - y0 + 1;
    if (lo.x == 0xffff) return;   // nothing kept (a screen is at most 16384 wide)
    if (w * h > kDirectBox) {
        direct_walk<G>(t, keep, area, FoldPlane{a});
        return;
    }
    for (int p = tid; p < w * h; p += 256) L.key[p] = ~0ull;
    __syncthreads();
    direct_walk<G>(t, keep, area, FoldBox{a, L, x0, y0, w});
    __syncthreads();
    for (int p = tid; p < w * h; p += 256) {
        const unsigned long long k = L.key[p];
        const int y = p / w, x = p - y * w;
        if (k != ~0ull) direct_min(a.key + (size_t)(x0 + x) + (size_t)(y0 + y) * a.W, k);
    }
}

// Triangle g staged from its face, and its vertex ids and draw.
__device__ __forceinline__ int4 direct_face(const DevDraw *draws, int d, const int4 *screen, int g, int W, int H, TriL &t)
{
    const DevDraw &dr = draws[d];
    const int f = g - dr.tri_base;
    const int4 tv = make_int4(dr.vert_base + dr.vi[3 * f], dr.vert_base + dr.vi[3 * f + 1],
                              dr.vert_base + dr.vi[3 * f + 2], d);
    stage_tri(t, g, screen[tv.x], screen[tv.y], screen[tv.z], W, H);
    return tv;
}

// Item k of triangle t by one wavefront.  DEEP: where the plane already holds
// a smaller key the atomic is left out.
template <bool DEEP, typename Fold>
__device__ __forceinline__ void direct_item(const TriL &t, int k, const Fold &fold)
{
    const int bx = t.bb0 & 0xffff, by = t.bb0 >> 16, w = (t.bb1 & 0xffff) - bx + 1, h = (t.bb1 >> 16) - by + 1;
    const int nx = (w + kDirectItemW - 1) / kDirectItemW;
    const int ox = k % nx * kDirectItemW, oy = k / nx * kDirectItemH;
    const int x = ox + (int)(threadIdx.x & 63);
    if (x >= w) return;
    const int y1 = imin(oy + kDirectItemH, h);
    if (!fold.wants(bx + x, by + oy, by + y1)) return;
    constexpr int kRows = DEEP ? 4 : 1;   // their keys load together
    for (int y = oy; y < y1; y += kRows) {
        unsigned long long held[kRows];
#pragma unroll
        for (int e = 0; e < kRows; ++e) held[e] = DEEP ? fold.held(bx + x, by + imin(y + e, y1 - 1)) : ~0ull;
#pragma unroll
        for (int e = 0; e < kRows; ++e) {
            float b0, b1, b2;
            if (y + e < y1 && cover(t, bx + x, by + y + e, b0, b1, b2))
                fold(t, bx + x, by + y + e, tri_depth(t, b0, b1, b2), held[e]);
        }
    }
}

// The items of a pass's large triangles shared out to the launch's wavefronts.
// of(d): the arguments of draw d's target.  Where the items cover the targets
// several times over (deep_items, pass_plan.hpp) the fold is bound by the
// atomics' traffic: a key is read before, and a wavefront takes runs of up to 16
// items (one search and one triangle's set-up a run or triangle): 64 full screens
// of 3840 x 2160 2.69 -> 1.02 ms.  With fewer an item's own time counts, to which
// the read would add (640 x 400 frame 102 -> 111 us), and runs would put covered
// items beside covered ones (24 views' shadow maps 81 -> 90).  Up to 64
// triangles' starts are kept in the lanes.
template <typename Fold, typename Args, typename Of>
__device__ __forceinline__ void direct_big(const Args &p, const Of &of)
{
    const unsigned long long claims = p.ctr->claims, n = claims & ((1ull << kBigShift) - 1ull);
    const uint32_t n_big = (uint32_t)(claims >> kBigShift);
    const unsigned long long waves = (unsigned long long)gridDim.x * (blockDim.x >> 6);
    const bool deep = n >= p.deep_from, few = n_big <= 64;
    const unsigned long long rounds = (n + 16 * waves - 1) / (16 * waves);
    const unsigned long long run = deep ? (n + rounds * waves - 1) / (rounds * waves) : 1;
    const uint32_t lane = threadIdx.x & 63;
    const unsigned long long start = few && lane < n_big ? p.big_start[lane] : ~0ull;
    const uint32_t tri = few && lane < n_big ? p.big_tri[lane] : 0u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    for (unsigned long long i = wave * run; i < n; i += waves * run) {
        const unsigned long long end = i + run < n ? i + run : n;
        uint32_t b = few ? (uint32_t)__popcll(__ballot(start <= i)) - 1u : owner_of(p.big_start, n_big, i);
        for (unsigned long long k = i; k < end; ++b) {
            const unsigned long long first = few ? lane_u64(start, b) : p.big_start[b];
            const unsigned long long next = b + 1 >= n_big ? n : few ? lane_u64(start, b + 1) : p.big_start[b + 1];
            const int g = few ? __builtin_amdgcn_readlane((int)tri, b) : (int)p.big_tri[b];
            const int d = draw_of(p.draws, p.n_draws, g);
            const DirectArgs a = of(d);
            TriL t;
            direct_face(a.draws, d, a.screen, g, a.W, a.H, t);
            if (deep)
                for (; k < end && k < next; ++k) direct_item<true>(t, (int)(k - first), Fold{a});
            else
                for (; k < end && k < next; ++k) direct_item<false>(t, (int)(k - first), Fold{a});
        }
    }
}

// A pixel's winner: its triangle (-1: none), vertex ids and draw, weights;
// with the direct rasteriser also its depth as the fold leaves it, and
// whether the pixel has a NaN mark.
struct Winner {
    int g;
    int4 tv;
    Vec3 b;
    float depth;
    bool mark;
};

// The winner of pixel i = (px, py) from its key.  Wavefronts whose winners
// belong to one draw find it once.
__device__ __forceinline__ Winner direct_winner(const DevDraw *draws, int n_draws, const unsigned long long *key,
                                                const unsigned long long *fix, const int4 *screen, int W, int H, size_t i,
                                                int px, int py)
{
    Winner w;
    unsigned long long k = key[i];
    bool nan = false;
    w.mark = (k >> 32) == 0ull && fix;
    if ((k >> 32) == 0ull) {
        const unsigned long long after = fix ? fix[i] : ~0ull;
        nan = after == ~0ull;
        w.g = nan ? (int)~(uint32_t)k : (int)(uint32_t)after - 1;
        k = after;
    } else {
        w.g = (int)(uint32_t)k - 1;
    }
    w.depth = 3.40282347e+38f;
    if (w.g < 0) return w;
    const int d0 = draw_of(draws, n_draws, __builtin_amdgcn_readfirstlane(w.g));
    const int f0 = w.g - draws[d0].tri_base;
    const int d = f0 >= 0 && f0 < draws[d0].n_faces ? d0 : draw_of(draws, n_draws, w.g);
    TriL t;
    w.tv = direct_face(draws, d, screen, w.g, W, H, t);
    w.b = vec3(0.f, 0.f, 0.f);
    cover(t, px, py, w.b.x, w.b.y, w.b.z);
    w.depth = depth_from_order((uint32_t)(k >> 32));
    if (nan || w.depth == 0.f) w.depth = tri_depth(t, w.b.x, w.b.y, w.b.z);   // NaN, or a zero with its sign
    return w;
}

// Barycentric weights of the winning triangle at (px,py), recomputed with the
// same staged arithmetic as the coverage loop.
__device__ __forceinline__ Vec3 winner_bary(const int4 *__restrict__ screen,
                                            const int4 *__restrict__ tri_v, int g, int W, int H,
                                            int px, int py, int4 &tv)
{
    tv = tri_v[g];
    TriL t;
    stage_tri(t, g, screen[tv.x], screen[tv.y], screen[tv.z], W, H);
    float b0 = 0.f, b1 = 0.f, b2 = 0.f;
    cover(t, px, py, b0, b1, b2);
    return vec3(b0, b1, b2);
}

// The winner of pixel i = (x, y), and the end of its resolve: the depth
// target, and the second plane all ones again (last, so that the loads
// between keep their scalar form).
template <bool DIRECT>
__device__ __forceinline__ Winner resolve_winner(const ResolveArgs &a, size_t i, int x, int y)
{
    if (DIRECT) return direct_winner(a.draws, a.n_draws, a.key, a.fix, a.screen, a.W, a.H, i, x, y);
    Winner w;
    w.g = a.vis[i];
    if (w.g >= 0) w.b = winner_bary(a.screen, a.tri_v, w.g, a.W, a.H, x, y, w.tv);
    return w;
}

template <bool DIRECT>
__device__ __forceinline__ void resolve_end(const ResolveArgs &a, size_t i, const Winner &w)
{
    if (!DIRECT) return;
    a.depth[i] = w.depth;
    if (w.mark) a.fix[i] = ~0ull;
}

// GShader::ProcessFragment + the seven buffer writes (gshader.h:95-202,
// forkergl.cpp:211-223) for the winner (face f of draw dr, material m,
// barycentrics b) at pixel i: the 19 G-buffer planes.
template <bool CORNER>
__device__ __forceinline__ void gbuffer_shade(const ResolveArgs &a, const FrameUniforms &u, const DevDraw &dr,
                                              const DevMaterial &m, int f, const int4 &tv, const Vec3 &b, size_t i,
                                              size_t P)
{
    float *gb = a.gbuf;
    Varying v0 = main_vertex<CORNER>(dr, u, a.vary, tv.x, f, 0);
    Varying v1 = main_vertex<CORNER>(dr, u, a.vary, tv.y, f, 1);
    Varying v2 = main_vertex<CORNER>(dr, u, a.vary, tv.z, f, 2);
    const DevBundle &bn = m.bundle[dr.support_pbr ? 1 : 0];
    FragGeom fg = frag_geometry(dr, u, a.textures, v0, v1, v2, b, m.map_bump, bn);
    Vec3 albedo, emissive, param;
    float type;
    if (dr.support_pbr) {
        albedo = (bn.has & kBundleA) ? fg.maps.a
               : m.map_base >= 0     ? tex_sample(a.textures, m.map_base, fg.uv)
                                     : vec3(m.albedo[0], m.albedo[1], m.albedo[2]);
        emissive = m.map_pbr_ke >= 0 ? tex_sample(a.textures, m.map_pbr_ke, fg.uv)
                                     : vec3(m.ke[0], m.ke[1], m.ke[2]);
        float rough = (bn.has & kBundleZ) ? fg.maps.z
                    : m.map_rough >= 0    ? tex_samplef(a.textures, m.map_rough, fg.uv) : m.roughness;
        float metal = (bn.has & kBundleY) ? fg.maps.y
                    : m.map_metal >= 0    ? tex_samplef(a.textures, m.map_metal, fg.uv) : m.metalness;
        float ao = m.map_ao >= 0 ? tex_samplef(a.textures, m.map_ao, fg.uv) : 1.f;
        param = vec3(ao, metal, rough);
        type = 1.f;
    } else {
        emissive = m.map_ke >= 0 ? tex_sample(a.textures, m.map_ke, fg.uv)
                                 : vec3(m.ke[0], m.ke[1], m.ke[2]);
        albedo = (bn.has & kBundleA) ? fg.maps.a
               : m.map_kd >= 0       ? tex_sample(a.textures, m.map_kd, fg.uv)
                                     : vec3(m.kd[0], m.kd[1], m.kd[2]);
        float shin = (bn.has & kBundleZ) ? fg.maps.z + 5
                   : m.map_ks >= 0       ? tex_samplef(a.textures, m.map_ks, fg.uv) + 5 : 1.f;
        param = vec3(1.f, m.ks[0], shin);
        type = 0.f;
    }
    gb[0 * P + i] = fg.normal.x; gb[1 * P + i] = fg.normal.y; gb[2 * P + i] = fg.normal.z;
    gb[3 * P + i] = fg.pos.x; gb[4 * P + i] = fg.pos.y; gb[5 * P + i] = fg.pos.z;
    if (u.shadow_on) {
        gb[6 * P + i] = fg.lndc.x; gb[7 * P + i] = fg.lndc.y; gb[8 * P + i] = fg.lndc.z;
    } else if (a.fresh) {
        gb[6 * P + i] = 0.f; gb[7 * P + i] = 0.f; gb[8 * P + i] = 0.f;
    }
    gb[9 * P + i] = albedo.x; gb[10 * P + i] = albedo.y; gb[11 * P + i] = albedo.z;
    gb[12 * P + i] = emissive.x; gb[13 * P + i] = emissive.y; gb[14 * P + i] = emissive.z;
    gb[15 * P + i] = param.x; gb[16 * P + i] = param.y; gb[17 * P + i] = param.z;
    gb[18 * P + i] = type;
}

// Geometry pass resolve of pixel (x,y); a pixel with no fragment gets the
// cleared values when `fresh`.  When every active lane of the wavefront
// resolves a face of the same draw with the same material (the common case:
// neighbouring pixels show the same mesh), the draw and material records are
// addressed through readfirstlane, so their fields (matrices, flags, texture
// descriptors) come in as scalar loads instead of one vector load per field.
// DIRECT: winners come from the direct rasteriser's keys, and the depth
// target is written here.
template <bool DIRECT, bool CORNER>
__device__ __forceinline__ void gbuffer_px(const ResolveArgs &a, const FrameUniforms &u, int x, int y)
{
    const size_t i = (size_t)x + (size_t)y * a.W;
    const size_t P = (size_t)a.W * a.H;
    float *gb = a.gbuf;
    const Winner w = resolve_winner<DIRECT>(a, i, x, y);
    if (w.g < 0) {
        if (a.fresh)
            for (int c = 0; c < kGbufPlanes; ++c) gb[c * P + i] = 0.f;
        resolve_end<DIRECT>(a, i, w);
        return;
    }
    const int d0 = __builtin_amdgcn_readfirstlane(w.tv.w);
    if (__ballot(w.tv.w != d0) == 0ull) {
        const DevDraw &dr = a.draws[d0];
        const int f = w.g - dr.tri_base;
        const int mi = dr.face_mat[f];
        const int m0 = __builtin_amdgcn_readfirstlane(mi);
        if (__ballot(mi != m0) == 0ull) {
            gbuffer_shade<CORNER>(a, u, dr, a.materials[m0], f, w.tv, w.b, i, P);
            resolve_end<DIRECT>(a, i, w);
            return;
        }
    }
    const DevDraw &dr = a.draws[w.tv.w];
    const int f = w.g - dr.tri_base;
    gbuffer_shade<CORNER>(a, u, dr, a.materials[dr.face_mat[f]], f, w.tv, w.b, i, P);
    resolve_end<DIRECT>(a, i, w);
}

}  // namespace fgl
