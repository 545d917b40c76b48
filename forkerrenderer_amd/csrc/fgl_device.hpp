// fgl_device.hpp -- device-resident scene data and the per-pixel programs of
// the reference's shaders, written for gfx950.
#pragma once

#include "fgl_math.hpp"

namespace fgl {

constexpr int kMaxLights = 4;
constexpr int kMaxDisk = 64;

// Texture in HBM: one packed texel per uint32 (r | g<<8 | b<<16), row y at y*w.
// TGAImage::Get's byte order (B,G,R; grey sets only b) is resolved at upload
// (src/tgaimage.h:149-181).
struct DevTexture {
    const uint32_t *texels;   // r | g << 8 | b << 16 per texel
    const uint8_t *zb;        // the b byte alone (what SampleFloat reads), 1 B per texel
    int w, h, wrap, filter;
};

// The maps that a shader samples at one coordinate, when they share size, wrap
// and filter, as one array: per texel colour A's r, g, b and map Z's byte,
// then the normal map's r, g, b and map Y's byte.  Texels lie in 4 x 4 blocks
// of 128 bytes: a bilinear sample of all of them takes four 8-byte loads from
// 1.6 cache lines on average, where separate row-major maps took 16 loads
// from 8 lines or more.
constexpr int kBundleA = 1, kBundleZ = 2, kBundleN = 4, kBundleY = 8;

struct DevBundle {
    const uint2 *t;          // nullptr: no bundle
    int w, h, wrap, filter;
    int has;                 // kBundle* of the maps it holds
    int pad;
};

struct DevMaterial {
    float ka[3], kd[3], ks[3], ke[3];
    int map_kd, map_ks, map_ke, map_bump;
    float pbr_ke[3], albedo[3], roughness, metalness;
    int map_base, map_rough, map_metal, map_ao, map_pbr_ke;
    // Blinn-Phong (A diffuse, Z specular), PBR (A base, Z roughness, Y metalness)
    DevBundle bundle[2];
};

// One draw of a pass: a model's SoA attribute arrays, face index streams and
// uniforms.  vert_base/tri_base place it in the pass-wide vertex/triangle order.
struct DevDraw {
    const float *pos, *uv, *nrm, *tan;
    const int *vi, *ti, *ni, *face_mat;
    // per face, the attributes the main vertex programs read, 9 float4: for
    // each corner (uv, n.xy), (n.z, t.xyz), the normal and tangent normalised as
    // ProcessVertex does, then the three positions (corner_form alone reads
    // them) -- one 144-byte record instead of four arrays behind three index streams
    const float4 *corner;
    // the faces in spatial order: position indices (as vi) and the face
    const int4 *tri;
    int n_pos, n_faces, vert_base, tri_base;
    int has_tangents, support_pbr;
    int view;      // batched views: index of the draw's view (0 otherwise)
    int pad0;
    float model[16];
    float normal[9];
    float lm[16];  // light_space * model (DepthShader, src/shaders/depthshader.h:23-25)
};

struct DevLight {
    int type;
    float vec[3];
    float color[3];
};

struct DevShadowCfg {
    int mode, grid, n_blocker, n_pcf;
    float pcf_filter, area_light;
    double blocker_filter, pcss_filter;
    float blocker_disk[2 * kMaxDisk];
    float pcf_disk[2 * kMaxDisk];
    // blocker_disk[i] * blocker_filter in double, narrowed to float (the
    // reference's per-sample offset; the same for every pixel)
    float blocker_off[2 * kMaxDisk];
};

struct FrameUniforms {
    float view[16], proj[16], light_space[16], viewport[16], shadow_viewport[16];
    float vp[16];  // proj * view (SetViewProjectionMatrix, src/render.cpp:115)
    float eye[3];
    int shadow_on;
    int n_lights, W, H, SW, SH;
    DevLight lights[kMaxLights];
    DevShadowCfg shadow;
};

// ---------------- textures (src/texture.h:41-145) ----------------

__device__ __forceinline__ Vec3 texel_rgb(const DevTexture &t, int x, int y)
{
    if (x < 0 || y < 0 || x >= t.w || y >= t.h) return vec3(0.f, 0.f, 0.f);
    uint32_t p = t.texels[(size_t)x + (size_t)y * t.w];
    return vec3((float)(p & 255u), (float)((p >> 8) & 255u), (float)((p >> 16) & 255u));
}

template <typename Tex>   // DevTexture or DevBundle
__device__ __forceinline__ Vec2 wrap_coord(const Tex &t, Vec2 c)
{
    if (t.wrap == 1) return vec2(c.x - floorf(c.x), c.y - floorf(c.y));
    if (t.wrap == 2) {
        int xi = trunc_int(floorf(c.x)), yi = trunc_int(floorf(c.y));
        float rx = c.x - (float)xi, ry = c.y - (float)yi;
        return vec2((xi % 2 == 0) ? rx : 1.f - rx, (yi % 2 == 0) ? ry : 1.f - ry);
    }
    if (t.wrap == 3) return vec2(clampf(c.x, 0.f, 1.f), clampf(c.y, 0.f, 1.f));
    return c;
}

__device__ __forceinline__ Vec3 filter_color(const DevTexture &t, Vec2 c)
{
    float w = (float)(t.w - 0.001), h = (float)(t.h - 0.001);
    if (t.filter == 1) {
        float px = c.x * w, py = c.y * h;
        float tlx = floorf(px - 0.5f), tly = floorf(py - 0.5f);
        float tx = px - (tlx + 0.5f);
        float ty = py - (tly + 0.5f);
        int s0x = trunc_int(tlx), s0y = trunc_int(tly);
        int s1x = trunc_int(tlx + 1.f), s2y = trunc_int(tly + 1.f);
        int s1y = s0y, s2x = s0x, s3x = s1x, s3y = s2y;
        if (t.wrap != 0) {
            s0x = clampi(s0x, 0, t.w - 1); s0y = clampi(s0y, 0, t.h - 1);
            s1x = clampi(s1x, 0, t.w - 1); s1y = clampi(s1y, 0, t.h - 1);
            s2x = clampi(s2x, 0, t.w - 1); s2y = clampi(s2y, 0, t.h - 1);
            s3x = clampi(s3x, 0, t.w - 1); s3y = clampi(s3y, 0, t.h - 1);
        }
        Vec3 c0 = texel_rgb(t, s0x, s0y), c1 = texel_rgb(t, s1x, s1y);
        Vec3 c2 = texel_rgb(t, s2x, s2y), c3 = texel_rgb(t, s3x, s3y);
        Vec3 cx1 = lerp3(tx, c0, c1), cx2 = lerp3(tx, c2, c3);
        return lerp3(ty, cx1, cx2);
    }
    return texel_rgb(t, trunc_int(floorf(c.x * w)), trunc_int(floorf(c.y * h)));
}

// filter_color's third channel alone, from the 1-byte plane: the same
// texel coordinates and the same per-channel arithmetic (lerp3 is
// component-wise), a quarter of the bytes.
__device__ __forceinline__ float texel_z(const DevTexture &t, int x, int y)
{
    if (x < 0 || y < 0 || x >= t.w || y >= t.h) return 0.f;
    return (float)t.zb[(size_t)x + (size_t)y * t.w];
}

__device__ __forceinline__ float lerp1(float t, float a, float b) { return a * (1 - t) + b * t; }

__device__ __forceinline__ float filter_z(const DevTexture &t, Vec2 c)
{
    float w = (float)(t.w - 0.001), h = (float)(t.h - 0.001);
    if (t.filter == 1) {
        float px = c.x * w, py = c.y * h;
        float tlx = floorf(px - 0.5f), tly = floorf(py - 0.5f);
        float tx = px - (tlx + 0.5f);
        float ty = py - (tly + 0.5f);
        int s0x = trunc_int(tlx), s0y = trunc_int(tly);
        int s1x = trunc_int(tlx + 1.f), s2y = trunc_int(tly + 1.f);
        int s1y = s0y, s2x = s0x, s3x = s1x, s3y = s2y;
        if (t.wrap != 0) {
            s0x = clampi(s0x, 0, t.w - 1); s0y = clampi(s0y, 0, t.h - 1);
            s1x = clampi(s1x, 0, t.w - 1); s1y = clampi(s1y, 0, t.h - 1);
            s2x = clampi(s2x, 0, t.w - 1); s2y = clampi(s2y, 0, t.h - 1);
            s3x = clampi(s3x, 0, t.w - 1); s3y = clampi(s3y, 0, t.h - 1);
        }
        float c0 = texel_z(t, s0x, s0y), c1 = texel_z(t, s1x, s1y);
        float c2 = texel_z(t, s2x, s2y), c3 = texel_z(t, s3x, s3y);
        float cx1 = lerp1(tx, c0, c1), cx2 = lerp1(tx, c2, c3);
        return lerp1(ty, cx1, cx2);
    }
    return texel_z(t, trunc_int(floorf(c.x * w)), trunc_int(floorf(c.y * h)));
}

// Texture::Sample / SampleFloat (src/texture.h:41-51)
__device__ __forceinline__ Vec3 tex_sample(const DevTexture *texs, int id, Vec2 uv)
{
    const DevTexture &t = texs[id];
    return divs3(filter_color(t, wrap_coord(t, uv)), 255.f);
}
__device__ __forceinline__ float tex_samplef(const DevTexture *texs, int id, Vec2 uv)
{
    const DevTexture &t = texs[id];
    return filter_z(t, wrap_coord(t, uv)) / 255.f;
}

// Every map of a bundle at one coordinate: the values tex_sample (A, N) and
// tex_samplef (Z, Y) give, by the same texel coordinates and arithmetic
// (lerp3 is component-wise).
struct BundleSample {
    Vec3 a, n;
    float z, y;
};

__host__ __device__ __forceinline__ size_t bundle_index(int w, int x, int y)
{
    return ((size_t)(y >> 2) * ((w + 3) >> 2) + (x >> 2)) * 16 + (y & 3) * 4 + (x & 3);
}

__device__ __forceinline__ uint2 bundle_texel(const DevBundle &t, int x, int y)
{
    if (x < 0 || y < 0 || x >= t.w || y >= t.h) return make_uint2(0u, 0u);
    return t.t[bundle_index(t.w, x, y)];
}

__device__ __forceinline__ BundleSample bundle_sample(const DevBundle &t, Vec2 uv)
{
    const Vec2 c = wrap_coord(t, uv);
    const float w = (float)(t.w - 0.001), h = (float)(t.h - 0.001);
    float v[8];
    if (t.filter == 1) {
        const float px = c.x * w, py = c.y * h;
        const float tlx = floorf(px - 0.5f), tly = floorf(py - 0.5f);
        const float tx = px - (tlx + 0.5f), ty = py - (tly + 0.5f);
        int x0 = trunc_int(tlx), y0 = trunc_int(tly), x1 = trunc_int(tlx + 1.f), y1 = trunc_int(tly + 1.f);
        if (t.wrap != 0) {
            x0 = clampi(x0, 0, t.w - 1); x1 = clampi(x1, 0, t.w - 1);
            y0 = clampi(y0, 0, t.h - 1); y1 = clampi(y1, 0, t.h - 1);
        }
        const uint2 t00 = bundle_texel(t, x0, y0), t10 = bundle_texel(t, x1, y0);
        const uint2 t01 = bundle_texel(t, x0, y1), t11 = bundle_texel(t, x1, y1);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int s = 8 * (k & 3);
            auto ch = [&](uint2 q) { return (float)(((k < 4 ? q.x : q.y) >> s) & 255u); };
            v[k] = lerp1(ty, lerp1(tx, ch(t00), ch(t10)), lerp1(tx, ch(t01), ch(t11)));
        }
    } else {
        const uint2 q = bundle_texel(t, trunc_int(floorf(c.x * w)), trunc_int(floorf(c.y * h)));
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = (float)(((k < 4 ? q.x : q.y) >> (8 * (k & 3))) & 255u);
    }
    BundleSample o;
    o.a = divs3(vec3(v[0], v[1], v[2]), 255.f);
    o.z = v[3] / 255.f;
    o.n = divs3(vec3(v[4], v[5], v[6]), 255.f);
    o.y = v[7] / 255.f;
    return o;
}

// ---------------- vertex programs ----------------

// Varyings of one vertex after ProcessVertex with perspective-correct
// interpolation enabled (src/shaders/gshader.h:41-92).
struct Varying {
    Vec3 ws, nws, tws, lndc;
    Vec2 uv;
    float oow;
};

// BlinnPhong/PBR/G ProcessVertex (phongshader.h:35-85, pbrshader.h:35-85,
// gshader.h:41-92), the part that depends on the position p alone: its NDC, and
// the varyings as two float4 (position / w and 1 / w, light NDC / w).
__device__ __forceinline__ Vec4 main_position(const DevDraw &d, const FrameUniforms &u, Vec4 p, float4 &v0, float4 &v1)
{
    Vec4 ws = mv4(d.model, p);
    Vec4 cs = mv4(u.proj, mv4(u.view, ws));
    Vec4 l = vec4(0.f, 0.f, 0.f, 0.f);
    if (u.shadow_on) {
        l = mv4(u.light_space, ws);
        l = divs4(l, l.w);
    }
    const float oow = recip(cs.w);
    ws = scale4(ws, oow);
    if (u.shadow_on) l = scale4(l, oow);
    v0 = make_float4(ws.x, ws.y, ws.z, oow);
    v1 = make_float4(l.x, l.y, l.z, 0.f);
    return divs4(cs, cs.w);
}

// main_position of vertex vi; vary (v0, v1 of each vertex; null where the
// resolve makes them, corner_form) also takes its varyings.
__device__ __forceinline__ Vec4 main_vertex_pass(const DevDraw &d, const FrameUniforms &u, int vi, float4 *vary)
{
    float4 v0, v1;
    const Vec4 ndc = main_position(d, u, vec4(d.pos[3 * vi], d.pos[3 * vi + 1], d.pos[3 * vi + 2], 1.f), v0, v1);
    if (vary) {
        const size_t v = 2 * ((size_t)d.vert_base + vi);
        vary[v] = v0;
        vary[v + 1] = v1;
    }
    return ndc;
}

// Corner k of face f, a corner at vertex v of the pass's varyings, with its
// attributes as Mesh::TexCoord / Normal / Tangent fetch them (mesh.cpp:34-56).
// CORNER: the varyings made here from the position in the corner's record
// (corner_form, pass_plan.hpp) instead of read from the vertex pass's.
template <bool CORNER>
__device__ __forceinline__ Varying main_vertex(const DevDraw &d, const FrameUniforms &u, const float4 *vary, int v, int f,
                                               int k)
{
    Varying o;
    const float4 *face = d.corner + (size_t)f * 9;
    const float4 r0 = face[2 * k], r1 = face[2 * k + 1];
    float4 p0, p1;
    if (CORNER) {
        const float4 r2 = face[6 + k];
        (void)main_position(d, u, vec4(r2.x, r2.y, r2.z, 1.f), p0, p1);
    } else {
        p0 = vary[2 * (size_t)v];
        p1 = vary[2 * (size_t)v + 1];
    }
    const float oow = p0.w;
    o.ws = vec3(p0.x, p0.y, p0.z);
    o.lndc = vec3(p1.x, p1.y, p1.z);
    o.oow = oow;
    o.uv = vec2(r0.x * oow, r0.y * oow);
    o.nws = scale3(mv3(d.normal, vec3(r0.z, r0.w, r1.x)), oow);
    o.tws = vec3(0.f, 0.f, 0.f);
    if (d.has_tangents) o.tws = scale3(mv3(d.normal, vec3(r1.y, r1.z, r1.w)), oow);
    return o;
}

// DepthShader::ProcessVertex (src/shaders/depthshader.h:21-28)
__device__ __forceinline__ Vec4 depth_ndc(const DevDraw &d, int vi)
{
    Vec4 p = vec4(d.pos[3 * vi], d.pos[3 * vi + 1], d.pos[3 * vi + 2], 1.f);
    Vec4 cs = mv4(d.lm, p);
    return divs4(cs, cs.w);
}

// ---------------- fragment geometry (gshader.h:95-141) ----------------

struct FragGeom {
    Vec3 pos, normal, lndc;
    Vec2 uv;
    BundleSample maps;   // the material's bundle at uv, when it has one
};

__device__ __forceinline__ FragGeom frag_geometry(const DevDraw &d, const FrameUniforms &u,
                                                  const DevTexture *texs, const Varying &v0,
                                                  const Varying &v1, const Varying &v2, Vec3 b,
                                                  int normal_map, const DevBundle &bundle)
{
    FragGeom g;
    Vec3 pws = interp3(v0.ws, v1.ws, v2.ws, b);
    Vec2 uv = interp2(v0.uv, v1.uv, v2.uv, b);
    Vec3 nws = interp3(v0.nws, v1.nws, v2.nws, b);
    float w = recip(dot3(vec3(v0.oow, v1.oow, v2.oow), b));
    pws = scale3(pws, w);
    uv.x *= w;
    uv.y *= w;
    if (bundle.t) g.maps = bundle_sample(bundle, uv);
    nws = scale3(nws, w);
    Vec3 N = norm3(nws);
    Vec3 normal = N;
    if (d.has_tangents && normal_map >= 0) {
        Vec3 tws = scale3(interp3(v0.tws, v1.tws, v2.tws, b), w);
        Vec3 T = norm3(add3(tws, vec3(0.001f, 0.001f, 0.001f)));
        T = norm3(sub3(T, scale3(N, dot3(T, N))));
        Vec3 B = norm3(cross3(N, T));
        Vec3 s = (bundle.has & kBundleN) ? g.maps.n : tex_sample(texs, normal_map, uv);
        s = norm3(sub3(scale3(s, 2.f), vec3(1.f, 1.f, 1.f)));
        normal = norm3(vec3(dot3(vec3(T.x, B.x, N.x), s), dot3(vec3(T.y, B.y, N.y), s),
                            dot3(vec3(T.z, B.z, N.z), s)));
    }
    g.pos = pws;
    g.normal = normal;
    g.uv = uv;
    g.lndc = vec3(0.f, 0.f, 0.f);
    if (u.shadow_on) g.lndc = scale3(interp3(v0.lndc, v1.lndc, v2.lndc, b), w);
    return g;
}

// ---------------- shadows (src/shaders/shadow.cpp:23-131) ----------------

__device__ __forceinline__ float sample_shadow(const float *map, int SW, int SH, float u, float v)
{
    // A NaN coordinate is treated as out of the map (the reference would
    // index with INT_MIN).
    if (!(u >= 0.f && u <= 1.f && v >= 0.f && v <= 1.f)) return __builtin_inff();
    int w = (int)((float)SW - 0.001f);
    int h = (int)((float)SH - 0.001f);
    int x = (int)((float)w * u);
    int y = (int)((float)h * v);
    float dd = map[(size_t)x + (size_t)y * SW];
    // (double)dd < 0.001: 0.001f is the float just above 0.001 (the one just
    // below is 0.00099999993), so for a float dd the two tests agree, NaN
    // included.
    return (dd < 0.001f) ? 1.f : dd;
}

__device__ __forceinline__ float pcf_disk(const float *map, int SW, int SH, Vec3 sc, float bias,
                                          float filter, const float *disk, int n)
{
    float vis = 0.f;
    float inv = 1.f / (float)n;
    for (int i = 0; i < n; ++i) {
        float s = sample_shadow(map, SW, SH, sc.x + disk[2 * i] * filter,
                                sc.y + disk[2 * i + 1] * filter);
        if (sc.z <= s + bias) vis += inv;
    }
    return vis;
}

// PCSS blocker term (FindAverageBlockDepth, shadow.cpp:65-91): the average
// depth of the samples that block, 0 when none does.  `disk` holds the
// offsets already scaled (blocker_off: the unit-disk samples times
// blocker_filter in double, as the reference scales them).
__device__ __forceinline__ float pcss_blocker_depth(const FrameUniforms &u, const float *map, Vec3 sc, float bias,
                                                    const float *disk, int n)
{
    float blocker = 0.f, nb = 0.f;
    for (int i = 0; i < n; ++i) {
        const float ou = disk[2 * i];
        const float ov = disk[2 * i + 1];
        float su = sc.x + ou;
        float sv = sc.y + ov;
        float s = sample_shadow(map, u.SW, u.SH, su, sv);
        if (sc.z > s + bias) {
            blocker += s;
            nb += 1.f;
        }
    }
    return (nb < 1.f) ? 0.f : blocker / nb;
}

// Accepted vectors of the random stream, in stream order, in chunks: chunk
// c's lie at v + c * stride * D (D floats each), prefix[c] of them before it;
// at least kStreamRun more follow each chunk's own (the next chunk's first),
// so a run of that many starting in a chunk is contiguous.  Chunks keep their
// tries' expected share within a fraction of a percent, so the chunk of a
// vector is guessed from it (inv: chunks per vector) and settled by the
// prefixes.
constexpr int kStreamRun = 128;
static_assert(kStreamRun >= 2 * kMaxDisk, "a point's blocker and PCF samples in one run");

struct StreamVectors {
    const float *v;
    const uint32_t *prefix;
    uint32_t chunks, stride;
    float inv;
};

template <int D>
__device__ __forceinline__ const float *stream_at(const StreamVectors &s, uint32_t j)
{
    uint32_t c = (uint32_t)((float)j * s.inv);
    c = c < s.chunks ? c : s.chunks - 1;
    while (c > 0 && j < s.prefix[c]) --c;
    while (c + 1 < s.chunks && j >= s.prefix[c + 1]) ++c;
    return s.v + ((size_t)c * s.stride + (j - s.prefix[c])) * D;
}

// The pairs from j on that lie in one run: their address and how many.
struct StreamRun {
    const float *v;
    uint32_t left;
};

__device__ __forceinline__ StreamRun stream_run(const StreamVectors &s, uint32_t j)
{
    uint32_t c = (uint32_t)((float)j * s.inv);
    c = c < s.chunks ? c : s.chunks - 1;
    while (c > 0 && j < s.prefix[c]) --c;
    while (c + 1 < s.chunks && j >= s.prefix[c + 1]) ++c;
    return StreamRun{s.v + ((size_t)c * s.stride + (j - s.prefix[c])) * 2, s.prefix[c + 1] - j};
}

// The random stream's samples (modes 4 and 5) are each pixel's own, 512
// bytes or more apart between neighbouring lanes: read one sample per load,
// every load would fetch a cache line per lane.  So they are taken
// kStreamGroup at a time: the group's pairs, then its texels, are loaded
// before any is used (a texel of a sample off the map is read at index 0 and
// replaced by +inf, as sample_shadow returns it), and a pixel's lines are
// used while they are cached.  The arithmetic and its order per sample are
// those of the reference's FindAverageBlockDepth and PCF (pcss_blocker_depth
// with the offsets scaled per sample, pcf_disk).
constexpr int kStreamGroup = 8;

// Shadow-map texel of (su, sv) as sample_shadow indexes it; in = on the map.
__device__ __forceinline__ size_t shadow_texel(int SW, int w, int h, float su, float sv, bool &in)
{
    in = su >= 0.f && su <= 1.f && sv >= 0.f && sv <= 1.f;
    const int x = in ? (int)((float)w * su) : 0, y = in ? (int)((float)h * sv) : 0;
    return (size_t)x + (size_t)y * SW;
}

__device__ __forceinline__ float shadow_value(bool in, float dd) { return !in ? __builtin_inff() : ((dd < 0.001f) ? 1.f : dd); }

// The (2 R + 1)^2 grid around sc: a row's and a column's coordinate, test and
// index are made once, not for every texel, and a row's texels are loaded
// together (adding 0 leaves the sum as it is).  5 x 5, 1280 x 800 lighting 39 -> 32
// us, 24 views 491 -> 422.
template <int R>
__device__ __forceinline__ float pcf_grid(const FrameUniforms &u, const float *map, Vec3 sc, float bias, float tu, float tv,
                                          float inv)
{
    const int w = (int)((float)u.SW - 0.001f), h = (int)((float)u.SH - 0.001f);
    int x[2 * R + 1];
    bool ix[2 * R + 1];
#pragma unroll
    for (int d = -R; d <= R; ++d) {
        const float su = sc.x + (float)d * tu;
        ix[d + R] = su >= 0.f && su <= 1.f;
        x[d + R] = ix[d + R] ? (int)((float)w * su) : 0;
    }
    float vis = 0.f;
#pragma unroll
    for (int d = -R; d <= R; ++d) {
        const float sv = sc.y + (float)d * tv;
        const bool iy = sv >= 0.f && sv <= 1.f;
        const float *row = map + (size_t)(iy ? (int)((float)h * sv) : 0) * u.SW;
        float dd[2 * R + 1];
#pragma unroll
        for (int k = 0; k < 2 * R + 1; ++k) dd[k] = row[x[k]];
#pragma unroll
        for (int k = 0; k < 2 * R + 1; ++k) vis += sc.z <= shadow_value(ix[k] && iy, dd[k]) + bias ? inv : 0.f;
    }
    return vis;
}

// pcss_blocker_depth over stream samples (unit-disk samples scaled here in
// double, as the reference scales them).
__device__ __forceinline__ float pcss_blocker_stream(const FrameUniforms &u, const float *map, Vec3 sc, float bias,
                                                     const float *disk, int n)
{
    const DevShadowCfg &c = u.shadow;
    const float2 *d = (const float2 *)disk;
    const int w = (int)((float)u.SW - 0.001f), h = (int)((float)u.SH - 0.001f);
    float blocker = 0.f, nb = 0.f;
    int i = 0;
    for (; i + kStreamGroup <= n; i += kStreamGroup) {
        float2 ds[kStreamGroup];
#pragma unroll
        for (int e = 0; e < kStreamGroup; ++e) ds[e] = d[i + e];
        float dd[kStreamGroup];
        bool in[kStreamGroup];
#pragma unroll
        for (int e = 0; e < kStreamGroup; ++e) {
            const float su = sc.x + (float)((double)ds[e].x * c.blocker_filter);
            const float sv = sc.y + (float)((double)ds[e].y * c.blocker_filter);
            dd[e] = map[shadow_texel(u.SW, w, h, su, sv, in[e])];
        }
#pragma unroll
        for (int e = 0; e < kStreamGroup; ++e) {
            const float s = shadow_value(in[e], dd[e]);
            if (sc.z > s + bias) {
                blocker += s;
                nb += 1.f;
            }
        }
    }
    for (; i < n; ++i) {
        const float su = sc.x + (float)((double)d[i].x * c.blocker_filter);
        const float sv = sc.y + (float)((double)d[i].y * c.blocker_filter);
        const float s = sample_shadow(map, u.SW, u.SH, su, sv);
        if (sc.z > s + bias) {
            blocker += s;
            nb += 1.f;
        }
    }
    return (nb < 1.f) ? 0.f : blocker / nb;
}

// pcf_disk over stream samples.
__device__ __forceinline__ float pcf_stream(const float *map, int SW, int SH, Vec3 sc, float bias, float filter,
                                            const float *disk, int n)
{
    const float2 *d = (const float2 *)disk;
    const int w = (int)((float)SW - 0.001f), h = (int)((float)SH - 0.001f);
    float vis = 0.f;
    const float inv = 1.f / (float)n;
    int i = 0;
    for (; i + kStreamGroup <= n; i += kStreamGroup) {
        float2 ds[kStreamGroup];
#pragma unroll
        for (int e = 0; e < kStreamGroup; ++e) ds[e] = d[i + e];
        float dd[kStreamGroup];
        bool in[kStreamGroup];
#pragma unroll
        for (int e = 0; e < kStreamGroup; ++e)
            dd[e] = map[shadow_texel(SW, w, h, sc.x + ds[e].x * filter, sc.y + ds[e].y * filter, in[e])];
#pragma unroll
        for (int e = 0; e < kStreamGroup; ++e)
            if (sc.z <= shadow_value(in[e], dd[e]) + bias) vis += inv;
    }
    for (; i < n; ++i) {
        const float s = sample_shadow(map, SW, SH, sc.x + d[i].x * filter, sc.y + d[i].y * filter);
        if (sc.z <= s + bias) vis += inv;
    }
    return vis;
}

// Shadow coordinate and slope bias (CalculateShadowVisibility, shadow.cpp:109-117).
__device__ __forceinline__ Vec3 shadow_coord(Vec3 ndc) { return add3(scale3(ndc, 0.5f), vec3(0.5f, 0.5f, 0.5f)); }
__device__ __forceinline__ float shadow_bias(Vec3 n, Vec3 l) { return smax(0.009f * (1.f - dot3(n, l)), 0.007f); }

// STREAM: the kernel runs with the random stream's samples (modes 4 and 5),
// `rdisk` being this pixel's: the PCF samples, or the blocker samples
// followed by the PCF ones.  MODE: the filter the kernel is compiled for (one
// filter's registers cost the others occupancy: with a grid unrolled beside
// it, PCSS lighting at 3840 x 2160 took 294 us, not 215); -1 reads it from the
// settings, without the stream filters, which only STREAM kernels have.
template <bool STREAM, int MODE>
__device__ __forceinline__ float shadow_visibility(const FrameUniforms &u, const float *map,
                                                   Vec3 ndc, Vec3 n, Vec3 l, const float *rdisk)
{
    const DevShadowCfg &c = u.shadow;
    const int mode = MODE >= 0 ? MODE : c.mode;
    Vec3 sc = shadow_coord(ndc);
    float bias = shadow_bias(n, l);
    if (mode == 1) return pcf_disk(map, u.SW, u.SH, sc, bias, c.pcf_filter, c.pcf_disk, c.n_pcf);
    if (mode == 4) {
        if constexpr (STREAM) return pcf_stream(map, u.SW, u.SH, sc, bias, c.pcf_filter, rdisk, c.n_pcf);
        return 1.f;
    }
    if (mode == 5) {
        if constexpr (STREAM) {
            const float dB = pcss_blocker_stream(u, map, sc, bias, rdisk, c.n_blocker);
            if ((double)dB < 0.001) return 1.f;
            float pen = (sc.z - dB) * c.area_light / dB;
            float filter = (float)(c.pcss_filter * (double)pen);
            return pcf_stream(map, u.SW, u.SH, sc, bias, filter, rdisk + 2 * c.n_blocker, c.n_pcf);
        }
        return 1.f;
    }
    if (mode == 2) {
        const float dB = pcss_blocker_depth(u, map, sc, bias, c.blocker_off, c.n_blocker);
        if ((double)dB < 0.001) return 1.f;
        float pen = (sc.z - dB) * c.area_light / dB;
        float filter = (float)(c.pcss_filter * (double)pen);
        return pcf_disk(map, u.SW, u.SH, sc, bias, filter, c.pcf_disk, c.n_pcf);
    }
    if (mode == 3) {
        const float inv = 1.f / (float)(c.grid * c.grid);
        const float tu = 1.f / (float)u.SW, tv = 1.f / (float)u.SH;
        if (c.grid == 5) return pcf_grid<2>(u, map, sc, bias, tu, tv, inv);
        if (c.grid == 3) return pcf_grid<1>(u, map, sc, bias, tu, tv, inv);
        const int r = c.grid / 2;
        float vis = 0.f;
        for (int dy = -r; dy <= r; ++dy)
            for (int dx = -r; dx <= r; ++dx) {
                float s = sample_shadow(map, u.SW, u.SH, sc.x + (float)dx * tu, sc.y + (float)dy * tv);
                if (sc.z <= s + bias) vis += inv;
            }
        return vis;
    }
    float s = sample_shadow(map, u.SW, u.SH, sc.x, sc.y);
    return (sc.z <= s + bias) ? 1.f : 0.f;
}

// ---------------- lighting (phongshader.h:171-215, pbrshader.h:182-288) ----------------

// powf(x, y) for the non-negative (or NaN) bases of the shading code, as
// exp2(y * log2(x)) with the hardware base-2 log and exp: a few ulps from the
// correctly rounded power, which the 8-bit output absorbs (a result moves by
// at most one 8-bit step, and only at a quantisation boundary), in ~8
// operations instead of the ~160 of the general powf.  pow(x, 0) = 1;
// denormal x and results below 2^-126 are rescaled (the hardware log and exp
// take and give normal floats only).
__device__ __forceinline__ float pow_pos(float x, float y)
{
    if (y == 0.f) return 1.f;
    const bool sub = x < 0x1p-126f;
    const float lx = __builtin_amdgcn_logf(sub ? x * 0x1p32f : x) - (sub ? 32.f : 0.f);
    const float e = y * lx;
    const bool tiny = e < -126.f;
    return __builtin_amdgcn_exp2f(tiny ? e + 32.f : e) * (tiny ? 0x1p-32f : 1.f);
}

__device__ __forceinline__ Vec3 pow3f(Vec3 a, float p)
{
    return vec3(pow_pos(a.x, p), pow_pos(a.y, p), pow_pos(a.z, p));
}

__device__ __forceinline__ Vec3 tonemap_gamma(Vec3 c)
{
    c = vec3(c.x / (c.x + 1.f), c.y / (c.y + 1.f), c.z / (c.z + 1.f));
    return clamp01_3(pow3f(c, 1.f / 2.2f));
}

__device__ __forceinline__ Vec3 bp_term(Vec3 L, Vec3 H, Vec3 N, float vis, Vec3 dl, Vec3 el,
                                        float ao, float ks, float shin, Vec3 lc, int shadow_on,
                                        bool with_emissive)
{
    float diff = smax(0.f, dot3(L, N));
    float spec = pow_pos(smax(0.f, dot3(H, N)), shin);
    Vec3 diffuse = scale3(scale3(dl, diff), ao);
    Vec3 specular = scale3(vec3(ks, ks, ks), spec);
    if (shadow_on) {
        float sh = (1 - vis) * 0.6f;
        float vv = 1 - sh;
        diffuse = scale3(diffuse, vv);
        specular = scale3(specular, vv);
    }
    Vec3 t = add3(diffuse, specular);
    if (with_emissive) t = add3(t, el);
    return mul3(t, lc);
}

__device__ __forceinline__ Vec3 pbr_lo(Vec3 L, Vec3 V, Vec3 H, Vec3 N, float vis, Vec3 al,
                                       float metal, float rough, Vec3 rad, int shadow_on)
{
    const float InvPi = (float)0.31830988618379067154;
    float NdotV = smax(dot3(N, V), 0.f);
    float NdotL = smax(dot3(N, L), 0.f);
    float NdotH = smax(dot3(N, H), 0.f);
    float HdotV = smax(dot3(H, V), 0.f);
    Vec3 F0 = lerp3(metal, vec3(0.04f, 0.04f, 0.04f), al);
    float a = rough * rough;
    float a2 = a * a;
    float NdotH2 = NdotH * NdotH;
    float den = (NdotH2 * (a2 - 1.f) + 1.f);
    float den2 = den * den;
    float NDF = a2 * InvPi / den2;
    float ka = rough + 1.f;
    float k = ka * ka / 8.f;
    float g1 = NdotV / (NdotV * (1 - k) + k);
    float g2 = NdotL / (NdotL * (1 - k) + k);
    float G = g1 * g2;
    float omh = smax(1.f - HdotV, 0.f);
    float p5 = pow_pos(omh, 5.f);
    Vec3 F = add3(F0, scale3(sub3(vec3(1.f, 1.f, 1.f), F0), p5));
    Vec3 DGF = scale3(F, NDF * G);
    float denom = 4 * NdotV * NdotL + 0.001f;
    Vec3 spec = divs3(DGF, denom);
    Vec3 kd = scale3(sub3(vec3(1.f, 1.f, 1.f), F), 1.f - metal);
    Vec3 brdf = add3(scale3(mul3(kd, al), InvPi), spec);
    Vec3 Lo = scale3(mul3(brdf, rad), NdotL);
    if (shadow_on) {
        float sh = (1 - vis) * 0.6f;
        float vv = 1 - sh;
        Lo = scale3(Lo, vv);
    }
    return Lo;
}

__device__ __forceinline__ Vec3 light_dir(const DevLight &l, Vec3 P)
{
    if (l.type == 0) return norm3(sub3(vec3(l.vec[0], l.vec[1], l.vec[2]), P));
    return norm3(vec3(-l.vec[0], -l.vec[1], -l.vec[2]));
}

// One surface point lit by every light.  With a single point light this is
// the reference's CalculateLight; `deferred_quirk` passes viewDir in the
// Blinn-Phong halfway slot as DrawScreenSpacePixels does (forkergl.cpp:369).
template <bool STREAM = false, int MODE = -1>
__device__ __forceinline__ Vec3 shade_point(const FrameUniforms &u, const float *smap, bool pbr,
                                            bool deferred_quirk, Vec3 P, Vec3 N, Vec3 lndc,
                                            Vec3 albedo, Vec3 emissive, Vec3 param,
                                            const float *rdisk = nullptr)
{
    const float gamma = (float)2.2;
    Vec3 Vd = norm3(sub3(vec3(u.eye[0], u.eye[1], u.eye[2]), P));
    // light 0's visibility, the same for both models
    float vis0 = 0.f;
    if (u.shadow_on && u.n_lights > 0)
        vis0 = shadow_visibility<STREAM, MODE>(u, smap, lndc, N, light_dir(u.lights[0], P), rdisk);
    if (!pbr) {
        Vec3 dl = pow3f(albedo, gamma);
        Vec3 el = pow3f(emissive, gamma);
        Vec3 c = scale3(mul3(vec3(0.3f, 0.3f, 0.3f), dl), param.x);
        for (int i = 0; i < u.n_lights; ++i) {
            const DevLight &l = u.lights[i];
            Vec3 L = light_dir(l, P);
            const float vis = !u.shadow_on ? 0.f : i == 0 ? vis0 : 1.f;
            Vec3 H = deferred_quirk ? Vd : norm3(add3(L, Vd));
            c = add3(c, bp_term(L, H, N, vis, dl, el, param.x, param.y, param.z,
                                vec3(l.color[0], l.color[1], l.color[2]), u.shadow_on, i == 0));
        }
        return tonemap_gamma(c);
    }
    Vec3 al = pow3f(albedo, gamma);
    Vec3 el = pow3f(emissive, gamma);
    Vec3 Lo = vec3(0.f, 0.f, 0.f);
    for (int i = 0; i < u.n_lights; ++i) {
        const DevLight &l = u.lights[i];
        Vec3 L = light_dir(l, P);
        const float vis = !u.shadow_on ? 0.f : i == 0 ? vis0 : 1.f;
        Vec3 H = norm3(add3(L, Vd));
        Vec3 lo = pbr_lo(L, Vd, H, N, vis, al, param.y, param.z,
                         vec3(l.color[0], l.color[1], l.color[2]), u.shadow_on);
        Lo = (i == 0) ? lo : add3(Lo, lo);
    }
    Vec3 color = Lo;
    color = add3(color, scale3(mul3(vec3(0.3f, 0.3f, 0.3f), al), param.x));
    color = add3(color, el);
    return tonemap_gamma(color);
}

// Pixels of a launch over 64 x 4 blocks, as the resolves and the lighting take
// them.  Workgroups are dealt round-robin to the 8 XCDs: each XCD takes runs of
// 16 blocks, 64 x 64 pixels of a column, so that what neighbouring pixels share
// (vertices, texture blocks, shadow texels) is fetched into one XCD's L2
// (rows of blocks in launch order -> this, 3840 x 2160: shadow targets 48 -> 31
// us, lighting 223 -> 216; 1280 x 800: G-buffer 43 -> 38).  A wavefront
// takes 64/WT rows of WT pixels: 16 where it mostly gathers (lighting; 64 x 1
// -> 16 x 4 at 1920 x 1080 82 -> 71 us), 32 where it writes 19 planes as well
// (16 x 4 in the G-buffer resolve at 3840 x 2160: 303 -> 340 us).
constexpr int kChunkBlocks = 16;
__device__ __forceinline__ int chunk_remap(int id, int n)
{
    constexpr int C = kChunkBlocks;
    const int g = id / (8 * C) * (8 * C);
    return g + 8 * C > n ? id : g + (id & 7) * C + ((id >> 3) & (C - 1));
}

template <int WT>
__device__ __forceinline__ void block_px(int b, int nby, int &x, int &y)
{
    static_assert(WT == 16 || WT == 32, "4 wavefronts make 64 x 4");
    const int t = threadIdx.x, w = t >> 6;
    x = b / nby * 64 + w * WT % 64 + (t & (WT - 1));
    y = b % nby * 4 + (WT == 32 ? (w >> 1) * 2 : 0) + (t & 63) / WT;
}

template <int WT>
__device__ __forceinline__ void grid_px(int &x, int &y)
{
    block_px<WT>(chunk_remap(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y), gridDim.y, x, y);
}

// A workgroup's barrier that orders its LDS accesses alone: a __syncthreads()
// also waits for the global stores before it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

}  // namespace fgl
