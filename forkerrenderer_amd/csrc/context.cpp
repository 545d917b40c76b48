// context.cpp -- the fgl_* C ABI: device resources, ForkerGL-style state, pass
// orchestration on one HIP stream, readback, scene rendering.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <climits>
#include <cstddef>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <atomic>
#include <chrono>
#include <string>
#include <utility>
#include <mutex>
#include <vector>

#include "../../include/fgl.h"
#include "ctx_internal.hpp"
#include "mt_jump.hpp"
#include "fgl_kernels.hpp"
#include "host_io.hpp"

using namespace fgl;

namespace {

struct DevBuf {
    void *p = nullptr;
    size_t cap = 0;
};

constexpr int kFewVertices = 256;

struct ModelRes {
    float *pos = nullptr, *uv = nullptr, *nrm = nullptr, *tan = nullptr;
    int *vi = nullptr, *ti = nullptr, *ni = nullptr, *fmat = nullptr;
    int4 *tri = nullptr;       // the faces in spatial order
    float *corner = nullptr;   // per face corner: uv, normal, tangent, position (12 floats)
    int n_pos = 0, n_faces = 0;
    bool has_tan = false, pbr = false;
    // extent of the faces' corners and the longest face edge; bounded: they
    // are finite
    double lo[3], hi[3], edge = 0.0;
    bool bounded = false;
    std::vector<float> few;    // the positions, of a model with at most kFewVertices
};

struct TimedKernel {
    std::string name;
    hipEvent_t a, b;
};

}  // namespace

struct fgl_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    int TS = 16;

    std::vector<DevTexture> textures;
    std::vector<void *> texture_mem;
    DevBuf d_textures;
    bool textures_dirty = true;
    std::vector<DevMaterial> materials;
    DevBuf d_materials;
    bool materials_dirty = true;
    std::vector<ModelRes> models;
    // map bundles made so far, by their texture ids (A, Z, N, Y; -1: not held)
    struct Bundle {
        int ids[4];
        DevBundle b;
    };
    std::vector<Bundle> bundles;

    // ForkerGL state
    int W = 0, H = 0, SW = 0, SH = 0;
    float viewport[16], shadow_viewport[16], view[16], proj[16], light_space[16];
    float eye[3] = {0.f, 0.f, 0.f};
    std::vector<fgl_light> lights;
    int shadow_on = 1;
    fgl_shadow_cfg shadow_cfg;

    // targets
    DevBuf depth, fb, gbuf, ao, blur_tmp, shadow, shadow_depth, img, vis;
    int img_w = 0, img_h = 0;
    // Clears requested by fgl_init_* / fgl_clear_color that have not been
    // written yet: the next pass that covers every pixel applies them.
    bool pend_depth = false, pend_gbuf = false, pend_fb = false, pend_ao = false, pend_shadow = false;
    float fb_clear[3] = {0.f, 0.f, 0.f};
    int TS_shadow = 16;

    // current pass
    int pass = -1;
    struct Rec {
        int model;
        float m[16];
        bool has_normal;   // the shader's uNormalMatrix was given
        float n[9];
    };
    std::vector<Rec> draws;

    // pass scratch
    DevBuf d_draws, screen, rect, counts, offs, scan_tmp, keys, vals, keys_alt, vals_alt, sort_tmp,
        tile_start, tile_end, tri_v, big_list, counters, ndc_z, vary;
    // the direct rasteriser: pixel keys, NaN plane (all ones between passes),
    // large triangles, two passes' counters used in turn
    DevBuf key, key_nan, big, direct_ctr;
    size_t frame_px = 0;   // pixels of the frame begun, where its size is known before the shadow pass
    int direct_turn = 0;
    // forward pass with a stochastic shadow filter: per-pixel passing counts
    // (+ scan scratch), the passing fragments (triangle ids then pixels) and
    // the sort's other copy, its scratch, their shadow inputs, and each
    // winner's sample offset
    DevBuf frag_cnt, frag_tri, frag_alt, frag_tmp, frag_planes, frag_offs_px;
    bool frag_sorted_alt = false;
    std::vector<DevDraw> last_draws;
    uint32_t *h_total = nullptr;
    // pass counts published by the device into coherent pinned memory
    // (pair count, big-triangle count, sequence number), polled by the host
    uint32_t *h_pub = nullptr, *d_pub = nullptr;
    uint32_t pub_seq = 0;
    // the reference's random stream (device MtState), its sample buffers,
    // the PCSS sample offsets, the DoSSAO powf table
    DevBuf rng, rng_samples, rng_offs, ssao_pow3;
    uint32_t rng_seed = 5489u;
    // the parallel generator: base sequence, jumped chunk arrays, the chunks'
    // kept vectors, their counts and checkpoints, the jump polynomials uploaded
    // so far; the last fill and the vectors asked of it, for its commit
    DevBuf mt_base, mt_states, mt_vec, mt_ck, pcss_mm;
    DevBuf mt_lists[2];          // the jumps' read lists for the two chunk lengths
    int mt_lists_n[2] = {0, 0};
    MtFill fill{};
    uint32_t fill_n = 0;

    // device address of the allocation-free entry point's scratch array
    float *noalloc_scratch = nullptr;
    int number = 0;   // of this context among its device's (0: none was free)
    // what its calls have used of that array, and the event that other contexts'
    // calls wait for where they use the same
    size_t scratch_lo = 0, scratch_hi = 0;
    hipEvent_t scratch_event = nullptr;
    // neural AO still on its network grid (lao != nullptr): the AO target's
    // content until something reads or replaces it; owner = the network
    // whose buffers hold it
    NetAo ao_net{};
    const void *ao_net_owner = nullptr;
    std::vector<void *> naos;   // networks created on this context
    std::vector<void *> batches;

    // timing
    bool timing = false;
    std::string timing_only;   // empty: every timed kernel
    std::vector<TimedKernel> timed;
};

// Scratch of fgl_ssao_noalloc: the unblurred AO that the separable blur
// reads, FGL_SSAO_NOALLOC_MAX_PIXELS floats on every device the library runs
// on, held until the process ends.  On the host `scratch` names a stand-in,
// not device memory: host code only ever uses the address that
// hipGetSymbolAddress returns for the current device (scratch_address).
static __device__ __align__(256) float scratch[FGL_SSAO_NOALLOC_MAX_PIXELS];

static constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static float *g_scratch_ptr[kMaxDevices] = {};

// Address of `scratch` on `device`, which must be the current device; looked
// up once per device.
static hipError_t scratch_address(int device, float **out)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    if (!g_scratch_ptr[device]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_ptr[device] = (float *)p;
    }
    *out = g_scratch_ptr[device];
    return hipSuccess;
}

// Contexts on a device are numbered (the lowest free number), so that their
// calls use different parts of `scratch` where it holds a part for each: parts
// are the frame rounded up to a power of two, by the number.  Where two
// contexts' parts meet all the same (scratch_use), their calls are ordered.
static std::vector<fgl_ctx *> g_scratch_users[kMaxDevices];
static uint64_t g_ctx_numbers[kMaxDevices] = {};

static int take_number(int device)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    uint64_t &used = g_ctx_numbers[device];
    if (~used == 0) return 0;
    const int k = __builtin_ctzll(~used);
    used |= 1ull << k;
    return k + 1;
}

static void give_number(int device, int number)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (number > 0) g_ctx_numbers[device] &= ~(1ull << (number - 1));
}

// The part of `scratch` for a call of c on n pixels; c's stream waits for the
// calls of other contexts that used any of it.  The caller holds g_scratch_mu
// until its own launches are enqueued, so an event recorded on a context's
// stream comes after all of them.
static hipError_t scratch_use(fgl_ctx *c, size_t n, float **out)
{
    size_t part = 1 << 16;
    while (part < n) part *= 2;
    const size_t parts = FGL_SSAO_NOALLOC_MAX_PIXELS / part;   // n is at most that, a power of two
    const size_t lo = (c->number > 0 ? (size_t)(c->number - 1) % parts : 0) * part, hi = lo + n;
    for (fgl_ctx *o : g_scratch_users[c->device]) {
        if (o == c || o->scratch_hi <= lo || hi <= o->scratch_lo) continue;
        hipError_t e = hipEventRecord(o->scratch_event, o->stream);
        if (e == hipSuccess) e = hipStreamWaitEvent(c->stream, o->scratch_event, 0);
        if (e != hipSuccess) return e;
    }
    if (c->scratch_hi == 0) {
        g_scratch_users[c->device].push_back(c);
        c->scratch_lo = lo;
    }
    c->scratch_lo = lo < c->scratch_lo ? lo : c->scratch_lo;
    c->scratch_hi = hi > c->scratch_hi ? hi : c->scratch_hi;
    *out = c->noalloc_scratch + lo;
    return hipSuccess;
}

// c's stream is idle and takes no more calls.
static void scratch_leave(fgl_ctx *c)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    std::vector<fgl_ctx *> &users = g_scratch_users[c->device];
    for (size_t k = 0; k < users.size(); ++k)
        if (users[k] == c) {
            users.erase(users.begin() + (long)k);
            break;
        }
}

static int fail(fgl_ctx *c, int code, const std::string &msg)
{
    if (c) c->err = msg;
    return code;
}

#define HIPCHK(ctx, expr)                                                                   \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess)                                                               \
            return fail(ctx, FGL_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

static int ensure(fgl_ctx *c, DevBuf &b, size_t bytes)
{
    if (bytes <= b.cap && b.p) return FGL_OK;
    if (b.p) {
        HIPCHK(c, hipStreamSynchronize(c->stream));   // no kernel may still use it
        (void)hipFree(b.p);
        b.p = nullptr;
        b.cap = 0;
    }
    size_t want = bytes < 256 ? 256 : bytes;
    if (hipMalloc(&b.p, want) != hipSuccess) {
        b.p = nullptr;
        return fail(c, FGL_ERR_NOMEM, "hipMalloc of " + std::to_string(want) + " bytes failed");
    }
    b.cap = want;
    return FGL_OK;
}

// ensure() for memory that the caller can do without: no error without it.
static bool room(fgl_ctx *c, DevBuf &b, size_t bytes)
{
    if (bytes <= b.cap && b.p) return true;
    if (b.p) {
        if (hipStreamSynchronize(c->stream) != hipSuccess) return false;
        (void)hipFree(b.p);
        b.p = nullptr;
        b.cap = 0;
    }
    if (hipMalloc(&b.p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        b.p = nullptr;
        return false;
    }
    b.cap = bytes;
    return true;
}

static void free_buf(DevBuf &b)
{
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.cap = 0;
}

// ---------------- timing ----------------

struct KernelTimer {
    fgl_ctx *c;
    TimedKernel tk;
    bool on;
    KernelTimer(fgl_ctx *ctx, const char *name)
        : c(ctx), on(ctx->timing && (ctx->timing_only.empty() || ctx->timing_only == name))
    {
        if (!on) return;
        tk.name = name;
        // a diagnostic: when its events cannot be made, the span is not timed
        if (hipEventCreate(&tk.a) != hipSuccess) {
            on = false;
            return;
        }
        if (hipEventCreate(&tk.b) != hipSuccess || hipEventRecord(tk.a, c->stream) != hipSuccess) {
            (void)hipEventDestroy(tk.a);
            on = false;
        }
    }
    ~KernelTimer()
    {
        if (!on) return;
        (void)hipEventRecord(tk.b, c->stream);
        c->timed.push_back(tk);
    }
};

// Two device counters to the host without a stream synchronisation: a
// one-thread kernel writes them and a fresh sequence number into coherent
// pinned memory, and the host polls for the sequence number (the GPU then
// idles only for the poll and the next launch, not for a full
// synchronisation).  A poll that outlasts a second falls back to
// synchronising the stream, which reports a failed kernel.
static int read_counts(fgl_ctx *c, const uint32_t *a, const uint32_t *b, uint32_t &va, uint32_t &vb)
{
    const uint32_t seq = ++c->pub_seq;
    launch_publish2(a, b, seq, c->d_pub, c->stream);
    HIPCHK(c, hipGetLastError());
    volatile uint32_t *pub = c->h_pub;
    auto t0 = std::chrono::steady_clock::now();
    for (uint32_t spin = 0; pub[2] != seq; ++spin) {
        if ((spin & 1023u) == 1023u &&
            std::chrono::steady_clock::now() - t0 > std::chrono::seconds(1)) {
            HIPCHK(c, hipStreamSynchronize(c->stream));
            if (pub[2] != seq) return fail(c, FGL_ERR_DEVICE, "pass counts were not published");
            break;
        }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    va = pub[0];
    vb = pub[1];
    return FGL_OK;
}

// Restarts the context's random stream at its seed (std::mt19937(seed)).
static int rng_restart(fgl_ctx *c)
{
    MtState st;
    mt_seed_state(c->rng_seed, st);
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(c->rng.p, &st, sizeof(st), hipMemcpyHostToDevice));
    return FGL_OK;
}

template <typename T>
static int upload_array(fgl_ctx *c, T **dst, const T *src, size_t n)
{
    *dst = nullptr;
    HIPCHK(c, hipMalloc((void **)dst, (n ? n : 1) * sizeof(T)));
    if (n) HIPCHK(c, hipMemcpy(*dst, src, n * sizeof(T), hipMemcpyHostToDevice));
    return FGL_OK;
}

extern "C" {

int fgl_ctx_create(int device, fgl_ctx **out)
{
    if (!out) return FGL_ERR_INVALID;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return FGL_ERR_DEVICE;
    if (device < 0 || device >= n) return FGL_ERR_INVALID;
    if (hipSetDevice(device) != hipSuccess) return FGL_ERR_DEVICE;
    fgl_ctx *c = new fgl_ctx();
    c->device = device;
    if (scratch_address(device, &c->noalloc_scratch) != hipSuccess) {
        delete c;
        return FGL_ERR_DEVICE;
    }
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return FGL_ERR_DEVICE;
    }
    if (hipHostMalloc((void **)&c->h_total, sizeof(uint32_t) * 4, hipHostMallocDefault) != hipSuccess) {
        (void)hipStreamDestroy(c->stream);
        delete c;
        return FGL_ERR_NOMEM;
    }
    if (hipHostMalloc((void **)&c->h_pub, 64, hipHostMallocCoherent | hipHostMallocMapped) != hipSuccess ||
        hipHostGetDevicePointer((void **)&c->d_pub, c->h_pub, 0) != hipSuccess ||
        hipEventCreateWithFlags(&c->scratch_event, hipEventDisableTiming) != hipSuccess) {
        if (c->h_pub) (void)hipHostFree(c->h_pub);
        (void)hipHostFree(c->h_total);
        (void)hipStreamDestroy(c->stream);
        delete c;
        return FGL_ERR_NOMEM;
    }
    c->number = take_number(device);
    std::memset(c->h_pub, 0, 64);
    float I[16] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1};
    std::memcpy(c->viewport, I, sizeof(I));
    std::memcpy(c->shadow_viewport, I, sizeof(I));
    std::memcpy(c->view, I, sizeof(I));
    std::memcpy(c->proj, I, sizeof(I));
    std::memcpy(c->light_space, I, sizeof(I));
    std::memset(&c->shadow_cfg, 0, sizeof(c->shadow_cfg));
    // Render::DoSSAO's 1 - occlusion is k/32 (k = 0..32, exact); its
    // Pow(x, 3) is the host libm's powf, as in the reference.
    float pow3[33];
    for (int k = 0; k <= 32; ++k) {
        float occ = 0.f;
        for (int j = 0; j < k; ++j) occ += (1.f / 32) * 1.f;
        pow3[k] = powf(1.f - occ, 3);
    }
    if (ensure(c, c->ssao_pow3, sizeof(pow3)) || ensure(c, c->rng, sizeof(MtState)) ||
        hipMemcpy(c->ssao_pow3.p, pow3, sizeof(pow3), hipMemcpyHostToDevice) != hipSuccess ||
        rng_restart(c) != FGL_OK) {
        fgl_ctx_destroy(c);
        return FGL_ERR_NOMEM;
    }
    *out = c;
    return FGL_OK;
}

void fgl_ctx_destroy(fgl_ctx *c)
{
    if (!c) return;
    for (void *n : c->naos) nao_detach(n);   // networks outliving their context stop using it
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    scratch_leave(c);
    for (void *b : c->batches) batch_detach(b);
    for (void *p : c->texture_mem) (void)hipFree(p);
    for (auto &m : c->models) {
        (void)hipFree(m.pos); (void)hipFree(m.uv); (void)hipFree(m.nrm);
        if (m.tan) (void)hipFree(m.tan);
        (void)hipFree(m.vi); (void)hipFree(m.ti); (void)hipFree(m.ni); (void)hipFree(m.fmat); (void)hipFree(m.corner); (void)hipFree(m.tri);
    }
    DevBuf *bufs[] = {&c->d_textures, &c->d_materials, &c->depth, &c->fb, &c->gbuf, &c->ao,
                      &c->blur_tmp, &c->shadow, &c->shadow_depth, &c->img, &c->vis, &c->d_draws,
                      &c->rng, &c->rng_samples, &c->rng_offs, &c->ssao_pow3,
                      &c->mt_base, &c->mt_states, &c->mt_vec, &c->mt_ck, &c->pcss_mm, &c->mt_lists[0], &c->mt_lists[1],
                      &c->screen, &c->rect, &c->counts, &c->offs, &c->scan_tmp, &c->keys,
                      &c->vals, &c->keys_alt, &c->vals_alt, &c->sort_tmp, &c->tile_start,
                      &c->tile_end, &c->tri_v, &c->big_list, &c->counters, &c->ndc_z, &c->vary,
                      &c->key, &c->key_nan, &c->big, &c->direct_ctr,
                      &c->frag_cnt, &c->frag_tri, &c->frag_alt, &c->frag_tmp, &c->frag_planes,
                      &c->frag_offs_px};
    for (DevBuf *b : bufs) free_buf(*b);
    for (auto &t : c->timed) { (void)hipEventDestroy(t.a); (void)hipEventDestroy(t.b); }
    if (c->h_total) (void)hipHostFree(c->h_total);
    if (c->h_pub) (void)hipHostFree(c->h_pub);
    (void)hipEventDestroy(c->scratch_event);
    (void)hipStreamDestroy(c->stream);
    give_number(c->device, c->number);
    delete c;
}

const char *fgl_last_error(const fgl_ctx *c) { return c ? c->err.c_str() : "null context"; }

int fgl_sync(fgl_ctx *c)
{
    if (!c) return FGL_ERR_INVALID;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return FGL_OK;
}

int fgl_set_tile_size(fgl_ctx *c, int tile)
{
    if (!c) return FGL_ERR_INVALID;
    if (tile != 8 && tile != 16 && tile != 32) return fail(c, FGL_ERR_INVALID, "tile must be 8, 16 or 32");
    c->TS = tile;
    c->TS_shadow = tile;
    return FGL_OK;
}

int fgl_set_pass_tile_size(fgl_ctx *c, int pass, int tile)
{
    if (!c) return FGL_ERR_INVALID;
    if (tile != 8 && tile != 16 && tile != 32) return fail(c, FGL_ERR_INVALID, "tile must be 8, 16 or 32");
    if (pass == FGL_PASS_SHADOW) c->TS_shadow = tile;
    else if (pass == FGL_PASS_FORWARD || pass == FGL_PASS_GEOMETRY) c->TS = tile;
    else return fail(c, FGL_ERR_INVALID, "pass has no raster stage");
    return FGL_OK;
}

int fgl_get_pass_tile_size(fgl_ctx *c, int pass, int *tile)
{
    if (!c || !tile) return FGL_ERR_INVALID;
    *tile = (pass == FGL_PASS_SHADOW) ? c->TS_shadow : c->TS;
    return FGL_OK;
}

// ---------------- resources ----------------

int fgl_upload_texture(fgl_ctx *c, int w, int h, int bpp, const uint8_t *bytes, int wrap,
                       int filter, int *out_id)
{
    if (!c || !bytes || !out_id) return FGL_ERR_INVALID;
    if (w <= 0 || h <= 0 || (bpp != 1 && bpp != 3 && bpp != 4) || wrap < 0 || wrap > 3 ||
        filter < 0 || filter > 1)
        return fail(c, FGL_ERR_INVALID, "bad texture parameters");
    std::vector<uint32_t> packed((size_t)w * h);
    std::vector<uint8_t> zb((size_t)w * h);
    for (size_t i = 0; i < packed.size(); ++i) {
        const uint8_t *p = bytes + i * bpp;
        uint32_t b = p[0], g = bpp > 1 ? p[1] : 0, r = bpp > 2 ? p[2] : 0;
        packed[i] = r | (g << 8) | (b << 16);
        zb[i] = (uint8_t)b;
    }
    void *mem = nullptr, *zmem = nullptr;
    HIPCHK(c, hipMalloc(&mem, packed.size() * 4));
    c->texture_mem.push_back(mem);
    HIPCHK(c, hipMalloc(&zmem, zb.size()));
    c->texture_mem.push_back(zmem);
    HIPCHK(c, hipMemcpy(mem, packed.data(), packed.size() * 4, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(zmem, zb.data(), zb.size(), hipMemcpyHostToDevice));
    DevTexture t;
    t.texels = (const uint32_t *)mem;
    t.zb = (const uint8_t *)zmem;
    t.w = w; t.h = h; t.wrap = wrap; t.filter = filter;
    c->textures.push_back(t);
    c->textures_dirty = true;
    *out_id = (int)c->textures.size() - 1;
    return FGL_OK;
}

int fgl_upload_material(fgl_ctx *c, const fgl_material *m, int *out_id)
{
    if (!c || !m || !out_id) return FGL_ERR_INVALID;
    const int32_t ids[] = {m->map_kd, m->map_ks, m->map_ke, m->map_bump, m->map_base,
                           m->map_rough, m->map_metal, m->map_ao, m->map_pbr_ke};
    for (int id : ids)
        if (id < -1 || id >= (int)c->textures.size())
            return fail(c, FGL_ERR_INVALID, "material references an unknown texture id");
    DevMaterial d{};
    static_assert(offsetof(DevMaterial, bundle) >= sizeof(fgl_material) &&
                      offsetof(DevMaterial, map_pbr_ke) == offsetof(fgl_material, map_pbr_ke), "material layout");
    std::memcpy((void *)&d, m, sizeof(fgl_material));
    c->materials.push_back(d);
    c->materials_dirty = true;
    *out_id = (int)c->materials.size() - 1;
    return FGL_OK;
}

// The bundle (DevBundle) of material k's maps for the Blinn-Phong (0) or PBR
// (1) shaders, made on first use from the maps that share the first one's
// size, wrap and filter; a single map has none, and maps without room for it go
// on by themselves.
static int ensure_bundle(fgl_ctx *c, int k, int pbr)
{
    DevMaterial &m = c->materials[k];
    if (m.bundle[pbr].t) return FGL_OK;
    fgl_ctx::Bundle n{{pbr ? m.map_base : m.map_kd, pbr ? m.map_rough : m.map_ks, m.map_bump, pbr ? m.map_metal : -1}, {}};
    const DevTexture *first = nullptr, *t[4];
    int maps = 0;
    for (int j = 0; j < 4; ++j) {
        t[j] = n.ids[j] >= 0 ? &c->textures[n.ids[j]] : nullptr;
        if (t[j] && !first) first = t[j];
        if (t[j] && (t[j]->w != first->w || t[j]->h != first->h || t[j]->wrap != first->wrap || t[j]->filter != first->filter)) {
            t[j] = nullptr;
            n.ids[j] = -1;
        }
        if (t[j]) {
            n.b.has |= 1 << j;
            ++maps;
        }
    }
    if (maps < 2) return FGL_OK;
    for (const fgl_ctx::Bundle &o : c->bundles)
        if (std::memcmp(o.ids, n.ids, sizeof(n.ids)) == 0) {
            m.bundle[pbr] = o.b;
            c->materials_dirty = true;
            return FGL_OK;
        }
    const int w = first->w, h = first->h;
    void *mem = nullptr;
    if (hipMalloc(&mem, (size_t)((w + 3) / 4) * ((h + 3) / 4) * 16 * sizeof(uint2)) != hipSuccess) {
        (void)hipGetLastError();
        return FGL_OK;
    }
    c->texture_mem.push_back(mem);
    launch_bundle(w, h, t[0] ? t[0]->texels : nullptr, t[1] ? t[1]->zb : nullptr, t[2] ? t[2]->texels : nullptr,
                  t[3] ? t[3]->zb : nullptr, (uint2 *)mem, c->stream);
    HIPCHK(c, hipGetLastError());
    n.b.t = (const uint2 *)mem;
    n.b.w = w;
    n.b.h = h;
    n.b.wrap = first->wrap;
    n.b.filter = first->filter;
    c->bundles.push_back(n);
    m.bundle[pbr] = n.b;
    c->materials_dirty = true;
    return FGL_OK;
}

// The faces in the order of a Morton curve through their first corners (10
// bits an axis of the model's extent; face order breaks ties), and each
// position's place in the order of first use (unused positions last).
static void spatial_order(const fgl_model_desc *d, std::vector<int32_t> &order, std::vector<int32_t> &rank)
{
    const size_t nf = (size_t)d->n_faces;
    float lo[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, hi[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
    for (size_t f = 0; f < nf; ++f)
        for (int j = 0; j < 3; ++j) {
            const float x = d->pos[3 * (size_t)d->vi[3 * f] + j];
            if (x < lo[j]) lo[j] = x;
            if (x > hi[j]) hi[j] = x;
        }
    float scale[3];
    for (int j = 0; j < 3; ++j) {
        scale[j] = 1023.f / (hi[j] - lo[j]);
        if (!std::isfinite(scale[j])) scale[j] = 0.f;
    }
    auto spread = [](uint32_t x) {
        x = (x | x << 16) & 0x030000ffu;
        x = (x | x << 8) & 0x0300f00fu;
        x = (x | x << 4) & 0x030c30c3u;
        return (x | x << 2) & 0x09249249u;
    };
    std::vector<uint32_t> key(nf), key2(nf);
    std::vector<int32_t> tmp(nf);
    order.resize(nf);
    for (size_t f = 0; f < nf; ++f) {
        uint32_t q[3];
        for (int j = 0; j < 3; ++j) {
            const float x = (d->pos[3 * (size_t)d->vi[3 * f] + j] - lo[j]) * scale[j];
            q[j] = x >= 0.f && x <= 1023.f ? (uint32_t)x : 0u;   // also a NaN
        }
        key[f] = spread(q[0]) | spread(q[1]) << 1 | spread(q[2]) << 2;
        order[f] = (int32_t)f;
    }
    for (int shift = 0; shift < 30; shift += 10) {   // stable counting sort, ten bits a pass
        uint32_t at[1025] = {0};
        for (size_t f = 0; f < nf; ++f) ++at[(key[f] >> shift & 1023u) + 1];
        for (int k = 0; k < 1024; ++k) at[k + 1] += at[k];
        for (size_t f = 0; f < nf; ++f) {
            const uint32_t o = at[key[f] >> shift & 1023u]++;
            key2[o] = key[f];
            tmp[o] = order[f];
        }
        key.swap(key2);
        order.swap(tmp);
    }
    rank.assign((size_t)d->n_pos, -1);
    int32_t next = 0;
    for (size_t k = 0; k < nf; ++k)
        for (int j = 0; j < 3; ++j) {
            int32_t &r = rank[d->vi[3 * (size_t)order[k] + j]];
            if (r < 0) r = next++;
        }
    for (int32_t &r : rank)
        if (r < 0) r = next++;
}

int fgl_upload_model(fgl_ctx *c, const fgl_model_desc *d, int *out_id)
{
    if (!c || !d || !out_id) return FGL_ERR_INVALID;
    if (d->n_pos <= 0 || d->n_uv <= 0 || d->n_nrm <= 0 || d->n_faces < 0 || !d->pos || !d->uv ||
        !d->nrm || (d->n_faces > 0 && (!d->vi || !d->ti || !d->ni || !d->face_material)))
        return fail(c, FGL_ERR_INVALID, "bad model description");
    size_t nf = (size_t)d->n_faces;
    for (size_t i = 0; i < 3 * nf; ++i)
        if (d->vi[i] < 0 || d->vi[i] >= d->n_pos || d->ti[i] < 0 || d->ti[i] >= d->n_uv ||
            d->ni[i] < 0 || d->ni[i] >= d->n_nrm)
            return fail(c, FGL_ERR_INVALID, "face index out of range");
    for (size_t f = 0; f < nf; ++f)
        if (d->face_material[f] < 0 || d->face_material[f] >= (int)c->materials.size())
            return fail(c, FGL_ERR_INVALID, "face material out of range");
    ModelRes m;
    int rc;
    for (size_t f = 0; f < nf; ++f)
        if ((f == 0 || d->face_material[f] != d->face_material[f - 1]) &&
            (rc = ensure_bundle(c, d->face_material[f], d->support_pbr != 0)))
            return rc;
    // The positions are kept in the order the faces, taken in spatial order,
    // first use them, so that neighbouring triangles' vertex records are
    // neighbours; vi indexes that order.
    std::vector<int32_t> order, rank, vi;
    std::vector<float> pos;
    spatial_order(d, order, rank);
    pos.resize(3 * (size_t)d->n_pos);
    for (int k = 0; k < d->n_pos; ++k) std::memcpy(&pos[3 * (size_t)rank[k]], d->pos + 3 * (size_t)k, 3 * sizeof(float));
    vi.resize(3 * nf);
    for (size_t k = 0; k < 3 * nf; ++k) vi[k] = rank[d->vi[k]];
    std::vector<int4> tri(nf);
    for (size_t k = 0; k < nf; ++k) {
        const int f = order[k];
        tri[k] = make_int4(vi[3 * (size_t)f], vi[3 * (size_t)f + 1], vi[3 * (size_t)f + 2], f);
    }
    if ((rc = upload_array(c, &m.pos, pos.data(), pos.size()))) return rc;
    if ((rc = upload_array(c, &m.tri, tri.data(), nf))) return rc;
    if ((rc = upload_array(c, &m.uv, d->uv, 2 * (size_t)d->n_uv))) return rc;
    if ((rc = upload_array(c, &m.nrm, d->nrm, 3 * (size_t)d->n_nrm))) return rc;
    if (d->tan) {   // in the positions' order
        for (int k = 0; k < d->n_pos; ++k)
            std::memcpy(&pos[3 * (size_t)rank[k]], d->tan + 3 * (size_t)k, 3 * sizeof(float));
        if ((rc = upload_array(c, &m.tan, pos.data(), pos.size()))) return rc;
    }
    if ((rc = upload_array(c, &m.vi, (const int *)vi.data(), 3 * nf))) return rc;
    if ((rc = upload_array(c, &m.ti, (const int *)d->ti, 3 * nf))) return rc;
    if ((rc = upload_array(c, &m.ni, (const int *)d->ni, 3 * nf))) return rc;
    if ((rc = upload_array(c, &m.fmat, (const int *)d->face_material, nf))) return rc;
    HIPCHK(c, hipMalloc((void **)&m.corner, (nf ? 3 * nf * 12 : 1) * sizeof(float)));
    launch_corners(m.pos, m.uv, m.nrm, m.tan, m.vi, m.ti, m.ni, 3 * nf, (float4 *)m.corner, c->stream);
    HIPCHK(c, hipGetLastError());
    for (int k = 0; k < 3; ++k) {
        m.lo[k] = HUGE_VAL;
        m.hi[k] = -HUGE_VAL;
    }
    bool finite = nf > 0;
    double edge2 = 0.0;
    for (size_t f = 0; f < nf; ++f) {
        const float *p[3];
        for (int k = 0; k < 3; ++k) p[k] = d->pos + 3 * (size_t)d->vi[3 * f + k];
        for (int k = 0; k < 3; ++k) {
            double e2 = 0.0;
            for (int j = 0; j < 3; ++j) {
                const double x = p[k][j], e = x - p[(k + 1) % 3][j];
                finite = finite && std::isfinite(x);
                m.lo[j] = x < m.lo[j] ? x : m.lo[j];
                m.hi[j] = x > m.hi[j] ? x : m.hi[j];
                e2 += e * e;
            }
            edge2 = e2 > edge2 ? e2 : edge2;
        }
    }
    m.edge = std::sqrt(edge2);
    m.bounded = finite;
    if (d->n_pos <= kFewVertices) m.few.assign(d->pos, d->pos + 3 * (size_t)d->n_pos);
    m.n_pos = d->n_pos;
    m.n_faces = d->n_faces;
    m.has_tan = d->tan != nullptr;
    m.pbr = d->support_pbr != 0;
    c->models.push_back(m);
    *out_id = (int)c->models.size() - 1;
    return FGL_OK;
}

// ---------------- state ----------------

static int flush_pass(fgl_ctx *c);

// Writes the clear values still pending on the targets named by the flags.
static int materialize(fgl_ctx *c, bool depth, bool gbuf, bool fb, bool ao, bool shadow)
{
    const size_t P = (size_t)c->W * c->H, SP = (size_t)c->SW * c->SH;
    if (depth && c->pend_depth) { launch_fill_f32((float *)c->depth.p, FLT_MAX, P, c->stream); c->pend_depth = false; }
    if (gbuf && c->pend_gbuf) { launch_fill_f32((float *)c->gbuf.p, 0.f, kGbufPlanes * P, c->stream); c->pend_gbuf = false; }
    if (fb && c->pend_fb) {
        for (int k = 0; k < 3; ++k) launch_fill_f32((float *)c->fb.p + k * P, c->fb_clear[k], P, c->stream);
        c->pend_fb = false;
    }
    if (ao && c->ao_net.lao) {
        nao_launch_up(c->ao_net, c->W, c->H, (float *)c->ao.p, c->stream);
        c->ao_net = NetAo{};
        c->ao_net_owner = nullptr;
    }
    if (ao && c->pend_ao) { launch_fill_f32((float *)c->ao.p, 1.f, P, c->stream); c->pend_ao = false; }
    if (shadow && c->pend_shadow) {
        launch_fill_f32((float *)c->shadow.p, 0.f, SP, c->stream);
        launch_fill_f32((float *)c->shadow_depth.p, FLT_MAX, SP, c->stream);
        c->pend_shadow = false;
    }
    HIPCHK(c, hipGetLastError());
    return FGL_OK;
}

// InitFrameBuffer (zero), InitDepthBuffer (FLT_MAX), InitGeometryBuffers
// (zero, AO one): recorded, then written by the first pass that covers the
// targets (or materialised before any partial use).
int fgl_init_targets(fgl_ctx *c, int w, int h)
{
    if (!c) return FGL_ERR_INVALID;
    if (w <= 0 || h <= 0 || w > 16384 || h > 16384) return fail(c, FGL_ERR_INVALID, "bad target size");
    int rc = flush_pass(c);
    if (rc) return rc;
    size_t P = (size_t)w * h;
    if ((rc = ensure(c, c->depth, P * 4)) || (rc = ensure(c, c->fb, 3 * P * 4)) ||
        (rc = ensure(c, c->gbuf, kGbufPlanes * P * 4)) || (rc = ensure(c, c->ao, P * 4)) ||
        (rc = ensure(c, c->blur_tmp, P * 4)))
        return rc;
    c->W = w;
    c->H = h;
    c->pend_depth = c->pend_gbuf = c->pend_fb = c->pend_ao = true;
    c->ao_net = NetAo{};
    c->ao_net_owner = nullptr;
    c->fb_clear[0] = c->fb_clear[1] = c->fb_clear[2] = 0.f;
    return FGL_OK;
}

// One of InitFrameBuffer / InitDepthBuffer / InitGeometryBuffers
// (forkergl.cpp:55-81).  The main targets share one size; initialising one
// at a new size re-initialises all of them.
int fgl_init_buffer(fgl_ctx *c, int which, int w, int h)
{
    if (!c) return FGL_ERR_INVALID;
    if (which == FGL_TARGET_SHADOW) return fgl_init_shadow_buffer(c, w, h);
    if (which != FGL_TARGET_FRAME && which != FGL_TARGET_DEPTH && which != FGL_TARGET_GBUFFER)
        return fail(c, FGL_ERR_INVALID, "fgl_init_buffer: FRAME, DEPTH, GBUFFER or SHADOW");
    if (!c->depth.p || w != c->W || h != c->H) return fgl_init_targets(c, w, h);
    int rc = flush_pass(c);
    if (rc) return rc;
    if (which == FGL_TARGET_FRAME) {
        c->pend_fb = true;
        c->fb_clear[0] = c->fb_clear[1] = c->fb_clear[2] = 0.f;
    } else if (which == FGL_TARGET_DEPTH) {
        c->pend_depth = true;
    } else {
        c->pend_gbuf = c->pend_ao = true;
        c->ao_net = NetAo{};
        c->ao_net_owner = nullptr;
    }
    return FGL_OK;
}

int fgl_init_shadow_buffer(fgl_ctx *c, int w, int h)
{
    if (!c) return FGL_ERR_INVALID;
    if (w <= 0 || h <= 0 || w > 16384 || h > 16384) return fail(c, FGL_ERR_INVALID, "bad shadow size");
    int rc = flush_pass(c);
    if (rc) return rc;
    size_t P = (size_t)w * h;
    if ((rc = ensure(c, c->shadow, P * 4)) || (rc = ensure(c, c->shadow_depth, P * 4))) return rc;
    c->SW = w;
    c->SH = h;
    c->pend_shadow = true;
    return FGL_OK;
}

int fgl_clear_color(fgl_ctx *c, float r, float g, float b)
{
    if (!c || !c->fb.p) return fail(c, FGL_ERR_INVALID, "targets not initialised");
    int rc = flush_pass(c);
    if (rc) return rc;
    c->fb_clear[0] = r;
    c->fb_clear[1] = g;
    c->fb_clear[2] = b;
    c->pend_fb = true;  // overwrites every pixel, so it replaces any pending clear
    return FGL_OK;
}

// The draws recorded so far were issued under the current ForkerGL state
// (in the reference each draw runs at once with its shader's uniforms,
// src/model.cpp:77-90).  A setter that changes state the pending draws read
// (matrices, viewport, eye, lights, shadow settings) rasterises them first,
// so every draw sees the values set before it; setting an equal value keeps
// the pass batched.
static int flush_if_changed(fgl_ctx *c, const void *cur, const void *next, size_t bytes)
{
    if (c->draws.empty() || std::memcmp(cur, next, bytes) == 0) return FGL_OK;
    return flush_pass(c);
}

int fgl_set_viewport(fgl_ctx *c, int shadow, int x, int y, int w, int h)
{
    if (!c) return FGL_ERR_INVALID;
    float vp[16];
    make_viewport(x, y, w, h, vp);
    float *dst = shadow ? c->shadow_viewport : c->viewport;
    int rc = flush_if_changed(c, dst, vp, sizeof(vp));
    if (rc) return rc;
    std::memcpy(dst, vp, sizeof(vp));
    return FGL_OK;
}

int fgl_set_matrix(fgl_ctx *c, int which, const float m[16])
{
    if (!c || !m) return FGL_ERR_INVALID;
    float *dst = which == FGL_MAT_VIEW ? c->view
               : which == FGL_MAT_PROJ ? c->proj
               : which == FGL_MAT_LIGHT_SPACE ? c->light_space : nullptr;
    if (!dst) return fail(c, FGL_ERR_INVALID, "unknown matrix");
    int rc = flush_if_changed(c, dst, m, 16 * sizeof(float));
    if (rc) return rc;
    std::memcpy(dst, m, 16 * sizeof(float));
    return FGL_OK;
}

int fgl_set_eye(fgl_ctx *c, const float eye[3])
{
    if (!c || !eye) return FGL_ERR_INVALID;
    int rc = flush_if_changed(c, c->eye, eye, 3 * sizeof(float));
    if (rc) return rc;
    std::memcpy(c->eye, eye, 3 * sizeof(float));
    return FGL_OK;
}

int fgl_set_lights(fgl_ctx *c, int n, const fgl_light *lights)
{
    if (!c || n < 0 || n > FGL_MAX_LIGHTS || (n && !lights)) return fail(c, FGL_ERR_INVALID, "bad lights");
    if (!c->draws.empty() &&
        (n != (int)c->lights.size() || (n && std::memcmp(c->lights.data(), lights, n * sizeof(fgl_light)) != 0))) {
        int rc = flush_pass(c);
        if (rc) return rc;
    }
    c->lights.assign(lights, lights + n);
    return FGL_OK;
}

int fgl_set_shadow(fgl_ctx *c, int on, const fgl_shadow_cfg *cfg)
{
    if (!c) return FGL_ERR_INVALID;
    if (cfg) {
        if (cfg->mode < 0 || cfg->mode > 5 || cfg->n_blocker < 0 || cfg->n_blocker > FGL_MAX_DISK ||
            cfg->n_pcf < 0 || cfg->n_pcf > FGL_MAX_DISK || (cfg->mode == 3 && (cfg->grid < 1 || cfg->grid > 9)) ||
            ((cfg->mode == 1 || cfg->mode == 2 || cfg->mode >= 4) && cfg->n_pcf < 1) ||
            (cfg->mode == 5 && cfg->n_blocker < 1))
            return fail(c, FGL_ERR_INVALID, "bad shadow filter configuration");
    }
    if (!c->draws.empty() && ((on ? 1 : 0) != c->shadow_on ||
                              (cfg && std::memcmp(cfg, &c->shadow_cfg, sizeof(fgl_shadow_cfg)) != 0))) {
        int rc = flush_pass(c);
        if (rc) return rc;
    }
    if (cfg) c->shadow_cfg = *cfg;
    c->shadow_on = on ? 1 : 0;
    return FGL_OK;
}

static void build_uniforms(fgl_ctx *c, FrameUniforms &u)
{
    std::memset(&u, 0, sizeof(u));
    std::memcpy(u.view, c->view, sizeof(u.view));
    std::memcpy(u.proj, c->proj, sizeof(u.proj));
    std::memcpy(u.light_space, c->light_space, sizeof(u.light_space));
    std::memcpy(u.viewport, c->viewport, sizeof(u.viewport));
    std::memcpy(u.shadow_viewport, c->shadow_viewport, sizeof(u.shadow_viewport));
    mat_mul(c->proj, c->view, u.vp);
    std::memcpy(u.eye, c->eye, sizeof(u.eye));
    u.shadow_on = c->shadow_on;
    u.n_lights = (int)c->lights.size();
    for (int i = 0; i < u.n_lights; ++i) {
        u.lights[i].type = c->lights[i].type;
        std::memcpy(u.lights[i].vec, c->lights[i].vec, sizeof(float) * 3);
        std::memcpy(u.lights[i].color, c->lights[i].color, sizeof(float) * 3);
    }
    u.W = c->W;
    u.H = c->H;
    u.SW = c->SW;
    u.SH = c->SH;
    const fgl_shadow_cfg &s = c->shadow_cfg;
    u.shadow.mode = s.mode;
    u.shadow.grid = s.grid;
    u.shadow.n_blocker = s.n_blocker;
    u.shadow.n_pcf = s.n_pcf;
    u.shadow.pcf_filter = s.pcf_filter;
    u.shadow.area_light = s.area_light;
    u.shadow.blocker_filter = s.blocker_filter;
    u.shadow.pcss_filter = s.pcss_filter;
    std::memcpy(u.shadow.blocker_disk, s.blocker_disk, sizeof(u.shadow.blocker_disk));
    std::memcpy(u.shadow.pcf_disk, s.pcf_disk, sizeof(u.shadow.pcf_disk));
    for (int i = 0; i < 2 * kMaxDisk; ++i)
        u.shadow.blocker_off[i] = (float)((double)s.blocker_disk[i] * s.blocker_filter);
}

static int upload_tables(fgl_ctx *c)
{
    int rc;
    if (c->textures_dirty) {
        if ((rc = ensure(c, c->d_textures, (c->textures.size() + 1) * sizeof(DevTexture)))) return rc;
        if (!c->textures.empty())
            HIPCHK(c, hipMemcpyAsync(c->d_textures.p, c->textures.data(),
                                     c->textures.size() * sizeof(DevTexture),
                                     hipMemcpyHostToDevice, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        c->textures_dirty = false;
    }
    if (c->materials_dirty) {
        if ((rc = ensure(c, c->d_materials, (c->materials.size() + 1) * sizeof(DevMaterial)))) return rc;
        if (!c->materials.empty())
            HIPCHK(c, hipMemcpyAsync(c->d_materials.p, c->materials.data(),
                                     c->materials.size() * sizeof(DevMaterial),
                                     hipMemcpyHostToDevice, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        c->materials_dirty = false;
    }
    return FGL_OK;
}

// ---------------- passes ----------------

static int flush_pass(fgl_ctx *c);

int fgl_begin_pass(fgl_ctx *c, int pass)
{
    if (!c) return FGL_ERR_INVALID;
    if (pass != FGL_PASS_FORWARD && pass != FGL_PASS_GEOMETRY && pass != FGL_PASS_LIGHTING &&
        pass != FGL_PASS_SHADOW)
        return fail(c, FGL_ERR_INVALID, "unknown pass");
    int rc = flush_pass(c);
    if (rc) return rc;
    c->pass = pass;
    return FGL_OK;
}

int fgl_draw_model(fgl_ctx *c, int model, const float model_matrix[16])
{
    if (!c || !model_matrix) return FGL_ERR_INVALID;
    if (model < 0 || model >= (int)c->models.size()) return fail(c, FGL_ERR_INVALID, "unknown model");
    if (c->pass != FGL_PASS_FORWARD && c->pass != FGL_PASS_GEOMETRY && c->pass != FGL_PASS_SHADOW)
        return fail(c, FGL_ERR_INVALID, "no raster pass begun");
    fgl_ctx::Rec r;
    r.model = model;
    std::memcpy(r.m, model_matrix, sizeof(r.m));
    r.has_normal = false;
    c->draws.push_back(r);
    return FGL_OK;
}

int fgl_draw_model_normal(fgl_ctx *c, int model, const float model_matrix[16], const float normal_matrix[9])
{
    if (!c || !normal_matrix) return FGL_ERR_INVALID;
    int rc = fgl_draw_model(c, model, model_matrix);
    if (rc) return rc;
    c->draws.back().has_normal = true;
    std::memcpy(c->draws.back().n, normal_matrix, sizeof(c->draws.back().n));
    return FGL_OK;
}

static int bits_for(uint32_t n)
{
    int b = 0;
    while (b < 32 && (n >> b) != 0) ++b;
    return b;
}

// Draw record of one model instance (bases left zero): Model::Render's
// per-draw state -- model matrix, its normal matrix, light * model.
static void fill_draw(fgl_ctx *c, const ModelRes &m, const float M[16], DevDraw &d)
{
    std::memset(&d, 0, sizeof(d));
    d.pos = m.pos; d.uv = m.uv; d.nrm = m.nrm; d.tan = m.tan;
    d.vi = m.vi; d.ti = m.ti; d.ni = m.ni; d.face_mat = m.fmat;
    d.corner = (const float4 *)m.corner;
    d.tri = m.tri;
    d.n_pos = m.n_pos;
    d.n_faces = m.n_faces;
    d.has_tangents = m.has_tan;
    d.support_pbr = m.pbr;
    std::memcpy(d.model, M, sizeof(d.model));
    make_normal_matrix(d.model, d.normal);
    mat_mul(c->light_space, d.model, d.lm);
}

// The stream's next n vectors (RandomVectorInUnitDisk for D = 2,
// RandomVectorInUnitSphere for D = 3) in stream order (c->fill), without
// consuming them: rng_take then moves the stream past the first m <= n.  The
// draws are generated in parallel chunks of K blocks, each chunk's first
// window reached by a jump from the context's next draw (rng.hip,
// mt_jump.hpp); the draws needed are estimated from the acceptance rate (pi/4
// for the disk, pi/6 for the sphere) with a margin, and doubled in the rare
// case that too few tries are kept.  A chunk's generation takes time in
// proportion to K (0.27 us per 454 words with a workgroup a CU, 0.36 with two),
// and the jumps (three workgroups each, one per CU) some 0.25 us a chunk: K =
// 256 while 256 chunks of it cover the request, else 512.
static constexpr int kMtChunkShort = 256, kMtChunkLong = 512;

static int rng_fill(fgl_ctx *c, int D, uint32_t n)
{
    int rc;
    c->fill = MtFill{};
    c->fill.D = D;
    c->fill_n = 0;
    if (n == 0) return FGL_OK;
    const double keep = D == 2 ? 0.78539816339744831 : 0.52359877559829887;
    uint64_t R = (uint64_t)((double)n * D / keep * 1.01) + 4096;
    for (;;) {
        const int kind = R <= 256ull * 624 * kMtChunkShort ? 0 : 1;
        const uint64_t C = 624ull * (kind ? kMtChunkLong : kMtChunkShort);
        const uint64_t Nc = (R + C - 1) / C;
        int K = kind ? kMtChunkLong : kMtChunkShort;
        if (Nc == 1) K = (int)((R + 623) / 624);   // one chunk: only the blocks needed
        const uint64_t len = Nc * (uint64_t)K * 624;
        if (len + 624 >= 0xffffffffull || Nc > 0x7fffffffull)
            return fail(c, FGL_ERR_CAPACITY, "random stream: too many draws in one request");
        MtFill f;
        f.D = D;
        f.chunks = (uint32_t)Nc;
        f.T = (uint32_t)K * 624u / (uint32_t)D;
        f.stride = (f.T + kStreamRun + 3u) & ~3u;
        f.n_ck = mt_checkpoints(f.T * (uint32_t)D);
        const size_t cks = (size_t)Nc * f.n_ck;
        if ((rc = ensure(c, c->mt_vec, (size_t)Nc * f.stride * D * sizeof(float))) ||
            (rc = ensure(c, c->mt_ck, (cks * 625 + 2 * (size_t)Nc + 1) * 4)) ||
            (rc = ensure(c, c->mt_base, (size_t)kMtBaseWords * 4)))
            return rc;
        f.out = (float *)c->mt_vec.p;
        f.ck_words = (uint32_t *)c->mt_ck.p;
        f.ck_kept = f.ck_words + cks * 624;
        f.kept = f.ck_kept + cks;
        f.prefix = f.kept + Nc;
        uint32_t *base = (uint32_t *)c->mt_base.p;
        const uint32_t *states = nullptr;
        launch_mt_base((const MtState *)c->rng.p, Nc > 1 ? (uint32_t)kMtBaseWords : 624u, base, c->stream);
        if (Nc > 1) {
            const int nj = (int)Nc - 1;
            if (nj > c->mt_lists_n[kind]) {
                std::vector<uint64_t> polys;
                if (!mt_jump_polys(C, nj, polys))
                    return fail(c, FGL_ERR_DEVICE, "random stream: no characteristic polynomial");
                c->mt_lists_n[kind] = 0;
                if ((rc = ensure(c, c->mt_lists[kind], (size_t)nj * (kMtListMax * 2 + kMtListStarts * 4)))) return rc;
                // the polynomials pass through the vectors' space, which the
                // fill writes after the lists are made
                static_assert(624 * kMtChunkShort / 3 * 4 >= kMtPolyWords * 8, "a chunk's vectors hold a polynomial");
                HIPCHK(c, hipMemcpyAsync(f.out, polys.data(), (size_t)nj * kMtPolyWords * 8, hipMemcpyHostToDevice, c->stream));
                uint16_t *entries = (uint16_t *)c->mt_lists[kind].p;
                launch_mt_lists((const uint64_t *)f.out, nj, entries, (uint32_t *)(entries + (size_t)nj * kMtListMax), c->stream);
                HIPCHK(c, hipStreamSynchronize(c->stream));
                c->mt_lists_n[kind] = nj;
            }
            if ((rc = ensure(c, c->mt_states, (size_t)Nc * kMtStateWords * 4))) return rc;
            const uint16_t *entries = (const uint16_t *)c->mt_lists[kind].p;
            launch_mt_jump(base, entries, (const uint32_t *)(entries + (size_t)c->mt_lists_n[kind] * kMtListMax), nj,
                           (uint32_t *)c->mt_states.p, c->stream);
            states = (const uint32_t *)c->mt_states.p;
        }
        launch_mt_fill(base, states, f, c->stream);
        HIPCHK(c, hipMemcpyAsync(c->h_total, f.prefix + Nc, 4, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        if (c->h_total[0] >= n) {
            c->fill = f;
            c->fill_n = n;
            HIPCHK(c, hipGetLastError());
            return FGL_OK;
        }
        R *= 2;
    }
}

static int rng_take(fgl_ctx *c, uint32_t m)
{
    if (m == 0) return FGL_OK;
    if (m > c->fill_n) return fail(c, FGL_ERR_INVALID, "random stream: taking more vectors than were drawn");
    launch_mt_commit((MtState *)c->rng.p, c->fill, m, c->stream);
    HIPCHK(c, hipGetLastError());
    return FGL_OK;
}

// The stochastic shadow filters' unit-disk samples for n shading points in
// the order they shade -- the lighting pass's pixels in row order, or the
// forward pass's passing fragments in raster order -- drawn from the
// context's stream, which ends past exactly the samples the points use.  g:
// the points' normal, world position and light NDC as planes of stride n
// (read for PCSS only).  ss: point i's samples start at pair ss.offs[i]
// (PCSS; offs[n] = the total) or at i * ss.stride (PCF).
static constexpr uint32_t kSegmentMax = kPcssSegmentMax;   // undecided PCSS points per walk segment, at most

static int stochastic_shadow_samples(fgl_ctx *c, const FrameUniforms &u, const float *g, size_t n, ShadowSamples &ss)
{
    int rc;
    const int mode = c->shadow_cfg.mode;
    const uint32_t nb = (uint32_t)c->shadow_cfg.n_blocker, np = (uint32_t)c->shadow_cfg.n_pcf;
    if (mode == FGL_SHADOW_REF_PCF) {
        const size_t total = n * np;
        if (total > 0xffffffffull) return fail(c, FGL_ERR_CAPACITY, "stochastic shadows: too many samples");
        if ((rc = rng_fill(c, 2, (uint32_t)total)) || (rc = rng_take(c, (uint32_t)total))) return rc;
        ss = {c->fill.vectors(), nullptr, np};
        return FGL_OK;
    }
    // PCSS takes n_pcf more samples only where its blocker search finds a
    // blocker.  Points the shadow map decides alone are counted in parallel;
    // the most samples the points can need (n_pcf more for every undecided
    // one) are drawn without consuming them; the undecided points are walked
    // in order; then the stream moves past exactly the samples used.
    if (n * (nb + np) > 0xffffffffull) return fail(c, FGL_ERR_CAPACITY, "stochastic shadows: too many samples");
    const size_t words = scan_tmp_words(n + 1), n4 = (n + 4) & ~(size_t)3;
    const size_t seg_words = 2 * (size_t)kSegmentMax + 2 * kPcssChainFbits + kPcssChainRes + 2 * ((size_t)kSegmentMax + 2) + 4;
    if ((rc = ensure(c, c->rng_offs, (6 * n4 + 4 * n4 + seg_words + words) * sizeof(uint32_t)))) return rc;
    uint32_t *base = (uint32_t *)c->rng_offs.p, *upos = base + n4, *list = upos + n4;
    uint32_t *found = list + n4, *offs = found + n4, *pbase = offs + n4;
    float4 *pt = (float4 *)(pbase + n4);
    unsigned long long *masks = (unsigned long long *)(pt + n4);
    unsigned long long *fbits = masks + kSegmentMax;
    uint32_t *res = (uint32_t *)(fbits + kPcssChainFbits);
    uint32_t *pred = res + kPcssChainRes;
    uint32_t *seg_out = pred + 2 * ((size_t)kSegmentMax + 2);
    uint32_t *tmp = seg_out + 4;
    int bx = 0, by = 0;
    float2 *mm = nullptr;   // without it (no room) every texel is read
    if (n > 0 && u.shadow_on && u.n_lights > 0 && pcss_windows(u, n, bx, by) &&
        room(c, c->pcss_mm, (size_t)u.SW * u.SH * sizeof(float2))) {
        mm = (float2 *)c->pcss_mm.p;
        launch_pcss_minmax(u, (const float *)c->shadow.p, bx, by, mm, c->stream);
    }
    launch_pcss_classify(u, g, n, (const float *)c->shadow.p, mm, bx, by, base, upos, c->stream);
    launch_exclusive_scan(base, base, n, tmp, c->stream);
    launch_exclusive_scan(upos, upos, n, tmp, c->stream);
    launch_pcss_compact(upos, n, list, c->stream);
    HIPCHK(c, hipMemcpyAsync(c->h_total, base + n, 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipMemcpyAsync(c->h_total + 1, upos + n, 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    const uint32_t n_unc = c->h_total[1];
    // the decided points' samples and n_blocker per undecided point, plus
    // n_pcf per undecided point: every offset the walk evaluates reads
    // inside it (point k of the undecided ones at most n_pcf k past its base)
    const size_t most = (size_t)c->h_total[0] + (size_t)np * n_unc;
    if ((rc = rng_fill(c, 2, (uint32_t)most))) return rc;
    const StreamVectors pairs = c->fill.vectors();
    // the undecided points in order, a segment at a time (shade.hip): the
    // band of miss counts each point is evaluated at follows the miss rate
    // seen so far
    launch_pcss_points(u, g, n, base, list, n_unc, pt, pbase, c->stream);
    uint32_t s0 = 0, M0 = 0, seg = kSegmentMax / 4;
    float rate = 0.25f;
    while (s0 < n_unc) {
        const uint32_t L = n_unc - s0 < seg ? n_unc - s0 : seg;
        launch_pcss_segment(u, (const float *)c->shadow.p, pairs, pt, pbase, s0, L, M0, rate, pred, tmp, masks, fbits,
                            res, found, seg_out, c->stream);
        HIPCHK(c, hipMemcpyAsync(c->h_total, seg_out, 8, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        const uint32_t s1 = c->h_total[0], M1 = c->h_total[1];
        if (s1 <= s0 || s1 > n_unc) return fail(c, FGL_ERR_DEVICE, "stochastic shadows: the PCSS walk did not advance");
        if (s1 - s0 >= 64) rate = (float)(M1 - M0) / (float)(s1 - s0);
        // the next segment: longer while whole segments settle, shorter when few of it did
        if (s1 - s0 == L && seg < kSegmentMax) seg *= 2;
        else if (4 * (s1 - s0) < L && seg > 1024) seg /= 2;
        s0 = s1;
        M0 = M1;
    }
    launch_exclusive_scan(found, found, n_unc, tmp, c->stream);
    launch_pcss_offsets(base, upos, found, np, n, offs, c->stream);
    HIPCHK(c, hipMemcpyAsync(c->h_total, offs + n, 4, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if ((rc = rng_take(c, c->h_total[0]))) return rc;
    ss = {pairs, offs, 0};
    return FGL_OK;
}

// Model to clip space of one draw in double precision, and the same product
// of absolute values, which bounds what the vertex stage's roundings can move.
struct ClipBound {
    double m[16], a[16];
};

// Rows r0 .. 3 of x y (depths_finite needs the last, of absolute values the last
// two).
static void mat_mul_d(const double *x, const float *y, double *o, bool absolute, int r0 = 0)
{
    for (int r = r0; r < 4; ++r)
        for (int j = 0; j < 4; ++j) {
            double v = 0.0;
            for (int k = 0; k < 4; ++k) {
                const double e = x[4 * r + k] * (double)y[4 * k + j];
                v += absolute ? std::fabs(e) : e;
            }
            o[4 * r + j] = v;
        }
}

// The pass's camera (model matrix still to come).
static ClipBound camera_bound(const fgl_ctx *c, bool shadow)
{
    const double I[16] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1};
    ClipBound b, p;
    mat_mul_d(I, shadow ? c->light_space : c->proj, b.m, false);
    mat_mul_d(I, shadow ? c->light_space : c->proj, b.a, true);
    if (shadow) return b;
    mat_mul_d(b.m, c->view, p.m, false);
    mat_mul_d(b.a, c->view, p.a, true);
    return p;
}

// Share of the vertex stage's largest intermediate that its roundings cannot
// reach (they are about a millionth of it).
constexpr double kClipMargin = 1e-4;

// Whether every vertex of m's faces has a finite window depth below 1e30: then
// no fragment's depth is NaN.  The model's extent is tried, which has to lie on
// one side of the camera plane; where it does not, each vertex of models of few
// vertices (a ground plane the camera stands on).  The extent first: 4,096 draws
// of 162 vertices, 640 x 400 view 6.4 -> 2.5 ms.
static bool depths_finite(const ModelRes &m, const ClipBound &b)
{
    if (!m.bounded) return false;
    auto far_from_camera = [&](const double lo[3], const double hi[3]) {
        double w = b.m[15], ext = 0.0, mag = b.a[15], z = b.a[11], top = 0.0;
        for (int j = 0; j < 3; ++j) {
            const double most = std::fmax(std::fabs(lo[j]), std::fabs(hi[j]));
            w += b.m[12 + j] * 0.5 * (lo[j] + hi[j]);
            ext += std::fabs(b.m[12 + j]) * 0.5 * (hi[j] - lo[j]);
            mag += b.a[12 + j] * most;
            z += b.a[8 + j] * most;
            top += most;
        }
        const double least = std::fabs(w) - ext;
        return least > kClipMargin * mag && z < 1e30 * least && least > 1e-30 && mag < 1e30 && top < 1e30;
    };
    if (far_from_camera(m.lo, m.hi)) return true;
    if (m.few.empty()) return false;
    for (size_t k = 0; k < m.few.size(); k += 3) {
        const double p[3] = {m.few[k], m.few[k + 1], m.few[k + 2]};
        if (!far_from_camera(p, p)) return false;
    }
    return true;
}

// The tile lists refuse a pass with 2^32 - 1 or more (tile, triangle) pairs,
// whatever rasterises it: a pass that could have as many goes to the lists,
// which count them.  pairs_bound bounds the pairs of m's faces: each face by
// the tiles its window rectangle can meet, from the model's extent and its
// longest edge, when all of the extent is in front of the camera; by the
// whole screen otherwise.
static double pairs_bound(const ModelRes &m, const ClipBound &b, const float vp[16], int W, int H, int TS)
{
    const double tx = (W + TS - 1) / TS, ty = (H + TS - 1) / TS;
    double all = tx * ty;
    if (!m.bounded) return all * m.n_faces;
    double wmin = HUGE_VAL, nx = 0.0, ny = 0.0;
    for (int k = 0; k < 8; ++k) {
        const double p[4] = {k & 1 ? m.hi[0] : m.lo[0], k & 2 ? m.hi[1] : m.lo[1], k & 4 ? m.hi[2] : m.lo[2], 1.0};
        double q[4], mag = 0.0;
        for (int r = 0; r < 4; ++r) {
            q[r] = 0.0;
            for (int j = 0; j < 4; ++j) q[r] += b.m[4 * r + j] * p[j];
        }
        for (int j = 0; j < 4; ++j) mag += b.a[12 + j] * std::fabs(p[j]);
        if (!(q[3] > kClipMargin * mag) || !std::isfinite(q[0]) || !std::isfinite(q[1])) return all * m.n_faces;
        wmin = std::fmin(wmin, q[3]);
        nx = std::fmax(nx, std::fabs(q[0] / q[3]));
        ny = std::fmax(ny, std::fabs(q[1] / q[3]));
    }
    // |x/w - x'/w'| <= (|x - x'| + |x'/w'| |w - w'|) / w over an edge
    double row[4];
    for (int r = 0; r < 4; ++r)
        row[r] = std::sqrt(b.m[4 * r] * b.m[4 * r] + b.m[4 * r + 1] * b.m[4 * r + 1] + b.m[4 * r + 2] * b.m[4 * r + 2]);
    const double ex = std::fabs((double)vp[0]) * (row[0] + nx * row[3]) * m.edge / wmin;
    const double ey = std::fabs((double)vp[5]) * (row[1] + ny * row[3]) * m.edge / wmin;
    const double face = std::fmin(tx, (1.01 * ex + 4.0) / TS + 2.0) * std::fmin(ty, (1.01 * ey + 4.0) / TS + 2.0);
    if (face < all) all = face;   // also when face is NaN
    return all * m.n_faces;
}

// What a pass's draws allow: its pairs are sure to be fewer than the lists
// can hold; no fragment can have a NaN depth.
static void bound_pass(const fgl_ctx *c, bool shadow, long long nt, int W, int H, int TS, bool &pairs_fit, bool &no_nan)
{
    const double most = 4294967295.0;
    const bool count = (double)nt * ((W + TS - 1) / TS) * ((H + TS - 1) / TS) >= most;
    const ClipBound cam = camera_bound(c, shadow);
    double sum = 0.0;
    no_nan = true;
    for (const fgl_ctx::Rec &r : c->draws) {
        const ModelRes &m = c->models[r.model];
        ClipBound b;
        if (!count && !no_nan) break;
        mat_mul_d(cam.m, r.m, b.m, false, count ? 0 : 3);
        mat_mul_d(cam.a, r.m, b.a, true, count ? 0 : 2);
        no_nan = no_nan && depths_finite(m, b);
        if (count) sum += pairs_bound(m, b, shadow ? c->shadow_viewport : c->viewport, W, H, TS);
    }
    pairs_fit = !count || sum < most;
}

// The direct rasteriser's launches of a pass: the draws' triangle groups and
// vertex blocks, and where each draw's begin.
struct DirectGrid {
    int lanes;
    long long groups, vblocks;
    bool corner;   // varyings from the corner records (corner_form)
    DrawStarts group_starts, vblock_starts;
};

static void free_direct(fgl_ctx *c)
{
    (void)hipStreamSynchronize(c->stream);   // no kernel may still use it
    (void)hipGetLastError();                 // of the allocation that failed
    for (DevBuf *b : {&c->key, &c->big, &c->key_nan, &c->direct_ctr}) free_buf(*b);
}

// Memory for a direct pass; without it the tile lists, which need none of this,
// take the pass.
static bool direct_room(fgl_ctx *c, size_t px, long long nt, bool no_nan)
{
    // a shadow pass already takes what its frame's main pass will: growing the
    // planes between them waits for the stream and frees
    const size_t most = px > c->frame_px ? px : c->frame_px;
    const size_t nan_cap = c->key_nan.cap;
    const bool first = !c->direct_ctr.p;
    if ((room(c, c->key, most * 8) || room(c, c->key, px * 8)) && room(c, c->big, (size_t)nt * 12) && room(c, c->direct_ctr, 2 * sizeof(DirectCtr)) &&
        (no_nan || room(c, c->key_nan, px * 8))) {
        if (first) launch_fill_u32((uint32_t *)c->direct_ctr.p, 0u, 2 * sizeof(DirectCtr) / 4, c->stream);
        if (c->key_nan.cap != nan_cap)
            launch_fill_u32((uint32_t *)c->key_nan.p, 0xffffffffu, c->key_nan.cap / 4, c->stream);
        return true;
    }
    free_direct(c);
    return false;
}

// The pass's fragments through the direct rasteriser (direct_room): its keys
// are left for the resolve, the shadow pass's targets are written.
static void direct_pass(fgl_ctx *c, const FrameUniforms &u, int n_draws, const DirectGrid &g, long long nt, bool shadow,
                        bool no_nan, int W, int H)
{
    const size_t px = (size_t)W * H;
    DirectCtr *ctr = (DirectCtr *)c->direct_ctr.p;
    DirectArgs a;
    a.draws = (const DevDraw *)c->d_draws.p;
    a.n_draws = n_draws;
    a.screen = (const int4 *)c->screen.p;
    a.key = (unsigned long long *)c->key.p;
    a.fix = no_nan ? nullptr : (unsigned long long *)c->key_nan.p;
    a.deep_from = (unsigned long long)deep_items((long long)px);
    a.big_start = (unsigned long long *)c->big.p;
    a.big_tri = (uint32_t *)(a.big_start + nt);
    a.ctr = ctr + c->direct_turn;
    a.W = W;
    a.H = H;
    c->direct_turn ^= 1;
    {
        KernelTimer t(c, "vertex");
        launch_direct_vertex(shadow, (int)g.vblocks, u, (int4 *)c->screen.p,
                             shadow ? (float *)c->ndc_z.p : nullptr, g.corner || shadow ? nullptr : (float4 *)c->vary.p, a,
                             g.vblock_starts, ctr + c->direct_turn, c->stream);
    }
    KernelTimer t(c, shadow ? "raster_shadow" : "raster");
    launch_direct(a, g.group_starts, g.lanes, (int)g.groups, nt, c->stream);
    if (shadow)
        launch_direct_shadow(a, (const float *)c->ndc_z.p, (float *)c->shadow_depth.p, (float *)c->shadow.p, c->stream);
}

// The pass through the tile lists; with stoch also the sequence of passing
// fragments (n_frag of them).
static int list_pass(fgl_ctx *c, const FrameUniforms &u, int n_draws, int max_pos, int max_faces, long long nt, bool shadow,
                     int W, int H, bool fresh, bool stoch, uint32_t &n_frag)
{
    const int TS = shadow ? c->TS_shadow : c->TS;
    const int tiles_x = (W + TS - 1) / TS, tiles_y = (H + TS - 1) / TS;
    const uint32_t ntiles = (uint32_t)(tiles_x * tiles_y);
    int rc;
    if ((rc = ensure(c, c->rect, (size_t)nt * sizeof(uint2))) ||
        (rc = ensure(c, c->counts, (size_t)nt * 4)) || (rc = ensure(c, c->offs, ((size_t)nt + 1) * 4)) ||
        (rc = ensure(c, c->scan_tmp, scan_tmp_words((size_t)nt) * 4)) ||
        (rc = ensure(c, c->tile_start, (size_t)ntiles * 4)) ||
        (rc = ensure(c, c->tile_end, (size_t)ntiles * 4)) ||
        (rc = ensure(c, c->tri_v, (size_t)nt * sizeof(int4))) ||
        (rc = ensure(c, c->big_list, (size_t)nt * 4)) || (rc = ensure(c, c->counters, 64)) ||
        (!shadow && (rc = ensure(c, c->vis, (size_t)W * H * 4))))
        return rc;
    const DevDraw *ddraws = (const DevDraw *)c->d_draws.p;
    uint32_t *big_count = (uint32_t *)c->counters.p;
    {
        KernelTimer t(c, "vertex");
        launch_vertex(shadow, ddraws, n_draws, max_pos, u, (int4 *)c->screen.p,
                      shadow ? (float *)c->ndc_z.p : nullptr, shadow ? nullptr : (float4 *)c->vary.p, big_count,
                      c->stream);
    }
    {
        KernelTimer t(c, "setup");
        launch_setup(ddraws, n_draws, max_faces, (const int4 *)c->screen.p, W, H, TS,
                     (uint2 *)c->rect.p, (uint32_t *)c->counts.p, (int4 *)c->tri_v.p,
                     (uint32_t *)c->big_list.p, big_count, c->stream);
    }
    {
        KernelTimer t(c, "scan");
        launch_exclusive_scan((const uint32_t *)c->counts.p, (uint32_t *)c->offs.p, (size_t)nt,
                              (uint32_t *)c->scan_tmp.p, c->stream);
    }
    uint32_t npairs = 0, n_big = 0;
    if ((rc = read_counts(c, (const uint32_t *)c->offs.p + nt, big_count, npairs, n_big))) return rc;
    if (npairs == 0xffffffffu)
        return fail(c, FGL_ERR_CAPACITY, "the pass has 2^32 - 1 or more (tile, triangle) pairs; use a larger tile");
    if ((rc = ensure(c, c->keys, (size_t)npairs * 4 + 4)) || (rc = ensure(c, c->vals, (size_t)npairs * 4 + 4)) ||
        (rc = ensure(c, c->keys_alt, (size_t)npairs * 4 + 4)) ||
        (rc = ensure(c, c->vals_alt, (size_t)npairs * 4 + 4)) ||
        (rc = ensure(c, c->sort_tmp, radix_tmp_words(npairs) * 4)))
        return rc;
    {
        KernelTimer t(c, "emit");
        launch_emit((const uint32_t *)c->offs.p, (int)nt, (const uint2 *)c->rect.p, tiles_x,
                    (const uint32_t *)c->big_list.p, n_big, (uint32_t *)c->keys.p,
                    (uint32_t *)c->vals.p, (uint32_t *)c->tile_start.p, (uint32_t *)c->tile_end.p,
                    (int)ntiles, c->stream);
    }
    {
        KernelTimer t(c, "sort");
        launch_radix_sort((uint32_t *)c->keys.p, (uint32_t *)c->vals.p, (uint32_t *)c->keys_alt.p,
                          (uint32_t *)c->vals_alt.p, npairs, bits_for(ntiles - 1),
                          (uint32_t *)c->sort_tmp.p, c->stream);
    }
    {
        KernelTimer t(c, "tile_ranges");
        launch_tile_ranges((const uint32_t *)c->keys.p, npairs, nullptr, (uint32_t *)c->tile_start.p,
                           (uint32_t *)c->tile_end.p, c->stream);
    }
    if (stoch) {
        // the passing fragments in raster order: count, scan, emit, sort
        KernelTimer t(c, "frag_walk");
        const size_t P = (size_t)W * H;
        if ((rc = ensure(c, c->frag_cnt, (P + 1 + scan_tmp_words(P)) * 4))) return rc;
        uint32_t *cnt = (uint32_t *)c->frag_cnt.p;
        FragWalkArgs fw;
        std::memset(&fw, 0, sizeof(fw));
        fw.screen = (const int4 *)c->screen.p;
        fw.tri_v = (const int4 *)c->tri_v.p;
        fw.vals = (const uint32_t *)c->vals.p;
        fw.tile_start = (const uint32_t *)c->tile_start.p;
        fw.tile_end = (const uint32_t *)c->tile_end.p;
        fw.W = W;
        fw.H = H;
        fw.tiles_x = tiles_x;
        fw.tiles_y = tiles_y;
        fw.fresh = fresh;
        fw.depth = (const float *)c->depth.p;
        fw.count = cnt;
        launch_frag_walk(false, TS, fw, c->stream);
        launch_exclusive_scan(cnt, cnt, P, cnt + P + 1, c->stream);
        HIPCHK(c, hipMemcpyAsync(c->h_total, cnt + P, 4, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        n_frag = c->h_total[0];
        if (n_frag == 0xffffffffu) return fail(c, FGL_ERR_CAPACITY, "stochastic shadows: too many passing fragments");
        if ((rc = ensure(c, c->frag_tri, (size_t)n_frag * 8 + 8)) ||
            (rc = ensure(c, c->frag_alt, (size_t)n_frag * 8 + 8)) ||
            (rc = ensure(c, c->frag_tmp, radix_tmp_words(n_frag) * 4)))
            return rc;
        uint32_t *ftri = (uint32_t *)c->frag_tri.p, *fq = ftri + n_frag;
        uint32_t *atri = (uint32_t *)c->frag_alt.p, *aq = atri + n_frag;
        fw.base = cnt;
        fw.tri_out = ftri;
        fw.q_out = fq;
        launch_frag_walk(true, TS, fw, c->stream);
        c->frag_sorted_alt = launch_radix_sort_impl(ftri, fq, atri, aq, n_frag, nullptr, bits_for((uint32_t)(nt - 1)),
                                                    (uint32_t *)c->frag_tmp.p, c->stream) != 0;
    }
    RasterArgs a;
    std::memset(&a, 0, sizeof(a));
    a.draws = ddraws;
    a.n_draws = n_draws;
    a.screen = (const int4 *)c->screen.p;
    a.tri_v = (const int4 *)c->tri_v.p;
    a.vals = (const uint32_t *)c->vals.p;
    a.tile_start = (const uint32_t *)c->tile_start.p;
    a.tile_end = (const uint32_t *)c->tile_end.p;
    a.W = W;
    a.H = H;
    a.tiles_x = tiles_x;
    a.tiles_y = tiles_y;
    a.fresh = fresh;
    a.depth = shadow ? (float *)c->shadow_depth.p : (float *)c->depth.p;
    a.vis = (int *)c->vis.p;
    a.shadow_out = (float *)c->shadow.p;
    a.ndc_z = shadow ? (const float *)c->ndc_z.p : nullptr;
    {
        KernelTimer t(c, shadow ? "raster_shadow" : "raster");
        launch_raster(shadow, TS, a, c->stream);
    }
    return FGL_OK;
}

static int flush_pass(fgl_ctx *c)
{
    if (c->draws.empty()) return FGL_OK;
    const int pass = c->pass == FGL_PASS_SHADOW ? kPassShadow
                   : c->pass == FGL_PASS_GEOMETRY ? kPassGeometry : kPassForward;
    const bool shadow = pass == kPassShadow;
    const int W = shadow ? c->SW : c->W, H = shadow ? c->SH : c->H;
    if (W <= 0 || H <= 0 || (shadow && !c->shadow.p) || (!shadow && !c->depth.p)) {
        c->draws.clear();
        return fail(c, FGL_ERR_INVALID, "render targets not initialised for this pass");
    }
    if (pass == kPassForward && c->shadow_on && !c->shadow.p) {
        c->draws.clear();
        return fail(c, FGL_ERR_INVALID, "forward pass with shadows needs a shadow buffer");
    }
    // The forward shaders with a stochastic shadow filter draw samples for
    // every fragment that passes the depth test, in raster order: the pass
    // replays that sequence (k_frag_walk) to find each winner's samples.
    const bool stoch = pass == kPassForward && c->shadow_on && !c->lights.empty() &&
                       (c->shadow_cfg.mode == FGL_SHADOW_REF_PCF || c->shadow_cfg.mode == FGL_SHADOW_REF_PCSS);
    if (stoch && (size_t)c->W * c->H > 0xffffffffull) {
        c->draws.clear();
        return fail(c, FGL_ERR_CAPACITY, "stochastic shadows in the forward pass: too many pixels");
    }
    int rc = upload_tables(c);
    if (rc) return rc;

    // draw table in submission order
    std::vector<DevDraw> dd(c->draws.size());
    long long nt = 0, nv = 0, tris = 0;
    int max_pos = 0, max_faces = 0;
    for (const fgl_ctx::Rec &r : c->draws) tris += c->models[r.model].n_faces;
    DirectGrid grid = {direct_lanes(tris, tris, (long long)W * H, shadow), 0, 0, corner_form((long long)W * H, tris),
                       {}, {}};
    for (int k = 1; k < kFewDraws; ++k) grid.group_starts.few[k] = grid.vblock_starts.few[k] = INT_MAX;
    for (size_t i = 0; i < c->draws.size(); ++i) {
        const ModelRes &m = c->models[c->draws[i].model];
        DevDraw &d = dd[i];
        fill_draw(c, m, c->draws[i].m, d);
        if (c->draws[i].has_normal) std::memcpy(d.normal, c->draws[i].n, sizeof(d.normal));
        d.vert_base = (int)nv;
        d.tri_base = (int)nt;
        if (i < kFewDraws) {
            grid.vblock_starts.few[i] = (int)grid.vblocks;
            grid.group_starts.few[i] = (int)grid.groups;
        }
        grid.vblocks += vertex_blocks(d.n_pos);
        grid.groups += direct_groups(d.n_faces, grid.lanes);
        nt += m.n_faces;
        nv += m.n_pos;
        max_pos = m.n_pos > max_pos ? m.n_pos : max_pos;
        max_faces = m.n_faces > max_faces ? m.n_faces : max_faces;
    }
    const int n_draws = (int)c->draws.size();
    bool fits, no_nan;
    bound_pass(c, shadow, nt, W, H, shadow ? c->TS_shadow : c->TS, fits, no_nan);
    c->draws.clear();
    if (nt > 0x7fffffffLL || nv > 0x7fffffffLL) return fail(c, FGL_ERR_CAPACITY, "pass too large");
    // Whether this pass starts from the cleared targets: then it writes
    // every pixel (winner or clear value) and no separate clear runs.
    bool fresh;
    if (shadow) {
        fresh = c->pend_shadow;
    } else if (pass == kPassGeometry) {
        if (c->pend_depth != c->pend_gbuf && (rc = materialize(c, true, true, false, false, false))) return rc;
        fresh = c->pend_depth;
    } else {
        if (c->pend_depth != c->pend_fb && (rc = materialize(c, true, false, true, false, false))) return rc;
        if (c->shadow_on && (rc = materialize(c, false, false, false, false, true))) return rc;
        fresh = c->pend_depth;
    }
    if (nt == 0) return FGL_OK;

    if (dd.size() != c->last_draws.size() ||
        std::memcmp(dd.data(), c->last_draws.data(), dd.size() * sizeof(DevDraw)) != 0) {
        // The records, then where each draw's workgroups begin (DrawStarts): the
        // vertex pass's, the triangle groups' at 1, 4 and 16 lanes.  Nothing of it
        // is one pass's own: the shadow pass's table serves the main pass.
        KernelTimer t(c, "draw_table");
        const size_t n = dd.size(), records = n * sizeof(DevDraw);
        std::vector<char> table(records + 4 * n * sizeof(int));
        std::memcpy(table.data(), dd.data(), records);
        int *starts = (int *)(table.data() + records);
        long long at[4] = {0, 0, 0, 0};
        for (size_t i = 0; i < n; ++i) {
            for (int k = 0; k < 4; ++k) starts[k * n + i] = (int)at[k];
            at[0] += vertex_blocks(dd[i].n_pos);
            for (int lanes : {1, 4, 16}) at[1 + lanes_slot(lanes)] += direct_groups(dd[i].n_faces, lanes);
        }
        c->last_draws.clear();   // nothing is known of the table until it is written
        if ((rc = ensure(c, c->d_draws, table.size()))) return rc;
        HIPCHK(c, hipStreamSynchronize(c->stream));
        HIPCHK(c, hipMemcpy(c->d_draws.p, table.data(), table.size(), hipMemcpyHostToDevice));
        c->last_draws = dd;
    }

    FrameUniforms u;
    build_uniforms(c, u);
    // A pass from cleared targets folds its fragments into a key plane; one
    // that goes on from earlier depths, or replays the fragment sequence, takes
    // the tile lists.
    const DevDraw *ddraws = (const DevDraw *)c->d_draws.p;
    grid.vblock_starts.table = (const int *)(ddraws + n_draws);
    grid.group_starts.table = grid.vblock_starts.table + (size_t)(1 + lanes_slot(grid.lanes)) * n_draws;
    const size_t px = (size_t)W * H;
    if ((rc = ensure(c, c->screen, (size_t)nv * sizeof(int4))) || (shadow && (rc = ensure(c, c->ndc_z, (size_t)nv * 4))) ||
        (!shadow && (rc = ensure(c, c->vary, (size_t)nv * 2 * sizeof(float4)))))
        return rc;
    const bool direct = fresh && !stoch && fits && nt <= kDirectTrisMost && launch_fits(grid.groups) &&
                        launch_fits(grid.vblocks + clear_blocks((long long)px)) && direct_room(c, px, nt, no_nan);
    uint32_t n_frag = 0;
    if (direct) {
        direct_pass(c, u, n_draws, grid, nt, shadow, no_nan, W, H);
    } else {
        rc = list_pass(c, u, n_draws, max_pos, max_faces, nt, shadow, W, H, fresh, stoch, n_frag);
        if (rc == FGL_ERR_NOMEM && c->key.p) {   // with the direct rasteriser's memory given back
            free_direct(c);
            rc = list_pass(c, u, n_draws, max_pos, max_faces, nt, shadow, W, H, fresh, stoch, n_frag);
        }
        if (rc) return rc;
    }
    if (shadow) {
        c->pend_shadow = false;
    } else {
        ResolveArgs r;
        std::memset(&r, 0, sizeof(r));
        r.draws = ddraws;
        r.n_draws = n_draws;
        r.screen = (const int4 *)c->screen.p;
        r.tri_v = (const int4 *)c->tri_v.p;
        r.vary = direct && grid.corner ? nullptr : (const float4 *)c->vary.p;
        r.vis = (const int *)c->vis.p;
        if (direct) {
            r.key = (unsigned long long *)c->key.p;
            r.fix = no_nan ? nullptr : (unsigned long long *)c->key_nan.p;
            r.depth = (float *)c->depth.p;
        }
        r.W = W;
        r.H = H;
        r.fresh = fresh;
        std::memcpy(r.clear, c->fb_clear, sizeof(r.clear));
        r.gbuf = (float *)c->gbuf.p;
        r.fb = (float *)c->fb.p;
        r.materials = (const DevMaterial *)c->d_materials.p;
        r.textures = (const DevTexture *)c->d_textures.p;
        r.shadow_map = (const float *)c->shadow.p;
        if (pass == kPassGeometry) {
            KernelTimer t(c, "gbuffer_resolve");
            launch_gbuffer_resolve(r, u, c->stream);
            c->pend_gbuf = false;
        } else {
            if (stoch) {
                // each winner's samples: the offset of its fragment in the sequence
                KernelTimer t(c, "shadow_samples");
                const size_t P = (size_t)W * H;
                if ((rc = ensure(c, c->frag_offs_px, P * 4))) return rc;
                uint32_t *offs_px = (uint32_t *)c->frag_offs_px.p;
                launch_fill_u32(offs_px, 0u, P, c->stream);
                uint32_t *ftri = (uint32_t *)(c->frag_sorted_alt ? c->frag_alt.p : c->frag_tri.p), *fq = ftri + n_frag;
                const float *planes = nullptr;
                if (c->shadow_cfg.mode == FGL_SHADOW_REF_PCSS) {
                    if ((rc = ensure(c, c->frag_planes, (size_t)9 * n_frag * sizeof(float) + 4))) return rc;
                    launch_frag_shadow_inputs(r, u, ftri, fq, n_frag, (float *)c->frag_planes.p, c->stream);
                    planes = (const float *)c->frag_planes.p;
                }
                ShadowSamples ss = {};
                if ((rc = stochastic_shadow_samples(c, u, planes, n_frag, ss))) return rc;
                launch_frag_pixel_offsets(ftri, fq, n_frag, W, H, (const int *)c->vis.p, ss.offs, ss.stride, offs_px,
                                          c->stream);
                r.ss = {ss.sv, offs_px, 0};
            }
            KernelTimer t(c, "forward_resolve");
            launch_forward_resolve(r, u, c->stream);
            c->pend_fb = false;
        }
        c->pend_depth = false;
    }
    HIPCHK(c, hipGetLastError());
    return FGL_OK;
}

int fgl_end_pass(fgl_ctx *c)
{
    if (!c) return FGL_ERR_INVALID;
    return flush_pass(c);
}

int fgl_draw_screen_space_pixels(fgl_ctx *c)
{
    if (!c) return FGL_ERR_INVALID;
    int rc = flush_pass(c);
    if (rc) return rc;
    if (!c->gbuf.p) return fail(c, FGL_ERR_INVALID, "targets not initialised");
    if (c->shadow_on && !c->shadow.p) return fail(c, FGL_ERR_INVALID, "shadows on but no shadow buffer");
    if ((rc = materialize(c, false, true, false, false, c->shadow_on != 0))) return rc;
    FrameUniforms u;
    build_uniforms(c, u);
    ShadowSamples ss = {};
    const int mode = c->shadow_cfg.mode;
    if (c->shadow_on && !c->lights.empty() && (mode == FGL_SHADOW_REF_PCF || mode == FGL_SHADOW_REF_PCSS)) {
        // the filters' unit-disk samples from the stream, pixels in row order
        KernelTimer t(c, "shadow_samples");
        if ((rc = stochastic_shadow_samples(c, u, (const float *)c->gbuf.p, (size_t)c->W * c->H, ss))) return rc;
    }
    {
        KernelTimer t(c, "lighting");
        // a pending network AO is interpolated from its grid by the lighting
        // pass itself (the same values the up pass would write)
        launch_lighting(u, (const float *)c->gbuf.p, (const float *)c->ao.p, c->pend_ao ? 1 : 0, c->ao_net,
                        (const float *)c->shadow.p, ss, (float *)c->fb.p, c->stream);
    }
    c->pend_fb = false;  // every pixel written
    HIPCHK(c, hipGetLastError());
    return FGL_OK;
}

int fgl_ssao(fgl_ctx *c, const fgl_ssao_cfg *cfg)
{
    if (!c || !cfg) return FGL_ERR_INVALID;
    if ((!cfg->stochastic && (cfg->n_kernel < 1 || cfg->n_kernel > 64)) || cfg->blur < 0 || cfg->blur > 2 ||
        (cfg->blur == 2 && (cfg->blur_radius < 1 || cfg->blur_radius > 8)))
        return fail(c, FGL_ERR_INVALID, "bad SSAO configuration");
    int rc = flush_pass(c);
    if (rc) return rc;
    if (!c->gbuf.p) return fail(c, FGL_ERR_INVALID, "targets not initialised");
    if ((rc = materialize(c, true, true, false, false, false))) return rc;
    c->pend_ao = false;  // every pixel written
    c->ao_net = NetAo{};
    c->ao_net_owner = nullptr;
    FrameUniforms u;
    build_uniforms(c, u);
    SsaoArgs sa;
    sa.n_kernel = cfg->n_kernel;
    std::memcpy(sa.kernel, cfg->kernel, sizeof(sa.kernel));
    std::memcpy(sa.noise, cfg->noise, sizeof(sa.noise));
    sa.radius = cfg->radius;
    sa.bias = cfg->bias;
    sa.range = cfg->range;
    sa.kmax = 0.f;
    for (int k = 0; k < 3 * sa.n_kernel; ++k) {
        const float a = std::fabs(sa.kernel[k]);
        if (!(a <= sa.kmax)) sa.kmax = a;   // a NaN component makes kmax NaN
    }
    // the whole AO stage (SSAO and blur, with the gap between them) as one span
    KernelTimer stage(c, "ssao_blur");
    if (cfg->stochastic) {
        // 32 hemisphere samples per pixel, pixels in row order, from the stream
        const size_t n = (size_t)c->W * c->H * 32;
        if (n > 0xffffffffull) return fail(c, FGL_ERR_CAPACITY, "stochastic SSAO: too many samples");
        KernelTimer t(c, "ssao_reference");
        if ((rc = rng_fill(c, 3, (uint32_t)n)) || (rc = rng_take(c, (uint32_t)n))) return rc;
        launch_ssao_reference(u, c->fill.vectors(), (const float *)c->ssao_pow3.p,
                              (const float *)c->depth.p, (const float *)c->gbuf.p, (float *)c->ao.p, c->stream);
    } else {
        KernelTimer t(c, "ssao");
        launch_ssao(u, sa, (const float *)c->depth.p, (const float *)c->gbuf.p, (float *)c->ao.p, c->stream);
    }
    if (cfg->blur == 1) {
        KernelTimer t(c, "blur_reference");
        launch_blur_recursive((float *)c->ao.p, c->W, c->H, c->stream);
    } else if (cfg->blur == 2) {
        KernelTimer t(c, "blur_gaussian");
        // one pass into the spare plane, which then becomes the AO target
        launch_blur_separable((const float *)c->ao.p, (float *)c->blur_tmp.p, c->W, c->H,
                                 cfg->blur_weights, cfg->blur_radius, c->stream);
        std::swap(c->ao, c->blur_tmp);
    }
    HIPCHK(c, hipGetLastError());
    return FGL_OK;
}

int fgl_ssao_noalloc(fgl_ctx *c, int w, int h, const float view[16], const float proj[16],
                     const float *depth, const float *gbuf, float *ao, const fgl_ssao_cfg *cfg)
{
    if (!c) return FGL_ERR_INVALID;
    if (!cfg || !view || !proj || !depth || !gbuf || !ao) return fail(c, FGL_ERR_INVALID, "null argument");
    if (w <= 0 || h <= 0) return fail(c, FGL_ERR_INVALID, "bad frame size");
    if ((long long)w * h > FGL_SSAO_NOALLOC_MAX_PIXELS)
        return fail(c, FGL_ERR_CAPACITY, "frame larger than FGL_SSAO_NOALLOC_MAX_PIXELS (" +
                                             std::to_string(FGL_SSAO_NOALLOC_MAX_PIXELS) + " pixels)");
    if (cfg->stochastic)
        return fail(c, FGL_ERR_INVALID, "the stochastic SSAO draws from the context's stream: use fgl_ssao");
    if (cfg->n_kernel < 1 || cfg->n_kernel > 64 || cfg->blur < 0 || cfg->blur > 2 ||
        (cfg->blur == 2 && (cfg->blur_radius < 1 || cfg->blur_radius > 8)))
        return fail(c, FGL_ERR_INVALID, "bad SSAO configuration");
    if (!c->noalloc_scratch) return fail(c, FGL_ERR_DEVICE, "no scratch address for this device");
    FrameUniforms u;
    std::memset(&u, 0, sizeof(u));
    std::memcpy(u.view, view, sizeof(u.view));
    std::memcpy(u.proj, proj, sizeof(u.proj));
    mat_mul(proj, view, u.vp);
    make_viewport(0, 0, w, h, u.viewport);
    u.W = w;
    u.H = h;
    SsaoArgs sa;
    sa.n_kernel = cfg->n_kernel;
    std::memcpy(sa.kernel, cfg->kernel, sizeof(sa.kernel));
    std::memcpy(sa.noise, cfg->noise, sizeof(sa.noise));
    sa.radius = cfg->radius;
    sa.bias = cfg->bias;
    sa.range = cfg->range;
    sa.kmax = 0.f;
    for (int k = 0; k < 3 * sa.n_kernel; ++k) {
        const float a = std::fabs(sa.kernel[k]);
        if (!(a <= sa.kmax)) sa.kmax = a;
    }
    // The separable blur reads the unblurred AO from the scratch array; the
    // SSAO kernel writes every pixel of it first, so nothing is cleared.
    float *raw = ao;
    std::unique_lock<std::mutex> lock(g_scratch_mu, std::defer_lock);
    if (cfg->blur == 2) {
        lock.lock();
        HIPCHK(c, scratch_use(c, (size_t)w * h, &raw));
    }
    launch_ssao(u, sa, depth, gbuf, raw, c->stream);
    if (cfg->blur == 1)
        launch_blur_recursive(ao, w, h, c->stream);
    else if (cfg->blur == 2)
        launch_blur_separable(raw, ao, w, h, cfg->blur_weights, cfg->blur_radius, c->stream);
    HIPCHK(c, hipGetLastError());
    return FGL_OK;
}

int fgl_resolve(fgl_ctx *c, int k)
{
    if (!c) return FGL_ERR_INVALID;
    int rc = flush_pass(c);
    if (rc) return rc;
    if (!c->fb.p) return fail(c, FGL_ERR_INVALID, "targets not initialised");
    if (k < 1 || k > 16 || c->W / k <= 0 || c->H / k <= 0) return fail(c, FGL_ERR_INVALID, "bad SSAA factor");
    int ow = c->W / k, oh = c->H / k;
    if ((rc = materialize(c, false, false, true, false, false))) return rc;
    if ((rc = ensure(c, c->img, (size_t)ow * oh * 3))) return rc;
    c->img_w = ow;
    c->img_h = oh;
    KernelTimer t(c, "resolve");
    launch_resolve((const float *)c->fb.p, c->W, c->H, k, (uint8_t *)c->img.p, c->stream);
    HIPCHK(c, hipGetLastError());
    return FGL_OK;
}

// ---------------- readback ----------------

static int target_ptr(fgl_ctx *c, int which, void **p, size_t *bytes)
{
    size_t P = (size_t)c->W * c->H, SP = (size_t)c->SW * c->SH;
    switch (which) {
    case FGL_TARGET_FRAME: *p = c->fb.p; *bytes = 3 * P * 4; break;
    case FGL_TARGET_DEPTH: *p = c->depth.p; *bytes = P * 4; break;
    case FGL_TARGET_SHADOW: *p = c->shadow.p; *bytes = SP * 4; break;
    case FGL_TARGET_SHADOW_DEPTH: *p = c->shadow_depth.p; *bytes = SP * 4; break;
    case FGL_TARGET_GBUFFER: *p = c->gbuf.p; *bytes = kGbufPlanes * P * 4; break;
    case FGL_TARGET_AO: *p = c->ao.p; *bytes = P * 4; break;
    case FGL_TARGET_IMAGE: *p = c->img.p; *bytes = (size_t)c->img_w * c->img_h * 3; break;
    default: return fail(c, FGL_ERR_INVALID, "unknown target");
    }
    if (!*p) return fail(c, FGL_ERR_INVALID, "target not initialised");
    return FGL_OK;
}

int fgl_target_bytes(fgl_ctx *c, int which, size_t *out)
{
    if (!c || !out) return FGL_ERR_INVALID;
    void *p;
    return target_ptr(c, which, &p, out);
}

int fgl_read_target(fgl_ctx *c, int which, void *dst, size_t bytes)
{
    if (!c || !dst) return FGL_ERR_INVALID;
    int rc = flush_pass(c);
    if (rc) return rc;
    void *p;
    size_t n;
    if ((rc = target_ptr(c, which, &p, &n))) return rc;
    if (bytes != n) return fail(c, FGL_ERR_INVALID, "size mismatch: target has " + std::to_string(n) + " bytes");
    if ((rc = materialize(c, which == FGL_TARGET_DEPTH, which == FGL_TARGET_GBUFFER,
                          which == FGL_TARGET_FRAME, which == FGL_TARGET_AO,
                          which == FGL_TARGET_SHADOW || which == FGL_TARGET_SHADOW_DEPTH)))
        return rc;
    HIPCHK(c, hipMemcpyAsync(dst, p, n, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return FGL_OK;
}

int fgl_write_target(fgl_ctx *c, int which, const void *src, size_t bytes)
{
    if (!c || !src) return FGL_ERR_INVALID;
    if (which == FGL_TARGET_IMAGE) return fail(c, FGL_ERR_INVALID, "image target is read-only");
    int rc = flush_pass(c);
    if (rc) return rc;
    void *p;
    size_t n;
    if ((rc = target_ptr(c, which, &p, &n))) return rc;
    if (bytes != n) return fail(c, FGL_ERR_INVALID, "size mismatch: target has " + std::to_string(n) + " bytes");
    // the whole target is replaced; a shadow target's companion is materialised
    if (which == FGL_TARGET_SHADOW || which == FGL_TARGET_SHADOW_DEPTH) {
        if ((rc = materialize(c, false, false, false, false, true))) return rc;
    }
    if (which == FGL_TARGET_DEPTH) c->pend_depth = false;
    if (which == FGL_TARGET_GBUFFER) c->pend_gbuf = false;
    if (which == FGL_TARGET_FRAME) c->pend_fb = false;
    if (which == FGL_TARGET_AO) {
        c->pend_ao = false;
        c->ao_net = NetAo{};
        c->ao_net_owner = nullptr;
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(p, src, n, hipMemcpyHostToDevice));
    return FGL_OK;
}

int fgl_enable_timing(fgl_ctx *c, int on)
{
    if (!c) return FGL_ERR_INVALID;
    c->timing = on != 0;
    return FGL_OK;
}

int fgl_time_only(fgl_ctx *c, const char *name)
{
    if (!c) return FGL_ERR_INVALID;
    c->timing_only = name ? name : "";
    return FGL_OK;
}

int fgl_rng_seed(fgl_ctx *c, uint32_t seed)
{
    if (!c) return FGL_ERR_INVALID;
    int rc = flush_pass(c);
    if (rc) return rc;
    c->rng_seed = seed;
    return rng_restart(c);
}

int fgl_rng_vectors(fgl_ctx *c, int kind, uint32_t n, float *out)
{
    if (!c || (kind != 2 && kind != 3) || (n && !out)) return FGL_ERR_INVALID;
    int rc = flush_pass(c);
    if (rc) return rc;
    if (n == 0) return FGL_OK;
    const size_t bytes = (size_t)n * kind * sizeof(float);
    if ((rc = ensure(c, c->rng_samples, bytes))) return rc;
    if ((rc = rng_fill(c, kind, n)) || (rc = rng_take(c, n))) return rc;
    launch_mt_gather(c->fill, n, (float *)c->rng_samples.p, c->stream);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(out, c->rng_samples.p, bytes, hipMemcpyDeviceToHost));
    return FGL_OK;
}

int fgl_rng_draws(fgl_ctx *c, uint64_t *out)
{
    if (!c || !out) return FGL_ERR_INVALID;
    int rc = flush_pass(c);
    if (rc) return rc;
    MtState st;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    HIPCHK(c, hipMemcpy(&st, c->rng.p, sizeof(st), hipMemcpyDeviceToHost));
    *out = st.draws;
    return FGL_OK;
}

int fgl_read_timings(fgl_ctx *c, char (*names)[32], float *ms, int cap, int *out_n)
{
    if (!c || !out_n) return FGL_ERR_INVALID;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    int n = 0;
    for (auto &t : c->timed) {
        if (n < cap && names && ms) {
            float v = 0.f;
            (void)hipEventElapsedTime(&v, t.a, t.b);
            std::snprintf(names[n], 32, "%s", t.name.c_str());
            ms[n] = v;
        }
        ++n;
        (void)hipEventDestroy(t.a);
        (void)hipEventDestroy(t.b);
    }
    c->timed.clear();
    *out_n = n;
    return FGL_OK;
}

int fgl_copy_benchmark(fgl_ctx *c, size_t bytes, int iters, float *ms_per_iter)
{
    if (!c || bytes < 16 || iters < 1) return FGL_ERR_INVALID;
    void *a = nullptr, *b = nullptr;
    HIPCHK(c, hipMalloc(&a, bytes));
    if (hipMalloc(&b, bytes) != hipSuccess) {
        (void)hipFree(a);
        return fail(c, FGL_ERR_NOMEM, "copy buffer");
    }
    launch_fill_f32((float *)a, 1.f, bytes / 4, c->stream);
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    launch_copy(a, b, bytes, c->stream);
    (void)hipEventRecord(e0, c->stream);
    for (int i = 0; i < iters; ++i) launch_copy(a, b, bytes, c->stream);
    (void)hipEventRecord(e1, c->stream);
    (void)hipEventSynchronize(e1);
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    if (ms_per_iter) *ms_per_iter = ms / iters;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(a);
    (void)hipFree(b);
    return FGL_OK;
}

int fgl_check_recip(fgl_ctx *c, uint64_t *compared, uint64_t *mismatches, uint64_t *fast_path)
{
    if (!c) return FGL_ERR_INVALID;
    int rc = flush_pass(c);
    if (rc) return rc;
    unsigned long long *d = nullptr, h[3] = {0, 0, 0};
    HIPCHK(c, hipMalloc(&d, sizeof(h)));
    hipError_t e = hipMemcpyAsync(d, h, sizeof(h), hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) {
        launch_check_recip(d, c->stream);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    (void)hipFree(d);
    if (e != hipSuccess) return fail(c, FGL_ERR_DEVICE, hipGetErrorString(e));
    if (compared) *compared = h[0];
    if (mismatches) *mismatches = h[1];
    if (fast_path) *fast_path = h[2];
    return FGL_OK;
}

int fgl_sort_pairs(fgl_ctx *c, uint32_t *keys, uint32_t *vals, size_t n, int bits)
{
    if (!c || (n && (!keys || !vals)) || n > 0x80000000ull || bits < 1 || bits > 32) return FGL_ERR_INVALID;
    if (n == 0) return FGL_OK;
    int rc = flush_pass(c);
    if (rc) return rc;
    const size_t bytes = n * 4;
    const size_t tmp_bytes = radix_tmp_words(n) * 4;
    void *buf[5] = {nullptr, nullptr, nullptr, nullptr, nullptr};
    const size_t sz[5] = {bytes, bytes, bytes, bytes, tmp_bytes};
    for (int i = 0; i < 5; ++i)
        if (hipMalloc(&buf[i], sz[i]) != hipSuccess) {
            for (int j = 0; j < i; ++j) (void)hipFree(buf[j]);
            return fail(c, FGL_ERR_NOMEM, "sort buffers");
        }
    hipError_t e = hipMemcpyAsync(buf[0], keys, bytes, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(buf[1], vals, bytes, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) {
        launch_radix_sort((uint32_t *)buf[0], (uint32_t *)buf[1], (uint32_t *)buf[2], (uint32_t *)buf[3], n, bits,
                          (uint32_t *)buf[4], c->stream);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(keys, buf[0], bytes, hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(vals, buf[1], bytes, hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    for (int i = 0; i < 5; ++i) (void)hipFree(buf[i]);
    if (e != hipSuccess) return fail(c, FGL_ERR_DEVICE, hipGetErrorString(e));
    return FGL_OK;
}

}  // extern "C"

namespace fgl {

int ctx_view(fgl_ctx *c, CtxView *v, bool need_ao)
{
    int rc = flush_pass(c);
    if (rc) return rc;
    if (!c->depth.p) return fail(c, FGL_ERR_INVALID, "targets not initialised");
    if ((rc = materialize(c, true, true, false, need_ao, false))) return rc;
    v->stream = c->stream;
    v->W = c->W;
    v->H = c->H;
    v->depth = (float *)c->depth.p;
    v->gbuf = (float *)c->gbuf.p;
    v->ao = (float *)c->ao.p;
    v->fb = (float *)c->fb.p;
    std::memcpy(v->view, c->view, sizeof(v->view));
    std::memcpy(v->proj, c->proj, sizeof(v->proj));
    std::memcpy(v->viewport, c->viewport, sizeof(v->viewport));
    return FGL_OK;
}

void ctx_ao_written(fgl_ctx *c)
{
    c->pend_ao = false;
    c->ao_net = NetAo{};
    c->ao_net_owner = nullptr;
}

void ctx_ao_from_network(fgl_ctx *c, const NetAo &net, const void *owner)
{
    c->pend_ao = false;
    c->ao_net = net;
    c->ao_net_owner = owner;
}

void ctx_drop_network_ao(fgl_ctx *c, const void *owner)
{
    if (c->ao_net_owner != owner) return;
    c->ao_net = NetAo{};
    c->ao_net_owner = nullptr;
}

int ctx_settle_network_ao(fgl_ctx *c, const void *owner)
{
    if (!c->ao_net.lao || c->ao_net_owner != owner) return FGL_OK;
    return materialize(c, false, false, false, true, false);
}

void ctx_register_nao(fgl_ctx *c, void *n) { c->naos.push_back(n); }

static void unregister(std::vector<void *> &list, void *p)
{
    for (size_t k = 0; k < list.size(); ++k)
        if (list[k] == p) {
            list.erase(list.begin() + (long)k);
            break;
        }
}

void ctx_unregister_nao(fgl_ctx *c, void *n) { unregister(c->naos, n); }

void ctx_register_batch(fgl_ctx *c, void *b) { c->batches.push_back(b); }

void ctx_unregister_batch(fgl_ctx *c, void *b) { unregister(c->batches, b); }

int ctx_fail(fgl_ctx *c, int code, const char *msg) { return fail(c, code, msg); }

void ctx_uniforms(fgl_ctx *c, FrameUniforms *u) { build_uniforms(c, *u); }

int ctx_draw_record(fgl_ctx *c, int model, const float M[16], DevDraw *out)
{
    if (model < 0 || model >= (int)c->models.size()) return fail(c, FGL_ERR_INVALID, "unknown model");
    fill_draw(c, c->models[model], M, *out);
    return FGL_OK;
}

void ctx_begin_frame(fgl_ctx *c, int w, int h) { c->frame_px = (size_t)w * h; }

std::mutex &ctx_order_mutex() { return g_scratch_mu; }

bool ctx_depths_finite(fgl_ctx *c, int model, const float M[16], bool shadow)
{
    const ClipBound cam = camera_bound(c, shadow);
    ClipBound b;
    mat_mul_d(cam.m, M, b.m, false, 3);
    mat_mul_d(cam.a, M, b.a, true, 2);
    return depths_finite(c->models[model], b);
}

int ctx_tables(fgl_ctx *c, const DevMaterial **materials, const DevTexture **textures)
{
    int rc = upload_tables(c);
    if (rc) return rc;
    *materials = (const DevMaterial *)c->d_materials.p;
    *textures = (const DevTexture *)c->d_textures.p;
    return FGL_OK;
}

hipStream_t ctx_stream(fgl_ctx *c) { return c->stream; }
bool ctx_timing(fgl_ctx *c) { return c->timing && c->timing_only.empty(); }

CtxTimer::CtxTimer(fgl_ctx *c, const char *name) : impl_(name ? new KernelTimer(c, name) : nullptr) {}
CtxTimer::~CtxTimer() { delete static_cast<KernelTimer *>(impl_); }

}  // namespace fgl

extern "C" {

// ---------------- scenes ----------------

struct fgl_scene {
    HostScene s;
};

int fgl_scene_load(const char *path, fgl_scene **out, char *err, size_t err_len)
{
    return fgl_scene_load_with(path, FGL_WRAP_NONE, FGL_FILTER_NEAREST, out, err, err_len);
}

int fgl_scene_load_with(const char *path, int wrap, int filter, fgl_scene **out, char *err, size_t err_len)
{
    if (!path || !out || wrap < FGL_WRAP_NONE || wrap > FGL_WRAP_CLAMP || filter < FGL_FILTER_NEAREST ||
        filter > FGL_FILTER_LINEAR)
        return FGL_ERR_INVALID;
    *out = nullptr;
    fgl_scene *sc = new fgl_scene();
    std::string e;
    if (!load_scene(path, sc->s, e, wrap, filter)) {
        if (err && err_len) std::snprintf(err, err_len, "%s", e.c_str());
        delete sc;
        return FGL_ERR_IO;
    }
    *out = sc;
    return FGL_OK;
}

void fgl_scene_free(fgl_scene *s) { delete s; }

int fgl_scene_info_get(const fgl_scene *s, fgl_scene_info *out)
{
    if (!s || !out) return FGL_ERR_INVALID;
    *out = s->s.info;
    return FGL_OK;
}

int fgl_scene_model(const fgl_scene *s, int i, fgl_model_desc *d, float mm[16])
{
    if (!s || !d || i < 0 || i >= (int)s->s.models.size()) return FGL_ERR_INVALID;
    const HostModel &m = *s->s.models[i];
    d->n_pos = (int)m.pos.size() / 3;
    d->n_uv = (int)m.uv.size() / 2;
    d->n_nrm = (int)m.nrm.size() / 3;
    d->n_faces = m.n_faces();
    d->pos = m.pos.data();
    d->uv = m.uv.data();
    d->nrm = m.nrm.data();
    d->tan = m.has_tangents ? m.tan.data() : nullptr;
    d->vi = m.vi.data();
    d->ti = m.ti.data();
    d->ni = m.ni.data();
    d->face_material = m.face_mat.data();
    d->support_pbr = m.support_pbr;
    if (mm) std::memcpy(mm, s->s.model_mats[i].data(), 16 * sizeof(float));
    return FGL_OK;
}

int fgl_scene_material(const fgl_scene *s, int i, fgl_material *out)
{
    if (!s || !out || i < 0 || i >= (int)s->s.materials.size()) return FGL_ERR_INVALID;
    *out = s->s.materials[i];
    return FGL_OK;
}

int fgl_scene_texture(const fgl_scene *s, int i, int *w, int *h, int *bpp, int *wrap, int *filter,
                      const uint8_t **bytes)
{
    if (!s || i < 0 || i >= (int)s->s.textures.size()) return FGL_ERR_INVALID;
    const HostTexture &t = s->s.textures[i];
    if (w) *w = t.w;
    if (h) *h = t.h;
    if (bpp) *bpp = t.bpp;
    if (wrap) *wrap = t.wrap;
    if (filter) *filter = t.filter;
    if (bytes) *bytes = t.bytes.data();
    return FGL_OK;
}

static int upload_scene(fgl_ctx *c, fgl_scene *sc)
{
    HostScene &s = sc->s;
    if (s.uploaded_ctx == c) return FGL_OK;
    int rc;
    std::vector<int> tex_id(s.textures.size()), mat_id(s.materials.size());
    for (size_t i = 0; i < s.textures.size(); ++i) {
        const HostTexture &t = s.textures[i];
        if ((rc = fgl_upload_texture(c, t.w, t.h, t.bpp, t.bytes.data(), t.wrap, t.filter, &tex_id[i])))
            return rc;
    }
    for (size_t i = 0; i < s.materials.size(); ++i) {
        fgl_material m = s.materials[i];
        int32_t *maps[] = {&m.map_kd, &m.map_ks, &m.map_ke, &m.map_bump, &m.map_base,
                           &m.map_rough, &m.map_metal, &m.map_ao, &m.map_pbr_ke};
        for (int32_t *p : maps)
            if (*p >= 0) *p = tex_id[*p];
        if ((rc = fgl_upload_material(c, &m, &mat_id[i]))) return rc;
    }
    s.dev_models.clear();
    std::vector<std::pair<const HostModel *, int>> done;
    for (size_t i = 0; i < s.models.size(); ++i) {
        const HostModel *hm = s.models[i].get();
        int id = -1;
        for (auto &p : done)
            if (p.first == hm) id = p.second;
        if (id < 0) {
            std::vector<int32_t> fm(hm->face_mat.size());
            for (size_t f = 0; f < fm.size(); ++f) fm[f] = mat_id[hm->face_mat[f]];
            fgl_model_desc d;
            fgl_scene_model(sc, (int)i, &d, nullptr);
            d.face_material = fm.data();
            if ((rc = fgl_upload_model(c, &d, &id))) return rc;
            done.push_back({hm, id});
        }
        s.dev_models.push_back(id);
    }
    s.uploaded_ctx = c;
    return FGL_OK;
}

int fgl_scene_upload(fgl_ctx *c, fgl_scene *sc, int32_t *model_ids)
{
    if (!c || !sc) return FGL_ERR_INVALID;
    int rc = upload_scene(c, sc);
    if (rc) return rc;
    if (model_ids)
        for (size_t i = 0; i < sc->s.dev_models.size(); ++i) model_ids[i] = sc->s.dev_models[i];
    return FGL_OK;
}

// Render::Render (src/render.cpp:40-58) with the scene's extension settings.
int fgl_render_scene(fgl_ctx *c, fgl_scene *sc)
{
    if (!c || !sc) return FGL_ERR_INVALID;
    int rc;
    if ((rc = upload_scene(c, sc))) return rc;
    const fgl_scene_info &I = sc->s.info;
    // one Render::Render run: the reference's stream starts fresh
    if ((I.ssao_on && I.ssao.stochastic) || (I.shadow_on && I.shadow.mode >= FGL_SHADOW_REF_PCF))
        if ((rc = rng_restart(c))) return rc;
    const int k = I.ssaa_on ? I.ssaa_k : 1;
    if (k < 1) return fail(c, FGL_ERR_INVALID, "bad SSAA factor");
    const int W = I.width * k, H = I.height * k;
    const float ratio = (float)I.width / I.height;
    // Preconfigure (render.cpp:33-38)
    fgl_set_viewport(c, 0, 0, 0, W, H);
    c->frame_px = (size_t)W * H;
    const int S = I.shadow_map_size > 0 ? I.shadow_map_size : 0;
    fgl_set_viewport(c, 1, 0, 0, S ? S : W, S ? S : H);
    fgl_set_lights(c, I.n_lights, I.lights);
    fgl_set_eye(c, I.eye);
    if ((rc = fgl_set_shadow(c, I.shadow_on, &I.shadow))) return rc;
    // DoShadowPass (render.cpp:60-97)
    if (I.shadow_on) {
        if ((rc = fgl_init_shadow_buffer(c, S ? S : W, S ? S : H))) return rc;
        float V[16], P[16], L[16];
        const float origin[3] = {0.f, 0.f, 0.f}, up[3] = {0.f, 1.f, 0.f};
        make_lookat(I.lights[0].vec, origin, up, V);
        make_ortho(-3.0f * ratio, 3.0f * ratio, -3.0f, 3.0f, 0.1f, 20.f, P);
        mat_mul(P, V, L);
        fgl_set_matrix(c, FGL_MAT_LIGHT_SPACE, L);
        fgl_begin_pass(c, FGL_PASS_SHADOW);
        for (size_t i = 0; i < sc->s.models.size(); ++i)
            if ((rc = fgl_draw_model(c, sc->s.dev_models[i], sc->s.model_mats[i].data()))) return rc;
        if ((rc = fgl_end_pass(c))) return rc;
    }
    // camera (render.cpp:106-115)
    float V[16], P[16];
    const float up[3] = {0.f, 1.f, 0.f};
    make_lookat(I.eye, I.look_at, up, V);
    if (I.camera_ortho) make_ortho(-1.f * ratio, 1.f * ratio, -1.f, 1.f, 0.01f, 20.f, P);
    else make_perspective(45.f, ratio, 0.01f, 20.f, P);
    fgl_set_matrix(c, FGL_MAT_VIEW, V);
    fgl_set_matrix(c, FGL_MAT_PROJ, P);
    if ((rc = fgl_init_targets(c, W, H))) return rc;
    if (!I.deferred) {
        // DoForwardPass (render.cpp:99-157)
        if ((rc = fgl_clear_color(c, 0.12f, 0.12f, 0.12f))) return rc;
        fgl_begin_pass(c, FGL_PASS_FORWARD);
        for (size_t i = 0; i < sc->s.models.size(); ++i)
            if ((rc = fgl_draw_model(c, sc->s.dev_models[i], sc->s.model_mats[i].data()))) return rc;
        if ((rc = fgl_end_pass(c))) return rc;
    } else {
        // DoGeometryPass + DoLightingPass (render.cpp:159-212)
        fgl_begin_pass(c, FGL_PASS_GEOMETRY);
        for (size_t i = 0; i < sc->s.models.size(); ++i)
            if ((rc = fgl_draw_model(c, sc->s.dev_models[i], sc->s.model_mats[i].data()))) return rc;
        if ((rc = fgl_end_pass(c))) return rc;
        fgl_begin_pass(c, FGL_PASS_LIGHTING);
        if (I.ssao_on && (rc = fgl_ssao(c, &I.ssao))) return rc;
        if ((rc = fgl_draw_screen_space_pixels(c))) return rc;
    }
    // DoSSAA (render.cpp:291-343); k = 1 quantises only
    return fgl_resolve(c, k);
}

// ---------------- host helpers ----------------

void fgl_make_model_matrix(float tx, float ty, float tz, float r, float s, float out[16])
{
    make_model_matrix(tx, ty, tz, r, s, out);
}
void fgl_make_lookat(const float eye[3], const float center[3], const float up[3], float out[16])
{
    make_lookat(eye, center, up, out);
}
void fgl_make_perspective(float fov, float aspect, float n, float f, float out[16])
{
    make_perspective(fov, aspect, n, f, out);
}
void fgl_make_ortho(float l, float r, float b, float t, float n, float f, float out[16])
{
    make_ortho(l, r, b, t, n, f, out);
}
void fgl_mat_mul(const float a[16], const float b[16], float out[16]) { mat_mul(a, b, out); }
void fgl_make_normal_matrix(const float m[16], float out[9]) { make_normal_matrix(m, out); }

int fgl_tga_write(const char *path, int w, int h, int bpp, const uint8_t *bytes, int rle)
{
    if (!path || !bytes || w <= 0 || h <= 0 || (bpp != 1 && bpp != 3 && bpp != 4)) return FGL_ERR_INVALID;
    return tga_write(path, w, h, bpp, bytes, rle != 0) ? FGL_OK : FGL_ERR_IO;
}

}  // extern "C"
