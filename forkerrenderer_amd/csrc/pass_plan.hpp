// Host-side sizes of a pass's launches (no HIP: also compiled by the tests).
#pragma once

namespace fgl {

// A launch's work-items count in 32 bits along x: so many workgroups of 256.
constexpr long long kMaxBlocks = 0xffffffffLL / 256;
constexpr bool launch_fits(long long blocks) { return blocks <= kMaxBlocks; }

// Lanes per triangle of the direct rasteriser: n_faces that share a target of
// `pixels`, in a pass of n_tri triangles.  A triangle's pixels are its lanes'
// serial work, its set-up every lane's; so by the pixels a face has (of a shadow
// map, which holds the whole light volume, the scene covers a third of what it
// covers of a view).  Passes of few triangles leave the chip idle with fewer lanes.
// One sphere that fills the view, 16 / 4 / 1 lanes, us of the pass's raster
// launches:
//   faces      pixels a face    view                     pixels a face   shadow map
//   20,480     12               11.4 / 11.9 / 41.0       20              19.2 / 15.3 / 37.2
//   81,920     0.5              15.6 / 10.4 / 10.6       0.8             19.6 / 18.6 / 17.0
//   81,920     3.1              17.0 / 11.9 / 22.5       5               20.8 / 18.2 / 22.2
//   81,920     12               21.4 / 19.1 / 49.8       20              25.7 / 21.3 / 50.3
//   81,920     25               23.8 / 39.8 / 60.7       45              32.1 / 29.2 / 62.6
//   327,680    0.8              42.5 / 18.8 / 13.2       1.2             46.5 / 21.6 / 18.5
//   327,680    6.3              49.1 / 26.6 / 83.7       11              58.6 / 35.7 / 39.6
//   327,680    25               70.6 / 100 / 131         45              110 / 98 / 158
//   1,310,720  1.6              145 / 55.5 / 38.0        2.8             162 / 69.8 / 46.4
//   1,310,720  6.3              175 / 83 / 221           11              214 / 123 / 131
// Between 12 and 25 pixels a batch places the upper line: 16 lanes from 16, 24, 48
// pixels a face on, 64 views 9.13, 9.06, 9.07 ms, 24 views 2.102, 2.079, 2.099.
constexpr long long kDirectFew = 32768;
constexpr int direct_lanes(long long n_tri, long long n_faces, long long pixels, bool shadow)
{
    const long long px2 = 2 * pixels / (shadow ? 3 : 1);   // in halves
    return n_tri <= kDirectFew || px2 >= 48 * n_faces ? 16 : px2 >= 5 * n_faces ? 4 : 1;
}

// Whether a main pass's resolve makes the varyings that depend on a position
// from the corner records, instead of reading what the vertex pass made of each
// vertex.  Where faces are a pixel or two, a pixel's three corners are gathers of
// their own: the corner records (one more line, some 120 operations a corner)
// cost less than the vertices' (three more lines), and the vertex pass writes 32
// bytes a vertex less.  Where more pixels share a vertex it is the other way.
// G-buffer resolve and main vertex pass, from vertices / from corners, us:
// 3840 x 2160, 64 objects of 81,920 faces (1.6 pixels a face) 297 / 250, 1920 x
// 1080 (0.4) 108 / 76; 25 objects, 3840 x 2160 (4) 248 / 222.  With shadows, whose
// light positions add to a corner's operations: 3840 x 2160 frame (1.6) 1,450 /
// 1,413; 1280 x 800 (3.1) 329 / 330; 1914 x 1206 forward (13) 326 / 334.
// In a batch by view: 64 views, none / by this rule / all from corners 9.22 /
// 9.13 / 9.16 ms.
constexpr bool corner_form(long long pixels, long long n_tri) { return pixels < 2 * n_tri; }

// Items (64 x 16 pixels) of large triangles that cover targets of so many pixels
// three times over.
constexpr long long deep_items(long long pixels) { return 3 * (pixels / 1024 + 1); }

// Triangles of a pass that the direct rasteriser's claims count.
constexpr long long kDirectTrisMost = (1LL << 30) - 1;

// Their place among 1, 4 and 16.
constexpr int lanes_slot(int lanes) { return lanes == 16 ? 2 : lanes == 4 ? 1 : 0; }

// Workgroups of a draw: 256 / lanes triangles each; 256 vertices each.
constexpr long long direct_groups(int n_faces, int lanes) { return ((long long)n_faces * lanes + 255) / 256; }
constexpr long long vertex_blocks(int n_pos) { return ((long long)n_pos + 255) / 256; }

// The key plane's clearing (8 keys a thread, at least one workgroup).
constexpr long long kClearKeys = 8;
constexpr long long clear_blocks(long long keys) { return (keys + 256 * kClearKeys - 1) / (256 * kClearKeys); }

}  // namespace fgl
