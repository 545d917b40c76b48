// Host-side sizes of a pass's launches (no HIP: also compiled by the tests).
#pragma once

namespace fgl {

// A launch's work-items count in 32 bits along x: so many workgroups of 256.
constexpr long long kMaxBlocks = 0xffffffffLL / 256;
constexpr bool launch_fits(long long blocks) { return blocks <= kMaxBlocks; }

// Lanes per triangle of the direct rasteriser in a pass of n_tri triangles: as
// many as fill the chip (a triangle's pixels are its lanes' serial work).
constexpr long long kDirectTris16 = 32768, kDirectTris4 = 262144;
constexpr int direct_lanes(long long n_tri) { return n_tri <= kDirectTris16 ? 16 : n_tri <= kDirectTris4 ? 4 : 1; }

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
// 1,413; 1280 x 800 (3.1) 329 / 330; 24 views (5.4) 3,099 / 3,136; 1914 x 1206
// forward (13) 326 / 334.
constexpr bool corner_form(long long pixels, long long n_tri) { return pixels < 2 * n_tri; }

// Items (64 x 16 pixels) of large triangles that cover targets of so many pixels
// three times over.
constexpr long long deep_items(long long pixels) { return 3 * (pixels / 1024 + 1); }

// Triangles of a pass that the direct rasteriser's claims count.
constexpr long long kDirectTrisMost = (1LL << 30) - 1;

// Workgroups of a draw: 256 / lanes triangles each; 256 vertices each.
constexpr long long direct_groups(int n_faces, int lanes) { return ((long long)n_faces * lanes + 255) / 256; }
constexpr long long vertex_blocks(int n_pos) { return ((long long)n_pos + 255) / 256; }

// The key plane's clearing (8 keys a thread, at least one workgroup).
constexpr long long kClearKeys = 8;
constexpr long long clear_blocks(long long keys) { return (keys + 256 * kClearKeys - 1) / (256 * kClearKeys); }

}  // namespace fgl
