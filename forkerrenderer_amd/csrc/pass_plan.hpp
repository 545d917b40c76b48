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
