// spec_tiles.h - how the specular filter's mips are cut into tiles, for one map
// (specular_split_kernel) and for a batch of probes (probe_batch_kernel): the
// tiles, the rule for a texel per wave, and a batch's work items.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

#include "hvx_internal.h"
#include "hvx_math.h"

namespace hvx {

constexpr uint32_t kNarrowFace = 6688;  // largest face whose cube level is smaller than 4 GiB

#ifndef HVX_SPEC_TPW
#define HVX_SPEC_TPW 4
#endif
constexpr int kSpecTPW = HVX_SPEC_TPW;  // texels per wave: 4, 8 or 16
static_assert(kSpecTPW == 4 || kSpecTPW == 8 || kSpecTPW == 16, "HVX_SPEC_TPW is 4, 8 or 16");
template <int TPW> struct SpecShape {
    static constexpr int kSPR = 64 / TPW;                         // samples per texel per round
    static constexpr int kTW = TPW >= 8 ? 8 : (TPW >= 4 ? 4 : 1);  // tile width (texels)
    static constexpr int kRPW = TPW / kTW;                        // texel rows per wave
    static constexpr int kTH = 4 * kRPW;                          // tile height: four waves
    static constexpr int kRow = 4 * kSPR + 4;                     // floats per texel row of the LDS buffer (padded)
};
// Small maps wait for their rounds (a texel's 1,024 samples are 64 of them with
// four texels to a wave) with most of the card idle: there a wave takes one
// texel and 64 samples a round. What is left of a round's gain past the starts
// of four times the waves grows with the samples and falls with the tiles. us
// of the whole call with four / one:
//   16^2 x 2 (24 tiles) and 256 samples 67 / 34, 64^2 x 2 (384): 16 samples 13.0 /
//   17.2, 64: 19.3 / 20.3, 1,024: 102 / 98, 64^2 x 7 (522): 64 samples 18.2 / 20.4,
//   1,024: 107 / 89, 80^2 x 2 (600): 64 samples 20.7 / 24.0, 256: 51 / 47, 90^2 x 4
//   from 1000^2 (1,134): 128 samples 74 / 65, 1,024: 462 / 375, 100^2 x 7 (1,398):
//   128 samples 35 / 40, 1,024: 187 / 170, but 110^2 x 3 (1,470) 243 / 259, 128^2 x 2
//   (1,536): 64 samples 29 / 43, 1,024: 275 / 305
constexpr uint32_t kSpecFewTiles = 1500;
inline bool spec_few(uint32_t tiles, uint32_t n) { return tiles <= kSpecFewTiles && 9ull * n >= tiles; }

// Tiles of one mip of size Sm: kTW x kTH texels, taken face by face in
// supertiles of 16 x 16 tiles (row-major supertiles, row-major tiles in each;
// the last column and row of supertiles are as wide and high as is left).
struct SpecTileGeom {
    uint32_t tiles_x, tiles_y, per_face;
};
template <int TPW> HVX_HD SpecTileGeom spec_tile_geom(uint32_t Sm) {
    constexpr uint32_t kTW = SpecShape<TPW>::kTW, kTH = SpecShape<TPW>::kTH;
    SpecTileGeom g;
    g.tiles_x = (Sm + kTW - 1) / kTW;
    g.tiles_y = (Sm + kTH - 1) / kTH;
    g.per_face = g.tiles_x * g.tiles_y;
    return g;
}
// Tile index (< 6 per_face) -> (face, tx, ty).
HVX_HD void spec_tile_at(const SpecTileGeom& g, uint32_t k, uint32_t& face, uint32_t& tx, uint32_t& ty) {
    face = k / g.per_face;
    const uint32_t kk = k % g.per_face, row = kk / (16u * g.tiles_x), kr = kk % (16u * g.tiles_x);
    const uint32_t high = g.tiles_y - 16u * row < 16u ? g.tiles_y - 16u * row : 16u;
    const uint32_t col = kr / (16u * high), kc = kr % (16u * high);
    const uint32_t wide = g.tiles_x - 16u * col < 16u ? g.tiles_x - 16u * col : 16u;
    tx = 16u * col + kc % wide;
    ty = 16u * row + kc / wide;
}

// A batch's work items (probe, mip, range): mip 0 as ranges of `texels` texels,
// other mips as runs of tiles of at most about `texels` texels, fewer where
// `slots` workgroups would get less than 64 runs each (at the end of the batch
// the card waits for the last of them: 16 probes 512^2 -> 256^2 x 9 take 13.7 ms
// with 16 runs each, 12.6 with 64). Each mip's items are dealt in eight contiguous
// runs, one per XCD (xcd_begin[x]: the first of XCD x's items), as
// specular_split_kernel does, and what is left over goes round the XCDs: tiles of
// one mip cost about the same, those of different mips up to several times each
// other, and mip 0 next to nothing, so no estimate of costs is needed (with the
// batch cut into eight runs of equal estimated cost: 18.9 ms; 256 probes of 64^2
// to 512^2 73.6 ms, 63.0 so; one call after the other 12.7 and 66.5). Returns
// whether a wave takes one texel (few tiles in the whole batch).
inline bool make_probe_items(const ProbeJob* jobs, uint32_t n_probes, uint32_t texels, uint32_t slots,
                             std::vector<ProbeItem>& items, uint32_t xcd_begin[9]) {
    uint64_t tiles = 0;
    uint32_t samples = 0;
    for (uint32_t p = 0; p < n_probes; ++p) {
        samples = std::max(samples, jobs[p].n);
        for (uint32_t m = 1; m < jobs[p].mips; ++m)
            tiles += 6u * (uint64_t)spec_tile_geom<kSpecTPW>(std::max(jobs[p].So >> m, 1u)).per_face;
    }
    const bool one = tiles <= kSpecFewTiles && spec_few((uint32_t)tiles, samples);
    const uint32_t tile_texels = one ? SpecShape<1>::kTW * SpecShape<1>::kTH
                                     : SpecShape<kSpecTPW>::kTW * SpecShape<kSpecTPW>::kTH;
    if (one) tiles *= kSpecTPW;
    const uint64_t spread = std::max<uint64_t>(tiles / (64ull * std::max(slots, 1u)), 1u);
    const uint32_t per_item = (uint32_t)std::min<uint64_t>(std::max(texels / tile_texels, 1u), spread);
    std::vector<ProbeItem> run[8];
    uint32_t next[2] = {0, 0};  // the XCD of the next item left over: of mips 0, of other mips
    for (uint32_t p = 0; p < n_probes; ++p)
        for (uint32_t m = 0; m < jobs[p].mips; ++m) {
            const uint32_t Sm = std::max(jobs[p].So >> m, 1u), per = m ? per_item : texels;
            const uint32_t total = m == 0 ? 6u * Sm * Sm
                                          : 6u * (one ? spec_tile_geom<1>(Sm) : spec_tile_geom<kSpecTPW>(Sm)).per_face;
            const uint32_t n = (total + per - 1) / per, left = n % 8u;
            uint32_t k = 0;
            for (uint32_t x = 0; x < 8; ++x) {
                const bool extra = (x + 8u - next[m > 0]) % 8u < left;
                for (const uint32_t end = k + n / 8u + (extra ? 1u : 0u); k < end; ++k)
                    run[x].push_back({p, m, k * per, std::min(per, total - k * per)});
            }
            next[m > 0] = (next[m > 0] + left) % 8u;
        }
    items.clear();
    for (uint32_t x = 0; x < 8; ++x) {
        xcd_begin[x] = (uint32_t)items.size();
        items.insert(items.end(), run[x].begin(), run[x].end());
    }
    xcd_begin[8] = (uint32_t)items.size();
    return one;
}

}  // namespace hvx
