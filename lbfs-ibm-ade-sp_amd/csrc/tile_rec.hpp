// One tile of the device layout: where its cells, faces, halos and boundary
// faces start, and where its slot patterns lie (tiles of the same shape share
// one pattern).
#pragma once

namespace lbfs {

struct TileRec {
    int c0, nc;    // first cell, cells
    int f0, nf;    // first face of the list, faces
    int h0;        // first entry of its halo ids:
    int nh, n2;    // the cells across the border that the faces reach, then the cells beyond them that
                   // those cells' gradients reach
    int b0, nif;   // first entry of the boundary-face ids, interior faces (the others follow them)
    int s0;        // first of the tile's nc + nh gradient slots among all tiles'
    int pf, pc, pn;  // first entries of the face, cell and gradient slot patterns
    int pad[3];
};

// The fused fluid pass keeps the gradients of a tile and its halo (48 B a slot)
// and its face fluxes (16 B) in LDS, up to 96 KiB; larger tiles run two passes.
// (Its table of cell ids comes on top: such a tile has at most 2048 slots, which
// reach at most 12288 cells more, 56 KiB.)
constexpr bool fused_tile_fits(int slots, int faces) { return 48 * (long long)slots + 16 * (long long)faces <= 96 * 1024; }

}  // namespace lbfs
