// tile_cut.hip -- cuts the active output rows of a rulebook into tiles of equal WORK for the MFMA
// gather-GEMM.
//
// The GEMM kernel gives every workgroup a run of consecutive output rows.  With runs of equal length the
// busiest compute unit of the headline frame issues 37 % more MFMA blocks than the average one (pairs per
// row vary between 1 and 27 with the local density of the scene), and the launch lasts as long as the
// busiest unit.  Here every row gets the weight  pairs(row) + row_weight  and the rows are cut where the
// running sum crosses multiples of W = ceil(total / T), T = the tile count the equal-length rule would
// use (tile_plan() with the target height the caller names).  The per-row constant is the caller's: what a row
// costs its GEMM kernel beside its pairs (4 pairs' worth on conv_wide.hip); it also keeps sparse runs from growing far
// beyond the kernel's tile capacity.  Runs that still do are walked in capacity-sized pieces by the kernel, so any
// cut is correct.
//
// The weights come with the rulebook (lookups, coord.hip) or from a pass over it (tile_weights); tile_cuts then re-derives
// a chunk's offset and the total from the sums over 64 rows (a few hundred values), scans its rows, and the first row of
// every tile writes start[tile]; the last active row writes the end marker and the tile count.
// Region layout (int32): [0] tile count (0 = no cuts: the kernel falls back to equal lengths), [1] W,
// [2] total weight, [3] unused, [4 ..] start[0 .. count], then w[max_voxels], wsum[max_voxels / 64].
#include "coord.h"

namespace sessd {

static int max_tiles(int max_voxels) { return max_voxels / kGemmMinTileRows + 1024 + 1; }

size_t tile_cut_bytes(int max_voxels) {
    const size_t ints = 4 + (size_t)max_tiles(max_voxels) + 1 + (size_t)max_voxels + (size_t)ceil_div(max_voxels, 64);
    return align_up(ints * sizeof(int32_t));
}

int32_t* tile_weight_array(void* region, int max_voxels) { return static_cast<int32_t*>(region) + 4 + max_tiles(max_voxels) + 1; }
int32_t* tile_weight_sums(void* region, int max_voxels) { return tile_weight_array(region, max_voxels) + max_voxels; }

CutPart make_cut_part(const int32_t* num_out, int K, int max_voxels, int target_rows, int row_weight, int wide, void* region) {
    CutPart c;
    c.num = num_out;
    c.max_voxels = max_voxels;
    c.K = K;
    c.num_cu = gemm_compute_units() / (wide ? wide : 1);
    c.target = target_rows;  // (>= kGemmMinTileRows: the cut table has room for the tiles of any row count)
    c.row_weight = row_weight;
    c.wide = wide ? 1 : 0;
    c.w = tile_weight_array(region, max_voxels);
    c.wsum = tile_weight_sums(region, max_voxels);
    c.hdr = static_cast<int32_t*>(region);
    const int blocks = ceil_div(max_voxels, 256);
    c.blocks = blocks < 512 ? blocks : 512;
    return c;
}

}  // namespace sessd
