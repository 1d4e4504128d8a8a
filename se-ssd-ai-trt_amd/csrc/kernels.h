// kernels.h -- launchers of the gather-GEMM kernels (conv_gemm.hip) used by both conv plugins.
#pragma once

#include <cstring>

#include "common.h"

namespace sessd {

struct GemmArgs {
    const void* in_feat;     // [max_voxels][cin]   FP32 or FP16
    void* out_feat;          // [max_voxels][cout]  FP32 or FP16
    const int32_t* nbr;      // [K][max_voxels] input row feeding (offset k, output row), -1 = none
    const int32_t* num_out;  // device scalar: active output rows
    int max_voxels;
    int K, cin, cout;
    int in_type, out_type;   // SESSD_FLOAT / SESSD_HALF
    const float* w_f32;      // [K][cin][cout]
    const __half* w_f16;     // same layout, rounded to half (used when in_type is HALF)
    const void* w_packed;    // MFMA operand order, or null
    bool halves_finite = false;  // all of w_f16, hence of w_f32: 0 x w is 0 (a kernel may multiply absent neighbours as rows of zeros)
    bool strided = false;    // the rows are others than the input's: fewer neighbours each
    const float* scale;      // [cout] or null
    const float* shift;      // [cout] or null
    int relu;
    int write_pad_rows;      // rows >= *num_out get epilogue(0) (the reference zero-fills them)
    int force_valu;          // skip the MFMA kernels (cross-check)
    const int32_t* tiles;    // tile cuts of this rulebook (tile_cut.hip) or null: tiles of equal length
    DenseTarget dense;       // dense.dense != null: also scatter the rows there (MFMA kernel only)
};

// Tiling of the MFMA gather-GEMM: n active rows on num_cu compute units are cut into num_cu * r tiles,
// r = the smallest tiles-per-CU count that keeps the mean tile at or below the target height, so that every
// CU gets the same number of tiles (a fixed 32-row tiling leaves e.g. 529 tiles for 256 CUs: some CUs run
// three tiles, most two, and the kernel lasts as long as the three).
// The target is the tile capacity of the kernel the rulebook's owner runs (gemm_wide_tile_rows()): the tallest
// tiles the quantisation to whole tiles per CU allows.  Any cut is correct for any kernel: runs longer than
// a kernel's capacity are walked in pieces.
constexpr int kGemmMinTileRows = 48;  // smallest capacity of any kernel: bounds the tile count
constexpr int kGemmMaxOffsets = 27;  // kernel volumes the rulebook holds (3 x 3 x 3)
struct TilePlan {
    int count;   // tiles
    int height;  // rows per tile when all tiles have the same length
};
__host__ __device__ inline TilePlan tile_plan(int n, int num_cu, int target) {
    TilePlan p;
    if (n <= 0) {
        p.count = num_cu;
        p.height = 1;
        return p;
    }
    const int r = (n + num_cu * target - 1) / (num_cu * target);
    p.count = num_cu * r;
    p.height = (n + p.count - 1) / p.count;
    return p;
}
// The FP32 kernel (conv_wide.hip) with few rows and 64 or more output columns: the 64 columns of a tile are dealt to two workgroups,
// so that the tiles stay tall enough to fill their 16-pair blocks while every compute unit has work and reads only its
// columns of the weights.  At the bound a tile has 75 rows (the kernel holds 128 with half of the columns, 112 with 128 channels): beyond
// it the blocks of the unsplit tiles are full enough (64 -> 64 at 3 815 rows 12.2 us split, 14.8 not; at 8 330 16.8, 17.6; at 9 145
// 17.0, 17.6; at 10 070 18.3, 18.0).
// A kernel volume with fewer offsets than could be dealt to the waves (the 3x1x1 layer) is not split.
constexpr int kWideSplitRows = 75, kWideSplitMinOffsets = 16;
__host__ __device__ inline int wide_log2_split(int n, int K, int num_cu) {
    if (num_cu % 2 || K < kWideSplitMinOffsets) return 0;
    return n <= num_cu / 2 * kWideSplitRows ? 1 : 0;
}
int gemm_compute_units();

// bytes of a layer's workspace for the equal-work tile cuts of its rulebook (tile_cut.hip, coord.h); the region's first
// word is the tile count, 0 = none
size_t tile_cut_bytes(int max_voxels);

// picks the kernel for the layer shape; returns SESSD_E_UNSUPPORTED for dtype pairs not covered, and when a
// dense target is set but the layer does not run on the MFMA kernel (see gemm_runs_on_mfma)
int launch_gather_gemm(const GemmArgs& a, hipStream_t stream);
bool gemm_runs_on_mfma(int K, int cin, int cout, int in_type, int out_type);
// whether the layer runs on one of the FP16 kernels (conv_tile.hip, conv_tall.hip) that cut their own tiles: a rulebook
// whose owner does needs no equal-work cuts
bool gemm_cuts_own_tiles(int K, int cin, int cout, int in_type, int out_type);
// whether the layer runs on conv_wide.hip's kernel (where the two above leave it), that kernel's tile capacity, how many rows it
// takes, and whether it multiplies 16-bit parts of FP32 operands, which need weights of a form of their own
bool gemm_runs_wide(int K, int cin, int cout, int in_type, int out_type);
int gemm_wide_tile_rows(int cin, int cout, int type);
bool gemm_wide_takes_rows(int max_voxels, int cin, int cout, int in_type);
bool wide_splits(int cin);
size_t wide_weight_bytes(int K, int cin, int cout);
void pack_wide_weights(const float* w, int K, int cin, int cout, void* dst);

// size in bytes of the packed weight copy for this shape/dtype (0 = shape runs on the VALU path)
size_t packed_weight_bytes(int K, int cin, int cout, int dtype);
// host-side packing into MFMA operand order; dst has packed_weight_bytes() bytes
void pack_weights(const float* w, int K, int cin, int cout, int dtype, void* dst);

// The nearest half, ties to even, as bits, and its value.  (Host code: the weights of a backbone are 500 000 and more, and the
// compiler's conversion is a call.)
inline uint16_t nearest_half(float v, float* value) {
    uint32_t u;
    std::memcpy(&u, &v, 4);
    const uint32_t sign = u & 0x80000000u, mag = u ^ sign;
    uint32_t h, back;
    if (mag >= 0x477ff000u) {  // beyond the largest half, infinite or NaN
        h = mag > 0x7f800000u ? 0x7e00u : 0x7c00u;
        back = mag > 0x7f800000u ? 0x7fc00000u : 0x7f800000u;
    } else if (mag >= 0x38800000u) {
        back = (mag + 0xfffu + ((mag >> 13) & 1u)) & ~0x1fffu;
        h = (back - 0x38000000u) >> 13;
    } else {  // a multiple of 2^-24, the unit of the last place of 1/2
        float f;
        std::memcpy(&f, &mag, 4);
        f += 0.5f;
        std::memcpy(&h, &f, 4);
        h -= 0x3f000000u;
        f -= 0.5f;
        std::memcpy(&back, &f, 4);
    }
    back |= sign;
    std::memcpy(value, &back, 4);
    return (uint16_t)(h | sign >> 16);
}
// rulebook export (reference layout indice_pairs[K][2][max_voxels], indice_num[K])
size_t export_scratch_bytes(int K, int max_voxels);
int launch_export_rulebook(const int32_t* nbr, const int32_t* num_out, int K, int max_voxels,
                           void* scratch, int32_t* indice_pairs, uint32_t* indice_num,
                           hipStream_t stream);

// indice_num[k] only (pairs per offset), same scratch as the export
int launch_count_pairs(const int32_t* nbr, const int32_t* num_out, int K, int max_voxels, void* scratch,
                       uint32_t* indice_num, hipStream_t stream);

}  // namespace sessd
