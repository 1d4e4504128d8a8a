// conv_tall.hip -- gather-GEMM for 3x3x3 layers with few channels (FP16 Cin 16 or 32, FP32 Cin 4 and 16 -> 16): all of W in LDS, no barrier
// between the offsets.
//
//     out[o][:] = epilogue( sum_k  in[nbr[k][o]][:] @ W[k] )
//
// W is 7 to 110 KB and one workgroup a compute unit keeps all of it, so that its waves meet only once, in front of the first product.
//   * A workgroup owns a run of output rows, 16 at a time (a block) for each of its eight waves, and all columns; the accumulators stay
//     in registers over all offsets: no compaction, no partial tiles.  A row without a neighbour contributes a zero operand (a buffer
//     load that points out of range: zeros, no memory touched), so the matrix cores multiply two to four times the useful pairs -- in
//     FP16, and in FP32 with so few channels, they have the headroom.
//   * A step is four offsets.  Lane (i, q) of a wave requests all 32 or 64 bytes of the neighbour of row i at offset 4 step + q, and the inner
//     dimension of an MFMA is eight channels of each of the four offsets: the lane's own list entries are all that it needs, no other
//     lane's, and W is in LDS as the host has packed it (lane (i, q) reads the operand that holds these channels of W[4 step + q]).
//     In FP32 an MFMA takes one channel of each of the four offsets.  Rows are requested two steps (eight offsets) ahead, those of up to
//     32 bytes three, all of them by straight-line code: the compiler's waits are exact.
//   * With few rows (up to four blocks a workgroup, 16 384 rows on 256 units; up to two, 8 192) two or four waves share a block and take
//     every second or fourth step; their sums are added in LDS.  (Workgroups of four waves, coord.hip: 8 192 and 4 096 rows.)
//   * W, the row count and, behind that, the lists are on their way together; the first rows are requested in front of the barrier.
//   * The rows beyond the active ones are written by four waves of their own.
// What bounds it from some 40 000 rows up are the requests for rows in four cache lookups a row (coalesced ones, with a 4 x 4
// transposition in registers, took longer: 49 874 rows 8.4 -> 9.5 us) and the reads of W from LDS (two blocks a wave: 8.4 -> 8.7), below
// the trips to memory: row count, lists, rows.
// Measured against the kernel with a barrier and 2 or 4 KB of W an offset that these layers ran on, launches back to back, 32 -> 32 and
// 32 -> 64: 801 rows 5.05 -> 3.5 us and 5.9 -> 4.8, 13 907 rows 5.3 -> 4.7 and 6.2 -> 6.25, 26 575 rows 7.1 -> 5.7 and 7.9 -> 7.3,
// 49 874 rows 11.2 -> 8.4 and 13.1 -> 10.9, 74 606 rows 13.9 -> 10.9 and 16.1 -> 13.4; frames of 60 000 points 229.6 -> 224.9.
// 16 -> 16 and 16 -> 32 against conv_wide.hip's pair lists (a quarter of the neighbours is there): 1 947 rows 5.0 -> 2.9 us and 5.2 -> 3.2,
// 16 198 rows 7.2 -> 3.3 and 8.1 -> 3.7, 60 000 rows 10.4 -> 4.9 and 11.9 -> 5.8; frames of 60 000 points 225.9 -> 215.7.
// FP32, launches back to back, pair lists -> here: 4 -> 16 at 933 rows 4.7 -> 3.2 us, 16 569 6.5 -> 4.3, 41 489 9.3 -> 6.2, 92 422 16.0 -> 9.2; 4 -> 32
// 5.3 -> 3.9, 8.2 -> 5.8, 11.0 -> 8.9, 21.0 -> 13.9; 16 -> 16 4.8 -> 3.7, 7.2 -> 6.8, 10.8 -> 10.1, 20.1 -> 16.8 (16 -> 32 would multiply
// twelve times its pairs).  That is at a frame's sites, where up to a quarter of the neighbours is there.  With all of them 30 000 rows 10.7 -> 4.5, 13.0 -> 6.2,
// 13.0 -> 7.3; without any 4 -> 16 6.1 -> 4.5, 60 000 rows 8.0 -> 6.8, but 4 -> 32 6.2 -> 6.2 and 8.3 -> 10.0, 16 -> 16 6.7 -> 7.1 and 8.7 -> 11.8: the host knows rows
// and not neighbours.  Distance from 64-bit sums at 41 489 rows 0.645e-7 -> 0.634e-7, 0.640e-7 -> 0.621e-7, 0.803e-7 -> 0.753e-7, at 933 to 51 443 rows 0.56-0.66e-7 ->
// 0.55-0.66e-7, 0.54-0.67e-7 -> 0.55-0.64e-7, 0.72-0.81e-7 -> 0.65-0.76e-7 (sites at random, 8 192 rows with a sixth of the neighbours, of a sum's per offset: 0.88 -> 0.92, 0.88 ->
// 0.93, 0.93 -> 0.79; 30 000 rows 0.76 -> 0.76, 0.77 -> 0.77, 0.83 -> 0.78).
// In a frame two of these layers share launches with passes over coordinates (coord.hip).  Frames on two streams in which they cannot, here / pair lists there:
// three SubM layers in front 2 000 points 171.0 / 173.3 us, 20 000 260.7 / 257.6, 80 000 389.0 / 392.7, a SubM layer on a grid of its own 2 000 202.7 / 205.6, 20 000 283.6 /
// 288.5, 80 000 423.4 / 427.9, on hashes 2 000 197.7 / 195.2, 20 000 291.1 / 290.9, FP16 60 000 points, nothing shared, 194.6 / 202.5.
// The waves are eight because the coordinate passes beside them need registers (12: the same times, and 504 of 512 taken).
// Summation order per output element.  FP16: a wave's steps ascending, in a step the channels eight at a time.  FP32: a step has a sum for each of
// the four channels of a 16-byte piece, over the pieces ascending, of four offsets at a time; (0 + 1) + (2 + 3) goes to one of two totals in turn (4 -> 16: of
// four), and the totals are added two by two at the end.  Where waves share a block, to the first one's sum those of the others, the last one's
// first.  Fixed for a row count and a grid, run-to-run identical; in a launch with more or fewer rows, or on another number of compute units or of
// waves a workgroup, the same row may be summed in another of the three orders.
// (The ring of conv_tile.hip, faster from 64 channels up, has too little work per row here.)
#include "conv_tall.h"

namespace sessd {

namespace {

constexpr int kWaves = 8;     // that multiply
constexpr int kPadWaves = 4;  // that write the rows beyond the active ones

template <int CIN, int COUT, typename T, typename TO, bool PAD>
__global__ void __launch_bounds__((kWaves + (PAD ? kPadWaves : 0)) * 64)
conv_tall(const int32_t* __restrict__ num_out, const int32_t* __restrict__ nbr, const void* __restrict__ in,
          const void* __restrict__ Wp, int max_voxels, int relu, void* __restrict__ out,
          const float* __restrict__ scale, const float* __restrict__ shift, DenseTarget dt) {
    __shared__ tall::Lds<CIN, COUT, T, kWaves> lds;
    TallArgs g;
    g.num_out = num_out;
    g.nbr = nbr;
    g.in = in;
    g.w = Wp;
    g.max_voxels = max_voxels;
    g.relu = relu;
    g.out = out;
    g.scale = scale;
    g.shift = shift;
    tall::workgroup<CIN, COUT, T, TO, kWaves, PAD ? kPadWaves : 0>(g, dt, blockIdx.x, gridDim.x, lds);
}

template <int CIN, int COUT, typename T, typename TO = T>
int launch(const GemmArgs& a, hipStream_t stream) {
    auto go = [&](auto pad) {
        hipLaunchKernelGGL((conv_tall<CIN, COUT, T, TO, decltype(pad)::value>), dim3(gemm_compute_units()),
                           dim3((kWaves + (decltype(pad)::value ? kPadWaves : 0)) * 64), 0, stream, a.num_out, a.nbr,
                           a.in_feat, a.w_packed, a.max_voxels, a.relu, a.out_feat, a.scale,
                           a.shift, a.dense);
    };
    a.write_pad_rows ? go(std::true_type{}) : go(std::false_type{});
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

}  // namespace

bool gemm_runs_tall(int K, int cin, int cout) { return K == tall::KC && ((cin == 32 && (cout == 64 || cout == 32)) || (cin == 16 && (cout == 16 || cout == 32))); }

constexpr int kFewStridedRows = 8192;

bool tall_takes(const GemmArgs& a) {
    // (0 x infinity: with weights that are not finite an absent neighbour may not be a row of zeros)
    if (!a.w_packed || !a.halves_finite || a.force_valu || a.K != tall::KC) return false;
    if ((reinterpret_cast<uintptr_t>(a.in_feat) | reinterpret_cast<uintptr_t>(a.out_feat)) & 15) return false;
    if ((size_t)a.max_voxels * a.cin * dtype_size(a.in_type) >= tall::kOutOfRange) return false;
    if ((size_t)a.max_voxels * (tall::KC * sizeof(int32_t)) >= tall::kOutOfRange) return false;
    if (a.in_type == SESSD_HALF) return a.out_type == SESSD_HALF && gemm_runs_tall(a.K, a.cin, a.cout);
    if (a.cin == 4) return a.cout == 16 || a.cout == 32;
    // (a strided layer's rows have one to three neighbours at a frame's sites, a SubM layer's up to seven: the pair lists are short.  A call, rulebook included, here / there, at a frame's sites
    // 1 000 rows 21.2 / 22.7 us, 5 000 24.6 / 25.4, 12 000 28.3 / 28.1, 27 585 36.9 / 35.2, 49 642 47.4 / 45.8, 92 422 69.2 / 64.9; isolated ones 5 000 26.7 / 26.6,
    // 60 000 79.4 / 69.7.  The host knows the rows that the tensors hold.  4 -> 16 at 27 585 32.9 / 34.3, 92 422 62.0 / 64.9, isolated 60 000 70.7 / 69.6)
    return a.out_type == SESSD_FLOAT && a.cin == 16 && a.cout == 16 && (!a.strided || a.max_voxels <= kFewStridedRows);
}

TallArgs tall_args(const GemmArgs& a) {
    TallArgs g;
    g.num_out = a.num_out;
    g.nbr = a.nbr;
    g.in = a.in_feat;
    g.w = a.w_packed;
    g.out = a.out_feat;
    g.scale = a.scale;
    g.shift = a.shift;
    g.max_voxels = a.max_voxels;
    g.relu = a.relu;
    return g;
}

int launch_tall(const GemmArgs& a, hipStream_t stream) {
    if (!tall_takes(a)) return SESSD_E_UNSUPPORTED;
    if (a.cin == 4 && a.out_type == SESSD_HALF) return a.cout == 16 ? launch<4, 16, float, __half>(a, stream) : launch<4, 32, float, __half>(a, stream);
    if (a.cin == 4) return a.cout == 16 ? launch<4, 16, float>(a, stream) : launch<4, 32, float>(a, stream);
    if (a.in_type == SESSD_FLOAT) return launch<16, 16, float>(a, stream);
    if (a.cin == 32) return a.cout == 64 ? launch<32, 64, __half>(a, stream) : launch<32, 32, __half>(a, stream);
    return a.cout == 16 ? launch<16, 16, __half>(a, stream) : launch<16, 32, __half>(a, stream);
}

}  // namespace sessd
