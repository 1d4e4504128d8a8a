// conv_wide.hip -- gather-GEMM of the FP32 layers from 16 -> 32 up and of all that conv_tile.hip and conv_tall.hip do not take (kernel
// volumes other than theirs, weights that are not finite as halves, large strided FP32 layers 16 -> 16).
//
//     out[o][:] = epilogue( sum_k  in[nbr[k][o]][:] @ W[k] )
//
// A workgroup owns a tile of consecutive output rows (from the rulebook's equal-work cuts, tile_cut.hip, or of equal length)
// and up to 64 columns.  The tile's neighbour lists are compacted per offset with wave64 ballots into pair lists in LDS; the
// offsets are dealt to the waves; a wave multiplies 16 pairs at a time with all columns and adds the block into a partial
// tile of its own in LDS (so the order of every sum is fixed); the partial tiles are summed in a fixed order, scale/shift/ReLU
// follow, each row is stored once.  Results are bit-identical run to run.
//
// Products.  The FP32 matrix instruction does 32 multiply-adds a cycle and SIMD, the 16-bit ones 512.  From 32 channels up both
// operands are split into three BF16 parts of eight bits each, x = x0 + x1 + x2 exactly, and the six largest products of
// parts are added in FP32, smallest first (v_mfma_f32_16x16x32_bf16; 6/16 of the FP32 instruction's time).  What is left out is
// below 2^-23 of a product, and BF16 has FP32's range, so that this holds for every element by itself, whatever the others
// of its row or column are.  What does not fit -- numbers below 2^-110 whose last bits lie under BF16's smallest number,
// infinities and NaN, sums that overflow on the way -- comes out as something that is not finite, and such elements are
// summed again, plainly (direct_sum()).  Two FP16 parts of operands scaled by row and column are three products (64 -> 64 at 17 262
// rows 19.1 us, 24.9 so; the FP32 instruction 32.2) but hold an element to 2^-24 of its row's largest and not of itself: one channel
// at 1e8 beside others at 1 cost these 5e-5 of their sums.  Cin 4 and 16: the FP32 instruction (it is not what they wait for).
// Distance from the sums in 64 bits, 2-norm, FP32 instruction and parts: 64 -> 64 1.27e-7, 0.72e-7; 128 -> 128 1.31e-7, 0.81e-7; 32 -> 32
// 0.93e-7, 0.67e-7.
//
// What bounds it: a block of 64 -> 64 is 768 cycles of MFMA (with half of them left out the launch above took 20.0 us of 24.9), the rest a wave's
// instructions and LDS.  Hence
//   * a wave takes all 64 columns: rows are requested, permuted and split once;
//   * as many waves as LDS holds partial tiles of: eight up to 72 rows and where two workgroups share the columns, seven up to 82, six up
//     to the 96 that a tile of all columns can have (with six on four SIMDs, two of these work alone and slower.  64 -> 64 at 11 252 rows
//     19.6 -> 18.8 us, 14 629 22.9 -> 21.9; 128 -> 128 at 14 629 69.7 -> 66.1; frames of 20 000 points 271 -> 266; up to 4 200 rows the
//     call with its pad rows 13.9 -> 14.2, frames of 2 000 points the same).  Longer runs are walked in two halves rather than in 96
//     rows and the rest (64 -> 64 at 21 591 rows 38.6 -> 34.4);
//   * a block's MFMAs are one column block after the other.  Under those of the next one a column block's sums are added to the partial
//     tile (filling pairs add to a row of their own, so that no branch is in the way) and, where the registers do not hold two
//     sets of weights (64 x 64), the next offset's weights of its columns requested if this is the offset's last block; else these
//     are requested with the offset's first into a second set.  The next block's rows are permuted and those of the block after it
//     requested under the last MFMAs, and split behind them (32 -> 32 at 62 674 rows 32.4 -> 30.6 us, 64 -> 64 at 21 591 34.3 -> 32.9, frames of
//     80 000 points 424 -> 410.  Split between the MFMAs instead: the same, the SIMD's other wave has filled those slots already);
//   * the last, incomplete round of the offsets goes to the waves 0, 1, ..: a SIMD serves its older wave first (64 -> 64 at 4 217 rows 14.3 ->
//     13.6 us, 7 236 17.2 -> 16.7; frames of 2 000 points 190.7 -> 186.7);
//   * a wave's blocks and offsets are listed once, a lane each, and read with readlane: the loop has no other bookkeeping.
// Up to 32 columns two to four workgroups share a unit, as many as the rows need: only where one tile for each unit would be higher than a
// tile can be does a second one begin (32 -> 32, eight waves, 4 208 rows: one workgroup a unit 7.9 us, two 10.7).  Beyond what they hold
// together a launch is two rounds of tiles, of which the second costs its lists and sums again; the tiles are therefore as high, or the
// workgroups as many, as the LDS takes: 16 columns 2 x 128 rows (60 000 rows, 4 -> 16 12.7 -> 10.3 us, 16 -> 16 15.2 -> 12.4 against 2 x 112),
// 4 -> 32 4 x 64 (54 613 rows 16.2 -> 12.7 against 2 x 64), 32 -> 32 3 x 80 (40 088 rows 26.1 -> 21.5, 60 727 33.3 -> 28.4 against 2 x 64; frames of
// 40 000 points 331 -> 324; of 80 000 398 and 405 where the rows are more than the 61 440 that three workgroups a unit hold, the same where
// they are fewer).  What LDS and registers they leave is what the coordinate passes of a frame's other branch run in: 32 -> 32 with eight waves is the faster launch (15.9 us against 17.1 at
// 28 043 rows) and makes the slower frame (20 000 points: 283 us against 274); 4 -> 32 likewise (487 against 475).  16 -> 32 with four waves and
// 3 x 80 rows: 54 613 rows 18.4 -> 17.4 us, but 17 132 rows 9.0 -> 11.4.
// FP16 features have so little in each block that with up to 32 columns four waves and 64 rows do: four workgroups share a unit, with up to 40 KB of
// LDS each.  3x3x3 layers are faster without pair lists (16 -> 16 at 60 000 rows 4.9 us on conv_tall.hip, 10.4 here; 32 -> 32 at 49 874 8.4 there,
// at 45 874 18 here) and come here where a weight is infinite or NaN as a half, and an absent neighbour must not be a row of zeros.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <utility>
#include <vector>

#include "pad_rows.h"

namespace sessd {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2b __attribute__((ext_vector_type(2)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef unsigned int v2u32 __attribute__((__vector_size__(8)));
typedef unsigned int v4u32 __attribute__((__vector_size__(16)));

constexpr int kMaxK = kGemmMaxOffsets;
constexpr unsigned kOutOfRange = 0x80000000u;  // beyond any buffer the kernel is given (launch() checks)
constexpr int kRawBuffer = 0x00020000;         // descriptor word 3: raw 32-bit data format, no swizzle

// how a layer's products are made: FP32 MFMA, or 16-bit MFMA on operands split into parts
enum Arith { kPlain, kThirds, kFp16 };
constexpr Arith arith(int cin) { return cin >= 32 ? kThirds : kPlain; }  // (of FP32 features)

// an entry of a pair list: input row << bits | row in the tile
constexpr uint32_t kNoPair = 0xffffff00u;  // fills up a list's last block (no input row has that number: gemm_wide_takes_rows())
constexpr int pair_row_bits(int tile_rows) { return tile_rows <= 64 ? 6 : 7; }

template <typename T, int CIN, int COUT>  // T: the input features' type
struct Shape {
    static constexpr Arith kArith = sizeof(T) == 2 ? kFp16 : arith(CIN);
    static constexpr int kWeightBytes = CIN * COUT * (kArith == kFp16 ? 2 : (kArith == kThirds ? 6 : 4));  // of an offset
    static constexpr int kWgCols = COUT < 64 ? COUT : 64;  // columns of a workgroup (before the split of short tiles)
    static constexpr int kColGroups = COUT / kWgCols;      // workgroups beside each other
    // (32 columns: four waves with 4 and 32 channels, whose launches are long enough for the frame's other branch to need the LDS)
    static constexpr int kWaves = kWgCols == 64 ? 8 : (sizeof(T) == 2 || (COUT == 32 && CIN != 16) ? 4 : 8);
    static constexpr int kThreads = kWaves * 64;
    static constexpr int kParts = CIN > 64 ? CIN / 64 : 1;  // of the inner dimension, taken one after the other
    static constexpr int CP = CIN / kParts;                 // channels of a part
    // Rows of a tile at most, and workgroups that can share a compute unit.  64 columns: as many waves multiply as the LDS holds partial
    // tiles of the tile's rows, eight up to 72 rows and kFewestWaves with kWholeRows; with half of the columns always all.
    static constexpr int kTileRows = kWgCols == 64 ? (kParts > 1 ? 112 : 128) : (sizeof(T) == 2 ? 64 : (kWgCols == 16 ? 128 : (CIN == 32 ? 80 : 64)));
    static constexpr int kWholeRows = kWgCols == 64 ? 96 : kTileRows;
    static constexpr int kFewestWaves = kWgCols == 64 ? 6 : kWaves;
    static constexpr int kPartRows = kFewestWaves * kWholeRows;  // of all partial tiles together
    static constexpr int kPerUnit = kWgCols == 64 ? 1 : (sizeof(T) == 2 || (CIN == 4 && COUT == 32) ? 4 : (CIN == 32 ? 3 : 2));
    static constexpr int kMaxBlk = kTileRows / 16;
    static constexpr int kRowBits = pair_row_bits(kTileRows);
    static constexpr int kNone = kMaxK * kTileRows * 4;  // an item with no pairs
    static constexpr int kRowBytes = CIN * (int)sizeof(T), kPartBytes = CP * (int)sizeof(T);
    static constexpr int kLaneBytes = kPartBytes < 64 ? kPartBytes / 4 : 16;  // of a row that a lane requests at a time; of a weight operand as well
    static constexpr int G = kPartBytes / (4 * kLaneBytes);  // requests for a part
    static constexpr int kMaxSplit = kWgCols == 64 ? 1 : 0;  // log2 of the column parts that short tiles are split into
    static_assert(kTileRows <= 128 && kTileRows % 16 == 0, "the lists are staged in two halves of 64 rows");
    static_assert((CP == 4 || CP % 16 == 0) && (kArith == kPlain || kArith == kFp16 || CP % 32 == 0) && COUT % kWgCols == 0, "whole MFMA steps and column groups");
    static_assert(kTileRows <= 1 << kRowBits, "a pair holds its row in the tile");
    static_assert((kMaxK + kWaves - 1) / kWaves * kMaxBlk * kParts + 2 <= 64 &&
                  (kMaxK + kFewestWaves - 1) / kFewestWaves * (kWholeRows / 16) * kParts + 2 <= 64, "an item a lane");
    static_assert(kMaxSplit == 0 || kWaves * kTileRows <= 2 * kPartRows, "partial tiles of half of the columns");
};

__device__ __forceinline__ void buffer_load(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, int (&v)[4]) {
    const v4u32 t = __builtin_amdgcn_raw_buffer_load_b128(r, byte_offset, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (int)t[e];
}
__device__ __forceinline__ void buffer_load(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, int (&v)[2]) {
    const v2u32 t = __builtin_amdgcn_raw_buffer_load_b64(r, byte_offset, 0, 0);
    v[0] = (int)t[0];
    v[1] = (int)t[1];
}
__device__ __forceinline__ void buffer_load(__amdgpu_buffer_rsrc_t r, unsigned byte_offset, int (&v)[1]) {
    v[0] = (int)__builtin_amdgcn_raw_buffer_load_b32(r, byte_offset, 0, 0);
}
__device__ __forceinline__ void store4(float* dst, const float (&o)[4]) { *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]); }
__device__ __forceinline__ void store4(__half* dst, const float (&o)[4]) {
    union {
        __half2 h[2];
        uint2 u;
    } p;
    p.h[0] = __floats2half2_rn(o[0], o[1]);
    p.h[1] = __floats2half2_rn(o[2], o[3]);
    *reinterpret_cast<uint2*>(dst) = p.u;
}

constexpr unsigned kUpperHalves = 0x07060302u;  // v_perm_b32: the upper half of the second word, then that of the first

template <typename V>
__device__ __forceinline__ V operand8(const int* w) {
    const int4 v = make_int4(w[0], w[1], w[2], w[3]);
    return __builtin_bit_cast(V, v);
}

// What a lane holds of a 16-pair block's rows (take(): in operand order) and of an offset's weights, and the products of the two.
template <typename S, int NB, Arith>
struct Products;

// FP16 features: their own MFMA
template <typename S, int NB>
struct Products<S, NB, kFp16> {
    static constexpr int G = S::G, E = S::kLaneBytes / 4, kWords = G * E, kPieces = G;
    static __device__ __forceinline__ void take(const int (&a)[G][E], int (&p)[kWords]) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < E; ++e) p[g * E + e] = a[g][e];
    }
    static __device__ __forceinline__ void multiply(const int (&w)[G][NB][E], const int (&x)[kWords], v4f (&acc)[NB]) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                if constexpr (E == 4) {
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand8<v8h>(w[g][nb]), operand8<v8h>(x + g * E), acc[nb], 0, 0, 0);
                } else {
                    const int2 a = make_int2(w[g][nb][0], w[g][nb][1]), b = make_int2(x[g * E], x[g * E + 1]);
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(v4h, a), __builtin_bit_cast(v4h, b), acc[nb], 0, 0, 0);
                }
            }
    }
};

// FP32 MFMA
template <typename S, int NB>
struct Products<S, NB, kPlain> {
    static constexpr int G = S::G, E = S::kLaneBytes / 4, kWords = G * E, kPieces = G;  // (pieces: weight operands a column block)
    static __device__ __forceinline__ void take(const int (&a)[G][E], int (&p)[kWords]) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < E; ++e) p[g * E + e] = a[g][e];
    }
    static __device__ __forceinline__ void multiply(const int (&w)[G][NB][E], const int (&x)[kWords], v4f (&acc)[NB]) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < E; ++e)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(__int_as_float(w[g][nb][e]), __int_as_float(x[g * E + e]), acc[nb], 0, 0, 0);
    }
};

// BF16 MFMA on three parts of eight bits each, x = x0 + x1 + x2: x0 cut off (rounded, the largest numbers would become
// infinite), x1 rounded, x2 what is left, which eight bits hold unless it reaches below BF16's smallest number; such a row becomes
// NaN.  The six largest products of parts, smallest first.
template <typename S, int NB>
struct Products<S, NB, kThirds> {
    static constexpr int G = S::G, E = 4, C = S::CP / 32, kWords = G * 6, kPieces = 3 * C;  // (words: x0, x1, x2)
    static __device__ __forceinline__ void take(const int (&a)[G][E], int (&p)[kWords]) {
        uint32_t left = 0;  // (of any element beyond the three parts: the low half of a word)
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const uint32_t u0 = (uint32_t)a[g][2 * e], u1 = (uint32_t)a[g][2 * e + 1];
                const int at = 2 * g + e;
                p[at] = (int)__builtin_amdgcn_perm(u1, u0, kUpperHalves);
                v2f r = {__uint_as_float(u0) - __uint_as_float(u0 & 0xffff0000u), __uint_as_float(u1) - __uint_as_float(u1 & 0xffff0000u)};
                int w = __builtin_bit_cast(int, __builtin_convertvector(r, v2b));
                asm("" : "+v"(w));
                p[2 * G + at] = w;
                const uint32_t r0 = __float_as_uint(r.x - __int_as_float(w << 16)), r1 = __float_as_uint(r.y - __int_as_float(w & (int)0xffff0000));
                p[4 * G + at] = (int)__builtin_amdgcn_perm(r1, r0, kUpperHalves);
                left |= r0 | r1;
            }
        p[kWords - 1] |= left & 0xffffu ? 0x7fff : 0;  // (the last word: what waits for all of them is last)
    }
    // the MFMAs of a block in their order: one column block after the other, whose weights are free behind it
    static constexpr int kSteps = 6 * C * NB;
    static __device__ __forceinline__ void step(int n, const int (&w)[3 * C][NB][E], const int (&x)[kWords], v4f (&acc)[NB]) {
        constexpr int kPart[6][2] = {{0, 2}, {1, 1}, {2, 0}, {0, 1}, {1, 0}, {0, 0}};  // of w, of x
        const int nb = n / (6 * C), t = n / C % 6, c = n % C;
        acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operand8<v8b>(w[kPart[t][0] * C + c][nb]),
                                                          operand8<v8b>(x + 2 * G * kPart[t][1] + 4 * c), acc[nb], 0, 0, 0);
    }
};

// f(0), f(1) .. f(N - 1), the numbers as types
template <typename F, int... N>
__device__ __forceinline__ void unrolled(F f, std::integer_sequence<int, N...>) {
    (f(std::integral_constant<int, N>{}), ...);
}

// One wave's share of a tile: the pairs of the offsets dealt to it, times its columns -- 16-column blocks nb0 .. nb0 + NB - 1
// of the layer -- into its partial tile `part` (rows of 16 NB floats).  waves: among which the offsets are dealt; most: blocks that an
// offset can have in this tile; spare: a row for what filling pairs add.
template <typename S, int COUT, int NB, typename Pads>
__device__ __forceinline__ void multiply(__amdgpu_buffer_rsrc_t rs_in, __amdgpu_buffer_rsrc_t rs_w, const uint32_t* s_pair,
                                         const int32_t* s_blk, int K, int wave, int waves, int lane, int nb0, int most, float* part, float* spare, Pads& pads) {
    using P = Products<S, NB, S::kArith>;
    constexpr int kParts = S::kParts, G = S::G, E = S::kLaneBytes / 4, kTileRows = S::kTileRows;
    constexpr int kSets = P::kPieces * NB * E > 64 ? 1 : 2;  // of weights: the registers do not hold two of the largest
    constexpr int NBT = COUT / 16;                   // 16-column blocks of the layer
    constexpr int kSlots = NB * 4;                   // 16-byte slots of a row of the partial tile
    const int i = lane & 15;  // pair inside a 16-pair block
    const int q = lane >> 4;  // channel group of a step

    // offsets of this wave: ranked by their number of 16-pair blocks (ballots: lane k holds offset k)
    // and dealt in that order back and forth over the waves (0 1 2 3 3 2 1 0 ...; or 3 2 1 0 0 1 2 3 ...)
    const int blocks_of = lane < K ? s_blk[lane] : 0;
    uint32_t mask;
    {
        int rank = 0, ahead = 0;
        for (int size = most; size >= 1; --size) {
            const uint64_t m = __ballot(blocks_of == size);
            const int before = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, ahead));
            if (blocks_of == size) rank = before;
            ahead += __popcll(m);
        }
        int r2 = rank;
        if constexpr (S::kFewestWaves == S::kWaves) {
            r2 = rank % (2 * waves);
        } else {  // (without a division: fewer than three rounds)
            static_assert(kMaxK <= 6 * S::kFewestWaves, "rounds");
            r2 -= r2 >= 4 * waves ? 4 * waves : 0;
            r2 -= r2 >= 2 * waves ? 2 * waves : 0;
        }
        // (the last round, of few offsets, begins with the first wave: the older waves of a SIMD are served first and end earlier)
        const int lists = __popcll(__ballot(blocks_of > 0));
        int rounds = 0;
#pragma unroll
        for (int n = 0; n * S::kFewestWaves < kMaxK; ++n) rounds += lists > n * waves;
        const bool back = (r2 >= waves) != (rounds % 2 == 0);
        const int in_round = r2 < waves ? r2 : r2 - waves;
        const int w = back ? waves - 1 - in_round : in_round;
        mask = (uint32_t)__ballot(blocks_of > 0 && w == wave);
    }
    if (!mask) return;
    // An item is a 16-pair block of an offset (and of a part of the channels); a stage is an offset (and a part).  An offset's blocks
    // are walked once for each part.  Lane t: where item t's pairs begin in s_pair, and its part; lane s: stage s.
    int items = 0, stages = 0, item_at = S::kNone, stage_at = -1, stage_items = 0;
    while (mask) {
        const int k = __ffs(mask) - 1;
        mask &= ~(1u << k);
        const int n = __builtin_amdgcn_readlane(blocks_of, k);
#pragma unroll
        for (int part_no = 0; part_no < kParts; ++part_no) {
            const int t = lane - items;
            if (t >= 0 && t < n) item_at = ((k * kTileRows + t * 16) * 4) | part_no;
            if (lane == stages) {
                stage_at = k * kParts + part_no;
                stage_items = n;
            }
            items += n;
            ++stages;
        }
    }
    // Rows are requested with four neighbouring lanes on the 64 contiguous bytes of one row (lane l: pair l / 4 of
    // the block, bytes 16 * (l % 4) ..): the cache looks up one line per group of four lanes.  In the MFMA's
    // operand order -- lane l: pair l % 16, bytes 16 * (l / 16) .. -- the four lanes of a group name four
    // different rows and the same request takes four lookups: 18 instead of 48 bytes per cycle and compute unit,
    // measured.  The operand order is restored by a lane permutation when the rows have arrived.
    // Filling pairs ask out of range (such a request returns zeros and touches no memory).
    const char* pairs = reinterpret_cast<const char*>(s_pair);
    auto entry_at = [&](int it, int j4) -> uint32_t { return *reinterpret_cast<const uint32_t*>(pairs + (kParts > 1 ? it & ~3 : it) + j4); };
    auto load_a = [&](int it, uint32_t entry, int (&a)[G][E]) {
        const unsigned row = (entry >> S::kRowBits) * (unsigned)S::kRowBytes + (kParts > 1 ? (unsigned)(it & 3) * (unsigned)S::kPartBytes : 0u);
        const unsigned at = entry < kNoPair ? row + (lane & 3) * (unsigned)S::kLaneBytes : kOutOfRange;
#pragma unroll
        for (int g = 0; g < G; ++g) buffer_load(rs_in, at + g * 64u, a[g]);
    };
    auto stage_weights = [&](int stage) -> unsigned {  // (stage < 0: nothing to fetch)
        return stage >= 0 ? (unsigned)(((stage * P::kPieces * NBT + nb0) * 64 + lane) * S::kLaneBytes) : kOutOfRange;
    };
    auto load_b1 = [&](unsigned at, int (&b)[P::kPieces][NB][E], int nb) {
#pragma unroll
        for (int c = 0; c < P::kPieces; ++c) buffer_load(rs_w, at + (c * NBT + nb) * (64u * S::kLaneBytes), b[c][nb]);
    };
    auto load_b = [&](int stage, int (&b)[P::kPieces][NB][E]) {
        const unsigned at = stage_weights(stage);
#pragma unroll
        for (int c = 0; c < P::kPieces; ++c)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) buffer_load(rs_w, at + (c * NBT + nb) * (64u * S::kLaneBytes), b[c][nb]);
    };
    const int from_lane4 = (4 * i + q) * 4;  // ds_bpermute address: this lane's operand sits in lane 4 * i + q
    const int request4 = lane & ~3, operand4 = i * 4;  // this lane's pair of a block in the request's and in the operands' order, times 4
    int d0 = __builtin_amdgcn_readlane(item_at, 0), d1 = __builtin_amdgcn_readlane(item_at, 1), d2;
    int a[G][E], p[P::kWords], b0[P::kPieces][NB][E], b1[kSets == 2 ? P::kPieces : 1][NB][E];
    auto take = [&]() {  // (permuted before they are split: two words instead of three)
        int row[G][E];
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < E; ++e) row[g][e] = __builtin_amdgcn_ds_bpermute(from_lane4, a[g][e]);
        P::take(row, p);
#pragma unroll
        for (int w = 0; w < P::kWords; ++w) asm volatile("" : "+v"(p[w]));  // (here, not where they are used: `a` is free for the next request)
    };
    load_a(d0, entry_at(d0, request4), a);
    load_b(__builtin_amdgcn_readlane(stage_at, 0), b0);
    uint32_t next_entry = entry_at(d1, request4);
    __builtin_amdgcn_sched_barrier(0);
    take();
    __builtin_amdgcn_sched_barrier(0);
    load_a(d1, next_entry, a);
    int t = 0, stage = 0;

    // `use`: the weights of the item's stage; `fill`: those of the next one, requested behind its first block, or, where there is one
    // set, behind its last
    auto plain_item = [&](const int (&use)[P::kPieces][NB][E], int (&fill)[P::kPieces][NB][E], bool request) {
        if constexpr (S::kArith != kThirds) {
            d2 = __builtin_amdgcn_readlane(item_at, t + 2);
            ++t;
            next_entry = entry_at(d2, request4);
            const uint32_t mine = entry_at(d0, operand4);
            const int r = (int)(mine & ((1u << S::kRowBits) - 1u));
            float4* const dst = reinterpret_cast<float4*>(part) + r * kSlots;
            float4 sum[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) sum[nb] = dst[(nb * 4 + q) ^ (r & (kSlots - 1))];
            v4f acc[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = (v4f){0.f, 0.f, 0.f, 0.f};
            P::multiply(use, p, acc);
            take();  // (of d1's rows)
            __builtin_amdgcn_sched_barrier(0);  // (or the requests below take other registers)
            if (request) load_b(__builtin_amdgcn_readlane(stage_at, stage + 1), fill);
            // (behind the weights in either case: what the waits count is then the same for every item)
            load_a(d2, next_entry, a);
            pads.step();  // (behind what the next item waits for)
            if (mine < kNoPair) {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    float4 v = sum[nb];
                    v.x += acc[nb][0];
                    v.y += acc[nb][1];
                    v.z += acc[nb][2];
                    v.w += acc[nb][3];
                    dst[(nb * 4 + q) ^ (r & (kSlots - 1))] = v;
                }
            }
            d0 = d1;
            d1 = d2;
        }
    };
    // The same with what there is to do between the MFMAs in its place: a column block's sums are added under the products of the
    // next, the rows permuted and requested under the last.
    auto dense_item = [&](const int (&use)[P::kPieces][NB][E], int (&fill)[P::kPieces][NB][E], auto request) {
        if constexpr (S::kArith == kThirds) {
            constexpr int kBlockSteps = P::kSteps / NB, kAddAt = kBlockSteps / 3, kRowsAt = P::kSteps - P::kSteps / 12;
            d2 = __builtin_amdgcn_readlane(item_at, t + 2);
            ++t;
            next_entry = entry_at(d2, request4);
            const uint32_t mine = entry_at(d0, operand4);
            const unsigned next = stage_weights(request.value ? __builtin_amdgcn_readlane(stage_at, stage + 1) : -1);
            const int r = (int)(mine & ((1u << S::kRowBits) - 1u));
            float4* const dst = mine < kNoPair ? reinterpret_cast<float4*>(part) + r * kSlots : reinterpret_cast<float4*>(spare);
            float4 sum[NB];
            v4f acc[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) acc[nb] = (v4f){0.f, 0.f, 0.f, 0.f};
            auto add = [&](int nb) {
                float4 v = sum[nb];
                v.x += acc[nb][0];
                v.y += acc[nb][1];
                v.z += acc[nb][2];
                v.w += acc[nb][3];
                dst[(nb * 4 + q) ^ (r & (kSlots - 1))] = v;
            };
            int row[G][E];
            __builtin_amdgcn_sched_barrier(0);
            unrolled([&](auto n_c) {
                constexpr int n = decltype(n_c)::value;
                P::step(n, use, p, acc);
                if constexpr (n == 1) {
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) sum[nb] = dst[(nb * 4 + q) ^ (r & (kSlots - 1))];
                }
                if constexpr (request.value && kSets == 1 && n % kBlockSteps == kBlockSteps - 1) load_b1(next, fill, n / kBlockSteps);
                if constexpr (n >= kBlockSteps && n % kBlockSteps == kAddAt) add(n / kBlockSteps - 1);
                if constexpr (n == kRowsAt) {
#pragma unroll
                    for (int g = 0; g < G; ++g)
#pragma unroll
                        for (int e = 0; e < E; ++e) row[g][e] = __builtin_amdgcn_ds_bpermute(from_lane4, a[g][e]);
                    if constexpr (request.value && kSets == 2) load_b(__builtin_amdgcn_readlane(stage_at, stage + 1), fill);
                    load_a(d2, next_entry, a);
                    pads.step();  // (behind what the next item waits for)
                }
                __builtin_amdgcn_sched_barrier(0);
            }, std::make_integer_sequence<int, P::kSteps>{});
            add(NB - 1);
            P::take(row, p);
#pragma unroll
            for (int w = 0; w < P::kWords; ++w) asm volatile("" : "+v"(p[w]));
            d0 = d1;
            d1 = d2;
        }
    };
    auto run_stage = [&](const int (&use)[P::kPieces][NB][E], int (&fill)[P::kPieces][NB][E]) -> bool {
        const int n = __builtin_amdgcn_readlane(stage_items, stage);
        if constexpr (S::kArith == kThirds) {
            if constexpr (kSets == 2) dense_item(use, fill, std::true_type{});
            for (int j = 1; j < n; ++j) dense_item(use, fill, std::false_type{});
            if constexpr (kSets == 1) dense_item(use, fill, std::true_type{});
        } else {
            for (int j = 0; j < n; ++j) plain_item(use, fill, j == (kSets == 2 ? 0 : n - 1));
        }
        return ++stage < stages;
    };
    if constexpr (kSets == 2)
        while (run_stage(b0, b1) && run_stage(b1, b0)) {}
    else
        while (run_stage(b0, b0)) {}
}

// Four output elements of a row as plain FP32 sums (nbr: the row's neighbour at offset 0; the others follow max_voxels apart).  Bound
// by the reads of W, 16 channels of it on their way at a time: where every row of a 64 -> 64 layer at 17 262 rows needs it the
// launch takes 279 us (one channel at a time 679), with NaN or infinities in every row 66 (132), with none 25.
template <int CIN, int COUT>
__device__ __forceinline__ void direct_sum(const float* __restrict__ in, const float* __restrict__ w, const int32_t* __restrict__ nbr,
                                           int max_voxels, int K, int col, float (&o)[4]) {
    constexpr int kAtOnce = 16;
    o[0] = o[1] = o[2] = o[3] = 0.f;
    int next = nbr[0];
    for (int k = 0; k < K; ++k) {
        const int idx = next;
        if (k + 1 < K) next = nbr[(size_t)(k + 1) * max_voxels];
        if (idx < 0) continue;
        const float4* x4 = reinterpret_cast<const float4*>(in + (size_t)idx * CIN);
        const float* wk = w + (size_t)k * CIN * COUT + col;
        float sum[4] = {0.f, 0.f, 0.f, 0.f};  // (in three levels: fewer roundings follow each other)
#pragma unroll 1
        for (int c0 = 0; c0 < CIN; c0 += kAtOnce) {
            float t[4] = {0.f, 0.f, 0.f, 0.f};
            float4 x[kAtOnce / 4], y[kAtOnce];
#pragma unroll
            for (int c = 0; c < kAtOnce / 4; ++c) x[c] = x4[c0 / 4 + c];
#pragma unroll
            for (int c = 0; c < kAtOnce; ++c) y[c] = *reinterpret_cast<const float4*>(wk + (size_t)(c0 + c) * COUT);
#pragma unroll
            for (int c = 0; c < kAtOnce; ++c) {
                const float v = reinterpret_cast<const float*>(x)[c];
                t[0] = fmaf(v, y[c].x, t[0]);
                t[1] = fmaf(v, y[c].y, t[1]);
                t[2] = fmaf(v, y[c].z, t[2]);
                t[3] = fmaf(v, y[c].w, t[3]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += t[e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += sum[e];
        if (o[0] != o[0] && o[1] != o[1] && o[2] != o[2] && o[3] != o[3]) break;  // (NaN from here on)
    }
}

// The number of workgroups and what is done to the sums, in one argument that is in a register when the kernel starts.  As arguments of their own
// scale, shift and relu were compared with 0 in front of the loops (no store can change them), which was a trip to memory between the cuts and the
// requests for the lists: frames of 2 000 points 167.0 -> 164.3 us, 5 000 189.0 -> 187.6; 20 000 255.9 -> 254.9 and 80 000 381 -> 380, which is within
// what runs of one side differ by (copies of the pointers inside the loops instead: scalar registers spill, 2 000 points 1.014x).
constexpr unsigned kUnitsMask = 0xffffffu, kHasScale = 1u << 24, kHasShift = 2u << 24, kRelu = 4u << 24;

// DENSE: the epilogue also scatters the rows into a dense tensor (the layer in front of sparse2Dense).  PAD: the rows beyond the
// active ones are written too.  Variants of their own: what they need in registers is missing in the launches without.
template <int CIN, int COUT, typename T, typename TO, bool DENSE, bool PAD>
__global__ void __launch_bounds__((Shape<T, CIN, COUT>::kThreads), (Shape<T, CIN, COUT>::kWaves * Shape<T, CIN, COUT>::kPerUnit / 4))
conv_wide(const int32_t* __restrict__ num_out, const int32_t* __restrict__ tiles, const int32_t* __restrict__ nbr,
          const void* __restrict__ Wp, const T* __restrict__ in, int max_voxels, int K, unsigned units_and_flags, TO* __restrict__ out,
          const float* __restrict__ w_f32, const float* __restrict__ scale, const float* __restrict__ shift, DenseTarget dt) {
    const int units = (int)(units_and_flags & kUnitsMask);
    const bool has_scale = units_and_flags & kHasScale, has_shift = units_and_flags & kHasShift, relu = units_and_flags & kRelu;
    using S = Shape<T, CIN, COUT>;
    constexpr int kWgCols = S::kWgCols, kMaxSplit = S::kMaxSplit, kTileRows = S::kTileRows, kWaves = S::kWaves, kThreads = S::kThreads;
    // (one block more: all of it filling pairs)
    __shared__ uint32_t s_pair[kMaxK * kTileRows + 16];  // compacted pair lists: pair j of offset k
    __shared__ int32_t s_blk[kMaxK + 5];            // 16-pair blocks per offset
    __shared__ float s_epi[3 * COUT];
    __shared__ __align__(16) float s_part[S::kPartRows * kWgCols + (S::kArith == kThirds ? kWgCols : 0)];  // (and the spare row)

    // The row count, the number of cuts and the cuts of this workgroup's first tile under each split it may be part of are one
    // trip to memory: without a branch around any of them (no cuts: the row count's word in their place; with branches they and the
    // arguments that do not fit in registers were six trips, 2 700 cycles).
    const int32_t* const cuts = tiles ? tiles : num_out;
    const unsigned has_cuts = tiles ? 1 : 0;
    int n = *num_out;
    int cut_count = cuts[0];
    // Workgroups of `units` tiles for each 64 columns of the layer; what follows counts inside one such group.
    int block = blockIdx.x, col0 = 0;
    if constexpr (COUT > kWgCols) {
        col0 = block / units * kWgCols;
        block %= units;
    }
    int cut_begin[kMaxSplit + 1], cut_end[kMaxSplit + 1], tile_of[kMaxSplit + 1];
#pragma unroll
    for (int s = 0; s <= kMaxSplit; ++s) {
        tile_of[s] = s && block >= units >> 1 ? block - (units >> 1) : block;
        const unsigned at = tiles ? 4u + (unsigned)tile_of[s] : 0u;
        cut_begin[s] = cuts[at];
        cut_end[s] = cuts[at + has_cuts];
    }
#pragma unroll
    for (int s = 0; s <= kMaxSplit; ++s) asm volatile("" : "+s"(n), "+s"(cut_count), "+s"(cut_begin[s]), "+s"(cut_end[s]));
    cut_count = tiles ? cut_count : 0;
    n = n < 0 ? 0 : (n > max_voxels ? max_voxels : n);
    // Column parts: 1 << lsplit workgroups share a tile.  The parts of a tile are row_groups apart in the grid, which
    // puts them on one XCD (workgroups are dealt round robin over eight): they read the same rows.
    const int lsplit = kMaxSplit ? wide_log2_split(n, K, units) : 0;
    const int row_groups = units >> lsplit;  // workgroups of one column part
    const int first_tile = tile_of[kMaxSplit ? lsplit : 0];
    const int first_begin = cut_begin[kMaxSplit ? lsplit : 0], first_end = cut_end[kMaxSplit ? lsplit : 0];
    const int part_id = lsplit && block >= row_groups ? 1 : 0;
    const int thread = threadIdx.x, own_wave = __builtin_amdgcn_readfirstlane(thread >> 6);  // (tells the compiler that it is wave-uniform)

    // The grid is one workgroup per compute unit (a workgroup takes most of a unit's LDS, so workgroups with no
    // tile would queue behind the busy ones just to return); a workgroup walks tiles first_tile, first_tile +
    // row_groups, ...: runs of rows from the rulebook's equal-work cuts, or runs of equal length.
    // (Workgroups share a unit only where one tile for each unit would be higher than they are: a tile's weights are the same for any height.)
    int walkers = row_groups;
    if (S::kPerUnit > 1 && cut_count == 0) {
        const int per_unit = (n + units / S::kPerUnit * kTileRows - 1) / (units / S::kPerUnit * kTileRows);
        walkers = units / S::kPerUnit * (per_unit < 1 ? 1 : (per_unit > S::kPerUnit ? S::kPerUnit : per_unit));
    }
    TilePlan plan = {0, 0};
    if (cut_count == 0) plan = tile_plan(n, walkers, kMaxSplit && lsplit ? kTileRows : S::kWholeRows);
    const int tile_count = cut_count > 0 ? cut_count : (n > 0 ? plan.count : 0);
    bool idle = true;  // (no rows)
    // Rows beyond the active ones: beside the products of a workgroup's first tile where there are as many of them as of the others, else
    // behind its last.  A step is paid for with every block of pairs, whether the wave has anything left to write or not.  Behind / beside:
    // 64 -> 64 at 30 000 rows, 2 000 to write 29.3 / 29.6 us, 20 000 29.6 / 29.4, 50 000 30.8 / 29.8; 32 -> 32 12.2 / 12.6, 12.5 / 12.7, 13.0 / 12.8;
    // 4 -> 16 at 8 000 rows, 8 000 to write 5.7 / 5.5, at 50 000 rows 9.7 / 9.8, 150 000 to write 11.2 / 10.8.  In a full tensor 64 -> 64 at
    // 50 000 rows 45.1 (46.2 with a step for every block).
    const bool beside = PAD && max_voxels - n >= n && PadRows<TO, COUT>::reach(n, max_voxels);
    for (int tile = first_tile; tile < tile_count; tile += walkers) {
    int run_begin, run_end;
    if (cut_count > 0) {
        run_begin = tile == first_tile ? first_begin : tiles[4 + tile];
        run_end = tile == first_tile ? first_end : tiles[5 + tile];
    } else {
        run_begin = tile * plan.height;
        run_end = run_begin + plan.height < n ? run_begin + plan.height : n;
    }
    // a run longer than the tile capacity (sparse stretches under equal-work cuts) is walked in pieces, of equal length if two do
    const int capacity = kMaxSplit && lsplit ? kTileRows : S::kWholeRows, length = run_end - run_begin;
    const int piece = length <= capacity ? capacity : (length <= 2 * capacity ? (length + 1) >> 1 : capacity);
    for (int row0 = run_begin; row0 < run_end; row0 += piece) {
    const int rows = run_end - row0 < piece ? run_end - row0 : piece;

    // ---- stage + compact: a wave turns an offset's neighbour list (two halves of 64 rows) into a pair list ----
    constexpr int kListsPerWave = (kMaxK + kWaves - 1) / kWaves;
    int staged[kListsPerWave][2];
    auto ask = [&](int h) {
        uint64_t at = reinterpret_cast<uint64_t>(nbr) + 4 * ((uint64_t)(uint32_t)own_wave * (uint32_t)max_voxels + (uint32_t)(row0 + 64 * h));
#pragma unroll
        for (int s = 0; s < kListsPerWave; ++s) {
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                reinterpret_cast<void*>(at), 0, own_wave + s * kWaves < K ? (rows - 64 * h) * 4 : 0, kRawBuffer);
            staged[s][h] = (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (thread & 63) * 4, 0, 0);
            at += 4 * (uint64_t)kWaves * (uint32_t)max_voxels;
        }
    };
    const bool tall = kTileRows > 64 && rows > 64;  // (more than one half)
    ask(0);
    if (tall) ask(1);
    // What everything else is computed from is hidden from the compiler until these requests are out: it would compute it in front of
    // the loops, 200 instructions and the trip to memory of the arguments that are not in registers.  (64 -> 64 at 2 448 rows 10.9 ->
    // 10.2 us, 8 662 18.8 -> 18.0, 17 262 25.0 -> 24.5; frames of 2 000 points 193.2 -> 187.9, 20 000 279.9 -> 273.8.  One asm for each: an
    // asm that also has a vector operand makes the scalar ones divergent.)
    __builtin_amdgcn_sched_barrier(0);
    int tid = thread, wave = own_wave, volume = K, split = __builtin_amdgcn_readfirstlane(lsplit), part_of = __builtin_amdgcn_readfirstlane(part_id);
    asm volatile("" : "+v"(tid));
    asm volatile("" : "+s"(wave));
    asm volatile("" : "+s"(volume));
    asm volatile("" : "+s"(split));
    asm volatile("" : "+s"(part_of));
    if constexpr (!kMaxSplit) split = part_of = 0;
    const int lane = tid & 63;
    const int cols = kWgCols >> split, col_first = col0 + part_of * cols;  // columns of this workgroup
    // this thread's epilogue columns (the same for every row it stores): within the part, and of the layer
    const int lvec = (kWgCols == 64 ? 4 : (kWgCols == 32 ? 3 : 2)) - split;  // log2 of the part's 4-column vectors
    const int vec = tid & ((1 << lvec) - 1), ec4 = col_first + vec * 4;
    const __amdgpu_buffer_rsrc_t rs_in = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<T*>(in), 0, (int)((size_t)max_voxels * S::kRowBytes), kRawBuffer);
    const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(Wp), 0, (int)((size_t)volume * S::kWeightBytes), kRawBuffer);
    const bool first = idle;
    idle = false;
    if (tid < 16) s_pair[kMaxK * kTileRows + tid] = kNoPair;
    // zero this wave's partial tile (while the lists are on their way)
    int waves = kWaves, part_rows = kTileRows;
    if constexpr (kMaxSplit) {
        part_rows = rows;
        waves = split || rows * 8 <= S::kPartRows ? 8 : (rows * 7 <= S::kPartRows ? 7 : 6);
        static_assert(kWaves == 8 && S::kFewestWaves == 6, "waves");
    }
    float* part = s_part + wave * part_rows * cols;
    for (int t = lane; t < (wave < waves ? rows << lvec : 0); t += 64) reinterpret_cast<float4*>(part)[t] = make_float4(0.f, 0.f, 0.f, 0.f);
    float epi_scale = 1.f, epi_shift = 0.f, epi_col = 1.f;
    if (row0 == run_begin && tid < COUT) {
        if (has_scale) epi_scale = scale[tid];
        if (has_shift) epi_shift = shift[tid];
        if (S::kArith == kThirds) epi_col = reinterpret_cast<const float*>(static_cast<const char*>(Wp) + (size_t)volume * S::kWeightBytes)[tid];
    }
    auto compact = [&](auto halves) {
#pragma unroll
        for (int s = 0; s < kListsPerWave; ++s) {
            const int k = wave + s * kWaves;
            if (k >= volume) break;
            int base = 0;
#pragma unroll
            for (int h = 0; h < decltype(halves)::value; ++h) {
                const int v = h * 64 + lane < rows ? staged[s][h] : -1;
                const uint64_t m = __ballot(v >= 0);
                const int j = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, base));
                if (v >= 0) s_pair[k * kTileRows + j] = ((uint32_t)v << S::kRowBits) | (uint32_t)(h * 64 + lane);
                base += __popcll(m);
            }
            const int blocks = (base + 15) >> 4;
            if (base + lane < blocks * 16) s_pair[k * kTileRows + base + lane] = kNoPair;
            if (lane == 0) s_blk[k] = blocks;
        }
    };
    if (tall) compact(std::integral_constant<int, 2>{});
    else compact(std::integral_constant<int, 1>{});
    if (row0 == run_begin && tid < COUT) {
        s_epi[tid] = epi_scale;
        s_epi[COUT + tid] = epi_shift;
        s_epi[2 * COUT + tid] = epi_col;
    }
    __syncthreads();
    auto products = [&](auto& p) {
        if constexpr (kMaxSplit)
            if (split) multiply<S, COUT, kWgCols / 32>(rs_in, rs_w, s_pair, s_blk, volume, wave, waves, lane, col_first / 16, (rows + 15) >> 4, part, s_part + S::kPartRows * kWgCols, p);
        if (!kMaxSplit || !split) multiply<S, COUT, kWgCols / 16>(rs_in, rs_w, s_pair, s_blk, volume, wave, waves, lane, col_first / 16, (rows + 15) >> 4, part, s_part + S::kPartRows * kWgCols, p);
    };
    if (PAD && beside && first) {
        PadRows<TO, COUT> pads;
        pads.begin(out, n, max_voxels, blockIdx.x * kWaves + wave, (unsigned)(units * S::kColGroups) * kWaves);
        pads.layer(s_epi, has_scale, has_shift, relu);
        products(pads);
        pads.rest();
    } else {
        NoPadRows none;
        products(none);
    }
    __syncthreads();

    // fixed-order sum of the waves' partial tiles, epilogue, coalesced stores; the sums of kAtOnce vectors are read together
    constexpr int kAtOnce = 2;
    float e_scale[4], e_shift[4], e_col[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        e_scale[e] = s_epi[ec4 + e];
        e_shift[e] = s_epi[COUT + ec4 + e];
        e_col[e] = s_epi[2 * COUT + ec4 + e];
    }
    auto sums_of = [&](int r) {
        const float4* col = reinterpret_cast<const float4*>(s_part) + (r << lvec) + (vec ^ (r & ((1 << lvec) - 1)));
        float4 p4[kWaves];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) p4[w] = w < S::kFewestWaves || w < waves ? col[w * (part_rows << lvec)] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int m = kWaves; m > 1; m = (m + 1) / 2)  // (folded: fewer roundings follow each other)
#pragma unroll
            for (int w = 0; w < m / 2; ++w) {
                p4[w].x += p4[m - 1 - w].x;
                p4[w].y += p4[m - 1 - w].y;
                p4[w].z += p4[m - 1 - w].z;
                p4[w].w += p4[m - 1 - w].w;
            }
        return p4[0];
    };
    auto finite = [&](float (&o)[4]) {
        bool all = true;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o[e] *= e_col[e];
            all = all && (__float_as_uint(o[e]) & 0x7f800000u) != 0x7f800000u;
        }
        return all;
    };
    auto put = [&](int r, float (&o)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float s = o[e];
            if (has_scale) s = s * e_scale[e];
            if (has_shift) s = s + e_shift[e];
            if (relu) s = s > 0.f ? s : 0.f;
            o[e] = s;
        }
        store4(out + (size_t)(row0 + r) * COUT + ec4, o);
        if (DENSE && dt.dense) {  // the sparse2Dense scatter of this row, fused (uniform branch)
            const int4 cc = reinterpret_cast<const int4*>(dt.coors)[row0 + r];  // (b,z,y,x)
            if (cc.x != 0 || cc.y < 0 || cc.y >= dt.D || cc.z < 0 || cc.z >= dt.H || cc.w < 0 || cc.w >= dt.W) {
                if (dt.status && ec4 == 0) atomicOr(dt.status, SESSD_STATUS_BAD_COORD);
            } else {
                TO* d = static_cast<TO*>(dt.dense) + ((size_t)cc.y * dt.Hp + cc.z + dt.pad_top) * dt.Wp + cc.w + dt.pad_left;
                const size_t plane = (size_t)dt.D * dt.Hp * dt.Wp;  // channel stride
#pragma unroll
                for (int e = 0; e < 4; ++e) d[(size_t)(ec4 + e) * plane] = (TO)o[e];
            }
        }
    };
    bool again = false;
    for (int v0 = tid; v0 < rows << lvec; v0 += kAtOnce * kThreads) {
        float4 sums[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int r = (v0 + u * kThreads) >> lvec;
            sums[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (r >= rows) break;
            sums[u] = sums_of(r);
        }
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int r = (v0 + u * kThreads) >> lvec;
            if (r >= rows) break;
            float o[4] = {sums[u].x, sums[u].y, sums[u].z, sums[u].w};
            if constexpr (S::kArith == kThirds) again |= !finite(o);
            put(r, o);
        }
    }
    // Parts of an infinity, of a row that is not all in its parts, or a sum beyond the range on the way: the products themselves, by the
    // thread that has stored the row before.  (A loop of its own: inside the one above frames took 0.5 % longer.)
    if constexpr (S::kArith == kThirds) {
        if (__any(again))
            for (int v = tid; v < rows << lvec; v += kThreads) {
                const int r = v >> lvec;
                const float4 sum = sums_of(r);
                float o[4] = {sum.x, sum.y, sum.z, sum.w};
                if (finite(o)) continue;
                const float* w = w_f32;
                asm volatile("" : "+s"(w));  // (or its offsets are computed, and it is waited for, at the kernel's head)
                direct_sum<CIN, COUT>(in, w, nbr + row0 + r, max_voxels, volume, ec4, o);
                put(r, o);
            }
    }
    __syncthreads();  // the next piece reuses the lists and partial tiles
    }
    }
    if (PAD && n < max_voxels && (idle || !beside)) {
        if (idle) {  // (no tile has staged scale and shift)
            if (thread < COUT) {
                s_epi[thread] = has_scale ? scale[thread] : 1.f;
                s_epi[COUT + thread] = has_shift ? shift[thread] : 0.f;
            }
            __syncthreads();
        }
        write_pad_rows<TO, COUT>(out, n, max_voxels, blockIdx.x * kThreads + thread, (unsigned)(units * S::kColGroups) * kThreads, s_epi, has_scale,
                                 has_shift, relu);
    }
}

template <int CIN, int COUT, typename T = float, typename TO = T>
int launch(const GemmArgs& a, hipStream_t stream) {
    // operands are addressed with 32-bit byte offsets, 2^31 means "out of range"
    if (!gemm_wide_takes_rows(a.max_voxels, CIN, COUT, a.in_type) || (size_t)a.K * Shape<T, CIN, COUT>::kWeightBytes >= kOutOfRange)
        return SESSD_E_UNSUPPORTED;
    using S = Shape<T, CIN, COUT>;
    const int units = gemm_compute_units() * S::kPerUnit / S::kColGroups;
    const unsigned units_and_flags = (unsigned)units | (a.scale ? kHasScale : 0) | (a.shift ? kHasShift : 0) | (a.relu ? kRelu : 0);
    auto go = [&](auto dense, auto pad) {
        hipLaunchKernelGGL((conv_wide<CIN, COUT, T, TO, decltype(dense)::value, decltype(pad)::value>), dim3((unsigned)(units * S::kColGroups)),
                           dim3(S::kThreads), 0, stream, a.num_out, a.tiles, a.nbr, a.w_packed, static_cast<const T*>(a.in_feat),
                           a.max_voxels, a.K, units_and_flags, static_cast<TO*>(a.out_feat), a.w_f32, a.scale, a.shift, a.dense);
    };
    if (a.dense.dense) a.write_pad_rows ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
    else a.write_pad_rows ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
    SESSD_HIP_TRY(hipGetLastError());
    return SESSD_OK;
}

}  // namespace

bool gemm_runs_wide(int K, int cin, int cout, int in_type, int out_type) {
    if (K > kMaxK) return false;
    if (cin == 4) return in_type == SESSD_FLOAT && (cout == 16 || cout == 32);  // (the first layer of an FP16 pipeline as well)
    if (in_type != out_type) return false;
    const int shapes[][2] = {{16, 16}, {16, 32}, {32, 32}, {32, 64}, {64, 64}, {64, 128}, {128, 128}};
    for (auto& s : shapes)
        if (s[0] == cin && s[1] == cout) return true;
    return false;
}

// (a kernel that has a shape to itself takes more; the pipeline asks before it relies on the fused scatter)
bool gemm_wide_takes_rows(int max_voxels, int cin, int cout, int in_type) {
    return (uint32_t)max_voxels <= kNoPair >> pair_row_bits(gemm_wide_tile_rows(cin, cout, in_type)) &&
           (size_t)max_voxels * cin * (in_type == SESSD_HALF ? 2 : 4) < kOutOfRange;
}

int gemm_wide_tile_rows(int cin, int cout, int type) {
    if (cout >= 64) return Shape<float, 64, 64>::kWholeRows;
    if (type == SESSD_HALF) return Shape<__half, 16, 16>::kTileRows;
    if (cout == 16) return Shape<float, 16, 16>::kTileRows;
    return cin == 32 ? Shape<float, 32, 32>::kTileRows : Shape<float, 16, 32>::kTileRows;
}

bool wide_splits(int cin) { return arith(cin) != kPlain; }
size_t wide_weight_bytes(int K, int cin, int cout) { return (size_t)K * cin * cout * 6 + cout * sizeof(float); }

// W in parts and in operand order: Wp[k][64 channels][part][step][16-column block][lane][8], element j of lane l being channel
// 32 step + 16 (j / 4) + 4 (l / 16) + j % 4 (the channels that the lane permutation of the rows brings there), column
// 16 block + l % 16; behind them a factor for each column.  Three parts hold a number from 2^-110 up.  A column with smaller
// ones is multiplied by a power of two (its largest to 2^30), and divided by it where the sums are; what is too small even then
// becomes NaN, and the column's sums are made plainly.
void pack_wide_weights(const float* w, int K, int cin, int cout, void* dst) {
    std::vector<float> up(cout, 1.f), big(cout, 0.f), small(cout, 1.f);  // (the columns' largest finite and smallest magnitudes)
    for (size_t t = 0; t < (size_t)K * cin; ++t)
        for (int col = 0; col < cout; ++col) {
            const float v = std::fabs(w[t * cout + col]), finite = v <= 3.402823466e38f ? v : 0.f, some = v > 0.f ? v : 1.f;
            big[col] = finite > big[col] ? finite : big[col];
            small[col] = some < small[col] ? some : small[col];
        }
    float* down = reinterpret_cast<float*>(static_cast<char*>(dst) + (size_t)K * cin * cout * 6);
    for (int col = 0; col < cout; ++col) {
        int e = 0;
        if (small[col] < std::ldexp(1.f, -110)) e = std::min(std::max(30 - std::ilogb(big[col]), 0), 126);
        up[col] = std::ldexp(1.f, e);
        down[col] = std::ldexp(1.f, -e);
    }
    const int cp = cin > 64 ? 64 : cin, steps = cp / 32, blocks = cout / 16;
    uint16_t* o = static_cast<uint16_t*>(dst);
    const size_t part_size = (size_t)steps * blocks * 512;
    auto nearest = [](uint32_t u) { return (u + 0x7fffu + ((u >> 16) & 1u)) & 0xffff0000u; };  // BF16 in the upper half
    std::vector<uint32_t> parts(3 * (size_t)cout);
    uint32_t *p0 = parts.data(), *p1 = p0 + cout, *p2 = p1 + cout;
    for (int k = 0; k < K; ++k)
        for (int ch = 0; ch < cin; ++ch, w += cout) {
            // (without branches: the weights of a backbone are 500 000 and more)
            for (int col = 0; col < cout; ++col) {
                float v = w[col] * up[col], part;
                uint32_t u, rest;
                std::memcpy(&u, &v, 4);
                const uint32_t mag = u & 0x7fffffffu;
                const uint32_t first = mag < 0x7f7f8000u ? nearest(u) : u & 0xffff0000u;  // (rounded, the largest would be infinite)
                std::memcpy(&part, &first, 4);
                v -= part;
                std::memcpy(&u, &v, 4);
                p1[col] = nearest(u);
                std::memcpy(&part, &p1[col], 4);
                v -= part;
                std::memcpy(&rest, &v, 4);
                p2[col] = rest;
                p0[col] = mag >= 0x7f800000u || (rest & 0xffffu) ? 0x7fc00000u : first;
            }
            const int in_part = ch % cp, in_step = in_part % 32;
            const int first_lane = in_step % 16 / 4 * 16, j = in_step / 16 * 4 + in_step % 4;
            uint16_t* at = o + (size_t)(k * (cin / cp) + ch / cp) * 3 * part_size + (size_t)(in_part / 32) * blocks * 512 + first_lane * 8 + j;
            for (int col = 0; col < cout; ++col) {
                uint16_t* to = at + (size_t)(col / 16) * 512 + col % 16 * 8;
                to[0] = (uint16_t)(p0[col] >> 16);
                to[part_size] = (uint16_t)(p1[col] >> 16);
                to[2 * part_size] = (uint16_t)(p2[col] >> 16);
            }
        }
}

int launch_wide(const GemmArgs& a, hipStream_t stream) {
    if (!a.w_packed || !gemm_runs_wide(a.K, a.cin, a.cout, a.in_type, a.out_type)) return SESSD_E_UNSUPPORTED;
    if ((reinterpret_cast<uintptr_t>(a.in_feat) | reinterpret_cast<uintptr_t>(a.out_feat)) & 15) return SESSD_E_UNSUPPORTED;
    if (a.cin == 4 && a.out_type == SESSD_HALF) return a.cout == 16 ? launch<4, 16, float, __half>(a, stream) : launch<4, 32, float, __half>(a, stream);
    if (a.cin == 4) return a.cout == 16 ? launch<4, 16>(a, stream) : launch<4, 32>(a, stream);
#define SESSD_CASE(CI, CO) \
    if (a.cin == CI && a.cout == CO) return a.in_type == SESSD_HALF ? launch<CI, CO, __half>(a, stream) : launch<CI, CO>(a, stream)
    SESSD_CASE(16, 16);
    SESSD_CASE(16, 32);
    SESSD_CASE(32, 32);
    SESSD_CASE(32, 64);
    SESSD_CASE(64, 64);
    SESSD_CASE(64, 128);
    SESSD_CASE(128, 128);
#undef SESSD_CASE
    return SESSD_E_UNSUPPORTED;
}

}  // namespace sessd
