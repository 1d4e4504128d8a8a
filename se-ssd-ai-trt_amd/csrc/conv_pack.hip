// conv_pack.hip -- which layer shapes the matrix-core kernels take, and their weights in operand order.
#include "kernels.h"

namespace sessd {

namespace {

bool mfma_shape(int K, int cin, int cout) {
    if (K > kGemmMaxOffsets) return false;
    if (cin == 4) return cout == 16 || cout == 32;  // FP32 operands whatever the pipeline's feature dtype
    const int shapes[][2] = {{16, 16}, {16, 32}, {32, 32}, {32, 64}, {64, 64}, {64, 128}, {128, 128}};
    for (auto& s : shapes)
        if (s[0] == cin && s[1] == cout) return true;
    return false;
}

// channels per MFMA step and elements per lane
void chunk_shape(int dtype, int cin, int* channels, int* lane_elems) {
    if (cin == 4) {
        *channels = 4;
        *lane_elems = 1;
    } else if (dtype == SESSD_FLOAT || cin == 16) {
        *channels = 16;
        *lane_elems = 4;
    } else {
        *channels = 32;
        *lane_elems = 8;
    }
}

}  // namespace

int gemm_compute_units() {
    static int cu = 0;
    if (cu == 0) {
        int dev = 0, v = 0;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
            cu = v;
        else
            cu = 256;
    }
    return cu;
}

bool gemm_runs_on_mfma(int K, int cin, int cout, int in_type, int out_type) {
    if (!mfma_shape(K, cin, cout)) return false;
    return in_type == out_type || (cin == 4 && in_type == SESSD_FLOAT && out_type == SESSD_HALF);
}

size_t packed_weight_bytes(int K, int cin, int cout, int dtype) {
    if (!mfma_shape(K, cin, cout)) return 0;
    if (dtype == SESSD_FLOAT && wide_splits(cin)) return wide_weight_bytes(K, cin, cout);
    return (size_t)K * cin * cout * (dtype == SESSD_HALF && cin != 4 ? sizeof(__half) : sizeof(float));
}

// Operand order: Wp[k][g][nb][lane][e] = W[k][C*g + E*(lane/16) + e][16nb + lane%16] with C channels per
// K-chunk and E elements per lane (FP32: 16/4, FP16: 32/8, FP16 with Cin = 16: 16/4, Cin = 4: 4/1).  Cin = 4
// always takes FP32 operands (the voxel means are FP32); in an FP16 pipeline its weights are the
// half-rounded values, as in every other layer of that pipeline.  FP32 from Cin 32 up: pack_wide_weights().
void pack_weights(const float* w, int K, int cin, int cout, int dtype, void* dst) {
    if (dtype == SESSD_FLOAT && wide_splits(cin)) return pack_wide_weights(w, K, cin, cout, dst);
    int C, E;
    chunk_shape(dtype, cin, &C, &E);
    const int G = cin / C, NB = cout / 16;
    for (int k = 0; k < K; ++k)
        for (int g = 0; g < G; ++g)
            for (int nb = 0; nb < NB; ++nb)
                for (int lane = 0; lane < 64; ++lane)
                    for (int e = 0; e < E; ++e) {
                        const size_t o = ((((size_t)k * G + g) * NB + nb) * 64 + lane) * E + e;
                        const float v = w[((size_t)k * cin + C * g + E * (lane / 16) + e) * cout + 16 * nb + lane % 16];
                        float near = v;
                        const uint16_t h = dtype == SESSD_HALF ? nearest_half(v, &near) : (uint16_t)0;
                        if (dtype == SESSD_HALF && cin != 4) static_cast<uint16_t*>(dst)[o] = h;
                        else static_cast<float*>(dst)[o] = near;
                    }
}

}  // namespace sessd
