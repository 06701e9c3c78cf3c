// Occupancy-grid maintenance (reference src/utils/occupancy-grid-kernels.cu,
// src/utils/bit-utils.*, src/core/trainer.cu:221-311) and the analytic
// Gaussian-blob field used for synthetic scenes.
#pragma clang fp contract(off)

#include "common.hpp"

namespace tn {

// density *= factor for every cascade (reference :16-34); float4 streaming
__global__ void occ_decay_kernel(uint64_t n, float factor, float* __restrict__ density) {
    const uint64_t i = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i + 3 < n) {
        float4 v = *reinterpret_cast<float4*>(density + i);
        v.x *= factor;
        v.y *= factor;
        v.z *= factor;
        v.w *= factor;
        *reinterpret_cast<float4*>(density + i) = v;
    } else {
        for (uint64_t j = i; j < n; ++j) density[j] *= factor;
    }
}

// jittered point in cell idx of `level` (three uniforms u), normalised by the
// training box, not clamped (reference :38-76, occupancy-grid.cuh:167-182)
TN_DEVICE void cell_point(uint32_t idx, int res, int level, float inv_aabb, const float u[3], float p[3]) {
    const float inv_res = 1.0f / (float)res;
    const int half_res = res / 2;
    const float level_size = (float)(1 << level);
    const float voxel = level_size * inv_res;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const int ic = (int)compact_bits10(idx >> c);
        const float v = (float)(ic - half_res) * voxel;
        const float x = v + u[c] * voxel;
        p[c] = (x * inv_aabb) + 0.5f;
    }
}

__global__ void occ_sample_points_kernel(uint32_t n_cells, uint32_t B, uint32_t start_idx, int res, int level,
                                         float inv_aabb, const float* __restrict__ random, float* __restrict__ pos) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_cells) return;
    const float u[3] = {random[i], random[i + B], random[i + 2 * B]};
    float p[3];
    cell_point(i + start_idx, res, level, inv_aabb, u, p);
    pos[i] = p[0];
    pos[i + B] = p[1];
    pos[i + 2 * B] = p[2];
}

// elements g .. g + 3 of the uniform stream keyed by (k0, k1): one block of it
// when g is a multiple of four, else two
TN_DEVICE void uniform4(uint64_t g, uint32_t k0, uint32_t k1, float u[4]) {
    const uint64_t block = g >> 2;
    uint32_t c[8] = {(uint32_t)block, (uint32_t)(block >> 32), 0u, 0u, 0u, 0u, 0u, 0u};
    philox4x32_10(c, k0, k1);
    const uint32_t m = (uint32_t)g & 3u;
    if (m != 0u) {
        c[4] = (uint32_t)(block + 1);
        c[5] = (uint32_t)((block + 1) >> 32);
        philox4x32_10(c + 4, k0, k1);
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        u[k] = u32_to_unit(m == 0u ? c[k] : m == 1u ? c[k + 1] : m == 2u ? c[k + 2] : c[k + 3 < 8 ? k + 3 : 7]);
}

// The two passes of a grid refresh around the network, drawing their uniforms
// themselves: cell i takes elements i, B + i, 2B + i (its point) and 3B + i (the
// subset rule) of the stream from `offset` on. Four cells per thread share the
// generator's blocks of four; each launch is as long as a launch is (5 us for
// 262,144 cells, their bytes take 1). A fill of 4B uniforms that both passes
// read was a third such launch per chunk: a refresh of three cascades of 128^3
// cells took 1.97 ms with it and 1.92 without.
__global__ void occ_draw_points_kernel(uint32_t n_cells, uint32_t B, uint32_t start_idx, int res, int level,
                                       float inv_aabb, uint32_t k0, uint32_t k1, uint64_t offset,
                                       float* __restrict__ pos) {
    const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= n_cells) return;
    float u[3][4], p[3][4];
#pragma unroll
    for (int c = 0; c < 3; ++c) uniform4(offset + (uint64_t)c * B + i, k0, k1, u[c]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float uk[3] = {u[0][k], u[1][k], u[2][k]};
        float q[3];
        cell_point(i + k + start_idx, res, level, inv_aabb, uk, q);
#pragma unroll
        for (int c = 0; c < 3; ++c) p[c][k] = q[c];
    }
    if ((B & 3u) == 0u && i + 4 <= n_cells) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
            *reinterpret_cast<float4*>(pos + (uint64_t)c * B + i) = make_float4(p[c][0], p[c][1], p[c][2], p[c][3]);
    } else {
        for (uint32_t k = 0; k < 4 && i + k < n_cells; ++k)
            for (int c = 0; c < 3; ++c) pos[(uint64_t)c * B + i + k] = p[c][k];
    }
}

// the reference's random subset rule once training is past warm-up (:79-115)
TN_DEVICE bool cell_sampled(float r, uint8_t bits, int level) {
    if (r > 0.5f) return false;
    return r < 0.25f || ((bits >> level) & 1u) != 0u;
}

// sigma_cell = max(sigma_cell, exp(min(s,12)-1)) (reference :79-115)
TN_DEVICE float updated_density(float raw, float density) { return fmaxf(__expf(fminf(raw, 12.0f) - 1.0f), density); }

template <typename TIn>
__global__ void occ_update_density_kernel(uint32_t n_cells, uint32_t start_idx, uint32_t volume, int level,
                                          int sample_all, const float* __restrict__ random,
                                          const TIn* __restrict__ raw, const uint8_t* __restrict__ bits,
                                          float* __restrict__ density) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_cells) return;
    const uint32_t idx = i + start_idx;
    if (!sample_all && !cell_sampled(random[i], bits[idx], level)) return;
    float* p = density + (uint64_t)level * volume + idx;
    *p = updated_density((float)raw[i], *p);
}

template <typename TIn>
__global__ void occ_draw_update_kernel(uint32_t n_cells, uint32_t B, uint32_t start_idx, uint32_t volume, int level,
                                       int sample_all, uint32_t k0, uint32_t k1, uint64_t offset,
                                       const TIn* __restrict__ raw, const uint8_t* __restrict__ bits,
                                       float* __restrict__ density) {
    const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= n_cells) return;
    float u[4];
    if (!sample_all) uniform4(offset + 3 * (uint64_t)B + i, k0, k1, u);
    const uint32_t idx = i + start_idx;
    float* const p = density + (uint64_t)level * volume + idx;
    const bool whole = i + 4 <= n_cells;
    if (sample_all && whole && ((start_idx | volume) & 3u) == 0u) {
        float4 v = *reinterpret_cast<const float4*>(p);
        v.x = updated_density((float)raw[i], v.x);
        v.y = updated_density((float)raw[i + 1], v.y);
        v.z = updated_density((float)raw[i + 2], v.z);
        v.w = updated_density((float)raw[i + 3], v.w);
        *reinterpret_cast<float4*>(p) = v;
        return;
    }
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (i + k < n_cells && (sample_all || cell_sampled(u[k], bits[idx + k], level)))
            p[k] = updated_density((float)raw[i + k], p[k]);
}

// byte = sum_k [density_k > threshold] << k (reference :118-141); one thread
// per 4 cells so the byte stores are one 32-bit store
__global__ void occ_bits_kernel(uint32_t volume, int n_levels, float thr, const float* __restrict__ density,
                                uint8_t* __restrict__ bits) {
    const uint32_t i4 = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i4 >= volume) return;
    if (i4 + 3 < volume) {
        uint32_t packed = 0;
        for (int l = 0; l < n_levels; ++l) {
            const float4 d = *reinterpret_cast<const float4*>(density + (uint64_t)l * volume + i4);
            packed |= (uint32_t)(d.x > thr) << l;
            packed |= (uint32_t)(d.y > thr) << (l + 8);
            packed |= (uint32_t)(d.z > thr) << (l + 16);
            packed |= (uint32_t)(d.w > thr) << (l + 24);
        }
        *reinterpret_cast<uint32_t*>(bits + i4) = packed;
    } else {
        for (uint32_t i = i4; i < volume; ++i) {
            uint8_t b = 0;
            for (int l = 0; l < n_levels; ++l) b |= (uint8_t)((density[(uint64_t)l * volume + i] > thr) << l);
            bits[i] = b;
        }
    }
}

// population count of a byte array into out[0] (u64 via 32-bit atomics on
// two words is avoided: one workgroup per chunk writes a partial, a second
// launch sums the partials)
constexpr int kPopThreads = 256;
__global__ void popcount_partial_kernel(uint64_t n, const uint8_t* __restrict__ bytes, uint32_t* __restrict__ part) {
    __shared__ uint32_t sm[kPopThreads / 64];
    const uint64_t base = (uint64_t)blockIdx.x * kPopThreads * 16;
    uint32_t c = 0;
    for (int k = 0; k < 4; ++k) {
        const uint64_t i = base + ((uint64_t)k * kPopThreads + threadIdx.x) * 4;
        if (i + 3 < n) c += __popc(*reinterpret_cast<const uint32_t*>(bytes + i));
        else
            for (uint64_t j = i; j < n; ++j) c += __popc((uint32_t)bytes[j]);
    }
    for (int d = 32; d >= 1; d >>= 1) c += __shfl_down(c, d, 64);
    if (__lane_id() == 0) sm[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = sm[0] + sm[1] + sm[2] + sm[3];
}

__global__ void popcount_final_kernel(uint32_t n_part, const uint32_t* __restrict__ part, uint32_t* __restrict__ out) {
    __shared__ uint32_t sm[16];
    uint32_t c = 0;
    for (uint32_t i = threadIdx.x; i < n_part; i += blockDim.x) c += part[i];
    for (int d = 32; d >= 1; d >>= 1) c += __shfl_down(c, d, 64);
    if (__lane_id() == 0) sm[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t t = 0;
        for (uint32_t k = 0; k < blockDim.x / 64; ++k) t += sm[k];
        out[0] = t;
    }
}

// ---------------------------------------------------------------------------
// analytic blob field: blob k = {cx, cy, cz, s, p, r, g, b} (world units)
// ---------------------------------------------------------------------------
constexpr int kMaxBlobs = 256;

TN_DEVICE void blob_field(const float* __restrict__ bl, uint32_t nb, float x, float y, float z, float& sigma,
                          float& r, float& g, float& b) {
    float s = 0.0f, sr = 0.0f, sg = 0.0f, sb = 0.0f;
    for (uint32_t k = 0; k < nb; ++k) {
        const float* q = bl + 8 * k;
        const float dx = x - q[0], dy = y - q[1], dz = z - q[2];
        const float d2 = dx * dx + dy * dy + dz * dz;
        const float rho = q[4] * __expf(-d2 / (2.0f * q[3] * q[3]));
        s += rho;
        sr += rho * q[5];
        sg += rho * q[6];
        sb += rho * q[7];
    }
    sigma = s;
    const float inv = s > 0.0f ? 1.0f / s : 0.0f;
    r = sr * inv;
    g = sg * inv;
    b = sb * inv;
}

// density of the blob field at every cell centre of every cascade
__global__ void blob_density_grid_kernel(uint32_t volume, int n_levels, int res, const float* __restrict__ blobs,
                                         uint32_t nb, float* __restrict__ density) {
    __shared__ float sb[kMaxBlobs * 8];
    for (uint32_t k = threadIdx.x; k < nb * 8; k += blockDim.x) sb[k] = blobs[k];
    __syncthreads();
    const uint64_t gi = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= (uint64_t)volume * n_levels) return;
    const int level = (int)(gi / volume);
    const uint32_t idx = (uint32_t)(gi % volume);
    const float cell = (float)(1 << level) / (float)res;
    const float x = ((float)(int)compact_bits10(idx >> 0) - (float)(res / 2) + 0.5f) * cell;
    const float y = ((float)(int)compact_bits10(idx >> 1) - (float)(res / 2) + 0.5f) * cell;
    const float z = ((float)(int)compact_bits10(idx >> 2) - (float)(res / 2) + 0.5f) * cell;
    float sigma, r, g, b;
    blob_field(sb, nb, x, y, z, sigma, r, g, b);
    density[gi] = sigma;
}

// sigma and rgb of the blob field at sample positions given in normalised
// [0,1] box coordinates (world = (p - 0.5) * aabb)
__global__ void blob_eval_kernel(const uint32_t* __restrict__ info, uint32_t n_max, uint32_t B, float aabb,
                                 const float* __restrict__ blobs, uint32_t nb, const float* __restrict__ pos,
                                 float* __restrict__ sigma, float* __restrict__ rgb) {
    __shared__ float sb[kMaxBlobs * 8];
    for (uint32_t k = threadIdx.x; k < nb * 8; k += blockDim.x) sb[k] = blobs[k];
    __syncthreads();
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n = info ? min(info[1], n_max) : n_max;
    if (i >= n) return;
    const float x = (pos[i] - 0.5f) * aabb, y = (pos[i + B] - 0.5f) * aabb, z = (pos[i + 2 * B] - 0.5f) * aabb;
    float s, r, g, b;
    blob_field(sb, nb, x, y, z, s, r, g, b);
    sigma[i] = s;
    rgb[i] = r;
    rgb[i + B] = g;
    rgb[i + 2 * B] = b;
}

}  // namespace tn

using namespace tn;

extern "C" int tn_occ_decay(tn_occupancy_grid_t grid, float factor, hipStream_t stream) {
    TN_CHECK_ARG(grid.density && grid.n_levels >= 1 && grid.resolution >= 2);
    const uint64_t n = (uint64_t)grid.n_levels * grid.resolution * grid.resolution * grid.resolution;
    occ_decay_kernel<<<blocks_for((n + 3) / 4, 256), 256, 0, stream>>>(n, factor, grid.density);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_occ_sample_points(uint32_t n_cells, uint32_t stride, uint32_t start_idx, tn_occupancy_grid_t grid,
                                    int level, float inv_aabb, const float* random, float* pos, hipStream_t stream) {
    TN_CHECK_ARG(random && pos && n_cells <= stride && level >= 0 && level < grid.n_levels);
    const uint32_t volume = (uint32_t)(grid.resolution * grid.resolution * grid.resolution);
    TN_CHECK_ARG((uint64_t)start_idx + n_cells <= volume);
    if (n_cells == 0) return TN_OK;
    occ_sample_points_kernel<<<blocks_for(n_cells, 256), 256, 0, stream>>>(n_cells, stride, start_idx, grid.resolution,
                                                                           level, inv_aabb, random, pos);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

// As tn_occ_sample_points with `random` the 4 stride uniforms of tn_fill_uniform at (seed, offset)
extern "C" int tn_occ_draw_points(uint32_t n_cells, uint32_t stride, uint32_t start_idx, tn_occupancy_grid_t grid,
                                  int level, float inv_aabb, uint64_t seed, uint64_t offset, float* pos,
                                  hipStream_t stream) {
    TN_CHECK_ARG(pos && n_cells <= stride && level >= 0 && level < grid.n_levels);
    TN_CHECK_ARG((reinterpret_cast<uintptr_t>(pos) & 15) == 0);
    const uint32_t volume = (uint32_t)(grid.resolution * grid.resolution * grid.resolution);
    TN_CHECK_ARG((uint64_t)start_idx + n_cells <= volume);
    if (n_cells == 0) return TN_OK;
    occ_draw_points_kernel<<<blocks_for(((uint64_t)n_cells + 3) / 4, 256), 256, 0, stream>>>(
        n_cells, stride, start_idx, grid.resolution, level, inv_aabb, (uint32_t)seed, (uint32_t)(seed >> 32), offset,
        pos);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

// As tn_occ_update_density with `random` the last `stride` of those uniforms
extern "C" int tn_occ_draw_update(int raw_dtype, uint32_t n_cells, uint32_t stride, uint32_t start_idx,
                                  tn_occupancy_grid_t grid, int level, int sample_all_cells, uint64_t seed,
                                  uint64_t offset, const void* raw_density, hipStream_t stream) {
    TN_CHECK_ARG(raw_density && grid.density && grid.bitfield && level >= 0 && level < grid.n_levels);
    TN_CHECK_ARG(n_cells <= stride && (reinterpret_cast<uintptr_t>(grid.density) & 15) == 0);
    const uint32_t volume = (uint32_t)(grid.resolution * grid.resolution * grid.resolution);
    TN_CHECK_ARG((uint64_t)start_idx + n_cells <= volume);
    if (raw_dtype != 0 && raw_dtype != 1) return TN_ERR_INVALID_ARGUMENT;
    if (n_cells == 0) return TN_OK;
    const unsigned blocks = blocks_for(((uint64_t)n_cells + 3) / 4, 256);
    const uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
    if (raw_dtype == 0)
        occ_draw_update_kernel<float><<<blocks, 256, 0, stream>>>(
            n_cells, stride, start_idx, volume, level, sample_all_cells, k0, k1, offset,
            static_cast<const float*>(raw_density), grid.bitfield, grid.density);
    else
        occ_draw_update_kernel<_Float16><<<blocks, 256, 0, stream>>>(
            n_cells, stride, start_idx, volume, level, sample_all_cells, k0, k1, offset,
            static_cast<const _Float16*>(raw_density), grid.bitfield, grid.density);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

// raw_dtype: 0 = fp32 network output, 1 = fp16
extern "C" int tn_occ_update_density(int raw_dtype, uint32_t n_cells, uint32_t start_idx, tn_occupancy_grid_t grid,
                                     int level, int sample_all_cells, const float* random, const void* raw_density,
                                     hipStream_t stream) {
    TN_CHECK_ARG(random && raw_density && grid.density && grid.bitfield && level >= 0 && level < grid.n_levels);
    const uint32_t volume = (uint32_t)(grid.resolution * grid.resolution * grid.resolution);
    TN_CHECK_ARG((uint64_t)start_idx + n_cells <= volume);
    if (n_cells == 0) return TN_OK;
    if (raw_dtype == 0)
        occ_update_density_kernel<float><<<blocks_for(n_cells, 256), 256, 0, stream>>>(
            n_cells, start_idx, volume, level, sample_all_cells, random, static_cast<const float*>(raw_density),
            grid.bitfield, grid.density);
    else if (raw_dtype == 1)
        occ_update_density_kernel<_Float16><<<blocks_for(n_cells, 256), 256, 0, stream>>>(
            n_cells, start_idx, volume, level, sample_all_cells, random, static_cast<const _Float16*>(raw_density),
            grid.bitfield, grid.density);
    else
        return TN_ERR_INVALID_ARGUMENT;
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_occ_update_bits(tn_occupancy_grid_t grid, float threshold, hipStream_t stream) {
    TN_CHECK_ARG(grid.density && grid.bitfield && grid.n_levels >= 1 && grid.n_levels <= 8);
    const uint32_t volume = (uint32_t)(grid.resolution * grid.resolution * grid.resolution);
    occ_bits_kernel<<<blocks_for((volume + 3) / 4, 256), 256, 0, stream>>>(volume, grid.n_levels, threshold,
                                                                            grid.density, grid.bitfield);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" size_t tn_popcount_workspace_bytes(uint64_t n_bytes) {
    return (size_t)blocks_for(n_bytes, kPopThreads * 16) * sizeof(uint32_t);
}

// number of set bits in n_bytes bytes -> *out (device u32)
extern "C" int tn_popcount(const uint8_t* bytes, uint64_t n_bytes, uint32_t* out, void* workspace,
                           size_t workspace_bytes, hipStream_t stream) {
    TN_CHECK_ARG(bytes && out && workspace && n_bytes > 0);
    if (workspace_bytes < tn_popcount_workspace_bytes(n_bytes)) return TN_ERR_OUT_OF_MEMORY;
    const unsigned nb = blocks_for(n_bytes, kPopThreads * 16);
    popcount_partial_kernel<<<nb, kPopThreads, 0, stream>>>(n_bytes, bytes, static_cast<uint32_t*>(workspace));
    popcount_final_kernel<<<1, 1024, 0, stream>>>(nb, static_cast<uint32_t*>(workspace), out);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_blob_density_grid(tn_occupancy_grid_t grid, const float* blobs, uint32_t n_blobs,
                                    hipStream_t stream) {
    TN_CHECK_ARG(grid.density && blobs && n_blobs >= 1 && n_blobs <= kMaxBlobs);
    const uint32_t volume = (uint32_t)(grid.resolution * grid.resolution * grid.resolution);
    const uint64_t n = (uint64_t)volume * grid.n_levels;
    blob_density_grid_kernel<<<blocks_for(n, 256), 256, 0, stream>>>(volume, grid.n_levels, grid.resolution, blobs,
                                                                      n_blobs, grid.density);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_blob_eval(const uint32_t* info, uint32_t n_max, uint32_t stride, float aabb, const float* blobs,
                            uint32_t n_blobs, const float* pos, float* sigma, float* rgb, hipStream_t stream) {
    TN_CHECK_ARG(blobs && pos && sigma && rgb && n_blobs >= 1 && n_blobs <= kMaxBlobs && n_max <= stride);
    if (n_max == 0) return TN_OK;
    blob_eval_kernel<<<blocks_for(n_max, 256), 256, 0, stream>>>(info, n_max, stride, aabb, blobs, n_blobs, pos,
                                                                  sigma, rgb);
    TN_CHECK_LAUNCH();
    return TN_OK;
}
