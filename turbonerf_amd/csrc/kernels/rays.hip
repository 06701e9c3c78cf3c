// Training-ray generation: seeded uniforms and camera rays clipped to the
// training box (reference src/utils/training-batch-kernels.cuh:82-187,
// src/models/camera.cuh:94-141, src/core/trainer.cu:45-62).
#pragma clang fp contract(off)

#include "camera.hpp"
#include "common.hpp"

namespace tn {

// out[j] = uniform element (offset + j) of the stream keyed by seed.
// One thread produces four consecutive elements from one Philox block.
__global__ void uniform_kernel(uint64_t n, uint32_t k0, uint32_t k1, uint64_t offset, float* __restrict__ out) {
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t first_block = offset >> 2;
    const uint64_t block = first_block + tid;
    uint32_t c[4] = {(uint32_t)block, (uint32_t)(block >> 32), 0u, 0u};
    philox4x32_10(c, k0, k1);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint64_t g = block * 4 + w;
        if (g < offset) continue;
        const uint64_t j = g - offset;
        if (j < n) out[j] = u32_to_unit(c[w]);
    }
}

// The same stream at an offset read on the device (each replay of a captured
// call draws at the offset that the one before left); the grid covers any alignment.
__global__ void uniform_dev_kernel(uint64_t n, uint32_t k0, uint32_t k1, const unsigned long long* __restrict__ d_off,
                                   float* __restrict__ out) {
    const uint64_t offset = *d_off;
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t block = (offset >> 2) + tid;
    if (block > (offset + n - 1) >> 2) return;
    uint32_t c[4] = {(uint32_t)block, (uint32_t)(block >> 32), 0u, 0u};
    philox4x32_10(c, k0, k1);
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint64_t g = block * 4 + w;
        if (g < offset) continue;
        const uint64_t j = g - offset;
        if (j < n) out[j] = u32_to_unit(c[w]);
    }
}

__global__ void counter_add_kernel(unsigned long long* __restrict__ c, unsigned long long inc) { *c += inc; }

// where a training ray's data go (SoA, stride B)
struct RayOut {
    float* __restrict__ pix_rgba;
    uint32_t* __restrict__ ray_img_id;
    float* __restrict__ ori;
    float* __restrict__ dir;
    float* __restrict__ ray_t;
    float* __restrict__ ray_tmax;
    uint8_t* __restrict__ ray_alive;
};

// Ray i of n_rays through the pixel that the uniform `u` picks; returns the
// pixel's alpha and leaves the ray alive only if it meets the box.
TN_DEVICE float training_ray(uint32_t i, uint32_t n_rays, float u, uint32_t B, uint32_t n_images, uint32_t n_pix,
                             int32_t img_w, float n_rays_per_image, const tn_bbox_t* __restrict__ bbox,
                             const tn_camera_t* __restrict__ cams, const uint8_t* __restrict__ images,
                             const RayOut& o) {
    // rays are split evenly over the images (reference trainer.cu:60); a
    // non-positive n_rays_per_image asks for that split of the device count
    const float nrpi = n_rays_per_image > 0.0f ? n_rays_per_image : (float)n_rays / (float)n_images;

    uint32_t image_idx = (uint32_t)((float)i / nrpi);
    if (image_idx >= n_images) image_idx = n_images - 1;
    const float p = (float)n_pix * u;
    const float w = (float)img_w;
    const float x = fmodf(p, w);
    const float y = p / w;  // not floored, as in the reference (its quirk Q5)

    const tn_camera_t cam = cams[image_idx];
    float ox, oy, oz, dx, dy, dz;
    camera_ray(cam, x, y, ox, oy, oz, dx, dy, dz);
    const float idx = 1.0f / dx, idy = 1.0f / dy, idz = 1.0f / dz;
    float tmin, tmax;
    const tn_bbox_t bb = *bbox;
    // a ray that misses the box has no samples; its target is cleared so the
    // reported loss does not pick up a pixel left over from an earlier batch
    // (the reference leaves the stale value in place; gradients are the same)
    bool hit = bbox_intersect(bb, ox, oy, oz, idx, idy, idz, tmin, tmax);
    const float t_max = fminf(cam.far_plane - cam.near_plane, tmax);
    const float t = fmaxf(0.0f, tmin + 1e-5f);
    hit = hit && !(t_max < t);
    if (!hit) {
        o.ray_alive[i] = 0;
        o.pix_rgba[i] = 0.0f;
        o.pix_rgba[i + B] = 0.0f;
        o.pix_rgba[i + 2 * B] = 0.0f;
        o.pix_rgba[i + 3 * B] = 0.0f;
        return 0.0f;
    }
    const uint64_t lp = min((uint64_t)p, (uint64_t)n_pix - 1);
    const uchar4 px = reinterpret_cast<const uchar4*>(images)[(uint64_t)n_pix * image_idx + lp];
    o.pix_rgba[i] = (float)px.x / 255.0f;
    o.pix_rgba[i + B] = (float)px.y / 255.0f;
    o.pix_rgba[i + 2 * B] = (float)px.z / 255.0f;
    o.pix_rgba[i + 3 * B] = (float)px.w / 255.0f;
    o.ori[i] = ox;
    o.ori[i + B] = oy;
    o.ori[i + 2 * B] = oz;
    o.dir[i] = dx;
    o.dir[i + B] = dy;
    o.dir[i + 2 * B] = dz;
    o.ray_t[i] = t;
    o.ray_tmax[i] = t_max;
    o.ray_alive[i] = 1;
    o.ray_img_id[i] = image_idx;
    return (float)px.w / 255.0f;
}

__global__ void init_training_rays_kernel(uint32_t n_rays_max, const uint32_t* __restrict__ d_n_rays,
                                          uint32_t B, uint32_t n_images, uint32_t n_pix, int32_t img_w,
                                          float n_rays_per_image, const tn_bbox_t* __restrict__ bbox,
                                          const tn_camera_t* __restrict__ cams,
                                          const uint8_t* __restrict__ images, const float* __restrict__ random,
                                          RayOut o) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n_rays = d_n_rays ? min(*d_n_rays, n_rays_max) : n_rays_max;
    if (i >= n_rays) return;
    training_ray(i, n_rays, random[i], B, n_images, n_pix, img_w, n_rays_per_image, bbox, cams, images, o);
}

// element `offset` of the uniform stream keyed by (k0, k1)
TN_DEVICE float uniform_at(uint64_t offset, uint32_t k0, uint32_t k1) {
    const uint64_t block = offset >> 2;
    uint32_t c[4] = {(uint32_t)block, (uint32_t)(block >> 32), 0u, 0u};
    philox4x32_10(c, k0, k1);
    const uint32_t w = (uint32_t)offset & 3u;
    return u32_to_unit(w == 0 ? c[0] : w == 1 ? c[1] : w == 2 ? c[2] : c[3]);
}

// A training batch's rays in one launch: ray i draws its four uniforms
// (elements i, B + i, 2B + i and 3B + i of the stream at *d_off: the pixel and
// the background colour), is formed, and is dropped by the alpha rule below.
// Only the uniforms of the rays in use are drawn; filling the whole capacity
// wrote 4 MB beside the network kernels (21 us there) for some 3,000 rays, and
// the fill, the counter, the rays and the rule were four launches.
__global__ void training_rays_kernel(uint32_t n_rays_max, const uint32_t* __restrict__ d_n_rays, uint32_t B,
                                     uint32_t n_images, uint32_t n_pix, int32_t img_w,
                                     const tn_bbox_t* __restrict__ bbox, const tn_camera_t* __restrict__ cams,
                                     const uint8_t* __restrict__ images, uint32_t k0, uint32_t k1,
                                     const unsigned long long* __restrict__ d_off, float alpha_threshold,
                                     float selection_probability, float* __restrict__ random, RayOut o) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n_rays = min(*d_n_rays, n_rays_max);
    if (i >= n_rays) return;
    const uint64_t off = *d_off;
    float u[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        u[k] = uniform_at(off + i + (uint64_t)k * B, k0, k1);
        random[i + (uint64_t)k * B] = u[k];
    }
    const float alpha = training_ray(i, n_rays, u[0], B, n_images, n_pix, img_w, -1.0f, bbox, cams, images, o);
    if (alpha_threshold < 1.0f && selection_probability < 1.0f && alpha < alpha_threshold && u[1] > selection_probability)
        o.ray_alive[i] = 0;
}

// Rays below the alpha threshold are kept only with the given probability
// (reference training-batch-kernels.cuh:189-208).
__global__ void deactivate_rays_kernel(uint32_t n_rays_max, const uint32_t* __restrict__ d_n_rays, uint32_t B,
                                       float alpha_threshold, float selection_probability,
                                       const float* __restrict__ pix_rgba, const float* __restrict__ random,
                                       uint8_t* __restrict__ ray_alive) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n_rays = d_n_rays ? min(*d_n_rays, n_rays_max) : n_rays_max;
    if (i >= n_rays) return;
    if (pix_rgba[3 * B + i] < alpha_threshold && random[i] > selection_probability) ray_alive[i] = 0;
}

}  // namespace tn

using namespace tn;

extern "C" int tn_fill_uniform(uint64_t n, uint64_t seed, uint64_t offset, float* out, hipStream_t stream) {
    TN_CHECK_ARG(out != nullptr);
    if (n == 0) return TN_OK;
    const uint64_t first_block = offset >> 2;
    const uint64_t last_block = (offset + n - 1) >> 2;
    const uint64_t n_threads = last_block - first_block + 1;
    uniform_kernel<<<blocks_for(n_threads, 256), 256, 0, stream>>>(n, (uint32_t)seed, (uint32_t)(seed >> 32),
                                                                   offset, out);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_fill_uniform_dev(uint64_t n, uint64_t seed, unsigned long long* d_offset, float* out,
                                   hipStream_t stream) {
    TN_CHECK_ARG(out != nullptr && d_offset != nullptr);
    if (n == 0) return TN_OK;
    uniform_dev_kernel<<<blocks_for(n / 4 + 2, 256), 256, 0, stream>>>(n, (uint32_t)seed, (uint32_t)(seed >> 32),
                                                                      d_offset, out);
    counter_add_kernel<<<1, 1, 0, stream>>>(d_offset, (unsigned long long)n);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_init_training_rays(uint32_t n_rays_max, const uint32_t* d_n_rays, uint32_t stride,
                                     uint32_t n_images, uint32_t n_pixels_per_image, int32_t img_w,
                                     int32_t img_h, float n_rays_per_image, const tn_bbox_t* bbox,
                                     const tn_camera_t* cameras, const uint8_t* images, const float* random,
                                     float* pix_rgba, uint32_t* ray_img_id, float* ori, float* dir,
                                     float* ray_t, float* ray_tmax, uint8_t* ray_alive, hipStream_t stream) {
    TN_CHECK_ARG(bbox && cameras && images && random && pix_rgba && ray_img_id && ori && dir && ray_t &&
                 ray_tmax && ray_alive);
    TN_CHECK_ARG(n_rays_max <= stride && n_images > 0 && img_w > 0 && img_h > 0);
    TN_CHECK_ARG(n_pixels_per_image == (uint32_t)img_w * (uint32_t)img_h);
    if (n_rays_max == 0) return TN_OK;
    init_training_rays_kernel<<<blocks_for(n_rays_max, 256), 256, 0, stream>>>(
        n_rays_max, d_n_rays, stride, n_images, n_pixels_per_image, img_w, n_rays_per_image, bbox, cameras,
        images, random, RayOut{pix_rgba, ray_img_id, ori, dir, ray_t, ray_tmax, ray_alive});
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_training_rays(uint32_t n_rays_max, const uint32_t* d_n_rays, uint32_t stride, uint32_t n_images,
                                uint32_t n_pixels_per_image, int32_t img_w, int32_t img_h, const tn_bbox_t* bbox,
                                const tn_camera_t* cameras, const uint8_t* images, uint64_t seed,
                                const unsigned long long* d_offset, float alpha_threshold,
                                float selection_probability, float* random, float* pix_rgba, uint32_t* ray_img_id,
                                float* ori, float* dir, float* ray_t, float* ray_tmax, uint8_t* ray_alive,
                                hipStream_t stream) {
    TN_CHECK_ARG(bbox && cameras && images && random && pix_rgba && ray_img_id && ori && dir && ray_t &&
                 ray_tmax && ray_alive && d_n_rays && d_offset);
    TN_CHECK_ARG(n_rays_max <= stride && n_images > 0 && img_w > 0 && img_h > 0);
    TN_CHECK_ARG(n_pixels_per_image == (uint32_t)img_w * (uint32_t)img_h);
    if (n_rays_max == 0) return TN_OK;
    training_rays_kernel<<<blocks_for(n_rays_max, 256), 256, 0, stream>>>(
        n_rays_max, d_n_rays, stride, n_images, n_pixels_per_image, img_w, bbox, cameras, images, (uint32_t)seed,
        (uint32_t)(seed >> 32), d_offset, alpha_threshold, selection_probability, random,
        RayOut{pix_rgba, ray_img_id, ori, dir, ray_t, ray_tmax, ray_alive});
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_deactivate_rays(uint32_t n_rays_max, const uint32_t* d_n_rays, uint32_t stride,
                                  float alpha_threshold, float selection_probability, const float* pix_rgba,
                                  const float* random, uint8_t* ray_alive, hipStream_t stream) {
    TN_CHECK_ARG(pix_rgba && random && ray_alive && n_rays_max <= stride);
    if (n_rays_max == 0) return TN_OK;
    deactivate_rays_kernel<<<blocks_for(n_rays_max, 256), 256, 0, stream>>>(
        n_rays_max, d_n_rays, stride, alpha_threshold, selection_probability, pix_rgba, random, ray_alive);
    TN_CHECK_LAUNCH();
    return TN_OK;
}
