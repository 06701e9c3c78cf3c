// Occupancy-grid ray marching and compacted sample generation
// (reference src/utils/training-batch-kernels.cuh:212-481,
//  src/core/occupancy-grid.cuh:150-282, src/core/trainer.cu:102-216).
//
// The count and generate passes run the same DDA with contraction disabled,
// so the samples written by the generate pass are exactly the ones counted.
// The exclusive scan and the prefix selection run on the device and leave
// (n_rays, n_samples) in a device-side tn_batch_info, so a training step has
// no host round trip between marching and the network.
#pragma clang fp contract(off)

#include "common.hpp"

namespace tn {

// Level k of the grid spans 2^k box units, and a point's level (grid_level_at)
// is the first with 2^k / 2 > |coordinate| and 2^k inv_res > dt. That only adds
// k to exponents, so levels are held as the exponent field of a float,
// kLevel0 + k << 23, and what is scaled by 2^k or 2^-k follows from it by one
// integer addition.
constexpr uint32_t kExponent = 0xFF800000u;  // sign and exponent
constexpr int kLevel0 = 0x3E800000;          // 0.25: a coordinate in [0.5, 1) is level 1's

struct MarchGrid {
    const uint8_t* bits;
    int top;         // the highest level
    float res_f;
    float inv_res;
    float half_res;
    uint32_t lim;
    float level_scale;  // the cascade is chosen from dt * level_scale
    int dt_bias;        // bits of (dt * level_scale) - dt_bias: the level that dt asks for, rounded down to an exponent
    int res_bias;       // res_bias - level: bits of res 2^-k
    int cell_bias;      // cell_bias + level: bits of 2^k / res
};

TN_DEVICE MarchGrid make_grid(const tn_occupancy_grid_t& g) {
    MarchGrid m;
    m.bits = g.bitfield;
    m.top = kLevel0 + ((g.n_levels - 1) << 23);
    m.res_f = (float)g.resolution;
    m.inv_res = 1.0f / m.res_f;
    m.half_res = 0.5f * m.res_f;
    m.lim = (uint32_t)g.resolution - 1u;
    m.level_scale = g.level_dt_scale > 0.0f ? g.level_dt_scale : 1.0f;
    m.dt_bias = __float_as_int(m.inv_res) - (1 << 23) - kLevel0;
    m.res_bias = __float_as_int(m.res_f) + kLevel0;
    m.cell_bias = __float_as_int(m.inv_res) - kLevel0;
    return m;
}

// What a marching kernel is compiled for. SEVERAL cascades; POW2: the
// resolution is a power of two, so that (x 2^-k + 1/2) res is one fused
// multiply-add with the same rounding; DT: a step may be longer than a cell of
// level 0 and so decide the level (training in a large box; a render's steps
// are normalised by the scene size and never are).
template <bool SEVERAL_, bool POW2_, bool DT_>
struct GridForm {
    static constexpr bool SEVERAL = SEVERAL_, POW2 = POW2_, DT = DT_;
};
// fn with the form for a launch on `grid`
template <typename Fn>
inline void with_grid_form(const tn_occupancy_grid_t& grid, float dt_max, Fn fn) {
    const bool pow2 = (grid.resolution & (grid.resolution - 1)) == 0;
    const float level_scale = grid.level_dt_scale > 0.0f ? grid.level_dt_scale : 1.0f;
    if (grid.n_levels == 1) {
        if (pow2) fn(GridForm<false, true, false>{});
        else fn(GridForm<false, false, false>{});
    } else if (!pow2) {
        fn(GridForm<true, false, true>{});
    } else if (dt_max * level_scale < 1.0f / (float)grid.resolution) {
        fn(GridForm<true, true, false>{});
    } else {
        fn(GridForm<true, true, true>{});
    }
}

// Marching follows the reference's serial recurrence exactly (contraction
// off, same operation order): at a ray's t, an occupied cell gives a sample
// and t += dt(t), an empty one a skip by the distance to the next cell
// boundary, divided by dt_min rounding upwards and multiplied back (reference
// src/core/occupancy-grid.cuh:243-282). What bounds
// it is the length of that dependent chain, several hundred steps for a ray
// through a mostly empty box, so everything but the chain itself is taken off
// it:
//  * a group of G lanes shares a ray. It forms G steps of the recurrence on
//    the assumption that the cells on the way stay occupied (a run of
//    samples) or empty (a skip), lane j keeping the j-th t, and then tests the
//    G points side by side: one gather of occupancy bits for G steps. The
//    leading points that bear the assumption out are taken, and the group goes
//    on from the first that does not;
//  * a skip step needs three axes' distances to their next cell boundary. Lane
//    j of a group works on axis j % 4 (2 and 3 alike) and the minimum is taken
//    across the quad, which leaves about a third of the instructions;
//  * the step's division by dt_min, rounded upwards, is by a constant: its
//    reciprocal is formed once (div_up);
//  * the cascade of a point is formed from exponents, without a loop, and
//    where the resolution is a power of two or a step cannot decide the
//    cascade, the kernels are compiled without what that takes (GridForm);
//  * the groups of a wave that run and those that skip share a block's test,
//    whose loads do not wait for the tests against the box and the ray's end.
// A skip step is 20 vector instructions in one cascade and 28 or 34 in several;
// a test about 80 and one load. Few rays are bound by the latency of the
// chain and of that load, many rays by instruction issue: 65,000 rays through
// a 16-unit scene issued vector instructions in nine cycles of ten.
// A wave per ray that looked every skip step's cell up in turn took 214 us to
// count and 116 us to generate a batch of 4,369 rays through a unit box with
// 8 blobs, and 120 us to count 53 rays; this takes 49, 40 and 39 us. A render
// pass of 65,000 rays in the 16-unit scene takes 290 us to count (380 with 24
// and 36 instructions per skip step and a test for runs and skips each).
// G and T by the number of rays: see kGroup16Rays.
struct MarchStep {
    float cone, dt_lo, dt_max;  // steps of samples: t cone within [dt_lo, dt_max]
    float dt_min, inv_dt_min;   // skips: whole multiples of dt_min
};
// dt_lo is dt_min, but no more than dt_max, where every step is dt_max (get_dt)
TN_DEVICE MarchStep make_step(float cone, float dt_min, float dt_max) {
    return {cone, fminf(dt_min, dt_max), dt_max, dt_min, 1.0f / dt_min};
}

struct MarchRay {
    float ox, oy, oz, dx, dy, dz;
};

// a / b rounded towards +infinity for positive a and b = dt_min, given y =
// RN(1 / b): q0 = RN(a y) is within 2 ulp; one correction by its residual
// leaves a neighbour of a / b (or a / b itself), and the sign of that
// neighbour's residual, which one fused multiply-add gives exactly, tells
// whether it lies below (Boldo & Muller, "Exact and approximated error of the
// FMA", IEEE TC 2011).
TN_DEVICE float div_up(float a, float b, float y) {
    const float q0 = a * y;
    const float q = __builtin_fmaf(__builtin_fmaf(-q0, b, a), y, q0);
    const uint32_t below = __float_as_uint(__builtin_fmaf(q, b, -a)) >> 31;  // q b < a
    return __uint_as_float(__float_as_uint(q) + below);
}

// get_dt
TN_DEVICE float step_dt(const MarchStep& st, float t) {
    return __builtin_amdgcn_fmed3f(t * st.cone, st.dt_lo, st.dt_max);
}
TN_DEVICE uint32_t abs_bits(float v) { return __float_as_uint(v) & 0x7FFFFFFFu; }

// the level, as kLevel0 + k << 23, of a point whose largest |coordinate| has the bits m, at t
template <typename F>
TN_DEVICE int level_bits(const MarchGrid& g, const MarchStep& st, uint32_t m, float t) {
    int e = (int)m;
    if constexpr (F::DT) e = max(e, __float_as_int(step_dt(st, t) * g.level_scale) - g.dt_bias);
    // (as floats: these are powers of two, infinity or below level 0)
    return __float_as_int(__builtin_amdgcn_fmed3f(__int_as_float(e & (int)kExponent), __int_as_float(kLevel0),
                                                  __int_as_float(g.top)));
}

// (v 2^-k + 1/2) res, k the level of `level`
template <typename F>
TN_DEVICE float cell_coord(const MarchGrid& g, float v, int level) {
    if constexpr (F::POW2)
        return __builtin_fmaf(v, F::SEVERAL ? __int_as_float(g.res_bias - level) : g.res_f, g.half_res);
    if constexpr (F::SEVERAL) v *= __int_as_float(0x3F800000 + kLevel0 - level);
    return (v + 0.5f) * g.res_f;
}
// index of a cell coordinate: truncated, at least 0 (the conversion takes
// negative values and NaN to 0), at most the last
TN_DEVICE uint32_t cell_index(const MarchGrid& g, float c) {
    uint32_t i;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(i) : "v"(c));
    return min(i, g.lim);
}
// Every third bit of a word. The empty assembly keeps the compiler from
// merging the stages into more instructions and the last one into a multiply,
// which takes as long as four.
TN_DEVICE uint32_t spread_bits(uint32_t v) {
    v = (v | (v << 16)) & 0x030000FFu;
    asm("" : "+v"(v));
    v = (v | (v << 8)) & 0x0300F00Fu;
    asm("" : "+v"(v));
    v = (v | (v << 4)) & 0x030C30C3u;
    asm("" : "+v"(v));
    v = (v | (v << 2)) & 0x09249249u;
    asm("" : "+v"(v));
    return v;
}

// occupancy of the cell at (x, y, z)
template <typename F>
TN_DEVICE bool point_occupied(const MarchGrid& g, const MarchStep& st, float t, float x, float y, float z) {
    int level = kLevel0;
    if constexpr (F::SEVERAL) level = level_bits<F>(g, st, max(max(abs_bits(x), abs_bits(y)), abs_bits(z)), t);
    const uint32_t xu = spread_bits(cell_index(g, cell_coord<F>(g, x, level)));
    const uint32_t yu = spread_bits(cell_index(g, cell_coord<F>(g, y, level)));
    const uint32_t zu = spread_bits(cell_index(g, cell_coord<F>(g, z, level)));
    const uint32_t bits = g.bits[xu | (yu << 1) | (zu << 2)];
    return ((F::SEVERAL ? bits >> ((level - kLevel0) >> 23) : bits) & 1u) != 0u;
}

// The distance to the next cell boundary along one axis, gc the coordinate in
// cells, h = copysign(0.5, d), id = 1 / d, k the cell's side: in one cascade of
// a power-of-two resolution the side is a constant power of two below 1 and
// already in id, which rounds alike.
template <typename F>
TN_DEVICE float axis_distance(float gc, float h, float id, float k) {
    const float d = (floorf(h + gc + 0.5f) - gc) * id;
    return F::POW2 && !F::SEVERAL ? d : k * d;
}

// max(lo, minimum of v over the quad), a NaN (a ray along a cell face) left out
// as fminf and fmaxf do. In assembly because fminf of a lane-permuted value
// costs a move and a quieting max besides; the two wait states that a DPP read
// needs after a vector write are part of it.
TN_DEVICE float quad_min_above(float v, float lo) {
    float a, b;
    asm("s_nop 1\n\t"
        "v_min_f32_dpp %0, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_min_f32_dpp %1, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "v_max_f32 %1, %3, %1"
        : "=&v"(a), "=&v"(b)
        : "v"(v), "s"(lo));
    return b;
}
TN_DEVICE uint32_t quad_max(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));     // lanes 1 0 3 2
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));  // lanes 2 3 0 1
}

// the group's bits of `ballot`
template <int G>
TN_DEVICE uint32_t group_bits(uint64_t ballot) {
    const uint32_t lane = __lane_id();
    const uint32_t half = lane < 32u ? (uint32_t)ballot : (uint32_t)(ballot >> 32);
    return (half >> (lane & 31u & ~(uint32_t)(G - 1))) & ((1u << G) - 1u);
}
// v of the group's lane j
template <int G>
TN_DEVICE float group_get(float v, uint32_t j) {
    return __shfl(v, (int)((__lane_id() & ~(uint32_t)(G - 1)) + j), 64);
}

// One ray per group, all 64 / G of a wave at once, G steps per block of a skip
// and G T per block of a run. Emits through `emit(n, t)`
// (lane-wise: sample n of the lane's ray at t). COUNT: stops at t_max, at
// the box and at max_n samples; otherwise (the generate pass) takes max_n
// samples, and one outside the box, which the count pass cannot have counted,
// would be emitted without advancing. Each run of samples without a skip in
// between goes to `log` (its first t and sample, and the t after its last), in
// pieces of at most G T. Returns the ray's sample count.
struct NoLog {
    TN_DEVICE void run(bool, float, uint32_t, float) {}
};
template <int G, int T, typename F, bool COUNT, typename Emit, typename Log>
TN_DEVICE uint32_t march_group(bool active, const MarchRay& r, float t, float t_max, uint32_t max_n,
                               const tn_bbox_t& bbox, const MarchGrid& g, const MarchStep& st, Emit emit, Log& log) {
    constexpr uint32_t S = G * T;  // samples per block of a run
    const uint32_t lane = __lane_id(), j = lane & (uint32_t)(G - 1), axis = lane & 3u;
    const float oa = axis == 0 ? r.ox : axis == 1 ? r.oy : r.oz;
    const float da = axis == 0 ? r.dx : axis == 1 ? r.dy : r.dz;
    const float ha = 0.5f * copysignf(1.0f, da);
    float ida = 1.0f / da;
    if constexpr (F::POW2 && !F::SEVERAL) ida *= g.inv_res;  // see axis_distance
    uint32_t n = 0;
    bool done = !active, skip = false, open = false;  // open: the last block's run goes on
    for (;;) {
        const uint64_t runs = __builtin_amdgcn_ballot_w64(!done && !skip);
        const uint64_t skips = __builtin_amdgcn_ballot_w64(!done && skip);
        if ((runs | skips) == 0ull) break;
        float tj[T];  // of the lane's samples j, j + G, ... of the block
        float t_end = t;
#pragma unroll
        for (int q = 0; q < T; ++q) tj[q] = t;
        if (runs != 0ull) {
            // a run: the t's after so many more samples
            if (st.dt_lo == st.dt_max) {
#pragma unroll
                for (uint32_t k = 0; k < S; ++k) {
                    tj[k / G] = j >= k % G ? t_end : tj[k / G];
                    t_end += st.dt_max;
                }
            } else {
#pragma unroll
                for (uint32_t k = 0; k < S; ++k) {
                    tj[k / G] = j >= k % G ? t_end : tj[k / G];
                    t_end += step_dt(st, t_end);
                }
            }
        }
        if (skips != 0ull) {
            // a skip from an empty cell: lane j's t after j + 1 steps
            float tc = t, ts = t;
#pragma unroll
            for (uint32_t k = 0; k < (uint32_t)G; ++k) {
                const float p = oa + tc * da;
                int level = kLevel0;
                float cell = g.inv_res;
                if constexpr (F::SEVERAL) {
                    level = level_bits<F>(g, st, quad_max(abs_bits(p)), tc);
                    cell = __int_as_float(g.cell_bias + level);
                }
                const float gc = cell_coord<F>(g, p, level);
                const float d = quad_min_above(axis_distance<F>(gc, ha, ida, cell), st.dt_min);
                tc += div_up(d, st.dt_min, st.inv_dt_min) * st.dt_min;
                ts = j == k ? tc : ts;
            }
            tj[0] = skip ? ts : tj[0];
            t_end = skip ? tc : t_end;
        }
        // one test for both: f is the first step that ends the group's run or
        // skip. The cells are looked up for every lane (their indices are
        // clamped), so that a block's loads are in flight together.
        uint64_t stop = 0, in = 0;
        const uint32_t whole = skip ? (uint32_t)G : S;
        bool occ[T];
#pragma unroll
        for (int q = 0; q < T; ++q) {
            if (q > 0 && runs == 0ull) break;
            const float x = r.ox + tj[q] * r.dx, y = r.oy + tj[q] * r.dy, z = r.oz + tj[q] * r.dz;
            occ[q] = point_occupied<F>(g, st, tj[q], x, y, z);
            const bool within = !done && (skip || j + q * G < max_n - n) && (!COUNT || tj[q] < t_max) &&
                                bbox_contains(bbox, x, y, z);
            in |= (uint64_t)group_bits<G>(__builtin_amdgcn_ballot_w64(within)) << (q * G);
        }
#pragma unroll
        for (int q = 0; q < T; ++q) {
            if (q > 0 && runs == 0ull) break;
            stop |= (uint64_t)group_bits<G>(__builtin_amdgcn_ballot_w64(occ[q] == skip)) << (q * G);
        }
        stop |= ~in;  // a skip's bits from G on and a block's from S on are set
        if (skip) stop |= ~0ull << G;
        const uint32_t f = stop != 0ull ? min((uint32_t)__builtin_ctzll(stop), whole) : whole;
        const bool in_f = f < whole && ((in >> f) & 1ull) != 0ull;
        float t_f = t_end;
#pragma unroll
        for (int q = 0; q < T; ++q) {
            const float v = group_get<G>(tj[q], f & (uint32_t)(G - 1));
            t_f = f < whole && f / G == (uint32_t)q ? v : t_f;
        }
        if (!done) {
            if (!skip) {
#pragma unroll
                for (int q = 0; q < T; ++q)
                    if (j + q * G < f) emit(n + j + q * G, tj[q]);
                if (f != 0u) log.run(!open, t, n, t_f);
                open = f == S;
                n += f;
            }
            t = t_f;
            if (f < whole) {
                if (in_f) {
                    skip = !skip;
                } else {
                    if (!COUNT)
                        for (uint32_t k = n + j; k < max_n; k += (uint32_t)G) emit(k, t);
                    done = true;
                }
            }
        }
    }
    return n;
}

constexpr int kMarchWaves = 4;  // waves per workgroup
// The marching kernels are launched on at most TN_TUNE_MARCH_MAX_BLOCKS
// workgroups and stride over the live rays: the ray count lives on the device,
// and a grid sized for the largest batch would launch a wave per possible ray,
// nearly all of which exit at once yet occupy the dispatcher beside the
// network kernels.
inline unsigned march_blocks(uint32_t n_rays_max) {
    return std::min(blocks_for((uint64_t)n_rays_max * 16, 64 * kMarchWaves), (unsigned)tune_value(TN_TUNE_MARCH_MAX_BLOCKS));
}

// A group of 16 halves the tests per step and so a ray's latency, one of 8 the
// waves that a large pass needs; with few rays, a run goes on for 32 samples
// at a time, two tests per lane. Measured, count pass in us with groups of 16
// by two tests, of 16 and of 8 (unit box with 8 blobs; all of it occupied;
// 16-unit box with 5 cascades and 128 small blobs): 2,048 rays 39 / 40 / 60,
// 29 / 34 / 60 and 106 / 103 / 134, 8,192 rays 51 / 47 / 62, 33 / 38 / 60 and
// 113 / 106 / 134, 16,384 rays 52 / 45 / 43, 13 / 14 / 19 and 125 / 118 / 144,
// 32,768 rays 56 / 51 / 43, 20 / 20 / 20 and 155 / 147 / 146, 131,072 rays
// 121 / 111 / 70, 47 / 49 / 38 and 319 / 305 / 208. Groups of 16 by four tests
// gain 2 us of 29 where all is occupied and lose 4 to 6 elsewhere, groups of
// 8 by two lose above 16,384 rays; groups of 4, 32 and 64 and a ray per lane
// were slower at every size.
constexpr uint32_t kTwoBlockRays = 4096;
constexpr uint32_t kGroup16Rays = 24576;

TN_DEVICE MarchRay load_ray(bool active, uint32_t i, uint32_t B, const float* __restrict__ ori,
                            const float* __restrict__ dir) {
    return active ? MarchRay{ori[i], ori[i + B], ori[i + 2 * B], dir[i], dir[i + B], dir[i + 2 * B]}
                  : MarchRay{0.0f, 0.0f, 0.0f, 1.0f, 1.0f, 1.0f};
}

// What the count pass leaves of a ray for the generate pass (16 records of 8
// bytes, one 128-byte line per ray): record 0 the number of runs and the t
// after the last sample, records 1 to 15 each run's first t and sample. Within
// a run the t's follow from its first one alone, so the generate pass neither
// skips through empty cells nor looks up occupancy again. A ray of more runs
// (their number is still counted) is marched a second time.
constexpr uint32_t kRunRecords = 16;
struct RunLog {
    uint2* rec;  // the ray's records; null in all lanes but the group's first
    uint32_t n = 0;
    float t_end = 0.0f;
    TN_DEVICE void run(bool first, float t, uint32_t sample, float t_after) {
        if (first) {
            ++n;
            if (rec && n < kRunRecords) rec[n] = make_uint2(__float_as_uint(t), sample);
        }
        t_end = t_after;
    }
    TN_DEVICE void close() {
        if (rec) rec[0] = make_uint2(n, __float_as_uint(t_end));
    }
};

struct MarchCountArgs {
    uint32_t n_rays, B, max_steps;
    const float *dir, *tmax, *ori, *t;
    uint8_t* alive;
    uint32_t* n_steps;
    uint2* runs;  // null: none wanted
};

template <int G, int T, typename F>
TN_DEVICE void march_count_rays(const MarchCountArgs& a, const tn_bbox_t& bbox, const MarchGrid& g,
                                const MarchStep& st) {
    const uint32_t n_threads = gridDim.x * blockDim.x, tid = blockIdx.x * blockDim.x + threadIdx.x;
    // whole waves: every lane of a wave takes part in the group operations
    for (uint32_t w = tid & ~63u; w / G < a.n_rays; w += n_threads) {
        const uint32_t i = (w + (tid & 63u)) / G;
        const bool own = i < a.n_rays, first = (tid & (uint32_t)(G - 1)) == 0;
        const bool active = own && a.alive[i] != 0;
        const MarchRay r = load_ray(active, i, a.B, a.ori, a.dir);
        RunLog log{a.runs && active && first ? a.runs + (uint64_t)i * kRunRecords : nullptr};
        const uint32_t n = march_group<G, T, F, true>(active, r, active ? a.t[i] : 0.0f, active ? a.tmax[i] : 0.0f,
                                                    a.max_steps, bbox, g, st, [](uint32_t, float) {}, log);
        log.close();
        if (own && first) {
            if (active && n == 0) a.alive[i] = 0;
            a.n_steps[i] = n;
        }
    }
}

template <typename F>
__global__ void __launch_bounds__(64 * kMarchWaves)
march_count_kernel(uint32_t n_rays_max, const uint32_t* __restrict__ d_n_rays, uint32_t B, tn_bbox_t bbox,
                   tn_occupancy_grid_t grid, float cone, float dt_min, float dt_max, uint32_t max_steps,
                   const float* __restrict__ dir, const float* __restrict__ ray_tmax, uint8_t* __restrict__ ray_alive,
                   const float* __restrict__ ori, const float* __restrict__ ray_t, uint32_t* __restrict__ n_steps,
                   uint2* __restrict__ runs) {
    const uint32_t n_rays = d_n_rays ? min(*d_n_rays, n_rays_max) : n_rays_max;
    const MarchGrid g = make_grid(grid);
    const MarchStep st = make_step(cone, dt_min, dt_max);
    const MarchCountArgs a = {n_rays, B, max_steps, dir, ray_tmax, ori, ray_t, ray_alive, n_steps, runs};
    if (n_rays <= kTwoBlockRays) march_count_rays<16, 2, F>(a, bbox, g, st);
    else if (n_rays <= kGroup16Rays) march_count_rays<16, 1, F>(a, bbox, g, st);
    else march_count_rays<8, 1, F>(a, bbox, g, st);
}

// ---------------------------------------------------------------------------
// exclusive scan + prefix selection. Three launches: per-tile sums, a single
// workgroup scanning the tile sums (at most kScanTile tiles), and a per-tile
// scan that writes offsets and picks the last ray whose offset is below the
// sample budget.
// ---------------------------------------------------------------------------
constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr uint32_t kScanTile = kScanThreads * kScanItems;  // 4096 rays per tile

// inclusive scan of one value per thread across a 256-thread block
TN_DEVICE uint32_t block_inclusive_scan(uint32_t v, uint32_t* smem /*[kScanThreads/64]*/, uint32_t& total) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wid = threadIdx.x >> 6;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(v, d, 64);
        if (lane >= (uint32_t)d) v += o;
    }
    if (lane == 63) smem[wid] = v;
    __syncthreads();
    uint32_t pre = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) {
        const uint32_t s = smem[w];
        if ((uint32_t)w < wid) pre += s;
        total += s;
    }
    __syncthreads();
    return v + pre;
}

__global__ void scan_tile_sums_kernel(uint32_t n, const uint32_t* __restrict__ d_n, const uint32_t* __restrict__ vals,
                                      uint32_t* __restrict__ tile_sums) {
    __shared__ uint32_t smem[kScanThreads / 64];
    if (d_n) n = min(*d_n, n);
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t j = base + k;
        if (j < n) s += vals[j];
    }
    uint32_t total;
    block_inclusive_scan(s, smem, total);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

__global__ void scan_tile_prefix_kernel(uint32_t n_tiles, uint32_t* __restrict__ tile_sums) {
    __shared__ uint32_t smem[kScanThreads / 64];
    uint32_t carry = 0;
    for (uint32_t base = 0; base < n_tiles; base += kScanThreads) {
        const uint32_t j = base + threadIdx.x;
        const uint32_t v = j < n_tiles ? tile_sums[j] : 0u;
        uint32_t total;
        const uint32_t inc = block_inclusive_scan(v, smem, total);
        if (j < n_tiles) tile_sums[j] = carry + inc - v;  // exclusive
        carry += total;
    }
}

// info[0] = n_rays kept, info[1] = n_samples, info[2] = status, info[3] =
// rays scanned (the batch's generated ray count).
// mode 0 (training, the reference's rule): j = last ray whose offset is below
//   max_samples; rays [0, j) are kept and n_samples = offset[j].
// mode 1 (rendering): every ray whose samples end within max_samples is kept.
__global__ void scan_write_select_kernel(uint32_t n, const uint32_t* __restrict__ d_n,
                                         const uint32_t* __restrict__ vals,
                                         const uint32_t* __restrict__ tile_prefix, uint32_t max_samples, int mode,
                                         uint32_t* __restrict__ offsets, uint32_t* __restrict__ info) {
    __shared__ uint32_t smem[kScanThreads / 64];
    if (d_n) n = min(*d_n, n);
    if (blockIdx.x == 0 && threadIdx.x == 0) info[3] = n;
    const uint32_t base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t j = base + k;
        v[k] = j < n ? vals[j] : 0u;
        s += v[k];
    }
    uint32_t total;
    const uint32_t inc = block_inclusive_scan(s, smem, total);
    uint64_t run = (uint64_t)tile_prefix[blockIdx.x] + inc - s;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint32_t j = base + k;
        if (j < n) {
            const uint32_t off = (uint32_t)min(run, (uint64_t)0xFFFFFFFFu);
            offsets[j] = off;
            const uint64_t next = run + v[k];
            // offsets are non-decreasing, so exactly one ray is the last with
            // offset < max_samples; the reference keeps the rays before it.
            if (mode == 0) {
                const bool last_lt = off < max_samples && (j + 1 == n || next >= max_samples);
                if (last_lt) {
                    info[0] = j;
                    info[1] = off;
                    info[2] = j == 0 ? (uint32_t)TN_ERR_NO_RAYS : (off == 0 ? (uint32_t)TN_ERR_NO_SAMPLES : 0u);
                }
            } else {
                // ends are non-decreasing: the last ray ending within budget is unique
                const uint64_t after = (j + 1 < n) ? next + vals[j + 1] : ~0ull;
                const bool last_fit = next <= max_samples && (j + 1 == n || after > max_samples);
                if (last_fit) {
                    info[0] = j + 1;
                    info[1] = (uint32_t)next;
                    info[2] = next == 0 ? (uint32_t)TN_ERR_NO_SAMPLES : 0u;
                }
                if (j == 0 && v[k] > max_samples) {
                    info[0] = 0;
                    info[1] = 0;
                    info[2] = (uint32_t)TN_ERR_NO_RAYS;
                }
            }
            run = next;
        }
    }
}

struct MarchGenerateArgs {
    uint32_t n_rays, B;
    const float *ori, *dir, *t;
    const uint32_t *offset, *n_steps;
    const uint8_t* alive;
    uint32_t* out_ray;
    float* out_t;
};

template <int G, int T, typename F>
TN_DEVICE void march_generate_rays(const MarchGenerateArgs& a, const tn_bbox_t& bbox, const MarchGrid& g,
                                   const MarchStep& st) {
    const uint32_t n_threads = gridDim.x * blockDim.x, tid = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t w = tid & ~63u; w / G < a.n_rays; w += n_threads) {
        const uint32_t i = (w + (tid & 63u)) / G;
        const bool active = i < a.n_rays && a.alive[i] != 0;
        const MarchRay r = load_ray(active, i, a.B, a.ori, a.dir);
        const uint32_t off = active ? a.offset[i] : 0u;
        NoLog log;
        march_group<G, T, F, false>(active, r, active ? a.t[i] : 0.0f, INFINITY, active ? a.n_steps[i] : 0u, bbox, g, st,
                                  [&](uint32_t n, float t) {
                                      a.out_t[off + n] = t;
                                      a.out_ray[off + n] = i;
                                  },
                                  log);
    }
}

template <typename F>
__global__ void __launch_bounds__(64 * kMarchWaves)
march_generate_kernel(uint32_t n_rays_max, const uint32_t* __restrict__ info, uint32_t B, tn_bbox_t bbox,
                      tn_occupancy_grid_t grid, float dt_min, float dt_max, float cone, const float* __restrict__ ori,
                      const float* __restrict__ dir, const float* __restrict__ ray_t,
                      const uint32_t* __restrict__ ray_offset, const uint8_t* __restrict__ ray_alive,
                      const uint32_t* __restrict__ n_ray_steps, uint32_t* __restrict__ out_ray,
                      float* __restrict__ out_t) {
    const uint32_t n_rays = min(info[0], n_rays_max);
    const MarchGrid g = make_grid(grid);
    const MarchStep st = make_step(cone, dt_min, dt_max);
    const MarchGenerateArgs a = {n_rays, B, ori, dir, ray_t, ray_offset, n_ray_steps, ray_alive, out_ray, out_t};
    if (n_rays <= kTwoBlockRays) march_generate_rays<16, 2, F>(a, bbox, g, st);
    else if (n_rays <= kGroup16Rays) march_generate_rays<16, 1, F>(a, bbox, g, st);
    else march_generate_rays<8, 1, F>(a, bbox, g, st);
}

// Sample-parallel second half of generation: from each sample's t and ray
// (left in out_img_id by the marching pass) write the network inputs and the
// distortion loss's normalised midpoints and steps. The ray's span ends where
// its last sample's step ends, fl(t_last + dt(t_last)), which is where the
// marching pass's t stood after its last emission.
__global__ void march_expand_kernel(uint32_t n_rays_max, uint32_t SB_max, const uint32_t* __restrict__ info,
                                    uint32_t B, uint32_t SB, float inv_aabb, float dt_min, float dt_max, float cone,
                                    const uint32_t* __restrict__ ray_img_id, const float* __restrict__ ori,
                                    const float* __restrict__ dir, const float* __restrict__ ray_t,
                                    const uint32_t* __restrict__ ray_offset, const uint32_t* __restrict__ n_ray_steps,
                                    uint32_t* __restrict__ out_img_id, const float* __restrict__ out_t,
                                    float* __restrict__ out_pos, float* __restrict__ out_dir, float* __restrict__ out_dt,
                                    float* __restrict__ out_m_norm, float* __restrict__ out_dt_norm) {
    const uint32_t sid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t n_samples = min(info[1], SB_max);
    if (sid >= n_samples) return;
    const uint32_t r = out_img_id[sid];
    if (r >= n_rays_max) return;  // defensive: every sample below n_samples was written by the marching pass
    const float t = out_t[sid];
    const float dt = get_dt(t, cone, dt_min, dt_max);
    const float x = ori[r] + t * dir[r];
    const float y = ori[r + B] + t * dir[r + B];
    const float z = ori[r + 2 * B] + t * dir[r + 2 * B];
    const float t_min = ray_t[r];
    const float t_last = out_t[ray_offset[r] + n_ray_steps[r] - 1u];
    const float t_max = t_last + get_dt(t_last, cone, dt_min, dt_max);
    const float t_span = fmaxf(t_max - t_min, 1e-6f);
    out_img_id[sid] = ray_img_id[r];
    out_dt[sid] = inv_aabb * dt;
    out_pos[sid] = fminf(fmaxf(x * inv_aabb + 0.5f, 0.0f), 1.0f);
    out_pos[sid + SB] = fminf(fmaxf(y * inv_aabb + 0.5f, 0.0f), 1.0f);
    out_pos[sid + 2 * SB] = fminf(fmaxf(z * inv_aabb + 0.5f, 0.0f), 1.0f);
    out_dir[sid] = 0.5f * dir[r] + 0.5f;
    out_dir[sid + SB] = 0.5f * dir[r + B] + 0.5f;
    out_dir[sid + 2 * SB] = 0.5f * dir[r + 2 * B] + 0.5f;
    out_m_norm[sid] = fminf(fmaxf(((t + 0.5f * dt) - t_min) / t_span, 0.0f), 1.0f);
    out_dt_norm[sid] = dt / t_span;
}

// Where a sample's words go; the normalised steps, t and image ids may be null
// (a render reads none).
struct SampleOut {
    uint32_t* __restrict__ img_id;
    float *__restrict__ t, *__restrict__ pos, *__restrict__ dir, *__restrict__ dt, *__restrict__ m_norm,
        *__restrict__ dt_norm;
    uint32_t SB;
};

// Sample sid at t of a ray that starts at t_min and whose last sample's step
// ends at t_end (march_expand_kernel's expressions)
TN_DEVICE void write_sample(const SampleOut& o, uint32_t sid, float t, const MarchRay& r, float t_min, float t_end,
                            uint32_t img, float inv_aabb, const MarchStep& st) {
    if (sid >= o.SB) return;
    const float dt = step_dt(st, t);
    const float x = r.ox + t * r.dx, y = r.oy + t * r.dy, z = r.oz + t * r.dz;
    const float t_span = fmaxf(t_end - t_min, 1e-6f);
    if (o.img_id) o.img_id[sid] = img;
    if (o.t) o.t[sid] = t;
    o.dt[sid] = inv_aabb * dt;
    o.pos[sid] = fminf(fmaxf(x * inv_aabb + 0.5f, 0.0f), 1.0f);
    o.pos[sid + o.SB] = fminf(fmaxf(y * inv_aabb + 0.5f, 0.0f), 1.0f);
    o.pos[sid + 2 * (uint64_t)o.SB] = fminf(fmaxf(z * inv_aabb + 0.5f, 0.0f), 1.0f);
    o.dir[sid] = 0.5f * r.dx + 0.5f;
    o.dir[sid + o.SB] = 0.5f * r.dy + 0.5f;
    o.dir[sid + 2 * (uint64_t)o.SB] = 0.5f * r.dz + 0.5f;
    if (o.m_norm) o.m_norm[sid] = fminf(fmaxf(((t + 0.5f * dt) - t_min) / t_span, 0.0f), 1.0f);
    if (o.dt_norm) o.dt_norm[sid] = dt / t_span;
}

// The generate pass from the count pass's runs: 16 lanes per ray form 16 t's of
// a run at a time and write the samples' words at once, in rows of 16. Bound
// by the serial chain of 15 step sizes per 16 samples and the 36 or 52 bytes
// per sample; 8 lanes per ray would halve the rows, 64 quadruple the chain.
// Against marching again and expanding in a second launch, per pass: 23 us
// (was 36 + 4) for a training step of 1,900 rays, 24 (was 39 + 10) for 20,000
// rendered rays, 32 (was 39 + 25) for 130,000 rays and 4.2 M samples, 43 (was
// 168 + 14) in a scene of 16 units, where most steps are skips. The count
// pass's 128 bytes per ray cost it 1 to 2 us.
template <typename F>
TN_DEVICE void march_generate_from_runs(uint32_t n_rays, uint32_t B, const tn_bbox_t& bbox, const MarchGrid& g,
                                        const MarchStep& st, float inv_aabb, const float* __restrict__ ori,
                                        const float* __restrict__ dir, const float* __restrict__ ray_t,
                                        const uint32_t* __restrict__ ray_offset, const uint8_t* __restrict__ ray_alive,
                                        const uint32_t* __restrict__ n_ray_steps,
                                        const uint32_t* __restrict__ ray_img_id, const uint2* __restrict__ runs,
                                        const SampleOut& o) {
    constexpr int G = 16;
    const uint32_t n_threads = gridDim.x * blockDim.x, tid = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t j = tid & (uint32_t)(G - 1);
    for (uint32_t w = tid & ~63u; w / G < n_rays; w += n_threads) {
        const uint32_t i = (w + (tid & 63u)) / G;
        const bool active = i < n_rays && ray_alive[i] != 0;
        const MarchRay r = load_ray(active, i, B, ori, dir);
        const uint32_t off = active ? ray_offset[i] : 0u, ns = active ? n_ray_steps[i] : 0u;
        const uint32_t img = active && o.img_id ? ray_img_id[i] : 0u;
        const float t_min = active ? ray_t[i] : 0.0f;
        const uint2 rec = active ? runs[(uint64_t)i * kRunRecords + j] : make_uint2(0u, 0u);
        const float rec_t = __uint_as_float(rec.x), rec_n = __uint_as_float(rec.y);
        const uint32_t nr = __float_as_uint(group_get<G>(rec_t, 0));
        const float t_end = group_get<G>(rec_n, 0);
        const bool again = nr >= kRunRecords;  // more runs than records
        auto emit = [&](uint32_t n, float t) { write_sample(o, off + n, t, r, t_min, t_end, img, inv_aabb, st); };
        uint32_t q = 0, n = 0, n1 = 0;  // run, next sample, the run's end
        float t = 0.0f;
        bool done = !active || again;
        while (__ballot(!done) != 0ull) {
            // (all lanes: the group reads its records across lanes)
            const bool next = n == n1;
            const uint32_t q1 = next ? q + 1 : q;
            const float t_q = group_get<G>(rec_t, min(q1, (uint32_t)G - 1u));
            const uint32_t n_q = __float_as_uint(group_get<G>(rec_n, min(q1 + 1u, (uint32_t)G - 1u)));
            if (next) {
                q = q1;
                t = t_q;
                n1 = q < nr ? n_q : ns;
            }
            float tj = t;
            if (st.dt_lo == st.dt_max) {
#pragma unroll
                for (uint32_t k = 0; k + 1 < (uint32_t)G; ++k) tj = j > k ? tj + st.dt_max : tj;
            } else {
#pragma unroll
                for (uint32_t k = 0; k + 1 < (uint32_t)G; ++k) tj = j > k ? tj + step_dt(st, tj) : tj;
            }
            const uint32_t f = min((uint32_t)G, n1 - n);
            if (!done && j < f) emit(n + j, tj);
            const float t16 = group_get<G>(tj + step_dt(st, tj), (uint32_t)G - 1u);
            n += f;
            t = t16;  // used only when the run goes on past 16 samples
            done = done || n >= ns || (n == n1 && q >= nr);
        }
        if (__ballot(active && again) != 0ull) {
            NoLog log;
            march_group<G, 1, F, false>(active && again, r, t_min, INFINITY, ns, bbox, g, st, emit, log);
        }
    }
}

template <typename F>
__global__ void __launch_bounds__(64 * kMarchWaves)
march_generate_runs_kernel(uint32_t n_rays_max, const uint32_t* __restrict__ info, uint32_t B, tn_bbox_t bbox,
                           float inv_aabb, tn_occupancy_grid_t grid, float dt_min, float dt_max, float cone,
                           const uint32_t* __restrict__ ray_img_id, const float* __restrict__ ori,
                           const float* __restrict__ dir, const float* __restrict__ ray_t,
                           const uint32_t* __restrict__ ray_offset, const uint8_t* __restrict__ ray_alive,
                           const uint32_t* __restrict__ n_ray_steps, const uint2* __restrict__ runs, SampleOut o) {
    const uint32_t n_rays = min(info[0], n_rays_max);
    const MarchGrid g = make_grid(grid);
    const MarchStep st = make_step(cone, dt_min, dt_max);
    march_generate_from_runs<F>(n_rays, B, bbox, g, st, inv_aabb, ori, dir, ray_t, ray_offset, ray_alive, n_ray_steps,
                                ray_img_id, runs, o);
}

// Next step's ray count: the rays that would fill the sample budget at this
// step's samples-per-ray rate, with 1/8 headroom so the prefix selection
// usually has rays to spare (replaces the reference's host-side estimate,
// trainer.cu:133-140).
TN_DEVICE uint32_t estimate_rays(uint32_t n_rays, uint32_t n_samples, uint32_t max_samples, uint32_t cap,
                                 uint32_t min_rays) {
    uint32_t est = cap;
    if (n_samples > 0 && n_rays > 0) {
        const double per = (double)n_rays / (double)n_samples;
        const double e = per * (double)max_samples * 1.125 + 64.0;
        est = e >= (double)cap ? cap : (uint32_t)e;
    }
    if (est < min_rays) est = min_rays;
    if (est > cap) est = cap;
    return est;
}

__global__ void estimate_rays_kernel(const uint32_t* __restrict__ info, uint32_t max_samples, uint32_t cap,
                                     uint32_t min_rays, uint32_t* __restrict__ n_rays_next) {
    *n_rays_next = estimate_rays(info[0], info[1], max_samples, cap, min_rays);
}

// A training batch's selection in one launch of one workgroup: the exclusive
// scan of the rays' step counts, the reference's selection (mode 0 of
// scan_write_select_kernel), the next batch's ray count and the advance of the
// uniform stream. A batch has some thousands of rays, so a launch costs more
// than the scan: three scan launches, the estimate and the counter took 5 us
// each; more rays than one round of the workgroup (16,384) take 3 us more per
// round.
constexpr int kSelectThreads = 1024;
__global__ void __launch_bounds__(kSelectThreads)
batch_select_kernel(uint32_t n_max, const uint32_t* d_n, const uint32_t* __restrict__ vals, uint32_t max_samples,
                    uint32_t* __restrict__ offsets, uint32_t* __restrict__ info, uint32_t cap, uint32_t min_rays,
                    uint32_t* n_rays_next, unsigned long long* __restrict__ rng, unsigned long long rng_advance) {
    __shared__ uint32_t wsum[kSelectThreads / 64];
    __shared__ uint32_t kept[2];
    const uint32_t n = min(*d_n, n_max), lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    if (threadIdx.x < 2) kept[threadIdx.x] = 0u;
    uint64_t carry = 0;  // samples of the rounds before
    for (uint32_t base = 0; base < n; base += kSelectThreads * kScanItems) {
        const uint32_t j0 = base + threadIdx.x * kScanItems;
        uint32_t v[kScanItems], s = 0;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            v[k] = j0 + k < n ? vals[j0 + k] : 0u;
            s += v[k];
        }
        uint32_t inc = s;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(inc, d, 64);
            if (lane >= (uint32_t)d) inc += o;
        }
        __syncthreads();  // wsum is free, kept cleared
        if (lane == 63) wsum[wid] = inc;
        __syncthreads();
        uint64_t run = carry + inc - s;
        uint32_t total = 0;
#pragma unroll
        for (uint32_t w = 0; w < kSelectThreads / 64; ++w) {
            const uint32_t x = wsum[w];
            run += w < wid ? x : 0u;
            total += x;
        }
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            const uint32_t j = j0 + k;
            if (j >= n) break;
            const uint32_t off = (uint32_t)min(run, (uint64_t)0xFFFFFFFFu);
            offsets[j] = off;
            const uint64_t next = run + v[k];
            // exactly one ray is the last with offset < max_samples; the rays before it are kept
            if (off < max_samples && (j + 1 == n || next >= max_samples)) {
                kept[0] = j;
                kept[1] = off;
            }
            run = next;
        }
        carry += total;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t nr = kept[0], ns = kept[1];
        if (n > 0) {
            info[0] = nr;
            info[1] = ns;
            info[2] = nr == 0 ? (uint32_t)TN_ERR_NO_RAYS : (ns == 0 ? (uint32_t)TN_ERR_NO_SAMPLES : 0u);
        }
        info[3] = n;
        *n_rays_next = estimate_rays(info[0], info[1], max_samples, cap, min_rays);
        if (rng) *rng += rng_advance;
    }
}

__global__ void accumulate_samples_kernel(const uint32_t* __restrict__ info, unsigned long long* __restrict__ total) {
    total[0] += (unsigned long long)info[1];
}

__global__ void batch_tail_kernel(const uint32_t* __restrict__ info, uint32_t first, uint32_t* __restrict__ tail) {
    const uint32_t n = info[1];
    tail[0] = info[0];
    tail[1] = n > first ? n - first : 0u;
    tail[2] = info[2];
    tail[3] = info[3];
}

__global__ void batch_info_kernel(uint32_t n_rays, uint32_t n_samples, uint32_t* __restrict__ info) {
    info[0] = n_rays;
    info[1] = n_samples;
    info[2] = 0u;
    info[3] = n_rays;
}

}  // namespace tn

using namespace tn;

extern "C" int tn_batch_info(uint32_t n_rays, uint32_t n_samples, uint32_t* info, hipStream_t stream) {
    TN_CHECK_ARG(info);
    batch_info_kernel<<<1, 1, 0, stream>>>(n_rays, n_samples, info);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

// total[0] += info[1] on the device (running count of trained samples)
extern "C" int tn_accumulate_samples(const uint32_t* info, unsigned long long* total, hipStream_t stream) {
    TN_CHECK_ARG(info && total);
    accumulate_samples_kernel<<<1, 1, 0, stream>>>(info, total);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_batch_tail(const uint32_t* info, uint32_t first, uint32_t* tail_info, hipStream_t stream) {
    TN_CHECK_ARG(info && tail_info && info != tail_info);
    batch_tail_kernel<<<1, 1, 0, stream>>>(info, first, tail_info);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

static int march_count(uint32_t n_rays_max, const uint32_t* d_n_rays, uint32_t stride, tn_bbox_t bbox,
                       tn_occupancy_grid_t grid, float cone_angle, float dt_min, float dt_max, uint32_t max_steps,
                       const float* dir, const float* ray_tmax, uint8_t* ray_alive, const float* ori,
                       const float* ray_t, uint32_t* n_steps, void* runs, hipStream_t stream) {
    TN_CHECK_ARG(dir && ray_tmax && ray_alive && ori && ray_t && n_steps && grid.bitfield);
    TN_CHECK_ARG(n_rays_max <= stride && grid.n_levels >= 1 && grid.n_levels <= 8);
    TN_CHECK_ARG(grid.resolution >= 2 && grid.resolution <= 1024 && dt_min > 0.0f && dt_max >= dt_min);
    if (n_rays_max == 0) return TN_OK;
    with_grid_form(grid, dt_max, [&](auto form) {
        march_count_kernel<decltype(form)><<<march_blocks(n_rays_max), 64 * kMarchWaves, 0, stream>>>(
            n_rays_max, d_n_rays, stride, bbox, grid, cone_angle, dt_min, dt_max, max_steps, dir, ray_tmax,
            ray_alive, ori, ray_t, n_steps, static_cast<uint2*>(runs));
    });
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_march_count(uint32_t n_rays_max, const uint32_t* d_n_rays, uint32_t stride,
                              tn_bbox_t bbox, tn_occupancy_grid_t grid, float cone_angle, float dt_min,
                              float dt_max, uint32_t max_steps, const float* dir, const float* ray_tmax,
                              uint8_t* ray_alive, const float* ori, const float* ray_t, uint32_t* n_steps,
                              hipStream_t stream) {
    return march_count(n_rays_max, d_n_rays, stride, bbox, grid, cone_angle, dt_min, dt_max, max_steps, dir, ray_tmax,
                       ray_alive, ori, ray_t, n_steps, nullptr, stream);
}

extern "C" size_t tn_march_runs_bytes(uint32_t n_rays_max) { return (size_t)n_rays_max * kRunRecords * sizeof(uint2); }

extern "C" int tn_march_count_runs(uint32_t n_rays_max, const uint32_t* d_n_rays, uint32_t stride, tn_bbox_t bbox,
                                   tn_occupancy_grid_t grid, float cone_angle, float dt_min, float dt_max,
                                   uint32_t max_steps, const float* dir, const float* ray_tmax, uint8_t* ray_alive,
                                   const float* ori, const float* ray_t, uint32_t* n_steps, void* runs,
                                   size_t runs_bytes, hipStream_t stream) {
    TN_CHECK_ARG(runs && (reinterpret_cast<uintptr_t>(runs) & 127) == 0);
    if (runs_bytes < tn_march_runs_bytes(n_rays_max)) return TN_ERR_OUT_OF_MEMORY;
    return march_count(n_rays_max, d_n_rays, stride, bbox, grid, cone_angle, dt_min, dt_max, max_steps, dir, ray_tmax,
                       ray_alive, ori, ray_t, n_steps, runs, stream);
}

extern "C" size_t tn_scan_workspace_bytes(uint32_t n) {
    const uint32_t tiles = (n + kScanTile - 1) / kScanTile;
    return (size_t)(tiles == 0 ? 1 : tiles) * sizeof(uint32_t);
}

extern "C" int tn_scan_select(int mode, uint32_t n_rays, const uint32_t* d_n_rays, const uint32_t* n_steps,
                              uint32_t max_samples, uint32_t* ray_offset, uint32_t* info, void* workspace,
                              size_t workspace_bytes, hipStream_t stream) {
    TN_CHECK_ARG(mode == 0 || mode == 1);
    TN_CHECK_ARG(n_steps && ray_offset && info && workspace && n_rays > 0 && max_samples > 0);
    if (workspace_bytes < tn_scan_workspace_bytes(n_rays)) return TN_ERR_OUT_OF_MEMORY;
    const uint32_t tiles = (n_rays + kScanTile - 1) / kScanTile;
    uint32_t* tile_sums = static_cast<uint32_t*>(workspace);
    scan_tile_sums_kernel<<<tiles, kScanThreads, 0, stream>>>(n_rays, d_n_rays, n_steps, tile_sums);
    scan_tile_prefix_kernel<<<1, kScanThreads, 0, stream>>>(tiles, tile_sums);
    scan_write_select_kernel<<<tiles, kScanThreads, 0, stream>>>(n_rays, d_n_rays, n_steps, tile_sums, max_samples,
                                                                 mode, ray_offset, info);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_march_generate(uint32_t n_rays_max, const uint32_t* info, uint32_t stride,
                                 uint32_t sample_stride, tn_bbox_t bbox,
                                 float inv_aabb, tn_occupancy_grid_t grid, float dt_min, float dt_max,
                                 float cone_angle, const uint32_t* ray_img_id, const float* ori,
                                 const float* dir, const float* ray_t, const uint32_t* ray_offset,
                                 const uint8_t* ray_alive, const uint32_t* n_ray_steps, uint32_t* out_img_id,
                                 float* out_t, float* out_pos, float* out_dir, float* out_dt,
                                 float* out_m_norm, float* out_dt_norm, hipStream_t stream) {
    TN_CHECK_ARG(ray_img_id && ori && dir && ray_t && ray_offset && ray_alive && n_ray_steps && out_img_id &&
                 out_t && out_pos && out_dir && out_dt && out_m_norm && out_dt_norm && grid.bitfield);
    TN_CHECK_ARG(n_rays_max <= stride && grid.n_levels >= 1 && grid.n_levels <= 8 && dt_min > 0.0f);
    TN_CHECK_ARG(info != nullptr && sample_stride > 0);
    if (n_rays_max == 0) return TN_OK;
    with_grid_form(grid, dt_max, [&](auto form) {
        march_generate_kernel<decltype(form)><<<march_blocks(n_rays_max), 64 * kMarchWaves, 0, stream>>>(
            n_rays_max, info, stride, bbox, grid, dt_min, dt_max, cone_angle, ori, dir, ray_t, ray_offset, ray_alive,
            n_ray_steps, out_img_id, out_t);
    });
    march_expand_kernel<<<blocks_for(sample_stride, 256), 256, 0, stream>>>(
        n_rays_max, sample_stride, info, stride, sample_stride, inv_aabb, dt_min, dt_max, cone_angle, ray_img_id, ori,
        dir, ray_t, ray_offset, n_ray_steps, out_img_id, out_t, out_pos, out_dir, out_dt, out_m_norm, out_dt_norm);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_march_generate_runs(uint32_t n_rays_max, const uint32_t* info, uint32_t stride,
                                      uint32_t sample_stride, tn_bbox_t bbox, float inv_aabb,
                                      tn_occupancy_grid_t grid, float dt_min, float dt_max, float cone_angle,
                                      const uint32_t* ray_img_id, const float* ori, const float* dir,
                                      const float* ray_t, const uint32_t* ray_offset, const uint8_t* ray_alive,
                                      const uint32_t* n_ray_steps, const void* runs, size_t runs_bytes,
                                      uint32_t* out_img_id, float* out_t, float* out_pos, float* out_dir,
                                      float* out_dt, float* out_m_norm, float* out_dt_norm, hipStream_t stream) {
    TN_CHECK_ARG(ori && dir && ray_t && ray_offset && ray_alive && n_ray_steps && out_pos && out_dir && out_dt &&
                 grid.bitfield && (!out_img_id || ray_img_id));
    TN_CHECK_ARG(n_rays_max <= stride && grid.n_levels >= 1 && grid.n_levels <= 8 && dt_min > 0.0f && dt_max >= dt_min);
    TN_CHECK_ARG(info != nullptr && sample_stride > 0 && runs && (reinterpret_cast<uintptr_t>(runs) & 127) == 0);
    if (runs_bytes < tn_march_runs_bytes(n_rays_max)) return TN_ERR_OUT_OF_MEMORY;
    if (n_rays_max == 0) return TN_OK;
    with_grid_form(grid, dt_max, [&](auto form) {
        march_generate_runs_kernel<decltype(form)><<<march_blocks(n_rays_max), 64 * kMarchWaves, 0, stream>>>(
            n_rays_max, info, stride, bbox, inv_aabb, grid, dt_min, dt_max, cone_angle, ray_img_id, ori, dir, ray_t,
            ray_offset, ray_alive, n_ray_steps, static_cast<const uint2*>(runs),
            SampleOut{out_img_id, out_t, out_pos, out_dir, out_dt, out_m_norm, out_dt_norm, sample_stride});
    });
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_batch_select(uint32_t n_rays_max, const uint32_t* d_n_rays, const uint32_t* n_steps,
                               uint32_t max_samples, uint32_t* ray_offset, uint32_t* info, uint32_t cap,
                               uint32_t min_rays, uint32_t* n_rays_next, unsigned long long* d_offset,
                               uint64_t advance, hipStream_t stream) {
    TN_CHECK_ARG(d_n_rays && n_steps && ray_offset && info && n_rays_next && n_rays_max > 0 && max_samples > 0 && cap > 0);
    batch_select_kernel<<<1, kSelectThreads, 0, stream>>>(n_rays_max, d_n_rays, n_steps, max_samples, ray_offset, info,
                                                          cap, min_rays, n_rays_next, d_offset,
                                                          (unsigned long long)advance);
    TN_CHECK_LAUNCH();
    return TN_OK;
}

extern "C" int tn_estimate_rays(const uint32_t* info, uint32_t max_samples, uint32_t cap, uint32_t min_rays,
                                uint32_t* n_rays_next, hipStream_t stream) {
    TN_CHECK_ARG(info && n_rays_next && cap > 0);
    estimate_rays_kernel<<<1, 1, 0, stream>>>(info, max_samples, cap, min_rays, n_rays_next);
    TN_CHECK_LAUNCH();
    return TN_OK;
}
