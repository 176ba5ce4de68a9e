// tgk_fast.hip -- the fast tracking path.
//
// * Persistent lanes: a grid sized to fill the GPU once; every wavefront
//   claims seeds from a device queue (one atomic per wavefront refill) and
//   each lane starts a new streamline as soon as its previous one stops, so
//   streamlines of very different lengths (5 to 3000 steps) do not leave
//   lanes idle until the longest of a wavefront ends.
// * Per-lane cell cache: mask value and the voxel's model coefficients stay
//   on chip (LDS at order 8, registers at order 12 and for DTI) until the
//   point crosses into another cell (about every ten steps at step 0.1).
// * Transcendental-free SH model (tgk_fast_model.h), hardware exp2/log2/cos
//   where the reference calls exp/log/cos, FP64 arc length; the four
//   orientation updates (Transport, Diffusion, Probabilistic, Deterministic).
// * Where a launch has fewer streamlines than lanes, or is left with few, lanes
//   (Probabilistic, Deterministic: track_group_kernel) or wavefronts (SH
//   Transport, Diffusion: track_split_fast_kernel) share a streamline's steps.
// * Seed-major dense output rows, compacted into ragged points afterwards.
// * The boundary connectome's tracking loop on the same machinery
//   (connectome_fast_kernel); its hits pass is the plain path's.
//
// Compiled with -ffp-contract=on: a product and a sum in one expression
// become an fma as the source writes them. With =fast the compiler also
// fused across statements, and chose differently in kernel variants that
// differ only in where a row waits (LDS or registers), which changed a few
// trajectories in the last bit; with =on every variant rounds alike.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

#include "tgk_fast_model.h"
#include "tgk_internal.h"
#include "tgk.h"
#include "tgk_sh_basis.h"

namespace tgk {

namespace {

using fast::Order;

__device__ __forceinline__ void store_row(float *dense, int64_t g, uint32_t n_points, uint32_t n, V3 p)
{
    float *dst = dense + (g * (int64_t)n_points + n) * 3;
    dst[0] = p.x;
    dst[1] = p.y;
    dst[2] = p.z;
}

__device__ __forceinline__ int64_t mask_cell(const MaskView &m, V3 p)
{
    const float rx = floorf(affine_row(m.inv, 0, p) + 0.5f);
    const float ry = floorf(affine_row(m.inv, 1, p) + 0.5f);
    const float rz = floorf(affine_row(m.inv, 2, p) + 0.5f);
    // Bitwise &: all three coordinates are computed anyway, and a branch per
    // test costs more than the tests.
    if (!((rx >= 0.0f) & (rx < (float)m.dims[0]) & (ry >= 0.0f) & (ry < (float)m.dims[1]) & (rz >= 0.0f) &
          (rz < (float)m.dims[2])))
        return -1;
    return ((int64_t)(uint32_t)rx * m.dims[1] + (uint32_t)ry) * m.dims[2] + (uint32_t)rz;
}

// Cell ids of the tracking kernel are 32-bit: the fast path takes mask and
// field grids of fewer than 2^32 - 2 voxels.
constexpr uint32_t NO_CELL = 0xffffffffu;     // outside the grid

// The cell of rounded voxel coordinates (rx, ry, rz) on a grid, C order.
__device__ __forceinline__ uint32_t grid_cell(float rx, float ry, float rz, const uint32_t dims[3])
{
    // Bitwise &: all three coordinates are computed anyway, and a branch per
    // test costs more than the tests.
    if (!((rx >= 0.0f) & (rx < (float)dims[0]) & (ry >= 0.0f) & (ry < (float)dims[1]) & (rz >= 0.0f) &
          (rz < (float)dims[2])))
        return NO_CELL;
    return ((uint32_t)rx * dims[1] + (uint32_t)ry) * dims[2] + (uint32_t)rz;
}

// Saved points are stored in groups. A lane appends a 12-byte point about
// every 2.5 steps to its own row, and the grid's 262,144 lanes keep more
// partly written lines open than L2 holds, so single-point stores were
// written back to memory in partial lines several times each (20.9 GB
// written for 6 GB of points at 1M seeds). A group of four is four
// consecutive points starting at a multiple of four, 48 bytes, stored as
// three 16-byte stores when its address is 16-byte aligned (always, for a
// 16-byte aligned buffer and n_points a multiple of 4): 8.2 GB written, and
// 24.2 -> 21.1 ms per launch. The order-12 kernels and the Probabilistic
// and Deterministic ones, whose registers the group would push past a wave
// boundary, store single points.
template <int MODEL, int ALGO, int LMAX> constexpr int point_group()
{
    return (MODEL == MODEL_SH && LMAX == 12) || ALGO == ALGO_PROBABILISTIC || ALGO == ALGO_DETERMINISTIC ? 1 : 4;
}

template <int G> struct Lane {
    int32_t g;          // seed being tracked (-1: idle); calls take fewer than 2^31 seeds
    V3 point, o;
    V3 previous;        // the last step's start (mesh domains: the segment tested against the boundary)
    uint2 rng;
    double time;
    uint32_t n, steps;
    uint32_t field_cell; // cell ids of `point` (UNSET_CELL: none yet); their data is requested by request_cells
    uint32_t mask_cell;
    uint32_t mask_value; // the mask at mask_cell (0 outside the mask image)
    SegmentCandidates near;  // mesh domains: of the last tested segment's start
    bool field_ok;       // `point` is inside the field image
    bool row_read;       // request_cells read a row / a mask value this iteration
    bool mask_read;
    // The last `held` saved points not yet stored, oldest first, in
    // group[G - held ..]; their indices are n - held .. n - 1.
    // `store_due`: n is a multiple of G, so they close a group.
    V3 group[G];
    uint32_t held;
    bool store_due;
};

template <int G> __device__ __forceinline__ void hold_point(Lane<G> &L, V3 q)
{
#pragma unroll
    for (int i = 0; i + 1 < G; i++)
        L.group[i] = L.group[i + 1];
    L.group[G - 1] = q;
    L.held = min(L.held + 1u, (uint32_t)G);
    L.n++;
    L.store_due = L.n % G == 0;
}

// Stores the held points: a whole aligned group of four as three float4
// stores, otherwise one point at a time (a single-point group, the first
// group after a resumption, or what a stopping or saved streamline holds).
template <int G> __device__ __forceinline__ void store_held(const TrackLaunch &p, Lane<G> &L)
{
    float *row = p.points + ((int64_t)L.g * p.n_points + (L.n - L.held)) * 3;
    if (G == 4 && L.held == G && (reinterpret_cast<uintptr_t>(row) & 15u) == 0) {
        float4 *dst = reinterpret_cast<float4 *>(row);
        const V3 *q = L.group;
        dst[0] = make_float4(q[0].x, q[0].y, q[0].z, q[G > 1 ? 1 : 0].x);
        dst[1] = make_float4(q[G > 1 ? 1 : 0].y, q[G > 1 ? 1 : 0].z, q[G > 2 ? 2 : 0].x, q[G > 2 ? 2 : 0].y);
        dst[2] = make_float4(q[G > 2 ? 2 : 0].z, q[G - 1].x, q[G - 1].y, q[G - 1].z);
    } else {
#pragma unroll
        for (int i = 0; i < G; i++) {
            if ((uint32_t)i >= G - L.held) {
                float *dst = row + 3 * (i - (G - (int)L.held));
                dst[0] = L.group[i].x;
                dst[1] = L.group[i].y;
                dst[2] = L.group[i].z;
            }
        }
    }
    L.held = 0;
    L.store_due = false;
}

// A closed group is stored in the iteration after its last point is saved,
// right after that iteration's wait for its cell data: every iteration
// waits (s_waitcnt vmcnt(0)) for the data requested in the previous one,
// and vector stores count under the same counter, so a store issued at the
// end of an iteration would hold the next one at that wait.
template <int G> __device__ __forceinline__ void store_due_group(const TrackLaunch &p, Lane<G> &L)
{
    if (L.store_due)
        store_held(p, L);
}

// A streamline in flight when a generation of the persistent launch ends
// (see track_fast_kernel): everything its lane needs to resume it, in four
// float4 (the previous point only for mesh domains). Its held points are
// stored first; the cell data are requested again on resumption.
template <int DOMAIN, int G> __device__ __forceinline__ void save_lane(float4 *slot, const Lane<G> &L)
{
    const uint64_t tb = (uint64_t)__double_as_longlong(L.time);
    const V3 prev = DOMAIN == DOMAIN_MESH ? L.previous : v3(0.0f, 0.0f, 0.0f);
    slot[0] = make_float4(L.point.x, L.point.y, L.point.z, L.o.x);
    slot[1] = make_float4(L.o.y, L.o.z, prev.x, prev.y);
    slot[2] = make_float4(prev.z, __uint_as_float((uint32_t)tb), __uint_as_float((uint32_t)(tb >> 32)),
                          __uint_as_float((uint32_t)L.g));
    slot[3] = make_float4(__uint_as_float(L.n), __uint_as_float(L.steps), __uint_as_float(L.rng.x),
                          __uint_as_float(L.rng.y));
}

template <int DOMAIN, int G> __device__ __forceinline__ void resume_lane(const float4 *slot, Lane<G> &L)
{
    const float4 a = slot[0], b = slot[1], c = slot[2], d = slot[3];
    L.point = v3(a.x, a.y, a.z);
    L.o = v3(a.w, b.x, b.y);
    if constexpr (DOMAIN == DOMAIN_MESH)
        L.previous = v3(b.z, b.w, c.x);
    L.time = __longlong_as_double((long long)(((uint64_t)__float_as_uint(c.z) << 32) | __float_as_uint(c.y)));
    L.g = (int32_t)__float_as_uint(c.w);
    L.n = __float_as_uint(d.x);
    L.steps = __float_as_uint(d.y);
    L.rng = make_uint2(__float_as_uint(d.z), __float_as_uint(d.w));
    L.held = 0;
    L.store_due = false;
}

// One iteration of the reference loop (tracking.py:121-147) for a lane with
// a streamline in flight; on termination the lane's results are written and
// the lane becomes idle (L.g = -1).
// Where a lane keeps its cell's coefficients between steps: SH rows of
// order 8 mostly in LDS (float4 columns, one per lane, read back every
// step), so no large register array is carried around the loop; DTI rows
// and order-12 rows in registers.
template <int MODEL, int LMAX> constexpr bool rows_in_lds() { return MODEL == MODEL_SH && LMAX == 8; }
// Threads per block of the fast kernels.
template <int LMAX> constexpr int fast_block() { return 256; }
// float4 columns of a row kept in LDS. At order 8, 10 of the 12 (the first
// 40 of 45 coefficients): 40 KiB per 256-lane block, so four blocks share a
// CU's 160 KiB and each SIMD runs four waves (at 109 VGPRs the registers
// would allow it; the full 48-float row would allow three). The other 5
// coefficients stay in registers.
template <int MODEL, int LMAX> constexpr int lds_vectors() { return rows_in_lds<MODEL, LMAX>() ? 10 : 0; }

// Launch shapes of the order-8 SH Transport and Diffusion tracking kernels,
// chosen per runtime (tgk_runtime_set_fast_shape, the autotuner): lanes per
// block and float4 columns of the row in LDS. Shape 0 is the default above;
// the others trade LDS per block against blocks per CU, or coefficients in
// LDS against registers. Which lane tracks which streamline, and where its
// coefficients wait between steps, changes no result.
struct FastShape {
    int block;
    int lds_vectors;
};
constexpr FastShape FAST_SHAPES[FAST_SHAPE_COUNT] = {{256, 10}, {128, 10}, {512, 10}, {256, 8}, {256, 11}};
template <int MODEL, int ALGO, int LMAX> constexpr bool shaped()
{
    return MODEL == MODEL_SH && LMAX == 8 && (ALGO == ALGO_TRANSPORT || ALGO == ALGO_DIFFUSION);
}
template <int MODEL, int ALGO, int LMAX, int S> constexpr int shape_block()
{
    return shaped<MODEL, ALGO, LMAX>() ? FAST_SHAPES[S].block : fast_block<LMAX>();
}
template <int MODEL, int ALGO, int LMAX, int S> constexpr int shape_lds_vectors()
{
    return shaped<MODEL, ALGO, LMAX>() ? FAST_SHAPES[S].lds_vectors : lds_vectors<MODEL, LMAX>();
}

// Column j of a row from memory into LDS for every lane of the wavefront
// that executes it. The instruction's immediate offset is added to both the
// memory address and the LDS base, so all columns share one vector address
// (the row) and the LDS base is set 16 * j below column j's slot.
template <int BLOCK, int... J>
__device__ __forceinline__ void dma_columns(const void *row, uint32_t wave_base, std::integer_sequence<int, J...>)
{
    (__builtin_amdgcn_global_load_lds(
         row, (__attribute__((address_space(3))) void *)(uintptr_t)(wave_base + (uint32_t)(J * BLOCK * 16 - J * 16)),
         16, J * 16, 0),
     ...);
}

// A cell's row into the lane's cache on a cell change: the first LDS_VEC
// float4 columns of an SH row to LDS (column j of a lane at j * BLOCK +
// lane), the rest to registers; DTI rows to registers.
template <int MODEL, int LMAX, int LDS_VEC = lds_vectors<MODEL, LMAX>(), int BLOCK = fast_block<LMAX>()>
__device__ __forceinline__ void load_row(const float *__restrict__ coeffs, int64_t cell, uint32_t cstride, float *q,
                                         float4 *__restrict__ lds_rows)
{
    constexpr int TERMS = Order<LMAX>::TERMS;
    constexpr int VEC = Order<LMAX>::STRIDE / 4;
    const float4 *row = reinterpret_cast<const float4 *>(coeffs + cell * (int64_t)cstride);
    if constexpr (MODEL == MODEL_SH) {
        // Straight from memory into LDS (no registers held while the loads
        // are in flight): each lane's 16 bytes land at the instruction's
        // wave-uniform LDS base + 16 * lane, i.e. column j of the lane's
        // slot. Lanes that do not reload are masked off and keep theirs.
        // The wavefront's slot base is a scalar: its first lane's byte
        // offset in the block's rows plus the rows' LDS address.
        typedef __attribute__((address_space(3))) char lds_char;
        const uint32_t wave_base =
            (uint32_t)__builtin_amdgcn_readfirstlane((int)((threadIdx.x & ~63u) * 16u)) +
            (uint32_t)(uintptr_t)(lds_char *)lds_rows;
        dma_columns<BLOCK>(static_cast<const void *>(row), wave_base, std::make_integer_sequence<int, LDS_VEC>{});
#pragma unroll
        for (int j = LDS_VEC; j < VEC; j++) {
            const float4 v = row[j];
            if (4 * j < TERMS)
                q[4 * j] = v.x;
            if (4 * j + 1 < TERMS)
                q[4 * j + 1] = v.y;
            if (4 * j + 2 < TERMS)
                q[4 * j + 2] = v.z;
            if (4 * j + 3 < TERMS)
                q[4 * j + 3] = v.w;
        }
    } else {
        const float4 a = row[0], b = row[1];
        q[0] = a.x;
        q[1] = a.y;
        q[2] = a.z;
        q[3] = a.w;
        q[4] = b.x;
        q[5] = b.y;
    }
}

// The LDS part of the cached row back into q, every step.
template <int MODEL, int LMAX, int LDS_VEC = lds_vectors<MODEL, LMAX>(), int BLOCK = fast_block<LMAX>()>
__device__ __forceinline__ void read_row(float *q, const float4 *__restrict__ lds_rows)
{
    constexpr int TERMS = Order<LMAX>::TERMS;
    if constexpr (LDS_VEC > 0) {
        // Loads into LDS (load_row) complete under vmcnt, which the compiler
        // does not wait on before these reads of the same LDS: wait here
        // (s_waitcnt vmcnt(0); expcnt and lgkmcnt left at their maxima).
        __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
        for (int j = 0; j < LDS_VEC; j++) {
            const float4 v = lds_rows[j * BLOCK + threadIdx.x];
            if (4 * j < TERMS)
                q[4 * j] = v.x;
            if (4 * j + 1 < TERMS)
                q[4 * j + 1] = v.y;
            if (4 * j + 2 < TERMS)
                q[4 * j + 2] = v.z;
            if (4 * j + 3 < TERMS)
                q[4 * j + 3] = v.w;
        }
    }
}

// One orientation update on the fast model. Transport and Diffusion take
// their normal draws (fast::draw_noise) from the caller, already drawn;
// Probabilistic draws from `rng` as it goes.
template <int MODEL, int ALGO, int LMAX>
__device__ __forceinline__ V3 update_orientation(const AlgoParams &a, const float *q, V3 o, uint2 &rng,
                                                 const fast::Noise &nz)
{
    if constexpr (ALGO == ALGO_PROBABILISTIC) {
        return fast::probabilistic<MODEL, LMAX>(a, q, o, rng);
    } else if constexpr (ALGO == ALGO_DETERMINISTIC) {
        return fast::deterministic<MODEL, LMAX>(a, q, o);
    } else if constexpr (MODEL == MODEL_SH) {
        return fast::sh_update<ALGO, LMAX>(a, q, o, nz);
    } else {
        const fast::Direction dir = fast::direction_of(o);
        return fast::update<ALGO>(a, fast::dti_model(q, o, dir), dir, o, nz);
    }
}

template <int MODEL, int ALGO, int LMAX>
__device__ __forceinline__ V3 update_orientation(const AlgoParams &a, const float *q, V3 o, uint2 &rng)
{
    const fast::Noise nz = fast::draw_noise<ALGO>(a, rng);
    return update_orientation<MODEL, ALGO, LMAX>(a, q, o, rng, nz);
}

// Requests the data of L.point's cells one iteration before the loop needs
// it: the mask value when the mask cell changes, the coefficient row when
// the field cell changes (into LDS or registers, see load_row). Their
// memory latency then overlaps the rest of the step, and of the next one
// up to the model evaluation, instead of stalling the wavefront, which
// nearly every step holds at least one lane entering a new cell.
// The voxel coordinates come from one evaluation of the field's inverse
// affine; the mask's, when it is the same matrix (shared_affine: every
// image-domain workload that tracks in its field's grid), reuses it. The mask
// rounds floor(v + 0.5) (domain.py:369), the field rint(v) (field.py:97).
template <int MODEL, int DOMAIN, int LMAX, int G, int LDS_VEC, int BLOCK>
__device__ __forceinline__ void request_cells(const TrackLaunch &p, bool shared_affine,
                                              const float *__restrict__ coeffs, uint32_t cstride, Lane<G> &L, float *q,
                                              float4 *__restrict__ lds_rows)
{
    const float fx = affine_row(p.field.inv, 0, L.point);
    const float fy = affine_row(p.field.inv, 1, L.point);
    const float fz = affine_row(p.field.inv, 2, L.point);
    if constexpr (DOMAIN == DOMAIN_MASK) {
        float mx = fx, my = fy, mz = fz;
        if (!shared_affine) {
            mx = affine_row(p.mask.inv, 0, L.point);
            my = affine_row(p.mask.inv, 1, L.point);
            mz = affine_row(p.mask.inv, 2, L.point);
        }
        const uint32_t cell = grid_cell(floorf(mx + 0.5f), floorf(my + 0.5f), floorf(mz + 0.5f), p.mask.dims);
        if (cell != L.mask_cell) {
            L.mask_cell = cell;
            L.mask_value = cell != NO_CELL ? (uint32_t)p.mask.mask[cell] : 0u;
            L.mask_read = cell != NO_CELL;
        }
    }
    const uint32_t cell = grid_cell(rintf(fx), rintf(fy), rintf(fz), p.field.dims);
    L.field_ok = cell != NO_CELL;
    if (cell != NO_CELL && cell != L.field_cell) {
        L.field_cell = cell;
        load_row<MODEL, LMAX, LDS_VEC, BLOCK>(coeffs, (int64_t)cell, cstride, q, lds_rows);
        L.row_read = true;
    }
}

// The tests that end a streamline before its next update, in the reference's
// order (tracking.py:121-133): the row or the step count is full, the point
// left the mask or the last segment hit the boundary (`hit` then names the
// triangle), the point left the field. seg_* is wave_segment_test's answer.
// (Written to its reference in every branch, `hit` costs the mesh kernels
// registers: order-12 Transport between two surfaces, 150k seeds, 14.6 against
// 15.4 ms.)
template <int DOMAIN, int G>
__device__ __forceinline__ bool stop_test(const TrackLaunch &p, const Lane<G> &L, bool seg_decided, bool seg_found,
                                          uint32_t seg_tri, uint32_t &hit_triangle)
{
    uint32_t hit = NO_HIT;
    bool stop = !(L.n < p.n_points && L.steps < p.max_steps);
    if (!stop) {
        if constexpr (DOMAIN == DOMAIN_MASK) {
            stop = L.mask_value == 0u;
        } else if (L.steps > 0) {
            // The start cell's candidate list (wave_segment_test) answers
            // segments up to `reach` long; longer segments, or starts off the
            // grid, traverse the BVH.
            if (seg_found) {
                hit = seg_tri;
                stop = true;
            } else if (!seg_decided) {
                uint32_t tri;
                float t;
                const float dx = L.point.x - L.previous.x, dy = L.point.y - L.previous.y,
                            dz = L.point.z - L.previous.z;
                if (!mesh_far(p.mesh, L.previous, dx * dx + dy * dy + dz * dz) &&
                    bvh_segment_hit(p.mesh, L.previous, L.point, tri, t)) {
                    hit = tri;
                    stop = true;
                }
            }
        }
    }
    if (!stop)
        stop = !L.field_ok;
    hit_triangle = hit;
    return stop;
}

// The arguments f of a kernel (its only parameter) read afresh, for what few
// iterations use: kept in scalar registers over the loop they push hot values
// out of them, into vector lanes, an instruction and a wait per use (26 SGPRs
// spilled on mask domains and 102 on mesh domains, SH Diffusion; now 0 and
// 31). 145 x 174 x 145 DTI Transport, 500k seeds: 8.73 -> 8.59 ms; SH45
// Transport between two surfaces, 300k seeds: 10.2 -> 9.5. A Deterministic
// step holds them: its wavefronts iterate over few lanes at a time, and waited
// for the arguments at each track's end (DTI, 2906 seeds: 2.70 against 2.54 ms
// per call).
template <int ALGO, class Launch> __device__ __forceinline__ const Launch &cold(const Launch &f)
{
    if constexpr (ALGO == ALGO_DETERMINISTIC)
        return f;
    auto *args = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    return *(const Launch *)args;
}

// nz: this step's Diffusion draws, made by the caller before anything that
// waits on memory, so they cover the latency of the cell data
// request_cells asked for.
template <int MODEL, int ALGO, int DOMAIN, int LMAX, int G, int LDS_VEC, int BLOCK>
__device__ __forceinline__ void advance(const FastLaunch &f, const float *__restrict__ coeffs, uint32_t cstride,
                                        Lane<G> &L, float *q, float4 *__restrict__ lds_rows, const fast::Noise &nz,
                                        bool seg_decided, bool seg_found, uint32_t seg_tri)
{
    const TrackLaunch &p = f.track;
    uint32_t hit;
    const bool stop = stop_test<DOMAIN>(p, L, seg_decided, seg_found, seg_tri, hit);
    if (stop) {
        const TrackLaunch &c = cold<ALGO>(f).track;
        store_held(c, L);
        c.lengths[L.g] = L.n;
        c.steps[L.g] = L.steps;
        c.hits[L.g] = hit;
        L.g = -1;
        return;
    }
    read_row<MODEL, LMAX, LDS_VEC, BLOCK>(q, lds_rows);
    store_due_group(p, L);
    L.o = update_orientation<MODEL, ALGO, LMAX>(p.algo, q, L.o, L.rng, nz);
    L.steps++;
    if constexpr (DOMAIN == DOMAIN_MESH)
        L.previous = L.point;
    const float step = p.algo.step_size;
    L.point = v3(L.point.x + step * L.o.x, L.point.y + step * L.o.y, L.point.z + step * L.o.z);
    L.time += (double)step;
    if (L.time >= (double)p.save_at) {
        L.time -= (double)p.save_at;
        const float t = (float)L.time;
        hold_point(L, v3(L.point.x - t * L.o.x, L.point.y - t * L.o.y, L.point.z - t * L.o.z));
    }
    request_cells<MODEL, DOMAIN, LMAX, G, LDS_VEC, BLOCK>(p, f.shared_affine != 0, coeffs, cstride, L, q, lds_rows);
}

// Waves per SIMD the compiler must fit: the order-8 SH Transport and
// Diffusion kernels fit 128 VGPRs without spilling when held to four waves,
// the most their 40 KiB of LDS per block allows (134-140 otherwise, three
// waves). Held to three, the order-12 Transport and Diffusion kernels take
// 168 VGPRs (170-185 otherwise, two waves) and the order-8 Probabilistic
// one 151-155 (168-181, two waves); held to four, Probabilistic ran 3%
// slower. The DTI kernels (90-115 VGPRs, four or five waves) ran 4% slower
// held to seven waves and 19% slower held to eight (spills).
// A launch shape that puts more of the row in LDS allows fewer blocks per
// CU (160 KiB of LDS each): shape 4 (44 coefficients) three waves per SIMD.
template <int MODEL, int ALGO, int DOMAIN, int LMAX, int S = 0> constexpr int fast_min_waves()
{
    if constexpr (MODEL == MODEL_SH && LMAX == 12 && (ALGO == ALGO_TRANSPORT || ALGO == ALGO_DIFFUSION))
        return 3;
    if constexpr (MODEL == MODEL_SH && LMAX == 8 && (ALGO == ALGO_TRANSPORT || ALGO == ALGO_DIFFUSION)) {
        constexpr int block = FAST_SHAPES[S].block;
        constexpr int per_cu = 163840 / (FAST_SHAPES[S].lds_vectors * block * 16);
        constexpr int waves = per_cu * (block / 64) / 4;
        return waves < 4 ? waves : 4;
    }
    if constexpr (MODEL == MODEL_SH && LMAX == 8 && ALGO == ALGO_PROBABILISTIC)
        return 3;
    return 1;
}

// The persistent launch runs in generations (launch_fast): generation 0
// claims seeds; each later one claims the streamlines the previous one left
// in flight. Once all of a generation's work is claimed, lanes go idle as
// their streamlines end, while a wavefront keeps issuing for its longest
// one: on the 1M-seed benchmark workload half the launch would run with
// its lanes ever sparser. So when the generation's live lanes fall below
// `stop_below` (half its work), every wavefront saves its live lanes and
// ends, and the next generation resumes them packed into full wavefronts,
// a quarter or half as many per SIMD, each running correspondingly faster.
// The last generation, or one with little work, runs to completion, by
// track_split_fast_kernel where there is one. Which lane tracks which
// streamline, and when, changes no result.
template <int MODEL, int ALGO, int DOMAIN, int LMAX, int S>
__global__ __launch_bounds__((shape_block<MODEL, ALGO, LMAX, S>()))
__attribute__((amdgpu_waves_per_eu(fast_min_waves<MODEL, ALGO, DOMAIN, LMAX, S>())))
void track_fast_kernel(FastLaunch f)
{
    constexpr int BLOCK = shape_block<MODEL, ALGO, LMAX, S>();
    constexpr int LDS_VEC = shape_lds_vectors<MODEL, ALGO, LMAX, S>();
    __shared__ float4 lds_rows[LDS_VEC > 0 ? LDS_VEC * BLOCK : 1];
    const TrackLaunch &p = f.track;
    const int lane_id = __lane_id();
    const float *coeffs = static_cast<const float *>(f.coeffs);
    const uint32_t cstride = f.coeff_stride;

    // This generation's work: seeds, or the previous generation's saved
    // streamlines, claimed through f.claims. Streamlines that end or are
    // saved are counted in f.ended: FAST_END_SHARDS counters a cache line
    // apart, each wavefront adding to one of them in batches, so that no
    // single word takes every wavefront's updates.
    const bool resume = f.cont_in != nullptr;
    const uint32_t n_work = resume ? *f.cont_in_count : (uint32_t)p.n_seeds;
    uint32_t stop_below = 0;
    if (!f.last) {
        const uint64_t lanes = (uint64_t)gridDim.x * blockDim.x;
        const uint32_t half = (uint32_t)((resume ? (uint64_t)n_work : min((uint64_t)n_work, lanes)) / 2);
        stop_below = half >= f.min_repack ? half : 0u;
    }
    uint32_t *const my_shard =
        f.ended + ((blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) % FAST_END_SHARDS) * FAST_END_STRIDE;

    constexpr int G = point_group<MODEL, ALGO, LMAX>();
    Lane<G> L;
    L.g = -1;
    // An idle lane's position is read (never used) by the wavefront-wide
    // boundary test before its first seed.
    L.point = L.previous = v3(0.0f, 0.0f, 0.0f);
    L.steps = 0;
    L.held = 0;
    L.store_due = false;
    L.row_read = false;
    L.mask_read = false;
    // Rows and mask values this wavefront read (wave-uniform sums).
    uint64_t rows_read = 0, masks_read = 0;
    float q[MODEL == MODEL_SH ? Order<LMAX>::TERMS : 6];
    bool drained = false;
    uint32_t ended_pending = 0;     // ended here and not yet added to the shard
    uint32_t iteration = 0;
    uint32_t live_seen = 0xffffffffu;  // the generation's streamlines in flight at the last count
    bool counting = false;          // shard reads issued, to be summed next iteration
    uint32_t shard_value = 0;

    while (true) {
        // Refill idle lanes, one atomic per wavefront.
        const uint64_t need = __ballot(L.g < 0);
        if (need != 0 && !drained) {
            const FastLaunch &c = cold<ALGO>(f);
            const int leader = __ffsll((unsigned long long)need) - 1;
            const uint32_t count = (uint32_t)__popcll(need);
            uint32_t base = 0;
            if (lane_id == leader)
                base = atomicAdd(c.claims, count);
            base = __shfl(base, leader);
            if ((uint64_t)base + count >= (uint64_t)n_work)
                drained = true;
            if (L.g < 0) {
                const uint32_t rank = (uint32_t)__popcll(need & ((1ull << lane_id) - 1ull));
                const uint64_t j = (uint64_t)base + rank;
                if (j < (uint64_t)n_work) {
                    if (resume) {
                        resume_lane<DOMAIN, G>(c.cont_in + FAST_CONTINUATION_VEC4 * j, L);
                    } else {
                        const uint64_t g = j;
                        L.g = (int32_t)g;
                        const float4 s0 = reinterpret_cast<const float4 *>(c.track.seeds)[2 * g];
                        const float4 s1 = reinterpret_cast<const float4 *>(c.track.seeds)[2 * g + 1];
                        L.point = v3(s0.x, s0.y, s0.z);
                        L.o = v3(s1.x, s1.y, s1.z);
                        L.previous = L.point;
                        if constexpr (ALGO == ALGO_DIFFUSION || ALGO == ALGO_PROBABILISTIC)
                            L.rng = seed_stream(c.track, c.track.first_seed + L.g);
                        L.time = 0.0;
                        L.n = 0;
                        L.steps = 0;
                        L.held = 0;
                        hold_point(L, L.point);  // the seed is the streamline's first point
                    }
                    L.field_cell = UNSET_CELL;
                    L.mask_cell = UNSET_CELL;
                    L.mask_value = 0;
                    L.near.cell = UNSET_CELL;
                    request_cells<MODEL, DOMAIN, LMAX, G, LDS_VEC, BLOCK>(p, f.shared_affine != 0, coeffs, cstride,
                                                                          L, q, lds_rows);
                }
            }
        }
        const uint64_t live = __ballot(L.g >= 0);
        if (live == 0)
            break;
        // The draws need no memory: made first, they cover the latency of
        // the cell data and shard counts requested last iteration. The
        // stream before them is what a saved streamline resumes from.
        // Only live lanes draw: an idle lane's stream is not initialised (an
        // all-zero MWC64X state never leaves zero, and randn would spin).
        const uint2 rng_before = L.rng;
        fast::Noise nz{0.0f, 0.0f};
        if (L.g >= 0)
            nz = fast::draw_noise<ALGO>(p.algo, L.rng);
        if (counting) {
            // Every claim was made before the shards were read, so the
            // streamlines in flight are the work minus those that left.
            uint32_t left = shard_value;
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1)
                left += __shfl_xor(left, d);
            live_seen = n_work - min(left, n_work);
            counting = false;
        }
        if (live_seen < stop_below) {
            // Few streamlines left in flight: end the generation, handing
            // this wavefront's to the next one.
            const FastLaunch &c = cold<ALGO>(f);
            const int leader = __ffsll((unsigned long long)live) - 1;
            const uint32_t count = (uint32_t)__popcll(live);
            uint32_t base = 0;
            if (lane_id == leader) {
                base = atomicAdd(c.cont_out_count, count);
                atomicAdd(my_shard, ended_pending + count);
            }
            base = __shfl(base, leader);
            if (L.g >= 0) {
                store_held(c.track, L);
                L.rng = rng_before;
                save_lane<DOMAIN, G>(c.cont_out +
                              FAST_CONTINUATION_VEC4 *
                                  ((uint64_t)base + (uint32_t)__popcll(live & ((1ull << lane_id) - 1ull))),
                          L);
            }
            ended_pending = 0;
            break;
        }
        bool seg_decided = false, seg_found = false;
        uint32_t seg_tri = 0;
        if constexpr (DOMAIN == DOMAIN_MESH)
            wave_segment_test(p.mesh, L.previous, L.point, L.g >= 0 && L.steps > 0, L.near, seg_decided, seg_found,
                              seg_tri);
        if (L.g >= 0)
            advance<MODEL, ALGO, DOMAIN, LMAX, G, LDS_VEC, BLOCK>(f, coeffs, cstride, L, q, lds_rows, nz,
                                                                 seg_decided, seg_found, seg_tri);
        rows_read += (uint64_t)__popcll(__ballot(L.row_read));
        masks_read += (uint64_t)__popcll(__ballot(L.mask_read));
        L.row_read = false;
        L.mask_read = false;
        ended_pending += (uint32_t)__popcll(live & ~__ballot(L.g >= 0));
        // Once every claim is made, every eighth iteration: add this
        // wavefront's ended streamlines to its shard and read all shards
        // (summed next iteration, after the draws).
        if (stop_below != 0 && drained && (++iteration & 7u) == 0u) {
            if (ended_pending != 0 && lane_id == 0)
                atomicAdd(my_shard, ended_pending);
            ended_pending = 0;
            shard_value = lane_id < FAST_END_SHARDS
                              ? __hip_atomic_load(f.ended + lane_id * FAST_END_STRIDE, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : 0u;
            counting = true;
        }
    }
    if (stop_below != 0 && ended_pending != 0 && lane_id == 0)
        atomicAdd(my_shard, ended_pending);
    // A lane that stopped may have requested a row for its last point; the
    // wavefront waits for every load into LDS before it ends, so none lands
    // in LDS another workgroup has been given.
    __builtin_amdgcn_s_waitcnt(0);
    // The wavefront's memory reads of rows and mask values, one atomic each
    // (the launch's totals price the bytes the cell cache had to fetch).
    if (lane_id == 0) {
        atomicAdd(&cold<ALGO>(f).stats[0], (unsigned long long)rows_read);
        atomicAdd(&cold<ALGO>(f).stats[1], (unsigned long long)masks_read);
    }
}

// Order-8 SH Transport and Diffusion, 64 streamlines to a block of four
// wavefronts that share out each step: 0, 1 and 2 evaluate orders 0-2, 3-5
// and 6-8 of the model from their parts of the row, 3 draws the noise, tests
// the boundary, stores the points and reads ahead. All hold the streamlines'
// state and do the rest of the step alike; the parts go through LDS, one
// barrier per step (two buffers: a wavefront writes the next step's parts
// while another still reads this one's).
//
// A lone wavefront of track_fast_kernel issues its 650 instructions per step
// at about one per four cycles and then waits for the row, a third of the
// step. Here the chain is some 300 instructions, and the row comes from the
// CU's own cache where the streamline keeps its direction: 145 x 174 x 145
// SH45 Diffusion, 5000 seeds, 3000 steps at most: 5.2 -> 3.8 ms per call;
// 32^3 SH45 Transport, 10k seeds: 5.1 -> 3.95.
// Bound by that chain: row, three orders, exchange, sums, exponential map.
// Every sum keeps its order: same bits.
constexpr int FAST_SPLIT_WAVES = 4;
// float4 columns FIRST .. FIRST + N - 1 of a row, and its coefficients from
// the first of them on.
template <int FIRST, int N> __device__ __forceinline__ void load_part(const float4 *row, float4 *part)
{
#pragma unroll
    for (int j = 0; j < N; j++)
        part[j] = row[FIRST + j];
}

template <int FIRST, int N> __device__ __forceinline__ void read_part(const float4 *part, float *q)
{
#pragma unroll
    for (int j = 0; j < N; j++) {
        q[4 * (FIRST + j)] = part[j].x;
        q[4 * (FIRST + j) + 1] = part[j].y;
        q[4 * (FIRST + j) + 2] = part[j].z;
        q[4 * (FIRST + j) + 3] = part[j].w;
    }
}

__device__ __forceinline__ void put_term(float4 *at, const fast::CartesianTerm &t)
{
    *at = make_float4(t.v, t.gx, t.gy, t.gz);
}

template <int M> __device__ __forceinline__ void add_put_term(const float4 *at, fast::Cartesian &g)
{
    const float4 t = *at;
    fast::add_term<M>(fast::CartesianTerm{t.x, t.y, t.z, t.w}, g);
}

template <int ALGO, int DOMAIN>
__global__ __launch_bounds__(64 * FAST_SPLIT_WAVES) void track_split_fast_kernel(FastLaunch f)
{
    constexpr int LMAX = 8;
    __shared__ float4 terms[2][7][64];       // orders 0-2 summed, then orders 3 to 8
    __shared__ float2 noise[2][64];
    __shared__ uint32_t test[2][64];         // mask domains: the mask value; mesh domains: the triangle hit
    const TrackLaunch &p = f.track;
    const int lane = threadIdx.x & 63;
    const int role = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const float *coeffs = static_cast<const float *>(f.coeffs);
    const uint32_t cstride = f.coeff_stride;
    const float step = p.algo.step_size;
    const bool resume = f.cont_in != nullptr;
    const uint32_t n_work = resume ? f.tail[0] : (uint32_t)p.n_seeds;
    const float4 *const saved = resume && f.tail[1] != 0 ? f.cont[1] : f.cont[0];
    uint64_t reads = 0;                      // rows (wavefront 0), mask values (2)
    int buffer = 0;
    for (uint32_t base = blockIdx.x * 64; base < n_work; base += gridDim.x * 64) {
        const uint32_t j = base + lane;
        bool live = j < n_work;
        Lane<1> L;
        L.g = 0;
        L.point = L.o = L.previous = v3(0.0f, 0.0f, 0.0f);
        L.rng = make_uint2(0u, 0u);
        L.time = 0.0;
        L.n = L.steps = 0;
        if (live) {
            if (resume) {
                resume_lane<DOMAIN, 1>(saved + FAST_CONTINUATION_VEC4 * (uint64_t)j, L);
            } else {
                L.g = (int32_t)j;
                const float4 s0 = reinterpret_cast<const float4 *>(p.seeds)[2 * (uint64_t)j];
                const float4 s1 = reinterpret_cast<const float4 *>(p.seeds)[2 * (uint64_t)j + 1];
                L.point = L.previous = v3(s0.x, s0.y, s0.z);
                L.o = v3(s1.x, s1.y, s1.z);
                if (ALGO == ALGO_DIFFUSION && role == 3)
                    L.rng = seed_stream(p, p.first_seed + L.g);
                L.n = 1;
            }
        }
        float *const row = p.points + (int64_t)L.g * p.n_points * 3;
        if (live && !resume && role == 3) {
            row[0] = L.point.x;
            row[1] = L.point.y;
            row[2] = L.point.z;
        }
        L.field_cell = L.mask_cell = L.near.cell = UNSET_CELL;
        L.mask_value = 0;
        float4 part[6];
#pragma unroll
        for (int i = 0; i < 6; i++)
            part[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float ahead0 = 0.0f, ahead1 = 0.0f;
        // As track_fast_kernel counts: a streamline's first two requests, made
        // in one iteration there, count once, and a mask value not at all
        // when the second leaves the image.
        uint64_t first = 0;
        int request = 0;
        const auto count_reads = [&](bool read, bool left) {
            const uint64_t lanes = __ballot(read);
            reads += (uint64_t)__popcll(request == 1 ? lanes & ~first : lanes);
            if (request == 1)
                reads -= (uint64_t)__popcll(__ballot(left) & first);
            first = lanes;
            request = min(request + 1, 2);
        };
        // The loads above end here: a wait left to their first use would
        // stand inside the loop, where it waits for everything in flight.
        __builtin_amdgcn_s_waitcnt(0);
        while (true) {
            // This point's cells, and its row's part on a change of cell.
            uint32_t cell = NO_CELL;
            {
                const float fx = affine_row(p.field.inv, 0, L.point);
                const float fy = affine_row(p.field.inv, 1, L.point);
                const float fz = affine_row(p.field.inv, 2, L.point);
                cell = grid_cell(rintf(fx), rintf(fy), rintf(fz), p.field.dims);
                if (DOMAIN == DOMAIN_MASK && role == 2) {
                    float mx = fx, my = fy, mz = fz;
                    if (f.shared_affine == 0) {
                        mx = affine_row(p.mask.inv, 0, L.point);
                        my = affine_row(p.mask.inv, 1, L.point);
                        mz = affine_row(p.mask.inv, 2, L.point);
                    }
                    const uint32_t m =
                        grid_cell(floorf(mx + 0.5f), floorf(my + 0.5f), floorf(mz + 0.5f), p.mask.dims);
                    const bool read = live && m != L.mask_cell && m != NO_CELL;
                    count_reads(read, live && m == NO_CELL && m != L.mask_cell);
                    if (live && m != L.mask_cell) {
                        L.mask_cell = m;
                        L.mask_value = 0;
                        if (m != NO_CELL)
                            L.mask_value = p.mask.mask[m];
                    }
                }
            }
            const bool change = live && cell != NO_CELL && cell != L.field_cell;
            if (role == 0)
                count_reads(change, false);
            if (change) {
                L.field_cell = cell;
                const float4 *at = reinterpret_cast<const float4 *>(coeffs + (int64_t)cell * cstride);
                if (role == 0)
                    load_part<0, 6>(at, part);
                else if (role == 1)
                    load_part<5, 5>(at, part);
                else if (role == 2)
                    load_part<9, 3>(at, part);
            }
            const V3 n = fast::unit_direction(L.o);
            const float w = n.z * n.z;
            float q[48];
            if (role == 0) {
                read_part<0, 6>(part, q);
                const fast::Cartesian g = fast::sh_cartesian<LMAX, 2>(q, n);
                terms[buffer][0][lane] = make_float4(g.value, g.gx, g.gy, g.gz);
            } else if (role < 3) {
                // u^2, as the sums over all orders reach it.
                float pr = n.x * n.x - n.y * n.y, pi = n.x * n.y + n.y * n.x;
                if (role == 1) {
                    read_part<5, 5>(part, q);
                    put_term(&terms[buffer][1][lane], fast::sh_cartesian_term<LMAX, 3>(q, n.z, w, n.x, n.y, pr, pi));
                    put_term(&terms[buffer][2][lane], fast::sh_cartesian_term<LMAX, 4>(q, n.z, w, n.x, n.y, pr, pi));
                    put_term(&terms[buffer][3][lane], fast::sh_cartesian_term<LMAX, 5>(q, n.z, w, n.x, n.y, pr, pi));
                } else {
                    read_part<9, 3>(part, q);
#pragma unroll
                    for (int m = 3; m <= 5; m++) {
                        const float ur = pr * n.x - pi * n.y;
                        pi = pr * n.y + pi * n.x;
                        pr = ur;
                    }
                    put_term(&terms[buffer][4][lane], fast::sh_cartesian_term<LMAX, 6>(q, n.z, w, n.x, n.y, pr, pi));
                    put_term(&terms[buffer][5][lane], fast::sh_cartesian_term<LMAX, 7>(q, n.z, w, n.x, n.y, pr, pi));
                    put_term(&terms[buffer][6][lane], fast::sh_cartesian_term<LMAX, 8>(q, n.z, w, n.x, n.y, pr, pi));
                    if constexpr (DOMAIN == DOMAIN_MASK)
                        test[buffer][lane] = L.mask_value;
                }
            } else {
                if constexpr (ALGO == ALGO_DIFFUSION) {
                    fast::Noise nz{0.0f, 0.0f};
                    if (live)
                        nz = fast::draw_noise<ALGO>(p.algo, L.rng);
                    noise[buffer][lane] = make_float2(nz.r1, nz.r2);
                }
                if constexpr (DOMAIN == DOMAIN_MESH) {
                    bool decided = false, found = false;
                    uint32_t tri = 0, hit = NO_HIT;
                    wave_segment_test(p.mesh, L.previous, L.point, live && L.steps > 0, L.near, decided, found, tri);
                    if (live && L.steps > 0 && L.n < p.n_points && L.steps < p.max_steps) {
                        if (found) {
                            hit = tri;
                        } else if (!decided) {
                            float t;
                            const float dx = L.point.x - L.previous.x, dy = L.point.y - L.previous.y,
                                        dz = L.point.z - L.previous.z;
                            if (!mesh_far(p.mesh, L.previous, dx * dx + dy * dy + dz * dz) &&
                                bvh_segment_hit(p.mesh, L.previous, L.point, tri, t))
                                hit = tri;
                        }
                    }
                    test[buffer][lane] = hit;
                }
            }
            __syncthreads();
            uint32_t hit = NO_HIT;
            bool stop = !(L.n < p.n_points && L.steps < p.max_steps) || cell == NO_CELL;
            if constexpr (DOMAIN == DOMAIN_MASK) {
                stop = stop || test[buffer][lane] == 0u;
            } else {
                hit = test[buffer][lane];
                stop = stop || hit != NO_HIT;
            }
            if (live && stop) {
                live = false;
                if (role == 3) {
                    p.lengths[L.g] = L.n;
                    p.steps[L.g] = L.steps;
                    p.hits[L.g] = hit;
                }
            }
            if (__ballot(live) == 0)
                break;
            const float4 g0 = terms[buffer][0][lane];
            fast::Cartesian g{g0.x, g0.y, g0.z, g0.w};
            add_put_term<3>(&terms[buffer][1][lane], g);
            add_put_term<4>(&terms[buffer][2][lane], g);
            add_put_term<5>(&terms[buffer][3][lane], g);
            add_put_term<6>(&terms[buffer][4][lane], g);
            add_put_term<7>(&terms[buffer][5][lane], g);
            add_put_term<8>(&terms[buffer][6][lane], g);
            fast::Noise nz{0.0f, 0.0f};
            if constexpr (ALGO == ALGO_DIFFUSION) {
                const float2 drawn = noise[buffer][lane];
                nz = fast::Noise{drawn.x, drawn.y};
            }
            buffer ^= 1;
            if (live) {
                L.o = fast::cartesian_turn<ALGO>(p.algo, n, g, L.o, nz);
                L.steps++;
                if constexpr (DOMAIN == DOMAIN_MESH)
                    L.previous = L.point;
                L.point = v3(L.point.x + step * L.o.x, L.point.y + step * L.o.y, L.point.z + step * L.o.z);
                L.time += (double)step;
                const bool save = L.time >= (double)p.save_at;
                if (save)
                    L.time -= (double)p.save_at;
                if (role == 3) {
                    // The last step's reads ahead have arrived (waited for
                    // here, before the store that would be waited for too).
                    asm volatile("" ::"v"(ahead0), "v"(ahead1));
                    if (save) {
                        const float t = (float)L.time;
                        float *at = row + 3 * (int64_t)L.n;
                        at[0] = L.point.x - t * L.o.x;
                        at[1] = L.point.y - t * L.o.y;
                        at[2] = L.point.z - t * L.o.z;
                    }
                    // The lines of the row one straight step ahead, towards this
                    // CU, a step before the others ask for them.
                    const V3 next = v3(L.point.x + step * L.o.x, L.point.y + step * L.o.y, L.point.z + step * L.o.z);
                    const uint32_t c = grid_cell(rintf(affine_row(p.field.inv, 0, next)),
                                                 rintf(affine_row(p.field.inv, 1, next)),
                                                 rintf(affine_row(p.field.inv, 2, next)), p.field.dims);
                    if (c != NO_CELL && c != L.field_cell) {
                        const float *at = coeffs + (int64_t)c * cstride;
                        ahead0 = at[0];
                        ahead1 = at[32];
                    }
                }
                L.n += save ? 1u : 0u;
            }
        }
        // Ended at the break after a barrier: every wavefront is past the
        // parts it reads there but this one's buffer, so the next 64
        // streamlines start on the other.
        buffer ^= 1;
    }
    if (lane == 0 && reads != 0) {
        if (role == 0)
            atomicAdd(&f.stats[0], (unsigned long long)reads);
        else if (role == 2)
            atomicAdd(&f.stats[1], (unsigned long long)reads);
    }
}

// Streamlines tracked by lane groups: fast::GROUP_LANES lanes hold one
// streamline's state between them, share out the evaluations of its update
// and do the rest of the step alike (same data, same arithmetic; the first
// lane of the group stores). One lane per streamline runs a Probabilistic
// step's 64 candidates one after another, 38 us of latency, and a
// Deterministic wavefront its slowest lane's iterations and line search, 70
// us, and a launch lasts as long as its longest streamline's steps, mostly
// with idle lanes: 46 ms for 150k SH45 Probabilistic seeds of 235 steps on
// average and 1200 at most, 206 ms for 100k Deterministic ones of 850 steps
// and 3000 at most. Eight lanes take about an eighth of that latency per
// step, for no more evaluations in all (the one-lane Probabilistic form
// evaluates a block of candidates twice, the Deterministic one waits for its
// wavefront): 16.1 and 32.4 ms, bound by VALU issue (about 1700 instructions
// per Probabilistic step of a wavefront's eight streamlines, 950 per
// Deterministic iteration) and by the longest streamlines.
template <int MODEL, int ALGO, int DOMAIN, int LMAX>
__global__ __launch_bounds__(256) void track_group_kernel(FastLaunch f)
{
    constexpr int W = fast::GROUP_LANES;
    const TrackLaunch &p = f.track;
    const int lane_id = __lane_id();
    const int sub = lane_id % W;
    const bool leader = sub == 0;
    const float *coeffs = static_cast<const float *>(f.coeffs);
    const uint64_t to_lane = f.group_jump[sub], to_end = f.group_jump[W];
    const float one_minus_cos_max = 1.0f - tgk_cosf(p.algo.max_angle);
    const float step = p.algo.step_size;

    Lane<1> L;
    L.g = -1;
    L.point = L.previous = v3(0.0f, 0.0f, 0.0f);
    L.steps = 0;
    L.row_read = false;
    L.mask_read = false;
    uint64_t rows_read = 0, masks_read = 0;
    float q[MODEL == MODEL_SH ? Order<LMAX>::TERMS : 6];
    bool drained = false;
    // Iterations the current update has done; -1: the next step begins.
    // A pass of the loop does one (a Probabilistic update is one), so that
    // groups whose updates take few go on to their next step while others
    // still iterate.
    int iteration = -1;

    while (true) {
        // Refill idle groups, one atomic per wavefront.
        const uint64_t need = __ballot(leader && L.g < 0);
        if (need != 0 && !drained) {
            const int first = __ffsll((unsigned long long)need) - 1;
            const uint32_t count = (uint32_t)__popcll(need);
            uint32_t base = 0;
            if (lane_id == first)
                base = atomicAdd(f.claims, count);
            base = __shfl(base, first);
            if ((uint64_t)base + count >= (uint64_t)p.n_seeds)
                drained = true;
            if (L.g < 0) {
                const uint64_t g = (uint64_t)base + (uint32_t)__popcll(need & ((1ull << (lane_id - sub)) - 1ull));
                if (g < (uint64_t)p.n_seeds) {
                    L.g = (int32_t)g;
                    const float4 s0 = reinterpret_cast<const float4 *>(p.seeds)[2 * g];
                    const float4 s1 = reinterpret_cast<const float4 *>(p.seeds)[2 * g + 1];
                    L.point = v3(s0.x, s0.y, s0.z);
                    L.o = v3(s1.x, s1.y, s1.z);
                    L.previous = L.point;
                    if constexpr (ALGO == ALGO_PROBABILISTIC)
                        L.rng = seed_stream(p, p.first_seed + L.g);
                    L.time = 0.0;
                    L.n = 1;  // the seed is the streamline's first point
                    L.steps = 0;
                    if (leader)
                        store_row(p.points, L.g, p.n_points, 0, L.point);
                    L.field_cell = UNSET_CELL;
                    L.mask_cell = UNSET_CELL;
                    L.mask_value = 0;
                    L.near.cell = UNSET_CELL;
                    request_cells<MODEL, DOMAIN, LMAX, 1, 0, 256>(p, f.shared_affine != 0, coeffs, f.coeff_stride, L,
                                                                  q, nullptr);
                }
            }
        }
        if (__ballot(L.g >= 0) == 0)
            break;
        const bool starting = L.g >= 0 && iteration < 0;
        bool seg_decided = false, seg_found = false;
        uint32_t seg_tri = 0;
        if constexpr (DOMAIN == DOMAIN_MESH) {
            // Asked once per group.
            wave_segment_test(p.mesh, L.previous, L.point, leader && starting && L.steps > 0, L.near, seg_decided,
                              seg_found, seg_tri);
            seg_decided = __shfl((int)seg_decided, 0, W) != 0;
            seg_found = __shfl((int)seg_found, 0, W) != 0;
            seg_tri = __shfl(seg_tri, 0, W);
        }
        if (starting) {
            uint32_t hit;
            if (stop_test<DOMAIN>(p, L, seg_decided, seg_found, seg_tri, hit)) {
                if (leader) {
                    p.lengths[L.g] = L.n;
                    p.steps[L.g] = L.steps;
                    p.hits[L.g] = hit;
                }
                L.g = -1;
            } else {
                iteration = 0;
                if constexpr (ALGO == ALGO_DETERMINISTIC)
                    L.o = fast::deterministic_start(L.o);
            }
        }
        if (L.g >= 0) {
            bool more = false;
            if constexpr (ALGO == ALGO_PROBABILISTIC)
                L.o = fast::probabilistic_group<MODEL, LMAX>(p.algo, q, L.o, L.rng, to_lane, to_end,
                                                            one_minus_cos_max, sub);
            else if (iteration < p.algo.max_iterations)
                more = fast::deterministic_iteration<LMAX>(p.algo, q, L.o, sub) &&
                       iteration + 1 < p.algo.max_iterations;
            iteration++;
            if (!more) {
                iteration = -1;
                L.steps++;
                if constexpr (DOMAIN == DOMAIN_MESH)
                    L.previous = L.point;
                L.point = v3(L.point.x + step * L.o.x, L.point.y + step * L.o.y, L.point.z + step * L.o.z);
                L.time += (double)step;
                if (L.time >= (double)p.save_at) {
                    L.time -= (double)p.save_at;
                    const float t = (float)L.time;
                    if (leader)
                        store_row(p.points, L.g, p.n_points, L.n,
                                  v3(L.point.x - t * L.o.x, L.point.y - t * L.o.y, L.point.z - t * L.o.z));
                    L.n++;
                }
                request_cells<MODEL, DOMAIN, LMAX, 1, 0, 256>(p, f.shared_affine != 0, coeffs, f.coeff_stride, L, q,
                                                              nullptr);
            }
        }
        // Counted once per step, as one lane per streamline counts them.
        const bool ended = iteration < 0;
        rows_read += (uint64_t)__popcll(__ballot(leader && ended && L.row_read));
        masks_read += (uint64_t)__popcll(__ballot(leader && ended && L.mask_read));
        if (ended) {
            L.row_read = false;
            L.mask_read = false;
        }
    }
    if (lane_id == 0) {
        atomicAdd(&f.stats[0], (unsigned long long)rows_read);
        atomicAdd(&f.stats[1], (unsigned long long)masks_read);
    }
}

// A generation of the connectome or TOD kernel, as one wavefront sees it: the
// tracks in flight over the launch, from shards that every wavefront adds its
// ended tracks to, and the cut once fewer than stop_below are left.
struct Generation {
    uint64_t n_work;
    uint32_t stop_below;      // 0: run to the end
    uint32_t pending = 0;     // ended here and not yet added to the shard
    uint32_t value = 0;       // this lane's shard as last read
    uint32_t iteration = 0;
    bool reading = false;     // shards read, to be summed next iteration
    uint32_t in_flight = 0xffffffffu;

    __device__ __forceinline__ Generation(uint64_t work, bool last, uint32_t min_repack)
    {
        n_work = work;
        const uint64_t half = min(n_work, (uint64_t)gridDim.x * blockDim.x) / 2;
        stop_below = !last && half >= min_repack ? (uint32_t)half : 0u;
    }
    static __device__ __forceinline__ uint32_t *shard(uint32_t *ended)
    {
        return ended + ((blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) % FAST_END_SHARDS) * FAST_END_STRIDE;
    }
    // Whether the wavefront hands its tracks over now.
    __device__ __forceinline__ bool over()
    {
        if (reading) {
            uint32_t left = value;
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1)
                left += __shfl_xor(left, d);
            in_flight = (uint32_t)min(n_work - min((uint64_t)left, n_work), (uint64_t)0xffffffffu);
            reading = false;
        }
        return in_flight < stop_below;
    }
    // The `live` lanes' tracks leave: the slot of this lane's among `saved`.
    __device__ __forceinline__ uint64_t hand_over(uint64_t live, uint32_t *ended, uint32_t *saved)
    {
        const int leader = __ffsll((unsigned long long)live) - 1;
        uint32_t base = 0;
        if (__lane_id() == leader) {
            base = atomicAdd(saved, (uint32_t)__popcll(live));
            atomicAdd(shard(ended), pending + (uint32_t)__popcll(live));
        }
        pending = 0;
        return (uint64_t)__shfl(base, leader) + (uint32_t)__popcll(live & ((1ull << __lane_id()) - 1ull));
    }
    // Once every claim is made, every 32nd iteration: this wavefront's ended
    // tracks to its shard, and all shards read. (Every eighth, 300k SH15
    // Transport tracks of at most 500 steps took 4.3 ms, 3.9 so.)
    template <int ALGO, class Launch> __device__ __forceinline__ void count(const Launch &f, bool drained)
    {
        if (stop_below != 0 && drained && (++iteration & 31u) == 0u) {
            uint32_t *const ended = cold<ALGO>(f).ended;
            flush(ended);
            value = __lane_id() < FAST_END_SHARDS
                        ? __hip_atomic_load(ended + __lane_id() * FAST_END_STRIDE, __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT)
                        : 0u;
            reading = true;
        }
    }
    __device__ __forceinline__ void flush(uint32_t *ended)
    {
        if (stop_below != 0 && pending != 0 && __lane_id() == 0)
            atomicAdd(shard(ended), pending);
        pending = 0;
    }
};

// The one generation of a launch that is never cut short.
struct WholeLaunch {
    uint64_t n_work;

    __device__ __forceinline__ WholeLaunch(uint64_t work, bool, uint32_t) { n_work = work; }
};

// tracking.py:457-558 (kernel connectome) on the fast model: the plain
// connectome kernel's loop (mask, field, update, finite and length test,
// move) with the tracking kernel's persistent lanes, cell cache and
// polynomial model. A finished track leaves the same record in its seed's
// output slots as on the plain path (last segment, start barycentrics,
// start triangle, length test) for the shared hits kernel.
//
// Run in generations where it pays (in_generations), as track_fast_kernel: a
// launch ends with its longest tracks, whose step takes four times as long
// while every wavefront of a SIMD keeps a few lanes alive. A track cut short
// waits in its seed's record (rows[2..7]: steps, noise state, orientation), its
// seed in a list in the columns' slots, which only the hits kernel fills.
// 97 x 116 x 97 SH45 Diffusion, 300k seeds, 3000 steps at most: 10.9 ms per call
// in one launch, 8.7 so, of which the last generation's lone wavefronts, at
// 1.9 us per step of the longest tracks, take some 4. The count costs 11 to 13
// VGPRs and as many scalar registers, so launches in one generation run a
// kernel without it (200k DTI Transport tracks: 6.2 against 5.5 ms).
template <int MODEL, int ALGO, int LMAX, bool GENERATIONS>
__global__ __launch_bounds__(fast_block<LMAX>()) void connectome_fast_kernel(FastConnectomeLaunch f)
{
    __shared__ float4 lds_rows[rows_in_lds<MODEL, LMAX>() ? lds_vectors<MODEL, LMAX>() * fast_block<LMAX>() : 1];
    const ConnectomeLaunch &c = f.connectome;
    const float *coeffs = static_cast<const float *>(f.coeffs);
    const uint32_t cstride = f.coeff_stride;
    const float step = c.algo.step_size;
    const int lane_id = __lane_id();
    const bool resume = GENERATIONS && f.list_in != nullptr;
    std::conditional_t<GENERATIONS, Generation, WholeLaunch> work(
        resume ? (uint64_t)*f.list_in_count : (uint64_t)c.n_seeds, f.last, f.min_repack);

    int64_t g = -1;
    bool drained = false;
    uint64_t live = 0;
    uint2 rng = make_uint2(0u, 0u);
    V3 point = v3(0.0f, 0.0f, 0.0f), o = point, previous = point;
    uint32_t tracked = 0, start_triangle = 0;
    float b0 = 0.0f, b1 = 0.0f, b2 = 0.0f;
    int64_t field_cell = -2, cached_mask_cell = -2;
    bool mask_inside = false;
    float q[MODEL == MODEL_SH ? Order<LMAX>::TERMS : 6];

    while (true) {
        const uint64_t need = __ballot(g < 0);
        if constexpr (GENERATIONS)
            work.pending += (uint32_t)__popcll(live & need);
        // Refill idle lanes, one atomic per wavefront.
        if (need != 0 && !drained) {
            const FastConnectomeLaunch &rare = cold<ALGO>(f);
            const ConnectomeLaunch &c = rare.connectome;
            const int leader = __ffsll((unsigned long long)need) - 1;
            const uint32_t wanted = (uint32_t)__popcll(need);
            uint32_t base = 0;
            if (lane_id == leader)
                base = atomicAdd(c.queue, wanted);
            base = __shfl(base, leader);
            if ((uint64_t)base + wanted >= work.n_work)
                drained = true;
            if (g < 0) {
                const uint64_t claimed = (uint64_t)base + (uint64_t)__popcll(need & ((1ull << lane_id) - 1ull));
                if (claimed < work.n_work) {
                    if (resume) {
                        g = (int64_t)rare.list_in[claimed];
                        const float *w = c.weights + 9 * g;
                        const int32_t *r = c.rows + 9 * g;
                        previous = v3(w[0], w[1], w[2]);
                        point = v3(w[3], w[4], w[5]);
                        b0 = w[6];
                        b1 = w[7];
                        b2 = w[8];
                        start_triangle = (uint32_t)r[0];
                        tracked = (uint32_t)r[2];
                        rng = make_uint2((uint32_t)r[3], (uint32_t)r[4]);
                        o = v3(__int_as_float(r[5]), __int_as_float(r[6]), __int_as_float(r[7]));
                    } else {
                        g = (int64_t)claimed;
                        rng = rng_init(c.rng_seed, (uint32_t)g);
                        const BoundarySample sample = sample_boundary(c.boundary.vertices, c.boundary.triangles,
                                                                      c.cumulative, c.n_triangles, rng);
                        point = sample.point;
                        o = sample.orientation;
                        previous = point;
                        tracked = 0;
                        start_triangle = sample.triangle;
                        b0 = sample.bary[0];
                        b1 = sample.bary[1];
                        b2 = sample.bary[2];
                    }
                    field_cell = -2;
                    cached_mask_cell = -2;
                    mask_inside = false;
                }
            }
        }
        live = __ballot(g >= 0);
        if (live == 0)
            break;
        if constexpr (GENERATIONS) {
            if (work.over()) {
                // Few tracks left in flight: hand this wavefront's over.
                const FastConnectomeLaunch &rare = cold<ALGO>(f);
                const uint64_t slot = work.hand_over(live, rare.ended, rare.list_out_count);
                if (g >= 0) {
                    rare.list_out[slot] = (uint32_t)g;
                    float *w = rare.connectome.weights + 9 * g;
                    int32_t *r = rare.connectome.rows + 9 * g;
                    w[0] = previous.x;
                    w[1] = previous.y;
                    w[2] = previous.z;
                    w[3] = point.x;
                    w[4] = point.y;
                    w[5] = point.z;
                    w[6] = b0;
                    w[7] = b1;
                    w[8] = b2;
                    r[0] = (int32_t)start_triangle;
                    r[2] = (int32_t)tracked;
                    r[3] = (int32_t)rng.x;
                    r[4] = (int32_t)rng.y;
                    r[5] = __float_as_int(o.x);
                    r[6] = __float_as_int(o.y);
                    r[7] = __float_as_int(o.z);
                }
                break;
            }
            work.template count<ALGO>(f, drained);
        }
        if (g < 0)
            continue;
        bool stop = tracked >= c.n_steps;
        if (!stop) {
            const int64_t cell = mask_cell(c.mask, point);
            if (cell != cached_mask_cell) {
                cached_mask_cell = cell;
                mask_inside = cell >= 0 && c.mask.mask[cell] != 0;
            }
            stop = !mask_inside;
        }
        int64_t cell = -1;
        if (!stop) {
            cell = field_voxel(c.field, point);
            stop = cell < 0;
        }
        if (!stop) {
            if (cell != field_cell) {
                field_cell = cell;
                load_row<MODEL, LMAX>(coeffs, cell, cstride, q, lds_rows);
            }
            read_row<MODEL, LMAX>(q, lds_rows);
            o = update_orientation<MODEL, ALGO, LMAX>(c.algo, q, o, rng);
            stop = !(__builtin_isfinite(o.x) && __builtin_isfinite(o.y) && __builtin_isfinite(o.z)) ||
                   length3(o) < 0.5f;
        }
        if (!stop) {
            previous = point;
            point.x += step * o.x;
            point.y += step * o.y;
            point.z += step * o.z;
            tracked++;
            continue;
        }
        // (Read afresh, few tracks' ends, one after another, waited for them:
        // 117 tracks 1.26 against 1.14 ms.)
        const ConnectomeLaunch &c = GENERATIONS ? cold<ALGO>(f).connectome : f.connectome;
        float *record = c.weights + 9 * g;
        record[0] = previous.x;
        record[1] = previous.y;
        record[2] = previous.z;
        record[3] = point.x;
        record[4] = point.y;
        record[5] = point.z;
        record[6] = b0;
        record[7] = b1;
        record[8] = b2;
        c.rows[9 * g] = (int32_t)start_triangle;
        c.rows[9 * g + 1] = (float)tracked * step < c.min_length ? 0 : 1;
        g = -1;
    }
    if constexpr (GENERATIONS)
        work.flush(cold<ALGO>(f).ended);
}

// tracking.py:262-357 (kernel tod) on the fast model: the plain TOD
// kernel's loop (tod_kernel: mask, field and output cell, flush on leaving a
// cell, deposit, update, finite and length test, move, flush at the end)
// with persistent lanes and the polynomial model. The deposit is the
// reference's 45-term SH basis at the step's orientation (fast::sh45_basis,
// from z and powers of x + iy instead of angles), added to the lane's run
// (acc = Y on entering a cell, acc += Y after); runs are flushed through the
// LDS stages of flush_runs. The row stays in registers: the LDS holds the
// stages.
//
// Run in generations as connectome_fast_kernel, where there is also room for
// the tracks cut short (three float4 each); their runs are flushed first. 97 x
// 116 x 97 SH45 Diffusion, 300k seeds, 3000 steps at most: 16.8 ms per call in
// one launch, 15.3 so. Order-8 SH Transport and Diffusion are then held to
// three waves per SIMD (168 VGPRs; 172 and two otherwise).
template <int MODEL, int ALGO, int LMAX, bool GENERATIONS>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(
    GENERATIONS && LMAX == 8 && (ALGO == ALGO_TRANSPORT || ALGO == ALGO_DIFFUSION) ? 3 : 1)))
void tod_fast_kernel(FastTodLaunch f)
{
    __shared__ RunStage stages[4];
    RunStage &stage = stages[threadIdx.x >> 6];
    const TodLaunch &t = f.tod;
    const float *coeffs = static_cast<const float *>(f.coeffs);
    const uint32_t cstride = f.coeff_stride;
    const float step = t.algo.step_size;
    const int lane_id = __lane_id();
    const bool resume = GENERATIONS && f.saved_in != nullptr;
    std::conditional_t<GENERATIONS, Generation, WholeLaunch> work(
        resume ? (uint64_t)*f.saved_in_count : (uint64_t)t.n_seeds, f.last, f.min_repack);

    int64_t g = -1;
    bool drained = false;
    uint64_t in_flight = 0;
    uint2 rng = make_uint2(0u, 0u);
    V3 point = v3(0.0f, 0.0f, 0.0f), o = point;
    uint32_t k = 0;
    int64_t previous = -1;
    int64_t field_cell = -2, cached_mask_cell = -2;
    bool mask_inside = false;
    float q[MODEL == MODEL_SH ? Order<LMAX>::TERMS : 6];
    float acc[45];
#pragma unroll
    for (int i = 0; i < 45; i++)
        acc[i] = 0.0f;

    while (true) {
        const uint64_t need = __ballot(g < 0);
        if constexpr (GENERATIONS)
            work.pending += (uint32_t)__popcll(in_flight & need);
        // Refill idle lanes, one atomic per wavefront.
        if (need != 0 && !drained) {
            const FastTodLaunch &rare = cold<ALGO>(f);
            const TodLaunch &t = rare.tod;
            const int leader = __ffsll((unsigned long long)need) - 1;
            const uint32_t wanted = (uint32_t)__popcll(need);
            uint32_t base = 0;
            if (lane_id == leader)
                base = atomicAdd(t.queue, wanted);
            base = __shfl(base, leader);
            if ((uint64_t)base + wanted >= work.n_work)
                drained = true;
            if (g < 0) {
                const uint64_t claimed = (uint64_t)base + (uint64_t)__popcll(need & ((1ull << lane_id) - 1ull));
                if (claimed < work.n_work) {
                    g = (int64_t)claimed;
                    if (resume) {
                        const float4 *slot = rare.saved_in + 3 * claimed;
                        const float4 a = slot[0], b = slot[1], c = slot[2];
                        point = v3(a.x, a.y, a.z);
                        o = v3(a.w, b.x, b.y);
                        rng = make_uint2(__float_as_uint(b.z), __float_as_uint(b.w));
                        k = __float_as_uint(c.x);
                    } else {
                        rng = rng_init(t.rng_seed, (uint32_t)g);
                        const BoundarySample sample =
                            sample_boundary(t.vertices, t.triangles, t.cumulative, t.n_triangles, rng);
                        point = sample.point;
                        o = sample.orientation;
                        k = 0;
                    }
                    previous = -1;
                    field_cell = -2;
                    cached_mask_cell = -2;
                    mask_inside = false;
                }
            }
        }
        in_flight = __ballot(g >= 0);
        if (in_flight == 0)
            break;
        if constexpr (GENERATIONS) {
            if (work.over()) {
                // Few tracks left in flight: hand this wavefront's over.
                flush_runs(g >= 0 && previous >= 0, previous, acc, t.coefficients, stage);
                const FastTodLaunch &rare = cold<ALGO>(f);
                const uint64_t slot = work.hand_over(in_flight, rare.ended, rare.saved_out_count);
                if (g >= 0) {
                    float4 *saved = rare.saved_out + 3 * slot;
                    saved[0] = make_float4(point.x, point.y, point.z, o.x);
                    saved[1] = make_float4(o.y, o.z, __uint_as_float(rng.x), __uint_as_float(rng.y));
                    saved[2] = make_float4(__uint_as_float(k), 0.0f, 0.0f, 0.0f);
                }
                break;
            }
            work.template count<ALGO>(f, drained);
        }
        const bool live = g >= 0;
        bool stop = false;
        int64_t voxel = -1, cell = -1;
        if (live) {
            stop = k >= t.n_steps;
            if (!stop) {
                const int64_t mc = mask_cell(t.mask, point);
                if (mc != cached_mask_cell) {
                    cached_mask_cell = mc;
                    mask_inside = mc >= 0 && t.mask.mask[mc] != 0;
                }
                stop = !mask_inside;
            }
            if (!stop) {
                voxel = field_voxel(t.field, point);
                stop = voxel < 0;
            }
            if (!stop)
                cell = output_cell(t.grid, point);  // -1 off the grid
        }
        // Leaving a cell (for another or for no cell) ends its run.
        flush_runs(live && !stop && previous >= 0 && cell != previous, previous, acc, t.coefficients, stage);
        if (live && !stop) {
            const bool in_grid = cell >= 0;
            // On the grid: a new run starts from the basis (keep 0) or the
            // run goes on (keep 1); off it, the run is left as it is.
            const float keep = in_grid && cell != previous ? 0.0f : 1.0f;
            previous = cell;
            fast::sh45_basis(o, in_grid ? 1.0f : 0.0f, [&](int i, float y) { acc[i] = fmaf(acc[i], keep, y); });
            if (voxel != field_cell) {
                field_cell = voxel;
                load_row<MODEL, LMAX, 0>(coeffs, voxel, cstride, q, nullptr);
            }
            o = update_orientation<MODEL, ALGO, LMAX>(t.algo, q, o, rng);
            stop = !(__builtin_isfinite(o.x) && __builtin_isfinite(o.y) && __builtin_isfinite(o.z)) ||
                   length3(o) < 0.5f;
            if (!stop) {
                point.x += step * o.x;
                point.y += step * o.y;
                point.z += step * o.z;
                k++;
            }
        }
        // The end of a track ends its run.
        const bool ended = live && stop;
        flush_runs(ended && previous >= 0, previous, acc, t.coefficients, stage);
        if (ended)
            g = -1;
    }
    if constexpr (GENERATIONS)
        work.flush(cold<ALGO>(f).ended);
}

// Clears a generation's claim counter, ended-streamline shards and
// saved-streamline count; before generation 0 also the launch's row and mask
// read totals. One block of 64 threads. Streamlines that the generation would run
// to their ends (fewer than twice min_repack, or the last generation's) go to
// track_split_fast_kernel instead where it may take them (up to split_limit):
// their buffer and number to f.tail, and none to this generation.
__global__ void zero_generation(FastLaunch f, bool first, uint32_t split_limit)
{
    const int t = threadIdx.x;
    if (t < FAST_END_SHARDS)
        f.ended[t * FAST_END_STRIDE] = 0u;
    if (t == 0) {
        *f.claims = 0u;
        if (first) {
            f.stats[0] = 0ull;
            f.stats[1] = 0ull;
            f.tail[0] = 0u;
        } else {
            const uint32_t work = *f.cont_in_count;
            if (work != 0 && work <= split_limit && (f.last || work / 2 < f.min_repack)) {
                f.tail[0] = work;
                f.tail[1] = f.cont_in == f.cont[1];
                *f.cont_in_count = 0u;
            }
        }
        *f.cont_out_count = 0u;
    }
}

__global__ void zero_product_generation(uint32_t *queue, uint32_t *ended, uint32_t *list_count)
{
    if (threadIdx.x < FAST_END_SHARDS)
        ended[threadIdx.x * FAST_END_STRIDE] = 0u;
    if (threadIdx.x == 0) {
        *queue = 0u;
        *list_count = 0u;
    }
}

// Dense seed-major rows -> ragged points. One wavefront per streamline copies
// its lengths[g] * 3 floats, coalesced on both sides, eight loads in flight
// per lane before their stores (a load-store pair per iteration left the
// copy latency-bound).
__global__ __launch_bounds__(256) void compact_seed_major_kernel(const float *__restrict__ dense, int64_t n_seeds,
                                                                 uint32_t n_points,
                                                                 const uint32_t *__restrict__ lengths,
                                                                 const int64_t *__restrict__ offsets,
                                                                 float *__restrict__ out)
{
    constexpr int UNROLL = 8;
    const int lane = threadIdx.x & 63;
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
    const int64_t capacity = n_seeds * (int64_t)n_points * 3;
    for (int64_t g = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); g < n_seeds; g += waves) {
        // Lengths are clamped to the row and writes to the output capacity,
        // whatever the caller's lengths and offsets hold: only i in [lo, hi)
        // is copied, for which 0 <= first + i < capacity.
        const int64_t count = (int64_t)min(lengths[g], n_points) * 3;
        const float *src = dense + g * (int64_t)n_points * 3;
        const int64_t first = offsets[g] * 3;
        const int64_t lo = first < 0 ? -first : 0;
        const int64_t hi = min(count, capacity - first);
        for (int64_t base = lo + lane; base < hi; base += 64 * UNROLL) {
            float v[UNROLL];
#pragma unroll
            for (int k = 0; k < UNROLL; k++) {
                const int64_t i = base + 64 * k;
                v[k] = i < hi ? src[i] : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < UNROLL; k++) {
                const int64_t i = base + 64 * k;
                if (i < hi)
                    out[first + i] = v[k];
            }
        }
    }
}

// out[v, r] = sum_i T[r, i] c[v, i] in FP64 for the SH -> polynomial map of
// order L (T row-major TERMS x TERMS in global memory, wave-uniform reads);
// coefficients past the field's K are zero, rows past TERMS of the padded
// stride are zero.
template <int L>
__global__ __launch_bounds__(256) void sh_to_poly_kernel(const float *__restrict__ field, int64_t n_voxels,
                                                         uint32_t stride, uint32_t K, const double *__restrict__ T,
                                                         float *__restrict__ out, uint32_t out_stride)
{
    constexpr int TERMS = Order<L>::TERMS;
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n_voxels)
        return;
    double c[TERMS];
#pragma unroll
    for (int i = 0; i < TERMS; i++)
        c[i] = i < (int)K ? (double)field[v * stride + i] : 0.0;
    float *dst = out + v * out_stride;
    for (int r = 0; r < TERMS; r++) {
        double acc = 0.0;
#pragma unroll
        for (int i = 0; i < TERMS; i++)
            acc += T[r * TERMS + i] * c[i];
        dst[r] = (float)acc;
    }
    for (uint32_t r = TERMS; r < out_stride; r++)
        dst[r] = 0.0f;
}

__global__ void copy_rows_kernel(const float *__restrict__ field, int64_t n_voxels, uint32_t stride,
                                 float *__restrict__ out, uint32_t out_stride)
{
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n_voxels)
        return;
    for (uint32_t r = 0; r < out_stride; r++)
        out[v * out_stride + r] = r < stride ? field[v * stride + r] : 0.0f;
}

// T[r, i]: coefficient r of the polynomial layout of order L
// (tgk_fast_model.h) per unit SH coefficient i (MRtrix order). The real
// harmonic of order m > 0 is sqrt(2) N_lm P_l^m(z) cos(m phi) (sin for -m)
// with P_l^m = (-1)^m s^m d^m P_l / dz^m and
// N_lm = sqrt((2l+1)/(4 pi) (l-m)!/(l+m)!).
template <int L> std::vector<double> sh_to_poly_matrix()
{
    using O = Order<L>;
    constexpr int TERMS = O::TERMS;
    std::vector<double> T((size_t)TERMS * TERMS, 0.0);
    for (int l = 0; l <= L; l += 2) {
        const std::vector<double> P = shb::legendre(l);
        for (int m = 0; m <= l; m++) {
            const double N = std::sqrt((2.0 * l + 1.0) / (4.0 * M_PI) * shb::factorial(l - m) / shb::factorial(l + m));
            const double F = N * (m == 0 ? 1.0 : std::sqrt(2.0)) * ((m & 1) ? -1.0 : 1.0);
            const int parity = m & 1;
            for (int side = 0; side < (m == 0 ? 1 : 2); side++) {
                const int column = l * (l + 1) / 2 + (side == 0 ? m : -m);
                const int base = side == 0 ? O::a_offset(m) : O::b_offset(m);
                for (int j = 0; j < O::poly_terms(m); j++) {
                    const int power = parity + 2 * j;
                    if (power + m > l)
                        continue;
                    const double coefficient = P[power + m] * shb::factorial(power + m) / shb::factorial(power);
                    T[(size_t)(base + j) * TERMS + column] += F * coefficient;
                }
            }
        }
    }
    return T;
}

// The map of order L on the current device, uploaded on first use and kept
// for the life of the process. Runtimes on different threads may ask for it
// at once: the first upload per device happens under a lock.
template <int L> hipError_t device_matrix(const double **out)
{
    static const double *matrices[64] = {};
    static std::mutex lock;
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess)
        return e;
    if (device < 0 || device >= 64)
        return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> guard(lock);
    if (!matrices[device]) {
        const std::vector<double> T = sh_to_poly_matrix<L>();
        void *ptr = nullptr;
        e = hipMalloc(&ptr, T.size() * sizeof(double));
        if (e != hipSuccess)
            return e;
        e = hipMemcpy(ptr, T.data(), T.size() * sizeof(double), hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            (void)hipFree(ptr);
            return e;
        }
        matrices[device] = static_cast<const double *>(ptr);
    }
    *out = matrices[device];
    return hipSuccess;
}

// Blocks of `block` threads of a kernel that fill the current device once,
// and the device's CUs, computed on first use per device (atomically
// published: runtimes on other threads may read it).
template <auto KERNEL> hipError_t fill_grid(int block, int *blocks, int *cus = nullptr)
{
    static std::atomic<uint64_t> cache[64] = {};
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess)
        return e;
    if (device < 0 || device >= 64)
        return hipErrorInvalidDevice;
    if (cache[device].load(std::memory_order_acquire) == 0) {
        int per_cu = 0;
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(KERNEL), block, 0);
        if (e != hipSuccess)
            return e;
        int count = 0;
        e = hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device);
        if (e != hipSuccess)
            return e;
        count = std::max(count, 1);
        cache[device].store((uint64_t)count << 32 | (uint32_t)(count * std::max(per_cu, 1)),
                            std::memory_order_release);
    }
    const uint64_t found = cache[device].load(std::memory_order_acquire);
    *blocks = (int)(uint32_t)found;
    if (cus)
        *cus = (int)(found >> 32);
    return hipSuccess;
}

// A^k 2^64 mod M for MWC64X (mwc64x_jump).
uint64_t jump_multiplier(uint64_t k)
{
    constexpr uint64_t A = 4294883355u, M = (A << 32) - 1;
    auto times = [](uint64_t a, uint64_t b) { return (uint64_t)((unsigned __int128)a * b % M); };
    uint64_t result = (uint64_t)(((unsigned __int128)1 << 64) % M);
    for (uint64_t power = A; k != 0; k >>= 1, power = times(power, power))
        if (k & 1)
            result = times(result, power);
    return result;
}

// Whether a launch tracks by lane groups. Probabilistic: a group's step costs
// some 500 instructions beside its candidates: with 16 candidates or fewer
// that shows once the streamlines fill the GPU one to a lane (SH45, 600k
// seeds, one lane per streamline against groups: 12.2 and 17.2 ms with 8
// candidates, 20.7 and 19.9 with 16, 35.3 and 30.7 with 32, 68.9 and 44.8
// with 64; 20k seeds: 3.9 and 2.7 with 2, 48.2 and 7.5 with 64). Past 64
// candidates a lane's share no longer fits its registers.
// Deterministic: every launch of the order-8 SH model (5k, 100k, 600k and
// 1.5M seeds: 162, 206, 339 and 648 ms one lane per streamline, 13, 32, 113
// and 257 ms by groups). Order 12 and DTI keep one lane per streamline: their
// gradients are contracted otherwise (deterministic_iteration), and the DTI
// evaluations are too short to share out (600k seeds: 47 against 64 ms).
constexpr int64_t GROUP_FEW_SEEDS = 65536;
template <int MODEL, int ALGO, int LMAX> constexpr bool groupable()
{
    return ALGO == ALGO_PROBABILISTIC || (ALGO == ALGO_DETERMINISTIC && MODEL == MODEL_SH && LMAX == 8);
}
template <int ALGO> bool grouped(const TrackLaunch &p)
{
    if (ALGO == ALGO_PROBABILISTIC)
        return p.algo.n_samples <= fast::GROUP_LANES * fast::GROUP_CANDIDATES &&
               (p.algo.n_samples > 16 || p.n_seeds <= GROUP_FEW_SEEDS);
    return true;
}

// The grid: whole blocks per CU, as many as the seeds fill and at most three
// (Probabilistic) or what fits, four (Deterministic). A launch ends with its
// longest streamline, whose steps take longer the more wavefronts share its
// SIMD, and the queue refills what ends early: 150k seeds of the 97 x 116 x
// 97 SH45 Probabilistic workload took 22.8, 17.3, 17.4 and 18.4 ms at one to
// four blocks per CU, 600k seeds 49.6, 45.0 and 45.6 ms at two to four, and
// 20k seeds (625 blocks' worth) 7.2 ms at two blocks per CU and 9.3 ms at 625
// blocks; Deterministic 50.6, 35.3, 32.4 and 32.9 ms with 100k seeds and 261,
// 154, 124 and 113 ms with 600k.
template <int ALGO> constexpr int group_blocks_per_cu() { return ALGO == ALGO_DETERMINISTIC ? 4 : 3; }
template <int MODEL, int ALGO, int DOMAIN, int LMAX>
hipError_t launch_group(const FastLaunch &f, FastPlan &plan, hipStream_t stream)
{
    int fill = 0, cus = 0;
    const hipError_t e = fill_grid<track_group_kernel<MODEL, ALGO, DOMAIN, LMAX>>(256, &fill, &cus);
    if (e != hipSuccess || plan.query)
        return e;
    plan.form = TGK_FAST_FORM_GROUPS;
    const int64_t needed = (f.track.n_seeds * fast::GROUP_LANES + 255) / 256;
    int grid_blocks = plan.tuned ? 0 : plan.grid_blocks;
    if (grid_blocks <= 0)
        grid_blocks = (int)std::min<int64_t>(std::min(fill, group_blocks_per_cu<ALGO>() * cus),
                                             std::max<int64_t>(needed / cus, 1) * cus);
    FastLaunch g = f;
    if (ALGO == ALGO_PROBABILISTIC) {
        const uint64_t per_lane = ((uint64_t)f.track.algo.n_samples + fast::GROUP_LANES - 1) / fast::GROUP_LANES;
        for (int b = 0; b < fast::GROUP_LANES; b++)
            g.group_jump[b] = jump_multiplier(2 * per_lane * b);
        g.group_jump[fast::GROUP_LANES] = jump_multiplier(2 * (uint64_t)f.track.algo.n_samples);
    }
    g.cont_out_count = f.cont_count[0];
    zero_generation<<<1, 64, 0, stream>>>(g, true, 0u);
    track_group_kernel<MODEL, ALGO, DOMAIN, LMAX>
        <<<(unsigned)std::min<int64_t>(grid_blocks, needed), 256, 0, stream>>>(g);
    return hipGetLastError();
}

// Streamlines that track_split_fast_kernel takes at most, a launch's all or
// its last ones: two wavefronts per SIMD where one lane per streamline leaves
// half the SIMDs idle. Mask domains, 145 x 174 x 145 SH45 Diffusion, one lane
// per streamline against split: 28k seeds 5.4 and 4.2 ms, the last ones of
// 100k 6.2 and 5.8, of 1M 22.5 and 21.9 (21.95 taken from 49152 on, 22.15
// from 65536); mesh domains, whose one-lane step is longer: 40k seeds 7.3 and
// 6.6 ms, the last ones of 500k 12.85 and 12.77 from 65536 on.
template <int DOMAIN> constexpr uint32_t split_lanes() { return DOMAIN == DOMAIN_MESH ? 65536 : 32768; }
// A grid, a shape other than 0 or a threshold that was set chooses the kernel
// that has them for few seeds too, unless it was set for large launches.
template <int MODEL, int ALGO, int DOMAIN, int LMAX, int S>
hipError_t launch_fast(const FastLaunch &f, FastPlan &plan, hipStream_t stream)
{
    constexpr int BLOCK = shape_block<MODEL, ALGO, LMAX, S>();
    int grid_blocks = plan.grid_blocks;
    if (grid_blocks <= 0) {
        const hipError_t e = fill_grid<track_fast_kernel<MODEL, ALGO, DOMAIN, LMAX, S>>(BLOCK, &grid_blocks);
        if (e != hipSuccess)
            return e;
    }
    plan.lanes = (int64_t)grid_blocks * BLOCK;
    if (plan.query)
        return hipSuccess;
    // Generation g resumes what g - 1 saved in cont[(g - 1) % 2] and saves
    // into cont[g % 2], whose count (generation g - 2's, consumed by g - 1)
    // it clears first.
    // A first generation that is never cut short (half its resident work
    // below the repack threshold) is the only one.
    const uint64_t first_work = std::min<uint64_t>((uint64_t)f.track.n_seeds, (uint64_t)grid_blocks * BLOCK);
    int generations = first_work / 2 >= f.min_repack ? FAST_GENERATIONS : 1;
    FastLaunch gen = f;
    constexpr bool SPLIT = shaped<MODEL, ALGO, LMAX>();
    const bool split_all = SPLIT && f.track.n_seeds <= split_lanes<DOMAIN>() &&
                           (plan.tuned || (plan.grid_blocks <= 0 && S == 0 && (generations == 1 || !plan.repack_set)));
    plan.form = split_all ? TGK_FAST_FORM_SPLIT : TGK_FAST_FORM_LANES;
    if (split_all)
        generations = 1;
    // What the last generation can be handed (see above).
    const bool split_last = SPLIT && generations > 1 &&
                            ((int64_t)grid_blocks * BLOCK >> (FAST_GENERATIONS - 1)) <= split_lanes<DOMAIN>();
    for (int g = 0; g < generations; g++) {
        gen.cont_in = g == 0 ? nullptr : f.cont[(g - 1) % 2];
        gen.cont_in_count = g == 0 ? nullptr : f.cont_count[(g - 1) % 2];
        gen.cont_out = f.cont[g % 2];
        gen.cont_out_count = f.cont_count[g % 2];
        gen.last = g == generations - 1;
        const uint32_t split_limit = !SPLIT ? 0u : gen.last && split_last ? 0xffffffffu : split_lanes<DOMAIN>();
        zero_generation<<<1, 64, 0, stream>>>(gen, g == 0, split_limit);
        const int blocks_g = std::max(1, grid_blocks >> g);
        if (!split_all && !(gen.last && split_last))
            track_fast_kernel<MODEL, ALGO, DOMAIN, LMAX, S><<<blocks_g, BLOCK, 0, stream>>>(gen);
    }
    if constexpr (SPLIT) {
        if (split_all || generations > 1) {
            gen.cont_in = split_all ? nullptr : f.cont[0];
            track_split_fast_kernel<ALGO, DOMAIN>
                <<<(unsigned)((std::min<uint64_t>(first_work, split_lanes<DOMAIN>()) + 63) / 64), 64 * FAST_SPLIT_WAVES, 0,
                   stream>>>(gen);
        }
    }
    return hipGetLastError();
}

// By lane groups where they track, else one lane per streamline.
template <int MODEL, int ALGO, int DOMAIN, int LMAX, int S>
hipError_t launch_tracks(const FastLaunch &f, FastPlan &plan, hipStream_t stream)
{
    if constexpr (groupable<MODEL, ALGO, LMAX>()) {
        // Queried for every launch: a later one may be grouped.
        if (plan.query || grouped<ALGO>(f.track)) {
            const hipError_t e = launch_group<MODEL, ALGO, DOMAIN, LMAX>(f, plan, stream);
            if (e != hipSuccess || !plan.query)
                return e;
        }
        if constexpr (ALGO == ALGO_DETERMINISTIC)
            return hipSuccess;  // plan.lanes = 0: groups save no streamlines
    }
    if constexpr (!groupable<MODEL, ALGO, LMAX>() || ALGO != ALGO_DETERMINISTIC)
        return launch_fast<MODEL, ALGO, DOMAIN, LMAX, S>(f, plan, stream);
}

template <int MODEL, int ALGO, int DOMAIN>
hipError_t launch_fast_order(const FastLaunch &f, FastPlan &plan, hipStream_t stream)
{
    if constexpr (MODEL == MODEL_SH) {
        if (f.sh_order == 12)
            return launch_tracks<MODEL, ALGO, DOMAIN, 12, 0>(f, plan, stream);
    }
    if constexpr (shaped<MODEL, ALGO, 8>()) {
        switch (f.shape) {
        case 1: return launch_tracks<MODEL, ALGO, DOMAIN, 8, 1>(f, plan, stream);
        case 2: return launch_tracks<MODEL, ALGO, DOMAIN, 8, 2>(f, plan, stream);
        case 3: return launch_tracks<MODEL, ALGO, DOMAIN, 8, 3>(f, plan, stream);
        case 4: return launch_tracks<MODEL, ALGO, DOMAIN, 8, 4>(f, plan, stream);
        default: break;
        }
    }
    return launch_tracks<MODEL, ALGO, DOMAIN, 8, 0>(f, plan, stream);
}

template <int MODEL, int ALGO>
hipError_t launch_fast_domain(const FastLaunch &f, FastPlan &plan, hipStream_t stream)
{
    if (f.track.domain_kind == DOMAIN_MESH)
        return launch_fast_order<MODEL, ALGO, DOMAIN_MESH>(f, plan, stream);
    return launch_fast_order<MODEL, ALGO, DOMAIN_MASK>(f, plan, stream);
}

template <int MODEL>
hipError_t launch_fast_algo(const FastLaunch &f, FastPlan &plan, hipStream_t stream)
{
    switch (f.track.algo.algorithm) {
    case ALGO_DIFFUSION: return launch_fast_domain<MODEL, ALGO_DIFFUSION>(f, plan, stream);
    case ALGO_PROBABILISTIC: return launch_fast_domain<MODEL, ALGO_PROBABILISTIC>(f, plan, stream);
    case ALGO_DETERMINISTIC: return launch_fast_domain<MODEL, ALGO_DETERMINISTIC>(f, plan, stream);
    default: return launch_fast_domain<MODEL, ALGO_TRANSPORT>(f, plan, stream);
    }
}

hipError_t dispatch_fast(const FastLaunch &f, FastPlan &plan, hipStream_t stream)
{
    if (f.track.algo.model == MODEL_DTI)
        return launch_fast_algo<MODEL_DTI>(f, plan, stream);
    return launch_fast_algo<MODEL_SH>(f, plan, stream);
}

// Whether a connectome or TOD launch of the SH model, `lanes` tracks at a
// time, runs in generations: where half its lanes, and half of those, still
// fill wavefronts for half the SIMDs, and where tracks are long. Packing lanes
// costs 0.2 to 0.4 ms a launch. Tracks that soon leave a small grid, or that
// most lanes take to a low limit, leave less than that to gain: 135k to 300k
// SH28 Transport and SH45 Diffusion tracks ran at 0.88 to 1.05 of the speed of
// one generation where at most 200 to 800 steps cross the mask's grid or are
// taken, and at 0.99 to 1.24 from 850 on; 40k to 100k tracks at 0.83 to 1.00.
// In connectomes a step of many Probabilistic candidates takes so long that a
// limit of 300 steps suffices (135k and 200k tracks: 0.91 to 0.97 with 160,
// 1.00 to 1.63 with 320 to 1200). Deterministic launches always run in one:
// their lanes iterate one by one, and packed they wait for more of the others
// (135k and 200k tracks: 0.75 to 1.34, with no order in it).
template <int MODEL, int ALGO> constexpr bool cut_short()
{
    return MODEL == MODEL_SH && ALGO != ALGO_DETERMINISTIC;
}
bool in_generations(const MaskView &mask, const AlgoParams &a, uint32_t n_steps, int64_t lanes, bool many_candidates)
{
    constexpr double LONG_TRACK = 840.0;
    if (lanes < 4 * (int64_t)FAST_MIN_REPACK_PRODUCT)
        return false;
    if (many_candidates && n_steps >= 300)
        return true;
    const float *m = mask.inv;
    const double det = (double)m[0] * ((double)m[5] * m[10] - (double)m[6] * m[9]) -
                       (double)m[1] * ((double)m[4] * m[10] - (double)m[6] * m[8]) +
                       (double)m[2] * ((double)m[4] * m[9] - (double)m[5] * m[8]);
    const double edge = std::cbrt((double)mask.dims[0] * mask.dims[1] * mask.dims[2] / std::fabs(det));
    return std::min((double)n_steps, edge / a.step_size) >= LONG_TRACK;
}

// Connectome launches: the persistent grid of the kernel's occupancy
// (cached per device), at most one lane per seed, then the hits pass. Launches
// in one generation (DTI always, as track launches) run the kernel without the
// counting.
template <int MODEL, int ALGO, int LMAX>
hipError_t launch_connectome_fast_kernel(const FastConnectomeLaunch &f, hipStream_t stream)
{
    constexpr int BLOCK = fast_block<LMAX>();
    const int64_t n = f.connectome.n_seeds, needed = (n + BLOCK - 1) / BLOCK;
    int fill = 0;
    FastConnectomeLaunch gen = f;
    int generations = 0;
    if constexpr (cut_short<MODEL, ALGO>()) {
        if (const hipError_t e = fill_grid<connectome_fast_kernel<MODEL, ALGO, LMAX, true>>(BLOCK, &fill))
            return e;
        const int64_t blocks = std::min<int64_t>(fill, needed);
        gen.min_repack = FAST_MIN_REPACK_PRODUCT;
        if (in_generations(f.connectome.mask, f.connectome.algo, f.connectome.n_steps, std::min(n, blocks * BLOCK),
                           ALGO == ALGO_PROBABILISTIC && f.connectome.algo.n_samples > 16))
            generations = FAST_GENERATIONS;
        uint32_t *const lists[2] = {reinterpret_cast<uint32_t *>(f.connectome.cols),
                                    reinterpret_cast<uint32_t *>(f.connectome.cols) + n};
        for (int g = 0; g < generations; g++) {
            gen.list_in = g == 0 ? nullptr : lists[(g - 1) % 2];
            gen.list_in_count = f.list_counts + (g + 1) % 2;
            gen.list_out = lists[g % 2];
            gen.list_out_count = f.list_counts + g % 2;
            gen.last = g == generations - 1;
            zero_product_generation<<<1, 64, 0, stream>>>(f.connectome.queue, f.ended, gen.list_out_count);
            connectome_fast_kernel<MODEL, ALGO, LMAX, true>
                <<<(unsigned)std::max<int64_t>(1, blocks >> g), BLOCK, 0, stream>>>(gen);
        }
    }
    if (generations == 0) {
        if (const hipError_t e = fill_grid<connectome_fast_kernel<MODEL, ALGO, LMAX, false>>(BLOCK, &fill))
            return e;
        zero_product_generation<<<1, 64, 0, stream>>>(f.connectome.queue, f.ended, f.list_counts);
        connectome_fast_kernel<MODEL, ALGO, LMAX, false>
            <<<(unsigned)std::min<int64_t>(fill, needed), BLOCK, 0, stream>>>(gen);
    }
    if (const hipError_t e = hipGetLastError())
        return e;
    return launch_connectome_hits(f.connectome, stream);
}

template <int MODEL, int ALGO>
hipError_t launch_connectome_fast_order(const FastConnectomeLaunch &f, hipStream_t stream)
{
    if constexpr (MODEL == MODEL_SH) {
        if (f.sh_order == 12)
            return launch_connectome_fast_kernel<MODEL, ALGO, 12>(f, stream);
    }
    return launch_connectome_fast_kernel<MODEL, ALGO, 8>(f, stream);
}

template <int MODEL>
hipError_t launch_connectome_fast_algo(const FastConnectomeLaunch &f, hipStream_t stream)
{
    switch (f.connectome.algo.algorithm) {
    case ALGO_DIFFUSION: return launch_connectome_fast_order<MODEL, ALGO_DIFFUSION>(f, stream);
    case ALGO_PROBABILISTIC: return launch_connectome_fast_order<MODEL, ALGO_PROBABILISTIC>(f, stream);
    case ALGO_DETERMINISTIC: return launch_connectome_fast_order<MODEL, ALGO_DETERMINISTIC>(f, stream);
    default: return launch_connectome_fast_order<MODEL, ALGO_TRANSPORT>(f, stream);
    }
}

// TOD launches: as connectome launches, in generations where there is room
// for the tracks cut short (at most half the lanes).
template <int MODEL, int ALGO, int LMAX> hipError_t launch_tod_fast_kernel(const FastTodLaunch &f, hipStream_t stream)
{
    const int64_t n = f.tod.n_seeds, needed = (n + 255) / 256;
    int fill = 0;
    FastTodLaunch gen = f;
    if constexpr (cut_short<MODEL, ALGO>()) {
        if (const hipError_t e = fill_grid<tod_fast_kernel<MODEL, ALGO, LMAX, true>>(256, &fill))
            return e;
        const int64_t blocks = std::min<int64_t>(fill, needed), lanes = std::min(n, blocks * 256);
        gen.min_repack = FAST_MIN_REPACK_PRODUCT;
        if ((uint64_t)(lanes / 2) <= f.saved_room &&
            in_generations(f.tod.mask, f.tod.algo, f.tod.n_steps, lanes, false)) {
            for (int g = 0; g < FAST_GENERATIONS; g++) {
                gen.saved_in = g == 0 ? nullptr : f.saved[(g - 1) % 2];
                gen.saved_in_count = f.saved_counts + (g + 1) % 2;
                gen.saved_out = f.saved[g % 2];
                gen.saved_out_count = f.saved_counts + g % 2;
                gen.last = g == FAST_GENERATIONS - 1;
                zero_product_generation<<<1, 64, 0, stream>>>(f.tod.queue, f.ended, gen.saved_out_count);
                tod_fast_kernel<MODEL, ALGO, LMAX, true>
                    <<<(unsigned)std::max<int64_t>(1, blocks >> g), 256, 0, stream>>>(gen);
            }
            return hipGetLastError();
        }
    }
    if (const hipError_t e = fill_grid<tod_fast_kernel<MODEL, ALGO, LMAX, false>>(256, &fill))
        return e;
    zero_product_generation<<<1, 64, 0, stream>>>(f.tod.queue, f.ended, f.saved_counts);
    tod_fast_kernel<MODEL, ALGO, LMAX, false><<<(unsigned)std::min<int64_t>(fill, needed), 256, 0, stream>>>(gen);
    return hipGetLastError();
}

template <int MODEL, int ALGO>
hipError_t launch_tod_fast_order(const FastTodLaunch &f, hipStream_t stream)
{
    if constexpr (MODEL == MODEL_SH) {
        if (f.sh_order == 12)
            return launch_tod_fast_kernel<MODEL, ALGO, 12>(f, stream);
    }
    return launch_tod_fast_kernel<MODEL, ALGO, 8>(f, stream);
}

template <int MODEL>
hipError_t launch_tod_fast_algo(const FastTodLaunch &f, hipStream_t stream)
{
    switch (f.tod.algo.algorithm) {
    case ALGO_DIFFUSION: return launch_tod_fast_order<MODEL, ALGO_DIFFUSION>(f, stream);
    case ALGO_PROBABILISTIC: return launch_tod_fast_order<MODEL, ALGO_PROBABILISTIC>(f, stream);
    case ALGO_DETERMINISTIC: return launch_tod_fast_order<MODEL, ALGO_DETERMINISTIC>(f, stream);
    default: return launch_tod_fast_order<MODEL, ALGO_TRANSPORT>(f, stream);
    }
}

}  // namespace

hipError_t launch_track_fast(const FastLaunch &f, FastPlan &plan, hipStream_t stream)
{
    if (f.track.n_seeds == 0 && !plan.query)
        return hipSuccess;
    if (f.track.n_seeds >= (int64_t)1 << 31)
        return hipErrorInvalidValue;
    return dispatch_fast(f, plan, stream);
}

hipError_t launch_connectome_fast(const FastConnectomeLaunch &f, hipStream_t stream)
{
    if (f.connectome.n_seeds == 0)
        return hipSuccess;
    if (f.connectome.algo.model == MODEL_DTI)
        return launch_connectome_fast_algo<MODEL_DTI>(f, stream);
    return launch_connectome_fast_algo<MODEL_SH>(f, stream);
}

hipError_t launch_tod_fast(const FastTodLaunch &f, hipStream_t stream)
{
    if (f.tod.n_seeds == 0)
        return hipSuccess;
    if (f.tod.algo.model == MODEL_DTI)
        return launch_tod_fast_algo<MODEL_DTI>(f, stream);
    return launch_tod_fast_algo<MODEL_SH>(f, stream);
}

hipError_t launch_compact_seed_major(const float *dense, int64_t n_seeds, uint32_t n_points,
                                     const uint32_t *lengths, const int64_t *offsets, float *out,
                                     hipStream_t stream)
{
    if (n_seeds == 0)
        return hipSuccess;
    const int64_t blocks = (n_seeds + 3) / 4;
    compact_seed_major_kernel<<<(unsigned)(blocks < 65536 ? blocks : 65536), 256, 0, stream>>>(
        dense, n_seeds, n_points, lengths, offsets, out);
    return hipGetLastError();
}

hipError_t launch_field_transform(const float *field, int64_t n_voxels, uint32_t stride, int32_t model, int32_t K,
                                  int32_t sh_order, void *out, uint32_t out_stride, hipStream_t stream)
{
    if (n_voxels == 0)
        return hipSuccess;
    const unsigned blocks = (unsigned)((n_voxels + 255) / 256);
    if (model == MODEL_SH) {
        const double *T = nullptr;
        hipError_t e = sh_order == 12 ? device_matrix<12>(&T) : device_matrix<8>(&T);
        if (e != hipSuccess)
            return e;
        if (sh_order == 12)
            sh_to_poly_kernel<12><<<blocks, 256, 0, stream>>>(field, n_voxels, stride, (uint32_t)K, T,
                                                              static_cast<float *>(out), out_stride);
        else
            sh_to_poly_kernel<8><<<blocks, 256, 0, stream>>>(field, n_voxels, stride, (uint32_t)K, T,
                                                             static_cast<float *>(out), out_stride);
    } else {
        copy_rows_kernel<<<blocks, 256, 0, stream>>>(field, n_voxels, stride, static_cast<float *>(out), out_stride);
    }
    return hipGetLastError();
}

}  // namespace tgk
