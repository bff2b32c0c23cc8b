// Device kernels of the near-field direct path, hand-written for gfx950.
//
//   k_gather_sinks / k_gather_sources   pencil gathers from device-resident
//       PosXYZ slabs into padded float4 pencil streams (the device-side form of
//       SinkPencilPlan/SourcePencilPlan::copy_into_pinned_memory,
//       PencilPlan.cc:22-90, 214-255), plus a bounding box per 64-source block.
//   k_gather_sources_binned  the batched path's source stream: each cell's
//       particles in x-bin order, FP64 cell offsets, block boxes.
//   k_plain      one 64-sink block per workgroup, one launch per SIC: the
//       structure of ComputeDirects (PencilKernel.cu:97-189) with the
//       reference's pair forms (DirectGPUKernels.cuh) and BLOCK_ACCUM tiles.
//   k_coadd_plain  FP32 co-add of the W partials per sink in the reference's
//       k order (PencilPlan.cc:140-207 as driven by PencilTask.cu:237-247).
//   k_batched    persistent kernel draining work queues dealt from a list sorted by cost;
//       FP32 tile sums accumulated into FP64 per-pencil partials.
//   k_coadd_f64  FP64 reduction of the W partials per sink.
//
// Pair kernel, all forms: d = source - sink, a -= g(r) d, w += max(0, b2 - r^2).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "nf_internal.h"

namespace nf {
namespace {

constexpr int kWave = 64;
constexpr float kFar = 1.0e30f;  // x of a padding source: its pair terms are exact zeros

// Read-only data of a launch is addressed through the constant address space:
// the backend then loads wave-uniform addresses with scalar loads (s_load)
// and divergent ones with global loads, even when the pointer itself came
// from memory (the SIC view table) rather than from a kernel argument.
// (The qualifiers exist only in the device compilation pass of this file.)
#if defined(__HIP_DEVICE_COMPILE__)
#define NF_CONST __attribute__((address_space(4)))
#define NF_GLOBAL __attribute__((address_space(1)))
#else
#define NF_CONST
#define NF_GLOBAL
#endif
template <typename T>
__device__ __forceinline__ const NF_CONST T *cptr(const void *p) {
    return (const NF_CONST T *)(p);
}

// Transcendentals at raised wave priority.  gfx950 issues plain FP32 VALU
// instructions of two waves of a SIMD together (16 v_mul_f32 of VGPRs take 37
// cycles with 8 waves, 2.3 each; 4.3 each when every one reads an SGPR), but
// after a v_rsq_f32 that the arbiter interleaves with other waves the SIMD
// falls back to one instruction per 4 cycles: v_rsq + 11 v_mul take 53 cycles.
// s_setprio around it keeps the pairing: a pair of 11 VALU instructions and a
// v_rsq takes 34-37 cycles instead of 41-54.  The s_setprio after it is also
// the wait state that a VALU use of a transcendental's result needs.
#if defined(__HIP_DEVICE_COMPILE__)
#define NF_TRANS1(op, a) asm("s_setprio 3\n\t" op " %0, %0\n\ts_setprio 0" : "+v"(a))
#define NF_TRANS2(op, a, b) asm("s_setprio 3\n\t" op " %0, %0\n\t" op " %1, %1\n\ts_setprio 0" : "+v"(a), "+v"(b))
#else
#define NF_TRANS1(op, a) (void)(a)
#define NF_TRANS2(op, a, b) (void)(a), (void)(b)
#endif
__device__ __forceinline__ float sqrt_(float x) {
    NF_TRANS1("v_sqrt_f32", x);
    return x;
}
__device__ __forceinline__ float rcp(float x) {
    NF_TRANS1("v_rcp_f32", x);
    return x;
}
__device__ __forceinline__ float clamp01(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, 1.0f); }

// A SIC's counts: from device memory when it was planned on the device
// without a host round trip (its host-side fields are then bounds), else
// the host's.  plan_bad: its launch group holds a cell outside its slab.
__device__ __forceinline__ bool plan_bad(const DevPlan &pl) { return pl.dbad && *cptr<int32_t>(pl.dbad) != 0; }
__device__ __forceinline__ int sink_blocks(const DevPlan &pl) {
    return pl.dtot ? (int)cptr<GPlanTotals>(pl.dtot)->sink_blocks : pl.nsink_blocks;
}
__device__ __forceinline__ int src_blocks(const DevPlan &pl) {
    return pl.dtot ? (int)cptr<GPlanTotals>(pl.dtot)->source_blocks : pl.nsrc_blocks;
}
__device__ __forceinline__ int coadd_chunks(const DevPlan &pl) {
    return pl.dtot ? (int)cptr<GPlanTotals>(pl.dtot)->chunks : pl.n_coadd_chunks;
}

// ---------------------------------------------------------------------------
// Gathers
// ---------------------------------------------------------------------------

// Particle i of a pencil: its cell c (pre[c] <= i < pre[c+1]) and slab index,
// by selects over the wave-uniform plan p.  False past the pencil's last.
template <typename Plan>
__device__ __forceinline__ bool plan_cell(const Plan &p, int W, int i, int &c, uint64_t &idx) {
    uint32_t start = p.cell[0].start;
    int pre = 0, total = 0;
    c = 0;
#pragma unroll
    for (int cc = 0; cc < NF_MAX_WIDTH; cc++) {
        if (cc >= W) break;
        const bool in = i >= total;
        c = in ? cc : c;
        pre = in ? total : pre;
        start = in ? p.cell[cc].start : start;
        total += p.cell[cc].N;
    }
    idx = (uint64_t)start + (uint64_t)(i - pre);
    return i < total;
}

// Position of particle idx of a slab of n particles: PosXYZ (X|Y|Z) or, with
// aos, posstruct (x,y,z interleaved).
__device__ __forceinline__ float3 slab_xyz(const float *P, uint64_t n, uint64_t idx, int aos) {
    if (aos) return make_float3(P[3 * idx], P[3 * idx + 1], P[3 * idx + 2]);
    return make_float3(P[idx], P[n + idx], P[2 * n + idx]);
}

// Padded blocks per wave of the plain path's gathers (blocks, not pencils, so
// that a heavy pencil spreads over many waves): a block's chain of
// dependent loads (its parent pencil, the pencil's plan, then the positions) is
// short on work, so four go side by side.  The parents and plans are wave
// uniform and come by scalar loads; with them in vector registers and the cell
// found by a loop, a SIC of a 256^3 box took 38 us (sources) and 34 us (sinks)
// where it now takes 13.8 and 8.1 us, 2.7 and 3.6 TB/s.  (One or two blocks a
// wave: the same.)
constexpr int kGatherBlocks = 4;

__global__ __launch_bounds__(256) void k_gather_sinks(DevPlan pl, const float *__restrict__ slab, uint64_t n,
                                                      int aos, float4 *__restrict__ out, float cellsize) {
    const int b0 = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (int)(threadIdx.x / kWave)) * kGatherBlocks;
    const int nsb = sink_blocks(pl);
    if (b0 >= nsb || plan_bad(pl)) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int W = pl.W;
    int par[kGatherBlocks];
#pragma unroll
    for (int u = 0; u < kGatherBlocks; u++) par[u] = cptr<int32_t>(pl.parent)[min(b0 + u, nsb - 1)];
    uint64_t idx[kGatherBlocks];
    int dcell[kGatherBlocks];
    bool live[kGatherBlocks];
#pragma unroll
    for (int u = 0; u < kGatherBlocks; u++) {
        const int s = par[u];
        const nf_sink_plan p = cptr<nf_sink_plan>(pl.sink_plan)[s];
        const int i = (b0 + u) * kWave - cptr<int32_t>(pl.sink_set_start)[s] + lane;  // index within the pencil
        int c;
        live[u] = plan_cell(p, W, i, c, idx[u]) && b0 + u < nsb;
        dcell[u] = c - pl.R;
    }
    float3 q[kGatherBlocks];
#pragma unroll
    for (int u = 0; u < kGatherBlocks; u++)
        q[u] = live[u] ? slab_xyz(slab, n, idx[u], aos) : make_float3(0.f, 0.f, 0.f);
#pragma unroll
    for (int u = 0; u < kGatherBlocks; u++) {
        if (b0 + u >= nsb) break;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (live[u]) {
            float z = q[u].z;
            const float dz = (float)dcell[u] * cellsize;  // PencilPlan.cc:43-50: FLOAT, added if nonzero
            if (dz != 0.f) z = z + dz;
            v = make_float4(q[u].x, q[u].y, z, 0.f);
        }
        out[(int64_t)(b0 + u) * kWave + lane] = v;
    }
}

__device__ __forceinline__ const float *slab_ptr(const DevSlabs &sl, int c) {
    return c == 0 ? sl.pos[0] : c == 1 ? sl.pos[1] : c == 2 ? sl.pos[2] : c == 3 ? sl.pos[3] : sl.pos[4];
}
__device__ __forceinline__ uint64_t slab_n(const DevSlabs &sl, int c) {
    return c == 0 ? sl.n[0] : c == 1 ? sl.n[1] : c == 2 ? sl.n[2] : c == 3 ? sl.n[3] : sl.n[4];
}

// Wave-wide min / max (every lane of the wave active), wave-uniform result:
// four DPP steps leave each 16-lane row's extremum in all its lanes
// (quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror, row_mirror), then
// the four rows' values are read out.  No LDS round trips, unlike a
// __shfl_xor butterfly (ds_bpermute per step).
template <bool MAX, int CTRL>
__device__ __forceinline__ float dpp_step(float v) {
    const int x = __builtin_bit_cast(int, v);
    const float u = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(x, x, CTRL, 0xF, 0xF, false));
    return MAX ? fmaxf(v, u) : fminf(v, u);
}
template <bool MAX>
__device__ __forceinline__ float wave_reduce(float v) {
    v = dpp_step<MAX, 0xB1>(v);   // quad_perm [1,0,3,2]
    v = dpp_step<MAX, 0x4E>(v);   // quad_perm [2,3,0,1]
    v = dpp_step<MAX, 0x141>(v);  // row_half_mirror
    v = dpp_step<MAX, 0x140>(v);  // row_mirror
    const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 0));
    const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 16));
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 32));
    const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 48));
    return MAX ? fmaxf(fmaxf(r0, r1), fmaxf(r2, r3)) : fminf(fminf(r0, r1), fminf(r2, r3));
}
__device__ __forceinline__ float wave_min(float v) { return wave_reduce<false>(v); }
__device__ __forceinline__ float wave_max(float v) { return wave_reduce<true>(v); }

// Plain-path source stream, in the reference's order.  One wave per
// kGatherBlocks padded 64-source blocks; it writes each block and its
// bounding box (padding excluded): box[2b] = min, box[2b+1] = max.
__global__ __launch_bounds__(256) void k_gather_sources(DevPlan pl, DevSlabs sl, float4 *__restrict__ out,
                                                        float4 *__restrict__ box, float cellsize) {
    const int b0 = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (int)(threadIdx.x / kWave)) * kGatherBlocks;
    const int nqb = src_blocks(pl);
    if (b0 >= nqb || plan_bad(pl)) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int W = pl.W;
    int par[kGatherBlocks];
#pragma unroll
    for (int u = 0; u < kGatherBlocks; u++) par[u] = cptr<int32_t>(pl.src_parent)[min(b0 + u, nqb - 1)];
    uint64_t idx[kGatherBlocks];
    int cc[kGatherBlocks];
    bool live[kGatherBlocks];
#pragma unroll
    for (int u = 0; u < kGatherBlocks; u++) {
        const int s = max(par[u], 0);  // a block no pencil covers (s < 0) is never read: left unwritten
        const nf_source_plan p = cptr<nf_source_plan>(pl.src_plan)[s];
        const int i = (b0 + u) * kWave - cptr<int32_t>(pl.src_set_start)[s] + lane;
        live[u] = plan_cell(p, W, i, cc[u], idx[u]) && b0 + u < nqb && par[u] >= 0;
    }
    float3 q[kGatherBlocks];
#pragma unroll
    for (int u = 0; u < kGatherBlocks; u++)
        q[u] = live[u] ? slab_xyz(slab_ptr(sl, cc[u]), slab_n(sl, cc[u]), idx[u], sl.aos)
                       : make_float3(0.f, 0.f, 0.f);
    const float inf = __builtin_huge_valf();
#pragma unroll
    for (int u = 0; u < kGatherBlocks; u++) {
        const int b = b0 + u;
        if (b >= nqb) break;
        if (par[u] < 0) continue;
        float4 v = make_float4(kFar, 0.f, 0.f, 0.f);
        const bool real = live[u];
        if (real) {
            float x = q[u].x;
            const float dx = (float)(cc[u] - pl.R) * cellsize;  // PencilPlan.cc:226-238
            if (dx != 0.f) x = x + dx;
            v = make_float4(x, q[u].y, q[u].z, 0.f);
        }
        out[(int64_t)b * kWave + lane] = v;
        const float mnx = wave_min(real ? v.x : inf), mny = wave_min(real ? v.y : inf),
                    mnz = wave_min(real ? v.z : inf);
        const float mxx = wave_max(real ? v.x : -inf), mxy = wave_max(real ? v.y : -inf),
                    mxz = wave_max(real ? v.z : -inf);
        if (lane == 0) {
            box[2 * (int64_t)b] = make_float4(mnx, mny, mnz, 0.f);
            box[2 * (int64_t)b + 1] = make_float4(mxx, mxy, mxz, 0.f);
        }
    }
}

// Batched-path source stream.  Each cell's particles are ordered by
// kXBins equal x-bins of the cell (a stable counting sort: within a bin
// the reference's order), so a 64-source block that straddles two cells
// takes an x-slice of each rather than all of one: tighter block boxes, so
// more sink-block/source-block pairs clear the softening and density radii
// and run the fast pair form.  Cells above kBinnedCellMax = 128 particles
// keep the reference's order: a replay of the mode split on a clustered box
// gained little from sorting them.
// Cell offsets are added in FP64 (x + dc/cpd, rounded once).
//
// A wave fills a range of a pencil's 64-source blocks: it loads each binned
// cell that reaches into the range once (two 64-particle chunks each, all
// cells' loads in flight together), ranks every particle within its cell
// (ballots per bin), writes the ones whose slots fall in the range, and
// reduces the box of each block of the range over the particles that land
// in it (the pencil's slots run cell after cell, so its blocks are met in
// order).  The last block's padding slots take kFar.
//
// One wave per source pencil fills the pencil's first kSegBlocks blocks;
// one wave per kSegBlocks blocks of the stream fills the blocks that lie
// beyond the first kSegBlocks of their pencil.  So every block is written
// by one wave, and a pencil of large cells (a clustered box's halos put
// thousands of particles in a cell) spreads over many waves instead of
// holding one for the whole launch.
constexpr int kXBins = 8;
constexpr int kBinnedCellMax = 2 * kWave;
constexpr int kSegBlocks = kGatherSegBlocks;

__device__ __forceinline__ int xbin(float x, float cpdf) {  // x cell-centred; out-of-cell x clamps
    const float t = floorf((x * cpdf + 0.5f) * (float)kXBins);
    return (int)fminf(fmaxf(t, 0.f), (float)(kXBins - 1));
}
__device__ __forceinline__ uint64_t ballot(bool p) { return __builtin_amdgcn_ballot_w64(p); }
__device__ __forceinline__ int lanes_below(uint64_t m) {  // set bits of m below this lane
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// The box of the block being filled: each lane's running min/max over its
// sources in the block, reduced across the wave once, when the next block
// starts or the pencil ends.
struct BlockBox {
    int open = -1;
    float mn[3], mx[3];
    __device__ __forceinline__ void reset() {
        mn[0] = mn[1] = mn[2] = __builtin_huge_valf();
        mx[0] = mx[1] = mx[2] = -__builtin_huge_valf();
    }
    // Make b the open block (b >= open; the pencil's blocks are met in order).
    __device__ __forceinline__ void to(int b, float4 *box, int64_t gb0, int lane) {
        if (b == open) return;
        flush(box, gb0, lane);
        open = b;
        reset();
    }
    __device__ __forceinline__ void add(bool in, float x, float y, float z) {
        if (!in) return;
        mn[0] = fminf(mn[0], x), mn[1] = fminf(mn[1], y), mn[2] = fminf(mn[2], z);
        mx[0] = fmaxf(mx[0], x), mx[1] = fmaxf(mx[1], y), mx[2] = fmaxf(mx[2], z);
    }
    __device__ __forceinline__ void flush(float4 *box, int64_t gb0, int lane) {
        if (open < 0) return;
        const float4 lo = make_float4(wave_min(mn[0]), wave_min(mn[1]), wave_min(mn[2]), 0.f);
        const float4 hi = make_float4(wave_max(mx[0]), wave_max(mx[1]), wave_max(mx[2]), 0.f);
        if (lane == 0) {
            box[2 * (gb0 + open)] = lo;
            box[2 * (gb0 + open) + 1] = hi;
        }
    }
};

// A pencil of at most one block (total <= 64 sources): a source to a lane, all
// cells at once.  A lane's rank among its cell's lanes comes from the same 8
// ballots, cut down to the cell: 100 instructions instead of 5 x 70 and one
// load instead of one after the other per cell.  A launch group of sparse SICs
// (129^2 pencils of 25 sources each): 105 -> 52 us on average.
__device__ __forceinline__ void gather_small_pencil(const DevPlan &pl, const DevSlabs &sl, const nf_source_plan &p,
                                                    const int *pre, int total, float4 *__restrict__ dst,
                                                    float4 *__restrict__ box, float cpdf, double invcpd, int lane) {
    int c = 0, first = 0, next = pre[1];
    uint32_t start = p.cell[0].start;
    const float *P = sl.pos[0];
    uint64_t ns = sl.n[0];
#pragma unroll
    for (int k = 1; k < NF_MAX_WIDTH; k++) {
        const bool in = lane >= pre[k] && pre[k + 1] > pre[k];
        c = in ? k : c;
        first = in ? pre[k] : first;
        next = in ? pre[k + 1] : next;
        start = in ? p.cell[k].start : start;
        P = in ? sl.pos[k] : P;
        ns = in ? sl.n[k] : ns;
    }
    const bool live = lane < total;
    const float3 q = live ? slab_xyz(P, ns, (uint64_t)start + (uint64_t)(lane - first), sl.aos)
                          : make_float3(0.f, 0.f, 0.f);
    const int bin = live ? xbin(q.x, cpdf) : -1;
    const int n = next - first;
    const uint64_t cell = (n >= kWave ? ~0ull : (1ull << n) - 1) << first;
    const uint64_t below = cell & ((1ull << lane) - 1);
    int rank = 0;
#pragma unroll
    for (int k = 0; k < kXBins; k++) {
        const uint64_t m = ballot(bin == k);
        rank += __builtin_popcountll(m & (k < bin ? cell : k == bin ? below : 0ull));
    }
    const float x = (float)((double)q.x + (double)(c - pl.R) * invcpd);
    dst[live ? first + rank : lane] = live ? make_float4(x, q.y, q.z, 0.f) : make_float4(kFar, 0.f, 0.f, 0.f);
    const float inf = __builtin_huge_valf();
    const float4 lo = make_float4(wave_min(live ? x : inf), wave_min(live ? q.y : inf), wave_min(live ? q.z : inf), 0.f);
    const float4 hi =
        make_float4(wave_max(live ? x : -inf), wave_max(live ? q.y : -inf), wave_max(live ? q.z : -inf), 0.f);
    if (lane == 0) {
        box[0] = lo;
        box[1] = hi;
    }
}

// Blocks [blo, bhi) of pencil s (pencil-relative; bhi may pass its end);
// RANGED false: the whole pencil, without the range tests.
template <bool RANGED>
__device__ __forceinline__ void gather_pencil_binned(const DevPlan &pl, const DevSlabs &sl, float4 *__restrict__ out,
                                                     float4 *__restrict__ box, float cpdf, double invcpd, int s,
                                                     int lane, int blo, int bhi) {
    const int W = pl.W;
    const nf_source_plan p = cptr<nf_source_plan>(pl.src_plan)[s];
    int pre[NF_MAX_WIDTH + 1];
    pre[0] = 0;
#pragma unroll
    for (int c = 0; c < NF_MAX_WIDTH; c++) pre[c + 1] = pre[c] + (c < W ? p.cell[c].N : 0);
    const int total = pre[NF_MAX_WIDTH];
    // the slots to fill
    const int lo = RANGED ? blo * kWave : 0, hi = !RANGED || bhi >= (total + kWave - 1) / kWave ? total : bhi * kWave;
    if (lo >= hi) return;
    const int start = cptr<int32_t>(pl.src_set_start)[s];  // the pencil's first slot, a multiple of 64
    float4 *dst = out + start;
    const int64_t gb0 = start / kWave;
    if (total <= kWave) {  // (its range is the whole pencil)
        gather_small_pencil(pl, sl, p, pre, total, dst, box + 2 * gb0, cpdf, invcpd, lane);
        return;
    }
    const int last = (total - 1) / kWave;
    if ((!RANGED || (last >= blo && last < bhi)) && last * kWave + lane >= total)
        dst[last * kWave + lane] = make_float4(kFar, 0.f, 0.f, 0.f);
    auto overlaps = [&](int c) { return !RANGED || (pre[c] < hi && pre[c + 1] > lo); };
    // the binned cells' particles (two chunks each) all load before any is ranked
    float3 q[NF_MAX_WIDTH][2];
#pragma unroll
    for (int c = 0; c < NF_MAX_WIDTH; c++) {
        const int n = pre[c + 1] - pre[c];
        q[c][0] = q[c][1] = make_float3(0.f, 0.f, 0.f);
        if (n > 0 && n <= kBinnedCellMax && overlaps(c)) {
            const float *P = slab_ptr(sl, c);
            const uint64_t ns = slab_n(sl, c), first = p.cell[c].start;
            if (lane < n) q[c][0] = slab_xyz(P, ns, first + (uint64_t)lane, sl.aos);
            if (lane + kWave < n) q[c][1] = slab_xyz(P, ns, first + (uint64_t)(lane + kWave), sl.aos);
        }
    }
    BlockBox bb;
    // The sources at slots s0 (and s1, if in1) of this lane: into the stream
    // and into the boxes of the blocks from slot a to slot z, as far as they
    // lie in the range.
    auto place = [&](int a, int z, bool in0, int s0, float3 v0, bool in1, int s1, float3 v1) {
        if (RANGED) {
            in0 = in0 && s0 >= lo && s0 < hi;
            in1 = in1 && s1 >= lo && s1 < hi;
            a = max(a, lo);
            z = min(z, hi - 1);
        }
        if (in0) dst[s0] = make_float4(v0.x, v0.y, v0.z, 0.f);
        if (in1) dst[s1] = make_float4(v1.x, v1.y, v1.z, 0.f);
        for (int b = a / kWave; b <= z / kWave; b++) {
            bb.to(b, box, gb0, lane);
            bb.add(in0 && s0 / kWave == b, v0.x, v0.y, v0.z);
            bb.add(in1 && s1 / kWave == b, v1.x, v1.y, v1.z);
        }
    };
    auto shifted = [&](float3 v, int c) {
        return make_float3((float)((double)v.x + (double)(c - pl.R) * invcpd), v.y, v.z);
    };
#pragma unroll
    for (int c = 0; c < NF_MAX_WIDTH; c++) {
        const int n = pre[c + 1] - pre[c];
        if (n == 0 || !overlaps(c)) continue;
        if (n <= kBinnedCellMax) {
            const int bin0 = lane < n ? xbin(q[c][0].x, cpdf) : -1;
            const int bin1 = lane + kWave < n ? xbin(q[c][1].x, cpdf) : -1;
            int rank0 = 0, rank1 = 0, acc = 0;
#pragma unroll
            for (int k = 0; k < kXBins; k++) {  // within a bin, chunk 0 ranks before chunk 1
                const uint64_t m0 = ballot(bin0 == k);
                if (bin0 == k) rank0 = acc + lanes_below(m0);
                acc += __builtin_popcountll(m0);
                if (n > kWave) {
                    const uint64_t m1 = ballot(bin1 == k);
                    if (bin1 == k) rank1 = acc + lanes_below(m1);
                    acc += __builtin_popcountll(m1);
                }
            }
            place(pre[c], pre[c + 1] - 1, bin0 >= 0, pre[c] + rank0, shifted(q[c][0], c), bin1 >= 0,
                  pre[c] + rank1, shifted(q[c][1], c));
            continue;
        }
        // a large cell: the reference's order, 64 at a time (the chunks
        // that reach into the range)
        const float *P = slab_ptr(sl, c);
        const uint64_t ns = slab_n(sl, c), first = p.cell[c].start;
        for (int i0 = RANGED ? max(lo - pre[c], 0) & ~(kWave - 1) : 0; i0 < n && (!RANGED || pre[c] + i0 < hi);
             i0 += kWave) {
            const bool in = i0 + lane < n;
            const float3 v = in ? slab_xyz(P, ns, first + (uint64_t)(i0 + lane), sl.aos) : make_float3(0.f, 0.f, 0.f);
            place(pre[c] + i0, pre[c] + min(n, i0 + kWave) - 1, in, pre[c] + i0 + lane, shifted(v, c), false, 0,
                  v);
        }
    }
    bb.flush(box, gb0, lane);
}

// Wave w of a SIC's source gather: w < nsrc_sets fills pencil w (its first
// kSegBlocks blocks if the gather is segmented); wave nsrc_sets + j fills,
// of the stream's blocks [j kSegBlocks, (j + 1) kSegBlocks), those beyond
// their pencil's first kSegBlocks.  Grid: gather_waves() waves.  SEG false:
// no SIC of the launch is segmented, and the kernel holds only the
// whole-pencil code (the segmented code's scalar registers would cost the
// whole-pencil waves an eighth of their occupancy).
template <bool SEG>
__device__ __forceinline__ void gather_wave(const DevPlan &pl, const DevSlabs &sl, float4 *__restrict__ out,
                                            float4 *__restrict__ box, float cpdf, double invcpd, int w, int lane) {
    if (!SEG) {
        gather_pencil_binned<false>(pl, sl, out, box, cpdf, invcpd, w, lane, 0, 0);
        return;
    }
    if (w < pl.nsrc_sets) {
        if (gather_segmented(pl.max_src_blocks))
            gather_pencil_binned<true>(pl, sl, out, box, cpdf, invcpd, w, lane, 0, kSegBlocks);
        else
            gather_pencil_binned<false>(pl, sl, out, box, cpdf, invcpd, w, lane, 0, 0);
        return;
    }
    // Only the pencil of the segment's first block can reach kSegBlocks past
    // its own start within the segment: a pencil that starts later in it
    // ends its first kSegBlocks blocks beyond the segment's end.
    const int b0 = (w - pl.nsrc_sets) * kSegBlocks;
    if (b0 >= src_blocks(pl)) return;
    const int s = cptr<int32_t>(pl.src_parent)[b0];
    if (s < 0) return;  // a block of no pencil
    const int f = cptr<int32_t>(pl.src_set_start)[s] / kWave;
    const int e = f + (cptr<int32_t>(pl.src_set_count)[s] + kWave - 1) / kWave;
    const int lo = max(b0, f + kSegBlocks), hi = min(b0 + kSegBlocks, e);
    if (lo < hi) gather_pencil_binned<true>(pl, sl, out, box, cpdf, invcpd, s, lane, lo - f, hi - f);
}

// Clears the batched launch's queues and, for a census build, its census; for a
// device-planned list, copies its length into counter[1], or 0 when the group
// holds a cell outside its slab.  The first workgroup of the gather does it
// (a launch of its own took 4 us, and a gap), or k_zero_counter.
constexpr int kCensusOffset = kCensusBytes / 4;  // int32 units
constexpr int kQueueOffset = kQueueBytes / 4, kQueueStride = kQueueLine / 4;
__device__ __forceinline__ void clear_queues(const QueueClear &qc, int t) {
    int32_t *const c = qc.counter;
    if (t < kQueues) c[kQueueOffset + t * kQueueStride] = 0;
    if (t != 0) return;
    if (qc.dnitems) c[1] = (qc.dbad && *qc.dbad != 0) ? 0 : *qc.dnitems;
    if (qc.census) {
        unsigned long long *cs = reinterpret_cast<unsigned long long *>(c + kCensusOffset);
        for (int f = 0; f < 4; f++) cs[f] = 0;
    }
}

// At most 96 SGPRs: above that the segmented form loses a wave per SIMD.  Both
// forms of the group's gather (below) are faster for it although they spill 6
// and 90 scalars into VGPR lanes (0 and 32 without the cap): with / without,
// 512^3 slabs 70.7 / 73.4 us on average, clustered slabs 49.2 / 50.1 us, the
// segmented gather of one CPD 255 slab 210 / 220 us.  One SIC's: no difference
// beyond the builds' own (whole pencils 15.8 us, segmented 19.5-20.5 us).
template <bool SEG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_sgpr(96))) void k_gather_sources_binned(
    DevPlan pl, DevSlabs sl, float4 *__restrict__ out, float4 *__restrict__ box, float cpdf, double invcpd,
    QueueClear qc) {
    if (blockIdx.x == 0 && qc.counter) clear_queues(qc, threadIdx.x);
    const int w = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (int)(threadIdx.x / kWave));
    if (w >= gather_waves(pl.nsrc_sets, pl.nsrc_blocks, pl.max_src_blocks) || plan_bad(pl)) return;
    gather_wave<SEG>(pl, sl, out, box, cpdf, invcpd, w, threadIdx.x & (kWave - 1));
}

// The SIC of a group-wide launch that wave w belongs to: the last i with
// first[i] <= w (first[] ascending, first[n] the total), by bisection.
__device__ __forceinline__ int group_sic_of(const int32_t *first, int n, int w) {
    const NF_CONST int32_t *f = cptr<int32_t>(first);
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (f[mid] <= w) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Every SIC's source gather of a launch group in one launch: a group of
// small SICs (a clustered box's) fills the GPU where one SIC's pencils do not.
template <bool SEG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_num_sgpr(96))) void k_gather_sources_binned_group(
    const GroupSic *__restrict__ g, const int32_t *__restrict__ first, int n, float cpdf, double invcpd,
    QueueClear qc) {
    if (blockIdx.x == 0 && qc.counter) clear_queues(qc, threadIdx.x);
    const int w = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (int)(threadIdx.x / kWave));
    if (w >= cptr<int32_t>(first)[n]) return;
    const int i = group_sic_of(first, n, w);
    const DevPlan pl = cptr<GroupSic>(g)[i].pl;
    const DevSlabs sl = cptr<GroupSic>(g)[i].sl;
    void *const sources4 = cptr<GroupSic>(g)[i].sources4;
    const int s = w - cptr<int32_t>(first)[i];
    if (s >= gather_waves(pl.nsrc_sets, pl.nsrc_blocks, pl.max_src_blocks) || plan_bad(pl)) return;
    float4 *src = static_cast<float4 *>(sources4);
    gather_wave<SEG>(pl, sl, src, src + (size_t)pl.nsrc_blocks * NF_BLOCK_SIZE, cpdf, invcpd, s,
                     threadIdx.x & (kWave - 1));  // the block boxes follow the stream
}

// ---------------------------------------------------------------------------
// Plain path: the reference's structure and pair forms
// ---------------------------------------------------------------------------

// What a source tile needs, decided from the tile's bounding box:
//   kNoDensity  unsoftened branch only, no FOF density (no pair within b)
//   kDensity    unsoftened branch only, with the FOF density term
//   kExact      the full softened form with the density term
// The unsoftened branch equals the full form for every pair with r > e (cubic
// spline: r > 2 e).
constexpr int kNoDensity = 0, kDensity = 1, kExact = 2;

// Squared distances above which a form's unsoftened branch is exact and the
// density term zero.  Both carry a relative margin far above FP32 rounding of
// the box corners and of r^2.
struct FormRadii {
    float soft2, dens2;
};
FormRadii form_radii(int softening, const PairConst &pc, float dens_b2) {
    const double eps = (double)pc.eps;
    FormRadii f;
    f.soft2 = softening == NF_SOFT_SINGLE_SPLINE  ? (float)((1.0 / eps) * 1.01)
              : softening == NF_SOFT_CUBIC_SPLINE ? (float)(4.0 / (eps * eps) * 1.01)
                                                  : 0.f;
    f.dens2 = dens_b2 > 0.f ? (float)((double)dens_b2 * 1.01) : -1.f;
    return f;
}
// The form a source tile needs, from the squared gap between its bounding box
// and the sinks'.
template <int SOFT>
__device__ __forceinline__ int form_of(const FormRadii &fr, float gap2) {
    if constexpr (SOFT == NF_SOFT_SINGLE_SPLINE || SOFT == NF_SOFT_CUBIC_SPLINE)
        if (!(gap2 > fr.soft2)) return kExact;
    return gap2 <= fr.dens2 ? kDensity : kNoDensity;
}

// DirectGPUKernels.cuh direct_density<0>: single spline :68-108, Plummer
// :144-174, cubic spline :20-66, cubic Plummer :110-143.  rsqrt is the
// hardware v_rsq_f32 (the reference uses its own platform's fast rsqrtf).  The
// reference's operations in its order; a form leaves out the branches that no
// pair of its tile takes, so every tile's sums are bitwise the full form's.
template <int SOFT, int MODE>
__device__ __forceinline__ void ref_d(float sx, float sy, float sz, float kx, float ky, float kz, const PairConst &pc,
                                      float &dx, float &dy, float &dz, float &r2, float &aw) {
    dx = kx - sx, dy = ky - sy, dz = kz - sz;  // (minus the reference's d: a += f d, exactly)
    r2 = dx * dx + dy * dy + dz * dz;
    if (MODE != kNoDensity && r2 < pc.b2) aw = aw + pc.b2 - r2;
}
// The argument of the form's first transcendental, and f from its value t.
template <int SOFT>
__device__ __forceinline__ float ref_arg(float r2, const PairConst &pc) {
    if constexpr (SOFT == NF_SOFT_SINGLE_SPLINE) return r2 * pc.eps + 1e-32f;
    else if constexpr (SOFT == NF_SOFT_PLUMMER) return r2 + pc.eps;
    else if constexpr (SOFT == NF_SOFT_CUBIC_SPLINE) return r2;
    else return r2 + 1e-16f;
}
template <int SOFT, int MODE>
__device__ __forceinline__ float ref_f(float q, float t, const PairConst &pc) {
    if constexpr (SOFT == NF_SOFT_SINGLE_SPLINE) {
        const float f3 = t * t * t;
        if constexpr (MODE != kExact) return f3;
        return (q > 1.0f) ? f3 : (-15.0f * t + 6.0f) * q + 10.0f;
    } else if constexpr (SOFT == NF_SOFT_PLUMMER) {
        return t * t * t;
    } else if constexpr (SOFT == NF_SOFT_CUBIC_SPLINE) {
        const float f3 = t * t * t;
        if constexpr (MODE != kExact) return f3;
        const float u = pc.eps * sqrt_(q);  // eps_inv / rinv
        if (u >= 2.0f) return f3;
        if (u >= 1.0f) {
            const float u3 = u * u * u;
            return f3 * ((float)(-1.0 / 15.0) + (float)(8.0 / 3.0) * u3 - 3.0f * u3 * u +
                         (float)(6.0 / 5.0) * u3 * u * u - (float)(1.0 / 6.0) * u3 * u3);
        }
        return pc.eps * pc.eps * pc.eps * ((float)(4.0 / 3.0) - (float)(6.0 / 5.0) * u * u + 0.5f * u * u * u);
    } else {  // cubic Plummer
        float r = q;
        r *= r * t;
        r += pc.eps;
        return rcp(r);
    }
}
// P sources against the lane's sink, in order.
template <int SOFT, int MODE, int P>
__device__ __forceinline__ void ref_pairs(const NF_CONST float4 *sp, float yo, float4 k, const PairConst &pc,
                                          float &ax, float &ay, float &az, float &aw) {
    float dx[P], dy[P], dz[P], q[P], t[P];
#pragma unroll
    for (int i = 0; i < P; i++) {
        const float4 s = sp[i];
        float r2;
        ref_d<SOFT, MODE>(s.x, s.y + yo, s.z, k.x, k.y, k.z, pc, dx[i], dy[i], dz[i], r2, aw);
        t[i] = q[i] = ref_arg<SOFT>(r2, pc);
    }
    if constexpr (P == 1) NF_TRANS1("v_rsq_f32", t[0]);
#pragma unroll
    for (int i = 0; i + 1 < P; i += 2) NF_TRANS2("v_rsq_f32", t[i], t[i + 1]);
#pragma unroll
    for (int i = 0; i < P; i++) {
        const float f = ref_f<SOFT, MODE>(q[i], t[i], pc);
        ax += f * dx[i];
        ay += f * dy[i];
        az += f * dz[i];
    }
}
// A tile of 64 sources (FullDirectTile with BLOCK_ACCUM), or the first cnt of
// one (PartialDirectTile, straight into the sink's sums).
template <int SOFT, int MODE>
__device__ __forceinline__ void ref_tile(const NF_CONST float4 *sp, int cnt, float yo, float4 k, const PairConst &pc,
                                         float &ax, float &ay, float &az, float &aw) {
    if (cnt == kWave) {
        float tx = 0.f, ty = 0.f, tz = 0.f;
        for (int i = 0; i < kWave; i += 16)
#pragma unroll
            for (int q = 0; q < 16; q += 2) ref_pairs<SOFT, MODE, 2>(sp + i + q, yo, k, pc, tx, ty, tz, aw);
        ax += tx;
        ay += ty;
        az += tz;
        return;
    }
    int i = 0;
    for (; i + 4 <= cnt; i += 4) {
        ref_pairs<SOFT, MODE, 2>(sp + i, yo, k, pc, ax, ay, az, aw);
        ref_pairs<SOFT, MODE, 2>(sp + i + 2, yo, k, pc, ax, ay, az, aw);
    }
    for (; i < cnt; i++) ref_pairs<SOFT, MODE, 1>(sp + i, yo, k, pc, ax, ay, az, aw);
}

// One 64-sink block per wave, every source pencil in turn.  VALU-bound: the
// full form of the single spline is 21 VALU instructions and a v_rsq_f32 per
// pair, of which the unsoftened form without the density needs 13; 78% of a
// uniform box's tiles take that one.  Eight slabs of a uniform 256^3 box: 7.95 ms as one loop of
// full forms, 5.89 with the v_rsq at raised priority, 4.55 with the forms.
template <int SOFT>
__global__ __launch_bounds__(64) void k_plain(DevPlan pl, PairConst pc, FormRadii fr,
                                              const float4 *__restrict__ sinks, const float4 *__restrict__ src,
                                              float4 *__restrict__ out) {
    const int blk = blockIdx.x;
    if (blk >= sink_blocks(pl) || plan_bad(pl)) return;
    const int lane = threadIdx.x;
    const int s = cptr<int32_t>(pl.parent)[blk];
    const int id = blk * kWave + lane;
    const float4 k = sinks[id];  // padded ids hold zeros (PencilKernel.cu:109-117)
    const bool real = (uint32_t)id < cptr<uint32_t>(pl.sink_idmax)[s];
    const float inf = __builtin_huge_valf();
    const float lx = wave_min(real ? k.x : inf), ly = wave_min(real ? k.y : inf), lz = wave_min(real ? k.z : inf);
    const float hx = wave_max(real ? k.x : -inf), hy = wave_max(real ? k.y : -inf), hz = wave_max(real ? k.z : -inf);
    const NF_CONST float4 *sources = cptr<float4>(src);
    const NF_CONST float4 *box = sources + (int64_t)pl.nsrc_blocks * kWave;  // box_after
    float ax = 0.f, ay = 0.f, az = 0.f, aw = 0.f;
    const int W = pl.W;
    for (int c = s * W; c < s * W + W; c++) {
        const int si = cptr<int32_t>(pl.ilist)[c];
        const float yo = cptr<float>(pl.yoff)[c];
        const int st = cptr<int32_t>(pl.src_set_start)[si], n = cptr<int32_t>(pl.src_set_count)[si];
        int forms = 0;  // lane i: the form of tile (b & ~63) + i
        for (int b = 0; b * kWave < n; b++) {
            if ((b & (kWave - 1)) == 0) {
                forms = 0;
                if ((b + lane) * kWave < n) {
                    const int64_t gb = (int64_t)st / kWave + b + lane;
                    const float4 ql = box[2 * gb], qh = box[2 * gb + 1];
                    const float gx = fmaxf(0.f, fmaxf(ql.x - hx, lx - qh.x));
                    const float gy = fmaxf(0.f, fmaxf(ql.y + yo - hy, ly - (qh.y + yo)));
                    const float gz = fmaxf(0.f, fmaxf(ql.z - hz, lz - qh.z));
                    forms = form_of<SOFT>(fr, gx * gx + gy * gy + gz * gz);
                }
            }
            const int form = __builtin_amdgcn_readlane(forms, b & (kWave - 1));
            const NF_CONST float4 *sp = sources + st + b * kWave;
            const int cnt = min(kWave, n - b * kWave);
            if (form == kNoDensity) ref_tile<SOFT, kNoDensity>(sp, cnt, yo, k, pc, ax, ay, az, aw);
            else if (form == kDensity) ref_tile<SOFT, kDensity>(sp, cnt, yo, k, pc, ax, ay, az, aw);
            else ref_tile<SOFT, kExact>(sp, cnt, yo, k, pc, ax, ay, az, aw);
        }
    }
    if (real) out[id] = make_float4(ax, ay, az, aw);
}

// The co-adds give a chunk (up to 64 particles of a sink cell) to LANES lanes:
// a whole wave, or 16 lanes where cells hold few particles (launch_coadd_*).
//
// Addresses of the W partials of the sinks of cell (j_low + j, z): the cell is
// at position c of pencil k = z - c (mod cpd).  Lane c < W of the chunk's lanes
// looks pencil k up, all of them at once (one lookup after the other took
// 13 us of a 980-sink SIC's co-add).  base: the padded slot of the cell's first
// particle in pencil k; with planes, split: the first of the cell's particles
// (its own numbering) whose partial there is not spread over the source
// pencils' planes.  Every lane gets the cell's slab start and its count (0 if
// not `on`).  Every lane of the wave must call it.
struct PartialSlots {
    int base, split;  // lane c's
    uint32_t cstart;
    int cn;
};
template <int LANES>
__device__ __forceinline__ PartialSlots partial_slots(const DevPlan &pl, bool on, int cell, int l, bool planes) {
    const int z = cell % pl.Nk, c = min(l, pl.W - 1), k = z >= c ? z - c : z - c + pl.cpd;
    const int s = cell - z + k;
    PartialSlots p{0, 0, 0, 0};
    int n = 0;
    uint64_t nsrc = 0;
    if (on) {
        const nf_cell_plan own = pl.sink_plan[s].cell[0];  // pencil k starts with cell k = z - c
        p.base = pl.sink_set_start[s];
        p.cstart = own.start;
        n = own.N;
        if (planes) {
            p.split = pl.sink_set_count[s];
#pragma unroll
            for (int y = 0; y < NF_MAX_WIDTH; y++)
                if (y < pl.W) nsrc += (uint64_t)pl.src_set_count[pl.ilist[s * pl.W + y]];
        }
    }
    int off = 0;  // the pencil's cells before this one: cells z - c .. z - 1
#pragma unroll
    for (int i = 1; i < NF_MAX_WIDTH; i++) {
        const int ni = __shfl(n, i, LANES);
        off += c >= i ? ni : 0;
    }
    p.base += off;
    p.split = planes && y_split(nsrc, pl.y_cost) ? tile_sinks(p.split) - off : 0;
    p.cstart = __shfl(p.cstart, 0, LANES);
    p.cn = __shfl(n, 0, LANES);
    return p;
}

// RescaleAndCoAddAcceleration (kick.cpp:96-105) on one sink's float4, with
// the FLOAT3p1 rules (float3p1.cpp:41-56): x, y, z = (a * inv_eps3 + far) *
// rescale in float, each operation rounded on its own (no contraction), and
// w -= DensityKernelRad2 in double.
__device__ __forceinline__ float4 apply_kick(float4 a, const KickArgs &k, int64_t row) {
#pragma clang fp contract(off)
    if (!k.on) return a;
    if (k.near_out)  // the NearAcc record: FLOAT3p1 *= FLOAT scales xyz only
        reinterpret_cast<float4 *>(k.near_out)[row] =
            make_float4(a.x * k.inv_eps3, a.y * k.inv_eps3, a.z * k.inv_eps3, a.w);
    const float *f = k.far + 3 * (row - k.far_base);
    a.x = (a.x * k.inv_eps3 + f[0]) * k.rescale;
    a.y = (a.y * k.inv_eps3 + f[1]) * k.rescale;
    a.z = (a.z * k.inv_eps3 + f[2]) * k.rescale;
    a.w = (float)((double)a.w - k.density_rad2);
    return a;
}

// FP32 co-add in the reference's order: the pencils of a skewer are applied
// in increasing k, the first one setting the value and the rest adding.  For
// cell z that is c = min(z, W-1) .. 0, then W-1 .. z+1.
template <int LANES>
__global__ __launch_bounds__(256) void k_coadd_plain(DevPlan pl, const float4 *__restrict__ part,
                                                     float4 *__restrict__ acc, KickArgs kick) {
    const int q = (int)((blockIdx.x * 256 + threadIdx.x) / LANES), l = threadIdx.x % LANES;
    const int nq = coadd_chunks(pl);
    if ((int)(blockIdx.x * 256 + (threadIdx.x & ~(kWave - 1))) / LANES >= nq || plan_bad(pl)) return;
    const bool on = q < nq;
    const int cell = on ? pl.coadd_chunk[2 * q] : 0, first = on ? pl.coadd_chunk[2 * q + 1] : 0;
    const PartialSlots ps = partial_slots<LANES>(pl, on, cell, l, false);
    const int W = pl.W, m = min(cell % pl.Nk, W - 1);
    int base[NF_MAX_WIDTH];  // in that order
#pragma unroll
    for (int t = 0; t < NF_MAX_WIDTH; t++) base[t] = __shfl(ps.base, t <= m ? m - t : max(W + m - t, 0), LANES);
    for (int i = first + l, e = min(first + kWave, ps.cn); i < e; i += LANES) {
        float4 a = part[base[0] + i];
#pragma unroll
        for (int t = 1; t < NF_MAX_WIDTH; t++) {
            if (t >= W) break;
            const float4 p = part[base[t] + i];
            a.x += p.x;
            a.y += p.y;
            a.z += p.z;
            a.w += p.w;
        }
        acc[ps.cstart + i] = apply_kick(a, kick, (int64_t)ps.cstart + i);
    }
}

// FP64 co-add: sum of the W double partials, scaled back to the reference's
// units (out_scale applies to a, not to w).  q, l: the lane's chunk (on: it is
// one) and its place among the chunk's lanes.  PLANES: the partials have planes
// per source pencil; a launch that has them is small and waits for its loads,
// so a sink's loads go out W partials at a time, a plane after the other (a
// 980-sink SIC's co-add 13.5 -> 9.8 us; two planes at a time 8.7, but 29 instead
// of 20 us for a group of eight 64^3 SICs, at 210 registers).
template <int LANES, bool PLANES>
__device__ __forceinline__ void coadd_chunk_f64(const DevPlan &pl, const double *__restrict__ part, double out_scale,
                                                float4 *__restrict__ acc, const KickArgs &kick, int q, bool on,
                                                int l) {
    const int cell = on ? pl.coadd_chunk[2 * q] : 0, first = on ? pl.coadd_chunk[2 * q + 1] : 0;
    const PartialSlots ps = partial_slots<LANES>(pl, on, cell, l, PLANES);
    const int W = pl.W;
    int base[NF_MAX_WIDTH], split[NF_MAX_WIDTH];
#pragma unroll
    for (int c = 0; c < NF_MAX_WIDTH; c++) {
        base[c] = __shfl(ps.base, c, LANES);
        split[c] = PLANES ? __shfl(ps.split, c, LANES) : 0;
    }
    for (int i = first + l, e = min(first + kWave, ps.cn); i < e; i += LANES) {
        double h[NF_MAX_WIDTH][4];
        auto partial = [&](int c, int y, double *out) {
            const double *p =
                part + 4 * ((int64_t)base[c < W ? c : 0] + i) + (y > 0 && y < W && i < split[c] ? y * pl.y_plane : 0);
#pragma unroll
            for (int t = 0; t < 4; t++) out[t] = p[t];
        };
#pragma unroll
        for (int c = 0; c < NF_MAX_WIDTH; c++) partial(c, 0, h[c]);
        if constexpr (PLANES)
#pragma unroll
            for (int y = 1; y < NF_MAX_WIDTH; y++) {
                double g[NF_MAX_WIDTH][4];
#pragma unroll
                for (int c = 0; c < NF_MAX_WIDTH; c++) partial(c, y, g[c]);
#pragma unroll
                for (int c = 0; c < NF_MAX_WIDTH; c++)
                    if (y < W && i < split[c])
#pragma unroll
                        for (int t = 0; t < 4; t++) h[c][t] += g[c][t];
            }
        double a[4] = {0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < NF_MAX_WIDTH; c++) {
            if (c >= W) break;
#pragma unroll
            for (int t = 0; t < 4; t++) a[t] += h[c][t];
        }
        const float4 r =
            make_float4((float)(a[0] * out_scale), (float)(a[1] * out_scale), (float)(a[2] * out_scale), (float)a[3]);
        acc[ps.cstart + i] = apply_kick(r, kick, (int64_t)ps.cstart + i);
    }
}

template <int LANES, bool PLANES>
__global__ __launch_bounds__(256) void k_coadd_f64(DevPlan pl, const double *__restrict__ part, double out_scale,
                                                   float4 *__restrict__ acc, KickArgs kick) {
    const int q = (int)((blockIdx.x * 256 + threadIdx.x) / LANES);
    const int nq = coadd_chunks(pl);
    if ((int)(blockIdx.x * 256 + (threadIdx.x & ~(kWave - 1))) / LANES >= nq || plan_bad(pl)) return;
    coadd_chunk_f64<LANES, PLANES>(pl, part, out_scale, acc, kick, q, q < nq, threadIdx.x % LANES);
}

// Every SIC's FP64 co-add of a launch group in one launch.
template <int LANES, bool PLANES>
__global__ __launch_bounds__(256) void k_coadd_f64_group(const GroupSic *__restrict__ g,
                                                         const int32_t *__restrict__ first, int n) {
    const int w = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (int)(threadIdx.x / kWave));
    if (w >= cptr<int32_t>(first)[n]) return;
    const int i = group_sic_of(first, n, w);
    const DevPlan pl = cptr<GroupSic>(g)[i].pl;
    const int q0 = (w - cptr<int32_t>(first)[i]) * (kWave / LANES), nq = coadd_chunks(pl);
    if (q0 >= nq || plan_bad(pl)) return;
    const int lane = threadIdx.x & (kWave - 1), q = q0 + lane / LANES;
    const KickArgs kick = cptr<GroupSic>(g)[i].kick;
    coadd_chunk_f64<LANES, PLANES>(pl, static_cast<const double *>(cptr<GroupSic>(g)[i].partial),
                                   cptr<GroupSic>(g)[i].out_scale, reinterpret_cast<float4 *>(cptr<GroupSic>(g)[i].acc4),
                                   kick, q, q < nq, lane % LANES);
}

// ---------------------------------------------------------------------------
// Batched path
// ---------------------------------------------------------------------------

// Pair kernel in box units.  r2 carries pc.r2add; for the single spline the
// result is g/e^3 (the e^3 is restored in the co-add).  MODE: the tile's form,
// as on the plain path.

// A pair in four steps, so that the transcendentals of two pairs can run in
// one raised stretch (35.9 -> 35.4 cycles per pair):
// 1. d = sink - source (so that a += g d, and no operand of an FMA carries a
//    sign), r2 and the density term;
template <int MODE>
__device__ __forceinline__ void pair_r2(float sx, float sy, float sz, float kx, float ky, float kz,
                                        const PairConst &pc, float &dx, float &dy, float &dz, float &r2, float &aw) {
    dx = kx - sx;
    dy = ky - sy;
    dz = kz - sz;
    r2 = fmaf(dx, dx, pc.r2add);
    r2 = fmaf(dy, dy, r2);
    r2 = fmaf(dz, dz, r2);
    if constexpr (MODE != kNoDensity) aw += clamp01(pc.b2x - r2);
}
// 2. f = 1/r, or r for the cubic Plummer form;
template <int SOFT>
__device__ __forceinline__ void pair_f(float &a, float &b) {
    if constexpr (SOFT == NF_SOFT_CUBIC_PLUMMER) NF_TRANS2("v_sqrt_f32", a, b);
    else NF_TRANS2("v_rsq_f32", a, b);
}
// 3. g from r2 and f;
template <int SOFT, int MODE>
__device__ __forceinline__ float pair_g(float r2, float f, const PairConst &pc) {
    if constexpr (SOFT == NF_SOFT_CUBIC_PLUMMER) {
        // r2 already holds + TAU2.  r^3 as r2*sqrt(r2), so a padding source
        // (r2 = inf) gives 1/inf = 0, not inf*0.
        return rcp(fmaf(r2, f, pc.eps));
    }
    const float f3 = f * f * f;
    if constexpr (MODE != kExact || SOFT == NF_SOFT_PLUMMER) {
        return f3;
    } else if constexpr (SOFT == NF_SOFT_SINGLE_SPLINE) {
        return fminf(f3, fmaf(fmaf(pc.c1, f, pc.c2), r2, pc.c3));
    } else {
        // Cubic spline, u = r/e: f^3 beyond 2, below it e^-3 times a cubic in u
        // (from 1 on, with the -1/(15 u^3) of the middle piece as -f^3/15, and
        // 8/3 - 3 u + 6/5 u^2 - u^3/6 about u = 3/2, where its terms are no
        // larger than its values: about 0 they cancel to a 50th).
        // Selects, not branches: nearly every wave has lanes in each piece.  A
        // padding source (r2 = inf, f = 0) has u = NaN and takes f^3 = 0.
        const float u = r2 * f * pc.eps;
        const float t = u - 1.5f;
        const float mid = fmaf(fmaf(fmaf((float)(-1.0 / 6.0), t, 0.45f), t, -0.525f), t, (float)(73.0 / 240.0));
        const float in = fmaf(fmaf(0.5f, u, (float)(-6.0 / 5.0)), u * u, (float)(4.0 / 3.0));
        const bool outer = u >= 1.0f;
        const float soft = fmaf(outer ? mid : in, pc.c3, outer ? f3 * (float)(-1.0 / 15.0) : 0.0f);
        return u < 2.0f ? soft : f3;
    }
}
// 4. the force sums.
__device__ __forceinline__ void pair_sum(float g, float dx, float dy, float dz, float &ax, float &ay, float &az) {
    ax = fmaf(g, dx, ax);
    ay = fmaf(g, dy, ay);
    az = fmaf(g, dz, az);
}

// Four sources in scalar registers, by one load.
struct Sources4 {
    float4 s[4];
    __device__ __forceinline__ void load(const NF_CONST float4 *p) {
        typedef float F32x16 __attribute__((ext_vector_type(16)));
        const F32x16 v = *(const NF_CONST F32x16 *)p;
#pragma unroll
        for (int i = 0; i < 4; i++) s[i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], 0.f);
    }
};

// The pairs of P sources (at sp) with the S sinks of a lane, sink slots below
// S/2 in form MLO and the others in MHI.
template <int SOFT, int MLO, int MHI, int S, int P, typename SrcP>
__device__ __forceinline__ void pair_group(SrcP sp, const float *kx, const float *ky,
                                           const float *kz, const PairConst &pc, float *bx, float *by, float *bz,
                                           float *tw) {
    constexpr int N = P * S;
    static_assert(N % 2 == 0, "pairs two by two");
    float dx[N], dy[N], dz[N], r2[N], f[N];
#pragma unroll
    for (int t = 0; t < N; t++) {
        const int u = t % S;
        const float4 sv = sp[t / S];
        if (u < S / 2) pair_r2<MLO>(sv.x, sv.y, sv.z, kx[u], ky[u], kz[u], pc, dx[t], dy[t], dz[t], r2[t], tw[u]);
        else pair_r2<MHI>(sv.x, sv.y, sv.z, kx[u], ky[u], kz[u], pc, dx[t], dy[t], dz[t], r2[t], tw[u]);
        f[t] = r2[t];
    }
#pragma unroll
    for (int t = 0; t < N; t += 2) pair_f<SOFT>(f[t], f[t + 1]);
#pragma unroll
    for (int t = 0; t < N; t++) {
        const int u = t % S;
        const float g = u < S / 2 ? pair_g<SOFT, MLO>(r2[t], f[t], pc) : pair_g<SOFT, MHI>(r2[t], f[t], pc);
        pair_sum(g, dx[t], dy[t], dz[t], bx[u], by[u], bz[u]);
    }
}

struct BatchCtx {
    PairConst pc;
    double invcpd;
    FormRadii fr;
};

// A sink pencil's cells, for reading its sinks straight from the slab.
struct SinkCells {
    uint32_t start[NF_MAX_WIDTH];
    int pre[NF_MAX_WIDTH + 1];  // sinks before each cell
};
__device__ __forceinline__ SinkCells sink_cells(const SicView &v, int s) {
    const nf_sink_plan p = cptr<nf_sink_plan>(v.sink_plan)[s];
    SinkCells sc;
    sc.pre[0] = 0;
#pragma unroll
    for (int c = 0; c < NF_MAX_WIDTH; c++) {
        sc.start[c] = p.cell[c].start;
        sc.pre[c + 1] = sc.pre[c] + (c < v.W ? p.cell[c].N : 0);
    }
    return sc;
}
// Sink i of the pencil: its slab position with z moved into the pencil's
// central cell by the FP64 offset (c - R)/cpd, rounded once.
__device__ __forceinline__ float3 pencil_sink(const SicView &v, const SinkCells &sc, int i, double invcpd) {
    // The cell holding sink i, by selects over the (wave-uniform) cell table:
    // no indexed private array.
    int c = 0, pre = 0;
    uint32_t start = sc.start[0];
#pragma unroll
    for (int cc = 1; cc < NF_MAX_WIDTH; cc++) {
        const bool in = cc < v.W && i >= sc.pre[cc];
        c = in ? cc : c;
        pre = in ? sc.pre[cc] : pre;
        start = in ? sc.start[cc] : start;
    }
    const float3 q = slab_xyz(v.sink_slab, v.sink_n, (uint64_t)start + (uint64_t)(i - pre), v.aos);
    return make_float3(q.x, q.y, (float)((double)q.z + (double)(c - v.R) * invcpd));
}

// A sink pencil's W source pencils: lane y holds pencil y's first slot and
// count, pre[y] the 64-source blocks before pencil y (wave-uniform).  The
// lookups of all W pencils are in flight together: a chain of two loads per
// item, not per pencil.
struct SourceRows {
    int start, count;            // per lane
    int pre[NF_MAX_WIDTH + 1];
    __device__ __forceinline__ int start_of(int y) const { return __builtin_amdgcn_readlane(start, y); }
    __device__ __forceinline__ int count_of(int y) const { return __builtin_amdgcn_readlane(count, y); }
};
__device__ __forceinline__ SourceRows source_rows(const SicView &v, int s, int lane) {
    SourceRows r;
    r.start = r.count = 0;
    if (lane < v.W) {
        const int si = cptr<int32_t>(v.ilist)[s * v.W + lane];
        r.start = cptr<int32_t>(v.src_set_start)[si];
        r.count = cptr<int32_t>(v.src_set_count)[si];
    }
    r.pre[0] = 0;
#pragma unroll
    for (int y = 0; y < NF_MAX_WIDTH; y++) r.pre[y + 1] = r.pre[y] + (r.count_of(y) + kWave - 1) / kWave;
    return r;
}
// The pair forms of blocks p, p + 1, ... p + 63 of the pencils' blocks taken
// one after the other, one per lane: form_lo | form_hi << 2 against the sinks'
// boxes (x and y: bl, bh; z per half of the sink slots).
struct SinkBox {
    float lx, ly, hx, hy, lz0, hz0, lz1, hz1;
};
template <int SOFT, bool HALVES>
__device__ __forceinline__ int block_forms(const BatchCtx &cx, const SicView &v, const SourceRows &r,
                                           const SinkBox &k, int p, int lane) {
    const NF_CONST float4 *box = cptr<float4>(v.box4);
    const int i = p + lane;
    int y = 0, first = 0;
#pragma unroll
    for (int c = 1; c < NF_MAX_WIDTH; c++) {
        const bool in = i >= r.pre[c];
        y = in ? c : y;
        first = in ? r.pre[c] : first;
    }
    const int start = __shfl(r.start, y);
    if (i >= r.pre[NF_MAX_WIDTH]) return 0;
    const int64_t gb = (int64_t)start / kWave + (i - first);
    const float4 ql = box[2 * gb], qh = box[2 * gb + 1];
    const double yo = (double)(y - v.R) * cx.invcpd;
    const float sly = (float)((double)k.ly - yo), shy = (float)((double)k.hy - yo);
    const float gx = fmaxf(0.f, fmaxf(ql.x - k.hx, k.lx - qh.x));
    const float gy = fmaxf(0.f, fmaxf(ql.y - shy, sly - qh.y));
    const float gxy = gx * gx + gy * gy;
    const float gz1 = fmaxf(0.f, fmaxf(ql.z - k.hz1, k.lz1 - qh.z));
    const int mh = form_of<SOFT>(cx.fr, gxy + gz1 * gz1);
    int ml = mh;
    if (HALVES) {
        const float gz0 = fmaxf(0.f, fmaxf(ql.z - k.hz0, k.lz0 - qh.z));
        ml = form_of<SOFT>(cx.fr, gxy + gz0 * gz0);
    }
    return ml | (mh << 2);
}

// Pair interactions a wave has computed in each pair form (kNoDensity,
// kDensity, kExact) and in short tails: wave-uniform, so the counts live in
// scalar registers and cost no VALU work.  Counted only by the census
// instantiations of k_batched: eight more 64-bit scalars push the single
// spline's S = 2 kernel into SGPR and VGPR spills that cost it 7%.
struct Census {
    uint64_t form[3];
    uint64_t tail;
};
__device__ __forceinline__ void census_add(Census &c, int mode, uint64_t n) {
    c.form[0] += mode == kNoDensity ? n : 0;
    c.form[1] += mode == kDensity ? n : 0;
    c.form[2] += mode == kExact ? n : 0;
}

// One source tile (cnt <= 64 sources) against the S sinks
// of every lane; sources are wave-uniform loads (scalar cache).  The force
// terms of each batch of kSrcBatch sources are summed on their own before
// they join the tile sum, for one add per component per batch.  On random
// terms a sum of 4 batch sums of 16 terms carries 1.7-2.3x less FP32
// rounding than one running sum of 64 terms, and 1.0-1.1x the rounding of 8
// batch sums of 8 terms, which cost 1% more kernel time.  Sink slots
// u < S/2 take pair form MLO, the others MHI (S = 1: MHI); every form gives
// the same value for the pairs its box test admits, so the split changes
// which code runs, not the result.  The last batch stops at the first multiple
// of 4 past the cnt % kSrcBatch real sources: the padding sources give exact
// zeros, so how many of them are taken changes no sum.
//
// The sources of full batches come four to a scalar load, the next four asked
// for before these are summed: left to itself the compiler loads two sources
// some 10 to 25 instructions before it waits for them, and the scalar cache
// misses on most (a pencil is read once per item).  One batch stands in the
// code, not the four of a block: the nine form pairs at S = 2 are 60 KB of the
// 64 KB that two CUs' instruction cache holds, unrolled 87 KB.  Direct kernel
// of eight 512^3 slabs at S = 1 / 2 / 4: 15.24 / 14.08 / 15.30 -> 14.13 / 13.66
// / 14.64 ms; of radius-1 slabs with 512 particles a cell 8.97 / 8.91 / 11.19
// -> 8.44 / 8.45 / 9.17 ms.  (The 512^3 slabs at S = 2 otherwise: unrolled
// 13.77; eight sources a load, which spills scalar registers, 14.71; half a
// batch in the code 13.83; the remainder in the same loop 14.39; sources
// through LDS 14.11.)
constexpr int kSrcBatch = 16;
template <int SOFT, int MLO, int MHI, int S>
__device__ __forceinline__ void full_tile(const NF_CONST float4 *sp, int cnt, const float *kx, const float *ky,
                                          const float *kz, const PairConst &pc, float *tx, float *ty, float *tz,
                                          float *tw) {
    constexpr int P = S == 1 ? 2 : 1;  // sources per pair_group
    const int fullb = cnt & ~(kSrcBatch - 1);
    Sources4 sb[2];
    if (fullb > 0) sb[0].load(sp);
#pragma unroll 1
    for (int i = 0; i < fullb; i += kSrcBatch) {
        float bx[S], by[S], bz[S];
#pragma unroll
        for (int u = 0; u < S; u++) bx[u] = by[u] = bz[u] = 0.f;
#pragma unroll
        for (int h = 0; h < kSrcBatch / 4; h++) {
            // (after a whole block's last batch the first sources again: in bounds, not used)
            sb[(h + 1) & 1].load(sp + (h < kSrcBatch / 4 - 1 ? i + 4 * h + 4 : (i + kSrcBatch) % kWave));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < 4; q += P)
                pair_group<SOFT, MLO, MHI, S, P>(sb[h & 1].s + q, kx, ky, kz, pc, bx, by, bz, tw);
        }
#pragma unroll
        for (int u = 0; u < S; u++) {
            tx[u] += bx[u];
            ty[u] += by[u];
            tz[u] += bz[u];
        }
    }
    if (cnt > fullb) {
        float bx[S], by[S], bz[S];
#pragma unroll
        for (int u = 0; u < S; u++) bx[u] = by[u] = bz[u] = 0.f;
        // (by 4, the last of them padding: one wait for scalar loads per 4 sources)
#pragma unroll 1
        for (int q = fullb; q < cnt; q += 4)
#pragma unroll
            for (int k = 0; k < 4; k += P)
                pair_group<SOFT, MLO, MHI, S, P>(sp + q + k, kx, ky, kz, pc, bx, by, bz, tw);
#pragma unroll
        for (int u = 0; u < S; u++) {
            tx[u] += bx[u];
            ty[u] += by[u];
            tz[u] += bz[u];
        }
    }
}

// A tile with the modes of its two halves of sink slots.
template <int SOFT, int S>
__device__ __forceinline__ void mixed_tile(int mlo, int mhi, const NF_CONST float4 *sp, int cnt, const float *kx,
                                           const float *ky, const float *kz, const PairConst &pc, float *tx,
                                           float *ty, float *tz, float *tw) {
    if (S == 1 || mlo == mhi) {
        if (mhi == kNoDensity) full_tile<SOFT, kNoDensity, kNoDensity, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
        else if (mhi == kDensity) full_tile<SOFT, kDensity, kDensity, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
        else full_tile<SOFT, kExact, kExact, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
    } else if (mlo == kNoDensity) {
        if (mhi == kDensity) full_tile<SOFT, kNoDensity, kDensity, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
        else full_tile<SOFT, kNoDensity, kExact, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
    } else if (mlo == kDensity) {
        if (mhi == kNoDensity) full_tile<SOFT, kDensity, kNoDensity, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
        else full_tile<SOFT, kDensity, kExact, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
    } else {
        if (mhi == kNoDensity) full_tile<SOFT, kExact, kNoDensity, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
        else full_tile<SOFT, kExact, kDensity, S>(sp, cnt, kx, ky, kz, pc, tx, ty, tz, tw);
    }
}

// Register tile: 64*S sinks of one pencil on the lanes; sources are wave
// uniform and come through the scalar cache.
// It meets source pencils [y0, y1); hsum: the lane's place in the wave's LDS
// accumulators, 4 S of them 64 apart.
template <int SOFT, int S, bool CENSUS>
__device__ __forceinline__ void full_item(const BatchCtx &cx, const SicView &v, const WorkItem &w, int nsink, int y0,
                                          int y1, double *hsum, int lane, Census &cen) {
    const NF_CONST float4 *src = cptr<float4>(v.sources4);
    NF_GLOBAL double *out = (NF_GLOBAL double *)v.partial;
    const int s = w.sinkset;
    const int base = cptr<int32_t>(v.sink_set_start)[s] + w.first;
    const SourceRows rows = source_rows(v, s, lane);
    // nsink: 64*S, or fewer for a masked tail tile
    const uint64_t n_lo = (uint64_t)min(nsink, kWave * (S / 2)), n_hi = (uint64_t)nsink - n_lo;  // sinks per half
    const SinkCells sc = sink_cells(v, s);
    float kx[S], ky[S], kz[S];
    // The sinks' box: x and y over all slots, z per half of the slots (the
    // slots run along the pencil, z), so each half of a tile can take its
    // own pair form.
    float blx = __builtin_huge_valf(), bly = blx, bhx = -blx, bhy = -blx;
    float blz0 = blx, bhz0 = -blx, blz1 = blx, bhz1 = -blx;
#pragma unroll
    for (int u = 0; u < S; u++) {
        // Lanes past nsink repeat sink 0 (inside the box, results not stored).
        const int ki = lane + kWave * u < nsink ? lane + kWave * u : 0;
        const float3 k = pencil_sink(v, sc, w.first + ki, cx.invcpd);
        kx[u] = k.x;
        ky[u] = k.y;
        kz[u] = k.z;
        blx = fminf(blx, k.x);
        bly = fminf(bly, k.y);
        bhx = fmaxf(bhx, k.x);
        bhy = fmaxf(bhy, k.y);
        if (u < S / 2) {
            blz0 = fminf(blz0, k.z);
            bhz0 = fmaxf(bhz0, k.z);
        } else {
            blz1 = fminf(blz1, k.z);
            bhz1 = fmaxf(bhz1, k.z);
        }
    }
    blx = wave_min(blx);
    bly = wave_min(bly);
    bhx = wave_max(bhx);
    bhy = wave_max(bhy);
    blz1 = wave_min(blz1);
    bhz1 = wave_max(bhz1);
    if (S > 1) {
        blz0 = wave_min(blz0);
        bhz0 = wave_max(bhz0);
    }

    // Each block's FP32 tile sum joins an FP64 sum: a convert and an add per
    // component, which gfx950 issues at nearly the FP32 rate (a TwoSum merge
    // into an FP32 (hi, lo) pair is 7 instructions and carries fewer bits).
    // The FOF density w too: in a dense halo a sink meets thousands of pairs
    // within b, and one FP32 running sum of them drifts by ~1e-5.  The FP64
    // sums are one source pencil's; the pencils' are added up in LDS, whose
    // registers the tile loop has no room for.
    const SinkBox kbox = {blx, bly, bhx, bhy, blz0, bhz0, blz1, bhz1};
    int p = 0;  // the item's blocks: p next, counted from source pencil 0
#pragma unroll
    for (int y = 0; y < NF_MAX_WIDTH; y++) p = y < y0 ? rows.pre[y + 1] : p;
    int modes = 0, pm0 = p;  // lane i: forms of block pm0 - 64 + i
    for (int y = y0; y < y1; y++) {
        const int st = rows.start_of(y), n = rows.count_of(y);
        double hx[S], hy[S], hz[S], hw[S];
#pragma unroll
        for (int u = 0; u < S; u++) hx[u] = hy[u] = hz[u] = hw[u] = 0.0;
        // Source y + (y-R)/cpd == sink y - (y-R)/cpd on the other side; the
        // cell-centre offset is formed in FP64.
        const double yo = (double)(y - v.R) * cx.invcpd;
        float kyy[S];
#pragma unroll
        for (int u = 0; u < S; u++) kyy[u] = (float)((double)ky[u] - yo);
        const int nblk = (n + kWave - 1) / kWave;
        for (int b = 0; b < nblk; b++, p++) {
            // Lane i decides the pair forms of block i of the item's source
            // blocks (64 per pass): one vector pass instead of a wave-uniform
            // box test and a dependent box load per block.
            if (p == pm0) {
                modes = block_forms<SOFT, (S > 1)>(cx, v, rows, kbox, p, lane);
                pm0 += kWave;
            }
            const int pm = __builtin_amdgcn_readlane(modes, (p - pm0) & (kWave - 1));
            const int mlo = pm & 3, mhi = pm >> 2;
            const NF_CONST float4 *sp = src + st + b * kWave;
            const int cnt = min(kWave, n - b * kWave);
            if constexpr (CENSUS) {
                census_add(cen, mlo, n_lo * (uint64_t)cnt);
                census_add(cen, mhi, n_hi * (uint64_t)cnt);
            }
            float tx[S], ty[S], tz[S], tw[S];
#pragma unroll
            for (int u = 0; u < S; u++) tx[u] = ty[u] = tz[u] = tw[u] = 0.f;
            mixed_tile<SOFT, S>(mlo, mhi, sp, cnt, kx, kyy, kz, cx.pc, tx, ty, tz, tw);
#pragma unroll
            for (int u = 0; u < S; u++) {
                hx[u] += (double)tx[u];
                hy[u] += (double)ty[u];
                hz[u] += (double)tz[u];
                hw[u] += (double)tw[u];
            }
        }
#pragma unroll
        for (int u = 0; u < S; u++) {
            const double h[4] = {hx[u], hy[u], hz[u], hw[u]};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                double *const a = hsum + kWave * (4 * u + c);
                *a = y == y0 ? h[c] : *a + h[c];
            }
        }
    }
    if (y1 - y0 < v.W) out += y0 * v.y_plane;
#pragma unroll
    for (int u = 0; u < S; u++) {
        if (lane + kWave * u >= nsink) continue;
        NF_GLOBAL double *o = out + 4 * (int64_t)(base + lane + kWave * u);
#pragma unroll
        for (int c = 0; c < 4; c++) o[c] = hsum[kWave * (4 * u + c)];
    }
}

// Short tail of a pencil (r < kTailLanes sinks): the sinks sit two to a lane
// on L = ceil(r / 2) lanes, the wave holds G = 64 / L such groups, and group g
// takes every G-th source of a block, from source g on.  One pass over the
// sources whatever r is, all lanes busy but 64 - L G and one slot of an odd r.
// A block's 64 sources are loaded one to a lane, the next block's while this
// one is summed, and handed to the groups through the wave's LDS (one 16 B read
// per two pairs of a lane, the same address on a group's lanes).  Each block's
// FP32 sums join FP64 sums per lane, as a register tile's do, and a tree over
// the groups adds those.
//
// Against the sources on 16-lane groups with up to 8 sinks per pass, which this
// replaces: the direct kernel of 24 sparse slabs (129^2 pencils of 25 sinks
// each) 3.30 -> 1.27 ms, of eight 512^3 slabs 14.77 -> 14.08 ms (the tails
// alone took 1.25 ms of that).  With every group loading its sources itself,
// two loads ahead, a lone tail of 36 sinks and 500 sources took 35 us; through
// LDS 23 us, and the sparse slabs 1.06 -> 0.97 ms.
template <int SOFT, int MODE>
__device__ __forceinline__ void tail_block(const float4 *bp, int cnt, int G, int full, int grp, const float *kx,
                                           const float *ky, const float *kz, const PairConst &pc, float *tx,
                                           float *ty, float *tz, float *tw) {
    auto pairs = [&](float4 sv) {
        float dx[2], dy[2], dz[2], r2[2], f[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            pair_r2<MODE>(sv.x, sv.y, sv.z, kx[u], ky[u], kz[u], pc, dx[u], dy[u], dz[u], r2[u], tw[u]);
            f[u] = r2[u];
        }
        pair_f<SOFT>(f[0], f[1]);
#pragma unroll
        for (int u = 0; u < 2; u++)
            pair_sum(pair_g<SOFT, MODE>(r2[u], f[u], pc), dx[u], dy[u], dz[u], tx[u], ty[u], tz[u]);
    };
    constexpr int kAhead = 2;  // reads in flight
    int i = 0;
    for (; i + kAhead <= full; i += kAhead) {
        float4 sv[kAhead];
#pragma unroll
        for (int q = 0; q < kAhead; q++) sv[q] = bp[(i + q) * G + grp];
#pragma unroll
        for (int q = 0; q < kAhead; q++) pairs(sv[q]);
    }
    for (; i * G < cnt; i++) {  // the last steps: a group past the block's sources takes a padding source
        float4 sv = bp[min(i * G + grp, kWave - 1)];
        if (i * G + grp >= cnt) sv.x = kFar;
        pairs(sv);
    }
}

// block: the wave's 64 float4 in LDS.
template <int SOFT, bool CENSUS>
__device__ __forceinline__ void tail_item(const BatchCtx &cx, const SicView &v, const WorkItem &w, float4 *block,
                                          int lane, Census &cen) {
    const NF_CONST float4 *src = cptr<float4>(v.sources4);
    NF_GLOBAL double *out = (NF_GLOBAL double *)v.partial;
    const int s = w.sinkset;
    const int base = cptr<int32_t>(v.sink_set_start)[s] + w.first;
    const SourceRows rows = source_rows(v, s, lane);
    const int r = w.nsink;
    const int L = (r + 1) / 2, G = kWave / L;
    const int g = lane / L, slot = lane - g * L;
    const int grp = min(g, G - 1);  // (lanes past the last group repeat it, and join no sum)
    const SinkCells sc = sink_cells(v, s);
    float kx[2], ky[2], kz[2];
    float blx = __builtin_huge_valf(), bly = blx, blz = blx, bhx = -blx, bhy = -blx, bhz = -blx;
#pragma unroll
    for (int u = 0; u < 2; u++) {  // (an odd r repeats its last sink in the free slot, not stored)
        const float3 k = pencil_sink(v, sc, w.first + min(slot + u * L, r - 1), cx.invcpd);
        kx[u] = k.x;
        ky[u] = k.y;
        kz[u] = k.z;
        blx = fminf(blx, k.x);
        bly = fminf(bly, k.y);
        blz = fminf(blz, k.z);
        bhx = fmaxf(bhx, k.x);
        bhy = fmaxf(bhy, k.y);
        bhz = fmaxf(bhz, k.z);
    }
    blz = wave_min(blz);
    bhz = wave_max(bhz);
    const SinkBox kbox = {wave_min(blx), wave_min(bly), wave_max(bhx), wave_max(bhy), blz, bhz, blz, bhz};
    double h[2][4] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
    const int W = v.W, full64 = kWave / G;
    // The next block's sources, one to a lane: from block `at` on (the blocks
    // of a pencil follow each other; ny, nleft: its pencil and blocks to come).
    int ny = -1, nleft = 0, at = 0;
    float4 ahead = make_float4(kFar, 0.f, 0.f, 0.f);
    auto load_next = [&] {
        while (nleft == 0 && ++ny < W) {
            nleft = (rows.count_of(ny) + kWave - 1) / kWave;
            at = rows.start_of(ny);
        }
        if (ny >= W) return;
        ahead = src[at + lane];
        at += kWave;
        nleft--;
    };
    load_next();
    int modes = 0, p = 0;
    for (int y = 0; y < W; y++) {
        const int n = rows.count_of(y);
        const double yo = (double)(y - v.R) * cx.invcpd;
        float kyy[2];
#pragma unroll
        for (int u = 0; u < 2; u++) kyy[u] = (float)((double)ky[u] - yo);
        const int nblk = (n + kWave - 1) / kWave;
        for (int b = 0; b < nblk; b++, p++) {
            if ((p & (kWave - 1)) == 0) modes = block_forms<SOFT, false>(cx, v, rows, kbox, p, lane);
            const int mode = __builtin_amdgcn_readlane(modes, p & (kWave - 1)) & 3;
            const int cnt = min(kWave, n - b * kWave);
            if constexpr (CENSUS) {
                census_add(cen, mode, (uint64_t)r * (uint64_t)cnt);
                cen.tail += (uint64_t)r * (uint64_t)cnt;
            }
            // (LDS is in order within the wave: the block's reads follow its
            // write, and the next block's write follows them.)
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            block[lane] = ahead;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            load_next();
            const float4 *bp = block;
            const int full = cnt == kWave ? full64 : cnt / G;
            float tx[2] = {0.f, 0.f}, ty[2] = {0.f, 0.f}, tz[2] = {0.f, 0.f}, tw[2] = {0.f, 0.f};
            if (mode == kNoDensity)
                tail_block<SOFT, kNoDensity>(bp, cnt, G, full, grp, kx, kyy, kz, cx.pc, tx, ty, tz, tw);
            else if (mode == kDensity)
                tail_block<SOFT, kDensity>(bp, cnt, G, full, grp, kx, kyy, kz, cx.pc, tx, ty, tz, tw);
            else
                tail_block<SOFT, kExact>(bp, cnt, G, full, grp, kx, kyy, kz, cx.pc, tx, ty, tz, tw);
#pragma unroll
            for (int u = 0; u < 2; u++) {
                h[u][0] += (double)tx[u];
                h[u][1] += (double)ty[u];
                h[u][2] += (double)tz[u];
                h[u][3] += (double)tw[u];
            }
        }
    }
    // The last block's reads come before whatever the wave's next item writes
    // there: full_item's sums are doubles, which the compiler may take for
    // other memory than these float4.
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int m = G; m > 1;) {  // groups [half, m) onto [0, m - half)
        const int half = (m + 1) / 2;
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const double o = __shfl(h[u][c], lane + half * L);
                if (g + half < m) h[u][c] += o;
            }
        m = half;
    }
    if (g > 0) return;
#pragma unroll
    for (int u = 0; u < 2; u++) {
        if (slot + u * L >= r) continue;
        NF_GLOBAL double *o = out + 4 * (int64_t)(base + slot + u * L);
#pragma unroll
        for (int c = 0; c < 4; c++) o[c] = h[u][c];
    }
}

// Occupancy target WPE (waves per SIMD): more resident waves hide the v_rsq
// and scalar-load latencies, as long as the tile loops' registers fit (6 waves:
// 80 VGPRs; 4: 128).  Only the cubic spline spills VGPRs, 4 of them at S = 1 and
// 2; S = 4 keeps 4 waves, which measured faster than 5.
constexpr int batched_waves_per_eu(int /*soft*/, int s) { return s == 4 ? 4 : 6; }

}  // namespace

int batched_kernel_waves(int softening, int sinks_per_lane) {
    return batched_waves_per_eu(softening, sinks_per_lane);
}

namespace {

// Persistent kernel: every wave pops items (of any SIC of the group) until
// the queue is empty.  CENSUS: count the pair interactions of each pair form
// into census (the diagnostic instantiations; the results are the same).
// nitems < 0 means a list of at most -nitems items whose length the prologue
// wrote into counter[1]; a census build adds its counts into the four uint64
// at counter + kCensusOffset.
//
// Wave g takes item g first, without an atomic, then pops the rest of the list
// from queue g mod kQueues, whose items are every kQueues-th one.  Atomics on
// one address retire one per 11.7 ns (28 cycles) whatever the grid, so a
// single queue held 6,144 waves for 72 us at their first pop and a list of
// short items (133,000 in a launch group of sparse cells) for 1.6 ms; 16
// queues on cache lines of their own pop 16 times as fast.  Waves do not look
// into other queues when theirs is empty: the queues deal the cost-sorted list
// out item by item, so they end within about an item of each other.  (Dealing
// it to one queue per XCD in chunks of 8 to 128 consecutive items, which share
// source pencils, measured 11% slower.)
template <int SOFT, int S, int WPE, bool CENSUS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, 8))) void k_batched(
    BatchCtx cx, const SicView *__restrict__ views, const WorkItem *__restrict__ items, int32_t nitems,
    int32_t *__restrict__ counter) {
    const int lane = threadIdx.x & (kWave - 1);
    extern __shared__ double hsums[];  // per wave 4 S x 64: full_item's sums over the source pencils
    double *const hsum = hsums + (threadIdx.x / kWave) * (4 * S * kWave) + lane;
    if (nitems < 0) nitems = min(-nitems, *cptr<int32_t>(counter + 1));
    Census cen = {{0, 0, 0}, 0};
    const int wpw = blockDim.x / kWave, nwaves = gridDim.x * wpw;
    const int g = __builtin_amdgcn_readfirstlane(blockIdx.x * wpw + (int)(threadIdx.x / kWave));
    const int nq = min(kQueues, nwaves), q = g % nq;  // (a grid of fewer waves serves as many queues)
    int it = g;
    for (;;) {
        if (it >= nitems) {
            if (CENSUS && lane == 0) {
                unsigned long long *census = reinterpret_cast<unsigned long long *>(counter + kCensusOffset);
                for (int f = 0; f < 3; f++)
                    if (cen.form[f]) atomicAdd(census + f, (unsigned long long)cen.form[f]);
                if (cen.tail) atomicAdd(census + 3, (unsigned long long)cen.tail);
            }
            return;
        }
        const WorkItem w = cptr<WorkItem>(items)[it];
        const int kind = w.kind_sic & 3;
        const SicView v = cptr<SicView>(views)[w.kind_sic >> 2];
        if (kind == 0) {
            full_item<SOFT, S, CENSUS>(cx, v, w, w.nsink, 0, v.W, hsum, lane, cen);
        } else if (kind >= 2) {  // one-wave tiles, whole or against one source pencil
            const int y = w.nsink >> 8;
            full_item<SOFT, 1, CENSUS>(cx, v, w, w.nsink & 255, y, kind == 2 ? v.W : y + 1, hsum, lane, cen);
        } else tail_item<SOFT, CENSUS>(cx, v, w, reinterpret_cast<float4 *>(hsum - lane), lane, cen);
        int j = 0;
        if (lane == 0) j = atomicAdd(counter + kQueueOffset + q * kQueueStride, 1);
        it = nwaves + __builtin_amdgcn_readfirstlane(j) * nq + q;
    }
}

// The batched launch's prologue where no gather before it cleared the queues
// (a kernel, so that it can sit in a captured graph).
__global__ void k_zero_counter(QueueClear qc) { clear_queues(qc, threadIdx.x); }

// Pair-math probe: the register-tile loop of k_batched alone (16-source batch
// sums, 64-source FP32 tile sums accumulated in FP64), one pair form for
// every block, on sinks and sources that stay in the caches.  Each wave holds
// 64 S sinks and makes `passes` passes over `nsrc` sources (a multiple of
// 64); lane 0 of each wave stores a checksum so that nothing is optimised
// away.  Its rate is the ceiling of the tile loop at that tile and occupancy.
template <int SOFT, int S, int MODE, int WPE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE, 8))) void k_probe(
    PairConst pc, const float4 *__restrict__ src, int nsrc, int passes, double *__restrict__ out) {
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = blockIdx.x * (blockDim.x / kWave) + (int)(threadIdx.x / kWave);
    float kx[S], ky[S], kz[S];
#pragma unroll
    for (int u = 0; u < S; u++) {  // sinks spread over a cell-sized box around the sources
        const int i = lane + kWave * u + 7 * wave;
        kx[u] = 0.004f * (float)((i * 37) % 101) / 101.f - 0.002f;
        ky[u] = 0.004f * (float)((i * 53) % 103) / 103.f - 0.002f;
        kz[u] = 0.004f * (float)((i * 71) % 107) / 107.f - 0.002f;
    }
    double hx[S], hy[S], hz[S], hw[S];
#pragma unroll
    for (int u = 0; u < S; u++) hx[u] = hy[u] = hz[u] = hw[u] = 0.0;
    const NF_CONST float4 *sp = cptr<float4>(src);
    for (int p = 0; p < passes; p++)
        for (int b = 0; b < nsrc; b += kWave) {
            float tx[S], ty[S], tz[S], tw[S];
#pragma unroll
            for (int u = 0; u < S; u++) tx[u] = ty[u] = tz[u] = tw[u] = 0.f;
            full_tile<SOFT, MODE, MODE, S>(sp + b, kWave, kx, ky, kz, pc, tx, ty, tz, tw);
#pragma unroll
            for (int u = 0; u < S; u++) {
                hx[u] += (double)tx[u];
                hy[u] += (double)ty[u];
                hz[u] += (double)tz[u];
                hw[u] += (double)tw[u];
            }
        }
    double c = 0.0;
#pragma unroll
    for (int u = 0; u < S; u++) c += hx[u] + hy[u] + hz[u] + hw[u];
    for (int off = 32; off >= 1; off >>= 1) c += __shfl_xor(c, off);
    if (lane == 0) out[wave] = c;
}

template <int S, int MODE, int WPE>
int run_probe_t(const PairConst &pc, double *rate) {
    // 25 ms a launch at S = 2 on a full GPU: two passes, 0.4 ms, read 10-20% less
    // than the loop's rate (4.35e12 interactions/s unsoftened at 6 waves).
    constexpr int kSrc = 1024, kPasses = 128;
    int ncu = device_cu_count(), bpc = 0;
    if (ncu <= 0) return (int)hipErrorNoDevice;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&bpc, k_probe<NF_SOFT_SINGLE_SPLINE, S, MODE, WPE>,
                                                                256, 0);
    if (e != hipSuccess) return (int)e;
    const int grid = ncu * std::max(1, bpc);
    float4 h[kSrc];
    for (int i = 0; i < kSrc; i++)  // sources in the same box, none within the softening of a sink
        h[i] = make_float4(0.004f * (float)((i * 29) % 97) / 97.f - 0.002f + 2e-5f,
                           0.004f * (float)((i * 31) % 89) / 89.f - 0.002f + 2e-5f,
                           0.004f * (float)((i * 43) % 83) / 83.f - 0.002f + 2e-5f, 0.f);
    float4 *src = nullptr;
    double *out = nullptr;
    hipEvent_t a = nullptr, b = nullptr;
    float ms = 0.f;
    if ((e = hipMalloc(&src, sizeof h)) == hipSuccess && (e = hipMalloc(&out, sizeof(double) * grid * 4)) == hipSuccess &&
        (e = hipMemcpy(src, h, sizeof h, hipMemcpyHostToDevice)) == hipSuccess &&
        (e = hipEventCreate(&a)) == hipSuccess && (e = hipEventCreate(&b)) == hipSuccess) {
        // a warm-up launch, then the timed one
        hipLaunchKernelGGL((k_probe<NF_SOFT_SINGLE_SPLINE, S, MODE, WPE>), dim3(grid), dim3(256), 0, nullptr, pc, src,
                           kSrc, kPasses, out);
        (void)hipEventRecord(a, nullptr);
        hipLaunchKernelGGL((k_probe<NF_SOFT_SINGLE_SPLINE, S, MODE, WPE>), dim3(grid), dim3(256), 0, nullptr, pc, src,
                           kSrc, kPasses, out);
        (void)hipEventRecord(b, nullptr);
        e = hipEventSynchronize(b);
        if (e == hipSuccess) e = hipEventElapsedTime(&ms, a, b);
    }
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
    if (src) (void)hipFree(src);
    if (out) (void)hipFree(out);
    if (e != hipSuccess) return (int)e;
    *rate = (double)grid * 4.0 * 64.0 * S * (double)kSrc * kPasses / (ms * 1e-3);
    return 0;
}

template <int SOFT>
int launch_plain_t(const DevPlan &pl, const PairConst &pc, const void *sinks4, const void *sources4, void *partial4,
                   hipStream_t st) {
    if (pl.nsink_blocks == 0) return 0;
    hipLaunchKernelGGL(k_plain<SOFT>, dim3(pl.nsink_blocks), dim3(kWave), 0, st, pl, pc, form_radii(SOFT, pc, pc.b2),
                       static_cast<const float4 *>(sinks4), static_cast<const float4 *>(sources4),
                       static_cast<float4 *>(partial4));
    return (int)hipGetLastError();
}

}  // namespace

int device_cu_count() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return n;
}

int launch_gather(const DevPlan &pl, const DevSlabs &sl, bool batched_stream, void *sinks4, void *sources4,
                  const QueueClear &qc, void *stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    const float cellsize = (float)(1.0 / (double)pl.cpd);
    const double invcpd = 1.0 / (double)pl.cpd;
    float4 *box = static_cast<float4 *>(box_after(sources4, pl.nsrc_blocks));
    auto grid_of = [](int blocks, int per_wave = kGatherBlocks) {  // 4 waves per workgroup
        return dim3((unsigned)((blocks + 4 * per_wave - 1) / (4 * per_wave)));
    };
    if (sinks4 && pl.nsink_blocks > 0) {
        const dim3 grid = grid_of(pl.nsink_blocks);
        hipLaunchKernelGGL(k_gather_sinks, grid, dim3(256), 0, st, pl, sl.pos[pl.R], sl.n[pl.R], sl.aos,
                           static_cast<float4 *>(sinks4), cellsize);
    }
    if (pl.nsrc_blocks > 0) {
        const dim3 grid = grid_of(pl.nsrc_blocks);
        if (batched_stream) {
            const dim3 bgrid((unsigned)((gather_waves(pl.nsrc_sets, pl.nsrc_blocks, pl.max_src_blocks) + 3) / 4));
            if (gather_segmented(pl.max_src_blocks))
                hipLaunchKernelGGL(k_gather_sources_binned<true>, bgrid, dim3(256), 0, st, pl, sl,
                                   static_cast<float4 *>(sources4), box, (float)pl.cpd, invcpd, qc);
            else
                hipLaunchKernelGGL(k_gather_sources_binned<false>, bgrid, dim3(256), 0, st, pl, sl,
                                   static_cast<float4 *>(sources4), box, (float)pl.cpd, invcpd, qc);
        }
        else
            hipLaunchKernelGGL(k_gather_sources, grid, dim3(256), 0, st, pl, sl, static_cast<float4 *>(sources4),
                               box, cellsize);
    }
    return (int)hipGetLastError();
}

int launch_gather_group(const GroupSic *g, const int32_t *first, int n, int total, int cpd, bool segmented,
                        const QueueClear &qc, void *stream) {
    if (total <= 0) return 0;
    const dim3 grid((unsigned)((total + 3) / 4));
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (segmented)
        hipLaunchKernelGGL(k_gather_sources_binned_group<true>, grid, dim3(256), 0, st, g, first, n, (float)cpd,
                           1.0 / (double)cpd, qc);
    else
        hipLaunchKernelGGL(k_gather_sources_binned_group<false>, grid, dim3(256), 0, st, g, first, n, (float)cpd,
                           1.0 / (double)cpd, qc);
    return (int)hipGetLastError();
}

int launch_coadd_group(const GroupSic *g, const int32_t *first, int n, int total, int lanes, bool planes,
                       void *stream) {
    if (total <= 0) return 0;
    const auto kern = lanes == 16 ? (planes ? k_coadd_f64_group<16, true> : k_coadd_f64_group<16, false>)
                                  : (planes ? k_coadd_f64_group<64, true> : k_coadd_f64_group<64, false>);
    hipLaunchKernelGGL(kern, dim3((unsigned)((total + 3) / 4)), dim3(256), 0, static_cast<hipStream_t>(stream), g,
                       first, n);
    return (int)hipGetLastError();
}

int launch_plain(const DevPlan &pl, int softening, const PairConst &pc, const void *sinks4, const void *sources4,
                 void *partial4, void *stream) {
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (softening) {
        case NF_SOFT_PLUMMER: return launch_plain_t<NF_SOFT_PLUMMER>(pl, pc, sinks4, sources4, partial4, st);
        case NF_SOFT_SINGLE_SPLINE:
            return launch_plain_t<NF_SOFT_SINGLE_SPLINE>(pl, pc, sinks4, sources4, partial4, st);
        case NF_SOFT_CUBIC_SPLINE:
            return launch_plain_t<NF_SOFT_CUBIC_SPLINE>(pl, pc, sinks4, sources4, partial4, st);
        case NF_SOFT_CUBIC_PLUMMER:
            return launch_plain_t<NF_SOFT_CUBIC_PLUMMER>(pl, pc, sinks4, sources4, partial4, st);
        default: return (int)hipErrorInvalidValue;
    }
}

int launch_coadd_plain(const DevPlan &pl, const void *partial4, float *acc4, const KickArgs &kick, int lanes,
                       void *stream) {
    if (pl.n_coadd_chunks == 0) return 0;
    const dim3 grid((unsigned)((group_coadd_waves(pl, lanes) + 3) / 4));
    hipStream_t st = static_cast<hipStream_t>(stream);
    const float4 *part = static_cast<const float4 *>(partial4);
    float4 *acc = reinterpret_cast<float4 *>(acc4);
    if (lanes == 16) hipLaunchKernelGGL(k_coadd_plain<16>, grid, dim3(256), 0, st, pl, part, acc, kick);
    else hipLaunchKernelGGL(k_coadd_plain<64>, grid, dim3(256), 0, st, pl, part, acc, kick);
    return (int)hipGetLastError();
}

int launch_coadd_f64(const DevPlan &pl, const void *partial_d4, double out_scale, float *acc4,
                     const KickArgs &kick, int lanes, void *stream) {
    if (pl.n_coadd_chunks == 0) return 0;
    const dim3 grid((unsigned)((group_coadd_waves(pl, lanes) + 3) / 4));
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool planes = pl.y_plane != 0;
    const auto kern = lanes == 16 ? (planes ? k_coadd_f64<16, true> : k_coadd_f64<16, false>)
                                  : (planes ? k_coadd_f64<64, true> : k_coadd_f64<64, false>);
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, pl, static_cast<const double *>(partial_d4), out_scale,
                       reinterpret_cast<float4 *>(acc4), kick);
    return (int)hipGetLastError();
}

template <int SOFT, int S, bool CENSUS>
static int launch_batched_k(const BatchCtx &cx, const TileShape &ts, const SicView *views, const WorkItem *items,
                            int32_t nitems, const QueueClear &qc, bool cleared, hipStream_t st) {
    constexpr auto kern = k_batched<SOFT, S, batched_waves_per_eu(SOFT, S), CENSUS>;
    // Workgroups of 1, 2 or 4 waves; each wave pops its own items, so the
    // size only changes how the dispatcher places the persistent grid.
    const int wpw = ts.waves_per_wg == 1 || ts.waves_per_wg == 2 ? ts.waves_per_wg : 4;
    const int threads = kWave * wpw;
    const size_t lds = sizeof(double) * 4 * S * threads;
    int blocks_per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks_per_cu, kern, threads, lds) != hipSuccess ||
        blocks_per_cu <= 0)
        blocks_per_cu = 1;
    if (ts.waves_per_cu > 0) blocks_per_cu = std::max(1, std::min(blocks_per_cu, ts.waves_per_cu / wpw));
    const int ncu = device_cu_count();
    int grid = std::max(1, ncu) * blocks_per_cu;
    const int need = (nitems + wpw - 1) / wpw;
    if (grid > need) grid = std::max(1, need);
    static_assert(kCensusBytes + 32 <= kQueueBytes && kQueues <= kWave, "census before the queues, one lane per queue");
    if (!cleared) hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(kWave), 0, st, qc);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, st, cx, views, items, qc.dnitems ? -nitems : nitems,
                       qc.counter);
    return (int)hipGetLastError();
}

template <int SOFT, int S>
static int launch_batched_s(const BatchCtx &cx, const TileShape &ts, const SicView *views, const WorkItem *items,
                            int32_t nitems, const QueueClear &qc, bool cleared, hipStream_t st) {
    if (qc.census) return launch_batched_k<SOFT, S, true>(cx, ts, views, items, nitems, qc, cleared, st);
    return launch_batched_k<SOFT, S, false>(cx, ts, views, items, nitems, qc, cleared, st);
}

template <int SOFT>
static int launch_batched_soft(const BatchCtx &cx, const TileShape &ts, const SicView *views, const WorkItem *items,
                               int32_t nitems, const QueueClear &qc, bool cleared, hipStream_t st) {
    switch (ts.sinks_per_lane) {
        case 1: return launch_batched_s<SOFT, 1>(cx, ts, views, items, nitems, qc, cleared, st);
        case 2: return launch_batched_s<SOFT, 2>(cx, ts, views, items, nitems, qc, cleared, st);
        case 4: return launch_batched_s<SOFT, 4>(cx, ts, views, items, nitems, qc, cleared, st);
        default: return (int)hipErrorInvalidValue;
    }
}

// The single-spline pair-math probe at (sinks per lane, pair form, waves per
// SIMD): pair interactions per second over the whole GPU.
int run_pair_probe(const PairConst &pc, int sinks_per_lane, int mode, int waves_per_simd, double *rate) {
#define NF_PROBE(S_, M_, W_) \
    if (sinks_per_lane == S_ && mode == M_ && waves_per_simd == W_) return run_probe_t<S_, M_, W_>(pc, rate);
#define NF_PROBE_W(S_, M_) NF_PROBE(S_, M_, 4) NF_PROBE(S_, M_, 6) NF_PROBE(S_, M_, 8)
#define NF_PROBE_M(S_) NF_PROBE_W(S_, kNoDensity) NF_PROBE_W(S_, kDensity) NF_PROBE_W(S_, kExact)
    NF_PROBE_M(1)
    NF_PROBE_M(2)
    NF_PROBE_M(4)
#undef NF_PROBE_M
#undef NF_PROBE_W
#undef NF_PROBE
    return (int)hipErrorInvalidValue;
}

int launch_batched(const SicView *views, int cpd, int softening, const PairConst &pc, const TileShape &ts,
                   const WorkItem *items, int32_t nitems, const QueueClear &qc, bool cleared, void *stream) {
    if (nitems == 0) return 0;
    hipStream_t st = static_cast<hipStream_t>(stream);
    BatchCtx cx;
    cx.pc = pc;
    cx.invcpd = 1.0 / (double)cpd;
    cx.fr = form_radii(softening, pc, pc.b2x);  // (density is nonzero only for r^2 + r2add < b2x)
    switch (softening) {
        case NF_SOFT_PLUMMER: return launch_batched_soft<NF_SOFT_PLUMMER>(cx, ts, views, items, nitems, qc, cleared, st);
        case NF_SOFT_SINGLE_SPLINE:
            return launch_batched_soft<NF_SOFT_SINGLE_SPLINE>(cx, ts, views, items, nitems, qc, cleared, st);
        case NF_SOFT_CUBIC_SPLINE:
            return launch_batched_soft<NF_SOFT_CUBIC_SPLINE>(cx, ts, views, items, nitems, qc, cleared, st);
        case NF_SOFT_CUBIC_PLUMMER:
            return launch_batched_soft<NF_SOFT_CUBIC_PLUMMER>(cx, ts, views, items, nitems, qc, cleared, st);
        default: return (int)hipErrorInvalidValue;
    }
}

}  // namespace nf
