// Batched ensembles: many independent simulations of uneven grid size and
// particle count advance together, two launches for the particles and four for
// the fields.
//
// Storage: every simulation's particle planes are a slice of one set of batch
// planes (PicBatchSim::particle_offset) and every field component a slice of
// one batch array (PicBatchSim::field_offset), each in the single-simulation
// layout.  The descriptor table lives in device memory.
//
// Particle phase: a work list of (simulation, block) items covers every
// simulation's slots in blocks of kThreads * rounds.  Items of first-order 1-D and
// 2-D members take a block each (planar_chunk, as the single simulation does); a
// fixed grid of persistent blocks walks the list for the others (fused_block_boxed).
//
// Field phase: the grid part of time_loop_electrodynamic's Esirkepov branch
// (evolve.py:70-97) as four launches over all members: J fold, B half step with
// J's guard cells, E step, B half step, none of which needs a barrier inside.
#include "pic_field_ops.h"
#include "pic_planar.h"

#include <algorithm>

namespace {

constexpr int kFieldThreads = 256;
// Blocks of a pass, shared out over the members.  A block costs 3.6 ns to start
// whether it has points or not, and four a CU hide the latency: the four passes
// of 2048 members of 64 cells take 161 us with one block a member, 304 with four
// and 717 with sixteen; 256 of 32 x 32 167 / 87 / 128; one of 512 x 512 69 with
// 1024, 466 with 64.
constexpr int kFieldBlocks = 1024;

struct BatchFields {
    const float* E[3];
    float* B[3];
    float* Bh[3];
    float* J[3];
    float* Eo[3];
};

__device__ inline FieldPtrs batch_field_ptrs(const float* const E[3], const float* const B[3], int64_t off) {
    FieldPtrs fp;
    for (int c = 0; c < 3; ++c) {
        fp.E[c] = E[c] + off;
        fp.B[c] = B[c] + off;
        fp.Ee[c] = nullptr;
        fp.Be[c] = nullptr;
    }
    return fp;
}

__device__ inline PicParticles offset_particles(const PicParticles& p, int64_t off) {
    PicParticles q;
    for (int a = 0; a < 3; ++a) {
        q.x[a] = p.x[a] + off;
        q.u[a] = p.u[a] + off;
    }
    q.active = p.active + off;
    return q;
}

struct BatchParticleArgs {
    PicParticles in, out;
    const float* E[3];
    const float* B[3];
    float* J[3];
};

// A member's table entry as constant memory: the kernels do not write the
// table, and without saying so each of its values is loaded again, by vector
// loads, after every store.
__device__ inline const PicBatchSim& member(const PicBatchSim* sims, int sim) {
    typedef const __attribute__((address_space(4))) PicBatchSim ConstSim;
    return *(const PicBatchSim*)((ConstSim*)(sims + __builtin_amdgcn_readfirstlane(sim)));
}

// Whether any of the block's work items (every gridDim.x-th) is left by the planar kernel.
__device__ inline bool any_item(const PicBatchSim* __restrict__ sims, const int32_t* __restrict__ work,
                                int32_t n_work) {
    bool any = false;
    for (int64_t w = blockIdx.x + (int64_t)threadIdx.x * gridDim.x; w < n_work; w += (int64_t)kThreads * gridDim.x)
        any = any || !planar_covers(sims[work[2 * w]].desc);
    return __syncthreads_or(any) != 0;
}

// The items of first-order 1-D and 2-D members, a block each: the chunks of planar_kernel.
template <int kRounds>
__global__ __launch_bounds__(kPlanarBlock, 2) void batch_planar_kernel(const PicBatchSim* __restrict__ sims,
                                                                   const int32_t* __restrict__ work,
                                                                   BatchParticleArgs args) {
    constexpr int kP = kRounds == 2 ? 1 : 2, kChunk = kPlanarBlock * kP;
    __shared__ PlanarShared<kP, kPlanarBlock> sh;
    const int32_t w = blockIdx.x;
    const PicBatchSim& bs = member(sims, work[2 * w]);
    const PicDesc& d = bs.desc;
    const int kind = fused_kind(d);
    if (kind == 1 || kind == 2) {
        const int64_t poff = bs.particle_offset, foff = bs.field_offset;
        const int64_t n = (int64_t)bs.species.count * bs.species.slots;
        const PicParticles in = offset_particles(args.in, poff);
        const PicParticles out = offset_particles(args.out, poff);
        const FieldPtrs fp = batch_field_ptrs(args.E, args.B, foff);
        float* const J[3] = {args.J[0] + foff, args.J[1] + foff, args.J[2] + foff};
        const bool vec_ok = groups_aligned(in, out);
        for (int r = 0; r < kThreads * kRounds / kChunk; ++r) {
            const uint32_t base = (uint32_t)work[2 * w + 1] * (uint32_t)(kThreads * kRounds) + (uint32_t)(r * kChunk);
            if (base >= n) break;
            if (kind == 2) planar_chunk<2, kP, kPlanarBlock>(d, bs.species, in, fp, out, J, n, base, vec_ok, sh);
            else planar_chunk<1, kP, kPlanarBlock>(d, bs.species, in, fp, out, J, n, base, vec_ok, sh);
        }
    }
}

// The other items: fused_block_boxed (J accumulated in an LDS box sized to the
// item's particles).
template <int kRounds>
__global__ __launch_bounds__(kThreads, 1) void batch_fused_kernel(const PicBatchSim* __restrict__ sims,
                                                                  const int32_t* __restrict__ work, int32_t n_work,
                                                                  BatchParticleArgs args) {
    __shared__ FusedShared<kRounds> sh;
    __shared__ float box[kRangeBoxCap];
    __shared__ int bmin[3], bmax[3];
    if (!any_item(sims, work, n_work)) return;
    for (int32_t w = blockIdx.x; w < n_work; w += gridDim.x) {
        const int sim = work[2 * w];
        const uint32_t blk = (uint32_t)work[2 * w + 1];
        const PicBatchSim& bs = sims[sim];
        const PicDesc& d = bs.desc;
        if (planar_covers(d)) continue;
        const int64_t poff = bs.particle_offset, foff = bs.field_offset;
        const int64_t n = (int64_t)bs.species.count * bs.species.slots;
        const PicParticles in = offset_particles(args.in, poff);
        const PicParticles out = offset_particles(args.out, poff);
        const FieldPtrs fp = batch_field_ptrs(args.E, args.B, foff);
        float* const J[3] = {args.J[0] + foff, args.J[1] + foff, args.J[2] + foff};
        const uint32_t base = blk * (uint32_t)(kThreads * kRounds);
        fused_block_boxed<kRounds>(d, bs.species, in, fp, out, J, n, base, sh, box, bmin, bmax);
        __syncthreads();   // the next item reuses the shared queue and box
    }
}

// Array point of number t in a box of e[] points from index o.
__device__ inline void box_point(const int e1, const int e2, int o, uint32_t t, int& i, int& j, int& k) {
    const uint32_t r = t / (uint32_t)e2;
    k = (int)(t - r * (uint32_t)e2) + o;
    j = (int)(r % (uint32_t)e1) + o;
    i = (int)(r / (uint32_t)e1) + o;
}

// Pass 0: J's guard cells folded into the interior with the particle codes
// (Esirkepov.py:357-359); 1: B_h = B - (dt/2) curl E (evolve.py:88) and J's
// guard cells; 2: E' = E + dt (C^2 curl B_h - J/eps) (:92); 3: B = B_h - (dt/2)
// curl E' (:96).  gridDim.x blocks share a member's points; blockIdx.y is the
// member.  Pass 0 has a thread per interior cell and component (a guard cell
// belongs to one cell, so nothing it reads is written by another); the others
// have a thread per array point, which stores the value of the interior point
// its coordinates map to.  1-D and 2-D members have 25 and 5 points a cell along
// their reduced axes, contiguous in memory: stored by the cell's own thread they
// took a strided store each, and the four passes of 2048 members of 64 cells
// 2.6 ms (a block per member with barriers between the passes: 397 us; now 161),
// of 64 members of 256 x 32 cells 152 (646, 141), of one of 512 x 512 1505 (15685,
// 69).
template <int kPass>
__global__ __launch_bounds__(kFieldThreads) void batch_field_kernel(const PicBatchSim* __restrict__ sims,
                                                                     BatchFields bf) {
    const PicDesc& d = member(sims, blockIdx.y).desc;
    const int64_t off = member(sims, blockIdx.y).field_offset;
    const uint32_t points = kPass == 0 ? (uint32_t)(d.n[0] * d.n[1] * d.n[2]) : (uint32_t)field_size(d);
    const uint32_t t0 = blockIdx.x * kFieldThreads + threadIdx.x, step = gridDim.x * kFieldThreads;
    if (blockIdx.x * kFieldThreads >= points) return;
    // FP64 divisions: by one thread of the block
    __shared__ YeeConst y;
    if (kPass != 0 && threadIdx.x == 0) y = yee_const(d);
    const float* E[3];
    float *B[3], *Bh[3], *J[3], *Eo[3];
    for (int c = 0; c < 3; ++c) {
        E[c] = bf.E[c] + off;
        B[c] = bf.B[c] + off;
        Bh[c] = bf.Bh[c] + off;
        J[c] = bf.J[c] + off;
        Eo[c] = bf.Eo[c] + off;
    }
    int mode[3], i, j, k;
    for (int a = 0; a < 3; ++a) mode[a] = refresh_mode(d, a, 1);
    if constexpr (kPass == 0) {
        int sign[3];
        for (int a = 0; a < 3; ++a) sign[a] = fold_sign(d, a, 1);
        float* const f = blockIdx.z == 0 ? J[0] : (blockIdx.z == 1 ? J[1] : J[2]);
        for (uint32_t t = t0; t < points; t += step) {
            box_point(d.n[1], d.n[2], d.g, t, i, j, k);
            if (has_images(d, 0, i) || has_images(d, 1, j) || has_images(d, 2, k))
                f[fidx(d, i, j, k)] = folded_at(d, mode, sign, f, i, j, k);
        }
    } else {
        __syncthreads();
        for (uint32_t t = t0; t < points; t += step) {
            box_point(d.dims[1], d.dims[2], 0, t, i, j, k);
            const int si = ghost_source(i, d.n[0], d.g, y.mode[0]), sj = ghost_source(j, d.n[1], d.g, y.mode[1]);
            const int sk = ghost_source(k, d.n[2], d.g, y.mode[2]);
            float v[3] = {0.0f, 0.0f, 0.0f};
            if (si >= 0 && sj >= 0 && sk >= 0) {
                if constexpr (kPass == 1) yee_b_value(d, y, E, B, v, si, sj, sk);
                else if constexpr (kPass == 2) yee_e_value(d, y, E, Bh, J, v, si, sj, sk);
                else yee_b_value(d, y, Eo, Bh, v, si, sj, sk);
            }
            float* const* out = kPass == 1 ? Bh : (kPass == 2 ? Eo : B);
            for (int c = 0; c < 3; ++c) out[c][t] = v[c];
            if constexpr (kPass == 1) {
                const int pi = ghost_source(i, d.n[0], d.g, mode[0]), pj = ghost_source(j, d.n[1], d.g, mode[1]);
                const int pk = ghost_source(k, d.n[2], d.g, mode[2]);
                if (pi == i && pj == j && pk == k) continue;
                const bool zero = pi < 0 || pj < 0 || pk < 0;
                const int64_t src = zero ? t : fidx(d, pi, pj, pk);
                for (int c = 0; c < 3; ++c) J[c][t] = zero ? 0.0f : J[c][src];
            }
        }
    }
}

bool batch_desc_ok(const PicDesc& d) {
    if (d.g < 1 || d.shape_factor < 1 || d.shape_factor > 2) return false;
    bool any = false;
    for (int a = 0; a < 3; ++a) {
        if (d.n[a] < 1 || d.dims[a] != d.n[a] + 2 * d.g) return false;
        if (d.n[a] > 1 && d.n[a] < d.g) return false;
        if (d.bc[a] != 0 || d.pbc[a] != 0) return false;   // periodic fields and particles
        any = any || d.n[a] > 1;
    }
    return any && d.alpha == 1.0;                           // digital filter is the identity
}

}  // namespace

extern "C" {

int pic_batch_check(const PicBatchSim* sims, int32_t n_sims, int64_t particle_slots, int64_t field_elems) {
    PIC_REQUIRE(sims && n_sims > 0);
    for (int32_t s = 0; s < n_sims; ++s) {
        const PicBatchSim& b = sims[s];
        PIC_REQUIRE(batch_desc_ok(b.desc));
        PIC_REQUIRE(b.species.count >= 1 && b.species.count <= PIC_MAX_SPECIES && b.species.slots >= 0);
        const int64_t n = (int64_t)b.species.count * b.species.slots;
        PIC_REQUIRE(b.particle_offset >= 0 && b.particle_offset + n <= particle_slots);
        PIC_REQUIRE(b.field_offset >= 0 && b.field_offset + field_size(b.desc) <= field_elems);
        PIC_REQUIRE(n < ((int64_t)1 << 31) - 8 * kThreads && field_size(b.desc) < ((int64_t)1 << 31));
    }
    return 0;
}

int pic_batch_fused_push_esirkepov(const PicBatchSim* sims, const int32_t* work, int32_t n_work, int32_t rounds,
                                   int32_t grid, const PicParticles* in, const float* const E[3],
                                   const float* const B[3], PicParticles* out, float* const J[3], void* stream) {
    PIC_REQUIRE(sims && work && n_work >= 0 && grid > 0 && in && out && E && B && J);
    PIC_REQUIRE(rounds == 2 || rounds == 4 || rounds == 8);
    for (int a = 0; a < 3; ++a) PIC_REQUIRE(E[a] && B[a] && J[a] && in->x[a] != out->x[a] && in->u[a] != out->u[a]);
    PIC_REQUIRE(in->active != out->active);
    if (n_work == 0) return 0;
    BatchParticleArgs args;
    args.in = *in;
    args.out = *out;
    for (int c = 0; c < 3; ++c) {
        args.E[c] = E[c];
        args.B[c] = B[c];
        args.J[c] = J[c];
    }
    hipStream_t st = as_stream(stream);
    const int g = grid < n_work ? grid : n_work;
    // items of a launch with a block each: a launch of 2^32 threads would run the remainder only, without an error
    constexpr int32_t kItems = 1 << 22;
    static_assert((int64_t)kItems * kPlanarBlock < ((int64_t)1 << 32), "threads of a launch");
#define PIC_BATCH_FUSED(R)                                                                                       \
    do {                                                                                                         \
        for (int32_t at = 0; at < n_work; at += std::min(kItems, n_work - at))                                   \
            hipLaunchKernelGGL(batch_planar_kernel<R>, dim3((unsigned)std::min(kItems, n_work - at)),            \
                               dim3(kPlanarBlock), 0, st, sims, work + 2 * (int64_t)at, args);                   \
        hipLaunchKernelGGL(batch_fused_kernel<R>, dim3(g), dim3(kThreads), 0, st, sims, work, n_work, args);     \
    } while (0)
    if (rounds == 2) PIC_BATCH_FUSED(2);
    else if (rounds == 4) PIC_BATCH_FUSED(4);
    else PIC_BATCH_FUSED(8);
#undef PIC_BATCH_FUSED
    PIC_CHECK_LAUNCH();
    return 0;
}

int pic_batch_field_step(const PicBatchSim* sims, int32_t n_sims, const float* const E_in[3], float* const B[3],
                         float* const B_half[3], float* const J[3], float* const E_out[3], void* stream) {
    PIC_REQUIRE(sims && n_sims > 0 && E_in && B && B_half && J && E_out);
    BatchFields bf;
    for (int c = 0; c < 3; ++c) {
        PIC_REQUIRE(E_in[c] && B[c] && B_half[c] && J[c] && E_out[c]);
        bf.E[c] = E_in[c];
        bf.B[c] = B[c];
        bf.Bh[c] = B_half[c];
        bf.J[c] = J[c];
        bf.Eo[c] = E_out[c];
    }
    for (int c = 0; c < 3; ++c)
        for (int e = 0; e < 3; ++e) PIC_REQUIRE((const float*)E_out[e] != E_in[c] && B_half[e] != B[c]);
    hipStream_t st = as_stream(stream);
    constexpr int kRowsMax = 65535;      // members per launch (grid rows)
    for (int32_t first = 0; first < n_sims; first += kRowsMax) {
        const PicBatchSim* part = sims + first;
        const int members = n_sims - first < kRowsMax ? n_sims - first : kRowsMax;
        const int per = std::max(kFieldBlocks / members, 1);
        const dim3 grid((unsigned)per, (unsigned)members), fold((unsigned)per, (unsigned)members, 3);
        hipLaunchKernelGGL(batch_field_kernel<0>, fold, dim3(kFieldThreads), 0, st, part, bf);
        hipLaunchKernelGGL(batch_field_kernel<1>, grid, dim3(kFieldThreads), 0, st, part, bf);
        hipLaunchKernelGGL(batch_field_kernel<2>, grid, dim3(kFieldThreads), 0, st, part, bf);
        hipLaunchKernelGGL(batch_field_kernel<3>, grid, dim3(kFieldThreads), 0, st, part, bf);
    }
    PIC_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
