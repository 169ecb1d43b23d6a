// Single-simulation launch of the fused particle phase (the block function
// and its design notes live in pic_fused_block.h).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "pic_exact_grid.h"
#include "pic_fused_block.h"
#include "pic_planar.h"

namespace {

// kRounds: particle slots per thread (block = kThreads * kRounds slots);
// kMinBlocks: resident-block target handed to the register allocator.
template <int kDims, int kRounds, int kMinBlocks>
__global__ __launch_bounds__(kThreads, kMinBlocks) void fused_push_esirkepov_v2(PicDesc d, PicSpecies sp,
                                                                                 PicParticles in, FieldPtrs fp,
                                                                                 PicParticles out, float* Jx,
                                                                                 float* Jy, float* Jz, int64_t n) {
    __shared__ FusedShared<kRounds> sh;
    const uint32_t base = blockIdx.x * (uint32_t)(kThreads * kRounds);   // n < 2^31 is checked at launch
    const GlobalSink sink{{Jx, Jy, Jz}};
    fused_block<kDims, kRounds>(d, sp, in, fp, out, sink, n, base, sh);
}

// Tile-ordered launch (particles sorted by pic_tile_keys): block b owns the
// slot range [starts[b], starts[b+1]) of one (species, tile) pair, i.e. the
// particles that were in that T^3-cell tile at the last sort.  Run sums and
// face-crossing deposits accumulate in an LDS box of (T+4)^3 nodes per
// component (the tile, one node below and three above for drift and the
// crossing frame); deposits that fall outside it go straight to J.  The box is
// added into J once per block, so J atomics scale with the tile surface
// instead of with the number of runs.
struct TileGeom {
    int T;
    int tiles;          // tiles per species
    int nt[3];          // tiles per axis
};

template <int kRounds, int kT, int kMinBlocks>
__global__ __launch_bounds__(kThreads, kMinBlocks) void fused_tiled_kernel(PicDesc d, PicSpecies sp, PicParticles in,
                                                                  FieldPtrs fp, PicParticles out, float* Jx,
                                                                  float* Jy, float* Jz,
                                                                  const int32_t* __restrict__ starts, TileGeom tg) {
    constexpr int kB = kT + 4;
    constexpr int kBox = 3 * kB * kB * kB;
    constexpr int kFB = kT + 4;
    constexpr int kFV = kFB * kFB * kFB;
    __shared__ FusedShared<kRounds> sh;
    __shared__ float box[kBox];
    __shared__ float fbox[6 * kFV];
    const int b = blockIdx.x;
    const int64_t begin = starts[b], end = starts[b + 1];
    if (begin >= end) return;
    const int t = b % (tg.tiles + 1);
    int o[3] = {0, 0, 0}, fo[3] = {0, 0, 0};
    if (t < tg.tiles) {
        const int tx = t / (tg.nt[1] * tg.nt[2]), ty = (t / tg.nt[2]) % tg.nt[1], tz = t % tg.nt[2];
        const int c0[3] = {tx * kT, ty * kT, tz * kT};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            o[a] = c0[a] + d.g - 1;
            fo[a] = c0[a] + d.g - 2;
        }
    }
    for (int e = threadIdx.x; e < kBox; e += kThreads) box[e] = 0.0f;
    // E+E_ext, B+B_ext on the (T+4)^3 nodes from T+g-2 (gather anchors of the
    // tile's particles, drifted by up to a cell, and their +1 neighbours)
    for (int e = threadIdx.x; e < 6 * kFV; e += kThreads) {
        const int c = e / kFV, r = e % kFV;
        const int i = pmod(fo[0] + r / (kFB * kFB), d.dims[0]), j = pmod(fo[1] + (r / kFB) % kFB, d.dims[1]);
        const int k = pmod(fo[2] + r % kFB, d.dims[2]);
        const int64_t id = fidx(d, i, j, k);
        const float* F = c < 3 ? fp.E[c] : fp.B[c - 3];
        const float* Fe = c < 3 ? fp.Ee[c] : fp.Be[c - 3];
        float v = F[id];
        if (Fe) v += Fe[id];
        fbox[e] = v;
    }
    __syncthreads();
    const BoxSink sink{{Jx, Jy, Jz}, box, {o[0], o[1], o[2]}, kB};
    const FieldBox fb{fbox, {fo[0], fo[1], fo[2]}, kFB};
    for (int64_t base = begin; base < end; base += kThreads * kRounds) {
        fused_block<3, kRounds, BoxSink, true>(d, sp, in, fp, out, sink, end, (uint32_t)base, sh, fb);
        __syncthreads();
    }
    float* const J[3] = {Jx, Jy, Jz};
    for (int e = threadIdx.x; e < kBox; e += kThreads) {
        const float v = box[e];
        if (v == 0.0f) continue;
        const int c = e / (kB * kB * kB), r = e % (kB * kB * kB);
        deposit_at(J[c], d, o[0] + r / (kB * kB), o[1] + (r / kB) % kB, o[2] + r % kB, v);
    }
}

// One particle of the tile kernel through the general route: global gather
// with FP64 anchors, push, 3-slot (or 5-slot) Esirkepov deposit, position
// update, boundaries and store.  Run by fused_tile_rare_kernel for the rare
// particles the tile kernel's fast loop does not cover.
template <class Sink>
__device__ inline void tile_particle_general(const PicDesc& d, const SpeciesK& k, const PicParticles& in,
                                             const FieldPtrs& fp, const PicParticles& out, const Sink& sink,
                                             int64_t i, int64_t src) {
    double xo[3];
    load_pos(in, src, xo);
    float v[3] = {in.u[0][src], in.u[1][src], in.u[2][src]};
    CicAxis gc[3], gv[3];
    int anc[3], anv[3];
    float dc[3], dv[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float x = (float)xo[a];
        cic_axis(x, (float)d.org_c[a], (float)(1.0 / d.sp_c[a]), d.org_c[a], d.sp_c[a], d.dims[a], gc[a], anc[a],
                 dc[a]);
        cic_axis(x, (float)d.org_v[a], (float)(1.0 / d.sp_v[a]), d.org_v[a], d.sp_v[a], d.dims[a], gv[a], anv[a],
                 dv[a]);
    }
    float E[3], B[3];
    E[0] = gather_cic(fp.E[0], fp.Ee[0], d, gv[0], gc[1], gc[2]);
    E[1] = gather_cic(fp.E[1], fp.Ee[1], d, gc[0], gv[1], gc[2]);
    E[2] = gather_cic(fp.E[2], fp.Ee[2], d, gc[0], gc[1], gv[2]);
    B[0] = gather_cic(fp.B[0], fp.Be[0], d, gc[0], gv[1], gv[2]);
    B[1] = gather_cic(fp.B[1], fp.Be[1], d, gv[0], gc[1], gv[2]);
    B[2] = gather_cic(fp.B[2], fp.Be[2], d, gv[0], gv[1], gc[2]);
    float nv[3] = {v[0], v[1], v[2]};
    push_velocity(nv, E, B, k.h, d);
#pragma unroll
    for (int a = 0; a < 3; ++a)
        if ((k.uu >> a) & 1u) v[a] = nv[a];
    double xn[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) xn[a] = ((k.ux >> a) & 1u) ? step_pos(xo[a], (double)v[a], d.dt) : xo[a];
    CrossAxis cx, cy, cz;
    bool ok = cross_axis(xo[0], xn[0], d.org_c[0], d.sp_c[0], 1.0 / d.d[0], (float)d.org_c[0],
                         (float)(1.0 / d.sp_c[0]), cx);
    ok = cross_axis(xo[1], xn[1], d.org_c[1], d.sp_c[1], 1.0 / d.d[1], (float)d.org_c[1], (float)(1.0 / d.sp_c[1]),
                    cy) && ok;
    ok = cross_axis(xo[2], xn[2], d.org_c[2], d.sp_c[2], 1.0 / d.d[2], (float)d.org_c[2], (float)(1.0 / d.sp_c[2]),
                    cz) && ok;
    if (ok) {
        crossing_deposit(d, k.qw, cx, cy, cz, sink);
    } else {
        float* const J[3] = {sink.J[0], sink.J[1], sink.J[2]};
        esirkepov_particle(d, k.qw, xo, xn, v, J);
    }
    bool act = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) apply_axis_boundary(d.pbc[a], d.wind[a], xn[a], v[a], act);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        out.x[a][i] = act ? (float)xn[a] : 0.0f;
        out.u[a][i] = act ? v[a] : 0.0f;
    }
    out.active[i] = act ? 1 : 0;
}

__device__ inline void rare_push(int32_t* rare, int64_t i) {
    const int p = atomicAdd(rare, 1);
    rare[1 + p] = (int32_t)i;
}

// LDS accumulators of the current boxes.  ds_add_f64 takes 0.24-0.36 cycles per
// lane on this card and ds_add_f32 3.0, so the 4-cell tiles sum in FP64; the
// 8-cell tiles keep FP32, whose box leaves room for two blocks per CU.
template <int kT>
using BoxSum = std::conditional_t<kT == 4, double, float>;

// Face-crossing deposit (the 54 terms of crossing_deposit) straight into the
// LDS box when the particle's 3x3x3 frame lies inside it: one base address,
// the term offsets are compile-time constants, no per-term bounds checks.
// pre[c] = -(q w / (d_p d_q dt)) as in SpeciesK.
template <int kC, int kB, class T>
__device__ inline void crossing_component_box(const float pre, const CrossAxis& A, const CrossAxis& P,
                                              const CrossAxis& Q, T* p) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float ci = i == 0 ? A.C0 : A.C1;
        if (ci == 0.0f) continue;
        const float w = pre * ci;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float y = P.S0[j] * Q.S0[k] + 0.5f * (P.S0[j] * Q.D[k] + P.D[j] * Q.S0[k]) +
                                (1.0f / 3.0f) * P.D[j] * Q.D[k];
                const int dx = kC == 0 ? i : j;
                const int dy = kC == 0 ? j : (kC == 1 ? i : k);
                const int dz = kC == 2 ? i : k;
                box_add(p + kC * kB * kB * kB + (dx * kB + dy) * kB + dz, w * y);
            }
            __builtin_amdgcn_sched_barrier(0);   // bound the live terms to one row of three
        }
    }
}

// Adds the moments of a cell's regular particles into the four nodes of each
// component: per component M = sum p (1, A_p, A_q, A_p A_q + d_p d_q / 12) with
// p the current of the particle and A_p, A_q its upper weights along the other
// axes, so node (1,1) is M3, (1,0) M1 - M3, (0,1) M2 - M3, (0,0) the rest.
template <int kB, class T>
__device__ inline void flush_moments(T* p, const float m[12]) {
    constexpr int kB3 = kB * kB * kB, s[3] = {kB * kB, kB, 1};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const int sp = s[c == 0 ? 1 : 0], sq = s[c == 2 ? 1 : 2];
        const float v10 = m[4 * c + 1] - m[4 * c + 3], v01 = m[4 * c + 2] - m[4 * c + 3];
        box_add(p + c * kB3, (m[4 * c] - m[4 * c + 1]) - v01);
        box_add(p + c * kB3 + sq, v01);
        box_add(p + c * kB3 + sp, v10);
        box_add(p + c * kB3 + sp + sq, m[4 * c + 3]);
        __builtin_amdgcn_sched_barrier(0);   // bound the live FP64 values to one component
    }
}

// Particles of a chunk that do not stay in their cell: slot offset from the
// chunk base and pushed velocity; the queue's pass reloads the old position.
// A full queue sends further particles to the rare list.
constexpr int kCrossCap = 512;
struct CrossQueue {
    int slot[kCrossCap];
    float v[3][kCrossCap];
    int n;
};

// Slots of a block of a tile kernel, whose grid has a block per (species, tile)
// and, in front of them, kOutside for the slots of each species that no tile
// holds: empty ones for the most part, whose number grows where an open box
// absorbs particles.  One block per species took longer over them than the tiles
// (160 x 96 x 96 with 4 per cell and PML, six steps: 2.9 ms on new particles, 3.7
// on a plasma that had lost some, 2.9 shared out).
constexpr int kOutside = 128;           // a multiple of 8: the tiles' blocks keep their XCDs

__device__ inline bool tile_slots(const int32_t* __restrict__ starts, const TileGeom& tg, int& s, int& t,
                                  int64_t& begin, int64_t& end) {
    const int bx = (int)blockIdx.x, ranges = tg.tiles + 1, count = (int)gridDim.x / (ranges + kOutside);
    if (bx < count * kOutside) {
        s = bx / kOutside;
        t = tg.tiles;
        const int64_t b0 = starts[s * ranges + t], b1 = starts[s * ranges + t + 1], lo = b0 & ~(int64_t)3;
        const int64_t share = ((b1 - lo + kOutside - 1) / kOutside + 3) & ~(int64_t)3;
        begin = max(b0, lo + share * (bx % kOutside));
        end = min(b1, lo + share * (bx % kOutside + 1));
    } else {
        const int b = xcd_block(bx - count * kOutside, count * ranges);
        s = b / ranges;
        t = b % ranges;
        begin = starts[b];
        end = t < tg.tiles ? starts[b + 1] : begin;
    }
    return begin < end;
}

// Tile-ordered launch: gather + push + Esirkepov + position update +
// boundaries.  Block b owns the sorted slot range [starts[b], starts[b+1]) of
// one (species, tile) pair: the particles that were in that T^3-cell tile at the
// last sort.  Fields are gathered from an LDS box of the (T+4)^3 nodes around
// the tile, J is summed in an LDS box of the same nodes and added into the
// arrays once per block.  Thread t of a chunk owns kP
// consecutive slots, loaded and stored with one access per plane (16 bytes of four);
// sorted slots of one cell are contiguous, so a thread's particles mostly share
// a cell and their twelve moments (flush_moments) are summed in registers, added
// into the box when the cell changes and, after a sum over equal cells of
// neighbouring lanes, at the end of the group.
//
// A particle that leaves its cell, or ends within 2^-19 spacings of a face, is
// queued with its velocity and deposited in the 3-slot frame after the chunk,
// by lanes that all do so (in the particle's own iteration that code would run
// for one lane of most waves).  One whose anchors leave the field box, whose
// frame leaves the current box, that moves its anchor by two or finds the queue
// full is put on the rare list (rare[0] = count, slots from rare[1]) and run
// whole by fused_tile_rare_kernel, which overwrites what is stored here.
//
// Bound by VALU instructions (577 per 64 particles, 81 % of the fastest launch at
// 256^3 with 32; the LDS and memory traffic overlap them).  Summing cell moments in registers, FP64 box adds in
// place of ds_add_f32 and a queue of (slot, velocity) took 128^3 with 2 x 16
// particles per cell from 1963 to 1548 us (43 G particles/s, 2.2 TB/s) and
// 256^3 with 32 from 12.1 to 9.7 ms; FP64 anchors in the same kernel take
// 160 x 96 x 96 with 4 per cell from 1132 to 396 us, one slot a thread there to 315.  kExact: FP32 anchors of an
// exact grid, else FP64 ones (TileGrid).  kAll: no species has a frozen axis.
template <int kT, bool kGather, bool kExact, bool kAll, int kP>
__global__ __launch_bounds__(kThreads, kT == 4 ? 4 : 2) void fused_tile_exact_kernel(
    PicDesc d, PicParticles in, FieldPtrs fp, PicParticles out, float* Jx, float* Jy, float* Jz,
    const int32_t* __restrict__ starts, TileGeom tg, TileGrid grid, int32_t* __restrict__ rare, int vec_ok,
    SpeciesTable st, const int32_t* __restrict__ gather) {
    constexpr int kB = kT + 4;                     // nodes per axis of both boxes
    constexpr int kB3 = kB * kB * kB;
    constexpr int kChunk = kThreads * kP;          // a thread owns kP consecutive slots
    // unrolled, the slots need no register shifts (128^3, 2 x 16 particles per cell: 1590 -> 1550 us,
    // 256^3, 32: 11.0 -> 9.7 ms); with FP64 anchors the rolled loop is shorter on the clock (396, 438 us)
    constexpr int kUnroll = kExact ? kP : 1;
    using Sum = BoxSum<kT>;
    __shared__ CrossQueue sh;
    __shared__ Sum box[3 * kB3];
    __shared__ float fbox[6 * kB3];
    int s, t;
    int64_t begin, end;
    if (!tile_slots(starts, tg, s, t, begin, end)) return;
    int fo[3] = {0, 0, 0};
    // interior: every particle the fast path handles (anchors inside the field
    // box, cells c0 - 2 .. c0 + T + 1, an anchor step of at most one) stays
    // inside [-W/2, W/2) on every axis, so its particle boundaries do nothing
    // and are skipped (a block-uniform branch)
    bool interior = t < tg.tiles;
    if (t < tg.tiles) {
        const int c0[3] = {(t / (tg.nt[1] * tg.nt[2])) * kT, ((t / tg.nt[2]) % tg.nt[1]) * kT, (t % tg.nt[2]) * kT};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            fo[a] = c0[a] + d.g - 2;
            interior = interior && c0[a] >= 3 && c0[a] + kT + 3 <= d.n[a];
        }
    }
    // Positions whose anchors on both node lines lie in the field box and whose
    // nodes lie in the arrays.  The bounds are rounded up, so an FP32 position
    // is inside exactly when its value is; off an exact grid a margin keeps the
    // rounding of the vertex line out.
    float nb[3], xlo[3], xhi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double org = d.org_c[a], sp = d.sp_c[a], margin = kExact ? 0.0 : 1.0e-6 * sp;
        nb[a] = uniform((float)(fo[a] * sp + org));
        xlo[a] = uniform(__double2float_ru(fmax(fo[a] * sp + org + 0.5 * sp, org) + margin));
        xhi[a] = uniform(__double2float_ru(min(fo[a] + kB - 1, d.dims[a] - 1) * sp + org - margin));
    }
    // the first group is loaded before the field box is filled: both wait for memory together
    float PX[3][kP], PU[3][kP];
    uint32_t pact;
    const auto inside = [&](int64_t s0) { return kP > 1 && vec_ok && s0 >= begin && s0 + kP <= end; };
    const int64_t first = begin & ~(int64_t)(kP - 1);
    const int64_t g0 = first + (int64_t)kP * (int)threadIdx.x;
    load_group<kP, kGather>(in, gather, g0, begin, end, inside(g0), PX, PU, pact);
    for (int e = threadIdx.x; e < 3 * kB3; e += kThreads) box[e] = (Sum)0;
    fill_field_box<kB>(d, fp, fo, fbox);
    const SpeciesK& k = st.k[s];

    for (int64_t base = first; base < end; base += kChunk) {
        if (threadIdx.x == 0) sh.n = 0;
        __syncthreads();    // also orders the box fills before the first deposits
        float acc[12];
#pragma unroll
        for (int m = 0; m < 12; ++m) acc[m] = 0.0f;
        int cell = -1;
        const int64_t s0 = base + (int64_t)kP * (int)threadIdx.x;
        const bool full = inside(s0);
        if (base != first) load_group<kP, kGather>(in, gather, s0, begin, end, full, PX, PU, pact);
        // One particle per iteration (the loop stays rolled to bound register
        // pressure): slot j's inputs are taken from the front of PX/PU/pact,
        // which shift by one, and its outputs enter at the back, so after kP
        // iterations PX/PU/oact hold the outputs in slot order for the vector
        // stores.  Slots sent to the rare list are stored as zeros here and
        // rewritten by the rare kernel.
        uint32_t oact = 0u;
#pragma unroll kUnroll
        for (int j = 0; j < kP; ++j) {
            const float xf[3] = {PX[0][0], PX[1][0], PX[2][0]};
            float v[3] = {PU[0][0], PU[1][0], PU[2][0]};
            const bool act0 = (pact & 0xffu) != 0u;
            pact >>= 8;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
#pragma unroll
                for (int q = 0; q + 1 < kP; ++q) {
                    PX[a][q] = PX[a][q + 1];
                    PU[a][q] = PU[a][q + 1];
                }
            }
            float ox[3] = {0.0f, 0.0f, 0.0f}, ou[3] = {0.0f, 0.0f, 0.0f};
            uint32_t oa = 0u;
            do {
            if (!act0) break;          // inactive, or outside [begin, end)
            // ---- anchors on both node lines (grid_and_stencil.py:92-166)
            bool fast = true;
#pragma unroll
            for (int a = 0; a < 3; ++a) fast = fast & (xf[a] >= xlo[a]) & (xf[a] < xhi[a]);
            float f[3], dc[3], qm[3], dv[3];
            bool up[3];
#pragma unroll
            for (int a = 0; a < 3; ++a)
                fast = tile_anchor<kExact>(grid, a, xf[a], nb[a], (float)fo[a], f[a], dc[a], qm[a], up[a], dv[a]) & fast;
            if (!fast) {
                rare_push(rare, s0 + j);
                break;
            }
            const int at = (int)fmaf(f[0], (float)(kB * kB), fmaf(f[1], (float)kB, f[2]));
            // ---- gather (boris.py:302-433) from the tile's field box
            float E[3], Bf[3];
            {
                CicAxis gc[3], gv[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    gc[a].w0 = fmaf(-dc[a], grid.isp[a], 1.0f);
                    gc[a].w1 = dc[a] * grid.isp[a];
                    gv[a].w0 = fmaf(-dv[a], grid.isp[a], 1.0f);
                    gv[a].w1 = dv[a] * grid.isp[a];
                }
                const int lx = up[0] ? 0 : kB * kB, ly = up[1] ? 0 : kB, lz = up[2] ? 0 : 1;   // vertex node below
                E[0] = gather_at<kB>(fbox + at - lx, gv[0], gc[1], gc[2]);
                E[1] = gather_at<kB>(fbox + kB3 + at - ly, gc[0], gv[1], gc[2]);
                E[2] = gather_at<kB>(fbox + 2 * kB3 + at - lz, gc[0], gc[1], gv[2]);
                Bf[0] = gather_at<kB>(fbox + 3 * kB3 + at - ly - lz, gc[0], gv[1], gv[2]);
                Bf[1] = gather_at<kB>(fbox + 4 * kB3 + at - lx - lz, gv[0], gc[1], gv[2]);
                Bf[2] = gather_at<kB>(fbox + 5 * kB3 + at - lx - ly, gv[0], gv[1], gc[2]);
            }
            // ---- push (boris.py:14-124), masked by update_u (particle_push.py:134-142)
            float nv[3] = {v[0], v[1], v[2]};
            push_velocity(nv, E, Bf, k.h, d);
#pragma unroll
            for (int a = 0; a < 3; ++a)
                if (kAll || ((k.uu >> a) & 1u)) v[a] = nv[a];
            // ---- regular case: the new position stays in the old cell, away from its
            // faces by more than the FP64 rounding of floor((x - origin)/spacing).
            // The FP32 offset from the cell's middle is within 2^-22 spacings of the
            // FP64 one, the band 2^-19 wide; a particle in the band takes the queue,
            // which treats a stay in the cell like any other step
            bool regular = true;
            float D[3], A[3], qn[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const float dvt = kAll || ((k.ux >> a) & 1u) ? v[a] * grid.dt32 : 0.0f;
                qn[a] = qm[a] + dvt;
                regular = regular & (fabsf(qn[a]) < grid.lim[a]);
                D[a] = dvt * grid.inv_d[a];
                A[a] = fmaf(0.5f, D[a], dc[a] * grid.inv_d[a]);      // upper weight S0 + d/2
            }
            if (regular) {
                // difference-form Esirkepov weights of a particle that stays in its
                // cell (Esirkepov.py:158-214): for component c over the other axes p, q,
                // W = D_c (S0p S0q + (S0p dq + dp S0q)/2 + dp dq/3) with d = -D, +D at
                // slots 0, 1, i.e. W = D_c (Ap Aq + dp dq/12) with A = S0 + d/2;
                // J_c = -(q/(d_p d_q dt)) W at slot a only.  The lower weight is 1 - A,
                // so the four nodes are linear in the four moments below
                if (at != cell) {
                    if (cell >= 0) flush_moments<kB>(box + cell, acc);
#pragma unroll
                    for (int m = 0; m < 12; ++m) acc[m] = 0.0f;
                    cell = at;
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const int o1 = c == 0 ? 1 : 0, o2 = c == 2 ? 1 : 2;
                    const float pc = k.pre[c] * (-D[c]);
                    const float y = fmaf(A[o1], A[o2], D[o1] * (D[o2] * (1.0f / 12.0f)));
                    acc[4 * c] += pc;
                    acc[4 * c + 1] = fmaf(pc, A[o1], acc[4 * c + 1]);
                    acc[4 * c + 2] = fmaf(pc, A[o2], acc[4 * c + 2]);
                    acc[4 * c + 3] = fmaf(pc, y, acc[4 * c + 3]);
                }
            } else {
                // queued only if the frame of the pass lies in the box and the anchor
                // moves by at most one, so that how many particles are rare does not
                // depend on the order in which the queue fills (within the band of a
                // face the pass has the last word)
                bool near = true;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const float low = f[a] - (qn[a] < 0.0f ? 1.0f : 0.0f);
                    near = near & (low >= 0.0f) & (low <= kB - 3.0f) & (fabsf(D[a]) < 0.99f);
                }
                const int slot = near ? atomicAdd(&sh.n, 1) : kCrossCap;
                if (slot >= kCrossCap) {
                    rare_push(rare, s0 + j);
                    break;
                }
                sh.slot[slot] = (int)(s0 - base) + j;
#pragma unroll
                for (int a = 0; a < 3; ++a) sh.v[a][slot] = v[a];
            }
            // ---- position update + particle boundaries (particle_tile_communication.py)
            bool act = true;
            double xn[3];
#pragma unroll
            for (int a = 0; a < 3; ++a)
                xn[a] = kAll || ((k.ux >> a) & 1u) ? step_pos((double)xf[a], (double)v[a], d.dt) : (double)xf[a];
            if (!interior) {
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    // the asm keeps the remainder's loop-invariant half (a dozen vector
                    // registers) from being hoisted into every block
                    double wind = d.wind[a];
                    asm volatile("" : "+s"(wind));
                    if (d.pbc[a] == 0) periodic_wrap(wind, xn[a]);
                    else apply_axis_boundary(d.pbc[a], wind, xn[a], v[a], act);
                }
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                ox[a] = act ? (float)xn[a] : 0.0f;
                ou[a] = act ? v[a] : 0.0f;
            }
            oa = act ? 1u : 0u;
            } while (false);
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                PX[a][kP - 1] = ox[a];
                PU[a][kP - 1] = ou[a];
            }
            oact = (oact >> 8) | (oa << (8 * (kP - 1)));
        }
        store_group<kP>(out, s0, begin, end, full, PX, PU, oact);
        // the thread's last cell: equal cells of four neighbouring lanes are summed
        // first (over sixteen the two further steps cost more than the adds saved)
        if (row_run_sums<4>(cell, acc) && cell >= 0) flush_moments<kB>(box + cell, acc);
        __syncthreads();
        // ---- queued particles (3-slot frame, Esirkepov.py:105-331)
        const int nq = min(sh.n, kCrossCap);
        for (int q = threadIdx.x; q < nq; q += kThreads) {
            const int64_t i = base + sh.slot[q], src = kGather ? (int64_t)gather[i] : i;
            CrossAxis ca[3];
            bool ok = true;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const double xo = (double)in.x[a][src];
                const double xn = kAll || ((k.ux >> a) & 1u) ? step_pos(xo, (double)sh.v[a][q], d.dt) : xo;
                ok = cross_axis(xo, xn, grid.org64[a], grid.sp64[a], grid.inv_d64[a], grid.org32[a], grid.isp[a], ca[a]) && ok;
                ok = ok && (unsigned)(ca[a].b - fo[a]) <= (unsigned)(kB - 3);
            }
            if (!ok) {
                rare_push(rare, i);
                continue;
            }
            Sum* p = box + ((ca[0].b - fo[0]) * kB + ca[1].b - fo[1]) * kB + ca[2].b - fo[2];
            crossing_component_box<0, kB>(k.pre[0], ca[0], ca[1], ca[2], p);
            crossing_component_box<1, kB>(k.pre[1], ca[1], ca[0], ca[2], p);
            crossing_component_box<2, kB>(k.pre[2], ca[2], ca[0], ca[1], p);
        }
        __syncthreads();
    }
    flush_current_box<kB>(d, fo, box, Jx, Jy, Jz);
}

// The rare list of fused_tile_exact_kernel: each listed particle runs the
// general route with its deposit added straight into J.
__global__ __launch_bounds__(kThreads) void fused_tile_rare_kernel(PicDesc d, PicSpecies sp, PicParticles in,
                                                                   FieldPtrs fp, PicParticles out, float* Jx,
                                                                   float* Jy, float* Jz,
                                                                   const int32_t* __restrict__ rare,
                                                                   const int32_t* __restrict__ gather) {
    const int n = rare[0];
    const GlobalSink sink{{Jx, Jy, Jz}};
    for (int q = blockIdx.x * kThreads + threadIdx.x; q < n; q += gridDim.x * kThreads) {
        const int64_t i = rare[1 + q];
        const SpeciesK k = species_constants(d, sp, species_of(i, sp.slots, sp.count));
        tile_particle_general(d, k, in, fp, out, sink, i, gather ? (int64_t)gather[i] : i);
    }
}

__global__ void zero_count_kernel(int32_t* c) { *c = 0; }

// Direct-current branch of time_loop_electrodynamic (evolve.py:44-67) on
// tile-sorted particles of a 3-D first-order grid, fused: gather from the
// tile's LDS field box, push, x += v dt/2 (FP64, rounded to FP32 like
// pic_advance_positions), particle boundaries, the J_from_rhov deposit at the
// half position (J_from_rhov.py:88-200: node weights 1 - dn/d, dn/d and face
// weights 1 - df/d, df/d with df = dn - d/2 on the 2x2x2 nodes of the centre
// anchor), x += v dt/2, boundaries, store.  Slots, boxes and anchors as in
// fused_tile_exact_kernel; the 24 node values of a cell are summed in registers
// over a thread's particles and four lanes, then added into the J box, whose
// one more node per axis takes half positions.  Particles the fast loop does not
// cover are listed for fused_direct_rare_kernel.
// Bound by VALU instructions.  13.8M particles on 96 x 80 x 112 cells of 0.1:
// 392 us with FP64 anchors (1.8 TB/s); as separate push, advance, boundary and
// deposit launches, whose deposit added with ds_add_f32, 3100 us.
template <int kT, bool kGather, bool kExact, bool kAll>
__global__ __launch_bounds__(kThreads, kT == 4 ? 4 : 2) void fused_tile_direct_kernel(
    PicDesc d, PicParticles in, FieldPtrs fp, PicParticles out, float* Jx, float* Jy, float* Jz,
    const int32_t* __restrict__ starts, TileGeom tg, TileGrid grid, int32_t* __restrict__ rare, int vec_ok,
    SpeciesTable st, const int32_t* __restrict__ gather) {
    constexpr int kP = 4;
    constexpr int kB = kT + 5;                     // nodes per axis of the current box
    constexpr int kB3 = kB * kB * kB;
    constexpr int kF = kT + 4;                     // and of the field box
    constexpr int kF3 = kF * kF * kF;
    constexpr int kChunk = kThreads * kP;
    constexpr int kUnroll = kExact ? kP : 1;       // as in fused_tile_exact_kernel
    using Sum = BoxSum<kT>;
    __shared__ Sum box[3 * kB3];
    __shared__ float fbox[6 * kF3];
    int s, t;
    int64_t begin, end;
    if (!tile_slots(starts, tg, s, t, begin, end)) return;
    int fo[3] = {0, 0, 0};
    // interior: a fast-path particle (anchors inside the field box, cells
    // c0 - 2 .. c0 + T + 1) that moves less than a cell per step stays inside
    // [-W/2, W/2) on every axis, so its particle boundaries do nothing
    bool interior = t < tg.tiles;
    if (t < tg.tiles) {
        const int c0[3] = {(t / (tg.nt[1] * tg.nt[2])) * kT, ((t / tg.nt[2]) % tg.nt[1]) * kT, (t % tg.nt[2]) * kT};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            fo[a] = c0[a] + d.g - 2;
            interior = interior && c0[a] >= 3 && c0[a] + kT + 3 <= d.n[a];
        }
    }
    // old positions as in fused_tile_exact_kernel; half positions: centre anchor and the node above in the J box
    float nb[3], xlo[3], xhi[3], hhi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double org = d.org_c[a], sp = d.sp_c[a], margin = kExact ? 0.0 : 1.0e-6 * sp;
        nb[a] = uniform((float)(fo[a] * sp + org));
        xlo[a] = uniform(__double2float_ru(fmax(fo[a] * sp + org + 0.5 * sp, org) + margin));
        xhi[a] = uniform(__double2float_ru(min(fo[a] + kF - 1, d.dims[a] - 1) * sp + org - margin));
        hhi[a] = uniform(__double2float_ru((fo[a] + kB - 1) * sp + org - margin));
    }
    const auto inside = [&](int64_t s0) { return vec_ok && s0 >= begin && s0 + kP <= end; };
    const int64_t first = begin & ~(int64_t)(kP - 1);
    const int64_t g0 = first + (int64_t)kP * (int)threadIdx.x;
    float PX[3][kP], PU[3][kP];
    uint32_t pact;
    load_group<kP, kGather>(in, gather, g0, begin, end, inside(g0), PX, PU, pact);
    for (int e = threadIdx.x; e < 3 * kB3; e += kThreads) box[e] = (Sum)0;
    fill_field_box<kF>(d, fp, fo, fbox);
    __syncthreads();
    const SpeciesK& k = st.k[s];
    const double hdt = 0.5 * d.dt;
    const auto flush = [&](int cell, const float* acc) {
        Sum* p = box + cell;
#pragma unroll
        for (int m = 0; m < 24; ++m) {
            const int n = m & 7;
            box_add(p + (m >> 3) * kB3 + ((n >> 2) * kB + ((n >> 1) & 1)) * kB + (n & 1), acc[m]);
            if ((m & 3) == 3) __builtin_amdgcn_sched_barrier(0);   // bound the live FP64 values
        }
    };

    for (int64_t base = first; base < end; base += kChunk) {
        const int64_t s0 = base + (int64_t)kP * (int)threadIdx.x;
        const bool full = inside(s0);
        if (base != first) load_group<kP, kGather>(in, gather, s0, begin, end, full, PX, PU, pact);
        float acc[24];
#pragma unroll
        for (int m = 0; m < 24; ++m) acc[m] = 0.0f;
        int cell = -1;
        uint32_t oact = 0u;
#pragma unroll kUnroll
        for (int j = 0; j < kP; ++j) {
            const float xf[3] = {PX[0][0], PX[1][0], PX[2][0]};
            float v[3] = {PU[0][0], PU[1][0], PU[2][0]};
            const bool act0 = (pact & 0xffu) != 0u;
            pact >>= 8;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
#pragma unroll
                for (int q = 0; q + 1 < kP; ++q) {
                    PX[a][q] = PX[a][q + 1];
                    PU[a][q] = PU[a][q + 1];
                }
            }
            float ox[3] = {0.0f, 0.0f, 0.0f}, ou[3] = {0.0f, 0.0f, 0.0f};
            uint32_t oa = 0u;
            do {
            if (!act0) break;
            bool fast = true;
#pragma unroll
            for (int a = 0; a < 3; ++a) fast = fast & (xf[a] >= xlo[a]) & (xf[a] < xhi[a]);
            float f[3], dc[3], qm[3], dv[3];
            bool up[3];
#pragma unroll
            for (int a = 0; a < 3; ++a)
                fast = tile_anchor<kExact>(grid, a, xf[a], nb[a], (float)fo[a], f[a], dc[a], qm[a], up[a], dv[a]) & fast;
            if (!fast) {
                rare_push(rare, s0 + j);
                break;
            }
            float E[3], Bf[3];
            {
                const int at = (int)fmaf(f[0], (float)(kF * kF), fmaf(f[1], (float)kF, f[2]));
                CicAxis gc[3], gv[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    gc[a].w0 = fmaf(-dc[a], grid.isp[a], 1.0f);
                    gc[a].w1 = dc[a] * grid.isp[a];
                    gv[a].w0 = fmaf(-dv[a], grid.isp[a], 1.0f);
                    gv[a].w1 = dv[a] * grid.isp[a];
                }
                // off an exact grid the particles are those of pic_push bit for bit
                constexpr CicRounding kE1 = kExact ? kPlain : kSecond, kBs = kExact ? kPlain : kMagnetic;
                const int lx = up[0] ? 0 : kF * kF, ly = up[1] ? 0 : kF, lz = up[2] ? 0 : 1;   // vertex node below
                E[0] = gather_at<kF>(fbox + at - lx, gv[0], gc[1], gc[2]);
                E[1] = gather_at<kF, kE1>(fbox + kF3 + at - ly, gc[0], gv[1], gc[2]);
                E[2] = gather_at<kF>(fbox + 2 * kF3 + at - lz, gc[0], gc[1], gv[2]);
                Bf[0] = gather_at<kF, kBs>(fbox + 3 * kF3 + at - ly - lz, gc[0], gv[1], gv[2]);
                Bf[1] = gather_at<kF, kBs>(fbox + 4 * kF3 + at - lx - lz, gv[0], gc[1], gv[2]);
                Bf[2] = gather_at<kF, kBs>(fbox + 5 * kF3 + at - lx - ly, gv[0], gv[1], gc[2]);
            }
            float nv[3] = {v[0], v[1], v[2]};
            push_velocity(nv, E, Bf, k.h, d);
#pragma unroll
            for (int a = 0; a < 3; ++a)
                if (kAll || ((k.uu >> a) & 1u)) v[a] = nv[a];
            // ---- x += v dt/2, boundaries (evolve.py:48-52)
            bool act = true;
            bool skip_bc = interior;
#pragma unroll
            for (int a = 0; a < 3; ++a) skip_bc = skip_bc & (fabsf(v[a]) * grid.dt32 < 0.99f * grid.sp[a]);
            const auto half_step = [&](float (&x)[3]) {
                double p[3];
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    p[a] = kAll || ((k.ux >> a) & 1u) ? (double)(float)step_pos((double)x[a], (double)v[a], hdt)
                                                      : (double)x[a];
                if (!skip_bc) {
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        double wind = d.wind[a];
                        asm volatile("" : "+s"(wind));      // see fused_tile_exact_kernel
                        if (d.pbc[a] == 0) periodic_wrap(wind, p[a]);
                        else apply_axis_boundary(d.pbc[a], wind, p[a], v[a], act);
                    }
                }
#pragma unroll
                for (int a = 0; a < 3; ++a) x[a] = (float)p[a];
            };
            float xh[3] = {xf[0], xf[1], xf[2]};
            half_step(xh);
            if (act) {
                // ---- J_from_rhov at the half position
                float dn[3];
                bool inbox = true;
#pragma unroll
                for (int a = 0; a < 3; ++a) inbox = inbox & (xh[a] >= nb[a]) & (xh[a] < hhi[a]);
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    inbox = tile_anchor<kExact>(grid, a, xh[a], nb[a], (float)fo[a], f[a], dn[a], qm[a], up[a], dv[a]) &
                            inbox & (f[a] >= 0.0f) & (f[a] <= kB - 2.0f);
                if (!inbox) {
                    rare_push(rare, s0 + j);
                    break;
                }
                const int at = (int)fmaf(f[0], (float)(kB * kB), fmaf(f[1], (float)kB, f[2]));
                if (at != cell) {
                    if (cell >= 0) flush(cell, acc);
#pragma unroll
                    for (int m = 0; m < 24; ++m) acc[m] = 0.0f;
                    cell = at;
                }
                float wn[3][2], wf[3][2];
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    wn[a][1] = dn[a] * grid.inv_d[a];
                    wn[a][0] = 1.0f - wn[a][1];
                    wf[a][1] = (dn[a] - grid.half[a]) * grid.inv_d[a];
                    wf[a][0] = 1.0f - wf[a][1];
                }
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const float qv = k.q_dv * v[c];
#pragma unroll
                    for (int n = 0; n < 4; ++n) {
                        const int xi = n >> 1, yi = n & 1;
                        const float w = qv * (c == 0 ? wf[0][xi] : wn[0][xi]) * (c == 1 ? wf[1][yi] : wn[1][yi]);
                        acc[8 * c + 2 * n] = fmaf(w, c == 2 ? wf[2][0] : wn[2][0], acc[8 * c + 2 * n]);
                        acc[8 * c + 2 * n + 1] = fmaf(w, c == 2 ? wf[2][1] : wn[2][1], acc[8 * c + 2 * n + 1]);
                    }
                }
                // ---- x += v dt/2, boundaries (evolve.py:62-66)
                half_step(xh);
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    ox[a] = act ? xh[a] : 0.0f;
                    ou[a] = act ? v[a] : 0.0f;
                }
                oa = act ? 1u : 0u;
            }
            } while (false);
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                PX[a][kP - 1] = ox[a];
                PU[a][kP - 1] = ou[a];
            }
            oact = (oact >> 8) | (oa << (8 * (kP - 1)));
        }
        store_group<kP>(out, s0, begin, end, full, PX, PU, oact);
        if (row_run_sums<4>(cell, acc) && cell >= 0) flush(cell, acc);
    }
    __syncthreads();
    flush_current_box<kB>(d, fo, box, Jx, Jy, Jz);
}

// The rare list of fused_tile_direct_kernel: each listed particle runs the
// direct branch through the general route (global gather, FP64 anchors, the
// 3^3 deposit into J).
template <bool kExact>
__global__ __launch_bounds__(kThreads) void fused_direct_rare_kernel(PicDesc d, PicSpecies sp, PicParticles in,
                                                                     FieldPtrs fp, PicParticles out, float* Jx,
                                                                     float* Jy, float* Jz,
                                                                     const int32_t* __restrict__ rare,
                                                                     const int32_t* __restrict__ gather) {
    const int n = rare[0];
    const GlobalSink sink{{Jx, Jy, Jz}};
    for (int q = blockIdx.x * kThreads + threadIdx.x; q < n; q += gridDim.x * kThreads) {
        const int64_t i = rare[1 + q];
        const int64_t src = gather ? (int64_t)gather[i] : i;      // input slot (a re-bin's permutation)
        const SpeciesK k = species_constants(d, sp, species_of(i, sp.slots, sp.count));
        double pos[3];
        load_pos(in, src, pos);
        float v[3] = {in.u[0][src], in.u[1][src], in.u[2][src]};
        float E[3], B[3];
        CicAxis gc[3], gv[3];
        for (int a = 0; a < 3; ++a) {
            int an;
            float dl;
            cic_axis((float)pos[a], (float)d.org_c[a], (float)(1.0 / d.sp_c[a]), d.org_c[a], d.sp_c[a], d.dims[a],
                     gc[a], an, dl);
            cic_axis((float)pos[a], (float)d.org_v[a], (float)(1.0 / d.sp_v[a]), d.org_v[a], d.sp_v[a], d.dims[a],
                     gv[a], an, dl);
        }
        E[0] = gather_cic(fp.E[0], fp.Ee[0], d, gv[0], gc[1], gc[2]);
        E[1] = gather_cic<kExact ? kPlain : kSecond>(fp.E[1], fp.Ee[1], d, gc[0], gv[1], gc[2]);
        E[2] = gather_cic(fp.E[2], fp.Ee[2], d, gc[0], gc[1], gv[2]);
        B[0] = gather_cic<kExact ? kPlain : kMagnetic>(fp.B[0], fp.Be[0], d, gc[0], gv[1], gv[2]);
        B[1] = gather_cic<kExact ? kPlain : kMagnetic>(fp.B[1], fp.Be[1], d, gv[0], gc[1], gv[2]);
        B[2] = gather_cic<kExact ? kPlain : kMagnetic>(fp.B[2], fp.Be[2], d, gv[0], gv[1], gc[2]);
        float nv[3] = {v[0], v[1], v[2]};
        push_velocity(nv, E, B, k.h, d);
        for (int a = 0; a < 3; ++a)
            if ((k.uu >> a) & 1u) v[a] = nv[a];
        bool act = true;
        double xh[3];
        for (int a = 0; a < 3; ++a) {
            xh[a] = ((k.ux >> a) & 1u) ? (double)(float)step_pos(pos[a], (double)v[a], 0.5 * d.dt) : pos[a];
            apply_axis_boundary(d.pbc[a], d.wind[a], xh[a], v[a], act);
            xh[a] = (double)(float)xh[a];
        }
        if (act) {
            direct_deposit(d, k.q_dv, xh, v, sink);
            for (int a = 0; a < 3; ++a) {
                double t2 = ((k.ux >> a) & 1u) ? (double)(float)step_pos(xh[a], (double)v[a], 0.5 * d.dt) : xh[a];
                apply_axis_boundary(d.pbc[a], d.wind[a], t2, v[a], act);
                xh[a] = t2;
            }
        }
        for (int a = 0; a < 3; ++a) {
            out.x[a][i] = act ? (float)xh[a] : 0.0f;
            out.u[a][i] = act ? v[a] : 0.0f;
        }
        out.active[i] = act ? 1 : 0;
    }
}

// 1-D and 2-D first-order runs: a chunk of slots per block.
template <int kDims, int kP, int kBlk>
__global__ __launch_bounds__(kBlk, 1024 / kBlk) void planar_kernel(PicDesc d, PicSpecies sp, PicParticles in, FieldPtrs fp,
                                                             PicParticles out, float* Jx, float* Jy, float* Jz,
                                                             int64_t n, int vec_ok) {
    __shared__ PlanarShared<kP, kBlk> sh;
    float* const J[3] = {Jx, Jy, Jz};
    planar_chunk<kDims, kP, kBlk>(d, sp, in, fp, out, J, n, blockIdx.x * (uint32_t)(kBlk * kP), vec_ok != 0, sh);
}

// Slot-ordered launch of the general path (any shape and reduced axes): each
// block accumulates J in an LDS box sized to its particles.
template <int kRounds>
__global__ __launch_bounds__(kThreads, 1) void fused_boxed_kernel(PicDesc d, PicSpecies sp, PicParticles in,
                                                                  FieldPtrs fp, PicParticles out, float* Jx,
                                                                  float* Jy, float* Jz, int64_t n) {
    __shared__ FusedShared<kRounds> sh;
    __shared__ float box[kRangeBoxCap];
    __shared__ int bmin[3], bmax[3];
    float* const J[3] = {Jx, Jy, Jz};
    fused_block_boxed<kRounds>(d, sp, in, fp, out, J, n, blockIdx.x * (uint32_t)(kThreads * kRounds), sh, box, bmin,
                               bmax);
}

}  // namespace

extern "C" {

// A launch of 2^32 threads or more would run the remainder only, without an error (tiles of 4^3 cells: 1024^3).
static bool tile_grid_ok(int64_t blocks, int32_t species) {
    return (blocks + (int64_t)kOutside * species) * kThreads < ((int64_t)1 << 32);
}

// node_values: 1-D and 2-D first-order sets too form J's node values particle by particle.
static int fused_esirkepov(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                           const float* const E[3], const float* const B[3], const float* const E_ext[3],
                           const float* const B_ext[3], PicParticles* out, float* const J[3], bool node_values,
                           void* stream) {
    PIC_REQUIRE(desc_ok(desc) && particles_ok(sp, in) && particles_ok(sp, out) && E && B && J);
    PIC_REQUIRE(desc->n[0] > 1 || desc->n[1] > 1 || desc->n[2] > 1);
    const bool empty = (int64_t)sp->count * sp->slots == 0;
    for (int a = 0; a < 3; ++a)
        PIC_REQUIRE(E[a] && B[a] && J[a] && (empty || (in->x[a] != out->x[a] && in->u[a] != out->u[a])));
    PIC_REQUIRE(empty || in->active != out->active);
    PIC_REQUIRE(field_size(*desc) < ((int64_t)1 << 31));
    int64_t n = (int64_t)sp->count * sp->slots;
    PIC_REQUIRE(n < ((int64_t)1 << 31) - 8 * kThreads);
    if (n == 0) return 0;
    const int kind = fused_kind(*desc);
    hipStream_t st = as_stream(stream);
    FieldPtrs fp = make_fields(E, B, E_ext, B_ext);
#define PIC_FUSED_LAUNCH(DIMS, R, MB)                                                                           \
    hipLaunchKernelGGL((fused_push_esirkepov_v2<DIMS, R, MB>), dim3(grid_1d(n, kThreads * R)), dim3(kThreads), 0, \
                       st, *desc, *sp, *in, fp, *out, J[0], J[1], J[2], n)
    if (kind == 3) {
        switch (desc->variant) {
            case 1: PIC_FUSED_LAUNCH(3, 4, 3); break;
            case 2: PIC_FUSED_LAUNCH(3, 4, 4); break;
            case 3: PIC_FUSED_LAUNCH(3, 8, 1); break;
            case 4: PIC_FUSED_LAUNCH(3, 2, 1); break;
            case 5: PIC_FUSED_LAUNCH(3, 8, 3); break;
            default: PIC_FUSED_LAUNCH(3, 4, 1); break;
        }
    } else if (kind != 0 && !node_values && planar_covers(*desc)) {
        // chunks of 1024 slots amortise ranges and boxes once they still make four blocks a CU; smaller
        // sets take 256, for more blocks (262k slots: 1024 of them, all resident at once)
        const bool large = n >= (int64_t)1 << 20;
        const int vec_ok = groups_aligned(*in, *out);
#define PIC_PLANAR(DIMS, P, BLK)                                                                                  \
    hipLaunchKernelGGL((planar_kernel<DIMS, P, BLK>), dim3(grid_1d(n, BLK * P)), dim3(BLK), 0, st, *desc, *sp, *in, \
                       fp, *out, J[0], J[1], J[2], n, vec_ok)
        if (kind == 2 && large) PIC_PLANAR(2, 2, kPlanarBlock);
        else if (kind == 2) PIC_PLANAR(2, 1, kThreads);
        else if (large) PIC_PLANAR(1, 2, kPlanarBlock);
        else PIC_PLANAR(1, 1, kThreads);
#undef PIC_PLANAR
    } else {
        hipLaunchKernelGGL(fused_boxed_kernel<4>, dim3(grid_1d(n, kThreads * 4)), dim3(kThreads), 0, st, *desc, *sp,
                           *in, fp, *out, J[0], J[1], J[2], n);
    }
#undef PIC_FUSED_LAUNCH
    PIC_CHECK_LAUNCH();
    return 0;
}

int pic_fused_push_esirkepov(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                             const float* const E[3], const float* const B[3], const float* const E_ext[3],
                             const float* const B_ext[3], PicParticles* out, float* const J[3], void* stream) {
    return fused_esirkepov(desc, sp, in, E, B, E_ext, B_ext, out, J, false, stream);
}

int pic_fused_push_esirkepov_nodes(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                   const float* const E[3], const float* const B[3], const float* const E_ext[3],
                                   const float* const B_ext[3], PicParticles* out, float* const J[3], void* stream) {
    return fused_esirkepov(desc, sp, in, E, B, E_ext, B_ext, out, J, true, stream);
}

static int fused_direct_tiled(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                              const float* const E[3], const float* const B[3], const float* const E_ext[3],
                              const float* const B_ext[3], PicParticles* out, float* const J[3], int32_t tile,
                              const int32_t* starts, int32_t min_blocks, int32_t* workspace, const int32_t* gather,
                              bool general, void* stream) {
    PIC_REQUIRE(desc_ok(desc) && particles_ok(sp, in) && particles_ok(sp, out) && E && B && J && starts && workspace);
    PIC_REQUIRE(fused_kind(*desc) == 3 && (tile == 4 || tile == 8) && (min_blocks == 1 || min_blocks == 4));
    ExactGrid eg;
    TileGrid grid;
    const bool exact = make_exact_grid(*desc, eg) && desc->d[0] == desc->sp_c[0] && desc->d[1] == desc->sp_c[1] &&
                       desc->d[2] == desc->sp_c[2];
    PIC_REQUIRE((exact || general) && make_tile_grid(*desc, exact, grid));
    const bool empty = (int64_t)sp->count * sp->slots == 0;
    for (int a = 0; a < 3; ++a)
        PIC_REQUIRE(E[a] && B[a] && J[a] && (empty || (in->x[a] != out->x[a] && in->u[a] != out->u[a])));
    PIC_REQUIRE(empty || in->active != out->active);
    PIC_REQUIRE(field_size(*desc) < ((int64_t)1 << 31));
    int64_t n = (int64_t)sp->count * sp->slots;
    PIC_REQUIRE(n < ((int64_t)1 << 31) - 8 * kThreads);
    if (n == 0) return 0;
    TileGeom tg;
    tg.T = tile;
    for (int a = 0; a < 3; ++a) tg.nt[a] = (desc->n[a] + tile - 1) / tile;
    tg.tiles = tg.nt[0] * tg.nt[1] * tg.nt[2];
    const int64_t blocks = (int64_t)sp->count * (tg.tiles + 1);
    PIC_REQUIRE(tile_grid_ok(blocks, sp->count));
    hipStream_t st = as_stream(stream);
    FieldPtrs fp = make_fields(E, B, E_ext, B_ext);
    const int vec_ok = groups_aligned(*in, *out, gather);
    hipLaunchKernelGGL(zero_count_kernel, dim3(1), dim3(1), 0, st, workspace);
    const SpeciesTable stab = species_table(*desc, *sp);
    bool all = true;
    for (int s = 0; s < sp->count; ++s) all = all && stab.k[s].ux == 7u && stab.k[s].uu == 7u;
#define PIC_DIRECT_LAUNCH(T, GA, EX, ALL)                                                                        \
    hipLaunchKernelGGL((fused_tile_direct_kernel<T, GA, EX, ALL>), dim3((unsigned)(blocks + kOutside * sp->count)), dim3(kThreads), 0, st, \
                       *desc, *in, fp, *out, J[0], J[1], J[2], starts, tg, grid, workspace, vec_ok, stab, gather)
#define PIC_DIRECT_ALL(T, GA, EX)                          \
    do {                                                   \
        if (all) PIC_DIRECT_LAUNCH(T, GA, EX, true);       \
        else PIC_DIRECT_LAUNCH(T, GA, EX, false);          \
    } while (0)
    // a gathered launch is only made on exact grids
#define PIC_DIRECT_SHAPE(T)                           \
    do {                                              \
        if (!exact) PIC_DIRECT_ALL(T, false, false);  \
        else if (gather) PIC_DIRECT_ALL(T, true, true); \
        else PIC_DIRECT_ALL(T, false, true);          \
    } while (0)
    if (tile == 8) PIC_DIRECT_SHAPE(8);
    else PIC_DIRECT_SHAPE(4);
#undef PIC_DIRECT_SHAPE
#undef PIC_DIRECT_ALL
#undef PIC_DIRECT_LAUNCH
    const int64_t rare_grid = std::min<int64_t>(std::max<int64_t>(grid_1d(n, kThreads), 1), 1024);
    hipLaunchKernelGGL(exact ? fused_direct_rare_kernel<true> : fused_direct_rare_kernel<false>,
                       dim3((unsigned)rare_grid), dim3(kThreads), 0, st, *desc, *sp, *in, fp, *out, J[0], J[1], J[2],
                       workspace, gather);
    PIC_CHECK_LAUNCH();
    return 0;
}

int pic_fused_push_direct_tiled(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                const float* const E[3], const float* const B[3], const float* const E_ext[3],
                                const float* const B_ext[3], PicParticles* out, float* const J[3], int32_t tile,
                                const int32_t* starts, int32_t min_blocks, int32_t* workspace, void* stream) {
    return fused_direct_tiled(desc, sp, in, E, B, E_ext, B_ext, out, J, tile, starts, min_blocks, workspace, nullptr,
                              false, stream);
}

int pic_fused_push_direct_tiled_general(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                        const float* const E[3], const float* const B[3], const float* const E_ext[3],
                                        const float* const B_ext[3], PicParticles* out, float* const J[3],
                                        int32_t tile, const int32_t* starts, int32_t* workspace, void* stream) {
    return fused_direct_tiled(desc, sp, in, E, B, E_ext, B_ext, out, J, tile, starts, 1, workspace, nullptr, true,
                              stream);
}

int pic_fused_push_direct_tiled_gather(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                       const int32_t* gather, const float* const E[3], const float* const B[3],
                                       const float* const E_ext[3], const float* const B_ext[3], PicParticles* out,
                                       float* const J[3], int32_t tile, const int32_t* starts, int32_t min_blocks,
                                       int32_t* workspace, void* stream) {
    PIC_REQUIRE(sp && (gather || (int64_t)sp->count * sp->slots == 0));
    return fused_direct_tiled(desc, sp, in, E, B, E_ext, B_ext, out, J, tile, starts, min_blocks, workspace, gather,
                              false, stream);
}

int pic_tile_general_grid(const PicDesc* desc) {
    TileGrid grid;
    return desc && desc_ok(desc) && fused_kind(*desc) == 3 && make_tile_grid(*desc, false, grid) ? 1 : 0;
}

int pic_tile_exact_grid(const PicDesc* desc) {
    ExactGrid eg;
    return desc && desc_ok(desc) && make_exact_grid(*desc, eg) ? 1 : 0;
}

// The tile kernel chooses its launch shape by the slots of a tile: rounds and
// min_blocks are those of the strided kernel.
static void launch_tile_esirkepov(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                  const FieldPtrs& fp, const PicParticles* out, float* const J[3],
                                  const int32_t* starts, const TileGeom& tg, const TileGrid& grid, bool exact,
                                  int32_t* workspace, const int32_t* gather, int64_t blocks,
                                  hipStream_t st) {
    const int vec_ok = groups_aligned(*in, *out, gather);
    hipLaunchKernelGGL(zero_count_kernel, dim3(1), dim3(1), 0, st, workspace);
    const SpeciesTable stab = species_table(*desc, *sp);
    bool all = true;
    for (int s = 0; s < sp->count; ++s) all = all && stab.k[s].ux == 7u && stab.k[s].uu == 7u;
    // Slots per thread by the mean of a block: with four a block of few slots ran in one or two of its waves.
    // 96^3, 2 / 4 / 8 / 10 per cell (128 / 256 / 512 / 640 slots): 285 / 301 / 348 / 370 us a step with four,
    // 215 / 255 / 335 / 371 by this rule (FP64 anchors 304 / 322 / 384 / 413 and 221 / 262 / 357 / 418).  Tiles of 8^3
    // cells, the phase alone, 64 / 128 / 256 / 384 / 512 slots: 105 / 118 / 137 / 144 / 150 us with four, 85 / 100 /
    // 119 / 126 / 146 by the rule (FP64 anchors 106 / 120 / 138 / 145 / 151 and 86 / 98 / 120 / 128 / 146)
    const int64_t mean = (int64_t)sp->count * sp->slots / blocks;
#define PIC_EXACT_SLOTS(T, GA, EX, ALL, P)                                                                      \
    hipLaunchKernelGGL((fused_tile_exact_kernel<T, GA, EX, ALL, P>), dim3((unsigned)(blocks + kOutside * sp->count)), dim3(kThreads), 0, st, \
                       *desc, *in, fp, *out, J[0], J[1], J[2], starts, tg, grid, workspace, vec_ok, stab, gather)
#define PIC_EXACT_LAUNCH(T, GA, EX, ALL)                                \
    do {                                                                \
        if (mean <= kThreads) PIC_EXACT_SLOTS(T, GA, EX, ALL, 1);       \
        else if (mean <= 2 * kThreads) PIC_EXACT_SLOTS(T, GA, EX, ALL, 2); \
        else PIC_EXACT_SLOTS(T, GA, EX, ALL, 4);                        \
    } while (0)
#define PIC_EXACT_ALL(T, GA, EX)                          \
    do {                                                     \
        if (all) PIC_EXACT_LAUNCH(T, GA, EX, true);       \
        else PIC_EXACT_LAUNCH(T, GA, EX, false);          \
    } while (0)
    // a gathered launch is only made on exact grids
#define PIC_EXACT_SHAPE(T)                                \
    do {                                                     \
        if (!exact) PIC_EXACT_ALL(T, false, false);       \
        else if (gather) PIC_EXACT_ALL(T, true, true);    \
        else PIC_EXACT_ALL(T, false, true);               \
    } while (0)
    if (tg.T == 8) PIC_EXACT_SHAPE(8);
    else PIC_EXACT_SHAPE(4);
#undef PIC_EXACT_SHAPE
#undef PIC_EXACT_ALL
#undef PIC_EXACT_LAUNCH
#undef PIC_EXACT_SLOTS
}

static int fused_esirkepov_tiled(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                 const float* const E[3], const float* const B[3], const float* const E_ext[3],
                                 const float* const B_ext[3], PicParticles* out, float* const J[3], int32_t tile,
                                 const int32_t* starts, int32_t rounds, int32_t min_blocks, int32_t* workspace,
                                 const int32_t* gather, bool general, void* stream) {
    PIC_REQUIRE(desc_ok(desc) && particles_ok(sp, in) && particles_ok(sp, out) && E && B && J && starts);
    PIC_REQUIRE(fused_kind(*desc) == 3 && (tile == 4 || tile == 8) &&
                (rounds == 2 || rounds == 4 || rounds == 8));
    PIC_REQUIRE(min_blocks == 1 || min_blocks == 3 || min_blocks == 4);
    const bool empty = (int64_t)sp->count * sp->slots == 0;
    for (int a = 0; a < 3; ++a)
        PIC_REQUIRE(E[a] && B[a] && J[a] && (empty || (in->x[a] != out->x[a] && in->u[a] != out->u[a])));
    PIC_REQUIRE(empty || in->active != out->active);
    PIC_REQUIRE(field_size(*desc) < ((int64_t)1 << 31));
    int64_t n = (int64_t)sp->count * sp->slots;
    PIC_REQUIRE(n < ((int64_t)1 << 31) - 8 * kThreads);
    if (n == 0) return 0;
    TileGeom tg;
    tg.T = tile;
    for (int a = 0; a < 3; ++a) tg.nt[a] = (desc->n[a] + tile - 1) / tile;
    tg.tiles = tg.nt[0] * tg.nt[1] * tg.nt[2];
    const int64_t blocks = (int64_t)sp->count * (tg.tiles + 1);
    PIC_REQUIRE(tile_grid_ok(blocks, sp->count));
    hipStream_t st = as_stream(stream);
    FieldPtrs fp = make_fields(E, B, E_ext, B_ext);
#define PIC_TILED_LAUNCH(R, T, MB)                                                                              \
    hipLaunchKernelGGL((fused_tiled_kernel<R, T, MB>), dim3((unsigned)blocks), dim3(kThreads), 0, st, *desc, *sp, \
                       *in, fp, *out, J[0], J[1], J[2], starts, tg)
#define PIC_TILED_MB(R, T)                              \
    do {                                                \
        if (min_blocks == 3) PIC_TILED_LAUNCH(R, T, 3); \
        else if (min_blocks == 4) PIC_TILED_LAUNCH(R, T, 4); \
        else PIC_TILED_LAUNCH(R, T, 1);                 \
    } while (0)
    ExactGrid eg;
    TileGrid grid;
    const bool exact = desc->variant != 1 && make_exact_grid(*desc, eg);
    if ((exact || general) && make_tile_grid(*desc, exact, grid)) {
        PIC_REQUIRE(workspace);
        launch_tile_esirkepov(desc, sp, in, fp, out, J, starts, tg, grid, exact, workspace, gather, blocks, st);
        const int64_t rare_grid = std::min<int64_t>(std::max<int64_t>(grid_1d(n, kThreads), 1), 1024);
        hipLaunchKernelGGL(fused_tile_rare_kernel, dim3((unsigned)rare_grid), dim3(kThreads), 0, st, *desc, *sp, *in,
                           fp, *out, J[0], J[1], J[2], workspace, gather);
    } else if (tile == 8) {
        if (rounds == 2) PIC_TILED_MB(2, 8);
        else PIC_TILED_MB(4, 8);
    } else {
        if (rounds == 2) PIC_TILED_MB(2, 4);
        else PIC_TILED_MB(4, 4);
    }
#undef PIC_TILED_MB
#undef PIC_TILED_LAUNCH
    PIC_CHECK_LAUNCH();
    return 0;
}

int pic_fused_push_esirkepov_tiled(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                   const float* const E[3], const float* const B[3], const float* const E_ext[3],
                                   const float* const B_ext[3], PicParticles* out, float* const J[3], int32_t tile,
                                   const int32_t* starts, int32_t rounds, int32_t min_blocks, int32_t* workspace,
                                   void* stream) {
    return fused_esirkepov_tiled(desc, sp, in, E, B, E_ext, B_ext, out, J, tile, starts, rounds, min_blocks,
                                 workspace, nullptr, false, stream);
}

int pic_fused_push_esirkepov_tiled_general(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                           const float* const E[3], const float* const B[3],
                                           const float* const E_ext[3], const float* const B_ext[3],
                                           PicParticles* out, float* const J[3], int32_t tile, const int32_t* starts,
                                           int32_t rounds, int32_t* workspace, void* stream) {
    return fused_esirkepov_tiled(desc, sp, in, E, B, E_ext, B_ext, out, J, tile, starts, rounds, 4, workspace, nullptr,
                                 true, stream);
}

int pic_fused_push_esirkepov_tiled_gather(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                          const int32_t* gather, const float* const E[3], const float* const B[3],
                                          const float* const E_ext[3], const float* const B_ext[3],
                                          PicParticles* out, float* const J[3], int32_t tile, const int32_t* starts,
                                          int32_t rounds, int32_t min_blocks, int32_t* workspace, void* stream) {
    ExactGrid eg;
    PIC_REQUIRE(desc && desc_ok(desc) && sp && desc->variant != 1 && make_exact_grid(*desc, eg));
    PIC_REQUIRE(gather || (int64_t)sp->count * sp->slots == 0);
    return fused_esirkepov_tiled(desc, sp, in, E, B, E_ext, B_ext, out, J, tile, starts, rounds, min_blocks,
                                 workspace, gather, false, stream);
}

}  // extern "C"
