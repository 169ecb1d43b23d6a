// Particle phase of first-order 1-D and 2-D runs (active axes x or x, y) in slot
// order: gather, push, Esirkepov deposit, position update and boundaries of a
// chunk of kBlk * kP slots per block.
//
// The block bounds the cells of its slots.  Sorted particles cover a few cells
// or rows, so E + E_ext, B + B_ext of the range and the J of the range fit in LDS
// (kBoxed): a particle then reads LDS where it read 24 array values, and J, summed
// in FP64 (ds_add_f64, a tenth of the time of ds_add_f32 on this card), is added
// into the arrays once per block.  A wider range keeps an FP32 J box, or none, and
// gathers from the arrays.  As in the 3-D tile kernel a thread owns kP consecutive
// slots, the moments of a cell's particles are summed in registers and over
// neighbouring lanes, anchors are relative to the box and exact wherever an FP64
// evaluation could decide otherwise, and particles that leave their cell are
// queued and deposited in the 3-slot frame by lanes that all do so.
//
// Bound by the latency of a chunk's stages, so blocks are kept at sixteen waves
// a CU.  64 members of up to 256 x 32 cells, 8.7M slots in order: 329 to 343 us,
// 852 us where each 256 slots were scanned by lane shuffles into an FP32 box; 262k
// slots on 64 x 64: 25 us, 52 us before.  (A node's value is a difference of FP32
// moments, so one of small weight carries the rounding of the cell's current; J
// is as far from its FP64 value as sums of single node values, 4.2e-7 against
// 4.9e-7 in the norm for two beams on 64 x 64.)  As slots lose their order ranges widen:
// 80 KB of boxes (2 x 512 threads a CU) hold them longer than 40 KB (4 x 256, 10 %
// faster in order, 25 % slower after 400 steps).
#pragma once
#include "pic_fused_block.h"

namespace {

constexpr int kPlanarBlock = 512;

// Bytes of a block's boxes: what leaves sixteen waves a CU beside a queue as long as the chunk.  A boxed node holds
// 6 FP32 and 3 FP64 values.
template <int kP, int kBlk>
constexpr int kPlanarLds = ((160 << 10) / (1024 / kBlk) - 1536 - kBlk * kP * 14) / 48 * 48;
template <int kP, int kBlk>
constexpr int kPlanarNodes = kPlanarLds<kP, kBlk> / 48;

// Grid constants of an active axis (the terms of TileGrid).
struct PlanarAxis {
    double org, sp, half, inv_d64;
    float isp, bias, edge, lim, inv_d, org32;
};

// False where the vertex line is not the centre line shifted by half a spacing up to rounding.
__host__ __device__ inline bool planar_axis(const PicDesc& d, int a, PlanarAxis& p) {
    const double org = d.org_c[a], sp = d.sp_c[a], off = d.org_v[a] - org - 0.5 * sp;
    p.org = org;
    p.sp = sp;
    p.half = 0.5 * sp;
    p.inv_d64 = 1.0 / d.d[a];
    p.isp = (float)(1.0 / sp);
    p.bias = 0x1p-22f * ((float)(fabs(org) / sp) + d.dims[a] + 32.0f);
    p.edge = (float)((0.5 - 0x1p-20) * sp);
    p.lim = (float)((0.5 - 0x1p-19) * sp);
    p.inv_d = (float)(1.0 / d.d[a]);
    p.org32 = (float)org;
    return sp > 0.0 && d.d[a] > 0.0 && d.dims[a] <= (1 << 20) && fabs(off) <= 1.0e-7 * sp &&
           fabs(d.sp_v[a] - sp) * d.dims[a] <= 1.0e-7 * sp && fabs(org) <= 4.0e6 * sp;
}

__host__ __device__ inline bool planar_covers(const PicDesc& d) {
    const int kind = fused_kind(d);
    PlanarAxis p;
    return (kind == 1 || kind == 2) && planar_axis(d, 0, p) && (kind == 1 || planar_axis(d, 1, p));
}

template <int kP, int kBlk>
struct PlanarShared {
    alignas(16) char box[kPlanarLds<kP, kBlk>];
    float v[3][kBlk * kP];
    uint16_t slot[kBlk * kP];
    SpeciesK spk[PIC_MAX_SPECIES];
    PlanarAxis ax[2];
    int q_n, ok[2], lo[2], hi[2];
};

template <int kDims>
struct PlanarMoments {
    static constexpr int kN = kDims == 2 ? 8 : 5;
};

// J of the nodes a cell's particles share, from their moments: 2-D Jx (1, A_y), Jy (1, A_x), Jz (1, A_x, A_y,
// A_x A_y + d_x d_y / 12), 1-D Jx (1), Jy, Jz (1, A_x); a node's value is the product of A or 1 - A.
template <int kDims, class Sink>
__device__ __forceinline__ void flush_planar(const PicDesc& d, const Sink& sink, int i, int j, const float* m) {
    const int g = d.g;
    if constexpr (kDims == 2) {
        sink.add(d, 0, i, j, g, m[0] - m[1]);
        sink.add(d, 0, i, j + 1, g, m[1]);
        sink.add(d, 1, i, j, g, m[2] - m[3]);
        sink.add(d, 1, i + 1, j, g, m[3]);
        sink.add(d, 2, i, j, g, (m[4] - m[5]) - (m[6] - m[7]));
        sink.add(d, 2, i + 1, j, g, m[5] - m[7]);
        sink.add(d, 2, i, j + 1, g, m[6] - m[7]);
        sink.add(d, 2, i + 1, j + 1, g, m[7]);
    } else {
        sink.add(d, 0, i, g, g, m[0]);
        sink.add(d, 1, i, g, g, m[1] - m[2]);
        sink.add(d, 1, i + 1, g, g, m[2]);
        sink.add(d, 2, i, g, g, m[3] - m[4]);
        sink.add(d, 2, i + 1, g, g, m[4]);
    }
}

// One component from its box plane at p (row stride e1): the sums of gather_n.
template <int kDims>
__device__ __forceinline__ float planar_gather(const float* p, int e1, const float (&wx)[2], const float (&wy)[2]) {
    if constexpr (kDims == 2) {
        const float a = mix<true>(wy[0], p[0], wy[1], p[1]), b = mix<true>(wy[0], p[e1], wy[1], p[e1 + 1]);
        return mix<true>(wx[0], a, wx[1], b);
    } else {
        return mix<true>(wx[0], p[0], wx[1], p[1]);
    }
}

// The slots of a chunk.  kBoxed: fields at fbox, J into sink's FP64 box; e[] are its extents, o[] its origin.
template <int kDims, int kP, int kBlk, bool kBoxed, class Sink>
__device__ __forceinline__ void planar_slots(const PicDesc& d, const PicSpecies& sp, const PicParticles& in,
                                    const FieldPtrs& fp, const PicParticles& out, const Sink& sink, int64_t n,
                                    uint32_t base, bool full, float (&PX)[3][kP], float (&PU)[3][kP], uint32_t pact,
                                    PlanarShared<kP, kBlk>& sh, const float* fbox, const int (&o)[2], const int (&e)[2]) {
    constexpr int kN = PlanarMoments<kDims>::kN;
    const int vol = kDims == 2 ? e[0] * e[1] : e[0];
    const float dt32 = (float)d.dt;
    float isp[kDims], bias[kDims], edge[kDims], lim[kDims], inv_d[kDims], nb[kDims];
#pragma unroll
    for (int a = 0; a < kDims; ++a) {
        const PlanarAxis& x = sh.ax[a];
        isp[a] = uniform(x.isp);
        bias[a] = uniform(x.bias);
        edge[a] = uniform(x.edge);
        lim[a] = uniform(x.lim);
        inv_d[a] = uniform(x.inv_d);
        nb[a] = uniform((float)node_coord(o[a], x.sp, x.org));
    }
    const uint32_t i0 = base + (uint32_t)(kP * threadIdx.x);
    int s = species_of(i0, sp.slots, sp.count);
    int64_t s_end = (int64_t)(s + 1) * sp.slots;
    float acc[kN];
#pragma unroll
    for (int m = 0; m < kN; ++m) acc[m] = 0.0f;
    int cell = -1;
    // a cell's key: its place in the box, or in the arrays with a margin
    const int row = kBoxed ? e[1] : d.dims[1] + 16;
    const auto flush = [&]() {
        const int i = kDims == 2 ? cell / row : cell, j = kDims == 2 ? cell % row : 0;
        flush_planar<kDims>(d, sink, kBoxed ? i + o[0] : i - 8, kBoxed ? j + o[1] : j - 8, acc);
    };
    uint32_t oact = 0u;
#pragma unroll
    for (int j = 0; j < kP; ++j) {
        const float xf[3] = {PX[0][j], PX[1][j], PX[2][j]};
        float v[3] = {PU[0][j], PU[1][j], PU[2][j]};
        const bool act0 = ((pact >> (8 * j)) & 0xffu) != 0u;
        while (s + 1 < sp.count && (int64_t)i0 + j >= s_end) {
            ++s;
            s_end += sp.slots;
        }
        PX[0][j] = PX[1][j] = PX[2][j] = PU[0][j] = PU[1][j] = PU[2][j] = 0.0f;
        if (!act0) continue;
        const SpeciesK& k = sh.spk[s];
        float dc[kDims], qm[kDims], E[3], B[3];
        int key = -2;
        if constexpr (kBoxed) {
            // ---- anchors relative to the box (tile_anchor); the exact division where it could round either way
            int f[2] = {0, 0};
            bool up[2] = {true, true};
            float wc[2][2], wv[2][2];
#pragma unroll
            for (int a = 0; a < kDims; ++a) {
                const PlanarAxis& x = sh.ax[a];
                int fa = (int)floorf(fmaf(xf[a] - nb[a], isp[a], bias[a]));
                fa = min(max(fa, 1), e[a] - 3);
                double dd = (double)xf[a] - node_coord(fa + o[a], x.sp, x.org);
                float q = (float)(dd - x.half);
                if (!(fabsf(q) < edge[a])) {
                    fa = min(max(anchor_of((double)xf[a], x.org, x.sp, 1) - o[a], 1), e[a] - 3);
                    dd = (double)xf[a] - node_coord(fa + o[a], x.sp, x.org);
                    q = (float)(dd - x.half);
                }
                f[a] = fa;
                dc[a] = (float)dd;
                qm[a] = q;
                up[a] = q >= 0.0f;
                const float dv = (float)(up[a] ? dd - x.half : dd - x.half + x.sp);
                wc[a][0] = fmaf(-dc[a], isp[a], 1.0f);
                wc[a][1] = dc[a] * isp[a];
                wv[a][0] = fmaf(-dv, isp[a], 1.0f);
                wv[a][1] = dv * isp[a];
            }
            if constexpr (kDims == 1) {
#pragma unroll
                for (int q = 0; q < 2; ++q) wc[1][q] = wv[1][q] = 0.0f;
            }
            key = kDims == 2 ? f[0] * e[1] + f[1] : f[0];
            const int lx = up[0] ? 0 : (kDims == 2 ? e[1] : 1), ly = kDims == 1 || up[1] ? 0 : 1;
            const float* p = fbox + key;
            E[0] = planar_gather<kDims>(p - lx, e[1], wv[0], wc[1]);
            E[1] = planar_gather<kDims>(p + vol - ly, e[1], wc[0], wv[1]);
            E[2] = planar_gather<kDims>(p + 2 * vol, e[1], wc[0], wc[1]);
            B[0] = planar_gather<kDims>(p + 3 * vol - ly, e[1], wc[0], wv[1]);
            B[1] = planar_gather<kDims>(p + 4 * vol - lx, e[1], wv[0], wc[1]);
            B[2] = planar_gather<kDims>(p + 5 * vol - lx - ly, e[1], wv[0], wv[1]);
        } else {
            CicAxis gc[3], gv[3];
            int anc[2] = {0, 0}, anv;
            float dv;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if (a < kDims) {
                    cic_axis(xf[a], sh.ax[a].org32, isp[a], d.org_c[a], d.sp_c[a], d.dims[a], gc[a], anc[a], dc[a]);
                    cic_axis(xf[a], (float)d.org_v[a], isp[a], d.org_v[a], d.sp_v[a], d.dims[a], gv[a], anv, dv);
                    qm[a] = dc[a] - (float)sh.ax[a].half;
                } else {
                    reduced_cic(d.g, gc[a]);
                    reduced_cic(d.g, gv[a]);
                }
            }
            constexpr int NY = kDims;
            const uint32_t sy = (uint32_t)d.dims[2], sx = (uint32_t)d.dims[1] * sy;
            E[0] = gather_n<2, NY, 1>(fp.E[0], fp.Ee[0], sx, sy, gv[0], gc[1], gc[2]);
            E[1] = gather_n<2, NY, 1>(fp.E[1], fp.Ee[1], sx, sy, gc[0], gv[1], gc[2]);
            E[2] = gather_n<2, NY, 1>(fp.E[2], fp.Ee[2], sx, sy, gc[0], gc[1], gv[2]);
            B[0] = gather_n<2, NY, 1>(fp.B[0], fp.Be[0], sx, sy, gc[0], gv[1], gv[2]);
            B[1] = gather_n<2, NY, 1>(fp.B[1], fp.Be[1], sx, sy, gv[0], gc[1], gv[2]);
            B[2] = gather_n<2, NY, 1>(fp.B[2], fp.Be[2], sx, sy, gv[0], gv[1], gc[2]);
            bool near = true;
#pragma unroll
            for (int a = 0; a < kDims; ++a) near = near & (anc[a] >= -8) & (anc[a] < d.dims[a] + 8);
            if (near) key = kDims == 2 ? (anc[0] + 8) * row + anc[1] + 8 : anc[0] + 8;
        }
        // ---- push (boris.py:14-124), masked by update_u (particle_push.py:134-142)
        float nv[3] = {v[0], v[1], v[2]};
        push_velocity(nv, E, B, k.h, d);
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if ((k.uu >> a) & 1u) v[a] = nv[a];
        // ---- a particle that stays in its cell, away from the faces (see fused_tile_exact_kernel)
        bool regular = key >= 0;
        float D[2] = {0.0f, 0.0f}, A[2] = {0.0f, 0.0f};
#pragma unroll
        for (int a = 0; a < kDims; ++a) {
            const float dvt = (k.ux >> a) & 1u ? v[a] * dt32 : 0.0f;
            regular = regular & (fabsf(qm[a] + dvt) < lim[a]);
            D[a] = dvt * inv_d[a];
            A[a] = fmaf(0.5f, D[a], dc[a] * inv_d[a]);
        }
        if (regular) {
            if (key != cell) {
                if (cell >= 0) flush();
#pragma unroll
                for (int m = 0; m < kN; ++m) acc[m] = 0.0f;
                cell = key;
            }
            const float px = k.pre[0] * (-D[0]), pz = k.q_dv * v[2];
            acc[0] += px;
            if constexpr (kDims == 2) {
                const float py = k.pre[1] * (-D[1]);
                acc[1] = fmaf(px, A[1], acc[1]);
                acc[2] += py;
                acc[3] = fmaf(py, A[0], acc[3]);
                acc[4] += pz;
                acc[5] = fmaf(pz, A[0], acc[5]);
                acc[6] = fmaf(pz, A[1], acc[6]);
                acc[7] = fmaf(pz, fmaf(A[0], A[1], D[0] * (D[1] * (1.0f / 12.0f))), acc[7]);
            } else {
                const float py = k.q_dv * v[1];
                acc[1] += py;
                acc[2] = fmaf(py, A[0], acc[2]);
                acc[3] += pz;
                acc[4] = fmaf(pz, A[0], acc[4]);
            }
        } else {
            const int q = atomicAdd(&sh.q_n, 1);
            sh.slot[q] = (uint16_t)(kP * threadIdx.x + j);
#pragma unroll
            for (int a = 0; a < 3; ++a) sh.v[a][q] = v[a];
        }
        // ---- position update + particle boundaries (particle_tile_communication.py)
        bool act = true;
        double xn[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            xn[a] = ((k.ux >> a) & 1u) ? step_pos((double)xf[a], (double)v[a], d.dt) : (double)xf[a];
            double wind = d.wind[a];
            asm volatile("" : "+v"(wind));      // see fused_tile_exact_kernel
            if (d.pbc[a] == 0) periodic_wrap(wind, xn[a]);
            else apply_axis_boundary(d.pbc[a], wind, xn[a], v[a], act);
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            PX[a][j] = act ? (float)xn[a] : 0.0f;
            PU[a][j] = act ? v[a] : 0.0f;
        }
        oact |= (act ? 1u : 0u) << (8 * j);
    }
    if constexpr (kP > 1) {
        store_group<kP>(out, i0, 0, n, full, PX, PU, oact);
    } else if (i0 < n) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            out.x[a][i0] = PX[a][0];
            out.u[a][i0] = PU[a][0];
        }
        out.active[i0] = (uint8_t)oact;
    }
    // equal cells of neighbouring lanes first: sixteen lanes, or four of four slots each
    if (row_run_sums<kP < 4 ? 16 : 4>(cell, acc) && cell >= 0) flush();
    __syncthreads();
    // ---- queued particles (Esirkepov.py:105-331)
    const int nq = sh.q_n;
    for (int q = threadIdx.x; q < nq; q += kBlk) {
        const uint32_t i = base + (uint32_t)sh.slot[q];
        const SpeciesK& k = sh.spk[species_of(i, sp.slots, sp.count)];
        const float v[3] = {sh.v[0][q], sh.v[1][q], sh.v[2][q]};
        double xo[3], xn[3];
        load_pos(in, i, xo);
#pragma unroll
        for (int a = 0; a < 3; ++a) xn[a] = ((k.ux >> a) & 1u) ? step_pos(xo[a], (double)v[a], d.dt) : xo[a];
        CrossAxis c[2];
        bool ok = true;
#pragma unroll
        for (int a = 0; a < kDims; ++a) {
            const PlanarAxis& x = sh.ax[a];
            ok = cross_axis(xo[a], xn[a], x.org, x.sp, x.inv_d64, x.org32, x.isp, c[a]) && ok;
        }
        if (ok) {
            crossing_deposit_reduced<kDims>(d, k, v, c[0], c[kDims - 1], sink);
        } else {
            float* const J[3] = {sink.J[0], sink.J[1], sink.J[2]};
            esirkepov_particle(d, k.qw, xo, xn, v, J);   // moved two or more cells
        }
    }
    __syncthreads();
}

// One step of a minimum and maximum over rows of 16 lanes (every lane receives it after steps 1, 2, 4, 8).
template <int kOff>
__device__ inline void row_min_max(int& lo, int& hi) {
    lo = min(lo, __builtin_amdgcn_update_dpp(lo, lo, 0x120 + kOff, 0xf, 0xf, false));     // row_ror
    hi = max(hi, __builtin_amdgcn_update_dpp(hi, hi, 0x120 + kOff, 0xf, 0xf, false));
}

// Adds the non-zero values of a range box into J.
template <int kBlk, class Sink>
__device__ inline void flush_range_box(const PicDesc& d, const Sink& sink, int vol) {
    for (int e = threadIdx.x; e < 3 * vol; e += kBlk) {
        const float val = (float)sink.box[e];
        if (val == 0.0f) continue;
        const int c = e / vol, r = e % vol;
        deposit_at(sink.J[c], d, sink.o[0] + r / sink.e[1], sink.o[1] + r % sink.e[1], sink.o[2], val);
    }
}

template <int kDims, int kP, int kBlk>
__device__ __forceinline__ void planar_chunk(const PicDesc& d, const PicSpecies& sp, const PicParticles& in,
                                    const FieldPtrs& fp, const PicParticles& out, float* const J[3], int64_t n,
                                    uint32_t base, bool vec_ok, PlanarShared<kP, kBlk>& sh) {
    const uint32_t i0 = base + (uint32_t)(kP * threadIdx.x);
    const bool full = kP > 1 && vec_ok && (int64_t)i0 + kP <= n;
    float PX[3][kP], PU[3][kP];
    uint32_t pact;
    load_group<kP, false>(in, nullptr, i0, 0, n, full, PX, PU, pact);
    // constants: the axes by one wave, the species by another
    if (threadIdx.x < 2) {
        sh.lo[threadIdx.x] = INT_MAX;
        sh.hi[threadIdx.x] = INT_MIN;
        sh.ok[threadIdx.x] = (int)threadIdx.x >= kDims || planar_axis(d, threadIdx.x, sh.ax[threadIdx.x]);
    } else if (threadIdx.x == 2) {
        sh.q_n = 0;
    } else if (threadIdx.x >= 64 && (int)threadIdx.x - 64 < sp.count) {
        sh.spk[threadIdx.x - 64] = species_constants(d, sp, threadIdx.x - 64);
    }
    __syncthreads();
    if (!sh.ok[0] || !sh.ok[1]) return;      // (the general kernel's)
    // ---- range of the centre anchors (FP32 estimate, within one of the anchor below kFar, four times the longest
    // axis; a chunk with a particle beyond gets no box, so no anchor is taken relative to a clamped range)
    constexpr int kFar = 1 << 22;
    int lo[2] = {INT_MAX, INT_MAX}, hi[2] = {INT_MIN, INT_MIN};
#pragma unroll
    for (int a = 0; a < kDims; ++a) {
        const float org = sh.ax[a].org32, isp = sh.ax[a].isp;
#pragma unroll
        for (int j = 0; j < kP; ++j) {
            if (((pact >> (8 * j)) & 0xffu) == 0u) continue;
            const int c = (int)fminf(fmaxf(floorf((PX[a][j] - org) * isp), -(float)kFar), (float)kFar);
            lo[a] = min(lo[a], c);
            hi[a] = max(hi[a], c);
        }
        // over rows of 16 lanes, then one lane a row
        row_min_max<1>(lo[a], hi[a]);
        row_min_max<2>(lo[a], hi[a]);
        row_min_max<4>(lo[a], hi[a]);
        row_min_max<8>(lo[a], hi[a]);
        if ((threadIdx.x & 15) == 0) {
            atomicMin(&sh.lo[a], lo[a]);
            atomicMax(&sh.hi[a], hi[a]);
        }
    }
    __syncthreads();
    // two nodes below and three above: the estimate's rounding, the stencil, a face crossing
    int o[2] = {0, d.g}, e[2] = {1, 1};
    int64_t vol = 1;
    const bool any = sh.lo[0] <= sh.hi[0];
    bool far = false;
#pragma unroll
    for (int a = 0; a < kDims; ++a) {
        far = far || (any && (sh.lo[a] <= -kFar || sh.hi[a] >= kFar));
        o[a] = __builtin_amdgcn_readfirstlane(any ? sh.lo[a] - 2 : 0);
        e[a] = __builtin_amdgcn_readfirstlane(any ? sh.hi[a] - sh.lo[a] + 6 : 6);
        vol *= e[a];
    }
    if (far) vol = INT64_MAX / 64;
    if (vol <= kPlanarNodes<kP, kBlk>) {
        float* fbox = reinterpret_cast<float*>(sh.box);
        double* box = reinterpret_cast<double*>(sh.box + 24 * kPlanarNodes<kP, kBlk>);
        const int v = (int)vol;
        // all loads of the arrays in flight before the first is used
        constexpr int kR = (kPlanarNodes<kP, kBlk> + kBlk - 1) / kBlk;
        float val[kR][6];
        int off[kR];
#pragma unroll
        for (int q = 0; q < kR; ++q) {
            const int r = min((int)threadIdx.x + q * kBlk, v - 1);
            off[q] = (int)fidx(d, pmod(o[0] + r / e[1], d.dims[0]),
                               kDims == 2 ? pmod(o[1] + r % e[1], d.dims[1]) : d.g, d.g);
#pragma unroll
            for (int c = 0; c < 6; ++c) val[q][c] = (c < 3 ? fp.E[c] : fp.B[c - 3])[off[q]];
        }
        for (int r = threadIdx.x; r < 3 * v; r += kBlk) box[r] = 0.0;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const float* Fe = c < 3 ? fp.Ee[c] : fp.Be[c - 3];
#pragma unroll
            for (int q = 0; q < kR; ++q) {
                const int r = (int)threadIdx.x + q * kBlk;
                if (Fe) val[q][c] += Fe[off[q]];
                if (r < v) fbox[c * v + r] = val[q][c];
            }
        }
        __syncthreads();
        const RangeBoxSink<double> sink{{J[0], J[1], J[2]}, box, {o[0], o[1], d.g}, {e[0], e[1], 1}, true};
        planar_slots<kDims, kP, kBlk, true>(d, sp, in, fp, out, sink, n, base, full, PX, PU, pact, sh, fbox, o, e);
        flush_range_box<kBlk>(d, sink, v);
    } else if (24 * vol <= kPlanarLds<kP, kBlk>) {
        double* box = reinterpret_cast<double*>(sh.box);
        const int v = (int)vol;
        for (int r = threadIdx.x; r < 3 * v; r += kBlk) box[r] = 0.0;
        __syncthreads();
        const RangeBoxSink<double> sink{{J[0], J[1], J[2]}, box, {o[0], o[1], d.g}, {e[0], e[1], 1}, true};
        planar_slots<kDims, kP, kBlk, false>(d, sp, in, fp, out, sink, n, base, full, PX, PU, pact, sh, nullptr, o, e);
        flush_range_box<kBlk>(d, sink, v);
    } else {
        float* box = reinterpret_cast<float*>(sh.box);
        const bool on = 12 * vol <= kPlanarLds<kP, kBlk>;
        const int v = on ? (int)vol : 0;
        for (int r = threadIdx.x; r < 3 * v; r += kBlk) box[r] = 0.0f;
        __syncthreads();
        const RangeBoxSink<float> sink{{J[0], J[1], J[2]}, box, {o[0], o[1], d.g}, {e[0], e[1], 1}, on};
        planar_slots<kDims, kP, kBlk, false>(d, sp, in, fp, out, sink, n, base, full, PX, PU, pact, sh, nullptr, o, e);
        flush_range_box<kBlk>(d, sink, v);
    }
    __syncthreads();   // the next chunk reuses the boxes and the queue
}

}  // namespace
