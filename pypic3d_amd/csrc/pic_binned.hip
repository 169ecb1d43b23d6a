// Deposits of particles in any slot order (3-D), and the fused push +
// Esirkepov phase built on them.
//
// What bounds a deposit straight into the arrays is the rate of global float
// atomics: about 20 G/s on this card whatever the order of the particles
// (rho, 16.8M particles in cell order: 7.3 ms; 4.2M in random order: 1.7 ms;
// the 12 values of the Esirkepov deposit, 4.2M random: 2.6 ms).  Here the
// particles are first split into bins of cells (tiles):
//   count    reads the positions, one LDS histogram per chunk of slots, one
//            global atomic per (chunk, tile);
//   scan     one block: first record and first work item of every tile;
//   scatter  ranks the chunk's particles in LDS, reserves the chunk's share
//            of each tile with one returning atomic, writes one record
//            (position, velocity or charge) per particle: a chunk's records of
//            a tile are contiguous, so L2 merges their lines;
//   deposit  one block per work item (records of one tile) adds into an LDS
//            box and the box once into the arrays.
// The boxes are FP64: an LDS float atomic takes 3 cycles per lane on this
// card, whatever its address (ds_add_f32, 192 cycles a wave), a double one 0.24
// to 0.36 (ds_add_f64, 16 to 23), so the wider sum is also the faster one.
// Equal tiles, then equal cells, in neighbouring lanes are combined first
// (row_run_position, row_run_sums), so sorted input does not serialise on one
// LDS word.  Per particle this moves 13 bytes (count), 25-50 (scatter) and 16
// or 32 (deposit).
#include "pic_fused_block.h"

namespace {

// Box nodes below the tile's first cell and in all beyond its edge: points a,
// a+1 (first order) or a-1 .. a+1 of an anchor a from the tile or, after a
// step, next to it.
__host__ __device__ inline int box_margin(int shape) { return shape == 1 ? 1 : 2; }
__host__ __device__ inline int box_pad(int shape) { return shape == 1 ? 3 : 5; }
constexpr int kMaxTiles = 8192;         // LDS histogram of 32 KB beside a chunk's 16 KB of places
constexpr int kQueue = 2048;            // face crossings held by a block, 4 KB
constexpr int kMaxBoxBytes = 59 * 1024; // with the queue below the 64 KB of a launch
constexpr int kItem = 8192;             // records per work item
// Threads of the kernels that work on an item's LDS box: a box is used by one
// block, so the waves that hide the latency of a CU have to come from that
// block (4.2M records in random order, 512 items: 403 us with 256 threads).
constexpr int kWide = 1024;

struct BinGeom {
    int T[3], shift[3], nt[3], e[3];    // tile edge (a power of two), tiles per axis, box extent per axis
    int tiles, box, margin;             // tiles, box nodes per component, nodes below the tile
    float org[3], isp[3];
};

// Tiles of 8^3 cells; edges double (x first) until the histogram fits.
bool bin_geom(const PicDesc& d, int comps, BinGeom& g) {
    for (int a = 0; a < 3; ++a) g.shift[a] = 3;
    g.margin = box_margin(d.shape_factor);
    for (int turn = 0;; ++turn) {
        int64_t tiles = 1;
        g.box = 1;
        for (int a = 0; a < 3; ++a) {
            g.T[a] = 1 << g.shift[a];
            // cells -g .. n+g-1 of the centre line belong to the tiles of their clamped index
            g.nt[a] = (d.n[a] + g.T[a] - 1) / g.T[a];
            g.e[a] = g.T[a] + box_pad(d.shape_factor);
            g.org[a] = (float)d.org_c[a];
            g.isp[a] = (float)(1.0 / d.sp_c[a]);
            tiles *= g.nt[a];
            g.box *= g.e[a];
        }
        if ((int64_t)g.box * comps * 8 > kMaxBoxBytes) return false;
        if (tiles <= kMaxTiles) {
            g.tiles = (int)tiles;
            return true;
        }
        ++g.shift[turn % 3];
    }
}

// Tile of a position from the FP32 estimate of its centre-line anchor; a
// particle whose nodes leave the tile's box deposits straight into the arrays,
// so the estimate need not be exact.
__device__ inline int tile_of(const PicDesc& d, const BinGeom& g, const float x[3]) {
    int t[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float f = fminf(fmaxf(floorf((x[a] - g.org[a]) * g.isp[a]), 0.0f), 1.0e6f);
        const int c = min(max((int)f - d.g, 0), d.n[a] - 1);
        t[a] = c >> g.shift[a];
    }
    return (t[0] * g.nt[1] + t[1]) * g.nt[2] + t[2];
}

struct BinWork {
    uint32_t* random;   // [1] the slots are in no cell order (bin_sample_kernel)
    uint32_t* count;    // [tiles] counts, then the cursors of the scatter
    uint32_t* first;    // [tiles + 1] first record of a tile
    uint32_t* item;     // [tiles + 1] first work item of a tile
    float4* rec;        // records
    uint32_t* place;    // [slots] record of a slot (the push through tiles only)
};

// Bytes of the flag and the three tables, and of n records.
int64_t bin_tables(int tiles) { return (((int64_t)(3 * (tiles + 1) + 1) * 4 + 255) / 256) * 256; }

enum RecordKind : int { REC_RHO = 0, REC_DIRECT = 1, REC_ESIRKEPOV = 2, REC_PUSH = 3 };

int64_t bin_records(int kind, int64_t n) { return n * (kind == REC_RHO ? 16 : 32); }

BinWork bin_work(void* ws, int tiles, int kind, int64_t n) {
    BinWork w;
    w.random = static_cast<uint32_t*>(ws);
    w.count = w.random + 1;
    w.first = w.count + tiles + 1;
    w.item = w.first + tiles + 1;
    char* rec = static_cast<char*>(ws) + bin_tables(tiles);
    w.rec = reinterpret_cast<float4*>(rec);
    w.place = reinterpret_cast<uint32_t*>(rec + bin_records(kind, n));
    return w;
}

// Clears the counts; one block also samples the slot order: pairs of
// consecutive slots spread over the set.  A sorted set has almost every pair in
// one tile, positions drawn over the domain almost none; half way between, the
// gather in slot order (33 ps a particle sorted, 160 ps random) and the push
// through tiles cost about the same.
constexpr int kSamples = 1024;

__global__ __launch_bounds__(kSamples) void bin_start_kernel(PicDesc d, BinGeom g, PicParticles in, BinWork w,
                                                              int64_t n) {
    for (int e = blockIdx.x * kSamples + threadIdx.x; e < g.tiles; e += gridDim.x * kSamples) w.count[e] = 0u;
    if (blockIdx.x) return;
    __shared__ int pairs, split;
    if (threadIdx.x == 0) pairs = split = 0;
    __syncthreads();
    const int64_t i = (n - 1) / kSamples * threadIdx.x;
    if (i + 1 < n && in.active[i] && in.active[i + 1]) {
        const float x0[3] = {in.x[0][i], in.x[1][i], in.x[2][i]};
        const float x1[3] = {in.x[0][i + 1], in.x[1][i + 1], in.x[2][i + 1]};
        atomicAdd(&pairs, 1);
        if (tile_of(d, g, x0) != tile_of(d, g, x1)) atomicAdd(&split, 1);
    }
    __syncthreads();
    if (threadIdx.x == 0) *w.random = 2 * split > pairs ? 1u : 0u;
}

// A chunk is kThreads * kItems consecutive slots.
template <int kItems>
__global__ __launch_bounds__(kThreads) void bin_count_kernel(PicDesc d, BinGeom g, PicParticles in,
                                                              uint32_t* __restrict__ count, int64_t n,
                                                              const uint32_t* run) {
    extern __shared__ uint32_t hist[];
    if (run && !*run) return;
    for (int e = threadIdx.x; e < g.tiles; e += kThreads) hist[e] = 0u;
    __syncthreads();
    const int64_t b0 = (int64_t)blockIdx.x * (kThreads * kItems);
    for (int k = 0; k < kItems; ++k) {
        const int64_t i = b0 + k * kThreads + threadIdx.x;
        int t = -1;
        if (i < n && in.active[i]) {
            const float x[3] = {in.x[0][i], in.x[1][i], in.x[2][i]};
            t = tile_of(d, g, x);
        }
        int p, q;
        row_run_position(t, p, q);
        if (t >= 0 && q == 1) atomicAdd(&hist[t], (uint32_t)p);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < g.tiles; e += kThreads)
        if (hist[e]) atomicAdd(&count[e], hist[e]);
}

// One block: exclusive prefix of the counts and of the work items per tile;
// the counts become the scatter's cursors.
__global__ __launch_bounds__(1024) void bin_scan_kernel(BinWork w, int tiles, const uint32_t* run) {
    __shared__ uint32_t sc[1024], si[1024];
    if (run && !*run) return;
    uint32_t carry = 0u, carry_item = 0u;
    for (int base = 0; base < tiles; base += 1024) {
        const int e = base + (int)threadIdx.x;
        const uint32_t c = e < tiles ? w.count[e] : 0u, m = (c + kItem - 1) / kItem;
        sc[threadIdx.x] = c;
        si[threadIdx.x] = m;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {
            const uint32_t ac = (int)threadIdx.x >= off ? sc[threadIdx.x - off] : 0u;
            const uint32_t ai = (int)threadIdx.x >= off ? si[threadIdx.x - off] : 0u;
            __syncthreads();
            sc[threadIdx.x] += ac;
            si[threadIdx.x] += ai;
            __syncthreads();
        }
        if (e < tiles) {
            const uint32_t f = carry + sc[threadIdx.x] - c;
            w.first[e] = f;
            w.count[e] = f;
            w.item[e] = carry_item + si[threadIdx.x] - m;
        }
        carry += sc[1023];
        carry_item += si[1023];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        w.first[tiles] = carry;
        w.item[tiles] = carry_item;
    }
}

// Ranks the chunk's slots by tile: afterwards place[s] is the record index of
// local slot s (kNoRecord: inactive or past the end).
constexpr uint32_t kNoRecord = 0xffffffffu;

template <int kItems>
__device__ inline void chunk_places(const PicDesc& d, const BinGeom& g, const PicParticles& in, int64_t b0, int64_t n,
                                    uint32_t* __restrict__ cursor, uint32_t* hist, uint32_t* place) {
    for (int e = threadIdx.x; e < g.tiles; e += kThreads) hist[e] = 0u;
    __syncthreads();
    const int lane = (int)(threadIdx.x & 63u);
    for (int k = 0; k < kItems; ++k) {
        const int s = k * kThreads + (int)threadIdx.x;
        const int64_t i = b0 + s;
        int t = -1;
        if (i < n && in.active[i]) {
            const float x[3] = {in.x[0][i], in.x[1][i], in.x[2][i]};
            t = tile_of(d, g, x);
        }
        int p, q;
        row_run_position(t, p, q);
        uint32_t base = 0u;
        if (t >= 0 && q == 1) base = atomicAdd(&hist[t], (uint32_t)p);
        base = (uint32_t)__shfl((int)base, lane + q - 1);      // the run's last lane holds its first rank
        // 14 bits of tile (tiles <= 8192), 18 bits of rank inside the chunk
        place[s] = t >= 0 ? ((uint32_t)t << 18) | (base + (uint32_t)p - 1u) : kNoRecord;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < g.tiles; e += kThreads)
        if (hist[e]) hist[e] = atomicAdd(&cursor[e], hist[e]);
    __syncthreads();
    for (int k = 0; k < kItems; ++k) {
        const int s = k * kThreads + (int)threadIdx.x;
        if (place[s] != kNoRecord) place[s] = hist[place[s] >> 18] + (place[s] & 0x3ffffu);
    }
}

// rho: (x, q w / dV).  J_from_rhov: (x, 0), (q w / dV v, 0).  Esirkepov and
// push: (x, species), (v, 0).
template <int kKind>
__device__ inline void write_record(float4* __restrict__ rec, uint32_t at, const float x[3], const float v[3], float qd,
                                    int s) {
    if constexpr (kKind == REC_RHO) {
        rec[at] = make_float4(x[0], x[1], x[2], qd);
    } else if constexpr (kKind == REC_DIRECT) {
        rec[2 * (int64_t)at] = make_float4(x[0], x[1], x[2], 0.0f);
        rec[2 * (int64_t)at + 1] = make_float4(qd * v[0], qd * v[1], qd * v[2], 0.0f);
    } else {
        rec[2 * (int64_t)at] = make_float4(x[0], x[1], x[2], __int_as_float(s));
        rec[2 * (int64_t)at + 1] = make_float4(v[0], v[1], v[2], 0.0f);
    }
}

// kPlaces: the record index of every slot is kept for bin_return_kernel.
template <int kItems, int kKind, bool kPlaces>
__global__ __launch_bounds__(kThreads) void bin_scatter_kernel(PicDesc d, BinGeom g, PicSpecies sp, SpeciesTable st,
                                                                PicParticles in, BinWork w, int64_t n,
                                                                const uint32_t* run) {
    extern __shared__ uint32_t lds[];
    if (run && !*run) return;
    uint32_t* place = lds;
    uint32_t* hist = lds + kThreads * kItems;
    const int64_t b0 = (int64_t)blockIdx.x * (kThreads * kItems);
    chunk_places<kItems>(d, g, in, b0, n, w.count, hist, place);
    for (int k = 0; k < kItems; ++k) {
        const int sl = k * kThreads + (int)threadIdx.x;
        const uint32_t at = place[sl];
        const int64_t i = b0 + sl;
        if constexpr (kPlaces) {
            if (i < n) w.place[i] = at;
        }
        if (at == kNoRecord) continue;
        const int s = species_of(i, sp.slots, sp.count);
        const float x[3] = {in.x[0][i], in.x[1][i], in.x[2][i]};
        float v[3] = {0.0f, 0.0f, 0.0f};
        if constexpr (kKind != REC_RHO) {
#pragma unroll
            for (int a = 0; a < 3; ++a) v[a] = in.u[a][i];
        }
        write_record<kKind>(w.rec, at, x, v, st.k[s].q_dv, s);
    }
}

// x += v dt and the particle boundaries (particle_tile_communication.py).
__device__ inline void move_and_store(const PicDesc& d, const SpeciesK& k, const float x[3], float v[3],
                                      const PicParticles& out, int64_t i) {
    bool act = true;
    double xn[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        xn[a] = ((k.ux >> a) & 1u) ? step_pos((double)x[a], (double)v[a], d.dt) : (double)x[a];
        apply_axis_boundary(d.pbc[a], d.wind[a], xn[a], v[a], act);
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        out.x[a][i] = act ? (float)xn[a] : 0.0f;
        out.u[a][i] = act ? v[a] : 0.0f;
    }
    out.active[i] = act ? 1 : 0;
}

// Gather + push + position update + boundaries in slot order, with the
// Esirkepov record (old position, pushed velocity) of every active particle.
template <int kItems, int kShape>
__global__ __launch_bounds__(kThreads) void bin_push_kernel(PicDesc d, BinGeom g, PicSpecies sp, SpeciesTable st,
                                                             PicParticles in, FieldPtrs fp, PicParticles out, BinWork w,
                                                             int64_t n, const uint32_t* skip) {
    extern __shared__ uint32_t lds[];
    if (skip && *skip) return;
    uint32_t* place = lds;
    uint32_t* hist = lds + kThreads * kItems;
    const int64_t b0 = (int64_t)blockIdx.x * (kThreads * kItems);
    chunk_places<kItems>(d, g, in, b0, n, w.count, hist, place);
#pragma unroll 1
    for (int k = 0; k < kItems; ++k) {
        const int sl = k * kThreads + (int)threadIdx.x;
        const int64_t i = b0 + sl;
        if (i >= n) break;
        const uint32_t at = place[sl];
        if (at == kNoRecord) {
#pragma unroll
            for (int a = 0; a < 3; ++a) out.x[a][i] = out.u[a][i] = 0.0f;
            out.active[i] = 0;
            continue;
        }
        const int s = species_of(i, sp.slots, sp.count);
        const float x[3] = {in.x[0][i], in.x[1][i], in.x[2][i]};
        float v[3] = {in.u[0][i], in.u[1][i], in.u[2][i]};
        float E[3], B[3];
        gather_points<kShape, uint32_t>(d, fp, x, E, B);
        float nv[3] = {v[0], v[1], v[2]};
        push_velocity(nv, E, B, st.k[s].h, d);
#pragma unroll
        for (int a = 0; a < 3; ++a)
            if ((st.k[s].uu >> a) & 1u) v[a] = nv[a];
        write_record<REC_ESIRKEPOV>(w.rec, at, x, v, 0.0f, s);
        move_and_store(d, st.k[s], x, v, out, i);
    }
}

// Record range and box origin of a work item.
struct Item {
    uint32_t begin, end;
    int o[3];
};

__device__ inline bool find_item(const PicDesc& d, const BinGeom& g, const BinWork& w, uint32_t b, Item& it) {
    if (b >= w.item[g.tiles]) return false;
    int lo = 0, hi = g.tiles;              // last tile whose first item is <= b and which has one
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (w.item[mid] <= b) lo = mid;
        else hi = mid;
    }
    it.begin = w.first[lo] + (b - w.item[lo]) * (uint32_t)kItem;
    it.end = min(it.begin + (uint32_t)kItem, w.first[lo + 1]);
    const int t[3] = {lo / (g.nt[1] * g.nt[2]), (lo / g.nt[2]) % g.nt[1], lo % g.nt[2]};
#pragma unroll
    for (int a = 0; a < 3; ++a) it.o[a] = t[a] * g.T[a] + d.g - g.margin;
    return true;
}

// Box index of the first stencil point and the weights of one axis and node
// line; false if a point lies outside the box.
template <int kShape>
__device__ inline bool line_points(float x, double org, double sp, int o, int e, int& first,
                                   float (&w)[PointAxis<kShape>::kN]) {
    const float isp32 = (float)(1.0 / sp);
    const int a = anchor_fast(x, (float)org, isp32, org, sp, kShape);
    const double dl = (double)x - node_coord(a, sp, org);
    if constexpr (kShape == 1) {
        const float r = (float)dl * isp32;
        first = a - o;
        w[0] = 1.0f - r;
        w[1] = r;
        return (unsigned)first < (unsigned)(e - 1);
    } else {
        double s[3];
        shape3(dl * (1.0 / sp), 2, s);
        first = a - 1 - o;
#pragma unroll
        for (int q = 0; q < 3; ++q) w[q] = (float)s[q];
        return (unsigned)first < (unsigned)(e - 2);
    }
}

template <int kN, CicRounding kR>
__device__ inline float box_value(const float* p, int plane, int row, const float (&wx)[kN], const float (&wy)[kN],
                                  const float (&wz)[kN]) {
    return stencil_sum<kN, kR>(wx, wy, wz, [&](int i, int j, float (&v)[kN]) {
#pragma unroll
        for (int k = 0; k < kN; ++k) v[k] = p[i * plane + j * row + k];
    });
}

// One block per work item: E + E_ext and B + B_ext of the tile's box in LDS
// (52 KB), gather, push, and the velocity written back into the record.  A slot
// in no cell order reads 24 stencil rows of the arrays, a line each (4.2M
// particles on 64^3: 665 us); through the box the fields are read once a tile.
template <int kShape>
__global__ __launch_bounds__(kWide) void bin_tile_push_kernel(PicDesc d, BinGeom g, SpeciesTable st, FieldPtrs fp,
                                                               BinWork w) {
    extern __shared__ float box[];
    if (!*w.random) return;
    Item it;
    if (!find_item(d, g, w, blockIdx.x, it)) return;
    const int plane = g.e[1] * g.e[2];
    for (int r = threadIdx.x; r < g.box; r += kWide) {
        const int i = pmod(it.o[0] + r / plane, d.dims[0]), j = pmod(it.o[1] + (r % plane) / g.e[2], d.dims[1]);
        const int64_t t = fidx(d, i, j, pmod(it.o[2] + r % g.e[2], d.dims[2]));
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const float* F = c < 3 ? fp.E[c] : fp.B[c - 3];
            const float* X = c < 3 ? fp.Ee[c] : fp.Be[c - 3];
            box[c * g.box + r] = X ? F[t] + X[t] : F[t];
        }
    }
    __syncthreads();
    constexpr int kN = PointAxis<kShape>::kN;
    for (uint32_t r = it.begin + threadIdx.x; r < it.end; r += kWide) {
        const float4 a = w.rec[2 * (int64_t)r], b = w.rec[2 * (int64_t)r + 1];
        const SpeciesK& k = st.k[__float_as_int(a.w)];
        const float x[3] = {a.x, a.y, a.z};
        float v[3] = {b.x, b.y, b.z}, E[3], B[3];
        int pc[3], pv[3];
        float wc[3][kN], wv[3][kN];
        bool in = true;
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            in = line_points<kShape>(x[m], d.org_c[m], d.sp_c[m], it.o[m], g.e[m], pc[m], wc[m]) && in;
            in = line_points<kShape>(x[m], d.org_v[m], d.sp_v[m], it.o[m], g.e[m], pv[m], wv[m]) && in;
        }
        if (in) {
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                // E[m] on the vertex line of its own axis, B[m] of the other two
                const auto pick = [&](int axis, bool vertex) { return vertex ? pv[axis] : pc[axis]; };
                const int e0 = pick(0, m == 0), e1 = pick(1, m == 1), e2 = pick(2, m == 2);
                const int b0 = pick(0, m != 0), b1 = pick(1, m != 1), b2 = pick(2, m != 2);
                const float* pe = box + m * g.box + (e0 * g.e[1] + e1) * g.e[2] + e2;
                E[m] = m == 1 ? box_value<kN, kSecond>(pe, plane, g.e[2], wc[0], wv[1], wc[2])
                              : box_value<kN, kPlain>(pe, plane, g.e[2], m == 0 ? wv[0] : wc[0], wc[1],
                                                      m == 2 ? wv[2] : wc[2]);
                B[m] = box_value<kN, kMagnetic>(box + (3 + m) * g.box + (b0 * g.e[1] + b1) * g.e[2] + b2, plane, g.e[2],
                                     m != 0 ? wv[0] : wc[0], m != 1 ? wv[1] : wc[1], m != 2 ? wv[2] : wc[2]);
            }
        } else {
            gather_points<kShape, uint32_t>(d, fp, x, E, B);
        }
        float nv[3] = {v[0], v[1], v[2]};
        push_velocity(nv, E, B, k.h, d);
#pragma unroll
        for (int m = 0; m < 3; ++m)
            if ((k.uu >> m) & 1u) v[m] = nv[m];
        w.rec[2 * (int64_t)r + 1] = make_float4(v[0], v[1], v[2], 0.0f);
    }
}

// Back to slot order: the pushed velocity from the slot's record, then the
// position update and boundaries (kMove) or the velocity alone.
template <bool kMove>
__global__ void bin_return_kernel(PicDesc d, PicSpecies sp, SpeciesTable st, PicParticles in, PicParticles out,
                                  BinWork w, int64_t n) {
    if (!*w.random) return;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t at = w.place[i];
    if constexpr (kMove) {
        if (at == kNoRecord) {
#pragma unroll
            for (int a = 0; a < 3; ++a) out.x[a][i] = out.u[a][i] = 0.0f;
            out.active[i] = 0;
            return;
        }
        const float4 r = w.rec[2 * (int64_t)at + 1];
        const float x[3] = {in.x[0][i], in.x[1][i], in.x[2][i]};
        float v[3] = {r.x, r.y, r.z};
        move_and_store(d, st.k[species_of(i, sp.slots, sp.count)], x, v, out, i);
    } else {
        float4 r;
        if (at != kNoRecord) r = w.rec[2 * (int64_t)at + 1];
        else r = make_float4(in.u[0][i], in.u[1][i], in.u[2][i], 0.0f);
        out.u[0][i] = r.x;
        out.u[1][i] = r.y;
        out.u[2][i] = r.z;
    }
}

// LDS box of a tile: kC components of e[0] x e[1] x e[2] nodes from array
// index o; nodes outside go straight to the arrays.
template <int kC>
struct TileBox {
    float* J[3];
    double* box;
    int o[3], e[3];
    int vol;
    __device__ inline void add(const PicDesc& d, int c, int i, int j, int k, float v) const {
        if (v == 0.0f) return;
        const int bi = i - o[0], bj = j - o[1], bk = k - o[2];
        if ((unsigned)bi < (unsigned)e[0] && (unsigned)bj < (unsigned)e[1] && (unsigned)bk < (unsigned)e[2])
            unsafeAtomicAdd(&box[c * vol + (bi * e[1] + bj) * e[2] + bk], (double)v);
        else
            deposit_at(J[c], d, i, j, k, v);
    }
};

// Node weights, and for J_from_rhov the face weights (rho.py:72-153,
// J_from_rhov.py:88-200), of the kPoints = 2 (CIC: a, a+1) or 3 (TSC: a-1 ..
// a+1) points of one axis; first is the first point's array index.
template <int kShape, bool kFace>
struct NodePoints {
    static constexpr int kN = kShape == 1 ? 2 : 3;
    int first;
    float wn[kN], wf[kN];
    __device__ inline void set(double pos, double org, double sp, double dd, float org32, float isp32) {
        const int a = anchor_fast((float)pos, org32, isp32, org, sp, kShape);
        double w[3];
        shape3((pos - node_coord(a, sp, org)) / dd, kShape, w);
        first = kShape == 1 ? a : a - 1;
#pragma unroll
        for (int q = 0; q < kN; ++q) wn[q] = (float)w[q + 3 - kN];
        if constexpr (kFace) {
            shape3(face_offset(pos, org, a, dd) / dd, kShape, w);
#pragma unroll
            for (int q = 0; q < kN; ++q) wf[q] = (float)w[q + 3 - kN];
        }
    }
};

template <int kC>
__device__ inline void flush_tile_box(const PicDesc& d, const TileBox<kC>& s) {
    const int plane = s.e[1] * s.e[2];
    for (int r = threadIdx.x; r < s.vol; r += kWide) {
        const int i = r / plane, j = (r - i * plane) / s.e[2], k = r % s.e[2];
#pragma unroll
        for (int c = 0; c < kC; ++c) {
            const float v = (float)s.box[c * s.vol + r];
            if (v != 0.0f) deposit_at(s.J[c], d, s.o[0] + i, s.o[1] + j, s.o[2] + k, v);
        }
    }
}

// rho (kC = 1) and J_from_rhov (kC = 3).  First order: the kC * 8 values of
// particles with one anchor in neighbouring lanes are summed before the LDS
// atomics; second order adds each value by itself.
template <int kC, int kShape>
__global__ __launch_bounds__(kWide) void bin_node_kernel(PicDesc d, BinGeom g, BinWork w, float* J0, float* J1,
                                                             float* J2) {
    extern __shared__ double node_box[];
    double* const box = node_box;
    Item it;
    if (!find_item(d, g, w, blockIdx.x, it)) return;
    for (int e = threadIdx.x; e < kC * g.box; e += kWide) box[e] = 0.0;
    __syncthreads();
    const TileBox<kC> sink{{J0, J1, J2}, box, {it.o[0], it.o[1], it.o[2]}, {g.e[0], g.e[1], g.e[2]}, g.box};
    for (uint32_t r0 = it.begin; r0 < it.end; r0 += kWide) {
        const uint32_t r = r0 + threadIdx.x;
        const bool live = r < it.end;
        float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f), b = a;
        if (live) {
            if constexpr (kC == 1) {
                a = w.rec[r];
                b.x = a.w;
            } else {
                a = w.rec[2 * (int64_t)r];
                b = w.rec[2 * (int64_t)r + 1];
            }
        }
        const float x[3] = {a.x, a.y, a.z}, q[3] = {b.x, b.y, b.z};
        NodePoints<kShape, kC == 3> ax[3];
#pragma unroll
        for (int m = 0; m < 3; ++m)
            ax[m].set((double)x[m], d.org_c[m], d.sp_c[m], d.d[m], g.org[m], g.isp[m]);
        if constexpr (kShape == 1) {
            float val[8 * kC];
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const int i = m >> 2, j = (m >> 1) & 1, k = m & 1;
                if constexpr (kC == 1) {
                    val[m] = q[0] * ax[0].wn[i] * ax[1].wn[j] * ax[2].wn[k];
                } else {
                    val[m] = q[0] * ax[0].wf[i] * ax[1].wn[j] * ax[2].wn[k];
                    val[8 + m] = q[1] * ax[0].wn[i] * ax[1].wf[j] * ax[2].wn[k];
                    val[16 + m] = q[2] * ax[0].wn[i] * ax[1].wn[j] * ax[2].wf[k];
                }
            }
            const int bi = ax[0].first - it.o[0], bj = ax[1].first - it.o[1], bk = ax[2].first - it.o[2];
            const bool in = (unsigned)bi < (unsigned)(g.e[0] - 1) && (unsigned)bj < (unsigned)(g.e[1] - 1) &&
                            (unsigned)bk < (unsigned)(g.e[2] - 1);
            const int at = (bi * g.e[1] + bj) * g.e[2] + bk;
            const int key = !live ? -1 : (in ? at : -2 - (int)(threadIdx.x & 63u));
            if (row_run_sums(key, val) && live) {
#pragma unroll
                for (int m = 0; m < 8 * kC; ++m) {
                    const int c = m >> 3, i = (m >> 2) & 1, j = (m >> 1) & 1, k = m & 1;
                    if (in) unsafeAtomicAdd(&box[c * g.box + at + (i * g.e[1] + j) * g.e[2] + k], (double)val[m]);
                    else deposit_at(sink.J[c], d, ax[0].first + i, ax[1].first + j, ax[2].first + k, val[m]);
                }
            }
        } else if (live) {
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const int ix = ax[0].first + i, iy = ax[1].first + j, iz = ax[2].first + k;
                        if constexpr (kC == 1) {
                            sink.add(d, 0, ix, iy, iz, q[0] * ax[0].wn[i] * ax[1].wn[j] * ax[2].wn[k]);
                        } else {
                            sink.add(d, 0, ix, iy, iz, q[0] * ax[0].wf[i] * ax[1].wn[j] * ax[2].wn[k]);
                            sink.add(d, 1, ix, iy, iz, q[1] * ax[0].wn[i] * ax[1].wf[j] * ax[2].wn[k]);
                            sink.add(d, 2, ix, iy, iz, q[2] * ax[0].wn[i] * ax[1].wn[j] * ax[2].wf[k]);
                        }
                    }
        }
    }
    __syncthreads();
    flush_tile_box(d, sink);
}

// Esirkepov deposit of the records (Esirkepov.py:105-331).  First order: a
// particle that stays in its cell adds the twelve values of the regular case
// (as fused_block does), summed over equal cells of neighbouring lanes; any
// other is queued (record index inside the item) and deposited when the queue
// could not hold another pass, or after the last: in the 3-slot frame, or in
// the 5-slot frame into the arrays when it moved a cell or more.  Second order:
// the 5-slot frame with its live slots only.  4.2M particles in random order on
// 64^3: 403 us with FP32 boxes, 132 us with FP64 ones.
template <int kShape>
__global__ __launch_bounds__(kWide) void bin_esirkepov_kernel(PicDesc d, BinGeom g, SpeciesTable st, BinWork w,
                                                                  float* Jx, float* Jy, float* Jz) {
    extern __shared__ double esir_box[];
    double* const box = esir_box;
    __shared__ uint16_t queue[kShape == 1 ? kQueue : 1];
    __shared__ int added[3];
    Item it;
    if (!find_item(d, g, w, blockIdx.x, it)) return;
    for (int e = threadIdx.x; e < 3 * g.box; e += kWide) box[e] = 0.0;
    if (threadIdx.x < 3) added[threadIdx.x] = 0;
    __syncthreads();
    const TileBox<3> sink{{Jx, Jy, Jz}, box, {it.o[0], it.o[1], it.o[2]}, {g.e[0], g.e[1], g.e[2]}, g.box};
    const float fdt = (float)d.dt;
    // Queued particles, the same number in every thread: those of the passes before
    // (held) and of this one, counted in added[pass].  After a pass's barrier every
    // wave reads that count and, held being equal, drains or goes on with the others.
    // A wave that goes on adds to the next count, and clears the one after it, which
    // was last read before the barrier it has just passed; the third was read by
    // waves that may not have read it yet, so two counts would not do.
    int held = 0, pass = 0;
    const auto drain = [&]() {
        for (int q = threadIdx.x; q < held; q += kWide) {
            const int64_t r = it.begin + queue[q];
            const float4 a = w.rec[2 * r], b = w.rec[2 * r + 1];
            const SpeciesK& k = st.k[__float_as_int(a.w)];
            const double xo[3] = {(double)a.x, (double)a.y, (double)a.z};
            const float v[3] = {b.x, b.y, b.z};
            double xn[3];
            CrossAxis ca[3];
            bool ok = true;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                xn[c] = ((k.ux >> c) & 1u) ? step_pos(xo[c], (double)v[c], d.dt) : xo[c];
                ok = cross_axis(xo[c], xn[c], d.org_c[c], d.sp_c[c], 1.0 / d.d[c], g.org[c], g.isp[c], ca[c]) && ok;
            }
            float* const J[3] = {Jx, Jy, Jz};
            if (ok) crossing_deposit(d, k.qw, ca[0], ca[1], ca[2], sink);
            else esirkepov_particle(d, k.qw, xo, xn, v, J);
        }
    };
    for (uint32_t r0 = it.begin; r0 < it.end; r0 += kWide) {
        const uint32_t r = r0 + threadIdx.x;
        const bool live = r < it.end;
        float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f), b = a;
        if (live) {
            a = w.rec[2 * (int64_t)r];
            b = w.rec[2 * (int64_t)r + 1];
        }
        const SpeciesK& k = st.k[__float_as_int(a.w)];
        const float x[3] = {a.x, a.y, a.z}, v[3] = {b.x, b.y, b.z};
        if constexpr (kShape == 1) {
            bool regular = live;
            int an[3];
            float A[3][2], D[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                const bool ux = (k.ux >> m) & 1u;
                an[m] = anchor_fast(x[m], g.org[m], g.isp[m], d.org_c[m], d.sp_c[m], 1);
                const float inv_d = (float)(1.0 / d.d[m]);
                const float r0m = (float)((double)x[m] - node_coord(an[m], d.sp_c[m], d.org_c[m])) * inv_d;
                const float dvt = ux ? v[m] * fdt : 0.0f;
                const double xn = ux ? step_pos((double)x[m], (double)v[m], d.dt) : (double)x[m];
                const int a1 = anchor_est((x[m] + dvt - g.org[m]) * g.isp[m],
                                          (fabsf(x[m]) + fabsf(dvt) + fabsf(g.org[m])) * g.isp[m], xn, d.org_c[m],
                                          d.sp_c[m], 1);
                regular = regular && a1 == an[m];
                D[m] = dvt * inv_d;
                A[m][1] = r0m + 0.5f * D[m];
                A[m][0] = 1.0f - r0m - 0.5f * D[m];
            }
            float val[12];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int o1 = c == 0 ? 1 : 0, o2 = c == 2 ? 1 : 2;
                const float pre = k.pre[c] * (-D[c]);
                const float e = D[o1] * D[o2] * (1.0f / 12.0f);
                val[c * 4 + 0] = pre * fmaf(A[o1][0], A[o2][0], e);
                val[c * 4 + 1] = pre * fmaf(A[o1][0], A[o2][1], -e);
                val[c * 4 + 2] = pre * fmaf(A[o1][1], A[o2][0], -e);
                val[c * 4 + 3] = pre * fmaf(A[o1][1], A[o2][1], e);
            }
            const int bi = an[0] - it.o[0], bj = an[1] - it.o[1], bk = an[2] - it.o[2];
            const bool in = (unsigned)bi < (unsigned)(g.e[0] - 1) && (unsigned)bj < (unsigned)(g.e[1] - 1) &&
                            (unsigned)bk < (unsigned)(g.e[2] - 1);
            const int at = (bi * g.e[1] + bj) * g.e[2] + bk;
            const int next = pass == 2 ? 0 : pass + 1;
            if (threadIdx.x == 0) added[next] = 0;
            if (live && !regular) queue[held + atomicAdd(&added[pass], 1)] = (uint16_t)(r - it.begin);
            const int key = !regular ? -1 - (int)(threadIdx.x & 63u) : (in ? at : -128 - (int)(threadIdx.x & 63u));
            if (row_run_sums(key, val) && regular) {
#pragma unroll
                for (int m = 0; m < 12; ++m) {
                    int dx, dy, dz;
                    RegularLayout<3>::delta(m, dx, dy, dz);
                    if (in) unsafeAtomicAdd(&box[(m >> 2) * g.box + at + (dx * g.e[1] + dy) * g.e[2] + dz], (double)val[m]);
                    else deposit_at(sink.J[m >> 2], d, an[0] + dx, an[1] + dy, an[2] + dz, val[m]);
                }
            }
            __syncthreads();
            held += added[pass];
            pass = next;
            const bool last = r0 + kWide >= it.end;
            if (last || held > kQueue - kWide) {    // room for a whole pass
                drain();
                __syncthreads();                    // before the next pass queues over what was read
                held = 0;
            }
        } else if (live) {
            double xo[3], xn[3];
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                xo[m] = (double)x[m];
                xn[m] = ((k.ux >> m) & 1u) ? step_pos(xo[m], (double)v[m], d.dt) : xo[m];
            }
            esirkepov_second_order(d, k, xo, xn, v, sink);
        }
    }
    __syncthreads();
    flush_tile_box(d, sink);
}

// Clear, sample, count and scan; the caller's scatter and deposit follow.  run
// (optional): a device flag without which the launches do nothing.
template <int kItems>
int bin_prepare(const PicDesc* desc, const BinGeom& g, const PicParticles* in, const BinWork& w, int64_t n,
                const uint32_t* run, hipStream_t s) {
    hipLaunchKernelGGL(bin_start_kernel, dim3(4), dim3(kSamples), 0, s, *desc, g, *in, w, n);
    hipLaunchKernelGGL(bin_count_kernel<kItems>, dim3((unsigned)grid_1d(n, kThreads * kItems)), dim3(kThreads),
                       (size_t)g.tiles * 4, s, *desc, g, *in, w.count, n, run);
    hipLaunchKernelGGL(bin_scan_kernel, dim3(1), dim3(1024), 0, s, w, g.tiles, run);
    PIC_CHECK_LAUNCH();
    return 0;
}

// Slots per chunk: large chunks make long runs per tile, small ones fill the
// chip when there are few particles.
inline bool small_set(int64_t n) { return n < (int64_t)1 << 21; }
constexpr int kSmall = 4, kLarge = 16;

template <int kItems, int kKind, bool kPlaces>
void launch_scatter(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const BinGeom& g,
                    const BinWork& w, int64_t n, const uint32_t* run, hipStream_t s) {
    hipLaunchKernelGGL((bin_scatter_kernel<kItems, kKind, kPlaces>), dim3((unsigned)grid_1d(n, kThreads * kItems)),
                       dim3(kThreads), (size_t)(g.tiles + kThreads * kItems) * 4, s, *desc, g, *sp,
                       species_table(*desc, *sp), *in, w, n, run);
}

template <int kKind>
int bin_scatter(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const BinGeom& g, const BinWork& w,
                int64_t n, hipStream_t s) {
    int rc;
    if (small_set(n)) {
        rc = bin_prepare<kSmall>(desc, g, in, w, n, nullptr, s);
        launch_scatter<kSmall, kKind, false>(desc, sp, in, g, w, n, nullptr, s);
    } else {
        rc = bin_prepare<kLarge>(desc, g, in, w, n, nullptr, s);
        launch_scatter<kLarge, kKind, false>(desc, sp, in, g, w, n, nullptr, s);
    }
    if (rc) return rc;
    PIC_CHECK_LAUNCH();
    return 0;
}

unsigned item_grid(const BinGeom& g, int64_t n) { return (unsigned)(g.tiles + n / kItem + 1); }

// Slots are numbered in 32 bits; larger sets keep the slot-ordered kernels.
constexpr int64_t kMaxSlots = ((int64_t)1 << 31) - 8 * kThreads;

// The six field components and the three current components of a box are held
// one after the other, never together.
bool binned_ok(const PicDesc* d, int kind, BinGeom& g) {
    return desc_ok(d) && d->n[0] > 1 && d->n[1] > 1 && d->n[2] > 1 && field_size(*d) < ((int64_t)1 << 30) &&
           bin_geom(*d, kind == REC_RHO ? 1 : 3, g);
}

// Below this the push runs in slot order: the launches of the push through
// tiles cost more than the lines they save.
constexpr int64_t kTilePushSlots = (int64_t)1 << 18;
constexpr int kMaxFieldBoxBytes = 64 * 1024;

bool tile_push_ok(const BinGeom& g, int64_t n) {
    return n >= kTilePushSlots && (int64_t)g.box * 6 * 4 <= kMaxFieldBoxBytes;
}

// Push through tiles (where the sampled slot order is random): scatter with
// places, gather + push per item.
template <int kItems, int kKind>
void launch_tile_push(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const FieldPtrs& fp,
                      const BinGeom& g, const BinWork& w, int64_t n, hipStream_t s) {
    launch_scatter<kItems, kKind, true>(desc, sp, in, g, w, n, w.random, s);
    const SpeciesTable st = species_table(*desc, *sp);
    const size_t lds = (size_t)g.box * 6 * 4;
    if (desc->shape_factor == 1)
        hipLaunchKernelGGL(bin_tile_push_kernel<1>, dim3(item_grid(g, n)), dim3(kWide), lds, s, *desc, g, st, fp, w);
    else
        hipLaunchKernelGGL(bin_tile_push_kernel<2>, dim3(item_grid(g, n)), dim3(kWide), lds, s, *desc, g, st, fp, w);
}

template <int kC>
int node_deposit(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, float* const J[3], void* ws,
                 int64_t ws_bytes, hipStream_t s) {
    constexpr int kKind = kC == 1 ? REC_RHO : REC_DIRECT;
    BinGeom g;
    PIC_REQUIRE(binned_ok(desc, kKind, g) && particles_ok(sp, in) && ws);
    PIC_REQUIRE(ws_bytes >= pic_binned_workspace_bytes(desc, sp, kKind));
    const int64_t n = (int64_t)sp->count * sp->slots;
    if (n == 0) return 0;
    PIC_REQUIRE(n < kMaxSlots);
    const BinWork w = bin_work(ws, g.tiles, kKind, n);
    const int rc = bin_scatter<kKind>(desc, sp, in, g, w, n, s);
    if (rc) return rc;
    const size_t lds = (size_t)g.box * kC * 8;
    if (desc->shape_factor == 1)
        hipLaunchKernelGGL((bin_node_kernel<kC, 1>), dim3(item_grid(g, n)), dim3(kWide), lds, s, *desc, g, w, J[0],
                           J[1], J[2]);
    else
        hipLaunchKernelGGL((bin_node_kernel<kC, 2>), dim3(item_grid(g, n)), dim3(kWide), lds, s, *desc, g, w, J[0],
                           J[1], J[2]);
    PIC_CHECK_LAUNCH();
    return 0;
}

int esirkepov_items(const PicDesc* desc, const PicSpecies* sp, const BinGeom& g, const BinWork& w, float* const J[3],
                    int64_t n, hipStream_t s) {
    const SpeciesTable st = species_table(*desc, *sp);
    const size_t lds = (size_t)g.box * 3 * 8;
    if (desc->shape_factor == 1)
        hipLaunchKernelGGL(bin_esirkepov_kernel<1>, dim3(item_grid(g, n)), dim3(kWide), lds, s, *desc, g, st, w, J[0],
                           J[1], J[2]);
    else
        hipLaunchKernelGGL(bin_esirkepov_kernel<2>, dim3(item_grid(g, n)), dim3(kWide), lds, s, *desc, g, st, w, J[0],
                           J[1], J[2]);
    PIC_CHECK_LAUNCH();
    return 0;
}

template <int kItems>
int fused_binned(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const FieldPtrs& fp,
                 const PicParticles* out, const BinGeom& g, const BinWork& w, int64_t n, hipStream_t s) {
    const int rc = bin_prepare<kItems>(desc, g, in, w, n, nullptr, s);
    if (rc) return rc;
    const SpeciesTable st = species_table(*desc, *sp);
    const bool tiles = tile_push_ok(g, n);
    const dim3 grid((unsigned)grid_1d(n, kThreads * kItems));
    const size_t lds = (size_t)(g.tiles + kThreads * kItems) * 4;
    const uint32_t* skip = tiles ? w.random : nullptr;
    if (desc->shape_factor == 1)
        hipLaunchKernelGGL((bin_push_kernel<kItems, 1>), grid, dim3(kThreads), lds, s, *desc, g, *sp, st, *in, fp,
                           *out, w, n, skip);
    else
        hipLaunchKernelGGL((bin_push_kernel<kItems, 2>), grid, dim3(kThreads), lds, s, *desc, g, *sp, st, *in, fp,
                           *out, w, n, skip);
    if (tiles) {
        launch_tile_push<kItems, REC_ESIRKEPOV>(desc, sp, in, fp, g, w, n, s);
        hipLaunchKernelGGL(bin_return_kernel<true>, dim3((unsigned)grid_1d(n, kThreads)), dim3(kThreads), 0, s, *desc,
                           *sp, st, *in, *out, w, n);
    }
    PIC_CHECK_LAUNCH();
    return 0;
}

}  // namespace

// The push in slot order, run where *skip is 0 (pic_particles.hip).
int pic_push_unless(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const float* const E[3],
                    const float* const B[3], const float* const E_ext[3], const float* const B_ext[3],
                    float* const u_out[3], const uint32_t* skip, void* stream);

extern "C" {

int64_t pic_binned_workspace_bytes(const PicDesc* desc, const PicSpecies* sp, int32_t kind) {
    BinGeom g;
    if (!desc || !sp || kind < 0 || kind > 3 || !binned_ok(desc, kind, g)) return -1;
    const int64_t n = (int64_t)sp->count * sp->slots;
    if (n >= kMaxSlots || (kind == REC_PUSH && !tile_push_ok(g, n))) return -1;
    return bin_tables(g.tiles) + bin_records(kind, n) + (kind >= REC_ESIRKEPOV && tile_push_ok(g, n) ? 4 * n : 0);
}

int pic_deposit_rho_binned(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, float* rho,
                           void* workspace, int64_t workspace_bytes, void* stream) {
    PIC_REQUIRE(rho);
    float* const J[3] = {rho, rho, rho};
    return node_deposit<1>(desc, sp, in, J, workspace, workspace_bytes, as_stream(stream));
}

int pic_deposit_direct_binned(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, float* const J[3],
                              void* workspace, int64_t workspace_bytes, void* stream) {
    PIC_REQUIRE(J && J[0] && J[1] && J[2]);
    return node_deposit<3>(desc, sp, in, J, workspace, workspace_bytes, as_stream(stream));
}

int pic_deposit_esirkepov_binned(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, float* const J[3],
                                 void* workspace, int64_t workspace_bytes, void* stream) {
    BinGeom g;
    PIC_REQUIRE(binned_ok(desc, REC_ESIRKEPOV, g) && particles_ok(sp, in) && J && J[0] && J[1] && J[2] && workspace);
    PIC_REQUIRE(workspace_bytes >= pic_binned_workspace_bytes(desc, sp, REC_ESIRKEPOV));
    const int64_t n = (int64_t)sp->count * sp->slots;
    if (n == 0) return 0;
    PIC_REQUIRE(n < kMaxSlots);
    hipStream_t s = as_stream(stream);
    const BinWork w = bin_work(workspace, g.tiles, REC_ESIRKEPOV, n);
    const int rc = bin_scatter<REC_ESIRKEPOV>(desc, sp, in, g, w, n, s);
    return rc ? rc : esirkepov_items(desc, sp, g, w, J, n, s);
}

int pic_push_binned(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in, const float* const E[3],
                    const float* const B[3], const float* const E_ext[3], const float* const B_ext[3],
                    float* const u_out[3], void* workspace, int64_t workspace_bytes, void* stream) {
    BinGeom g;
    PIC_REQUIRE(binned_ok(desc, REC_PUSH, g) && particles_ok(sp, in) && E && B && u_out && workspace);
    for (int a = 0; a < 3; ++a) PIC_REQUIRE(E[a] && B[a] && u_out[a]);
    const int64_t need = pic_binned_workspace_bytes(desc, sp, REC_PUSH), n = (int64_t)sp->count * sp->slots;
    PIC_REQUIRE(need > 0 && workspace_bytes >= need && n < kMaxSlots);
    hipStream_t s = as_stream(stream);
    const BinWork w = bin_work(workspace, g.tiles, REC_PUSH, n);
    const FieldPtrs fp = make_fields(E, B, E_ext, B_ext);
    int rc;
    if (small_set(n)) {
        rc = bin_prepare<kSmall>(desc, g, in, w, n, w.random, s);
        launch_tile_push<kSmall, REC_PUSH>(desc, sp, in, fp, g, w, n, s);
    } else {
        rc = bin_prepare<kLarge>(desc, g, in, w, n, w.random, s);
        launch_tile_push<kLarge, REC_PUSH>(desc, sp, in, fp, g, w, n, s);
    }
    if (rc) return rc;
    PicParticles out = *in;
    for (int a = 0; a < 3; ++a) out.u[a] = u_out[a];
    hipLaunchKernelGGL(bin_return_kernel<false>, dim3((unsigned)grid_1d(n, kThreads)), dim3(kThreads), 0, s, *desc,
                       *sp, species_table(*desc, *sp), *in, out, w, n);
    PIC_CHECK_LAUNCH();
    return pic_push_unless(desc, sp, in, E, B, E_ext, B_ext, u_out, w.random, stream);
}

int pic_fused_push_esirkepov_binned(const PicDesc* desc, const PicSpecies* sp, const PicParticles* in,
                                    const float* const E[3], const float* const B[3], const float* const E_ext[3],
                                    const float* const B_ext[3], PicParticles* out, float* const J[3], void* workspace,
                                    int64_t workspace_bytes, void* stream) {
    BinGeom g;
    PIC_REQUIRE(binned_ok(desc, REC_ESIRKEPOV, g) && particles_ok(sp, in) && particles_ok(sp, out));
    PIC_REQUIRE(E && B && J && workspace);
    const int64_t n = (int64_t)sp->count * sp->slots;
    for (int a = 0; a < 3; ++a)
        PIC_REQUIRE(E[a] && B[a] && J[a] && (n == 0 || (in->x[a] != out->x[a] && in->u[a] != out->u[a])));
    PIC_REQUIRE(n == 0 || in->active != out->active);
    PIC_REQUIRE(n < kMaxSlots);
    PIC_REQUIRE(workspace_bytes >= pic_binned_workspace_bytes(desc, sp, REC_ESIRKEPOV));
    if (n == 0) return 0;
    hipStream_t s = as_stream(stream);
    const BinWork w = bin_work(workspace, g.tiles, REC_ESIRKEPOV, n);
    const FieldPtrs fp = make_fields(E, B, E_ext, B_ext);
    const int rc = small_set(n) ? fused_binned<kSmall>(desc, sp, in, fp, out, g, w, n, s)
                                : fused_binned<kLarge>(desc, sp, in, fp, out, g, w, n, s);
    return rc ? rc : esirkepov_items(desc, sp, g, w, J, n, s);
}

}  // extern "C"
