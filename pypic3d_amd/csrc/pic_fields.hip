// Field kernels: fill, ghost refresh/fold, conducting walls, filters, Yee
// curl updates and the electrostatic centred gradient.
//
// The Yee kernels read neighbours through ghost_source(), i.e. they see the
// values a freshly refreshed copy of the input would hold
// (first_order_yee.py:31, :115 refresh before differencing), so the caller's
// input arrays are never modified -- the reference is functional.
#include "pic_field_ops.h"

#include <algorithm>

namespace {

using namespace pic;

constexpr int kBlock = 256;

template <class T>
__global__ void fill_kernel(T* __restrict__ p, int64_t n, T v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}

// Zeros in up to three components, two 16-byte stores per thread and pass.
template <class T>
__global__ void zero_fields_kernel(T* f0, T* f1, T* f2, int64_t n, int vec) {
    T* const f[3] = {f0, f1, f2};
    T* const p = f[blockIdx.y];
    if (!p) return;
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    constexpr int kPer = 16 / sizeof(T);
    const int64_t nv = vec ? n / kPer : 0;
    for (int64_t i = t0; i < nv; i += stride) reinterpret_cast<float4*>(p)[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int64_t i = nv * kPer + t0; i < n; i += stride) p[i] = (T)0;
}

struct Modes {
    int mode[3], sign[3];
};

// Ghost refresh of up to three fields in one launch (ghost_cells.py:142-215):
// a ghost cell takes the value of the interior cell its coordinates map to, or
// 0 across a non-periodic axis, so no axis waits for another.  Threads number
// the ghost cells: the x slabs, the y slabs of the rest, then the z ends of the
// interior lines.  With a row of 64 threads per (i, j) line, four of them at
// work in an interior one, a component of 4096 x 4096 x 1 took 2411 us
// (this: 245), of 512 x 512 x 59 40 us (12); a launch per axis took 596 and 31.
template <class T, class Idx>
__global__ void refresh_kernel(PicDesc d, Modes md, T* f0, T* f1, T* f2, Idx gx, Idx gxy, Idx ghosts) {
    T* const f[3] = {f0, f1, f2};
    const Idx g2 = 2 * d.g, d1 = d.dims[1], d2 = d.dims[2];
    const auto outside = [&](int l, int n) { return l < d.g ? l : n + l; };
    for (Idx t = (Idx)blockIdx.x * blockDim.x + threadIdx.x; t < ghosts; t += (Idx)gridDim.x * blockDim.x) {
        int i, j, k;
        if (t < gx) {
            const Idx r = t / d2;
            k = (int)(t - r * d2);
            j = (int)(r % d1);
            i = outside((int)(r / d1), d.n[0]);
        } else if (t < gxy) {
            const Idx u = t - gx, r = u / d2;
            k = (int)(u - r * d2);
            j = outside((int)(r % g2), d.n[1]);
            i = (int)(r / g2) + d.g;
        } else {
            const Idx u = t - gxy, r = u / g2, n1 = d.n[1];
            k = outside((int)(u - r * g2), d.n[2]);
            j = (int)(r % n1) + d.g;
            i = (int)(r / n1) + d.g;
        }
        const int si = ghost_source(i, d.n[0], d.g, md.mode[0]), sj = ghost_source(j, d.n[1], d.g, md.mode[1]);
        const int sk = ghost_source(k, d.n[2], d.g, md.mode[2]);
        const bool zero = si < 0 || sj < 0 || sk < 0;
        const int64_t dst = fidx(d, i, j, k), src = zero ? dst : fidx(d, si, sj, sk);
#pragma unroll
        for (int c = 0; c < 3; ++c)
            if (f[c]) f[c][dst] = zero ? (T)0 : f[c][src];
    }
}

// Fold and refresh of up to three fields in one launch: the thread of an
// interior cell with images adds them into it and writes the refreshed value
// back to all of them (each ghost cell belongs to one interior cell, so no
// other thread touches them).  Replaces 18 launches of a step (fold and refresh
// per axis and component).  Threads number the cells with images only: the x
// shell, then the y and the z shell of the rest; a thread's eight loads are
// independent.  (With a row of 64 threads per (i, j), four of them working in
// the z shell, the launch took 259 us at 256^3.)
template <class T>
__global__ void finish_kernel(PicDesc d, Modes md, T* f0, T* f1, T* f2, uint32_t mx, uint32_t my, uint32_t mz) {
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;     // mx + my + mz < 2^31 is checked at launch
    const uint32_t s1 = shell_count(d, 1), s2 = shell_count(d, 2);
    int i, j, k;
    if (t < mx) {
        const uint32_t r = t / d.n[2];
        k = (int)(t - r * d.n[2]) + d.g;
        j = (int)(r % d.n[1]) + d.g;
        i = shell_index(d, 0, (int)(r / d.n[1]));
    } else if (t < mx + my) {
        t -= mx;
        const uint32_t r = t / d.n[2];
        k = (int)(t - r * d.n[2]) + d.g;
        j = shell_index(d, 1, (int)(r % s1));
        i = (int)(r / s1) + 2 * d.g;
    } else {
        t -= mx + my;
        if (t >= mz) return;
        const uint32_t n1 = d.n[1] - s1, r = t / s2;
        k = shell_index(d, 2, (int)(t - r * s2));
        j = (int)(r % n1) + 2 * d.g;
        i = (int)(r / n1) + 2 * d.g;
    }
    T* const f = blockIdx.y == 0 ? f0 : (blockIdx.y == 1 ? f1 : f2);
    if (f) finish_point(d, md.mode, md.sign, f, i, j, k);
}

// Tangential E on the conducting walls set to zero, with its ghost images
// (first_order_yee.py:80-92 and the refresh after it); a row of threads per line along z.
constexpr int kRowThreads = 64, kRows = 4;

// Row of a thread of a row_grid launch; its index fits 32 bits where it is below rows.
__device__ inline bool grid_row(int64_t rows, int& row) {
    const int64_t r = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * kRows + threadIdx.y;
    row = (int)r;
    return r < rows;
}

template <class T>
__global__ void walls_kernel(PicDesc d, Modes md, T* f0, T* f1, T* f2) {
    int row;
    if (!grid_row((int64_t)d.n[0] * d.n[1], row)) return;
    const int i = row / d.n[1] + d.g, j = row % d.n[1] + d.g;
    const bool all = (d.bc[0] == 1 && (i == d.g || i == d.n[0] + d.g - 1)) ||
                     (d.bc[1] == 1 && (j == d.g || j == d.n[1] + d.g - 1));
    const int m = all ? d.n[2] : 2;               // other rows: the z walls only
    T* const f[3] = {f0, f1, f2};
    const T none[1] = {(T)0};
    for (int q = threadIdx.x; q < m; q += kRowThreads) {
        const int k = all || q == 0 ? d.g + q : d.n[2] + d.g - 1;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            T* const out[1] = {f[c]};
            if (on_wall(d, c, i, j, k)) store_refreshed<1>(d, md.mode, out, i, j, k, none);
        }
    }
}

// ghost_cells.py:218-289: one axis of the fold (non-reduced axis).
template <class T>
__global__ void fold_axis_kernel(PicDesc d, T* f, int axis, int bc) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= fold_elems(d, axis)) return;
    fold_elem(d, f, axis, bc, t);
}

// ghost_cells.py:218-235: fold of a reduced (single-cell) axis.
template <class T>
__global__ void fold_reduced_kernel(PicDesc d, T* f, int axis, int bc) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= fold_elems(d, axis)) return;
    fold_reduced_elem(d, f, axis, bc, t);
}

// Zero the wall planes g and n+g-1 of one axis (ghost_cells.py:344-362).
template <class T>
__global__ void zero_planes_kernel(PicDesc d, T* f, int axis) {
    int da, db;
    other_dims(d, axis, da, db);
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)2 * da * db) return;
    int which = (int)(t / ((int64_t)da * db));
    int64_t r = t - (int64_t)which * da * db;
    int b = (int)(r % db);
    int a = (int)(r / db);
    int pos = which == 0 ? d.g : d.n[axis] + d.g - 1;
    f[slab_to_index(d, axis, pos, a, b)] = (T)0;
}

// Fill the ghosts of one axis from the adjacent interior plane
// (ghost_cells.py:365-386).
template <class T>
__global__ void constant_ghosts_kernel(PicDesc d, T* f, int axis) {
    int g = d.g, n = d.n[axis];
    int da, db;
    other_dims(d, axis, da, db);
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)2 * g * da * db) return;
    int b = (int)(t % db);
    int64_t r = t / db;
    int a = (int)(r % da);
    int l = (int)(r / da);
    int dst = l < g ? l : n + l;
    int src = l < g ? g : n + g - 1;
    f[slab_to_index(d, axis, dst, a, b)] = f[slab_to_index(d, axis, src, a, b)];
}

// filters.py:234-291 at interior point t: the 3x3x3 correlation of f.
template <bool kBilinear, class T>
__device__ inline T filter_at(const PicDesc& d, const T* __restrict__ in, int64_t t, T alpha) {
    const int64_t sx = (int64_t)d.dims[1] * d.dims[2], sy = d.dims[2];
    if constexpr (kBilinear) {
        const T w1[3] = {(T)1, (T)2, (T)1};
        T acc = (T)0;
        for (int a = -1; a <= 1; ++a)
            for (int b = -1; b <= 1; ++b)
                for (int c = -1; c <= 1; ++c)
                    acc += (w1[a + 1] * w1[b + 1] * w1[c + 1] / (T)64) * in[t + a * sx + b * sy + c];
        return acc;
    } else {
        T nw = ((T)1 - alpha) / (T)6;
        T faces = in[t - sx] + in[t + sx] + in[t - sy] + in[t + sy] + in[t - 1] + in[t + 1];
        return alpha * in[t] + nw * faces;
    }
}

// interior <- filter; ghosts copied.
template <bool kBilinear, class T>
__global__ void filter_kernel(PicDesc d, const T* __restrict__ in, T* __restrict__ out, T alpha) {
    int64_t total = field_size(d);
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    int k = (int)(t % d.dims[2]);
    int64_t r = t / d.dims[2];
    int j = (int)(r % d.dims[1]);
    int i = (int)(r / d.dims[1]);
    int g = d.g;
    bool inside = i >= g && i < d.n[0] + g && j >= g && j < d.n[1] + g && k >= g && k < d.n[2] + g;
    out[t] = inside ? filter_at<kBilinear>(d, in, t, alpha) : in[t];
}

// Interior array point of a thread of an interior_grid launch: one grid row per
// (i, j) line along z, or, where the z lines are shorter than a wave (2-D and
// 1-D runs have one cell there), threads numbered over all points.
__device__ inline bool interior_point(const PicDesc& d, int flat, int& i, int& j, int& k) {
    if (flat) {
        const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, r = t / (uint32_t)d.n[2];
        k = (int)(t - r * (uint32_t)d.n[2]) + d.g;
        j = (int)(r % (uint32_t)d.n[1]) + d.g;
        i = (int)(r / (uint32_t)d.n[1]) + d.g;
        return i < d.n[0] + d.g;
    }
    k = (int)(blockIdx.x * blockDim.x + threadIdx.x) + d.g;
    j = blockIdx.y + d.g;
    i = blockIdx.z + d.g;
    return k < d.n[2] + d.g;
}

template <class T>
struct F3T {
    const T* p[3];
};
template <class T>
struct W3T {
    T* p[3];
};
using F3 = F3T<float>;
using W3f = W3T<float>;
struct W6f {
    float* p[6];
};

// Filter of up to three components into other arrays with their guard cells
// refreshed, and the conducting walls of E where asked for: one launch for the
// filter, refresh, wall and copy-back launches of every component.
template <bool kBilinear, class T>
__global__ void filter_refresh_kernel(PicDesc d, Modes md, F3T<T> in, W3T<T> out, T alpha, int walls, int flat) {
    int i, j, k;
    if (!interior_point(d, flat, i, j, k)) return;
    const int64_t t = fidx(d, i, j, k);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        if (!in.p[c]) continue;
        const T v[1] = {walls && on_wall(d, c, i, j, k) ? (T)0 : filter_at<kBilinear>(d, in.p[c], t, alpha)};
        T* const o[1] = {out.p[c]};
        store_refreshed<1>(d, md.mode, o, i, j, k, v);
    }
}

// The Yee updates store each point with its ghost images (store_refreshed), so
// no refresh launch follows them: bound by memory, 36 and 48 bytes per cell.
// first_order_yee.py:96-142: B_out = B_in - (dt/2) curl E (forward diffs).
template <class T>
__global__ void yee_b_kernel(PicDesc d, YeeConstT<T> y, F3T<T> E, F3T<T> B, W3T<T> out, int flat) {
    int i, j, k;
    if (interior_point(d, flat, i, j, k)) yee_b_point(d, y, E.p, B.p, out.p, i, j, k);
}

// first_order_yee.py:12-72: E_out = E_in + dt (C^2 curl B - J/eps) (backward diffs).
template <class T>
__global__ void yee_e_kernel(PicDesc d, YeeConstT<T> y, F3T<T> E, F3T<T> B, F3T<T> J, W3T<T> out, int flat) {
    int i, j, k;
    if (interior_point(d, flat, i, j, k)) yee_e_point(d, y, E.p, B.p, J.p, out.p, i, j, k);
}

__global__ void yee_b_pml_kernel(PicDesc d, YeeConst y, PmlArgs pml, F3 E, F3 B, W3f out, int flat) {
    int i, j, k;
    if (interior_point(d, flat, i, j, k)) yee_b_point_pml(d, y, pml, E.p, B.p, out.p, i, j, k);
}

__global__ void yee_e_pml_kernel(PicDesc d, YeeConst y, PmlArgs pml, F3 E, F3 B, F3 J, W3f out, int flat) {
    int i, j, k;
    if (interior_point(d, flat, i, j, k)) yee_e_point_pml(d, y, pml, E.p, B.p, J.p, out.p, i, j, k);
}

// stretch_spatial_derivative over six interior derivative arrays in place
// (apply_tiled_pml_to_e_curl / _b_curl without the curl assembly).
__global__ void pml_stretch_kernel(PicDesc d, PmlArgs pml, W6f dv, int flat) {
    int i, j, k;
    if (!interior_point(d, flat, i, j, k)) return;
    const int64_t mi = ((int64_t)(i - d.g) * d.n[1] + (j - d.g)) * d.n[2] + (k - d.g);
    float v[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) v[q] = dv.p[q][mi];
    pml_stretch6(d, pml, i, j, k, v);
#pragma unroll
    for (int q = 0; q < 6; ++q) dv.p[q][mi] = v[q];
}

// electrostatic_yee.py:212-246: E interior = -(phi[+1]-phi[-1])/(2d), reading
// phi's own (already boundary-applied) ghosts.
__global__ void efield_from_phi_kernel(PicDesc d, Modes md, const float* __restrict__ phi, float* __restrict__ ex,
                                       float* __restrict__ ey, float* __restrict__ ez, float h2x, float h2y,
                                       float h2z, int flat) {
    int i, j, k;
    if (!interior_point(d, flat, i, j, k)) return;
    int64_t c = fidx(d, i, j, k);
    const int64_t sx = (int64_t)d.dims[1] * d.dims[2], sy = d.dims[2];
    const float v[3] = {-1.0f * (phi[c + sx] - phi[c - sx]) * h2x, -1.0f * (phi[c + sy] - phi[c - sy]) * h2y,
                        -1.0f * (phi[c + 1] - phi[c - 1]) * h2z};
    float* const out[3] = {ex, ey, ez};
    store_refreshed<3>(d, md.mode, out, i, j, k, v);
}

bool desc_ok(const PicDesc* d) {
    if (!d) return false;
    if (d->g < 1) return false;
    for (int a = 0; a < 3; ++a) {
        if (d->n[a] < 1 || d->dims[a] != d->n[a] + 2 * d->g) return false;
        // a non-reduced axis narrower than the guard band would alias slabs
        if (d->n[a] > 1 && d->n[a] < d->g) return false;
    }
    return true;
}

// flags[0], flags[1]: whether any value of f[0..2], of f[3..5] is not zero (NaN is not).  flags are cleared before.
template <class T>
struct Six {
    const T* f[6];
};

template <class T>
__global__ void any_nonzero_kernel(Six<T> p, int64_t n, int32_t* flags) {
    bool any[2] = {false, false};
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
#pragma unroll
        for (int c = 0; c < 6; ++c) any[c / 3] = any[c / 3] | (p.f[c][i] != (T)0);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (__any(any[q]) && (threadIdx.x & 63) == 0) flags[q] = 1;
}

__global__ void clear_flags_kernel(int32_t* flags) { flags[threadIdx.x] = 0; }

template <class T>
int any_nonzero_t(const PicDesc* desc, const T* const a[3], const T* const b[3], int32_t* flags, hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && a && b && flags);
    Six<T> p;
    for (int c = 0; c < 3; ++c) {
        PIC_REQUIRE(a[c] && b[c]);
        p.f[c] = a[c];
        p.f[3 + c] = b[c];
    }
    const int64_t n = field_size(*desc);
    hipLaunchKernelGGL(clear_flags_kernel, dim3(1), dim3(2), 0, s, flags);
    const int64_t blocks = std::min<int64_t>((n + 1023) / 1024, 2048);
    hipLaunchKernelGGL(any_nonzero_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, s, p, n, flags);
    PIC_CHECK_LAUNCH();
    return 0;
}

}  // namespace

// Host-side launch sequences, for the FP32 (float) and FP64 (double) fields.
static Modes modes(const PicDesc* d, int bc_type) {
    Modes m;
    for (int a = 0; a < 3; ++a) {
        m.mode[a] = refresh_mode(*d, a, bc_type);
        m.sign[a] = fold_sign(*d, a, bc_type);
    }
    return m;
}

// Blocks of kRows rows, in two grid axes: one alone would pass 2^32 threads from 2^28 rows on (a 2-D run of
// 16384^2 cells).
static dim3 row_grid(int64_t rows) {
    const int64_t blocks = (rows + kRows - 1) / kRows, x = std::min<int64_t>(blocks, 1 << 20);
    return dim3((unsigned)x, (unsigned)((blocks + x - 1) / x));
}

template <class T>
static int refresh_t(const PicDesc* d, T* f0, T* f1, T* f2, int bc_type, hipStream_t s) {
    const int64_t g2 = 2 * d->g, gx = g2 * d->dims[1] * d->dims[2], gxy = gx + d->n[0] * g2 * d->dims[2];
    const int64_t ghosts = gxy + (int64_t)d->n[0] * d->n[1] * g2;
    const dim3 grid((unsigned)std::min<int64_t>((ghosts + kBlock - 1) / kBlock, 1 << 20));
    // 32-bit numbers where the last step past the end stays below 2^32
    if (ghosts < ((int64_t)1 << 31))
        hipLaunchKernelGGL((refresh_kernel<T, uint32_t>), grid, dim3(kBlock), 0, s, *d, modes(d, bc_type), f0, f1, f2,
                           (uint32_t)gx, (uint32_t)gxy, (uint32_t)ghosts);
    else
        hipLaunchKernelGGL((refresh_kernel<T, uint64_t>), grid, dim3(kBlock), 0, s, *d, modes(d, bc_type), f0, f1, f2,
                           (uint64_t)gx, (uint64_t)gxy, (uint64_t)ghosts);
    PIC_CHECK_LAUNCH();
    return 0;
}

template <class T>
static int zero_fields_t(const PicDesc* desc, T* const f[3], hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && f);
    const int64_t n = field_size(*desc);
    const int vec = ((((uintptr_t)f[0]) | ((uintptr_t)f[1]) | ((uintptr_t)f[2])) & 15u) == 0;
    const int64_t blocks = grid_1d(n / 8 + 1, kBlock);
    hipLaunchKernelGGL(zero_fields_kernel<T>, dim3((unsigned)(blocks > 4096 ? 4096 : blocks), 3), dim3(kBlock), 0, s,
                       f[0], f[1], f[2], n, vec);
    PIC_CHECK_LAUNCH();
    return 0;
}

template <class T>
static int finish_t(const PicDesc* desc, T* const f[3], int bc_type, hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && f && (bc_type == 0 || bc_type == 1));
    const int64_t s0 = shell_count(*desc, 0), s1 = shell_count(*desc, 1), s2 = shell_count(*desc, 2);
    const int64_t n0 = desc->n[0], n1 = desc->n[1], n2 = desc->n[2];
    const int64_t mx = s0 * n1 * n2, my = (n0 - s0) * s1 * n2, mz = (n0 - s0) * (n1 - s1) * s2;
    PIC_REQUIRE(mx + my + mz < ((int64_t)1 << 31));
    hipLaunchKernelGGL(finish_kernel<T>, dim3((unsigned)grid_1d(mx + my + mz, kBlock), 3), dim3(kBlock), 0, s, *desc,
                       modes(desc, bc_type), f[0], f[1], f[2], (uint32_t)mx, (uint32_t)my, (uint32_t)mz);
    PIC_CHECK_LAUNCH();
    return 0;
}

template <class T>
static int walls_t(const PicDesc* desc, T* const E[3], hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && E && E[0] && E[1] && E[2]);
    if (desc->bc[0] != 1 && desc->bc[1] != 1 && desc->bc[2] != 1) return 0;
    PIC_REQUIRE((int64_t)desc->n[0] * desc->n[1] < ((int64_t)1 << 31));
    hipLaunchKernelGGL(walls_kernel<T>, row_grid((int64_t)desc->n[0] * desc->n[1]), dim3(kRowThreads, kRows), 0, s,
                       *desc, modes(desc, 0), E[0], E[1], E[2]);
    PIC_CHECK_LAUNCH();
    return 0;
}

// Shared with other translation units.
int pic_refresh_fields(const PicDesc* d, float* f0, float* f1, float* f2, int bc_type, hipStream_t s) {
    return refresh_t<float>(d, f0, f1, f2, bc_type, s);
}

// Lines shorter than a wave would leave most of its lanes idle (64 x 64 x 1: one
// of 64, 7.2 us per update against 4 us numbered over all points); at 64 cells
// and more a line per grid row needs no division per thread.
static int interior_flat(const PicDesc* d) {
    return d->n[2] < 64 && (int64_t)d->n[0] * d->n[1] * d->n[2] < ((int64_t)1 << 31) ? 1 : 0;
}

static dim3 interior_grid(const PicDesc* d, int block) {
    if (interior_flat(d)) return dim3((unsigned)grid_1d((int64_t)d->n[0] * d->n[1] * d->n[2], block));
    return dim3((unsigned)((d->n[2] + block - 1) / block), (unsigned)d->n[1], (unsigned)d->n[0]);
}

static int interior_block(const PicDesc* d) { return d->n[2] >= 128 ? 128 : 64; }

template <class T>
static int fill_t(T* ptr, int64_t n, T value, hipStream_t s) {
    PIC_REQUIRE(ptr != nullptr && n >= 0);
    if (n == 0) return 0;
    int blocks = grid_1d(n, kBlock);
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(fill_kernel<T>, dim3(blocks), dim3(kBlock), 0, s, ptr, n, value);
    PIC_CHECK_LAUNCH();
    return 0;
}

template <class T>
static int halo_refresh_t(const PicDesc* desc, T* field, int bc_type, hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && field && (bc_type == 0 || bc_type == 1));
    return refresh_t<T>(desc, field, nullptr, nullptr, bc_type, s);
}

template <class T>
static int halo_fold_t(const PicDesc* desc, T* field, int bc_type, hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && field && (bc_type == 0 || bc_type == 1));
    for (int axis = 0; axis < 3; ++axis) {
        int bc = bc_type == 0 ? desc->bc[axis] : desc->pbc[axis];
        int da = desc->dims[axis == 0 ? 1 : 0], db = desc->dims[axis == 2 ? 1 : 2];
        if (desc->n[axis] == 1) {
            hipLaunchKernelGGL(fold_reduced_kernel<T>, dim3(grid_1d((int64_t)da * db, kBlock)), dim3(kBlock), 0, s,
                               *desc, field, axis, bc);
        } else {
            hipLaunchKernelGGL(fold_axis_kernel<T>, dim3(grid_1d((int64_t)desc->g * da * db, kBlock)), dim3(kBlock),
                               0, s, *desc, field, axis, bc);
        }
        PIC_CHECK_LAUNCH();
    }
    return 0;
}

template <class T>
static int zero_boundary_t(const PicDesc* desc, T* field, int axis, hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && field && axis >= 0 && axis < 3);
    if (desc->bc[axis] == 1) {
        int da = desc->dims[axis == 0 ? 1 : 0], db = desc->dims[axis == 2 ? 1 : 2];
        hipLaunchKernelGGL(zero_planes_kernel<T>, dim3(grid_1d((int64_t)2 * da * db, kBlock)), dim3(kBlock), 0, s,
                           *desc, field, axis);
        PIC_CHECK_LAUNCH();
    }
    return refresh_t<T>(desc, field, nullptr, nullptr, 0, s);
}

template <class T>
static int constant_boundary_t(const PicDesc* desc, T* field, int axis, hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && field && axis >= 0 && axis < 3);
    int rc = refresh_t<T>(desc, field, nullptr, nullptr, 0, s);
    if (rc) return rc;
    if (desc->bc[axis] == 1) {
        int da = desc->dims[axis == 0 ? 1 : 0], db = desc->dims[axis == 2 ? 1 : 2];
        hipLaunchKernelGGL(constant_ghosts_kernel<T>, dim3(grid_1d((int64_t)2 * desc->g * da * db, kBlock)),
                           dim3(kBlock), 0, s, *desc, field, axis);
        PIC_CHECK_LAUNCH();
    }
    return 0;
}

template <bool kBilinear, class T>
static int filter_t(const PicDesc* desc, const T* in, T* out, double alpha, hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && in && out && in != out);
    int64_t n = field_size(*desc);
    hipLaunchKernelGGL((filter_kernel<kBilinear, T>), dim3(grid_1d(n, kBlock)), dim3(kBlock), 0, s, *desc, in, out,
                       (T)alpha);
    PIC_CHECK_LAUNCH();
    return 0;
}

template <class T>
static int filter_refresh_t(const PicDesc* desc, const T* const in[3], T* const out[3], int bilinear, double alpha,
                            int bc_type, int walls, hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && in && out && (bc_type == 0 || bc_type == 1));
    for (int c = 0; c < 3; ++c) {
        PIC_REQUIRE((in[c] != nullptr) == (out[c] != nullptr));
        for (int e = 0; e < 3; ++e) PIC_REQUIRE(!in[c] || (const T*)out[e] != in[c]);
    }
    const int block = interior_block(desc);
    const F3T<T> from{{in[0], in[1], in[2]}};
    const W3T<T> to{{out[0], out[1], out[2]}};
    if (bilinear)
        hipLaunchKernelGGL((filter_refresh_kernel<true, T>), interior_grid(desc, block), dim3(block), 0, s, *desc,
                           modes(desc, bc_type), from, to, (T)alpha, walls, interior_flat(desc));
    else
        hipLaunchKernelGGL((filter_refresh_kernel<false, T>), interior_grid(desc, block), dim3(block), 0, s, *desc,
                           modes(desc, bc_type), from, to, (T)alpha, walls, interior_flat(desc));
    PIC_CHECK_LAUNCH();
    return 0;
}

template <class T>
static int yee_b_t(const PicDesc* desc, const T* const E[3], const T* const B_in[3], T* const B_out[3],
                   hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && E && B_in && B_out);
    for (int c = 0; c < 3; ++c) PIC_REQUIRE(E[c] && B_in[c] && B_out[c]);
    for (int c = 0; c < 3; ++c)
        for (int e = 0; e < 3; ++e) PIC_REQUIRE((const T*)B_out[c] != E[e]);
    int block = interior_block(desc);
    hipLaunchKernelGGL(yee_b_kernel<T>, interior_grid(desc, block), dim3(block), 0, s, *desc, yee_const<T>(*desc),
                       F3T<T>{{E[0], E[1], E[2]}}, F3T<T>{{B_in[0], B_in[1], B_in[2]}},
                       W3T<T>{{B_out[0], B_out[1], B_out[2]}}, interior_flat(desc));
    PIC_CHECK_LAUNCH();
    return 0;
}

template <class T>
static int yee_e_t(const PicDesc* desc, const T* const E_in[3], const T* const B[3], const T* const J[3],
                   T* const E_out[3], hipStream_t s) {
    PIC_REQUIRE(desc_ok(desc) && E_in && B && J && E_out);
    for (int c = 0; c < 3; ++c) PIC_REQUIRE(E_in[c] && B[c] && J[c] && E_out[c]);
    for (int c = 0; c < 3; ++c)
        for (int e = 0; e < 3; ++e) PIC_REQUIRE((const T*)E_out[c] != B[e] && (const T*)E_out[c] != J[e]);
    int block = interior_block(desc);
    hipLaunchKernelGGL(yee_e_kernel<T>, interior_grid(desc, block), dim3(block), 0, s, *desc, yee_const<T>(*desc),
                       F3T<T>{{E_in[0], E_in[1], E_in[2]}}, F3T<T>{{B[0], B[1], B[2]}}, F3T<T>{{J[0], J[1], J[2]}},
                       W3T<T>{{E_out[0], E_out[1], E_out[2]}}, interior_flat(desc));
    PIC_CHECK_LAUNCH();
    return 0;
}

extern "C" {

int pic_abi_version(void) { return PIC_ABI_VERSION; }

int pic_fill_f32(float* ptr, int64_t n, float value, void* stream) { return fill_t(ptr, n, value, as_stream(stream)); }

int pic_halo_refresh(const PicDesc* desc, float* field, int bc_type, void* stream) {
    return halo_refresh_t(desc, field, bc_type, as_stream(stream));
}

int pic_halo_refresh_f64(const PicDesc* desc, double* field, int bc_type, void* stream) {
    return halo_refresh_t(desc, field, bc_type, as_stream(stream));
}

int pic_halo_fold(const PicDesc* desc, float* field, int bc_type, void* stream) {
    return halo_fold_t(desc, field, bc_type, as_stream(stream));
}

int pic_halo_fold_f64(const PicDesc* desc, double* field, int bc_type, void* stream) {
    return halo_fold_t(desc, field, bc_type, as_stream(stream));
}

int pic_zero_boundary(const PicDesc* desc, float* field, int axis, void* stream) {
    return zero_boundary_t(desc, field, axis, as_stream(stream));
}

int pic_zero_boundary_f64(const PicDesc* desc, double* field, int axis, void* stream) {
    return zero_boundary_t(desc, field, axis, as_stream(stream));
}

int pic_constant_boundary(const PicDesc* desc, float* field, int axis, void* stream) {
    return constant_boundary_t(desc, field, axis, as_stream(stream));
}

int pic_constant_boundary_f64(const PicDesc* desc, double* field, int axis, void* stream) {
    return constant_boundary_t(desc, field, axis, as_stream(stream));
}

int pic_filter_digital(const PicDesc* desc, const float* in, float* out, double alpha, void* stream) {
    return filter_t<false>(desc, in, out, alpha, as_stream(stream));
}

int pic_filter_digital_f64(const PicDesc* desc, const double* in, double* out, double alpha, void* stream) {
    return filter_t<false>(desc, in, out, alpha, as_stream(stream));
}

int pic_filter_bilinear(const PicDesc* desc, const float* in, float* out, void* stream) {
    return filter_t<true>(desc, in, out, 1.0, as_stream(stream));
}

int pic_filter_bilinear_f64(const PicDesc* desc, const double* in, double* out, void* stream) {
    return filter_t<true>(desc, in, out, 1.0, as_stream(stream));
}

int pic_zero_fields(const PicDesc* desc, float* const f[3], void* stream) {
    return zero_fields_t(desc, f, as_stream(stream));
}

int pic_zero_fields_f64(const PicDesc* desc, double* const f[3], void* stream) {
    return zero_fields_t(desc, f, as_stream(stream));
}

int pic_any_nonzero(const PicDesc* desc, const float* const a[3], const float* const b[3], int32_t* flags,
                    void* stream) {
    return any_nonzero_t(desc, a, b, flags, as_stream(stream));
}

int pic_any_nonzero_f64(const PicDesc* desc, const double* const a[3], const double* const b[3], int32_t* flags,
                        void* stream) {
    return any_nonzero_t(desc, a, b, flags, as_stream(stream));
}

int pic_finish_current(const PicDesc* desc, float* const f[3], int bc_type, void* stream) {
    return finish_t(desc, f, bc_type, as_stream(stream));
}

int pic_finish_current_f64(const PicDesc* desc, double* const f[3], int bc_type, void* stream) {
    return finish_t(desc, f, bc_type, as_stream(stream));
}

int pic_filter_refresh(const PicDesc* desc, const float* const in[3], float* const out[3], int bilinear, double alpha,
                       int bc_type, int walls, void* stream) {
    return filter_refresh_t(desc, in, out, bilinear, alpha, bc_type, walls, as_stream(stream));
}

int pic_filter_refresh_f64(const PicDesc* desc, const double* const in[3], double* const out[3], int bilinear,
                           double alpha, int bc_type, int walls, void* stream) {
    return filter_refresh_t(desc, in, out, bilinear, alpha, bc_type, walls, as_stream(stream));
}

int pic_conducting_walls(const PicDesc* desc, float* const E[3], void* stream) {
    return walls_t(desc, E, as_stream(stream));
}

int pic_conducting_walls_f64(const PicDesc* desc, double* const E[3], void* stream) {
    return walls_t(desc, E, as_stream(stream));
}

int pic_yee_update_b(const PicDesc* desc, const float* const E[3], const float* const B_in[3], float* const B_out[3],
                     void* stream) {
    return yee_b_t(desc, E, B_in, B_out, as_stream(stream));
}

int pic_yee_update_b_f64(const PicDesc* desc, const double* const E[3], const double* const B_in[3],
                         double* const B_out[3], void* stream) {
    return yee_b_t(desc, E, B_in, B_out, as_stream(stream));
}

int pic_yee_update_e(const PicDesc* desc, const float* const E_in[3], const float* const B[3], const float* const J[3],
                     float* const E_out[3], void* stream) {
    return yee_e_t(desc, E_in, B, J, E_out, as_stream(stream));
}

int pic_yee_update_e_f64(const PicDesc* desc, const double* const E_in[3], const double* const B[3],
                         const double* const J[3], double* const E_out[3], void* stream) {
    return yee_e_t(desc, E_in, B, J, E_out, as_stream(stream));
}

static bool pml_ok(const PicPml* pml) {
    if (!pml) return false;
    for (int q = 0; q < 6; ++q)
        if (!pml->mem[q]) return false;
    for (int a = 0; a < 3; ++a)
        if (!pml->sigma[a]) return false;
    return true;
}

static PmlArgs pml_args(const PicDesc* desc, const PicPml* pml) {
    PmlArgs a;
    for (int q = 0; q < 6; ++q) a.mem[q] = pml->mem[q];
    for (int c = 0; c < 3; ++c) {
        a.sigma[c] = pml->sigma[c];
        a.line[c] = pml->sigma_line[c];
    }
    a.dt = (float)desc->dt;          // the stretch uses the full step in both updates (PML.py:291, 337)
    return a;
}

int pic_yee_update_b_pml(const PicDesc* desc, const float* const E[3], const float* const B_in[3],
                         float* const B_out[3], const PicPml* pml, void* stream) {
    PIC_REQUIRE(desc_ok(desc) && E && B_in && B_out && pml_ok(pml));
    for (int c = 0; c < 3; ++c) PIC_REQUIRE(E[c] && B_in[c] && B_out[c]);
    for (int c = 0; c < 3; ++c)
        for (int e = 0; e < 3; ++e) PIC_REQUIRE((const float*)B_out[c] != E[e]);
    hipStream_t s = as_stream(stream);
    int block = interior_block(desc);
    hipLaunchKernelGGL(yee_b_pml_kernel, interior_grid(desc, block), dim3(block), 0, s, *desc, yee_const(*desc),
                       pml_args(desc, pml), F3{{E[0], E[1], E[2]}}, F3{{B_in[0], B_in[1], B_in[2]}},
                       W3f{{B_out[0], B_out[1], B_out[2]}}, interior_flat(desc));
    PIC_CHECK_LAUNCH();
    return 0;
}

int pic_yee_update_e_pml(const PicDesc* desc, const float* const E_in[3], const float* const B[3],
                         const float* const J[3], float* const E_out[3], const PicPml* pml, void* stream) {
    PIC_REQUIRE(desc_ok(desc) && E_in && B && J && E_out && pml_ok(pml));
    for (int c = 0; c < 3; ++c) PIC_REQUIRE(E_in[c] && B[c] && J[c] && E_out[c]);
    for (int c = 0; c < 3; ++c)
        for (int e = 0; e < 3; ++e) PIC_REQUIRE((const float*)E_out[c] != B[e] && (const float*)E_out[c] != J[e]);
    hipStream_t s = as_stream(stream);
    int block = interior_block(desc);
    hipLaunchKernelGGL(yee_e_pml_kernel, interior_grid(desc, block), dim3(block), 0, s, *desc, yee_const(*desc),
                       pml_args(desc, pml), F3{{E_in[0], E_in[1], E_in[2]}}, F3{{B[0], B[1], B[2]}},
                       F3{{J[0], J[1], J[2]}}, W3f{{E_out[0], E_out[1], E_out[2]}}, interior_flat(desc));
    PIC_CHECK_LAUNCH();
    return 0;
}

int pic_pml_stretch(const PicDesc* desc, float* const deriv[6], const PicPml* pml, void* stream) {
    PIC_REQUIRE(desc_ok(desc) && deriv && pml_ok(pml));
    W6f dv;
    for (int q = 0; q < 6; ++q) {
        PIC_REQUIRE(deriv[q]);
        dv.p[q] = deriv[q];
    }
    hipStream_t s = as_stream(stream);
    int block = interior_block(desc);
    hipLaunchKernelGGL(pml_stretch_kernel, interior_grid(desc, block), dim3(block), 0, s, *desc, pml_args(desc, pml),
                       dv, interior_flat(desc));
    PIC_CHECK_LAUNCH();
    return 0;
}

int pic_efield_from_phi(const PicDesc* desc, const float* phi, float* const E[3], void* stream) {
    PIC_REQUIRE(desc_ok(desc) && phi && E && E[0] && E[1] && E[2]);
    hipStream_t s = as_stream(stream);
    int block = interior_block(desc);
    hipLaunchKernelGGL(efield_from_phi_kernel, interior_grid(desc, block), dim3(block), 0, s, *desc, modes(desc, 0), phi,
                       E[0], E[1], E[2], (float)(1.0 / (2.0 * desc->d[0])), (float)(1.0 / (2.0 * desc->d[1])),
                       (float)(1.0 / (2.0 * desc->d[2])), interior_flat(desc));
    PIC_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
