// Per-element field operations shared by the single-simulation kernels
// (pic_fields.hip) and the ensembles' field passes (pic_batch.hip).  Each
// function handles one element id `t` or one point (i, j, k); callers map
// threads to them.  The scalar type T is float for the FP32 path and double for
// the FP64 path.
#pragma once
#include "pic_common.h"

namespace pic {

__device__ inline int64_t slab_to_index(const PicDesc& d, int axis, int pos, int a, int b) {
    if (axis == 0) return fidx(d, pos, a, b);
    if (axis == 1) return fidx(d, a, pos, b);
    return fidx(d, a, b, pos);
}

__host__ __device__ inline void other_dims(const PicDesc& d, int axis, int& da, int& db) {
    da = d.dims[axis == 0 ? 1 : 0];
    db = d.dims[axis == 2 ? 1 : 2];
}

// Number of element ids of the fold on one axis.
__host__ __device__ inline int64_t fold_elems(const PicDesc& d, int axis) {
    int da, db;
    other_dims(d, axis, da, db);
    return d.n[axis] == 1 ? (int64_t)da * db : (int64_t)d.g * da * db;
}

__device__ inline void atomic_add_t(float* p, float v) { unsafeAtomicAdd(p, v); }
__device__ inline void atomic_add_t(double* p, double v) { unsafeAtomicAdd(p, v); }

// ghost_cells.py:218-289: fold element t (< fold_elems) of a non-reduced axis.
// bc: 0 periodic self-exchange, 1 conducting reflection, other: dropped.
template <class T>
__device__ inline void fold_elem(const PicDesc& d, T* f, int axis, int bc, int64_t t) {
    int g = d.g, n = d.n[axis];
    int da, db;
    other_dims(d, axis, da, db);
    int b = (int)(t % db);
    int64_t r = t / db;
    int a = (int)(r % da);
    int l = (int)(r / da);
    int64_t lo_i = slab_to_index(d, axis, l, a, b);
    int64_t hi_i = slab_to_index(d, axis, n + g + l, a, b);
    T lo = f[lo_i];
    T hi = f[hi_i];
    f[lo_i] = (T)0;
    f[hi_i] = (T)0;
    if (bc == 0) {
        atomic_add_t(&f[slab_to_index(d, axis, n + l, a, b)], lo);
        atomic_add_t(&f[slab_to_index(d, axis, g + l, a, b)], hi);
    } else if (bc == 1) {
        atomic_add_t(&f[slab_to_index(d, axis, g + l, a, b)], -lo);
        atomic_add_t(&f[slab_to_index(d, axis, n + l, a, b)], -hi);
    }
}

// ghost_cells.py:218-235: fold element t of a reduced (single-cell) axis.
template <class T>
__device__ inline void fold_reduced_elem(const PicDesc& d, T* f, int axis, int bc, int64_t t) {
    int g = d.g;
    int da, db;
    other_dims(d, axis, da, db);
    int b = (int)(t % db);
    int a = (int)(t / db);
    T lower = (T)0, upper = (T)0;
    for (int l = 0; l < g; ++l) {
        int64_t i0 = slab_to_index(d, axis, l, a, b);
        int64_t i1 = slab_to_index(d, axis, 1 + g + l, a, b);
        lower += f[i0];
        upper += f[i1];
        f[i0] = (T)0;
        f[i1] = (T)0;
    }
    T s = lower + upper;
    int64_t c = slab_to_index(d, axis, g, a, b);
    if (bc == 0) f[c] += s;
    else if (bc == 1) f[c] += -s;
}

// ---- images: the ghost cells that belong to an interior cell --------------
// On every axis each ghost index belongs to exactly one interior index: its
// periodic partner, the cell at the same depth inside a non-periodic wall, or
// index g of a reduced axis.  The product over the axes assigns every ghost
// cell of the array to one interior cell.  A refreshed field holds the interior
// value at all images across periodic axes and 0 where a non-periodic axis is
// crossed (the x -> y -> z sequence of ghost_cells.py:142-215 composed), and
// the fold adds the images into the interior cell (:218-289), so the thread of
// an interior cell can do both in place without a second launch.

__device__ inline int image_count(const PicDesc& d, int axis) { return d.n[axis] == 1 ? 2 * d.g : 2; }

// Image q of interior index i along an axis; -1 if there is none.
__device__ inline int image_index(const PicDesc& d, int axis, int mode, int i, int q) {
    const int g = d.g, n = d.n[axis];
    if (n == 1) return q < g ? q : q + 1;
    if (q == 0) return i < 2 * g ? (mode == MODE_PERIODIC ? i + n : i - g) : -1;
    return i >= n ? (mode == MODE_PERIODIC ? i - n : i + g) : -1;
}

// Whether interior index i has images on an axis.
__device__ inline bool has_images(const PicDesc& d, int axis, int i) {
    return d.n[axis] == 1 || i < 2 * d.g || i >= d.n[axis];
}

// The image of an interior index on an axis of at least two guard bands, which
// has at most one; -1 if it has none.
__device__ inline int single_image(const PicDesc& d, int axis, int mode, int i) {
    const int g = d.g, n = d.n[axis];
    if (i < 2 * g) return mode == MODE_PERIODIC ? i + n : i - g;
    if (i >= n) return mode == MODE_PERIODIC ? i - n : i + g;
    return -1;
}

// Every axis with at most one image per cell (uniform over a launch).
__device__ inline bool single_images(const PicDesc& d) {
    return d.n[0] >= 2 * d.g && d.n[1] >= 2 * d.g && d.n[2] >= 2 * d.g;
}

// Stores v[] at interior cell (i, j, k) of kC components and at all its images
// (v across periodic axes, 0 across others): the refresh that would follow.
template <int kC, class T>
__device__ inline void store_refreshed(const PicDesc& d, const int mode[3], T* const out[kC], int i, int j, int k,
                                       const T v[kC]) {
    const auto put = [&](int ii, int jj, int kk, bool zero) {
        const int64_t t = fidx(d, ii, jj, kk);
#pragma unroll
        for (int m = 0; m < kC; ++m) out[m][t] = zero ? (T)0 : v[m];
    };
    put(i, j, k, false);
    if (single_images(d)) {
        const int ii = single_image(d, 0, mode[0], i), jj = single_image(d, 1, mode[1], j);
        const int kk = single_image(d, 2, mode[2], k);
        const bool zi = mode[0] == MODE_ZERO, zj = mode[1] == MODE_ZERO, zk = mode[2] == MODE_ZERO;
        if (kk >= 0) put(i, j, kk, zk);
        if (jj >= 0) {
            put(i, jj, k, zj);
            if (kk >= 0) put(i, jj, kk, zj || zk);
        }
        if (ii >= 0) {
            put(ii, j, k, zi);
            if (kk >= 0) put(ii, j, kk, zi || zk);
            if (jj >= 0) {
                put(ii, jj, k, zi || zj);
                if (kk >= 0) put(ii, jj, kk, zi || zj || zk);
            }
        }
        return;
    }
    if (!(has_images(d, 0, i) || has_images(d, 1, j) || has_images(d, 2, k))) return;
    const int n0 = image_count(d, 0), n1 = image_count(d, 1), n2 = image_count(d, 2);
    for (int a = -1; a < n0; ++a) {
        const int ii = a < 0 ? i : image_index(d, 0, mode[0], i, a);
        if (ii < 0) continue;
        for (int b = -1; b < n1; ++b) {
            const int jj = b < 0 ? j : image_index(d, 1, mode[1], j, b);
            if (jj < 0) continue;
            for (int e = -1; e < n2; ++e) {
                const int kk = e < 0 ? k : image_index(d, 2, mode[2], k, e);
                if (kk < 0 || (a < 0 && b < 0 && e < 0)) continue;
                put(ii, jj, kk, (a >= 0 && mode[0] == MODE_ZERO) || (b >= 0 && mode[1] == MODE_ZERO) ||
                                    (e >= 0 && mode[2] == MODE_ZERO));
            }
        }
    }
}

// Interior value of the fold of f at (i, j, k): the cell plus its images, each
// axis' images with the sign of its code (0 periodic: +, 1 conducting /
// reflecting: -, other: dropped), x summed first as the sequential fold does.
template <class T>
__device__ inline T folded_at(const PicDesc& d, const int mode[3], const int sign[3], const T* f, int i, int j,
                              int k) {
    if (single_images(d)) {
        // the up to eight cells as independent loads
        const int at[3][2] = {{i, sign[0] ? single_image(d, 0, mode[0], i) : -1},
                              {j, sign[1] ? single_image(d, 1, mode[1], j) : -1},
                              {k, sign[2] ? single_image(d, 2, mode[2], k) : -1}};
        T v[2][2][2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int a = 0; a < 2; ++a)
                    v[e][b][a] = (a && at[0][1] < 0) || (b && at[1][1] < 0) || (e && at[2][1] < 0)
                                     ? (T)0
                                     : f[fidx(d, at[0][a], at[1][b], at[2][e])];
        T plane[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const T l0 = v[e][0][0] + (sign[0] < 0 ? -v[e][0][1] : v[e][0][1]);
            const T l1 = v[e][1][0] + (sign[0] < 0 ? -v[e][1][1] : v[e][1][1]);
            plane[e] = l0 + (sign[1] < 0 ? -l1 : l1);
        }
        return plane[0] + (sign[2] < 0 ? -plane[1] : plane[1]);
    }
    T total = (T)0;
    const int n0 = sign[0] ? image_count(d, 0) : 0, n1 = sign[1] ? image_count(d, 1) : 0;
    const int n2 = sign[2] ? image_count(d, 2) : 0;
    for (int e = -1; e < n2; ++e) {
        const int kk = e < 0 ? k : image_index(d, 2, mode[2], k, e);
        if (kk < 0) continue;
        T plane = (T)0;
        for (int b = -1; b < n1; ++b) {
            const int jj = b < 0 ? j : image_index(d, 1, mode[1], j, b);
            if (jj < 0) continue;
            T line = (T)0;
            for (int a = -1; a < n0; ++a) {
                const int ii = a < 0 ? i : image_index(d, 0, mode[0], i, a);
                if (ii < 0) continue;
                const T v = f[fidx(d, ii, jj, kk)];
                line += a >= 0 && sign[0] < 0 ? -v : v;
            }
            plane += b >= 0 && sign[1] < 0 ? -line : line;
        }
        total += e >= 0 && sign[2] < 0 ? -plane : plane;
    }
    return total;
}

// Fold and refresh of f at interior cell (i, j, k), in place; nothing to do
// (and nothing read) where the cell has no images.
template <class T>
__device__ inline void finish_point(const PicDesc& d, const int mode[3], const int sign[3], T* f, int i, int j, int k) {
    if (!(has_images(d, 0, i) || has_images(d, 1, j) || has_images(d, 2, k))) return;
    const T v[1] = {folded_at(d, mode, sign, f, i, j, k)};
    T* const out[1] = {f};
    store_refreshed<1>(d, mode, out, i, j, k, v);
}

// Interior indices of an axis with images, and the s-th of them; the others
// are 2g .. n-1.
__host__ __device__ inline int shell_count(const PicDesc& d, int axis) {
    return d.n[axis] < 2 * d.g ? d.n[axis] : 2 * d.g;
}
__device__ inline int shell_index(const PicDesc& d, int axis, int s) {
    return s < d.g || d.n[axis] < 2 * d.g ? d.g + s : d.n[axis] + s - d.g;
}

// Sign of each axis' images in a fold with the particle (bc_type 1) or field codes.
__host__ __device__ inline int fold_sign(const PicDesc& d, int axis, int bc_type) {
    const int bc = bc_type == 0 ? d.bc[axis] : d.pbc[axis];
    return bc == 0 ? 1 : (bc == 1 ? -1 : 0);
}

// Whether component c of E is tangential to a conducting wall at (i, j, k)
// (first_order_yee.py:80-92: zero on the planes g and n+g-1).
__device__ inline bool on_wall(const PicDesc& d, int c, int i, int j, int k) {
    const int at[3] = {i, j, k};
#pragma unroll
    for (int a = 0; a < 3; ++a)
        if (a != c && d.bc[a] == 1 && (at[a] == d.g || at[a] == d.n[a] + d.g - 1)) return true;
    return false;
}

// Value of a refreshed copy of f at (i,j,k) where exactly one coordinate may
// sit one cell outside the interior along `axis`.
template <class T>
__device__ inline T refreshed_at(const T* __restrict__ f, const PicDesc& d, const int mode[3], int i, int j, int k,
                                 int axis) {
    int c[3] = {i, j, k};
    int src = ghost_source(c[axis], d.n[axis], d.g, mode[axis]);
    if (src < 0) return (T)0;
    c[axis] = src;
    return f[fidx(d, c[0], c[1], c[2])];
}

template <class T>
struct YeeConstT {
    T hdt, dt, c2, inv_eps, id[3];
    int mode[3];
};
using YeeConst = YeeConstT<float>;

template <class T = float>
__host__ __device__ inline YeeConstT<T> yee_const(const PicDesc& d) {
    YeeConstT<T> y;
    y.hdt = (T)(d.dt / 2);
    y.dt = (T)d.dt;
    y.c2 = (T)(d.C * d.C);
    y.inv_eps = (T)(1.0 / d.eps);
    for (int a = 0; a < 3; ++a) {
        y.id[a] = (T)(1.0 / d.d[a]);
        y.mode[a] = refresh_mode(d, a, 0);
    }
    return y;
}

// first_order_yee.py:96-142 at interior array point (i, j, k):
// v = B_in - (dt/2) curl E with forward differences.
template <class T>
__device__ inline void yee_b_value(const PicDesc& d, const YeeConstT<T>& y, const T* const E[3], const T* const B[3],
                                   T v[3], int i, int j, int k) {
    int64_t c = fidx(d, i, j, k);
    T ex = E[0][c], ey = E[1][c], ez = E[2][c];
    T ez_yp = refreshed_at(E[2], d, y.mode, i, j + 1, k, 1);
    T ey_zp = refreshed_at(E[1], d, y.mode, i, j, k + 1, 2);
    T ex_zp = refreshed_at(E[0], d, y.mode, i, j, k + 1, 2);
    T ez_xp = refreshed_at(E[2], d, y.mode, i + 1, j, k, 0);
    T ey_xp = refreshed_at(E[1], d, y.mode, i + 1, j, k, 0);
    T ex_yp = refreshed_at(E[0], d, y.mode, i, j + 1, k, 1);
    T curl_x = (ez_yp - ez) * y.id[1] - (ey_zp - ey) * y.id[2];
    T curl_y = (ex_zp - ex) * y.id[2] - (ez_xp - ez) * y.id[0];
    T curl_z = (ey_xp - ey) * y.id[0] - (ex_yp - ex) * y.id[1];
    v[0] = B[0][c] - y.hdt * curl_x;
    v[1] = B[1][c] - y.hdt * curl_y;
    v[2] = B[2][c] - y.hdt * curl_z;
}

// The point stored with its guard images (out may be B: only the point itself is read from it).
template <class T>
__device__ inline void yee_b_point(const PicDesc& d, const YeeConstT<T>& y, const T* const E[3], const T* const B[3],
                                   T* const out[3], int i, int j, int k) {
    T v[3];
    yee_b_value(d, y, E, B, v, i, j, k);
    store_refreshed<3>(d, y.mode, out, i, j, k, v);
}

// first_order_yee.py:12-72 at interior array point (i, j, k):
// v = E_in + dt (C^2 curl B - J/eps) with backward differences.
template <class T>
__device__ inline void yee_e_value(const PicDesc& d, const YeeConstT<T>& y, const T* const E[3], const T* const B[3],
                                   const T* const J[3], T v[3], int i, int j, int k) {
    int64_t c = fidx(d, i, j, k);
    T bx = B[0][c], by = B[1][c], bz = B[2][c];
    T bz_ym = refreshed_at(B[2], d, y.mode, i, j - 1, k, 1);
    T by_zm = refreshed_at(B[1], d, y.mode, i, j, k - 1, 2);
    T bx_zm = refreshed_at(B[0], d, y.mode, i, j, k - 1, 2);
    T bz_xm = refreshed_at(B[2], d, y.mode, i - 1, j, k, 0);
    T by_xm = refreshed_at(B[1], d, y.mode, i - 1, j, k, 0);
    T bx_ym = refreshed_at(B[0], d, y.mode, i, j - 1, k, 1);
    T curl_x = (bz - bz_ym) * y.id[1] - (by - by_zm) * y.id[2];
    T curl_y = (bx - bx_zm) * y.id[2] - (bz - bz_xm) * y.id[0];
    T curl_z = (by - by_xm) * y.id[0] - (bx - bx_ym) * y.id[1];
    v[0] = E[0][c] + (y.c2 * curl_x - J[0][c] * y.inv_eps) * y.dt;
    v[1] = E[1][c] + (y.c2 * curl_y - J[1][c] * y.inv_eps) * y.dt;
    v[2] = E[2][c] + (y.c2 * curl_z - J[2][c] * y.inv_eps) * y.dt;
}

template <class T>
__device__ inline void yee_e_point(const PicDesc& d, const YeeConstT<T>& y, const T* const E[3], const T* const B[3],
                                   const T* const J[3], T* const out[3], int i, int j, int k) {
    T v[3];
    yee_e_value(d, y, E, B, J, v, i, j, k);
    store_refreshed<3>(d, y.mode, out, i, j, k, v);
}

// PML coordinate stretch of the six curl derivatives (PML.py:251-359): for a
// derivative d along axis a at interior point (i, j, k), with b = exp(-sigma_a
// dt) from the ghosted profile of axis a, the ADE memory becomes
// m' = b m + (b - 1) d and the derivative d + m'.  Derivative order (and memory
// order): d?z/dy, d?y/dz, d?x/dz, d?z/dx, d?y/dx, d?x/dy; curl = (d0 - d1,
// d2 - d3, d4 - d5).  mem[] are interior (Nx, Ny, Nz) arrays updated in place.
// line[a] (optional) holds profile a along its own axis, for profiles that do
// not vary along the other two: one cached value per point instead of three
// reads of field-shaped arrays.
struct PmlArgs {
    float* mem[6];
    const float* sigma[3];
    const float* line[3];
    float dt;
};

__device__ inline void pml_stretch6(const PicDesc& d, const PmlArgs& pml, int i, int j, int k, float dv[6]) {
    const int64_t c = fidx(d, i, j, k);
    const int64_t mi = ((int64_t)(i - d.g) * d.n[1] + (j - d.g)) * d.n[2] + (k - d.g);
    const int idx[3] = {i, j, k};
    float b[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) b[a] = expf(-(pml.line[a] ? pml.line[a][idx[a]] : pml.sigma[a][c]) * pml.dt);
    constexpr int kAxis[6] = {1, 2, 2, 0, 0, 1};
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const float bb = b[kAxis[q]];
        const float m = bb * pml.mem[q][mi] + (bb - 1.0f) * dv[q];
        if (bb != 1.0f) pml.mem[q][mi] = m;     // sigma = 0: m' = m, nothing to write
        dv[q] += m;
    }
}

// yee_b_point with the PML stretch of the E derivatives (first_order_yee.py:127-142).
__device__ inline void yee_b_point_pml(const PicDesc& d, const YeeConst& y, const PmlArgs& pml,
                                       const float* const E[3], const float* const B[3], float* const out[3], int i,
                                       int j, int k) {
    int64_t c = fidx(d, i, j, k);
    float ex = E[0][c], ey = E[1][c], ez = E[2][c];
    float dv[6] = {(refreshed_at(E[2], d, y.mode, i, j + 1, k, 1) - ez) * y.id[1],
                   (refreshed_at(E[1], d, y.mode, i, j, k + 1, 2) - ey) * y.id[2],
                   (refreshed_at(E[0], d, y.mode, i, j, k + 1, 2) - ex) * y.id[2],
                   (refreshed_at(E[2], d, y.mode, i + 1, j, k, 0) - ez) * y.id[0],
                   (refreshed_at(E[1], d, y.mode, i + 1, j, k, 0) - ey) * y.id[0],
                   (refreshed_at(E[0], d, y.mode, i, j + 1, k, 1) - ex) * y.id[1]};
    pml_stretch6(d, pml, i, j, k, dv);
    const float v[3] = {B[0][c] - y.hdt * (dv[0] - dv[1]), B[1][c] - y.hdt * (dv[2] - dv[3]),
                        B[2][c] - y.hdt * (dv[4] - dv[5])};
    store_refreshed<3>(d, y.mode, out, i, j, k, v);
}

// yee_e_point with the PML stretch of the B derivatives (first_order_yee.py:49-72).
__device__ inline void yee_e_point_pml(const PicDesc& d, const YeeConst& y, const PmlArgs& pml,
                                       const float* const E[3], const float* const B[3], const float* const J[3],
                                       float* const out[3], int i, int j, int k) {
    int64_t c = fidx(d, i, j, k);
    float bx = B[0][c], by = B[1][c], bz = B[2][c];
    float dv[6] = {(bz - refreshed_at(B[2], d, y.mode, i, j - 1, k, 1)) * y.id[1],
                   (by - refreshed_at(B[1], d, y.mode, i, j, k - 1, 2)) * y.id[2],
                   (bx - refreshed_at(B[0], d, y.mode, i, j, k - 1, 2)) * y.id[2],
                   (bz - refreshed_at(B[2], d, y.mode, i - 1, j, k, 0)) * y.id[0],
                   (by - refreshed_at(B[1], d, y.mode, i - 1, j, k, 0)) * y.id[0],
                   (bx - refreshed_at(B[0], d, y.mode, i, j - 1, k, 1)) * y.id[1]};
    pml_stretch6(d, pml, i, j, k, dv);
    const float v[3] = {E[0][c] + (y.c2 * (dv[0] - dv[1]) - J[0][c] * y.inv_eps) * y.dt,
                        E[1][c] + (y.c2 * (dv[2] - dv[3]) - J[1][c] * y.inv_eps) * y.dt,
                        E[2][c] + (y.c2 * (dv[4] - dv[5]) - J[2][c] * y.inv_eps) * y.dt};
    store_refreshed<3>(d, y.mode, out, i, j, k, v);
}

}  // namespace pic
