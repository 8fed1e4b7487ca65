// kernels.hpp - gfx950 kernels of the three leapfrog loops.
//
// Field and operator values are of type T (double on the plain path, float on
// the fast path); every reduction accumulates in double. Incidence is stored
// as int32 indices plus signs: 2-bit codes packed four to a byte
// (0 = absent, 1 = +1, 3 = -1) for the fixed-width FIT stencils, int8 per
// entry for the CSR incidence of the tetrahedral meshes.
#pragma once

#include "common.hpp"

#include <algorithm>

namespace tfd {

__device__ __forceinline__ double sgn2(uint32_t code) {
    // 0 -> 0, 1 -> +1, 3 -> -1
    return code == 1 ? 1.0 : (code == 3 ? -1.0 : 0.0);
}

// Value injected at a source edge for the current step: sum of its terms of
// carrier(source, step) * weight.
__device__ __forceinline__ double source_value(int tb, int te, const int32_t* __restrict__ term_src,
                                               const double* __restrict__ term_w,
                                               const double* __restrict__ carr_step) {
    double v = 0;
    for (int t = tb; t < te; ++t) v += carr_step[term_src[t]] * term_w[t];
    return v;
}

// Device state of one CG solve (kernels in sell.hpp). Each kernel writes one
// fp64 partial per block; the next kernel sums them (every block, in index
// order, so all blocks take the same decision) - no cross-block fences.
struct CgState {
    double rr0;        // ||r0||^2 of this solve
    double gam[2];     // r.u of pass it, slot it&1
    double alpha[2];   // step length of pass it, slot it&1
    double beta[2];    // beta of pass it, slot it&1 (learned passes)
    double relres;     // ||r||/||r0|| at the last stop test
    double tol;
    int32_t maxiter;
    int32_t iter;      // iterations done when the solve stopped
    int32_t done;
    int32_t need_conv;  // the solve must meet tol (learned solves; Jacobi ones may stop at maxiter)
    int32_t rr0_given;  // rr0 holds the warm-start residual of an extrapolated start (cg_set_rr0_kernel)
};

// Guard of the kernels a gfdtd step enqueues ahead of the host's check of
// the previous CG solve (gf_scatter of that step, the next step's
// dga_curl, sell_n, probe_kernel, gf_inject and gf_rhs_init): they run only
// if that solve has stopped, and, for a solve that must meet the tolerance,
// met it. Otherwise they return at once and the host enqueues them again
// once the solve is complete. A null guard always passes.
__device__ __forceinline__ bool cg_guard_ok(const CgState* g) {
    return !g || (g->done && (!g->need_conv || g->relres <= g->tol));
}

// Extrapolated start of a gfdtd solve (an option of the fast path; the
// stop test stays relative to the warm-start residual b - A U_old). On the
// free rows x holds U_n (the warm start), h1 = U_{n-1}, h2 = U_{n-2}:
// order 1: x0 = 2 U_n - U_{n-1}; order 2: x0 = 3 U_n - 3 U_{n-1} + U_{n-2};
// order 0: x unchanged. d = x0 - U_n as the rounded x0 gives it (exact when
// x0 and U_n lie within a factor of two, Sterbenz), for r0 - A d; the
// history then shifts by one step. Guard as in cg_guard_ok.
template <typename T>
__global__ void __launch_bounds__(kBlock) cg_extrap_kernel(int32_t n, T* __restrict__ x, T* __restrict__ h1,
                                                           T* __restrict__ h2, T* __restrict__ d, int order,
                                                           const CgState* guard) {
    if (!cg_guard_ok(guard)) return;
    for (int32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const T xi = x[i], a = h1[i], b = h2[i];
        const double x0 = order == 2 ? 3.0 * (double)xi - 3.0 * (double)a + (double)b
                          : order == 1 ? 2.0 * (double)xi - (double)a
                                       : (double)xi;
        const T x0t = (T)x0;
        d[i] = (T)((double)x0t - (double)xi);
        x[i] = x0t;
        h2[i] = a;
        h1[i] = xi;
    }
}

// ------------------------------------------------------------------ FIT
//
// Grid order (tf_fit_ops edge_sid / face_sid): with the fields stored at
// the grid positions of their edges and faces, the four faces around an
// interior edge and the four edges of a face follow from the position.
// Slots: x edge (i,j,k): y faces (i,j,k-1), (i,j,k), z faces (i,j-1,k),
// (i,j,k); y edge: x faces (i,j,k-1), (i,j,k), z faces (i-1,j,k), (i,j,k);
// z edge: x faces (i,j-1,k), (i,j,k), y faces (i-1,j,k), (i,j,k). x face
// (i,j,k): y edges (i,j,k), (i,j,k+1), z edges (i,j,k), (i,j+1,k); y face:
// x edges (i,j,k), (i,j,k+1), z edges (i,j,k), (i+1,j,k); z face: x edges
// (i,j,k), (i,j+1,k), y edges (i,j,k), (i+1,j,k). Slots of boundary
// entities may lie outside the grid; those are never read (code 0).
// Division of n < 2^31 by a fixed divisor d >= 1 with a multiply-high and a
// shift (Granlund and Montgomery, "Division by invariant integers using
// multiplication", PLDI 1994): l = ceil(log2 d), m = 2^32 (2^l - d) / d + 1,
// n / d = (mulhi(m, n) + n) >> l; mulhi(m, n) < n, so the sum stays below
// 2^32.
struct FastDiv {
    uint32_t d, m, l;
};
inline FastDiv make_fastdiv(uint32_t d) {
    uint32_t l = 0;
    while (((uint64_t)1 << l) < d) ++l;
    const uint64_t m = ((((uint64_t)1 << l) - d) << 32) / d + 1;
    return FastDiv{d, (uint32_t)m, l};
}
__host__ __device__ inline uint32_t fastdiv(const FastDiv& f, uint32_t n) {
#if defined(__HIP_DEVICE_COMPILE__)
    const uint32_t t = __umulhi(f.m, n);
#else
    const uint32_t t = (uint32_t)(((uint64_t)f.m * n) >> 32);
#endif
    return (t + n) >> f.l;
}

struct FitGrid {
    int32_t nx, ny, nz;
    FastDiv dx, dx1, dy, dy1;  // by nx, nx + 1, ny, ny + 1
};
inline FitGrid make_fit_grid(int32_t nx, int32_t ny, int32_t nz) {
    return FitGrid{nx, ny, nz, make_fastdiv(nx), make_fastdiv(nx + 1), make_fastdiv(ny), make_fastdiv(ny + 1)};
}
// n = q d + r with the fixed divisor of f
__host__ __device__ inline void fit_divmod(const FastDiv& f, uint32_t n, uint32_t& q, uint32_t& r) {
    q = fastdiv(f, n);
    r = n - q * f.d;
}
// Items of each direction in grid order: x, y, z edges (faces = false) or
// x, y, z faces (faces = true).
__host__ __device__ inline void fit_counts(const FitGrid g, bool faces, uint32_t n[3]) {
    const uint32_t nx = g.nx, ny = g.ny, nz = g.nz;
    if (faces) {
        n[0] = (nx + 1) * ny * nz; n[1] = nx * (ny + 1) * nz; n[2] = nx * ny * (nz + 1);
    } else {
        n[0] = nx * (ny + 1) * (nz + 1); n[1] = (nx + 1) * ny * (nz + 1); n[2] = (nx + 1) * (ny + 1) * nz;
    }
}
// Block mapping for grid order. The items of one direction are stored k-plane
// by k-plane, so the XCD that takes the x-th eighth of the blocks of each of
// the three directions works on one k-slab of the grid, and the neighbours its
// items gather (faces of an edge, edges of a face) stay in its own L2; with a
// single contiguous range per XCD, each gathered plane would be read through
// the L2s of two XCDs. Workgroup b runs on XCD b % 8 and takes the (b / 8)-th
// block of `per` items of that XCD's list (its x, then y, then z blocks). The
// grid has 8 * (longest list) workgroups (slab_grid).
__host__ __device__ inline uint32_t slab_len(uint32_t n, uint32_t x, uint32_t per) {
    const uint32_t nb = (n + per - 1) / per;
    return (x + 1) * nb / kXcd - x * nb / kXcd;
}
inline int slab_grid(const uint32_t n[3], uint32_t per) {
    uint32_t m = 1;
    for (uint32_t x = 0; x < (uint32_t)kXcd; ++x)
        m = std::max(m, slab_len(n[0], x, per) + slab_len(n[1], x, per) + slab_len(n[2], x, per));
    return (int)(m * kXcd);
}
// The XCD's list interleaves the three directions block by block (x, y, z,
// x, y, z, ...; the longer directions' last few blocks follow), so that all
// three advance through the slab's planes together and a plane of gathered
// neighbours, read by two directions, is fetched once while it is in L2.
// dir: the workgroup's direction (-1: none), first: its first item there.
template <uint32_t per>
__device__ __forceinline__ void slab_block(int b, const uint32_t n[3], int& dir, uint32_t& first) {
    const uint32_t x = (uint32_t)b % kXcd, i = (uint32_t)b / kXcd;
    uint32_t lo[3], len[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        const uint32_t nb = (n[t] + per - 1) / per;
        lo[t] = x * nb / kXcd;
        len[t] = (x + 1) * nb / kXcd - lo[t];
    }
    const uint32_t m = min(len[0], min(len[1], len[2]));
    uint32_t j = 0;
    dir = -1;
    if (i < 3 * m) {
        dir = (int)(i % 3);
        j = i / 3;
    } else {
        uint32_t k = i - 3 * m;
#pragma unroll
        for (int u = 0; u < 3; ++u) {
            if (dir < 0 && k < len[u] - m) {
                dir = u;
                j = m + k;
            } else if (dir < 0) {
                k -= len[u] - m;
            }
        }
    }
    first = dir < 0 ? 0 : ((dir == 0 ? lo[0] : dir == 1 ? lo[1] : lo[2]) + j) * per;
}

// 32-bit index arithmetic: grid order is used only when edge and face
// counts are below 2^31 (fit_grid_codes).
__host__ __device__ inline bool fit_edge_slots(const FitGrid g, uint32_t s, int32_t f[4]) {
    const uint32_t nx = g.nx, ny = g.ny, nz = g.nz;
    const uint32_t nEx = nx * (ny + 1) * (nz + 1), nEy = (nx + 1) * ny * (nz + 1);
    const uint32_t nFx = (nx + 1) * ny * nz, nFy = nx * (ny + 1) * nz;
    auto xf = [&](uint32_t i, uint32_t j, uint32_t k) { return (int32_t)((k * ny + j) * (nx + 1) + i); };
    auto yf = [&](uint32_t i, uint32_t j, uint32_t k) { return (int32_t)(nFx + (k * (ny + 1) + j) * nx + i); };
    auto zf = [&](uint32_t i, uint32_t j, uint32_t k) { return (int32_t)(nFx + nFy + (k * ny + j) * nx + i); };
    // out-of-grid slots (boundary edges: false) wrap around in unsigned
    // arithmetic; they are computed but never read
    auto mid = [](uint32_t a, uint32_t n) { return a > 0 && a < n; };
    uint32_t i, j, k, t;
    if (s < nEx) {
        fit_divmod(g.dx, s, t, i);
        fit_divmod(g.dy1, t, k, j);
        f[0] = yf(i, j, k - 1); f[1] = yf(i, j, k); f[2] = zf(i, j - 1, k); f[3] = zf(i, j, k);
        return mid(j, ny) && mid(k, nz);
    } else if (s < nEx + nEy) {
        fit_divmod(g.dx1, s - nEx, t, i);
        fit_divmod(g.dy, t, k, j);
        f[0] = xf(i, j, k - 1); f[1] = xf(i, j, k); f[2] = zf(i - 1, j, k); f[3] = zf(i, j, k);
        return mid(i, nx) && mid(k, nz);
    } else {
        fit_divmod(g.dx1, s - nEx - nEy, t, i);
        fit_divmod(g.dy1, t, k, j);
        f[0] = xf(i, j - 1, k); f[1] = xf(i, j, k); f[2] = yf(i - 1, j, k); f[3] = yf(i, j, k);
        return mid(i, nx) && mid(j, ny);
    }
}
__host__ __device__ inline void fit_face_slots(const FitGrid g, uint32_t s, int32_t e[4]) {
    const uint32_t nx = g.nx, ny = g.ny, nz = g.nz;
    const uint32_t nEx = nx * (ny + 1) * (nz + 1), nEy = (nx + 1) * ny * (nz + 1);
    const uint32_t nFx = (nx + 1) * ny * nz, nFy = nx * (ny + 1) * nz;
    auto xe = [&](uint32_t i, uint32_t j, uint32_t k) { return (int32_t)((k * (ny + 1) + j) * nx + i); };
    auto ye = [&](uint32_t i, uint32_t j, uint32_t k) { return (int32_t)(nEx + (k * ny + j) * (nx + 1) + i); };
    auto ze = [&](uint32_t i, uint32_t j, uint32_t k) {
        return (int32_t)(nEx + nEy + (k * (ny + 1) + j) * (nx + 1) + i);
    };
    uint32_t i, j, k, t;
    if (s < nFx) {
        fit_divmod(g.dx1, s, t, i);
        fit_divmod(g.dy, t, k, j);
        e[0] = ye(i, j, k); e[1] = ye(i, j, k + 1); e[2] = ze(i, j, k); e[3] = ze(i, j + 1, k);
    } else if (s < nFx + nFy) {
        fit_divmod(g.dx, s - nFx, t, i);
        fit_divmod(g.dy1, t, k, j);
        e[0] = xe(i, j, k); e[1] = xe(i, j, k + 1); e[2] = ze(i, j, k); e[3] = ze(i + 1, j, k);
    } else {
        fit_divmod(g.dx, s - nFx - nFy, t, i);
        fit_divmod(g.dy, t, k, j);
        e[0] = xe(i, j, k); e[1] = xe(i, j + 1, k); e[2] = ye(i, j, k); e[3] = ye(i + 1, j, k);
    }
}

// The two updates, with the fused multiply-add written out so that every
// kernel rounds them alike: ca u + cb c and cm f - dt c.
__device__ __forceinline__ double fit_e_new(double ca, double u, double cb, double c) {
    return __builtin_fma(ca, u, cb * c);
}
__device__ __forceinline__ double fit_b_new(double cm, double f, double dtc) { return __builtin_fma(cm, f, -dtc); }

// One special item of the E phase (D:1850-1895): uncommon h-source edges and
// e / j source edges, with their own face lists and fp64 coefficients:
//   kind 0 (h):  U = ca*U_old + cb*(sum s_k F + src)     (ca = M_h M_q, cb = M_h dt)
//   kind 1 (e):  U = src
//   kind 2 (j):  U = ca*U_old + cb*(sum s_k F - src)     (common coefficients)
struct FitSpecial {
    int32_t n;
    const int32_t* edge;
    const int4* f4;
    const uint8_t* sg;
    const double* ca;
    const double* cb;
    const int8_t* kind;
    const int32_t* tb;
    const int32_t* te;
    const int32_t* term_src;
    const double* term_w;
};
template <typename T>
__device__ __forceinline__ double fit_special(const FitSpecial& sp, int32_t i, double uold, double src,
                                              const T* __restrict__ Fv) {
    const int k = sp.kind[i];
    if (k == 1) return src;
    const int4 f = sp.f4[i];
    const uint32_t s = sp.sg[i];
    double c = 0;
    if (s & 3) c += sgn2(s & 3) * (double)Fv[f.x];
    if ((s >> 2) & 3) c += sgn2((s >> 2) & 3) * (double)Fv[f.y];
    if ((s >> 4) & 3) c += sgn2((s >> 4) & 3) * (double)Fv[f.z];
    if ((s >> 6) & 3) c += sgn2((s >> 6) & 3) * (double)Fv[f.w];
    c += k == 0 ? src : -src;
    return fit_e_new(sp.ca[i], uold, sp.cb[i], c);
}
// Source value of a special item from one carrier row.
__device__ __forceinline__ double fit_source(const FitSpecial& sp, int32_t i, const double* __restrict__ carr) {
    return source_value(sp.tb[i], sp.te[i], sp.term_src, sp.term_w, carr);
}

// E phase of the index-table layout (D:1850-1895). The first sp_blocks
// workgroups take the special items, so that their longer dependent chains
// (source value, Poynting sum) start with the launch instead of trailing it;
// the rest cover every edge in index order (XCD-mapped among themselves).
// Edges whose sign byte is 0 (pec / source / non-common) are left to the
// special items. U = ca*U_old + cb*(sum_k s_k F[f_k])
//   common:   ca = upml^2 M_h M_q, cb = upml^3 M_h dt, s = dual_curl*(+,-,+,-)
template <typename T>
__global__ void __launch_bounds__(kBlock) fit_e_kernel(int32_t n_edges, int32_t sp_blocks,
                                                       const uint8_t* __restrict__ sg, const T* __restrict__ ca,
                                                       const T* __restrict__ cb, const int4* __restrict__ f4,
                                                       const T* __restrict__ Fv, T* __restrict__ U, FitSpecial sp,
                                                       const double* __restrict__ carr_step,
                                                       double* __restrict__ poy_part) {
    const int hb = (int)blockIdx.x;
    if (hb >= sp_blocks) {
        const int32_t e = xcd_block_of(hb - sp_blocks, (int)gridDim.x - sp_blocks) * kBlock + threadIdx.x;
        if (e >= n_edges) return;
        const uint32_t s = sg[e];
        if (s == 0) return;
        const int4 f = f4[e];
        double c = sgn2(s & 3) * (double)Fv[f.x] + sgn2((s >> 2) & 3) * (double)Fv[f.y] +
                   sgn2((s >> 4) & 3) * (double)Fv[f.z] + sgn2((s >> 6) & 3) * (double)Fv[f.w];
        U[e] = (T)fit_e_new((double)ca[e], (double)U[e], (double)cb[e], c);
        return;
    }
    __shared__ double red[kBlock / kWave];
    const int32_t i = hb * kBlock + threadIdx.x;
    double poy = 0;
    if (i < sp.n) {
        const int32_t e = sp.edge[i];
        const double src = fit_source(sp, i, carr_step);
        const double uold = (double)U[e];
        const double unew = fit_special<T>(sp, i, uold, src, Fv);
        U[e] = (T)unew;
        // Poynting term 0.5*(U_old+U)*curl_fb, nonzero on h-source edges only (D:1901)
        if (sp.kind[i] == 0) poy = 0.5 * (uold + (double)(T)unew) * src;
    }
    const double s = block_sum(poy, red);
    if (threadIdx.x == 0) poy_part[hb] = s;
}

// H phase over tbc faces (D:1908-1915), index-table layout:
// B = cm*F_old - dt*sum s_k U[e_k]; F = cn*B with cm = M_mu*fpml,
// cn = fpml*M_nu, s = curl*(+,-,+,-).
template <typename T>
__global__ void __launch_bounds__(kBlock) fit_h_kernel(int32_t n_faces, const uint8_t* __restrict__ sg,
                                                       const T* __restrict__ cm, const T* __restrict__ cn,
                                                       const int4* __restrict__ e4, const T* __restrict__ U,
                                                       T* __restrict__ Fv, T* __restrict__ B, double dt) {
    const int32_t f = xcd_block() * kBlock + threadIdx.x;
    if (f >= n_faces) return;
    const uint32_t s = sg[f];
    if (s == 0) return;
    const int4 e = e4[f];
    double c = sgn2(s & 3) * (double)U[e.x] + sgn2((s >> 2) & 3) * (double)U[e.y] +
               sgn2((s >> 4) & 3) * (double)U[e.z] + sgn2((s >> 6) & 3) * (double)U[e.w];
    const double b = fit_b_new((double)cm[f], (double)Fv[f], dt * c);
    B[f] = (T)b;
    Fv[f] = (T)((double)cn[f] * b);
}

// ------------------------------------------------------------------ probes
// One thread per (probe, component): E from U, H from B (D:2400-2470,
// D:3093-3158). Output sample layout [probe][6].
struct ProbeDev {
    int32_t ne, nh;
    int32_t e_idx[12];
    double e_w[12][3];
    int32_t h_idx[6];
    double h_w[6][3];
};

// Component c of probe q. All loads are issued before the first is used (the
// terms' sum keeps its order): as a loop of dependent loads the 12 terms of a
// FIT probe took 8.6 us a launch.
template <typename T>
__device__ __forceinline__ double probe_value(const ProbeDev& q, int c, const T* __restrict__ U,
                                              const T* __restrict__ B) {
    const bool e = c < 3;
    const int n = e ? q.ne : q.nh, cc = e ? c : c - 3;
    double v = 0;
    if (e) {
        T x[12];
        double w[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            x[k] = U[k < n ? q.e_idx[k] : 0];
            w[k] = q.e_w[k][cc];
        }
#pragma unroll
        for (int k = 0; k < 12; ++k)
            if (k < n) v += (double)x[k] * w[k];
    } else {
        T x[6];
        double w[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            x[k] = B[k < n ? q.h_idx[k] : 0];
            w[k] = q.h_w[k][cc];
        }
#pragma unroll
        for (int k = 0; k < 6; ++k)
            if (k < n) v += (double)x[k] * w[k];
    }
    return v;
}

template <typename T>
__global__ void probe_kernel(int32_t n_probes, const ProbeDev* __restrict__ pr, const T* __restrict__ U,
                             const T* __restrict__ B, double* __restrict__ out, const CgState* guard) {
    if (!cg_guard_ok(guard)) return;
    const int32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_probes * 6) return;
    out[t] = probe_value<T>(pr[t / 6], t % 6, U, B);
}

// Sampling inside a step's kernels: workgroups of the launch evaluate the
// probes for the output sample *slot (negative: none), components [c0, c0 + nc)
// of each (0..2 from U, 3..5 from B). The probes and the sample buffer are read
// from device memory, so that captured steps follow a change of either. As a
// launch of its own a sample cost 5 us of host-launched step at 16^3, and kept
// the steps out of the graph.
struct SampleRef {
    const ProbeDev* probes;
    double* out;
    int32_t n_probes;
};
template <typename T>
__device__ __forceinline__ void sample_probes(const SampleRef* __restrict__ ref, const int64_t* __restrict__ slot,
                                              int32_t t, int c0, int nc, const T* __restrict__ U,
                                              const T* __restrict__ B) {
    const int64_t sl = *slot;
    const SampleRef r = *ref;
    const int32_t p = t / nc, c = c0 + t % nc;
    if (sl < 0 || p >= r.n_probes) return;
    r.out[(sl * r.n_probes + p) * 6 + c] = probe_value<T>(r.probes[p], c, U, B);
}

// A sample taken by workgroups appended to another kernel's grid.
template <typename T>
struct SampleArgs {
    int32_t blocks = 0;
    const SampleRef* ref = nullptr;
    const int64_t* slot = nullptr;
    const T* U = nullptr;
    const T* B = nullptr;
};

template <typename T>
__global__ void __launch_bounds__(kBlock) probe_tail_kernel(const SampleRef* __restrict__ ref,
                                                            const int64_t* __restrict__ slot, int c0, int nc,
                                                            const T* __restrict__ U, const T* __restrict__ B) {
    sample_probes<T>(ref, slot, (int32_t)(blockIdx.x * kBlock + threadIdx.x), c0, nc, U, B);
}

// ------------------------------------------------------------------ FIT, grid order
// Constants of one entity. With media that are uniform per region they take
// few distinct values: each entity then stores the 16-bit number of its entry
// (id 0: not updated) and a workgroup keeps the table in LDS. At most kPalMax
// entries (8 KB in fp64; a cavity holds 2 to 4, a random medium's E side one
// per edge), else id 1 and plain arrays.
template <typename T>
struct FitPal {
    T c0, c1;  // E: ca, cb; H: cm, cn
};
constexpr int kPalMax = 512;

// How a grid-order kernel finds an item's constants and the order and signs of
// its sum. kFitPal: palette; kFitPlain: plain arrays; both sum in the mesher's
// order with one sign per direction. kFitCoded: plain arrays, and the id is the
// item's own code: slot map (2 bits per position of the sum) << 8 | signs (2
// bits per position: 1 -> +1, 2 -> -1, 0 -> 0), for problems numbered in any
// other way (a step on 96^3 random media: fp64 39 us, fp32 24; with the index
// tables 50 and 35). kFitPlainNt, kFitCodedNt: the plain arrays are loaded
// non-temporally (fit_non_temporal).
enum FitMode { kFitPal, kFitPlain, kFitPlainNt, kFitCoded, kFitCodedNt };
constexpr bool fit_coded_mode(FitMode m) { return m == kFitCoded || m == kFitCodedNt; }
template <FitMode M, typename T>
__device__ __forceinline__ T fit_coef(const T* p) {
    if constexpr (M == kFitPlainNt || M == kFitCodedNt) return __builtin_nontemporal_load(p);
    else return *p;
}
template <typename T>
__device__ __forceinline__ double coded_sum(uint32_t code, T v0, T v1, T v2, T v3) {
    double c = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t m = code >> (8 + 2 * q);
        const T v = m & 2 ? (m & 1 ? v3 : v2) : (m & 1 ? v1 : v0);
        c += sgn2((code >> (2 * q)) & 3) * (double)v;
    }
    return c;
}

// id[at[i]] = val[i] (faces that become probed or stop to be)
__global__ void __launch_bounds__(kBlock) set_ids_kernel(int32_t n, const int32_t* __restrict__ at,
                                                         const uint16_t* __restrict__ val, uint16_t* __restrict__ id) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) id[at[i]] = val[i];
}

// spv[i] = source value of special item i from one carrier row.
__global__ void __launch_bounds__(kBlock) fit_src_kernel(FitSpecial sp, const double* __restrict__ carr,
                                                         double* __restrict__ spv) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < sp.n) spv[i] = fit_source(sp, i, carr);
}

// What the two kernels of a step share. A kernel starts with cold L2 (the
// other XCDs wrote part of what it reads), so on grids up to about 64^3 each
// dependent load level costs about 0.8 us of a 5 us launch. Everything an item
// needs is therefore loaded at once: its neighbours' positions follow from its
// own (clamped at the boundary, where nothing of them is used), the palette
// goes to LDS meanwhile, and source values are prepared a step ahead. Larger
// grids are bound by bytes: an fp64 item moves 26 (E) and 26 (H) with palettes,
// against 42 and 50 with plain coefficients and B stored every step.
// One step (both kernels, in a graph): 64^3 fp64 12.1 us, fp32 9.8 us; 161^3
// random media fp64 137 us. With codes read before the neighbours, five-load
// source chains and one item per thread: 15.4, 12.0 and 185 us.
template <typename T>
struct FitStep {
    FitGrid g;
    int32_t sp_blocks, probe_blocks, src_blocks;
    int32_t n_pal;        // entries of pal
    uint32_t flag;        // H: ids from here on are probed faces
    const uint16_t* id;
    const FitPal<T>* pal;
    const T* c0;          // plain coefficients (no palette)
    const T* c1;
    double sg[3];         // sign of the sums per direction (H: times dt)
    FitSpecial sp;
    const double* spv;
    double* spv_next;
    const double* carr_next;
    double* poy_part;
    const SampleRef* ref;
    const int64_t* slot;  // E: of the step before (its B); H: of this step (its U)
};

// Palette into LDS (before the loads that follow are waited for).
template <typename T, FitMode M>
__device__ __forceinline__ void fit_pal_load(const FitStep<T>& a, FitPal<T>* __restrict__ lds) {
    if constexpr (M == kFitPal)
        for (int t = (int)threadIdx.x; t < a.n_pal; t += kBlock) lds[t] = a.pal[t];
}

// E phase (D:1850-1895). Workgroups: the special items first (their chains are
// the longest), then the H components of the sample of the step before, then
// the edges, N per thread, by slab_block. U = ca U + cb c, c the signed sum of
// the edge's four faces in the order 0, 2, 3, 1 of fit_edge_slots with signs
// +, -, +, - and the direction's sign, checked when the context is created
// (kFitCoded: in the edge's own order and signs). Special items take their
// source value from spv.
template <typename T, FitMode M, int N>
__global__ void __launch_bounds__(kBlock) fit_e_grid_kernel(FitStep<T> a, const T* __restrict__ Fv, T* __restrict__ U,
                                                            const T* __restrict__ B) {
    __shared__ FitPal<T> pal[M == kFitPal ? kPalMax : 1];
    __shared__ double red[kBlock / kWave];
    const int hb = (int)blockIdx.x;
    if (hb < a.sp_blocks) {
        const int32_t i = hb * kBlock + threadIdx.x;
        double poy = 0;
        if (i < a.sp.n) {
            const int32_t e = a.sp.edge[i];
            const double src = a.spv[i], uold = (double)U[e];
            const double unew = fit_special<T>(a.sp, i, uold, src, Fv);
            U[e] = (T)unew;
            // Poynting term 0.5*(U_old+U)*curl_fb, nonzero on h-source edges only (D:1901)
            if (a.sp.kind[i] == 0) poy = 0.5 * (uold + (double)(T)unew) * src;
        }
        const double s = block_sum(poy, red);
        if (threadIdx.x == 0) a.poy_part[hb] = s;
        return;
    }
    if (hb < a.sp_blocks + a.probe_blocks) {
        sample_probes<T>(a.ref, a.slot, (hb - a.sp_blocks) * kBlock + (int)threadIdx.x, 3, 3, (const T*)nullptr, B);
        return;
    }
    uint32_t cnt[3], first;
    int dir;
    fit_counts(a.g, false, cnt);
    slab_block<N * kBlock>(hb - a.sp_blocks - a.probe_blocks, cnt, dir, first);
    if (dir < 0) return;
    const uint32_t nx = a.g.nx, ny = a.g.ny, nz = a.g.nz;
    const uint32_t nF1 = (nx + 1) * ny * nz, nF2 = nF1 + nx * (ny + 1) * nz;
    const uint32_t n = dir == 0 ? cnt[0] : dir == 1 ? cnt[1] : cnt[2];
    const uint32_t base = dir == 0 ? 0 : dir == 1 ? cnt[0] : cnt[0] + cnt[1];
    const double sg = a.sg[dir];
    fit_pal_load<T, M>(a, pal);
    uint32_t id[N];
    T u[N], v0[N], v1[N], v2[N], v3[N];
    FitPal<T> q[N];
#pragma unroll
    for (int m = 0; m < N; ++m) {
        // an item past the end repeats the last one's loads
        const uint32_t r = min(first + m * kBlock + threadIdx.x, n - 1), s = base + r;
        uint32_t i, j, k, t, f0, f1, f2, f3;
        bool in;  // all four faces exist
        if (dir == 0) {
            fit_divmod(a.g.dx, r, t, i);
            fit_divmod(a.g.dy1, t, k, j);
            in = j > 0 && j < ny && k > 0 && k < nz;
            f1 = nF1 + (k * (ny + 1) + j) * nx + i;
            f0 = f1 - (ny + 1) * nx;
            f3 = nF2 + (k * ny + j) * nx + i;
            f2 = f3 - nx;
        } else if (dir == 1) {
            fit_divmod(a.g.dx1, r, t, i);
            fit_divmod(a.g.dy, t, k, j);
            in = i > 0 && i < nx && k > 0 && k < nz;
            f1 = (k * ny + j) * (nx + 1) + i;
            f0 = f1 - ny * (nx + 1);
            f3 = nF2 + (k * ny + j) * nx + i;
            f2 = f3 - 1;
        } else {
            fit_divmod(a.g.dx1, r, t, i);
            fit_divmod(a.g.dy1, t, k, j);
            in = i > 0 && i < nx && j > 0 && j < ny;
            f1 = (k * ny + j) * (nx + 1) + i;
            f0 = f1 - (nx + 1);
            f3 = nF1 + (k * (ny + 1) + j) * nx + i;
            f2 = f3 - 1;
        }
        id[m] = a.id[s];
        u[m] = U[s];
        v0[m] = Fv[in ? f0 : 0];
        v1[m] = Fv[in ? f1 : 0];
        v2[m] = Fv[in ? f2 : 0];
        v3[m] = Fv[in ? f3 : 0];
        if constexpr (M != kFitPal) q[m] = FitPal<T>{fit_coef<M>(a.c0 + s), fit_coef<M>(a.c1 + s)};
    }
    if constexpr (M == kFitPal) __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) {
        const uint32_t r = first + m * kBlock + threadIdx.x;
        if constexpr (M == kFitPal) q[m] = pal[id[m]];
        const double c = fit_coded_mode(M)
                             ? coded_sum(id[m], v0[m], v1[m], v2[m], v3[m])
                             : sg * ((((double)v0[m] - (double)v2[m]) + (double)v3[m]) - (double)v1[m]);
        if (r < n && id[m]) U[base + r] = (T)fit_e_new((double)q[m].c0, (double)u[m], (double)q[m].c1, c);
    }
}

// H phase over tbc faces (D:1908-1915): B = cm F_old - dt c, F = cn B, c the
// signed sum of the face's four edges (order and signs as in the E phase).
// The loop itself never reads B, so it is stored only where something reads it
// before the next step overwrites it: on probed faces (id >= flag) every step
// and on every face with store_b (the run's last step, energy samples) or
// kFitCoded, whose ids have no room for the flag. The
// first workgroups take the U components of this step's sample and the next
// step's source values.
template <typename T, FitMode M, int N>
__global__ void __launch_bounds__(kBlock) fit_h_grid_kernel(FitStep<T> a, int store_b, const T* __restrict__ U,
                                                            T* __restrict__ Fv, T* __restrict__ B) {
    __shared__ FitPal<T> pal[M == kFitPal ? kPalMax : 1];
    const int hb = (int)blockIdx.x;
    if (hb < a.src_blocks) {
        const int32_t i = hb * kBlock + threadIdx.x;
        if (i < a.sp.n) a.spv_next[i] = fit_source(a.sp, i, a.carr_next);
        return;
    }
    if (hb < a.src_blocks + a.probe_blocks) {
        sample_probes<T>(a.ref, a.slot, (hb - a.src_blocks) * kBlock + (int)threadIdx.x, 0, 3, U, (const T*)nullptr);
        return;
    }
    uint32_t cnt[3], first;
    int dir;
    fit_counts(a.g, true, cnt);
    slab_block<N * kBlock>(hb - a.src_blocks - a.probe_blocks, cnt, dir, first);
    if (dir < 0) return;
    const uint32_t nx = a.g.nx, ny = a.g.ny, nz = a.g.nz;
    const uint32_t nE1 = nx * (ny + 1) * (nz + 1), nE2 = nE1 + (nx + 1) * ny * (nz + 1);
    const uint32_t n = dir == 0 ? cnt[0] : dir == 1 ? cnt[1] : cnt[2];
    const uint32_t base = dir == 0 ? 0 : dir == 1 ? cnt[0] : cnt[0] + cnt[1];
    const double sg = a.sg[dir];
    fit_pal_load<T, M>(a, pal);
    uint32_t id[N];
    T fo[N], v0[N], v1[N], v2[N], v3[N];
    FitPal<T> q[N];
#pragma unroll
    for (int m = 0; m < N; ++m) {
        const uint32_t r = min(first + m * kBlock + threadIdx.x, n - 1), s = base + r;
        uint32_t i, j, k, t, e0, e1, e2, e3;
        if (dir == 0) {
            fit_divmod(a.g.dx1, r, t, i);
            fit_divmod(a.g.dy, t, k, j);
            e0 = nE1 + (k * ny + j) * (nx + 1) + i;
            e1 = e0 + ny * (nx + 1);
            e2 = nE2 + (k * (ny + 1) + j) * (nx + 1) + i;
            e3 = e2 + (nx + 1);
        } else if (dir == 1) {
            fit_divmod(a.g.dx, r, t, i);
            fit_divmod(a.g.dy1, t, k, j);
            e0 = (k * (ny + 1) + j) * nx + i;
            e1 = e0 + (ny + 1) * nx;
            e2 = nE2 + (k * (ny + 1) + j) * (nx + 1) + i;
            e3 = e2 + 1;
        } else {
            fit_divmod(a.g.dx, r, t, i);
            fit_divmod(a.g.dy, t, k, j);
            e0 = (k * (ny + 1) + j) * nx + i;
            e1 = e0 + nx;
            e2 = nE1 + (k * ny + j) * (nx + 1) + i;
            e3 = e2 + 1;
        }
        id[m] = a.id[s];
        fo[m] = Fv[s];
        v0[m] = U[e0];
        v1[m] = U[e1];
        v2[m] = U[e2];
        v3[m] = U[e3];
        if constexpr (M != kFitPal) q[m] = FitPal<T>{fit_coef<M>(a.c0 + s), fit_coef<M>(a.c1 + s)};
    }
    if constexpr (M == kFitPal) __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m) {
        const uint32_t r = first + m * kBlock + threadIdx.x;
        if constexpr (M == kFitPal) q[m] = pal[id[m] >= a.flag ? id[m] - a.flag : id[m]];
        const double c = fit_coded_mode(M) ? coded_sum(id[m], v0[m], v1[m], v2[m], v3[m])
                                        : (((double)v0[m] - (double)v2[m]) + (double)v3[m]) - (double)v1[m];
        const double b = fit_b_new((double)q[m].c0, (double)fo[m], sg * c);
        if (r < n && id[m]) {
            if (fit_coded_mode(M) || store_b || id[m] >= a.flag) B[base + r] = (T)b;
            Fv[base + r] = (T)((double)q[m].c1 * b);
        }
    }
}

// ------------------------------------------------------------------ DGA
// Sources of the lossless dga step. h sources add Fb to curl_f (Ctb Fb, one +1
// per boundary edge), e sources set U (class-4 edges). As a kernel between
// sell_ct and sell_h they cost a launch of 4.2 us a step; now the h values of a
// step are left by the step before, in fp64, at 64 slots per Ct slice that has
// any (fbv, fb_pos), and sell_ct adds them to its rows, while workgroups
// appended to it set the e values and form the first Poynting half.
struct InjItems {
    int32_t n = 0;
    const int32_t* edge = nullptr;
    const int8_t* kind = nullptr;
    const int32_t* tb = nullptr;
    const int32_t* te = nullptr;
    const int32_t* term_src = nullptr;
    const double* term_w = nullptr;
};
__device__ __forceinline__ double inj_value(const InjItems& q, int32_t i, const double* __restrict__ carr) {
    return source_value(q.tb[i], q.te[i], q.term_src, q.term_w, carr);
}
template <typename T>
struct CtSources {
    int32_t blocks = 0;                    // appended workgroups
    InjItems q;
    const int32_t* slice_slot = nullptr;   // per Ct slice: its slot of fbv, or -1 (null: no h sources)
    const int32_t* fb_pos = nullptr;       // per item
    const double* fbv = nullptr;
    const double* carr_step = nullptr;
    T* U = nullptr;
    double* poy_part = nullptr;
};
template <typename T>
__device__ __forceinline__ void ct_source_block(const CtSources<T>& a, int32_t blk, double* red) {
    const int32_t i = blk * kBlock + (int32_t)threadIdx.x;
    double poy = 0;
    if (i < a.q.n) {
        const int32_t e = a.q.edge[i];
        // the Poynting partial uses U before the E update: 0.5*U_old*fb
        if (a.q.kind[i] == 0) poy = 0.5 * (double)a.U[e] * a.fbv[a.fb_pos[i]];
        else a.U[e] = (T)inj_value(a.q, i, a.carr_step);
    }
    const double s = block_sum(poy, red);
    if (threadIdx.x == 0) a.poy_part[blk] = s;
}

// The h values of the first step of a run.
__global__ void __launch_bounds__(kBlock) dga_src_kernel(InjItems q, const int32_t* __restrict__ fb_pos,
                                                         const double* __restrict__ carr, double* __restrict__ fbv) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < q.n && q.kind[i] == 0) fbv[fb_pos[i]] = inj_value(q, i, carr);
}

// Before the loop every source edge takes its e-source sum at t = 0
// (D:746-765), which is 0 on an h edge.
template <typename T>
__global__ void __launch_bounds__(kBlock) dga_init_kernel(InjItems q, const double* __restrict__ carr,
                                                          T* __restrict__ U) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < q.n) U[q.edge[i]] = q.kind[i] == 0 ? (T)0 : (T)inj_value(q, i, carr);
}

// ---- lossy dga: fractional unknowns (D:883-920, tf_dga_frac)
// Sources of a lossy dga step. h edges add their value to curl_f and give the
// first Poynting partial, 0.5*U_old*fb; the other kinds write their value into the
// edge's U_frac entry slot[e] (U_d of a class-4 edge, U_a of a class-1
// edge; none for classes 2/3, whose entries the update rebuilds from their
// old values, D:888-890). With init (the pass before the loop, D:726-790)
// every source edge writes its e-source value at t = 0 (0 unless an e
// source) into all of its fractional entries, half of it into U_c entries
// ([q0, q1)); mu_a / mu_b are the entries of each edge's Mu row.
template <typename T>
__global__ void __launch_bounds__(kBlock) frac_inject_kernel(
    int32_t n_inj, const int32_t* __restrict__ inj_edge, const int8_t* __restrict__ inj_kind,
    const int32_t* __restrict__ inj_tb, const int32_t* __restrict__ inj_te, const int32_t* __restrict__ term_src,
    const double* __restrict__ term_w, const double* __restrict__ carr_step, T* __restrict__ curl_f,
    const T* __restrict__ U, T* __restrict__ Uf, const int32_t* __restrict__ slot, const int32_t* __restrict__ mu_a,
    const int32_t* __restrict__ mu_b, int32_t q0, int32_t q1, double* __restrict__ poy_part, int init) {
    __shared__ double red[kBlock / kWave];
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    double poy = 0;
    if (i < n_inj) {
        const int32_t e = inj_edge[i];
        const double v = source_value(inj_tb[i], inj_te[i], term_src, term_w, carr_step);
        if (init) {
            const double u = inj_kind[i] == 0 ? 0.0 : v;
            for (int32_t c : {mu_a[e], mu_b[e]})
                if (c >= 0) Uf[c] = (T)(c >= q0 && c < q1 ? 0.5 * u : u);
        } else if (inj_kind[i] == 0) {
            curl_f[e] = (T)((double)curl_f[e] + v);
            poy = 0.5 * (double)U[e] * v;
        } else if (slot[e] >= 0) {
            Uf[slot[e]] = (T)v;
        }
    }
    const double s = block_sum(poy, red);
    if (threadIdx.x == 0) poy_part[blockIdx.x] = s;
}

// out[e] = X[a[e]] (+ X[b[e]] when b[e] >= 0) for the n entities of list
// (null: every entity): U = Mu U_frac, F = Tf F_frac (rows of one or two unit
// entries).
template <typename T>
__global__ void __launch_bounds__(kBlock) frac_gather_kernel(int32_t n, const int32_t* __restrict__ list,
                                                             const int32_t* __restrict__ a,
                                                             const int32_t* __restrict__ b, const T* __restrict__ X,
                                                             T* __restrict__ out) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int32_t e = list ? list[i] : i, j = b[e];
    out[e] = j >= 0 ? (T)((double)X[a[e]] + (double)X[j]) : X[a[e]];
}

// Source work taken by workgroups appended to dga_curl_kernel's grid (after
// the face workgroups in logical order), one injection item per thread:
//   mode 1 (dga): the second Poynting half of the step, 0.5 U_new v on the
//     h-source edges, and (fbv) their values of the next step;
//   mode 2 (gfdtd, fem): the step's sources as gf_inject_kernel forms them
//     (fb, dir_new and the Poynting term from U_old).
// One fp64 partial per appended workgroup into poy_part; mode 0: none.
template <typename T>
struct CurlSources {
    int32_t n_inj = 0;
    int32_t mode = 0;
    const int32_t* edge = nullptr;
    const int8_t* kind = nullptr;
    const int32_t* tb = nullptr;
    const int32_t* te = nullptr;
    const int32_t* term_src = nullptr;
    const double* term_w = nullptr;
    const double* carr_step = nullptr;
    const double* carr_prev = nullptr;  // mode 2: the previous step's carriers (null at step 1)
    T* fb = nullptr;
    T* dir_new = nullptr;
    int32_t delta = 0;                  // mode 2, fem: an h edge's forcing is Fb - Fb_old
    double* poy_part = nullptr;
    double* fbv = nullptr;              // mode 1: h values of the next step (CtSources)
    const int32_t* fb_pos = nullptr;
    const double* carr_next = nullptr;
};

// gfdtd sources of one item (D:1478-1502): returns its Poynting term.
template <typename T>
__device__ __forceinline__ double gf_source_item(int32_t i, const int32_t* __restrict__ inj_edge,
                                                 const int8_t* __restrict__ inj_kind, const int32_t* __restrict__ inj_tb,
                                                 const int32_t* __restrict__ inj_te,
                                                 const int32_t* __restrict__ term_src,
                                                 const double* __restrict__ term_w, const double* __restrict__ carr_step,
                                                 const double* __restrict__ carr_prev, T* __restrict__ fb,
                                                 T* __restrict__ dir_new, const T* __restrict__ U, int delta) {
    const int32_t e = inj_edge[i];
    const double v = source_value(inj_tb[i], inj_te[i], term_src, term_w, carr_step);
    if (inj_kind[i] == 0) {
        const double vo = carr_prev ? source_value(inj_tb[i], inj_te[i], term_src, term_w, carr_prev) : 0.0;
        fb[e] = (T)(delta ? v - vo : v);
        return (double)U[e] * (0.5 * (v + vo));
    }
    if (inj_kind[i] == 2) {
        fb[e] = (T)(-v);  // current I at t (D:1491-1492): -dt I joins dt Ctb Fb in Psi
    } else {
        dir_new[e] = (T)v;
    }
    return 0.0;
}

// curl_u = C U (3 signed edges per face), B -= dt*curl_u (D:902-910).
template <typename T>
__global__ void __launch_bounds__(kBlock) dga_curl_kernel(int32_t n_faces, const int32_t* __restrict__ c_col,
                                                          const int8_t* __restrict__ c_sg, const T* __restrict__ U,
                                                          T* __restrict__ curl_u, T* __restrict__ B, double dt,
                                                          const double* __restrict__ face_dt, const CgState* guard,
                                                          CurlSources<T> py) {
    if (!cg_guard_ok(guard)) return;
    // the appended workgroups are the last ones dispatched, spread over the
    // XCDs; the face workgroups keep the XCD-aware map over their own count
    const int face_blocks = (n_faces + kBlock - 1) / kBlock;
    if (py.mode && (int)blockIdx.x >= face_blocks) {
        __shared__ double red[kBlock / kWave];
        const int lb = (int)blockIdx.x;
        const int32_t i = (lb - face_blocks) * kBlock + threadIdx.x;
        double poy = 0;
        if (i < py.n_inj) {
            if (py.mode == 1) {
                if (py.kind[i] == 0) {
                    const int32_t tb = py.tb[i], te = py.te[i];
                    if (py.fbv) {
                        const int32_t at = py.fb_pos[i];
                        poy = 0.5 * (double)U[py.edge[i]] * py.fbv[at];
                        py.fbv[at] = source_value(tb, te, py.term_src, py.term_w, py.carr_next);
                    } else {
                        poy = 0.5 * (double)U[py.edge[i]] *
                              source_value(tb, te, py.term_src, py.term_w, py.carr_step);
                    }
                }
            } else {
                poy = gf_source_item<T>(i, py.edge, py.kind, py.tb, py.te, py.term_src, py.term_w, py.carr_step,
                                        py.carr_prev, py.fb, py.dir_new, U, py.delta);
            }
        }
        const double s = block_sum(poy, red);
        if (threadIdx.x == 0) py.poy_part[lb - face_blocks] = s;
        return;
    }
    const int32_t f = xcd_block_of((int)blockIdx.x, py.mode ? face_blocks : (int)gridDim.x) * kBlock + threadIdx.x;
    if (f >= n_faces) return;
    const int32_t* c = c_col + 3 * (int64_t)f;
    double cu;
    if (c_sg) {
        const int8_t* s = c_sg + 3 * (int64_t)f;
        cu = (double)s[0] * (double)U[c[0]] + (double)s[1] * (double)U[c[1]] + (double)s[2] * (double)U[c[2]];
    } else {
        // every tet face has the fixed pattern +1,-1,+1 on (p0p1, p0p2, p1p2) (D:6345-6352)
        cu = (double)U[c[0]] - (double)U[c[1]] + (double)U[c[2]];
    }
    curl_u[f] = (T)cu;
    B[f] = (T)((double)B[f] - (face_dt ? face_dt[f] : dt) * cu);
}

// ------------------------------------------------------------------ gfdtd
__device__ __forceinline__ double sum_partials(const double* __restrict__ part, int n, double* red) {
    double v = 0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) v += part[i];
    v = block_sum(v, red);
    __shared__ double bcast;
    if (threadIdx.x == 0) bcast = v;
    __syncthreads();
    v = bcast;
    __syncthreads();
    return v;
}

// U[free[k]] = x[k]; Dirichlet edges take their new values.
// U_older (fem, or null): the old U of every written edge is kept first
// (U_older = U_old, D:1764).
template <typename T>
__global__ void gf_scatter_kernel(int32_t n_free, const int32_t* __restrict__ free_edge, const T* __restrict__ x,
                                  T* __restrict__ U, int32_t n_dir, const int32_t* __restrict__ dir_edge,
                                  const T* __restrict__ dir_new, const CgState* guard, T* __restrict__ U_older) {
    if (!cg_guard_ok(guard)) return;
    const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_free) {
        const int32_t e = free_edge[i];
        if (U_older) U_older[e] = U[e];
        U[e] = x[i];
    } else if (i - n_free < n_dir) {
        const int32_t e = dir_edge[i - n_free];
        if (U_older) U_older[e] = U[e];
        U[e] = dir_new[e];
    }
}

// The same in edge order: edge e takes x[edge_row[e]], or its new
// Dirichlet value when edge_row[e] < 0. The free rows are ordered for the
// gathers of the CG, not by edge, so one thread per edge gathers from x and
// writes U (and U_older) in whole cache lines.
template <typename T>
__global__ void gf_scatter_edges_kernel(int32_t n_edges, const int32_t* __restrict__ edge_row,
                                        const T* __restrict__ x, T* __restrict__ U, const T* __restrict__ dir_new,
                                        const CgState* guard, T* __restrict__ U_older) {
    if (!cg_guard_ok(guard)) return;
    const int32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n_edges) return;
    const int32_t r = edge_row[e];
    if (U_older) U_older[e] = U[e];
    U[e] = r >= 0 ? x[r] : dir_new[e];
}

// fem: the vectors the step's initial residual gathers (U = U_old here, Src
// = the Dirichlet values at the new time): free edges W = W2 = U - U_older;
// Dirichlet edges W = 2 U - U_older - Src, W2 = Src - U_older, so that with
// x0 = U_old on the free edges
//   Psi_f - A x0 = 1/dt^2 (E W)_f - 0.5/dt (SigMat W2)_f - (Ct N C U_old)_f
//                  + 1/dt (Ctb (Fb - Fb_old) - I)_f
// without the cancelling 2/dt^2 E U_old - A x0 of the reference's Psi
// (D:1731-1733). guard as in cg_guard_ok.
// One thread per edge; edge_row[e] < 0 marks a Dirichlet edge.
template <typename T>
__global__ void fem_w_kernel(int32_t n_edges, const int32_t* __restrict__ edge_row, const T* __restrict__ U,
                             const T* __restrict__ U_older, const T* __restrict__ src, T* __restrict__ W,
                             T* __restrict__ W2, const CgState* guard) {
    if (!cg_guard_ok(guard)) return;
    const int32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n_edges) return;
    if (edge_row[e] >= 0) {
        const T v = (T)((double)U[e] - (double)U_older[e]);
        W[e] = v;
        W2[e] = v;
    } else {
        const double u = U[e], uo = U_older[e], sv = src[e];
        W[e] = (T)((u - uo) + (u - sv));
        W2[e] = (T)(sv - uo);
    }
}

// gfdtd sources at step i (D:1478-1502): fb, the edge-indexed forcing
// Ctb Fb - I of Psi (h sources at t - dt/2: Fb; j dipoles at t: -I), and
// dir_new (e sources); the Poynting term U_old . 0.5 Ctb (Fb + Fb_old)
// (D:1518) with fb_old from the previous step's carriers. With delta (fem,
// D:1701-1733) an h edge's forcing is Fb - Fb_old.
template <typename T>
__global__ void __launch_bounds__(kBlock) gf_inject_kernel(
    int32_t n_inj, const int32_t* __restrict__ inj_edge, const int8_t* __restrict__ inj_kind,
    const int32_t* __restrict__ inj_tb, const int32_t* __restrict__ inj_te, const int32_t* __restrict__ term_src,
    const double* __restrict__ term_w, const double* __restrict__ carr_step, const double* __restrict__ carr_prev,
    T* __restrict__ fb, T* __restrict__ dir_new, const T* __restrict__ U, double* __restrict__ poy_part,
    const CgState* guard, int delta) {
    if (!cg_guard_ok(guard)) return;
    __shared__ double red[kBlock / kWave];
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    double poy = 0;
    if (i < n_inj)
        poy = gf_source_item<T>(i, inj_edge, inj_kind, inj_tb, inj_te, term_src, term_w, carr_step, carr_prev, fb,
                                dir_new, U, delta);
    const double s = block_sum(poy, red);
    if (threadIdx.x == 0) poy_part[blockIdx.x] = s;
}

// ------------------------------------------------------------------ state
// A field in the caller's numbering and in fp64: out[i] = x[pos[i]] (pos null:
// the same order), and the other way round. The permutation and the conversion
// run here, bound by the gather (161^3 fp64, 300 MB: 1 ms), so that the host
// only receives the bytes.
template <typename T, typename O>
__global__ void __launch_bounds__(kBlock) state_gather_kernel(int64_t n, const int32_t* __restrict__ pos,
                                                              const T* __restrict__ x, O* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = (O)x[pos ? pos[i] : i];
}
template <typename T>
__global__ void __launch_bounds__(kBlock) state_scatter_kernel(int64_t n, const int32_t* __restrict__ pos,
                                                               const double* __restrict__ in, T* __restrict__ x) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) x[pos ? pos[i] : i] = (T)in[i];
}

// ------------------------------------------------------------------ energy
// part[block] = sum over this block's entries of w_i x_i^2 (fp64).
template <typename T>
__global__ void __launch_bounds__(kBlock) weighted_sq_kernel(int64_t n, const T* __restrict__ x,
                                                             const double* __restrict__ w,
                                                             double* __restrict__ part) {
    __shared__ double red[kBlock / kWave];
    double acc = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const double v = (double)x[i];
        acc += w[i] * v * v;
    }
    acc = block_sum(acc, red);
    if (threadIdx.x == 0) part[blockIdx.x] = acc;
}

}  // namespace tfd
