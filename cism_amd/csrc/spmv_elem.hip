// spmv_elem.hip -- FP64 product with an assembled 3-D system in element form.
//
// The assembled Blatter-Pattyn operator is a sum over the elements, and all
// that k_elem computes for one is the factor f = efvs w detJ / vol0 at its 8
// quadrature points: on a rectilinear vertex grid the rest of the element
// matrix follows from the surface and thickness at its four corner columns
// (glissade_velo_higher.F90:8001-8123 with the Jacobian of :6508-6732).  The
// product therefore needs 64 bytes of f per node instead of the 448 of the
// half-stored rows: strain rates at the points, times f, gathered back.
//
// Bound.  At 1024^2 x 11 k_spmv_sym64 (the rows) streams 5.5 GB and re-reads
// partner rows, 9.2 GB in all.  This kernel moves about 1.3 GB and is bound
// by its ~350 FP64 instructions per element at two wavefronts per SIMD.  At
// 512^2 x 11 a product takes about 97 us against 332 us for the rows, and a
// solve 49.3 against 88.9 ms; 8 Picard iterations at 193^2 x 11 with a sliding
// law 70.4 against 104 ms.
//
// Split.  One lane per cell column, marching down the element layers; one
// wavefront per row of 64 cells, EL_J rows per workgroup.  A vertex needs the
// four cells around it: the east neighbour's part comes by a lane shuffle,
// the north neighbour row's through LDS, so a tile of 64 x EL_J cells gives
// 63 x (EL_J - 1) vertices and only its rim cells are computed twice.
//
// Sum factorisation.  On each level the corner values are turned into the
// horizontal derivatives at the Gauss abscissae and the values at the four
// horizontal points (8 numbers per component, used by the layers above and
// below); in a layer, u_x and u_y at the 8 points are two-point
// interpolations of those, and the vertical difference does not depend on
// the vertical abscissa.  The way back is the transpose, so the operator is
// symmetric by construction.
#include "cismgpu_internal.h"

namespace cg {

constexpr int EL_J = 8;

__host__ __device__ inline int elem_tiles_i(const Dims& d) { return (d.nxo + WAVE - 2) / (WAVE - 1); }
__host__ __device__ inline int elem_blocks(const Dims& d) { return elem_tiles_i(d) * ((d.nyo + EL_J - 2) / (EL_J - 1)); }

// Levels per workgroup.  A share of kper levels below the first redoes the
// layer above it, and one workgroup fits a CU, so the time goes as rounds of
// 256 workgroups times layers per workgroup; the smallest product wins (one
// layer stands for the start of a workgroup).
inline int elem_split(const Dims& d) {
    int best = d.nz;
    long long cost = -1;
    for (int kper = d.nz; kper >= 1; --kper) {
        const long long shares = (d.nz + kper - 1) / kper;
        const long long c = (elem_blocks(d) * shares + 255) / 256 * (kper + (shares > 1 ? 2 : 1));
        if (cost < 0 || c < cost) { cost = c; best = kper; }
    }
    return best;
}
inline int elem_parts(const Dims& d, int kper) { return elem_blocks(d) * ((d.nz + kper - 1) / kper); }

// What the short cuts of the assembly rest on, counted: count[0] the vertices
// whose x varies along j or whose y varies along i (the element form needs a
// rectilinear vertex grid), count[1] the owned inactive vertices of active
// cells.  The rows of those are zero (k_rows) while the element form would
// give them their cells' part, and their neighbours' rows couple to them, so
// the matrix is not symmetric off the rim either.
__global__ void k_form_check(Dims d, AsmDev in, unsigned long long* __restrict__ count) {
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    unsigned long long bent = 0, gap = 0;
    if (t < (long long)d.nvx * d.nvy) {
        const long long i0 = t % d.nvx, j0 = t / d.nvx;
        bent = (in.xV[t] != in.xV[i0] || in.yV[t] != in.yV[j0 * d.nvx]) ? 1ull : 0ull;
        const int i = 1 + (int)i0, j = 1 + (int)j0;
        auto cell_on = [&](int ci, int cj) { return cell_in_range(d, in.nhalo, ci, cj) && in.acell[c2(d, ci, cj)]; };
        if (!in.avert[t] && i >= d.ilo && i <= d.ihi && j >= d.jlo && j <= d.jhi)
            gap = (cell_on(i, j) || cell_on(i + 1, j) || cell_on(i, j + 1) || cell_on(i + 1, j + 1)) ? 1ull : 0ull;
    }
    for (int off = WAVE / 2; off > 0; off >>= 1) {
        bent += __shfl_down(bent, off, WAVE);
        gap += __shfl_down(gap, off, WAVE);
    }
    if (threadIdx.x % WAVE == 0 && bent) atomicAdd(count, bent);
    if (threadIdx.x % WAVE == 0 && gap) atomicAdd(count + 1, gap);
}

// Horizontal values of one component on one level: x derivative at the two s
// abscissae, y derivative at the two r abscissae, value at the four points
// (order (-,-), (+,-), (+,+), (-,+)).
struct PlaneQ { double x[2], y[2], v[4]; };

__device__ __forceinline__ void plane_values(double sw, double se, double ne, double nw, double hx2, double hy2,
                                             PlaneQ& p) {
    const double g = 0.57735026918962576451;            // 1 / sqrt(3)
    const double es = se - sw, en = ne - nw;            // differences along the south and north edges
    const double m0 = (se + sw) + (ne + nw), mr = es + en, ms = (ne + nw) - (se + sw), mrs = en - es;
    p.x[0] = hx2 * (mr - g * mrs);                      // hx2 = 1 / (2 hx)
    p.x[1] = hx2 * (mr + g * mrs);
    p.y[0] = hy2 * (ms - g * mrs);
    p.y[1] = hy2 * (ms + g * mrs);
    const double a0 = m0 - g * ms, a1 = m0 + g * ms, b0 = mr - g * mrs, b1 = mr + g * mrs;
    p.v[0] = 0.25 * (a0 - g * b0);
    p.v[1] = 0.25 * (a0 + g * b0);
    p.v[2] = 0.25 * (a1 + g * b1);
    p.v[3] = 0.25 * (a1 - g * b1);
}

// The transpose: corner contributions (sw, se, ne, nw) of the plane duals.
__device__ __forceinline__ void plane_corners(const PlaneQ& p, double hx2, double hy2, double (&c)[4]) {
    const double g = 0.57735026918962576451;
    const double a0 = 0.25 * (p.v[0] + p.v[1]), a1 = 0.25 * (p.v[2] + p.v[3]);
    const double b0 = 0.25 * g * (p.v[1] - p.v[0]) + hx2 * p.x[0], b1 = 0.25 * g * (p.v[2] - p.v[3]) + hx2 * p.x[1];
    const double y0 = hy2 * p.y[0], y1 = hy2 * p.y[1];
    const double m0 = a0 + a1, ms = g * (a1 - a0) + (y0 + y1);
    const double mr = b0 + b1, mrs = g * ((b1 - b0) + (y1 - y0));
    c[0] = (m0 - mr) - (ms - mrs);
    c[1] = (m0 + mr) - (ms + mrs);
    c[2] = (m0 + mr) + (ms + mrs);
    c[3] = (m0 - mr) + (ms - mrs);
}

// MODE 1: y = A x with the (y, x) partials; MODE 2: r = b - A x with the
// (r, r) partials, as the row kernels.  bd: the basal friction term of the
// diagonal at the bed, per vertex.  The rows that the no-ice rule zeroes
// (k_matrix_noice_edge) need no case of their own: where one was not zero
// before, its neighbours still couple to it, the matrix is not symmetric and
// its rows are the only form.
template <int MODE>
__global__ __launch_bounds__(WAVE * EL_J) void k_spmv_elem(Dims d, AsmDev in, const double* __restrict__ E,
                                                           const double* __restrict__ bd,
                                                           const double* __restrict__ xu, const double* __restrict__ xv,
                                                           double* __restrict__ yu, double* __restrict__ yv,
                                                           const double* __restrict__ bu, const double* __restrict__ bv,
                                                           double* __restrict__ partials, int kper) {
    __shared__ double ex[2][2][EL_J][WAVE];
    const int nti = elem_tiles_i(d), nblk = elem_blocks(d);
    const int lin = xcd_remap(blockIdx.x, nblk);
    const int bx = lin % nti, by = lin / nti;
    const int k0 = blockIdx.y * kper, k1 = min(d.nz, k0 + kper);       // the levels of this share
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const int ci = d.ilo + bx * (WAVE - 1) + lane, cj = d.jlo + by * (EL_J - 1) + w;   // cell; its NE vertex is (ci, cj)
    const bool on = ci <= d.ihi + 1 && cj <= d.jhi + 1 && cell_in_range(d, in.nhalo, ci, cj) && in.acell[c2(d, ci, cj)];
    const bool out = lane < WAVE - 1 && w < EL_J - 1 && ci <= d.ihi && cj <= d.jhi;
    const double g = 0.57735026918962576451;
    double kq[4], zx[2], zy[2], tx[2], ty[2], hx2 = 0.0, hy2 = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) kq[q] = 0.0;
#pragma unroll
    for (int q = 0; q < 2; ++q) zx[q] = zy[q] = tx[q] = ty[q] = 0.0;
    long long c00 = 0;                                  // NE vertex of the cell, level 0
    if (on) {
        const long long p = v2(d, ci, cj), nvx = d.nvx;
        hx2 = 0.5 / (in.xV[p] - in.xV[p - 1]);
        hy2 = 0.5 / (in.yV[p] - in.yV[p - nvx]);
        PlaneQ s, h;
        plane_values(in.susrf[p - nvx - 1], in.susrf[p - nvx], in.susrf[p], in.susrf[p - 1], hx2, hy2, s);
        plane_values(in.sthck[p - nvx - 1], in.sthck[p - nvx], in.sthck[p], in.sthck[p - 1], hx2, hy2, h);
#pragma unroll
        for (int q = 0; q < 2; ++q) { zx[q] = s.x[q]; zy[q] = s.y[q]; tx[q] = h.x[q]; ty[q] = h.y[q]; }
#pragma unroll
        for (int q = 0; q < 4; ++q) kq[q] = 1.0 / h.v[q];
        c00 = vidx(d, 0, ci, cj);
    }
    const long long ne = (long long)(d.nz - 1) * d.nx * d.ny;
    const double* F = E + 9 * ne + (on ? elem_id(d, ci, cj, 1) : 0);
    const long long lay = (long long)d.nx * d.ny;
    auto plane = [&](int k, PlaneQ& pu, PlaneQ& pv) {
        double a[4] = {0.0, 0.0, 0.0, 0.0}, b[4] = {0.0, 0.0, 0.0, 0.0};
        if (on) {
            const long long c = c00 + k * d.plane;
            a[0] = xu[c - d.px - 1]; a[1] = xu[c - d.px]; a[2] = xu[c]; a[3] = xu[c - 1];
            b[0] = xv[c - d.px - 1]; b[1] = xv[c - d.px]; b[2] = xv[c]; b[3] = xv[c - 1];
        }
        plane_values(a[0], a[1], a[2], a[3], hx2, hy2, pu);
        plane_values(b[0], b[1], b[2], b[3], hx2, hy2, pv);
    };
    dd acc = {0.0, 0.0};
    // level k is complete: corners to the vertices, south parts to the wave of
    // the row below through LDS (two buffers: one barrier per level)
    auto finish = [&](int k, const PlaneQ& du, const PlaneQ& dv) {
        double cu[4], cv[4];
        plane_corners(du, hx2, hy2, cu);
        plane_corners(dv, hx2, hy2, cv);
        const double nu = cu[2] + __shfl_down(cu[3], 1, WAVE), nv = cv[2] + __shfl_down(cv[3], 1, WAVE);
        const double su = cu[1] + __shfl_down(cu[0], 1, WAVE), sv = cv[1] + __shfl_down(cv[0], 1, WAVE);
        ex[k & 1][0][w][lane] = su;
        ex[k & 1][1][w][lane] = sv;
        __syncthreads();
        if (out) {
            const long long c = vidx(d, k, ci, cj);
            double au = nu + ex[k & 1][0][w + 1][lane], av = nv + ex[k & 1][1][w + 1][lane];
            const double x0 = xu[c], x1 = xv[c];
            if (k == d.nz - 1) {
                const double s = bd[v2(d, ci, cj)];
                au = au + s * x0;
                av = av + s * x1;
            }
            if (MODE == 2) {
                const double r0 = bu[c] - au, r1 = bv[c] - av;
                yu[c] = r0;
                yv[c] = r1;
                acc = dd_add_d(acc, r0 * r0);
                acc = dd_add_d(acc, r1 * r1);
            } else {
                yu[c] = au;
                yv[c] = av;
                acc = dd_add_d(acc, au * x0);
                acc = dd_add_d(acc, av * x1);
            }
        }
    };
    PlaneQ Uu, Uv, Du, Dv;                              // upper level's values, and its duals so far
    const int ks = max(k0 - 1, 0);
    plane(ks, Uu, Uv);
#pragma unroll
    for (int q = 0; q < 2; ++q) Du.x[q] = Du.y[q] = Dv.x[q] = Dv.y[q] = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) Du.v[q] = Dv.v[q] = 0.0;
    const double wa = 0.5 * (1.0 + g), wb = 0.5 * (1.0 - g);   // weights of the near and far level at a point
#pragma unroll 1
    for (int k = ks; k < k1 && k + 1 < d.nz; ++k) {     // element layer between levels k and k + 1
        double f[8];
#pragma unroll
        for (int p = 0; p < 8; ++p) f[p] = on ? F[(long long)p * EQ * ne + k * lay] : 0.0;
        PlaneQ Lu, Lv, Eu, Ev;                          // lower level's values and duals
        plane(k + 1, Lu, Lv);
        const double s0 = in.sigma[k], s1 = in.sigma[k + 1], kz = 1.0 / (s1 - s0);
#pragma unroll
        for (int q = 0; q < 2; ++q) Eu.x[q] = Eu.y[q] = Ev.x[q] = Ev.y[q] = 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {                   // horizontal point (ri, si)
            const int ri = (q == 1 || q == 2) ? 1 : 0, si = q >= 2 ? 1 : 0;
            const double kk = kz * kq[q];
            const double uz = kk * (Uu.v[q] - Lu.v[q]), vz = kk * (Uv.v[q] - Lv.v[q]);
            double Gu = 0.0, Gv = 0.0;
#pragma unroll
            for (int t = 0; t < 2; ++t) {               // 0: lower point, 1: upper
                const double a = t ? wa : wb, b = t ? wb : wa;
                const double sg = a * s0 + b * s1;
                const double ax = zx[si] - sg * tx[si], ay = zy[ri] - sg * ty[ri];
                const double ux = (a * Uu.x[si] + b * Lu.x[si]) - ax * uz, uy = (a * Uu.y[ri] + b * Lu.y[ri]) - ay * uz;
                const double vx = (a * Uv.x[si] + b * Lv.x[si]) - ax * vz, vy = (a * Uv.y[ri] + b * Lv.y[ri]) - ay * vz;
                const double ff = f[q + 4 * t], f2 = 2.0 * ff;
                const double Fx = f2 * (2.0 * ux + vy), Fy = f2 * (2.0 * vy + ux), S = ff * (uy + vx);
                Gu += ff * uz - ax * Fx - ay * S;
                Gv += ff * vz - ax * S - ay * Fy;
                Du.x[si] += a * Fx; Eu.x[si] += b * Fx;
                Du.y[ri] += a * S;  Eu.y[ri] += b * S;
                Dv.x[si] += a * S;  Ev.x[si] += b * S;
                Dv.y[ri] += a * Fy; Ev.y[ri] += b * Fy;
            }
            Gu *= kk;
            Gv *= kk;
            Du.v[q] += Gu; Eu.v[q] = -Gu;
            Dv.v[q] += Gv; Ev.v[q] = -Gv;
        }
        if (k >= k0) finish(k, Du, Dv);
        Du = Eu; Dv = Ev; Uu = Lu; Uv = Lv;
    }
    if (k1 == d.nz) finish(d.nz - 1, Du, Dv);
    dd v[1] = {acc};
    block_reduce_dd<1, WAVE * EL_J>(v);
    if (threadIdx.x == 0) {
        partials[2 * (blockIdx.y * nblk + lin) + 0] = v[0].hi;
        partials[2 * (blockIdx.y * nblk + lin) + 1] = v[0].lo;
    }
}

}  // namespace cg
