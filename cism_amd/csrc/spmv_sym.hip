// spmv_sym.hip -- half-storage SpMV for the inner FP32 iterations.
//
// The assembled operator is symmetric: Auu = Auu^T, Avv = Avv^T, Auv = Avu^T
// (glissade_velo_higher.F90:10859-10864), so of the 27 neighbour couplings
// of a node only the centre and the 13 "upper" ones (m = 14..27 in the
// reference numbering, 0-based 13..26) need storing; the coupling of node r
// to its lower neighbour q = r + off(m), m < 13, is the transposed 2x2
// block of q's upper coupling 26 - m.  Storage (per owned row r, slot
// s = m - 13 for m >= 13):
//     Sq[((r/64)*14 + s)*256 + (r%64)*4 + c]
// slot 0 holds (uu, uv, vv, 0) of the centre, slots 1..13 the quads
// (uu, uv, vu, vv) of the upper couplings, so the matrix streams 224 B per
// node instead of 432.
//
// k_spmv_sym walks a column up the levels like k_spmv_q and loads the 13
// lower quads from the partner rows; k_spmv_symj (large grids) forms both
// products of a slot where it is read and passes the lower one on.  The
// products and their association (node_sum) are those of the full-storage
// kernel, so when the FP32 matrix is exactly symmetric (k_check_sym finds no
// mismatch) all three kernels give identical results; the solver uses this
// layout only then.  x is staged in LDS per tile with a one-vertex ring.
//
// Partner offsets within a level are 32-bit (po[] below): the half layouts
// are used only while one level of slots, nyo * nxp * 56 elements, stays
// below 2^31 (half_storage_fits); larger grids keep the full-row kernels.
#include "cismgpu_internal.h"

namespace cg {

constexpr int NSLOT = 14;

inline bool half_storage_fits(const Dims& d) {
    return (long long)d.nyo * d.nxp * NSLOT * 4 < (1LL << 31);
}

// partner column of row (i, j) at horizontal offset (iA, jA): its owned
// image (periodic rules) as jo*nxp + io, or -1 if it has no stored row
__device__ __forceinline__ int partner_col(const Dims& d, int i, int j) {
    if (!row_image(d, i, j)) return -1;
    return (j - d.jlo) * d.nxp + (i - d.ilo);
}

// Half-storage copy of the owned rows of the FP64 row-blocked matrix.
template <typename TA>
__global__ void k_convert_sym(long long nrows, const double* __restrict__ src, TA* __restrict__ dst) {
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;   // over nrows * 14 * 4
    if (t >= nrows * NSLOT * 4) return;
    const int c = (int)(t % 4);
    const long long u = t / 4;
    const int lane = (int)(u % WAVE);
    const long long v = u / WAVE;
    const int s = (int)(v % NSLOT);
    const long long rb = v / NSLOT;
    const double* row = src + rb * NCOEF * WAVE + lane;
    double val;
    if (s == 0) {   // centre: uu, uv, vv, 0
        const int blk = c == 0 ? 0 : (c == 1 ? 1 : 3);
        val = c == 3 ? 0.0 : row[(blk * 27 + 13) * WAVE];
    } else {
        val = row[(c * 27 + 13 + s) * WAVE];
    }
    dst[t] = to_lowp<TA>(val);
}

// Counts the couplings that the half storage cannot reproduce exactly in
// precision TA (float or double): a lower coupling whose transposed partner differs, a
// nonzero coupling to a node without a stored row, or Auv != Avu at the
// centre.  count[0] += mismatches.
template <typename TA>
__global__ void k_check_sym(Dims d, const double* __restrict__ A, unsigned long long* __restrict__ count) {
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    unsigned long long bad = 0;
    if (t < d.nrows) {
        const int io = (int)(t % d.nxp);
        const long long kj = t / d.nxp;
        const int jo = (int)(kj % d.nyo), k0 = (int)(kj / d.nyo);
        if (io < d.nxo) {
            const int i = d.ilo + io, j = d.jlo + jo;
            const double* a = A + ((t / WAVE) * NCOEF) * WAVE + (t % WAVE);
            auto rd = [](double x) { return to_lowp<TA>(x); };
            if (rd(a[(1 * 27 + 13) * WAVE]) != rd(a[(2 * 27 + 13) * WAVE])) ++bad;
            for (int m = 0; m < 13; ++m) {
                const int iA = m % 3 - 1, jA = (m / 3) % 3 - 1, kA = m / 9 - 1;
                if (k0 + kA < 0) continue;                   // stored as zero
                const double c0 = a[(0 * 27 + m) * WAVE], c1 = a[(1 * 27 + m) * WAVE];
                const double c2_ = a[(2 * 27 + m) * WAVE], c3 = a[(3 * 27 + m) * WAVE];
                int qi = i + iA, qj = j + jA;
                if (!row_image(d, qi, qj)) {
                    bad += (c0 != 0.0 || c1 != 0.0 || c2_ != 0.0 || c3 != 0.0) ? 1 : 0;
                    continue;
                }
                const double* q = row_ptr(d, A, k0 + kA, qi, qj);
                const int mm = 26 - m;
                if (rd(c0) != rd(q[(0 * 27 + mm) * WAVE]) || rd(c1) != rd(q[(2 * 27 + mm) * WAVE]) ||
                    rd(c2_) != rd(q[(1 * 27 + mm) * WAVE]) || rd(c3) != rd(q[(3 * 27 + mm) * WAVE]))
                    ++bad;
            }
        }
    }
    for (int off = WAVE / 2; off > 0; off >>= 1) bad += __shfl_down(bad, off, WAVE);
    if (threadIdx.x % WAVE == 0 && bad) atomicAdd(count, bad);
}

__device__ __forceinline__ void ld_slot(const float* p, float& a, float& b, float& c, float& e) { ld_quad(p, a, b, c, e); }

template <typename TA, int MODE>
__global__ __launch_bounds__(256, 4) void k_spmv_sym(Dims d, const TA* __restrict__ S, const float* __restrict__ xu,
                                                  const float* __restrict__ xv, float* __restrict__ yu,
                                                  float* __restrict__ yv, const float* __restrict__ bu,
                                                  const float* __restrict__ bv, double* __restrict__ partials,
                                                  int kper) {
    const int k0 = blockIdx.y * kper, k1 = min(d.nz, k0 + kper);   // the levels of this share
    // x of the tile (64 x 4 columns) plus a one-column ring, for levels k-1,
    // k, k+1, staged in LDS (a 3-level ring)
    __shared__ float xs[2][3][6][WAVE + 2];
    const int nbx = d.nxp / WAVE;
    const int nblk = nbx * ((d.nyo + 3) / 4);
    const int lin = xcd_remap(blockIdx.x, nblk);     // neighbouring tiles share an XCD's L2
    const int bx = lin % nbx, by = lin / nbx;
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const int io = bx * WAVE + lane;
    const int jo = by * 4 + w;
    const bool live = io < d.nxo && jo < d.nyo;
    const int i0 = d.ilo + bx * WAVE - 1, j0 = d.jlo + by * 4 - 1;   // vertex of xs[.][.][0][0]
    const long long pl = d.plane;
    // stage level kk (-1..nz) of x into ring slot kk+1 mod 3
    auto stage = [&](int kk) {
        const int slot = (kk + 1) % 3;
        for (int e = threadIdx.x; e < 6 * (WAVE + 2); e += 256) {
            const int r = e / (WAVE + 2), c = e % (WAVE + 2);
            const int vi = i0 + c, vj = j0 + r;
            float a = 0.f, b = 0.f;
            if (vi >= 1 && vi <= d.nvx && vj >= 1 && vj <= d.nvy) {
                const long long n = vidx(d, kk, vi, vj);
                a = xu[n];
                b = xv[n];
            }
            xs[0][slot][r][c] = a;
            xs[1][slot][r][c] = b;
        }
    };
    dd acc = {0.0, 0.0};
    int po[9];
    const long long LS = (long long)d.nyo * d.nxp / WAVE * (NSLOT * 4 * WAVE);   // elements per level
    if (live) {
        const int i = d.ilo + io, j = d.jlo + jo;
        // element offsets of the partner rows' slot 0 within a level, -1 when
        // the neighbour has no stored row; rows per level are a multiple of 64
#pragma unroll
        for (int h = 0; h < 9; ++h) {
            const int pc = partner_col(d, i + h % 3 - 1, j + h / 3 - 1);
            po[h] = pc < 0 ? -1 : (pc / WAVE) * (NSLOT * 4 * WAVE) + (pc % WAVE) * 4;
        }
    }
    stage(k0 - 1);
    stage(k0);
    for (int k = k0; k < k1; ++k) {
        stage(k + 1);
        __syncthreads();
        if (live) {
            const long long ck = vidx(d, k, d.ilo + io, d.jlo + jo);
            const TA* Sk = S + (long long)k * LS;     // level k
            const TA* Sb = Sk - LS;                   // level k - 1
            const float2 y = node_sum([&](int m, float2& g) {
                float cuu, cuv, cvu, cvv;
                if (m < 13) {
                    const int h = m % 9;
                    if (!(po[h] >= 0 && (m >= 9 || k > 0))) return;
                    float a, b, c, e;
                    ld_slot((m < 9 ? Sb : Sk) + po[h] + (13 - m) * (4 * WAVE), a, b, c, e);
                    cuu = a; cuv = c; cvu = b; cvv = e;     // transposed 2x2 block
                } else if (m == 13) {
                    float a, b, c, e;
                    ld_slot(Sk + po[4], a, b, c, e);
                    cuu = a; cuv = b; cvu = b; cvv = c;
                } else {
                    ld_slot(Sk + po[4] + (m - 13) * (4 * WAVE), cuu, cuv, cvu, cvv);
                }
                const int slot = (k + m / 9) % 3;              // level k + kA lives in slot (k + kA + 1) % 3
                const int r = w + 1 + ((m / 3) % 3 - 1), c = lane + 1 + (m % 3 - 1);
                g = add2(g, prod2(cuu, cuv, cvu, cvv, xs[0][slot][r][c], xs[1][slot][r][c]));
            });
            const float su = y.x, sv = y.y;
            if (MODE == 2) {
                const float ru = bu[ck] - su, rv = bv[ck] - sv;
                yu[ck] = ru;
                yv[ck] = rv;
                acc = dd_add_d(acc, dot2(ru, ru, rv, rv));
            } else {
                yu[ck] = su;
                yv[ck] = sv;
                if (MODE == 1) {
                    const int slot = (k + 1) % 3;
                    acc = dd_add_d(acc, dot2(su, xs[0][slot][w + 1][lane + 1], sv, xs[1][slot][w + 1][lane + 1]));
                }
            }
        }
        __syncthreads();   // the slot of level k-1 is restaged next
    }
    if (MODE != 0) {
        dd v[1] = {acc};
        block_reduce_dd<1, 256>(v);
        if (threadIdx.x == 0) {
            partials[2 * (blockIdx.y * nblk + lin) + 0] = v[0].hi;
            partials[2 * (blockIdx.y * nblk + lin) + 1] = v[0].lo;
        }
    }
}

// FP32 half storage, every slot read once.  A row's stored couplings serve two
// rows: its own sum, and the transposed block in the sum of the row it couples
// to.  Here the row that holds a slot forms both products and passes the two
// numbers on, instead of the other row fetching the four again: k_spmv_sym
// reads 4.1 GB a product at 1024^2 x 11, of 2.8 GB of slots and vectors.
//
// A workgroup takes 64 columns of a vertex row (lanes) on all levels (one
// wavefront each, at most SJ_WAVES; deeper columns are cut into shares, whose
// first wavefront recomputes the level above) and marches along j.  Products
// for the neighbouring lanes go by shuffle, for the next vertex row they stay
// in registers, for the level below they go through LDS (three pairs per lane
// and step, two buffers, one barrier per step).  What remains to be read twice
// are the columns next to the tile (five slots of one lane, four of another,
// per row) and one ghost row before and after the march; the march before,
// along the levels, re-read a tile's rim on every level.  A row waits one step
// for the products of the next row on the level above.
//
// At 1024^2 x 11 a product takes 561 us (4.94 TB/s of slots and vectors)
// against 691 us for k_spmv_sym and 651 us for the march along the levels that
// this replaced; 571 us with all loads of a row issued after the last one's
// products, 193^2 x 11 24.8 against 28.9 us.
//
// x of rows j-1 .. j+1 is in LDS, a ring of four rows.  Sums are associated as
// in the other FP32 products (node_sum), so the results are the same bits.
// Columns without a stored row (outside the owned region) hold zero slots; the
// image of a periodic neighbour is read where the shuffle has another row.
constexpr int SJ_WAVES = 12;

struct SjCut { int nj, jper, nk, kper, waves; };   // shares along j and k; wavefronts per workgroup

// 12 wavefronts with 168 registers fit a CU: the number of shares along j that
// takes the fewest steps in all, with two ghost rows per share.
inline SjCut symj_cut(const Dims& d) {
    SjCut c{};
    c.nk = d.nz <= SJ_WAVES ? 1 : (d.nz + SJ_WAVES - 2) / (SJ_WAVES - 1);
    c.kper = (d.nz + c.nk - 1) / c.nk;
    c.nk = (d.nz + c.kper - 1) / c.kper;
    c.waves = c.kper + (c.nk > 1 ? 1 : 0);
    const long long nb = (long long)(d.nxp / WAVE) * c.nk;
    const int per_cu = SJ_WAVES / c.waves;
    long long best = -1;
    for (int jper = d.nyo; jper >= 4 || jper == d.nyo; --jper) {
        const int nj = (d.nyo + jper - 1) / jper;
        const long long cost = (nb * nj + 256 * per_cu - 1) / (256 * per_cu) * (jper + 2);
        if (best < 0 || cost < best) { best = cost; c.jper = jper; c.nj = nj; }
        if (jper <= 1) break;
    }
    return c;
}
inline bool symj_fits(const Dims& d) { return (long long)d.nyo * d.nxp * NSLOT * 16 < (1LL << 31); }
inline int symj_blocks(const Dims& d, const SjCut& c) { return (d.nxp / WAVE) * c.nj * c.nk; }
inline size_t symj_lds(const SjCut& c) {
    return sizeof(float2) * (4 * (c.waves + 1) * (WAVE + 2) + 2 * 3 * c.waves * WAVE);
}

template <int MODE>
__global__ __launch_bounds__(WAVE * SJ_WAVES) void k_spmv_symj(Dims d, const float* __restrict__ S,
                                                               const float* __restrict__ xu, const float* __restrict__ xv,
                                                               float* __restrict__ yu, float* __restrict__ yv,
                                                               const float* __restrict__ bu, const float* __restrict__ bv,
                                                               double* __restrict__ partials, int jper, int kper) {
    extern __shared__ float2 sj_lds[];
    const int nw = blockDim.x / WAVE;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    auto xs = [&](int q, int l, int c) -> float2& {       // row q (ring of 4), level index l, column c - 1 of the tile
        return sj_lds[((q & 3) * (nw + 1) + l) * (WAVE + 2) + c];
    };
    float2* ex = sj_lds + 4 * (nw + 1) * (WAVE + 2);      // [2][3][nw][64]
    const int nbx = d.nxp / WAVE;
    const int lin = xcd_remap(blockIdx.x, gridDim.x);
    const int bx = lin % nbx, jt = lin / nbx;
    const int kc0 = blockIdx.y * kper, ghost = kc0 > 0 ? 1 : 0;
    const int kend = min(d.nz, kc0 + kper);
    const int k = kc0 - ghost + w;                        // level of this wavefront
    const bool kon = k < kend;
    const int io = bx * WAVE + lane, i = d.ilo + io;
    const bool live = io < d.nxo && kon;
    const int q0 = jt * jper, q1 = min(d.nyo, q0 + jper);
    const bool edge_l = lane == 0, edge_r = lane == WAVE - 1;
    const long long LS = (long long)d.nyo * d.nxp / WAVE * (NSLOT * 4 * WAVE);
    const float* Sk = S + (long long)(kon ? k : 0) * LS;
    // raw buffer over the level's slots (below 2 GiB, symj_fits): a load past
    // it reads zero, which is what a row that is not stored holds
    constexpr unsigned NONE = 0x80000000u;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)Sk, (short)0, (int)(LS * 4), 0x00020000);
    auto offset = [&](int col) { return col < 0 ? NONE : (unsigned)((col / WAVE) * (NSLOT * 4 * WAVE) + (col % WAVE) * 4) * 4u; };
    auto slot = [&](unsigned off, int s) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rs, off, s * (4 * WAVE * 4), 0);
        return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
    };
    float4 own[NSLOT], ed[5];
    // Offsets of row q's slots (o*: the ghost rows give only the slots that
    // couple into the share) and of the column next to the tile.
    unsigned of = NONE, ob = NONE, oo = NONE, oe = NONE;
    auto locate = [&](int q) {
        // the lane past the last owned column holds the row beyond it, if there is one (periodic)
        const unsigned o = offset(io <= d.nxo && kon && q <= q1 ? partner_col(d, i, d.jlo + q) : -1);
        of = q >= q1 ? NONE : o;
        ob = q < q0 ? NONE : o;
        oo = q < q0 ? NONE : of;
        // left: slots 1, 4, 7, 10, 13 of column i - 1 (coupling to i), right: 2, 5, 8, 11 of column i + 1
        const int ec = live && (edge_l || edge_r) && q <= q1 ? partner_col(d, edge_l ? i - 1 : i + 1, d.jlo + q) : -1;
        oe = ec < 0 ? NONE : offset(ec) + (edge_l ? 1u : 2u) * (4 * WAVE * 4);
    };
    auto refill = [&](int s) { own[s] = slot((s >= 2 && s <= 4) || s >= 11 ? of : s >= 5 && s <= 7 ? ob : oo, s); };
    auto refill_edge = [&](int e) { ed[e] = slot(e == 4 && !edge_l ? NONE : oe, 3 * e); };
    // x of row q, levels kl0 .. kl0 + nw, into LDS: at most XST values a thread
    constexpr int XST = 2;                 // (nw + 1) * 66 <= 2 * 64 * nw from two wavefronts on
    const int nst = (nw + 1) * (WAVE + 2);
    const int ci0 = d.ilo + bx * WAVE - 1, kl0 = kc0 - ghost;
    float2 xr_[XST];
    auto fetch = [&](int q) {
        const int vj = d.jlo + q;
#pragma unroll
        for (int u = 0; u < XST; ++u) {
            const int e = threadIdx.x + u * blockDim.x;
            const int l = e / (WAVE + 2), c = e % (WAVE + 2), vi = ci0 + c;
            xr_[u] = make_float2(0.f, 0.f);
            if (e < nst && vi >= 1 && vi <= d.nvx && vj >= 1 && vj <= d.nvy && kl0 + l <= d.nz) {
                const long long n = vidx(d, kl0 + l, vi, vj);
                xr_[u] = make_float2(xu[n], xv[n]);
            }
        }
    };
    auto put = [&](int q) {
#pragma unroll
        for (int u = 0; u < XST; ++u) {
            const int e = threadIdx.x + u * blockDim.x;
            if (e < nst) xs(q, e / (WAVE + 2), e % (WAVE + 2)) = xr_[u];
        }
    };
    auto prod = [](float cuu, float cuv, float cvu, float cvv, float2 x) { return prod2(cuu, cuv, cvu, cvv, x.x, x.y); };
    auto up = [&](float2 v) { return make_float2(__shfl_up(v.x, 1, WAVE), __shfl_up(v.y, 1, WAVE)); };
    auto down = [&](float2 v) { return make_float2(__shfl_down(v.x, 1, WAVE), __shfl_down(v.y, 1, WAVE)); };
    dd acc = {0.0, 0.0};
    float2 pend = make_float2(0.f, 0.f), xp = pend, Bp = pend, Ep = pend;
    for (int q = q0 - 2; q <= q0; ++q) {
        fetch(q);
        put(q);
    }
    locate(q0 - 1);
#pragma unroll
    for (int s = 0; s < NSLOT; ++s) refill(s);
#pragma unroll
    for (int e = 0; e < 5; ++e) refill_edge(e);
    __syncthreads();
    // Each group of slots is refilled with the next row's as soon as its
    // products are fixed, so loads are under way through the whole step; the
    // x row, whose LDS write must not wait for them, is fetched before.  The
    // barriers keep the compiler from moving the products below the loads
    // (and spilling the slots).
#define SJ_FIX(v) asm volatile("" : "+v"(v.x), "+v"(v.y))
#define SJ_FENCE __builtin_amdgcn_sched_barrier(0)
#pragma unroll 1
    for (int q = q0 - 1; q <= q1; ++q) {
        fetch(q + 2);
        locate(q + 1);
        const float2 x0 = xs(q, w, lane + 1);
        const float2 xl = xs(q, w, lane), xr = xs(q, w, lane + 2);
        auto c = [&](int s, int r, int l, int di) {        // own product
            return prod(own[s].x, own[s].y, own[s].z, own[s].w, xs(q + r, w + l, lane + 1 + di));
        };
        auto t = [&](float4 s, float2 x) { return prod(s.x, s.z, s.y, s.w, x); };   // transposed
        auto from_l = [&](int s, int e) {  // the column i - 1's product for this column
            const float2 v = up(t(own[s], x0)), m = t(ed[e], xl);
            return edge_l ? m : v;
        };
        auto from_r = [&](int s, int e) {  // the column i + 1's
            const float2 v = down(t(own[s], x0)), m = t(ed[e], xr);
            return edge_r ? m : v;
        };
        float2 U = prod(own[0].x, own[0].y, own[0].y, own[0].z, x0);
        U = add2(U, prod(own[1].x, own[1].y, own[1].z, own[1].w, xr));
        float2 L = from_l(1, 0);
        SJ_FIX(U); SJ_FIX(L); SJ_FENCE;
        refill(0); refill(1);
        SJ_FENCE;
        // row j + 1, this level
        U = add2(U, add2(add2(c(2, 1, 0, -1), c(3, 1, 0, 0)), c(4, 1, 0, 1)));
        float2 B = add2(add2(from_l(4, 1), t(own[3], x0)), from_r(2, 0));
        SJ_FIX(U); SJ_FIX(B); SJ_FENCE;
        refill(2); refill(3); refill(4); refill_edge(0);
        SJ_FENCE;
        // row j - 1, level k + 1
        U = add2(U, add2(add2(c(5, -1, 1, -1), c(6, -1, 1, 0)), c(7, -1, 1, 1)));
        float2 C = add2(add2(from_l(7, 2), t(own[6], x0)), from_r(5, 1));
        SJ_FIX(U); SJ_FIX(C); SJ_FENCE;
        refill(5); refill(6); refill(7); refill_edge(1);
        SJ_FENCE;
        // row j, level k + 1
        U = add2(U, add2(add2(c(8, 0, 1, -1), c(9, 0, 1, 0)), c(10, 0, 1, 1)));
        float2 D = add2(add2(from_l(10, 3), t(own[9], x0)), from_r(8, 2));
        SJ_FIX(U); SJ_FIX(D); SJ_FENCE;
        refill(8); refill(9); refill(10); refill_edge(2);
        SJ_FENCE;
        // row j + 1, level k + 1
        U = add2(U, add2(add2(c(11, 1, 1, -1), c(12, 1, 1, 0)), c(13, 1, 1, 1)));
        float2 E = add2(add2(from_l(13, 4), t(own[12], x0)), from_r(11, 3));
        const float2 V = add2(U, L);
        SJ_FIX(U); SJ_FIX(E); SJ_FENCE;
        refill(11); refill(12); refill(13); refill_edge(3); refill_edge(4);
        SJ_FENCE;
        float2* out = ex + (q & 1) * 3 * nw * WAVE + w * WAVE + lane;
        out[0] = C;
        out[nw * WAVE] = D;
        out[2 * nw * WAVE] = E;
        put(q + 2);
        __syncthreads();
        float2 Ci = make_float2(0.f, 0.f), Di = Ci, Ei = Ci;
        if (w > 0) {
            const float2* in = ex + (q & 1) * 3 * nw * WAVE + (w - 1) * WAVE + lane;
            Ci = in[0];
            Di = in[nw * WAVE];
            Ei = in[2 * nw * WAVE];
        }
        if (q > q0 && live && w >= ghost) {               // row q - 1 is complete
            const float2 y = add2(pend, Ci);
            const long long ck = vidx(d, k, i, d.jlo + q - 1);
            if (MODE == 2) {
                const float ru = bu[ck] - y.x, rv = bv[ck] - y.y;
                yu[ck] = ru;
                yv[ck] = rv;
                acc = dd_add_d(acc, dot2(ru, ru, rv, rv));
            } else {
                yu[ck] = y.x;
                yv[ck] = y.y;
                if (MODE == 1) {
                    acc = dd_add_d(acc, dot2(y.x, xp.x, y.y, xp.y));
                }
            }
        }
        pend = add2(add2(add2(V, Bp), Ep), Di);
        Bp = B;
        Ep = Ei;
        xp = x0;
    }
#undef SJ_FIX
#undef SJ_FENCE
    if (MODE != 0) {
        // one sum over the wavefronts, in wavefront order
        __shared__ dd sh[SJ_WAVES];
        for (int off = WAVE / 2; off > 0; off >>= 1) acc = dd_add(acc, dd_shfl_down(acc, off));
        if (lane == 0) sh[w] = acc;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int u = 1; u < nw; ++u) acc = dd_add(acc, sh[u]);
            const int b = blockIdx.y * gridDim.x + lin;
            partials[2 * b + 0] = acc.hi;
            partials[2 * b + 1] = acc.lo;
        }
    }
}

// FP64 half storage: the same slots with double quads,
//     Sd[((r/64)*14 + s)*256 + (r%64)*4 + c]
// (448 B per node instead of 864), for the FP64 solves when the FP64 matrix
// is exactly symmetric.  Sums in the order and with the values of k_spmv,
// so the results are identical.
__global__ void k_convert_sym64(long long nrows, const double* __restrict__ src, double* __restrict__ dst) {
    const long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    if (t >= nrows * NSLOT * 4) return;
    const int c = (int)(t % 4);
    const long long u = t / 4;
    const int lane = (int)(u % WAVE);
    const long long v = u / WAVE;
    const int s = (int)(v % NSLOT);
    const long long rb = v / NSLOT;
    const double* row = src + rb * NCOEF * WAVE + lane;
    double val;
    if (s == 0) {
        const int blk = c == 0 ? 0 : (c == 1 ? 1 : 3);
        val = c == 3 ? 0.0 : row[(blk * 27 + 13) * WAVE];
    } else {
        val = row[(c * 27 + 13 + s) * WAVE];
    }
    dst[t] = val;
}

__device__ __forceinline__ void ld_slot64(const double* p, double& a, double& b, double& c, double& e) {
    const double2 q0 = *reinterpret_cast<const double2*>(p);
    const double2 q1 = *reinterpret_cast<const double2*>(p + 2);
    a = q0.x; b = q0.y; c = q1.x; e = q1.y;
}

// Whole columns (SPLIT false) have a kernel of their own: with the first level
// and the share in variables it takes 114 registers for 98, and 384^2 x 24
// 462 us for 444, 640^2 x 11 538 for 524.
template <int MODE, bool SPLIT>
__global__ __launch_bounds__(256) void k_spmv_sym64(Dims d, const double* __restrict__ S,
                                                    const double* __restrict__ xu, const double* __restrict__ xv,
                                                    double* __restrict__ yu, double* __restrict__ yv,
                                                    const double* __restrict__ bu, const double* __restrict__ bv,
                                                    double* __restrict__ partials, int kper) {
    const int k0 = SPLIT ? blockIdx.y * kper : 0, k1 = SPLIT ? min(d.nz, k0 + kper) : d.nz;   // the levels of this share
    __shared__ double xs[2][3][6][WAVE + 2];
    const int nbx = d.nxp / WAVE;
    const int nblk = nbx * ((d.nyo + 3) / 4);
    const int lin = xcd_remap(blockIdx.x, nblk);
    const int bx = lin % nbx, by = lin / nbx;
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const int io = bx * WAVE + lane;
    const int jo = by * 4 + w;
    const bool live = io < d.nxo && jo < d.nyo;
    const int i0 = d.ilo + bx * WAVE - 1, j0 = d.jlo + by * 4 - 1;
    auto stage = [&](int kk) {
        const int slot = (kk + 1) % 3;
        for (int e = threadIdx.x; e < 6 * (WAVE + 2); e += 256) {
            const int r = e / (WAVE + 2), c = e % (WAVE + 2);
            const int vi = i0 + c, vj = j0 + r;
            double a = 0.0, b = 0.0;
            if (vi >= 1 && vi <= d.nvx && vj >= 1 && vj <= d.nvy) {
                const long long n = vidx(d, kk, vi, vj);
                a = xu[n];
                b = xv[n];
            }
            xs[0][slot][r][c] = a;
            xs[1][slot][r][c] = b;
        }
    };
    dd acc = {0.0, 0.0};
    int po[9];
    const long long LS = (long long)d.nyo * d.nxp / WAVE * (NSLOT * 4 * WAVE);
    if (live) {
        const int i = d.ilo + io, j = d.jlo + jo;
#pragma unroll
        for (int h = 0; h < 9; ++h) {
            const int pc = partner_col(d, i + h % 3 - 1, j + h / 3 - 1);
            po[h] = pc < 0 ? -1 : (pc / WAVE) * (NSLOT * 4 * WAVE) + (pc % WAVE) * 4;
        }
    }
    stage(k0 - 1);
    stage(k0);
    for (int k = k0; k < k1; ++k) {
        stage(k + 1);
        __syncthreads();
        if (live) {
            const long long ck = vidx(d, k, d.ilo + io, d.jlo + jo);
            const double* Sk = S + (long long)k * LS;
            const double* Sb = Sk - LS;
            double su = 0.0, sv = 0.0;
#pragma unroll
            for (int m = 0; m < 27; ++m) {
                double cuu = 0.0, cuv = 0.0, cvu = 0.0, cvv = 0.0;
                bool have = true;
                if (m < 13) {
                    const int h = m % 9;
                    have = po[h] >= 0 && (m >= 9 || k > 0);
                    if (have) {
                        double a, b, c, e;
                        ld_slot64((m < 9 ? Sb : Sk) + po[h] + (13 - m) * (4 * WAVE), a, b, c, e);
                        cuu = a; cuv = c; cvu = b; cvv = e;
                    }
                } else if (m == 13) {
                    double a, b, c, e;
                    ld_slot64(Sk + po[4], a, b, c, e);
                    cuu = a; cuv = b; cvu = b; cvv = c;
                } else {
                    ld_slot64(Sk + po[4] + (m - 13) * (4 * WAVE), cuu, cuv, cvu, cvv);
                }
                if (have) {
                    const int slot = (k + m / 9) % 3;
                    const int r = w + 1 + ((m / 3) % 3 - 1), c = lane + 1 + (m % 3 - 1);
                    const double xun = xs[0][slot][r][c], xvn = xs[1][slot][r][c];
                    su = su + cuu * xun + cuv * xvn;
                    sv = sv + cvu * xun + cvv * xvn;
                }
            }
            if (MODE == 2) {
                const double ru = bu[ck] - su, rv = bv[ck] - sv;
                yu[ck] = ru;
                yv[ck] = rv;
                acc = dd_add_d(acc, ru * ru);
                acc = dd_add_d(acc, rv * rv);
            } else {
                const bool zr = MODE == 3 && zero_halo(d, d.ilo + io, d.jlo + jo, 2);
                yu[ck] = zr ? 0.0 : su;
                yv[ck] = zr ? 0.0 : sv;
                if (MODE == 1 || MODE == 3) {
                    const int slot = (k + 1) % 3;
                    acc = dd_add_d(acc, su * xs[0][slot][w + 1][lane + 1]);
                    acc = dd_add_d(acc, sv * xs[1][slot][w + 1][lane + 1]);
                }
            }
        }
        __syncthreads();
    }
    if (MODE != 0) {
        dd v[1] = {acc};
        block_reduce_dd<1, 256>(v);
        if (threadIdx.x == 0) {
            const int b = SPLIT ? blockIdx.y * nblk + lin : lin;
            partials[2 * b + 0] = v[0].hi;
            partials[2 * b + 1] = v[0].lo;
        }
    }
}

}  // namespace cg
