// cmp_mg.hip - geometric multigrid V-cycle on dense domain-shaped grids, the preconditioner of the
// implicit Grad_Q solve (div(b grad Q) = Div_Jhat, the system the reference hands to AMReX's MLMG,
// source/Class_Compressible_PhaseField.cpp:2133-2310, include/Operators_LinearSystem/Solver_MLMG_AllLevels.H).
//
// Built twice, with CMP_KERNEL_DIM=2 and CMP_KERNEL_DIM=3. A level that covers its whole domain is
// gathered into a dense array (i fastest, no ghosts; the operator's periodic and Neumann sides are
// applied by index arithmetic, so no fill is needed), then coarsened by 2 in every direction while
// every extent is even: face coefficients of a coarse face are the mean of the fine faces on it,
// residuals restrict as the mean of the 2^DIM children, corrections prolong piecewise constant, the
// coarse operators are the same five- (seven-) point discretisation at the coarse spacing. The
// smoother is damped Jacobi, the same number of sweeps before and after the coarse correction, and
// the coarsest grid (at most 1024 cells) takes a fixed number of sweeps in one workgroup: the
// V-cycle is then a fixed symmetric positive definite operator, as a conjugate-gradient
// preconditioner must be. Every kernel returns at once when the solve's stop flag is set.
#include "cmp_kernels.hpp"

#ifndef CMP_KERNEL_DIM
#error "CMP_KERNEL_DIM must be 2 or 3"
#endif

namespace cmp {

namespace {

__device__ __forceinline__ double mg_wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// the block's sums of N values a thread -> part[m * nb + block]
template <int N>
__device__ __forceinline__ void mg_block_sums(const double (&w)[N], double* part, long long nb, long long blk)
{
    __shared__ double red[N][NT / 64];
#pragma unroll
    for (int m = 0; m < N; ++m) {
        const double t = mg_wave_sum(w[m]);
        if ((threadIdx.x & 63) == 0) red[m][threadIdx.x >> 6] = t;
    }
    __syncthreads();
    if (threadIdx.x < N) {
        const int m = threadIdx.x;
        double s = red[m][0];
#pragma unroll
        for (int v = 1; v < NT / 64; ++v) s += red[m][v];
        part[m * nb + blk] = s;
    }
}

template <int DIM>
__device__ __forceinline__ void mg_cell(const MgGrid& G, long long q, int& i, int& j, int& k)
{
    pos3(q, G.n[0], G.n[1], i, j, k);
    if (DIM != 3) k = 0;
}

__device__ __forceinline__ long long mg_idx(const MgGrid& G, int i, int j, int k)
{
    return (long long)i + (long long)G.n[0] * (j + (long long)G.n[1] * k);
}

// the face of direction d at the low side of cell (i,j,k): nodal extents n + e_d
__device__ __forceinline__ long long mg_face(const MgGrid& G, int d, int i, int j, int k)
{
    const int f0 = G.n[0] + (d == 0), f1 = G.n[1] + (d == 1);
    return (long long)i + (long long)f0 * (j + (long long)f1 * k);
}

// (A x)_c = -div(b grad x) at cell (i,j,k): sum_d (b_lo (x_c - x_m) - b_hi (x_p - x_c)) / h_d^2, with
// no flux through a Neumann domain face and periodic neighbours wrapped; x(i,j,k) the value at a cell
template <int DIM, typename X>
__device__ __forceinline__ double mg_apply(const MgGrid& G, const X& x, const double* const* b, int i, int j, int k)
{
    const int co[3] = {i, j, k};
    const double xc = x(i, j, k);
    double acc = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        int m[3] = {i, j, k}, p[3] = {i, j, k};
        const bool lo_dom = co[d] == 0, hi_dom = co[d] == G.n[d] - 1;
        m[d] = lo_dom ? G.n[d] - 1 : co[d] - 1;
        p[d] = hi_dom ? 0 : co[d] + 1;
        double flo = 0.0, fhi = 0.0;
        if (!lo_dom || G.periodic[d]) flo = b[d][mg_face(G, d, i, j, k)] * (xc - x(m[0], m[1], m[2]));
        if (!hi_dom || G.periodic[d]) {
            int f[3] = {i, j, k};
            f[d] += 1;
            fhi = b[d][mg_face(G, d, f[0], f[1], f[2])] * (x(p[0], p[1], p[2]) - xc);
        }
        acc += (flo - fhi) * G.ih2[d];
    }
    return acc;
}

// the values of a grid's array
struct MgValues {
    const MgGrid& G;
    const double* x;
    __device__ __forceinline__ double operator()(int i, int j, int k) const { return x[mg_idx(G, i, j, k)]; }
};

template <int DIM>
__global__ __launch_bounds__(NT) void k_mg_gather_r(PfGeom g, const double* __restrict__ sc,
                                                    const double* __restrict__ R, double* r0, MgGrid G)
{
    if (sc && sc[CG_DONE] != 0.0) return;
    long long q;
    const BoxDev ab = g.abox[cell_block(g.cmap, q)];
    const int n0 = ab.hi[0] - ab.lo[0] + 1, n1 = ab.hi[1] - ab.lo[1] + 1;
    const int n2 = (DIM == 3) ? ab.hi[2] - ab.lo[2] + 1 : 1;
    if (q >= (long long)n0 * n1 * n2) return;
    int i, j, k;
    pos3(q, n0, n1, i, j, k);
    i += ab.lo[0];
    j += ab.lo[1];
    k += ab.lo[2];
    r0[mg_idx(G, i - g.dlo[0], j - g.dlo[1], (DIM == 3) ? k - g.dlo[2] : 0)] = R[ab.off + fab_index(ab, i, j, k)];
}

template <int DIM>
__global__ __launch_bounds__(NT) void k_mg_scatter(PfGeom g, const double* __restrict__ x0, double* X, MgGrid G)
{
    long long q;
    const BoxDev ab = g.abox[cell_block(g.cmap, q)];
    const int n0 = ab.hi[0] - ab.lo[0] + 1, n1 = ab.hi[1] - ab.lo[1] + 1;
    const int n2 = (DIM == 3) ? ab.hi[2] - ab.lo[2] + 1 : 1;
    if (q >= (long long)n0 * n1 * n2) return;
    int i, j, k;
    pos3(q, n0, n1, i, j, k);
    i += ab.lo[0];
    j += ab.lo[1];
    k += ab.lo[2];
    X[ab.off + fab_index(ab, i, j, k)] = x0[mg_idx(G, i - g.dlo[0], j - g.dlo[1], (DIM == 3) ? k - g.dlo[2] : 0)];
}

// the box face buffer of direction D (cmp_face_layout, one component) -> the dense face array
template <int DIM, int D>
__global__ __launch_bounds__(NT) void k_mg_gather_b(PfGeom g, const double* __restrict__ Bf, double* b0, MgGrid G)
{
    const BoxDev ab = g.abox[blockIdx.y];
    const int n0 = ab.hi[0] - ab.lo[0] + 1 + (D == 0), n1 = ab.hi[1] - ab.lo[1] + 1 + (D == 1);
    const int n2 = (DIM == 3) ? ab.hi[2] - ab.lo[2] + 1 + (D == 2) : 1;
    const long long q = (long long)blockIdx.x * NT + threadIdx.x;
    if (q >= (long long)n0 * n1 * n2) return;
    int i, j, k;
    pos3(q, n0, n1, i, j, k);
    i += ab.lo[0];
    j += ab.lo[1];
    k += ab.lo[2];
    b0[mg_face(G, D, i - g.dlo[0], j - g.dlo[1], (DIM == 3) ? k - g.dlo[2] : 0)] = Bf[ab.goff[D] + q];
}

// a coarse face of direction d: the mean of the 2^(DIM-1) fine faces on it (the fine faces at twice
// its position along d, the two (four) transverse children)
template <int DIM>
__global__ __launch_bounds__(NT) void k_mg_restrict_b(const double* __restrict__ bf, double* bc, MgGrid Gf,
                                                      MgGrid Gc, int d)
{
    const int f0 = Gc.n[0] + (d == 0), f1 = Gc.n[1] + (d == 1), f2 = (DIM == 3) ? Gc.n[2] + (d == 2) : 1;
    const long long nf = (long long)f0 * f1 * f2;
    const int t1 = (d == 0) ? 1 : 0;                   // the transverse axes, t1 < t2
    const int t2 = (d == 2) ? 1 : 2;
    constexpr int NS = (DIM == 3) ? 4 : 2;
    for (long long q = (long long)blockIdx.x * NT + threadIdx.x; q < nf; q += (long long)gridDim.x * NT) {
        int co[3];
        pos3(q, f0, f1, co[0], co[1], co[2]);
        if (DIM != 3) co[2] = 0;
        double s = 0.0;
#pragma unroll
        for (int m = 0; m < NS; ++m) {
            int f[3] = {2 * co[0], 2 * co[1], 2 * co[2]};
            f[t1] += m & 1;
            if (DIM == 3) f[t2] += m >> 1;
            s += bf[mg_face(Gf, d, f[0], f[1], f[2])];
        }
        bc[q] = s * (1.0 / (double)NS);
    }
}

// 1 / diag(A): sum of b / h_d^2 over the cell's faces that carry a flux
template <int DIM>
__global__ __launch_bounds__(NT) void k_mg_diag(const double* __restrict__ b0, const double* __restrict__ b1,
                                                const double* __restrict__ b2, double* id, MgGrid G)
{
    const double* b[3] = {b0, b1, b2};
    for (long long q = (long long)blockIdx.x * NT + threadIdx.x; q < G.nc; q += (long long)gridDim.x * NT) {
        int i, j, k;
        mg_cell<DIM>(G, q, i, j, k);
        const int co[3] = {i, j, k};
        double s = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            int f[3] = {i, j, k};
            f[d] += 1;
            if (co[d] > 0 || G.periodic[d]) s += b[d][mg_face(G, d, i, j, k)] * G.ih2[d];
            if (co[d] < G.n[d] - 1 || G.periodic[d]) s += b[d][mg_face(G, d, f[0], f[1], f[2])] * G.ih2[d];
        }
        id[q] = (s > 0.0) ? 1.0 / s : 0.0;
    }
}

// one damped Jacobi sweep y = x + omega D^-1 (r - A x). FROM: x the array (MG_FROM_X), the sweep from zero
// omega D^-1 r (MG_FROM_ZERO) or the array plus the coarser grid's value at the parent cell
// (MG_FROM_COARSE), the last two computed where they are read: a launch and a pass over memory each against
// one or two more loads a neighbour: four launches a grid instead of six. It pays at all sizes (3D Grad_Q with the
// two computed in launches of their own / so: 32^3 1.67 / 1.56 ms, 64^3 2.88 / 2.70, 128^3 7.87 / 7.37, 256^3
// 51.3 / 50.1; before the dense CG and the one-workgroup coarse end 3.22, 4.83, 11.08, 62.2). SUMS: the last sweep
// of a CG's preconditioner adds up r.z, z and r as it goes.
template <int DIM, int FROM, bool SUMS>
__global__ __launch_bounds__(NT) void k_mg_smooth(const double* __restrict__ sc, const double* __restrict__ x,
                                                  double* __restrict__ y, const double* __restrict__ r,
                                                  const double* __restrict__ b0, const double* __restrict__ b1,
                                                  const double* __restrict__ b2, const double* __restrict__ id,
                                                  MgGrid G, double omega, const double* __restrict__ xc, MgGrid Gc,
                                                  double* part)
{
    if (sc && sc[CG_DONE] != 0.0) return;
    const double* b[3] = {b0, b1, b2};
    auto value = [&](int i, int j, int k) __attribute__((always_inline)) -> double {
        // (rounded as a value that was stored: no term of it is contracted into a difference)
#pragma clang fp contract(off)
        const long long c = mg_idx(G, i, j, k);
        if (FROM == MG_FROM_ZERO) return omega * id[c] * r[c];
        if (FROM == MG_FROM_COARSE) return x[c] + xc[mg_idx(Gc, i >> 1, j >> 1, (DIM == 3) ? (k >> 1) : 0)];
        return x[c];
    };
    double w[3] = {0.0, 0.0, 0.0};
    for (long long q = (long long)blockIdx.x * NT + threadIdx.x; q < G.nc; q += (long long)gridDim.x * NT) {
        int i, j, k;
        mg_cell<DIM>(G, q, i, j, k);
        const double z = value(i, j, k) + omega * id[q] * (r[q] - mg_apply<DIM>(G, value, b, i, j, k));
        y[q] = z;
        if (SUMS) {
            w[0] += r[q] * z;
            w[1] += z;
            w[2] += r[q];
        }
    }
    if (SUMS) mg_block_sums(w, part + gridDim.x, gridDim.x, blockIdx.x);
}

// rc = mean over the 2^DIM children of (r - A x)
template <int DIM>
__global__ __launch_bounds__(NT) void k_mg_resid_restrict(const double* __restrict__ sc, const double* __restrict__ x,
                                                          const double* __restrict__ r, const double* __restrict__ b0,
                                                          const double* __restrict__ b1, const double* __restrict__ b2,
                                                          MgGrid Gf, double* rc, MgGrid Gc)
{
    if (sc && sc[CG_DONE] != 0.0) return;
    const double* b[3] = {b0, b1, b2};
    constexpr int NCH = (DIM == 3) ? 8 : 4;
    for (long long q = (long long)blockIdx.x * NT + threadIdx.x; q < Gc.nc; q += (long long)gridDim.x * NT) {
        int I, J, K;
        mg_cell<DIM>(Gc, q, I, J, K);
        double s = 0.0;
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch) {
            const int i = 2 * I + (ch & 1), j = 2 * J + ((ch >> 1) & 1), k = (DIM == 3) ? 2 * K + (ch >> 2) : 0;
            const long long c = mg_idx(Gf, i, j, k);
            s += r[c] - mg_apply<DIM>(Gf, MgValues{Gf, x}, b, i, j, k);
        }
        rc[q] = s * (1.0 / (double)NCH);
    }
}

// The two legs of a 2D grid's visit, a launch each: a workgroup takes 32 x 8 cells and recomputes what its
// sweeps read beyond them (the first sweep on two cells around, the second on one), in LDS. Bound by launches
// and load latency on all grids but the largest: a launch is about 4 us whatever it does, and the legs were two
// launches each. 512 x 256 Grad_Q 2.00 -> 1.62 ms, eight cases' CAC steps 5.57 -> 4.97 ms, a hierarchy's 21.4 ->
// 19.6 ms. The arithmetic is k_mg_smooth's and k_mg_resid_restrict's.
static_assert(MGX * MGY == NT, "a cell a thread");

// coordinate i of direction d taken into the domain across a periodic side; false: no such cell
__device__ __forceinline__ bool mg_wrap(const MgGrid& G, int d, int& i)
{
    const int n = G.n[d];
    if (G.periodic[d]) i = (i < 0) ? i + n : (i >= n) ? i - n : i;
    return i >= 0 && i < n;
}

// mg_apply at cell (i,j) on values in LDS rows of W, x at the cell's
template <int W>
__device__ __forceinline__ double mg_apply_lds(const MgGrid& G, const double* x, const double* __restrict__ b0,
                                               const double* __restrict__ b1, int i, int j)
{
    const double xc = x[0];
    double acc = 0.0, flo = 0.0, fhi = 0.0;
    if (i > 0 || G.periodic[0]) flo = b0[mg_face(G, 0, i, j, 0)] * (xc - x[-1]);
    if (i < G.n[0] - 1 || G.periodic[0]) fhi = b0[mg_face(G, 0, i + 1, j, 0)] * (x[1] - xc);
    acc += (flo - fhi) * G.ih2[0];
    flo = fhi = 0.0;
    if (j > 0 || G.periodic[1]) flo = b1[mg_face(G, 1, i, j, 0)] * (xc - x[-W]);
    if (j < G.n[1] - 1 || G.periodic[1]) fhi = b1[mg_face(G, 1, i, j + 1, 0)] * (x[W] - xc);
    acc += (flo - fhi) * G.ih2[1];
    return acc;
}

// the sweep's start on the tile and two cells around (rows of MGX + 4), then one sweep on the tile and one cell
// around (rows of MGX + 2)
template <typename V>
__device__ __forceinline__ void mg_tile_sweep(const MgGrid& G, int i0, int j0, double* s0, double* s1, const V& value,
                                              const double* __restrict__ r, const double* __restrict__ id,
                                              const double* __restrict__ b0, const double* __restrict__ b1, double omega)
{
    for (int q = threadIdx.x; q < (MGX + 4) * (MGY + 4); q += NT) {
        int i = i0 - 2 + q % (MGX + 4), j = j0 - 2 + q / (MGX + 4);
        if (mg_wrap(G, 0, i) && mg_wrap(G, 1, j)) s0[q] = value(i, j);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < (MGX + 2) * (MGY + 2); q += NT) {
        const int li = q % (MGX + 2), lj = q / (MGX + 2);
        int i = i0 - 1 + li, j = j0 - 1 + lj;
        if (!mg_wrap(G, 0, i) || !mg_wrap(G, 1, j)) continue;
        const double* x = s0 + (lj + 1) * (MGX + 4) + li + 1;
        const long long c = mg_idx(G, i, j, 0);
        s1[q] = x[0] + omega * id[c] * (r[c] - mg_apply_lds<MGX + 4>(G, x, b0, b1, i, j));
    }
    __syncthreads();
}

__device__ __forceinline__ void mg_tile(const MgGrid& G, int& i0, int& j0)
{
    const int ntx = (G.n[0] + MGX - 1) / MGX, t = blockIdx.x;
    j0 = (t / ntx) * MGY;
    i0 = (t % ntx) * MGX;
}

__global__ __launch_bounds__(NT) void k_mg_down(const double* __restrict__ sc, double* __restrict__ y,
                                                const double* __restrict__ r, const double* __restrict__ b0,
                                                const double* __restrict__ b1, const double* __restrict__ id, MgGrid G,
                                                double omega, double* __restrict__ rc, MgGrid Gc)
{
    if (sc && sc[CG_DONE] != 0.0) return;
    __shared__ double s0[(MGX + 4) * (MGY + 4)], s1[(MGX + 2) * (MGY + 2)], res[MGX * MGY];
    int i0, j0;
    mg_tile(G, i0, j0);
    auto value = [&](int i, int j) __attribute__((always_inline)) -> double {
#pragma clang fp contract(off)
        const long long c = mg_idx(G, i, j, 0);
        return omega * id[c] * r[c];
    };
    mg_tile_sweep(G, i0, j0, s0, s1, value, r, id, b0, b1, omega);
    const int li = threadIdx.x % MGX, lj = threadIdx.x / MGX, i = i0 + li, j = j0 + lj;
    if (i < G.n[0] && j < G.n[1]) {
        const double* x = s1 + (lj + 1) * (MGX + 2) + li + 1;
        const long long c = mg_idx(G, i, j, 0);
        y[c] = x[0];
        res[threadIdx.x] = r[c] - mg_apply_lds<MGX + 2>(G, x, b0, b1, i, j);
    }
    __syncthreads();
    if (threadIdx.x >= NT / 4) return;
    const int ci = threadIdx.x % (MGX / 2), cj = threadIdx.x / (MGX / 2);
    if (i0 / 2 + ci >= Gc.n[0] || j0 / 2 + cj >= Gc.n[1]) return;
    const double* q = res + 2 * cj * MGX + 2 * ci;
    double s = q[0];
    s += q[1];
    s += q[MGX];
    s += q[MGX + 1];
    rc[mg_idx(Gc, i0 / 2 + ci, j0 / 2 + cj, 0)] = s * 0.25;
}

// SUMS: the partials of r.z, z and r, z the result, into part's second to fourth slots
template <bool SUMS>
__global__ __launch_bounds__(NT) void k_mg_up(const double* __restrict__ sc, const double* __restrict__ x1,
                                              double* __restrict__ y, const double* __restrict__ r,
                                              const double* __restrict__ b0, const double* __restrict__ b1,
                                              const double* __restrict__ id, MgGrid G, double omega,
                                              const double* __restrict__ xc, MgGrid Gc, double* part)
{
    if (sc && sc[CG_DONE] != 0.0) return;
    __shared__ double s0[(MGX + 4) * (MGY + 4)], s1[(MGX + 2) * (MGY + 2)];
    int i0, j0;
    mg_tile(G, i0, j0);
    auto value = [&](int i, int j) __attribute__((always_inline)) -> double {
        return x1[mg_idx(G, i, j, 0)] + xc[mg_idx(Gc, i >> 1, j >> 1, 0)];
    };
    mg_tile_sweep(G, i0, j0, s0, s1, value, r, id, b0, b1, omega);
    const int li = threadIdx.x % MGX, lj = threadIdx.x / MGX, i = i0 + li, j = j0 + lj;
    double w[3] = {0.0, 0.0, 0.0};
    if (i < G.n[0] && j < G.n[1]) {
        const double* x = s1 + (lj + 1) * (MGX + 2) + li + 1;
        const long long c = mg_idx(G, i, j, 0);
        const double rq = r[c], z = x[0] + omega * id[c] * (rq - mg_apply_lds<MGX + 2>(G, x, b0, b1, i, j));
        y[c] = z;
        w[0] = rq * z;
        w[1] = z;
        w[2] = rq;
    }
    if (SUMS) mg_block_sums(w, part + gridDim.x, gridDim.x, blockIdx.x);
}

// A cell of a grid with the coefficients its operator row reads, kept in registers over the phases of a
// visit: (A x)_c = sum_d (b_lo (x_c - x_m) - b_hi (x_p - x_c)) / h_d^2, a Neumann domain face with b = 0.
template <int DIM>
struct TailCell {
    int q;                  // -1: no cell
    unsigned edge;          // bit 2d / 2d + 1: at the low / high side of the domain along d
    double r, id, bl[DIM], bh[DIM];
};

template <int DIM>
__device__ __forceinline__ void tail_pos(const MgGrid& G, int q, int* c)
{
    // exact below 10^6: the quotient (q + 1/2) / n lies at least 1/(2 n) from an integer
    const float h = (float)q + 0.5f;
    const int a = (int)(h * __builtin_amdgcn_rcpf((float)G.n[0]));
    c[0] = q - a * G.n[0];
    c[1] = a;
    c[2] = 0;
    if (DIM == 3) {
        c[2] = (int)(h * __builtin_amdgcn_rcpf((float)(G.n[0] * G.n[1])));
        c[1] = a - c[2] * G.n[1];
    }
}

// b[d]: the grid's face coefficients
template <int DIM, typename B>
__device__ __forceinline__ TailCell<DIM> tail_cell(const MgGrid& G, int q, double r, double id, const B& b)
{
    TailCell<DIM> c;
    int p[3];
    tail_pos<DIM>(G, q, p);
    c.q = q;
    c.edge = 0u;
    c.r = r;
    c.id = id;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const bool lo = p[d] == 0, hi = p[d] == G.n[d] - 1;
        c.edge |= (lo ? 1u : 0u) << (2 * d) | (hi ? 2u : 0u) << (2 * d);
        int f[3] = {p[0], p[1], p[2]};
        c.bl[d] = (!lo || G.periodic[d]) ? b(d, (int)mg_face(G, d, f[0], f[1], f[2])) : 0.0;
        f[d] += 1;
        c.bh[d] = (!hi || G.periodic[d]) ? b(d, (int)mg_face(G, d, f[0], f[1], f[2])) : 0.0;
    }
    return c;
}

template <int DIM>
__device__ __forceinline__ double tail_apply(const MgGrid& G, const TailCell<DIM>& c, const double* x)
{
    const double xc = x[c.q];
    double acc = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const int s = (d == 0) ? 1 : ((d == 1) ? G.n[0] : G.n[0] * G.n[1]);
        const int wrap = (G.n[d] - 1) * s;   // (a Neumann side's neighbour counts nothing: b = 0)
        const int m = (c.edge >> (2 * d) & 1u) ? c.q + wrap : c.q - s;
        const int p = (c.edge >> (2 * d) & 2u) ? c.q - wrap : c.q + s;
        acc += (c.bl[d] * (xc - x[m]) - c.bh[d] * (x[p] - xc)) * G.ih2[d];
    }
    return acc;
}

// The coarse end of the V-cycle (MgTail) in one workgroup of 1024 threads. Bound by the latency of its many
// short phases, so: every grid's iterates live in LDS (the first grid's r, 1/diag and b in its threads'
// registers, at most four cells a thread; the others' in LDS), and the grids of at most 64 cells are one
// wave's, whose phases follow each other without a barrier (its LDS accesses execute in order). The arithmetic
// is the per-grid launches'. On one card 33 -> 14.5 us a
// visit from 64 x 32 cells, 70 -> 24.9 from 128 x 32.
constexpr int NTAIL = 1024;
template <int DIM>
__global__ __launch_bounds__(NTAIL) void k_mg_tail(MgTail t)
{
    if (t.sc && t.sc[CG_DONE] != 0.0) return;
    __shared__ double lds[MG_TAIL_LDS];
    constexpr int CPT = (int)(MG_TAIL_MAX_CELLS / NTAIL);
    constexpr int NCH = (DIM == 3) ? 8 : 4;
    const int tid = threadIdx.x;
    const double om = t.omega;
    const int last = t.nlev - 1;
    int w = 1;                      // the first grid (after grid 0) that one wave takes
    while (w <= last && t.G[w].nc > 64) ++w;
    // the coarser grids' inverse diagonals and face coefficients
    for (int m = 1; m < t.nlev; ++m) {
        const MgGrid& G = t.G[m];
        for (int q = tid; q < (int)G.nc; q += NTAIL) lds[t.loff[m][3] + q] = t.id[m][q];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            int nf = 1;
#pragma unroll
            for (int e = 0; e < DIM; ++e) nf *= G.n[e] + (e == d);
            for (int q = tid; q < nf; q += NTAIL) lds[t.loff[m][4 + d] + q] = t.b[m][d][q];
        }
    }
    // grid 0's cells
    const MgGrid& G0 = t.G[0];
    double* const a0 = lds + t.loff[0][0];
    double* const a1 = lds + t.loff[0][1];
    TailCell<DIM> c0[CPT];
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
        const int q = c * NTAIL + tid;
        c0[c].q = -1;
        if (q < (int)G0.nc)
            c0[c] = tail_cell<DIM>(G0, q, t.r[0][q], t.id[0][q], [&](int d, int f) { return t.b[0][d][f]; });
    }
    auto lds_cell = [&](int m, int q) __attribute__((always_inline)) {
        return tail_cell<DIM>(t.G[m], q, lds[t.loff[m][2] + q], lds[t.loff[m][3] + q],
                              [&](int d, int f) { return lds[t.loff[m][4 + d] + f]; });
    };
    // r of grid m + 1 from the residual of grid m (in its x0), the mean over the children
    auto restrict_to = [&](int m, int q) __attribute__((always_inline)) {
        const MgGrid& Gf = t.G[m];
        const double* res = lds + t.loff[m][0];
        int p[3];
        tail_pos<DIM>(t.G[m + 1], q, p);
        double sum = 0.0;
#pragma unroll
        for (int ch = 0; ch < NCH; ++ch)
            sum += res[(2 * p[0] + (ch & 1)) +
                       Gf.n[0] * ((2 * p[1] + ((ch >> 1) & 1)) + Gf.n[1] * ((DIM == 3) ? 2 * p[2] + (ch >> 2) : 0))];
        lds[t.loff[m + 1][2] + q] = sum * (1.0 / (double)NCH);
    };
    // grid m's x1 plus the coarser grid's result at the parent cell
    auto prolonged = [&](int m, int q) __attribute__((always_inline)) -> double {
        int p[3];
        tail_pos<DIM>(t.G[m], q, p);
        const MgGrid& Gc = t.G[m + 1];
        const double* xc = lds + t.loff[m + 1][(m + 1 == last) ? 0 : 1];
        return lds[t.loff[m][1] + q] + xc[(p[0] >> 1) + Gc.n[0] * ((p[1] >> 1) + Gc.n[1] * ((DIM == 3) ? p[2] >> 1 : 0))];
    };
    // one grid of at most n threads' cells (q = the thread's, when below nc): two sweeps from zero and the
    // residual; prolongation and two sweeps; the coarsest grid's sweeps
    auto down = [&](int m, int q, auto sync) __attribute__((always_inline)) {
        const MgGrid& G = t.G[m];
        double* x0 = lds + t.loff[m][0];
        double* x1 = lds + t.loff[m][1];
        const bool on = q < (int)G.nc;
        TailCell<DIM> c;
        c.q = -1;
        double v = 0.0;
        if (on) {
            c = lds_cell(m, q);
            v = om * c.id * c.r;
            x0[q] = v;
        }
        sync();
        if (on) x1[q] = v + om * c.id * (c.r - tail_apply<DIM>(G, c, x0));
        sync();
        if (on) x0[q] = c.r - tail_apply<DIM>(G, c, x1);
        sync();
        if (q < (int)t.G[m + 1].nc) restrict_to(m, q);
        sync();
    };
    auto up = [&](int m, int q, auto sync) __attribute__((always_inline)) {
        const MgGrid& G = t.G[m];
        double* x0 = lds + t.loff[m][0];
        double* x1 = lds + t.loff[m][1];
        const bool on = q < (int)G.nc;
        TailCell<DIM> c;
        c.q = -1;
        double v = 0.0;
        if (on) {
            c = lds_cell(m, q);
            v = prolonged(m, q);
            x1[q] = v;
        }
        sync();
        if (on) {
            v = v + om * c.id * (c.r - tail_apply<DIM>(G, c, x1));
            x0[q] = v;
        }
        sync();
        if (on) x1[q] = v + om * c.id * (c.r - tail_apply<DIM>(G, c, x0));
        sync();
    };
    auto bottom = [&](int q, auto sync) __attribute__((always_inline)) {
        const MgGrid& G = t.G[last];
        double* x0 = lds + t.loff[last][0];
        double* x1 = lds + t.loff[last][1];
        const bool on = q < (int)G.nc;
        TailCell<DIM> c;
        c.q = -1;
        double v = 0.0;
        if (on) {
            c = lds_cell(last, q);
            v = om * c.id * c.r;
        }
        for (int sw = 1; sw < t.sweeps; ++sw) {
            double* x = (sw & 1) ? x0 : x1;
            if (on) x[q] = v;
            sync();
            if (on) v = v + om * c.id * (c.r - tail_apply<DIM>(G, c, x));
        }
        sync();
        if (on) x0[q] = v;
        sync();
    };
    auto block_sync = [&]() { __syncthreads(); };
    auto wave_sync = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    if (last == 0) {
        // one grid: its sweeps from zero (nc <= 1024), r in place of a coarser grid's
        __syncthreads();
        double v = 0.0;
        if (c0[0].q >= 0) v = om * c0[0].id * c0[0].r;
        for (int sw = 1; sw < t.sweeps; ++sw) {
            double* x = (sw & 1) ? a0 : a1;
            if (c0[0].q >= 0) x[c0[0].q] = v;
            __syncthreads();
            if (c0[0].q >= 0) v = v + om * c0[0].id * (c0[0].r - tail_apply<DIM>(G0, c0[0], x));
        }
        if (c0[0].q >= 0) t.x0[0][c0[0].q] = v;
        return;
    }
    double v0[CPT];
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
        v0[c] = 0.0;
        if (c0[c].q >= 0) {
            v0[c] = om * c0[c].id * c0[c].r;
            a0[c0[c].q] = v0[c];
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CPT; ++c)
        if (c0[c].q >= 0) a1[c0[c].q] = v0[c] + om * c0[c].id * (c0[c].r - tail_apply<DIM>(G0, c0[c], a0));
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CPT; ++c)
        if (c0[c].q >= 0) a0[c0[c].q] = c0[c].r - tail_apply<DIM>(G0, c0[c], a1);
    __syncthreads();
    if (tid < (int)t.G[1].nc) restrict_to(0, tid);
    __syncthreads();
    for (int m = 1; m < w && m < last; ++m) down(m, tid, block_sync);
    if (w > last) {
        bottom(tid, block_sync);
    } else if (tid < 64) {
        for (int m = w; m < last; ++m) down(m, tid, wave_sync);
        bottom(tid, wave_sync);
        for (int m = last - 1; m >= w; --m) up(m, tid, wave_sync);
    }
    __syncthreads();
    for (int m = (w > last ? last : w) - 1; m >= 1; --m) up(m, tid, block_sync);
#pragma unroll
    for (int c = 0; c < CPT; ++c)
        if (c0[c].q >= 0) v0[c] = prolonged(0, c0[c].q);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CPT; ++c)
        if (c0[c].q >= 0) a1[c0[c].q] = v0[c];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CPT; ++c)
        if (c0[c].q >= 0) {
            v0[c] = v0[c] + om * c0[c].id * (c0[c].r - tail_apply<DIM>(G0, c0[c], a1));
            a0[c0[c].q] = v0[c];
        }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CPT; ++c)
        if (c0[c].q >= 0) t.x1[0][c0[c].q] = v0[c] + om * c0[c].id * (c0[c].r - tail_apply<DIM>(G0, c0[c], a0));
}

// the partial sums of one CG iteration's r.z, sum z and sum r (the second, third and fourth partial
// slots; the first holds r.r)
template <int DIM>
__global__ __launch_bounds__(NT) void k_cg_rz(PfGeom g, const double* __restrict__ sc, const double* __restrict__ R,
                                              const double* __restrict__ Z, double* part)
{
    if (sc && sc[CG_DONE] != 0.0) return;
    long long q;
    const BoxDev ab = g.abox[cell_block(g.cmap, q)];
    const int n0 = ab.hi[0] - ab.lo[0] + 1, n1 = ab.hi[1] - ab.lo[1] + 1;
    const int n2 = (DIM == 3) ? ab.hi[2] - ab.lo[2] + 1 : 1;
    double w[3] = {0.0, 0.0, 0.0};
    if (q < (long long)n0 * n1 * n2) {
        int i, j, k;
        pos3(q, n0, n1, i, j, k);
        i += ab.lo[0];
        j += ab.lo[1];
        k += ab.lo[2];
        const long long c = ab.off + fab_index(ab, i, j, k);
        const double r = R[c], z = Z[c];
        w[0] = r * z;
        w[1] = z;
        w[2] = r;
    }
    const long long nb = (long long)gridDim.x * gridDim.y;
    mg_block_sums(w, part + nb, nb, (long long)blockIdx.y * gridDim.x + blockIdx.x);
}

// ---- the iteration of a CG on one dense grid (a level that covers its domain) -------------------------
// Bound by its launches on all but the largest levels: on the dense arrays there are no ghost cells to fill,
// nothing to gather for or scatter from the V-cycle, and the direction's update is taken where ap reads it
// (p_old -> p, two arrays in turn), so that an iteration outside the V-cycle has three launches (four above
// 1024 partials a sum) where the box layout's had nine (eight cases' CAC steps 6.90 -> 5.55 ms).

// the partials of r.z, z and r (a preconditioner whose last launch is not a sweep of grid 0)
__global__ __launch_bounds__(NT) void k_dcg_sums(const double* __restrict__ sc, const double* __restrict__ r,
                                                 const double* __restrict__ z, long long nc, double* part)
{
    if (sc && sc[CG_DONE] != 0.0) return;
    double w[3] = {0.0, 0.0, 0.0};
    for (long long q = (long long)blockIdx.x * NT + threadIdx.x; q < nc; q += (long long)gridDim.x * NT) {
        w[0] += r[q] * z[q];
        w[1] += z[q];
        w[2] += r[q];
    }
    mg_block_sums(w, part + gridDim.x, gridDim.x, blockIdx.x);
}

// p = z - mean(z) + beta p_old; ap = -div(b grad p) with the box layout's arithmetic (k_cg_ap); partials of p.ap
template <int DIM>
__global__ __launch_bounds__(NT) void k_dcg_ap(const double* __restrict__ sc, const double* __restrict__ z,
                                               const double* __restrict__ pold, double* __restrict__ p,
                                               double* __restrict__ AP, const double* __restrict__ b0,
                                               const double* __restrict__ b1, const double* __restrict__ b2,
                                               MgGrid G, double dx0, double dx1, double dx2, double inv_n, double* part)
{
    if (sc[CG_DONE] != 0.0) return;
    const double be = sc[CG_BETA], zm = sc[CG_ZS] * inv_n;
    const double* b[3] = {b0, b1, b2};
    const double dx[3] = {dx0, dx1, dx2};
    auto value = [&](int i, int j, int k) __attribute__((always_inline)) -> double {
        const long long c = mg_idx(G, i, j, k);
        const double zc = z[c] - zm;
        return be != 0.0 ? fma(be, pold[c], zc) : zc;   // (the first direction: p_old holds nothing)
    };
    double w[1] = {0.0};
    for (long long q = (long long)blockIdx.x * NT + threadIdx.x; q < G.nc; q += (long long)gridDim.x * NT) {
        int i, j, k;
        mg_cell<DIM>(G, q, i, j, k);
        const int co[3] = {i, j, k};
        const double pc = value(i, j, k);
        double acc = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            int m[3] = {i, j, k}, n[3] = {i, j, k}, f[3] = {i, j, k};
            const bool lo = co[d] == 0, hi = co[d] == G.n[d] - 1;
            m[d] = lo ? G.n[d] - 1 : co[d] - 1;
            n[d] = hi ? 0 : co[d] + 1;
            f[d] += 1;
            const double fp = (hi && !G.periodic[d])
                                  ? 0.0
                                  : b[d][mg_face(G, d, f[0], f[1], f[2])] * (value(n[0], n[1], n[2]) - pc) / dx[d];
            const double fm = (lo && !G.periodic[d])
                                  ? 0.0
                                  : b[d][mg_face(G, d, i, j, k)] * (pc - value(m[0], m[1], m[2])) / dx[d];
            const double t = (fp - fm) / dx[d];
            acc = (d == 0) ? t : acc + t;
        }
        p[q] = pc;
        AP[q] = -acc;
        w[0] += pc * (-acc);
    }
    mg_block_sums(w, part, gridDim.x, blockIdx.x);
}

// x += al p, r -= al ap, partials of r.r into the first slot. nred > 0: p.ap is its nred partials' sum, taken
// by every block in the same order (a launch less; at most 1024 values, four a thread); else it is in sc.
__global__ __launch_bounds__(NT) void k_dcg_xr(double* __restrict__ sc, double* __restrict__ x,
                                               double* __restrict__ r, const double* __restrict__ p,
                                               const double* __restrict__ AP, long long nc, int nred,
                                               const double* __restrict__ pap_part, double* part)
{
    if (sc[CG_DONE] != 0.0) return;
    __shared__ double red[NT / 64];
    double pap;
    if (nred > 0) {
        double t = 0.0;
        for (int b = threadIdx.x; b < nred; b += NT) t += pap_part[b];
        t = mg_wave_sum(t);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
        __syncthreads();
        pap = red[0];
#pragma unroll
        for (int v = 1; v < NT / 64; ++v) pap += red[v];
        if (blockIdx.x == 0 && threadIdx.x == 0) sc[CG_PAP] = pap;
    } else {
        pap = sc[CG_PAP];
    }
    if (!(pap > 0.0)) return;
    const double al = sc[CG_RZ] / pap;
    double w[1] = {0.0};
    for (long long q = (long long)blockIdx.x * NT + threadIdx.x; q < nc; q += (long long)gridDim.x * NT) {
        x[q] += al * p[q];
        const double v = r[q] - al * AP[q];
        r[q] = v;
        w[0] += v * v;
    }
    mg_block_sums(w, part, gridDim.x, blockIdx.x);
}

// the four sums of an iteration in one workgroup, then its end; first: r.z and the means' sums alone (r.r of the
// initial residual is in sc), then the solve's start
__global__ __launch_bounds__(1024) void k_dcg_end(double* sc, const double* __restrict__ part, int nb, double maxit,
                                                  double inv_n, int first)
{
    if (!first && sc[CG_DONE] != 0.0) return;
    __shared__ double red[4][16];
    const int tid = threadIdx.x;
    double w[4] = {0.0, 0.0, 0.0, 0.0};
    for (int b = tid; b < nb; b += 1024) {
#pragma unroll
        for (int m = 0; m < 4; ++m)
            if (m > 0 || !first) w[m] += part[(long long)m * nb + b];
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const double t = mg_wave_sum(w[m]);
        if ((tid & 63) == 0) red[m][tid >> 6] = t;
    }
    __syncthreads();
    if (tid != 0) return;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        w[m] = red[m][0];
#pragma unroll
        for (int v = 1; v < 16; ++v) w[m] += red[m][v];
    }
    if (!first) sc[CG_RRNEW] = w[0];
    sc[first ? CG_RZ : CG_RZNEW] = w[1];
    sc[CG_ZS] = w[2];
    sc[CG_RS] = w[3];
    if (first)
        cg_start_step(sc, inv_n);
    else
        cg_end_step(sc, maxit, inv_n);
}

dim3 mg_grid(long long n) { return dim3((unsigned)mg_blocks(n)); }

dim3 box_grid(long long maxn, int nbox)
{
    long long b = (maxn + NT - 1) / NT;
    if (b < 1) b = 1;
    return dim3((unsigned)b, (unsigned)nbox);
}

}  // namespace

template <int DIM>
hipError_t launch_mg_dim(int op, const MgArgs& a, hipStream_t s)
{
    switch (op) {
    case MG_GATHER_R:
        hipLaunchKernelGGL((k_mg_gather_r<DIM>), cell_grid(a.g.cmap, a.g.ncmap, a.maxcells, a.g.nbox), dim3(NT), 0, s, a.g, a.sc, a.src,
                           a.dst, a.G);
        break;
    case MG_GATHER_B:
        hipLaunchKernelGGL((k_mg_gather_b<DIM, 0>), box_grid(a.maxfaces[0], a.g.nbox), dim3(NT), 0, s, a.g, a.src,
                           a.b[0], a.G);
        hipLaunchKernelGGL((k_mg_gather_b<DIM, 1>), box_grid(a.maxfaces[1], a.g.nbox), dim3(NT), 0, s, a.g, a.src,
                           a.b[1], a.G);
        if (DIM == 3)
            hipLaunchKernelGGL((k_mg_gather_b<DIM, (DIM == 3 ? 2 : 1)>), box_grid(a.maxfaces[2], a.g.nbox), dim3(NT),
                               0, s, a.g, a.src, a.b[2], a.G);
        break;
    case MG_RESTRICT_B:
        for (int d = 0; d < DIM; ++d) {
            long long nf = 1;
            for (int e = 0; e < DIM; ++e) nf *= a.Gc.n[e] + (e == d);
            hipLaunchKernelGGL((k_mg_restrict_b<DIM>), mg_grid(nf), dim3(NT), 0, s, a.b[d], a.bc[d], a.G, a.Gc, d);
        }
        break;
    case MG_DIAG:
        hipLaunchKernelGGL((k_mg_diag<DIM>), mg_grid(a.G.nc), dim3(NT), 0, s, a.b[0], a.b[1], a.b[2], a.dst, a.G);
        break;
    case MG_SMOOTH: if constexpr (DIM == 3) {
        if (a.part && a.from != MG_FROM_X) return hipErrorInvalidValue;
        const auto f = a.part                    ? k_mg_smooth<DIM, MG_FROM_X, true>
                       : a.from == MG_FROM_X    ? k_mg_smooth<DIM, MG_FROM_X, false>
                       : a.from == MG_FROM_ZERO ? k_mg_smooth<DIM, MG_FROM_ZERO, false>
                                                : k_mg_smooth<DIM, MG_FROM_COARSE, false>;
        hipLaunchKernelGGL(f, mg_grid(a.G.nc), dim3(NT), 0, s, a.sc, a.src, a.dst, a.r, a.b[0], a.b[1], a.b[2],
                           a.id, a.G, a.omega, a.xc, a.Gc, a.part);
        break;
    } else return hipErrorInvalidValue;
    case MG_RESID_RESTRICT: if constexpr (DIM == 3) {
        hipLaunchKernelGGL((k_mg_resid_restrict<DIM>), mg_grid(a.Gc.nc), dim3(NT), 0, s, a.sc, a.src, a.r, a.b[0],
                           a.b[1], a.b[2], a.G, a.dst, a.Gc);
        break;
    } else return hipErrorInvalidValue;
    case MG_DOWN: if constexpr (DIM == 2) {
        hipLaunchKernelGGL(k_mg_down, dim3((unsigned)mg_parts(2, a.G)), dim3(NT), 0, s, a.sc, a.dst, a.r, a.b[0],
                           a.b[1], a.id, a.G, a.omega, a.rw, a.Gc);
        break;
    } else return hipErrorInvalidValue;
    case MG_UP: if constexpr (DIM == 2) {
        hipLaunchKernelGGL((a.part ? k_mg_up<true> : k_mg_up<false>), dim3((unsigned)mg_parts(2, a.G)), dim3(NT), 0, s,
                           a.sc, a.src, a.dst, a.r, a.b[0], a.b[1], a.id, a.G, a.omega, a.xc, a.Gc, a.part);
        break;
    } else return hipErrorInvalidValue;
    case MG_SCATTER:
        hipLaunchKernelGGL((k_mg_scatter<DIM>), cell_grid(a.g.cmap, a.g.ncmap, a.maxcells, a.g.nbox), dim3(NT), 0, s,
                           a.g, a.src, a.dst, a.G);
        break;
    case MG_CG_RZ:
        hipLaunchKernelGGL((k_cg_rz<DIM>), cell_grid(a.g.cmap, a.g.ncmap, a.maxcells, a.g.nbox), dim3(NT), 0, s, a.g,
                           a.sc, a.r, a.dst, a.part);
        break;
    case MG_CG_SUMS:
        hipLaunchKernelGGL(k_dcg_sums, dim3((unsigned)mg_parts(DIM, a.G)), dim3(NT), 0, s, a.sc, a.r, a.src, a.G.nc, a.part);
        break;
    case MG_CG_AP:
        hipLaunchKernelGGL((k_dcg_ap<DIM>), dim3((unsigned)mg_parts(DIM, a.G)), dim3(NT), 0, s, a.sc, a.src, a.r, a.dst, a.rw, a.b[0],
                           a.b[1], a.b[2], a.G, a.g.dx[0], a.g.dx[1], a.g.dx[2], a.inv_n, a.part);
        break;
    case MG_CG_XR: {
        const int nb = mg_parts(DIM, a.G);
        hipLaunchKernelGGL(k_dcg_xr, dim3((unsigned)mg_parts(DIM, a.G)), dim3(NT), 0, s, a.scw, a.dst, a.rw, a.src, a.id, a.G.nc,
                           nb <= 1024 ? nb : 0, a.r, a.part);
        break;
    }
    case MG_CG_END:
        hipLaunchKernelGGL(k_dcg_end, dim3(1), dim3(1024), 0, s, a.scw, a.part, mg_parts(DIM, a.G), a.maxit,
                           a.inv_n, a.first);
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template hipError_t launch_mg_dim<CMP_KERNEL_DIM>(int, const MgArgs&, hipStream_t);

template <int DIM>
hipError_t launch_mg_tail_dim(const MgTail& t, hipStream_t s)
{
    if (t.nlev < 1 || t.nlev > MG_TAIL_MAX_LEVELS) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_mg_tail<DIM>), dim3(1), dim3(NTAIL), 0, s, t);
    return hipGetLastError();
}

template hipError_t launch_mg_tail_dim<CMP_KERNEL_DIM>(const MgTail&, hipStream_t);

}  // namespace cmp
