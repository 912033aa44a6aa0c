// hamr_adjoint.hip -- adjoint of one forward stage of the step (FP64).
//
// Forward stage (the predictor of the step with the full Dt):
//   fluxes F_d = HLL(PPM(P), face B) through every computed face,
//   corner EMF E(P, F) upwinded on the mass-flux signs,
//   face field  B_f' = B_f - Dt curl(E) / gdet_f,
//   U' = U(P) - Dt sum_d (F_d(c + e_d) - F_d(c)) / dx_d + Dt S(P), U'[B] = face average of B_f'.
// For a loss L = sum w . U' the kernels below form dL/dP and dL/dB_f (the face
// field at the start of the stage) in reverse order, recomputing the
// reconstructed states, fluxes and EMF selections from P instead of storing
// them.  The source term is zero in the flat metric the adjoint serves (a
// periodic box of one block).
//
// Every kernel gathers: a thread owns a cell, face or edge and reads what
// reaches it, with indices wrapped into the periodic box, so each of the box's
// n1 n2 n3 faces of a direction is taken once (its ghost copies and the copies on
// the upper boundary add up in their common weight) and nothing is
// accumulated by atomics: a call gives the same bits every time.
#include "hamr_adjoint.h"
#include "hamr_kernels_dev.h"

namespace hamr {

namespace {

// components of P that are reconstructed at a face: all but KTOT (which does not
// enter the stage) and the normal field; each takes two slabs of the faces' buffer
constexpr int kAdjRec = 7;
static_assert(kAdjXSlabs == 2 * kAdjRec, "two slabs per reconstructed component");

struct AdjArgs {
    int D[3], bs[3];
    int n;               // interior cells
    int64_t K;           // slab length of the context's arrays and the scratch
    int64_t Kw, Kg;      // slab length of the weights and of the gradients
    double dx[3], Dt, gam;
    const double *gcov, *gcon, *gdet;  // geometry slab 0
    int64_t kcol;
};

// periodic image inside the interior of an index at most bs cells outside
__device__ __forceinline__ int wrap1(int i, int bs) { return i < NG ? i + bs : i >= NG + bs ? i - bs : i; }

__device__ __forceinline__ uint32_t cell_of(const AdjArgs &A, int i, int j, int z)
{
    return ((uint32_t)i * A.D[1] + j) * A.D[2] + z;
}

// Interior cell number t (z fastest).
__device__ __forceinline__ void decode(const AdjArgs &A, int t, int &i, int &j, int &z)
{
    int a, b, c;
    region_index(t, A.bs[1], A.bs[2], a, b, c);
    i = a + NG;
    j = b + NG;
    z = c + NG;
}

__device__ __forceinline__ Geom<double> geom_at(const AdjArgs &A, int pos, uint32_t col)
{
    Geom<double> G;
#pragma unroll
    for (int s = 0; s < 10; s++) {
        G.gcov[s] = gld(A.gcov + ((int64_t)pos * 10 + s) * A.kcol, col);
        G.gcon[s] = gld(A.gcon + ((int64_t)pos * 10 + s) * A.kcol, col);
    }
    G.g = gld(A.gdet + (int64_t)pos * A.kcol, col);
    return G;
}

// 1 where a mass flux selects the lower side (the corner EMF's upwinding)
__device__ __forceinline__ double sel(const double *F, uint32_t g) { return (double)(gld(F, g) <= 0.0); }

// Adjoint of the field flux component of a face along DIR (stride sd) whose
// transverse direction has stride st: from the corner EMFs at both ends, e the
// EMF's adjoint and F the mass flux along the transverse direction.
__device__ __forceinline__ double field_flux(const double *e, const double *F, uint32_t g, uint32_t sd, uint32_t st)
{
    return 0.25 * (gld(e, g) * (1. + sel(F, g) + sel(F, g - sd))
                   + gld(e, g + st) * (3. - sel(F, g + st) - sel(F, g + st - sd)));
}

// Adjoint of a centre EMF component whose two transverse directions have strides
// sa, sb: from the four corners around the cell; Fa, Fb the mass fluxes along them.
__device__ __forceinline__ double centre_emf(const double *e, const double *Fa, const double *Fb, uint32_t g, uint32_t sa,
                                             uint32_t sb)
{
    const double a0 = sel(Fa, g), a1 = 1. - sel(Fa, g + sa), b0 = sel(Fb, g), b1 = 1. - sel(Fb, g + sb);
    return -0.25 * (gld(e, g) * (a0 + b0) + gld(e, g + sa) * (a1 + b0) + gld(e, g + sb) * (a0 + b1)
                    + gld(e, g + sa + sb) * (a1 + b1));
}

}  // namespace

// lE, the adjoint of the corner EMFs, at the corners [NG, NG + bs] (transpose of
// the face-field update and of the face average of U'[B]), and lps, the part of
// dL/dB_f that the updated face field carries over; zero in the ghosts.
__global__ void __launch_bounds__(256) k_adj_edge(AdjArgs A, const double *__restrict__ w, double *__restrict__ lE,
                                                  double *__restrict__ lps)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= A.D[0] * A.D[1] * A.D[2]) return;
    int i, j, z;
    region_index(t, A.D[1], A.D[2], i, j, z);
    if (i < NG || i > NG + A.bs[0] || j < NG || j > NG + A.bs[1] || z < NG || z > NG + A.bs[2]) {
        for (int d = 0; d < 3; d++) gst(lps + d * A.Kg, (uint32_t)t, 0.);
        return;
    }
    const int i0 = wrap1(i, A.bs[0]), j0 = wrap1(j, A.bs[1]), z0 = wrap1(z, A.bs[2]);
    const int im = wrap1(i0 - 1, A.bs[0]), jm = wrap1(j0 - 1, A.bs[1]), zm = wrap1(z0 - 1, A.bs[2]);
    const double *w0 = w + B1 * A.Kw, *w1 = w + B2 * A.Kw, *w2 = w + B3 * A.Kw;
    // face averages at the corner's cell c and its lower neighbours
    const uint32_t c = cell_of(A, i0, j0, z0), ci = cell_of(A, im, j0, z0), cj = cell_of(A, i0, jm, z0),
                   cz = cell_of(A, i0, j0, zm), cij = cell_of(A, im, jm, z0), ciz = cell_of(A, im, j0, zm),
                   cjz = cell_of(A, i0, jm, zm);
    const double v0 = 0.5 * (gld(w0, c) + gld(w0, ci)), v1 = 0.5 * (gld(w1, c) + gld(w1, cj)),
                 v2 = 0.5 * (gld(w2, c) + gld(w2, cz));
    const double v0j = 0.5 * (gld(w0, cj) + gld(w0, cij)), v0z = 0.5 * (gld(w0, cz) + gld(w0, ciz));
    const double v1i = 0.5 * (gld(w1, ci) + gld(w1, cij)), v1z = 0.5 * (gld(w1, cz) + gld(w1, cjz));
    const double v2i = 0.5 * (gld(w2, ci) + gld(w2, ciz)), v2j = 0.5 * (gld(w2, cj) + gld(w2, cjz));
    const double r1 = A.Dt / A.dx[0], r2 = A.Dt / A.dx[1], r3 = A.Dt / A.dx[2];
    gst(lE, (uint32_t)t, r3 * (v1 - v1z) - r2 * (v2 - v2j));
    gst(lE + A.K, (uint32_t)t, r1 * (v2 - v2i) - r3 * (v0 - v0z));
    gst(lE + 2 * A.K, (uint32_t)t, r2 * (v0 - v0j) - r1 * (v1 - v1i));
    const bool in = i == i0 && j == j0 && z == z0;
    const uint32_t col = (uint32_t)i * A.D[1] + j;
    gst(lps, (uint32_t)t, in ? gld(A.gdet + FACE1 * A.kcol, col) * v0 : 0.);
    gst(lps + A.Kg, (uint32_t)t, in ? gld(A.gdet + FACE2 * A.kcol, col) * v1 : 0.);
    gst(lps + 2 * A.Kg, (uint32_t)t, in ? gld(A.gdet + FACE3 * A.kcol, col) * v2 : 0.);
}

// lP (initialised here, zero in the ghosts) from U(P) and the centre EMF.
__global__ void __launch_bounds__(256) k_adj_cell(AdjArgs A, const double *__restrict__ p, const double *__restrict__ w,
                                                  const double *__restrict__ lE, const double *__restrict__ F1,
                                                  const double *__restrict__ F2, const double *__restrict__ F3,
                                                  double *__restrict__ lP)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= A.D[0] * A.D[1] * A.D[2]) return;
    int i, j, z;
    region_index(t, A.D[1], A.D[2], i, j, z);
    const uint32_t g = t;
    if (i < NG || i >= NG + A.bs[0] || j < NG || j >= NG + A.bs[1] || z < NG || z >= NG + A.bs[2]) {
        for (int k = 0; k < NPR; k++) gst(lP + k * A.Kg, g, 0.);
        return;
    }
    double pr[NPR], lU[NPR], lpr[NPR];
#pragma unroll
    for (int k = 0; k < NPR; k++) {
        const bool fld = k == B1 || k == B2 || k == B3;
        pr[k] = k == KTOT ? 0. : gld(p + k * A.K, g);
        lU[k] = fld ? 0. : gld(w + k * A.Kw, g);
    }
    const uint32_t sj = A.D[2], si = sj * A.D[1];
    const double e[3] = {centre_emf(lE, F2, F3, g, sj, 1), centre_emf(lE + A.K, F3, F1, g, 1, si),
                         centre_emf(lE + 2 * A.K, F2, F1, g, sj, si)};
    const Geom<double> G = geom_at(A, CENT, (uint32_t)i * A.D[1] + j);
    cell_vjp(pr, G, A.gam, lU, e, lpr);
    for (int k = 0; k < NPR; k++) gst(lP + k * A.Kg, g, lpr[k]);
}

// Reconstructed component number v of the faces along DIR.
template <int DIR> __device__ __forceinline__ constexpr int rec_comp(int v)
{
    return v < B1 ? v : v == 5 ? (DIR == 1 ? B2 : B1) : (DIR == 3 ? B2 : B3);
}

// One face of direction DIR: the flux's adjoint (from the divergence and the EMFs),
// HLL and the two face states, transposed into the adjoints of the face's
// reconstructed values: X[2 v] of the lower cell's upper value (left state), X[2 v
// + 1] of the upper cell's lower value; the normal field's goes into lps.
// Bound by the vector units and by latency: 2579 vector instructions a face (138 us
// of issue for the 128^3 box) at two waves per SIMD, the states of both sides being
// live across HLL; 305 us (790 us with the fluxes formed component by component,
// the partials of both parabolas per face and the sums by atomics).  The metric's
// loads moved up among the parabolas spill more: 342 us.
template <int DIR>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
k_adj_face(AdjArgs A, const double *__restrict__ p, const double *__restrict__ ps, const double *__restrict__ w,
           const double *__restrict__ lE, const double *__restrict__ F1, const double *__restrict__ F2,
           const double *__restrict__ F3, double *__restrict__ X, double *__restrict__ lps)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= A.n) return;
    int i, j, z;
    decode(A, t, i, j, z);
    const uint32_t g = cell_of(A, i, j, z), sj = A.D[2], si = sj * A.D[1];
    const uint32_t sd = DIR == 1 ? si : DIR == 2 ? sj : 1;
    double y[kAdjRec][6];
#pragma unroll
    for (int v = 0; v < kAdjRec; v++)
#pragma unroll
        for (int m = 0; m < 6; m++) y[v][m] = gld(p + rec_comp<DIR>(v) * A.K, g + (m - 3) * sd);
    const double bn = gld(ps + (DIR - 1) * A.K, g);
    const uint32_t gm = cell_of(A, DIR == 1 ? wrap1(i - 1, A.bs[0]) : i, DIR == 2 ? wrap1(j - 1, A.bs[1]) : j,
                                DIR == 3 ? wrap1(z - 1, A.bs[2]) : z);
    const double rate = A.Dt / A.dx[DIR - 1];
    double lf[NPR];
    bool any = false;
#pragma unroll
    for (int k = 0; k < NPR; k++)
        if (k < B1 || k == KTOT) lf[k] = rate * (gld(w + k * A.Kw, g) - gld(w + k * A.Kw, gm));
    lf[B1 + DIR - 1] = 0.;
    if (DIR == 1) {
        lf[B2] = -field_flux(lE + 2 * A.K, F2, g, si, sj);
        lf[B3] = field_flux(lE + A.K, F3, g, si, 1);
    } else if (DIR == 2) {
        lf[B3] = -field_flux(lE, F3, g, sj, 1);
        lf[B1] = field_flux(lE + 2 * A.K, F1, g, sj, si);
    } else {
        lf[B1] = -field_flux(lE + A.K, F1, g, 1, si);
        lf[B2] = field_flux(lE, F2, g, 1, sj);
    }
#pragma unroll
    for (int k = 0; k < NPR; k++) any |= lf[k] != 0.;
    if (!any) {  // nothing reaches the face: its states may be invalid
        for (int v = 0; v < 2 * kAdjRec; v++) gst(X + v * A.K, g, 0.);
        return;
    }
    double pl[NPR], pr[NPR], lpl[NPR], lpr[NPR], dum;
    pl[KTOT] = pr[KTOT] = 0.;
#pragma unroll
    for (int v = 0; v < kAdjRec; v++) {
        const int k = rec_comp<DIR>(v);
        para(y[v][0], y[v][1], y[v][2], y[v][3], y[v][4], dum, pl[k]);
        para(y[v][1], y[v][2], y[v][3], y[v][4], y[v][5], pr[k], dum);
    }
    pl[B1 + DIR - 1] = pr[B1 + DIR - 1] = bn;
    const Geom<double> G = geom_at(A, DIR == 1 ? FACE1 : DIR == 2 ? FACE2 : FACE3, (uint32_t)i * A.D[1] + j);
    hll_vjp(pl, pr, G, DIR, A.gam, lf, lpl, lpr);
    double *n = lps + (DIR - 1) * A.Kg;
    gst(n, g, gld(n, g) + (lpl[B1 + DIR - 1] + lpr[B1 + DIR - 1]));
#pragma unroll
    for (int v = 0; v < kAdjRec; v++) {
        gst(X + 2 * v * A.K, g, lpl[rec_comp<DIR>(v)]);
        gst(X + (2 * v + 1) * A.K, g, lpr[rec_comp<DIR>(v)]);
    }
}

// Reconstruction along x1 or x2, reverse: adds to lP what the face adjoints X of
// k_adj_face give through each cell's parabola, one component per blockIdx.y.  A
// thread takes `seg` cells of a line along DIR (lanes along z) and the two cells on
// either side, with the five sums that a parabola's stencil reaches in registers.
// Bound by memory: 128^3, 139 us for 0.6 GB (4.4 TB/s).  Tiles with the sums in LDS
// (28 cells of 16 z-lanes) took 194 us, segments of 16 cells with their loads not
// sent ahead 173.
template <int DIR>
__global__ void __launch_bounds__(256) k_adj_rec(AdjArgs A, const double *__restrict__ p, const double *__restrict__ X,
                                                 double *__restrict__ lP, int seg, int nseg)
{
    const int d = DIR - 1, o = 1 - d;  // this direction, the other of x1 and x2
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= nseg * A.bs[o] * A.bs[2]) return;
    int sg, a, z;
    region_index(t, A.bs[o], A.bs[2], sg, a, z);
    const int v = blockIdx.y, k = rec_comp<DIR>(v), n = A.bs[d];
    const double *q = p + k * A.K, *Xl = X + 2 * v * A.K, *Xr = Xl + A.K;
    double *out = lP + k * A.Kg;
    const uint32_t sj = A.D[2], si = sj * A.D[1], sd = DIR == 1 ? si : sj;
    const uint32_t base = cell_of(A, DIR == 1 ? NG : a + NG, DIR == 1 ? a + NG : NG, z + NG);
    const int c0 = sg * seg, len = n - c0 < seg ? n - c0 : seg;
    auto at = [&](int c) { return base + (c < 0 ? c + n : c >= n ? c - n : c) * sd; };
    double x[5], r[5] = {0., 0., 0., 0., 0.};
#pragma unroll
    for (int s = 0; s < 5; s++) x[s] = gld(q, at(c0 + s - 4));
    double ll = gld(Xr, at(c0 - 2)), lr = gld(Xl, at(c0 - 1));
#pragma unroll 2
    for (int m = -2; m < len + 2; m++) {
        // the next cell's values are on their way while this one's are worked on
        const double xn = gld(q, at(c0 + m + 3)), lln = gld(Xr, at(c0 + m + 1)), lrn = gld(Xl, at(c0 + m + 2));
        if (ll != 0. || lr != 0.) para_vjp(x, ll, lr, r);
        if (m >= 2) {
            const uint32_t g = base + (c0 + m - 2) * sd;
            gst(out, g, gld(out, g) + r[0]);
        }
#pragma unroll
        for (int s = 0; s < 4; s++) {
            r[s] = r[s + 1];
            x[s] = x[s + 1];
        }
        r[4] = 0.;
        x[4] = xn;
        ll = lln;
        lr = lrn;
    }
}

// The same along x3, a block taking `nrow` z-rows as a whole (len = bs3, halo = 0),
// or a window of len - 4 cells of one row with two on either side (halo = 2) where
// a row is longer than a block.
// Bound by memory: 128^3, 141 us (groups of 47 lanes with the sums by shuffles: 180).
constexpr int kAdjRow3 = 256;
__global__ void __launch_bounds__(kAdjRow3) k_adj_rec3(AdjArgs A, const double *__restrict__ p,
                                                       const double *__restrict__ X, double *__restrict__ lP, int len,
                                                       int nrow, int nwin, int halo)
{
    __shared__ double sh[4][kAdjRow3];
    const int t = threadIdx.x, sub = t / len, l = t - sub * len;
    const int row = blockIdx.x * nrow + sub;  // (i, j, window of the row)
    const bool live = sub < nrow && row < A.bs[0] * A.bs[1] * nwin;
    int i = 0, j = 0, win = 0;
    if (live) region_index(row, A.bs[1], nwin, i, j, win);
    const int v = blockIdx.y, k = rec_comp<3>(v);
    const int o = win * (len - 2 * halo) + l - halo;
    const int z = wrap1(NG + o, A.bs[2]);
    const uint32_t g = cell_of(A, i + NG, j + NG, z), gn = z + 1 == NG + A.bs[2] ? g + 1 - A.bs[2] : g + 1;
    double x[5], r[5] = {0., 0., 0., 0., 0.};
#pragma unroll
    for (int s = 0; s < 5; s++) x[s] = gld(p + k * A.K, g + s - 2);
    const double ll = gld(X + (2 * v + 1) * A.K, g), lr = gld(X + 2 * v * A.K, gn);
    if (ll != 0. || lr != 0.) para_vjp(x, ll, lr, r);
    sh[0][t] = r[0];
    sh[1][t] = r[1];
    sh[2][t] = r[3];
    sh[3][t] = r[4];
    __syncthreads();
    if (!live || l < halo || l >= len - halo || o >= A.bs[2]) return;
    // lanes of the cells at -2 .. 2: the row is periodic where the block holds all of it
    auto at = [&](int m) { const int q = l + m; return sub * len + (q < 0 ? q + len : q >= len ? q - len : q); };
    double sum = r[2] + (sh[3][at(-2)] + sh[2][at(-1)]);
    sum += sh[1][at(1)] + sh[0][at(2)];
    double *out = lP + k * A.Kg;
    gst(out, g, gld(out, g) + sum);
}

// ---------------------------------------------------------------------------
static inline dim3 g1(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

void launch_adjoint(const KParams &P, const BlockDev &B, double Dt, const double *p, const double *ps,
                    const double *F1, const double *F2, const double *F3, const double *w, int64_t Kw, double *lP,
                    double *lps, int64_t Kg, double *lE, double *X, hipStream_t s)
{
    AdjArgs A;
    for (int k = 0; k < 3; k++) {
        A.D[k] = B.D[k];
        A.bs[k] = B.bs[k];
        A.dx[k] = B.dx[k];
    }
    A.n = B.bs[0] * B.bs[1] * B.bs[2];
    A.K = B.ks;
    A.Kw = Kw;
    A.Kg = Kg;
    A.Dt = Dt;
    A.gam = P.gam;
    A.kcol = B.kcol;
    A.gcov = P.gcov + B.moff * NPOS * 10;
    A.gcon = P.gcon + B.moff * NPOS * 10;
    A.gdet = P.gdet + B.moff * NPOS;
    const int64_t N = (int64_t)A.D[0] * A.D[1] * A.D[2];
    // mass fluxes only: RHO is the first component
    hipLaunchKernelGGL(k_adj_edge, g1(N), dim3(256), 0, s, A, w, lE, lps);
    hipLaunchKernelGGL(k_adj_cell, g1(N), dim3(256), 0, s, A, p, w, lE, F1, F2, F3, lP);
    // the longest segments that still give the chip 4 wavefronts a SIMD, from 32
    // cells (4 cells of overlap in 32) down to 4: on 20x27x14 cells segments of 16
    // take 30 us, of 4 8 us; on 128^3 16 to 32 are alike
    int seg = 32;
    while (seg > 4 && (int64_t)kAdjRec * A.n / seg < 256 * 16 * 64) seg /= 2;
    int nseg[2];
    dim3 grec[2];
    for (int d = 0; d < 2; d++) {
        nseg[d] = (A.bs[d] + seg - 1) / seg;
        grec[d] = dim3((unsigned)(((int64_t)nseg[d] * A.bs[1 - d] * A.bs[2] + 255) / 256), kAdjRec);
    }
    hipLaunchKernelGGL(k_adj_face<1>, g1(A.n), dim3(256), 0, s, A, p, ps, w, lE, F1, F2, F3, X, lps);
    hipLaunchKernelGGL(k_adj_rec<1>, grec[0], dim3(256), 0, s, A, p, X, lP, seg, nseg[0]);
    hipLaunchKernelGGL(k_adj_face<2>, g1(A.n), dim3(256), 0, s, A, p, ps, w, lE, F1, F2, F3, X, lps);
    hipLaunchKernelGGL(k_adj_rec<2>, grec[1], dim3(256), 0, s, A, p, X, lP, seg, nseg[1]);
    hipLaunchKernelGGL(k_adj_face<3>, g1(A.n), dim3(256), 0, s, A, p, ps, w, lE, F1, F2, F3, X, lps);
    const int nwin = A.bs[2] <= kAdjRow3 ? 1 : (A.bs[2] + kAdjRow3 - 5) / (kAdjRow3 - 4), halo = nwin > 1 ? 2 : 0;
    const int len = (A.bs[2] + nwin - 1) / nwin + 2 * halo, nrow = kAdjRow3 / len;
    const int64_t nr = (int64_t)A.bs[0] * A.bs[1] * nwin;
    hipLaunchKernelGGL(k_adj_rec3, dim3((unsigned)((nr + nrow - 1) / nrow), kAdjRec), dim3((nrow * len + 63) / 64 * 64), 0,
                       s, A, p, X, lP, len, nrow, nwin, halo);
}

}  // namespace hamr
