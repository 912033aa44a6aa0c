// hamr_recon.h -- reconstruction, HLL flux and EMF kernels, templated on the
// arithmetic R of the face states (double: the FP64 step; float: the mixed
// step).  hamr_kernels.hip instantiates R = double, hamr_kernels_f32.hip
// R = float.  Both units are built without FMA contraction: the FP64 step
// follows the reference expression by expression, and in the FP32 fluxes
// contraction made the face-field error of one mixed step against the FP64
// step about 50 times larger (the corner EMFs difference fluxes of nearly
// equal size).
#pragma once

#include "hamr_hllc.h"
#include "hamr_kernels_dev.h"

namespace hamr {

// ---------------------------------------------------------------------------
// Fused PPM reconstruction + HLL flux through the lower dir-faces of a block:
// fluxcalcprep (GPU_program1.cu:78-190) and fluxcalc2D2 (:791-1068) in one pass,
// without the dq1/dq2 round trip through HBM.  Face range: [NG, NG+BS] along
// dir, [NG-1, NG+BS] across (the transverse ghost faces feed the corner EMFs).
//
// R is the arithmetic of reconstruction, state, fluxes and speeds: double for
// the FP64 step, float for the mixed step (primitives, face fields and metric
// are read in FP64 and rounded once; fluxes are stored as R).

// HLL flux through face `cell` (cell index of the face's upper cell; (i, j) its
// metric column) from the reconstructed states pl (lower side) and pr (upper
// side), fluxcalc2D2's flux and speed part (GPU_program1.cu:811-1045).  G: the
// metric at the face, bn: the face's normal field.  Stores the 9 fluxes, returns them
// in f and the face's largest signal speed.
template <int DIR, class R>
__device__ __forceinline__ R hll_face(const KParams &P, const BlockDev &B, const double *__restrict__ ps, R *pl,
                                      R *pr, int i, int j, int64_t cell, R *__restrict__ F, const Geom<R> &G,
                                      const R bn, R *f)
{
    const int64_t K = B.ks;
    pl[B1 + DIR - 1] = bn;
    pr[B1 + DIR - 1] = bn;
    if (DIR == 2 && (((B.pole & 1) && j == NG) || ((B.pole & 2) && j == NG + B.bs[1]))) {
        pl[B1] = R(0.);
        pr[B1] = R(0.);
    }
    const R gam = (R)P.gam;
    R t1[NPR], t2[NPR], t3[NPR], t4[NPR], cmax_l = R(0.), cmin_l = R(0.), cmax_r = R(0.), cmin_r = R(0.), dum;
    State<R> q;
    get_state(pl, G, q);
    primtoflux(pl, q, DIR, G, gam, t1, &cmax_l, &cmin_l);
    primtoflux(pl, q, 0, G, gam, t2, &dum, &dum);
    get_state(pr, G, q);
    primtoflux(pr, q, DIR, G, gam, t3, &cmax_r, &cmin_r);
    primtoflux(pr, q, 0, G, gam, t4, &dum, &dum);
    const R cmax = fabs(mymax(mymax(R(0.), cmax_l), cmax_r));
    const R cmin = fabs(mymax(mymax(R(0.), -cmin_l), -cmin_r));
    const R ctop = mymax(cmax, cmin);
    R *Fb = F + NPR * B.off;
    const Div<R> by_c(cmax + cmin + R(kSMALL));
#pragma unroll
    for (int k = 0; k < NPR; k++) {
        f[k] = by_c(cmax * t1[k] + cmin * t3[k] - cmax * cmin * (t4[k] - t2[k]));
        gst(Fb + (int64_t)k * K, (uint32_t)cell, f[k]);
    }
    return ctop;
}

// HLLC flux through the same face (fluxcalc2D_FT, GPU_hllc.h:3-247): the largest
// signal speed from the coordinate speeds as in hll_face, the flux from the
// orthonormal-frame solver of hamr_hllc.h with the face's tetrad.
template <int DIR, class R>
__device__ __forceinline__ R hllc_face(const KParams &P, const BlockDev &B, const double *__restrict__ ps, R *pl,
                                       R *pr, int i, int j, int64_t cell, R *__restrict__ F, const Geom<R> &G,
                                       const R bn, R *f)
{
    const int64_t K = B.ks;
    pl[B1 + DIR - 1] = bn;
    pr[B1 + DIR - 1] = bn;
    if (DIR == 2 && (((B.pole & 1) && j == NG) || ((B.pole & 2) && j == NG + B.bs[1]))) {
        pl[B1] = R(0.);
        pr[B1] = R(0.);
    }
    const int64_t col = (int64_t)i * B.D[1] + j;
    const R gam = (R)P.gam;
    State<R> ql, qr;
    get_state(pl, G, ql);
    get_state(pr, G, qr);
    R cmax_l, cmin_l, cmax_r, cmin_r;
    vchar_state(pl, ql, DIR, G, gam, &cmax_l, &cmin_l);
    vchar_state(pr, qr, DIR, G, gam, &cmax_r, &cmin_r);
    const R cmax = fabs(mymax(mymax(R(0.), cmax_l), cmax_r));
    const R cmin = fabs(mymax(mymax(R(0.), -cmin_l), -cmin_r));
    const R ctop = mymax(cmax, cmin);
    R mud[16], mudi[16];
    const double *T = P.tet + B.moff * 96 + (int64_t)(DIR - 1) * 32 * B.kcol + col;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        mud[e] = (R)T[(int64_t)e * B.kcol];
        mudi[e] = (R)T[(int64_t)(16 + e) * B.kcol];
    }
    R F1[NPR];
    hllc_frame_flux<DIR>(pl, pr, ql.ucon, ql.bcon, qr.ucon, qr.bcon, mud, mudi, face_velocity<DIR>(G.gcon), gam,
                         sizeof(R) == 4 ? G.oma : R(0.), F1);
    R *Fb = F + NPR * B.off + cell;
#pragma unroll
    for (int k = 0; k < NPR; k++) {
        f[k] = G.g * F1[k];
        Fb[(int64_t)k * K] = f[k];
    }
    return ctop;
}

// A wavefront's part in a Courant minimum, from its faces' largest signal speeds c (0:
// none): the step cour dx / c where it lies between 1e-6 and 1e9.  The quotient falls
// with c, so the faces' largest c gives their smallest step and one division serves the
// wavefront.
template <class R>
__device__ __forceinline__ void dt_reduce(const KParams &P, double dx, R c, unsigned long long *__restrict__ dtmin,
                                          int slot)
{
    const double cd = P.cour * dx;
    c = ((double)c > cd * 1.e-9 && (double)c < cd * 1.e6) ? c : R(0.);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) c = mymax(c, (R)__shfl_xor(c, off, 64));
    const double v = cd / (double)c;
    if ((threadIdx.x & 63) == 0 && v < 1.e9) atomicMin(&dtmin[slot], (unsigned long long)__double_as_longlong(v));
}

// The face's part in the blocks beside it along x1 and x2 (uniform grids): a face in
// the first or last row of a transverse direction is a ghost face of the block across
// that side, which does not compute it, and an x3 face at two sides one of the block
// across both.  Those blocks get its fluxes (share_face), and their Courant minima
// count it (share_dt, by the whole wavefront).  side[d]: the sides of direction d that
// the lane's face lies at, bit 0 the lower, bit 1 the upper.
template <int DIR, class R>
__device__ __forceinline__ void share_face(const KParams &P, const BlockDev &B, const int side[2], int cell, const R *f,
                                           R *__restrict__ F)
{
    const int64_t K = B.ks;
    int n[2], shift[2];
    auto put = [&](int m, int sh) {
        R *o = F + NPR * (m * K) + (cell + sh);
#pragma unroll
        for (int k = 0; k < NPR; k++) o[k * K] = f[k];
    };
#pragma unroll
    for (int d = 0; d < 2; d++) {
        if (d == DIR - 1 || !side[d]) continue;
        const bool lo = side[d] & 1;
        n[d] = lo ? B.nbr[2 * d] : B.nbr[2 * d + 1];
        shift[d] = (lo ? B.bs[d] : -B.bs[d]) * (d == 0 ? B.D[1] * B.D[2] : B.D[2]);
        put(n[d], shift[d]);
    }
    if (DIR == 3 && side[0] && side[1]) put(P.blk[n[0]].nbr[side[1] & 1 ? 2 : 3], shift[0] + shift[1]);
}
template <int DIR, class R>
__device__ __forceinline__ void share_dt(const KParams &P, const BlockDev &B, const int side[2], R c,
                                         unsigned long long *__restrict__ dtmin)
{
    if (!__any(side[0] | side[1])) return;
#pragma unroll
    for (int a = 0; a < 3; a++) {      // x1: beside, below, above
        if (DIR == 1 && a) continue;
#pragma unroll
        for (int b = 0; b < 3; b++) {  // x2
            if ((DIR == 2 && b) || (!a && !b)) continue;
            const bool in = (!a || (side[0] & a)) && (!b || (side[1] & b));
            if (!__any(in)) continue;
            int n = a ? B.nbr[a - 1] : B.nbr[2 + b - 1];
            if (a && b) n = P.blk[n].nbr[2 + b - 1];
            dt_reduce(P, B.dx[DIR - 1], in ? c : R(0.), dtmin, n * 3 + DIR - 1);
        }
    }
}

// One thread per face: both parabolas of the face's two cells.
//
// Bound by the float units (FP32: 1471-1543 instructions per face, x1, x2, x3 fluxes
// with the float unit busy 74, 78, 92% of the cycles, where float instructions alone
// reach 86-96%; FP64: 1.9e3, 55%, too few waves) and, beside it, by the latency of the
// stencil loads: the limiter's branches keep the compiler from moving a load above the
// previous variable's parabola, so that the 7 variables' loads waited one after another.
// The x1 faces read 2.8 GB where the others read 1.3-1.4 (384x192x192): a chunk of an XCD
// holds 3.5 of the planes that their stencils reach across.
// With all 42 issued first and the metric's 21 in the middle: x1, x2, x3 fluxes
// 418, 435, 400 -> 339, 346, 320 us (FP64, 256x128x128), 818, 855, 690 -> 768, 727,
// 594 us (mixed, 384x192x192).  At least 3 waves per SIMD (FP64: 162 VGPRs; FP32
// 92-104, four or five waves); held at four in FP64, or at five or six in FP32,
// they spill and run 8-25% slower.  Without the limiter's branches (selects) the
// loads are hoisted too far: spills, 15% slower.  A variant that marches each
// thread through a segment of faces along x1 or x2 and forms each cell's parabola
// once issues 29% fewer FP32 VALU instructions per face, but its carried state
// takes 157 registers (three waves) and it ran 7-35% slower.
// RS selects the Riemann solver: 0 HLL, 1 HLLC.  The FP64 HLLC kernel is held
// at two waves per SIMD (240 VGPRs, none spilled): 1.4x faster than one wave.  The
// FP32 HLLC kernel at four waves (128 VGPRs, 28 bytes of scratch) ran 4% faster than
// at three (139, none).
template <int DIR, class R, int RS, bool SHARE = false>
__device__ __forceinline__ void flux_item(const KParams &P, const int2 it, const double *__restrict__ p,
                                          const double *__restrict__ ps, R *__restrict__ F,
                                          unsigned long long *__restrict__ dtmin)
{
    const int n = it.x;
    const BlockDev &B = P.blk[n];
    // first face and number of faces along each direction: across DIR one ghost layer, with
    // SHARE along x1 and x2 only where no block of the grid is beyond that side
    int f0[3], nf[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const bool lo = d != DIR - 1 && !(SHARE && d < 2 && B.kind[2 * d] == FK_COPY);
        const bool hi = d != DIR - 1 && !(SHARE && d < 2 && B.kind[2 * d + 1] == FK_COPY);
        f0[d] = lo ? NG - 1 : NG;
        nf[d] = B.bs[d] + (d == DIR - 1 ? 1 : (int)lo + (int)hi);
    }
    const int t = it.y * blockDim.x + threadIdx.x;
    R ctop = R(0.);
    int side[2] = {0, 0};
    if (t < nf[0] * nf[1] * nf[2]) {
        int a, b, c;
        region_index(t, nf[1], nf[2], a, b, c);
        const int i = a + f0[0], j = b + f0[1], z = c + f0[2];
        const int64_t K = B.ks;
        const int64_t cell = ((int64_t)i * B.D[1] + j) * B.D[2] + z;
        const int64_t sd = (DIR == 1) ? (int64_t)B.D[1] * B.D[2] : (DIR == 2) ? (int64_t)B.D[2] : 1;
        const double *pb = p + NPR * B.off;
        R pl[NPR], pr[NPR];
        // every stencil value first, then the parabolas (KTOT enters no flux)
        double y[KTOT][6];
#pragma unroll
        for (int k = 0; k < KTOT; k++) {
            if (k == B1 + DIR - 1) continue;
            const double *q = pb + (int64_t)k * K;
#pragma unroll
            for (int m = 0; m < 6; m++) y[k][m] = gld(q + (m - 3) * sd, (uint32_t)cell);
        }
        auto one = [&](int k) {
            if (k == B1 + DIR - 1) return;  // the face-normal field comes from ps
            const R ym3 = (R)y[k][0], ym2 = (R)y[k][1], ym1 = (R)y[k][2], y0 = (R)y[k][3], yp1 = (R)y[k][4],
                    yp2 = (R)y[k][5];
            R l, r;
            para(ym3, ym2, ym1, y0, yp1, l, r);
            pl[k] = r;
            para(ym2, ym1, y0, yp1, yp2, l, r);
            pr[k] = l;
        };
#pragma unroll
        for (int k = 0; k < 4; k++) one(k);
        // the metric while the rest is reconstructed, in the registers the first stencils left
        const Geom<R> G = load_geom<R>(P, B, DIR == 1 ? FACE1 : DIR == 2 ? FACE2 : FACE3, (int64_t)i * B.D[1] + j);
        const R bn = (R)gld(ps + 3 * B.off + (DIR - 1) * K, (uint32_t)cell);
#pragma unroll
        for (int k = 4; k < KTOT; k++) one(k);
        R f[NPR];
        if constexpr (RS == 1) ctop = hllc_face<DIR>(P, B, ps, pl, pr, i, j, cell, F, G, bn, f);
        else ctop = hll_face<DIR>(P, B, ps, pl, pr, i, j, cell, F, G, bn, f);
        if constexpr (SHARE) {
            const int x[2] = {i, j};
#pragma unroll
            for (int d = 0; d < 2; d++)
                if (d != DIR - 1)
                    side[d] = (x[d] == NG && B.kind[2 * d] == FK_COPY ? 1 : 0)
                        | (x[d] == NG + B.bs[d] - 1 && B.kind[2 * d + 1] == FK_COPY ? 2 : 0);
            share_face<DIR>(P, B, side, (int)cell, f, F);
        }
    }
    if (dtmin) {
        dt_reduce(P, B.dx[DIR - 1], ctop, dtmin, n * 3 + DIR - 1);
        if constexpr (SHARE) share_dt<DIR>(P, B, side, ctop, dtmin);
    }
}

template <int DIR, class R, int RS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RS ? (sizeof(R) == 4 ? 4 : 2) : 3)))
k_flux(KParams P, WorkList wl, const double *__restrict__ p, const double *__restrict__ ps, R *__restrict__ F,
       unsigned long long *__restrict__ dtmin)
{
    FOR_ITEMS(wl) flux_item<DIR, R, RS>(P, wl_get(wl, w_), p, ps, F, dtmin);
}

// ---------------------------------------------------------------------------
// Line-staged reconstruction + Riemann flux: the faces, states and fluxes of
// k_flux, with each cell's MC slope and limited parabola formed once instead
// of once per face that reaches it.
//
// A work-list item is a tile (line_tiles): one segment of S consecutive faces
// along DIR on L consecutive lines of one row, a line being one transverse
// position of the face range, with one thread per cell of each line's S + 3
// cells f0 - 2 .. f0 + S (f0: the segment's first face, as the index of its
// upper cell).  In three steps, with a barrier between them:
//   1. every cell's MC slope from its own three-point stencil (read from
//      memory, rounded to R) into LDS;
//   2. cells f0 - 1 .. f0 + S - 1: the interface values of both boundaries
//      (the neighbours' slopes from LDS) and the limited parabola; the upper
//      edge goes to LDS, the lower edge stays in registers;
//   3. one thread per face (the face's upper cell): the lower cell's upper
//      edge from LDS and its own lower edge are the face states.
// Every value is para's expression on para's operands, so the states and
// fluxes are k_flux's bit for bit.  Thread t of a tile: line q and cell c
// (c = 0: cell f0 - 2) with t = c L + q for DIR = 1, 2 (consecutive threads
// on consecutive lines, i.e. consecutive z) and t = q (S + 3) + c for DIR = 3
// (consecutive threads along the z-row).  SC is the segment length when it is
// known at compile time (33: blocks of 32 or 64 cells along DIR; 17: 16
// cells), 0 otherwise.  A shorter last segment masks the cells past its faces.
template <int DIR, class R, int SC>
__device__ __forceinline__ void line_tile_states(const BlockDev &B, int item, const double *__restrict__ p, R *sm,
                                                 R *pl, R *pr, bool &fact, int64_t &cell, int &i, int &j)
{
    constexpr int T = kLineT, NV = NPR - 1;
    const int t = threadIdx.x;
    const LineTiles lt = line_tiles(B.bs[0], B.bs[1], B.bs[2], DIR);
    const int S = SC ? SC : lt.S, W = S + 3, L = SC ? T / (SC + 3) : lt.L;
    const int seg = item % lt.nseg, rest = item / lt.nseg, row = rest / lt.tpr, tb0 = (rest - row * lt.tpr) * L;
    const int nl = mymin(L, lt.n2 - tb0);
    const int nf = mymin(S, B.bs[DIR - 1] + 1 - seg * S);  // faces of this segment
    const int f0 = NG + seg * S;
    int q, c;
    if (DIR == 3) { q = t / W; c = t - q * W; }
    else { c = t / L; q = t - c * L; }
    const int sn = DIR == 3 ? 1 : L;  // LDS distance to the next cell along DIR
    const bool ok = q < nl && c < W;
    const bool slope = ok && c <= nf + 2, edge = ok && c >= 1 && c < nf + 2;
    fact = ok && c >= 2 && c < nf + 2;
    const int64_t D12 = (int64_t)B.D[1] * B.D[2];
    const int64_t sdir = DIR == 1 ? D12 : DIR == 2 ? (int64_t)B.D[2] : 1;
    const int64_t sq = DIR == 3 ? (int64_t)B.D[2] : 1;  // between consecutive lines of a row
    const int ta = row + NG - 1, tb = tb0 + NG - 1;
    const int64_t base = DIR == 1 ? (int64_t)ta * B.D[2] + tb : DIR == 2 ? (int64_t)ta * D12 + tb
                                                                         : (int64_t)ta * D12 + (int64_t)tb * B.D[2];
    const int pos = f0 - 2 + c;  // this thread's cell along DIR
    cell = base + q * sq + (int64_t)pos * sdir;
    i = DIR == 1 ? pos : ta;  // the face's metric column (i, j)
    j = DIR == 1 ? ta : DIR == 2 ? pos : tb + q;
    R *const DQ = sm, *const RE = sm + NV * T;
    const int64_t K = B.ks;
    const double *pc = p + NPR * B.off + cell;
    R ym[NV], y0[NV], yp[NV], dq[NV];
#pragma unroll
    for (int k = 0, v = 0; k < NPR; k++) {
        if (k == B1 + DIR - 1) continue;  // the face-normal field comes from ps
        if (slope) {
            const double *y = pc + (int64_t)k * K;
            ym[v] = (R)y[-sdir];
            y0[v] = (R)y[0];
            yp[v] = (R)y[sdir];
            dq[v] = mc_slope(ym[v], y0[v], yp[v]);
            DQ[v * T + t] = dq[v];
        }
        v++;
    }
    __syncthreads();
    R le[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
        if (edge) {
            R l, r;
            ppm_limit(y0[v], ppm_face(ym[v], y0[v], DQ[v * T + t - sn], dq[v]),
                      ppm_face(y0[v], yp[v], dq[v], DQ[v * T + t + sn]), l, r);
            le[v] = l;
            RE[v * T + t] = r;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0, v = 0; k < NPR; k++) {
        if (k == B1 + DIR - 1) continue;
        if (fact) {
            pl[k] = RE[v * T + t - sn];
            pr[k] = le[v];
        }
        v++;
    }
}

// Occupancy: four waves per SIMD in FP32 (128 VGPRs), two in FP64 (256 VGPRs and
// 360-552 bytes of scratch, HLLC 644-844).  The LDS of one tile:
// 2 (NPR - 1) kLineT values of R.
template <int DIR, class R, int RS>
__global__ void __launch_bounds__(kLineT) __attribute__((amdgpu_waves_per_eu(RS || sizeof(R) == 8 ? 2 : 4)))
k_flux_lines(KParams P, WorkList wl, const double *__restrict__ p, const double *__restrict__ ps, R *__restrict__ F,
             unsigned long long *__restrict__ dtmin)
{
    extern __shared__ double smem_d[];
    R *const sm = reinterpret_cast<R *>(smem_d);
    FOR_ITEMS(wl)
    {
        const int2 it = wl_get(wl, w_);
        const int n = it.x;
        const BlockDev &B = P.blk[n];
        const int nfd = B.bs[DIR - 1] + 1;
        R pl[NPR], pr[NPR];
        bool fact;
        int64_t cell;
        int i, j;
        if (nfd == 33 || nfd == 65) line_tile_states<DIR, R, 33>(B, it.y, p, sm, pl, pr, fact, cell, i, j);
        else if (nfd == 17) line_tile_states<DIR, R, 17>(B, it.y, p, sm, pl, pr, fact, cell, i, j);
        else line_tile_states<DIR, R, 0>(B, it.y, p, sm, pl, pr, fact, cell, i, j);
        R ctop = R(0.);
        if (fact) {
            const Geom<R> G = load_geom<R>(P, B, DIR == 1 ? FACE1 : DIR == 2 ? FACE2 : FACE3, (int64_t)i * B.D[1] + j);
            const R bn = (R)ps[3 * B.off + (DIR - 1) * (int64_t)B.ks + cell];
            R f[NPR];
            if constexpr (RS == 1) ctop = hllc_face<DIR>(P, B, ps, pl, pr, i, j, cell, F, G, bn, f);
            else ctop = hll_face<DIR>(P, B, ps, pl, pr, i, j, cell, F, G, bn, f);
        }
        if (dtmin) dt_reduce(P, B.dx[DIR - 1], ctop, dtmin, n * 3 + DIR - 1);
        // the next item's first barrier orders its LDS writes after these reads
    }
}

// ---------------------------------------------------------------------------
// Cell-centre EMF, consttransport1 (GPU_const_trans.h:63-119), cells [NG-1, NG+BS].
template <class R>
__device__ __forceinline__ void emf_centre_item(const KParams &P, const int2 it, const double *__restrict__ p,
                                                R *__restrict__ Ec)
{
    const BlockDev &B = P.blk[it.x];
    const int e1 = B.bs[0] + 2, e2 = B.bs[1] + 2, e3 = B.bs[2] + 2;
    const int t = it.y * blockDim.x + threadIdx.x;
    if (t >= e1 * e2 * e3) return;
    int a, b, c;
    region_index(t, e2, e3, a, b, c);
    const int i = a + NG - 1, j = b + NG - 1, z = c + NG - 1;
    const int64_t K = B.ks;
    const int64_t cell = ((int64_t)i * B.D[1] + j) * B.D[2] + z;
    const double *pb = p + NPR * B.off + cell;
    R pr[NPR];
#pragma unroll
    for (int k = 0; k < NPR; k++) pr[k] = (R)pb[(int64_t)k * K];
    const Geom<R> G = load_geom<R>(P, B, CENT, (int64_t)i * B.D[1] + j);
    R ucon[4], ucov[4], bcon[4];
    ucon_calc(pr, G, ucon);
    lower10(ucon, G.gcov, ucov);
    bcon_calc(pr, ucon, ucov, bcon);
    R *E = Ec + 3 * B.off + cell;
    E[0] = -G.g * (ucon[2] * bcon[3] - ucon[3] * bcon[2]);
    E[K] = -G.g * (ucon[3] * bcon[1] - ucon[1] * bcon[3]);
    E[2 * K] = -G.g * (ucon[1] * bcon[2] - ucon[2] * bcon[1]);
}

template <class R>
__global__ void __launch_bounds__(256) k_emf_centre(KParams P, WorkList wl, const double *__restrict__ p,
                                                    R *__restrict__ Ec)
{
    FOR_ITEMS(wl) emf_centre_item(P, wl_get(wl, w_), p, Ec);
}

// The three fluxes and the centre EMFs in one launch.  They depend on nothing of each
// other, so that a class's blocks start while the last ones of the class before
// still run, where as four launches each waited for the slowest block of the one
// before with the chip draining (a flux block runs 10 us or more on its own, and a
// grid of 64x32x32 zones fills the chip once).  The classes follow one another, the
// light one last; FP32 launches of four chunks or more per class go chunk by chunk,
// so that the primitives of a region come from the memory-side cache for three of
// their four readings (FP64 fluxes issue too long for that to show: 256x128x128
// 3.86 and 3.88 ms a step).  Classes in turn from one workgroup to the next run 8-20%
// slower: the three flux bodies do not fit the instruction cache together.
// Per pass, four launches -> one: 64x32x32 FP64 1.93 -> 1.66 ms, 42x25x39 blocks 4.82
// -> 4.28, 256x128x128 17.0 -> 16.5, HLLC 96x72x60 3.11 -> 2.71; mixed 384x192x192
// 42.5 -> 40.1, HLLC 256x128x128 14.8 -> 13.4; the step of 384x192x192 by chunk
// (items of 256): all 9.78 ms, 16384 9.72, 8192 9.53, 4096 9.32, 2048 9.40, 1024 9.45.
//
// SHARE (uniform grids): ghost faces along x1 and x2 beyond a side with a block are
// computed by that block only, which writes all their fluxes to both: 8% fewer faces on
// 32^3 blocks, 20% on 16x8x8.  Without and with it, ms a pass: 42x25x39 blocks FP64 4.18,
// 4.13; 256x128x128 FP64 16.03, 15.75, HLLC mixed 13.31, 13.18; HLLC 96x72x60 2.64, 2.58;
// 384x192x192 mixed 40.18, 39.86.  (With only the fluxes written that the face update's
// EMFs read: 0.1-0.7% less time, but stale values left in HAMR_F1-F3 and on edges of
// HAMR_EMF.)  Along x3 as well the blocks would write single values into the rows beside
// them: no faster than computing the two faces more per row (384x192x192 2.09 and 2.07
// ms a launch).
constexpr int kFrontChunk = 1 << 20;  // threads: 8192 items of the default 128
template <class R, int RS, bool SHARE>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RS ? (sizeof(R) == 4 ? 4 : 2) : 3)))
k_front(KParams P, FrontLists L, const double *__restrict__ p, const double *__restrict__ ps, R *__restrict__ F1,
        R *__restrict__ F2, R *__restrict__ F3, unsigned long long *__restrict__ dtmin, R *__restrict__ Ec)
{
    const int w = blockIdx.x;
    int cls, idx;
    if (w < 4 * L.chunked) {
        const int chunk = kFrontChunk / (int)blockDim.x, q = w / chunk;
        cls = q & 3;
        idx = (q >> 2) * chunk + (w - q * chunk);
    } else {
        idx = w - 4 * L.chunked;
        for (cls = 0; cls < 3 && idx >= L.wl[cls].n - L.chunked; cls++) idx -= L.wl[cls].n - L.chunked;
        idx += L.chunked;
    }
    const int2 it = wl_get(L.wl[cls], idx);
    if (cls == 0) flux_item<1, R, RS, SHARE>(P, it, p, ps, F1, dtmin);
    else if (cls == 1) flux_item<2, R, RS, SHARE>(P, it, p, ps, F2, dtmin);
    else if (cls == 2) flux_item<3, R, RS, SHARE>(P, it, p, ps, F3, dtmin);
    else emf_centre_item(P, it, p, Ec);
}

// Corner EMF upwinded on the mass-flux sign, consttransport2
// (GPU_const_trans.h:121-339) with the polar rule (:233-236); corners [NG, NG+BS].
template <class R>
__global__ void __launch_bounds__(256) k_emf_corner(KParams P, WorkList wl, const R *__restrict__ Ec,
                                                    const R *__restrict__ F1, const R *__restrict__ F2,
                                                    const R *__restrict__ F3, R *__restrict__ E)
{
    FOR_ITEMS(wl)
    {
        const int2 it = wl_get(wl, w_);
        const BlockDev &B = P.blk[it.x];
        const int e1 = B.bs[0] + 1, e2 = B.bs[1] + 1, e3 = B.bs[2] + 1;
        const int t = it.y * blockDim.x + threadIdx.x;
        if (t >= e1 * e2 * e3) continue;
        int a, b, c;
        region_index(t, e2, e3, a, b, c);
        const int i = a + NG, j = b + NG, z = c + NG;
        const int64_t g = ((int64_t)i * B.D[1] + j) * B.D[2] + z;
        const int64_t K = B.ks, si = (int64_t)B.D[1] * B.D[2], sj = B.D[2];
        const R *E1c = Ec + 3 * B.off, *E2c = E1c + K, *E3c = E2c + K;
        const R *f1 = F1 + NPR * B.off, *f2 = F2 + NPR * B.off, *f3 = F3 + NPR * B.off;
        const R *F1R = f1 + RHO * K, *F2R = f2 + RHO * K, *F3R = f3 + RHO * K;
        const R *F1B2 = f1 + B2 * K, *F1B3 = f1 + B3 * K;
        const R *F2B1 = f2 + B1 * K, *F2B3 = f2 + B3 * K;
        const R *F3B1 = f3 + B1 * K, *F3B2 = f3 + B2 * K;
        const R dEL13_1 = E1c[g] - F3B2[g];
        const R dEL13_2 = E1c[g - sj] - F3B2[g - sj];
        const R dER13_1 = F3B2[g] - E1c[g - 1];
        const R dER13_2 = F3B2[g - sj] - E1c[g - sj - 1];
        const R dEL12_1 = E1c[g] + F2B3[g];
        const R dEL12_2 = E1c[g - 1] + F2B3[g - 1];
        const R dER12_1 = -F2B3[g] - E1c[g - sj];
        const R dER12_2 = -F2B3[g - 1] - E1c[g - sj - 1];
        const R dEL21_1 = E2c[g] - F1B3[g];
        const R dEL21_2 = E2c[g - 1] - F1B3[g - 1];
        const R dER21_1 = F1B3[g] - E2c[g - si];
        const R dER21_2 = F1B3[g - 1] - E2c[g - si - 1];
        const R dEL23_1 = E2c[g] + F3B1[g];
        const R dEL23_2 = E2c[g - si] + F3B1[g - si];
        const R dER23_1 = -F3B1[g] - E2c[g - 1];
        const R dER23_2 = -F3B1[g - si] - E2c[g - si - 1];
        const R dEL31_1 = E3c[g] + F1B2[g];
        const R dEL31_2 = E3c[g - sj] + F1B2[g - sj];
        const R dER31_1 = -F1B2[g] - E3c[g - si];
        const R dER31_2 = -F1B2[g - sj] - E3c[g - si - sj];
        const R dEL32_1 = E3c[g] - F2B1[g];
        const R dEL32_2 = E3c[g - si] - F2B1[g - si];
        const R dER32_1 = F2B1[g] - E3c[g - sj];
        const R dER32_2 = F2B1[g - si] - E3c[g - si - sj];
#define LE(x) ((R)((x) <= R(0.)))
#define GT(x) ((R)((x) > R(0.)))
        R e1v = R(0.25) * ((-F2B3[g] - (dEL13_1 * LE(F2R[g]) + dEL13_2 * GT(F2R[g])))
            + (-F2B3[g - 1] + (dER13_1 * LE(F2R[g - 1]) + dER13_2 * GT(F2R[g - 1])))
            + (F3B2[g] - (dEL12_1 * LE(F3R[g]) + dEL12_2 * GT(F3R[g])))
            + (F3B2[g - sj] + (dER12_1 * LE(F3R[g - sj]) + dER12_2 * GT(F3R[g - sj]))));
        const R e2v = R(0.25) * ((-F3B1[g] - (dEL21_1 * LE(F3R[g]) + dEL21_2 * GT(F3R[g])))
            + (-F3B1[g - si] + (dER21_1 * LE(F3R[g - si]) + dER21_2 * GT(F3R[g - si])))
            + (F1B3[g] - (dEL23_1 * LE(F1R[g]) + dEL23_2 * GT(F1R[g])))
            + (F1B3[g - 1] + (dER23_1 * LE(F1R[g - 1]) + dER23_2 * GT(F1R[g - 1]))));
        R e3v = R(0.25) * ((F2B1[g] - (dEL31_1 * LE(F2R[g]) + dEL31_2 * GT(F2R[g])))
            + (F2B1[g - si] + (dER31_1 * LE(F2R[g - si]) + dER31_2 * GT(F2R[g - si])))
            + (-F1B2[g] - (dEL32_1 * LE(F1R[g]) + dEL32_2 * GT(F1R[g])))
            + (-F1B2[g - sj] + (dER32_1 * LE(F1R[g - sj]) + dER32_2 * GT(F1R[g - sj]))));
#undef LE
#undef GT
        if (((B.pole & 1) && j == NG) || ((B.pole & 2) && j == NG + B.bs[1])) {
            e3v = R(0.);
            e1v = R(-0.5) * (F2B3[g] + F2B3[g - 1]);
        }
        R *Eb = E + 3 * B.off + g;
        Eb[0] = e1v;
        Eb[K] = e2v;
        Eb[2 * K] = e3v;
    }
}

// Launchers of one arithmetic (R = double here and in hamr_kernels.hip, R =
// float in hamr_kernels_f32.hip).
template <int DIR, class R, int RS>
static void launch_flux_lines(const KParams &P, const Launch &L, const double *p, const double *ps, R *F,
                              unsigned long long *dtmin, hipStream_t s)
{
    const size_t lds = (size_t)2 * (NPR - 1) * kLineT * sizeof(R);
    hipLaunchKernelGGL((k_flux_lines<DIR, R, RS>), gdim(L), bdim(L), lds, s, P, L.wl, p, ps, F, dtmin);
}

template <class R>
void recon_flux(const KParams &P, int dir, const Launch &L, const double *p, const double *ps, R *F,
                unsigned long long *dtmin, hipStream_t s)
{
    if (L.wl.n <= 0) return;
    if (L.line) {
        if (P.riemann == 1) {
            if (dir == 1) launch_flux_lines<1, R, 1>(P, L, p, ps, F, dtmin, s);
            else if (dir == 2) launch_flux_lines<2, R, 1>(P, L, p, ps, F, dtmin, s);
            else launch_flux_lines<3, R, 1>(P, L, p, ps, F, dtmin, s);
            return;
        }
        if (dir == 1) launch_flux_lines<1, R, 0>(P, L, p, ps, F, dtmin, s);
        else if (dir == 2) launch_flux_lines<2, R, 0>(P, L, p, ps, F, dtmin, s);
        else launch_flux_lines<3, R, 0>(P, L, p, ps, F, dtmin, s);
        return;
    }
    if (P.riemann == 1) {
        if (dir == 1) hipLaunchKernelGGL((k_flux<1, R, 1>), gdim(L), bdim(L), 0, s, P, L.wl, p, ps, F, dtmin);
        else if (dir == 2) hipLaunchKernelGGL((k_flux<2, R, 1>), gdim(L), bdim(L), 0, s, P, L.wl, p, ps, F, dtmin);
        else hipLaunchKernelGGL((k_flux<3, R, 1>), gdim(L), bdim(L), 0, s, P, L.wl, p, ps, F, dtmin);
        return;
    }
    if (dir == 1) hipLaunchKernelGGL((k_flux<1, R, 0>), gdim(L), bdim(L), 0, s, P, L.wl, p, ps, F, dtmin);
    else if (dir == 2) hipLaunchKernelGGL((k_flux<2, R, 0>), gdim(L), bdim(L), 0, s, P, L.wl, p, ps, F, dtmin);
    else hipLaunchKernelGGL((k_flux<3, R, 0>), gdim(L), bdim(L), 0, s, P, L.wl, p, ps, F, dtmin);
}

template <class R>
void recon_front(const KParams &P, const Launch *L, bool share, const double *p, const double *ps, R *F1, R *F2,
                 R *F3, unsigned long long *dtmin, R *Ec, hipStream_t s)
{
    FrontLists f;
    int n = 0;
    for (int k = 0; k < 4; k++) {
        f.wl[k] = L[k].wl;
        n += L[k].wl.n;
    }
    f.chunked = L[0].wl.n;
    for (int k = 1; k < 4; k++) f.chunked = L[k].wl.n < f.chunked ? L[k].wl.n : f.chunked;
    const int chunk = kFrontChunk / L[0].threads;
    f.chunked = sizeof(R) == 4 && f.chunked >= 4 * chunk ? f.chunked / chunk * chunk : 0;
    if (n <= 0) return;
    const dim3 g((unsigned)n), b = bdim(L[0]);
    if (P.riemann == 1) {
        if (share) hipLaunchKernelGGL((k_front<R, 1, true>), g, b, 0, s, P, f, p, ps, F1, F2, F3, dtmin, Ec);
        else hipLaunchKernelGGL((k_front<R, 1, false>), g, b, 0, s, P, f, p, ps, F1, F2, F3, dtmin, Ec);
    } else {
        if (share) hipLaunchKernelGGL((k_front<R, 0, true>), g, b, 0, s, P, f, p, ps, F1, F2, F3, dtmin, Ec);
        else hipLaunchKernelGGL((k_front<R, 0, false>), g, b, 0, s, P, f, p, ps, F1, F2, F3, dtmin, Ec);
    }
}

template <class R>
void recon_emf_centre(const KParams &P, const Launch &L, const double *p, R *Ec, hipStream_t s)
{
    if (L.wl.n <= 0) return;
    hipLaunchKernelGGL((k_emf_centre<R>), gdim(L), bdim(L), 0, s, P, L.wl, p, Ec);
}

template <class R>
void recon_emf_corner(const KParams &P, const Launch &L, const R *Ec, const R *F1, const R *F2, const R *F3, R *E,
                      hipStream_t s)
{
    if (L.wl.n <= 0) return;
    hipLaunchKernelGGL((k_emf_corner<R>), gdim(L), bdim(L), 0, s, P, L.wl, Ec, F1, F2, F3, E);
}

// The FP32 instantiations (hamr_kernels_f32.hip).
void launch_flux_f32(const KParams &P, int dir, const Launch &L, const double *p, const double *ps, float *F,
                     unsigned long long *dtmin, hipStream_t s);
void launch_front_f32(const KParams &P, const Launch *L, bool share, const double *p, const double *ps, float *F1,
                      float *F2, float *F3, unsigned long long *dtmin, float *Ec, hipStream_t s);
void launch_emf_centre_f32(const KParams &P, const Launch &L, const double *p, float *Ec, hipStream_t s);
void launch_emf_corner_f32(const KParams &P, const Launch &L, const float *Ec, const float *F1, const float *F2,
                           const float *F3, float *E, hipStream_t s);

}  // namespace hamr
