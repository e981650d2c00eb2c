// Implicit energy step on the GPU: the matrix of EnergyDirectSolve
// (ThermalRoutines.c:185-390, theta = 1, transient, no air cells) applied
// matrix-free from the cell-face conductivities, solved with the
// Jacobi-preconditioned CG of SolveThermalPCG (ThermalSolver.c:338-480)
// started from the current temperature.
//
// Per iteration two launches on the context's stream:
//   apply  : the previous iteration's ||r|| / ||r0|| test, breakdown -3,
//            iteration limit and beta; p = z + beta p_old on the cell and its
//            four neighbours (the direction update, folded in here), q = A p,
//            block partials of p.q;
//   update : alpha = rz / p.q (breakdown -2); x += alpha p, r -= alpha q,
//            z = M^-1 r, block partials of r.r and r.z.
// Every block sums the previous kernel's partials itself, in one fixed order
// (at most TH_BLOCKS of them, read from L2), and takes the same decision;
// block 0 writes it down for the next kernel.  One-block kernels for those
// sums over 16k partials took 46 of an iteration's 144 us at 2047^2, and two
// launches of the four on small grids.  Once the control block says "done"
// every later launch returns at once, so the host queues iterations in
// batches and reads the control block between batches only.  Products and
// sums within a cell follow the reference's CSR row order (south, west,
// centre, east, north), so only the dot-product reductions round differently.
//
// Bound: memory.  apply streams 7 arrays of a cell (z, p_old, kx, kz, diag
// read, p, q written), update 8 (p, q, r, x, minv read, x, r, z written).
// Measured at 2047^2: apply 66 us, update 44 us (3.6 and 6.1 TB/s, the second
// helped by the last-level cache), against 57 + 16 + 38 + 30 us for the four
// kernels.  2048 blocks, or two or four cells of a thread loaded before any is
// stored, measured 70-77 and 47-49 us: the blocks then spread over more rows.
#include <cmath>

#include "mdg_internal.h"

namespace {

constexpr int TB = 512;

// State between kernels: [0] written by update (and the set-up), [1] by apply.
struct th_ctl {
    double rz, r0, rel_tol, alpha, beta;
    int done, its, it, max_its;
};

struct th_geom {
    int ncx, ncz, nx, nxvz;
    double idx2, idz2, dx;
};

// At most this many blocks (4 per CU, all resident).  Blocks are dispatched
// round-robin over the 8 XCDs; each XCD takes a contiguous band of the cells
// and its blocks walk it side by side in steps of TB, so that the rows above
// and below a block's cells are in the same L2 as the blocks that read them.
constexpr int TH_BLOCKS = 1024;
struct th_share {
    int lo, hi, step;      // cells lo + threadIdx.x, + step, ... below hi
};
__device__ inline th_share th_cells(int n) {
    const int nb = gridDim.x, xcd = blockIdx.x & 7, per = nb >> 3, rem = nb & 7;
    const int first = xcd * per + min(xcd, rem), mine = per + (xcd < rem ? 1 : 0);   // the XCD's blocks
    const long steps = (n + TB - 1) / TB;
    const int lo = (int)(steps * first / nb), hi = (int)(steps * (first + mine) / nb);
    return th_share{(lo + (int)(blockIdx.x >> 3)) * TB, min(n, hi * TB), mine * TB};
}

// Sums of a and b over the block, in every thread.
struct sum2 {
    double a, b;
};
__device__ inline sum2 block_sum2(double a, double b, double (*s)[2]) {
    for (int w = 32; w > 0; w >>= 1) {
        a += __shfl_xor(a, w);
        b += __shfl_xor(b, w);
    }
    if ((threadIdx.x & 63) == 0) {
        s[threadIdx.x >> 6][0] = a;
        s[threadIdx.x >> 6][1] = b;
    }
    __syncthreads();
    sum2 t{0.0, 0.0};
    for (int w = 0; w < TB / 64; w++) {
        t.a += s[w][0];
        t.b += s[w][1];
    }
    __syncthreads();
    return t;
}
// Totals of nb <= TH_BLOCKS partials, the same in every block and thread.
__device__ inline sum2 part_sum2(int nb, const double *__restrict__ pa, const double *__restrict__ pb, double (*s)[2]) {
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < nb; i += TB) {
        a += pa[i];
        if (pb) b += pb[i];
    }
    return block_sum2(a, b, s);
}

// Diagonal and boundary right-hand side of cell (k, l), in the order of the
// reference's assembly.
__device__ inline void th_diag(const th_geom &g, double rhoCp_dt, const double *__restrict__ kx,
                               const double *__restrict__ kz, const signed char *__restrict__ BT,
                               const double *__restrict__ BV, int k, int l, double *d, double *bbc) {
    const int c0 = (k + 1) + (l + 1) * (g.ncx + 2), c1 = k + (l + 1) * g.nx, c3 = k + l * g.nxvz + 1;
    const double AW = kx[c1], AE = kx[c1 + 1], AS = kz[c3], AN = kz[c3 + g.nxvz];
    double val = rhoCp_dt, b = 0.0;
    if (l > 0) val += AS * g.idz2;
    if (k > 0) val += AW * g.idx2;
    if (k < g.ncx - 1) val += AE * g.idx2;
    if (l < g.ncz - 1) val += AN * g.idz2;
    if (l == 0 && BT[c0 - (g.ncx + 2)] == 1) {
        val += 2.0 * AS * g.idz2;
        b += 2.0 * AS * g.idz2 * BV[c0 - (g.ncx + 2)];
    }
    if (l == 0 && BT[c0 - (g.ncx + 2)] == 0) b += -1.0 / g.dx * BV[c0 - (g.ncx + 2)];
    if (k == 0 && BT[c0 - 1] == 1) {
        val += 2.0 * AW * g.idx2;
        b += 2.0 * AW * g.idx2 * BV[c0 - 1];
    }
    if (k == g.ncx - 1 && BT[c0 + 1] == 1) {
        val += 2.0 * AE * g.idx2;
        b += 2.0 * AE * g.idx2 * BV[c0 + 1];
    }
    if (l == g.ncz - 1 && BT[c0 + (g.ncx + 2)] == 1) {
        val += 2.0 * AN * g.idz2;
        b += 2.0 * AN * g.idz2 * BV[c0 + (g.ncx + 2)];
    }
    *d = val;
    *bbc = b;
}

// Row c2 = (k, l) of A times v, with P(j) giving v at cell j.  At a wall the
// neighbour is the cell itself with a zero coefficient: its product adds a
// zero, and the loads of all five cells stay free of branches.
template <typename F>
__device__ inline double th_row(const th_geom &g, const double *__restrict__ kx, const double *__restrict__ kz,
                                double d, int k, int l, int c2, F P) {
    const int c1 = k + (l + 1) * g.nx, c3 = k + l * g.nxvz + 1;
    const bool S = l > 0, W = k > 0, E = k < g.ncx - 1, N = l < g.ncz - 1;
    const double aS = S ? -kz[c3] * g.idz2 : 0.0, aW = W ? -kx[c1] * g.idx2 : 0.0;
    const double aE = E ? -kx[c1 + 1] * g.idx2 : 0.0, aN = N ? -kz[c3 + g.nxvz] * g.idz2 : 0.0;
    double s = 0.0;
    s += aS * P(S ? c2 - g.ncx : c2);
    s += aW * P(W ? c2 - 1 : c2);
    s += d * P(c2);
    s += aE * P(E ? c2 + 1 : c2);
    s += aN * P(N ? c2 + g.ncx : c2);
    return s;
}

struct th_in {
    const double *rho, *Cp, *Qr, *Wd, *Ha, *kx, *kz, *BV;
    const signed char *BT;
};

// b, diag, M^-1, r = b - A x, z = M^-1 r, p = z; partials of r.r and r.z.
__global__ void __launch_bounds__(TB) k_th_setup(th_geom g, double dt, th_in in, const double *__restrict__ x,
                                                 double *__restrict__ diag, double *__restrict__ minv,
                                                 double *__restrict__ r, double *__restrict__ z,
                                                 double *__restrict__ p, double *__restrict__ part_rr,
                                                 double *__restrict__ part_rz) {
    __shared__ double s[TB / 64][2];
    const int n = g.ncx * g.ncz;
    const th_share c = th_cells(n);
    double rz = 0.0, rr = 0.0;
    for (int c2 = c.lo + threadIdx.x; c2 < c.hi; c2 += c.step) {
        const int k = c2 % g.ncx, l = c2 / g.ncx;
        const double rhoCp = in.rho[c2] * in.Cp[c2];
        double d, bbc;
        th_diag(g, rhoCp / dt, in.kx, in.kz, in.BT, in.BV, k, l, &d, &bbc);
        double b = rhoCp * x[c2] / dt;
        b += 1.0 * (in.Qr ? in.Qr[c2] : 0.0);
        if (in.Wd) b += in.Wd[c2];
        if (in.Ha) b += in.Ha[c2];
        b += 1.0 * bbc;
        const double mi = (fabs(d) > 1e-30) ? 1.0 / d : 1.0;
        const double ri = b - th_row(g, in.kx, in.kz, d, k, l, c2, [&](int j) { return x[j]; });
        diag[c2] = d;
        minv[c2] = mi;
        r[c2] = ri;
        const double zi = mi * ri;
        z[c2] = zi;
        p[c2] = zi;
        rz += ri * zi;
        rr += ri * ri;
    }
    const sum2 t = block_sum2(rr, rz, s);
    if (threadIdx.x == 0) {
        part_rr[blockIdx.x] = t.a;
        part_rz[blockIdx.x] = t.b;
    }
}

__global__ void __launch_bounds__(TB) k_th_start(int nb, const double *__restrict__ part_rr,
                                                 const double *__restrict__ part_rz, th_ctl *ctl) {
    __shared__ double s[TB / 64][2];
    const sum2 t = part_sum2(nb, part_rr, part_rz, s);
    if (threadIdx.x == 0) {
        const double r0 = sqrt(t.a);
        th_ctl c = ctl[0];
        c.rz = t.b;
        c.r0 = r0;
        c.it = 0;
        c.done = (r0 < 1e-30) ? 1 : 0;
        c.its = (r0 < 1e-30) ? 0 : -1;
        ctl[0] = c;
        ctl[1] = c;
    }
}

// FIRST: p = z (the set-up's), nothing to test.
template <bool FIRST>
__global__ void __launch_bounds__(TB) k_th_apply(th_geom g, const double *__restrict__ kx,
                                                 const double *__restrict__ kz, const double *__restrict__ diag,
                                                 const double *__restrict__ z, const double *__restrict__ pold,
                                                 double *__restrict__ pnew, double *__restrict__ q, int nb,
                                                 const double *__restrict__ part_rr, const double *__restrict__ part_rz,
                                                 double *__restrict__ part_pq, th_ctl *ctl) {
    __shared__ double s[TB / 64][2];
    sum2 t{0.0, 0.0};
    if (!FIRST) t = part_sum2(nb, part_rr, part_rz, s);   // before the test: one round of loads
    th_ctl c = ctl[0];
    if (c.done) return;
    if (!FIRST) {
        c.it++;
        if (sqrt(t.a) / c.r0 < c.rel_tol) {
            c.its = c.it;
            c.done = 1;
        } else if (fabs(c.rz) < 1e-30) {
            c.its = -3;
            c.done = 1;
        } else {
            c.beta = t.b / c.rz;
            c.rz = t.b;
            if (c.it >= c.max_its) c.done = 1;   // its stays -1
        }
    } else {
        c.beta = 0.0;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl[1] = c;
    if (c.done) return;
    const int n = g.ncx * g.ncz;
    const th_share sh = th_cells(n);
    const double beta = c.beta;
    double pq = 0.0;
    int c2 = sh.lo + threadIdx.x, l = c2 / g.ncx, k = c2 - l * g.ncx;
    const int dl = sh.step / g.ncx, dk = sh.step - dl * g.ncx;
    for (; c2 < sh.hi; c2 += sh.step) {
        auto P = [&](int j) { return z[j] + beta * pold[j]; };
        const double qi = th_row(g, kx, kz, diag[c2], k, l, c2, P);
        const double pi = P(c2);
        pnew[c2] = pi;
        q[c2] = qi;
        pq += pi * qi;
        k += dk;
        l += dl;
        if (k >= g.ncx) {
            k -= g.ncx;
            l++;
        }
    }
    t = block_sum2(pq, 0.0, s);
    if (threadIdx.x == 0) part_pq[blockIdx.x] = t.a;
}

__global__ void __launch_bounds__(TB) k_th_update(int n, const double *__restrict__ p, const double *__restrict__ q,
                                                  const double *__restrict__ minv, double *__restrict__ x,
                                                  double *__restrict__ r, double *__restrict__ z, int nb,
                                                  const double *__restrict__ part_pq, double *__restrict__ part_rr,
                                                  double *__restrict__ part_rz, th_ctl *ctl) {
    __shared__ double s[TB / 64][2];
    const double pq = part_sum2(nb, part_pq, nullptr, s).a;
    th_ctl c = ctl[1];
    if (!c.done) {
        if (fabs(pq) < 1e-30) {
            c.its = -2;
            c.done = 1;
        } else {
            c.alpha = c.rz / pq;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl[0] = c;
    if (c.done) return;
    const th_share sh = th_cells(n);
    const double alpha = c.alpha;
    double rr = 0.0, rz = 0.0;
    for (int i = sh.lo + threadIdx.x; i < sh.hi; i += sh.step) {
        x[i] += alpha * p[i];
        const double ri = r[i] - alpha * q[i];
        r[i] = ri;
        const double zi = minv[i] * ri;
        z[i] = zi;
        rr += ri * ri;
        rz += ri * zi;
    }
    const sum2 t = block_sum2(rr, rz, s);
    if (threadIdx.x == 0) {
        part_rr[blockIdx.x] = t.a;
        part_rz[blockIdx.x] = t.b;
    }
}

// What the next apply would decide, for the host: the state with that test
// taken, the ratio ||r|| / ||r0|| in beta.
__global__ void __launch_bounds__(TB) k_th_test(int nb, const double *__restrict__ part_rr, const th_ctl *__restrict__ ctl,
                                                th_ctl *__restrict__ out) {
    __shared__ double s[TB / 64][2];
    th_ctl c = ctl[0];
    const double rr = part_sum2(nb, part_rr, nullptr, s).a;
    if (threadIdx.x == 0) {
        if (!c.done) {
            c.it++;
            c.beta = sqrt(rr) / c.r0;
            if (c.beta < c.rel_tol) {
                c.its = c.it;
                c.done = 1;
            } else if (fabs(c.rz) < 1e-30) {
                c.its = -3;
                c.done = 1;
            } else if (c.it >= c.max_its) {
                c.done = 1;
            }
        }
        *out = c;
    }
}

}  // namespace

struct thermal_scratch {
    dbuf<double> in[8];   // staged inputs: rho, Cp, Qr, Wdiss, Ha, kx, kz, BCT_v
    dbuf<signed char> bt;
    dbuf<double> x, diag, minv, r, z, p[2], q, part[3];
    dbuf<th_ctl> ctl;
};

void mdg_thermal_release(mdg_ctx *c) {
    if (!c->thermal) return;
    thermal_scratch *s = c->thermal;
    for (auto &b : s->in) b.release();
    s->bt.release(); s->x.release(); s->diag.release(); s->minv.release(); s->r.release(); s->z.release();
    s->p[0].release(); s->p[1].release(); s->q.release(); s->part[0].release(); s->part[1].release(); s->part[2].release();
    s->ctl.release();
    delete s;
    c->thermal = nullptr;
}

extern "C" int mdg_energy_step(mdg_ctx *c, double dt, const double *rho_n, const double *Cp, const double *Qr,
                               const double *Wdiss, const double *Ha, const double *kx, const double *kz,
                               const signed char *BCT_t, const double *BCT_v, int max_its, double rel_tol, double *T,
                               int *its) {
    if (!c || !rho_n || !Cp || !kx || !kz || !BCT_t || !BCT_v || !T || !its)
        return mdg_fail(c, MDG_ERR_ARG, "bad argument");
    if (!(dt > 0.0) || max_its < 0 || !(rel_tol > 0.0))
        return mdg_fail(c, MDG_ERR_ARG, "dt and rel_tol must be positive, max_its non-negative");
    if (c->Ncx < 1 || c->Ncz < 1) return mdg_fail(c, MDG_ERR_STATE, "no grid");
    if (!c->thermal) c->thermal = new thermal_scratch();
    thermal_scratch &s = *c->thermal;
    const int ncx = c->Ncx, ncz = c->Ncz, n = ncx * ncz;
    const size_t nkx = (size_t)c->Nx * (c->Nz + 1), nkz = (size_t)(c->Nx + 1) * c->Nz;
    const size_t nbc = (size_t)(ncx + 2) * (ncz + 2);
    th_in in{};
    int rc;
    if ((rc = mdg_stage_in(c, rho_n, (size_t)n, s.in[0], &in.rho)) || (rc = mdg_stage_in(c, Cp, (size_t)n, s.in[1], &in.Cp)) ||
        (rc = mdg_stage_in(c, Qr, (size_t)n, s.in[2], &in.Qr)) ||
        (rc = mdg_stage_in(c, Wdiss, (size_t)n, s.in[3], &in.Wd)) ||
        (rc = mdg_stage_in(c, Ha, (size_t)n, s.in[4], &in.Ha)) || (rc = mdg_stage_in(c, kx, nkx, s.in[5], &in.kx)) ||
        (rc = mdg_stage_in(c, kz, nkz, s.in[6], &in.kz)) || (rc = mdg_stage_in(c, BCT_v, nbc, s.in[7], &in.BV)) ||
        (rc = mdg_stage_in(c, BCT_t, nbc, s.bt, &in.BT)))
        return rc;
    double *x = T;
    if (!mdg_is_device_ptr(T)) {
        HIPCHK(c, s.x.reserve((size_t)n));
        HIPCHK(c, hipMemcpyAsync(s.x.p, T, (size_t)n * 8, hipMemcpyHostToDevice, c->stream));
        x = s.x.p;
    }
    const int nb = std::min(TH_BLOCKS, mdg_grid1d(n, TB));
    HIPCHK(c, s.diag.reserve(n)); HIPCHK(c, s.minv.reserve(n)); HIPCHK(c, s.r.reserve(n));
    HIPCHK(c, s.z.reserve(n)); HIPCHK(c, s.p[0].reserve(n)); HIPCHK(c, s.p[1].reserve(n));
    HIPCHK(c, s.q.reserve(n));
    for (auto &p : s.part) HIPCHK(c, p.reserve(nb));
    HIPCHK(c, s.ctl.reserve(3));
    th_ctl h{};
    h.rel_tol = rel_tol;
    h.max_its = max_its;
    h.done = 0;
    h.its = -1;
    HIPCHK(c, hipMemcpyAsync(s.ctl.p, &h, sizeof h, hipMemcpyHostToDevice, c->stream));
    const th_geom g{ncx, ncz, c->Nx, c->Nx + 1, 1.0 / (c->dx * c->dx), 1.0 / (c->dz * c->dz), c->dx};
    double *rr = s.part[0].p, *rz = s.part[1].p, *pq = s.part[2].p;
    HIPCHK(c, hipEventRecord(c->ev0, c->stream));
    hipLaunchKernelGGL(k_th_setup, dim3(nb), dim3(TB), 0, c->stream, g, dt, in, (const double *)x, s.diag.p,
                       s.minv.p, s.r.p, s.z.p, s.p[0].p, rr, rz);
    hipLaunchKernelGGL(k_th_start, dim3(1), dim3(TB), 0, c->stream, nb, (const double *)rr, (const double *)rz, s.ctl.p);
    HIPCHK(c, hipGetLastError());
    // With max_its = 0 the reference's loop does not run: its = -1 unless
    // the start already has a zero residual.
    if (max_its == 0) {
        HIPCHK(c, hipMemcpyAsync(&h, s.ctl.p, sizeof h, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
    }
    int launched = 0, batch = 8, cur = 0;
    while (launched < max_its) {
        const int m = std::min(batch, max_its - launched);
        for (int i = 0; i < m; i++) {
            const bool first = launched + i == 0;
            hipLaunchKernelGGL(first ? k_th_apply<true> : k_th_apply<false>, dim3(nb), dim3(TB), 0, c->stream, g, in.kx, in.kz,
                               (const double *)s.diag.p, (const double *)s.z.p, (const double *)s.p[cur].p,
                               s.p[cur ^ 1].p, s.q.p, nb, (const double *)rr, (const double *)rz, pq, s.ctl.p);
            hipLaunchKernelGGL(k_th_update, dim3(nb), dim3(TB), 0, c->stream, n, (const double *)s.p[cur ^ 1].p,
                               (const double *)s.q.p, (const double *)s.minv.p, x, s.r.p, s.z.p, nb, (const double *)pq, rr, rz,
                               s.ctl.p);
            cur ^= 1;
        }
        hipLaunchKernelGGL(k_th_test, dim3(1), dim3(TB), 0, c->stream, nb, (const double *)rr, (const th_ctl *)s.ctl.p,
                           s.ctl.p + 2);
        HIPCHK(c, hipGetLastError());
        launched += m;
        HIPCHK(c, hipMemcpyAsync(&h, s.ctl.p + 2, sizeof h, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        if (h.done) break;
        // the next batch: as many as the mean rate so far still needs (an
        // iteration too many costs two empty launches, one too few a round trip)
        const double left = h.beta < 1.0 ? launched * (std::log(rel_tol) / std::log(h.beta) - 1.0) : batch;
        batch = (int)std::min(128.0, std::max(8.0, 1.02 * left + 1.0));
    }
    HIPCHK(c, hipEventRecord(c->ev1, c->stream));
    if (x != T) HIPCHK(c, hipMemcpyAsync(T, x, (size_t)n * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    float ms = 0.0f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    *its = h.its;
    return MDG_OK;
}
