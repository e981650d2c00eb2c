// Marker advection: V2P (ParticleRoutines.c:63-256) and the fourth-order
// Runge-Kutta step of RogerGuntherII (AdvectionRoutines.c:347-410) with
// isoutPart (AdvectionRoutines.c:320-341, non-periodic box).
//
// One thread per marker: the four V2P stages gather 2 x 4 velocities each
// from the Vx / Vz grids (read through L2; a sorted marker set keeps the
// gathers of a wavefront within a few grid rows) and the marker streams
// x, z, phase in and x, z, phase, vx, vz out: 44 B of HBM traffic per
// marker. The arithmetic is the reference's, in the same order, built
// without contraction, so positions and velocities match the CPU
// restatement bit for bit.
//
// Bound: FP64 issue. Each stage divides twelve times by a cell width; those
// divisions are xdiv_core's product and four fused multiply-adds (the same
// bits), and one test per stage, over the marker's coordinates and the four
// products of a velocity, says whether every one of them is in range (the
// coordinate tables are tested once, on the host); a marker that fails it
// repeats the stage with divisions. The reference's substitutions for air
// nodes (tag 30) are left out: mdg_set_bc accepts no such tag on velocity
// nodes, and reading the tags took 8 more gathers per stage.
// Measured with 37.7M markers on 2047^2, conservative interpolation:
// k_advect_rk4 3.26 ms with divisions and tags, 1.63 ms with exact_div tested
// division by division, 1.48 ms with one test per stage (about 1500 VALU
// instructions per marker, at the issue rate; 1.66 GB of marker streams would
// take 0.36 ms).
#include "exact_div.h"
#include "mdg_internal.h"

namespace {

struct v2p_grid {
    int Nx, Nz;                       // vertices
    exact_div dx, dz;
    const double *xg, *zg, *xvz, *zvx;
    double xmin, xmax, zmin, zmax;    // box of isoutPart
    int tables_ok;                    // every coordinate passes v2p_coord_ok
};

// The divisions of a stage: by exact_div's steps, collecting whether any
// numerator is out of their range, or by the division itself.
struct div_steps {
    bool bad;
    __device__ __forceinline__ double dist(double a, const exact_div &h) const { return xdiv_core(a, h); }
    __device__ __forceinline__ double prod(double a, const exact_div &h) {
        bad |= !xdiv_takes(a, h);
        return xdiv_core(a, h);
    }
};
struct div_plain {
    __device__ __forceinline__ double dist(double a, const exact_div &h) const { return a / h.b; }
    __device__ __forceinline__ double prod(double a, const exact_div &h) const { return a / h.b; }
};

__device__ __forceinline__ int v2p_cell(double q, int n) {
    int j = (int)ceil(q) - 1;
    if (j < 0) j = 0;
    if (j > n - 2) j = n - 2;
    return j;
}
// 0.5 pow(t - 0.5, 2): the square written as one product, the correctly
// rounded value the C library's pow returns for an exponent of 2
__device__ inline double v2p_corr(double t) {
    const double y = t - 0.5;
    return 0.5 * (y * y);
}

// One velocity component at a marker: F on an n1 x n2 node grid (stride s1
// along the component's own axis, s2 across it), cell (c1, c2), distances d1,
// t1 = d1 / h1 along it and t2 across it.  The correction of the second
// difference reads one node beyond the cell on the side the marker is on.
template <bool CONSERV, typename D>
__device__ __forceinline__ double v2p_comp(D &div, const double *__restrict__ F, int at, int s1, int s2, int c1, int n1,
                                           double d1, double t1, double t2, const exact_div &h1) {
    const double A0 = F[at], A1 = F[at + s1], B0 = F[at + s2], B1 = F[at + s1 + s2];
    double a = A0 * (1.0 - t1) + div.prod(A1 * d1, h1);
    double b = B0 * (1.0 - t1) + div.prod(B1 * d1, h1);
    if (CONSERV) {
        const bool up = t1 >= 0.5, on = up ? c1 < n1 - 2 : c1 > 0;
        const int far = at + (on ? (up ? 2 * s1 : -s1) : 0);
        const double Af = F[far], Bf = F[far + s2], w = v2p_corr(t1);
        const double ac = a + w * ((up ? A0 : Af) - 2.0 * (up ? A1 : A0) + (up ? Af : A1));
        const double bc = b + w * ((up ? B0 : Bf) - 2.0 * (up ? B1 : B0) + (up ? Bf : B1));
        a = on ? ac : a;
        b = on ? bc : b;
    }
    return (1.0 - t2) * a + t2 * b;
}

// V2P of one active marker (ParticleRoutines.c:76-252)
template <bool CONSERV, typename D>
__device__ __forceinline__ void v2p_with(D &div, const v2p_grid &g, const double *__restrict__ u,
                                         const double *__restrict__ v, double x, double z, double *vxm, double *vzm) {
    {
        const int Nx = g.Nx, Nz = g.Nz + 1;
        const int j = v2p_cell(div.dist(x - g.xg[0], g.dx), Nx), i = v2p_cell(div.dist(z - g.zvx[0], g.dz), Nz);
        const double dxm = fabs(x - g.xg[j]), dzm = fabs(z - g.zvx[i]);
        *vxm = v2p_comp<CONSERV>(div, u, j + i * Nx, 1, Nx, j, Nx, dxm, div.dist(dxm, g.dx), div.dist(dzm, g.dz), g.dx);
    }
    {
        const int Nx = g.Nx + 1, Nz = g.Nz;
        const int j = v2p_cell(div.dist(x - g.xvz[0], g.dx), Nx), i = v2p_cell(div.dist(z - g.zg[0], g.dz), Nz);
        const double dxm = fabs(x - g.xvz[j]), dzm = fabs(z - g.zg[i]);
        *vzm = v2p_comp<CONSERV>(div, v, j + i * Nx, Nx, 1, i, Nz, dzm, div.dist(dzm, g.dz), div.dist(dxm, g.dx), g.dz);
    }
}

// A coordinate whose distances to the table's entries are zero or in
// exact_div's range: zero, or of a size in [2^-400, 2^400).
__host__ __device__ inline bool v2p_coord_ok(double x) {
    return (xdiv_hi(x) & 0x7fffffffu) - ((uint32_t)(1023 - 400) << 20) < ((uint32_t)800 << 20) || x == 0.0;
}

template <bool CONSERV>
__device__ __forceinline__ void v2p_one(const v2p_grid &g, const double *__restrict__ u, const double *__restrict__ v,
                                        double x, double z, double *vxm, double *vzm) {
    div_steps steps{!(v2p_coord_ok(x) && v2p_coord_ok(z)) || !g.tables_ok};
    v2p_with<CONSERV>(steps, g, u, v, x, z, vxm, vzm);
    if (__builtin_expect(steps.bad, 0)) {
        div_plain plain;
        v2p_with<CONSERV>(plain, g, u, v, x, z, vxm, vzm);
    }
}

__device__ inline void isout(const v2p_grid &g, double x, double z, int *ph) {
    if (x < g.xmin || x > g.xmax || z < g.zmin || z > g.zmax) *ph = -1;
}

template <bool CONSERV>
__global__ void k_v2p(v2p_grid g, const double *__restrict__ u, const double *__restrict__ v, int n,
                      const double *__restrict__ x, const double *__restrict__ z, const int *__restrict__ phase,
                      double *__restrict__ vx, double *__restrict__ vz) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    double a = 0.0, b = 0.0;
    if (phase[k] != -1) v2p_one<CONSERV>(g, u, v, x[k], z[k], &a, &b);
    vx[k] = a;
    vz[k] = b;
}

// RogerGuntherII's loop body (AdvectionRoutines.c:372-405)
template <bool CONSERV>
__global__ void k_advect_rk4(v2p_grid g, const double *__restrict__ u, const double *__restrict__ v, double dt,
                             int n, double *__restrict__ x, double *__restrict__ z,
                             int *__restrict__ phase, double *__restrict__ vxo, double *__restrict__ vzo) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double xA = x[k], zA = z[k];
    double xk = xA, zk = zA, sx = 0.0, sz = 0.0;
    int ph = phase[k];
    // stages A, B, C, D: the sums VxA + 2 VxB + 2 VxC + VxD grow in order
#pragma unroll 1
    for (int s = 0; s < 4; s++) {
        if (ph != -1) {
            double a, b;
            v2p_one<CONSERV>(g, u, v, xk, zk, &a, &b);
            const double w = (s == 1 || s == 2) ? 2.0 : 1.0;
            sx = (s == 0) ? a : sx + w * a;
            sz = (s == 0) ? b : sz + w * b;
            if (s < 3) {
                const double h = (s == 2) ? 1.0 * dt : 0.5 * dt;
                xk = xA + h * a;
                zk = zA + h * b;
            }
        }
        if (s < 3) isout(g, xk, zk, &ph);
    }
    if (ph != -1) {
        const double VxA = (1.0 / 6.0) * sx, VzA = (1.0 / 6.0) * sz;
        xk = xA + dt * VxA;
        zk = zA + dt * VzA;
        if (vxo) vxo[k] = VxA;
        if (vzo) vzo[k] = VzA;
    }
    isout(g, xk, zk, &ph);
    x[k] = xk;
    z[k] = zk;
    phase[k] = ph;
}

bool tables_ok(const mdg_ctx *c) {
    for (const std::vector<double> *t : {&c->h_xg, &c->h_zg, &c->h_xvz, &c->h_zvx})
        if (!std::all_of(t->begin(), t->end(), v2p_coord_ok)) return false;
    return true;
}

v2p_grid make_grid(const mdg_ctx *c) {
    return v2p_grid{c->Nx, c->Nz, make_exact_div(c->dx), make_exact_div(c->dz), c->xg.p, c->zg.p, c->xvz.p, c->zvx.p,
                    c->xmin, c->xmax, c->zmin, c->zmax, tables_ok(c) ? 1 : 0};
}

// A caller's array as a device pointer: itself, or a device copy (copied in
// when `in`); copy_back returns a device copy's contents to the caller.
template <typename T>
int dev_view(mdg_ctx *c, T *user, size_t n, dbuf<T> &tmp, bool in, T **d) {
    if (!user) { *d = nullptr; return MDG_OK; }
    if (mdg_is_device_ptr(user)) { *d = user; return MDG_OK; }
    HIPCHK(c, tmp.reserve(n));
    if (in) HIPCHK(c, hipMemcpyAsync(tmp.p, user, n * sizeof(T), hipMemcpyHostToDevice, c->stream));
    *d = tmp.p;
    return MDG_OK;
}
template <typename T>
int copy_back(mdg_ctx *c, T *user, const T *d, size_t n) {
    if (user && d && d != user) HIPCHK(c, hipMemcpyAsync(user, d, n * sizeof(T), hipMemcpyDeviceToHost, c->stream));
    return MDG_OK;
}

}  // namespace

// staging buffers for host callers, one set per context (freed with it)
struct advect_scratch {
    dbuf<double> u, v, x, z, vx, vz;
    dbuf<int> ph;
};

static advect_scratch &scratch_of(mdg_ctx *c) {
    if (!c->advect) c->advect = new advect_scratch();
    return *c->advect;
}

void mdg_advect_release(mdg_ctx *c) {
    if (!c || !c->advect) return;
    advect_scratch *s = c->advect;
    s->u.release(); s->v.release(); s->x.release(); s->z.release(); s->vx.release(); s->vz.release(); s->ph.release();
    delete s;
    c->advect = nullptr;
}

extern "C" int mdg_v2p(mdg_ctx *c, const double *u, const double *v, int conserv_interp, int n, const double *x,
                       const double *z, const int *phase, double *vx, double *vz) {
    if (!c || !u || !v || !x || !z || !phase || !vx || !vz || n < 0) return mdg_fail(c, MDG_ERR_ARG, "bad argument");
    if (!c->have_bc) return mdg_fail(c, MDG_ERR_STATE, "mdg_set_bc has not been called");
    if (n == 0) return MDG_OK;
    advect_scratch &s = scratch_of(c);
    const size_t nu = (size_t)c->Nx * (c->Nz + 1), nv = (size_t)(c->Nx + 1) * c->Nz;
    const double *du, *dv, *dx_, *dz_;
    const int *dph;
    double *dvx, *dvz;
    int rc;
    if ((rc = mdg_stage_in(c, u, nu, s.u, &du)) || (rc = mdg_stage_in(c, v, nv, s.v, &dv)) ||
        (rc = mdg_stage_in(c, x, (size_t)n, s.x, &dx_)) || (rc = mdg_stage_in(c, z, (size_t)n, s.z, &dz_)) ||
        (rc = mdg_stage_in(c, phase, (size_t)n, s.ph, &dph)) || (rc = dev_view(c, vx, (size_t)n, s.vx, false, &dvx)) ||
        (rc = dev_view(c, vz, (size_t)n, s.vz, false, &dvz)))
        return rc;
    HIPCHK(c, hipEventRecord(c->ev0, c->stream));
    hipLaunchKernelGGL(conserv_interp == 1 ? k_v2p<true> : k_v2p<false>, dim3(mdg_grid1d(n, 256)), dim3(256), 0, c->stream,
                       make_grid(c), du, dv, n, dx_, dz_, dph, dvx, dvz);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipEventRecord(c->ev1, c->stream));
    if ((rc = copy_back(c, vx, (const double *)dvx, (size_t)n)) || (rc = copy_back(c, vz, (const double *)dvz, (size_t)n)))
        return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    float ms = 0.0f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    return MDG_OK;
}

extern "C" int mdg_advect_rk4(mdg_ctx *c, const double *u, const double *v, double dt, int conserv_interp, int n,
                              double *x, double *z, int *phase, double *vx, double *vz) {
    if (!c || !u || !v || !x || !z || !phase || n < 0) return mdg_fail(c, MDG_ERR_ARG, "bad argument");
    if (!c->have_bc) return mdg_fail(c, MDG_ERR_STATE, "mdg_set_bc has not been called");
    if (n == 0) return MDG_OK;
    advect_scratch &s = scratch_of(c);
    const size_t nu = (size_t)c->Nx * (c->Nz + 1), nv = (size_t)(c->Nx + 1) * c->Nz;
    const double *du, *dv;
    double *dx_, *dz_, *dvx, *dvz;
    int *dph;
    int rc;
    if ((rc = mdg_stage_in(c, u, nu, s.u, &du)) || (rc = mdg_stage_in(c, v, nv, s.v, &dv)) ||
        (rc = dev_view(c, x, (size_t)n, s.x, true, &dx_)) || (rc = dev_view(c, z, (size_t)n, s.z, true, &dz_)) ||
        (rc = dev_view(c, phase, (size_t)n, s.ph, true, &dph)) || (rc = dev_view(c, vx, (size_t)n, s.vx, true, &dvx)) ||
        (rc = dev_view(c, vz, (size_t)n, s.vz, true, &dvz)))
        return rc;
    HIPCHK(c, hipEventRecord(c->ev0, c->stream));
    hipLaunchKernelGGL(conserv_interp == 1 ? k_advect_rk4<true> : k_advect_rk4<false>, dim3(mdg_grid1d(n, 256)), dim3(256),
                       0, c->stream, make_grid(c), du, dv, dt, n, dx_, dz_, dph, dvx, dvz);
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipEventRecord(c->ev1, c->stream));
    if ((rc = copy_back(c, x, (const double *)dx_, (size_t)n)) || (rc = copy_back(c, z, (const double *)dz_, (size_t)n)) ||
        (rc = copy_back(c, phase, (const int *)dph, (size_t)n)) || (rc = copy_back(c, vx, (const double *)dvx, (size_t)n)) ||
        (rc = copy_back(c, vz, (const double *)dvz, (size_t)n)))
        return rc;
    HIPCHK(c, hipStreamSynchronize(c->stream));
    float ms = 0.0f;
    HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->last_ms = ms;
    return MDG_OK;
}
