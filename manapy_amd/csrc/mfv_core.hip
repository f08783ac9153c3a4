// libmfv core: error plumbing, mesh checks, generic operators (ghost fill, face->cell,
// least-squares gradient, Barth-Jespersen limiter) and linear advection.
//
// Every kernel runs one thread per cell (or per listed face) and gathers what it needs;
// nothing is scattered and no atomics touch floating-point sums, so results are
// deterministic and independent of the launch shape.
#include <stdarg.h>

#include <mutex>
#include <vector>

#include "mfv_common.hpp"

namespace mfv {

static thread_local char g_err[512] = "";

void set_error(const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int check_launch(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: %s", what, hipGetErrorString(e));
        return MFV_EHIP;
    }
    return MFV_OK;
}

int validate_mesh(const mfv_mesh *m, int need_lsq, int need_order_split, int need_order_sorted)
{
    MFV_REQUIRE(m != nullptr, "mesh descriptor is NULL");
    MFV_REQUIRE(m->dim == 2 || m->dim == 3, "mesh dim must be 2 or 3, got %d", m->dim);
    MFV_REQUIRE(m->nb_cells >= 0 && m->nb_faces >= 0, "negative mesh sizes");
    MFV_REQUIRE(m->max_cell_faces >= 1 && m->max_cell_faces <= 8, "max_cell_faces %d out of [1, 8]",
                m->max_cell_faces);
    MFV_REQUIRE(m->face_cells && m->face_name && m->face_normal && m->face_mesure && m->face_center &&
                    m->cell_center && m->cell_volume && m->cell_faces && m->cell_nfaces,
                "mesh descriptor has NULL geometry/connectivity pointers");
    if (need_lsq)
        MFV_REQUIRE(m->lsq_cells && m->lsq_ncells && m->lsq_ghosts && m->lsq_nghosts && m->face_ghost &&
                        m->lsq_width >= 0 && m->ghost_width >= 0,
                    "mesh descriptor lacks the least-squares stencil");
    if (need_order_split) MFV_REQUIRE(m->order_split, "mesh descriptor lacks order_split");
    if (need_order_sorted) MFV_REQUIRE(m->order_sorted, "mesh descriptor lacks order_sorted");
    return MFV_OK;
}

}  // namespace mfv

using namespace mfv;

extern "C" const char *mfv_version(void) { return "mfv 0.1 gfx950"; }
extern "C" const char *mfv_last_error(void) { return mfv::g_err; }

extern "C" int mfv_device_count(int *count_host)
{
    MFV_REQUIRE(count_host, "count_host is NULL");
    hipError_t e = hipGetDeviceCount(count_host);
    if (e != hipSuccess) {
        *count_host = 0;
        set_error("hipGetDeviceCount: %s", hipGetErrorString(e));
        return MFV_EHIP;
    }
    return MFV_OK;
}

// ---------------------------------------------------------------------------------------------
// ghost values (boundary/bc_utils.py:45-68), face->cell (ast/ast_utils.py:8-18)

__global__ void __launch_bounds__(kBlock) k_ghost_value(const int32_t *__restrict__ face_cells, int kind,
                                                         const double *__restrict__ src,
                                                         double *__restrict__ w_ghost,
                                                         const int32_t *__restrict__ faces, int n)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int f = faces[k];
    if (kind == 0) w_ghost[f] = src[face_cells[2 * f]];
    else if (kind == 1) w_ghost[f] = -1 * src[face_cells[2 * f]];
    else w_ghost[f] = src[f];
}

extern "C" int mfv_ghost_value(const mfv_mesh *m, int kind, const double *src, double *w_ghost,
                               const int32_t *faces, int nfaces, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    MFV_REQUIRE(kind >= 0 && kind <= 2, "ghost kind %d not in {0,1,2}", kind);
    MFV_REQUIRE(nfaces >= 0, "nfaces < 0");
    if (nfaces == 0) return MFV_OK;
    MFV_REQUIRE(src && w_ghost && faces, "NULL array");
    hipLaunchKernelGGL(k_ghost_value, dim3(grid_for(nfaces)), dim3(kBlock), 0, as_stream(stream), m->face_cells,
                       kind, src, w_ghost, faces, nfaces);
    return check_launch("k_ghost_value");
}

// All boundary locations of all fields of a step in one launch (blockIdx.y is the segment): a
// location has a few hundred faces, so a launch each is only launch time (20 of them took 43 us
// a step in the five-field shallow-water scheme at 200k cells, this one 3.4 us).
constexpr int kGhostSegs = 32;
struct GhostSegs {
    mfv_ghost_seg s[kGhostSegs];
};

__global__ void __launch_bounds__(kBlock) k_ghost_values(const int32_t *__restrict__ face_cells, GhostSegs g)
{
    const mfv_ghost_seg &s = g.s[blockIdx.y];
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= s.n) return;
    const int f = s.faces[k];
    double v;
    if (s.kind == 2) {
        v = s.w[f];
    } else {
        v = s.w[face_cells[2 * f]];
        if (s.kind == 1) v = -1 * v;
        if (s.kind == 3) v = v + s.cst[f] * s.dist[f];
    }
    s.ghost[f] = v;
}

extern "C" int mfv_ghost_values(const mfv_mesh *m, const mfv_ghost_seg *segs, int nseg, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    MFV_REQUIRE(nseg >= 0 && (nseg == 0 || segs), "segments missing");
    GhostSegs g;
    int n = 0, most = 0;
    for (int k = 0; k < nseg; k++) {
        const mfv_ghost_seg &s = segs[k];
        MFV_REQUIRE(s.kind >= 0 && s.kind <= 3, "ghost kind %d not in {0,1,2,3}", s.kind);
        MFV_REQUIRE(s.n >= 0, "nfaces < 0");
        MFV_REQUIRE(s.n == 0 || (s.faces && s.w && s.ghost && (s.kind != 3 || (s.cst && s.dist))), "NULL array");
    }
    for (int k = 0; k < nseg; k++) {
        if (segs[k].n > 0) {
            g.s[n++] = segs[k];
            most = segs[k].n > most ? segs[k].n : most;
        }
        if (n == kGhostSegs || (n > 0 && k == nseg - 1)) {
            hipLaunchKernelGGL(k_ghost_values, dim3(grid_for(most), n), dim3(kBlock), 0, as_stream(stream),
                               m->face_cells, g);
            if (int rc = check_launch("k_ghost_values")) return rc;
            n = most = 0;
        }
    }
    return MFV_OK;
}

__global__ void __launch_bounds__(kBlock) k_facetocell(Mesh m, const double *__restrict__ u_face,
                                                        double *__restrict__ u_c)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m.C) return;
    int nf = m.cell_nfaces[i];
    double s = 0.;
    for (int j = 0; j < nf; j++) s += u_face[m.cell_faces[(size_t)j * m.C + i]];
    u_c[i] = s / (double)nf;
}

extern "C" int mfv_facetocell(const mfv_mesh *m, const double *u_face, double *u_c, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    if (m->nb_cells == 0) return MFV_OK;
    MFV_REQUIRE(u_face && u_c, "NULL array");
    hipLaunchKernelGGL(k_facetocell, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream),
                       to_kernel(m), u_face, u_c);
    return check_launch("k_facetocell");
}

// ---------------------------------------------------------------------------------------------
// least-squares cell gradient (ast/functions2d.py:5-104, functions3d.py:4-120)

template <int DIM>
__device__ __forceinline__ void lsq_solve(const double (&I)[6], const double (&J)[3], double &gx, double &gy,
                                          double &gz)
{
    // I = {xx, yy, xy, zz, xz, yz}
    if (DIM == 2) {
        double dia = I[0] * I[1] - I[2] * I[2];
        gx = (I[1] * J[0] - I[2] * J[1]) / dia;
        gy = (I[0] * J[1] - I[2] * J[0]) / dia;
        gz = 0.;
    } else {
        double xx = I[0], yy = I[1], xy = I[2], zz = I[3], xz = I[4], yz = I[5];
        double dia = xx * yy * zz + 2. * xy * xz * yz - xx * (yz * yz) - yy * (xz * xz) - zz * (xy * xy);
        gx = ((yy * zz - yz * yz) * J[0] + (xz * yz - xy * zz) * J[1] + (xy * yz - xz * yy) * J[2]) / dia;
        gy = ((xz * yz - xy * zz) * J[0] + (xx * zz - xz * xz) * J[1] + (xy * xz - yz * xx) * J[2]) / dia;
        gz = ((xy * yz - xz * yy) * J[0] + (xy * xz - yz * xx) * J[1] + (xx * yy - xy * xy) * J[2]) / dia;
    }
}

template <int DIM>
__device__ __forceinline__ void lsq_accumulate(double (&I)[6], double (&J)[3], double jx, double jy, double jz,
                                               double dw)
{
    I[0] += jx * jx;
    I[1] += jy * jy;
    if (DIM == 3) I[3] += jz * jz;
    I[2] += (jx * jy);
    if (DIM == 3) {
        I[4] += (jx * jz);
        I[5] += (jy * jz);
    }
    J[0] += (jx * dw);
    J[1] += (jy * dw);
    if (DIM == 3) J[2] += (jz * dw);
}

template <int DIM>
__global__ void __launch_bounds__(kBlock) k_cell_gradient(Mesh m, const double *__restrict__ w_c,
                                                           const double *__restrict__ w_ghost,
                                                           double *__restrict__ wx, double *__restrict__ wy,
                                                           double *__restrict__ wz)
{
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= m.C) return;
    const double cx = m.cell_center[3 * i], cy = m.cell_center[3 * i + 1], cz = m.cell_center[3 * i + 2];
    const double wi = w_c[i];
    double I[6] = {0., 0., 0., 0., 0., 0.}, J[3] = {0., 0., 0.};
    const int nn = m.lsq_ncells[i];
    for (int j = 0; j < nn; j++) {
        int c = m.lsq_cells[(size_t)j * m.C + i];
        const double *p = m.cell_center + 3 * (size_t)c;
        lsq_accumulate<DIM>(I, J, p[0] - cx, p[1] - cy, DIM == 3 ? p[2] - cz : 0., w_c[c] - wi);
    }
    const int ng = m.lsq_nghosts[i];
    for (int j = 0; j < ng; j++) {
        int f = m.lsq_ghosts[(size_t)j * m.C + i];
        const double *p = m.face_ghost + 3 * (size_t)f;
        lsq_accumulate<DIM>(I, J, p[0] - cx, p[1] - cy, DIM == 3 ? p[2] - cz : 0., w_ghost[f] - wi);
    }
    double gx, gy, gz;
    lsq_solve<DIM>(I, J, gx, gy, gz);
    wx[i] = gx;
    wy[i] = gy;
    wz[i] = gz;
}

extern "C" int mfv_cell_gradient(const mfv_mesh *m, const double *w_c, const double *w_ghost, double *w_x,
                                 double *w_y, double *w_z, void *stream)
{
    if (int rc = validate_mesh(m, 1, 0, 0)) return rc;
    if (m->nb_cells == 0) return MFV_OK;
    MFV_REQUIRE(w_c && w_ghost && w_x && w_y && w_z, "NULL array");
    auto k = (m->dim == 2) ? k_cell_gradient<2> : k_cell_gradient<3>;
    hipLaunchKernelGGL(k, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream), to_kernel(m), w_c,
                       w_ghost, w_x, w_y, w_z);
    return check_launch("k_cell_gradient");
}

// ---------------------------------------------------------------------------------------------
// Barth-Jespersen limiter (ast/functions2d.py:280-325, functions3d.py:364-408)

template <int DIM>
__device__ __forceinline__ double barth_psi(const Mesh &m, int i, double wi, double gx, double gy, double gz,
                                            double w_max, double w_min)
{
    const double eps = (DIM == 2) ? 1e-8 : 1e-10;
    const double cx = m.cell_center[3 * i], cy = m.cell_center[3 * i + 1], cz = m.cell_center[3 * i + 2];
    const int nf = m.cell_nfaces[i];
    double psi = 1., psi_ij = 1.;
    for (int j = 0; j < nf; j++) {
        int f = m.cell_faces[(size_t)j * m.C + i];
        const double *fc = m.face_center + 3 * (size_t)f;
        double r1 = fc[0] - cx, r2 = fc[1] - cy;
        double delta2 = (DIM == 2) ? (gx * r1 + gy * r2) : (gx * r1 + gy * r2 + gz * (fc[2] - cz));
        if (fabs(delta2) < eps) {
            psi_ij = 1.;
        } else {
            if (delta2 > 0.) psi_ij = pmin(1., (w_max - wi) / delta2);
            if (delta2 < 0.) psi_ij = pmin(1., (w_min - wi) / delta2);
        }
        psi = pmin(psi, psi_ij);
    }
    return psi;
}

template <int DIM>
__global__ void __launch_bounds__(kBlock) k_barthlimiter(Mesh m, const double *__restrict__ w_c,
                                                          const double *__restrict__ w_ghost,
                                                          const double *__restrict__ wx,
                                                          const double *__restrict__ wy,
                                                          const double *__restrict__ wz, double *__restrict__ psi)
{
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= m.C) return;
    const double wi = w_c[i];
    double w_max = wi, w_min = wi;
    const int nf = m.cell_nfaces[i];
    for (int j = 0; j < nf; j++) {
        int f = m.cell_faces[(size_t)j * m.C + i];
        int nm = m.face_name[f];
        double a = w_c[m.face_cells[2 * f]];
        double b = (nm == 0 || nm > 10) ? w_c[m.face_cells[2 * f + 1]] : w_ghost[f];
        w_max = pmax(pmax(w_max, a), b);
        w_min = pmin(pmin(w_min, a), b);
    }
    psi[i] = barth_psi<DIM>(m, i, wi, wx[i], wy[i], DIM == 3 ? wz[i] : 0., w_max, w_min);
}

extern "C" int mfv_barthlimiter(const mfv_mesh *m, const double *w_c, const double *w_ghost, const double *w_x,
                                const double *w_y, const double *w_z, double *psi, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    if (m->nb_cells == 0) return MFV_OK;
    MFV_REQUIRE(w_c && w_ghost && w_x && w_y && w_z && psi, "NULL array");
    auto k = (m->dim == 2) ? k_barthlimiter<2> : k_barthlimiter<3>;
    hipLaunchKernelGGL(k, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream), to_kernel(m), w_c,
                       w_ghost, w_x, w_y, w_z, psi);
    return check_launch("k_barthlimiter");
}

// ---------------------------------------------------------------------------------------------
// gradient and limiter of NF fields in one pass (cell_gradient then barthlimiter, bit for bit)
//
// OWNER: a ghost takes its owner's value (Neumann everywhere), as the fused advection steps read
// it; RECORD > 0 then writes w, gx, gy, (gz,) psi as one record of that many doubles to gx[0], so
// that a step gathers a neighbour's from one line.

template <int NF>
struct GradArgs {
    const double *__restrict__ w[NF];
    const double *__restrict__ ghost[NF];
    double *__restrict__ gx[NF];
    double *__restrict__ gy[NF];
    double *__restrict__ gz[NF];
    double *__restrict__ psi[NF];
};

template <int DIM, int NF>
__device__ __forceinline__ void stencil_sums(const Mesh &m, const GradArgs<NF> &a, int i, double cx, double cy,
                                             double cz, const double (&wi)[NF], double (&I)[6], double (&J)[NF][3])
{
    constexpr int G = 8;
    const int nn = m.lsq_ncells[i];
    const int nmax = wave_max_int(nn);
    int c[G];
#pragma unroll
    for (int k = 0; k < G; k++) c[k] = (k < m.K) ? m.lsq_cells[(size_t)k * m.C + i] : 0;
    for (int j = 0; j < nmax; j += G) {
        double p[G][3], v[G][NF];
#pragma unroll
        for (int k = 0; k < G; k++) {
            const int q = (j + k < nn) ? c[k] : i;
            p[k][0] = m.cell_center[3 * (size_t)q];
            p[k][1] = m.cell_center[3 * (size_t)q + 1];
            if (DIM == 3) p[k][2] = m.cell_center[3 * (size_t)q + 2];
#pragma unroll
            for (int f = 0; f < NF; f++) v[k][f] = a.w[f][q];
        }
#pragma unroll
        for (int k = 0; k < G; k++) c[k] = (j + G + k < m.K) ? m.lsq_cells[(size_t)(j + G + k) * m.C + i] : 0;
#pragma unroll
        for (int k = 0; k < G; k++) {
            if (j + k >= nn) continue;
            const double jx = p[k][0] - cx, jy = p[k][1] - cy, jz = DIM == 3 ? p[k][2] - cz : 0.;
            lsq_accumulate<DIM>(I, J[0], jx, jy, jz, v[k][0] - wi[0]);
#pragma unroll
            for (int f = 1; f < NF; f++) {
                const double dw = v[k][f] - wi[f];
                J[f][0] += (jx * dw);
                J[f][1] += (jy * dw);
                if (DIM == 3) J[f][2] += (jz * dw);
            }
        }
    }
}

// The ghost part of the sums, after the cells'.
template <int DIM, int NF, bool OWNER>
__device__ __forceinline__ void ghost_sums(const Mesh &m, const GradArgs<NF> &a, int i, double cx, double cy, double cz,
                                           const double (&wi)[NF], double (&I)[6], double (&J)[NF][3])
{
    const int ng = m.lsq_nghosts[i], gmax = wave_max_int(ng);
    for (int j = 0; j < gmax; j++) {
        if (j >= ng) continue;
        const int q = m.lsq_ghosts[(size_t)j * m.C + i];
        const double *g = m.face_ghost + 3 * (size_t)q;
        const double jx = g[0] - cx, jy = g[1] - cy, jz = DIM == 3 ? g[2] - cz : 0.;
        const int o = OWNER ? m.face_cells[2 * (size_t)q] : q;
        lsq_accumulate<DIM>(I, J[0], jx, jy, jz, (OWNER ? a.w[0] : a.ghost[0])[o] - wi[0]);
#pragma unroll
        for (int f = 1; f < NF; f++) {
            const double dw = (OWNER ? a.w[f] : a.ghost[f])[o] - wi[f];
            J[f][0] += (jx * dw);
            J[f][1] += (jy * dw);
            if (DIM == 3) J[f][2] += (jz * dw);
        }
    }
}

// Gradient and limiter of cell i; sums(...) adds the stencil's cells.
template <int DIM, int NF, int MF, bool OWNER, int RECORD, class Sums>
__device__ __forceinline__ void gradient_cell(const Mesh &m, const GradArgs<NF> &a, int i, Sums sums)
{
    const double cx = m.cell_center[3 * (size_t)i], cy = m.cell_center[3 * (size_t)i + 1],
                 cz = m.cell_center[3 * (size_t)i + 2];
    const int nf = m.cell_nfaces[i];
    int fid[MF];
#pragma unroll
    for (int s = 0; s < MF; s++) {
        const int f = m.cell_faces[(size_t)min(s, m.MF - 1) * m.C + i];
        fid[s] = (s < nf) ? f : -1;
    }
    double wi[NF], I[6] = {0., 0., 0., 0., 0., 0.}, J[NF][3];
#pragma unroll
    for (int f = 0; f < NF; f++) {
        wi[f] = a.w[f][i];
        J[f][0] = J[f][1] = J[f][2] = 0.;
    }
    sums(cx, cy, cz, wi, I, J);
    ghost_sums<DIM, NF, OWNER>(m, a, i, cx, cy, cz, wi, I, J);
    // the faces: what lies on both sides, and the face's centre
    int2 ab[MF];
    int nm[MF];
    double r[MF][3];
#pragma unroll
    for (int s = 0; s < MF; s++) {
        const size_t f = fid[s] >= 0 ? fid[s] : 0;
        ab[s] = face_pair(m, f);
        nm[s] = m.face_name[f];
        r[s][0] = m.face_center[3 * f] - cx;
        r[s][1] = m.face_center[3 * f + 1] - cy;
        if (DIM == 3) r[s][2] = m.face_center[3 * f + 2] - cz;
    }
    const double eps = (DIM == 2) ? 1e-8 : 1e-10;
#pragma unroll
    for (int f = 0; f < NF; f++) {
        double wl[MF], wr[MF];
#pragma unroll
        for (int s = 0; s < MF; s++) {
            const bool has = fid[s] >= 0, inner = nm[s] == 0 || nm[s] > 10;
            wl[s] = a.w[f][has ? ab[s].x : i];
            const double *src = (has && !inner && !OWNER) ? a.ghost[f] : a.w[f];
            wr[s] = src[!has ? i : inner ? ab[s].y : OWNER ? ab[s].x : fid[s]];
        }
        double gx, gy, gz;
        lsq_solve<DIM>(I, J[f], gx, gy, gz);
        double hi = wi[f], lo = wi[f];
#pragma unroll
        for (int s = 0; s < MF; s++)
            if (fid[s] >= 0) {
                hi = pmax(pmax(hi, wl[s]), wr[s]);
                lo = pmin(pmin(lo, wl[s]), wr[s]);
            }
        double psi = 1., psi_ij = 1.;
#pragma unroll
        for (int s = 0; s < MF; s++)
            if (fid[s] >= 0) {
                const double delta2 =
                    (DIM == 2) ? (gx * r[s][0] + gy * r[s][1]) : (gx * r[s][0] + gy * r[s][1] + gz * r[s][2]);
                if (fabs(delta2) < eps) {
                    psi_ij = 1.;
                } else {
                    if (delta2 > 0.) psi_ij = pmin(1., (hi - wi[f]) / delta2);
                    if (delta2 < 0.) psi_ij = pmin(1., (lo - wi[f]) / delta2);
                }
                psi = pmin(psi, psi_ij);
            }
        if (RECORD) {
            double2 *q = reinterpret_cast<double2 *>(a.gx[f] + RECORD * (size_t)i);
            q[0] = make_double2(wi[f], gx);
            q[1] = DIM == 3 ? make_double2(gy, gz) : make_double2(gy, psi);
            if (DIM == 3) q[2] = make_double2(psi, 0.);
            continue;
        }
        a.gx[f][i] = gx;
        a.gy[f][i] = gy;
        if (DIM == 3 || !OWNER) a.gz[f][i] = gz;
        a.psi[f][i] = psi;
    }
}

template <int DIM, int NF, int MF, bool OWNER, int RECORD>
__global__ void __launch_bounds__(kBlock) k_gradient_limited(Mesh m, GradArgs<NF> a)
{
    const int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= m.C) return;
    gradient_cell<DIM, NF, MF, OWNER, RECORD>(
        m, a, i, [&](double cx, double cy, double cz, const double (&wi)[NF], double (&I)[6], double (&J)[NF][3]) {
            stencil_sums<DIM, NF>(m, a, i, cx, cy, cz, wi, I, J);
        });
}

// The same of one field on tetrahedra with the stencils' cells in LDS (mfv_stencil_tiles). A
// tetrahedron has some 70 vertex neighbours: gathered from memory they are 70 x 32 bytes a cell through
// an L1 that the block's neighbourhood does not fit, 441 MB at 197k cells, and neither fewer loads (x
// and y as one) nor more in flight made that faster. A block of 256 cells along a Morton curve reads
// about 1000 different cells: they are copied once (32 KB) and the stencil is 16-bit positions, half
// the bytes of the cell numbers. 197k cells: 54.8 -> 36.9 us. Same order of the sums, same bits.
struct StencilTiles {
    const int32_t *__restrict__ cell;   // [nt][kBlock] cell of each thread, -1 past the end
    const int32_t *__restrict__ eptr;   // [nt + 1]
    const int32_t *__restrict__ ext;    // cells a tile reads
    const uint32_t *__restrict__ pairs; // [K2][nt * kBlock] positions 2j and 2j + 1 in the tile's ext list
    int K2;
    size_t n;
};

template <bool OWNER, int RECORD>
__global__ void __launch_bounds__(kBlock) k_gradient_tiled(Mesh m, StencilTiles t, GradArgs<1> a)
{
    extern __shared__ double4 sten[];
    const int tile = xcd_block();
    const size_t row = (size_t)tile * kBlock + threadIdx.x;
    const int i = t.cell[row], e0 = t.eptr[tile], ne = t.eptr[tile + 1] - e0;
    constexpr int H = 4;  // words of two positions in flight
    uint32_t h[H];
#pragma unroll
    for (int k = 0; k < H; k++) h[k] = t.pairs[(size_t)min(k, t.K2 - 1) * t.n + row];
    for (int e = threadIdx.x; e < ne; e += 2 * kBlock) {
        const int f = min(e + kBlock, ne - 1);
        const size_t c = t.ext[e0 + e], d = t.ext[e0 + f];
        const double4 v = make_double4(m.cell_center[3 * c], m.cell_center[3 * c + 1], m.cell_center[3 * c + 2],
                                       a.w[0][c]),
                      u = make_double4(m.cell_center[3 * d], m.cell_center[3 * d + 1], m.cell_center[3 * d + 2],
                                       a.w[0][d]);
        sten[e] = v;
        sten[f] = u;
    }
    __syncthreads();
    if (i < 0) return;
    gradient_cell<3, 1, 4, OWNER, RECORD>(
        m, a, i, [&](double cx, double cy, double cz, const double (&wi)[1], double (&I)[6], double (&J)[1][3]) {
            const int nn = m.lsq_ncells[i];
            const int nmax = wave_max_int(nn);
            for (int j = 0; j < nmax; j += 2 * H) {
                double4 p[2 * H];
#pragma unroll
                for (int k = 0; k < H; k++) {
                    p[2 * k] = sten[h[k] & 0xffffu];
                    p[2 * k + 1] = sten[h[k] >> 16];
                }
#pragma unroll
                for (int k = 0; k < H; k++) h[k] = t.pairs[(size_t)min(j / 2 + H + k, t.K2 - 1) * t.n + row];
#pragma unroll
                for (int k = 0; k < 2 * H; k++) {
                    if (j + k >= nn) continue;
                    lsq_accumulate<3>(I, J[0], p[k].x - cx, p[k].y - cy, p[k].z - cz, p[k].w - wi[0]);
                }
            }
        });
}

// Doubles of a cell's record (w, gradient, psi) in the fused advection steps.
constexpr int adv_record(int dim) { return dim == 2 ? 4 : 8; }

template <int NF, bool OWNER = false, bool RECORD = false>
static int gradient_limited(const mfv_mesh *m, const GradArgs<NF> &a, hipStream_t st)
{
    const Mesh k = to_kernel(m);
    const dim3 g(grid_for(m->nb_cells)), b(kBlock);
#define LAUNCH(D, M) \
    hipLaunchKernelGGL((k_gradient_limited<D, NF, M, OWNER, RECORD ? adv_record(D) : 0>), g, b, 0, st, k, a)
    if (m->dim == 2) {
        if (m->max_cell_faces <= 3) LAUNCH(2, 3);
        else if (m->max_cell_faces == 4) LAUNCH(2, 4);
        else LAUNCH(2, 8);
    } else {
        if (m->max_cell_faces <= 4) LAUNCH(3, 4);
        else LAUNCH(3, 8);
    }
#undef LAUNCH
    return check_launch("k_gradient_limited");
}

template <bool OWNER, bool RECORD>
static int gradient_tiled(const mfv_mesh *m, const mfv_stencil_tiles *t, const GradArgs<1> &a, hipStream_t st)
{
    const StencilTiles k{t->cell, t->ext_ptr, t->ext_cells, t->pairs, t->nb_pairs, (size_t)t->nb_tiles * kBlock};
    hipLaunchKernelGGL((k_gradient_tiled<OWNER, RECORD ? adv_record(3) : 0>), dim3(t->nb_tiles), dim3(kBlock),
                       sizeof(double4) * (size_t)t->max_ext, st, to_kernel(m), k, a);
    return check_launch("k_gradient_tiled");
}

static int check_stencil_tiles(const mfv_mesh *m, const mfv_stencil_tiles *t)
{
    MFV_REQUIRE(m->dim == 3 && m->max_cell_faces <= 4, "stencil tiles are for tetrahedra");
    MFV_REQUIRE(t && t->cell && t->ext_ptr && t->ext_cells && t->pairs, "stencil tiles have NULL arrays");
    MFV_REQUIRE(t->tile_size == kBlock && t->nb_tiles == (m->nb_cells + kBlock - 1) / kBlock &&
                    t->nb_pairs == (m->lsq_width + 1) / 2 && t->nb_pairs >= 1,
                "stencil tiles were built for another mesh");
    MFV_REQUIRE(t->max_ext >= 1 && t->max_ext <= 2048, "stencil tiles read %d cells a block, at most 2048 fit the LDS",
                t->max_ext);
    return MFV_OK;
}

extern "C" int mfv_cell_gradient_tiled(const mfv_mesh *m, const mfv_stencil_tiles *t, const mfv_gradient_fields *f,
                                       void *stream)
{
    if (int rc = validate_mesh(m, 1, 0, 0)) return rc;
    if (int rc = check_stencil_tiles(m, t)) return rc;
    MFV_REQUIRE(f && f->w && f->ghost && f->gx && f->gy && f->gz && f->psi, "NULL array");
    if (m->nb_cells == 0) return MFV_OK;
    return gradient_tiled<false, false>(m, t, GradArgs<1>{{f->w}, {f->ghost}, {f->gx}, {f->gy}, {f->gz}, {f->psi}},
                                        as_stream(stream));
}

extern "C" int mfv_cell_gradient_limited(const mfv_mesh *m, int nfields, const mfv_gradient_fields *f, void *stream)
{
    if (int rc = validate_mesh(m, 1, 0, 0)) return rc;
    MFV_REQUIRE(nfields == 1 || nfields == 2, "nfields must be 1 or 2, got %d", nfields);
    MFV_REQUIRE(f, "fields missing");
    for (int k = 0; k < nfields; k++)
        MFV_REQUIRE(f[k].w && f[k].ghost && f[k].gx && f[k].gy && f[k].gz && f[k].psi, "NULL array");
    if (m->nb_cells == 0) return MFV_OK;
    if (nfields == 1)
        return gradient_limited<1>(m, GradArgs<1>{{f->w}, {f->ghost}, {f->gx}, {f->gy}, {f->gz}, {f->psi}},
                                   as_stream(stream));
    return gradient_limited<2>(m,
                               GradArgs<2>{{f[0].w, f[1].w}, {f[0].ghost, f[1].ghost}, {f[0].gx, f[1].gx},
                                           {f[0].gy, f[1].gy}, {f[0].gz, f[1].gz}, {f[0].psi, f[1].psi}},
                               as_stream(stream));
}

// ---------------------------------------------------------------------------------------------
// dt reduction helpers

__global__ void k_dt_reset(double *dt) { dt[0] = 1e6; }

__global__ void k_dt_ring_init(double *ring, const double *dt0)
{
    ring[0] = dt0[0];
    ring[1] = 1e6;
    ring[2] = 1e6;
    ring[3] = 0.;
}

extern "C" int mfv_dt_ring_init(double *dt_ring_p, const double *dt0, void *stream)
{
    MFV_REQUIRE(dt_ring_p && dt0, "NULL array");
    hipLaunchKernelGGL(k_dt_ring_init, dim3(1), dim3(1), 0, as_stream(stream), dt_ring_p, dt0);
    return check_launch("k_dt_ring_init");
}

extern "C" int mfv_dt_reset(double *dt, void *stream)
{
    MFV_REQUIRE(dt, "dt is NULL");
    hipLaunchKernelGGL(k_dt_reset, dim3(1), dim3(1), 0, as_stream(stream), dt);
    return check_launch("k_dt_reset");
}

namespace mfv {

// Per-wave dt partial minima live in one buffer per (device, stream): work queued on one
// stream runs in order, so the buffer is reused without a race, and calls on different
// streams never share one. A buffer only grows. A smaller buffer it replaces is never freed:
// a graph captured on that stream (by the caller, e.g. torch) may still hold its address and
// be replayed later, so retired buffers stay allocated until the process ends. Growth is by
// doubling, so the retired buffers together are smaller than the live one.
struct DtScratch {
    int dev;
    hipStream_t stream;
    double *ptr;
    size_t cap;
};
static std::mutex g_dt_mu;
static std::vector<DtScratch> g_dt_scr;
static std::vector<double *> g_dt_retired;

void graph_free(MfvGraph *g)
{
    if (!g) return;
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    if (g->stream) (void)hipStreamDestroy(g->stream);
    if (g->part) (void)hipFree(g->part);
    delete g;
}

int graph_begin(MfvGraph *g)
{
    hipError_t e = hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipStreamBeginCapture(g->stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) {
        set_error("graph capture setup: %s", hipGetErrorString(e));
        return MFV_EHIP;
    }
    return MFV_OK;
}

int graph_finish(MfvGraph *g, int rc)
{
    hipError_t e = hipStreamEndCapture(g->stream, &g->graph);
    if (rc != MFV_OK) return rc;
    if (e != hipSuccess) {
        set_error("graph capture: %s", hipGetErrorString(e));
        return MFV_EHIP;
    }
    e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        set_error("graph instantiate: %s", hipGetErrorString(e));
        return MFV_EHIP;
    }
    return MFV_OK;
}

double *dt_scratch(size_t nwaves, hipStream_t st)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        set_error("dt scratch: no current device");
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_dt_mu);
    DtScratch *e = nullptr;
    for (auto &x : g_dt_scr)
        if (x.dev == dev && x.stream == st) e = &x;
    if (!e) {
        g_dt_scr.push_back(DtScratch{dev, st, nullptr, 0});
        e = &g_dt_scr.back();
    }
    if (e->cap < nwaves) {
        const size_t cap = e->cap * 2 > nwaves ? e->cap * 2 : nwaves;
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone) {
            set_error("dt scratch: the stream is being captured and its partials buffer must grow to %zu doubles; "
                      "run one uncaptured call of the same size first",
                      nwaves);
            return nullptr;
        }
        if (e->ptr) g_dt_retired.push_back(e->ptr);
        e->ptr = nullptr;
        e->cap = 0;
        if (hipMalloc(reinterpret_cast<void **>(&e->ptr), cap * sizeof(double)) != hipSuccess) {
            set_error("dt scratch: hipMalloc of %zu doubles failed", cap);
            e->ptr = nullptr;
            return nullptr;
        }
        e->cap = cap;
    }
    return e->ptr;
}

__device__ __forceinline__ double dt_block_min(const double *__restrict__ part, size_t n)
{
    __shared__ double sh[1024];
    // four partials in flight per thread (the minimum of a set does not depend on the order)
    double m0 = __longlong_as_double(0x7ff0000000000000LL), m1 = m0, m2 = m0, m3 = m0;
    size_t j = threadIdx.x;
    for (; j + 3 * 1024 < n; j += 4 * 1024) {
        const double a = part[j], b = part[j + 1024], c = part[j + 2048], e = part[j + 3072];
        m0 = (a < m0) ? a : m0;
        m1 = (b < m1) ? b : m1;
        m2 = (c < m2) ? c : m2;
        m3 = (e < m3) ? e : m3;
    }
    for (; j < n; j += 1024) {
        const double v = part[j];
        m0 = (v < m0) ? v : m0;
    }
    m0 = (m1 < m0) ? m1 : m0;
    m2 = (m3 < m2) ? m3 : m2;
    const double m = (m2 < m0) ? m2 : m0;
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            const double o = sh[threadIdx.x + w];
            sh[threadIdx.x] = (o < sh[threadIdx.x]) ? o : sh[threadIdx.x];
        }
        __syncthreads();
    }
    return sh[0];
}

__global__ void __launch_bounds__(1024) k_dt_finish(const double *__restrict__ part, size_t n, double *__restrict__ out)
{
    const double r = dt_block_min(part, n);
    if (threadIdx.x == 0 && r < out[0]) out[0] = r;
}

// out[0] = min(1e6, min part), and then the same to host memory if given, in release order at system
// scope (k_dt_total's own start value: no launch to reset out[0] first).
__global__ void __launch_bounds__(1024) k_dt_total(const double *__restrict__ part, size_t n,
                                                   double *__restrict__ out, double *host)
{
    const double r = dt_block_min(part, n);
    if (threadIdx.x == 0) {
        const double dt = (r < 1e6) ? r : 1e6;
        out[0] = dt;
        if (host) __hip_atomic_store(host, dt, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

int dt_finish(const double *part, size_t n, double *out, hipStream_t st)
{
    if (int rc = check_launch("dt kernel")) return rc;
    hipLaunchKernelGGL(k_dt_finish, dim3(1), dim3(1024), 0, st, part, n, out);
    return check_launch("k_dt_finish");
}

}  // namespace mfv

namespace {

// One double of pinned host memory for a dt on its way to the host. A call takes a slot for as long
// as it waits; as many slots exist as calls have waited at once (threads).
std::mutex g_dt_slot_mu;
std::vector<double *> g_dt_slots;

double *take_dt_slot()
{
    {
        std::lock_guard<std::mutex> lock(g_dt_slot_mu);
        if (!g_dt_slots.empty()) {
            double *p = g_dt_slots.back();
            g_dt_slots.pop_back();
            return p;
        }
    }
    void *p = nullptr;
    const hipError_t e = hipHostMalloc(&p, sizeof(double), hipHostMallocPortable | hipHostMallocMapped);
    if (e != hipSuccess) {
        set_error("dt readback: hipHostMalloc: %s", hipGetErrorString(e));
        return nullptr;
    }
    return static_cast<double *>(p);
}

void give_dt_slot(double *p)
{
    std::lock_guard<std::mutex> lock(g_dt_slot_mu);
    g_dt_slots.push_back(p);
}

}  // namespace

// A dt that the host asks for is written to pinned memory by the fold itself: a copy to the caller's
// (pageable) double is a launch of its own. kIdle then waits for the stream, as any *_host output
// promises. kDt looks at the pinned word instead, which the fold stores last and with release order:
// whoever sees it also sees dt_dev and what the stream held before it, but the kernel itself may not have
// retired. Four 3D advection steps take 328 us with kIdle and 306 us with kDt, four of the SRNH scheme at
// 1k cells (eight dts) 338 and 278 us, of Euler at 8k 138 and 120, of advection-diffusion 332 and 240. The
// release order itself costs 0.35 us a dt (12.3 -> 12.6 us a call at 1k cells); a write-through store and a
// wait for it in its place the same.
int mfv::dt_total(const double *part, size_t n, double *dt_dev, double *dt_host, DtWait wait, hipStream_t st)
{
    double *slot = nullptr;
    volatile long long *word = nullptr;
    const long long kWaiting = 0x7ff8000000000001LL;  // a NaN: no dt has these bits
    if (dt_host) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone) {
            set_error("dt readback: the stream is being captured; the dt cannot be read on the host");
            return MFV_EHIP;
        }
        slot = take_dt_slot();
        if (!slot) return MFV_ENOMEM;
        word = reinterpret_cast<volatile long long *>(slot);
        *word = kWaiting;
    }
    hipLaunchKernelGGL(k_dt_total, dim3(1), dim3(1024), 0, st, part, n, dt_dev, slot);
    int rc = check_launch("dt kernel");
    if (slot) {
        if (rc == MFV_OK) {
            if (wait == kDt)
                for (int k = 0; k < 200000 && *word == kWaiting; k++) __builtin_ia32_pause();
            if (*word == kWaiting || wait == kIdle) {  // kDt: a long queue ahead, or an error
                const hipError_t e = hipStreamSynchronize(st);
                if (e != hipSuccess) {
                    set_error("dt readback: %s", hipGetErrorString(e));
                    return MFV_EHIP;  // the slot may still be written: it is not given back
                }
            }
            const long long w = *word;
            memcpy(dt_host, &w, sizeof(double));
        } else {
            (void)hipStreamSynchronize(st);
        }
        give_dt_slot(slot);
    }
    return rc;
}

// ---------------------------------------------------------------------------------------------
// advection (solvers/advec/fvm_utils.py)

// time_step (fvm_utils.py:293-309): the per-cell candidate; faces summed in faceid order.
template <int MF>
__device__ __forceinline__ double adv_cell_dt(const Mesh &m, int i, double u, double v, double w, double cfl)
{
    const int nf = m.cell_nfaces[i];
    int f[MF];
    double n[MF][3];
    cell_face_ids<MF>(m, i, nf, f);
#pragma unroll
    for (int j = 0; j < MF; j++)
#pragma unroll
        for (int d = 0; d < 3; d++) n[j][d] = m.face_normal[3 * (size_t)f[j] + d];
    double lam = 0.;
#pragma unroll
    for (int j = 0; j < MF; j++)
        if (j < nf) lam += fabs(u * n[j][0] + v * n[j][1] + w * n[j][2]);
    return cfl * m.cell_volume[i] / lam;
}

template <int MF>
__global__ void __launch_bounds__(kBlock) k_adv_time_step(Mesh m, const double *__restrict__ u,
                                                           const double *__restrict__ v,
                                                           const double *__restrict__ w, double cfl,
                                                           double *__restrict__ dtpart)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    double d = (i < m.C) ? adv_cell_dt<MF>(m, i, u[i], v[i], w[i], cfl) : 1e300;
    wave_min_part(dtpart, (size_t)i, d);
}

static int time_step(const mfv_mesh *m, const double *u, const double *v, const double *w, double cfl, double *dt_dev,
                     double *dt_host, DtWait wait, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    MFV_REQUIRE(u && v && w && dt_dev, "NULL array");
    const size_t nw = m->nb_cells ? waves_for(m->nb_cells) : 0;
    double *part = nullptr;
    if (nw) {
        part = dt_scratch(nw, as_stream(stream));
        if (!part) return MFV_ENOMEM;
        auto k = m->max_cell_faces <= 4 ? k_adv_time_step<4> : k_adv_time_step<8>;
        hipLaunchKernelGGL(k, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream), to_kernel(m), u, v, w,
                           cfl, part);
    }
    return dt_total(part, nw, dt_dev, dt_host, wait, as_stream(stream));
}

extern "C" int mfv_time_step(const mfv_mesh *m, const double *u, const double *v, const double *w, double cfl,
                             double *dt_dev, double *dt_host, void *stream)
{
    return time_step(m, u, v, w, cfl, dt_dev, dt_host, kIdle, stream);
}

extern "C" int mfv_time_step_polled(const mfv_mesh *m, const double *u, const double *v, const double *w, double cfl,
                                    double *dt_dev, double *dt_host, void *stream)
{
    return time_step(m, u, v, w, cfl, dt_dev, dt_host, kDt, stream);
}

// Residual of cell i by the upwind flux (compute_upwind_flux, fvm_utils.py:5-17) with the MUSCL
// reconstruction of explicitscheme_convective_{2d,3d}: contributions added in the reference's face
// order (inner faces by increasing id, then boundary faces by increasing id) so the sum is
// bit-identical to the face-ordered scatter rez[c0] -= F; rez[c1] += F.
// Only the side that the flow comes from is read: the face's sign is formed first, then the value
// (left = face_cells[f][0]; right = face_cells[f][1] or, on a boundary face, w_ghost[f]) and, at
// order 2, the gradient of that cell. ORDER 1 skips the gradient reads: the reference's term
// (order-1)*psi*(grad.r) is then 0 * 0 * 0 (psi and gradients stay zero when
// compute_cell_gradient is never called). OWNER_GHOST takes the Neumann ghost
// w_ghost[f] = w_c[face_cells[f][0]] on the fly.
// The loads of all faces leave together, level by level (ids, faces, upwind cells): 197k tetrahedra
// 24.6 -> 14.1 us, 100k triangles 8.9 -> 6.6 us against a loop over the faces that reads both sides.
template <int DIM, int ORDER, bool OWNER_GHOST, int MF>
__device__ __forceinline__ double adv_residual(const Mesh &m, int i, const double *__restrict__ w_c,
                                               const double *__restrict__ w_ghost, const double *__restrict__ uf,
                                               const double *__restrict__ vf, const double *__restrict__ wf,
                                               const double *__restrict__ gx, const double *__restrict__ gy,
                                               const double *__restrict__ gz, const double *__restrict__ psi,
                                               double om)
{
    const int nf = m.cell_nfaces[i];
    int f[MF], a[MF], up[MF];
    bool left[MF], ghost[MF];
    double sign[MF], r[MF][3], w[MF];
    ordered_face_ids<MF>(m, m.order_split, i, nf, f);
#pragma unroll
    for (int k = 0; k < MF; k++) {
        const int2 ab = face_pair(m, f[k]);
        const double *n = m.face_normal + 3 * (size_t)f[k];
        sign[k] = uf[f[k]] * n[0] + vf[f[k]] * n[1] + wf[f[k]] * n[2];
        if (ORDER == 2) {
#pragma unroll
            for (int d = 0; d < DIM; d++) r[k][d] = m.face_center[3 * (size_t)f[k] + d];
        }
        a[k] = ab.x;
        up[k] = ab.y;
    }
#pragma unroll
    for (int k = 0; k < MF; k++) {
        left[k] = sign[k] >= 0;
        ghost[k] = !left[k] && up[k] < 0;
        up[k] = (left[k] || ghost[k]) ? a[k] : up[k];
    }
#pragma unroll
    for (int k = 0; k < MF; k++) {
        const int c = up[k];
        w[k] = w_c[c];
        if (!OWNER_GHOST && ghost[k]) w[k] = w_ghost[f[k]];
        if (ORDER == 1) {
            w[k] = ghost[k] ? w[k] : w[k] + 0.;
            continue;
        }
        const double *cc = m.cell_center + 3 * (size_t)c;
        double full;
        if (DIM == 2)
            full = w[k] + om * psi[c] * (gx[c] * (r[k][0] - cc[0]) + gy[c] * (r[k][1] - cc[1]));
        else
            full = w[k] + om * psi[c] * (gx[c] * (r[k][0] - cc[0]) + gy[c] * (r[k][1] - cc[1]) + gz[c] * (r[k][2] - cc[2]));
        w[k] = ghost[k] ? w[k] : full;
    }
    double rez = 0.;
#pragma unroll
    for (int k = 0; k < MF; k++) {
        if (k >= nf) continue;
        const double flux = sign[k] * w[k];
        if (a[k] == i)
            rez -= flux;
        else
            rez += flux;
    }
    return rez;
}

template <int DIM, int MF>
__global__ void __launch_bounds__(kBlock) k_adv_residual(Mesh m, double *__restrict__ rez_w,
                                                          const double *__restrict__ w_c,
                                                          const double *__restrict__ w_ghost,
                                                          const double *__restrict__ uf,
                                                          const double *__restrict__ vf,
                                                          const double *__restrict__ wf,
                                                          const double *__restrict__ gx,
                                                          const double *__restrict__ gy,
                                                          const double *__restrict__ gz,
                                                          const double *__restrict__ psi, double om)
{
    int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= m.C) return;
    // the kernel-level entry point always evaluates the reference expression with its arrays
    rez_w[i] = adv_residual<DIM, 2, false, MF>(m, i, w_c, w_ghost, uf, vf, wf, gx, gy, gz, psi, om);
}

extern "C" int mfv_explicitscheme_convective(const mfv_mesh *m, double *rez_w, const double *w_c,
                                             const double *w_ghost, const double *u_face, const double *v_face,
                                             const double *w_face, const double *w_x, const double *w_y,
                                             const double *w_z, const double *psi, int order, void *stream)
{
    if (int rc = validate_mesh(m, 0, 1, 0)) return rc;
    if (m->nb_cells == 0) return MFV_OK;
    MFV_REQUIRE(rez_w && w_c && w_ghost && u_face && v_face && w_face && w_x && w_y && w_z && psi,
                "NULL array");
    double om = (double)(order - 1);
    const int MF = m->max_cell_faces;
    auto k = (m->dim == 2) ? (MF <= 3 ? k_adv_residual<2, 3> : MF <= 4 ? k_adv_residual<2, 4> : k_adv_residual<2, 8>)
                           : (MF <= 4 ? k_adv_residual<3, 4> : k_adv_residual<3, 8>);
    hipLaunchKernelGGL(k, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream), to_kernel(m), rez_w,
                       w_c, w_ghost, u_face, v_face, w_face, w_x, w_y, w_z, psi, om);
    return check_launch("k_adv_residual");
}

__global__ void __launch_bounds__(kBlock) k_update_new_value(int C, double *__restrict__ ne_c,
                                                              const double *__restrict__ rez,
                                                              const double *__restrict__ dissip,
                                                              const double *__restrict__ src, double dtime,
                                                              const double *__restrict__ dt_dev,
                                                              const double *__restrict__ vol)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= C) return;
    double dt = dt_dev ? dt_dev[0] : dtime;
    ne_c[i] += dt * ((rez[i] + dissip[i]) / vol[i] + src[i]);
}

extern "C" int mfv_update_new_value(const mfv_mesh *m, double *ne_c, const double *rez, const double *dissip,
                                    const double *src, double dtime, const double *dt_dev, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    if (m->nb_cells == 0) return MFV_OK;
    MFV_REQUIRE(ne_c && rez && dissip && src, "NULL array");
    hipLaunchKernelGGL(k_update_new_value, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream),
                       m->nb_cells, ne_c, rez, dissip, src, dtime, dt_dev, m->cell_volume);
    return check_launch("k_update_new_value");
}

// ----- fused advection step ------------------------------------------------------------------
// Neumann ghosts (w_ghost[f] = w[c0]) are read straight from the owner cell.

template <int DIM, int ORDER, int MF>
__global__ void __launch_bounds__(kBlock) k_adv_step(Mesh m, const double *__restrict__ w_in,
                                                      double *__restrict__ w_out, const double *__restrict__ uc,
                                                      const double *__restrict__ vc,
                                                      const double *__restrict__ wc,
                                                      const double *__restrict__ uf,
                                                      const double *__restrict__ vf,
                                                      const double *__restrict__ wf, double cfl, double om,
                                                      const double *__restrict__ scratch,
                                                      DtRing ring, double *__restrict__ dtpart)
{
    int i = xcd_block() * blockDim.x + threadIdx.x;
    ring_advance(ring);
    double dloc = 1e300;
    if (i < m.C) {
        const double *gx = scratch, *gy = scratch + m.C, *gz = scratch + 2 * (size_t)m.C;
        const double *psi = scratch + (size_t)DIM * m.C;
        double rez = adv_residual<DIM, ORDER, true, MF>(m, i, w_in, nullptr, uf, vf, wf, gx, gy, gz, psi, om);
        double dt = ring.cur[0];
        // update_new_value with the dissipative and source terms zero
        w_out[i] = w_in[i] + dt * ((rez + 0.) / m.cell_volume[i] + 0.);
        dloc = adv_cell_dt<MF>(m, i, uc[i], vc[i], wc[i], cfl);
    }
    wave_min_part(dtpart, (size_t)i, dloc);
}

extern "C" int mfv_advection_step(const mfv_mesh *m, const double *w_in, double *w_out, const double *u_c,
                                  const double *v_c, const double *w_c, const double *u_face,
                                  const double *v_face, const double *w_face, double cfl, int order,
                                  double *dt_ring_p, int step, double *scratch, void *stream)
{
    if (int rc = validate_mesh(m, order == 2, 1, 0)) return rc;
    MFV_REQUIRE(order == 1 || order == 2, "order must be 1 or 2");
    MFV_REQUIRE(w_in && w_out && w_in != w_out && u_c && v_c && w_c && u_face && v_face && w_face && dt_ring_p,
                "NULL or aliased array");
    DtRing r = dt_ring(dt_ring_p, step);
    MFV_REQUIRE(order == 1 || scratch, "order 2 needs a scratch of (dim+1)*C doubles");
    MFV_REQUIRE(!(m->dim == 2 && m->max_cell_faces > 4), "2D cells have at most 4 faces");
    if (m->nb_cells == 0) return MFV_OK;
    Mesh k = to_kernel(m);
    hipStream_t st = as_stream(stream);
    if (order == 2) {
        const size_t C = m->nb_cells;
        const GradArgs<1> a{{w_in}, {nullptr}, {scratch}, {scratch + C}, {scratch + 2 * C}, {scratch + m->dim * C}};
        if (int rc = gradient_limited<1, true>(m, a, st)) return rc;
    }
    const size_t nw = waves_for(m->nb_cells);
    double *part = dt_scratch(nw, as_stream(stream));
    if (!part) return MFV_ENOMEM;
    const bool few = m->max_cell_faces <= 4;
    auto ks = (m->dim == 2) ? ((order == 2) ? k_adv_step<2, 2, 4> : k_adv_step<2, 1, 4>)
              : few         ? ((order == 2) ? k_adv_step<3, 2, 4> : k_adv_step<3, 1, 4>)
                            : ((order == 2) ? k_adv_step<3, 2, 8> : k_adv_step<3, 1, 8>);
    hipLaunchKernelGGL(ks, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, st, k, w_in, w_out, u_c, v_c, w_c,
                       u_face, v_face, w_face, cfl, (double)(order - 1), scratch, r, part);
    if (int rc = check_launch("k_adv_step")) return rc;
    return dt_finish(part, nw, r.next, st);
}

// ----- nsteps advection steps ------------------------------------------------------------------
// The velocity does not change within a run, so what a face contributes of it is laid out once: for
// the r-th contribution of a cell's residual the cell whose value is carried (the upwind side), the
// flux velocity out of the cell, and at order 2 the face's centre as seen from the upwind cell. dt
// is one number for all steps. A step is then one launch (two at order 2) that reads 12 (28, 36)
// coalesced bytes a slot and gathers one value (record) a slot, where the general step gathers both
// sides of each face, its normal and velocities, and forms and reduces the same dt again. 100 steps
// at 80k triangles, order 1: 1022 -> 341 us, about what 100 launches in a row take. The sums are the general step's term for term: the
// outward velocity is the face's with its sign turned for the right-hand cell, which is exact.
namespace {

constexpr int kAdvNone = (int)0x80000000;  // no face in this position
// Cells up to which two steps go into one launch (k_adv_run_pair), 100 steps single and in pairs:
// triangles 1k 361 and 240 us, 20k 341 and 251, 80k 341 and 300, 131k 348 and 308, 200k 410 and 405,
// 400k 513 and 581; tetrahedra 10k 325 and 289, 48k 335 and 300, 162k 416 and 492.
constexpr int kAdvPairCells3 = 131072, kAdvPairCells4 = 65536;

struct AdvTable {
    int32_t *__restrict__ up;   // [MF][C] upwind cell; ~cell: its value without reconstruction (a ghost's)
    double *__restrict__ coef;  // [MF][C] velocity through the face, out of the cell
    double *__restrict__ r;     // [MF][DIM][C] face centre - upwind cell's centre (order 2)
    double *__restrict__ rec;   // [C][adv_record] w, gradient, psi (order 2)
};

size_t adv_table(const mfv_mesh *m, int order, double *ws, AdvTable *t)
{
    const size_t C = ((size_t)m->nb_cells + 1) & ~(size_t)1, MF = m->max_cell_faces;
    size_t n = 0;
    auto take = [&](size_t k) {
        n += k;
        return ws ? ws + n - k : nullptr;
    };
    t->rec = order == 2 ? take(C * adv_record(m->dim)) : nullptr;
    t->coef = take(MF * C);
    t->r = order == 2 ? take(MF * C * m->dim) : nullptr;
    t->up = reinterpret_cast<int32_t *>(take((MF * C + 1) / 2));
    return n;
}

template <int DIM, int ORDER>
__global__ void __launch_bounds__(kBlock) k_adv_table(Mesh m, AdvTable t, const double *__restrict__ uf,
                                                      const double *__restrict__ vf, const double *__restrict__ wf)
{
    const int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= m.C) return;
    const int nf = m.cell_nfaces[i];
    for (int r = 0; r < m.MF; r++) {
        const size_t q = (size_t)r * m.C + i;
        if (r >= nf) {
            t.up[q] = kAdvNone;
            t.coef[q] = 0.;
            if (ORDER == 2)
                for (int d = 0; d < DIM; d++) t.r[((size_t)r * DIM + d) * m.C + i] = 0.;
            continue;
        }
        const int f = m.cell_faces[(size_t)m.order_split[q] * m.C + i];
        const int a = m.face_cells[2 * (size_t)f], b = m.face_cells[2 * (size_t)f + 1];
        const double *n = m.face_normal + 3 * (size_t)f;
        const double sign = uf[f] * n[0] + vf[f] * n[1] + wf[f] * n[2];
        const bool left = sign >= 0;
        const int up = (left || b < 0) ? a : b;
        t.up[q] = (left || b >= 0) ? up : ~up;
        t.coef[q] = (a == i) ? sign : -sign;
        if (ORDER == 2) {
            for (int d = 0; d < DIM; d++)
                t.r[((size_t)r * DIM + d) * m.C + i] = m.face_center[3 * (size_t)f + d] - m.cell_center[3 * (size_t)up + d];
        }
    }
}

template <int DIM, int ORDER, int MF>
__global__ void __launch_bounds__(kBlock) k_adv_run(Mesh m, AdvTable t, const double *__restrict__ w_in,
                                                    double *__restrict__ w_out, DtRing ring, double om)
{
    const int i = xcd_block() * blockDim.x + threadIdx.x;
    const double dt = ring.cur[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) {  // the ring as a step that forms the same dt leaves it
        ring.spare[0] = 1e6;
        ring.time[0] += dt;
        ring.next[0] = dt;
    }
    if (i >= m.C) return;
    int up[MF];
    double c[MF], r[MF][DIM], w[MF];
#pragma unroll
    for (int s = 0; s < MF; s++) {
        const size_t row = min(s, m.MF - 1);
        const int u = t.up[row * m.C + i];
        up[s] = (s < m.MF) ? u : kAdvNone;
        c[s] = t.coef[row * m.C + i];
        if (ORDER == 2) {
#pragma unroll
            for (int d = 0; d < DIM; d++) r[s][d] = t.r[(row * DIM + d) * m.C + i];
        }
    }
    const double wi = w_in[i], vol = m.cell_volume[i];
#pragma unroll
    for (int s = 0; s < MF; s++) {
        const int q = up[s] == kAdvNone ? i : up[s] < 0 ? ~up[s] : up[s];
        if (ORDER == 1) {
            w[s] = w_in[q] + 0.;
            continue;
        }
        const double2 *p = reinterpret_cast<const double2 *>(t.rec + adv_record(DIM) * (size_t)q);
        const double2 a = p[0], b = p[1];
        double full;
        if (DIM == 2)
            full = a.x + om * b.y * (a.y * r[s][0] + b.x * r[s][1]);
        else
            full = a.x + om * p[2].x * (a.y * r[s][0] + b.x * r[s][1] + b.y * r[s][DIM - 1]);
        w[s] = up[s] < 0 ? a.x : full;
    }
    double rez = 0.;
#pragma unroll
    for (int s = 0; s < MF; s++)
        if (up[s] != kAdvNone) rez -= c[s] * w[s];
    w_out[i] = wi + dt * ((rez + 0.) / vol + 0.);
}

// Two first-order steps in one launch: a cell forms the first step's value of each cell that its second
// step takes (its own for the faces it flows out of), which costs up to four times the loads and no
// barrier, and is faster where a step is no more than its launch (100 steps at 80k triangles 341 -> 300
// us, at 1k 361 -> 240). Same expressions, same bits. The ring: as by the first of the two steps, whose spare slot (which the
// second would reset) is this launch's dt and is left to the single steps that end a run.
template <int MF>
__global__ void __launch_bounds__(kBlock) k_adv_run_pair(Mesh m, AdvTable t, const double *__restrict__ w_in,
                                                         double *__restrict__ w_out, DtRing ring)
{
    const int i = xcd_block() * blockDim.x + threadIdx.x;
    const double dt = ring.cur[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ring.next[0] = dt;
        ring.spare[0] = dt;  // the slot of the step after these two
        ring.time[0] += dt;
        ring.time[0] += dt;
    }
    if (i >= m.C) return;
    int up[MF];
    double c[MF];
    auto slots = [&](int q, int (&u)[MF], double (&k)[MF]) {
#pragma unroll
        for (int s = 0; s < MF; s++) {
            const size_t row = min(s, m.MF - 1);
            u[s] = (s < m.MF) ? t.up[row * m.C + q] : kAdvNone;
            k[s] = t.coef[row * m.C + q];
        }
    };
    auto cell = [&](int u, int own) { return u == kAdvNone ? own : u < 0 ? ~u : u; };
    slots(i, up, c);
    int u1[MF + 1][MF], at[MF + 1];
    double c1[MF + 1][MF], w1[MF + 1], v1[MF + 1], g1[MF + 1][MF];
    at[MF] = i;
#pragma unroll
    for (int s = 0; s < MF; s++) at[s] = cell(up[s], i);
#pragma unroll
    for (int q = 0; q <= MF; q++) {
        if (q < MF) slots(at[q], u1[q], c1[q]);
        w1[q] = w_in[at[q]];
        v1[q] = m.cell_volume[at[q]];
    }
#pragma unroll
    for (int s = 0; s < MF; s++) {
        u1[MF][s] = up[s];
        c1[MF][s] = c[s];
    }
#pragma unroll
    for (int q = 0; q <= MF; q++)
#pragma unroll
        for (int s = 0; s < MF; s++) g1[q][s] = w_in[cell(u1[q][s], at[q])] + 0.;
    auto stepped = [&](double w, double vol, const int (&u)[MF], const double (&k)[MF], const double (&g)[MF]) {
        double rez = 0.;
#pragma unroll
        for (int s = 0; s < MF; s++)
            if (u[s] != kAdvNone) rez -= k[s] * g[s];
        return w + dt * ((rez + 0.) / vol + 0.);
    };
#pragma unroll
    for (int q = 0; q <= MF; q++) w1[q] = stepped(w1[q], v1[q], u1[q], c1[q], g1[q]);
    double g[MF];
#pragma unroll
    for (int s = 0; s < MF; s++) g[s] = w1[s] + 0.;
    w_out[i] = stepped(w1[MF], v1[MF], up, c, g);
}

}  // namespace

static int check_advection_run(const mfv_mesh *m, int order)
{
    MFV_REQUIRE(order == 1 || order == 2, "order must be 1 or 2");
    if (int rc = validate_mesh(m, order == 2, 1, 0)) return rc;
    MFV_REQUIRE(!(m->dim == 2 && m->max_cell_faces > 4), "2D cells have at most 4 faces");
    return MFV_OK;
}

extern "C" int mfv_advection_run_size(const mfv_mesh *m, int order, size_t *doubles)
{
    if (int rc = check_advection_run(m, order)) return rc;
    MFV_REQUIRE(doubles, "NULL pointer");
    AdvTable t;
    *doubles = adv_table(m, order, nullptr, &t);
    return MFV_OK;
}

extern "C" int mfv_advection_run(const mfv_mesh *m, double *w_a, double *w_b, const double *u_face,
                                 const double *v_face, const double *w_face, int order, double *dt_ring_p, int nsteps,
                                 double *workspace, const mfv_stencil_tiles *tiles, void *stream)
{
    if (int rc = check_advection_run(m, order)) return rc;
    if (tiles)
        if (int rc = check_stencil_tiles(m, tiles)) return rc;
    MFV_REQUIRE(nsteps >= 0, "nsteps < 0");
    MFV_REQUIRE(w_a && w_b && w_a != w_b && u_face && v_face && w_face && dt_ring_p && workspace,
                "NULL or aliased array");
    MFV_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0, "workspace must be 16-byte aligned");
    if (m->nb_cells == 0 || nsteps == 0) return MFV_OK;
    const Mesh k = to_kernel(m);
    const hipStream_t st = as_stream(stream);
    const dim3 g(grid_for(m->nb_cells)), b(kBlock);
    AdvTable t;
    adv_table(m, order, workspace, &t);
    auto kt = m->dim == 2 ? (order == 2 ? k_adv_table<2, 2> : k_adv_table<2, 1>)
                          : (order == 2 ? k_adv_table<3, 2> : k_adv_table<3, 1>);
    hipLaunchKernelGGL(kt, g, b, 0, st, k, t, u_face, v_face, w_face);
    if (int rc = check_launch("k_adv_table")) return rc;
    const int MF = m->max_cell_faces;
    auto ks = m->dim == 2 ? (MF <= 3 ? (order == 2 ? k_adv_run<2, 2, 3> : k_adv_run<2, 1, 3>)
                                     : (order == 2 ? k_adv_run<2, 2, 4> : k_adv_run<2, 1, 4>))
                          : (MF <= 4 ? (order == 2 ? k_adv_run<3, 2, 4> : k_adv_run<3, 1, 4>)
                                     : (order == 2 ? k_adv_run<3, 2, 8> : k_adv_run<3, 1, 8>));
    double *in = w_a, *out = w_b;
    // an even number of pairs, so that the buffers end as after nsteps single ones, and a single last
    const int pairs = (order == 1 && MF <= 4 && m->nb_cells <= (MF <= 3 ? kAdvPairCells3 : kAdvPairCells4))
                          ? (nsteps - 1) / 2 / 2 * 2
                          : 0;
    auto kp = MF <= 3 ? k_adv_run_pair<3> : k_adv_run_pair<4>;
    for (int p = 0; p < pairs; p++) {
        hipLaunchKernelGGL(kp, g, b, 0, st, k, t, in, out, dt_ring(dt_ring_p, 2 * p));
        if (int rc = check_launch("k_adv_run_pair")) return rc;
        double *x = in;
        in = out;
        out = x;
    }
    for (int s = 2 * pairs; s < nsteps; s++) {
        if (order == 2) {
            const GradArgs<1> a{{in}, {nullptr}, {t.rec}, {nullptr}, {nullptr}, {nullptr}};
            const int rc = tiles ? gradient_tiled<true, true>(m, tiles, a, st) : gradient_limited<1, true, true>(m, a, st);
            if (rc) return rc;
        }
        hipLaunchKernelGGL(ks, g, b, 0, st, k, t, in, out, dt_ring(dt_ring_p, s), (double)(order - 1));
        if (int rc = check_launch("k_adv_run")) return rc;
        double *x = in;
        in = out;
        out = x;
    }
    return MFV_OK;
}
