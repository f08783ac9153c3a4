// libmfv shallow water with the reference's own numerical flux and source: the SRNH
// Roe-type flux on five fields (h, hu, hv, hc, Z), MUSCL on h and hc limited by hc's psi,
// the well-balanced bathymetry source of triangles, and update_SW.
//
// The residual is a cell-centric gather: each cell evaluates the flux of each of its faces
// in the face's own orientation (left = faces.cellid[f][0]) and adds -F (left) or +F
// (right) in the order of the reference's face loops (inner faces by id, then boundary
// faces by id), so the float64 sums follow the reference's scatter term by term. The flux
// takes the sign matrix in closed form where the reference solves a cubic with acos and cos,
// so parity with the CPU restatement is to rounding, not bitwise.
#include "mfv_common.hpp"

namespace mfv {

struct Fields5 {
    const double *__restrict__ f[5];
};
struct Out5 {
    double *__restrict__ f[5];
};

// Sign matrix of the Roe state times w_dif (shallowater/fvm_utils.py:220-327, As = 0), the rows
// of (h, hu, hv, hc); the flux does not use the Z row.
//
// The reference finds the eigenvalues of the (h, hu, Z) block as the roots of a cubic (acos, three
// cos, two pow) and divides by their differences some thirty times. With As = 0 the roots are
// u + c, u - c and 0, the one at 0 has sign 0, and sign(A) w_dif is the sum of the two acoustic
// waves' strengths times their signs:
//   w+ = sign(u + c) (dhu - (u - c) dh + c^2 dZ / (u + c)) / (2 c)
//   w- = sign(u - c) ((u + c) dh - c^2 dZ / (u - c) - dhu) / (2 c)
// Against the formulas in extended precision (200k random states) the float64 error is 1.7e-16
// relative here and 2.2e-16 for the cubic in subcritical flow; near u = c, where the cubic's roots
// cancel, 8e-15 and 6e-12. Eigenvalues below 1e-10 have sign 0, as in the reference; their term
// is left out, not multiplied by 0 (its quotient may be infinite).
__device__ __forceinline__ void srnh_sign_apply(double hroe, double u, double v, double c, double grav,
                                                const double *w_dif, double *out)
{
    const double eps = 1e-10;
    const double ss = grav * hroe, sound = sqrt(ss);
    const double lp = u + sound, lm = u - sound;
    const double half = 0.5 / sound, zz = ss * w_dif[4];
    const double sp = (lp < 0.) ? -half : half, sm = (lm < 0.) ? -half : half;
    const double wp = (fabs(lp) < eps) ? 0. : sp * (w_dif[1] - lm * w_dif[0] + zz / lp);
    const double wm = (fabs(lm) < eps) ? 0. : sm * (lp * w_dif[0] - zz / lm - w_dif[1]);
    const double s4 = (fabs(u) < eps) ? 0. : (u < 0.) ? -1. : 1.;
    const double tot = wp + wm, rest = tot - s4 * w_dif[0];
    out[0] = tot;
    out[1] = lp * wp + lm * wm;
    out[2] = v * rest + s4 * w_dif[2];
    out[3] = c * rest + s4 * w_dif[3];
}

// srnh_scheme (shallowater/fvm_utils.py:152-342): flux in the face orientation, |n| = mes. The
// Roe averages use h / sqrt(h) = sqrt(h) and the normal is scaled once, which leaves nine
// divisions. The reference's fifth flux is As = 0 times a finite term.
__device__ __forceinline__ void srnh_flux(double hu_l, double hu_r, double hv_l, double hv_r, double h_l, double h_r,
                                          double hc_l, double hc_r, double Z_l, double Z_r, double n0, double n1,
                                          double mes, double grav, double *flux)
{
    const double e0 = n0 / mes, e1 = n1 / mes;
    const double sl = sqrt(h_l), sr = sqrt(h_r);
    const double il = 1. / sl, ir = 1. / sr, is = 1. / (sl + sr);
    const double u_h = (hu_l * il + hu_r * ir) * is;
    const double v_h = (hv_l * il + hv_r * ir) * is;
    const double c_h = (hc_l * il + hc_r * ir) * is;
    const double un_h = u_h * e0 + v_h * e1;
    const double vn_h = v_h * e0 - u_h * e1;
    const double hroe = (h_l + h_r) / 2.;
    const double uleft = hu_l * e0 + hv_l * e1;
    const double vleft = hv_l * e0 - hu_l * e1;
    const double uright = hu_r * e0 + hv_r * e1;
    const double vright = hv_r * e0 - hu_r * e1;
    double w_dif[5], corr[4];
    w_dif[0] = h_r - h_l;
    w_dif[1] = uright - uleft;
    w_dif[2] = vright - vleft;
    w_dif[3] = hc_r - hc_l;
    w_dif[4] = Z_r - Z_l;
    srnh_sign_apply(hroe, un_h, vn_h, c_h, grav, w_dif, corr);
    const double w_h = hroe - corr[0] / 2.;
    const double w_u = (uleft + uright) / 2. - corr[1] / 2.;
    const double w_v = (vleft + vright) / 2. - corr[2] / 2.;
    const double w_c = (hc_l + hc_r) / 2. - corr[3] / 2.;
    const double unew = w_u * e0 - w_v * e1;
    const double vnew = w_u * e1 + w_v * e0;
    const double q_s = n0 * unew + n1 * vnew;
    const double q_h = q_s / w_h, p = 0.5 * grav * w_h * w_h;
    flux[0] = q_s;
    flux[1] = q_h * unew + p * n0;
    flux[2] = q_h * vnew + p * n1;
    flux[3] = q_h * w_c;
    flux[4] = 0. * (q_h * (unew * unew + vnew * vnew));
}

// explicitscheme_convective_SW (shallowater/fvm_utils.py:344-496), one cell per thread. 200k
// cells at order 2: 21.8 us, and 65 us with the cubic's acos, cos and pow; bound by what it gathers
// now (110 MB past the L2s at 5.2 TB/s, a copy's rate; vector issue 0.42), by its arithmetic before.
__global__ void __launch_bounds__(kBlock) k_srnh_convective(Mesh m, Out5 rez, Fields5 cell, Fields5 ghost,
                                                            const double *__restrict__ h_x,
                                                            const double *__restrict__ h_y,
                                                            const double *__restrict__ hc_x,
                                                            const double *__restrict__ hc_y,
                                                            const double *__restrict__ psi, double om, double grav)
{
    const int i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= m.C) return;
    const double *h = cell.f[0], *hu = cell.f[1], *hv = cell.f[2], *hc = cell.f[3], *Z = cell.f[4];
    const int nf = m.cell_nfaces[i];
    double acc[5] = {0., 0., 0., 0., 0.};
    for (int r = 0; r < nf; r++) {
        const int s = m.order_split[(size_t)r * m.C + i];
        const int f = m.cell_faces[(size_t)s * m.C + i];
        const int L = m.face_cells[2 * f], R = m.face_cells[2 * f + 1];
        const double *cf = m.face_center + 3 * (size_t)f;
        const double *cl = m.cell_center + 3 * (size_t)L;
        const double *nrm = m.face_normal + 3 * (size_t)f;
        const double mes = m.face_mesure[f];
        const double rl0 = cf[0] - cl[0], rl1 = cf[1] - cl[1];
        const double h_l = h[L] + om * psi[L] * (h_x[L] * rl0 + h_y[L] * rl1);
        const double hc_l = hc[L] + om * psi[L] * (hc_x[L] * rl0 + hc_y[L] * rl1);
        double fl[5];
        if (R >= 0) {
            const double *cr = m.cell_center + 3 * (size_t)R;
            const double rr0 = cf[0] - cr[0], rr1 = cf[1] - cr[1];
            const double h_r = h[R] + om * psi[R] * (h_x[R] * rr0 + h_y[R] * rr1);
            const double hc_r = hc[R] + om * psi[R] * (hc_x[R] * rr0 + hc_y[R] * rr1);
            srnh_flux(hu[L], hu[R], hv[L], hv[R], h_l, h_r, hc_l, hc_r, Z[L], Z[R], nrm[0], nrm[1], mes, grav, fl);
        } else {
            srnh_flux(hu[L], ghost.f[1][f], hv[L], ghost.f[2][f], h_l, ghost.f[0][f], hc_l, ghost.f[3][f], Z[L],
                      ghost.f[4][f], nrm[0], nrm[1], mes, grav, fl);
        }
        if (L == i) {
#pragma unroll
            for (int k = 0; k < 5; k++) acc[k] -= fl[k];
        } else {
#pragma unroll
            for (int k = 0; k < 5; k++) acc[k] += fl[k];
        }
    }
#pragma unroll
    for (int k = 0; k < 5; k++) rez.f[k][i] = acc[k];
}

// term_source_srnh_SW (shallowater/fvm_utils.py:44-148) for triangles. With quirk the
// neighbour of face slot j is cellfid[i][j] of the compacted neighbour list, negative
// entries wrapping to the end as Python indexing does; without, the cell across face j.
struct SrnhSource {
    const int32_t *__restrict__ nodeid;
    const int32_t *__restrict__ cellfid;
    const double *__restrict__ nf;
    const double *__restrict__ vertex;
    int nw, fw, quirk;
};

__device__ __forceinline__ void srnh_source_cell(const Mesh &m, const SrnhSource &t, int i,
                                                 const double *__restrict__ h, const double *__restrict__ Z,
                                                 const double *__restrict__ h_ghost,
                                                 const double *__restrict__ Z_ghost, double grav, double &src_hu,
                                                 double &src_hv)
{
    const double *G = m.cell_center + 3 * (size_t)i;
    double ss[3][2], zv[3], mata[3], matb[3];
    double c_1 = 0., c_2 = 0.;
    const double h_1p = h[i], z_1p = Z[i];
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const int f = m.cell_faces[(size_t)j * m.C + i];
        ss[j][0] = t.nf[(size_t)i * 9 + j * 3 + 0];
        ss[j][1] = t.nf[(size_t)i * 9 + j * 3 + 1];
        double h_p1, z_p1;
        if (m.face_name[f] == 0) {
            int nb;
            if (t.quirk) {
                nb = t.cellfid[(size_t)i * t.fw + j];
                if (nb < 0) nb += m.C;
            } else {
                const int L = m.face_cells[2 * f];
                nb = (L == i) ? m.face_cells[2 * f + 1] : L;
            }
            h_p1 = h[nb];
            z_p1 = Z[nb];
        } else {
            h_p1 = h_ghost[f];
            z_p1 = Z_ghost[f];
        }
        zv[j] = z_p1;
        mata[j] = h_p1 * ss[j][0];
        matb[j] = h_p1 * ss[j][1];
        c_1 = c_1 + (0.5 * (h_1p + h_p1) * 0.5 * (h_1p + h_p1)) * ss[j][0];
        c_2 = c_2 + (0.5 * (h_1p + h_p1) * 0.5 * (h_1p + h_p1)) * ss[j][1];
    }
    const double c_3 = 3.0 * h_1p;
    const double delta = (mata[1] * matb[2] - mata[2] * matb[1]) - (mata[0] * matb[2] - matb[0] * mata[2]) +
                         (mata[0] * matb[1] - matb[0] * mata[1]);
    const double deltax = c_3 * (mata[1] * matb[2] - mata[2] * matb[1]) - (c_1 * matb[2] - c_2 * mata[2]) +
                          (c_1 * matb[1] - c_2 * mata[1]);
    const double deltay = (c_1 * matb[2] - c_2 * mata[2]) - c_3 * (mata[0] * matb[2] - matb[0] * mata[2]) +
                          (mata[0] * c_2 - matb[0] * c_1);
    const double deltaz = (mata[1] * c_2 - matb[1] * c_1) - (mata[0] * c_2 - matb[0] * c_1) +
                          c_3 * (mata[0] * matb[1] - matb[0] * mata[1]);
    const double h_1 = deltax / delta, h_2 = deltay / delta, h_3 = deltaz / delta;
    const double z_1 = z_1p + h_1p - h_1;
    const double z_2 = z_1p + h_1p - h_2;
    const double z_3 = z_1p + h_1p - h_3;
    const double *b = t.vertex + 4 * (size_t)t.nodeid[(size_t)i * t.nw + 1];
    double ns[3][2];
    ns[0][0] = G[1] - b[1];
    ns[0][1] = -(G[0] - b[0]);
#pragma unroll
    for (int k = 0; k < 2; k++) {
        ns[1][k] = ns[0][k] - ss[1][k];
        ns[2][k] = ns[0][k] + ss[0][k];
    }
    double s_1[2], s_2[2], s_3[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        s_1[k] = 0.5 * h_1 * (zv[0] * ss[0][k] + z_2 * ns[0][k] + z_3 * -1. * ns[2][k]);
        s_2[k] = 0.5 * h_2 * (zv[1] * ss[1][k] + z_1 * -1. * ns[0][k] + z_3 * ns[1][k]);
        s_3[k] = 0.5 * h_3 * (zv[2] * ss[2][k] + z_1 * ns[2][k] + z_2 * -1. * ns[1][k]);
    }
    src_hu = -grav * (s_1[0] + s_2[0] + s_3[0]);
    src_hv = -grav * (s_1[1] + s_2[1] + s_3[1]);
}

__global__ void __launch_bounds__(kBlock) k_srnh_source(Mesh m, SrnhSource t, Out5 src, const double *__restrict__ h,
                                                        const double *__restrict__ Z,
                                                        const double *__restrict__ h_ghost,
                                                        const double *__restrict__ Z_ghost, double grav)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m.C) return;
    double s1, s2;
    srnh_source_cell(m, t, i, h, Z, h_ghost, Z_ghost, grav, s1, s2);
    src.f[0][i] = 0.;
    src.f[1][i] = s1;
    src.f[2][i] = s2;
    src.f[3][i] = 0.;
    src.f[4][i] = 0.;
}

// update_SW (shallowater/fvm_utils.py:3-14), all five fields.
__global__ void __launch_bounds__(kBlock) k_update_sw5(int C, Out5 st, Fields5 rez, Fields5 src,
                                                       const double *__restrict__ dissip_hc,
                                                       const double *__restrict__ corio_hu,
                                                       const double *__restrict__ corio_hv, double wind_hu,
                                                       double wind_hv, double dtime,
                                                       const double *__restrict__ dt_dev,
                                                       const double *__restrict__ vol)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= C) return;
    const double dt = dt_dev ? dt_dev[0] : dtime;
    const double v = vol[i];
    st.f[0][i] += dt * (rez.f[0][i] + src.f[0][i]) / v;
    st.f[1][i] += dt * ((rez.f[1][i] + src.f[1][i]) / v + corio_hu[i] + wind_hu);
    st.f[2][i] += dt * ((rez.f[2][i] + src.f[2][i]) / v + corio_hv[i] + wind_hv);
    st.f[3][i] += dt * (rez.f[3][i] + src.f[3][i] - dissip_hc[i]) / v;
    st.f[4][i] += dt * (rez.f[4][i] + src.f[4][i]) / v;
}

// ----- steps in a row --------------------------------------------------------------------------
// What the sequence of entry points does per step in a face pass and a cell pass. Every face is evaluated
// once (nine divisions and three roots) and gathered for once, where the cell-centric residual does
// both twice for inner faces: 51 MB past the L2s in the face pass, at the 5.2 TB/s of a copy, for the
// residual's 110; the cell pass moves 84 MB at 4.8. The cell pass then adds the three fluxes in the
// residual's order, forms the source term, updates into a second set of fields (its neighbours still
// read this one) and takes the next time step's candidate, which otherwise are a launch and a trip
// of ten arrays each. 200k cells, second order: 9.9 + 18.1 us a step for 21.4 + 11.2 + 7.4 + 8.7 us of the four
// kernels (run of 10 steps 785 -> 633 us). Same expressions, same bits.
__global__ void __launch_bounds__(kBlock) k_srnh_face(Mesh m, Fields5 cell, Fields5 ghost,
                                                      const double *__restrict__ h_x, const double *__restrict__ h_y,
                                                      const double *__restrict__ hc_x,
                                                      const double *__restrict__ hc_y,
                                                      const double *__restrict__ psi, double om, double grav,
                                                      double4 *__restrict__ flux)
{
    const int f = xcd_block() * blockDim.x + threadIdx.x;
    if (f >= m.F) return;
    const double *h = cell.f[0], *hu = cell.f[1], *hv = cell.f[2], *hc = cell.f[3], *Z = cell.f[4];
    const int2 lr = face_pair(m, f);
    const int L = lr.x, R = lr.y, r = R >= 0 ? R : L;
    const double *cf = m.face_center + 3 * (size_t)f, *cl = m.cell_center + 3 * (size_t)L,
                 *cr = m.cell_center + 3 * (size_t)r, *nrm = m.face_normal + 3 * (size_t)f;
    const double mes = m.face_mesure[f];
    const double rl0 = cf[0] - cl[0], rl1 = cf[1] - cl[1], rr0 = cf[0] - cr[0], rr1 = cf[1] - cr[1];
    const double hL = h[L], hcL = hc[L], huL = hu[L], hvL = hv[L], zL = Z[L];
    double h_r, hc_r, hu_r, hv_r, z_r;
    const double h_l = hL + om * psi[L] * (h_x[L] * rl0 + h_y[L] * rl1);
    const double hc_l = hcL + om * psi[L] * (hc_x[L] * rl0 + hc_y[L] * rl1);
    if (R >= 0) {
        h_r = h[R] + om * psi[R] * (h_x[R] * rr0 + h_y[R] * rr1);
        hc_r = hc[R] + om * psi[R] * (hc_x[R] * rr0 + hc_y[R] * rr1);
        hu_r = hu[R];
        hv_r = hv[R];
        z_r = Z[R];
    } else {
        h_r = ghost.f[0][f];
        hu_r = ghost.f[1][f];
        hv_r = ghost.f[2][f];
        hc_r = ghost.f[3][f];
        z_r = ghost.f[4][f];
    }
    double fl[5];
    srnh_flux(huL, hu_r, hvL, hv_r, h_l, h_r, hc_l, hc_r, zL, z_r, nrm[0], nrm[1], mes, grav, fl);
    flux[f] = make_double4(fl[0], fl[1], fl[2], fl[3]);
}

// dt: dts[k], or the minimum of the nfold partials of the step before, which is then written there.
__global__ void __launch_bounds__(kBlock) k_srnh_cell(Mesh m, SrnhSource t, Fields5 cell, Fields5 ghost, Out5 out,
                                                      const double4 *__restrict__ flux,
                                                      const double *__restrict__ dissip_hc,
                                                      const double *__restrict__ corio_hu,
                                                      const double *__restrict__ corio_hv, double grav, double cfl,
                                                      double *__restrict__ dt_k, const double *__restrict__ fold,
                                                      int nfold, double *__restrict__ dtpart)
{
    const int i = xcd_block() * blockDim.x + threadIdx.x;
    const double dt = nfold ? fold_min(fold, nfold) : dt_k[0];
    if (nfold && blockIdx.x == 0 && threadIdx.x == 0) dt_k[0] = dt;
    double d = 1e300;
    if (i < m.C) {
        int face[3];
        double4 fl[3];
        bool left[3];
#pragma unroll
        for (int r = 0; r < 3; r++)
            face[r] = m.cell_faces[(size_t)m.order_split[(size_t)r * m.C + i] * m.C + i];
#pragma unroll
        for (int r = 0; r < 3; r++) {
            fl[r] = flux[face[r]];
            left[r] = m.face_cells[2 * (size_t)face[r]] == i;
        }
        double s1, s2;
        srnh_source_cell(m, t, i, cell.f[0], cell.f[4], ghost.f[0], ghost.f[4], grav, s1, s2);
        double acc[5] = {0., 0., 0., 0., 0.};
#pragma unroll
        for (int r = 0; r < 3; r++) {
            // the fifth flux is 0 times a term of the momentum's, finite where the momentum flux is
            const double v[5] = {fl[r].x, fl[r].y, fl[r].z, fl[r].w, 0. * (fl[r].y + fl[r].z)};
#pragma unroll
            for (int k = 0; k < 5; k++) {
                if (left[r]) acc[k] -= v[k];
                else acc[k] += v[k];
            }
        }
        const double vol = m.cell_volume[i];
        double u[5];
#pragma unroll
        for (int k = 0; k < 5; k++) u[k] = cell.f[k][i];
        u[0] += dt * (acc[0] + 0.) / vol;
        u[1] += dt * ((acc[1] + s1) / vol + corio_hu[i] + 0.);
        u[2] += dt * ((acc[2] + s2) / vol + corio_hv[i] + 0.);
        u[3] += dt * (acc[3] + 0. - dissip_hc[i]) / vol;
        u[4] += dt * (acc[4] + 0.) / vol;
#pragma unroll
        for (int k = 0; k < 5; k++) out.f[k][i] = u[k];
        d = sw_cell_dt<3>(m, i, u[0], u[1], u[2], cfl, grav, 0., 0.);
    }
    wave_min_part(dtpart, (size_t)i, d);
}

}  // namespace mfv

using namespace mfv;

extern "C" int mfv_explicitscheme_convective_sw(const mfv_mesh *m, double *rez_h, double *rez_hu, double *rez_hv,
                                                double *rez_hc, double *rez_Z, const double *h_c,
                                                const double *hu_c, const double *hv_c, const double *hc_c,
                                                const double *Z_c, const double *h_ghost, const double *hu_ghost,
                                                const double *hv_ghost, const double *hc_ghost,
                                                const double *Z_ghost, const double *h_x, const double *h_y,
                                                const double *hc_x, const double *hc_y, const double *psi,
                                                double grav, int order, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    MFV_REQUIRE(m->dim == 2, "shallow water needs a 2D mesh");
    MFV_REQUIRE(order == 1 || order == 2, "order must be 1 or 2");
    MFV_REQUIRE(rez_h && rez_hu && rez_hv && rez_hc && rez_Z && h_c && hu_c && hv_c && hc_c && Z_c && h_ghost &&
                    hu_ghost && hv_ghost && hc_ghost && Z_ghost && h_x && h_y && hc_x && hc_y && psi,
                "NULL array");
    if (m->nb_cells == 0) return MFV_OK;
    Out5 rez{{rez_h, rez_hu, rez_hv, rez_hc, rez_Z}};
    Fields5 cell{{h_c, hu_c, hv_c, hc_c, Z_c}};
    Fields5 ghost{{h_ghost, hu_ghost, hv_ghost, hc_ghost, Z_ghost}};
    hipLaunchKernelGGL(k_srnh_convective, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream),
                       to_kernel(m), rez, cell, ghost, h_x, h_y, hc_x, hc_y, psi, (double)(order - 1), grav);
    return check_launch("k_srnh_convective");
}

extern "C" int mfv_term_source_srnh_sw(const mfv_mesh *m, double *src_h, double *src_hu, double *src_hv,
                                       double *src_hc, double *src_Z, const double *h_c, const double *Z_c,
                                       const double *h_ghost, const double *Z_ghost, const int32_t *nodeid, int nw,
                                       const int32_t *cellfid, int fw, const double *nf, const double *vertex,
                                       double grav, int quirk, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    MFV_REQUIRE(m->dim == 2 && m->max_cell_faces == 3,
                "term_source_srnh_SW is defined for triangles only (2D, 3 faces per cell)");
    MFV_REQUIRE(nw >= 3 && fw >= 3, "nodeid / cellfid widths must be >= 3 (got %d, %d)", nw, fw);
    MFV_REQUIRE(src_h && src_hu && src_hv && src_hc && src_Z && h_c && Z_c && h_ghost && Z_ghost && nodeid &&
                    cellfid && nf && vertex,
                "NULL array");
    if (m->nb_cells == 0) return MFV_OK;
    Out5 src{{src_h, src_hu, src_hv, src_hc, src_Z}};
    const SrnhSource t{nodeid, cellfid, nf, vertex, nw, fw, quirk};
    hipLaunchKernelGGL(k_srnh_source, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream), to_kernel(m),
                       t, src, h_c, Z_c, h_ghost, Z_ghost, grav);
    return check_launch("k_srnh_source");
}

extern "C" int mfv_update_sw5(const mfv_mesh *m, double *h_c, double *hu_c, double *hv_c, double *hc_c, double *Z_c,
                              const double *rez_h, const double *rez_hu, const double *rez_hv, const double *rez_hc,
                              const double *rez_Z, const double *src_h, const double *src_hu, const double *src_hv,
                              const double *src_hc, const double *src_Z, const double *dissip_hc,
                              const double *corio_hu, const double *corio_hv, double wind_hu, double wind_hv,
                              double dtime, const double *dt_dev, void *stream)
{
    if (int rc = validate_mesh(m, 0, 0, 0)) return rc;
    MFV_REQUIRE(h_c && hu_c && hv_c && hc_c && Z_c && rez_h && rez_hu && rez_hv && rez_hc && rez_Z && src_h &&
                    src_hu && src_hv && src_hc && src_Z && dissip_hc && corio_hu && corio_hv,
                "NULL array");
    if (m->nb_cells == 0) return MFV_OK;
    Out5 st{{h_c, hu_c, hv_c, hc_c, Z_c}};
    Fields5 rez{{rez_h, rez_hu, rez_hv, rez_hc, rez_Z}};
    Fields5 src{{src_h, src_hu, src_hv, src_hc, src_Z}};
    hipLaunchKernelGGL(k_update_sw5, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, as_stream(stream), m->nb_cells,
                       st, rez, src, dissip_hc, corio_hu, corio_hv, wind_hu, wind_hv, dtime, dt_dev,
                       m->cell_volume);
    return check_launch("k_update_sw5");
}

extern "C" int mfv_srnh_run(const mfv_mesh *m, const mfv_srnh_step *p, int order, double grav, double cfl, double *dts,
                            int nsteps, void *stream)
{
    if (int rc = validate_mesh(m, order == 2, 1, 0)) return rc;
    MFV_REQUIRE(m->dim == 2 && m->max_cell_faces == 3, "the SRNH steps are defined for triangles only");
    MFV_REQUIRE(order == 1 || order == 2, "order must be 1 or 2");
    MFV_REQUIRE(nsteps >= 0 && nsteps % 2 == 0, "nsteps %d must be even (the fields alternate)", nsteps);
    MFV_REQUIRE(p && dts, "NULL descriptor");
    for (int k = 0; k < 5; k++)
        MFV_REQUIRE(p->cell[k] && p->cell2[k] && p->ghost[k] && p->cell[k] != p->cell2[k], "NULL or aliased field");
    MFV_REQUIRE(p->h_x && p->h_y && p->h_z && p->h_psi && p->hc_x && p->hc_y && p->hc_z && p->hc_psi && p->dissip_hc &&
                    p->corio_hu && p->corio_hv && p->flux && p->nodeid && p->cellfid && p->nf && p->vertex,
                "NULL array");
    MFV_REQUIRE((reinterpret_cast<uintptr_t>(p->flux) & 31) == 0, "flux must be 32-byte aligned");
    MFV_REQUIRE(p->nodeid_width >= 3 && p->cellfid_width >= 3, "nodeid / cellfid widths must be >= 3");
    MFV_REQUIRE(p->nb_segs >= 0 && p->nb_segs <= 64 && (p->nb_segs == 0 || p->segs), "0 to 64 ghost segments, got %d",
                p->nb_segs);
    if (m->nb_cells == 0 || nsteps == 0) return MFV_OK;
    const Mesh k = to_kernel(m);
    const SrnhSource t{p->nodeid, p->cellfid, p->nf, p->vertex, p->nodeid_width, p->cellfid_width, p->quirk};
    const size_t nw = waves_for(m->nb_cells);
    const bool fold = nw <= (size_t)kFoldMax;
    const hipStream_t st = as_stream(stream);
    double *part = dt_scratch(fold ? 2 * nw : nw, st);
    if (!part) return MFV_ENOMEM;
    double4 *flux = reinterpret_cast<double4 *>(p->flux);
    for (int s = 0; s < nsteps; s++) {
        double *const *in = s & 1 ? p->cell2 : p->cell, *const *out = s & 1 ? p->cell : p->cell2;
        const Fields5 cell{{in[0], in[1], in[2], in[3], in[4]}};
        const Fields5 ghost{{p->ghost[0], p->ghost[1], p->ghost[2], p->ghost[3], p->ghost[4]}};
        mfv_ghost_seg segs[64];
        for (int q = 0; q < p->nb_segs; q++) {
            segs[q] = p->segs[q];
            for (int v = 0; v < 5; v++)
                if (segs[q].kind != 2 && segs[q].w == p->cell[v]) segs[q].w = in[v];
        }
        if (int rc = mfv_ghost_values(m, segs, p->nb_segs, stream)) return rc;
        if (order == 2) {
            const mfv_gradient_fields g[2] = {{in[0], p->ghost[0], p->h_x, p->h_y, p->h_z, p->h_psi},
                                              {in[3], p->ghost[3], p->hc_x, p->hc_y, p->hc_z, p->hc_psi}};
            if (int rc = mfv_cell_gradient_limited(m, 2, g, stream)) return rc;
        }
        hipLaunchKernelGGL(k_srnh_face, dim3(grid_for(m->nb_faces)), dim3(kBlock), 0, st, k, cell, ghost, p->h_x, p->h_y,
                           p->hc_x, p->hc_y, p->hc_psi, (double)(order - 1), grav, flux);
        double *mine = part + (fold && (s & 1) ? nw : 0), *last = part + (fold && !(s & 1) ? nw : 0);
        hipLaunchKernelGGL(k_srnh_cell, dim3(grid_for(m->nb_cells)), dim3(kBlock), 0, st, k, t, cell, ghost,
                           Out5{{out[0], out[1], out[2], out[3], out[4]}}, flux, p->dissip_hc, p->corio_hu, p->corio_hv,
                           grav, cfl, dts + s, last, fold && s > 0 ? (int)nw : 0, mine);
        if (int rc = check_launch("k_srnh_cell")) return rc;
        if (!fold || s == nsteps - 1)
            if (int rc = dt_total(mine, nw, dts + s + 1, nullptr, kIdle, st)) return rc;
    }
    return MFV_OK;
}

// ---------------------------------------------------------------------------------------------
// term_friction_SW, term_coriolis_SW, term_wind_SW (shallowater/fvm_utils.py:498-544)

__global__ void __launch_bounds__(kBlock) k_term_friction_sw(int C, const double *__restrict__ h,
                                                              double *__restrict__ hu, double *__restrict__ hv,
                                                              double grav, double eta, double time)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= C) return;
    const double ufric = hu[i] / h[i];
    const double vfric = hv[i] / h[i];
    const double hfric = h[i];
    const double A = 1 + time * grav * (eta * eta) * (sqrt(ufric * ufric + vfric * vfric) / pow(hfric, 4. / 3.));
    const double hutild = hu[i] / A;
    const double hvtild = hv[i] / A;
    hu[i] = hutild;
    hv[i] = hvtild;
}

__global__ void __launch_bounds__(kBlock) k_term_coriolis_sw(int C, const double *__restrict__ hu,
                                                              const double *__restrict__ hv,
                                                              double *__restrict__ corio_hu,
                                                              double *__restrict__ corio_hv,
                                                              const double *__restrict__ f_c, double f_const)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= C) return;
    const double f = f_c ? f_c[i] : f_const;
    corio_hu[i] = f * hu[i];
    corio_hv[i] = -f * hv[i];
}

__global__ void __launch_bounds__(kBlock) k_term_wind_sw(int C, double *__restrict__ Tx, double *__restrict__ Ty,
                                                          const double *__restrict__ wx,
                                                          const double *__restrict__ wy)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= C) return;
    const double ro_a = 1.25;
    const double u = wx[i], v = wy[i];
    const double nor = sqrt(u * u + v * v);
    const double Cw = ro_a * (0.75 + 0.067 * nor) * 1e-03;
    Tx[i] = Cw * u * nor;
    Ty[i] = Cw * v * nor;
}

extern "C" int mfv_term_friction_sw(int C, const double *h, double *hu, double *hv, double grav, double eta,
                                    double time, void *stream)
{
    MFV_REQUIRE(C >= 0, "negative cell count");
    if (C == 0) return MFV_OK;
    MFV_REQUIRE(h && hu && hv, "NULL array");
    hipLaunchKernelGGL(k_term_friction_sw, dim3(grid_for(C)), dim3(kBlock), 0, as_stream(stream), C, h, hu, hv, grav,
                       eta, time);
    return check_launch("k_term_friction_sw");
}

extern "C" int mfv_term_coriolis_sw(int C, const double *hu, const double *hv, double *corio_hu, double *corio_hv,
                                    const double *f_c, double f_const, void *stream)
{
    MFV_REQUIRE(C >= 0, "negative cell count");
    if (C == 0) return MFV_OK;
    MFV_REQUIRE(hu && hv && corio_hu && corio_hv, "NULL array");
    hipLaunchKernelGGL(k_term_coriolis_sw, dim3(grid_for(C)), dim3(kBlock), 0, as_stream(stream), C, hu, hv,
                       corio_hu, corio_hv, f_c, f_const);
    return check_launch("k_term_coriolis_sw");
}

extern "C" int mfv_term_wind_sw(int C, double *Tx, double *Ty, const double *wind_wx, const double *wind_wy,
                                void *stream)
{
    MFV_REQUIRE(C >= 0, "negative cell count");
    if (C == 0) return MFV_OK;
    MFV_REQUIRE(Tx && Ty && wind_wx && wind_wy, "NULL array");
    hipLaunchKernelGGL(k_term_wind_sw, dim3(grid_for(C)), dim3(kBlock), 0, as_stream(stream), C, Tx, Ty, wind_wx,
                       wind_wy);
    return check_launch("k_term_wind_sw");
}
