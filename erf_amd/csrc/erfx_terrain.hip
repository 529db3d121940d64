// erfx_terrain.hip -- terrain-following grid: the metrics of the node heights
// and the acoustic substep erf_fast_rhs_T (static terrain, unit map factors).
//
// The substep runs as two launches: theta extrapolation, the horizontal momentum
// increments and the new horizontal momenta on the faces; and the columns (in
// tiles whose lanes share a column's levels, or one lane each), which form Omega
// of the old increments and the horizontal divergence of the new ones, solve the
// implicit vertical system and update rho, rho*theta and rho*w.  Every
// expression keeps the reference's operation order (FP contraction is off),
// so each point carries the reference's rounding.
#include "erfx_internal.h"
#include "erfx_terrain.h"

namespace erfx {

// one lane per element of the layout, padding included
template <class F>
__global__ void __launch_bounds__(256) lin_kernel(long n, F g) {
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    if (q < n) g(q);
}

// make_J, make_areas, make_zcc (Source/Utils/ERF_TerrainMetrics.cpp:583-715):
// detJ and z_cc on cells (-1..nx, -1..ny, 0..nz), ax on x-faces (-1..nx+1),
// ay on y-faces (-1..ny+1); 1 (0 for z_cc) everywhere else, az = 1.
void terrain_metrics(const Params& P, const double* z_nd, double* detJ, double* ax, double* ay, double* az,
                     double* z_cc, double* mrx, double* mry, hipStream_t s) {
    if (rec_refuse("terrain metrics")) return;
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz, ng = L.ng;
    const long ne = L.ne, sy = L.sy, sz = L.sz;
    const double dzInv = 1.0 / P.cfg.dz;
    const double dxi = P.dxInv[0], dyi = P.dxInv[1], dzi = P.dxInv[2];
    const Zn z{z_nd, L};
    const unsigned nb = (unsigned)((ne + 255) / 256);
    auto f = [=] __device__(long q) {
        const int k = (int)(q / sz) - ng;
        const long rem = q % sz;
        const int j = (int)(rem / sy) - ng, i = (int)(rem % sy) - ng;
        const bool kin = k >= 0 && k <= nz;
        double J = 1.0, Zc = 0.0, Ax = 1.0, Ay = 1.0;
        if (kin && i >= -1 && i <= nx && j >= -1 && j <= ny) {
            J = .25 * dzInv * (z(i, j, k + 1) + z(i + 1, j, k + 1) + z(i, j + 1, k + 1) + z(i + 1, j + 1, k + 1)
                               - z(i, j, k) - z(i + 1, j, k) - z(i, j + 1, k) - z(i + 1, j + 1, k));
            Zc = .125 * (z(i, j, k) + z(i + 1, j, k) + z(i, j + 1, k) + z(i + 1, j + 1, k)
                         + z(i, j, k + 1) + z(i + 1, j, k + 1) + z(i, j + 1, k + 1) + z(i + 1, j + 1, k + 1));
        }
        if (kin && i >= -1 && i <= nx + 1 && j >= -1 && j <= ny)
            Ax = .5 * dzInv * (z(i, j, k + 1) + z(i, j + 1, k + 1) - z(i, j, k) - z(i, j + 1, k));
        if (kin && i >= -1 && i <= nx && j >= -1 && j <= ny + 1)
            Ay = .5 * dzInv * (z(i, j, k + 1) + z(i + 1, j, k + 1) - z(i, j, k) - z(i + 1, j, k));
        detJ[q] = J; z_cc[q] = Zc; ax[q] = Ax; ay[q] = Ay; az[q] = 1.0;
        const bool kv = k >= 0 && k <= nz - 1;
        mrx[q] = (kv && i >= 0 && i <= nx && j >= 0 && j <= ny - 1)
                     ? met::h_xi_Iface(z, i, j, k, dxi) / met::h_zeta_Iface(z, i, j, k, dzi) : 0.0;
        mry[q] = (kv && i >= 0 && i <= nx - 1 && j >= 0 && j <= ny)
                     ? met::h_eta_Jface(z, i, j, k, dyi) / met::h_zeta_Jface(z, i, j, k, dzi) : 0.0;
    };
    hipLaunchKernelGGL(lin_kernel<decltype(f)>, dim3(nb), dim3(256), 0, s, ne, f);
}

// erf_fast_rhs_T (Source/TimeIntegration/ERF_fast_rhs_T.cpp:39-704), GPU
// branch of the column solve.  For step > 0 prev and data alias (S_sum).
void fast_rhs_T(const Params& P, const FastWork& W, const TerrainWork& T, int step, int nrk,
                const erfx_state& slow_rhs, const erfx_state& prev, const erfx_state& stage, const double* prim,
                const double* pi_stage, const double* fc, const erfx_state& data, const erfx_state& scratch,
                double dtau, double beta_s, double facinv, hipStream_t s, const FastChain& ch) {
    (void)nrk;
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const long ne = L.ne, sy = L.sy, sz = L.sz;
    const double beta_1 = 0.5 * (1.0 - beta_s);
    const double beta_2 = 0.5 * (1.0 + beta_s);
    const double beta_d = 0.1;
    const double dxi = P.dxInv[0], dyi = P.dxInv[1], dzi = P.dxInv[2];
    const bool moist = P.moist;
    const Zn z{P.z_nd, L};
    const double* J = P.detJ;
    double* cc0 = data.cons;
    double* cc1 = data.cons + ne;
    const double* pc0 = prev.cons;
    const double* pc1 = prev.cons + ne;
    const double* sc0 = stage.cons;
    const double* sc1 = stage.cons + ne;
    double* lagged1 = scratch.cons + ne;
    double* du = T.du; double* dv = T.dv;
    double* nu = T.nu; double* nv = T.nv; double* om = T.om;
    double* wtop = T.wtop;
    double* trhs0 = W.trhs;
    double* trhs1 = W.trhs + ne;
    double* soln = W.soln;
    const double* pxm = prev.xmom; const double* pym = prev.ymom; const double* pzm = prev.zmom;
    const double* sxm = stage.xmom; const double* sym = stage.ymom; const double* szm = stage.zmom;
    const bool first = step == 0;
    // The substep chain (laterally periodic box, Dirichlet top): prev is S_sum as the
    // previous substep left it, without the apply_bcs between the two.  What
    // that apply_bcs would give, the kernels form as they read: ghost cells of
    // rho*theta are the periodic images (foextrap rows above and below), and
    // each momentum is put through the momentum -> velocity -> momentum round
    // trip with the face density of its periodic image
    // (ERF_MomentumToVelocity.cpp, ERF_VelocityToMomentum.cpp), so the rounding
    // is the reference's.  The horizontal momenta of prev are stage + nu, the sum
    // the previous substep would have stored: the chain keeps the increments nu,
    // nv alone and stores the momenta in its last substep.
    const bool rt = ch.rt_prev && step > 0;
    const double* prho = prev.cons;
    auto wrap_c = [=] __device__(int a, int n) { return a < 0 ? a + n : (a > n - 1 ? a - n : a); };
    auto wrap_f = [=] __device__(int a, int n) { return a < 0 ? a + n : (a > n ? a - n : a); };
    // rho*w on the top face of column (i, j) as the skipped apply_bcs leaves it
    // (Dirichlet top on a terrain grid, ERF_BoundaryConditions_zvel.cpp:220-257):
    // w = WFromOmega of the top value with u and v as the fill makes them --
    // prev's momenta over the face density of the images, the level above the
    // top from the xvel / yvel top rules -- then rho*w with the top cell's
    // density (the cell above it is a copy).  On a plane top the slopes vanish
    // and w is the Dirichlet value.
    const int xth = P.bck[0][5], yth = P.bck[1][5];
    const double xvh = P.vel_extdir[0][5], yvh = P.vel_extdir[1][5], zvh = P.vel_extdir[2][5];
    auto u_fill = [=] __device__(int ii, int jj, int kk) -> double {
        if (kk > nz - 1) {
            if (xth == EXT_DIR) return xvh;
            kk = nz - 1;
        }
        const int fi = wrap_f(ii, nx), cj = wrap_c(jj, ny);
        const double d = prho[L.ix(wrap_c(fi, nx), cj, kk)] + prho[L.ix(wrap_c(fi - 1, nx), cj, kk)];
        const long f = L.ix(fi, cj, kk);
        return (sxm[f] + nu[f]) * 2.0 / d;
    };
    auto v_fill = [=] __device__(int ii, int jj, int kk) -> double {
        if (kk > nz - 1) {
            if (yth == EXT_DIR) return yvh;
            kk = nz - 1;
        }
        const int ci = wrap_c(ii, nx), fj = wrap_f(jj, ny);
        const double d = prho[L.ix(ci, wrap_c(fj, ny), kk)] + prho[L.ix(ci, wrap_c(fj - 1, ny), kk)];
        const long f = L.ix(ci, fj, kk);
        return (sym[f] + nv[f]) * 2.0 / d;
    };
    auto pw_top = [=] __device__(int i, int j) -> double {
        const double w = met::w_from_omega(i, j, nz, zvh, u_fill, v_fill, z, dxi, dyi);
        const double r = prho[L.ix(i, j, nz - 1)];
        return w * 0.5 * (r + r);
    };

    // in the chain: rho*w of the top face of every column (read by the column
    // kernel), before the increments and the densities of prev are overwritten
    if (rt) {
        launch_box(Box(0, 0, 0, nx - 1, ny - 1, 0), s,
                   [=] __device__(int i, int j, int) { wtop[L.ix(i, j, -L.ng)] = pw_top(i, j); });
    }

    // :139-331 in one launch: theta extrapolated forward, the horizontal momentum
    // increments of prev (kept in du, dv for the column kernel, because the new
    // momenta overwrite prev when it aliases data) and the horizontal momenta with
    // the terrain-corrected pressure gradient.
    // HBM bound: 17 fields read and 6 (8 in a stage's last substep) written, where
    // increments and momenta in launches of their own moved 34 (512 x 512 x 96: 1418
    // us for the two, 1130 us as one).  Each lane marches
    // up a chunk of KC levels of its (i, j) and forms the extrapolated increment
    // of its own column and of the columns at i-1 and j-1, kept for levels k-1, k
    // and k+1 in registers, so every level is read once per chunk (the box order
    // would put the levels of the gradient's stencil a whole plane of tiles
    // apart); the columns shared by neighbouring lanes are L2 hits.
    const double* pq1 = prim + PRIM_Q1 * ne;
    const double* pq2 = prim + PRIM_Q2 * ne;
    const double* srx = slow_rhs.xmom;
    const double* sry = slow_rhs.ymom;
    double* axm = scratch.xmom;
    double* aym = scratch.ymom;
    double* dxm = data.xmom;
    double* dym = data.ymom;
    const double* mrx = P.mrx;
    const double* mry = P.mry;
    const double* drt = first ? pc1 : cc1;
    const bool store_mom = !ch.active || ch.last;
    constexpr int KC = 12;   // 512 x 512 x 96: 1147 us at 24 levels, 1130 at 12, 1142 at 8
    const int nch = (nz + KC - 1) / KC;
    launch_box(Box(0, 0, 0, nx, ny, nch - 1), s, [=] __device__(int i, int j, int c) {
        const int k0 = c * KC, k1 = k0 + KC < nz ? k0 + KC : nz;
        const bool xf = j <= ny - 1, yf = i <= nx - 1;
        long q = L.ix(i, j, k0);
        // the cells of the faces as offsets from q: c (i, j), x (i-1, j), y (i, j-1);
        // in the chain ghost cells are their periodic images
        const long oc = rt ? (i == nx ? -(long)nx : 0) + (j == ny ? -(long)ny * sy : 0) : 0;
        const long ox = (rt && i == 0) ? nx - 1 : -1;
        const long oy = (rt && j == 0) ? (long)(ny - 1) * sy : -sy;
        auto ext = [&](long a) {
            const double d = drt[a] - sc1[a];
            return first ? d : d + beta_d * (d - lagged1[a]);
        };
        // m / 0 / p: levels k-1 / k / k+1
        double ecm = 0.0, exm = 0.0, eym = 0.0;
        if (k0 > 0) {
            ecm = ext(q + oc - sz);
            if (xf) exm = ext(q + ox - sz);
            if (yf) eym = ext(q + oy - sz);
        }
        double ec0 = ext(q + oc);
        double ex0 = xf ? ext(q + ox) : 0.0;
        double ey0 = yf ? ext(q + oy) : 0.0;
        for (int k = k0; k < k1; ++k, q += sz) {
            // the level above the top is a copy of the top one in the chain
            const long up = (rt && k == nz - 1) ? 0 : sz;
            const double ecp = ext(q + oc + up);
            const double exp_ = xf ? ext(q + ox + up) : 0.0;
            const double eyp = yf ? ext(q + oy + up) : 0.0;
            // all loads of the level before its first store, which may alias them
            // as far as the compiler knows (a face outside its box reads inside
            // the layout; only its stores are guarded)
            const double sx = sxm[q], sy_ = sym[q], lx = srx[q], ly = sry[q], ax = axm[q], ay = aym[q];
            const double mx = mrx[q], my = mry[q];
            const double pc = pi_stage[q], px = pi_stage[q - 1], py = pi_stage[q - sy];
            double pmx, pmy, rc = 0.0, rx = 0.0, ry = 0.0;
            if (rt) {
                pmx = sx + nu[q];
                pmy = sy_ + nv[q];
                rc = prho[q + oc]; rx = prho[q + ox]; ry = prho[q + oy];
            } else {
                pmx = pxm[q];
                pmy = pym[q];
            }
            const double gp_xi = (ec0 - ex0) * dxi;
            const double gp_zeta_on_iface = (k == 0)
                ? 0.5 * dzi * (exp_ + ecp - ex0 - ec0)
                : 0.25 * dzi * (exp_ + ecp - exm - ecm);
            double gpx = gp_xi - mx * gp_zeta_on_iface;   // (h_xi / h_zeta) made once
            const double gp_eta = (ec0 - ey0) * dyi;
            const double gp_zeta_on_jface = (k == 0)
                ? 0.5 * dzi * (ecp + eyp - ec0 - ey0)
                : 0.25 * dzi * (ecp + eyp - ecm - eym);
            double gpy = gp_eta - my * gp_zeta_on_jface;   // (h_eta / h_zeta) made once
            if (moist) {
                gpx /= (1.0 + face_q(pq1, pq2, q, q - 1));
                gpy /= (1.0 + face_q(pq1, pq2, q, q - sy));
            }
            if (rt) {
                const double d = rc + rx, e = rc + ry;
                const double u = pmx * 2.0 / d, v = pmy * 2.0 / e;
                pmx = u * 0.5 * d;
                pmy = v * 0.5 * e;
            }
            const double ix = pmx - sx, iy = pmy - sy_;
            const double nx_ = ix + dtau * (-Gamma * R_d * (0.5 * (px + pc)) * gpx) + dtau * lx;
            const double ny_ = iy + dtau * (-Gamma * R_d * (0.5 * (py + pc)) * gpy) + dtau * ly;
            if (xf) {
                du[q] = ix;
                nu[q] = nx_;
                axm[q] = ax + facinv * nx_;
                if (store_mom) dxm[q] = sx + nx_;
            }
            if (yf) {
                dv[q] = iy;
                nv[q] = ny_;
                aym[q] = ay + facinv * ny_;
                if (store_mom) dym[q] = sy_ + ny_;
            }
            ecm = ec0; ec0 = ecp;
            exm = ex0; ex0 = exp_;
            eym = ey0; ey0 = eyp;
        }
    });
    // the ghost layer of the lagged increment and, in the first substep, of rho
    // and rho*theta (:139-152), which the chain reads at the images instead (written
    // with the column launch below)
    const LaggedShell shell{L, drt, sc1, lagged1, first ? cc0 : nullptr, pc0};

    // :414-669, one lane per (i, j) column.  The forward sweep makes, level by
    // level, Omega of the old increments (:460-484) on the face above, the
    // horizontal divergence of the area-weighted new increments (:414-457) in
    // the cell, the tridiagonal right-hand side on the face (:499-552) and the
    // elimination (:561-581, GPU branch); Omega, the divergences and the
    // solution are kept for the backward sweep: substitution, rho*w = stage +
    // WFromOmega on the interior faces (faces 0 and nz keep the stage value,
    // :620-633), the time-averaged Omega and the rho, rho*theta update (:640-669).
    const Fld fdu{du, L}, fdv{dv, L}, fnu{nu, L}, fnv{nv, L};
    const double* cr0 = first ? pc0 : cc0;   // rho, rho*theta at the substep's start
    const double* cr1 = first ? pc1 : cc1;
    const double halfg = fabs(0.5 * (-P.gravity));
    const double* sr0 = slow_rhs.cons;
    const double* sr1 = slow_rhs.cons + ne;
    const double* srz = slow_rhs.zmom;
    const double* fA = fc;
    const double* fB = fc + ne;
    const double* fC = fc + 2 * ne;
    const double* fP = fc + 3 * ne;
    const double* fQ = fc + 4 * ne;
    double* cz = data.zmom;
    double* azm = scratch.zmom;
    kt_start(P.timer, KT_FAST_COLUMN, s);
    // The tile form (launch_relay; the default for boxes of up to 96 levels), as
    // the flat grid's: 32 (or 16) columns per work-group of 8 waves, one lane per
    // column and chunk of levels.  Each lane reads its levels once -- node
    // heights, increments and theta of a level serve the level above from
    // registers -- and forms the divergences, Omega, the slope terms and the
    // tridiagonal rows; the chunks hand their top cell up through LDS; the sweeps
    // run from registers (short chunks from LDS); and each lane updates its cells
    // from what it holds.  Every value is the column kernel's expression, so the
    // results are bit-identical.  HBM bound: the form this replaced (64 columns,
    // rows swept in LDS, operands read again for the update) moved 49 fields on
    // 512 x 512 x 96 and took 2105 us where this takes 1464 (1692 with 16-column
    // tiles, whose rows are one cache line).
    const bool own = ch.own_coeffs;
    const double Dc = dtau * dtau * beta_2 * beta_2 * dzi;
    auto relay = [=] __device__(int i, int j, bool valid, int col, int chunk, double* lds, auto cmc, auto tcc) {
        constexpr int CM = decltype(cmc)::value;
        constexpr int TC = decltype(tcc)::value;
        constexpr int NCH = 512 / TC;
        constexpr int NA = CM > 4 ? 5 : 4;         // arrays in the lane's own LDS slots
        const int tid = (int)threadIdx.x;
        const int chl = tile_chunk(nz, NCH);
        const int ka = chunk * chl;
        const int kb = (ka + chl < nz ? ka + chl : nz) - 1;
        const bool has = ka <= kb;
        const bool work = valid && has;
        const bool top = has && kb == nz - 1;
        const long q0 = valid ? L.ix(i, j, 0) : 0;
        auto slot = [&](int a, int m) -> double& { return lds[(a * CM + m) * 512 + tid]; };
        auto below = [&](int a) -> double { return lds[(a * CM + chl - 1) * 512 + tid - TC]; };
        double* xch = lds + NA * CM * 512;
        constexpr int NX = NA == 5 ? 9 : 6;        // exchange rows; 6..8 hold this lane's own first cell
        double* carry = xch + NX * 512;
        enum { T0 = 0, T1, S0, S1, PX };
        double rhs[CM], av[CM], bv[CM], cv[CM], om[CM + 1], c0r[CM], c1r[CM], pp[CM], sz_[CM], Jr[CM], pyr[CM];
        double pxr[NA == 5 ? 1 : CM];
        double r_top = 0.0, a_top = 0.0, b_top = 0.0, s_top = 0.0;
        // of the chunk's first cell, until its face's row is finished
        double f_cP = 0.0, f_cQ = 0.0, f_ws = 0.0, f_dw = 0.0, f_drho = 0.0, f_drt = 0.0, f_q1 = 0.0, f_q2 = 0.0;
        double f_pm2 = 0.0, f_pm1 = 0.0, f_pp1 = 0.0;
        struct Cell { double drho, drt, s0, s1, t0, t1, q1, q2, om, J; };   // om: of the cell's lower face
        // row k of the system (:499-552): cell k is `c`, the cell below `b`; dw the
        // old rho*w increment, px, py the slope terms of the new increments
        auto row = [&](double cP, double cQ, double ws, double dw, double px, double py, const Cell& c, const Cell& b,
                       double om_p, double p_km2, double p_km1, double p_k, double p_kp1, double& a,
                       double& cc) -> double {
            const double ofw = (0. - px) - py;
            double detJ_on_kface = 0.5 * (c.J + b.J);
            if (moist) {
                double qf = 0.5 * (c.q1 + b.q1 + c.q2 + b.q2);
                cP /= (1.0 + qf);
                cQ /= (1.0 + qf);
            }
            double theta_t_lo = 0.5 * (p_km2 + p_km1);
            double theta_t_mid = 0.5 * (p_km1 + p_k);
            double theta_t_hi = 0.5 * (p_k + p_kp1);
            double R0_tmp = (-halfg * c.drho + cP * c.drt) * c.J
                          + (-halfg * b.drho + cQ * b.drt) * b.J;
            double R1_tmp = -halfg * (c.s0 * c.J + b.s0 * b.J)
                          + (cP * c.s1 * c.J + cQ * b.s1 * b.J);
            R1_tmp += (halfg) * (beta_1 * dzi * (om_p - b.om) + c.t0 + b.t0);
            R1_tmp += -(cP * (beta_1 * dzi * (om_p * theta_t_hi - c.om * theta_t_mid) + c.t1) +
                        cQ * (beta_1 * dzi * (c.om * theta_t_mid - b.om * theta_t_lo) + b.t1));
            if (own) {
                a = Dc * (halfg - cQ * theta_t_lo);
                cc = Dc * (-halfg + cP * theta_t_hi);
            }
            double r = detJ_on_kface * dw + dtau * (detJ_on_kface * ws + R0_tmp + dtau * beta_2 * R1_tmp);
            r += detJ_on_kface * ofw;
            return r;
        };
        // nodes of a level: z(i, j), z(i+1, j), z(i, j+1), z(i+1, j+1)
        struct Nodes { double a, b, c, d; };
        auto nodes = [&](long q) -> Nodes { return {z.z[q], z.z[q + 1], z.z[q + sy], z.z[q + 1 + sy]}; };
        auto slope_x = [&](const Nodes& n) { return 0.5 * dxi * (n.d + n.b - n.c - n.a); };   // met::zlo_xi
        auto slope_y = [&](const Nodes& n) { return 0.5 * dyi * (n.d + n.c - n.b - n.a); };   // met::zlo_eta
        // prev rho*w on face kf (q its index), with the densities above and below
        auto pw = [&](int kf, long q, double r_hi, double r_lo) -> double {
            if (!rt) return pzm[q];
            if (kf >= nz) return wtop[L.ix(i, j, -L.ng)];
            const double d = r_hi + r_lo;
            const double w = pzm[q] * 2.0 / d;
            return w * 0.5 * d;
        };
        // ---- phase 1: one reading of the chunk's levels ----
        if (work) {
            const long qa = q0 + (long)ka * sz;
            double p_m2 = ka > 1 ? prim[qa - 2 * sz] : prim[q0 - sz], p_m1 = prim[qa - sz], p_k = prim[qa];
            double c0_k = cr0[qa], sz_k = szm[qa];
            Nodes zk = nodes(qa);
            double du0 = du[qa], du1 = du[qa + 1], dv0 = dv[qa], dv1 = dv[qa + sy];
            double nu0 = 0.0, nu1 = 0.0, nv0 = 0.0, nv1 = 0.0;      // of the level below
            double dw_k = 0.0, om_k = 0.0;
            if (ka > 0) {
                const long ql = qa - sz;
                nu0 = nu[ql]; nu1 = nu[ql + 1]; nv0 = nv[ql]; nv1 = nv[ql + sy];
                dw_k = pw(ka, qa, c0_k, rt ? prho[ql] : 0.0) - sz_k;
                const double uu = 0.25 * (du[ql] + du[ql + 1] + du0 + du1);
                const double vv = 0.25 * (dv[ql] + dv[ql + sy] + dv0 + dv1);
                om_k = dw_k - slope_x(zk) * uu - slope_y(zk) * vv;
            }
            Cell b{};
            double o_top = 0.0, J_top = 0.0;
#pragma unroll
            for (int m = 0; m < CM; ++m) {
                const int k = ka + m;
                if (k > kb) break;
                const long q = q0 + (long)k * sz;
                const double ws = srz[q], cP = fP[q], cQ = fQ[q];
                bv[m] = fB[q];
                if (!own) { av[m] = fA[q]; cv[m] = fC[q]; }
                const double p_p = prim[q + sz], c0_p = cr0[q + sz], sz_p = szm[q + sz];
                const Nodes zn = nodes(q + sz);
                const double eu0 = du[q + sz], eu1 = du[q + sz + 1], ev0 = dv[q + sz], ev1 = dv[q + sz + sy];
                const double mu0 = nu[q], mu1 = nu[q + 1], mv0 = nv[q], mv1 = nv[q + sy];
                const double c1_k = cr1[q], st0 = sc0[q], st1 = sc1[q];
                const double pxm = prim[q - 1], pxp = prim[q + 1], pym = prim[q - sy], pyp = prim[q + sy];
                Cell c;
                c.s0 = sr0[q]; c.s1 = sr1[q]; c.J = J[q];
                c.q1 = 0.0; c.q2 = 0.0;
                if (moist) { c.q1 = pq1[q]; c.q2 = pq2[q]; }
                const double dw_p = pw(k + 1, q + sz, c0_p, c0_k) - sz_p;
                // horizontal divergence of the area-weighted new increments (:414-457)
                double h_xhi = 0.5 * dzi * (zn.b + zn.d - zk.b - zk.d);
                double h_xlo = 0.5 * dzi * (zn.a + zn.c - zk.a - zk.c);
                double h_yhi = 0.5 * dzi * (zn.c + zn.d - zk.c - zk.d);
                double h_ylo = 0.5 * dzi * (zn.a + zn.b - zk.a - zk.b);
                double xflux_lo = mu0 * h_xlo, xflux_hi = mu1 * h_xhi;
                double yflux_lo = mv0 * h_ylo, yflux_hi = mv1 * h_yhi;
                c.t0 = (xflux_hi - xflux_lo) * dxi + (yflux_hi - yflux_lo) * dyi;
                c.t1 = ((xflux_hi * (p_k + pxp) - xflux_lo * (p_k + pxm)) * dxi +
                        (yflux_hi * (p_k + pyp) - yflux_lo * (p_k + pym)) * dyi) * 0.5;
                // Omega of the old increments on the face above (:460-484)
                double om_p = dw_p;
                if (k < nz - 1) {
                    const double uu = 0.25 * (du0 + du1 + eu0 + eu1);
                    const double vv = 0.25 * (dv0 + dv1 + ev0 + ev1);
                    om_p = dw_p - slope_x(zn) * uu - slope_y(zn) * vv;
                }
                c.om = om_k;
                c.drho = c0_k - st0;
                c.drt = c1_k - st1;
                lagged1[q] = c.drt;
                // the slope terms of the lower face with the new increments
                double px = 0.0, py = 0.0;
                if (k > 0) {
                    px = slope_x(zk) * (0.25 * (nu0 + nu1 + mu0 + mu1));
                    py = slope_y(zk) * (0.25 * (nv0 + nv1 + mv0 + mv1));
                }
                if (m > 0) {
                    const int l = m > 0 ? m - 1 : 0;
                    b.t0 = slot(T0, l); b.t1 = slot(T1, l); b.s0 = slot(S0, l); b.s1 = slot(S1, l);
                    b.om = om[l]; b.J = Jr[l];
                    rhs[m] = row(cP, cQ, ws, dw_k, px, py, c, b, om_p, p_m2, p_m1, p_k, p_p, av[m], cv[m]);
                } else if (k == 0) {      // face 0
                    rhs[m] = dtau * ws;
                    if (own) { av[m] = 0.0; cv[m] = 0.0; }
                } else {
                    if constexpr (NA == 5) {
                        xch[6 * 512 + tid] = cP; xch[7 * 512 + tid] = cQ; xch[8 * 512 + tid] = ws;
                    } else {
                        f_cP = cP; f_cQ = cQ; f_ws = ws;
                    }
                    f_dw = dw_k; f_drho = c.drho; f_drt = c.drt;
                    f_q1 = c.q1; f_q2 = c.q2; f_pm2 = p_m2; f_pm1 = p_m1; f_pp1 = p_p;
                }
                slot(T0, m) = c.t0; slot(T1, m) = c.t1; slot(S0, m) = c.s0; slot(S1, m) = c.s1;
                if constexpr (NA == 5) slot(PX, m) = px; else pxr[m] = px;
                pyr[m] = py; Jr[m] = c.J;
                om[m] = om_k; om[m + 1] = om_p;
                o_top = om_k; J_top = c.J;
                c0r[m] = c0_k; c1r[m] = c1_k; pp[m] = p_k; sz_[m] = sz_k;
                tile_level_fence();
                b.drho = c.drho; b.drt = c.drt; b.q1 = c.q1; b.q2 = c.q2;
                p_m2 = p_m1; p_m1 = p_k; p_k = p_p;
                c0_k = c0_p; sz_k = sz_p; om_k = om_p; dw_k = dw_p;
                zk = zn;
                du0 = eu0; du1 = eu1; dv0 = ev0; dv1 = ev1;
                nu0 = mu0; nu1 = mu1; nv0 = mv0; nv1 = mv1;
            }
            // the top cell, for the chunk above
            xch[tid] = b.drho; xch[512 + tid] = b.drt; xch[2 * 512 + tid] = o_top; xch[3 * 512 + tid] = J_top;
            if (moist) { xch[4 * 512 + tid] = b.q1; xch[5 * 512 + tid] = b.q2; }
            if (top) {   // the top face: the right-hand side of its elimination step
                const long qt = q0 + (long)nz * sz;
                r_top = dtau * srz[qt];
                a_top = fA[qt];
                b_top = fB[qt];
            }
        }
        __syncthreads();
        if (work && ka > 0) {
            Cell c, b;
            b.drho = xch[tid - TC]; b.drt = xch[512 + tid - TC]; b.om = xch[2 * 512 + tid - TC];
            b.J = xch[3 * 512 + tid - TC];
            b.q1 = 0.0; b.q2 = 0.0;
            if (moist) { b.q1 = xch[4 * 512 + tid - TC]; b.q2 = xch[5 * 512 + tid - TC]; }
            b.t0 = below(T0); b.t1 = below(T1); b.s0 = below(S0); b.s1 = below(S1);
            c.drho = f_drho; c.drt = f_drt; c.q1 = f_q1; c.q2 = f_q2; c.om = om[0]; c.J = Jr[0];
            c.t0 = slot(T0, 0); c.t1 = slot(T1, 0); c.s0 = slot(S0, 0); c.s1 = slot(S1, 0);
            double px;
            if constexpr (NA == 5) {
                px = slot(PX, 0);
                f_cP = xch[6 * 512 + tid]; f_cQ = xch[7 * 512 + tid]; f_ws = xch[8 * 512 + tid];
            } else {
                px = pxr[0];
            }
            rhs[0] = row(f_cP, f_cQ, f_ws, f_dw, px, pyr[0], c, b, om[1], f_pm2, f_pm1, pp[0], f_pp1, av[0], cv[0]);
        }
        // ---- phase 2 ----
        double x_hi = 0.0;       // the solution on the chunk's upper face
        relay_solve<CM, TC>(carry, xch, true, nz, chl, col, valid, rhs, av, bv, cv, r_top, a_top, b_top, s_top, x_hi);
        // ---- phase 3: rho*w, the averaged Omega, rho and rho*theta of the chunk ----
        if (work) {
            if (top) {
                const long qt = q0 + (long)nz * sz;
                cz[qt] = szm[qt];
            }
            const double p_top = prim[q0 + (long)(kb + 1) * sz], p_bot = prim[q0 + (long)(ka - 1) * sz];
            double az[CM];
#pragma unroll
            for (int m = 0; m < CM; ++m)
                if (ka + m <= kb) az[m] = azm[q0 + (long)(ka + m) * sz];
#pragma unroll
            for (int m = 0; m < CM; ++m) {
                const int k = ka + m;
                if (k > kb) break;
                const long q = q0 + (long)k * sz;
                const bool last = k == kb;
                const double sol = rhs[m], sol_hi = last ? x_hi : rhs[m + 1 < CM ? m + 1 : m];
                const double pq = pp[m], p_hi = last ? p_top : pp[m + 1 < CM ? m + 1 : m];
                const double p_lo = m == 0 ? p_bot : pp[m > 0 ? m - 1 : 0];
                double px;
                if constexpr (NA == 5) px = slot(PX, m); else px = pxr[m];
                const double cz_k = (k >= 1) ? sz_[m] + ((sol + px) + pyr[m]) : sz_[m];
                double zflux_lo = beta_2 * sol + beta_1 * om[m];
                double zflux_hi = beta_2 * sol_hi + beta_1 * om[m + 1];
                double fast_rhs_rho = -(slot(T0, m) + (zflux_hi - zflux_lo) * dzi) / Jr[m];
                double fast_rhs_rhotheta = -(slot(T1, m) + 0.5 * (zflux_hi * (pq + p_hi) -
                                                                  zflux_lo * (pq + p_lo)) * dzi) / Jr[m];
                cz[q] = cz_k;
                azm[q] = az[m] + facinv * zflux_lo / (1.0 * 1.0);
                if (k == nz - 1) azm[q + sz] += facinv * zflux_hi / (1.0 * 1.0);
                cc0[q] = c0r[m] + dtau * (slot(S0, m) + fast_rhs_rho);
                cc1[q] = c1r[m] + dtau * (slot(S1, m) + fast_rhs_rhotheta);
            }
        }
    };
    // a recorded (batched) launch takes chunks of 6 levels in 32-column tiles, so
    // every member of a batch records the same kernel
    if (nz <= 96 && P.col_variant == COL_TILE) {
        if (!ch.active && g_rec) lagged_shell(shell, s);
        auto launch = [&](auto cmc, auto tcc) {
            constexpr int CM = decltype(cmc)::value;
            launch_relay<CM, decltype(tcc)::value, (CM > 4 ? 5 : 4), (CM > 4 ? 9 : 6)>(0, nx - 1, 0, ny - 1, s,
                [=] __device__(int i, int j, bool valid, int col, int chunk, double* lds) {
                    relay(i, j, valid, col, chunk, lds, cmc, tcc);
                }, ch.active ? 0u : shell.lanes(), shell);
        };
        using IC16 = std::integral_constant<int, 16>;
        using IC32 = std::integral_constant<int, 32>;
        using IC4 = std::integral_constant<int, 4>;
        using IC6 = std::integral_constant<int, 6>;
        if (!g_rec && tile_columns((long)nx * ny) == 16) launch(IC4{}, IC16{});   // 32 chunks: at most 3 levels each
        else if (!g_rec && tile_chunk(nz, 16) <= 4) launch(IC4{}, IC32{});
        else launch(IC6{}, IC32{});
    } else {
    if (!ch.active) lagged_shell(shell, s);
    launch_cols(0, nx - 1, 0, ny - 1, s, [=] __device__(int i, int j) {
        const long q0 = L.ix(i, j, 0);
        // Omega of the old increments on face kf (0 at the bottom, the rho*w
        // increment at the top, OmegaFromW between)
        // prev rho*w on interior face kf (round trip with the two cells' density
        // in the substep chain); the top face keeps what the last substep wrote
        auto pw = [&](int kf) -> double {
            const long q = q0 + (long)kf * sz;
            if (!rt) return pzm[q];
            if (kf >= nz) return wtop[L.ix(i, j, -L.ng)];
            const double d = prho[q] + prho[q - sz];
            const double w = pzm[q] * 2.0 / d;
            return w * 0.5 * d;
        };
        auto omega_old = [&](int kf) -> double {
            const long q = q0 + (long)kf * sz;
            if (kf == 0) return 0.;
            const double dwk = pw(kf) - szm[q];
            if (kf == nz) return dwk;
            return met::omega_from_w(i, j, kf, dwk, fdu, fdv, z, dxi, dyi);
        };
        // horizontal divergence of the new increments in cell k
        auto trhs_at = [&](int k, double& t0, double& t1) {
            const long q = q0 + (long)k * sz;
            double h_zeta_cc_xface_hi = 0.5 * dzi * (z(i + 1, j, k + 1) + z(i + 1, j + 1, k + 1) - z(i + 1, j, k) - z(i + 1, j + 1, k));
            double h_zeta_cc_xface_lo = 0.5 * dzi * (z(i, j, k + 1) + z(i, j + 1, k + 1) - z(i, j, k) - z(i, j + 1, k));
            double h_zeta_cc_yface_hi = 0.5 * dzi * (z(i, j + 1, k + 1) + z(i + 1, j + 1, k + 1) - z(i, j + 1, k) - z(i + 1, j + 1, k));
            double h_zeta_cc_yface_lo = 0.5 * dzi * (z(i, j, k + 1) + z(i + 1, j, k + 1) - z(i, j, k) - z(i + 1, j, k));
            double xflux_lo = nu[q] * h_zeta_cc_xface_lo / 1.0;
            double xflux_hi = nu[q + 1] * h_zeta_cc_xface_hi / 1.0;
            double yflux_lo = nv[q] * h_zeta_cc_yface_lo / 1.0;
            double yflux_hi = nv[q + sy] * h_zeta_cc_yface_hi / 1.0;
            double mfsq = 1.0 * 1.0;
            t0 = (xflux_hi - xflux_lo) * dxi * mfsq + (yflux_hi - yflux_lo) * dyi * mfsq;
            t1 = ((xflux_hi * (prim[q] + prim[q + 1]) - xflux_lo * (prim[q] + prim[q - 1])) * dxi * mfsq +
                  (yflux_hi * (prim[q] + prim[q + sy]) - yflux_lo * (prim[q] + prim[q - sy])) * dyi * mfsq) * 0.5;
        };
        // face 0 and cell 0
        double s_prev = (dtau * srz[q0]) * fB[q0];
        soln[q0] = s_prev;
        double om_km1 = 0.0, om_k = omega_old(1);
        om[q0] = om_km1;
        double t0_km1, t1_km1;
        trhs_at(0, t0_km1, t1_km1);
        trhs0[q0] = t0_km1;
        trhs1[q0] = t1_km1;
        double drho_km1 = cr0[q0] - sc0[q0], drt_km1 = cr1[q0] - sc1[q0];
        lagged1[q0] = drt_km1;
        double J_km1 = J[q0], s0_km1 = sr0[q0], s1_km1 = sr1[q0];
        double p_km2 = prim[q0 - sz], p_km1 = prim[q0];
        double q1_km1 = moist ? pq1[q0] : 0.0, q2_km1 = moist ? pq2[q0] : 0.0;
        // Each level reads everything it needs before its first store (the
        // stores may alias the inputs as far as the compiler knows, so a load
        // after a store waits for another round trip to memory).
        for (int k = 1; k <= nz - 1; ++k) {
            const long q = q0 + (long)k * sz;
            const double Jk = J[q], s0_k = sr0[q], s1_k = sr1[q], p_k = prim[q], p_kp1 = prim[q + sz];
            const double drho_k = cr0[q] - sc0[q], drt_k = cr1[q] - sc1[q];
            const double q1_k = moist ? pq1[q] : 0.0, q2_k = moist ? pq2[q] : 0.0;
            const double fP_k = fP[q], fQ_k = fQ[q], fA_k = fA[q], fB_k = fB[q], srz_k = srz[q];
            const double dw_k = pw(k) - szm[q];
            const double om_kp1 = omega_old(k + 1);
            double t0_k, t1_k;
            trhs_at(k, t0_k, t1_k);
            const double ofw = met::omega_from_w(i, j, k, 0., fnu, fnv, z, dxi, dyi);
            double detJ_on_kface = 0.5 * (Jk + J_km1);
            double coeff_P = fP_k;
            double coeff_Q = fQ_k;
            if (moist) {
                double qf = 0.5 * (q1_k + q1_km1 + q2_k + q2_km1);
                coeff_P /= (1.0 + qf);
                coeff_Q /= (1.0 + qf);
            }
            double theta_t_lo = 0.5 * (p_km2 + p_km1);
            double theta_t_mid = 0.5 * (p_km1 + p_k);
            double theta_t_hi = 0.5 * (p_k + p_kp1);
            double R0_tmp = (-halfg * drho_k + coeff_P * drt_k) * Jk
                          + (-halfg * drho_km1 + coeff_Q * drt_km1) * J_km1;
            double R1_tmp = -halfg * (s0_k * Jk + s0_km1 * J_km1)
                          + (coeff_P * s1_k * Jk + coeff_Q * s1_km1 * J_km1);
            R1_tmp += (halfg) * (beta_1 * dzi * (om_kp1 - om_km1) + t0_k + t0_km1);
            R1_tmp += -(coeff_P * (beta_1 * dzi * (om_kp1 * theta_t_hi - om_k * theta_t_mid) + t1_k) +
                        coeff_Q * (beta_1 * dzi * (om_k * theta_t_mid - om_km1 * theta_t_lo) + t1_km1));
            double rhs = detJ_on_kface * dw_k + dtau * (detJ_on_kface * srz_k + R0_tmp + dtau * beta_2 * R1_tmp);
            rhs += detJ_on_kface * ofw;
            s_prev = (rhs - fA_k * s_prev) * fB_k;
            om[q] = om_k;
            trhs0[q] = t0_k;
            trhs1[q] = t1_k;
            soln[q] = s_prev;
            lagged1[q] = drt_k;
            om_km1 = om_k; om_k = om_kp1;
            t0_km1 = t0_k; t1_km1 = t1_k;
            drho_km1 = drho_k; drt_km1 = drt_k;
            J_km1 = Jk; s0_km1 = s0_k; s1_km1 = s1_k;
            p_km2 = p_km1; p_km1 = p_k;
            q1_km1 = q1_k; q2_km1 = q2_k;
        }
        // top face: the last elimination step (no substitution there)
        const long qt = q0 + (long)nz * sz;
        double sol_hi = (dtau * srz[qt] - fA[qt] * s_prev) * fB[qt];
        cz[qt] = szm[qt];
        // one downward sweep: substitution, rho*w of face k, then the update
        // of cell k from its two faces
        double om_hi = om_k, p_hi = prim[qt];
        for (int k = nz - 1; k >= 0; --k) {
            const long q = q0 + k * sz;
            // loads first, as in the forward sweep
            const double soln_k = soln[q], fCB = fC[q] * fB[q], szm_k = szm[q], om_lo = om[q], azm_k = azm[q];
            const double Jq = J[q], pq = prim[q], p_lo = prim[q - sz], tr0 = trhs0[q], tr1 = trhs1[q];
            const double sr0_k = sr0[q], sr1_k = sr1[q], cc0_k = cr0[q], cc1_k = cr1[q];
            const double sol = soln_k - fCB * sol_hi;
            const double cz_k = (k >= 1) ? szm_k + met::w_from_omega(i, j, k, sol, fnu, fnv, z, dxi, dyi) : szm_k;
            double zflux_lo = beta_2 * sol + beta_1 * om_lo;
            double zflux_hi = beta_2 * sol_hi + beta_1 * om_hi;
            double fast_rhs_rho = -(tr0 + (zflux_hi - zflux_lo) * dzi) / Jq;
            double fast_rhs_rhotheta = -(tr1 + 0.5 * (zflux_hi * (pq + p_hi) -
                                                      zflux_lo * (pq + p_lo)) * dzi) / Jq;
            cz[q] = cz_k;
            azm[q] = azm_k + facinv * zflux_lo / (1.0 * 1.0);
            if (k == nz - 1) azm[q + sz] += facinv * zflux_hi / (1.0 * 1.0);
            cc0[q] = cc0_k + dtau * (sr0_k + fast_rhs_rho);
            cc1[q] = cc1_k + dtau * (sr1_k + fast_rhs_rhotheta);
            sol_hi = sol;
            om_hi = om_lo;
            p_hi = pq;
        }
    });
    }
    // algorithmic bytes per cell: the fields of the substep this kernel reads
    // (stage rho, rho*theta, rho*u, rho*v, rho*w; the previous rho*u, rho*v,
    // rho*w; the new rho*u, rho*v; the current rho, rho*theta; the slow RHS of
    // rho, rho*theta, rho*w; the averaged rho*w; z_nd, detJ; qv, qc when moist)
    // and writes (rho*w, averaged rho*w, rho, rho*theta), 8 B each
    kt_stop(P.timer, KT_FAST_COLUMN, s, (moist ? 24.0 : 22.0) * 8.0 * nx * ny * nz, "fast_rhs_T column");
}

}  // namespace erfx
