// erfx_fast.hip -- acoustic substep on a flat grid: make_fast_coeffs and
// erf_fast_rhs_N as gfx950 kernels.
//
// Launch structure per substep:
//   K1-2 x- and y-faces (one launch): Delta(rho theta) of the face's two cells
//       extrapolated forward, horizontal momentum update, written straight into
//       the current state (each lane reads prev and writes cur at its own
//       index, so the S_prev == S_data aliasing is safe)
//   K3-5 columns (tiles of columns whose lanes share a column's levels, or one
//       lane per column): horizontal divergence of the increments, tridiagonal
//       RHS, Thomas sweep, new rho*w, vertical fluxes, time-averaged rho*w, rho
//       and rho*theta update; the lagged Delta(rho theta), which K1-2 of this
//       substep has read, is replaced by the new one here, each cell by one lane
// The arithmetic of every point keeps the reference's operation order.
#include "erfx_common.h"
#include "erfx_internal.h"
#include <mutex>
#include <string>
#include <type_traits>

namespace erfx {

// make_fast_coeffs, flat branch (Source/TimeIntegration/ERF_make_fast_coeffs.cpp:158-200),
// GPU column recurrence (:214-242) and inversion (:287-290), fused into one
// column kernel.  fc comps: 0 A, 1 B (1/B on interior faces), 2 C, 3 P, 4 Q.
void make_fast_coeffs(const Params& P, double* fc, const erfx_state& stage, const double* prim,
                      const double* pi_stage, const double* r0, const double* pi0, double dtau, double beta_s,
                      hipStream_t s) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const long ne = L.ne, sz = L.sz;
    const double beta_2 = 0.5 * (1.0 + beta_s);
    const double c_v = P.cfg.c_p - R_d;
    const double dzi = P.dxInv[2];
    const double halfg = fabs(0.5 * (-P.gravity));
    const bool top_outflow = (P.cfg.bc[5] == ERFX_BC_OUTFLOW);
    const double* rt = stage.cons + ne;
    double* A = fc;
    double* B = fc + ne;
    double* Cc = fc + 2 * ne;
    double* Pc = fc + 3 * ne;
    double* Qc = fc + 4 * ne;
    const double D = dtau * dtau * beta_2 * beta_2 * dzi;
    const bool moist = P.moist;
    const double* pq1 = prim + PRIM_Q1 * ne;
    const double* pq2 = prim + PRIM_Q2 * ne;
    const double* J = P.terrain ? P.detJ : nullptr;
    // cell values of a level with theta of the level above, and the coefficients of
    // the face between `lo` and `hi`
    struct Lv { double r, pib, pis, rt_, pkp1, q1, q2; };
    struct Row { double a, b, c; };
    auto load = [=] __device__(long q, Lv& v) {
        v.r = r0[q]; v.pib = pi0[q]; v.pis = pi_stage[q]; v.rt_ = rt[q]; v.pkp1 = prim[q + sz];
        if (moist) { v.q1 = pq1[q]; v.q2 = pq2[q]; } else { v.q1 = 0.0; v.q2 = 0.0; }
    };
    // face q, theta at levels k-2 .. k
    auto face = [=] __device__(long q, const Lv& lo, const Lv& hi, double pr_km2, double pr_km1, double pr_k) {
        double rhobar_lo = lo.r, rhobar_hi = hi.r;
        double pibar_lo = lo.pib, pibar_hi = hi.pib;
        double pi_c = 0.5 * (lo.pis + hi.pis);
        double coeff_P, coeff_Q, detJ_on_kface = 1.0;
        if (J) {   // terrain (ERF_make_fast_coeffs.cpp:113-137)
            detJ_on_kface = 0.5 * (J[q] + J[q - sz]);
            double inv_detJ_on_kface = 1. / detJ_on_kface;
            coeff_P = -Gamma * R_d * dzi * inv_detJ_on_kface + halfg * R_d * rhobar_hi / (c_v * pibar_hi * hi.rt_);
            coeff_Q = Gamma * R_d * dzi * inv_detJ_on_kface + halfg * R_d * rhobar_lo / (c_v * pibar_lo * lo.rt_);
        } else {
            coeff_P = -Gamma * R_d * dzi + halfg * R_d * rhobar_hi / (c_v * pibar_hi * hi.rt_);
            coeff_Q = Gamma * R_d * dzi + halfg * R_d * rhobar_lo / (c_v * pibar_lo * lo.rt_);
        }
        coeff_P *= pi_c;
        coeff_Q *= pi_c;
        Row w;
        Pc[q] = coeff_P;
        Qc[q] = coeff_Q;
        if (moist) {   // ERF_make_fast_coeffs.cpp:183-188
            double qf = 0.5 * (hi.q1 + lo.q1 + hi.q2 + lo.q2);
            coeff_P /= (1.0 + qf);
            coeff_Q /= (1.0 + qf);
        }
        double theta_t_lo = 0.5 * (pr_km2 + pr_km1);
        double theta_t_mid = 0.5 * (pr_km1 + pr_k);
        double theta_t_hi = 0.5 * (pr_k + hi.pkp1);
        w.a = D * (halfg - coeff_Q * theta_t_lo);
        w.c = D * (-halfg + coeff_P * theta_t_hi);
        w.b = (J ? detJ_on_kface : 1.0) + D * (coeff_Q - coeff_P) * theta_t_mid;
        return w;
    };
    const double at = top_outflow ? -1.0 : 0.0;
    // Boxes of few columns: one lane per column and chunk of levels (launch_relay),
    // so a lane forms one to four rows instead of a whole column of them in
    // sequence; the recurrence, whose division per level is the serial part, runs
    // over LDS on one chunk's lanes and the inverses are taken in parallel again.
    // 64 x 64 x 64: 24.9 us one lane per column, 10.3 us; 161 x 97 x 63 moist: 39.8
    // us, 34.2 us.  Two tiles fit the LDS of a CU, so 512 of 32 columns fill the
    // chip once, and the line lies there, at 16,384 columns.  Tile | per-column form
    // at 64 levels, dry and moist: 127 x 127 21.0 | 27.7, 24.5 | 30.8 us; 128 x 128
    // 20.0 | 27.7, 23.8 | 30.8; 135 x 135 26.8 | 28.1, 30.6 | 30.8; 150 x 150
    // 28.3 | 28.3, 33.4 | 31.3; 181 x 181 dry 38.0 | 29.9.  At 16 and 40 levels, dry:
    // 127 x 127 7.0 | 9.3 and 13.1 | 18.7, 181 x 181 11.1 | 10.5 and 25.0 | 20.2.
    // Chunks of more than 4 levels were slower too (190 x 150 x 80: 86 us against 53
    // profiled).  The lanes of the per-column form fill the chip there and it reads
    // each level once (5.4 TB/s at 512 x 512 x 96).
    const long ncols = (long)nx * ny;
    auto tile = [=] __device__(int i, int j, bool valid, int col, int chunk, double* lds, auto cmc, auto tcc) {
        constexpr int CM = decltype(cmc)::value;
        constexpr int TC = decltype(tcc)::value;
        constexpr int R = relay_rows<CM, TC>() * TC;
        const int chl = tile_chunk(nz, 512 / TC);
        const int ka = chunk * chl;
        const int kb = (ka + chl < nz ? ka + chl : nz) - 1;
        const bool work = valid && ka <= kb;
        const long q0 = valid ? L.ix(i, j, 0) : 0;
        double* X = lds;            // a_k
        double* Y = lds + R;        // b_k, then the pivot
        double* Z = lds + 2 * R;    // c_k
        if (work) {
#pragma unroll
            for (int m = 0; m < CM; ++m) {
                const int k = ka + m;
                if (k > kb) break;
                const long q = q0 + (long)k * sz;
                if (k == 0) { A[q] = 0.0; B[q] = 1.0; Cc[q] = 0.0; continue; }
                Lv lo, hi;
                load(q - sz, lo);
                load(q, hi);
                const Row w = face(q, lo, hi, prim[q - 2 * sz], prim[q - sz], prim[q]);
                A[q] = w.a; Cc[q] = w.c;
                X[k * TC + col] = w.a; Y[k * TC + col] = w.b; Z[k * TC + col] = w.c;
            }
        }
        __syncthreads();
        if (chunk == 0 && valid) {
            double bet = 1.0, c_prev = 0.0;
            for (int k = 1; k <= nz - 1; ++k) {
                double gam = c_prev / bet;
                bet = Y[k * TC + col] - X[k * TC + col] * gam;
                Y[k * TC + col] = bet;
                c_prev = Z[k * TC + col];
            }
            const long qt = q0 + (long)nz * sz;     // the top face keeps B itself
            A[qt] = at; Cc[qt] = 0.0;
            double gam = c_prev / bet;
            B[qt] = 1.0 - at * gam;
        }
        __syncthreads();
        if (work) {
#pragma unroll
            for (int m = 0; m < CM; ++m) {
                const int k = ka + m;
                if (k > kb) break;
                if (k > 0) B[q0 + (long)k * sz] = 1.0 / Y[k * TC + col];   // interior faces store 1/B (:287-290)
            }
        }
    };
    if (!g_rec && nz <= 128 && (tile_columns(ncols) == 16 || (nz <= 64 && ncols <= 16384))) {
        auto launch = [&](auto cmc, auto tcc) {
            constexpr int CM = decltype(cmc)::value, TC = decltype(tcc)::value;
            launch_relay<CM, TC, 0, 0>(0, nx - 1, 0, ny - 1, s,
                [=] __device__(int i, int j, bool valid, int col, int chunk, double* lds) {
                    tile(i, j, valid, col, chunk, lds, cmc, tcc);
                });
        };
        using IC16 = std::integral_constant<int, 16>;
        using IC32 = std::integral_constant<int, 32>;
        using IC4 = std::integral_constant<int, 4>;
        if (tile_columns(ncols) == 16) launch(IC4{}, IC16{});
        else launch(IC4{}, IC32{});
        return;
    }
    launch_cols(0, nx - 1, 0, ny - 1, s, [=] __device__(int i, int j) {
        const long q0 = L.ix(i, j, 0);
        // bottom face, then the interior faces with the recurrence carried along
        A[q0] = 0.0; B[q0] = 1.0; Cc[q0] = 0.0;
        double bet = 1.0;
        double c_prev = 0.0;
        Lv lo;
        load(q0, lo);
        double pr_km2 = prim[q0 - sz], pr_km1 = prim[q0], pr_k = lo.pkp1;
        constexpr int RD = 4;
        Lv ring[RD];
#pragma unroll
        for (int d = 0; d < RD; ++d)
            if (1 + d <= nz - 1) load(q0 + (1 + d) * sz, ring[d]);
        for (int kb = 1; kb <= nz - 1; kb += RD) {
#pragma unroll
            for (int d = 0; d < RD; ++d) {
                const int k = kb + d;
                if (k > nz - 1) break;
                const long q = q0 + k * sz;
                const Lv v = ring[d];
                if (k + RD <= nz - 1) load(q + RD * sz, ring[d]);
                const Row w = face(q, lo, v, pr_km2, pr_km1, pr_k);
                A[q] = w.a;
                Cc[q] = w.c;
                double gam = c_prev / bet;
                bet = w.b - w.a * gam;
                c_prev = w.c;
                B[q] = 1.0 / bet;                        // interior faces store 1/B (:287-290)
                lo = v;
                pr_km2 = pr_km1; pr_km1 = pr_k; pr_k = v.pkp1;
            }
        }
        // top face keeps B itself
        const long qt = q0 + nz * sz;
        A[qt] = at; Cc[qt] = 0.0;
        double gam = c_prev / bet;
        B[qt] = 1.0 - at * gam;
    });
}

// no_substep_fun (Source/TimeIntegration/ERF_TI_no_substep_fun.H:88-126),
// fixed or no terrain: with substepping_type None each RK stage advances the
// fast variables with the slow right-hand side alone -- rho and rho*theta on
// the valid cells, each momentum on its nodal box -- in one launch.
void no_substep(const Params& P, const erfx_state& ssum, const erfx_state& sold, const erfx_state& fslow,
                double slow_dt, hipStream_t s) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const long ne = L.ne;
    launch_box(Box(0, 0, 0, nx, ny, nz), s, [=] __device__(int i, int j, int k) {
        const long q = L.ix(i, j, k);
        if (i <= nx - 1 && j <= ny - 1 && k <= nz - 1) {
            ssum.cons[q] = sold.cons[q] + slow_dt * (fslow.cons[q]);
            ssum.cons[q + ne] = sold.cons[q + ne] + slow_dt * (fslow.cons[q + ne]);
        }
        if (j <= ny - 1 && k <= nz - 1) ssum.xmom[q] = sold.xmom[q] + slow_dt * fslow.xmom[q];
        if (i <= nx - 1 && k <= nz - 1) ssum.ymom[q] = sold.ymom[q] + slow_dt * fslow.ymom[q];
        if (i <= nx - 1 && j <= ny - 1) ssum.zmom[q] = sold.zmom[q] + slow_dt * fslow.zmom[q];
    });
}

void fast_rhs_N(const Params& P, const FastWork& W, int step, int nrk, const erfx_state& slow_rhs,
                const erfx_state& prev, const erfx_state& stage, const double* prim, const double* pi_stage,
                const double* fc, const erfx_state& data, const erfx_state& scratch, double dtau,
                double beta_s, double facinv, hipStream_t s, const FastChain& ch) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const long ne = L.ne, sy = L.sy, sz = L.sz;
    const double beta_1 = 0.5 * (1.0 - beta_s);
    const double beta_2 = 0.5 * (1.0 + beta_s);
    const double beta_d = 0.1;
    const double dxi = P.dxInv[0], dyi = P.dxInv[1], dzi = P.dxInv[2];
    const bool implicit = P.cfg.implicit_substepping != 0;
    double* drw = W.drw;
    double* tr0 = W.trhs;
    double* tr1 = W.trhs + ne;
    double* soln = W.soln;
    const double* prt = prev.cons + ne;
    const double* srt = stage.cons + ne;
    double* lagged = scratch.cons + ne;

    // K1 + K2 (:115-257), one lane per x- and y-face.  Delta(rho theta) of a
    // cell, extrapolated forward with the lagged increment (:115-152), is formed
    // by each of the four faces that read it: 3 fields of neighbour reads, which
    // the four rows of a work-group share, in place of a field written and read
    // again by a launch of its own.  HBM bound at 13 fields read and 4 written
    // (256 x 256 x 128: 283 us as two launches, 250 us as one, 4.6 TB/s).  With
    // rt_prev the previous substep's apply_bcs is folded in: its momentum ->
    // velocity -> momentum round trip (ERF_MomentumToVelocity.cpp,
    // ERF_VelocityToMomentum.cpp) is applied to prev as it is read, and ghost cells
    // are read at their periodic images.
    const bool first = (nrk == 0 && step == 0);
    const bool rt = ch.rt_prev && step > 0;
    const bool use_lag = step > 0;
    const bool seed = ch.seed;
    const double* prho = prev.cons;
    const double gr = -Gamma * R_d;
    const bool moist = P.moist;
    const double* pq1 = prim + PRIM_Q1 * ne;
    const double* pq2 = prim + PRIM_Q2 * ne;
    // Every load is issued before the first store: the stores may alias the
    // inputs as far as the compiler knows, so loads of the y-face after the
    // stores of the x-face would wait for a second round trip to memory.  (The
    // loads of a face outside its box stay inside the layout; only the stores
    // are guarded.)
    const double *pxm = prev.xmom, *pym = prev.ymom, *sxm = stage.xmom, *sym = stage.ymom;
    const double *slx = slow_rhs.xmom, *sly = slow_rhs.ymom;
    double *axm = scratch.xmom, *aym = scratch.ymom, *dxm = data.xmom, *dym = data.ymom;
    launch_box(Box(0, 0, 0, nx, ny, nz - 1), s, [=] __device__(int i, int j, int k) {
        const long q = L.ix(i, j, k);
        // the faces' cells: c (i, j), x (i-1, j), y (i, j-1); images in the chain
        const long qc = rt ? q - (i == nx ? nx : 0) - (j == ny ? (long)ny * sy : 0) : q;
        const long qx = (rt && i == 0) ? q + nx - 1 : q - 1;
        const long qy = (rt && j == 0) ? q + (long)(ny - 1) * sy : q - sy;
        double pmx = pxm[q], pmy = pym[q];
        const double sx = sxm[q], sy_ = sym[q], lx = slx[q], ly = sly[q];
        const double ax = seed ? sx : axm[q], ay = seed ? sy_ : aym[q];
        double rc = 0.0, rx = 0.0, ry = 0.0;
        if (rt) { rc = prho[qc]; rx = prho[qx]; ry = prho[qy]; }
        double frx = 0.0, fry = 0.0;
        if (!first) {
            double ec = prt[qc] - srt[qc], ex = prt[qx] - srt[qx], ey = prt[qy] - srt[qy];
            const double pc = pi_stage[q], px = pi_stage[q - 1], py = pi_stage[q - sy];
            if (use_lag) {
                const double lc = lagged[qc], lgx = lagged[qx], lgy = lagged[qy];
                ec = ec + beta_d * (ec - lc);
                ex = ex + beta_d * (ex - lgx);
                ey = ey + beta_d * (ey - lgy);
            }
            double gpx = (ec - ex) * dxi, gpy = (ec - ey) * dyi;
            if (moist) {   // :215-219, :238-242
                gpx /= (1.0 + face_q(pq1, pq2, q, q - 1));
                gpy /= (1.0 + face_q(pq1, pq2, q, q - sy));
            }
            frx = gr * (0.5 * (px + pc)) * gpx;
            fry = gr * (0.5 * (py + pc)) * gpy;
        }
        if (rt) {
            const double d = rc + rx, e = rc + ry;
            const double u = pmx * 2.0 / d, v = pmy * 2.0 / e;
            pmx = u * 0.5 * d;
            pmy = v * 0.5 * e;
        }
        const double nu = first ? pmx - sx + dtau * lx : pmx - sx + dtau * frx + dtau * lx;
        const double nv = first ? pmy - sy_ + dtau * ly : pmy - sy_ + dtau * fry + dtau * ly;
        if (j <= ny - 1) {
            axm[q] = ax + facinv * nu;
            dxm[q] = sx + nu;
        }
        if (i <= nx - 1) {
            aym[q] = ay + facinv * nv;
            dym[q] = sy_ + nv;
        }
    });
    // the lagged increment's ghost layer, which the next substep reads unless it
    // reads the periodic images (written with the column launch below)
    const LaggedShell shell{L, prt, srt, lagged, nullptr, nullptr};

    // K3 + K4 + K5 fused per column (:328-357, :374-453, :518-536, :566-592).
    // One lane per (i, j) column.  Forward sweep: horizontal divergence of the
    // increments in cell k, tridiagonal RHS on face k, elimination.  Backward
    // sweep: substitution, new rho*w, vertical fluxes and the rho / rho*theta
    // update of cell k.  The loads of the next level are issued before the
    // arithmetic of the current one, so each lane keeps two levels of loads in
    // flight.  Every expression keeps the reference's operation order.
    const double halfg = fabs(0.5 * (-P.gravity));
    const double* A = fc;
    const double* iB = fc + ne;
    const double* Cc = fc + 2 * ne;
    const double* Pc = fc + 3 * ne;
    const double* Qc = fc + 4 * ne;
    const double* sr0 = slow_rhs.cons;
    const double* sr1 = slow_rhs.cons + ne;
    const double* pr0 = prev.cons;
    const double* st0 = stage.cons;
    double* cc0 = data.cons;
    double* cc1 = data.cons + ne;
    const double ch_w_lo = ch.w_lo, ch_w_hi = ch.w_hi;
    auto column = [=] __device__(int i, int j, auto depth) {
        const long q0 = L.ix(i, j, 0);
        // per-level loads of the forward sweep (face k and cell k)
        struct Fw {
            double P, Q, A, iB, ws, pkp1, pz, szz, pr, rkp1, st, prt_, srt_, s0, s1;
            double dxl, dxh, sxl, sxh, dyl, dyh, syl, syh, pc, pxm, pxp, pym, pyp;
            double q1, q2;   // qv, qc of cell k (moist only)
        };
        auto fload = [&](long q, Fw& v) {
            v.P = Pc[q]; v.Q = Qc[q]; v.A = A[q]; v.iB = iB[q]; v.ws = slow_rhs.zmom[q];
            v.pkp1 = prim[q + sz]; v.pz = prev.zmom[q + sz]; v.szz = stage.zmom[q + sz];
            v.pr = pr0[q]; v.rkp1 = rt ? pr0[q + sz] : 0.0;
            v.st = st0[q]; v.prt_ = prt[q]; v.srt_ = srt[q]; v.s0 = sr0[q]; v.s1 = sr1[q];
            v.dxl = data.xmom[q]; v.dxh = data.xmom[q + 1]; v.sxl = stage.xmom[q]; v.sxh = stage.xmom[q + 1];
            v.dyl = data.ymom[q]; v.dyh = data.ymom[q + sy]; v.syl = stage.ymom[q]; v.syh = stage.ymom[q + sy];
            v.pc = prim[q]; v.pxm = prim[q - 1]; v.pxp = prim[q + 1]; v.pym = prim[q - sy]; v.pyp = prim[q + sy];
            if (moist) { v.q1 = pq1[q]; v.q2 = pq2[q]; } else { v.q1 = 0.0; v.q2 = 0.0; }
        };
        // horizontal flux divergence of the increments (K3)
        auto hdiv = [&](const Fw& v, double& t0, double& t1) {
            double xflux_lo = v.dxl - v.sxl;
            double xflux_hi = v.dxh - v.sxh;
            double yflux_lo = v.dyl - v.syl;
            double yflux_hi = v.dyh - v.syh;
            double pc = v.pc;
            t0 = (xflux_hi - xflux_lo) * dxi + (yflux_hi - yflux_lo) * dyi;
            t1 = ((xflux_hi * (pc + v.pxp) - xflux_lo * (pc + v.pxm)) * dxi +
                  (yflux_hi * (pc + v.pyp) - yflux_lo * (pc + v.pym)) * dyi) * 0.5;
        };

        // prev rho*w at the face above a level's cell, after the round trip when
        // rt (interior: rho of the two cells; top: the Dirichlet w with the
        // foextrap ghost rho)
        auto w_above = [&](const Fw& v, int kf) {
            if (!rt) return v.pz;
            if (kf >= nz) return ch_w_hi * 0.5 * (v.pr + v.pr);
            double d = v.rkp1 + v.pr;
            double w = v.pz * 2.0 / d;
            return w * 0.5 * d;
        };
        Fw cur;
        fload(q0, cur);
        // face 0 (bottom row, :423-432) and cell 0
        double pz0 = rt ? ch_w_lo * 0.5 * (cur.pr + cur.pr) : prev.zmom[q0];
        double Om_km1 = pz0 - stage.zmom[q0];
        drw[q0] = Om_km1;
        double rhs0 = Om_km1 + dtau * cur.ws;
        double sol_prev = implicit ? rhs0 * cur.iB : rhs0;
        soln[q0] = sol_prev;
        double t0_km1, t1_km1;
        hdiv(cur, t0_km1, t1_km1);
        tr0[q0] = t0_km1;
        tr1[q0] = t1_km1;
        double drho_km1 = cur.pr - cur.st;
        double drt_km1 = cur.prt_ - cur.srt_;
        lagged[q0] = drt_km1;
        double s0_km1 = cur.s0, s1_km1 = cur.s1;
        double p_km2 = prim[q0 - sz], p_km1 = cur.pc, p_k = cur.pkp1;
        double q1_km1 = cur.q1, q2_km1 = cur.q2;
        double Om_k = w_above(cur, 1) - cur.szz;
        // ring of FD levels of loads in flight (slots indexed statically after unrolling)
        constexpr int FD = decltype(depth)::value;
        Fw ring[FD];
#pragma unroll
        for (int d = 0; d < FD; ++d)
            if (1 + d <= nz - 1) fload(q0 + (1 + d) * sz, ring[d]);
        for (int kb = 1; kb <= nz - 1; kb += FD) {
#pragma unroll
            for (int d = 0; d < FD; ++d) {
                const int k = kb + d;
                if (k > nz - 1) break;
                const long q = q0 + k * sz;
                Fw c = ring[d];
                if (k + FD <= nz - 1) fload(q + FD * sz, ring[d]);
                double t0_k, t1_k;
                hdiv(c, t0_k, t1_k);
                tr0[q] = t0_k;
                tr1[q] = t1_k;
                drw[q] = Om_k;
                double Om_kp1 = w_above(c, k + 1) - c.szz;
                double drho_k = c.pr - c.st;
                double drt_k = c.prt_ - c.srt_;
                lagged[q] = drt_k;
                double coeff_P = c.P, coeff_Q = c.Q;
                if (moist) {   // :379-384
                    double qf = 0.5 * (c.q1 + q1_km1 + c.q2 + q2_km1);
                    coeff_P /= (1.0 + qf);
                    coeff_Q /= (1.0 + qf);
                }
                double theta_t_lo = 0.5 * (p_km2 + p_km1);
                double theta_t_mid = 0.5 * (p_km1 + p_k);
                double theta_t_hi = 0.5 * (p_k + c.pkp1);
                double R0_tmp = coeff_P * drt_k + coeff_Q * drt_km1 - halfg * (drho_k + drho_km1);
                double R1_tmp = halfg * (-c.s0 - s0_km1 + t0_k + t0_km1) +
                                (coeff_P * (c.s1 - t1_k) + coeff_Q * (s1_km1 - t1_km1));
                R1_tmp += beta_1 * dzi * ((Om_kp1 - Om_km1) * halfg
                                          - (Om_kp1 * theta_t_hi - Om_k * theta_t_mid) * coeff_P
                                          - (Om_k * theta_t_mid - Om_km1 * theta_t_lo) * coeff_Q);
                double RHS = Om_k + dtau * (c.ws + R0_tmp + dtau * beta_2 * R1_tmp);
                double sol = implicit ? (RHS - c.A * sol_prev) * c.iB : RHS;
                soln[q] = sol;
                sol_prev = sol;
                p_km2 = p_km1; p_km1 = p_k; p_k = c.pkp1;
                q1_km1 = c.q1; q2_km1 = c.q2;
                Om_km1 = Om_k; Om_k = Om_kp1;
                drho_km1 = drho_k; drt_km1 = drt_k;
                s0_km1 = c.s0; s1_km1 = c.s1;
                t0_km1 = t0_k; t1_km1 = t1_k;
            }
        }
        // top face (:423-432): Om_k now holds face nz
        const long qt = q0 + nz * sz;
        double rhs_t = Om_k + dtau * slow_rhs.zmom[qt];
        double sol_t = implicit ? (rhs_t - A[qt] * sol_prev) * iB[qt] : rhs_t;
        data.zmom[qt] = stage.zmom[qt] + sol_t;
        drw[qt] = Om_k;

        // backward sweep with the cell update (K5)
        struct Bw { double so, C, iB, dw, szz, t0, t1, pc, pm, s0, s1, c0, c1; };
        auto bload = [&](long q, Bw& v) {
            v.so = soln[q]; v.C = Cc[q]; v.iB = iB[q]; v.dw = drw[q]; v.szz = stage.zmom[q];
            v.t0 = tr0[q]; v.t1 = tr1[q]; v.pc = prim[q]; v.pm = prim[q - sz]; v.s0 = sr0[q]; v.s1 = sr1[q];
            v.c0 = step == 0 ? prev.cons[q] : cc0[q];
            v.c1 = step == 0 ? prev.cons[q + ne] : cc1[q];
        };
        double sol_next = sol_t;
        double drw_next = Om_k;
        double p_next = prim[qt];
        constexpr int BD = decltype(depth)::value;
        Bw bring[BD];
#pragma unroll
        for (int d = 0; d < BD; ++d)
            if (nz - 1 - d >= 0) bload(q0 + (nz - 1 - d) * sz, bring[d]);
        for (int kb = nz - 1; kb >= 0; kb -= BD) {
#pragma unroll
            for (int d = 0; d < BD; ++d) {
                const int k = kb - d;
                if (k < 0) break;
                const long q = q0 + k * sz;
                Bw bc = bring[d];
                if (k - BD >= 0) bload(q - BD * sz, bring[d]);
                double sol = implicit ? bc.so - (bc.C * bc.iB) * sol_next : bc.so;
                double drw_k = bc.dw;
                data.zmom[q] = bc.szz + sol;
                double zflux_lo = beta_2 * sol + beta_1 * drw_k;
                double zflux_hi = beta_2 * sol_next + beta_1 * drw_next;
                scratch.zmom[q] = (seed ? bc.szz : scratch.zmom[q]) + facinv * zflux_lo / (1.0 * 1.0);
                if (k == nz - 1)
                    scratch.zmom[q + sz] = (seed ? stage.zmom : scratch.zmom)[q + sz] + facinv * zflux_hi / (1.0 * 1.0);
                double pcq = bc.pc;
                double t0 = bc.t0 + dzi * (zflux_hi - zflux_lo);
                double t1 = bc.t1 + 0.5 * dzi * (zflux_hi * (pcq + p_next) - zflux_lo * (pcq + bc.pm));
                double r_new = bc.c0 + dtau * (bc.s0 - t0);
                double rt_new = bc.c1 + dtau * (bc.s1 - t1);
                cc0[q] = r_new;
                cc1[q] = rt_new;
                sol_next = sol;
                drw_next = drw_k;
                p_next = pcq;
            }
        }
    };
    // The same column work as a tile of TC (64, 32 or 16) columns per work-group of 8
    // waves, the levels of a column split into 512 / TC chunks of at most CM, one
    // lane per chunk and column (launch_relay), for boxes of up to 128 levels:
    //  1. each lane reads its chunk's levels once and forms, as the column kernel
    //     does, the horizontal divergences of cell k, Omega of face k + 1 and the
    //     tridiagonal row of face k; the row of a chunk's first face, which needs
    //     the cell below, is finished after the chunks have passed each other
    //     their top cell in LDS;
    //  2. the elimination is relayed up the chunks and the substitution down them:
    //     each lane runs its own levels from registers and hands one value to the
    //     next chunk (chunks of up to 4 levels stage their rows in LDS instead,
    //     where the first chunk's lanes sweep them);
    //  3. each lane updates rho*w, the averaged rho*w, rho and rho*theta of its
    //     cells from what it still holds.
    // Every value is computed by the same expression as in the column kernel, so
    // the results are bit-identical.  The kernel is HBM bound.  Everything a level
    // needs later stays in the lane (registers, and four arrays in its own LDS
    // slots), so each field is read once: the form this replaced (64 columns, 12
    // levels per wave, rows staged in LDS and swept by one wave, operands read
    // again for the update) moved 36 fields on 256 x 256 x 80 and took 331 us where
    // this takes 280; the per-lane form moved 41 on 256 x 256 x 128 and took 503 us
    // against 394.  With the coefficients of make_fast_coeffs itself
    // (own_coeffs) a_k and c_k are formed again from P, Q and theta, by the
    // expressions that made them, instead of being read.
    const bool own = ch.own_coeffs;
    const bool separate = step > 0 && prev.cons != data.cons;   // a hook's separate buffers
    const double Dc = dtau * dtau * beta_2 * beta_2 * dzi;
    auto relay = [=] __device__(int i, int j, bool valid, int col, int chunk, double* lds, auto cmc, auto tcc) {
        constexpr int CM = decltype(cmc)::value;
        constexpr int TC = decltype(tcc)::value;   // columns per tile
        constexpr int NCH = 512 / TC;              // chunks of levels
        const int tid = (int)threadIdx.x;
        // read here once: in a batch captures are loads, and the wait for them in the
        // middle of the sweeps took 2% of the kernel
        const int mode = __builtin_amdgcn_readfirstlane((implicit ? 1 : 0) | (separate ? 2 : 0));
        const int chl = tile_chunk(nz, NCH);
        const int ka = chunk * chl;
        const int kb = (ka + chl < nz ? ka + chl : nz) - 1;
        const bool has = ka <= kb;
        const bool work = valid && has;
        const bool top = has && kb == nz - 1;
        const long q0 = valid ? L.ix(i, j, 0) : 0;
        // the lane's own LDS slots (array a, level m) and the exchange rows
        auto slot = [&](int a, int m) -> double& { return lds[(a * CM + m) * 512 + tid]; };
        auto below = [&](int a) -> double { return lds[(a * CM + chl - 1) * 512 + tid - TC]; };
        double* xch = lds + 4 * CM * 512;
        double* carry = xch + 5 * 512;
        enum { T0 = 0, T1, S0, S1 };
        double rhs[CM], av[CM], bv[CM], cv[CM], om[CM + 1], prr[CM], ptr_[CM], pp[CM], sz_[CM];
        double r_top = 0.0, a_top = 0.0, b_top = 0.0, s_top = 0.0;
        // of the chunk's first cell, until its face's row is finished
        double f_cP = 0.0, f_cQ = 0.0, f_ws = 0.0, f_drho = 0.0, f_drt = 0.0, f_q1 = 0.0, f_q2 = 0.0;
        double f_pm2 = 0.0, f_pm1 = 0.0, f_pp1 = 0.0;
        struct Cell { double drho, drt, s0, s1, t0, t1, q1, q2, om; };   // om: of the cell's lower face
        // row k of the system: cell k is `c`, the cell below `b`; om_p: Omega of face k + 1
        auto row = [&](double cP, double cQ, double ws, const Cell& c, const Cell& b, double om_p, double p_km2,
                       double p_km1, double p_k, double p_kp1, double& a, double& cc) -> double {
            if (moist) {   // :379-384
                double qf = 0.5 * (c.q1 + b.q1 + c.q2 + b.q2);
                cP /= (1.0 + qf);
                cQ /= (1.0 + qf);
            }
            double theta_t_lo = 0.5 * (p_km2 + p_km1);
            double theta_t_mid = 0.5 * (p_km1 + p_k);
            double theta_t_hi = 0.5 * (p_k + p_kp1);
            double R0_tmp = cP * c.drt + cQ * b.drt - halfg * (c.drho + b.drho);
            double R1_tmp = halfg * (-c.s0 - b.s0 + c.t0 + b.t0) +
                            (cP * (c.s1 - c.t1) + cQ * (b.s1 - b.t1));
            R1_tmp += beta_1 * dzi * ((om_p - b.om) * halfg
                                      - (om_p * theta_t_hi - c.om * theta_t_mid) * cP
                                      - (c.om * theta_t_mid - b.om * theta_t_lo) * cQ);
            if (own) {
                a = Dc * (halfg - cQ * theta_t_lo);
                cc = Dc * (-halfg + cP * theta_t_hi);
            }
            return c.om + dtau * (ws + R0_tmp + dtau * beta_2 * R1_tmp);
        };
        // ---- phase 1: one reading of the chunk's levels ----
        if (work) {
            const long qa = q0 + (long)ka * sz;
            double p_m2 = ka > 1 ? prim[qa - 2 * sz] : prim[q0 - sz], p_m1 = prim[qa - sz], p_k = prim[qa];
            double pr_k = pr0[qa];
            double sz_k = stage.zmom[qa];
            double om_k;
            {
                double pz = prev.zmom[qa];
                if (rt) {
                    if (ka == 0) {
                        pz = ch_w_lo * 0.5 * (pr_k + pr_k);
                    } else {
                        double d = pr_k + pr0[qa - sz];
                        double w = pz * 2.0 / d;
                        pz = w * 0.5 * d;
                    }
                }
                om_k = pz - sz_k;
            }
            Cell b{};
#pragma unroll
            for (int m = 0; m < CM; ++m) {
                const int k = ka + m;
                if (k > kb) break;
                const long q = q0 + (long)k * sz;
                const double ws = slow_rhs.zmom[q], cP = Pc[q], cQ = Qc[q];
                bv[m] = iB[q];
                if (!own) { av[m] = A[q]; cv[m] = Cc[q]; }
                const double p_p = prim[q + sz], pr_p = pr0[q + sz], sz_p = stage.zmom[q + sz];
                double pz = prev.zmom[q + sz];
                const double st = st0[q], pt = prt[q], srt_ = srt[q];
                Cell c;
                c.s0 = sr0[q]; c.s1 = sr1[q];
                const double dxl = data.xmom[q], dxh = data.xmom[q + 1], sxl = stage.xmom[q], sxh = stage.xmom[q + 1];
                const double dyl = data.ymom[q], dyh = data.ymom[q + sy], syl = stage.ymom[q], syh = stage.ymom[q + sy];
                const double pxm = prim[q - 1], pxp = prim[q + 1], pym = prim[q - sy], pyp = prim[q + sy];
                c.q1 = 0.0; c.q2 = 0.0;
                if (moist) { c.q1 = pq1[q]; c.q2 = pq2[q]; }
                // horizontal flux divergence of the increments (K3)
                double xflux_lo = dxl - sxl;
                double xflux_hi = dxh - sxh;
                double yflux_lo = dyl - syl;
                double yflux_hi = dyh - syh;
                c.t0 = (xflux_hi - xflux_lo) * dxi + (yflux_hi - yflux_lo) * dyi;
                c.t1 = ((xflux_hi * (p_k + pxp) - xflux_lo * (p_k + pxm)) * dxi +
                        (yflux_hi * (p_k + pyp) - yflux_lo * (p_k + pym)) * dyi) * 0.5;
                // Omega of the face above
                if (rt) {
                    if (k == nz - 1) {
                        pz = ch_w_hi * 0.5 * (pr_k + pr_k);
                    } else {
                        double d = pr_p + pr_k;
                        double w = pz * 2.0 / d;
                        pz = w * 0.5 * d;
                    }
                }
                const double om_p = pz - sz_p;
                c.om = om_k;
                c.drho = pr_k - st;
                c.drt = pt - srt_;
                lagged[q] = c.drt;
                if (m > 0) {
                    rhs[m] = row(cP, cQ, ws, c, b, om_p, p_m2, p_m1, p_k, p_p, av[m], cv[m]);
                } else if (k == 0) {   // face 0: the bottom row (:423-432)
                    rhs[m] = om_k + dtau * ws;
                    if (own) { av[m] = 0.0; cv[m] = 0.0; }
                } else {
                    f_cP = cP; f_cQ = cQ; f_ws = ws; f_drho = c.drho; f_drt = c.drt; f_q1 = c.q1; f_q2 = c.q2;
                    f_pm2 = p_m2; f_pm1 = p_m1; f_pp1 = p_p;
                }
                slot(T0, m) = c.t0; slot(T1, m) = c.t1; slot(S0, m) = c.s0; slot(S1, m) = c.s1;
                om[m] = om_k; om[m + 1] = om_p;
                prr[m] = pr_k; ptr_[m] = pt; pp[m] = p_k; sz_[m] = sz_k;
                tile_level_fence();
                b = c;
                p_m2 = p_m1; p_m1 = p_k; p_k = p_p;
                pr_k = pr_p; sz_k = sz_p; om_k = om_p;
            }
            // the top cell, for the chunk above
            xch[tid] = b.drho; xch[512 + tid] = b.drt; xch[2 * 512 + tid] = b.om;
            if (moist) { xch[3 * 512 + tid] = b.q1; xch[4 * 512 + tid] = b.q2; }
            if (top) {                         // the top face's row (:423-432)
                const long qt = q0 + (long)nz * sz;
                r_top = om_k + dtau * slow_rhs.zmom[qt];
                a_top = A[qt];
                b_top = iB[qt];
            }
        }
        __syncthreads();
        if (work && ka > 0) {
            Cell c, b;
            b.drho = xch[tid - TC]; b.drt = xch[512 + tid - TC]; b.om = xch[2 * 512 + tid - TC];
            b.q1 = 0.0; b.q2 = 0.0;
            if (moist) { b.q1 = xch[3 * 512 + tid - TC]; b.q2 = xch[4 * 512 + tid - TC]; }
            b.t0 = below(T0); b.t1 = below(T1); b.s0 = below(S0); b.s1 = below(S1);
            c.drho = f_drho; c.drt = f_drt; c.q1 = f_q1; c.q2 = f_q2; c.om = om[0];
            c.t0 = slot(T0, 0); c.t1 = slot(T1, 0); c.s0 = slot(S0, 0); c.s1 = slot(S1, 0);
            rhs[0] = row(f_cP, f_cQ, f_ws, c, b, om[1], f_pm2, f_pm1, pp[0], f_pp1, av[0], cv[0]);
        }
        // what phase 3 reads for the first time, in flight during the sweeps where
        // the registers allow it: the averaged rho*w, and theta above and below
        double az[CM], p_top = 0.0, p_bot = 0.0;
        auto load3 = [&]() {
            p_top = prim[q0 + (long)(kb + 1) * sz];
            p_bot = prim[q0 + (long)(ka - 1) * sz];
#pragma unroll
            for (int m = 0; m < CM; ++m)
                if (ka + m <= kb) az[m] = seed ? sz_[m] : scratch.zmom[q0 + (long)(ka + m) * sz];
            if (mode & 2) {    // the cells to update are not the ones read so far
#pragma unroll
                for (int m = 0; m < CM; ++m)
                    if (ka + m <= kb) {
                        prr[m] = cc0[q0 + (long)(ka + m) * sz];
                        ptr_[m] = cc1[q0 + (long)(ka + m) * sz];
                    }
            }
        };
        if (CM <= 6 && work) load3();
        // ---- phase 2: the sweeps ----
        double x_hi = 0.0;       // the solution on the chunk's upper face
        relay_solve<CM, TC>(carry, xch, (mode & 1) != 0, nz, chl, col, valid, rhs, av, bv, cv, r_top, a_top, b_top, s_top, x_hi);
        // ---- phase 3: the chunk's cells ----
        if (work) {
            if (CM > 6) load3();
            if (top) {
                const long qt = q0 + (long)nz * sz;
                data.zmom[qt] = stage.zmom[qt] + s_top;
            }
#pragma unroll
            for (int m = 0; m < CM; ++m) {
                const int k = ka + m;
                if (k > kb) break;
                const long q = q0 + (long)k * sz;
                const bool last = k == kb;
                const double sol = rhs[m], sol_next = last ? x_hi : rhs[m + 1 < CM ? m + 1 : m];
                const double pcq = pp[m], p_next = last ? p_top : pp[m + 1 < CM ? m + 1 : m];
                const double pm = m == 0 ? p_bot : pp[m > 0 ? m - 1 : 0];
                double zflux_lo = beta_2 * sol + beta_1 * om[m];
                double zflux_hi = beta_2 * sol_next + beta_1 * om[m + 1];
                double t0 = slot(T0, m) + dzi * (zflux_hi - zflux_lo);
                double t1 = slot(T1, m) + 0.5 * dzi * (zflux_hi * (pcq + p_next) - zflux_lo * (pcq + pm));
                data.zmom[q] = sz_[m] + sol;
                scratch.zmom[q] = az[m] + facinv * zflux_lo / (1.0 * 1.0);
                if (k == nz - 1)
                    scratch.zmom[q + sz] = (seed ? stage.zmom : scratch.zmom)[q + sz] + facinv * zflux_hi / (1.0 * 1.0);
                cc0[q] = prr[m] + dtau * (slot(S0, m) - t0);
                cc1[q] = ptr_[m] + dtau * (slot(S1, m) - t1);
            }
        }
    };
    // the variant: the sim's choice, or the next one to time while tuning
    int var = P.col_variant;
    int tag = -1;
    if (P.tuner && P.tuner->chosen < 0 && P.tuner->next < COL_NV * ColTuner::SAMPLES) {
        tag = P.tuner->next++;
        var = tag % COL_NV;
        (void)hipEventRecord(P.tuner->ev[2 * tag], s);
    }
    // The tile form takes up to 128 levels; a recorded (batched) launch up to 96,
    // always in 32-column tiles of 6 levels per chunk, so every member of a batch
    // records the same kernel.  Separate buffers and the explicit substep included:
    // 64 x 64 x 64 in separate buffers 27.6 us a substep, one lane per column 91.9
    // us; 190 x 150 x 80 199 and 248.
    if (var == COL_TILE && nz > (g_rec ? 96 : 128)) var = COL_FALLBACK;
    kt_start(P.timer, KT_FAST_COLUMN, s);
    if (var == COL_TILE) {
        if (!ch.active && g_rec) lagged_shell(shell, s);
        auto launch = [&](auto cmc, auto tcc) {
            launch_relay<decltype(cmc)::value, decltype(tcc)::value, 4, 5>(0, nx - 1, 0, ny - 1, s,
                [=] __device__(int i, int j, bool valid, int col, int chunk, double* lds) {
                    relay(i, j, valid, col, chunk, lds, cmc, tcc);
                }, ch.active ? 0u : shell.lanes(), shell);
        };
        using IC16 = std::integral_constant<int, 16>;
        using IC32 = std::integral_constant<int, 32>;
        using IC4 = std::integral_constant<int, 4>;
        using IC6 = std::integral_constant<int, 6>;
        using IC8 = std::integral_constant<int, 8>;
        // Up to 32 levels on many columns, 64 columns per tile: 8 chunks instead of
        // 16, of which short columns leave most idle, and up to 8 levels with the LDS
        // of one level a chunk, which lets two work-groups run on a CU.  In 64-column
        // tiles, in 32-column tiles: 512 x 512 x 4 86, 178 us; x 9 199, 274; x 16
        // 333, 388; x 32 630, 682; 96 x 96 x 20 18.8, 23.8 (more levels have no room
        // for their rows; fewer columns give fewer tiles than CUs: 64 x 64 x 32 in
        // 16-column tiles 17.3, one lane per column 51).
        using IC64 = std::integral_constant<int, 64>;
        if (!g_rec && tile_columns((long)nx * ny) == 16) launch(IC4{}, IC16{});   // 32 chunks: at most 4 levels each
        else if (!g_rec && tile_chunk(nz, 8) <= 1) launch(std::integral_constant<int, 1>{}, IC64{});
        else if (!g_rec && tile_chunk(nz, 8) <= 2) launch(std::integral_constant<int, 2>{}, IC64{});
        else if (!g_rec && tile_chunk(nz, 8) <= 4) launch(IC4{}, IC64{});
        else if (!g_rec && tile_chunk(nz, 16) <= 4) launch(IC4{}, IC32{});
        else if (tile_chunk(nz, 16) <= 6) launch(IC6{}, IC32{});
        else launch(IC8{}, IC32{});
    } else {
        if (!ch.active) lagged_shell(shell, s);
        const int width = COL_WIDTH[var];
        switch (COL_DEPTH[var]) {
        case 2:
            launch_cols(0, nx - 1, 0, ny - 1, s,
                        [=] __device__(int i, int j) { column(i, j, std::integral_constant<int, 2>{}); }, width);
            break;
        case 4:
            launch_cols(0, nx - 1, 0, ny - 1, s,
                        [=] __device__(int i, int j) { column(i, j, std::integral_constant<int, 4>{}); }, width);
            break;
        default:
            launch_cols(0, nx - 1, 0, ny - 1, s,
                        [=] __device__(int i, int j) { column(i, j, std::integral_constant<int, 3>{}); }, width);
            break;
        }
    }
    if (tag >= 0) (void)hipEventRecord(P.tuner->ev[2 * tag + 1], s);
    // algorithmic bytes per cell: the fields of the substep this kernel reads
    // (stage rho, rho*theta, rho*u, rho*v, rho*w; the previous rho*w; the new
    // rho*u, rho*v; the current rho, rho*theta; the slow RHS of rho, rho*theta,
    // rho*w; the averaged rho*w; qv, qc when moist) and writes (rho*w, averaged
    // rho*w, rho, rho*theta), 8 B each.  The tridiagonal coefficients, theta
    // and the sweep's intermediates are not counted.
    kt_stop(P.timer, KT_FAST_COLUMN, s, (moist ? 20.0 : 18.0) * 8.0 * nx * ny * nz, "fast_rhs_N column");
}

}  // namespace erfx

// ---- erf_fast_rhs_N with no device allocation ---------------------------------
// For callers that cannot allocate device memory (code under stream / graph
// capture, tight serving loops, harnesses that forbid hipMalloc): the work
// fields of the substep (the rho*w increment, the two horizontal divergences
// and the tridiagonal solution), 4 of the layout, live in one static device
// array instead of a context's workspace.
// Each GPU holds its own copy of the array until the process ends; calls on
// one GPU share it, so two calls that overlap on one GPU race.  No element of
// it needs to start at zero: every launch of the substep writes each element
// it reads (the column kernel its own column)
// before reading it, so whatever a previous call left there is never seen.
namespace erfx {
namespace noalloc {
constexpr size_t MAX_FIELD = (size_t(8) << 20) / 5;      // doubles of the largest box's layout
constexpr size_t SCRATCH_DOUBLES = 4 * MAX_FIELD;         // 51.2 MiB
constexpr int MAX_DEVICES = 64;
static __device__ __align__(256) double scratch[SCRATCH_DOUBLES];
// The array's device address per device, looked up once on the device's first
// call (the host-side name of a __device__ array is only a stand-in: passing it
// to a kernel would fault).
static double* g_ptr[MAX_DEVICES];
static std::mutex g_mu;

static int device_scratch(double** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= MAX_DEVICES) {
        set_error("erfx_fast_rhs_N_noalloc: device index beyond the table of scratch addresses");
        return ERFX_ERR_NODEVICE;
    }
    std::lock_guard<std::mutex> lock(g_mu);
    if (!g_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        g_ptr[dev] = static_cast<double*>(p);
    }
    *out = g_ptr[dev];
    return ERFX_OK;
}
}  // namespace noalloc

}  // namespace erfx

using namespace erfx;

extern "C" int erfx_fast_rhs_N_noalloc(const erfx_config* cfg, void* stream, int step, int nrk,
                                       const erfx_state* slow_rhs, const erfx_state* prev,
                                       const erfx_state* stage, const double* prim, const double* pi_stage,
                                       const double* fast_coeffs, erfx_state* data, erfx_state* scratch,
                                       double dtau, double beta_s, double facinv) {
    auto bad = [](const erfx_state* s) { return !s || !s->cons || !s->xmom || !s->ymom || !s->zmom; };
    if (!cfg || bad(slow_rhs) || bad(prev) || bad(stage) || bad(data) || bad(scratch) || !prim || !pi_stage ||
        !fast_coeffs) {
        set_error("null argument");
        return ERFX_ERR_ARG;
    }
    int rc = validate_config(*cfg);
    if (rc) return rc;
    if (cfg->use_terrain) { set_error("a terrain-following grid takes erf_fast_rhs_T"); return ERFX_ERR_STATE; }
    if (!(nrk > 0 || step == 0)) {
        set_error("the first RK stage takes a single substep (ERF_fast_rhs_N.cpp:106)");
        return ERFX_ERR_ARG;
    }
    erfx_layout lay;
    erfx_layout_for(cfg, &lay);
    const size_t ne = (size_t)lay.nelem;
    if (ne > noalloc::MAX_FIELD) {
        set_error("erfx_fast_rhs_N_noalloc: the box's layout has " + std::to_string(ne) +
                  " doubles a field, the static buffer holds " + std::to_string(noalloc::MAX_FIELD) +
                  " of each of its 4 (boxes up to about 108 x 108 x 108 cells)");
        return ERFX_ERR_ARG;
    }
    double* base = nullptr;
    rc = noalloc::device_scratch(&base);
    if (rc) return rc;
    Params P;
    make_params(*cfg, lay, P);
    FastWork W;
    W.drw = base;
    W.trhs = base + ne;          // two components
    W.soln = base + 3 * ne;
    fast_rhs_N(P, W, step, nrk, *slow_rhs, *prev, *stage, prim, pi_stage, fast_coeffs, *data, *scratch, dtau,
               beta_s, facinv, static_cast<hipStream_t>(stream));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, "kernel launch");
    return ERFX_OK;
}
