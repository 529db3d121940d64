// erfx_bc.hip -- ghost-cell fills, momentum <-> velocity conversion and
// cons_to_prim on the GPU (level 0, one box).
//
// The fills keep ERF's order -- periodic copy, lateral x, lateral y, vertical --
// because corner ghosts read values written by the earlier stages
// (ERF_PhysBCFunct.cpp:16-367).  Each stage is one launch over its ghost slabs.
#include "erfx_common.h"
#include "erfx_internal.h"
#include "erfx_terrain.h"

namespace erfx {

// FabArray::FillBoundary for one periodic box: ghost points whose periodic
// image lies in the valid region take that value.  Launched over the lateral
// ghost slabs of the periodic directions only (z is never periodic here).
void fill_boundary_periodic(const Params& P, double* a, int ncomp, int ng, int nodal_dir, hipStream_t s) {
    const Lay L = P.L;
    const int n0 = L.nx, n1 = L.ny, n2 = L.nz;
    const int vh0 = n0 - 1 + (nodal_dir == 0), vh1 = n1 - 1 + (nodal_dir == 1), vh2 = n2 - 1 + (nodal_dir == 2);
    const bool px = P.periodic[0], py = P.periodic[1];
    if (!px && !py) return;
    const long ne = L.ne;
    // ghost layers of z are not periodic: restrict to valid k
    if (px) {
        // i' in [0, 2ng): lo slab then hi slab
        Box b(0, -ng, 0, 2 * ng - 1, vh1 + ng, vh2);
        launch_box(b, s, [=] __device__(int ip, int j, int k) {
            int i = ip < ng ? ip - ng : vh0 + 1 + (ip - ng);
            int qi = i < 0 ? i + n0 : i - n0;
            int qj = j;
            if (py) { if (qj < 0) qj += n1; else if (qj > vh1) qj -= n1; }
            if (qi < 0 || qi > vh0 || qj < 0 || qj > vh1) return;
            long d = L.ix(i, j, k), sidx = L.ix(qi, qj, k);
            for (int c = 0; c < ncomp; ++c) a[d + c * ne] = a[sidx + c * ne];
        });
    }
    if (py) {
        Box b(-ng, 0, 0, vh0 + ng, 2 * ng - 1, vh2);
        launch_box(b, s, [=] __device__(int i, int jp, int k) {
            int j = jp < ng ? jp - ng : vh1 + 1 + (jp - ng);
            int qj = j < 0 ? j + n1 : j - n1;
            int qi = i;
            if (px) { if (qi < 0) qi += n0; else if (qi > vh0) qi -= n0; }
            if (qi < 0 || qi > vh0 || qj < 0 || qj > vh1) return;
            long d = L.ix(i, j, k), sidx = L.ix(qi, qj, k);
            for (int c = 0; c < ncomp; ++c) a[d + c * ne] = a[sidx + c * ne];
        });
    }
}

// ERFPhysBCFunct_cons::operator() with do_fb: FillBoundary of all components,
// then impose_lateral_cons_bcs (ERF_BoundaryConditions_cons.cpp:17-246) and
// impose_vertical_cons_bcs (:261-494) on components [icomp, icomp+ncomp).
// the ext_dir values of every cons component on face `ori`
struct ExtVals {
    double v[ERFX_NCONS_MOIST];
};
static ExtVals ext_vals(const Params& P, int ori) {
    ExtVals e;
    for (int n = 0; n < ERFX_NCONS_MOIST; ++n) e.v[n] = P.cons_extdir[n][ori];
    return e;
}

void fill_cons(const Params& P, double* c, int icomp, int ncomp, int ng, hipStream_t s) {
    fill_boundary_periodic(P, c, P.cfg.ncons, P.ng_cons, -1, s);
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const long ne = L.ne;
    if (!P.periodic[0]) {
        const int tl = P.bck[3][0], th = P.bck[3][3];
        Box b(0, -ng, 0, 2 * ng - 1, ny - 1 + ng, nz - 1);
        ExtVals xl = ext_vals(P, 0), xh = ext_vals(P, 3);
        launch_box(b, s, [=] __device__(int ip, int j, int k) {
            bool lo = ip < ng;
            int i = lo ? ip - ng : nx + (ip - ng);
            int t = lo ? tl : th;
            int src;
            if (t == EXT_DIR) {   // ERF_BoundaryConditions_cons.cpp:68-104
                const long d = L.ix(i, j, k);
                for (int n = icomp; n < icomp + ncomp; ++n) c[d + n * ne] = lo ? xl.v[n] : xh.v[n];
                return;
            }
            if (t == FOEXTRAP) src = lo ? 0 : nx - 1;
            else if (t == REFLECT_EVEN) src = lo ? -1 - i : 2 * (nx - 1) + 1 - i;
            else return;
            long d = L.ix(i, j, k), sidx = L.ix(src, j, k);
            for (int n = icomp; n < icomp + ncomp; ++n) c[d + n * ne] = c[sidx + n * ne];
        });
    }
    if (!P.periodic[1]) {
        const int tl = P.bck[3][1], th = P.bck[3][4];
        Box b(-ng, 0, 0, nx - 1 + ng, 2 * ng - 1, nz - 1);
        ExtVals yl = ext_vals(P, 1), yh = ext_vals(P, 4);
        launch_box(b, s, [=] __device__(int i, int jp, int k) {
            bool lo = jp < ng;
            int j = lo ? jp - ng : ny + (jp - ng);
            int t = lo ? tl : th;
            int src;
            if (t == EXT_DIR) {
                const long d = L.ix(i, j, k);
                for (int n = icomp; n < icomp + ncomp; ++n) c[d + n * ne] = lo ? yl.v[n] : yh.v[n];
                return;
            }
            if (t == FOEXTRAP) src = lo ? 0 : ny - 1;
            else if (t == REFLECT_EVEN) src = lo ? -1 - j : 2 * (ny - 1) + 1 - j;
            else return;
            long d = L.ix(i, j, k), sidx = L.ix(i, src, k);
            for (int n = icomp; n < icomp + ncomp; ++n) c[d + n * ne] = c[sidx + n * ne];
        });
    }
    {   // vertical: foextrap on both z faces for every supported face type
        Box b(-ng, -ng, 0, nx - 1 + ng, ny - 1 + ng, 2 * ng - 1);
        launch_box(b, s, [=] __device__(int i, int j, int kp) {
            bool lo = kp < ng;
            int k = lo ? kp - ng : nz + (kp - ng);
            int src = lo ? 0 : nz - 1;
            long d = L.ix(i, j, k), sidx = L.ix(i, j, src);
            for (int n = icomp; n < icomp + ncomp; ++n) c[d + n * ne] = c[sidx + n * ne];
        });
    }
}

// Tangential/normal face-velocity fills along one lateral or vertical
// direction.  `dir` is the fill direction, `nodal` whether the field is
// staggered along it.  Rules follow ERF_BoundaryConditions_{x,y,z}vel.cpp.
struct FaceFill {
    int tl, th;       // kinds on lo/hi sides
    double vl, vh;    // Dirichlet values
};

__device__ __forceinline__ double vel_rule_cell(const double* a, const Lay& L, int t, double v, bool lo,
                                                int dir, int i, int j, int k, int n) {
    // cell-centred along dir (tangential component): ghost m in [-ng,-1] or [n, n+ng-1]
    int p[3] = {i, j, k};
    int m = p[dir];
    int q = p[dir];
    double sgn = 1.0;
    if (t == EXT_DIR) return v;
    if (t == FOEXTRAP) q = lo ? 0 : n - 1;
    else if (t == REFLECT_EVEN) q = lo ? -1 - m : 2 * (n - 1) + 1 - m;
    else if (t == REFLECT_ODD) { q = lo ? -1 - m : 2 * (n - 1) + 1 - m; sgn = -1.0; }
    else return NAN;
    p[dir] = q;
    double val = a[L.ix(p[0], p[1], p[2])];
    return sgn < 0 ? -val : val;
}

// ERFPhysBCFunct_u/v::operator() for the velocity component `comp` (0 = x, 1 = y).
static void fill_hvel(const Params& P, double* a, int comp, int ng, hipStream_t s) {
    fill_boundary_periodic(P, a, 1, P.ng_vel, comp, s);
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int nn[3] = {nx, ny, nz};
    // extents of the staggered box
    const int hx = nx - 1 + (comp == 0), hy = ny - 1 + (comp == 1);
    for (int dir = 0; dir < 2; ++dir) {
        if (P.periodic[dir]) continue;
        const int tl = P.bck[comp][dir], th = P.bck[comp][dir + 3];
        const double vl = P.vel_extdir[comp][dir], vh = P.vel_extdir[comp][dir + 3];
        const int n = nn[dir];
        if (dir == comp) {
            // normal component: ghosts beyond the boundary faces plus the faces
            // themselves for ext_dir / neumann_int (ERF_BoundaryConditions_xvel.cpp:55-110)
            Box b = dir == 0 ? Box(0, -ng, 0, 2 * ng + 1, hy + ng, nz - 1) : Box(-ng, 0, 0, hx + ng, 2 * ng + 1, nz - 1);
            launch_box(b, s, [=] __device__(int i0, int j0, int k) {
                int pp = dir == 0 ? i0 : j0;
                bool lo = pp <= ng;              // ng ghosts + the lo face
                int m = lo ? pp - ng : n + (pp - ng - 1);   // lo: -ng..0 ; hi: n..n+ng
                int t = lo ? tl : th;
                double v = lo ? vl : vh;
                int p[3] = {i0, j0, k};
                p[dir] = m;
                bool face = lo ? (m == 0) : (m == n);
                auto at = [&](int q) { int r[3] = {p[0], p[1], p[2]}; r[dir] = q; return a[L.ix(r[0], r[1], r[2])]; };
                double val;
                if (face) {
                    if (t == EXT_DIR) val = v;
                    else if (t == NEUMANN_INT) val = lo ? (4.0 * at(1) - at(2)) / 3.0 : (4.0 * at(n - 1) - at(n - 2)) / 3.0;
                    else return;
                } else {
                    if (t == EXT_DIR) val = v;
                    else if (t == FOEXTRAP) val = at(lo ? 0 : n);
                    else if (t == REFLECT_EVEN) val = at(lo ? -m : 2 * n - m);
                    else if (t == REFLECT_ODD) val = -at(lo ? -m : 2 * n - m);
                    else if (t == NEUMANN_INT) val = lo ? (4.0 * at(1) - at(2)) / 3.0 : (4.0 * at(n - 1) - at(n - 2)) / 3.0;
                    else return;
                }
                a[L.ix(p[0], p[1], p[2])] = val;
            });
        } else {
            Box b = dir == 0 ? Box(0, -ng, 0, 2 * ng - 1, hy + ng, nz - 1) : Box(-ng, 0, 0, hx + ng, 2 * ng - 1, nz - 1);
            launch_box(b, s, [=] __device__(int i0, int j0, int k) {
                int pp = dir == 0 ? i0 : j0;
                bool lo = pp < ng;
                int m = lo ? pp - ng : n + (pp - ng);
                int p[3] = {i0, j0, k};
                p[dir] = m;
                double val = vel_rule_cell(a, L, lo ? tl : th, lo ? vl : vh, lo, dir, p[0], p[1], p[2], n);
                a[L.ix(p[0], p[1], p[2])] = val;
            });
        }
    }
    {   // vertical, over the full grown box (ERF_BoundaryConditions_xvel.cpp:200-245)
        const int tl = P.bck[comp][2], th = P.bck[comp][5];
        const double vl = P.vel_extdir[comp][2], vh = P.vel_extdir[comp][5];
        Box b(-ng, -ng, 0, hx + ng, hy + ng, 2 * ng - 1);
        launch_box(b, s, [=] __device__(int i, int j, int kp) {
            bool lo = kp < ng;
            int k = lo ? kp - ng : nz + (kp - ng);
            double val = vel_rule_cell(a, L, lo ? tl : th, lo ? vl : vh, lo, 2, i, j, k, nz);
            a[L.ix(i, j, k)] = val;
        });
    }
}

void fill_xvel(const Params& P, double* a, int ng, hipStream_t s) { fill_hvel(P, a, 0, ng, s); }
void fill_yvel(const Params& P, double* a, int ng, hipStream_t s) { fill_hvel(P, a, 1, ng, s); }

// ERFPhysBCFunct_w::operator() (ERF_PhysBCFunct.cpp:271-367) and
// ERF_BoundaryConditions_zvel.cpp:16-268: the box is clipped to k in [0, nz];
// w(k=0) always takes the zlo Dirichlet value, which on a terrain grid is
// Omega's, w following the slope of the filled u, v (:220-257).
void fill_zvel(const Params& P, double* a, int ng, hipStream_t s, const double* uf, const double* vf) {
    fill_boundary_periodic(P, a, 1, P.ng_vel, 2, s);
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int nn[2] = {nx, ny};
    for (int dir = 0; dir < 2; ++dir) {
        if (P.periodic[dir]) continue;
        const int tl = P.bck[2][dir], th = P.bck[2][dir + 3];
        const double vl = P.vel_extdir[2][dir], vh = P.vel_extdir[2][dir + 3];
        const int n = nn[dir];
        Box b = dir == 0 ? Box(0, -ng, 0, 2 * ng - 1, ny - 1 + ng, nz) : Box(-ng, 0, 0, nx - 1 + ng, 2 * ng - 1, nz);
        launch_box(b, s, [=] __device__(int i0, int j0, int k) {
            int pp = dir == 0 ? i0 : j0;
            bool lo = pp < ng;
            int m = lo ? pp - ng : n + (pp - ng);
            int p[3] = {i0, j0, k};
            p[dir] = m;
            double val = vel_rule_cell(a, L, lo ? tl : th, lo ? vl : vh, lo, dir, p[0], p[1], p[2], n);
            a[L.ix(p[0], p[1], p[2])] = val;
        });
    }
    const double vl = P.vel_extdir[2][2], vh = P.vel_extdir[2][5];
    const int th = P.bck[2][5];
    // both planes in one launch: kp = 0 -> k = 0, kp = 1 -> k = nz
    Box b(-ng, -ng, 0, nx - 1 + ng, ny - 1 + ng, 1);
    if (P.terrain) {
        const Zn z{P.z_nd, L};
        const Fld u{uf, L}, v{vf, L};
        const double dxi = P.dxInv[0], dyi = P.dxInv[1];
        launch_box(b, s, [=] __device__(int i, int j, int kp) {
            if (kp == 0) { a[L.ix(i, j, 0)] = met::w_from_omega(i, j, 0, vl, u, v, z, dxi, dyi); return; }
            if (th == EXT_DIR) a[L.ix(i, j, nz)] = met::w_from_omega(i, j, nz, vh, u, v, z, dxi, dyi);
            else if (th == NEUMANN_INT) a[L.ix(i, j, nz)] = (4.0 * a[L.ix(i, j, nz - 1)] - a[L.ix(i, j, nz - 2)]) / 3.0;
        });
        return;
    }
    launch_box(b, s, [=] __device__(int i, int j, int kp) {
        if (kp == 0) { a[L.ix(i, j, 0)] = vl; return; }
        if (th == EXT_DIR) a[L.ix(i, j, nz)] = vh;
        else if (th == NEUMANN_INT) a[L.ix(i, j, nz)] = (4.0 * a[L.ix(i, j, nz - 1)] - a[L.ix(i, j, nz - 2)]) / 3.0;
    });
}

// MomentumToVelocity (Source/Utils/ERF_MomentumToVelocity.cpp:24-96) on the
// valid faces; one launch covers the three staggered boxes.
void momentum_to_velocity(const Params& P, double* xv, double* yv, double* zv, const double* dens,
                          const double* xm, const double* ym, const double* zm, hipStream_t s) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    Box b(0, 0, 0, nx, ny, nz);
    launch_box(b, s, [=] __device__(int i, int j, int k) {
        long c = L.ix(i, j, k);
        if (j < ny && k < nz) xv[c] = xm[c] * 2.0 / (dens[c] + dens[c - 1]);
        if (i < nx && k < nz) yv[c] = ym[c] * 2.0 / (dens[c] + dens[c - L.sy]);
        if (i < nx && j < ny) zv[c] = zm[c] * 2.0 / (dens[c] + dens[c - L.sz]);
    });
}

// VelocityToMomentum (Source/Utils/ERF_VelocityToMomentum.cpp:24-114): faces
// of the valid box grown by g (w limited to k in [0, nz]).
void velocity_to_momentum(const Params& P, const double* xv, const double* yv, const double* zv, int gx,
                          int gz_w, const double* dens, double* xm, double* ym, double* zm, hipStream_t s) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int zlo_w = gz_w > 0 ? 0 : 0, zhi_w = nz;
    Box b(-gx, -gx, -gx, nx + gx, ny + gx, nz + gx);
    launch_box(b, s, [=] __device__(int i, int j, int k) {
        long c = L.ix(i, j, k);
        if (j <= ny - 1 + gx && k <= nz - 1 + gx) xm[c] = xv[c] * 0.5 * (dens[c] + dens[c - 1]);
        if (i <= nx - 1 + gx && k <= nz - 1 + gx) ym[c] = yv[c] * 0.5 * (dens[c] + dens[c - L.sy]);
        if (i <= nx - 1 + gx && j <= ny - 1 + gx && k >= zlo_w && k <= zhi_w && k >= -gz_w && k <= nz + gz_w)
            zm[c] = zv[c] * 0.5 * (dens[c] + dens[c - L.sz]);
    });
}

// The start of a step where the fills are fused: VelocityToMomentum of the old
// velocities, and on the valid faces the MomentumToVelocity and VelocityToMomentum
// that apply_bcs on the old state begins with (its new velocities xn, yn, zn).
// Bound by HBM: 512 x 512 x 96 345 us for the first part alone and 857 for the fill,
// 507 + 158 so.
void velocity_round_trip(const Params& P, const double* xv, const double* yv, const double* zv, int gx, int gz_w,
                         const double* dens, double* xm, double* ym, double* zm, double* xn, double* yn, double* zn,
                         hipStream_t s) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    launch_box(Box(-gx, -gx, -gx, nx + gx, ny + gx, nz + gx), s, [=] __device__(int i, int j, int k) {
        const long c = L.ix(i, j, k);
        const bool in = i >= 0 && j >= 0 && k >= 0 && i <= nx && j <= ny && k <= nz;
        if (j <= ny - 1 + gx && k <= nz - 1 + gx) {
            const double d = dens[c] + dens[c - 1];
            double m = xv[c] * 0.5 * d;
            if (in && j < ny && k < nz) {
                const double u = m * 2.0 / d;
                xn[c] = u;
                m = u * 0.5 * d;
            }
            xm[c] = m;
        }
        if (i <= nx - 1 + gx && k <= nz - 1 + gx) {
            const double d = dens[c] + dens[c - L.sy];
            double m = yv[c] * 0.5 * d;
            if (in && i < nx && k < nz) {
                const double v = m * 2.0 / d;
                yn[c] = v;
                m = v * 0.5 * d;
            }
            ym[c] = m;
        }
        if (i <= nx - 1 + gx && j <= ny - 1 + gx && k >= 0 && k <= nz && k >= -gz_w && k <= nz + gz_w) {
            const double d = dens[c] + dens[c - L.sz];
            double m = zv[c] * 0.5 * d;
            if (in && i < nx && j < ny && k > 0 && k < nz) {
                const double w = m * 2.0 / d;
                zn[c] = w;
                m = w * 0.5 * d;
            }
            zm[c] = m;
        }
    });
}

// The fused fills: every ghost value the generic sequences below leave behind,
// computed from valid data alone, so no lane reads a ghost another lane writes
// and one launch replaces the stages.  What a ghost point holds after
// FillBoundary, the lateral x fill, the lateral y fill and the vertical fill
// follows by resolving them in reverse: the vertical row takes the point's value
// on the nearest level, a point beyond a y face what the y rule reads (its
// periodic image on a periodic axis), that point's x position likewise.
bool bcs_fusable(const Params& P) {
    if (!P.periodic[0] && !P.periodic[1]) return false;
    if (g_rec && g_rec->generic_fills && !(P.periodic[0] && P.periodic[1])) return false;
    const int G = P.ng_cons > P.ng_vel ? P.ng_cons : P.ng_vel;
    if (P.L.nx < G + 1 || P.L.ny < G + 1 || P.L.nz < 2 * G) return false;
    for (int v = 0; v < 2; ++v)
        for (int o : {2, 5})
            if (P.bck[v][o] != EXT_DIR && P.bck[v][o] != FOEXTRAP) return false;
    if (P.bck[2][5] != EXT_DIR && P.bck[2][5] != NEUMANN_INT) return false;
    for (int d = 0; d < 2; ++d) {
        if (P.periodic[d]) continue;
        if (P.terrain) return false;
        for (int o : {d, d + 3})
            for (int f = 0; f < 4; ++f) {
                const int t = P.bck[f][o];
                if (t != EXT_DIR && t != FOEXTRAP && t != REFLECT_EVEN && !(f < 3 && t == REFLECT_ODD) &&
                    !(f == d && t == NEUMANN_INT))
                    return false;
            }
    }
    return P.cfg.ncons <= 8;
}
// periodic in x and y besides: the substeps of a stage can be chained
bool fast_bcs_fusable(const Params& P) { return P.periodic[0] && P.periodic[1] && bcs_fusable(P); }

struct ConsRows {
    int r[8];   // ghost cells filled by the lateral rules and the vertical rows, per component
};

// Lateral resolution of one box: the rules of each field on the four lateral
// faces.  Each `*_at` returns the value of a point of valid k at any lateral
// index, from `base` at valid points.  PER: both axes periodic (the rules drop
// out at compile time).
struct LatRules {
    int kind[4][6];                          // x-, y-, z-velocity, cons
    double vel[3][6];
    double ext[ERFX_NCONS_MOIST][6];
    bool px, py;
};
struct LatImages {                           // both axes periodic: no rule is read (nor passed to the kernels)
    static constexpr int kind[4][6] = {};
    static constexpr double vel[3][6] = {};
    static constexpr double ext[ERFX_NCONS_MOIST][6] = {};
    static constexpr bool px = true, py = true;
};
template <bool PER>
struct LatFill : std::conditional_t<PER, LatImages, LatRules> {
    using Rules = std::conditional_t<PER, LatImages, LatRules>;
    using Rules::kind;
    using Rules::vel;
    using Rules::ext;
    using Rules::px;
    using Rules::py;
    int nx, ny;
    static __device__ __forceinline__ int wrap(int a, int n, int hi) { return a < 0 ? a + n : (a > hi ? a - n : a); }
    // cell-centred along an axis of n cells: moves `a` to the source index, false
    // for a Dirichlet ghost; `neg` flips the sign (odd reflection)
    static __device__ __forceinline__ bool cell(int& a, int n, int tl, int th, bool per, bool& neg) {
        if (PER || per) { a = wrap(a, n, n - 1); return true; }
        if (a >= 0 && a <= n - 1) return true;
        const bool lo = a < 0;
        const int t = lo ? tl : th;
        if (t == EXT_DIR) return false;
        if (t == FOEXTRAP) a = lo ? 0 : n - 1;
        else { a = lo ? -1 - a : 2 * (n - 1) + 1 - a; neg ^= (t == REFLECT_ODD); }
        return true;
    }
    // moves (i, j) to the source of a cons ghost, false where the Dirichlet value v is it
    __device__ __forceinline__ bool cons_src(int n, int& i, int& j, double& v) const {
        bool neg = false;
        const bool jl = j < 0, il = i < 0;
        if (!cell(j, ny, kind[3][1], kind[3][4], py, neg)) { v = jl ? ext[n][1] : ext[n][4]; return false; }
        if (!cell(i, nx, kind[3][0], kind[3][3], px, neg)) { v = il ? ext[n][0] : ext[n][3]; return false; }
        return true;
    }
    template <class B>
    __device__ __forceinline__ double cons_at(int n, int i, int j, const B& base) const {
        double v = 0.0;
        return cons_src(n, i, j, v) ? base(i, j) : v;
    }
    // a velocity component along its own axis (faces 0..n) from base(face), which
    // is evaluated in one place (and once more for the Neumann rule), as it is the
    // kernel's largest expression; `rules` false: periodic images alone
    template <class B>
    static __device__ __forceinline__ double normal(int m, int n, int tl, int th, double vl, double vh, bool per,
                                                    bool rules, const B& base) {
        if (PER || per) return base(wrap(m, n, n));
        bool neu = false, odd = false;
        int a = m;
        const bool lo = m <= 0;
        if (rules && (m <= 0 || m >= n)) {
            const int t = lo ? tl : th;
            if (t == EXT_DIR) return lo ? vl : vh;
            if (t == NEUMANN_INT) { neu = true; a = lo ? 1 : n - 1; }
            else if (m < 0 || m > n) {
                a = t == FOEXTRAP ? (lo ? 0 : n) : (lo ? -m : 2 * n - m);
                odd = t == REFLECT_ODD;
            }
        }
        double v = base(a);
        if (neu) v = (4.0 * v - base(lo ? 2 : n - 2)) / 3.0;
        return odd ? -v : v;
    }
    template <class B>
    __device__ __forceinline__ double u_at(int i, int j, bool rules, const B& base) const {
        bool neg = false;
        int b = j;
        if (!cell(b, ny, kind[0][1], kind[0][4], py, neg)) return j < 0 ? vel[0][1] : vel[0][4];
        const double v = normal(i, nx, kind[0][0], kind[0][3], vel[0][0], vel[0][3], px, rules,
                                [&](int m) __attribute__((always_inline)) { return base(m, b); });
        return neg ? -v : v;
    }
    template <class B>
    __device__ __forceinline__ double v_at(int i, int j, bool rules, const B& base) const {
        // one axis is periodic, so the order of the two rules does not matter
        bool neg = false;
        int a = i;
        if (!cell(a, nx, kind[1][0], kind[1][3], px, neg)) return i < 0 ? vel[1][0] : vel[1][3];
        const double v = normal(j, ny, kind[1][1], kind[1][4], vel[1][1], vel[1][4], py, rules,
                                [&](int m) __attribute__((always_inline)) { return base(a, m); });
        return neg ? -v : v;
    }
    template <class B>
    __device__ __forceinline__ double w_at(int i, int j, const B& base) const {
        bool neg = false;
        int a = i, b = j;
        if (!cell(b, ny, kind[2][1], kind[2][4], py, neg)) return j < 0 ? vel[2][1] : vel[2][4];
        if (!cell(a, nx, kind[2][0], kind[2][3], px, neg)) return i < 0 ? vel[2][0] : vel[2][3];
        const double v = base(a, b);
        return neg ? -v : v;
    }
    // whether the face m of a component normal to an axis takes a rule there
    static __device__ __forceinline__ bool face_rule(int m, int n, int tl, int th, bool per) {
        if (PER || per) return false;
        const int t = m == 0 ? tl : th;
        return (m == 0 || m == n) && (t == EXT_DIR || t == NEUMANN_INT);
    }
};
template <bool PER>
static LatFill<PER> lat_fill(const Params& P) {
    LatFill<PER> F;
    F.nx = P.L.nx; F.ny = P.L.ny;
    if constexpr (!PER) {
        F.px = P.periodic[0]; F.py = P.periodic[1];
        for (int o = 0; o < 6; ++o) {
            for (int f = 0; f < 4; ++f) F.kind[f][o] = P.bck[f][o];
            for (int v = 0; v < 3; ++v) F.vel[v][o] = P.vel_extdir[v][o];
            for (int n = 0; n < ERFX_NCONS_MOIST; ++n) F.ext[n][o] = P.cons_extdir[n][o];
        }
    }
    return F;
}

// Ghost cells of cons and every velocity the fills define, in one launch.
//   RAW = false: the velocities are MomentumToVelocity of S's momenta on the
//   valid faces (ERF_MomentumToVelocity.cpp:24-96), ghosts filled from those;
//   RAW = true: the velocity arrays hold the valid faces already; only ghosts and
//   the faces a rule sets are written, and with S's momenta given (ngv is P.ng_vel
//   then) VelocityToMomentum of those, where the sequence applies it and on the
//   periodic images.
// ngv: ghost width of the rules and vertical rows; periodic images reach
// P.ng_vel (P.ng_cons for cons).  Points the sequences do not touch are not
// written.
template <bool PER, bool RAW>
static void fill_points(const Params& P, const erfx_state& S, double* xv, double* yv, double* zv, const ConsRows& R,
                        int rmax, int ngv, hipStream_t s) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int ngC = P.ng_cons, ngV = P.ng_vel;
    const int G = ngC > ngV ? ngC : ngV;
    const long ne = L.ne;
    const int nc = P.cfg.ncons;
    double* c = S.cons;
    double* xm = S.xmom;
    double* ym = S.ymom;
    double* zm = S.zmom;
    const LatFill<PER> F = lat_fill<PER>(P);
    const bool px = PER || P.periodic[0], py = PER || P.periodic[1];
    const int xtl = P.bck[0][2], xth = P.bck[0][5], ytl = P.bck[1][2], yth = P.bck[1][5];
    const double xvl = P.vel_extdir[0][2], xvh = P.vel_extdir[0][5];
    const double yvl = P.vel_extdir[1][2], yvh = P.vel_extdir[1][5];
    const double zvl = P.vel_extdir[2][2], zvh = P.vel_extdir[2][5];
    const int zth = P.bck[2][5];
    const int kz = rmax > ngv ? rmax : (ngv > 1 ? ngv : 1);
    const Box grown(-G, -G, -kz, nx + G, ny + G, nz - 1 + kz);
    const bool terr = PER && P.terrain;
    const Zn zt{P.z_nd, L};
    const double dxi = P.dxInv[0], dyi = P.dxInv[1];
    auto point = [=] __device__(int i, int j, int k) {
        // ghost depth along x and y of the cell and of the x- / y-face
        const int dxc = i < 0 ? -i : (i > nx - 1 ? i - (nx - 1) : 0), dyc = j < 0 ? -j : (j > ny - 1 ? j - (ny - 1) : 0);
        const int dxf = i < 0 ? -i : (i > nx ? i - nx : 0), dyf = j < 0 ? -j : (j > ny ? j - ny : 0);
        const long q = L.ix(i, j, k);
        const bool kval = k >= 0 && k <= nz - 1;
        const int depth = k < 0 ? -k : (k > nz - 1 ? k - nz + 1 : 0);   // vertical ghost row
        // within g of the valid box, reached by periodic images alone
        auto image = [&](int dx, int dy, int g) { return (dx == 0 || px) && (dy == 0 || py) && dx <= g && dy <= g; };
        // ---- cons ghosts
        if (kval && (dxc > 0 || dyc > 0)) {
            if (image(dxc, dyc, ngC)) {
                const long src = L.ix(LatFill<PER>::wrap(i, nx, nx - 1), LatFill<PER>::wrap(j, ny, ny - 1), k);
                for (int n = 0; n < nc; ++n) c[q + n * ne] = c[src + n * ne];
            } else if (!PER) {
                for (int n = 0; n < nc; ++n)
                    if (dxc <= R.r[n] && dyc <= R.r[n])
                        c[q + n * ne] = F.cons_at(n, i, j, [&](int a, int b) __attribute__((always_inline)) { return c[L.ix(a, b, k) + n * ne]; });
            }
        }
        if (depth > 0) {
            const int ks = k < 0 ? 0 : nz - 1;
            for (int n = 0; n < nc; ++n)
                if (depth <= R.r[n] && dxc <= R.r[n] && dyc <= R.r[n])
                    c[q + n * ne] = F.cons_at(n, i, j, [&](int a, int b) __attribute__((always_inline)) { return c[L.ix(a, b, ks) + n * ne]; });
        }
        // the velocities on valid faces
        auto rho = [&](int a, int b, int kk) __attribute__((always_inline)) {
            return F.cons_at(0, a, b, [&](int e, int f) __attribute__((always_inline)) { return c[L.ix(e, f, kk)]; });
        };
        auto u_of = [&](int fi, int jj, int kk) __attribute__((always_inline)) {
            const long f = L.ix(fi, jj, kk);
            if constexpr (RAW) return xv[f];
            else return xm[f] * 2.0 / (rho(fi, jj, kk) + rho(fi - 1, jj, kk));
        };
        auto v_of = [&](int ii, int fj, int kk) __attribute__((always_inline)) {
            const long f = L.ix(ii, fj, kk);
            if constexpr (RAW) return yv[f];
            else return ym[f] * 2.0 / (rho(ii, fj, kk) + rho(ii, fj - 1, kk));
        };
        auto w_of = [&](int ii, int jj, int fk) __attribute__((always_inline)) {
            const long f = L.ix(ii, jj, fk);
            if constexpr (RAW) return zv[f];
            const int kl = fk - 1 < 0 ? 0 : fk - 1, kh = fk > nz - 1 ? nz - 1 : fk;
            return zm[f] * 2.0 / (rho(ii, jj, kh) + rho(ii, jj, kl));
        };
        auto u_lat = [&](int ii, int jj, int kk, bool rules) __attribute__((always_inline)) {
            return F.u_at(ii, jj, rules, [&](int a, int b) __attribute__((always_inline)) { return u_of(a, b, kk); });
        };
        auto v_lat = [&](int ii, int jj, int kk, bool rules) __attribute__((always_inline)) {
            return F.v_at(ii, jj, rules, [&](int a, int b) __attribute__((always_inline)) { return v_of(a, b, kk); });
        };
        auto w_lat = [&](int ii, int jj, int kk) __attribute__((always_inline)) {
            return F.w_at(ii, jj, [&](int a, int b) __attribute__((always_inline)) { return w_of(a, b, kk); });
        };
        const bool lo = k < 0;
        const int kv = kval ? k : (lo ? 0 : nz - 1);     // the level a vertical row copies
        // ---- x-velocity: valid faces, images and rule ghosts, vertical rows
        const bool un = dxf <= ngv && dyc <= ngv;
        const bool ukeep = RAW && dxf == 0 && dyc == 0 && !LatFill<PER>::face_rule(i, nx, F.kind[0][0], F.kind[0][3], px);
        if (kval ? !ukeep && (un || image(dxf, dyc, ngV)) : depth <= ngv && un) {
            const double u = !kval && (lo ? xtl : xth) == EXT_DIR ? (lo ? xvl : xvh) : u_lat(i, j, kv, un);
            xv[q] = u;
            if (RAW && xm && (kval && image(dxf, dyc, ngV) || dxf <= 1 && dyc <= 1 && k >= -1 && k <= nz))
                xm[q] = u * 0.5 * (rho(i, j, kv) + rho(i - 1, j, kv));
        }
        // ---- y-velocity
        const bool vn = dxc <= ngv && dyf <= ngv;
        const bool vkeep = RAW && dxc == 0 && dyf == 0 && !LatFill<PER>::face_rule(j, ny, F.kind[1][1], F.kind[1][4], py);
        if (kval ? !vkeep && (vn || image(dxc, dyf, ngV)) : depth <= ngv && vn) {
            const double v = !kval && (lo ? ytl : yth) == EXT_DIR ? (lo ? yvl : yvh) : v_lat(i, j, kv, vn);
            yv[q] = v;
            if (RAW && xm && (kval && image(dxc, dyf, ngV) || dxc <= 1 && dyf <= 1 && k >= -1 && k <= nz))
                ym[q] = v * 0.5 * (rho(i, j, kv) + rho(i, j - 1, kv));
        }
        // ---- z-velocity (k = 0 takes the zlo value on the valid box grown by ngv)
        const bool near = dxc <= ngv && dyc <= ngv;
        const bool plane = near && (k == 0 || k == nz);
        if (k >= 0 && k <= nz && (near || image(dxc, dyc, ngV)) && !(RAW && dxc == 0 && dyc == 0 && !plane)) {
            double w;
            if (terr && plane && (k == 0 || zth == EXT_DIR)) {
                // terrain wall: WFromOmega with u, v as this launch leaves them
                auto uf = [&](int ii, int jj, int kk) __attribute__((always_inline)) {
                    const bool l = kk < 0, in = kk >= 0 && kk <= nz - 1;
                    return !in && (l ? xtl : xth) == EXT_DIR ? (l ? xvl : xvh)
                                                             : u_lat(ii, jj, in ? kk : (l ? 0 : nz - 1), true);
                };
                auto vf = [&](int ii, int jj, int kk) __attribute__((always_inline)) {
                    const bool l = kk < 0, in = kk >= 0 && kk <= nz - 1;
                    return !in && (l ? ytl : yth) == EXT_DIR ? (l ? yvl : yvh)
                                                             : v_lat(ii, jj, in ? kk : (l ? 0 : nz - 1), true);
                };
                w = met::w_from_omega(i, j, k, k == 0 ? zvl : zvh, uf, vf, zt, dxi, dyi);
            } else if (plane && k == 0) {
                w = zvl;
            } else if (plane && zth == EXT_DIR) {
                w = zvh;
            } else {
                w = w_lat(i, j, plane ? nz - 1 : k);   // (beyond `near` only images, where no rule applies)
                if (plane) w = (4.0 * w - w_lat(i, j, nz - 2)) / 3.0;
            }
            zv[q] = w;
            if (RAW && xm && (image(dxc, dyc, ngV) || dxc <= 1 && dyc <= 1))
                zm[q] = w * 0.5 * (rho(i, j, k > nz - 1 ? nz - 1 : k) + rho(i, j, k - 1 < 0 ? 0 : k - 1));
        }
    };
    if constexpr (!RAW) {
        launch_box(grown, s, point);
    } else {
        // only the points outside the core 1 .. nx-2, 1 .. ny-2, 1 .. nz-1, which no
        // rule touches: the levels below and above it, the rows beside it, the columns
        // beside those (512 x 512 x 96: 294 us over the whole box, 132 so; 161 x 97 x 63
        // with inflow 34 and 19).  One call of `point`: called from three places it is
        // no longer inlined, and its captures go through scratch (91 us).
        const int wx = nx + 1 + 2 * G, wy = ny + 1 + 2 * G, e = 2 * G + 3;   // e: columns or rows beside the core
        const unsigned nzp = (unsigned)(2 * kz + 1) * (unsigned)wy * (unsigned)wx;
        const unsigned nyp = (unsigned)(nz - 1) * (unsigned)e * (unsigned)wx;
        const unsigned nxp = (unsigned)(nz - 1) * (unsigned)(ny - 2) * (unsigned)e;
        auto beside = [=] __device__(int a, int n) { return a <= G ? a - G : n - 1 + (a - G - 1); };
        launch_grid((nzp + nyp + nxp + 255u) / 256u, s, [=] __device__(unsigned b) {
            unsigned t = b * 256u + threadIdx.x;
            int i, j, k;
            if (t < nzp) {
                i = (int)(t % wx) - G;
                const int r = (int)(t / wx), a = r / wy;
                j = r % wy - G;
                k = a <= kz ? a - kz : nz + (a - kz - 1);
            } else if ((t -= nzp) < nyp) {
                i = (int)(t % wx) - G;
                const int r = (int)(t / wx);
                j = beside(r % e, ny);
                k = 1 + r / e;
            } else if ((t -= nyp) < nxp) {
                i = beside((int)(t % e), nx);
                const int r = (int)(t / e);
                j = 1 + r % (ny - 2);
                k = 1 + r / (ny - 2);
            } else {
                return;
            }
            point(i, j, k);
        });
    }
}

// MomentumToVelocity and VelocityToMomentum of the valid faces, with the density
// ghosts the fill is about to write.  The z-faces of the bottom and the top take
// their rule there.
template <bool PER>
static void valid_faces(const Params& P, const erfx_state& S, double* xv, double* yv, double* zv, hipStream_t s) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const double* c = S.cons;
    double* xm = S.xmom;
    double* ym = S.ymom;
    double* zm = S.zmom;
    const LatFill<PER> F = lat_fill<PER>(P);
    launch_box(Box(0, 0, 0, nx, ny, nz - 1), s, [=] __device__(int i, int j, int k) {
        const long q = L.ix(i, j, k);
        auto rho = [&](int a, int b) __attribute__((always_inline)) {
            double v = 0.0;
            return F.cons_src(0, a, b, v) ? c[L.ix(a, b, k)] : v;
        };
        const double r = rho(i, j);
        if (j < ny) {
            const double d = r + rho(i - 1, j), u = xm[q] * 2.0 / d;
            xv[q] = u;
            xm[q] = u * 0.5 * d;
        }
        if (i < nx) {
            const double d = r + rho(i, j - 1), v = ym[q] * 2.0 / d;
            yv[q] = v;
            ym[q] = v * 0.5 * d;
        }
        if (i < nx && j < ny && k > 0) {
            const double d = r + c[q - L.sz], w = zm[q] * 2.0 / d;
            zv[q] = w;
            zm[q] = w * 0.5 * d;
        }
    });
}

// apply_bcs on a box with a periodic lateral axis in two launches instead of the
// ~30 of the generic sequence below, point for point what that leaves behind:
// fill_points, then the momenta: V2M where the sequence applies it, the periodic
// image's V2M on the FillBoundary layers.  `synced`: every component's ghosts
// take part in the one fill (its rho ghosts are valid on entry, as this forms
// them again).
//
// At the full velocity ghost width the work is split by place instead: the valid
// faces' momentum -> velocity -> momentum, point by point (valid_faces, or the
// kernel that wrote the momenta: `ready`), then everything else in one launch
// around the box.  512 x 512 x 96 with terrain: 857 us in the two launches over the
// grown box; 158 so, and 135 more in the kernel that wrote the momenta.  161 x 97 x
// 63 with inflow, where valid_faces does them: 49 us, and 20 + 26.  A narrower fill
// leaves ghosts of the unruled faces beyond its width and keeps the two launches.
template <bool PER>
static void apply_bcs_fused(const Params& P, const erfx_state& S, double* xv, double* yv, double* zv, int ngc,
                            int ngv, bool fast_only, bool synced, bool ready, hipStream_t s) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int ngC = P.ng_cons, ngV = P.ng_vel;
    const int G = ngC > ngV ? ngC : ngV;
    const long sy = L.sy, sz = L.sz;
    const int nc = P.cfg.ncons;
    // rows per component: rho by the first FillIntermediatePatch, the others by the second
    ConsRows R;
    const int ngu1 = ngc > ngv + 1 ? ngc : ngv + 1;
    const int ncomp2 = fast_only ? 1 : nc - 1;
    int rmax = 0;
    for (int n = 0; n < 8; ++n) {
        R.r[n] = n == 0 ? ngu1 : (n < 1 + ncomp2 && n < nc ? (synced ? ngu1 : ngc) : 0);
        if (R.r[n] > rmax) rmax = R.r[n];
    }
    if (ngv == ngV) {
        if (!ready) valid_faces<PER>(P, S, xv, yv, zv, s);
        fill_points<PER, true>(P, S, xv, yv, zv, R, rmax, ngv, s);
        return;
    }
    fill_points<PER, false>(P, S, xv, yv, zv, R, rmax, ngv, s);
    const double* c = S.cons;
    double* xm = S.xmom;
    double* ym = S.ymom;
    double* zm = S.zmom;
    const bool px = PER || P.periodic[0], py = PER || P.periodic[1];
    const Box grownB(-G, -G, -1, nx + G, ny + G, nz);
    launch_box(grownB, s, [=] __device__(int i, int j, int k) {
        const int dxc = i < 0 ? -i : (i > nx - 1 ? i - (nx - 1) : 0), dyc = j < 0 ? -j : (j > ny - 1 ? j - (ny - 1) : 0);
        const int dxf = i < 0 ? -i : (i > nx ? i - nx : 0), dyf = j < 0 ? -j : (j > ny ? j - ny : 0);
        const long q = L.ix(i, j, k);
        const bool kval = k >= 0 && k <= nz - 1;
        const int ic = px ? LatFill<PER>::wrap(i, nx, nx - 1) : i, jc = py ? LatFill<PER>::wrap(j, ny, ny - 1) : j;
        const int if_ = px ? LatFill<PER>::wrap(i, nx, nx) : i, jf = py ? LatFill<PER>::wrap(j, ny, ny) : j;
        // a FillBoundary layer: beyond the valid box, reached by periodic images alone
        auto image = [&](int dx, int dy) {
            return (dx > 0 || dy > 0) && (dx == 0 || px) && (dy == 0 || py) && dx <= ngV && dy <= ngV;
        };
        // VelocityToMomentum (ERF_VelocityToMomentum.cpp:24-114) at face index f
        auto xm_at = [&](long f) { return xv[f] * 0.5 * (c[f] + c[f - 1]); };
        auto ym_at = [&](long f) { return yv[f] * 0.5 * (c[f] + c[f - sy]); };
        auto zm_at = [&](long f) { return zv[f] * 0.5 * (c[f] + c[f - sz]); };
        if (kval && image(dxf, dyc)) xm[q] = xm_at(L.ix(if_, jc, k));
        else if (dxf <= 1 && dyc <= 1 && k >= -1 && k <= nz) xm[q] = xm_at(q);
        if (kval && image(dxc, dyf)) ym[q] = ym_at(L.ix(ic, jf, k));
        else if (dxc <= 1 && dyf <= 1 && k >= -1 && k <= nz) ym[q] = ym_at(q);
        if (k >= 0 && k <= nz) {
            if (image(dxc, dyc)) zm[q] = zm_at(L.ix(ic, jc, k));
            else if (dxc <= 1 && dyc <= 1) zm[q] = zm_at(q);
        }
    });
}

// ERF::FillIntermediatePatch, level 0 (ERF_FillIntermediatePatch.cpp:27-261).
void fill_intermediate_patch(const Params& P, const erfx_state& S, double* xv, double* yv, double* zv,
                             int ngc, int ngv, bool cons_only, int icomp, int ncomp, hipStream_t s) {
    if (!cons_only) momentum_to_velocity(P, xv, yv, zv, S.cons, S.xmom, S.ymom, S.zmom, s);
    fill_cons(P, S.cons, icomp, ncomp, ngc, s);
    if (!cons_only) {
        fill_xvel(P, xv, ngv, s);
        fill_yvel(P, yv, ngv, s);
        fill_zvel(P, zv, ngv, s, xv, yv);
        velocity_to_momentum(P, xv, yv, zv, 1, 0, S.cons, S.xmom, S.ymom, S.zmom, s);
    }
    fill_boundary_periodic(P, S.cons, P.cfg.ncons, P.ng_cons, -1, s);
    fill_boundary_periodic(P, S.xmom, 1, P.ng_vel, 0, s);
    fill_boundary_periodic(P, S.ymom, 1, P.ng_vel, 1, s);
    fill_boundary_periodic(P, S.zmom, 1, P.ng_vel, 2, s);
}

// apply_bcs (Source/TimeIntegration/ERF_TI_utils.H:53-150).
void apply_bcs(const Params& P, const erfx_state& S, double* xv, double* yv, double* zv, int ngc, int ngv,
               bool fast_only, bool synced, hipStream_t s, bool filled, bool ready) {
    // synced: the sequence reads the density ghosts as they are, which the fused
    // form forms again: the same where the caller says that they are filled
    if ((!synced || filled) && ngc >= 1 && ngv >= 1 && bcs_fusable(P)) {
        if (P.periodic[0] && P.periodic[1]) apply_bcs_fused<true>(P, S, xv, yv, zv, ngc, ngv, fast_only, synced, ready, s);
        else apply_bcs_fused<false>(P, S, xv, yv, zv, ngc, ngv, fast_only, synced, ready, s);
        return;
    }
    int scomp, ncomp, ngu;
    if (!synced) {
        ngu = ngc > ngv + 1 ? ngc : ngv + 1;
        fill_intermediate_patch(P, S, xv, yv, zv, ngu, 0, true, 0, 1, s);
    }
    if (synced) {
        scomp = 0;
        ncomp = fast_only ? 2 : P.cfg.ncons;
        ngu = ngc > ngv + 1 ? ngc : ngv + 1;
    } else {
        scomp = 1;
        ncomp = fast_only ? 1 : P.cfg.ncons - 1;
        ngu = ngc;
    }
    fill_intermediate_patch(P, S, xv, yv, zv, ngu, ngv, false, scomp, ncomp, s);
}

// ERF::FillPatch, level 0 at the old time (ERF_FillPatch.cpp:19-140).
void fill_patch(const Params& P, double* c, double* u, double* v, double* w, hipStream_t s) {
    if (bcs_fusable(P)) {
        const erfx_state S{c, nullptr, nullptr, nullptr};
        ConsRows R;
        for (int n = 0; n < 8; ++n) R.r[n] = n < P.cfg.ncons ? P.ng_cons : 0;
        if (P.periodic[0] && P.periodic[1]) fill_points<true, true>(P, S, u, v, w, R, P.ng_cons, P.ng_vel, s);
        else fill_points<false, true>(P, S, u, v, w, R, P.ng_cons, P.ng_vel, s);
        return;
    }
    fill_cons(P, c, 0, P.cfg.ncons, P.ng_cons, s);
    fill_xvel(P, u, P.ng_vel, s);
    fill_yvel(P, v, P.ng_vel, s);
    fill_zvel(P, w, P.ng_vel, s, u, v);
}

// cons_to_prim (ERF_TI_utils.H:4-45): prim on the box grown by ng, pi_stage
// on the box grown by one.  One launch covers both, and with `pp` the pressure
// perturbation that erf_slow_rhs_pre begins with (ERF_slow_rhs_pre.cpp:337-358),
// on cells grown by one from k = 0 up: this kernel waits for memory, that one for
// its powers (two launches and one: 64^3 22 and 19 us, 256 x 256 x 128 258 and 230,
// 512 x 512 x 96 moist 974 and 847).
void cons_to_prim(const Params& P, const double* c, double* prim, double* pi_stage, int ng, hipStream_t s, double* pp,
                  const double* p0) {
    const Lay L = P.L;
    const int nx = L.nx, ny = L.ny, nz = L.nz;
    const int nprim = P.cfg.ncons - 1;
    const long ne = L.ne;
    const double rdOcp = P.rdOcp;
    const bool moist = P.moist;
    Box b(-ng, -ng, -ng, nx - 1 + ng, ny - 1 + ng, nz - 1 + ng);
    launch_box(b, s, [=] __device__(int i, int j, int k) {
        long q = L.ix(i, j, k);
        double rho = c[q];
        double rho_theta = c[q + ne];
        prim[q] = rho_theta / rho;
        for (int n = 1; n < nprim; ++n) prim[q + n * ne] = c[q + (1 + n) * ne] / rho;
        if (i >= -1 && i <= nx && j >= -1 && j <= ny && k >= -1 && k <= nz)
            pi_stage[q] = eos_exner_of_rt(rho_theta, rdOcp);
        if (pp && i >= -1 && i <= nx && j >= -1 && j <= ny && k >= 0 && k <= nz)
            pp[q] = (moist ? eos_p_of_rt_qv(rho_theta, c[q + ERFX_RHOQ1 * ne] / rho) : eos_p_of_rt(rho_theta)) - p0[q];
    });
}

}  // namespace erfx

namespace erfx {

// Copy n doubles, 16 bytes per lane where both ends share their offset within
// 16 bytes (a field allocated with its rows shifted onto cache lines starts 8
// bytes into a 16-byte unit: its first double is then copied on its own), 8
// bytes per lane otherwise.  `first`/`stride` are the lane's index and the
// grid's width in lanes.
__device__ __forceinline__ void copy_span(double* dst, const double* src, long n, long first, long stride) {
    const unsigned long long as = reinterpret_cast<unsigned long long>(src);
    const unsigned long long ad = reinterpret_cast<unsigned long long>(dst);
    if (((as ^ ad) & 15ull) != 0) {
        for (long t = first; t < n; t += stride) dst[t] = src[t];
        return;
    }
    const long lead = (as & 15ull) ? 1 : 0;
    if (lead && first == 0 && n > 0) dst[0] = src[0];
    const long n2 = (n - lead) / 2;
    const double2* s2 = reinterpret_cast<const double2*>(src + lead);
    double2* d2 = reinterpret_cast<double2*>(dst + lead);
    for (long t = first; t < n2; t += stride) d2[t] = s2[t];
    const long tail = lead + 2 * n2;
    if (tail < n && first == 0) dst[tail] = src[tail];
}

__global__ void __launch_bounds__(256) copy_kernel(CopyList c) {
    const long stride = (long)gridDim.x * 256;
    for (int a = 0; a < c.count; ++a) copy_span(c.dst[a], c.src[a], c.n[a], (long)blockIdx.x * 256 + threadIdx.x, stride);
}

// batched form: each member's lists copied by its own range of work-groups
struct CopyItem {
    BHdr h;
    CopyList c;
};
__global__ void __launch_bounds__(256) copy_kernel_batch(const CopyItem* __restrict__ it,
                                                         const unsigned* __restrict__ starts, int n) {
    const CopyItem& m = batch_member(it, starts, n, blockIdx.x);
    const BHdr h = m.h;
    const CopyList& c = m.c;
    const long stride = (long)h.tiles * 256;
    const long first = (long)(blockIdx.x - h.t0) * 256 + threadIdx.x;
    for (int a = 0; a < c.count; ++a) copy_span(c.dst[a], c.src[a], c.n[a], first, stride);
}
static void copy_batch(const void* items, const unsigned* starts, int n, unsigned total, unsigned width,
                       hipStream_t s) {
    (void)width;
    hipLaunchKernelGGL(copy_kernel_batch, dim3(total), dim3(256), 0, s, static_cast<const CopyItem*>(items), starts,
                       n);
}

void copy_fields(const CopyList& c, hipStream_t s) {
    if (g_rec) {
        long nmax = 0;
        for (int a = 0; a < c.count; ++a) nmax = c.n[a] > nmax ? c.n[a] : nmax;
        const long want = (nmax / 2 + 255) / 256;
        CopyItem it{{{0, 0, 0}, {0, 0, 0}, 1u, 1u, 0u, (unsigned)(want < 1024 ? want : 1024)}, c};
        if (c.count == 0) it.h.tiles = 0;
        rec_push(&copy_batch, 256u, it);
        return;
    }
    if (c.count == 0) return;
    hipLaunchKernelGGL(copy_kernel, dim3(4096), dim3(256), 0, s, c);
}

}  // namespace erfx
