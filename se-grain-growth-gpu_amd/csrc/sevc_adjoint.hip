// sevc_adjoint.hip -- topology-fixed windows and their adjoint (extension).
//
// Within a window the topology is held fixed (no T1/T2/nucleation), dt is
// the fixed opts.dt and the velocity is the analytic model
//   x_{n+1} = dom_mod(x_n + dt * mu * F(x_n)),   F = -grad E,
//   E = sum_b gamma_b L_b + sum_g SE_g |A_g|,    gamma_b = e_b * GB_scaling.
// The reverse pass runs lambda_n = J_n^T lambda_{n+1} with
// J_n = I - dt mu H(x_n) (H the Hessian of E; dom_mod has derivative 1), and
// accumulates the parameter terms lambda_{n+1} . dx_{n+1}/dtheta.
//
// Every kernel takes the positions it works on explicitly (a checkpoint or
// a slot of the segment buffer), one lane per vertex / grain / edge, and
// evaluates the same operations in the same order as the oracle's
// orc_window_forward / orc_adjoint_window, so results are bit-identical.
#include <hip/hip_runtime.h>
#include "sevc_dev.h"

namespace sevc {

// Boundary energies for the window (compute_boundary_energies,
// calculus.h:104-114).
__global__ void k_win_prepare(Dev d) {
    TABLE_BLOCK(d.eblk, d.neb)
    if (i >= bd_.e || !d.benab[i]) return;
    const double e = (P.gb_eps == 0.0) ? 1.0 : boundary_compute_energy(d, i, P.gb_eps);
    d.ben[i] = e * P.gb_scaling;
}

// The window's topology is fixed, so what every step would look up again
// (a vertex's edges, their far ends, its place in its three grains' lists,
// the list neighbours there) is looked up once per window and kept in
// vertex order:
//   nbr[v]  (w0, w1, w2, code): the far ends of the vertex's edges and, per
//           grain slot j, which of them are the list's previous and next
//           vertex (code bits 4j..4j+1 and 4j+2..4j+3) and whether the slot
//           counts at all (bit 12 + j: the vertex is in the list and the
//           list has 3 entries or more); kWinOn: an enabled vertex;
//           kWinSearch: a list neighbour is not the end of one of the
//           vertex's edges (the steps then search the lists)
//   vse[j V + v]  stored energy of grain slot j
//   veb[j V + v]  d gamma_b / d GB_scaling of edge j (null when every member
//           has GB_eps = 0, where it is 1)
// and the grains' lists in one of two ways.  Where the vertices are ordered
// along the mesh (win_own_rule), a table block's 256 vertices have about 160
// grains between them, and the step's workgroup forms their area signs itself:
//   wb.count[lb]  grains at the enabled vertices of block lb, at most kWinGrains
//   wb.grain[lb kWinGrains + k]  the k-th one and its list's length (-1: disabled)
//   wb.list[(kq nvb + lb) kWinGrains + k]  entries 4 kq .. 4 kq + 3 of its list
//   wb.loc[v]  the block's numbers of the vertex's three grains, 10 bits each
// Each grain's area is then formed by 1.3 workgroups on average, but a step is
// one launch and its two chains of loads run side by side: 10,000 grains 6.2 us
// a step (areas 4.3 and step 4.7 as two launches), 40,000 8.2 (11.3); 16 members
// of 11,000 the same 20.  Otherwise
//   wl[kq G + g], wn[g]  the same per grain, for a launch of k_win_area per step.
constexpr int kWinOn = 1 << 16, kWinSearch = 1 << 15;
constexpr int kWinList = 12;                 // list entries held in the table (longer lists are read on)
constexpr int kWinGrains = kWinBlockGrains;
static_assert(kWinGrains == 3 * kBlock && kWinGrains <= 1024, "three grains a vertex, numbered in 10 bits");

__device__ __forceinline__ void win_list4(const Dev& d, int g, int n, int q, int (&e)[4]) {
    const int* L = glist(d, g);
#pragma unroll
    for (int r = 0; r < 4; r++) e[r] = 4 * q + r < n ? L[4 * q + r] : 0;
}

__global__ void __launch_bounds__(kBlock) k_win_table_v(Dev d, int4* nbr, double* vse, double* veb, WinBlocks wb) {
    TABLE_BLOCK(d.vblk, d.nvb)
    const int v = i;
    const bool in = i < bd_.e, on = in && d.ven[v] != 0;
    int vg[3] = {0, 0, 0};
    if (in && !on) nbr[v] = make_int4(v, v, v, 0);
    if (on) {
        int w[3], code = kWinOn;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int b = d.vb[3 * v + j];
            w[j] = other_end(d, b, v);
            if (veb) veb[(size_t)j * d.V + v] = (P.gb_eps == 0.0) ? 1.0 : boundary_compute_energy(d, b, P.gb_eps);
        }
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int g = d.vg[3 * v + j];
            const int n = d.glen[g];
            const int k = grain_contains_vertex(d, g, v);
            vg[j] = g;
            vse[(size_t)j * d.V + v] = d.gse[g];
            if (k < 0 || n < 3) continue;
            const int* L = glist(d, g);
            const int wp = L[(k + n - 1) % n], wn = L[(k + 1) % n];
            const int ip = wp == w[0] ? 0 : (wp == w[1] ? 1 : (wp == w[2] ? 2 : 3));
            const int in = wn == w[0] ? 0 : (wn == w[1] ? 1 : (wn == w[2] ? 2 : 3));
            if (ip == 3 || in == 3) code |= kWinSearch;
            code |= (ip << (4 * j)) | (in << (4 * j + 2)) | (1 << (12 + j));
        }
        nbr[v] = make_int4(w[0], w[1], w[2], code);
    }
    if (!wb.loc) return;
    // the block's grains, numbered by a table of the grains met so far
    constexpr int kSlots = 2048;
    __shared__ int key[kSlots], num[kSlots], met[kWinGrains], n_met;
    for (int h = (int)threadIdx.x; h < kSlots; h += kBlock) key[h] = -1;
    if (threadIdx.x == 0) n_met = 0;
    __syncthreads();
    int at[3] = {0, 0, 0};
    if (on)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            int h = (int)(((unsigned)vg[j] * 2654435761u) >> 16) & (kSlots - 1);
            for (;; h = (h + 1) & (kSlots - 1)) {
                const int was = atomicCAS(&key[h], -1, vg[j]);
                if (was == -1) {
                    num[h] = atomicAdd(&n_met, 1);
                    met[num[h]] = vg[j];
                }
                if (was == -1 || was == vg[j]) break;
            }
            at[j] = h;
        }
    __syncthreads();
    if (in) wb.loc[v] = on ? num[at[0]] | (num[at[1]] << 10) | (num[at[2]] << 20) : 0;
    const int n = n_met;
    if (threadIdx.x == 0) wb.count[lb_] = n;
    for (int k = (int)threadIdx.x; k < n; k += kBlock) {
        const int g = met[k], len = d.genab[g] ? d.glen[g] : -1;
        wb.grain[(size_t)lb_ * kWinGrains + k] = make_int2(g, len);
#pragma unroll
        for (int q = 0; q < kWinList / 4; q++) {
            int e[4];
            win_list4(d, g, len, q, e);
            wb.list[((size_t)q * d.nvb + lb_) * kWinGrains + k] = make_int4(e[0], e[1], e[2], e[3]);
        }
    }
}

__global__ void k_win_table_g(Dev d, int4* wl, int* wn) {
    TABLE_BLOCK(d.gblk, d.ngb)
    if (i >= bd_.e) return;
    const int n = d.genab[i] ? d.glen[i] : -1;
    wn[i] = n;
#pragma unroll
    for (int q = 0; q < kWinList / 4; q++) {
        int e[4];
        win_list4(d, i, n, q, e);
        wl[(size_t)q * d.G + i] = make_int4(e[0], e[1], e[2], e[3]);
    }
}

// Area of grain g (list length n > 0, its first entries in L) at positions X
// (compute_grain_areas, calculus.h:224-234).
__device__ __forceinline__ double win_area(const Dev& d, const double2* X2, int g, int n, const int (&L)[kWinList], double D) {
    double2 p[kWinList];
#pragma unroll
    for (int k = 0; k < kWinList; k++) p[k] = k < n ? X2[L[k]] : make_double2(0.0, 0.0);
    if (n <= 0) return 0.0;
    AreaAcc acc;
    acc.start(p[0].x, p[0].y);
#pragma unroll
    for (int k = 1; k < kWinList; k++)
        if (k < n) acc.push(p[k].x, p[k].y, D);
    if (n > kWinList) {
        const int* Lg = glist(d, g);
        for (int k = kWinList; k < n; k++) {
            const double2 q = X2[Lg[k]];
            acc.push(q.x, q.y, D);
        }
    }
    return acc.finish();
}

// Signs of the grain areas at positions X (the analytic force needs no more of
// them): neg[g] = 1 for a negative area, where the steps' workgroups do not form
// them themselves (wl given).  The areas go to `area` when given (the last step
// of the window's forward leaves them in the state).
__global__ void k_win_area(Dev d, const double* X, const int4* wl, const int* wn, uint8_t* neg, double* area) {
    TABLE_BLOCK(d.gblk, d.ngb)
    if (i >= bd_.e) return;
    const int n = wl ? wn[i] : (d.genab[i] ? d.glen[i] : -1);
    int L[kWinList];
#pragma unroll
    for (int q = 0; q < kWinList / 4; q++) {
        int e[4];
        if (wl) {
            const int4 t = wl[(size_t)q * d.G + i];
            e[0] = t.x; e[1] = t.y; e[2] = t.z; e[3] = t.w;
        } else {
            win_list4(d, i, n, q, e);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) L[4 * q + r] = e[r];
    }
    if (n < 0) return;
    const double a = win_area(d, reinterpret_cast<const double2*>(X), i, n, L, P.D);
    if (neg) neg[i] = a < 0 ? 1 : 0;
    if (area) area[i] = a;
}

// The list neighbours (previous, next) of v in its grain slot j, by search
// (kWinSearch vertices only).
__device__ __forceinline__ void win_search(const Dev& d, int v, int g, int* wp, int* wn) {
    const int n = d.glen[g], k = grain_contains_vertex(d, g, v);
    const int* L = glist(d, g);
    *wp = L[(k + n - 1) % n];
    *wn = L[(k + 1) % n];
}

// One of three values by a run-time index, by selects on values (indexing an
// array would put it into LDS or scratch).
__device__ __forceinline__ double2 pick3(double2 a, double2 b, double2 c, int k) {
    const double x = k == 0 ? a.x : (k == 1 ? b.x : c.x), y = k == 0 ? a.y : (k == 1 ? b.y : c.y);
    return make_double2(x, y);
}

// One window step x_n -> x_{n+1}: analytic velocity (calculus.h:143-154
// with the analytic model, the sums of analytic_force_at) and
// update_vertices_positions (calculus.h:391-404), written to a separate
// array so that neighbours still read x_n.  Disabled slots are copied.  The
// area signs of the vertex's three grains go to sgn, for the reverse step.
// kOwn: the workgroup forms them itself from its block's lists (wb), else they
// are in neg.  A step at 10,000 grains or fewer is bound by the latency of its
// launches and loads (an empty launch takes 4.5 us in a busy stream), so the
// areas' lists are read unconditionally, with the vertices' own data, and both
// gathers of positions are in flight together.
template <bool kOwn>
__global__ void __launch_bounds__(kBlock) k_win_step(Dev d, const double* X, const uint8_t* neg, WinBlocks wb,
                                                     const int4* nbr, const double* vse, const double* veb, double* Xn,
                                                     uint8_t* sgn, int write_vel) {
    TABLE_BLOCK(d.vblk, d.nvb)
    __shared__ uint8_t own[kOwn ? kWinGrains : 1];
    const bool in = i < bd_.e;
    const double2* X2 = reinterpret_cast<const double2*>(X);
    const int iv = in ? i : bd_.b;
    const int4 t = nbr[iv];
    const double2 p = X2[iv];
    double se[3], eb[3];
    uint8_t ng[3];
#pragma unroll
    for (int j = 0; j < 3; j++) {
        se[j] = vse[(size_t)j * d.V + iv];
        eb[j] = veb ? veb[(size_t)j * d.V + iv] : 1.0;
    }
    double2 q[3];
    if (kOwn) {
        const int loc = wb.loc[iv], n_own = wb.count[lb_];
        const size_t row = (size_t)lb_ * kWinGrains, qs = (size_t)d.nvb * kWinGrains;
        int k = (int)threadIdx.x;
        int2 gn = wb.grain[row + k];
        int4 l[kWinList / 4];
#pragma unroll
        for (int r = 0; r < kWinList / 4; r++) l[r] = wb.list[r * qs + row + k];
        q[0] = X2[t.x]; q[1] = X2[t.y]; q[2] = X2[t.z];
        while (k < n_own) {
            int L[kWinList];
#pragma unroll
            for (int r = 0; r < kWinList / 4; r++) {
                L[4 * r] = l[r].x; L[4 * r + 1] = l[r].y; L[4 * r + 2] = l[r].z; L[4 * r + 3] = l[r].w;
            }
            own[k] = win_area(d, X2, gn.x, gn.y, L, P.D) < 0 ? 1 : 0;
            k += kBlock;
            if (k >= n_own) break;
            gn = wb.grain[row + k];
#pragma unroll
            for (int r = 0; r < kWinList / 4; r++) l[r] = wb.list[r * qs + row + k];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 3; j++) ng[j] = own[(loc >> (10 * j)) & 1023];
    } else {
        int g[3];
#pragma unroll
        for (int j = 0; j < 3; j++) g[j] = d.vg[3 * iv + j];
        q[0] = X2[t.x]; q[1] = X2[t.y]; q[2] = X2[t.z];
#pragma unroll
        for (int j = 0; j < 3; j++) ng[j] = (t.w & kWinOn) ? neg[g[j]] : 0;
    }
    if (!in) return;
    if (!(t.w & kWinOn)) {
        reinterpret_cast<double2*>(Xn)[i] = p;
        return;
    }
    sgn[i] = (uint8_t)(ng[0] | (ng[1] << 1) | (ng[2] << 2));
    const double D = P.D, x = p.x, y = p.y;
    double ex = 0.0, ey = 0.0, gx = 0.0, gy = 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const double dx = wrapd(x, q[j].x, D), dy = wrapd(y, q[j].y, D);
        const double L = mag(dx, dy);
        const double gam = eb[j] * P.gb_scaling;
        if (L > 0) {
            ex += gam * (dx / L);
            ey += gam * (dy / L);
        }
    }
#pragma unroll
    for (int j = 0; j < 3; j++) {
        if (!((t.w >> (12 + j)) & 1)) continue;
        double2 a, b;
        if (t.w & kWinSearch) {
            int wp, wn;
            win_search(d, i, d.vg[3 * i + j], &wp, &wn);
            a = X2[wp];
            b = X2[wn];
        } else {
            a = pick3(q[0], q[1], q[2], (t.w >> (4 * j)) & 3);
            b = pick3(q[0], q[1], q[2], (t.w >> (4 * j + 2)) & 3);
        }
        const double dpx = wrapd(x, a.x, D), dpy = wrapd(y, a.y, D);
        const double dnx = wrapd(b.x, x, D), dny = wrapd(b.y, y, D);
        const double sg = ng[j] ? -1.0 : 1.0;
        const double c = se[j] * sg * 0.5;
        gx += c * (dpy + dny);
        gy += c * (-(dpx + dnx));
    }
    const double vx = -(ex + gx) * P.mobility, vy = -(ey + gy) * P.mobility;
    if (write_vel) reinterpret_cast<double2*>(d.vel)[i] = make_double2(vx, vy);
    double xn = x, yn = y;
    xn += vx * P.dt_max;
    yn += vy * P.dt_max;
    reinterpret_cast<double2*>(Xn)[i] = make_double2(dom_mod(xn, D), dom_mod(yn, D));
}

// Window end: step counter and time as k_end advances them per step.
__global__ void k_win_end(Dev d, int steps) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= d.B) return;
    const Params& P = d.prm[m];
    MState& M = d.ms[m];
    for (int k = 0; k < steps; k++) {
        M.n += 1;
        if (P.adaptive) M.t += P.dt_max;
        else M.t = M.n * P.dt_max;
    }
}

// lambda <- 0 on disabled slots; accumulators <- 0.
__global__ void k_win_init(Dev d, double* lam, double* acc_mu, double* acc_s, double* acc_se) {
    TABLE_BLOCK(d.vblk, d.nvb)
    if (i >= bd_.e) return;
    if (!d.ven[i]) {
        lam[2 * i] = 0.0;
        lam[2 * i + 1] = 0.0;
    }
    acc_mu[i] = 0.0;
    acc_s[i] = 0.0;
    for (int j = 0; j < 3; j++) acc_se[(size_t)j * d.V + i] = 0.0;
}

// One reverse step at vertex v, with lambda = dL/dx_{n+1} and the state
// x_n (positions X, area signs of the vertex's grains sgn):
//   lambda_n  = lambda - dt mu (H lambda)_v
//   acc_mu   += dt (lambda . F_v)
//   acc_s    += dt mu (lambda . dF_v/dGB_scaling),  dF_v/ds = -sum_b e_b u_b
//   acc_se_j += dt mu (lambda . dF_v/dSE_g),        dF_v/dSE_g = -sign(A_g) dA_g/dp_v
// An edge b to w (d = wrap(p_v - p_w), L = |d| > 0, u = d/L) adds
// (gamma_b / L)(I - u u^T)(lambda_v - lambda_w) to (H lambda)_v; a grain g
// with list neighbours prev, next adds
// SE_g sign(A_g)/2 (lambda_next.y - lambda_prev.y, lambda_prev.x - lambda_next.x).
__global__ void __launch_bounds__(kBlock) k_win_adjoint(Dev d, const double* X, const uint8_t* sgn, const int4* nbr,
                                                        const double* vse, const double* veb, const double* lam,
                                                        double* lam2, double* acc_mu, double* acc_s, double* acc_se) {
    TABLE_BLOCK(d.vblk, d.nvb)
    if (i >= bd_.e) return;
    const int v = i;
    const double2* X2 = reinterpret_cast<const double2*>(X);
    const double2* M2 = reinterpret_cast<const double2*>(lam);
    const int4 t = nbr[v];
    const double2 p = X2[v], l = M2[v];
    const int sb = sgn[v];
    double se[3], ebs[3], ase[3];
#pragma unroll
    for (int j = 0; j < 3; j++) {
        se[j] = vse[(size_t)j * d.V + v];
        ebs[j] = veb ? veb[(size_t)j * d.V + v] : 1.0;
        ase[j] = acc_se[(size_t)j * d.V + v];
    }
    const double am = acc_mu[v], as = acc_s[v];
    if (!(t.w & kWinOn)) {
        reinterpret_cast<double2*>(lam2)[v] = make_double2(0.0, 0.0);
        return;
    }
    const double2 q[3] = {X2[t.x], X2[t.y], X2[t.z]};
    const double2 m[3] = {M2[t.x], M2[t.y], M2[t.z]};
    const double D = P.D, mu = P.mobility, dt = P.dt_max, dtm = dt * mu;
    const double x = p.x, y = p.y;
    const double lx = l.x, ly = l.y;
    double ex = 0.0, ey = 0.0, gx = 0.0, gy = 0.0;
    double hex = 0.0, hey = 0.0, hgx = 0.0, hgy = 0.0, sx = 0.0, sy = 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const double dx = wrapd(x, q[j].x, D), dy = wrapd(y, q[j].y, D);
        const double L = mag(dx, dy);
        if (L > 0) {
            const double ux = dx / L, uy = dy / L;
            const double eb = ebs[j];
            const double gam = eb * P.gb_scaling;
            ex += gam * ux;
            ey += gam * uy;
            const double wx = lx - m[j].x, wy = ly - m[j].y;
            const double uw = ux * wx + uy * wy;
            const double c = gam / L;
            hex += c * (wx - ux * uw);
            hey += c * (wy - uy * uw);
            sx += eb * ux;
            sy += eb * uy;
        }
    }
#pragma unroll
    for (int j = 0; j < 3; j++) {
        if (!((t.w >> (12 + j)) & 1)) continue;
        double2 a, b, la, lb;
        if (t.w & kWinSearch) {
            int wp, wn;
            win_search(d, v, d.vg[3 * v + j], &wp, &wn);
            a = X2[wp];
            b = X2[wn];
            la = M2[wp];
            lb = M2[wn];
        } else {
            const int ip = (t.w >> (4 * j)) & 3, in = (t.w >> (4 * j + 2)) & 3;
            a = pick3(q[0], q[1], q[2], ip);
            b = pick3(q[0], q[1], q[2], in);
            la = pick3(m[0], m[1], m[2], ip);
            lb = pick3(m[0], m[1], m[2], in);
        }
        const double dpx = wrapd(x, a.x, D), dpy = wrapd(y, a.y, D);
        const double dnx = wrapd(b.x, x, D), dny = wrapd(b.y, y, D);
        const double sg = (sb >> j) & 1 ? -1.0 : 1.0;
        const double c = se[j] * sg * 0.5;
        gx += c * (dpy + dny);
        gy += c * (-(dpx + dnx));
        hgx += c * (lb.y - la.y);
        hgy += c * (la.x - lb.x);
        const double h = sg * 0.5;
        const double tse = -(lx * (h * (dpy + dny)) + ly * (h * (-(dpx + dnx))));
        acc_se[(size_t)j * d.V + v] = ase[j] + dtm * tse;
    }
    const double fx = -(ex + gx), fy = -(ey + gy);
    const double hx = hex + hgx, hy = hey + hgy;
    acc_mu[v] = am + dt * (lx * fx + ly * fy);
    acc_s[v] = as + dtm * (-(lx * sx + ly * sy));
    reinterpret_cast<double2*>(lam2)[v] = make_double2(lx - dtm * hx, ly - dtm * hy);
}

template __global__ void k_win_step<false>(Dev, const double*, const uint8_t*, WinBlocks, const int4*, const double*,
                                           const double*, double*, uint8_t*, int);
template __global__ void k_win_step<true>(Dev, const double*, const uint8_t*, WinBlocks, const int4*, const double*,
                                          const double*, double*, uint8_t*, int);

// Level 1 of the deterministic parameter sums: one lane per 256-vertex
// table block sums its enabled slots left to right (the chunks of the
// oracle's orc_sum_chunked).  part[lb] for mu, part[2*nvb + lb] for s.
__global__ void k_win_sum_l1(Dev d, const double* acc_mu, const double* acc_s, double* part) {
    const int lb = blockIdx.x * blockDim.x + threadIdx.x;
    if (lb >= d.nvb) return;
    const Blk bd = d.vblk[lb];
    double a = 0.0, b = 0.0;
    for (int v = bd.b; v < bd.e; v++)
        if (d.ven[v]) {
            a += acc_mu[v];
            b += acc_s[v];
        }
    part[lb] = a;
    part[2 * d.nvb + lb] = b;
}

// Upper levels per member (chunks of 256 partials left to right until one
// remains), one workgroup per member and quantity (blockIdx.y); levels
// alternate between two halves so no lane overwrites a value still read.
// out[2m] = dL/dGB_scaling, out[2m+1] = dL/dmobility.
__global__ void k_win_sum_up(Dev d, double* part, double* out) {
    const int m = blockIdx.x, which = blockIdx.y;      // 0: mu, 1: s
    if (m >= d.B) return;
    const int first = d.vblk_first[m];
    int cnt = d.vblk_first[m + 1] - first;
    double* src = part + 2 * (size_t)d.nvb * which + first;
    double* dst = src + d.nvb;
    while (cnt > 1) {
        const int nn = (cnt + 255) / 256;
        for (int c = threadIdx.x; c < nn; c += blockDim.x) {
            double s = 0.0;
            const int e = (c + 1) * 256 < cnt ? (c + 1) * 256 : cnt;
            for (int q = c * 256; q < e; q++) s += src[q];
            dst[c] = s;
        }
        __syncthreads();
        double* t = src;
        src = dst;
        dst = t;
        cnt = nn;
    }
    if (threadIdx.x == 0) out[2 * m + (which == 0 ? 1 : 0)] = cnt == 1 ? src[0] : 0.0;
}

// dL/dSE_g: the grain's vertices' terms summed in list order.
__global__ void k_win_dse(Dev d, const double* acc_se, double* dse) {
    TABLE_BLOCK(d.gblk, d.ngb)
    if (i >= bd_.e) return;
    double r = 0.0;
    if (d.genab[i]) {
        const int* L = glist(d, i);
        for (int k = 0; k < d.glen[i]; k++) {
            const int v = L[k];
            for (int j = 0; j < 3; j++)
                if (d.vg[3 * v + j] == i) {
                    r += acc_se[(size_t)j * d.V + v];
                    break;
                }
        }
    }
    dse[i] = r;
}

}  // namespace sevc

namespace sevc {

// ---------------------------------------------------------------------
// smooth area histogram loss (calibration), on the device
// ---------------------------------------------------------------------
//
// Member m: c_k = a_min + (k + 1/2)(a_max - a_min)/nb, width w,
//   h_k = (1/G) sum_g exp(-z_gk^2 / 2),  z_gk = (|A_g| - c_k)/w,
//   L   = sum_k (h_k - t_k)^2,
// over its enabled grains with at least 3 vertices (G of them).  Sums run in
// a fixed order (grain index within 256-grain blocks, then blocks), so the
// result does not depend on scheduling.

__device__ __forceinline__ double hist_centre(const double* rg, int nb, int k) {
    return rg[0] + (k + 0.5) * (rg[1] - rg[0]) / nb;
}

// Level 1: one workgroup per grain table block.  Stores the signed areas;
// part[lb*(nb+1) + k] = sum over the block's grains of exp(-z^2/2) for bin
// k, part[lb*(nb+1) + nb] = number of grains in the histogram.
__global__ void __launch_bounds__(256) k_hist_l1(Dev d, int nb, const double* ranges, double* hA, double* part) {
    __shared__ double a_s[kBlock];
    __shared__ unsigned char ok_s[kBlock];
    TABLE_BLOCK(d.gblk, d.ngb)
    const int t = threadIdx.x;
    const bool ok = i < bd_.e && d.genab[i] && d.glen[i] >= 3;
    double a = 0.0;
    if (ok) {
        a = grain_area_at(d, d.pos, i, P.D);
        hA[i] = a;
    } else if (i < bd_.e) {
        hA[i] = 0.0;
    }
    a_s[t] = fabs(a);
    ok_s[t] = ok ? 1 : 0;
    __syncthreads();
    const int n = bd_.e - bd_.b;
    const double* rg = ranges + 3 * bd_.m;
    if (t < nb) {
        const double c = hist_centre(rg, nb, t), w = rg[2];
        double s = 0.0;
        for (int q = 0; q < n; q++)
            if (ok_s[q]) {
                const double z = (a_s[q] - c) / w;
                s += sevc_exp(-0.5 * (z * z));
            }
        part[(size_t)lb_ * (nb + 1) + t] = s;
    } else if (t == nb) {
        int cnt = 0;
        for (int q = 0; q < n; q++) cnt += ok_s[q];
        part[(size_t)lb_ * (nb + 1) + nb] = cnt;
    }
}

// Level 2: one workgroup per member.  hist[m*nb+k] = h_k, res[m*nb+k] =
// h_k - t_k, loss[m] = sum_k (h_k - t_k)^2, gcount[m] = G.
__global__ void k_hist_member(Dev d, int nb, const double* part, const double* targets, double* hist, double* res,
                              double* loss, double* gcount) {
    __shared__ double r_s[kMaxHistBins];
    __shared__ double g_s;
    const int m = blockIdx.x;
    if (m >= d.B) return;
    const int first = d.gblk_first[m], cnt = d.gblk_first[m + 1] - first;
    const int t = threadIdx.x;
    if (t == nb) {
        double g = 0.0;
        for (int b = first; b < first + cnt; b++) g += part[(size_t)b * (nb + 1) + nb];
        g_s = g;
    }
    __syncthreads();
    if (t < nb) {
        double s = 0.0;
        for (int b = first; b < first + cnt; b++) s += part[(size_t)b * (nb + 1) + t];
        const double G = g_s > 0 ? g_s : 1.0;
        const double h = s / G;
        const double r = h - targets[(size_t)m * nb + t];
        hist[(size_t)m * nb + t] = h;
        res[(size_t)m * nb + t] = r;
        r_s[t] = r;
    }
    __syncthreads();
    if (t == 0) {
        double L = 0.0;
        for (int k = 0; k < nb; k++) L += r_s[k] * r_s[k];
        loss[m] = L;
        gcount[m] = g_s;
    }
}

// Per grain: wg = dL/dA_g = sign(A_g) sum_k 2 r_k exp(-z^2/2) (-z/w) / G.
__global__ void k_hist_weight(Dev d, int nb, const double* ranges, const double* hA, const double* res,
                              const double* gcount, double* wg) {
    TABLE_BLOCK(d.gblk, d.ngb)
    if (i >= bd_.e) return;
    if (!(d.genab[i] && d.glen[i] >= 3)) {
        wg[i] = 0.0;
        return;
    }
    const double* rg = ranges + 3 * bd_.m;
    const double* r = res + (size_t)bd_.m * nb;
    const double a = fabs(hA[i]), w = rg[2];
    const double G = gcount[bd_.m] > 0 ? gcount[bd_.m] : 1.0;
    double s = 0.0;
    for (int k = 0; k < nb; k++) {
        const double z = (a - hist_centre(rg, nb, k)) / w;
        s += 2.0 * r[k] * sevc_exp(-0.5 * (z * z)) * (-z / w);
    }
    s = s / G;
    wg[i] = hA[i] < 0 ? -s : s;
}

// Per vertex: dL/dp_v = sum over its grains of wg * dA_g/dp_v with
// dA/dx_v = (dy_prev + dy_next)/2, dA/dy_v = -(dx_prev + dx_next)/2.
__global__ void k_hist_seed(Dev d, const double* wg, double* seed) {
    TABLE_BLOCK(d.vblk, d.nvb)
    if (i >= bd_.e) return;
    const int v = i;
    double gx = 0.0, gy = 0.0;
    if (d.ven[v]) {
        const double D = P.D, x = d.pos[2 * v], y = d.pos[2 * v + 1];
        for (int j = 0; j < 3; j++) {
            const int g = d.vg[3 * v + j];
            const int n = d.glen[g];
            const int k = grain_contains_vertex(d, g, v);
            if (k < 0 || n < 3 || !d.genab[g]) continue;
            const int* L = glist(d, g);
            const int wp = L[(k + n - 1) % n], wn = L[(k + 1) % n];
            const double dpx = wrapd(x, d.pos[2 * wp], D), dpy = wrapd(y, d.pos[2 * wp + 1], D);
            const double dnx = wrapd(d.pos[2 * wn], x, D), dny = wrapd(d.pos[2 * wn + 1], y, D);
            const double c = wg[g] * 0.5;
            gx += c * (dpy + dny);
            gy += c * (-(dpx + dnx));
        }
    }
    seed[2 * v] = gx;
    seed[2 * v + 1] = gy;
}

}  // namespace sevc
