// tangent.hpp -- the fused tangent residual (JVP): values and tangents of
// FiniteVolume<Ibis::dual>::compute_dudt (src/solvers/solvers/
// steady_state.cpp:52-128) in three kernels, four when viscous.
//
// Included by residual.hip after the forward kernels, inside its anonymous
// namespace (it uses DevMesh, VarSet, FaceParams, ViscParams and the
// general path's device functions).
//
//   k_tan_state  the (value, tangent) pairs of the state: from prim and its
//                tangent, or from the conserved state and a Krylov vector;
//                a ghost's thread converts its valid cell itself and runs
//                both lists of boundary actions in registers
//   k_tan_cell   per tile: viscous gradients, then per reconstruction
//                variable the LSQ gradient, the limiter and the value on
//                each face of the cell
//   k_tan_visc   per face: the viscous terms (visc_face)
//   k_tan_face   per tile: every face's flux once, then the cells' sums, and
//                for a matvec vec / dt* - J vec directly
//
// Every expression is the general path's on ibis::Dual (run_general), in its
// order, so both give the same bits; what is saved is the passes over memory
// between its eight to eleven kernels: the gradients, limiters and fluxes
// of the pairs never go to memory, the face values (5 pairs per cell and
// face) go once.
#ifndef IBIS_TANGENT_HPP
#define IBIS_TANGENT_HPP

// where the state and its tangent come from
struct TanSource {
    const double* a;   // prim rows (7 x Nt), or the conserved rows ((dim+2) x Nt)
    const double* ad;  // prim_dot rows, or the Krylov vector (cell * (dim+2) + q)
    double R, Cv;
};

// the accessor of the boundary actions on register rows
struct TanGhost {
    ibis::Dual va[NPRIM], gr[NPRIM];
    __device__ __forceinline__ ibis::Dual v(int row) const { return va[row]; }
    __device__ __forceinline__ ibis::Dual g(int row) const { return gr[row]; }
    __device__ __forceinline__ void set(int row, ibis::Dual x) { gr[row] = x; }
};

// the primitive rows of cell c as k_to_dual, or k_seed_cons and
// k_cons_to_prim, give them (a ghost's conserved row is seeded with zero)
template <int DIM, bool CONS>
__device__ __forceinline__ void tan_load(const DevMesh& m, const TanSource& s, int c,
                                         ibis::Dual (&out)[NPRIM]) {
    if (CONS) {
        constexpr int NC = DIM + 2;
        ibis::Dual q[NC];
#pragma unroll
        for (int k = 0; k < NC; k++)
            q[k] = c < m.N ? ibis::Dual(s.a[(size_t)k * m.Nt + c], s.ad[(size_t)c * NC + k])
                           : ibis::Dual(0.0, 0.0);
        ibis::cons_to_prim_cell<ibis::Dual, DIM>(q, s.R, s.Cv, out);
    } else {
#pragma unroll
        for (int k = 0; k < NPRIM; k++)
            out[k] = ibis::Dual(s.a[(size_t)k * m.Nt + c], s.ad[(size_t)k * m.Nt + c]);
    }
}

// One thread per cell, ghosts included.  gpre (7 x G): the ghosts after the
// pre-reconstruction actions, which the convective part reads; prim's ghost
// rows end as after the viscous actions.  FL (null without reconstruction):
// the ghosts' face values.
template <int DIM, bool CONS>
__global__ void __launch_bounds__(BLOCK)
    k_tan_state(DevMesh m, TanSource s, const int* __restrict__ kinds,
                const double* __restrict__ pars, int ntab, int has_pre, int has_visc, GasParams gp,
                VarSet vs, ibis::Dual* __restrict__ prim, ibis::Dual* __restrict__ gpre,
                ibis::Dual* __restrict__ FL) {
    const int c = blockIdx.x * BLOCK + threadIdx.x;
    const int N = m.N, Nt = m.Nt, F = m.F, G = m.G;
    if (c >= Nt) return;
    TanGhost X;
    tan_load<DIM, CONS>(m, s, c, X.gr);
    const int b = c < N ? -1 : m.b_of_ghost[c - N];
    if (b < 0) {  // a valid cell, or a ghost that nothing reaches
#pragma unroll
        for (int k = 0; k < NPRIM; k++) prim[(size_t)k * Nt + c] = X.gr[k];
        return;
    }
    const int f = m.b_face[b], t = m.b_tag[b];
    tan_load<DIM, CONS>(m, s, m.b_valid[b], X.va);
    if (has_pre) bc_actions_on<ibis::Dual>(m, kinds, pars, gp, f, t, X);
#pragma unroll
    for (int k = 0; k < NPRIM; k++) gpre[(size_t)k * G + (c - N)] = X.gr[k];
    if (FL) {  // lin_interp of a ghost: no gradient, limiter 1
        const double dx = m.geom[9 * (size_t)F + f] - m.cen[c];
        const double dy = m.geom[10 * (size_t)F + f] - m.cen[Nt + c];
        const double dz = m.geom[11 * (size_t)F + f] - m.cen[2 * (size_t)Nt + c];
        const ibis::Dual gx(0.0), gy(0.0), gz(0.0);
#pragma unroll
        for (int v = 0; v < 5; v++) {
            ibis::Dual u = X.gr[0];  // a select chain keeps the rows in registers
#pragma unroll
            for (int k = 1; k < NPRIM; k++)
                if (vs.row[v] == k) u = X.gr[k];
            FL[soa_index(m, c, 0, v)] = u + ibis::Dual(1.0) * (gx * dx + gy * dy + gz * dz);
        }
    }
    if (has_visc)
        bc_actions_on<ibis::Dual>(m, kinds + ntab, pars + (size_t)ntab * IBIS_NPAR, gp, f, t, X);
#pragma unroll
    for (int k = 0; k < NPRIM; k++) prim[(size_t)k * Nt + c] = X.gr[k];
}

// faces of a cell that the tangent's cell kernel unrolls over
template <int DIM>
constexpr int tan_maxf() {
    return DIM == 2 ? 4 : MAXF;
}
// LDS of k_tan_cell: the staged variables of one phase (pairs) and the
// centroids of the tile's stencil
size_t tan_cell_lds(const DevMesh& D, bool recon) {
    return (size_t)(D.tile + D.maxhalo) * ((recon ? 5 : 4) * sizeof(ibis::Dual) + 3 * sizeof(double));
}

// One block per tile, one thread per cell.  The stencil goes to LDS in two
// phases that share its space, first T, vx, vy, vz for the viscous gradients
// (VISC), then the reconstruction variables (RECON); pairs of all nine at
// once would take 83 KB in 3D and leave one block per CU.  The LSQ weights
// and the face offsets are formed once and kept in registers, and the
// variables are worked through one after the other, so that only one
// variable's gradient, extremes and limiter (14 doubles of pairs) are live
// beside them: all five together would be 60.
template <int DIM, int LIM, bool RECON, bool VISC>
__global__ void __launch_bounds__(MAXTILE)
    k_tan_cell(DevMesh m, VarSet vs, const ibis::Dual* __restrict__ prim,
               const ibis::Dual* __restrict__ gpre, ibis::Dual* __restrict__ grad, double eps,
               double venkat_K, int freeze, const double* __restrict__ offs,
               ibis::Dual* __restrict__ FL) {
    extern __shared__ double soff[];
    using ibis::Dual;
    constexpr int MF = tan_maxf<DIM>();
    const int lb = xcd_block(m.ntiles);
    if (lb >= m.ntiles) return;
    const int TS = m.tile, N = m.N, Nt = m.Nt, G = m.G, SS = TS + m.maxhalo;
    const int i = lb * TS + threadIdx.x;
    const int il = i < N ? i : 0;  // past the last cell: cell 0's inputs, not used
    Dual* su = reinterpret_cast<Dual*>(soff);
    double* sc = soff + (size_t)2 * (RECON ? 5 : 4) * SS;
    const bool zflat = DIM == 2 && m.flat_z;
    const int h0 = m.halo_off[lb], nh = m.halo_off[lb + 1] - h0;
    const int nf = m.nfaces[il];
    int kst[MF];
#pragma unroll
    for (int j = 0; j < MF; j++) kst[j] = j < m.maxf ? m.nbr_lds[(size_t)j * N + il] : 0;
    const int vrow[4] = {P_T, P_VX, P_VY, P_VZ};
    auto put = [&](int k, int c, bool visc, bool first) {
        if (first) {
            sc[k] = m.cen[c];
            sc[SS + k] = m.cen[Nt + c];
            sc[2 * SS + k] = zflat ? 0.0 : m.cen[2 * (size_t)Nt + c];
        }
        if (visc) {
#pragma unroll
            for (int q = 0; q < 4; q++) su[q * SS + k] = prim[(size_t)vrow[q] * Nt + c];
        } else {
#pragma unroll
            for (int v = 0; v < 5; v++)
                su[v * SS + k] = VISC && c >= N ? gpre[(size_t)vs.row[v] * G + (c - N)]
                                                : prim[(size_t)vs.row[v] * Nt + c];
        }
    };
    auto stage = [&](bool visc, bool first) {
        if (i < N) put(threadIdx.x, i, visc, first);
        for (int k = threadIdx.x; k < nh; k += TS) put(TS + k, m.halo_ids[h0 + k], visc, first);
        __syncthreads();
    };
    stage(VISC, true);
    // LSQ weights of the cell's neighbours (k_cell_grad_var's expressions;
    // the factors from the staged centroids when the mesh's equal them)
    const double xi = sc[threadIdx.x], yi = sc[SS + threadIdx.x], zi = sc[2 * SS + threadIdx.x];
    double w[MF][3];
    {
        double r11 = 1.0, r12 = 0.0, r22 = 1.0, r13 = 0.0, r23 = 0.0, r33 = 0.0;
        if (m.lsq_from_cen) {
            double sxx = 0.0, sxy = 0.0, sxz = 0.0, syy = 0.0, syz = 0.0, szz = 0.0;
#pragma unroll
            for (int j = 0; j < MF; j++) {
                if (j < nf) {
                    const double dx = sc[kst[j]] - xi;
                    const double dy = sc[SS + kst[j]] - yi;
                    const double dz = sc[2 * SS + kst[j]] - zi;
                    sxx += dx * dx;
                    sxy += dx * dy;
                    sxz += dx * dz;
                    syy += dy * dy;
                    syz += dy * dz;
                    szz += dz * dz;
                }
            }
            r11 = sqrt(sxx);
            r12 = 1.0 / r11 * sxy;
            r22 = sqrt(syy - r12 * r12);
            if (DIM == 3) {
                r13 = 1.0 / r11 * sxz;
                r23 = 1.0 / r22 * (syz - r12 / r11 * sxz);
                r33 = sqrt(szz - (r13 * r13 + r23 * r23));
            }
        } else {
            r11 = m.lsq[il];
            r12 = m.lsq[N + il];
            r22 = m.lsq[2 * (size_t)N + il];
            if (DIM == 3) {
                r13 = m.lsq[3 * (size_t)N + il];
                r23 = m.lsq[4 * (size_t)N + il];
                r33 = m.lsq[5 * (size_t)N + il];
            }
        }
        const double beta = (r12 * r23 - r13 * r23) / (r11 * r22);  // GR/gradient.h:89 (sic)
        const double r11s = r11 * r11;
        const double i22 = 1.0 / (r22 * r22);
        const double q12 = r12 / r11;
        const double i33 = 1.0 / (r33 * r33);
        const double q23 = r23 / r22;
#pragma unroll
        for (int j = 0; j < MF; j++) {
            w[j][0] = w[j][1] = w[j][2] = 0.0;
            if (j < nf) {
                const double dx = sc[kst[j]] - xi;
                const double dy = sc[SS + kst[j]] - yi;
                const double dz = sc[2 * SS + kst[j]] - zi;
                const double alpha_1 = dx / r11s;
                const double alpha_2 = i22 * (dy - q12 * dx);
                double alpha_3 = 0.0;
                if (DIM == 3) alpha_3 = i33 * (dz - q23 * dy + beta * dx);
                w[j][0] = alpha_1 - q12 * alpha_2 + beta * alpha_3;
                w[j][1] = alpha_2 - q23 * alpha_3;
                w[j][2] = alpha_3;
            }
        }
    }
    // the LSQ gradient of one staged variable
    auto gradient = [&](const Dual* u, const Dual& ui, Dual& gx, Dual& gy, Dual& gz) {
        gx = gy = gz = Dual(0.0);
#pragma unroll
        for (int j = 0; j < MF; j++) {
            if (j < nf) {
                const Dual diff = u[kst[j]] - ui;
                gx += w[j][0] * diff;
                gy += w[j][1] * diff;
                gz += w[j][2] * diff;
            }
        }
    };
    // 2D: the convective vz gradient is its slot's value from before this
    // call's viscous gradients
    Dual vz_old[3];
    if (RECON && DIM == 2 && i < N) {
        const Dual* g = grad + (size_t)G_VZ * 3 * N;
        vz_old[0] = g[i];
        vz_old[1] = g[N + i];
        vz_old[2] = grad_z<Dual, DIM>(g, N, i);
    }
    if (VISC) {
        const int vslot[4] = {G_T, G_VX, G_VY, G_VZ};
        if (i < N) {
#pragma unroll
            for (int q = 0; q < 4; q++) {
                Dual gx, gy, gz;
                gradient(su + q * SS, su[q * SS + threadIdx.x], gx, gy, gz);
                Dual* g = grad + (size_t)vslot[q] * 3 * N;
                g[i] = gx;
                g[N + i] = gy;
                if (DIM == 3) g[2 * (size_t)N + i] = gz;  // 2D: +0, not stored (grad_z)
            }
        }
        if (!RECON) return;
        __syncthreads();  // the viscous variables are read: their LDS takes the others
        stage(false, false);
    }
    if (!RECON || i >= N) return;
    double ox[MF], oy[MF], oz[MF];
#pragma unroll
    for (int j = 0; j < MF; j++) {
        const int k = j < nf ? j : nf - 1;
        ox[j] = offs[(size_t)(k * 3 + 0) * N + i];
        oy[j] = offs[(size_t)(k * 3 + 1) * N + i];
        oz[j] = zflat ? 0.0 : offs[(size_t)(k * 3 + 2) * N + i];
    }
    double eps2 = 0.0;
    if (LIM == 2) {
        const double V = fabs(m.vol[i]);  // cell size h^dim = |V|
        const double K3 = venkat_K * venkat_K * venkat_K;
        eps2 = (DIM == 3) ? K3 * V : K3 * (V * sqrt(V));
    }
#pragma unroll
    for (int v = 0; v < 5; v++) {
        const Dual* u = su + v * SS;
        const Dual ui = u[threadIdx.x];
        Dual gx, gy, gz;
        if (DIM == 2 && v == 4) {
            gx = vz_old[0];
            gy = vz_old[1];
            gz = vz_old[2];
        } else {
            gradient(u, ui, gx, gy, gz);
        }
        Dual phi(1.0);
        if (LIM != 0) {
            Dual umin = ui, umax = ui;
#pragma unroll
            for (int j = 0; j < MF; j++) {
                if (j < nf) {
                    const Dual un = u[kst[j]];
                    umin = ibis::kmin(umin, un);
                    umax = ibis::kmax(umax, un);
                }
            }
            Dual bn(1.0), bd(1.0);
#pragma unroll
            for (int j = 0; j < MF; j++) {
                if (j >= nf) break;
                Dual d2 = gx * ox[j] + gy * oy[j] + gz * oz[j];
                if (LIM == 1) {  // Barth-Jespersen, FV/limiter.cpp:24-62
                    const int sg = (d2 > Dual(0.0)) - (d2 < Dual(0.0));
                    d2 = (double)sg * (fabs(d2) + eps);
                    if (sg > 0)
                        phi = ibis::kmin(phi, (umax - ui) / d2);
                    else if (sg < 0)
                        phi = ibis::kmin(phi, (umin - ui) / d2);
                } else {  // Venkatakrishnan
                    Dual d1;
                    if (d2 > Dual(0.0))
                        d1 = umax - ui;
                    else if (d2 < Dual(0.0))
                        d1 = umin - ui;
                    else
                        continue;
                    const Dual d1s = d1 * d1;
                    const Dual d2s = d2 * d2;
                    const Dual num = d1s + eps2 + 2.0 * (d1 * d2);
                    const Dual den = d1s + 2.0 * d2s + d1 * d2 + eps2;
                    if (ibis::venkat_take(num, den, bn, bd)) {
                        bn = num;
                        bd = den;
                    }
                }
            }
            if (LIM == 2) phi = bn / bd;
            if (freeze) phi.d = 0.0;
        }
#pragma unroll
        for (int j = 0; j < MF; j++) {
            if (j >= nf) break;
            FL[((size_t)j * 5 + v) * N + i] = ui + phi * (gx * ox[j] + gy * oy[j] + gz * oz[j]);
        }
    }
}

template <int DIM>
__global__ void __launch_bounds__(BLOCK)
    k_tan_visc(DevMesh m, ViscParams vp, const ibis::Dual* __restrict__ prim,
               const ibis::Dual* __restrict__ grad, ibis::Dual* __restrict__ vterm) {
    const int f = blockIdx.x * BLOCK + threadIdx.x;
    const int F = m.F;
    if (f >= F) return;
    ibis::Dual vt[DIM + 1];
    double rho_f, T_f;
    visc_face<ibis::Dual, DIM>(m, vp, prim, grad, f, m.L[f], m.R[f], vt, &rho_f, &T_f);
#pragma unroll
    for (int q = 0; q <= DIM; q++) vterm[(size_t)q * F + f] = vt[q];
}

// what k_tan_face writes: a JVP the rows of the residual and of its tangent, and
// the ghost rows of the caller's state and its tangent; a matvec (VEC) result =
// vec / dt_star - tangent
template <bool VEC>
struct TanOut {
    double *dudt, *dudt_dot, *prim, *prim_dot;
};
template <>
struct TanOut<true> {
    const double* vec;
    double* result;
    double dt_star;
};

// One block per tile: the flux of every face touching it, minus its viscous
// terms, times the area, into LDS; then each cell's sum in its own face
// order over its volume.  RECON reads the entry order's face data (value
// starts and geometry, k_entries); first order reads the cells' rows by face.
// VEC keeps only the tangents in LDS and writes the matvec's result. A JVP has
// blocks past the tiles' that copy the ghost rows of the pairs to the caller's
// rows: k_tan_state, which forms them, stores no half of a pair beside the whole
// pair, since ROCm 7.2's register allocator then marked one half undefined and
// stored what its register held by then.
template <int DIM, int FLUX, bool RECON, bool VISC, bool VEC>
__global__ void __launch_bounds__(MAXTILE)
    k_tan_face(DevMesh m, FaceParams fp, const int2* __restrict__ eidx,
               const double* __restrict__ egeom, const ibis::Dual* __restrict__ FL,
               const ibis::Dual* __restrict__ prim, const ibis::Dual* __restrict__ gpre,
               const ibis::Dual* __restrict__ vterm, TanOut<VEC> o) {
    extern __shared__ double sflux[];  // NC x maxtf tangents [, then the values]
    using ibis::Dual;
    constexpr int NC = DIM + 2;
    const int N = m.N, Nt = m.Nt, F = m.F, S = m.maxtf, NE = m.ntf;
    if constexpr (!VEC) {
        const int gb = (int)blockIdx.x - NXCD * ((m.ntiles + NXCD - 1) / NXCD);
        if (gb >= 0) {
            const int g = N + gb * (int)blockDim.x + (int)threadIdx.x;
            if (g >= Nt) return;
#pragma unroll
            for (int k = 0; k < NPRIM; k++) {
                const Dual x = prim[(size_t)k * Nt + g];
                o.prim[(size_t)k * Nt + g] = x.r;
                o.prim_dot[(size_t)k * Nt + g] = x.d;
            }
            return;
        }
    }
    const int t = xcd_block(m.ntiles);
    if (t >= m.ntiles) return;
    const int f0 = m.tile_face_off[t];
    const int nfl = m.tile_face_off[t + 1] - f0;
    double* sval = sflux + NC * S;
    for (int k = threadIdx.x; k < nfl; k += blockDim.x) {
        const int e = f0 + k;
        Dual st[2][NPRIM];
        double n[3], t1[3], t2[3], A;
        int f = 0;
        if (RECON) {
            const int2 bb = eidx[e];
            const bool swap = bb.y < 0;  // the first start is the right cell's
            const int gbase = m.maxf * 5 * N;
#pragma unroll
            for (int side = 0; side < 2; side++) {
                const int b = side ? (swap ? bb.x : bb.y) : (swap ? ~bb.y : bb.x);
                const size_t stride = b >= gbase ? (size_t)m.G : (size_t)N;
                Dual q[5];
#pragma unroll
                for (int v = 0; v < 5; v++) q[v] = FL[(size_t)b + v * stride];
                thermo_state<Dual>(fp, q[0], q[1], st[side]);
#pragma unroll
                for (int v = 0; v < 3; v++) st[side][ibis::S_U + v] = q[2 + v];
            }
            const double2* eg2 = reinterpret_cast<const double2*>(egeom);
            const double2 p0 = eg2[e];
            const bool planar = DIM == 2 && m.planar2d;
            double2 p1 = make_double2(0.0, 0.0), p2 = make_double2(0.0, 1.0);
            if (!planar) {
                p1 = eg2[(size_t)NE + e];
                p2 = eg2[2 * (size_t)NE + e];
            }
            A = egeom[(size_t)(planar ? 2 : 6) * NE + e];
            t1[0] = p0.x;
            t1[1] = p0.y;
            t1[2] = p1.x;
            t2[0] = p1.y;
            t2[1] = p2.x;
            t2[2] = p2.y;
            n[0] = t1[1] * t2[2] - t1[2] * t2[1];  // cross(tan1, tan2), GR/interface.h:249
            n[1] = t1[2] * t2[0] - t1[0] * t2[2];
            n[2] = t1[0] * t2[1] - t1[1] * t2[0];
            if (VISC) f = m.ent_faces[e];
        } else {
            f = m.tile_faces[e];
#pragma unroll
            for (int side = 0; side < 2; side++) {
                const int c = side ? m.R[f] : m.L[f];
                const Dual* p = VISC && c >= N ? gpre + (c - N) : prim + c;
                const size_t stride = VISC && c >= N ? (size_t)m.G : (size_t)Nt;
#pragma unroll
                for (int v = 0; v < NPRIM; v++) st[side][v] = p[v * stride];
            }
#pragma unroll
            for (int q = 0; q < 3; q++) {
                n[q] = m.geom[(size_t)q * F + f];
                t1[q] = m.geom[(size_t)(3 + q) * F + f];
                t2[q] = m.geom[(size_t)(6 + q) * F + f];
            }
            A = m.geom[12 * (size_t)F + f];
        }
        Dual res[NC];
        rotated_flux<Dual, DIM, FLUX>(fp, st[0], st[1], n, t1, t2, res);
#pragma unroll
        for (int q = 0; q < NC; q++) {
            if (VISC && q > 0) res[q] -= vterm[(size_t)(q - 1) * F + f];
            const Dual fa = res[q] * A;
            sflux[q * S + k] = fa.d;
            if (!VEC) sval[q * S + k] = fa.r;
        }
    }
    __syncthreads();
    const int c = t * m.tile + threadIdx.x;
    if ((int)threadIdx.x >= m.tile || c >= N) return;
    Dual d[NC];
#pragma unroll
    for (int q = 0; q < NC; q++) d[q] = Dual(0.0);
    const int nf = m.nfaces[c];
    const unsigned short* at = RECON ? m.ent_lds : m.cell_lds;
    for (int j = 0; j < nf; j++) {
        const int k = at[(size_t)j * N + c];
        const int s = m.ell_sign[(size_t)j * N + c];
#pragma unroll
        for (int q = 0; q < NC; q++) {
            const Dual fa(VEC ? 0.0 : sval[q * S + k], sflux[q * S + k]);
            d[q] += (s > 0) ? -fa : fa;  // == flux * (-area * outsign), exactly
        }
    }
    const double V = m.vol[c];
#pragma unroll
    for (int q = 0; q < NC; q++) {
        const Dual x = d[q] / V;
        if constexpr (VEC) {  // set_vector, steady_state.cpp:102-111
            const size_t v = (size_t)c * NC + q;
            o.result[v] = 1 / o.dt_star * o.vec[v] - x.d;
        } else {
            o.dudt[(size_t)q * Nt + c] = x.r;
            o.dudt_dot[(size_t)q * Nt + c] = x.d;
        }
    }
}

#endif
