// jfnk.hip -- FP64 Krylov solvers and the JFNK pseudo-transient step on the
// MI355X, around the residual and its tangent (residual.hip).
//
// Restates src/linear_algebra/linear_algebra/gmres.cpp:11-303 (GMRES and
// flexible GMRES with modified Gram-Schmidt Arnoldi, Givens rotations of
// the Hessenberg matrix on the host) and src/solvers/solvers/jfnk.cpp:24-93
// with the CFL schedules of src/solvers/solvers/cfl.cpp:9-83.
//
// Device design: the Krylov basis is one contiguous (m+1) x n FP64 block.
// Modified Gram-Schmidt is run with one reduction per Arnoldi step instead
// of one per basis vector: its coefficients solve the triangular system
// (I + L) h = V^T w, with L the strictly lower part of V^T V (Swirydowicz,
// Langou, Ananthan, Yang, Thomas, "Low synchronization Gram-Schmidt and
// generalized minimal residual algorithms", 2021), and the vector is then
// updated w += v_k (-h_k) in the order of k.  Every sum is deterministic
// (fixed grid, fixed tree).  A step is four launches whatever its length,
// and the host reads the new Hessenberg column once, for the rotations.
// All arithmetic is FP64.  On vectors of up to a few million entries the
// one-vector-at-a-time form is bound by its 3 (j + 1) dependent launches of
// about 3 us each: a JFNK step with 30 GMRES iterations on 73,728 unknowns
// took 6.02 ms with it and 2.65 ms with this one, 1.6 ms of both in the tangent
// operator on the general path (2.1 ms with the fused one); the errors against
// 64-bit references are the same (1.5e-15 of the state).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "ibis_internal.h"

namespace {

constexpr int RB = 256;      // threads per block
constexpr int RNB = 1024;    // blocks of the residual norms' first reduction stage (fixed)
constexpr int DNB = 256;     // most blocks a dot product is summed over (per group of vectors)
constexpr int VG = 8;        // basis vectors per block of k_mgs_dots
constexpr int SOLVE_T = 1024;  // threads of k_mgs_solve
constexpr int LDS_ROWS = 64;   // largest system k_mgs_solve keeps in LDS

#define HIP_TRY(expr)                                                             \
    do {                                                                          \
        hipError_t e_ = (expr);                                                   \
        if (e_ != hipSuccess) {                                                   \
            std::string m_ = std::string(#expr) + ": " + hipGetErrorString(e_);   \
            return ibis::fail(IBIS_ERR_HIP, m_.c_str());                          \
        }                                                                         \
    } while (0)

#define IBIS_TRY(expr)                      \
    do {                                    \
        ibis_status s_ = (expr);            \
        if (s_ != IBIS_OK) return s_;       \
    } while (0)

inline unsigned nblk(int64_t n) { return (unsigned)((n + RB - 1) / RB); }

__device__ __forceinline__ double block_sum(double v, double* sm) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sm[w] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < RB / 64; k++) v += sm[k];
    }
    return v;
}

// blocks over which the n entries of a vector are summed: 1024 entries a
// block (four per thread, so that a wave's reduction is paid once for them),
// at most DNB, which keeps the partial sums of a step (2 (j+1) DNB doubles)
// small enough for k_mgs_solve's one block
inline int dot_blocks(int64_t n) {
    const int64_t b = (n + 4 * RB - 1) / (4 * RB);
    return (int)std::min<int64_t>(b, DNB);
}

// blocks of the kernels that stream a vector and sum one value: one entry per
// thread up to 8 blocks per CU; k_normalise's every block adds up their sums
constexpr unsigned STREAM_NB = 2048;
inline unsigned stream_blocks(int64_t n) { return std::min(nblk(n), STREAM_NB); }

// Sums of 16 values over a wave by recursive halving: at each of the first
// four steps a lane keeps half of its values and adds the other half's of
// its partner, so 17 exchanges instead of 96.  Returns the sum of value
// (lane >> 2) of the wave, in its four lanes.
__device__ __forceinline__ double wave_sum16(double (&a)[16]) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int half = 8, off = 32; half >= 1; half >>= 1, off >>= 1) {
        const bool hi = lane & off;
#pragma unroll
        for (int q = 0; q < half; q++) {
            const double mine = hi ? a[q + half] : a[q];
            const double give = hi ? a[q] : a[q + half];
            a[q] = mine + __shfl_xor(give, off, 64);
        }
    }
    double v = a[0];
    v += __shfl_xor(v, 2, 64);
    v += __shfl_xor(v, 1, 64);
    return v;
}

// Partial sums of V^T w and V^T v_j for the vectors 8 y .. 8 y + 7 of the
// nv = j + 1 in the basis (y = blockIdx.y): value q < 8 of group y is
// v_{8y+q} . w, value 8 + q is v_{8y+q} . v_j, at
// partial[(16 y + value) * gridDim.x + blockIdx.x].  Bound by reading the
// basis once; groups of 8 keep 16 sums per thread in registers and give
// short vectors enough blocks. On those each thread has four entries: their
// 40 loads are issued together (139 VGPRs), one wait instead of four (30
// iterations on 73,728 unknowns 2310 -> 2225 us).
__global__ void __launch_bounds__(RB)
    k_mgs_dots(int64_t n, int nv, const double* __restrict__ V, const double* __restrict__ w,
               double* __restrict__ partial) {
    __shared__ double sm[RB / 64][16];
    const int g0 = blockIdx.y * VG;
    const double* vj = V + (size_t)(nv - 1) * n;
    const double* v[VG];  // past the last vector: the last again, not read back
#pragma unroll
    for (int q = 0; q < VG; q++) v[q] = V + (size_t)min(g0 + q, nv - 1) * n;
    double a[16];
#pragma unroll
    for (int q = 0; q < 16; q++) a[q] = 0.0;
    const int64_t step = (int64_t)gridDim.x * RB;
    int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x;
    for (; i + 3 * step < n; i += 4 * step) {
        double wi[4], vi[4], x[4][VG];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            wi[u] = w[i + u * step];
            vi[u] = vj[i + u * step];
#pragma unroll
            for (int q = 0; q < VG; q++) x[u][q] = v[q][i + u * step];
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int q = 0; q < VG; q++) {
                a[q] += x[u][q] * wi[u];
                a[VG + q] += x[u][q] * vi[u];
            }
    }
    for (; i < n; i += step) {
        const double wi = w[i], vi = vj[i];
#pragma unroll
        for (int q = 0; q < VG; q++) {
            const double x = v[q][i];
            a[q] += x * wi;
            a[VG + q] += x * vi;
        }
    }
    const double s = wave_sum16(a);
    const int lane = threadIdx.x & 63;
    if ((lane & 3) == 0) sm[threadIdx.x >> 6][lane >> 2] = s;
    __syncthreads();
    if (threadIdx.x < 16) {
        double t = sm[0][threadIdx.x];
        for (int k = 1; k < RB / 64; k++) t += sm[k][threadIdx.x];
        partial[((size_t)blockIdx.y * 16 + threadIdx.x) * gridDim.x + blockIdx.x] = t;
    }
}

// One block: the sums of k_mgs_dots' partials, the new row of L
// (L[j * ld + k] = v_j . v_k, k < j, kept for the later steps) and the
// forward substitution h_i = (V^T w)_i - sum_{k<i} L_ik h_k, the
// coefficients that subtracting the vectors one after the other gives.
// Up to LDS_ROWS vectors the system is in LDS and the substitution runs in
// one wave's registers; a longer one stays in memory and the block
// synchronises at each row.
__global__ void __launch_bounds__(SOLVE_T)
    k_mgs_solve(int nv, int nb, const double* __restrict__ partial, double* L, int ld, double* h) {
    __shared__ double sh[2 * LDS_ROWS + LDS_ROWS * (LDS_ROWS + 1)];
    const int j = nv - 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool small = nv <= LDS_ROWS;
    double* d = small ? sh : h;                                  // V^T w, then h
    double* row = small ? sh + LDS_ROWS : L + (size_t)j * ld;    // row j of L
    double* sL = sh + 2 * LDS_ROWS;                              // its other rows
    if (small)
        for (int e = threadIdx.x; e < j * LDS_ROWS; e += SOLVE_T) {
            const int r = e / LDS_ROWS, c = e % LDS_ROWS;
            if (c < r) sL[r * (LDS_ROWS + 1) + c] = L[(size_t)r * ld + c];
        }
    for (int k = wave; k < 2 * nv; k += SOLVE_T / 64) {
        const int i = k >> 1, dot = k & 1;  // dot 0: v_i . w, 1: v_i . v_j
        const double* p = partial + ((size_t)(i / VG) * 16 + dot * VG + i % VG) * nb;
        double s = 0.0;
        for (int b = lane; b < nb; b += 64) s += p[b];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) (dot ? row : d)[i] = s;
    }
    __syncthreads();
    if (small) {
        for (int k = threadIdx.x; k < j; k += SOLVE_T) L[(size_t)j * ld + k] = row[k];
        if (wave) return;
        double x = lane < nv ? d[lane] : 0.0;
        const double* lr = lane < j ? sL + lane * (LDS_ROWS + 1) : row;
        for (int i = 0; i < j; i++) {
            const double hi = __shfl(x, i, 64);
            if (lane > i && lane < nv) x -= lr[i] * hi;
        }
        if (lane < nv) h[lane] = x;
        return;
    }
    for (int i = 0; i < j; i++) {
        const double hi = d[i];
        for (int r = i + 1 + threadIdx.x; r <= j; r += SOLVE_T) d[r] -= L[(size_t)r * ld + i] * hi;
        __syncthreads();
    }
}

// w += v_k (-h_k) in the order of k (add_scaled_vector, gmres.cpp:147), and
// the partial sums of w . w
__global__ void __launch_bounds__(RB)
    k_mgs_update(int64_t n, int nv, const double* __restrict__ V, const double* __restrict__ h,
                 double* __restrict__ w, double* __restrict__ partial) {
    __shared__ double sm[RB / 64];
    double s = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) {
        double x = w[i];
        const double* v = V + i;
#pragma unroll 8
        for (int k = 0; k < nv; k++) x += v[(size_t)k * n] * (-h[k]);
        w[i] = x;
        s += x * x;
    }
    s = block_sum(s, sm);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// v = w (1 / |w|) with |w| from the nb partial sums of w . w
// (scale(w, v, 1 / h), gmres.cpp:150), summed by every block in the same
// order; the first block stores it to norm
__global__ void __launch_bounds__(RB)
    k_normalise(int64_t n, const double* __restrict__ w, const double* __restrict__ partial, int nb,
                double* __restrict__ v, double* __restrict__ norm) {
    __shared__ double sm[RB / 64];
    __shared__ double total;
    double s = 0.0;
    for (int k = threadIdx.x; k < nb; k += RB) s += partial[k];
    s = block_sum(s, sm);
    if (threadIdx.x == 0) total = sqrt(s);
    __syncthreads();
    const double f = 1.0 / total;
    if (blockIdx.x == 0 && threadIdx.x == 0) norm[0] = total;
    for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB)
        v[i] = w[i] * f;
}

// w = rhs - w (r0, gmres.cpp:17-19) and the partial sums of r0 . r0; w null:
// a zero initial vector, r0 is rhs
__global__ void __launch_bounds__(RB)
    k_sub(int64_t n, const double* __restrict__ rhs, double* __restrict__ w,
          double* __restrict__ partial) {
    __shared__ double sm[RB / 64];
    double s = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x; i < n; i += (int64_t)gridDim.x * RB) {
        double x = rhs[i];
        if (w) {
            x -= w[i];
            w[i] = x;
        }
        s += x * x;
    }
    s = block_sum(s, sm);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

__global__ void __launch_bounds__(RB) k_fill(int64_t n, double* __restrict__ a, double v) {
    const int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x;
    if (i < n) a[i] = v;
}

// w = V[:, 0:k] y (gemv, in column order), then x += w * 1.0
// (gmres.cpp:177-179)
__global__ void __launch_bounds__(RB)
    k_combine_add(int64_t n, int k, const double* __restrict__ V, const double* __restrict__ y,
                  double* __restrict__ w, double* __restrict__ x) {
    const int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int c = 0; c < k; c++) s += V[(size_t)c * n + i] * y[c];
    w[i] = s;
    x[i] += w[i] * 1.0;
}

// Jfnk::apply_update_ (jfnk.cpp:67-74): cons(cell, q) += dU[cell*nc + q]
__global__ void __launch_bounds__(RB)
    k_apply_update(int N, int Nt, int nc, const double* __restrict__ dU, double* __restrict__ cons) {
    const int i = blockIdx.x * RB + threadIdx.x;
    if (i >= N) return;
    for (int q = 0; q < nc; q++) cons[(size_t)q * Nt + i] += dU[(size_t)i * nc + q];
}

// ConservedQuantities::L2_norms partial sums (conserved_quantities.cpp:41-69):
// per block, the six sums (mass, mx, my, mz, energy, global)
__global__ void __launch_bounds__(RB)
    k_norm_partial(int N, int Nt, int dim, const double* __restrict__ dudt,
                   double* __restrict__ partial) {
    __shared__ double sm[RB / 64];
    double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int i = blockIdx.x * RB + threadIdx.x; i < N; i += RNB * RB) {
        const double m = dudt[i];
        const double mx = dudt[(size_t)Nt + i];
        const double my = dudt[2 * (size_t)Nt + i];
        const double mz = dim == 3 ? dudt[3 * (size_t)Nt + i] : 0.0;
        const double e = dudt[(size_t)(dim + 1) * Nt + i];
        s[0] += m * m;
        s[1] += mx * mx;
        s[2] += my * my;
        s[3] += mz * mz;
        s[4] += e * e;
        s[5] += m * m + mx * mx + my * my + mz * mz + e * e;
    }
    for (int q = 0; q < 6; q++) {
        const double t = block_sum(s[q], sm);
        if (threadIdx.x == 0) partial[(size_t)q * RNB + blockIdx.x] = t;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(RB)
    k_norm_final(const double* __restrict__ partial, double* __restrict__ out) {
    __shared__ double sm[RB / 64];
    for (int q = 0; q < 6; q++) {
        double s = 0.0;
        for (int k = threadIdx.x; k < RNB; k += RB) s += partial[(size_t)q * RNB + k];
        s = block_sum(s, sm);
        if (threadIdx.x == 0) out[q] = sqrt(s);
        __syncthreads();
    }
}

}  // namespace

// ===========================================================================
// GMRES / FGMRES
// ===========================================================================
struct ibis_gmres {
    int64_t n = 0;
    int m = 0;
    double tol = 0.0;
    double* V = nullptr;        // (m+1) x n Krylov basis
    double* Z = nullptr;        // m x n preconditioned vectors (FGMRES, on demand)
    double* w = nullptr;
    double* partial = nullptr;  // partial sums: 16 per group of VG basis vectors, DNB each
    double* L = nullptr;        // m x m: strictly lower part of V^T V
    double* hdev = nullptr;     // m + 2 Hessenberg column entries (device)
    double* ydev = nullptr;     // m
    double* hhost = nullptr;    // pinned copy of hdev
    std::vector<double> H;      // (m+1) x m, row-major
    std::vector<double> cs, sn, g;
};

static ibis_status read_dev(ibis_gmres* s, const double* dev, int k, hipStream_t st) {
    HIP_TRY(hipMemcpyAsync(s->hhost, dev, sizeof(double) * k, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    return IBIS_OK;
}

void ibis_gmres_destroy(ibis_gmres* g) {
    if (!g) return;
    for (void* p : {(void*)g->V, (void*)g->Z, (void*)g->w, (void*)g->partial, (void*)g->L,
                    (void*)g->hdev, (void*)g->ydev})
        if (p) (void)hipFree(p);
    if (g->hhost) (void)hipHostFree(g->hhost);
    delete g;
}

ibis_status ibis_gmres_create(int64_t num_vars, int32_t max_iters, double tol, ibis_gmres** out) {
    if (!out || num_vars <= 0 || max_iters <= 0)
        return ibis::fail(IBIS_ERR_INVALID, "ibis_gmres_create: invalid argument");
    ibis_gmres* g = new ibis_gmres();
    g->n = num_vars;
    g->m = (int)std::min<int64_t>(num_vars, max_iters);  // gmres.cpp:90
    g->tol = tol;
    const size_t n = (size_t)num_vars, m = (size_t)g->m;
    hipError_t e = hipMalloc((void**)&g->V, sizeof(double) * n * (m + 1));
    if (e == hipSuccess) e = hipMalloc((void**)&g->w, sizeof(double) * n);
    if (e == hipSuccess)
        e = hipMalloc((void**)&g->partial, sizeof(double) * ((m + VG - 1) / VG) * 16 * DNB);
    static_assert(STREAM_NB <= 16 * DNB, "one group's partial sums hold a streaming kernel's");
    if (e == hipSuccess) e = hipMalloc((void**)&g->L, sizeof(double) * m * m);
    if (e == hipSuccess) e = hipMalloc((void**)&g->hdev, sizeof(double) * (m + 2));
    if (e == hipSuccess) e = hipMalloc((void**)&g->ydev, sizeof(double) * (m + 1));
    if (e == hipSuccess) e = hipHostMalloc((void**)&g->hhost, sizeof(double) * (m + 2), hipHostMallocDefault);
    if (e != hipSuccess) {
        ibis_gmres_destroy(g);
        return ibis::fail(IBIS_ERR_HIP, hipGetErrorString(e));
    }
    g->H.assign((m + 1) * m, 0.0);
    g->cs.assign(m, 0.0);
    g->sn.assign(m, 0.0);
    g->g.assign(m + 1, 0.0);
    *out = g;
    return IBIS_OK;
}

// Orthonormalise w against the nv = j + 1 vectors of the basis and store
// the result as vector nv; hdev[0 .. nv] receives the Hessenberg column.
static ibis_status arnoldi(ibis_gmres* s, int nv, hipStream_t st) {
    const int64_t n = s->n;
    const int nb = dot_blocks(n);
    const unsigned ub = stream_blocks(n);
    k_mgs_dots<<<dim3(nb, (nv + VG - 1) / VG), RB, 0, st>>>(n, nv, s->V, s->w, s->partial);
    k_mgs_solve<<<1, SOLVE_T, 0, st>>>(nv, nb, s->partial, s->L, s->m, s->hdev);
    k_mgs_update<<<ub, RB, 0, st>>>(n, nv, s->V, s->hdev, s->w, s->partial);
    k_normalise<<<ub, RB, 0, st>>>(n, s->w, s->partial, (int)ub, s->V + (size_t)nv * n,
                                  s->hdev + nv);
    HIP_TRY(hipGetLastError());
    return IBIS_OK;
}

// One (F)GMRES solve.  With inner != nullptr the Krylov vectors are
// preconditioned by an inner GMRES solve of P z = v from z = 0.  x_is_zero:
// the caller has just zeroed x, so A x is zero and r0 is rhs itself.
static ibis_status gmres_run(ibis_gmres* s, ibis_matvec_fn A, void* ctx_a, const double* rhs,
                             double* x, bool x_is_zero, ibis_gmres* inner, ibis_matvec_fn P,
                             void* ctx_p, ibis_linear_result* res, hipStream_t st) {
    const int64_t n = s->n;
    const int m = s->m;
    ibis_stream_t sh = reinterpret_cast<ibis_stream_t>(st);
    if (inner && !s->Z) HIP_TRY(hipMalloc((void**)&s->Z, sizeof(double) * (size_t)n * m));
    std::fill(s->H.begin(), s->H.end(), 0.0);
    std::fill(s->g.begin(), s->g.end(), 0.0);
    auto Hm = [&](int i, int j) -> double& { return s->H[(size_t)i * m + j]; };
    // r0 = rhs - A x0, beta = |r0|, v_0 = r0 / beta (gmres.cpp:11-20, 130-135)
    if (!x_is_zero) IBIS_TRY(A(ctx_a, x, s->w, sh));
    const unsigned ub = stream_blocks(n);
    k_sub<<<ub, RB, 0, st>>>(n, rhs, x_is_zero ? nullptr : s->w, s->partial);
    k_normalise<<<ub, RB, 0, st>>>(n, x_is_zero ? rhs : s->w, s->partial, (int)ub, s->V, s->hdev);
    HIP_TRY(hipGetLastError());
    IBIS_TRY(read_dev(s, s->hdev, 1, st));
    const double beta = s->hhost[0];
    ibis_linear_result r{0, 0, s->tol, beta};
    if (beta < s->tol) {
        r.success = 1;
        *res = r;
        return IBIS_OK;
    }
    s->g[0] = beta;
    for (int j = 0; j < m; j++) {
        double* vj = s->V + (size_t)j * n;
        if (inner) {  // gmres.cpp:260-265
            double* zj = s->Z + (size_t)j * n;
            k_fill<<<nblk(n), RB, 0, st>>>(n, zj, 0.0);
            ibis_linear_result ri;
            IBIS_TRY(gmres_run(inner, P, ctx_p, vj, zj, true, nullptr, nullptr, nullptr, &ri, st));
            IBIS_TRY(A(ctx_a, zj, s->w, sh));
        } else {
            IBIS_TRY(A(ctx_a, vj, s->w, sh));
        }
        IBIS_TRY(arnoldi(s, j + 1, st));
        IBIS_TRY(read_dev(s, s->hdev, j + 2, st));
        for (int i = 0; i <= j + 1; i++) Hm(i, j) = s->hhost[i];
        // previous rotations on the new column, then this step's rotation
        // (apply_rotations_to_hessenberg_, gmres.cpp:22-74)
        for (int i = 0; i < j; i++) {
            const double a = Hm(i, j), b = Hm(i + 1, j);
            Hm(i, j) = s->cs[i] * a + s->sn[i] * b;
            Hm(i + 1, j) = -s->sn[i] * a + s->cs[i] * b;
        }
        const double denom = std::sqrt(Hm(j, j) * Hm(j, j) + Hm(j + 1, j) * Hm(j + 1, j));
        const double si = Hm(j + 1, j) / denom;
        const double ci = Hm(j, j) / denom;
        s->cs[j] = ci;
        s->sn[j] = si;
        Hm(j, j) = ci * Hm(j, j) + si * Hm(j + 1, j);
        Hm(j + 1, j) = 0.0;
        const double gj = s->g[j];
        s->g[j] = ci * gj;
        s->g[j + 1] = -si * gj;
        const double residual = std::fabs(s->g[j + 1]);
        r.residual = residual / beta;
        r.n_iters = j + 1;
        if (residual < s->tol * beta) {
            r.success = 1;
            break;
        }
    }
    // upper-triangular solve H y = g, then x += V y (or Z y)
    const int k = r.n_iters;
    std::vector<double> y(k, 0.0);
    y[k - 1] = s->g[k - 1] / Hm(k - 1, k - 1);
    for (int i = k - 2; i >= 0; i--) {
        double sum = s->g[i];
        for (int c = i + 1; c < k; c++) sum -= Hm(i, c) * y[c];
        y[i] = sum / Hm(i, i);
    }
    HIP_TRY(hipMemcpyAsync(s->ydev, y.data(), sizeof(double) * k, hipMemcpyHostToDevice, st));
    k_combine_add<<<nblk(n), RB, 0, st>>>(n, k, inner ? s->Z : s->V, s->ydev, s->w, x);
    HIP_TRY(hipGetLastError());
    // y is host memory: finish the copy before it goes out of scope
    HIP_TRY(hipStreamSynchronize(st));
    *res = r;
    return IBIS_OK;
}

ibis_status ibis_gmres_solve(ibis_gmres* g, ibis_matvec_fn A, void* ctx, const double* rhs,
                             double* x, ibis_linear_result* result, ibis_stream_t stream) {
    if (!g || !A || !rhs || !x || !result)
        return ibis::fail(IBIS_ERR_INVALID, "ibis_gmres_solve: null argument");
    return gmres_run(g, A, ctx, rhs, x, false, nullptr, nullptr, nullptr, result,
                     reinterpret_cast<hipStream_t>(stream));
}

ibis_status ibis_fgmres_solve(ibis_gmres* g, ibis_matvec_fn A, void* ctx_a, const double* rhs,
                              double* x, ibis_gmres* inner, ibis_matvec_fn P, void* ctx_p,
                              ibis_linear_result* result, ibis_stream_t stream) {
    if (!g || !A || !rhs || !x || !result || !inner || !P)
        return ibis::fail(IBIS_ERR_INVALID, "ibis_fgmres_solve: null argument");
    if (inner->n != g->n)
        return ibis::fail(IBIS_ERR_INVALID, "ibis_fgmres_solve: inner solver size differs");
    return gmres_run(g, A, ctx_a, rhs, x, false, inner, P, ctx_p, result,
                     reinterpret_cast<hipStream_t>(stream));
}

// ===========================================================================
// CFL schedules and JFNK
// ===========================================================================
static ibis_status cfl_eval(const ibis_jfnk_desc& d, double t, double* prev_cfl,
                            double* prev_res, double* out) {
    switch (d.cfl_kind) {
        case IBIS_CFL_CONSTANT:  // cfl.cpp:9-14
            *out = d.cfl_value;
            return IBIS_OK;
        case IBIS_CFL_LINEAR: {  // cfl.cpp:16-41
            const int n = d.n_cfl_points;
            if (t <= d.cfl_times[0]) {
                *out = d.cfl_values[0];
                return IBIS_OK;
            }
            if (t >= d.cfl_times[n - 1]) {
                *out = d.cfl_values[n - 1];
                return IBIS_OK;
            }
            for (int i = 0; i + 1 < n; i++) {
                if (t >= d.cfl_times[i] && t < d.cfl_times[i + 1]) {
                    const double frac = (t - d.cfl_times[i]) / (d.cfl_times[i + 1] - d.cfl_times[i]);
                    *out = d.cfl_values[i] + frac * (d.cfl_values[i + 1] - d.cfl_values[i]);
                    return IBIS_OK;
                }
            }
            return ibis::fail(IBIS_ERR_INVALID, "linear CFL schedule: times not increasing");
        }
        case IBIS_CFL_RESIDUAL: {  // cfl.cpp:43-68
            if (t > d.growth_threshold) {
                *prev_res = t;
                *out = *prev_cfl;
                return IBIS_OK;
            }
            const double ratio = *prev_res / t;
            double c = *prev_cfl * std::pow(ratio, d.power);
            c = (d.max_cfl < c) ? d.max_cfl : c;      // Ibis::min
            c = (d.start_cfl < c) ? c : d.start_cfl;  // Ibis::max
            *prev_res = t;
            *prev_cfl = c;
            *out = c;
            return IBIS_OK;
        }
        default:
            return ibis::fail(IBIS_ERR_INVALID, "Unknown CFL schedule");
    }
}

ibis_status ibis_cfl_eval(const ibis_jfnk_desc* desc, double t, double* previous_cfl,
                          double* previous_residual, double* cfl) {
    if (!desc || !previous_cfl || !previous_residual || !cfl)
        return ibis::fail(IBIS_ERR_INVALID, "ibis_cfl_eval: null argument");
    return cfl_eval(*desc, t, previous_cfl, previous_residual, cfl);
}

typedef ibis_steady_op SteadyCtx;

static ibis_status steady_mv(void* ctx, const double* v, double* w, ibis_stream_t st) {
    return ibis_steady_op_matvec(ctx, v, w, st);
}

ibis_status ibis_steady_op_matvec(void* ctx, const double* v, double* w, ibis_stream_t stream) {
    const ibis_steady_op* c = static_cast<const ibis_steady_op*>(ctx);
    if (!c) return ibis::fail(IBIS_ERR_INVALID, "ibis_steady_op_matvec: null operator");
    return ibis_steady_matvec(c->r, c->cons, v, w, c->dt_star, c->allow_reconstruction, stream);
}

namespace {
__global__ void __launch_bounds__(RB)
    k_dense_mv(int64_t n, const double* __restrict__ a, const double* __restrict__ v,
               double* __restrict__ w) {
    const int64_t i = (int64_t)blockIdx.x * RB + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    for (int64_t k = 0; k < n; k++) s += a[(size_t)i * n + k] * v[k];
    w[i] = s;
}
}  // namespace

ibis_status ibis_dense_matvec(void* ctx, const double* v, double* w, ibis_stream_t stream) {
    const ibis_dense_op* c = static_cast<const ibis_dense_op*>(ctx);
    if (!c || !c->a || !v || !w) return ibis::fail(IBIS_ERR_INVALID, "ibis_dense_matvec: null argument");
    k_dense_mv<<<nblk(c->n), RB, 0, reinterpret_cast<hipStream_t>(stream)>>>(c->n, c->a, v, w);
    HIP_TRY(hipGetLastError());
    return IBIS_OK;
}

struct ibis_jfnk {
    ibis_residual* r = nullptr;
    ibis_jfnk_desc d{};
    int dim = 0, N = 0, Nt = 0, nc = 0;
    int64_t nv = 0;
    ibis_gmres* outer = nullptr;
    ibis_gmres* inner = nullptr;
    double* rhs = nullptr;
    double* dU = nullptr;
    double* dudt = nullptr;
    double* partial = nullptr;
    double* norms_dev = nullptr;
    double* norms_host = nullptr;  // pinned
    double norms[IBIS_NNORMS] = {0};
    double initial_norms[IBIS_NNORMS] = {0};
    double prev_cfl = 0.0, prev_res = 1.0;  // ResidualBasedCfl state (cfl.cpp:43-50)
};

void ibis_jfnk_destroy(ibis_jfnk* j) {
    if (!j) return;
    ibis_gmres_destroy(j->outer);
    ibis_gmres_destroy(j->inner);
    for (void* p : {(void*)j->rhs, (void*)j->dU, (void*)j->dudt, (void*)j->partial,
                    (void*)j->norms_dev})
        if (p) (void)hipFree(p);
    if (j->norms_host) (void)hipHostFree(j->norms_host);
    delete j;
}

ibis_status ibis_jfnk_create(ibis_residual* r, const ibis_jfnk_desc* desc, ibis_jfnk** out) {
    if (!r || !desc || !out) return ibis::fail(IBIS_ERR_INVALID, "ibis_jfnk_create: null argument");
    const ibis_jfnk_desc& d = *desc;
    if (d.linear_solver != 0 && d.linear_solver != 1)
        return ibis::fail(IBIS_ERR_INVALID, "Unknown linear solver");
    if (d.cfl_kind < 0 || d.cfl_kind > 2) return ibis::fail(IBIS_ERR_INVALID, "Unknown CFL schedule");
    if (d.cfl_kind == IBIS_CFL_LINEAR && (d.n_cfl_points < 1 || d.n_cfl_points > IBIS_MAX_CFL_POINTS))
        return ibis::fail(IBIS_ERR_INVALID, "linear CFL schedule: bad number of points");
    int64_t sizes[5];
    IBIS_TRY(ibis_residual_sizes(r, sizes));
    ibis_jfnk* j = new ibis_jfnk();
    j->r = r;
    j->d = d;
    j->dim = (int)sizes[0];
    j->N = (int)sizes[1];
    j->Nt = (int)sizes[2];
    j->nc = j->dim + 2;
    j->nv = (int64_t)j->N * j->nc;
    j->prev_cfl = d.start_cfl;
    ibis_status s = ibis_gmres_create(j->nv, d.max_iters, d.tol, &j->outer);
    if (s == IBIS_OK && d.linear_solver == 1)
        s = ibis_gmres_create(j->nv, d.max_precond_iters, d.precond_tol, &j->inner);
    if (s != IBIS_OK) {
        ibis_jfnk_destroy(j);
        return s;
    }
    hipError_t e = hipMalloc((void**)&j->rhs, sizeof(double) * j->nv);
    if (e == hipSuccess) e = hipMalloc((void**)&j->dU, sizeof(double) * j->nv);
    if (e == hipSuccess) e = hipMalloc((void**)&j->dudt, sizeof(double) * j->nc * (size_t)j->Nt);
    if (e == hipSuccess) e = hipMemset(j->dudt, 0, sizeof(double) * j->nc * (size_t)j->Nt);
    if (e == hipSuccess) e = hipMalloc((void**)&j->partial, sizeof(double) * 6 * RNB);
    if (e == hipSuccess) e = hipMalloc((void**)&j->norms_dev, sizeof(double) * IBIS_NNORMS);
    if (e == hipSuccess)
        e = hipHostMalloc((void**)&j->norms_host, sizeof(double) * IBIS_NNORMS, hipHostMallocDefault);
    if (e != hipSuccess) {
        ibis_jfnk_destroy(j);
        return ibis::fail(IBIS_ERR_HIP, hipGetErrorString(e));
    }
    *out = j;
    return IBIS_OK;
}

// eval_rhs + L2_norms (jfnk.cpp:24-29, 60-63)
static ibis_status jfnk_rhs_norms(ibis_jfnk* j, double* prim, hipStream_t st) {
    IBIS_TRY(ibis_steady_rhs(j->r, prim, j->dudt, j->rhs, 1, reinterpret_cast<ibis_stream_t>(st)));
    k_norm_partial<<<RNB, RB, 0, st>>>(j->N, j->Nt, j->dim, j->dudt, j->partial);
    k_norm_final<<<1, RB, 0, st>>>(j->partial, j->norms_dev);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(j->norms_host, j->norms_dev, sizeof(double) * IBIS_NNORMS,
                           hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    // kernel order mass, mx, my, mz, energy, global
    for (int q = 0; q < IBIS_NNORMS; q++) j->norms[q] = j->norms_host[q];
    return IBIS_OK;
}

ibis_status ibis_jfnk_initialise(ibis_jfnk* j, double* cons, double* prim, double* norms,
                                 ibis_stream_t stream) {
    if (!j || !cons || !prim) return ibis::fail(IBIS_ERR_INVALID, "ibis_jfnk_initialise: null argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    IBIS_TRY(jfnk_rhs_norms(j, prim, st));
    std::memcpy(j->initial_norms, j->norms, sizeof(j->norms));
    if (norms) std::memcpy(norms, j->norms, sizeof(j->norms));
    return IBIS_OK;
}

ibis_status ibis_jfnk_step(ibis_jfnk* j, double* cons, double* prim, int64_t step,
                           ibis_linear_result* result, double* norms, double* dt_star_out,
                           ibis_stream_t stream) {
    if (!j || !cons || !prim) return ibis::fail(IBIS_ERR_INVALID, "ibis_jfnk_step: null argument");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    k_fill<<<nblk(j->nv), RB, 0, st>>>(j->nv, j->dU, 0.0);
    double stable_dt = 0.0;
    IBIS_TRY(ibis_estimate_dt(j->r, prim, &stable_dt, stream));
    // Jfnk::calculate_cfl (jfnk.h:39-47)
    double cfl = 0.0;
    if (j->d.cfl_kind == IBIS_CFL_RESIDUAL) {
        const double rel = j->norms[5] / j->initial_norms[5];
        IBIS_TRY(cfl_eval(j->d, rel, &j->prev_cfl, &j->prev_res, &cfl));
    } else {
        IBIS_TRY(cfl_eval(j->d, (double)step, &j->prev_cfl, &j->prev_res, &cfl));
    }
    const double dt_star = cfl * stable_dt;
    SteadyCtx sys{j->r, cons, dt_star, 1};
    SteadyCtx pre{j->r, cons, dt_star, 0};
    ibis_linear_result lr;
    if (j->d.linear_solver == 1)
        IBIS_TRY(gmres_run(j->outer, steady_mv, &sys, j->rhs, j->dU, true, j->inner, steady_mv,
                           &pre, &lr, st));
    else
        IBIS_TRY(gmres_run(j->outer, steady_mv, &sys, j->rhs, j->dU, true, nullptr, nullptr,
                           nullptr, &lr, st));
    k_apply_update<<<nblk(j->N), RB, 0, st>>>(j->N, j->Nt, j->nc, j->dU, cons);
    HIP_TRY(hipGetLastError());
    IBIS_TRY(ibis_cons_to_prim(j->r, cons, prim, stream));
    IBIS_TRY(jfnk_rhs_norms(j, prim, st));
    if (result) *result = lr;
    if (norms) std::memcpy(norms, j->norms, sizeof(j->norms));
    if (dt_star_out) *dt_star_out = dt_star;
    return IBIS_OK;
}
