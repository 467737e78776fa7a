// Level-1 / merged BiCGStab vector kernels with fused per-RHS dot partials, the
// single-workgroup finalize kernels that turn partials into the Krylov scalars and the
// convergence decision on the device, and the smoother / coarse-solve kernels.
//
// References: blas::axpby_z / axpbypcz / xdivy_z (src/blas/detail/blas_ext.inl:31-239),
// merged_bicgstab_group1/2/4/5 (src/blas/detail/specific/blas_merged_bicgstab.inl:33-257),
// merged_rbicgstab_group2 (src/blas/detail/specific/blas_merged_rbicgstab.inl:120-196),
// base_solver::convergence_check / converged (src/solvers/solver.h:173-241),
// merged_jacobi (src/blas/detail/specific/blas_merged_jacobi.inl:33-90),
// dense_Ax_y (src/blas2/detail/dense_matvec.inl:72-121), vector::convert
// (src/primitives/vector/operations/convert.inl:31-83).
//
// Every expression keeps the reference's operand order; the file is built with
// -ffp-contract=off so a*b+c rounds twice as in the reference's x86-64 build.
#include "xh_internal.hpp"
#include "xh_krylov.hpp"

#include <algorithm>

namespace xh {
namespace {

__device__ __forceinline__ int64_t logical_block() {
    const uint32_t G = gridDim.x, p = blockIdx.x;
    return (int64_t)(p & 7u) * (int64_t)(G >> 3) + (int64_t)(p >> 3);
}

template <int NV, int ND>
__device__ __forceinline__ void block_partials(double (&p)[ND], double *__restrict__ out,
                                               int64_t lb) {
    __shared__ double red[kBlock / 64][ND][NV];
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int off = NV; off < 64; off <<= 1)
            p[d] = p[d] + __shfl_xor(p[d], off, 64);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane < NV)
#pragma unroll
        for (int d = 0; d < ND; ++d)
            red[w][d][lane] = p[d];
    __syncthreads();
    if ((int)threadIdx.x < ND * NV) {
        const int d = threadIdx.x / NV, k = threadIdx.x % NV;
        double s = red[0][d][k];
#pragma unroll
        for (int q = 1; q < kBlock / 64; ++q)
            s = s + red[q][d][k];
        out[lb * (ND * NV) + d * NV + k] = s;
    }
}

enum Gate : int { GATE_NOT_DONE = 0, GATE_CONV_ALL = 1 };

template <int NV, int OP>
__global__ __launch_bounds__(kBlock) void k_vec(int64_t n, int64_t chunk, double *__restrict__ p,
                                                double *__restrict__ s,
                                                double *__restrict__ r,
                                                const double *__restrict__ r0,
                                                const double *__restrict__ v,
                                                const double *__restrict__ t,
                                                const double *__restrict__ p_,
                                                const double *__restrict__ s_,
                                                const SolverState *__restrict__ st, int gate,
                                                double *__restrict__ partials) {
    if (st->done)
        return;
    if (gate == GATE_CONV_ALL && !st->conv_all)
        return;
    constexpr int ND =
        (OP == V_XR_UPDATE || OP == V_R_UPDATE || OP == V_DOT1 || OP == V_COPY_DOT) ? 1
        : (OP == V_DOT2)                                                             ? 2
        : (OP == V_DOT3)                                                             ? 3
                                                                                     : 0;
    constexpr int RPB = kBlock / NV;
    constexpr bool X = OP == V_XR_UPDATE || OP == V_X_UPDATE || OP == V_GROUP5 || OP == V_CG_XR ||
                       OP == V_RB_UPDATE || OP == V_RB_UPDATE_MERGED;
    // global memory: a pointer read from memory would otherwise make flat accesses
    typedef __attribute__((address_space(1))) double gdouble;
    gdouble *__restrict__ x = X ? (gdouble *)st->x : nullptr;
    const int64_t lb = logical_block();
    const int64_t start = lb * chunk;
    const int64_t end = start + chunk < n ? start + chunk : n;
    const int tr = threadIdx.x / NV, k = threadIdx.x % NV;
    double part[ND > 0 ? ND : 1];
#pragma unroll
    for (int d = 0; d < (ND > 0 ? ND : 1); ++d)
        part[d] = 0.0;
    double c1 = 0, c2 = 0, c3 = 0;
    if constexpr (OP == V_S_UPDATE) {
        c1 = st->nalpha[k];
    } else if constexpr (OP == V_XR_UPDATE) {
        c1 = st->ac[k];
        c2 = st->oc[k];
        c3 = st->omega[k];
    } else if constexpr (OP == V_X_UPDATE) {
        c1 = st->ac[k];
        c2 = st->oc[k];
    } else if constexpr (OP == V_R_UPDATE) {
        c3 = st->omega[k];
    } else if constexpr (OP == V_P_UPDATE) {
        c1 = st->pcoef[k];
        c2 = st->beta[k];
    } else if constexpr (OP == V_GROUP5) {
        c1 = st->ac[k];
        c2 = st->oc[k];
        c3 = st->beta[k] * st->omega[k];
    } else if constexpr (OP == V_CG_XR) {
        c1 = st->ac[k];
        c2 = st->nalpha[k];
    } else if constexpr (OP == V_CG_P) {
        c1 = st->beta[k];
    } else if constexpr (OP == V_RB_UPDATE) {
        c1 = st->ac[k];
        c2 = st->oc[k];
        c3 = st->nomega[k];
    } else if constexpr (OP == V_RB_UPDATE_MERGED) {
        c1 = st->ac[k];
        c2 = st->oc[k];
        c3 = st->nomega[k];
    }
    // RBiCGStab step 25 coefficients: (-omega)*beta (ax_y(omega, beta, delta) with omega
    // negated) for the plain form, beta*omega for merged_rbicgstab_group2
    const double be = (OP == V_RB_UPDATE || OP == V_RB_UPDATE_MERGED) ? st->beta[k] : 0.0;
    const double d2 = (OP == V_RB_UPDATE) ? st->nomega[k] * be : 0.0;
    const double om = (OP == V_RB_UPDATE_MERGED) ? st->omega[k] : 0.0;
    const double bo = (OP == V_RB_UPDATE_MERGED) ? be * om : 0.0;
    // unrolled so that the loads of several rows are in flight together; each thread
    // still visits its rows, and adds its dot terms, in row order
#pragma unroll 4
    for (int64_t i = start + tr; i < end; i += RPB) {
        const size_t o = (size_t)i * NV + k;
        if constexpr (OP == V_S_UPDATE) {
            // axpby_z(a1, r, -alpha, v, s): s = 1*r + (-alpha)*v
            s[o] = r[o] + c1 * v[o];
        } else if constexpr (OP == V_XR_UPDATE) {
            // axpbypcz(ac, p_, oc, s_, a1, x) then merged_bicgstab_group4
            x[o] = c1 * p_[o] + c2 * s_[o] + x[o];
            const double rv = s[o] - c3 * t[o];
            r[o] = rv;
            part[0] = part[0] + rv * r0[o];
        } else if constexpr (OP == V_X_UPDATE) {
            x[o] = c1 * p_[o] + c2 * s_[o] + x[o];
        } else if constexpr (OP == V_R_UPDATE) {
            const double rv = s[o] - c3 * t[o];
            r[o] = rv;
            part[0] = part[0] + rv * r0[o];
        } else if constexpr (OP == V_P_UPDATE) {
            // axpbypcz(a1, r, -(omega*beta), v, beta, p)
            p[o] = r[o] + c1 * v[o] + c2 * p[o];
        } else if constexpr (OP == V_GROUP5) {
            x[o] += c1 * p[o] + c2 * s[o];
            p[o] = r[o] + st->beta[k] * p[o] - c3 * v[o];
        } else if constexpr (OP == V_DOT3) {
            const double tv = t[o], sv = s[o];
            part[0] = part[0] + tv * sv;
            part[1] = part[1] + tv * tv;
            part[2] = part[2] + sv * sv;
        } else if constexpr (OP == V_DOT1) {
            part[0] = part[0] + r[o] * r0[o];
        } else if constexpr (OP == V_CG_XR) {
            // axpby(alpha_conv, p, a1, x) ; axpby(-alpha, Ap, a1, r)
            x[o] = c1 * p_[o] + x[o];
            r[o] = c2 * t[o] + r[o];
        } else if constexpr (OP == V_DOT2) {
            const double rv = r[o], zv = r0[o];
            part[0] = part[0] + rv * zv;
            part[1] = part[1] + rv * rv;
        } else if constexpr (OP == V_CG_P) {
            p[o] = v[o] + c1 * p[o]; // axpby(a1, z, beta, p)
        } else if constexpr (OP == V_COPY_DOT) {
            const double zv = v[o];
            p[o] = zv;
            part[0] = part[0] + r[o] * zv;
        } else if constexpr (OP == V_COPY) {
            p[o] = v[o];
        } else if constexpr (OP == V_RB_UPDATE) {
            r[o] = c3 * t[o] + r[o];                  // 16: axpby(-omega, t, a1, r)
            x[o] = c1 * p[o] + c2 * p_[o] + x[o];     // 23: axpbypcz(ac, v_, oc, t_, a1, x)
            const double zn = p_[o] + c3 * s[o];      // 24: axpby(a1, t_, -omega, z)
            s[o] = zn;
            p[o] = zn + d2 * v[o] + be * p[o];        // 25: axpbypcz(a1, z, delta, s, beta, v_)
        } else if constexpr (OP == V_RB_UPDATE_MERGED) {
            r[o] = c3 * t[o] + r[o];                  // 16
            x[o] += c1 * p[o] + c2 * p_[o];           // group2: x += ac v_ + oc t_
            const double zn = p_[o] - om * s[o];      //         z = t_ - omega z
            s[o] = zn;
            p[o] = zn + be * p[o] - bo * v[o];        //         v_ = z + beta v_ - beta omega s
        }
    }
    if constexpr (ND > 0)
        block_partials<NV, ND>(part, partials, lb);
}

template <int NV>
int vec_nv(VecOp op, int64_t n, const VecArgs &a, int gate, hipStream_t s) {
    const int rpb = kBlock / NV;
    const bool dots = (op == V_XR_UPDATE || op == V_R_UPDATE || op == V_DOT1 || op == V_DOT3 ||
                       op == V_DOT2 || op == V_COPY_DOT);
    int64_t need = (n + rpb - 1) / rpb;
    int64_t g = std::min<int64_t>(need, dots ? g_tune.vec_dot_groups : 8192);
    g = std::max<int64_t>(8, (g + 7) / 8 * 8);
    int64_t chunk = (n + g - 1) / g;
    chunk = (chunk + rpb - 1) / rpb * rpb;
#define XH_VEC_CASE(OPV)                                                                        \
    case OPV:                                                                                   \
        hipLaunchKernelGGL((k_vec<NV, OPV>), dim3(g), dim3(kBlock), 0, s, n, chunk,             \
                           (double *)a.p, (double *)a.s, (double *)a.r,                         \
                           (const double *)a.r0, (const double *)a.v, (const double *)a.t,      \
                           (const double *)a.p_, (const double *)a.s_, a.st, gate, a.partials); \
        break;
    switch (op) {
        XH_VEC_CASE(V_S_UPDATE)
        XH_VEC_CASE(V_XR_UPDATE)
        XH_VEC_CASE(V_P_UPDATE)
        XH_VEC_CASE(V_X_UPDATE)
        XH_VEC_CASE(V_R_UPDATE)
        XH_VEC_CASE(V_GROUP5)
        XH_VEC_CASE(V_DOT3)
        XH_VEC_CASE(V_DOT1)
        XH_VEC_CASE(V_CG_XR)
        XH_VEC_CASE(V_DOT2)
        XH_VEC_CASE(V_CG_P)
        XH_VEC_CASE(V_COPY_DOT)
        XH_VEC_CASE(V_COPY)
        XH_VEC_CASE(V_RB_UPDATE)
        XH_VEC_CASE(V_RB_UPDATE_MERGED)
    default:
        return -1;
    }
#undef XH_VEC_CASE
    return dots ? (int)g : 0;
}

// ---- finalize: partial sums -> Krylov scalars and the convergence decision ----

__global__ __launch_bounds__(256) void k_finalize(int op, SolverState *__restrict__ st,
                                                  const double *__restrict__ partials,
                                                  int nparts, int nv) {
    finalize_body(op, st, partials, nparts, nv, fin_ndots(op) * nv);
}

// ---- smoother / coarse / conversion kernels ----

template <typename VT>
__global__ __launch_bounds__(kBlock) void k_cheb_init_zero(int64_t count, int nv,
                                                           const VT *__restrict__ b,
                                                           const VT *__restrict__ isd, VT c,
                                                           VT *__restrict__ r,
                                                           VT *__restrict__ u, int last,
                                                           const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    // get_residual with a zero-flagged x gives r = 1*b; r *= isd; t1 = c*r; t1 *= isd
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < count;
         e += (int64_t)gridDim.x * kBlock) {
        const VT di = isd[e / nv];
        const VT rv = b[e] * di;
        VT t1 = c * rv;
        t1 = t1 * di;
        if (!last)
            r[e] = rv;
        u[e] = t1;
    }
}

template <typename VT>
__global__ __launch_bounds__(kBlock) void k_jacobi(int64_t count, int nv, VT *__restrict__ x,
                                                   const VT *__restrict__ b,
                                                   const VT *__restrict__ r,
                                                   const VT *__restrict__ invd, VT relax,
                                                   int x_zero, const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < count;
         e += (int64_t)gridDim.x * kBlock) {
        const VT d = invd[e / nv];
        if (x_zero)
            x[e] = relax * d * b[e];
        else
            x[e] += relax * d * (b[e] - r[e]);
    }
}

// y = D x with one output per thread, which walks its n columns in memory: the small products,
// whose whole D is a tile or less, and products called on their own (dense_tiled)
template <typename VT, typename XT>
__global__ __launch_bounds__(kBlock) void k_dense_direct(int64_t n, int nv,
                                                         const VT *__restrict__ D,
                                                         const XT *__restrict__ x,
                                                         XT *__restrict__ y,
                                                         const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    const int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (e >= n * nv)
        return;
    const int64_t i = e / nv;
    const int k = (int)(e % nv);
    VT acc = VT(0);
    // j order as dense_Ax_y; unrolled so that many loads are in flight
#pragma unroll 16
    for (int64_t j = 0; j < n; ++j)
        acc = acc + D[i * n + j] * (VT)x[j * nv + k];
    y[e] = (XT)acc;
}

// y = D x, D dense n x n (the coarsest level's inverse, n of a few hundred): every output is
// a sum of n terms added one by one in column order (the rounding of dense_Ax_y), so the
// time cannot go below n dependent adds; what is left to hide is memory.  A workgroup owns
// RB rows and all NV right-hand sides (one output per thread) and walks the columns in
// tiles of TJ: D and x tiles go through double-buffered LDS, loaded NS tiles ahead into
// registers, all threads loading contiguous rows.  A small product runs two waves per
// workgroup, spread over the CUs; a large one shares each x tile among four.  One output
// per thread reading memory itself waited for a load round trip every 16 terms: n = 500,
// nv = 32, fp64: 23.7 us; here 12.8 (four waves and two tiles ahead: 13.8), of which the 500
// dependent adds behind their LDS reads take about 5.  XT: type of x and y in memory
// (float with a double D: the fp64 coarse solve of an fp32 hierarchy, each value converted
// once as a separate pass would).
template <int NV, int WV>
struct DenseShape {
    static constexpr int T = 64 * WV; // threads
    static constexpr int RB = T / NV < 32 ? T / NV : 32; // rows
};
template <typename VT, typename XT, int NV, int WV>
__global__ __launch_bounds__(64 * WV) void k_dense(int64_t n, const VT *__restrict__ D,
                                                   const XT *__restrict__ x, XT *__restrict__ y,
                                                   const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    constexpr int RB = DenseShape<NV, WV>::RB, T = 64 * WV, TJ = 64, NS = 4;
    constexpr int DS = TJ + 16 / (int)sizeof(VT); // padded D row: 16-byte aligned, spread banks
    constexpr int PX = (TJ * NV + T - 1) / T, PD = (RB * TJ + T - 1) / T;
    __shared__ __align__(16) VT sx[2][TJ * NV];
    __shared__ __align__(16) VT sd[2][RB * DS];
    const int tid = threadIdx.x;
    const int64_t i0 = (int64_t)blockIdx.x * RB;
    const int r = tid / NV, k = tid % NV; // the thread's output (threads past RB rows have none)
    VT rx[NS][PX], rd[NS][PD];
    // tile loads, clamped into the arrays: entries past column n - 1 or row n - 1 are
    // never used
    auto load = [&](int64_t j0, VT (&ax)[PX], VT (&ad)[PD]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < PX; ++u) {
            const int64_t e = j0 * NV + tid + u * T;
            ax[u] = (VT)x[e < n * NV ? e : n * NV - 1];
        }
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            const int e = tid + u * T, row = e / TJ, c = e % TJ;
            const int64_t i = i0 + row < n ? i0 + row : n - 1;
            const int64_t j = j0 + c < n ? j0 + c : n - 1;
            ad[u] = D[i * n + j];
        }
    };
    auto store = [&](int b, const VT (&ax)[PX], const VT (&ad)[PD]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < PX; ++u)
            if (TJ * NV % T == 0 || tid + u * T < TJ * NV)
                sx[b][tid + u * T] = ax[u];
#pragma unroll
        for (int u = 0; u < PD; ++u) {
            const int e = tid + u * T;
            if (RB * TJ % T == 0 || e < RB * TJ)
                sd[b][(e / TJ) * DS + e % TJ] = ad[u];
        }
    };
    VT acc = VT(0);
    const bool mine = r < RB && i0 + r < n;
    auto tile = [&](int b, int64_t j0) __attribute__((always_inline)) {
        const VT *px = sx[b] + k, *pd = sd[b] + (r < RB ? r : 0) * DS;
        const int m = (int)(n - j0 < TJ ? n - j0 : TJ);
        if (m == TJ) {
#pragma unroll 16
            for (int j = 0; j < TJ; ++j)
                acc = acc + pd[j] * px[j * NV];
        } else {
            for (int j = 0; j < m; ++j)
                acc = acc + pd[j] * px[j * NV];
        }
    };
#pragma unroll
    for (int q = 0; q < NS; ++q)
        load((int64_t)q * TJ, rx[q], rd[q]);
    for (int64_t j0 = 0; j0 < n; j0 += NS * TJ) {
#pragma unroll
        for (int q = 0; q < NS; ++q) {
            // an LDS buffer is written two tiles after its last reads, which the barrier
            // of the tile between them has ordered
            if (j0 + q * TJ < n) { // uniform
                store(q & 1, rx[q], rd[q]);
                load(j0 + (int64_t)(q + NS) * TJ, rx[q], rd[q]);
                __syncthreads();
                tile(q & 1, j0 + (int64_t)q * TJ);
            }
        }
    }
    if (mine)
        y[(i0 + r) * NV + k] = (XT)acc;
}

template <typename T1, typename T2>
__global__ __launch_bounds__(kBlock) void k_convert(int64_t count, const T1 *__restrict__ a,
                                                    T2 *__restrict__ b,
                                                    const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < count;
         e += (int64_t)gridDim.x * kBlock)
        b[e] = (T2)a[e];
}

// x_c[c][k] = x_full[col_ind[c] + off][k]: the column decode of a compressed block
// (col_ind[col[j]] + block_col_offset, csr_matrix.h:290-297) applied to the operand
template <typename T>
__global__ __launch_bounds__(kBlock) void k_gather_cols(int64_t count, int nv,
                                                        const uint32_t *__restrict__ col_ind,
                                                        int64_t off, const T *__restrict__ xf,
                                                        T *__restrict__ xc) {
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < count;
         e += (int64_t)gridDim.x * kBlock) {
        const int64_t c = e / nv, k = e - c * nv;
        xc[e] = xf[((int64_t)col_ind[c] + off) * nv + k];
    }
}

// b[p][k] = sum over the bumps of RHS k of a exp(-|x_p - c|^2 / (2 w^2)), cells within the
// box of half-width ceil(4w) around c only (cell centres at integer + 0.5)
__global__ __launch_bounds__(kBlock) void k_bumps(int nx, int ny, int nz, int nv, int maxb,
                                                  const int *__restrict__ count,
                                                  const double *__restrict__ P,
                                                  double *__restrict__ b) {
    const int64_t n = (int64_t)nx * ny * nz * nv;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * kBlock) {
        const int k = (int)(e % nv);
        const int64_t p = e / nv;
        const int x = (int)(p % nx), y = (int)((p / nx) % ny), z = (int)(p / ((int64_t)nx * ny));
        double s = 0.0;
        for (int q = 0; q < count[k]; ++q) {
            const double *Q = P + ((size_t)k * maxb + q) * 5;
            const double w = Q[3];
            const int64_t R = (int64_t)ceil(4.0 * w);
            if (x < (int64_t)Q[0] - R || x > (int64_t)Q[0] + R || y < (int64_t)Q[1] - R ||
                y > (int64_t)Q[1] + R || z < (int64_t)Q[2] - R || z > (int64_t)Q[2] + R)
                continue;
            const double dx = (double)x + 0.5 - Q[0], dy = (double)y + 0.5 - Q[1],
                         dz = (double)z + 0.5 - Q[2];
            s += Q[4] * exp(-(dx * dx + dy * dy + dz * dz) * (1.0 / (2.0 * w * w)));
        }
        b[e] = s;
    }
}

// x = u + x (the axpby(a1, t1, a1, x) that ends a Chebyshev application,
// chebyshev.inl:201-202)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_add(int64_t count, const T *__restrict__ u,
                                                T *__restrict__ x, const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < count;
         e += (int64_t)gridDim.x * kBlock)
        x[e] = u[e] + x[e];
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_fill0(int64_t count, T *__restrict__ b,
                                                  const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < count;
         e += (int64_t)gridDim.x * kBlock)
        b[e] = T(0);
}

int grid_for(int64_t count) {
    int64_t g = (count + kBlock - 1) / kBlock;
    g = std::min<int64_t>(g, 16384);
    return (int)std::max<int64_t>(1, g);
}

} // namespace

namespace {

// vectors of n x nv doubles each vector op reads plus writes, and its dot count
int vec_streams(VecOp op) {
    static const int rw[] = {3, 8, 4, 5, 4, 4, 7, 2, 2, 6, 2, 3, 3, 2, 11, 11};
    return (op >= 0 && op <= V_RB_UPDATE_MERGED) ? rw[op] : 0;
}
int vec_ndots(VecOp op) {
    return (op == V_XR_UPDATE || op == V_R_UPDATE || op == V_DOT1 || op == V_COPY_DOT) ? 1
           : op == V_DOT2                                                             ? 2
           : op == V_DOT3                                                             ? 3
                                                                                      : 0;
}
const char *vec_name(VecOp op) {
    static const char *names[] = {"V_S_UPDATE", "V_XR_UPDATE", "V_P_UPDATE", "V_GROUP1",
                                  "V_X_UPDATE", "V_R_UPDATE", "V_GROUP5", "V_DOT3", "V_DOT1",
                                  "V_CG_XR", "V_DOT2", "V_CG_P", "V_COPY_DOT", "V_COPY",
                                  "V_RB_UPDATE", "V_RB_UPDATE_MERGED"};
    return (op >= 0 && op <= V_RB_UPDATE_MERGED) ? names[op] : "V_?";
}

int vec_dispatch(VecOp op, int64_t n, int nv, const VecArgs &a, hipStream_t s) {
    const int gate = a.gate;
    const VecArgs &b = a;
    switch (nv) {
    case 1:
        return vec_nv<1>(op, n, b, gate, s);
    case 2:
        return vec_nv<2>(op, n, b, gate, s);
    case 4:
        return vec_nv<4>(op, n, b, gate, s);
    case 8:
        return vec_nv<8>(op, n, b, gate, s);
    case 16:
        return vec_nv<16>(op, n, b, gate, s);
    case 32:
        return vec_nv<32>(op, n, b, gate, s);
    case 64:
        return vec_nv<64>(op, n, b, gate, s);
    default:
        return -1;
    }
}

} // namespace

int vec_op(VecOp op, int64_t n, int nv, const VecArgs &a, hipStream_t s) {
    LedgerScope led(s);
    const int np = vec_dispatch(op, n, nv, a, s);
    if (led.on) {
        led.kernel = std::string("k_vec<") + std::to_string(nv) + "," + vec_name(op) + ">";
        led.bytes = (double)vec_streams(op) * n * nv * 8.0 +
                    (np > 0 ? (double)np * vec_ndots(op) * nv * 8.0 : 0.0);
    }
    return np;
}

void finalize(FinOp op, SolverState *st, const double *partials, int nparts, int nv,
              hipStream_t s) {
    LedgerScope led(s);
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(256), 0, s, (int)op, st, partials, nparts, nv);
    if (led.on) {
        led.kernel = "k_finalize";
        led.bytes = (double)nparts * fin_ndots(op) * nv * 8.0;
    }
}

void cheb_init_zero(int64_t n, int nv, int prec, const void *b, const void *isd, double c,
                    void *r, void *u_or_x, int last, const int *done, hipStream_t s) {
    const int64_t count = n * nv;
    LedgerScope led(s);
    if (led.on) {
        const double sv = prec == F64 ? 8.0 : 4.0;
        led.kernel = std::string("k_cheb_init_zero<") + prec_name(prec) + ">";
        led.bytes = sv * (double)(count * (last ? 2 : 3) + n); // b, isd ; u or x (and r)
    }
    if (prec == F64)
        hipLaunchKernelGGL(k_cheb_init_zero<double>, dim3(grid_for(count)), dim3(kBlock), 0, s,
                           count, nv, (const double *)b, (const double *)isd, c, (double *)r,
                           (double *)u_or_x, last, done);
    else
        hipLaunchKernelGGL(k_cheb_init_zero<float>, dim3(grid_for(count)), dim3(kBlock), 0, s,
                           count, nv, (const float *)b, (const float *)isd, (float)c,
                           (float *)r, (float *)u_or_x, last, done);
}

void jacobi_update(int64_t n, int nv, int prec, void *x, const void *b, const void *r,
                   const void *inv_diag, double relax, int x_zero, const int *done,
                   hipStream_t s) {
    const int64_t count = n * nv;
    LedgerScope led(s);
    if (led.on) {
        const double sv = prec == F64 ? 8.0 : 4.0;
        led.kernel = std::string("k_jacobi<") + prec_name(prec) + ">";
        // b, inverse diagonal ; x written (x and r read unless x is zero-flagged)
        led.bytes = sv * (double)(count * (x_zero ? 2 : 4) + n);
    }
    if (prec == F64)
        hipLaunchKernelGGL(k_jacobi<double>, dim3(grid_for(count)), dim3(kBlock), 0, s, count,
                           nv, (double *)x, (const double *)b, (const double *)r,
                           (const double *)inv_diag, relax, x_zero, done);
    else
        hipLaunchKernelGGL(k_jacobi<float>, dim3(grid_for(count)), dim3(kBlock), 0, s, count,
                           nv, (float *)x, (const float *)b, (const float *)r,
                           (const float *)inv_diag, (float)relax, x_zero, done);
}

// Whether the product runs in tiles (k_dense).  Inside a solve D has left the L2 caches since
// its last use, and the tiles, loaded four ahead, hide that: event-timed launches in us,
// direct / tiled: fp64 nv = 8, n = 45 7.7 / 6.4, nv = 64, n = 512 33 / 26, 1000 70 / 55; fp32 nv =
// 16, n = 512 18.6 / 16.7, 1728 64 / 46.  Only 64 right-hand sides and a D of less than a tile
// are better without (n = 33 6.4 / 9.2, 45 9.9 / 9.7).
// Called on its own, again on the same D (warm), a small product pays for the tiles'
// barriers, and with 64 right-hand sides, or 16 and 32 in fp32, a whole wave reads a row of D
// at once already.  us per call, direct / tiled: fp64 nv = 8, n = 48 14.6 / 14.7, 100 17.1 / 16.3,
// 500 33.6 / 26.1; nv = 64, n = 100 17.4 / 20.0, 1000 57.1 / 63.2, 1200 114 / 64; fp32 nv = 8, n = 160
// 15.6 / 15.7, 200 17.0 / 16.2; nv = 16, n = 500 22.9 / 24.8, 2500 65 / 77, 3000 110 / 89; nv = 32, n =
// 257 17.9 / 18.8, 500 23.0 / 22.3; nv = 64, n = 1000 34.4 / 41.7, 1200 50.5 / 41.0.
bool dense_tiled(int64_t n, int nv, int prec, bool warm) {
    if (!warm)
        return nv < 64 || n >= 40;
    if (nv == 64)
        return n >= 1100;
    if (prec == F64)
        return n >= 96;
    return n >= (nv <= 8 ? 180 : nv == 16 ? 2800 : 450);
}

template <typename VT, typename XT, int NV>
void dense_t(int64_t n, const void *D, const void *x, void *y, const int *done, hipStream_t s) {
    // two waves per workgroup while that gives at most 2 workgroups per CU
    constexpr int R1 = DenseShape<NV, 2>::RB, R4 = DenseShape<NV, 4>::RB;
    if (R1 == R4 || (n + R1 - 1) / R1 <= 512)
        hipLaunchKernelGGL((k_dense<VT, XT, NV, 2>), dim3((unsigned)((n + R1 - 1) / R1)), dim3(128),
                           0, s, n, (const VT *)D, (const XT *)x, (XT *)y, done);
    else
        hipLaunchKernelGGL((k_dense<VT, XT, NV, 4>), dim3((unsigned)((n + R4 - 1) / R4)), dim3(256),
                           0, s, n, (const VT *)D, (const XT *)x, (XT *)y, done);
}

template <typename VT, typename XT>
void dense_nv(int64_t n, int nv, const void *D, const void *x, void *y, bool tiled,
              const int *done, hipStream_t s) {
    if (!tiled) {
        const dim3 grid((unsigned)((n * nv + kBlock - 1) / kBlock));
        hipLaunchKernelGGL((k_dense_direct<VT, XT>), grid, dim3(kBlock), 0, s, n, nv, (const VT *)D,
                           (const XT *)x, (XT *)y, done);
        return;
    }
    switch (nv) {
    case 1:
        return dense_t<VT, XT, 1>(n, D, x, y, done, s);
    case 2:
        return dense_t<VT, XT, 2>(n, D, x, y, done, s);
    case 4:
        return dense_t<VT, XT, 4>(n, D, x, y, done, s);
    case 8:
        return dense_t<VT, XT, 8>(n, D, x, y, done, s);
    case 16:
        return dense_t<VT, XT, 16>(n, D, x, y, done, s);
    case 32:
        return dense_t<VT, XT, 32>(n, D, x, y, done, s);
    default:
        return dense_t<VT, XT, 64>(n, D, x, y, done, s);
    }
}

void dense_matvec(int64_t n, int nv, int prec, int xprec, const void *D, const void *x, void *y,
                  bool warm, const int *done, hipStream_t s) {
    LedgerScope led(s);
    const bool tiled = dense_tiled(n, nv, prec, warm);
    if (led.on) {
        const double sv = prec == F64 ? 8.0 : 4.0, sx = xprec == F64 ? 8.0 : 4.0;
        led.kernel = std::string(tiled ? "k_dense<" : "k_dense_direct<") +
                     prec_name(prec) + "," + prec_name(xprec) + ">";
        led.bytes = sv * (double)(n * n) + 2.0 * sx * (double)(n * nv); // D, x, y
    }
    if (prec == F64 && xprec == F64)
        dense_nv<double, double>(n, nv, D, x, y, tiled, done, s);
    else if (prec == F64)
        dense_nv<double, float>(n, nv, D, x, y, tiled, done, s);
    else
        dense_nv<float, float>(n, nv, D, x, y, tiled, done, s);
}

void convert(int64_t count, int from_prec, const void *src, void *dst, const int *done,
             hipStream_t s) {
    LedgerScope led(s);
    if (led.on) {
        led.kernel = from_prec == F64 ? "k_convert<double,float>" : "k_convert<float,double>";
        led.bytes = 12.0 * (double)count;
    }
    if (from_prec == F64)
        hipLaunchKernelGGL((k_convert<double, float>), dim3(grid_for(count)), dim3(kBlock), 0, s,
                           count, (const double *)src, (float *)dst, done);
    else
        hipLaunchKernelGGL((k_convert<float, double>), dim3(grid_for(count)), dim3(kBlock), 0, s,
                           count, (const float *)src, (double *)dst, done);
}

void add_vec(int64_t count, int prec, const void *u, void *x, const int *done, hipStream_t s) {
    LedgerScope led(s);
    if (led.on) {
        led.kernel = std::string("k_add<") + prec_name(prec) + ">";
        led.bytes = (prec == F64 ? 24.0 : 12.0) * (double)count;
    }
    if (prec == F64)
        hipLaunchKernelGGL(k_add<double>, dim3(grid_for(count)), dim3(kBlock), 0, s, count,
                           (const double *)u, (double *)x, done);
    else
        hipLaunchKernelGGL(k_add<float>, dim3(grid_for(count)), dim3(kBlock), 0, s, count,
                           (const float *)u, (float *)x, done);
}

void copy_vec(int64_t count, int prec, const void *src, void *dst, const int *done,
              hipStream_t s) {
    LedgerScope led(s);
    if (led.on) {
        led.kernel = std::string("k_convert<") + prec_name(prec) + "," + prec_name(prec) + ">";
        led.bytes = (prec == F64 ? 16.0 : 8.0) * (double)count;
    }
    if (prec == F64)
        hipLaunchKernelGGL((k_convert<double, double>), dim3(grid_for(count)), dim3(kBlock), 0,
                           s, count, (const double *)src, (double *)dst, done);
    else
        hipLaunchKernelGGL((k_convert<float, float>), dim3(grid_for(count)), dim3(kBlock), 0, s,
                           count, (const float *)src, (float *)dst, done);
}

void gather_cols(int64_t nc, int nv, int prec, const uint32_t *col_ind, int64_t off,
                 const void *x_full, void *x_c, hipStream_t s) {
    const int64_t count = nc * nv;
    if (count == 0)
        return;
    if (prec == F64)
        hipLaunchKernelGGL(k_gather_cols<double>, dim3(grid_for(count)), dim3(kBlock), 0, s,
                           count, nv, col_ind, off, (const double *)x_full, (double *)x_c);
    else
        hipLaunchKernelGGL(k_gather_cols<float>, dim3(grid_for(count)), dim3(kBlock), 0, s,
                           count, nv, col_ind, off, (const float *)x_full, (float *)x_c);
}

void eval_bumps(int nx, int ny, int nz, int nv, int maxb, const int *count, const double *P,
                double *b, hipStream_t s) {
    const int64_t n = (int64_t)nx * ny * nz * nv;
    hipLaunchKernelGGL(k_bumps, dim3(grid_for(n)), dim3(kBlock), 0, s, nx, ny, nz, nv, maxb,
                       count, P, b);
}

void fill_zero(int64_t count, int prec, void *dst, const int *done, hipStream_t s) {
    LedgerScope led(s);
    if (led.on) {
        led.kernel = std::string("k_fill0<") + prec_name(prec) + ">";
        led.bytes = (prec == F64 ? 8.0 : 4.0) * (double)count;
    }
    if (prec == F64)
        hipLaunchKernelGGL(k_fill0<double>, dim3(grid_for(count)), dim3(kBlock), 0, s, count,
                           (double *)dst, done);
    else
        hipLaunchKernelGGL(k_fill0<float>, dim3(grid_for(count)), dim3(kBlock), 0, s, count,
                           (float *)dst, done);
}

} // namespace xh
