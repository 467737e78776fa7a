// Multi-RHS CSR SpMV for few, long rows: the coarse levels of a hierarchy.
//
// Such a launch leaves most of the GPU idle; its time is the chain of memory round trips of
// one row.  The row-parallel kernel (xh_spmv.hip) gives a row L = NV/W lanes, which walk its
// entries in batches of 8: a 93-entry row waits 12 times.  Here a group of GL > L lanes
// owns the row: its lanes load the columns and values of up to CH entries at once, then
// all their x rows at once, round every product, and put the products in LDS by entry.  The
// first L lanes then add them one by one in stored order, so each RHS gets the sum of
// csr_Ax_y (src/blas2/detail/csr_matvec.inl:149-260) exactly, and run the epilogue, whose
// operands were loaded before the entries.  A row costs about three dependent memory
// round trips (row pointers, columns, x) instead of two per batch.
#include "xh_internal.hpp"
#include "xh_spmv_dev.hpp"

#include <algorithm>

namespace xh {
namespace {

// EPX: entries of a row loaded side by side (at most; 64 lanes hold 64 / L)
template <typename VT, int NV, int EPX>
struct WaveShape {
    static constexpr int W = Width<VT, NV>::value;
    static constexpr int L = NV / W;                       // lanes per entry and per sum
    static constexpr int EP = EPX * L > 64 ? 64 / L : EPX; // entries loaded side by side
    static constexpr int GL = EP * L;                      // lanes per row
    static constexpr int G = 64 / GL;                      // rows per wave
    static constexpr int CH = EPX == 16 && EP >= 4 ? 64 : 32; // entries per pass
    static constexpr int Q = CH / EP;                      // x loads in flight per lane
    // products of one row in LDS; the pad keeps the sums of the wave's rows on different
    // banks
    static constexpr int STRIDE = CH * NV + 16 / (int)sizeof(VT);
};

template <typename VT, typename IT, int NV, int OP, int EPX>
__global__ __launch_bounds__(64) void k_spmv_wave(
    const uint32_t *__restrict__ row, const IT *__restrict__ col, const VT *__restrict__ val,
    const uint32_t *__restrict__ pbase, int shift, int64_t nrows, const VT *__restrict__ x,
    void *__restrict__ yv, const VT *__restrict__ b, const VT *__restrict__ isd,
    const VT *__restrict__ rr, VT *__restrict__ out2, void *__restrict__ xupdv, VT c, int last,
    int x_zero, int out_f32, const int *__restrict__ done, VT c2) {
    using S = WaveShape<VT, NV, EPX>;
    constexpr int W = S::W, L = S::L, GL = S::GL, EP = S::EP, CH = S::CH, Q = S::Q;
    using P = Pack<VT, W>;
    __shared__ __align__(16) VT prod[S::G * S::STRIDE];
    if (done != nullptr && *done)
        return;
    const int lane = threadIdx.x, gl = lane % GL, el = gl / L, k0 = (gl % L) * W;
    const int64_t i = (int64_t)blockIdx.x * S::G + lane / GL;
    if (i >= nrows)
        return; // a whole group
    const uint32_t jb = row[i], je = row[i + 1];
    const uint32_t base = panel_base<IT>(pbase, shift, i);
    const size_t o = (size_t)i * NV + k0;
    const bool sums = el == 0; // the lanes that add and store
    EpiIn<VT, W> in;
    if (sums)
        epi_load<VT, NV, W, OP>(i, o, o, k0, in, yv, b, nullptr, isd, rr, out2, xupdv, last,
                                x_zero);
    uint32_t cq[Q];
    VT vq[Q];
    auto entries = [&](uint32_t j) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const uint32_t e = j + q * EP + el;
            if (e < je) {
                cq[q] = base + (uint32_t)col[e];
                vq[q] = val[e];
            }
        }
    };
    VT acc[W];
#pragma unroll
    for (int w = 0; w < W; ++w)
        acc[w] = VT(0);
    if (OP == OP_ADD && sums)
#pragma unroll
        for (int w = 0; w < W; ++w)
            acc[w] = in.a.v[w];
    VT *mine = prod + (lane / GL) * S::STRIDE;
    entries(jb);
    for (uint32_t j = jb; j < je; j += CH) {
        P xv[Q];
        VT dq[OP == OP_CHEBZ ? Q : 1];
        VT pv[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            pv[q] = vq[q];
            if (j + q * EP + el < je) {
                xv[q] = ld<VT, W>(x + (size_t)cq[q] * NV + k0);
                if constexpr (OP == OP_CHEBZ)
                    dq[q] = isd[cq[q]];
            }
        }
        entries(j + CH); // of the next pass, in flight with this pass's x
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (j + q * EP + el < je) {
                P p;
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    VT xw = xv[q].v[w];
                    if constexpr (OP == OP_CHEBZ) { // the zero-x first step's value
                        xw = xw * dq[q];
                        xw = c2 * xw;
                        xw = xw * dq[q];
                    }
                    p.v[w] = xw * pv[q];
                }
                *reinterpret_cast<P *>(mine + (q * EP + el) * NV + k0) = p;
            }
        // one wave: its LDS accesses complete in order, the fences keep the compiler's too
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (sums) {
            // batches of 8, the next one read while the current one is added; reads past
            // the row's last entry stay inside the pass's CH slots and are not added
            const int n = je - j < (uint32_t)CH ? (int)(je - j) : CH;
            auto batch = [&](P(&t)[8], int e) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    t[u] = *reinterpret_cast<const P *>(mine + ((e + u) & (CH - 1)) * NV + k0);
            };
            auto add = [&](const P(&t)[8], int m) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (u < m)
#pragma unroll
                        for (int w = 0; w < W; ++w)
                            acc[w] = acc[w] + t[u].v[w];
            };
            P t0[8], t1[8];
            batch(t0, 0);
            int e = 0;
            for (; e + 16 <= n; e += 16) {
                batch(t1, e + 8);
                add(t0, 8);
                batch(t0, e + 16);
                add(t1, 8);
            }
            if (e + 8 <= n) {
                batch(t1, e + 8);
                add(t0, 8);
                add(t1, n - e - 8);
            } else {
                add(t0, n - e);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    if (sums) {
        double part[1][W];
        row_epilogue<VT, NV, W, OP>(o, o, acc, part, in, yv, out2, (VT *)nullptr, xupdv, c, last,
                                    x_zero, out_f32);
    }
}

template <typename VT, typename IT, int NV, int OP, int EPX>
void launch_ep(const Mat &A, const void *x, void *y, const SpmvArgs &a, hipStream_t s) {
    constexpr int G = WaveShape<VT, NV, EPX>::G;
    hipLaunchKernelGGL((k_spmv_wave<VT, IT, NV, OP, EPX>), dim3((unsigned)((A.nrows + G - 1) / G)),
                       dim3(64), 0, s, A.row, (const IT *)A.col, (const VT *)A.val, A.panel_base,
                       A.panel_shift, A.nrows, (const VT *)x, y, (const VT *)a.b,
                       (const VT *)a.isd, (const VT *)a.r, (VT *)a.out2, a.xupd, (VT)a.c, a.last,
                       a.x_zero, a.out_f32, a.done, (VT)a.c2);
}

template <typename VT, typename IT, int NV, int OP>
void launch(const Mat &A, const void *x, void *y, const SpmvArgs &a, hipStream_t s) {
    // one lane per entry and many rows: 4 lanes per row, so a wave's instructions serve 16
    // rows (262144 rows of 26 entries, us with 16 / 4 lanes: fp64 nv = 2 43 / 36, fp32 nv = 1
    // 24 / 18, nv = 4 44 / 26); with fewer rows than fill the chip the longer batches lose
    if constexpr (WaveShape<VT, NV, 4>::L == 1)
        if (wave_entries(A, NV) == 4)
            return launch_ep<VT, IT, NV, OP, 4>(A, x, y, a, s);
    launch_ep<VT, IT, NV, OP, 16>(A, x, y, a, s);
}

template <typename VT, typename IT, int NV>
void by_op(const Mat &A, const void *x, void *y, SpmvOp op, const SpmvArgs &a, hipStream_t s) {
    switch (op) {
    case OP_SET:
        return launch<VT, IT, NV, OP_SET>(A, x, y, a, s);
    case OP_ADD:
        return launch<VT, IT, NV, OP_ADD>(A, x, y, a, s);
    case OP_RESID:
        return launch<VT, IT, NV, OP_RESID>(A, x, y, a, s);
    case OP_CHEB0:
        return launch<VT, IT, NV, OP_CHEB0>(A, x, y, a, s);
    case OP_CHEB:
        return launch<VT, IT, NV, OP_CHEB>(A, x, y, a, s);
    case OP_CHEBZ:
        return launch<VT, IT, NV, OP_CHEBZ>(A, x, y, a, s);
    default:
        return launch<VT, IT, NV, OP_CHEBR>(A, x, y, a, s);
    }
}

template <typename VT, typename IT>
void by_nv(const Mat &A, int nv, const void *x, void *y, SpmvOp op, const SpmvArgs &a,
           hipStream_t s) {
    switch (nv) {
    case 1:
        return by_op<VT, IT, 1>(A, x, y, op, a, s);
    case 2:
        return by_op<VT, IT, 2>(A, x, y, op, a, s);
    case 4:
        return by_op<VT, IT, 4>(A, x, y, op, a, s);
    case 8:
        return by_op<VT, IT, 8>(A, x, y, op, a, s);
    case 16:
        return by_op<VT, IT, 16>(A, x, y, op, a, s);
    case 32:
        return by_op<VT, IT, 32>(A, x, y, op, a, s);
    default:
        return by_op<VT, IT, 64>(A, x, y, op, a, s);
    }
}

} // namespace

// Where this kernel is the faster one.  A wave here costs the instructions of a whole row
// (the sum runs in L of its 64 lanes) and saves the row-parallel kernel's wait per 8 entries,
// so it pays while the launch has few rows, and fewer the shorter they are.  The caps are
// where the two kernels' times crossed on 4080 matrices of hierarchies (all operators,
// prolongations and restrictions of 7- and 27-point grids of 20^3 to 128^3), time of the
// row-parallel kernel over this one's: L = 1 32768 rows of 7 0.78, 32768 of 25 1.4, 21952 of 7
// 1.3; L = 2 (nv = 4, fp64) 9910 of 9 0.95, 7500 of 6 1.2, 17391 of 38 1.14, 27366 of 24 0.7; L = 4
// (nv = 8) 3470 of 8 0.95, 2500 of 7 1.2, 6912 of 17 0.86, 5700 of 22 1.2, 7000 of 30 1.25, 8500 of
// 30 0.9; L = 8 (nv = 16) 3470 of 12 0.88, 2500 of 13 1.35, 4375 of 56 1.0; L = 16 (nv = 32) 400 of
// 6 0.93, 400 of 10 1.05, 440 of 38 1.3, 2200 of 25 0.8.  Below 4 entries a row is one batch
// there.
// One right-hand side, and two in fp32, win at every size with long rows (262144 rows of 26:
// fp64 nv = 1 52.9 / 24.8, fp32 nv = 2 41.1 / 21.8; 163868 rows of 14: 15.0 / 13.0, 12.6 /
// 11.7), as the row-parallel kernel then has each lane load its own entries.  Two in fp64
// win past the cap from 18 entries per row (442368 rows of 18.6: 55.6 / 50.7, 110592 of 26:
// 22.2 / 17.9; but 119404 of 16: 13.9 / 16.7, 955225 of 16: 91.3 / 106.4), and against the
// neighbour codes from 2^17 rows (135000 of 26: 22.8 / 21.1, 262144: 47.8 / 36.2; but 64000: 9.4
// / 12.1, 110592: 14.4 / 18.0).
bool takes_wave(const Mat &A, SpmvOp op, int nv) {
    if (!(op == OP_SET || op == OP_ADD || op == OP_RESID || op == OP_CHEB0 || op == OP_CHEB ||
          op == OP_CHEBZ || op == OP_CHEBR) ||
        A.idx == IDX_U8 || A.row_ind != nullptr || g_tune.wave_enable == 0)
        return false;
    if (g_tune.wave_enable == 1)
        return true;
    if (g_tune.wide_batches == 0 || A.nnz < 4 * A.nrows)
        return false;
    const bool longrows = A.nnz >= 12 * A.nrows;
    if (longrows && (nv == 1 || (nv == 2 && (A.prec == F32 ||
                                             (A.nnz >= 18 * A.nrows &&
                                              (!takes_codes(A, op, nv) || A.nrows >= 1 << 17))))))
        return true;
    const int L = nv / std::min(nv, A.prec == F64 ? 2 : 4);
    if (A.gcode != nullptr && L > 1)
        return false;
    // most rows by entries per row: 4 to 12, 12 to 26, more
    static const int64_t cap[5][3] = {{24576, 32768, 32768}, // L = 1
                                      {8192, 20480, 20480},  // 2
                                      {3072, 6144, 7680},    // 4
                                      {2048, 3072, 4096},    // 8
                                      {768, 1536, 1536}};    // 16
    if (L > 16 || (L == 16 && A.nnz < 9 * A.nrows))
        return false;
    return A.nrows <= cap[__builtin_ctz(L)][!longrows ? 0 : A.nnz < 26 * A.nrows ? 1 : 2];
}

int wave_entries(const Mat &A, int nv) {
    const int L = nv / std::min(nv, A.prec == F64 ? 2 : 4);
    if (L == 1 && A.nrows > 65536)
        return 4;
    return 16;
}

void spmv_wave(const Mat &A, int nv, const void *x, void *y, SpmvOp op, const SpmvArgs &a,
               hipStream_t s) {
    if (A.prec == F64)
        A.idx == IDX_U16 ? by_nv<double, uint16_t>(A, nv, x, y, op, a, s)
                         : by_nv<double, uint32_t>(A, nv, x, y, op, a, s);
    else
        A.idx == IDX_U16 ? by_nv<float, uint16_t>(A, nv, x, y, op, a, s)
                         : by_nv<float, uint32_t>(A, nv, x, y, op, a, s);
}

} // namespace xh
