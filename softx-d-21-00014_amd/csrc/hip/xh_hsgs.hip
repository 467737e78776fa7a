// Hybrid symmetric Gauss-Seidel sweeps (csr_SGS, src/blas2/detail/csr_gs.inl:33-134, driven
// by blas2::SGS, src/blas2/blas2.h:185-281): rows in core blocks of B rows, each block swept
// forward then backward in order by one group of NV lanes (one lane per right-hand side),
// blocks independent.  Built with -ffp-contract=off: products rounded, then subtracted one
// by one in stored order, as the reference's x86-64 build.
#include "xh_internal.hpp"

#include <algorithm>

namespace xh {
namespace {

// HSGS: one group of NV lanes sweeps one core block forward then backward; the block's
// x lives in LDS, each lane only touches its own RHS column so no barrier is needed.
template <typename VT, typename IT, int NV>
__global__ __launch_bounds__(64) void k_hsgs_lds(const uint32_t *__restrict__ row,
                                                 const IT *__restrict__ col,
                                                 const VT *__restrict__ val,
                                                 const uint32_t *__restrict__ pbase, int shift,
                                                 const VT *__restrict__ invd, int64_t n,
                                                 int64_t B, const VT *__restrict__ t,
                                                 VT *__restrict__ x, int x_zero, VT relax,
                                                 const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    extern __shared__ unsigned char smem[];
    constexpr int G = 64 / NV;
    const int g = threadIdx.x / NV, k = threadIdx.x % NV;
    VT *xs = (VT *)smem + (size_t)g * B * NV;
    const int64_t blk = (int64_t)blockIdx.x * G + g;
    const int64_t lo = blk * B;
    if (lo >= n)
        return;
    const int64_t hi = lo + B < n ? lo + B : n;
    for (int64_t i = lo; i < hi; ++i)
        xs[(i - lo) * NV + k] = x_zero ? VT(0) : x[(size_t)i * NV + k];
    for (int sweep = 0; sweep < 2; ++sweep) {
        for (int64_t q = 0; q < hi - lo; ++q) {
            const int64_t i = sweep == 0 ? lo + q : hi - 1 - q;
            uint32_t base = 0;
            if constexpr (sizeof(IT) == 2)
                base = pbase[i >> shift];
            VT sum = t[(size_t)i * NV + k];
            // unrolled so that the row's column and value loads are in flight together;
            // the subtractions keep the stored order
#pragma unroll 8
            for (uint32_t j = row[i]; j < row[i + 1]; ++j) {
                const int64_t c = (int64_t)(base + (uint32_t)col[j]);
                if (c >= lo && c < hi)
                    sum = sum - xs[(c - lo) * NV + k] * val[j];
            }
            const VT coeff = relax * invd[i];
            xs[(i - lo) * NV + k] = xs[(i - lo) * NV + k] + coeff * sum;
        }
    }
    for (int64_t i = lo; i < hi; ++i)
        x[(size_t)i * NV + k] = xs[(i - lo) * NV + k];
}

// Copies count elements from global memory into LDS with the lanes lane, lane + nl, ...;
// U loads are issued before their LDS writes so that a copy costs count / (nl * U) memory
// round trips instead of one per element.  16-byte vectors where both ends are aligned.
// Loads and stores past the end re-read and re-write the last element (always in
// bounds, same value), so that no load can be moved behind a branch and the batch stays
// in flight together.
template <typename VT, int U>
__device__ inline void stage_copy(VT *__restrict__ dst, const VT *__restrict__ src,
                                  int64_t count, int lane, int nl) {
    int64_t done_el = 0;
    if ((((uintptr_t)src | (uintptr_t)dst) & 15) == 0) {
        const int64_t nvec = count * (int64_t)sizeof(VT) / 16;
        const uint4 *s4 = (const uint4 *)src;
        uint4 *d4 = (uint4 *)dst;
        for (int64_t b = lane; b < nvec; b += (int64_t)nl * U) {
            uint4 r[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t i = b + (int64_t)u * nl;
                r[u] = s4[i < nvec ? i : nvec - 1];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t i = b + (int64_t)u * nl;
                d4[i < nvec ? i : nvec - 1] = r[u];
            }
        }
        done_el = nvec * 16 / (int64_t)sizeof(VT);
    }
    for (int64_t b = done_el + lane; b < count; b += (int64_t)nl * U) {
        VT r[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = b + (int64_t)u * nl;
            r[u] = src[i < count ? i : count - 1];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = b + (int64_t)u * nl;
            dst[i < count ? i : count - 1] = r[u];
        }
    }
}

// The same sweeps on a core-block matrix (only entries inside the row's block, u32
// columns; each row padded to whole batches of KB entries, pads pointing at the block's
// end with value +0).  gw groups of NV lanes per wave, one core block each; a group first
// stages its block's x, row pointers, x offsets of the columns, values and inverse diagonal
// in LDS (loads issued in batches), with one more x row of zeros at local row nr for the
// pads, then sweeps from LDS.  Entry order and arithmetic as k_hsgs_lds: the products
// x_c * a_ic are rounded, then subtracted from t one by one in stored order; a pad
// subtracts +0 * +0 = +0, which changes no value.  ONE: every row is one batch.
//
// A sweep is a serial chain of rows, one wave per SIMD or less, so what a row costs is the
// LDS round trip of its x operands (they may name the row just written) and the issue of its
// ~6 instructions per entry.  What can be read ahead is: t of the next R rows from memory
// while R rows are swept, the row pointers two rows ahead, and the columns and values of
// the next batch (of this row or the next) while the current batch's x is in flight, so no
// batch waits for two dependent LDS reads.  Reading x a batch early too, and taking the
// previous row's new x from its register, removed the round trip but cost more
// instructions than it saved (32^3 finest sweep 40 -> 72 us).  KB is picked at upload
// (upload_core).  Each lane reads and writes only its own RHS column of x, so the sweep
// needs no barrier.  Measured (two sweeps over all blocks): 32^3 7-point, nv = 4, fp64:
// 147 us with k_hsgs_lds, 40 here; its 16^3 coarse level (24 entries per row) 270 -> 47;
// 96^3 27-point, nv = 32, fp32: 122 -> 116 (6144 waves, bound by the t, x streams at
// 0.4 of 8 TB/s and by issue).
template <typename VT, int NV, int KB, bool ONE>
__global__ __launch_bounds__(64) void k_hsgs_core(const uint32_t *__restrict__ row,
                                                  const uint32_t *__restrict__ col,
                                                  const VT *__restrict__ val,
                                                  const VT *__restrict__ invd, int64_t n,
                                                  int64_t B, int64_t E, size_t gbytes, int gw,
                                                  const VT *__restrict__ t,
                                                  VT *__restrict__ x, int x_zero, VT relax,
                                                  const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    constexpr int R = 16;
    extern __shared__ unsigned char smem[];
    const int g = threadIdx.x / NV, k = threadIdx.x % NV;
    // per group: x [B + 1][NV], values [E], inverse diagonal [B] (VT); x offsets of the
    // columns [E], row pointers [B + 1] (u32)
    VT *__restrict__ xs = (VT *)(smem + (size_t)g * gbytes);
    VT *__restrict__ cv = xs + (B + 1) * NV;
    VT *__restrict__ ivs = cv + E;
    uint32_t *__restrict__ cc = (uint32_t *)(ivs + B);
    uint32_t *__restrict__ rp = cc + E;
    const int64_t lo = ((int64_t)blockIdx.x * gw + g) * B;
    const bool active = g < gw && lo < n;
    const int nr = active ? (int)(lo + B < n ? B : n - lo) : 0;
    const uint32_t e0 = active ? row[lo] : 0u;
    const uint32_t ne = active ? row[lo + nr] - e0 : 0u;
    if (active) {
        for (int b = k; b <= nr && !ONE; b += NV * 8) {
            uint32_t r[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                r[u] = row[lo + (b + u * NV <= nr ? b + u * NV : nr)];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                rp[b + u * NV <= nr ? b + u * NV : nr] = r[u] - e0;
        }
        for (uint32_t b = k; b < ne; b += NV * 8u) {
            uint32_t c[8];
            VT v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const uint32_t i = b + u * NV < ne ? b + u * NV : ne - 1;
                c[u] = col[e0 + i];
                v[u] = val[e0 + i];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const uint32_t i = b + u * NV < ne ? b + u * NV : ne - 1;
                cc[i] = (c[u] - (uint32_t)lo) * NV;
                cv[i] = v[u];
            }
        }
        stage_copy<VT, 8>(ivs, invd + lo, nr, k, NV);
        if (x_zero)
            for (int q = 0; q < nr; ++q)
                xs[q * NV + k] = VT(0);
        else
            stage_copy<VT, 12>(xs, x + (size_t)lo * NV, (int64_t)nr * NV, k, NV);
        xs[nr * NV + k] = VT(0);
    }
    __syncthreads();
    const VT *__restrict__ tb = t + (size_t)lo * NV + k;
    for (int sweep = 0; sweep < 2 && nr > 0; ++sweep) {
        // step q of the sweep works on local row r0 + dir * q
        const int dir = sweep == 0 ? 1 : -1, r0 = sweep == 0 ? 0 : nr - 1;
        // the same, with steps past the end clamped to the last one
        auto row_of = [&](int q) { return r0 + dir * (q < nr ? q : nr - 1); };
        // first batch of local row l
        auto begin = [&](int l) { return ONE ? (uint32_t)(l * KB) : rp[l]; };
        VT tc[R], tn[R];
#pragma unroll
        for (int u = 0; u < R; ++u)
            tc[u] = tb[row_of(u) * NV];
        // the current row's batch (at j, row end je) and the next row's extent
        uint32_t c4[KB];
        VT v4[KB];
        auto fetch = [&](uint32_t at) __attribute__((always_inline)) {
#pragma unroll
            for (int v = 0; v < KB; ++v) {
                c4[v] = cc[at + v];
                v4[v] = cv[at + v];
            }
        };
        int lc = r0, ln = row_of(1);
        uint32_t j = begin(lc), je = ONE ? j + KB : rp[lc + 1];
        uint32_t nj = begin(ln), nje = ONE ? nj + KB : rp[ln + 1];
        VT di = ivs[lc];
        fetch(j);
        // sweeps the row lc with t value tv, then moves on; lnn is the row after the next
        auto step = [&](const VT tv, const int lnn) __attribute__((always_inline)) {
            VT sum = tv;
            const VT xo = xs[lc * NV + k];
            while (true) {
                VT p[KB];
#pragma unroll
                for (int v = 0; v < KB; ++v)
                    p[v] = xs[c4[v] + k] * v4[v];
                const bool more = !ONE && j + KB < je;
                fetch(more ? j + KB : nj);
#pragma unroll
                for (int v = 0; v < KB; ++v)
                    sum = sum - p[v];
                if (!more)
                    break;
                j += KB;
            }
            const VT ndi = ivs[ln];
            const VT coeff = relax * di;
            xs[lc * NV + k] = xo + coeff * sum;
            lc = ln;
            j = nj;
            je = nje;
            di = ndi;
            ln = lnn;
            nj = begin(ln);
            nje = ONE ? nj + KB : rp[ln + 1];
        };
        for (int q0 = 0; q0 < nr; q0 += R) {
            // t of the next R steps, in flight while these R rows are swept
            if (q0 + 2 * R <= nr) {
#pragma unroll
                for (int u = 0; u < R; ++u)
                    tn[u] = tb[(r0 + dir * (q0 + R + u)) * NV];
            } else {
#pragma unroll
                for (int u = 0; u < R; ++u)
                    tn[u] = tb[row_of(q0 + R + u) * NV];
            }
            if (q0 + R + 2 <= nr) {
#pragma unroll
                for (int u = 0; u < R; ++u)
                    step(tc[u], r0 + dir * (q0 + u + 2));
            } else {
#pragma unroll
                for (int u = 0; u < R; ++u)
                    if (q0 + u < nr)
                        step(tc[u], row_of(q0 + u + 2));
            }
#pragma unroll
            for (int u = 0; u < R; ++u)
                tc[u] = tn[u];
        }
    }
    for (int q = 0; q < nr; ++q)
        x[(size_t)(lo + q) * NV + k] = xs[q * NV + k];
}

// same sweep order on x in global memory, for blocks that do not fit in LDS
template <typename VT, typename IT, int NV>
__global__ __launch_bounds__(64) void k_hsgs_glb(const uint32_t *__restrict__ row,
                                                 const IT *__restrict__ col,
                                                 const VT *__restrict__ val,
                                                 const uint32_t *__restrict__ pbase, int shift,
                                                 const VT *__restrict__ invd, int64_t n,
                                                 int64_t B, const VT *__restrict__ t, VT *x,
                                                 int x_zero, VT relax,
                                                 const int *__restrict__ done) {
    if (done != nullptr && *done)
        return;
    constexpr int G = 64 / NV;
    const int g = threadIdx.x / NV, k = threadIdx.x % NV;
    const int64_t blk = (int64_t)blockIdx.x * G + g;
    const int64_t lo = blk * B;
    if (lo >= n)
        return;
    const int64_t hi = lo + B < n ? lo + B : n;
    if (x_zero)
        for (int64_t i = lo; i < hi; ++i)
            x[(size_t)i * NV + k] = VT(0);
    for (int sweep = 0; sweep < 2; ++sweep) {
        for (int64_t q = 0; q < hi - lo; ++q) {
            const int64_t i = sweep == 0 ? lo + q : hi - 1 - q;
            uint32_t base = 0;
            if constexpr (sizeof(IT) == 2)
                base = pbase[i >> shift];
            VT sum = t[(size_t)i * NV + k];
#pragma unroll 8
            for (uint32_t j = row[i]; j < row[i + 1]; ++j) {
                const int64_t c = (int64_t)(base + (uint32_t)col[j]);
                if (c >= lo && c < hi)
                    sum = sum - x[(size_t)c * NV + k] * val[j];
            }
            const VT coeff = relax * invd[i];
            x[(size_t)i * NV + k] = x[(size_t)i * NV + k] + coeff * sum;
        }
    }
}

template <typename VT, int NV, int KB>
void launch_core(const Mat &A, size_t gb, int gw, const void *t, void *x, int x_zero,
                 double relax, int64_t B, const int *done, hipStream_t s) {
    const int64_t nblk = (A.nrows + B - 1) / B;
    const dim3 grid((unsigned)((nblk + gw - 1) / gw));
    auto kern = A.core_rowmax <= KB ? k_hsgs_core<VT, NV, KB, true> : k_hsgs_core<VT, NV, KB, false>;
    hipLaunchKernelGGL(kern, grid, dim3(64), gw * gb, s, A.row, (const uint32_t *)A.col,
                       (const VT *)A.val, (const VT *)A.inv_diag, A.nrows, B, A.core_emax, gb,
                       gw, (const VT *)t, (VT *)x, x_zero, (VT)relax, done);
}

template <typename VT, typename IT, int NV>
const char *hsgs_t(const Mat &A, const void *t, void *x, int x_zero, double relax, int64_t B,
                   const int *done, hipStream_t s) {
    constexpr int G = 64 / NV;
    const int64_t nblk = (A.nrows + B - 1) / B;
    const int grid = (int)((nblk + G - 1) / G);
    const size_t lds = (size_t)64 * B * sizeof(VT);
    if constexpr (sizeof(IT) == 4) {
        // a padded core-block matrix of this block size whose blocks fit in LDS: staged sweeps
        const size_t gb = hsgs_core_bytes(B, NV, A.core_emax, sizeof(VT));
        if (A.core_B == B && gb <= kHsgsLds) {
            // blocks per wave: as many as the wave's lanes and 64 KB of LDS hold, but fewer
            // while there are not 2048 waves (2 per SIMD): a wave's time is its row chain,
            // the same for one block as for several
            const int64_t fit = std::min<int64_t>(G, kHsgsLds / gb);
            const int gw = (int)std::max<int64_t>(1, std::min<int64_t>(fit, nblk / 2048));
            switch (A.core_kb) {
            case 3:
                launch_core<VT, NV, 3>(A, gb, gw, t, x, x_zero, relax, B, done, s);
                return "k_hsgs_core";
            case 4:
                launch_core<VT, NV, 4>(A, gb, gw, t, x, x_zero, relax, B, done, s);
                return "k_hsgs_core";
            case 6:
                launch_core<VT, NV, 6>(A, gb, gw, t, x, x_zero, relax, B, done, s);
                return "k_hsgs_core";
            case 8:
                launch_core<VT, NV, 8>(A, gb, gw, t, x, x_zero, relax, B, done, s);
                return "k_hsgs_core";
            }
        }
    }
    if (lds <= 64 * 1024) {
        hipLaunchKernelGGL((k_hsgs_lds<VT, IT, NV>), dim3(grid), dim3(64), lds, s, A.row,
                           (const IT *)A.col, (const VT *)A.val, A.panel_base, A.panel_shift,
                           (const VT *)A.inv_diag, A.nrows, B, (const VT *)t, (VT *)x, x_zero,
                           (VT)relax, done);
        return "k_hsgs_lds";
    }
    hipLaunchKernelGGL((k_hsgs_glb<VT, IT, NV>), dim3(grid), dim3(64), 0, s, A.row,
                       (const IT *)A.col, (const VT *)A.val, A.panel_base, A.panel_shift,
                       (const VT *)A.inv_diag, A.nrows, B, (const VT *)t, (VT *)x, x_zero,
                       (VT)relax, done);
    return "k_hsgs_glb";
}

template <typename VT, typename IT>
const char *hsgs_nv(const Mat &A, int nv, const void *t, void *x, int x_zero, double relax, int64_t B,
             const int *done, hipStream_t s) {
    switch (nv) {
    case 1:
        return hsgs_t<VT, IT, 1>(A, t, x, x_zero, relax, B, done, s);
    case 2:
        return hsgs_t<VT, IT, 2>(A, t, x, x_zero, relax, B, done, s);
    case 4:
        return hsgs_t<VT, IT, 4>(A, t, x, x_zero, relax, B, done, s);
    case 8:
        return hsgs_t<VT, IT, 8>(A, t, x, x_zero, relax, B, done, s);
    case 16:
        return hsgs_t<VT, IT, 16>(A, t, x, x_zero, relax, B, done, s);
    case 32:
        return hsgs_t<VT, IT, 32>(A, t, x, x_zero, relax, B, done, s);
    case 64:
        return hsgs_t<VT, IT, 64>(A, t, x, x_zero, relax, B, done, s);
    default:
        return nullptr;
    }
}

} // namespace

int64_t hsgs_block_rows(int64_t n, int nblocks) {
    // misc::split_range<float64_t> (src/misc/misc.h:46-55)
    int64_t cs = n / nblocks;
    cs += 8 - (cs % 8);
    return cs;
}

void hsgs_sweeps(const Mat &A, int nv, const void *t, void *x, int x_zero, double relax,
                 int64_t B, const int *done, hipStream_t s) {
    LedgerScope led(s);
    const char *name;
    if (A.prec == F64)
        name = A.idx == IDX_U16 ? hsgs_nv<double, uint16_t>(A, nv, t, x, x_zero, relax, B, done, s)
                                : hsgs_nv<double, uint32_t>(A, nv, t, x, x_zero, relax, B, done, s);
    else
        name = A.idx == IDX_U16 ? hsgs_nv<float, uint16_t>(A, nv, t, x, x_zero, relax, B, done, s)
                                : hsgs_nv<float, uint32_t>(A, nv, t, x, x_zero, relax, B, done, s);
    if (led.on && name) {
        // the swept matrix (core blocks or the whole operator), its inverse diagonal, t ;
        // x written (and read unless zero-flagged)
        const double sv = A.prec == F64 ? 8.0 : 4.0, si = A.idx == IDX_U16 ? 2.0 : 4.0;
        const double V = (double)A.nrows * nv * sv;
        led.kernel = std::string(name) + "<" + prec_name(A.prec) + "," + std::to_string(nv) + ">";
        led.bytes = (double)A.nnz * (sv + si) + (double)(A.nrows + 1) * 4.0 +
                    (double)A.nrows * sv + V + (x_zero ? V : 2.0 * V);
    }
}

} // namespace xh
