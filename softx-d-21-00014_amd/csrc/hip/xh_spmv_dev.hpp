// Device code shared by the SpMV kernels: 16-byte packs of right-hand sides, the column
// panels, and the fused epilogues of a row.
#pragma once

#include "xh_internal.hpp"

namespace xh {
namespace {

template <typename T, int W>
struct alignas(sizeof(T) * W) Pack {
    T v[W];
};

template <typename T, int W>
__device__ __forceinline__ Pack<T, W> ld(const T *__restrict__ p) {
    return *reinterpret_cast<const Pack<T, W> *>(p);
}

// Results are streamed out with nontemporal stores, so they do not evict the x rows
// that later rows of the launch will read again from L2.
template <typename T, int W>
__device__ __forceinline__ void st(T *__restrict__ p, const Pack<T, W> &v) {
    typedef T vec __attribute__((ext_vector_type(W)));
    vec t;
#pragma unroll
    for (int w = 0; w < W; ++w)
        t[w] = v.v[w];
    __builtin_nontemporal_store(t, reinterpret_cast<vec *>(p));
}

// the code of a grid neighbour (Mat::gcode) in the place of a column index
struct GridCol {
    uint8_t code;
};

template <typename IT>
__device__ __forceinline__ uint32_t panel_base(const uint32_t *__restrict__ pb, int shift,
                                               int64_t i) {
    if constexpr (std::is_same<IT, GridCol>::value)
        return (uint32_t)i;
    else if constexpr (sizeof(IT) == 4)
        return 0u;
    else
        return pb[i >> shift];
}

template <typename VT, int NV>
struct Width {
    static constexpr int value = (16 / (int)sizeof(VT)) < NV ? (16 / (int)sizeof(VT)) : NV;
};

// Operands of the fused epilogue of one row, loaded by epi_load (right before the
// epilogue in k_spmv, a few passes ahead in k_spmv_sweep).
template <typename VT, int W>
struct EpiIn {
    Pack<VT, W> a, b, c;
    Pack<double, W> xd;
    VT di;
    VT al[W];
};

template <typename VT, int NV, int W, int OP>
__device__ __forceinline__ void epi_load(int64_t i, size_t o, size_t oy, int k0,
                                         EpiIn<VT, W> &in, const void *__restrict__ yv,
                                         const VT *__restrict__ b, const VT *__restrict__ o1,
                                         const VT *__restrict__ isd, const VT *__restrict__ rr,
                                         const VT *__restrict__ out2,
                                         const void *__restrict__ xupdv, int last, int x_zero) {
    if constexpr (OP == OP_ADD) {
        in.a = ld<VT, W>((const VT *)yv + oy);
    } else if constexpr (OP == OP_RESID || OP == OP_OFFBLOCK || OP == OP_RESID0) {
        in.a = ld<VT, W>(b + o);
    } else if constexpr (OP == OP_DOT1 || OP == OP_DOT3) {
        in.a = ld<VT, W>(o1 + o);
    } else if constexpr (OP == OP_RDOT4) {
        in.a = ld<VT, W>(b + o);
        in.b = ld<VT, W>(o1 + o);
        in.c = ld<VT, W>(out2 + o);
#pragma unroll
        for (int w = 0; w < W; ++w)
            in.al[w] = rr[k0 + w];
    } else if constexpr (OP == OP_CHEB0 || OP == OP_CHEB || OP == OP_CHEBZ || OP == OP_CHEBR) {
        in.di = isd[i];
        if constexpr (OP == OP_CHEB0 || OP == OP_CHEBZ || OP == OP_CHEBR)
            in.a = ld<VT, W>(b + o);
        else
            in.a = ld<VT, W>(rr + o);
        if (last && !x_zero) {
            in.b = ld<VT, W>((const VT *)xupdv + o);
        } else {
#pragma unroll
            for (int w = 0; w < W; ++w)
                in.b.v[w] = VT(0);
        }
    } else if constexpr (OP == OP_PROLONG32) {
        if (!x_zero)
            in.xd = ld<double, W>((const double *)yv + o);
    }
}

// The fused epilogue of one row: acc holds the row's W sums (y = A x, or y + A x for
// OP_ADD); o is the row's offset in the nv-interleaved vectors, oy that of the output row;
// `in` holds the operands epi_load read for the row.
template <typename VT, int NV, int W, int OP, int NP>
__device__ __forceinline__ void row_epilogue(
    size_t o, size_t oy, const VT (&acc)[W], double (&part)[NP][W],
    const EpiIn<VT, W> &in, void *__restrict__ yv, VT *__restrict__ out2,
    VT *__restrict__ out3, void *__restrict__ xupdv, VT c, int last, int x_zero, int out_f32) {
    using P = Pack<VT, W>;
    if constexpr (OP == OP_SET || OP == OP_ADD) {
        P yo;
#pragma unroll
        for (int w = 0; w < W; ++w)
            yo.v[w] = acc[w];
        st<VT, W>((VT *)yv + oy, yo);
    } else if constexpr (OP == OP_RESID || OP == OP_OFFBLOCK) {
        const P &bv = in.a;
        if (OP == OP_RESID && out_f32) {
            Pack<float, W> t;
#pragma unroll
            for (int w = 0; w < W; ++w)
                t.v[w] = (float)(bv.v[w] - acc[w]);
            st<float, W>((float *)yv + o, t);
        } else {
            P t;
#pragma unroll
            for (int w = 0; w < W; ++w)
                t.v[w] = bv.v[w] - acc[w];
            st<VT, W>((VT *)yv + o, t);
        }
    } else if constexpr (OP == OP_RESID0) {
        const P &bv = in.a;
        P t;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            t.v[w] = bv.v[w] - acc[w];
            part[0][w] = part[0][w] + (double)(t.v[w] * t.v[w]);
        }
        st<VT, W>((VT *)yv + o, t);
        st<VT, W>(out2 + o, t);
        st<VT, W>(out3 + o, t);
    } else if constexpr (OP == OP_DOT1) {
        const P &ov = in.a;
        P yo;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            yo.v[w] = acc[w];
            part[0][w] = part[0][w] + (double)(acc[w] * ov.v[w]);
        }
        st<VT, W>((VT *)yv + o, yo);
    } else if constexpr (OP == OP_DOT3) {
        const P &sv = in.a;
        P yo;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            yo.v[w] = acc[w];
            part[0][w] = part[0][w] + (double)(acc[w] * sv.v[w]);
            part[1][w] = part[1][w] + (double)(acc[w] * acc[w]);
            part[2][w] = part[2][w] + (double)(sv.v[w] * sv.v[w]);
        }
        st<VT, W>((VT *)yv + o, yo);
    } else if constexpr (OP == OP_RDOT4) {
        // RBiCGStab 12-13 (merged_rbicgstab_group1): r^ = r - alpha v, then
        // theta = (t, r^), phi = (t, t), psi = (t, r0), eta = (r^, r^)
        const P &vv = in.a, &r0v = in.b, &rv = in.c;
        P yo, rn;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            yo.v[w] = acc[w];
            rn.v[w] = rv.v[w] - in.al[w] * vv.v[w];
            part[0][w] = part[0][w] + (double)(acc[w] * rn.v[w]);
            part[1][w] = part[1][w] + (double)(acc[w] * acc[w]);
            part[2][w] = part[2][w] + (double)(acc[w] * r0v.v[w]);
            part[3][w] = part[3][w] + (double)(rn.v[w] * rn.v[w]);
        }
        st<VT, W>((VT *)yv + o, yo);
        st<VT, W>(out2 + o, rn);
    } else if constexpr (OP == OP_CHEB0) {
        // r = b - A x ; r *= isd ; t1 = c*r ; then t1 *= isd (u) or x (+)= t1*isd
        const VT di = in.di;
        const P &bv = in.a;
        P rv, t1;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            rv.v[w] = bv.v[w] - acc[w];
            rv.v[w] = rv.v[w] * di;
            t1.v[w] = c * rv.v[w];
            t1.v[w] = t1.v[w] * di;
        }
        // last: x (+)= t1 ; else r and u; one store through the selected pointer
        if (last && !x_zero) {
#pragma unroll
            for (int w = 0; w < W; ++w)
                t1.v[w] = t1.v[w] + in.b.v[w];
        }
        if (!last)
            st<VT, W>(out2 + o, rv);
        st<VT, W>((last ? (VT *)xupdv : (VT *)yv) + o, t1);
    } else if constexpr (OP == OP_CHEB || OP == OP_CHEBR) {
        // t2 = (A u)*isd ; t1 = c*r + t2 ; then u' = t1*isd or x (+)= t1*isd
        // (OP_CHEBR: r = b*isd here)
        const VT di = in.di;
        P r0 = in.a;
        if constexpr (OP == OP_CHEBR)
#pragma unroll
            for (int w = 0; w < W; ++w)
                r0.v[w] = r0.v[w] * di;
        P t1;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const VT t2 = acc[w] * di;
            t1.v[w] = c * r0.v[w] + t2;
            t1.v[w] = t1.v[w] * di;
        }
        if (last && !x_zero) {
#pragma unroll
            for (int w = 0; w < W; ++w)
                t1.v[w] = t1.v[w] + in.b.v[w];
        }
        st<VT, W>((last ? (VT *)xupdv : (VT *)yv) + o, t1);
    } else if constexpr (OP == OP_CHEBZ) {
        // r = b*isd (the zero-x first step's residual, stored for the later steps when
        // out2 is given and this step is not the last) ; t2 = (A u)*isd ; t1 = c*r + t2 ;
        // u' or x = t1*isd
        const VT di = in.di;
        P rv, t1;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            rv.v[w] = in.a.v[w] * di;
            const VT t2 = acc[w] * di;
            t1.v[w] = c * rv.v[w] + t2;
            t1.v[w] = t1.v[w] * di;
        }
        if (!last && out2 != nullptr)
            st<VT, W>(out2 + o, rv);
        st<VT, W>((last ? (VT *)xupdv : (VT *)yv) + o, t1);
    } else if constexpr (OP == OP_PROLONG32) {
        // VT = float: temp32 = P xH ; x64 = (double)temp32 + x64
        double *xd = (double *)yv;
        Pack<double, W> xo;
#pragma unroll
        for (int w = 0; w < W; ++w)
            xo.v[w] = x_zero ? (double)acc[w] : (double)acc[w] + in.xd.v[w];
        st<double, W>(xd + o, xo);
    }
}

} // namespace
} // namespace xh
