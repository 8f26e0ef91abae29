// rows.hpp -- sums over the rows and planes of a fine cone's coefficients, and the axis maps of the
// values -> coefficients transform, for orders known at run time: compiled per (first, second)
// fine order, or per number of inputs of an axis, with the rest in loops.  Shared by the
// single-column kernels (orders.hip) and those of several columns (columns.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "dev_common.hpp"

namespace ifgf
{
namespace dev
{
// a * b + c in one rounding
__device__ __forceinline__ float fma_r(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_r(double a, double b, double c) { return fma(a, b, c); }

// acc + a b, each rounding in its place: left to the compiler, the far field from the pair records and
// the one that locates the pairs fused different products of a b, and their results differed
template <typename R> __device__ __forceinline__ Cx<R> cmul_add(Cx<R> acc, Cx<R> a, Cx<R> b)
{
    return {acc.x + fma_r(a.x, b.x, -(a.y * b.y)), acc.y + fma_r(a.x, b.y, a.y * b.x)};
}

// A cone's coefficients are read a chunk ahead of the arithmetic, in two buffers of at most
// CHUNK complex values (96 bytes, 24 registers, each): whole axis-2 planes where one or more fit,
// else a plane's rows in equal parts
template <typename R> constexpr int CHUNK = sizeof(R) == 4 ? 12 : 6;

// Chebyshev values and sums of G points as the rows and planes of a cone go by
template <typename R, int O0, int O1, int G> struct ConeSum
{
    R t0[G][O0], t1[G][O1], x2[G], a2[G], b2[G];
    Cx<R> pl[G], out[G];
    __device__ __forceinline__ ConeSum(const R (&x0)[G], const R (&x1)[G], const R (&x2_)[G])
    {
#pragma unroll
        for (int g = 0; g < G; g++)
        {
            t0[g][0] = t1[g][0] = R(1);
            if constexpr (O0 > 1)
                t0[g][1] = x0[g];
#pragma unroll
            for (int i = 2; i < O0; i++)
                t0[g][i] = fma_r(R(2) * x0[g], t0[g][i - 1], -t0[g][i - 2]);
            if constexpr (O1 > 1)
                t1[g][1] = x1[g];
#pragma unroll
            for (int i = 2; i < O1; i++)
                t1[g][i] = fma_r(R(2) * x1[g], t1[g][i - 1], -t1[g][i - 2]);
            // T_i2 and T_i2-1 from (T_0, T_-1) = (1, x): the recurrence gives T_1 = x exactly
            x2[g] = x2_[g];
            a2[g] = R(1);
            b2[g] = x2_[g];
            out[g] = {R(0), R(0)};
        }
    }
    // row i1 of the current plane
    __device__ __forceinline__ void row(const Cx<R>* b, int i1)
    {
#pragma unroll
        for (int g = 0; g < G; g++)
        {
            Cx<R> sm = b[0];
#pragma unroll
            for (int i = 1; i < O0; i++)
            {
                sm.x = fma_r(b[i].x, t0[g][i], sm.x);
                sm.y = fma_r(b[i].y, t0[g][i], sm.y);
            }
            if (i1 == 0)
                pl[g] = sm;
            else
            {
                pl[g].x = fma_r(sm.x, t1[g][i1], pl[g].x);
                pl[g].y = fma_r(sm.y, t1[g][i1], pl[g].y);
            }
        }
    }
    __device__ __forceinline__ void end_plane()
    {
#pragma unroll
        for (int g = 0; g < G; g++)
        {
            out[g].x = fma_r(pl[g].x, a2[g], out[g].x);
            out[g].y = fma_r(pl[g].y, a2[g], out[g].y);
            const R t = fma_r(R(2) * x2[g], a2[g], -b2[g]);
            b2[g] = a2[g];
            a2[g] = t;
        }
    }
};

// The interpolant of one fine cone (coefficients c, index i0 + O0 (i1 + O1 i2)) at G points:
// sum c T_i0(x0) T_i1(x1) T_i2(x2), over i0, then i1, then i2, each coefficient read once for
// the G points.  A last chunk of several planes may run past the cone's coefficients (the
// coefficient buffers are padded by ROW_PAD entries) and uses none of what lies there.
// STRIDED: the coefficients are cs entries apart.
template <typename R, int O0, int O1, int G, bool STRIDED = false>
__device__ __forceinline__ void eval_planes(const Cx<R>* c, int o2, const R (&x0)[G],
                                            const R (&x1)[G], const R (&x2)[G], Cx<R> (&out)[G],
                                            int cs = 1)
{
    constexpr int NP = O0 * O1, CH = CHUNK<R>;
    const int st = STRIDED ? cs : 1;
    ConeSum<R, O0, O1, G> S(x0, x1, x2);
    // loads and arithmetic stay on their sides of a fence: the next chunk's loads are in flight
    // during this chunk's arithmetic
    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    if constexpr (NP <= CH)
    {
        // planes per chunk: a partly used last chunk reads for nothing, so few
        constexpr int PB = NP >= 6 ? 1 : (NP >= 3 ? 2 : 4);
        static_assert(PB * NP <= ROW_PAD, "the padding covers the last chunk");
        Cx<R> ba[PB * NP], bb[PB * NP];
        auto load = [&](Cx<R> (&b)[PB * NP])
        {
#pragma unroll
            for (int i = 0; i < PB * NP; i++)
                b[i] = c[i * st];
            c += PB * NP * st;
            fence();
        };
        auto sum = [&](const Cx<R> (&b)[PB * NP], int i2)
        {
#pragma unroll
            for (int k = 0; k < PB; k++)
            {
                if (k > 0 && i2 + k >= o2) // uniform
                    break;
#pragma unroll
                for (int i1 = 0; i1 < O1; i1++)
                    S.row(b + k * NP + i1 * O0, i1);
                S.end_plane();
            }
            fence();
        };
        load(ba);
#pragma unroll 1
        for (int i2 = 0;; i2 += 2 * PB)
        {
            if (i2 + PB >= o2)
            {
                sum(ba, i2);
                break;
            }
            load(bb);
            sum(ba, i2);
            if (i2 + 2 * PB >= o2)
            {
                sum(bb, i2 + PB);
                break;
            }
            load(ba);
            sum(bb, i2 + PB);
        }
    }
    else
    {
        constexpr int RM = CH / O0 < 1 ? 1 : CH / O0; // most rows per chunk
        constexpr int NCH = (O1 + RM - 1) / RM;       // chunks per plane
        constexpr int CR = (O1 + NCH - 1) / NCH;      // rows per chunk (the last may have fewer)
        Cx<R> b[2][CR * O0];
#pragma unroll
        for (int i = 0; i < CR * O0; i++)
            b[0][i] = c[i * st];
        fence();
        auto plane = [&](auto more)
        {
            constexpr bool MORE = decltype(more)::value;
#pragma unroll
            for (int j = 0; j < NCH; j++)
            {
                // the next chunk: of this plane, or the next plane's first
                const Cx<R>* p = c + (j + 1 < NCH ? (j + 1) * CR * O0 : NP) * st;
                const int nr = (j + 1 < NCH && (j + 2) * CR > O1) ? O1 - (j + 1) * CR : CR;
                if (MORE || j + 1 < NCH)
                {
#pragma unroll
                    for (int i = 0; i < CR * O0; i++)
                        if (i < nr * O0)
                            b[(j + 1) & 1][i] = p[i * st];
                }
                fence();
#pragma unroll
                for (int k = 0; k < CR; k++)
                    if (j * CR + k < O1)
                        S.row(b[j & 1] + k * O0, j * CR + k);
                fence();
            }
            S.end_plane();
            c += NP * st;
            if constexpr (MORE && (NCH & 1))
            {
#pragma unroll
                for (int i = 0; i < CR * O0; i++)
                    b[0][i] = b[1][i];
            }
        };
#pragma unroll 1
        for (int i2 = 0; i2 + 1 < o2; i2++)
            plane(std::true_type());
        plane(std::false_type());
    }
#pragma unroll
    for (int g = 0; g < G; g++)
        out[g] = S.out[g];
}

// The same sum at one point, the coefficients (in LDS, or in memory where several waves hide the
// wait) read up to about 20 at a time with nothing read ahead: fewer registers, as many waves
template <typename R, int O0, int O1>
__device__ __forceinline__ Cx<R> eval_point(const Cx<R>* c, int o2, R x0, R x1, R x2)
{
    constexpr int NP = O0 * O1, MOST = sizeof(R) == 4 ? 20 : 10;
    const R y0[1] = {x0}, y1[1] = {x1}, y2[1] = {x2};
    ConeSum<R, O0, O1, 1> S(y0, y1, y2);
    if constexpr (NP <= MOST)
    {
        constexpr int PB = MOST / NP > 4 ? 4 : MOST / NP; // planes per chunk
        static_assert(PB * NP <= ROW_PAD, "the padding covers the last chunk");
#pragma unroll 1
        for (int i2 = 0; i2 < o2; i2 += PB, c += PB * NP)
        {
            Cx<R> b[PB * NP];
#pragma unroll
            for (int i = 0; i < PB * NP; i++)
                b[i] = c[i];
#pragma unroll
            for (int k = 0; k < PB; k++)
            {
                if (k > 0 && i2 + k >= o2) // uniform
                    break;
#pragma unroll
                for (int i1 = 0; i1 < O1; i1++)
                    S.row(b + k * NP + i1 * O0, i1);
                S.end_plane();
            }
        }
    }
    else
    {
        constexpr int CR = MOST / O0 < 1 ? 1 : MOST / O0; // rows per chunk
#pragma unroll 1
        for (int i2 = 0; i2 < o2; i2++, c += NP)
        {
#pragma unroll
            for (int r = 0; r < O1; r += CR)
            {
                Cx<R> b[CR * O0];
#pragma unroll
                for (int i = 0; i < CR * O0; i++)
                    if (r * O0 + i < NP)
                        b[i] = c[r * O0 + i];
#pragma unroll
                for (int k = 0; k < CR; k++)
                    if (r + k < O1)
                        S.row(b + k * O0, r + k);
                __builtin_amdgcn_sched_barrier(0);
            }
            S.end_plane();
        }
    }
    return S.out[0];
}

// the same sum for first orders without a compiled kernel
template <typename R, int G>
__device__ __forceinline__ void eval_any(const Cx<R>* c, int o0, int o1, int o2,
                                         const R (&x0)[G], const R (&x1)[G], const R (&x2)[G],
                                         Cx<R> (&out)[G], int cs = 1)
{
    R a2[G], b2[G];
#pragma unroll
    for (int g = 0; g < G; g++)
    {
        a2[g] = R(1);
        b2[g] = x2[g];
        out[g] = {R(0), R(0)};
    }
    for (int i2 = 0; i2 < o2; i2++)
    {
        R a1[G], b1[G];
        Cx<R> pl[G];
#pragma unroll
        for (int g = 0; g < G; g++)
        {
            a1[g] = R(1);
            b1[g] = x1[g];
            pl[g] = {R(0), R(0)};
        }
        for (int i1 = 0; i1 < o1; i1++)
        {
            R a0[G], b0[G];
            Cx<R> sm[G];
#pragma unroll
            for (int g = 0; g < G; g++)
            {
                a0[g] = R(1);
                b0[g] = x0[g];
                sm[g] = {R(0), R(0)};
            }
            for (int i0 = 0; i0 < o0; i0++, c += cs)
            {
                const Cx<R> v = *c;
#pragma unroll
                for (int g = 0; g < G; g++)
                {
                    sm[g].x = fma_r(v.x, a0[g], sm[g].x);
                    sm[g].y = fma_r(v.y, a0[g], sm[g].y);
                    const R t = fma_r(R(2) * x0[g], a0[g], -b0[g]);
                    b0[g] = a0[g];
                    a0[g] = t;
                }
            }
#pragma unroll
            for (int g = 0; g < G; g++)
            {
                pl[g].x = fma_r(sm[g].x, a1[g], pl[g].x);
                pl[g].y = fma_r(sm[g].y, a1[g], pl[g].y);
                const R t = fma_r(R(2) * x1[g], a1[g], -b1[g]);
                b1[g] = a1[g];
                a1[g] = t;
            }
        }
#pragma unroll
        for (int g = 0; g < G; g++)
        {
            out[g].x = fma_r(pl[g].x, a2[g], out[g].x);
            out[g].y = fma_r(pl[g].y, a2[g], out[g].y);
            const R t = fma_r(R(2) * x2[g], a2[g], -b2[g]);
            b2[g] = a2[g];
            a2[g] = t;
        }
    }
}

// f(O0, O1) with the fine orders of the first two axes as compile-time constants: first orders
// 1 to 6 with second orders 1 to 10; (0, 0) for the others
template <int O0, class Fn> void with_second_order(int o1, const Fn& f)
{
#define IFGF_O1(N)                                                                              \
    case N:                                                                                     \
        return f(std::integral_constant<int, O0>(), std::integral_constant<int, N>())
    switch (o1)
    {
        IFGF_O1(1);
        IFGF_O1(2);
        IFGF_O1(3);
        IFGF_O1(4);
        IFGF_O1(5);
        IFGF_O1(6);
        IFGF_O1(7);
        IFGF_O1(8);
        IFGF_O1(9);
        IFGF_O1(10);
    }
#undef IFGF_O1
    f(std::integral_constant<int, 0>(), std::integral_constant<int, 0>());
}
template <class Fn> void with_orders(int o0, int o1, const Fn& f)
{
    switch (o0)
    {
    case 1:
        return with_second_order<1>(o1, f);
    case 2:
        return with_second_order<2>(o1, f);
    case 3:
        return with_second_order<3>(o1, f);
    case 4:
        return with_second_order<4>(o1, f);
    case 5:
        return with_second_order<5>(o1, f);
    case 6:
        return with_second_order<6>(o1, f);
    }
    f(std::integral_constant<int, 0>(), std::integral_constant<int, 0>());
}

// e / n for 0 <= e < 2^16 with inv = 1 / n (the half keeps the product off the integers)
__device__ __forceinline__ int div_small(int e, float inv)
{
    return int((float(e) + 0.5f) * inv);
}

// fn(H) with the high order of an axis as a compile-time constant (2 to 13; 0: any)
template <class Fn> __device__ __forceinline__ void with_high_order(int h, const Fn& fn)
{
#define IFGF_H(N)                                                                               \
    case N:                                                                                     \
        return fn(std::integral_constant<int, N>())
    switch (h) // uniform
    {
        IFGF_H(2);
        IFGF_H(3);
        IFGF_H(4);
        IFGF_H(5);
        IFGF_H(6);
        IFGF_H(7);
        IFGF_H(8);
        IFGF_H(9);
        IFGF_H(10);
        IFGF_H(11);
        IFGF_H(12);
        IFGF_H(13);
    }
#undef IFGF_H
    fn(std::integral_constant<int, 0>());
}

// out(j, sum_t W[j h + t] in[stride t]) for j < m: one pencil of an axis map.  H > 0 (= h): the
// pencil's inputs in registers, the map's rows in scalar registers (uniform addresses)
template <typename R, int H, class Out>
__device__ __forceinline__ void map_pencil(const R* __restrict__ W, int h, int m, const Cx<R>* in,
                                           int stride, const Out& out)
{
    if constexpr (H > 0)
    {
        Cx<R> v[H];
#pragma unroll
        for (int t = 0; t < H; t++)
            v[t] = in[t * stride];
#pragma unroll 3
        for (int j = 0; j < m; j++)
        {
            Cx<R> a = {R(0), R(0)};
#pragma unroll
            for (int t = 0; t < H; t++)
            {
                const R wv = W[j * H + t];
                a.x += wv * v[t].x;
                a.y += wv * v[t].y;
            }
            out(j, a);
        }
    }
    else
        for (int j = 0; j < m; j++)
        {
            Cx<R> a = {R(0), R(0)};
            for (int t = 0; t < h; t++)
            {
                const R wv = W[j * h + t];
                a.x += wv * in[t * stride].x;
                a.y += wv * in[t * stride].y;
            }
            out(j, a);
        }
}
} // namespace dev
} // namespace ifgf
