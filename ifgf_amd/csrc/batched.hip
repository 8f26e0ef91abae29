// batched.hip -- mult of several density columns (up to 32) at once on one plan.
//
// The same pipeline as the single-column mult, with every buffer column-minor for nc columns (the
// columns of the pass; nothing is padded): ws[i nc + r], result[t nc + r], V[(cone n_hi + q) nc +
// r], F[(slot n_lo + c) nc + r].  Whatever depends on the geometry only is computed once per
// (target, source), (node, source), (node, child) or (target, source box) and applied to the
// columns.  The near field and leaf sampling hold the columns' sums in registers (instances for
// 2, 4, 8, 16 and 32 columns, the densities padded with zeros in LDS); the upward pass, the
// transform and the far field are those of columns.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <vector>

#include "columns.hpp"
#include "dev_common.hpp"
#include "device.hpp"

namespace ifgf
{
namespace
{
using namespace dev;

template <typename R>
__global__ void k_gather_b(const double* __restrict__ w_in, const int64_t* __restrict__ perm,
                           Cx<R>* __restrict__ w_out, int64_t n, int rb, int ncol,
                           double im_sign)
{
    // w_in: ncol columns of n values in caller order; columns ncol..rb-1 are zero
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= n * rb)
        return;
    const int64_t i = e / rb;
    const int r = int(e - i * rb);
    Cx<R> v = {0, 0};
    if (r < ncol)
    {
        const double* p = w_in + 2 * (int64_t(r) * n + perm[i]);
        v = {R(p[0]), R(im_sign * p[1])};
    }
    w_out[e] = v;
}

// the near field's results plus the far field's of each target level, in order
template <typename R>
__global__ void k_scatter_b(const Cx<R>* __restrict__ res, const Cx<R>* __restrict__ far, int nlvl,
                            const int64_t* __restrict__ perm, double* __restrict__ out, int64_t n,
                            int rb, int ncol, double re_sign, double im_sign)
{
    const int64_t e = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (e >= n * rb)
        return;
    const int64_t i = e / rb;
    const int r = int(e - i * rb);
    if (r >= ncol)
        return;
    Cx<R> u = res[e];
    for (int l = 0; l < nlvl; l++)
        u = cadd(u, far[l * n * rb + e]);
    double* p = out + 2 * (int64_t(r) * n + perm[i]);
    p[0] = re_sign * double(u.x);
    p[1] = im_sign * double(u.y);
}

template <typename R> __global__ void k_zero_b(Cx<R>* p, int64_t n, Cx<R>* q, int64_t nq)
{
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        p[i] = {R(0), R(0)};
    else if (i - n < nq)
        q[i - n] = {R(0), R(0)};
}

// near field (ifgfoperator.hpp:900-960): as k_near (source leaves staged in LDS, lanes =
// (target, group)), the kernel value of each (source, target) pair applied to the RB columns
template <int KIND, typename R, int RB>
__global__ __launch_bounds__(64) void k_near_b(const WorkItem* __restrict__ items,
                                               int64_t nitems,
                                               const int32_t* __restrict__ near_off,
                                               const PointRun* __restrict__ near_run,
                                               const BoxGeo* __restrict__ geo,
                                               const double* __restrict__ spts,
                                               const double* __restrict__ snrm,
                                               const Cx<R>* __restrict__ w,
                                               const double* __restrict__ tpts,
                                               Cx<R>* __restrict__ result, int nc, KParams kp)
{
    constexpr bool NRM = KIND == KD || KIND == KC;
    __shared__ double sp[3 * 64];
    __shared__ double sn[NRM ? 3 * 64 : 1];
    __shared__ Cx<R> sw[64 * RB];
    const int64_t it = xcd_block(kp.xlg);
    if (it >= nitems)
        return;
    const WorkItem wi = items[it];
    const int lane = threadIdx.x;
    const int Tp = pow2_at_least(wi.count);
    const int ti = lane & (Tp - 1);
    const int grp = lane / Tp, ngrp = 64 / Tp;
    const bool valid = ti < wi.count;
    const int64_t t = int64_t(wi.first) + (valid ? ti : 0);
    const double y0 = tpts[3 * t], y1 = tpts[3 * t + 1], y2 = tpts[3 * t + 2];
    Cx<R> acc[RB];
#pragma unroll
    for (int r = 0; r < RB; r++)
        acc[r] = {0, 0};
    const int32_t j0 = near_off[wi.box], j1 = near_off[wi.box + 1];
    const KParams kb = with_k(kp, geo[wi.pad]);
    for (int32_t j = j0; j < j1; j++)
    {
        const int64_t b = near_run[j].begin, e = near_run[j].end;
        for (int64_t c0 = b; c0 < e; c0 += 64)
        {
            const int n = int(min<int64_t>(64, e - c0));
            __syncthreads();
            if (lane < n)
            {
                const int64_t i = c0 + lane;
                sp[3 * lane] = spts[3 * i];
                sp[3 * lane + 1] = spts[3 * i + 1];
                sp[3 * lane + 2] = spts[3 * i + 2];
                if constexpr (NRM)
                {
                    sn[3 * lane] = snrm[3 * i];
                    sn[3 * lane + 1] = snrm[3 * i + 1];
                    sn[3 * lane + 2] = snrm[3 * i + 2];
                }
            }
            for (int e2 = lane; e2 < n * RB; e2 += 64)
            {
                const int i = e2 / RB, r = e2 % RB;
                sw[e2] = r < nc ? w[(c0 + i) * nc + r] : Cx<R>{R(0), R(0)};
            }
            __syncthreads();
            for (int k = grp; k < n; k += ngrp)
            {
                const double d0 = sp[3 * k] - y0, d1 = sp[3 * k + 1] - y1, d2 = sp[3 * k + 2] - y2;
                double xn = 0;
                if constexpr (NRM)
                    xn = d0 * sn[3 * k] + d1 * sn[3 * k + 1] + d2 * sn[3 * k + 2];
                // (0 times the density would not do: it need not be finite)
                if (coincident<KIND>(R(d0) * R(d0) + R(d1) * R(d1) + R(d2) * R(d2)))
                    continue;
                const Cx<R> g = p2p<KIND, R>(kb, R(d0), R(d1), R(d2), xn, Cx<R>{1, 0});
#pragma unroll
                for (int r = 0; r < RB; r++)
                    acc[r] = cadd(acc[r], cmul(g, sw[k * RB + r]));
            }
        }
    }
#pragma unroll
    for (int r = 0; r < RB; r++)
        for (int m = Tp; m < 64; m <<= 1)
        {
            acc[r].x += __shfl_xor(acc[r].x, m, 64);
            acc[r].y += __shfl_xor(acc[r].y, m, 64);
        }
    if (grp == 0 && valid)
    {
        Cx<R>* o = result + t * nc;
#pragma unroll
        for (int r = 0; r < RB; r++)
            if (r < nc)
                o[r] = cadd(o[r], acc[r]);
    }
}

// leaf sampling (ifgfoperator.hpp:1057-1073): thread = high-order node, the factored kernel
// of each (node, source) pair applied to the RB columns staged in LDS
template <int KIND, typename R, int RB>
__global__ __launch_bounds__(128) void k_leaf_b(const int32_t* __restrict__ work, int64_t nwork,
                                                const ConeDev* __restrict__ cones,
                                                const BoxGeo* __restrict__ geo,
                                                const int64_t* __restrict__ sbeg,
                                                const int64_t* __restrict__ send,
                                                const double* __restrict__ spts,
                                                const double* __restrict__ snrm,
                                                const Cx<R>* __restrict__ w, NodeTabs tabs,
                                                Cx<R>* __restrict__ V, int nc, KParams kp)
{
    constexpr int CH = 64; // sources per LDS chunk
    __shared__ R sx[CH], sy[CH], sz[CH];
    __shared__ R nx[CH], ny[CH], nz[CH];
    __shared__ Cx<R> sw[CH * RB];
    const int64_t wi = xcd_block(kp.xlg);
    if (wi >= nwork)
        return;
    const int32_t g = work[wi];
    const ConeDev cn = cones[g];
    const BoxGeo B = geo[cn.box];
    const KParams kb = with_k(kp, B);
    const int64_t b0 = sbeg[cn.box], b1 = send[cn.box];
    for (int q0 = 0; q0 < kp.n_hi; q0 += 128)
    {
        const int q = q0 + threadIdx.x;
        const bool active = q < kp.n_hi;
        double yd[3] = {0, 0, 0}, rr = 1;
        if (active)
            cone_node(B, cn.cell, q, kp.ho0, kp.ho1, kp.ho2, tabs, false, yd, rr);
        const R y0 = R(yd[0]), y1 = R(yd[1]), y2 = R(yd[2]), dc = R(rr);
        Cx<R> acc[RB];
#pragma unroll
        for (int r = 0; r < RB; r++)
            acc[r] = {0, 0};
        for (int64_t c0 = b0; c0 < b1; c0 += CH)
        {
            const int n = int(min<int64_t>(CH, b1 - c0));
            __syncthreads();
            if (threadIdx.x < n)
            {
                const int64_t i = c0 + threadIdx.x;
                sx[threadIdx.x] = R(spts[3 * i] - B.ctr[0]);
                sy[threadIdx.x] = R(spts[3 * i + 1] - B.ctr[1]);
                sz[threadIdx.x] = R(spts[3 * i + 2] - B.ctr[2]);
                if (snrm)
                {
                    nx[threadIdx.x] = R(snrm[3 * i]);
                    ny[threadIdx.x] = R(snrm[3 * i + 1]);
                    nz[threadIdx.x] = R(snrm[3 * i + 2]);
                }
            }
            for (int e = threadIdx.x; e < n * RB; e += 128)
            {
                const int i = e / RB, r = e % RB;
                sw[e] = r < nc ? w[(c0 + i) * nc + r] : Cx<R>{R(0), R(0)};
            }
            __syncthreads();
            if (active)
                for (int k = 0; k < n; k++)
                {
                    R nn[3] = {0, 0, 0};
                    if (snrm)
                    {
                        nn[0] = nx[k];
                        nn[1] = ny[k];
                        nn[2] = nz[k];
                    }
                    const Cx<R> f = factored<KIND, R>(kb, y0, y1, y2, dc, sx[k], sy[k], sz[k],
                                                      nn, Cx<R>{1, 0});
#pragma unroll
                    for (int r = 0; r < RB; r++)
                        acc[r] = cadd(acc[r], cmul(f, sw[k * RB + r]));
                }
        }
        if (active)
        {
            Cx<R>* o = V + (int64_t(g) * kp.n_hi + q) * nc;
#pragma unroll
            for (int r = 0; r < RB; r++)
                if (r < nc)
                    o[r] = acc[r];
        }
    }
}

// ------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------
typedef float mf4 __attribute__((ext_vector_type(4)));

// one-wave workgroups: the wave's LDS writes complete before its later LDS reads (of other
// lanes' values) issue; the memory clobber keeps the compiler from moving LDS accesses across
__device__ __forceinline__ void lds_fence()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// values -> fine coefficients at orders (3,6,6)/(2,3,3) on FP32 MFMA (v_mfma_f32_16x16x4f32),
// one wave per (cone, 16 real columns): the three axis maps as 16 x 16 x 4 tiles, axis 1, then
// axis 2, then axis 0 (171 MFMAs when every sub-cone is active; the 6 x 3 and 9 x 6 maps fill
// 28% and 42% of a tile). Tile operands: lane l holds A[l % 16][l / 16] (map row, input index)
// and B[l / 16][l % 16] (input index, column); the result tile row 4 (l / 16) + i, column
// l % 16 is element i of lane l. The same map as k_transform_cols up to rounding (the axes in
// another order), and slower than it on the 32-column spheroid (9.0 against 6.1 ms per mult):
// the pass moves 19 GB (values read, coefficients of the active sub-cones written) and the
// arithmetic is not what bounds it. Kept for that comparison: it runs only when the
// environment variable IFGF_TRANSFORM_MFMA is set at the call (device_mult).
__global__ __launch_bounds__(64) void k_transform_mf(int64_t c0, int64_t c1, int NC,
                                                     const ConeDev* __restrict__ cones,
                                                     const float* __restrict__ V,
                                                     float* __restrict__ Fout,
                                                     const float* __restrict__ W, int xlg)
{
    const int NT = NC / 16; // NC: real columns, a multiple of 16
    constexpr int S1 = 100, S2 = 68; // padded row strides: lane groups 16 banks apart
    __shared__ float Y1[27 * S1];    // (t0, j1) x (t2, column)
    __shared__ float Y2[9 * S2];     // per j1: j2 x (t0, column)
    const int lane = threadIdx.x, g = lane >> 4, c = lane & 15;
    const int64_t blk = xcd_block(xlg);
    const int64_t cone = c0 + blk / NT;
    if (cone >= c1)
        return;
    const int n = int(blk % NT) * 16 + c;
    const uint32_t mask = cones[cone].mask;
    const int64_t base = cones[cone].fine_base;
    const float* W0 = W;      // 6 x 3
    const float* W1 = W + 18; // 9 x 6
    const float* W2 = W + 72; // 9 x 6
    const float a1a = c < 9 ? W1[c * 6 + g] : 0.f;
    const float a1b = (c < 9 && g < 2) ? W1[c * 6 + g + 4] : 0.f;
    const float a2a = c < 9 ? W2[c * 6 + g] : 0.f;
    const float a2b = (c < 9 && g < 2) ? W2[c * 6 + g + 4] : 0.f;
    const float a0 = (c < 6 && g < 3) ? W0[c * 3 + g] : 0.f;
    const float* v = V + cone * (108 * NC) + n;
    float b[18][2];
#pragma unroll
    for (int q = 0; q < 18; q++) // q = t0 + 3 t2
    {
        const int t0 = q % 3, t2 = q / 3;
        b[q][0] = v[(t0 + 3 * (g + 6 * t2)) * NC];
        b[q][1] = g < 2 ? v[(t0 + 3 * (g + 4 + 6 * t2)) * NC] : 0.f;
    }
#pragma unroll
    for (int q = 0; q < 18; q++)
    {
        const int t0 = q % 3, t2 = q / 3;
        mf4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a1a, b[q][0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a1b, b[q][1], acc, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++)
        {
            const int j1 = 4 * g + i;
            if (j1 < 9)
                Y1[(t0 * 9 + j1) * S1 + t2 * 16 + c] = acc[i];
        }
    }
    lds_fence();
    for (int j1 = 0; j1 < 9; j1++)
    {
        const int s1 = j1 / 3, m1 = j1 - 3 * s1;
        // sub-cones s0 + 3 s1 + 9 s2 for every s0, s2
        if (!((mask >> (3 * s1)) & 0x1C0E07u))
            continue;
#pragma unroll
        for (int t0 = 0; t0 < 3; t0++)
        {
            const float* y = Y1 + (t0 * 9 + j1) * S1 + c;
            mf4 acc = {0.f, 0.f, 0.f, 0.f};
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a2a, y[g * 16], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a2b, g < 2 ? y[(g + 4) * 16] : 0.f, acc,
                                                       0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++)
            {
                const int j2 = 4 * g + i;
                if (j2 < 9)
                    Y2[j2 * S2 + t0 * 16 + c] = acc[i];
            }
        }
        lds_fence();
        mf4 acc[9];
#pragma unroll
        for (int j2 = 0; j2 < 9; j2++)
        {
            acc[j2] = mf4{0.f, 0.f, 0.f, 0.f};
            acc[j2] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                a0, g < 3 ? Y2[j2 * S2 + g * 16 + c] : 0.f, acc[j2], 0, 0, 0);
        }
#pragma unroll
        for (int j2 = 0; j2 < 9; j2++)
        {
            const int s2 = j2 / 3, m2 = j2 - 3 * s2;
#pragma unroll
            for (int i = 0; i < 4; i++)
            {
                const int j0 = 4 * g + i;
                const int sub = (j0 >> 1) + 3 * s1 + 9 * s2;
                if (j0 < 6 && ((mask >> sub) & 1u))
                {
                    const int rk = __popc(mask & ((1u << sub) - 1u));
                    const int coef = (j0 & 1) + 2 * (m1 + 3 * m2);
                    Fout[((base + rk) * 18 + coef) * NC + n] = acc[j2][i];
                }
            }
        }
        lds_fence();
    }
}

// everything of a batched mult between the gather of the densities and the scatter of the
// results: it reads and writes only the batch buffers, so one captured graph per number of
// columns and form (few, tiles) serves every call with these buffers
template <int KIND, typename R, int RB>
void run_batched_core(DevicePlan& D, hipStream_t st, int nc, bool few, bool tiles)
{
    const KParams kp = kparams(D);
    const NodeTabs tabs{D.ho_nodes, D.trig_th, D.trig_ph};
    Cx<R>* ws = static_cast<Cx<R>*>(D.b_ws);
    Cx<R>* res = static_cast<Cx<R>*>(D.b_res);
    Cx<R>* V = static_cast<Cx<R>*>(D.b_V);
    Cx<R>* F = static_cast<Cx<R>*>(D.b_F);
    const int64_t nt = D.ntgt * nc, nf = nt * D.n_far_lvls;
    Cx<R>* far_res = res + nt;
    k_zero_b<R><<<dim3(unsigned((nt + nf + 255) / 256)), dim3(256), 0, st>>>(res, nt, far_res, nf);
    // near and far fields as in the single-column mult (SidePipe)
    const int overlap = D.n_near_items ? D.shape.overlap : 0;
    auto pipe = side_pipe(
        D, D.far_steps, st, overlap,
        [&](hipStream_t s)
        {
            if (D.n_near_items)
                k_near_b<KIND, R, RB><<<dim3(unsigned(D.n_near_items)), dim3(64), 0, s>>>(
                    D.near_items, D.n_near_items, D.near_off, D.near_run, D.geo, D.src_pts,
                    D.normals, ws, D.tgt_pts, res, nc, kp);
        },
        [&](int g, hipStream_t s) { launch_far_cols<R>(D, s, kp, g, F, far_res, nc, few); });
    if (overlap != 1)
        pipe.fork();
    if (D.n_leaf_cones)
        k_leaf_b<KIND, R, RB><<<dim3(unsigned(D.n_leaf_cones)), dim3(128), 0, st>>>(
            D.leaf_cones, D.n_leaf_cones, D.cones, D.geo, D.src_begin, D.src_end, D.src_pts,
            D.normals, ws, tabs, V, nc, kp);
    for (int l = D.levels - 1; l >= 0; l--)
    {
        const int64_t c0 = D.cone_lvl_off[l], c1 = D.cone_lvl_off[l + 1];
        launch_up_cols<R>(D, st, kp, l, F, V, nc);
        if (c1 > c0)
        {
            bool done = false;
            if constexpr (sizeof(R) == 4)
                if (tiles && nc % 8 == 0)
                {
                    k_transform_mf<<<dim3(unsigned((c1 - c0) * (nc / 8))), dim3(64), 0, st>>>(
                        c0, c1, 2 * nc, D.cones, reinterpret_cast<const float*>(V),
                        reinterpret_cast<float*>(F), static_cast<const float*>(D.wmat),
                        D.shape.xcd_log2);
                    done = true;
                }
            if (!done)
                launch_transform_cols<R>(D, st, kp, c0, c1, V, F, nc);
            pipe.fork();
        }
        pipe.ready(l);
    }
    pipe.finish();
}

// one batched mult: gather, the core (eagerly, or as the captured graph of this number of
// columns and form), scatter
template <int KIND, typename R, int RB>
void run_batched(DevicePlan& D, const double* w_dev, double* out_dev, int nc, int ncol,
                 hipStream_t st, int io, bool graph, bool few, bool tiles)
{
    Cx<R>* ws = static_cast<Cx<R>*>(D.b_ws);
    Cx<R>* res = static_cast<Cx<R>*>(D.b_res);
    const double in_im = (io & IO_CONJ_IN) ? -1.0 : 1.0;
    const double out_re = (io & IO_NEGATE_OUT) ? -1.0 : 1.0;
    const double out_im = out_re * ((io & IO_CONJ_OUT) ? -1.0 : 1.0);
    const int64_t ns = D.nsrc * nc, nt = D.ntgt * nc;
    k_gather_b<R><<<dim3(unsigned((ns + 255) / 256)), dim3(256), 0, st>>>(
        w_dev, D.src_perm, ws, D.nsrc, nc, ncol, in_im);
    if (graph)
    {
        auto& g = D.b_graphs[nc | (few ? 64 : 0) | (tiles ? 128 : 0)]; // nc <= 32
        if (!g.second)
        {
            // captured on the plan's capture stream (the caller's may be the null stream,
            // which cannot be captured); kernels and event waits only
            if (!D.cap_stream)
            {
                hipStream_t cs;
                HIP_OK(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
                D.cap_stream = cs;
            }
            hipStream_t cs = static_cast<hipStream_t>(D.cap_stream);
            HIP_OK(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal));
            run_batched_core<KIND, R, RB>(D, cs, nc, few, tiles);
            hipGraph_t gr = nullptr;
            HIP_OK(hipStreamEndCapture(cs, &gr));
            hipGraphExec_t ex = nullptr;
            HIP_OK(hipGraphInstantiate(&ex, gr, nullptr, nullptr, 0));
            g = {gr, ex};
        }
        HIP_OK(hipGraphLaunch(static_cast<hipGraphExec_t>(g.second), st));
    }
    else
        run_batched_core<KIND, R, RB>(D, st, nc, few, tiles);
    k_scatter_b<R><<<dim3(unsigned((nt + 255) / 256)), dim3(256), 0, st>>>(
        res, res + nt, D.n_far_lvls, D.tgt_perm, out_dev, D.ntgt, nc, ncol, out_re, out_im);
    HIP_OK(hipGetLastError());
}

template <typename R, int RB>
void run_kind(DevicePlan& D, const double* w, double* o, int nc, int ncol, hipStream_t st, int io,
              bool graph, bool few, bool tiles)
{
    switch (D.kind)
    {
    case KIND_HELMHOLTZ:
        return run_batched<KH, R, RB>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    case KIND_MODHELMHOLTZ:
        return run_batched<KM, R, RB>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    case KIND_LAPLACE:
        return run_batched<KL, R, RB>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    case KIND_DOUBLELAYER:
        return run_batched<KD, R, RB>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    case KIND_COMBINED:
        return run_batched<KC, R, RB>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    case KIND_GRAD:
        return run_batched<KG, R, RB>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    }
    throw std::runtime_error("unknown kernel kind");
}

template <typename R>
void run_width(DevicePlan& D, const double* w, double* o, int ncol, hipStream_t st, int io,
               bool graph, bool few, bool tiles)
{
    // the MFMA tiles take 8 columns at a time: zero columns fill the last
    int nc = tiles ? (ncol + 7) / 8 * 8 : ncol;
    if (nc > D.b_rb)
        nc = ncol;
    if (nc <= 2)
        return run_kind<R, 2>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    if (nc <= 4)
        return run_kind<R, 4>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    if (nc <= 8)
        return run_kind<R, 8>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    if (nc <= 16)
        return run_kind<R, 16>(D, w, o, nc, ncol, st, io, graph, few, tiles);
    run_kind<R, 32>(D, w, o, nc, ncol, st, io, graph, few, tiles);
}
} // namespace

void mult_batched(DevicePlan& D, const double* w_dev, double* out_dev, int ncol, void* stream,
                  int io, bool graph, bool few, bool tiles)
{
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (ncol < 1 || ncol > D.b_rb || ncol > MAX_COLUMNS)
        throw std::runtime_error("mult_batched: column count or buffers");
    if (D.prec == PREC_FP64)
        run_width<double>(D, w_dev, out_dev, ncol, st, io, graph, few, tiles);
    else
        run_width<float>(D, w_dev, out_dev, ncol, st, io, graph, few, tiles);
}
} // namespace ifgf
