// columns.hip -- the upward pass, the transform and the far field for several density columns at
// once, at any orders.
//
// What depends on the geometry only (table entries, cone lookups, cone location, Chebyshev values)
// is read or formed once for the columns; a fine cone's coefficients are read once for the nodes
// or targets of a thread that fall into it, nc consecutive columns on consecutive lanes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>

#include "columns.hpp"
#include "orders.hpp"
#include "rows.hpp"

namespace ifgf
{
namespace
{
using namespace dev;

// Upward pass with the grouped tables for cw of the nc columns (ifgfoperator.hpp:631-688,
// 1639-1705): a workgroup takes one parent cone (its UpDesc record) and a chunk of cw columns,
// thread = (group task, column); the children one after another, each adding its nodes' values
// times the transfer factors to part (a node is in one group of a child), so that one copy of the
// node values in LDS serves all eight.  Bound by memory: 32 columns, 262,144 points, (2,3,3), 29.5
// GB in 7.0 ms, 4.2 TB/s (a child cone is read by several parent cones).
template <typename R, int O0, int O1>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? (O0 * O1 <= 12 ? 4 : (O0 * O1 <= 18 ? 3 : 2)) : 2)))
void k_up_cols(
    const UpDesc* __restrict__ desc, const CellRef* __restrict__ ctab,
    const UpGrpOf<R>* __restrict__ grp, const Cx<R>* __restrict__ F, Cx<R>* __restrict__ V, int nc,
    int cw, int nch, KParams kp)
{
    constexpr int G = UpGrpOf<R>::N;
    constexpr int NW = int(sizeof(UpDesc) / 16);
    extern __shared__ __align__(16) unsigned char up_smem[];
    UpDesc& sd = *reinterpret_cast<UpDesc*>(up_smem);
    Cx<R>* part = reinterpret_cast<Cx<R>*>(up_smem + sizeof(UpDesc)); // node q, column r: q cw + r
    const int nhi = kp.n_hi, tid = threadIdx.x, nt = blockDim.x;
    const int64_t it = xcd_block(kp.xlg);
    const int64_t k = it / nch;
    const int col0 = int(it - k * nch) * cw;
    const int nw = nt / cw, w = tid / cw, r = tid - w * cw;
    const bool active = w < nw && col0 + r < nc;
    const int4* src = reinterpret_cast<const int4*>(desc + k);
    for (int i = tid; i < NW; i += nt)
        reinterpret_cast<int4*>(&sd)[i] = src[i];
    for (int i = tid; i < nhi * cw; i += nt)
        part[i] = {R(0), R(0)};
    __syncthreads();
    for (int c = 0; c < 8; c++)
    {
        const int t1 = active ? sd.tend[c] : 0;
        for (int t = (c ? sd.tend[c - 1] : 0) + w; t < t1; t += nw)
        {
            const UpGrpOf<R>* ep = grp + (sd.tg0[c] + t);
            const int4* ew = reinterpret_cast<const int4*>(ep);
            union
            {
                int4 w[4];
                struct
                {
                    int32_t cf, subd;
                    uint32_t q01, q23;
                    R x0[G], x1[G], x2[G];
                } f;
            } e;
#pragma unroll
            for (int i = 0; i < 4; i++)
                e.w[i] = ew[i];
            const int d = e.f.subd >> 8;
            int slot;
            if (d < UP_DMAX)
                slot = sd.slot[c][d];
            else
            {
                const int sub = e.f.subd & 255;
                const CellRef cr = ctab[sd.toff[c] + e.f.cf];
                slot = ((cr.mask >> sub) & 1u) ? cr.fine_base + __popc(cr.mask & ((1u << sub) - 1u))
                                               : -1;
            }
            if (slot < 0)
                continue;
            R x0[G], x1[G], x2[G];
#pragma unroll
            for (int g = 0; g < G; g++)
            {
                x0[g] = e.f.x0[g];
                x1[g] = e.f.x1[g];
                x2[g] = e.f.x2[g];
            }
            Cx<R> val[G];
            const Cx<R>* coef = F + int64_t(slot) * kp.n_lo * nc + (col0 + r);
            if constexpr (O0 > 0)
                eval_planes<R, O0, O1, G, true>(coef, kp.lo2, x0, x1, x2, val, nc);
            else
                eval_any<R, G>(coef, kp.lo0, kp.lo1, kp.lo2, x0, x1, x2, val, nc);
            R tr[G], ti[G];
#pragma unroll
            for (int g = 0; g < G; g++)
            {
                tr[g] = ep->tr[g];
                ti[g] = ep->ti[g];
            }
#pragma unroll
            for (int g = 0; g < G; g++)
            {
                const int q = int(((g < 2 ? e.f.q01 : e.f.q23) >> (16 * (g & 1))) & 0xffffu);
                if (q != 0xffff)
                    part[q * cw + r] = cadd(part[q * cw + r], cmul(val[g], Cx<R>{tr[g], ti[g]}));
            }
        }
        __syncthreads();
    }
    if (active)
        for (int q = w; q < nhi; q += nw)
            V[(int64_t(sd.g) * nhi + q) * nc + col0 + r] = part[q * cw + r];
}

// upward pass without tables (k_up): thread = (node, column), each locating the node in the
// children's grids itself
template <typename R>
__global__ __launch_bounds__(256) void k_up_cols_locate(const int32_t* __restrict__ work,
                                                        const ConeDev* __restrict__ cones,
                                                        const BoxGeo* __restrict__ geo,
                                                        const int32_t* __restrict__ child,
                                                        const CellRef* __restrict__ ctab,
                                                        NodeTabs tabs, const Cx<R>* __restrict__ F,
                                                        Cx<R>* __restrict__ V, int nc, int phase,
                                                        KParams kp)
{
    const int32_t g = work[xcd_block(kp.xlg)];
    const ConeDev cn = cones[g];
    const BoxGeo& P = geo[cn.box];
    for (int e = threadIdx.x; e < kp.n_hi * nc; e += 256)
    {
        const int q = e / nc, r = e - q * nc;
        double y[3], rp;
        cone_node(P, cn.cell, q, kp.ho0, kp.ho1, kp.ho2, tabs, true, y, rp);
        Cx<R> acc = {0, 0};
        for (int c = 0; c < 8; c++)
        {
            const int32_t ch = child[8 * cn.box + c];
            if (ch < 0)
                continue;
            const BoxGeo& C = geo[ch];
            Loc L;
            if (!locate(C, ctab, y[0] - C.ctr[0], y[1] - C.ctr[1], y[2] - C.ctr[2], kp.f0,
                        kp.f1, kp.f2, L))
                continue;
            const R x0[1] = {R(L.xi[0])}, x1[1] = {R(L.xi[1])}, x2[1] = {R(L.xi[2])};
            Cx<R> val[1];
            eval_any<R, 1>(F + int64_t(L.fine) * kp.n_lo * nc + r, kp.lo0, kp.lo1, kp.lo2, x0, x1,
                           x2, val, nc);
            Cx<R> tf;
            if (!phase)
                tf = {R(rp / L.r), R(0)};
            else
                tf = cscale(expmk<R>(P.k_re, P.k_im, R(L.r - rp)), R(rp / L.r));
            acc = cadd(acc, cmul(val[0], tf));
        }
        V[(int64_t(g) * kp.n_hi + q) * nc + r] = acc;
    }
}

// High-order values -> fine coefficients of the active sub-cones (k_transform_rows) of one cone and
// a chunk of cw columns per workgroup; thread = (pencil, column).  C: the orders and the chunk's
// columns as constants (Orders), or run-time values (AnyOrders).
// 32 columns, 262,144 points, (2,3,3): 6.0 ms, 3.1 TB/s; 7.4 with run-time values, bound by neither
// memory (2.6 TB/s) nor issue (328 vector instructions per ns) alone.
struct AnyOrders
{
    static constexpr int h0 = 0, h1 = 0, h2 = 0, l0 = 0, l1 = 0, l2 = 0, cw = 0;
};
template <int H0, int H1, int H2, int L0, int L1, int L2, int CW> struct Orders // fine factors 3
{
    static constexpr int h0 = H0, h1 = H1, h2 = H2, l0 = L0, l1 = L1, l2 = L2, cw = CW;
};
template <typename R, class C>
__global__ __launch_bounds__(256) void k_transform_cols(int64_t c0, int xsz,
                                                        const ConeDev* __restrict__ cones,
                                                        const Cx<R>* __restrict__ V,
                                                        Cx<R>* __restrict__ F,
                                                        const R* __restrict__ W, int nc, int cw_,
                                                        int nch, KParams kp)
{
    constexpr bool K = C::h0 > 0;
    extern __shared__ __align__(16) unsigned char tr_smem[];
    const int cw = K ? C::cw : cw_;
    Cx<R>* X = reinterpret_cast<Cx<R>*>(tr_smem);
    Cx<R>* Y = X + xsz * cw;
    const int h0 = K ? C::h0 : kp.ho0, h1 = K ? C::h1 : kp.ho1, h2 = K ? C::h2 : kp.ho2;
    const int l0 = K ? C::l0 : kp.lo0, l1 = K ? C::l1 : kp.lo1, l2 = K ? C::l2 : kp.lo2;
    const int f0 = K ? 3 : kp.f0, f1 = K ? 3 : kp.f1, f2 = K ? 3 : kp.f2;
    const int nh = h0 * h1 * h2, nlo = l0 * l1 * l2;
    const int m0 = f0 * l0, m1 = f1 * l1;
    const int64_t it = xcd_block(kp.xlg);
    const int64_t k = it / nch;
    const int col0 = int(it - k * nch) * cw, cn = K ? C::cw : min(cw, nc - col0);
    const int64_t cone = c0 + k;
    const int tid = threadIdx.x;
    // e / n (inv = 1 / n), by the constant where there is one
    auto div = [](int e, int n, float inv) { return K ? e / n : div_small(e, inv); };
    const float icn = 1.0f / float(cn);
    for (int e = tid; e < nh * cn; e += 256)
    {
        const int i = div(e, cn, icn), r = e - i * cn;
        X[i * cw + r] = V[(cone * nh + i) * nc + col0 + r];
    }
    __syncthreads();
    const R* W1 = W + m0 * h0;
    const R* W2 = W1 + m1 * h1;
    with_high_order(h0, [&](auto H)
                    {
                        for (int e = tid; e < h1 * h2 * cn; e += 256)
                        {
                            const int p = div(e, cn, icn), r = e - p * cn;
                            Cx<R>* y = Y + p * m0 * cw + r;
                            map_pencil<R, decltype(H)::value>(W, h0, m0, X + p * h0 * cw + r, cw,
                                                              [&](int j, Cx<R> a) { y[j * cw] = a; });
                        }
                    });
    __syncthreads();
    const float im0 = 1.0f / float(m0);
    with_high_order(h1, [&](auto H)
                    {
                        for (int e = tid; e < m0 * h2 * cn; e += 256)
                        {
                            const int p = div(e, cn, icn), r = e - p * cn;
                            const int i2 = div(p, m0, im0), j0 = p - i2 * m0;
                            Cx<R>* x = X + (j0 + m0 * m1 * i2) * cw + r;
                            map_pencil<R, decltype(H)::value>(
                                W1, h1, m1, Y + (j0 + m0 * h1 * i2) * cw + r, m0 * cw,
                                [&](int j, Cx<R> a) { x[j * m0 * cw] = a; });
                        }
                    });
    __syncthreads();
    const uint32_t mask = cones[cone].mask;
    const int64_t base = cones[cone].fine_base;
    const int l01 = l0 * l1;
    const float il0 = 1.0f / float(l0), il01 = 1.0f / float(l01), if0 = 1.0f / float(f0);
    with_high_order(h2, [&](auto H)
                    {
                        for (int e = tid; e < m0 * m1 * cn; e += 256)
                        {
                            // the pencils of one sub-cone column on consecutive lanes
                            const int p = div(e, cn, icn), r = e - p * cn;
                            const int s01 = div(p, l01, il01), m01 = p - s01 * l01;
                            const int s1 = div(s01, f0, if0), s0 = s01 - s1 * f0;
                            const int q1 = div(m01, l0, il0), q0 = m01 - q1 * l0;
                            const int j01 = s0 * l0 + q0 + m0 * (s1 * l1 + q1);
                            for (int s2 = 0; s2 < f2; s2++)
                            {
                                const int sub = s01 + f0 * f1 * s2;
                                if (!((mask >> sub) & 1u))
                                    continue;
                                const int rk = __popc(mask & ((1u << sub) - 1u));
                                Cx<R>* o = F + ((base + rk) * nlo + m01) * nc + col0 + r;
                                const int os = l01 * nc;
                                map_pencil<R, decltype(H)::value>(
                                    W2 + s2 * l2 * h2, h2, l2, X + j01 * cw + r, m0 * m1 * cw,
                                    [&](int j, Cx<R> a) { o[int64_t(j) * os] = a; });
                            }
                        }
                    });
}

// coefficients read together in the far field's evaluation
template <typename R> constexpr int FAR_CHUNK = sizeof(R) == 4 ? 24 : 12;

// Far field for nc columns (ifgfoperator.hpp:962-1012, 1708-1891).  Four waves; per step of four
// source boxes each wave locates the item's targets in one box (cone slot, Chebyshev values,
// centre factor into LDS), then thread = (run of tpt consecutive targets, column): the distinct
// cones of its targets (neighbours in Morton order, mostly one or two) one after another, each
// cone's coefficients read once, a chunk at a time, for all the run's targets in it.
template <typename R, int O0, int O1, bool FAST>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 3 : 2)))
void k_far_cols(
    const WorkItem* __restrict__ items, const int32_t* __restrict__ srange,
    const int32_t* __restrict__ far_src, const BoxGeo* __restrict__ geo,
    const CellRef* __restrict__ ctab, const Cx<R>* __restrict__ F,
    const double* __restrict__ tpts, const double* __restrict__ ang, int ang_base, int ang_n,
    const int64_t* __restrict__ rec_off, const FarRec<R>* __restrict__ rec,
    const Cx<R>* __restrict__ cfs, int phase, int nc, int tpt, int64_t ntgt,
    Cx<R>* __restrict__ far_res, KParams kp)
{
    constexpr int TM = 8; // targets per thread at most
    extern __shared__ __align__(16) unsigned char far_smem[];
    double* sang = reinterpret_cast<double*>(far_smem);
    // Chebyshev values T_1 .. of the three axes, ts per (box, target)
    R* s_t = reinterpret_cast<R*>(far_smem + ((ang_n + 1) & ~1) * sizeof(double));
    __shared__ int32_t s_slot[4][64];
    __shared__ Cx<R> s_cf[4][64];
    const int o0 = O0 > 0 ? O0 : kp.lo0, o1 = O0 > 0 ? O1 : kp.lo1, o2 = kp.lo2;
    const int ts = (o0 + o1 + o2 - 3) | 1;
    const int64_t it = xcd_block(kp.xlg);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    if constexpr (FAST)
        for (int i = tid; i < ang_n; i += 256)
            sang[i] = ang[ang_base + i];
    __syncthreads();
    const WorkItem wi = items[it];
    const bool tvalid = lane < wi.count;
    const int64_t t = int64_t(wi.first) + (tvalid ? lane : 0);
    const double y0 = tpts[3 * t], y1 = tpts[3 * t + 1], y2 = tpts[3 * t + 2];
    const int w = tid / nc, r = tid - w * nc;
    const int tgt0 = w * tpt;
    const int nt = w < 256 / nc ? max(0, min(tpt, wi.count - tgt0)) : 0; // this thread's targets
    Cx<R> acc[TM];
#pragma unroll
    for (int j = 0; j < TM; j++)
        acc[j] = {R(0), R(0)};
    const int32_t j0 = srange[2 * it], j1 = srange[2 * it + 1];
    for (int32_t jb = j0; jb < j1; jb += 4)
    {
        if (jb + wave < j1) // uniform per wave
        {
            const BoxGeo& B = geo[__builtin_amdgcn_readfirstlane(far_src[jb + wave])];
            bool ok = false;
            int slot = -1;
            double rr = 1, ri = 1;
            R x[3] = {R(0), R(0), R(0)};
            const int64_t e = rec ? rec_off[it] + int64_t(jb - j0 + wave) * wi.count + lane : 0;
            if (tvalid && rec) // the pairs' records
            {
                const FarRec<R> q = rec[e];
                ok = q.slot >= 0;
                slot = q.slot;
                x[0] = q.x0;
                x[1] = q.x1;
                x[2] = q.x2;
            }
            else if (tvalid)
            {
                if constexpr (FAST)
                {
                    LocF L;
                    const double* eth = sang + (2 * B.fth_off - ang_base);
                    const double* eph = sang + (2 * B.fph_off - ang_base);
                    ok = locate_fast(B, eth, eph, ctab, y0 - B.ctr[0], y1 - B.ctr[1],
                                     y2 - B.ctr[2], kp.f0, kp.f1, kp.f2, L);
                    slot = L.fine;
                    rr = L.r;
                    ri = L.rinv;
                    x[0] = R(L.xi[0]);
                    x[1] = R(L.xi[1]);
                    x[2] = R(L.xi[2]);
                }
                else
                {
                    Loc L;
                    ok = locate(B, ctab, y0 - B.ctr[0], y1 - B.ctr[1], y2 - B.ctr[2], kp.f0, kp.f1,
                                kp.f2, L);
                    slot = L.fine;
                    rr = L.r;
                    ri = 1.0 / L.r;
                    x[0] = R(L.xi[0]);
                    x[1] = R(L.xi[1]);
                    x[2] = R(L.xi[2]);
                }
            }
            s_slot[wave][lane] = ok ? slot : -1;
            if (ok)
            {
                R* T = s_t + (wave * 64 + lane) * ts;
                const int n[3] = {o0, o1, o2};
#pragma unroll
                for (int a = 0; a < 3; a++)
                {
                    R p = R(1), q = x[a]; // T_k-1, T_k
                    for (int k = 1; k < n[a]; k++)
                    {
                        *T++ = q;
                        const R v = fma_r(R(2) * x[a], q, -p);
                        p = q;
                        q = v;
                    }
                }
                if (rec)
                    s_cf[wave][lane] = cfs[e];
                else if (!phase)
                    s_cf[wave][lane] = {R(INV_4PI_D * ri), R(0)};
                else
                    s_cf[wave][lane] = cscale(expmk_far<R>(B.k_re, B.k_im, rr), R(INV_4PI_D * ri));
            }
        }
        __syncthreads();
        const int nb = min(4, j1 - jb);
        for (int b = 0; b < nb; b++)
        {
            int sl[TM];
            unsigned todo = 0;
#pragma unroll
            for (int j = 0; j < TM; j++)
            {
                sl[j] = -1;
                if (j < nt)
                    sl[j] = s_slot[b][tgt0 + j];
                todo |= unsigned(sl[j] >= 0) << j;
            }
            while (__any(todo != 0))
            {
                // the cone of the first target left, and the run's targets in it
                int cur = -1;
#pragma unroll
                for (int j = TM - 1; j >= 0; j--)
                    cur = ((todo >> j) & 1u) ? sl[j] : cur;
                unsigned m = 0;
#pragma unroll
                for (int j = 0; j < TM; j++)
                    m |= (unsigned(sl[j] == cur) << j) & todo;
                todo &= ~m;
                // (a thread with none left: cur = -1, m = 0; it reads slot 0 and adds nothing)
                const Cx<R>* c = F + int64_t(max(cur, 0)) * kp.n_lo * nc + r;
                const R* T0 = s_t + (b * 64 + tgt0) * ts;
                Cx<R> val[TM];
#pragma unroll
                for (int j = 0; j < TM; j++)
                    val[j] = {R(0), R(0)};
                if constexpr (O0 > 0)
                {
                    // chunks of whole planes, or of a plane's rows
                    constexpr int NP = O0 * O1, CH = FAR_CHUNK<R>;
                    constexpr int PB = NP <= CH ? (CH / NP > 4 ? 4 : CH / NP) : 1;
                    constexpr int RC = NP <= CH ? O1 : (CH / O0 < 1 ? 1 : CH / O0);
                    static_assert(PB * NP <= ROW_PAD || PB == 1, "the padding covers the last chunk");
#pragma unroll 1
                    for (int i2 = 0; i2 < o2; i2 += PB)
#pragma unroll
                        for (int r0 = 0; r0 < O1; r0 += RC)
                        {
                            Cx<R> cc[PB * RC * O0];
#pragma unroll
                            for (int i = 0; i < PB * RC * O0; i++)
                                if (PB > 1 || r0 * O0 + i < NP)
                                    cc[i] = c[(i2 * NP + r0 * O0 + i) * nc];
#pragma unroll
                            for (int j = 0; j < TM; j++)
                            {
                                if (!((m >> j) & 1u))
                                    continue;
                                const R* T = T0 + j * ts;
                                R u[O0], v[O1];
                                u[0] = v[0] = R(1);
#pragma unroll
                                for (int i = 1; i < O0; i++)
                                    u[i] = T[i - 1];
#pragma unroll
                                for (int i = 1; i < O1; i++)
                                    v[i] = T[O0 - 2 + i];
#pragma unroll
                                for (int k = 0; k < PB; k++)
                                {
                                    if (k > 0 && i2 + k >= o2) // uniform
                                        break;
                                    const R t2 = i2 + k ? T[O0 + O1 - 3 + i2 + k] : R(1);
                                    Cx<R> pl = {R(0), R(0)};
#pragma unroll
                                    for (int i1 = 0; i1 < RC; i1++)
                                        if (r0 + i1 < O1)
                                        {
                                            const Cx<R>* row = cc + (k * RC + i1) * O0;
                                            Cx<R> sm = row[0];
#pragma unroll
                                            for (int i = 1; i < O0; i++)
                                            {
                                                sm.x = fma_r(row[i].x, u[i], sm.x);
                                                sm.y = fma_r(row[i].y, u[i], sm.y);
                                            }
                                            pl.x = fma_r(sm.x, v[r0 + i1], pl.x);
                                            pl.y = fma_r(sm.y, v[r0 + i1], pl.y);
                                        }
                                    val[j].x = fma_r(pl.x, t2, val[j].x);
                                    val[j].y = fma_r(pl.y, t2, val[j].y);
                                }
                            }
                        }
                }
                else
                    for (int i2 = 0; i2 < o2; i2++)
                        for (int i1 = 0; i1 < o1; i1++)
                            for (int i0 = 0; i0 < o0; i0++, c += nc)
                            {
                                const Cx<R> v = *c;
#pragma unroll
                                for (int j = 0; j < TM; j++)
                                    if ((m >> j) & 1u)
                                    {
                                        const R* T = T0 + j * ts;
                                        R tt = i0 ? T[i0 - 1] : R(1);
                                        tt *= i1 ? T[o0 - 2 + i1] : R(1);
                                        tt *= i2 ? T[o0 + o1 - 3 + i2] : R(1);
                                        val[j].x = fma_r(v.x, tt, val[j].x);
                                        val[j].y = fma_r(v.y, tt, val[j].y);
                                    }
                            }
#pragma unroll
                for (int j = 0; j < TM; j++)
                    if ((m >> j) & 1u)
                        acc[j] = cmul_add(acc[j], val[j], s_cf[b][tgt0 + j]);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < TM; j++)
        if (j < nt)
        {
            Cx<R>* o = far_res + (wi.pad * ntgt + wi.first + tgt0 + j) * nc + r;
            *o = cadd(*o, acc[j]);
        }
}
typedef float mf4 __attribute__((ext_vector_type(4)));

// Far field for NC of the nc columns (blockIdx.y picks which), any orders: a workgroup per item, its
// waves sharing the item's sources; lanes = (target, run of sources) as in k_far_rec.  PLACE: where
// the pairs lie, read from their records (0) or, without those, located by locate_fast (1) or
// locate (2), so that the results do not depend on the room for records.  Per step the wave copies its lanes' distinct cones (up to most at a time, the NC
// columns' coefficients next to one another) to LDS and each lane adds coefficient times
// Chebyshev product for its target, one product for the columns.  Bound by the LDS reads (8 NC
// bytes per lane and coefficient).  Whole mult of 3 and 5 columns, with the kernels that evaluate
// 16 columns at a time -> with this one: 8.0 -> 4.1 and 9.1 -> 5.3 ms at (2,3,3), 262,144 points;
// 6.8 -> 3.3 and 7.7 -> 4.8 at (3,5,4), 100,000 points; FP64 at (3,5,4), 50,000 points, 6.9 -> 4.9
// and 10.3 -> 8.3.  NC of 8 and 16 instead (fewer groups, more registers and LDS per wave): 12
// columns 12.4 and 17.9 ms against 11.9.  Without records, where every group of columns locates
// the pairs: 3, 5 and 12 columns at (2,3,3) 8.6 -> 5.5, 9.8 -> 6.8 and 15.1 -> 14.4 ms, FP64 at
// (3,5,4), 50,000 points, 7.5 -> 6.0, 10.8 -> 10.0 and, slower, 18.0 -> 21.5.
template <typename R, int O0, int NC, int PLACE>
__global__ __launch_bounds__(512)
void k_far_few_cols(const WorkItem* __restrict__ items, const int32_t* __restrict__ srange,
                    const int32_t* __restrict__ far_src, const BoxGeo* __restrict__ geo,
                    const CellRef* __restrict__ ctab, const double* __restrict__ tpts,
                    const double* __restrict__ ang, int ang_base, int phase,
                    const int64_t* __restrict__ rec_off, const FarRec<R>* __restrict__ rec,
                    const Cx<R>* __restrict__ cfs, const Cx<R>* __restrict__ F, int nc, int most,
                    int stride, int64_t ntgt, Cx<R>* __restrict__ far_res, KParams kp)
{
    extern __shared__ __align__(16) unsigned char far_smem[];
    const int lane = int(threadIdx.x & 63), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wpb = int(blockDim.x >> 6);
    Cx<R>* sm = reinterpret_cast<Cx<R>*>(far_smem);
    Cx<R>* sc = sm + wave * most * stride;
    const int64_t it = xcd_block(kp.xlg);
    const int c0 = int(blockIdx.y) * NC, ncg = min(NC, nc - c0);
    const WorkItem wi = items[it];
    const int Tp = pow2_at_least(wi.count);
    const int ti = lane & (Tp - 1);
    const int grp = lane / Tp, ngrp = 64 / Tp;
    const bool valid = ti < wi.count;
    const int32_t j0 = srange[2 * it], n = srange[2 * it + 1] - j0;
    const int32_t ja = n * wave / wpb, jb = n * (wave + 1) / wpb;
    const FarRec<R>* rp = nullptr;
    const Cx<R>* cp = nullptr;
    double y0 = 0, y1 = 0, y2 = 0;
    if constexpr (PLACE == 0)
    {
        rp = rec + rec_off[it] + ti;
        cp = cfs + rec_off[it] + ti;
    }
    else if (valid)
    {
        const int64_t t = int64_t(wi.first) + ti;
        y0 = tpts[3 * t];
        y1 = tpts[3 * t + 1];
        y2 = tpts[3 * t + 2];
    }
    constexpr int ROWS = 64 / NC; // rows of NC columns the wave copies at a time
    const int n_lo = kp.n_lo;
    const int col = lane % NC, row0 = lane < ROWS * NC ? lane / NC : 4 * n_lo;
    Cx<R> acc[NC];
#pragma unroll
    for (int r = 0; r < NC; r++)
        acc[r] = {R(0), R(0)};
    int qs = -1;
    R q0 = R(0), q1 = R(0), q2 = R(0);
    Cx<R> cf = {R(0), R(0)};
    auto fetch = [&](int32_t j)
    {
        qs = -1;
        if (valid && j + grp < jb)
        {
            auto take = [&](const FarRec<R>& q)
            {
                qs = q.slot;
                q0 = q.x0;
                q1 = q.x1;
                q2 = q.x2;
            };
            if constexpr (PLACE == 0)
            {
                const int64_t e = int64_t(j + grp) * wi.count;
                take(rp[e]);
                cf = cp[e];
            }
            else
            {
                FarRec<R> q;
                place_pair<R, PLACE == 1>(geo[far_src[j0 + j + grp]], ctab, ang + ang_base, ang_base,
                                          y0, y1, y2, phase, kp, q, cf);
                take(q);
            }
        }
    };
    fetch(ja);
    for (int32_t j = ja; j < jb; j += ngrp)
    {
        const int fine = qs;
        const R x0 = q0, x1 = q1, x2 = q2;
        const Cx<R> cc = cf;
        fetch(j + ngrp);
        uint64_t rem = __ballot(fine >= 0);
        while (rem != 0)
        {
            int my = -1, nd = 0;
            int cs0 = 0, cs1 = 0, cs2 = 0, cs3 = 0;
#pragma unroll 1
            while (rem != 0 && nd < most)
            {
                const int f0 = __builtin_amdgcn_readlane(fine, __ffsll((unsigned long long)rem) - 1);
                const uint64_t m = __ballot(fine == f0);
                if (fine == f0)
                    my = nd;
                cs0 = nd == 0 ? f0 : cs0;
                cs1 = nd == 1 ? f0 : cs1;
                cs2 = nd == 2 ? f0 : cs2;
                cs3 = nd == 3 ? f0 : cs3;
                rem &= ~m;
                nd++;
            }
            // the staging writes stay behind the reads of the step before
            asm volatile("" ::: "memory");
#pragma unroll 4
            for (int k = row0; k < nd * n_lo; k += ROWS)
            {
                const int d = (k >= n_lo) + (k >= 2 * n_lo) + (k >= 3 * n_lo);
                const int f0 = d == 0 ? cs0 : (d == 1 ? cs1 : (d == 2 ? cs2 : cs3));
                const int i = k - d * n_lo;
                Cx<R> v = {R(0), R(0)};
                if (col < ncg)
                    v = F[(int64_t(f0) * n_lo + i) * nc + c0 + col];
                sc[d * stride + i * NC + col] = v;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (my >= 0)
            {
                const Cx<R>* l = sc + my * stride;
                Cx<R> p[NC];
#pragma unroll
                for (int r = 0; r < NC; r++)
                    p[r] = {R(0), R(0)};
                auto add = [&](R w)
                {
#pragma unroll
                    for (int r = 0; r < NC; r++)
                    {
                        const Cx<R> b = l[r];
                        p[r].x = fma_r(w, b.x, p[r].x);
                        p[r].y = fma_r(w, b.y, p[r].y);
                    }
                    l += NC;
                };
                // T_k T_j T_i from the recurrences of the three axes, each started from T_0 = 1
                // and T_-1 = x, the inner ones scaled by the outer's value
                R a2 = R(1), b2 = x2;
#pragma unroll 1
                for (int i2 = 0; i2 < kp.lo2; i2++)
                {
                    R a1 = a2, b1 = a2 * x1;
#pragma unroll 1
                    for (int i1 = 0; i1 < kp.lo1; i1++)
                    {
                        R a0 = a1, b0 = a1 * x0;
                        auto term = [&]()
                        {
                            add(a0);
                            const R t = fma_r(R(2) * x0, a0, -b0);
                            b0 = a0;
                            a0 = t;
                        };
                        if constexpr (O0 > 0)
                        {
#pragma unroll
                            for (int i0 = 0; i0 < O0; i0++)
                                term();
                        }
                        else
                        {
#pragma unroll 1
                            for (int i0 = 0; i0 < kp.lo0; i0++)
                                term();
                        }
                        const R t = fma_r(R(2) * x1, a1, -b1);
                        b1 = a1;
                        a1 = t;
                    }
                    const R t = fma_r(R(2) * x2, a2, -b2);
                    b2 = a2;
                    a2 = t;
                }
#pragma unroll
                for (int r = 0; r < NC; r++)
                    acc[r] = cmul_add(acc[r], p[r], cc);
            }
        }
    }
    for (int m = Tp; m < 64; m <<= 1)
    {
#pragma unroll
        for (int r = 0; r < NC; r++)
        {
            acc[r].x += __shfl_xor(acc[r].x, m, 64);
            acc[r].y += __shfl_xor(acc[r].y, m, 64);
        }
    }
    if (wpb > 1)
    {
        __syncthreads(); // the waves are done with their cones
#pragma unroll
        for (int r = 0; r < NC; r++)
            sm[(wave * NC + r) * 64 + lane] = acc[r];
        __syncthreads();
        if (wave)
            return;
        for (int w = 1; w < wpb; w++)
        {
#pragma unroll
            for (int r = 0; r < NC; r++)
                acc[r] = cadd(acc[r], sm[(w * NC + r) * 64 + lane]);
        }
    }
    if (grp == 0 && valid)
    {
        Cx<R>* res = far_res + (wi.pad * ntgt + wi.first + ti) * nc + c0;
#pragma unroll
        for (int r = 0; r < NC; r++)
            if (r < ncg)
                res[r] = cadd(res[r], acc[r]);
    }
}

// Far field for nc columns on the FP32 matrix cores (mixed form, any orders): per source box the
// item's targets are sums over a fine cone's n_lo coefficients, the same cone for many of them, so
// a block of 16 targets x 16 real columns is a product basis (16 x n_lo) times coefficients (n_lo x
// 16) on v_mfma_f32_16x16x4f32.  Four waves; per step of nbox source boxes a wave locates the
// item's targets in one box (or reads their records) and writes the products of their Chebyshev
// values to LDS (ks floats per target).  Then each wave takes one tile of 16 columns and its share
// of the four blocks of targets, and goes through the distinct cones of each box (2 to 3 for 64
// targets), 32 coefficients at a time: the next chunk's (or cone's, or box's) coefficients are
// loaded while the current ones are multiplied into every block that has targets in the cone,
// rows of other targets zeroed.
// The sums of a box times the centre factors are added up in registers.
// Lane l: g = l / 16, n = l % 16; A[row n], B[column n] at coefficient 8 c + 2 g + s in step s of
// chunk c (one 8-byte LDS read gives A for two steps), C[row 4 g + i][column n] in element i;
// real and imaginary parts are neighbouring columns.
// Bound by the waits for coefficients and LDS, not by the matrix rate (matrix cores busy 30% of
// the time, 2.6 TB/s): 32 columns, 262,144 points,
// (2,3,3), far phase 27 -> 11.9 ms (16.2 ms with
// k_far_cols); 5 columns, 49,999 points, (3,3,3): 2.6 -> 1.65 ms against k_far_cols.
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(4)))
void k_far_mfma(
    const WorkItem* __restrict__ items, const int32_t* __restrict__ srange,
    const int32_t* __restrict__ far_src, const BoxGeo* __restrict__ geo,
    const CellRef* __restrict__ ctab, const float* __restrict__ F,
    const double* __restrict__ tpts, const double* __restrict__ ang, int ang_base, int ang_n,
    const int64_t* __restrict__ rec_off, const FarRec<float>* __restrict__ rec,
    const Cx<float>* __restrict__ cfs, int phase, int nc, int nbox, int ks, int64_t ntgt,
    float* __restrict__ far_res, KParams kp)
{
    extern __shared__ __align__(16) unsigned char far_smem[];
    double* sang = reinterpret_cast<double*>(far_smem);
    float* s_b = reinterpret_cast<float*>(far_smem + ((ang_n + 1) & ~1) * sizeof(double));
    __shared__ int4 s_cone[4][64]; // a box's distinct cones: slot, the targets in it (64 bits)
    __shared__ int32_t s_nd[4];
    __shared__ uint64_t s_nv[4];   // the box's targets in no cone
    __shared__ Cx<float> s_cf[4][64];
    const int64_t it = xcd_block(kp.xlg);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int g = lane >> 4, n = lane & 15;
    for (int i = tid; i < ang_n; i += 256)
        sang[i] = ang[ang_base + i];
    __syncthreads();
    const WorkItem wi = items[it];
    const bool tvalid = lane < wi.count;
    const int64_t t = int64_t(wi.first) + (tvalid ? lane : 0);
    const double y0 = tpts[3 * t], y1 = tpts[3 * t + 1], y2 = tpts[3 * t + 2];
    const int nlo = kp.n_lo, ntile = (2 * nc + 15) / 16;
    const int rs = 2 * nc; // floats from one coefficient to the next
    // this wave's column tile and blocks: one tile per wave with 3 or 4 tiles (blocks 0 .. 3), two
    // waves per tile with 2, a block per wave with 1
    const int tile = ntile >= 3 ? wave : (ntile == 2 ? (wave & 1) : 0);
    unsigned blocks = ntile >= 3 ? 15u : (ntile == 2 ? 5u << (wave >> 1) : 1u << wave);
    blocks &= (1u << ((wi.count + 15) / 16)) - 1u;
    if (tile >= ntile)
        blocks = 0;
    const uint64_t mine = (((blocks & 1u) ? 0xffffull : 0) | ((blocks & 2u) ? 0xffffull << 16 : 0) |
                           ((blocks & 4u) ? 0xffffull << 32 : 0) |
                           ((blocks & 8u) ? 0xffffull << 48 : 0)); // the targets of the blocks
    // the products that are never written (targets outside the boxes' domains, past a row's end)
    // are multiplied by zero coefficients or into sums that are not used: they only have to be
    // finite
    for (int i = tid; i < nbox * 64 * ks + 16; i += 256)
        s_b[i] = 0.f;
    __syncthreads();
    mf4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++)
        acc[i] = mf4{0.f, 0.f, 0.f, 0.f};
    const int32_t j0 = srange[2 * it], j1 = srange[2 * it + 1];
    for (int32_t jb = j0; jb < j1; jb += nbox)
    {
        if (wave < nbox && jb + wave < j1) // uniform per wave
        {
            const BoxGeo& B = geo[__builtin_amdgcn_readfirstlane(far_src[jb + wave])];
            bool ok = false;
            LocF L;
            Cx<float> cf = {0.f, 0.f};
            if (tvalid && rec) // the pairs' records
            {
                const int64_t e = rec_off[it] + int64_t(jb - j0 + wave) * wi.count + lane;
                const FarRec<float> q = rec[e];
                cf = cfs[e];
                ok = q.slot >= 0;
                L.fine = q.slot;
                L.xi[0] = q.x0;
                L.xi[1] = q.x1;
                L.xi[2] = q.x2;
            }
            else if (tvalid)
                ok = locate_fast(B, sang + (2 * B.fth_off - ang_base),
                                 sang + (2 * B.fph_off - ang_base), ctab, y0 - B.ctr[0],
                                 y1 - B.ctr[1], y2 - B.ctr[2], kp.f0, kp.f1, kp.f2, L);
            {
                const int slot = ok ? L.fine : -1;
                const uint64_t act = __ballot(ok);
                uint64_t todo = act;
                int nd = 0;
                while (todo != 0) // uniform
                {
                    const int cur =
                        __builtin_amdgcn_readlane(slot, __ffsll((unsigned long long)todo) - 1);
                    const uint64_t m = __ballot(slot == cur);
                    todo &= ~m;
                    if (lane == 0)
                        s_cone[wave][nd] =
                            make_int4(cur, 0, int(uint32_t(m)), int(uint32_t(m >> 32)));
                    nd++;
                }
                if (lane == 0)
                {
                    s_nd[wave] = nd;
                    s_nv[wave] = ~act;
                }
            }
            if (ok)
            {
                float* b = s_b + (wave * 64 + lane) * ks;
                float a2 = 1.f, b2 = L.xi[2]; // T_i2, T_i2-1 (T_-1 = x)
                for (int i2 = 0; i2 < kp.lo2; i2++)
                {
                    float a1 = a2, b1 = a2 * L.xi[1]; // T_i2 T_i1, T_i2 T_i1-1
                    for (int i1 = 0; i1 < kp.lo1; i1++)
                    {
                        float a0 = a1, b0 = a1 * L.xi[0];
                        for (int i0 = 0; i0 < kp.lo0; i0++)
                        {
                            *b++ = a0;
                            const float v = fmaf(2.f * L.xi[0], a0, -b0);
                            b0 = a0;
                            a0 = v;
                        }
                        const float v = fmaf(2.f * L.xi[1], a1, -b1);
                        b1 = a1;
                        a1 = v;
                    }
                    const float v = fmaf(2.f * L.xi[2], a2, -b2);
                    b2 = a2;
                    a2 = v;
                }
                if (!rec && !phase)
                    cf = {float(INV_4PI_D * L.rinv), 0.f};
                else if (!rec)
                    cf = cscale(expmk_far<float>(B.k_re, B.k_im, L.r), float(INV_4PI_D * L.rinv));
            }
            s_cf[wave][lane] = cf;
        }
        __syncthreads();
        if (blocks != 0) // uniform
        {
            const int nb = min(nbox, j1 - jb);
            // the chunks of the step, in order: box nbx, its cone nd (slot ncur, this wave's
            // targets in it nm), the coefficients from nk on
            int nbx = -1, nd = 0, ndn = 0, ncur = 0, nk = 0;
            uint64_t nm = 0;
            auto next = [&]() -> bool
            {
                nk += 32;
                if (nm != 0 && nk < nlo)
                    return true;
                for (;;)
                {
                    while (nd >= ndn)
                    {
                        if (++nbx >= nb)
                            return false;
                        ndn = __builtin_amdgcn_readfirstlane(s_nd[nbx]);
                        nd = 0;
                    }
                    const int4 e = s_cone[nbx][nd++];
                    ncur = __builtin_amdgcn_readfirstlane(e.x);
                    nm = (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(e.w))) << 32 |
                          uint32_t(__builtin_amdgcn_readfirstlane(e.z))) & mine;
                    if (nm != 0)
                        break;
                }
                nk = 0;
                return true;
            };
            // uniform row addresses plus the lane's offset; columns past the last belong to the
            // next row and give sums that are not used, coefficients past the last are zeros
            const unsigned loff = unsigned(2 * g * rs + tile * 16 + n);
            const int lim = nlo - 2 * g, cs = nlo * rs;
            auto load = [&](float (&v)[8])
            {
                const float* Bp = F + int64_t(ncur) * cs + nk * rs;
#pragma unroll
                for (int q = 0; q < 8; q++)
                    v[q] = Bp[unsigned((8 * (q >> 1) + (q & 1)) * rs) + loff];
            };
            mf4 c[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
                c[i] = mf4{0.f, 0.f, 0.f, 0.f};
            const float sgn = (n & 1) ? 1.f : -1.f;
            float bv[8], bn[8];
            bool more = next();
            if (more)
                load(bn);
            while (more) // uniform
            {
                const int bx = nbx, k0 = nk;
                const uint64_t m = nm;
                // (rows past the last coefficient, of the next cone or the buffer's padding, are read
                // and replaced: a branch per load costs more)
#pragma unroll
                for (int q = 0; q < 8; q++)
                    bv[q] = k0 + 8 * (q >> 1) + (q & 1) < lim ? bn[q] : 0.f;
                more = next();
                if (more)
                    load(bn);
                const uint64_t other = ~(m | s_nv[bx]); // rows of other cones are zeroed
#pragma unroll
                for (int i = 0; i < 4; i++)
                {
                    const unsigned rows = unsigned(m >> (16 * i)) & 0xffffu;
                    if (rows == 0) // uniform
                        continue;
                    const bool keep = !((unsigned(other >> (16 * i)) >> n) & 1u);
                    const float* A = s_b + (bx * 64 + 16 * i + n) * ks + k0 + 2 * g;
#pragma unroll
                    for (int h = 0; h < 4; h++)
                    {
                        if (k0 + 8 * h >= nlo) // uniform
                            break;
                        float2 a = *reinterpret_cast<const float2*>(A + 8 * h);
                        a = make_float2(keep ? a.x : 0.f, keep ? a.y : 0.f);
                        c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, bv[2 * h], c[i], 0, 0, 0);
                        c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, bv[2 * h + 1], c[i], 0, 0,
                                                                    0);
                    }
                }
                if (!more || nbx != bx) // the box's sums are complete
                {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                    {
                        if (!((blocks >> i) & 1u)) // uniform
                            continue;
#pragma unroll
                        for (int e = 0; e < 4; e++)
                        {
                            const Cx<float> cf = s_cf[bx][16 * i + 4 * g + e];
                            const float own = c[i][e];
                            // the other part of the complex value: the neighbouring lane's
                            const float oth = __int_as_float(__builtin_amdgcn_mov_dpp(
                                __float_as_int(own), 0xB1, 0xF, 0xF, true));
                            acc[i][e] = fmaf(own, cf.x, fmaf(oth * sgn, cf.y, acc[i][e]));
                        }
                        c[i] = mf4{0.f, 0.f, 0.f, 0.f};
                    }
                }
            }
        }
        __syncthreads();
    }
    if (tile * 16 + n >= rs)
        return;
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
        if (!((blocks >> i) & 1u))
            continue;
#pragma unroll
        for (int e = 0; e < 4; e++)
        {
            const int row = 16 * i + 4 * g + e;
            if (row < wi.count)
            {
                float* o = far_res + (wi.pad * ntgt + wi.first + row) * rs + tile * 16 + n;
                *o += acc[i][e];
            }
        }
    }
}
} // namespace

namespace dev
{
constexpr size_t LDS_MAX = 160 * 1024; // gfx950: 160 KB of LDS per CU

// columns per workgroup: at most `most`, in as few equal chunks as that allows
static int column_chunk(int nc, int most)
{
    most = std::max(1, std::min(most, nc));
    const int chunks = (nc + most - 1) / most;
    return (nc + chunks - 1) / chunks;
}

template <typename R>
void launch_up_cols(DevicePlan& D, hipStream_t st, const KParams& kp, int level, const Cx<R>* F,
                    Cx<R>* V, int nc)
{
    const int64_t u0 = D.up_off[level], u1 = D.up_off[level + 1];
    const int64_t n = D.up_gl_off[level + 1] - D.up_gl_off[level];
    if (n > 0)
    {
        if (!D.up_tl_desc)
            throw std::runtime_error("upward pass: the per-cone records were not uploaded");
        // 8 columns of FP32 make 64-byte rows; the node values of the chunk fit 48 KB
        const size_t col = size_t(D.n_hi) * sizeof(Cx<R>);
        const int cw = column_chunk(nc, int(std::min<size_t>(8, 48 * 1024 / col)));
        const int nch = (nc + cw - 1) / cw;
        const size_t lds = sizeof(UpDesc) + cw * col;
        if (lds > LDS_MAX)
            throw std::runtime_error("interpolation orders too large for the upward kernel's LDS");
        const dim3 grid(unsigned(n * nch)), block(D.n_hi >= 200 ? 256 : 128);
        with_orders(D.lo[0], D.lo[1], [&](auto o0, auto o1)
                    {
                        constexpr int O0 = decltype(o0)::value, O1 = decltype(o1)::value;
                        if (lds > size_t(64) * 1024)
                            HIP_OK(hipFuncSetAttribute(
                                reinterpret_cast<const void*>(&k_up_cols<R, O0, O1>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
                        k_up_cols<R, O0, O1><<<grid, block, lds, st>>>(
                            D.up_tl_desc + D.up_gl_off[level], D.ctab,
                            static_cast<const UpGrpOf<R>*>(D.up_grp), F, V, nc, cw, nch, kp);
                    });
    }
    if (u1 > u0)
        k_up_cols_locate<R><<<dim3(unsigned(u1 - u0)), dim3(256), 0, st>>>(
            D.up_cones + u0, D.cones, D.geo, D.child, D.ctab,
            NodeTabs{D.ho_nodes, D.trig_th, D.trig_ph}, F, V, nc, D.kind != KL, kp);
}

template <typename R>
void launch_transform_cols(DevicePlan& D, hipStream_t st, const KParams& kp, int64_t c0, int64_t c1,
                           const Cx<R>* V, Cx<R>* F, int nc)
{
    const int h0 = D.ho[0], h1 = D.ho[1], h2 = D.ho[2];
    const int m0 = D.f[0] * D.lo[0], m1 = D.f[1] * D.lo[1];
    const int xsz = std::max(h0 * h1 * h2, m0 * m1 * h2);
    const int ysz = m0 * h1 * h2;
    const size_t col = size_t(xsz + ysz) * sizeof(Cx<R>);
    const int cw = column_chunk(nc, int(std::min<size_t>(8, 56 * 1024 / col)));
    const int nch = (nc + cw - 1) / cw;
    const size_t lds = cw * col;
    if (lds > LDS_MAX)
        throw std::runtime_error("interpolation orders too large for the transform kernel's LDS");
    auto go = [&](auto orders)
    {
        using C = decltype(orders);
        if (lds > size_t(64) * 1024)
            HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_transform_cols<R, C>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        k_transform_cols<R, C><<<dim3(unsigned((c1 - c0) * nch)), dim3(256), lds, st>>>(
            c0, xsz, D.cones, V, F, static_cast<const R*>(D.wmat), nc, cw, nch, kp);
    };
    // (constants gain nothing in FP64 and at the larger orders, whose chunks are narrower)
    if constexpr (sizeof(R) == 4)
        if (order_class(D) == 1 && cw == 8 && nc % 8 == 0)
            return go(Orders<3, 6, 6, 2, 3, 3, 8>());
    go(AnyOrders());
}

// k_far_few_cols for a call of at most FEW_COLUMNS columns, where a cone's coefficients for five
// columns fit the LDS; false otherwise
template <typename R>
static bool launch_far_few_cols(DevicePlan& D, hipStream_t st, const KParams& kp, int step,
                                const Cx<R>* F, Cx<R>* far_res, int nc)
{
    constexpr size_t CX = sizeof(Cx<R>);
    if ((size_t(D.n_lo) * 5 + 2) * CX > size_t(64) * 1024)
        return false;
    const DevicePlan::FarGroup& G = D.far_steps[step];
    const int64_t n = G.item1 - G.item0;
    // waves per item: as many for every number of columns, so that a column's sum does not depend
    // on the others; at most 128 KB of LDS
    int w = far_split(n);
    while (w > 1 && std::max<size_t>(12 * 1024, (size_t(D.n_lo) * 5 + 2) * CX) * w > 128 * 1024)
        w /= 2;
    // groups of at most five columns, as equal as they go
    const int gy = (nc + 4) / 5;
    auto go = [&](auto o0, auto ncc, auto place)
    {
        constexpr int O0 = decltype(o0)::value, NC = decltype(ncc)::value;
        constexpr int PLACE = decltype(place)::value;
        // 16-byte words, an odd number of them, so that the cones start in different banks
        const int stride = sizeof(R) == 4 ? (((D.n_lo * NC + 1) / 2) | 1) * 2 : (D.n_lo * NC) | 1;
        const size_t cone = size_t(stride) * CX;
        const int most = int(std::min<size_t>(4, std::max<size_t>(1, size_t(12) * 1024 / cone)));
        const size_t lds = std::max(cone * most * w, w > 1 ? size_t(w) * 64 * NC * CX : 0);
        if (lds > size_t(64) * 1024)
            HIP_OK(hipFuncSetAttribute(
                reinterpret_cast<const void*>(&k_far_few_cols<R, O0, NC, PLACE>),
                hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        k_far_few_cols<R, O0, NC, PLACE><<<dim3(unsigned(n), unsigned(gy)), dim3(64 * w), lds, st>>>(
            D.far_items + G.item0, D.far_srange + 2 * G.item0, D.far_src, D.geo, D.ctab, D.tgt_pts,
            D.fine_ang, G.ang_base, D.kind != KL, D.far_rec ? D.far_rec_off + G.item0 : nullptr,
            static_cast<const FarRec<R>*>(D.far_rec), static_cast<const Cx<R>*>(D.far_cf), F, nc,
            most, stride, D.ntgt, far_res, kp);
    };
    auto width = [&](auto o0, auto place)
    {
        switch ((nc + gy - 1) / gy)
        {
        case 5: go(o0, std::integral_constant<int, 5>(), place); break;
        case 4: go(o0, std::integral_constant<int, 4>(), place); break;
        default: go(o0, std::integral_constant<int, 3>(), place); break;
        }
    };
    auto cols = [&](auto o0)
    {
        if (D.far_rec)
            return width(o0, std::integral_constant<int, 0>());
        if constexpr (sizeof(R) == 4)
            if (G.ang_n > 0)
                return width(o0, std::integral_constant<int, 1>());
        width(o0, std::integral_constant<int, 2>());
    };
    switch (D.lo[0])
    {
    case 1: cols(std::integral_constant<int, 1>()); break;
    case 2: cols(std::integral_constant<int, 2>()); break;
    case 3: cols(std::integral_constant<int, 3>()); break;
    case 4: cols(std::integral_constant<int, 4>()); break;
    case 5: cols(std::integral_constant<int, 5>()); break;
    default: cols(std::integral_constant<int, 0>()); break;
    }
    return true;
}

template <typename R>
void launch_far_cols(DevicePlan& D, hipStream_t st, const KParams& kp, int step, const Cx<R>* F,
                     Cx<R>* far_res, int nc, bool few)
{
    if (few && launch_far_few_cols<R>(D, st, kp, step, F, far_res, nc))
        return;
    const DevicePlan::FarGroup& G = D.far_steps[step];
    const int64_t n = G.item1 - G.item0;
    const WorkItem* items = D.far_items + G.item0;
    const int32_t* srange = D.far_srange + 2 * G.item0;
    const int workers = 256 / nc; // nc <= 32: at least 8
    const int tpt = (64 + workers - 1) / workers;
    const int ts = (D.lo[0] + D.lo[1] + D.lo[2] - 3) | 1;
    const bool fast = sizeof(R) == 4 && G.ang_n > 0;
    const int an = fast ? G.ang_n : 0;
    const size_t lds = ((an + 1) & ~1) * sizeof(double) + size_t(4) * 64 * ts * sizeof(R);
    auto go = [&](auto kernel)
    {
        if (lds > size_t(64) * 1024)
            HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
        kernel<<<dim3(unsigned(n)), dim3(256), lds, st>>>(
            items, srange, D.far_src, D.geo, D.ctab, F, D.tgt_pts, D.fine_ang, G.ang_base, an,
            D.far_rec ? D.far_rec_off + G.item0 : nullptr,
            static_cast<const FarRec<R>*>(D.far_rec), static_cast<const Cx<R>*>(D.far_cf),
            D.kind != KL, nc, tpt, D.ntgt, far_res, kp);
    };
    if constexpr (sizeof(R) == 4)
    {
        // ks: an odd number of 8-byte words, so that the 16 rows of a block lie in different banks; as
        // many boxes per step (up to one per wave) as keep the products within 48 KB
        const int ks = 2 * (((D.n_lo + 1) / 2) | 1);
        const size_t box = size_t(64) * ks * sizeof(float), angb = ((an + 1) & ~1) * sizeof(double);
        const int nbox = int(std::min<size_t>(4, std::max<size_t>(1, 48 * 1024 / box)));
        const size_t mlds = angb + nbox * box + 64;
        if (fast && mlds <= LDS_MAX - 8192)
        {
            if (mlds > size_t(64) * 1024)
                HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_far_mfma),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, int(mlds)));
            k_far_mfma<<<dim3(unsigned(n)), dim3(256), mlds, st>>>(
                items, srange, D.far_src, D.geo, D.ctab, reinterpret_cast<const float*>(F),
                D.tgt_pts, D.fine_ang, G.ang_base, an,
                D.far_rec ? D.far_rec_off + G.item0 : nullptr,
                static_cast<const FarRec<float>*>(D.far_rec),
                static_cast<const Cx<float>*>(D.far_cf), D.kind != KL, nc, nbox, ks, D.ntgt,
                reinterpret_cast<float*>(far_res), kp);
        }
        else if (fast) // coefficients by the hundred
            go(&k_far_cols<R, 0, 0, true>);
        else // angle tables too large for LDS: rare
            go(&k_far_cols<R, 0, 0, false>);
    }
    else
        with_orders(D.lo[0], D.lo[1], [&](auto o0, auto o1)
                    { go(&k_far_cols<R, decltype(o0)::value, decltype(o1)::value, false>); });
}

#define IFGF_COLS(R)                                                                            \
    template void launch_up_cols<R>(DevicePlan&, hipStream_t, const KParams&, int,              \
                                    const Cx<R>*, Cx<R>*, int);                                 \
    template void launch_transform_cols<R>(DevicePlan&, hipStream_t, const KParams&, int64_t,   \
                                           int64_t, const Cx<R>*, Cx<R>*, int);                 \
    template void launch_far_cols<R>(DevicePlan&, hipStream_t, const KParams&, int,             \
                                     const Cx<R>*, Cx<R>*, int, bool);
IFGF_COLS(float)
IFGF_COLS(double)
#undef IFGF_COLS
} // namespace dev
} // namespace ifgf
