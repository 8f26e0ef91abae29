// orders.hip -- kernels that take the interpolation orders at run time.
//
// The tolerance estimate (ifgfoperator.hpp:108-244) raises each axis' order by itself, so the
// orders of an operator are any of hundreds of combinations and cannot all be compiled.  These
// kernels are compiled per pair of first fine orders (O0 1 to 6, O1 1 to 10; the others run one
// generic instance) and walk the third axis in a loop: the coefficients of a cone are O2 planes of
// O1 rows of O0 values, read a chunk ahead of the arithmetic, the Chebyshev values of the
// first two axes in registers, those of the third from their recurrence as the planes go by.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>

#include "orders.hpp"
#include "rows.hpp"

namespace ifgf
{
namespace
{
using namespace dev;

// Upward pass with the grouped tables at any orders (ifgfoperator.hpp:631-688, 1639-1705), as
// k_up_grp but for the orders: a workgroup takes K consecutive cones of the tiled list, each
// from its UpDesc record, and runs the cone's (child, group) tasks; a task reads its child
// cone's coefficients once for the group's nodes.  SEQ = false: all tasks at once, node q's value
// from child c in part[c n_hi + q], the eight then added in child order.  SEQ = true (n_hi too
// large for eight copies in LDS): the children one after another, each adding to part[q] (a
// node is in one group of a child, so no two threads add to the same place): the same sums.
// Bound by the vector-memory path (each coefficient is read once per group, 64 lanes wide): at
// (3,4,5), 1M points, 29 GB at 4.1 TB/s; at (5,5,5), combined field on a torus, 131,072 points, and in FP64
// by the waits for it (2.0 and 2.1 TB/s, 348 and 126 vector instructions per ns).  At (3,6,4), 1M points, 11.0 ms; 14.7 without the read-ahead, 16 ms when a
// chunk was read ahead past the last one; at (2,3,3) and (2,5,5) within 2% of k_up_grp without
// its transform.
template <typename R, int O0, int O1, bool SEQ>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? (O0 * O1 <= 20 ? 4 : 3) : 2)))
void k_up_rows(
    const UpDesc* __restrict__ desc, int64_t n, int K, const CellRef* __restrict__ ctab,
    const UpGrpOf<R>* __restrict__ grp, const Cx<R>* __restrict__ F, Cx<R>* __restrict__ V,
    KParams kp)
{
    constexpr int G = UpGrpOf<R>::N;
    constexpr int NW = int(sizeof(UpDesc) / 16);
    extern __shared__ __align__(16) unsigned char up_smem[];
    UpDesc& sd = *reinterpret_cast<UpDesc*>(up_smem);
    Cx<R>* part = reinterpret_cast<Cx<R>*>(up_smem + sizeof(UpDesc));
    const int nhi = kp.n_hi, o2 = kp.lo2;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int64_t first = xcd_block(kp.xlg) * K;
    const int count = int(min<int64_t>(K, n - first));
#pragma unroll 1
    for (int k = 0; k < count; k++)
    {
        const int4* src = reinterpret_cast<const int4*>(desc + first + k);
        for (int i = tid; i < NW; i += nt)
            reinterpret_cast<int4*>(&sd)[i] = src[i];
        for (int i = tid; i < (SEQ ? nhi : 8 * nhi); i += nt)
            part[i] = {R(0), R(0)};
        __syncthreads();
        auto task = [&](int t, int c)
        {
            // the record's header and coordinates at once (16-byte loads)
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
                return;
            R x0[G], x1[G], x2[G];
#pragma unroll
            for (int g = 0; g < G; g++)
            {
                x0[g] = e.f.x0[g];
                x1[g] = e.f.x1[g];
                x2[g] = e.f.x2[g];
            }
            Cx<R> val[G];
            const Cx<R>* coef = F + int64_t(slot) * kp.n_lo;
            if constexpr (O0 > 0)
                eval_planes<R, O0, O1, G>(coef, o2, x0, x1, x2, val);
            else
                eval_any<R, G>(coef, kp.lo0, kp.lo1, o2, x0, x1, x2, val);
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
                if (q == 0xffff) // an empty place
                    continue;
                const Cx<R> v = cmul(val[g], Cx<R>{tr[g], ti[g]});
                if constexpr (SEQ)
                    part[q] = cadd(part[q], v);
                else
                    part[c * nhi + q] = v;
            }
        };
        if constexpr (SEQ)
        {
            for (int c = 0; c < 8; c++)
            {
                const int t1 = sd.tend[c];
                for (int t = (c ? sd.tend[c - 1] : 0) + tid; t < t1; t += nt)
                    task(t, c);
                __syncthreads();
            }
        }
        else
        {
            const int tot = sd.tend[7];
            for (int t = tid; t < tot; t += nt)
            {
                int c = 0;
                while (t >= sd.tend[c])
                    c++;
                task(t, c);
            }
            __syncthreads();
        }
        for (int q = tid; q < nhi; q += nt)
        {
            Cx<R> a = part[q];
            if constexpr (!SEQ)
            {
#pragma unroll
                for (int c = 1; c < 8; c++)
                    a = cadd(a, part[c * nhi + q]);
            }
            V[int64_t(sd.g) * nhi + q] = a;
        }
        __syncthreads(); // before the next cone replaces sd and part
    }
}
// distinct cones per wave and source box copied to LDS
constexpr int FAR_STAGE = 4;

// the wave's LDS writes have completed before its next LDS reads (of what other lanes wrote)
// issue; the memory clobber keeps the compiler from moving LDS accesses across
__device__ __forceinline__ void wave_lds_wait()
{
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

// the nc coefficients of cones c0 .. c3 (the first nd of them) to LDS, `stride` entries apart, by
// the nact active lanes of a wave together; U: 16 bytes where a cone is whole 16-byte words
template <class U, typename R>
__device__ __forceinline__ void stage_cones(const Cx<R>* __restrict__ F, int c0, int c1, int c2,
                                            int c3, int nd, int nc, int stride, int rank, int nact,
                                            Cx<R>* sc)
{
    constexpr int E = int(sizeof(U) / sizeof(Cx<R>));
    static_assert(FAR_STAGE == 4, "four cones");
    const int nu = nc / E;
#pragma unroll 2
    for (int i = rank; i < nd * nu; i += nact)
    {
        const bool b1 = i >= nu, b2 = i >= 2 * nu, b3 = i >= 3 * nu;
        const int cf = b3 ? c3 : (b2 ? c2 : (b1 ? c1 : c0));
        const int d = int(b1) + int(b2) + int(b3), k = i - d * nu;
        *reinterpret_cast<U*>(sc + d * stride + E * k) =
            reinterpret_cast<const U*>(F + int64_t(cf) * nc)[k];
    }
}

// Far field at any orders (ifgfoperator.hpp:962-1012, 1708-1891): for each target of the item,
// the interpolants of its far source boxes times the centre factor.  One wave per item, or
// (split) all waves of the workgroup a run each of one item's sources, their sums added in order;
// the waves share the launch's angle tables in LDS (FAST: cones located by
// locate_fast; otherwise the exact locate).  With stage > 0 (cones of stage coefficients and
// more) the distinct cones of the wave's lanes, up to FAR_STAGE, are copied to LDS by all lanes
// together and each lane reads its own there, `stride` entries apart so that the same
// coefficient of different cones lies in different banks; a wave with more distinct cones, and
// every wave without staging, reads the coefficients from memory.
// Bound by memory latency and the cone location's arithmetic: waves per SIMD matter, so a point's
// coefficients are not all in registers (eval_point).  Far phase against the kernel that read each
// coefficient from memory in Clenshaw order: 24.8 -> 8.8 ms at (3,6,4), 1M points; 26 -> 6.8 ms at
// (5,5,5), combined field on a torus, 131,072 points; with a read-ahead in two buffers instead
// 27 registers spilled at (2,5,*).  At six coefficients a plane 8 waves per SIMD (4 registers
// spilled at (2,3)) against 7: far phase 4.74 -> 4.63 ms, whole mult 8.65 -> 8.43 at (2,3,3), 1M
// points; with fewer, slower (2.33 -> 2.38 at (2,2,2), 400,000 points).
template <typename R, int O0, int O1, bool FAST>
__global__ __launch_bounds__(512)
__attribute__((amdgpu_waves_per_eu(
    sizeof(R) == 4 ? (O0 * O1 == 6 ? 8 : 4) : (O0 * O1 > 24 ? 1 : 2))))
void k_far_rows(
    const WorkItem* __restrict__ items, int64_t nitems, const int32_t* __restrict__ srange,
    const int32_t* __restrict__ far_src, const BoxGeo* __restrict__ geo,
    const CellRef* __restrict__ ctab, const Cx<R>* __restrict__ F,
    const double* __restrict__ tpts, const double* __restrict__ ang, int ang_base, int ang_n,
    int stage, int stride, int phase, int split, int64_t ntgt, Cx<R>* __restrict__ far_res,
    KParams kp)
{
    extern __shared__ __align__(16) unsigned char far_smem[];
    double* sang = reinterpret_cast<double*>(far_smem);
    const int lane = int(threadIdx.x & 63), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wpb = int(blockDim.x >> 6);
    Cx<R>* sc = reinterpret_cast<Cx<R>*>(far_smem + ((ang_n + 1) & ~1) * sizeof(double)) +
                wave * (FAR_STAGE * stride + ROW_PAD);
    const int64_t it = split ? xcd_block(kp.xlg) : xcd_block(kp.xlg) * wpb + wave;
    if constexpr (FAST)
    {
        for (int i = threadIdx.x; i < ang_n; i += int(blockDim.x))
            sang[i] = ang[ang_base + i];
        __syncthreads();
    }
    if (it >= nitems)
        return;
    const WorkItem wi = items[it];
    const int Tp = pow2_at_least(wi.count);
    const int ti = lane & (Tp - 1);
    const int grp = lane / Tp, ngrp = 64 / Tp;
    const bool valid = ti < wi.count;
    const int64_t t = int64_t(wi.first) + (valid ? ti : 0);
    const double y0 = tpts[3 * t], y1 = tpts[3 * t + 1], y2 = tpts[3 * t + 2];
    Cx<R> acc = {0, 0};
    int32_t j0 = srange[2 * it], j1 = srange[2 * it + 1];
    if (split) // a run of the item's sources per wave
    {
        const int32_t n = j1 - j0, a = j0;
        j0 = a + n * wave / wpb;
        j1 = a + n * (wave + 1) / wpb;
    }
    auto body = [&](const BoxGeo& B)
    {
        int fine;
        double r, rinv;
        R x0[1], x1[1], x2[1];
        if constexpr (FAST)
        {
            LocF L;
            const double* eth = sang + (2 * B.fth_off - ang_base);
            const double* eph = sang + (2 * B.fph_off - ang_base);
            if (!locate_fast(B, eth, eph, ctab, y0 - B.ctr[0], y1 - B.ctr[1], y2 - B.ctr[2],
                             kp.f0, kp.f1, kp.f2, L))
                return;
            fine = L.fine;
            r = L.r;
            rinv = L.rinv;
            x0[0] = R(L.xi[0]);
            x1[0] = R(L.xi[1]);
            x2[0] = R(L.xi[2]);
        }
        else
        {
            Loc L;
            if (!locate(B, ctab, y0 - B.ctr[0], y1 - B.ctr[1], y2 - B.ctr[2], kp.f0, kp.f1, kp.f2,
                        L))
                return;
            fine = L.fine;
            r = L.r;
            rinv = 1.0 / L.r;
            x0[0] = R(L.xi[0]);
            x1[0] = R(L.xi[1]);
            x2[0] = R(L.xi[2]);
        }
        Cx<R> val[1];
        bool staged = false;
        if constexpr (sizeof(R) == 4)
            if (stage > 0)
            {
                const uint64_t act = __ballot(1);
                const int rank = __popcll(act & ((1ull << lane) - 1ull));
                const int nact = __popcll(act);
                uint64_t rem = act;
                int myslot = 0, nd = 0;
                int cs[FAR_STAGE] = {};
#pragma unroll 1
                while (rem != 0 && nd < FAR_STAGE)
                {
                    const int l0 = __ffsll((unsigned long long)rem) - 1;
                    const int f0 = __builtin_amdgcn_readlane(fine, l0);
                    const uint64_t m = __ballot(fine == f0);
                    if (fine == f0)
                        myslot = nd;
#pragma unroll
                    for (int e = 0; e < FAR_STAGE; e++)
                        cs[e] = nd == e ? f0 : cs[e];
                    rem &= ~m;
                    nd++;
                }
                if (rem == 0) // uniform
                {
                    if (kp.n_lo & 1)
                        stage_cones<float2>(F, cs[0], cs[1], cs[2], cs[3], nd, kp.n_lo, stride,
                                            rank, nact, sc);
                    else
                        stage_cones<float4>(F, cs[0], cs[1], cs[2], cs[3], nd, kp.n_lo, stride,
                                            rank, nact, sc);
                    wave_lds_wait();
                    const Cx<R>* c = sc + myslot * stride;
                    if constexpr (O0 > 0)
                        val[0] = eval_point<R, O0, O1>(c, kp.lo2, x0[0], x1[0], x2[0]);
                    else
                        eval_any<R, 1>(c, kp.lo0, kp.lo1, kp.lo2, x0, x1, x2, val);
                    staged = true;
                    // the next source box's staging writes stay behind this box's LDS reads
                    asm volatile("" ::: "memory");
                }
            }
        if (!staged)
        {
            const Cx<R>* c = F + int64_t(fine) * kp.n_lo;
            if constexpr (O0 > 0)
                val[0] = eval_point<R, O0, O1>(c, kp.lo2, x0[0], x1[0], x2[0]);
            else
                eval_any<R, 1>(c, kp.lo0, kp.lo1, kp.lo2, x0, x1, x2, val);
        }
        Cx<R> cf;
        if (!phase) // uniform
            cf = {R(INV_4PI_D * rinv), R(0)};
        else
            cf = cscale(expmk_far<R>(B.k_re, B.k_im, r), R(INV_4PI_D * rinv));
        acc = cmul_add(acc, val[0], cf);
    };
    // the next source box's index is loaded one box ahead, so that its geometry loads do not
    // wait for it
    if (ngrp == 1)
    {
        // uniform source box: scalar loads of its geometry
        int32_t sn = j0 < j1 ? far_src[j0] : 0;
        for (int32_t j = j0; j < j1; j++)
        {
            const int32_t sb = __builtin_amdgcn_readfirstlane(sn);
            if (j + 1 < j1)
                sn = far_src[j + 1];
            body(geo[sb]);
        }
    }
    else
    {
        int32_t sn = j0 + grp < j1 ? far_src[j0 + grp] : 0;
        for (int32_t j = j0 + grp; j < j1; j += ngrp)
        {
            const int32_t sb = sn;
            if (j + ngrp < j1)
                sn = far_src[j + ngrp];
            body(geo[sb]);
        }
        for (int m = Tp; m < 64; m <<= 1)
        {
            acc.x += __shfl_xor(acc.x, m, 64);
            acc.y += __shfl_xor(acc.y, m, 64);
        }
    }
    if (split)
    {
        __shared__ Cx<R> psum[8][64];
        psum[wave][lane] = acc;
        __syncthreads();
        if (wave)
            return;
        for (int w = 1; w < wpb; w++)
            acc = cadd(acc, psum[w][lane]);
    }
    if (grp == 0 && valid)
    {
        Cx<R>* res = far_res + wi.pad * ntgt + t;
        *res = cadd(*res, acc);
    }
}
// the pair records of the items of one far launch: one wave per item (the order of the records:
// DevicePlan::far_rec)
template <typename R, bool FAST>
__global__ __launch_bounds__(64) void k_far_record(
    const WorkItem* __restrict__ items, const int32_t* __restrict__ srange,
    const int64_t* __restrict__ rec_off, const int32_t* __restrict__ far_src,
    const BoxGeo* __restrict__ geo, const CellRef* __restrict__ ctab,
    const double* __restrict__ tpts, const double* __restrict__ ang, int ang_base, int ang_n,
    int phase, FarRec<R>* __restrict__ rec, Cx<R>* __restrict__ cfs, KParams kp)
{
    extern __shared__ double rec_ang[];
    const int64_t it = blockIdx.x;
    if constexpr (FAST)
    {
        for (int i = threadIdx.x; i < ang_n; i += 64)
            rec_ang[i] = ang[ang_base + i];
        __syncthreads();
    }
    const WorkItem wi = items[it];
    const int32_t j0 = srange[2 * it], n = srange[2 * it + 1] - j0;
    const int64_t off = rec_off[it];
    for (int e = threadIdx.x; e < n * wi.count; e += 64)
    {
        const int j = e / wi.count;
        const int64_t t = int64_t(wi.first) + (e - j * wi.count);
        FarRec<R> q;
        Cx<R> cf;
        place_pair<R, FAST>(geo[far_src[j0 + j]], ctab, FAST ? rec_ang : nullptr, ang_base,
                            tpts[3 * t], tpts[3 * t + 1], tpts[3 * t + 2], phase, kp, q, cf);
        rec[off + e] = q;
        cfs[off + e] = cf;
    }
}

// Far field from the pair records, any orders: as k_far_rows without the cone location.  A step
// reads the pairs' records (one step ahead), then their cones: with stage > 0 the distinct cones
// of the wave's lanes copied to LDS by all lanes together, otherwise each lane's from memory.
// Bound by memory at few coefficients, the records most of its traffic (4.0 TB/s at (3,4,5), 1M
// points); at (5,5,5) by the LDS reads (99 million, 1.3 of 2.4 ms at their rate) and the waits for
// them (1.9 TB/s, 195 vector instructions per ns).  Far phase against locating the cones in
// every mult: 7.5 -> 4.5 ms
// at (3,6,4), 1M points; 3.7 -> 2.4 ms at (2,3,3), 1M points; FP64 at (3,5,4), 99,991 points,
// 1.6 -> 0.63 ms.
template <typename R, int O0, int O1>
__global__ __launch_bounds__(512)
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? (O0 * O1 <= 9 ? 7 : 5) : 3)))
void k_far_rec(
    const WorkItem* __restrict__ items, int64_t nitems, const int32_t* __restrict__ srange,
    const int64_t* __restrict__ rec_off, const FarRec<R>* __restrict__ rec,
    const Cx<R>* __restrict__ cfs, const Cx<R>* __restrict__ F, int stage, int stride, int split,
    int64_t ntgt, Cx<R>* __restrict__ far_res, KParams kp)
{
    extern __shared__ __align__(16) unsigned char far_smem[];
    __shared__ Cx<R> psum[8][64];
    const int lane = int(threadIdx.x & 63), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wpb = int(blockDim.x >> 6);
    Cx<R>* sc = reinterpret_cast<Cx<R>*>(far_smem) + wave * (FAR_STAGE * stride + ROW_PAD);
    const int64_t it = split ? xcd_block(kp.xlg) : xcd_block(kp.xlg) * wpb + wave;
    if (it >= nitems)
        return;
    const WorkItem wi = items[it];
    const int Tp = pow2_at_least(wi.count);
    const int ti = lane & (Tp - 1);
    const int grp = lane / Tp, ngrp = 64 / Tp;
    const bool valid = ti < wi.count;
    const int32_t n = srange[2 * it + 1] - srange[2 * it];
    int32_t ja = 0, jb = n;
    if (split) // a run of the item's sources per wave
    {
        ja = n * wave / wpb;
        jb = n * (wave + 1) / wpb;
    }
    const FarRec<R>* rp = rec + rec_off[it] + ti;
    const Cx<R>* cp = cfs + rec_off[it] + ti;
    Cx<R> acc = {0, 0};
    FarRec<R> q;
    Cx<R> cf;
    auto fetch = [&](int32_t j)
    {
        q.slot = -1;
        if (valid && j + grp < jb)
        {
            const int64_t e = int64_t(j + grp) * wi.count;
            q = rp[e];
            cf = cp[e];
        }
    };
    fetch(ja);
    for (int32_t j = ja; j < jb; j += ngrp)
    {
        const int fine = q.slot;
        const R x0 = q.x0, x1 = q.x1, x2 = q.x2;
        const Cx<R> c0 = cf;
        fetch(j + ngrp);
        const Cx<R>* c = F + int64_t(fine) * kp.n_lo;
        bool staged = false;
        if (stage > 0)
        {
            uint64_t rem = __ballot(fine >= 0);
            int myslot = 0, nd = 0;
            int cs[FAR_STAGE] = {};
#pragma unroll 1
            while (rem != 0 && nd < FAR_STAGE)
            {
                const int f0 = __builtin_amdgcn_readlane(fine, __ffsll((unsigned long long)rem) - 1);
                const uint64_t m = __ballot(fine == f0);
                if (fine == f0)
                    myslot = nd;
#pragma unroll
                for (int e = 0; e < FAR_STAGE; e++)
                    cs[e] = nd == e ? f0 : cs[e];
                rem &= ~m;
                nd++;
            }
            if (rem == 0) // uniform
            {
                if (sizeof(R) == 4 && (kp.n_lo & 1))
                    stage_cones<typename std::conditional<sizeof(R) == 4, float2, float4>::type>(
                        F, cs[0], cs[1], cs[2], cs[3], nd, kp.n_lo, stride, lane,
                                        64, sc);
                else
                    stage_cones<float4>(F, cs[0], cs[1], cs[2], cs[3], nd, kp.n_lo, stride, lane,
                                        64, sc);
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                staged = true;
                if (fine >= 0)
                {
                    const Cx<R>* l = sc + myslot * stride;
                    Cx<R> v[1];
                    if constexpr (O0 > 0)
                        v[0] = eval_point<R, O0, O1>(l, kp.lo2, x0, x1, x2);
                    else
                    {
                        const R y0[1] = {x0}, y1[1] = {x1}, y2[1] = {x2};
                        eval_any<R, 1>(l, kp.lo0, kp.lo1, kp.lo2, y0, y1, y2, v);
                    }
                    acc = cmul_add(acc, v[0], c0);
                }
                // the next step's staging writes stay behind this step's LDS reads
                asm volatile("" ::: "memory");
            }
        }
        if (!staged && fine >= 0)
        {
            Cx<R> v[1];
            if constexpr (O0 > 0)
                v[0] = eval_point<R, O0, O1>(c, kp.lo2, x0, x1, x2);
            else
            {
                const R y0[1] = {x0}, y1[1] = {x1}, y2[1] = {x2};
                eval_any<R, 1>(c, kp.lo0, kp.lo1, kp.lo2, y0, y1, y2, v);
            }
            acc = cmul_add(acc, v[0], c0);
        }
    }
    for (int m = Tp; m < 64; m <<= 1)
    {
        acc.x += __shfl_xor(acc.x, m, 64);
        acc.y += __shfl_xor(acc.y, m, 64);
    }
    if (split)
    {
        psum[wave][lane] = acc;
        __syncthreads();
        if (wave)
            return;
        for (int w = 1; w < wpb; w++)
            acc = cadd(acc, psum[w][lane]);
    }
    if (grp == 0 && valid)
    {
        Cx<R>* res = far_res + wi.pad * ntgt + wi.first + ti;
        *res = cadd(*res, acc);
    }
}

// High-order values -> fine coefficients of the active sub-cones at any orders and factors
// (chebinterp.hpp:176-250, ifgfoperator.hpp:1539-1637), separable per axis as k_transform_t: one
// thread per pencil and axis, cpb cones per workgroup (X: xsz entries per cone, the values, then
// the axis-1 stage; Y: ysz, the axis-0 stage; the axis-2 stage goes to memory).  Each axis has
// its loop compiled per number of inputs, chosen once by a uniform switch: an input is read from
// LDS once for all its outputs and the map's entries are scalar operands, where one thread per
// output read both from LDS for every product.  Bound by LDS (2 to 4 cycles of bank conflicts per
// instruction) and vector issue (390 per ns), at 2.7 to 3.0 TB/s.
// 1M points, (6,9,7)/(3,6,4): 16.8 -> 4.7 ms; torus, 131,072 points, (8,8,8)/(5,5,5): 3.8 ->
// 0.94 ms.
template <typename R>
__global__ __launch_bounds__(256) void k_transform_rows(int64_t c0, int64_t c1, int cpb, int xsz,
                                                        int ysz, const ConeDev* __restrict__ cones,
                                                        const Cx<R>* __restrict__ V,
                                                        Cx<R>* __restrict__ F,
                                                        const R* __restrict__ W, KParams kp)
{
    extern __shared__ __align__(16) unsigned char tr_smem[];
    Cx<R>* X = reinterpret_cast<Cx<R>*>(tr_smem);
    Cx<R>* Y = X + cpb * xsz;
    const int h0 = kp.ho0, h1 = kp.ho1, h2 = kp.ho2, nh = kp.n_hi;
    const int l0 = kp.lo0, l1 = kp.lo1, l2 = kp.lo2;
    const int m0 = kp.f0 * l0, m1 = kp.f1 * l1, m2 = kp.f2 * l2;
    const int64_t first = c0 + xcd_block(kp.xlg) * cpb;
    const int ncone = int(min<int64_t>(cpb, c1 - first));
    const int tid = threadIdx.x;
    for (int k = 0; k < ncone; k++)
        for (int i = tid; i < nh; i += 256)
            X[k * xsz + i] = V[(first + k) * nh + i];
    __syncthreads();
    const R* W1 = W + m0 * h0;
    const R* W2 = W1 + m1 * h1;
    {
        const int np = h1 * h2;
        const float inv = 1.0f / float(np);
        with_high_order(h0, [&](auto H)
                        {
                            for (int e = tid; e < ncone * np; e += 256)
                            {
                                const int k = div_small(e, inv), p = e - k * np;
                                Cx<R>* y = Y + k * ysz + p * m0;
                                map_pencil<R, decltype(H)::value>(
                                    W, h0, m0, X + k * xsz + p * h0, 1,
                                    [&](int j, Cx<R> a) { y[j] = a; });
                            }
                        });
    }
    __syncthreads();
    {
        const int np = m0 * h2;
        const float inv = 1.0f / float(np), inv0 = 1.0f / float(m0);
        with_high_order(h1, [&](auto H)
                        {
                            for (int e = tid; e < ncone * np; e += 256)
                            {
                                const int k = div_small(e, inv), p = e - k * np;
                                const int i2 = div_small(p, inv0), j0 = p - i2 * m0;
                                Cx<R>* x = X + k * xsz + j0 + m0 * m1 * i2;
                                map_pencil<R, decltype(H)::value>(
                                    W1, h1, m1, Y + k * ysz + j0 + m0 * h1 * i2, m0,
                                    [&](int j, Cx<R> a) { x[j * m0] = a; });
                            }
                        });
    }
    __syncthreads();
    {
        const int np = m0 * m1, l01 = l0 * l1;
        const float inv = 1.0f / float(np), il0 = 1.0f / float(l0), il01 = 1.0f / float(l01),
                    if0 = 1.0f / float(kp.f0);
        with_high_order(h2, [&](auto H)
                        {
                            for (int e = tid; e < ncone * np; e += 256)
                            {
                                const int k = div_small(e, inv), p = e - k * np;
                                // the pencils of one sub-cone column on consecutive lanes: their
                                // coefficients are consecutive in memory
                                const int s01 = div_small(p, il01), m01 = p - s01 * l01;
                                const int s1 = div_small(s01, if0), s0 = s01 - s1 * kp.f0;
                                const int q1 = div_small(m01, il0), q0 = m01 - q1 * l0;
                                const int j01 = s0 * l0 + q0 + m0 * (s1 * l1 + q1);
                                const ConeDev cn = cones[first + k];
                                for (int s2 = 0; s2 < kp.f2; s2++)
                                {
                                    const int sub = s01 + kp.f0 * kp.f1 * s2;
                                    if (!((cn.mask >> sub) & 1u))
                                        continue;
                                    const int rk = __popc(cn.mask & ((1u << sub) - 1u));
                                    Cx<R>* o = F + int64_t(cn.fine_base + rk) * kp.n_lo + m01;
                                    map_pencil<R, decltype(H)::value>(
                                        W2 + s2 * l2 * h2, h2, l2, X + k * xsz + j01, np,
                                        [&](int j, Cx<R> a) { o[l01 * j] = a; });
                                }
                            }
                        });
    }
}
} // namespace

namespace dev
{
template <typename R>
void launch_up_rows(DevicePlan& D, hipStream_t st, const KParams& kp, int level, const Cx<R>* F,
                    Cx<R>* V)
{
    const int64_t n = D.up_gl_off[level + 1] - D.up_gl_off[level];
    if (n == 0)
        return;
    if (!D.up_tl_desc)
        throw std::runtime_error("upward pass: the per-cone records were not uploaded");
    const size_t full = sizeof(UpDesc) + 8 * size_t(D.n_hi) * sizeof(Cx<R>);
    const bool seq = full > size_t(48) * 1024;
    const size_t lds = seq ? sizeof(UpDesc) + size_t(D.n_hi) * sizeof(Cx<R>) : full;
    constexpr size_t LDS_MAX = 160 * 1024; // gfx950: 160 KB of LDS per CU
    if (lds > LDS_MAX)
        throw std::runtime_error("interpolation orders too large for the upward kernel's LDS");
    const int K = up_cones_per_block(D, n);
    const dim3 grid(unsigned((n + K - 1) / K)), block(seq ? 256 : 128);
    const UpDesc* desc = D.up_tl_desc + D.up_gl_off[level];
    const auto* grp = static_cast<const UpGrpOf<R>*>(D.up_grp);
    with_orders(D.lo[0], D.lo[1], [&](auto o0, auto o1)
                {
                    constexpr int O0 = decltype(o0)::value, O1 = decltype(o1)::value;
                    if (lds > size_t(64) * 1024)
                        HIP_OK(hipFuncSetAttribute(
                            reinterpret_cast<const void*>(&k_up_rows<R, O0, O1, true>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
                    if (seq)
                        k_up_rows<R, O0, O1, true><<<grid, block, lds, st>>>(desc, n, K, D.ctab,
                                                                             grp, F, V, kp);
                    else
                        k_up_rows<R, O0, O1, false><<<grid, block, lds, st>>>(desc, n, K, D.ctab,
                                                                              grp, F, V, kp);
                });
}
template void launch_up_rows<float>(DevicePlan&, hipStream_t, const KParams&, int,
                                    const Cx<float>*, Cx<float>*);
template void launch_up_rows<double>(DevicePlan&, hipStream_t, const KParams&, int,
                                     const Cx<double>*, Cx<double>*);

template <typename R>
void launch_far_rows(DevicePlan& D, hipStream_t st, const KParams& kp, int group, const Cx<R>* F,
                     Cx<R>* far_res)
{
    const DevicePlan::FarGroup& G = D.far_steps[group];
    const int64_t n = G.item1 - G.item0;
    const int split = far_split(n);
    const int phase = D.kind != KL;
    const WorkItem* items = D.far_items + G.item0;
    const int32_t* srange = D.far_srange + 2 * G.item0;
    if constexpr (sizeof(R) == 4)
        if (G.ang_n > 0)
        {
            const int wpb = split > 1 ? split : D.shape.far_waves;
            const int stage = D.n_lo >= 40 && D.n_lo <= 400 ? D.n_lo : 0;
            // entries from one staged cone to the next: 16-byte words, an odd number of them
            // mod 8, so that the four cones' words start in different banks
            const int stride = stage ? (((D.n_lo + 1) / 2) | 1) * 2 : 0;
            const size_t lds = ((G.ang_n + 1) & ~1) * sizeof(double) +
                               (stage ? size_t(wpb) * (FAR_STAGE * stride + ROW_PAD) * sizeof(Cx<R>)
                                      : 0);
            with_orders(D.lo[0], D.lo[1], [&](auto o0, auto o1)
                        {
                            constexpr int O0 = decltype(o0)::value, O1 = decltype(o1)::value;
                            if (lds > size_t(64) * 1024)
                                HIP_OK(hipFuncSetAttribute(
                                    reinterpret_cast<const void*>(&k_far_rows<R, O0, O1, true>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
                            k_far_rows<R, O0, O1, true>
                                <<<dim3(unsigned(split > 1 ? n : (n + wpb - 1) / wpb)),
                                   dim3(64 * wpb), lds, st>>>(
                                    items, n, srange, D.far_src, D.geo, D.ctab, F, D.tgt_pts,
                                    D.fine_ang, G.ang_base, G.ang_n, stage, stride, phase,
                                    split > 1, D.ntgt, far_res, kp);
                        });
            return;
        }
    auto slow = [&](auto o0, auto o1)
    {
        constexpr int O0 = decltype(o0)::value, O1 = decltype(o1)::value;
        k_far_rows<R, O0, O1, false><<<dim3(unsigned(n)), dim3(64 * split), 0, st>>>(
            items, n, srange, D.far_src, D.geo, D.ctab, F, D.tgt_pts, D.fine_ang, 0, 0, 0, 0,
            phase, split > 1, D.ntgt, far_res, kp);
    };
    if constexpr (sizeof(R) == 4) // angle tables too large for LDS: rare
        slow(std::integral_constant<int, 0>(), std::integral_constant<int, 0>());
    else
        with_orders(D.lo[0], D.lo[1], slow);
}
template void launch_far_rows<float>(DevicePlan&, hipStream_t, const KParams&, int,
                                     const Cx<float>*, Cx<float>*);
template void launch_far_rows<double>(DevicePlan&, hipStream_t, const KParams&, int,
                                      const Cx<double>*, Cx<double>*);

template <typename R>
void launch_transform_rows(DevicePlan& D, hipStream_t st, const KParams& kp, int64_t c0, int64_t c1,
                           const Cx<R>* V, Cx<R>* F)
{
    const int h0 = D.ho[0], h1 = D.ho[1], h2 = D.ho[2];
    const int m0 = D.f[0] * D.lo[0], m1 = D.f[1] * D.lo[1];
    const int xsz = std::max(h0 * h1 * h2, m0 * m1 * h2);
    const int ysz = m0 * h1 * h2;
    const size_t per_cone = size_t(xsz + ysz) * sizeof(Cx<R>);
    // several cones fill the threads where one cone's pencils do not; 32 KB keeps 5 workgroups
    // per CU
    const int cpb = int(std::max<size_t>(1, std::min<size_t>(8, (32 * 1024) / per_cone)));
    const size_t lds = cpb * per_cone;
    constexpr size_t LDS_MAX = 160 * 1024; // gfx950: 160 KB of LDS per CU
    if (lds > LDS_MAX)
        throw std::runtime_error("interpolation orders too large for the transform kernel's LDS");
    if (lds > size_t(64) * 1024)
        HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(&k_transform_rows<R>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    k_transform_rows<R><<<dim3(unsigned((c1 - c0 + cpb - 1) / cpb)), dim3(256), lds, st>>>(
        c0, c1, cpb, xsz, ysz, D.cones, V, F, static_cast<const R*>(D.wmat), kp);
}
template void launch_transform_rows<float>(DevicePlan&, hipStream_t, const KParams&, int64_t,
                                           int64_t, const Cx<float>*, Cx<float>*);
template void launch_transform_rows<double>(DevicePlan&, hipStream_t, const KParams&, int64_t,
                                            int64_t, const Cx<double>*, Cx<double>*);

template <typename R> void record_far(DevicePlan& D)
{
    const KParams kp = kparams(D);
    const int phase = D.kind != KL;
    for (const DevicePlan::FarGroup& G : D.far_steps)
    {
        const dim3 grid(unsigned(G.item1 - G.item0));
        const int64_t i0 = G.item0;
        auto* rec = static_cast<FarRec<R>*>(D.far_rec);
        auto* cf = static_cast<Cx<R>*>(D.far_cf);
        if (sizeof(R) == 4 && G.ang_n > 0)
            k_far_record<R, true><<<grid, dim3(64), size_t(G.ang_n) * sizeof(double)>>>(
                D.far_items + i0, D.far_srange + 2 * i0, D.far_rec_off + i0, D.far_src, D.geo,
                D.ctab, D.tgt_pts, D.fine_ang, G.ang_base, G.ang_n, phase, rec, cf, kp);
        else
            k_far_record<R, false><<<grid, dim3(64)>>>(
                D.far_items + i0, D.far_srange + 2 * i0, D.far_rec_off + i0, D.far_src, D.geo,
                D.ctab, D.tgt_pts, D.fine_ang, 0, 0, phase, rec, cf, kp);
        HIP_OK(hipGetLastError());
    }
}
template void record_far<float>(DevicePlan&);
template void record_far<double>(DevicePlan&);

template <typename R>
void launch_far_rec(DevicePlan& D, hipStream_t st, const KParams& kp, int group, const Cx<R>* F,
                    Cx<R>* far_res)
{
    const DevicePlan::FarGroup& G = D.far_steps[group];
    const int64_t n = G.item1 - G.item0;
    const int split = far_split(n);
    const int wpb = split > 1 ? split : D.shape.far_waves;
    // (staging from 16 coefficients on: far phase at (2,3,3), 262,144 points, 0.76 against 0.98 ms
    // with every lane reading its cone from memory; at (2,5,5), 1M points, 3.5 against 6.7 ms)
    // up to 112 KB per workgroup
    const int stride = (((D.n_lo + 1) / 2) | 1) * 2;
    const size_t staged = size_t(wpb) * (FAR_STAGE * stride + ROW_PAD) * sizeof(Cx<R>);
    const int stage = D.n_lo >= 16 && staged <= size_t(112) * 1024 ? D.n_lo : 0;
    const size_t lds = stage ? staged : 0;
    with_orders(D.lo[0], D.lo[1], [&](auto o0, auto o1)
                {
                    constexpr int O0 = decltype(o0)::value, O1 = decltype(o1)::value;
                    if (lds > size_t(64) * 1024)
                        HIP_OK(hipFuncSetAttribute(
                            reinterpret_cast<const void*>(&k_far_rec<R, O0, O1>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
                    k_far_rec<R, O0, O1>
                        <<<dim3(unsigned(split > 1 ? n : (n + wpb - 1) / wpb)), dim3(64 * wpb),
                           lds, st>>>(D.far_items + G.item0, n, D.far_srange + 2 * G.item0,
                                      D.far_rec_off + G.item0,
                                      static_cast<const FarRec<R>*>(D.far_rec),
                                      static_cast<const Cx<R>*>(D.far_cf), F, stage, stride,
                                      split > 1, D.ntgt, far_res, kp);
                });
}
template void launch_far_rec<float>(DevicePlan&, hipStream_t, const KParams&, int,
                                    const Cx<float>*, Cx<float>*);
template void launch_far_rec<double>(DevicePlan&, hipStream_t, const KParams&, int,
                                     const Cx<double>*, Cx<double>*);
} // namespace dev
} // namespace ifgf
