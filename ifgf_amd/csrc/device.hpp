// device.hpp -- device-resident plan and the mult pipeline (host-side declarations).
#pragma once

#include <cstdint>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "plan.hpp"

namespace ifgf
{
enum Precision
{
    PREC_FP64 = 0,  // every step in FP64 (the plain form)
    PREC_MIXED = 1  // FP32 arithmetic; FP64 for cone coordinates, phases and box geometry
};

// geometry and cone grid of one source box, as read by the kernels
struct BoxGeo
{
    double ctr[3];
    double H;
    double lo[3];     // cone domain (s, theta, phi)
    double hi[3];
    double hf[3];     // fine cell widths
    double inv_hf[3]; // 1 / hf (cell search; exact division near cell boundaries)
    double hc[3];     // coarse cell widths
    int32_t nf[3];    // fine cells per axis
    int32_t nc[3];    // coarse cells per axis
    int64_t table_off;
    int32_t th_off;   // node-angle tables of the coarse grid (cos/sin per cell and node)
    int32_t ph_off;
    int32_t fth_off;  // fine-grid theta table: (cos, sin) of the nf1+1 cell edges, then centres
    int32_t fph_off;  // fine-grid phi table: the same for the nf2 cells
    double k_re, k_im, kappa; // wavenumber of the box's geometry (e^{-k d}; kappa: real form)
};

struct ConeDev
{
    int32_t box;
    int32_t cell;      // coarse cell id within the box grid
    uint32_t mask;     // active fine sub-cones
    int32_t fine_base; // first fine slot
};

// coarse cell of a box grid, as the cone lookups read it: the fine slots of its cone in one
// load (mask 0: no cone in the cell)
struct CellRef
{
    int32_t fine_base;
    uint32_t mask;
};

struct WorkItem // a chunk of at most 64 consecutive target points of one target box
{
    int32_t box;   // target box (global id in the target tree)
    int32_t first; // first target point (sorted order)
    int32_t count; // 1..64
    int32_t pad;
};

struct PointRun // consecutive source points [begin, end) in Morton order
{
    int32_t begin, end;
};

// Launch shapes of the mult's kernels: choices that change speed but not results, picked by
// device_autotune (measured on the operator itself), set by the caller, or where the upload
// starts from something else than these defaults (device_upload).
struct LaunchShape
{
    int xcd_log2 = 4; // work items dealt to the XCDs in runs of 2^xcd_log2 (0: plain order)
    int cpb = 0;      // transform: cones per workgroup (0: the order class's default)
    int up_k = 16;    // upward: parent cones per workgroup, at most (2, 4, 8 or 16)
    int rb = 0;       // batched: most columns per pass (8 or 32; 0: 32)
    int far_waves = 1; // far field: waves (items) per workgroup, sharing the LDS tables of the
                       // launches that locate the pairs
    int overlap = 1;   // far field on a second stream beside the upward chain, with the near
                       // field there too (1) or first on the main stream (2); 0: one stream
};
// tiles of the grouped upward kernels' work list: parent boxes (in Morton order within a level)
// x cells (table index) per tile
constexpr int UP_TILE_BOXES = 16;
constexpr int UP_TILE_CELLS = 128;

// What k_up_grp and k_up_rows need of a parent cone before its tasks, per entry of the tiled
// upward list, computed at upload from the plan's fixed tables: read as one
// 16-byte-aligned record instead of a chain of dependent loads (cone -> box -> children ->
// their tables -> the (cell, octant) rows -> the listed child cones' slots).
// entries allocated past the fine coefficients: kernels that read a cone's coefficients a chunk
// of rows at a time may read up to this far past the last cone's (and use none of it)
constexpr int ROW_PAD = 40;
constexpr int UP_DMAX = 32; // listed child cones per (parent cone, child) with a slot here
struct alignas(16) UpDesc
{
    int64_t toff[8];          // child c's coarse-cell table offset (-1: no child c)
    int32_t tg0[8];           // the group record of child c's task t is tg0[c] + t
    int32_t tend[8];          // child c's tasks end at tend[c] (prefix over the children)
    int32_t g;                // the parent cone
    uint32_t mask;            // its active fine sub-cones
    int32_t fine_base;        // its first fine slot
    int32_t pad;
    int32_t slot[8][UP_DMAX]; // fine slot of listed child cone d of child c (-1: inactive)
};
static_assert(sizeof(UpDesc) == 1168, "UpDesc is 73 16-byte words");

// bytes of the fixed device scratch of the allocation-free mult (device_mult_noalloc): the
// Morton-order densities and results of one column (64 MiB: n_src + n_tgt up to 8,388,576
// points in the mixed form, 4,194,272 in FP64)
constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(64) << 20;

struct DevicePlan
{
    int device = -1; // HIP device of the upload
    int prec = PREC_MIXED;
    int kind = 0;
    double k_re = 0, k_im = 0; // e^{-k d}
    double kappa = 0;
    int dx = -1;
    int ho[3], lo[3], f[3];
    int n_hi = 0, n_lo = 0, nsub = 0;
    int64_t nsrc = 0, ntgt = 0;
    int levels = 0;
    int64_t n_cones = 0, n_fine = 0;

    // device arrays (raw pointers owned by this struct)
    double* src_pts = nullptr;   // sorted, xyz
    double* tgt_pts = nullptr;
    double* normals = nullptr;   // sorted source normals (DL, CF) or null
    int64_t* src_perm = nullptr;
    int64_t* tgt_perm = nullptr;
    int64_t* src_begin = nullptr; // per source box
    int64_t* src_end = nullptr;
    int32_t* child = nullptr;     // 8 per source box
    BoxGeo* geo = nullptr;
    ConeDev* cones = nullptr;
    CellRef* ctab = nullptr;      // per box: dense coarse-cell table (BoxGeo::table_off)
    double* ho_nodes = nullptr;   // n_hi x 3 reference nodes in [-1,1]^3
    double* trig_th = nullptr;    // (cos, sin) of theta at coarse cell / node, per grid class
    double* trig_ph = nullptr;    // (cos, sin) of phi
    double* fine_ang = nullptr;   // fine-grid edge / centre (cos, sin) tables
    void* wmat = nullptr;         // axis maps (R): W0 | W1 | W2
    int woff[4] = {0, 0, 0, 0};

    // the upward geometry tables of every part (a level of one geometry) regrouped by child cone
    // (UpGrp / UpGrpD records): one read of a child cone's coefficients serves the nodes that
    // fall into it
    void* up_grp = nullptr;
    // the parent cones with a table, per level (up_gl_off) in tiles of UP_TILE_BOXES boxes x
    // UP_TILE_CELLS cells
    std::vector<int64_t> up_gl_off;
    UpDesc* up_tl_desc = nullptr; // one record per cone of the list

    int32_t* leaf_cones = nullptr;
    int64_t n_leaf_cones = 0;
    // per level, the cones whose values -> coefficients transform runs on its own (non-leaf
    // cones without an upward table) when leaf sampling and k_up_grp transform theirs
    int32_t* tr_list = nullptr;
    std::vector<int64_t> tr_list_off;
    WorkItem* leaf_boxes = nullptr; // leaf boxes with active cones: (box, first cone, count)
    int64_t n_leaf_boxes = 0;
    int32_t* up_cones = nullptr;             // non-leaf cones without a table, level-major
    std::vector<int64_t> up_off;             // per level, into up_cones
    std::vector<int64_t> cone_lvl_off;       // per level, global cone range

    int32_t* far_src = nullptr;   // far source boxes, by target box then source box
    int32_t* far_srange = nullptr; // per far item: its sources far_src[2i] .. far_src[2i + 1]
    // near sources by target box: runs of consecutive points near_run[near_off[t]] ..
    // near_run[near_off[t + 1]], near_pts[t] points in all
    int32_t* near_off = nullptr;
    PointRun* near_run = nullptr;
    int32_t* near_pts = nullptr;
    WorkItem* far_items = nullptr;
    // the far launches, deepest source level first: the items of one source level (of one target
    // level each where their angle tables would not fit LDS together); a launch can run as soon
    // as its source level's coefficients exist.  A target point is in boxes of several levels, so
    // the items of target level t (WorkItem::pad: its index among the target levels with far
    // items) add to their own results, far_res[pad * ntgt ..], and the scatter sums the levels in
    // order.
    struct FarGroup
    {
        int64_t item0, item1; // far_items[item0 .. item1)
        int ang_base, ang_n;  // the sources' angle tables staged in LDS (mixed form; 0: none)
        int src_level;
    };
    std::vector<FarGroup> far_steps;
    // Where each (target, far source box) pair lies, in the order of the far items (item i's
    // records from far_rec_off[i] on, its targets fastest): the fine slot and local coordinates
    // (FarRec) and the centre factor.  All from the geometry and the wavenumber, so recorded once
    // at upload by the location the far field would otherwise repeat in every mult; null when
    // they would take more than a quarter of the free device memory less 4 GiB (24 bytes a pair in
    // the mixed form, 48 in FP64), or were refused.
    int64_t* far_rec_off = nullptr;
    void* far_rec = nullptr; // FarRec<R>
    void* far_cf = nullptr;  // Cx<R>
    int n_far_lvls = 0;
    void* far_res = nullptr; // n_far_lvls * ntgt complex (R)
    WorkItem* near_items = nullptr;
    int64_t n_near_items = 0;

    // work buffers of the single-column mult
    void* wsorted = nullptr;  // N complex (R)
    void* result = nullptr;   // M complex (R)
    void* V = nullptr;        // n_cones * n_hi complex (R)
    void* F = nullptr;        // n_fine * n_lo complex (R)
    // level storage (ring): instead of every level's values and coefficients, V holds the values
    // of one level and F_bank[l & 1] the fine coefficients of level l (a level's coefficients
    // are read only by the upward pass of the level above and the far field of that source
    // level); for operators whose coefficients of all levels exceed the device memory
    bool ring = false;
    void* F_bank[2] = {nullptr, nullptr};
    std::vector<int64_t> fine_lvl_off;    // per level, global fine-slot range
    std::vector<int64_t> leaf_lvl_off;    // per level, range of leaf_boxes
    std::vector<void*> ev_far_done;       // ring on two streams: far groups of a source level done
    int64_t bytes_total = 0;

    // the single-column mult's core captured as a graph (on first use with graphs enabled),
    // and the batched mult's core for the current batch buffers, per number of columns (at most
    // MAX_COLUMNS) and the forms of mult_batched: hipGraph_t, hipGraphExec_t
    void* graph = nullptr;
    void* graph_exec = nullptr;
    std::map<int, std::pair<void*, void*>> b_graphs;
    void* cap_stream = nullptr; // hipStream_t of the capture
    // the second stream of the overlapped near field and its fork / join events
    void* side_stream = nullptr;
    void* ev_fork = nullptr;
    void* ev_near = nullptr;
    std::vector<void*> ev_level; // per source level: its coefficients are written

    LaunchShape shape;
    bool shape_chosen = false; // by device_set_shape, not the upload
    // per-phase device times of this operator's last timed mult (ms: near, leaf, upward,
    // transform, far, total); force_timing: time the phases of the next mults (autotuner)
    float last_ms[6] = {0, 0, 0, 0, 0, 0};
    bool force_timing = false;

    // staging of host densities and results of single-column mults (first use)
    double *h_in = nullptr, *h_out = nullptr;

    // work buffers of the batched mult (up to b_rb columns, column-minor; the results followed by
    // the far results of each target level), allocated on first use; b_in / b_out stage host
    // densities and results
    int b_rb = 0;
    void *b_ws = nullptr, *b_res = nullptr, *b_V = nullptr, *b_F = nullptr;
    double *b_in = nullptr, *b_out = nullptr;
    int64_t b_bytes = 0;
    // the most columns asked for so far, and whether with host densities: memory may have allowed
    // fewer (ensure_batch)
    int b_asked = 0;
    bool b_asked_host = false;
};

// ring: 0 = every level resident when it fits the device memory, else level storage;
// 1 = level storage (DevicePlan::ring).  records: lay down the far pair records where memory allows
std::string device_upload(const Plan& P, int precision, DevicePlan& D, int ring, bool records);
void device_free(DevicePlan& D);
// coarse cones of one mult's standalone values -> coefficients transform (all of them unless
// leaf sampling and the grouped upward kernel transform their own)
int64_t device_transform_cones(const DevicePlan& D);
// batched mult (batched.hip): ncol <= b_rb columns of device densities
constexpr int MAX_COLUMNS = 32;
// calls of at most this many columns take the far field by groups of columns (k_far_few_cols), the
// others 16 real columns at a time.  Whole mult of 8, 12 and 16 columns by groups / by tiles:
// 7.9 / 10.2, 11.9 / 14.6 and 16.4 / 16.1 ms at (2,3,3), 262,144 points; 7.3 / 8.6, 11.5 / 11.6 and
// 15.0 / 13.3 at (3,5,4), 100,000 points; FP64 at (3,5,4), 50,000 points, 11.6 / 12.3, 17.2 / 17.3
// and 21.8 / 19.9.
constexpr int FEW_COLUMNS = 12;
// few: of a call of at most FEW_COLUMNS; tiles: the transform on MFMA tiles
void mult_batched(DevicePlan& D, const double* w_dev, double* out_dev, int ncol, void* stream,
                  int io, bool graph, bool few, bool tiles);
// w: complex128 (host or device), out: complex128 (host or device); nrhs columns of length
// N / M stored one after another.  io: IO_* bits applied while the densities are gathered and
// the results scattered (conjugations and a sign, for adjoint products).
enum
{
    IO_CONJ_IN = 1,
    IO_CONJ_OUT = 2,
    IO_NEGATE_OUT = 4
};
std::string device_mult(DevicePlan& D, const void* w, void* out, int64_t nrhs, bool device_ptrs,
                        void* stream, int io = 0, bool graph = false);
// One column of device densities into device results with no device allocation: the staging
// vectors live in the library's fixed per-device scratch (NOALLOC_SCRATCH_BYTES; larger
// operators are refused), everything on `stream`, no phase timing, no graph.  Calls that
// overlap on one GPU race on the scratch.  The current device must be the upload's.
std::string device_mult_noalloc(DevicePlan& D, const double* w_dev, double* out_dev,
                                void* stream);
// Apply a launch shape (validated; an unknown choice is an error).  Drops a captured graph.
std::string device_set_shape(DevicePlan& D, const LaunchShape& s);
// Drop the captured graphs of the single-column and batched mults (after a change of their
// kernel arguments).
void device_drop_graph(DevicePlan& D);
// Time the candidate shapes on this operator with synthetic densities (nrhs columns, each
// candidate `reps` times, the fastest kept), one choice after another: the XCD run length on
// the whole mult, then the transform's cones per workgroup, the upward cones per item and the
// far field's waves per workgroup on their phases, then (nrhs >= 3) the batched columns per
// pass.  Leaves the best shape applied.
std::string device_autotune(DevicePlan& D, int64_t nrhs, int reps, LaunchShape& best);
// per-phase timings of the last mult (ms): near, leaf, upward, transform, far, total
void device_last_timings(const DevicePlan& D, double* out6);
bool device_available();

// The source or target octree of init on the device (tree.hip): the same Tree as build_tree
// (identical permutation, boxes and point ranges).  Returns "" or an error.
std::string device_build_tree(const double* pts, int64_t n, int64_t max_leaf, Tree& T);
// The cone marking of build_cones on the device (cones.hip): the same bitmaps as the host's.
ConeMarker make_device_cone_marker();
// The interaction lists on the device (pairs.hip): the same sorted lists as build_interactions.
std::string device_build_interactions(Plan& P);
// all three device builders
inline PlanBuilders device_plan_builders()
{
    PlanBuilders b;
    b.tree = device_build_tree;
    b.pairs = device_build_interactions;
    b.cones = make_device_cone_marker();
    return b;
}
} // namespace ifgf
