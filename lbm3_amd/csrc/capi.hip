// C ABI of the hot path (include/lbm3mi.h): simulation objects, level import,
// the per-step driver with 2:1 sub-cycling, observables and timing.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <vector>
#include <mutex>
#include <new>
#include "sim.hpp"
#include "levelargs.hpp"

namespace lbm3 {

static thread_local std::string g_error;

int set_error(int code, const std::string &msg)
{
    g_error = msg;
    return code;
}

int check_hip(hipError_t e, const char *what)
{
    if (e == hipSuccess) return 0;
    (void)hipGetLastError();   // reported here: the next launch's check must not find it again
    return set_error(LBM3_E_HIP, std::string(what) + ": " + hipGetErrorString(e));
}

#define HIPCHK(expr)                                  \
    do {                                              \
        const int rc_ = check_hip((expr), #expr);     \
        if (rc_) return rc_;                          \
    } while (0)

size_t storage_bytes(int storage)
{
    switch (storage) {
    case LBM3_STORE_F16: case LBM3_STORE_BF16: case LBM3_STORE_F16C: return 2;
    case LBM3_STORE_F64: return 8;
    default: return 4;
    }
}
size_t compute_bytes(int storage) { return storage == LBM3_STORE_F64 ? 8 : 4; }

// 16-bit encoding: deviation from the shifted equilibrium at rho = 1 and the
// case's reference velocity, in units of the weight
Codec make_codec(const lbm3_case &c, int storage)
{
    Codec k;
    for (int q = 0; q < 27; ++q) {
        k.off[q] = feq_shifted<float>(q, 0.f, c.storeRef[0], c.storeRef[1], c.storeRef[2]);
        k.w[q] = weight<float>(q);
        k.iw[q] = 1.f / k.w[q];
        if (storage == LBM3_STORE_F16C) {   // the f16c bit pattern is that of the value times 2^-112
            k.w[q] = std::ldexp(k.w[q], 112);
            k.iw[q] = std::ldexp(k.iw[q], -112);
        }
    }
    for (int a = 0; a < 3; ++a) k.u[a] = c.storeRef[a];
    return k;
}


template <class T> static int upload(DBuf<T> &b, const T *host, long long n, hipStream_t s)
{
    HIPCHK(b.alloc(n));
    if (n > 0 && host) HIPCHK(hipMemcpyAsync(b.p, host, sizeof(T) * (size_t)n, hipMemcpyHostToDevice, s));
    return 0;
}

// the bulk kernel's skip masks and block rows, from the current cell records
static int refresh_bulk_mask(Sim &s, Level &l)
{
    const long long blocks = (l.N + 255) / 256;
    if (l.waveRow.n < 4 * blocks) HIPCHK(l.waveRow.alloc(blocks > 0 ? 4 * blocks : 4));
    if (l.bulkSkip.n < 4 * blocks) HIPCHK(l.bulkSkip.alloc(blocks > 0 ? 4 * blocks : 4));
    if (l.openInBulk && l.openBits.n < 4 * blocks) HIPCHK(l.openBits.alloc(blocks > 0 ? 4 * blocks : 4));
    if (l.rotorInBulk && l.rotorBits.n < 4 * blocks) HIPCHK(l.rotorBits.alloc(blocks > 0 ? 4 * blocks : 4));
    launch_bulk_mask(l.cellRow.p, l.N, l.bulkSkip.p, l.waveRow.p, l.openInBulk ? l.openBits.p : nullptr,
                     l.rotorInBulk ? l.rotorBits.p : nullptr, s.stream);
    return check_hip(hipGetLastError(), "bulk mask");
}

// the open-boundary records the level's open cells index: the level's own list
// (built from the rule table or the case's getOpenBC hook), else the rule table
static int upload_open_records(Sim &s, Level &l)
{
    std::vector<OpenBCRecord> rec;
    if (!l.openBC.empty()) {
        for (const lbm3_bc &b : l.openBC) rec.push_back(open_record(b));
    } else {
        for (int r = 0; r <= s.C.nOpenRules; ++r) rec.push_back(open_record(open_bc(s.C, r)));
    }
    for (OpenBCRecord &r : rec) {
        r.impedance = s.C.openScheme == LBM3_OPEN_IMPEDANCE;
        r.tolerance = s.C.rhoReflectionTolerance;
    }
    if (upload(l.openRecords, rec.data(), (long long)rec.size(), s.stream)) return LBM3_E_HIP;
    return 0;
}

int hook_local_bc(Sim &s, int level, LocalBC &bulk, LocalBC (&wb)[32]);   // casehooks.hip
int hook_initial_fields(Sim &s, int level, DBuf<float> &fields4);

// getLocalBC per (level, wall id): the rule table, or the case's own hook
static int setup_local_bc(Sim &s, int level)
{
    Level &l = s.L[level];
    LocalBC wb[32];
    l.wallVel.release();
    if (s.hooks.local_bc) {
        if (const int rc = hook_local_bc(s, level, l.bulk, wb)) return rc;
    } else {
        l.bulk = local_bc(s.C, level, -1);
        for (int w = 0; w < 32; ++w) wb[w] = local_bc(s.C, level, w);
    }
    set_relax(l.bulk, double(l.info.nu));
    for (int w = 0; w < 32; ++w) set_relax(wb[w], double(l.info.nu));
    if (upload(l.wallBC, wb, 32, s.stream)) return LBM3_E_HIP;
    return 0;
}

static int settle_open(Sim &s, int L);

static int prepare_open_fusion(Sim &s, int L);

// entry points of casehooks.hip and serve.hip into this file
int prepare_cells(Sim &s, int level) { return prepare_open_fusion(s, level); }   // serve.hip
int upload_open_records_of(Sim &s, Level &l) { return upload_open_records(s, l); }
int settle_open_level(Sim &s, int level) { return settle_open(s, level); }
int setup_local_bc_of(Sim &s, int level) { return setup_local_bc(s, level); }

// derived per-level tables: local BC, open-BC records, force accumulators, populations
int finish_level_setup(Sim &s, int level)
{
    Level &l = s.L[level];
    l.geom = LevelGeom{l.info.res, l.info.ox, l.info.oy, l.info.oz, l.info.dtPhys, l.info.cellCountX, l.info.cellCountY,
                       l.info.cellCountZ};
    if (l.N > (1LL << 31) - 1 - LBM3_TILE) return set_error(LBM3_E_MEMORY, "a level exceeds 2^31 cells");
    if (const int rc = setup_local_bc(s, level)) return rc;
    HIPCHK(l.cellRow.alloc(l.N > 0 ? l.N : 1));
    HIPCHK(l.rowTab.alloc(l.nRows + kRowPad));
    launch_fast_topo(topo_of(l), l.nRows, l.wallMap.p, nullptr, nullptr, l.cellRow.p, l.rowTab.p, s.stream);
    if (const int rc = refresh_bulk_mask(s, l)) return rc;
    // interface neighbour tables that read this level are derived again
    l.F2C.nbReady = l.C2F.nbReady = false;
    if (level > 0) s.L[level - 1].F2C.nbReady = s.L[level - 1].C2F.nbReady = false;
    l.rotors.clear();              // rotors belong to the grid they were built on
    l.rotorDev.release();
    l.rotorCellCount = 0;
    l.openFusionChecked = false;
    l.imagesReady = false;
    l.ghostsStale = false;
    l.shared = false;
    l.fusedOpen = false;
    l.openInBulk = false;
    l.rotorInBulk = false;
    l.openSettled = true;
    HIPCHK(l.openNb.alloc(2LL * (l.nOpen > 0 ? l.nOpen : 1)));
    launch_open_nb(topo_of(l), l.nOpen, l.openCell.p, l.openNb.p, s.stream);
    HIPCHK(hipGetLastError());
    if (const int rc = upload_open_records(s, l)) return rc;
    // radial profiles of the rule table (the case's own hook returns final values)
    OpenProfiles prof{};
    bool profiled = false;
    for (int r = 0; r < s.C.nOpenRules && !s.hooks.open_bc; ++r) {
        prof.p[r] = s.C.openRules[r].profile;
        profiled = profiled || prof.p[r].radius > 0.f;
    }
    l.openScale.release();
    if (profiled && l.nOpen > 0) {
        HIPCHK(l.openScale.alloc(l.nOpen));
        launch_open_scale(topo_of(l), l.geom, l.nOpen, l.openCell.p, l.openMeta.p, prof, l.openScale.p, s.stream);
        HIPCHK(hipGetLastError());
    }
    HIPCHK(l.gWall.alloc(3LL * (l.W > 0 ? l.W : 1)));
    HIPCHK(hipMemsetAsync(l.gWall.p, 0, sizeof(double) * (size_t)l.gWall.n, s.stream));
    HIPCHK(l.openRefs.alloc(2LL * (l.nOpen > 0 ? l.nOpen : 1) * (long long)compute_bytes(s.storage)));
    HIPCHK(hipMemsetAsync(l.openRefs.p, 0, (size_t)l.openRefs.n, s.stream));
    HIPCHK(l.openCum.alloc(2LL * (l.nOpen > 0 ? l.nOpen : 1)));
    HIPCHK(hipMemsetAsync(l.openCum.p, 0, sizeof(double) * (size_t)l.openCum.n, s.stream));
    HIPCHK(l.f.alloc(27LL * padded_cells(l.N) * (long long)storage_bytes(s.storage)));
    l.built = true;
    return 0;
}



static int settle_open(Sim &s, int L);

static bool wide_of(const Sim &s, const Level &l)
{
    return 27LL * padded_cells(l.N) * (long long)storage_bytes(s.storage) > 0xFFFFFFFFLL;
}

// The launch choices of a level that nobody chose (lbm3_set_tune, lbm3_autotune).
// Times are us per step on this GPU, FP32 unless said otherwise:
// * one launch per step: the wall-adjacent cells in blocks ahead of the bulk
//   blocks, the open cells and the rotor cells in the bulk kernel.  Against
//   groups of open cells, wall cells and rotor cells on side streams: sphere
//   96x48x48 57 -> 24, 186x92x84 (K17) 86 -> 57, 256x128x128 179 -> 155 (FP16
//   126 -> 94), two-level rotor duct 427 -> 286, and the smallest boxes too:
//   sphere 48x24x24 34 -> 18.  FP64: 48x24x24 48 -> 14, 256x128x128 445 -> 328.
// * the levels in order on one stream: three-level sphere 344, with a stream
//   per level 384.
// * block order: one contiguous part per XCD, swept backwards every other step
//   (order 3), so that each XCD's L2 and the last-level cache still hold what
//   the step starts on: 64^3 vortex 14.9 against 18.3 in plain order, 118^3 57 /
//   63, sphere 260x130x130 (453 MiB) 171 / 174.  The plain order swept backwards (2)
//   wins above about 512 MiB of populations, 272x136x136 (518 MiB) 201 / 203,
//   300x150x150 272 / 287, FP64 140^3 vortex (590 MiB) 204 / 217, and where rotors
//   make some parts slower than others: rotor duct 286 / 306.
// * occupancy cap of the bulk kernel (40 KiB of LDS per block, four blocks per
//   CU: their tiles then fit an XCD's L2), each where one simulation alone on the
//   GPU is faster with it: above 640 MiB, 300x150x150 (695 MiB) 272 against 273,
//   340x170x170 411 / 418, 400x200x200 659 / 695 (288x144x144 of 615 MiB 237 /
//   230); on refined levels with walls above 256 MiB, three-level sphere 88 across
//   (317 MiB) 757 / 767, 100 across 1106 / 1112; and on levels of 64 to 256 MiB
//   without open cells, 92^3 vortex (86 MiB) 30.4 / 30.8, 118^3 53 / 57, 130^3
//   (237 MiB) 72 / 91, FP64 104^3 73 / 76 (80^3 of 57 MiB 23.0 / 22.3, 140^3 of 295
//   MiB 122 / 117).  Several simulations at once on streams of their own want it
//   earlier: three 272x136x136 in turn 231 / 266.  Never for 16-bit storage,
//   whose kernels are bound by instructions: FP16 272x136x136 159 / 137,
//   360x180x180 357 / 285.
// The levels' wall cells on a side stream, as the three-level sphere above 200
// MiB had them for several simulations at once (three in turn, 88 across, 833
// against 894), cost one alone 783 against 757, FP64 64 across 685 against 606.
Sim::Tune tune_of(const Sim &s, const Level &l)
{
    if (s.tuneChosen) return s.tune;
    constexpr long long MiB = 1LL << 20;
    const long long size = (long long)storage_bytes(s.storage), bytes = 27 * size * l.N;
    Sim::Tune t;
    t.overlap = 3;
    t.ordered = true;
    // the same on every level: a new layout rebuilds all of them (same_open_layout)
    for (int L = 0; L < s.levels; ++L) t.rotorInBulk |= s.L[L].rotors.empty() ? 0 : 1;
    t.openGroup = 1;
    t.openSplit = s.ownSplit;
    t.xcdRemap = !l.rotors.empty() || bytes > 512 * MiB ? 2 : 3;
    const bool refined = s.levels > 1 && l.W > 0 && l.rotors.empty();
    const bool cap = bytes > 640 * MiB || (!l.openInBulk && bytes > 64 * MiB && (refined || bytes <= 256 * MiB));
    t.bulkLds = size >= 4 && cap ? LBM3_BULK_LDS : 0;
    return t;
}

// Whether the bulk kernel can step the periodic ghosts from their source cells
// (one launch per step instead of a copy after each): a single level that is a
// full box of plain fluid cells where ghosts and sources lie.  Levels with
// wall-adjacent or rotor cells, whose kernels could step a ghost, an interface
// that reads ghosts, or 64-bit offsets keep the copy.
static int prepare_images(Sim &s, Level &l)
{
    l.imagesReady = false;
    const long long box = (long long)l.info.cellCountX * l.info.cellCountY * l.info.cellCountZ;
    if (l.nPeriodic == 0 || s.levels != 1 || l.W > 0 || !l.rotors.empty() || l.laneRot || l.N != box || wide_of(s, l)) return 0;
    const long long words = 4 * ((l.N + 255) / 256);
    DBuf<int> flag;
    HIPCHK(flag.alloc(1));
    // where the tables do not fit beside the level the copy needs none
    if (l.ghostSkip.alloc(words) != hipSuccess || l.imageSources.alloc(words) != hipSuccess ||
        l.imageHead.alloc(l.N) != hipSuccess || l.imageInfo.alloc(l.nPeriodic) != hipSuccess ||
        l.imageNb.alloc(2LL * l.nPeriodic) != hipSuccess) {
        (void)hipGetLastError();
        l.ghostSkip.release();
        l.imageSources.release();
        l.imageHead.release();
        l.imageInfo.release();
        l.imageNb.release();
        return 0;
    }
    HIPCHK(hipMemsetAsync(flag.p, 0, sizeof(int), s.stream));
    HIPCHK(hipMemsetAsync(l.imageSources.p, 0, sizeof(uint64_t) * (size_t)words, s.stream));
    HIPCHK(hipMemcpyAsync(l.ghostSkip.p, l.bulkSkip.p, sizeof(uint64_t) * (size_t)words, hipMemcpyDeviceToDevice, s.stream));
    FastTopo ft{};
    ft.N = l.N;
    ft.cellRow = l.cellRow.p;
    ft.rows = l.rowTab.p;
    ft.skip = l.bulkSkip.p;
    ft.nRows = l.nRows;
    launch_images(topo_of(l), ft, l.geom, l.nPeriodic, l.perIndex.p, l.perSource.p, l.ghostSkip.p, l.imageSources.p,
                  l.imageHead.p, l.imageInfo.p, l.imageNb.p, flag.p, s.stream);
    HIPCHK(hipGetLastError());
    int bad = 0;
    HIPCHK(hipMemcpyAsync(&bad, flag.p, sizeof(int), hipMemcpyDeviceToHost, s.stream));
    HIPCHK(hipStreamSynchronize(s.stream));
    l.imagesReady = bad == 0;
    return 0;
}

// Decide which special cells of level L get kernels of their own and rebuild
// the per-cell records the bulk kernel skips them by:
// * the cells a rotor can reach at some angle (record -4, k_rotor_cells);
// * on level 0, the open-boundary cells (record -(8 + open index),
//   k_open_groups over aligned groups of cells around them, which applies the
//   boundary condition when it next loads the cell), unless an open cell is wall-adjacent or reachable by a rotor, or a
//   periodic copy or an interface transfer touches one (those passes read or
//   write whole cells and need the condition applied in the same step).
static int prepare_open_fusion(Sim &s, int L)
{
    Level &l = s.L[L];
    const Sim::Tune tune = tune_of(s, l);
    if (const int rc = settle_open(s, L)) return rc;   // a condition pending under the old records
    l.openFusionChecked = true;
    l.imagesReady = false;
    l.fusedOpen = false;
    l.openInBulk = false;
    l.laneRot = false;
    l.rotorInBulk = false;
    l.openSettled = true;
    l.rotorCellCount = 0;
    const uint8_t *cand = nullptr;
    if (!l.rotors.empty()) {
        RotorReachSet R{};
        R.n = (int)l.rotors.size();
        for (int r = 0; r < R.n; ++r) {
            const RotorDev &d = l.rotors[r].dev;
            R.r[r] = RotorReach{{d.xMin, d.yMin, d.zMin}, {d.xMax, d.yMax, d.zMax}, {d.ox, d.oy, d.oz}, d.axis};
        }
        HIPCHK(l.rotorCand.alloc(l.N > 0 ? l.N : 1));
        launch_rotor_reach(topo_of(l), l.geom, R, l.rotorCand.p, s.stream);
        cand = l.rotorCand.p;
    }
    DBuf<int> openOf;
    bool fuse = false;
    // without room for the index the open cells keep their pass after streaming
    bool index = L == 0 && l.nOpen > 0;
    if (index && openOf.alloc(l.N) != hipSuccess) {
        (void)hipGetLastError();
        index = false;
    }
    if (index) {
        DBuf<int> flag;
        HIPCHK(flag.alloc(1));
        HIPCHK(hipMemsetAsync(openOf.p, 0xFF, sizeof(int) * (size_t)l.N, s.stream));
        HIPCHK(hipMemsetAsync(flag.p, 0, sizeof(int), s.stream));
        launch_scatter_index(l.openCell.p, l.nOpen, openOf.p, s.stream);
        const FastTopo t{l.N, l.cellRow.p, l.rowTab.p};
        const int *wm = l.wallMap.p;
        int *fl = flag.p;
        launch_open_conflicts(l.openCell.p, l.nOpen, 3, openOf.p, wm, cand, t, fl, s.stream);
        if (cand) launch_open_conflicts(l.openCell.p, l.nOpen, 4, openOf.p, wm, cand, t, fl, s.stream);
        launch_open_conflicts(l.perIndex.p, l.nPeriodic, 0, openOf.p, wm, cand, t, fl, s.stream);
        launch_open_conflicts(l.perSource.p, l.nPeriodic, 0, openOf.p, wm, cand, t, fl, s.stream);
        launch_open_conflicts(l.F2C.index.p, l.F2C.interfaceCount, 0, openOf.p, wm, cand, t, fl, s.stream);
        launch_open_conflicts(l.C2F.index.p, l.C2F.interfaceCount, 2, openOf.p, wm, cand, t, fl, s.stream);
        launch_open_conflicts(l.C2F.leftoverParent.p, l.C2F.leftoverCount, 0, openOf.p, wm, cand, t, fl, s.stream);
        launch_open_conflicts(l.C2F.leftoverNbrI.p, l.C2F.leftoverCount, 1, openOf.p, wm, cand, t, fl, s.stream);
        launch_open_conflicts(l.C2F.leftoverNbrJ.p, l.C2F.leftoverCount, 1, openOf.p, wm, cand, t, fl, s.stream);
        launch_open_conflicts(l.C2F.leftoverNbrK.p, l.C2F.leftoverCount, 1, openOf.p, wm, cand, t, fl, s.stream);
        int conflicts = 0;
        HIPCHK(hipMemcpyAsync(&conflicts, flag.p, sizeof(int), hipMemcpyDeviceToHost, s.stream));
        HIPCHK(hipStreamSynchronize(s.stream));
        // the open-cell kernel uses 32-bit buffer offsets
        fuse = conflicts == 0 && !wide_of(s, l);
    }
    l.nFusedEntries = l.nSepEntries = 0;
    l.fusedEntries.release();
    l.sepEntries.release();
    if (fuse && tune.openSplit == 1) {
        // cells on the x faces (one per row end: every access of theirs is a
        // line of its own) leave the open-cell kernel: the bulk kernel steps
        // them and a pass after streaming completes them
        std::vector<uint32_t> meta((size_t)l.nOpen);
        HIPCHK(hipMemcpyAsync(meta.data(), l.openMeta.p, sizeof(uint32_t) * meta.size(), hipMemcpyDeviceToHost, s.stream));
        HIPCHK(hipStreamSynchronize(s.stream));
        std::vector<int> fusedList, sepList;
        for (int x = 0; x < l.nOpen; ++x)
            (LBM3_BT_NORMAL[meta[(size_t)x] & 31u][0] != 0 ? sepList : fusedList).push_back(x);
        if (!sepList.empty()) {
            if (upload(l.fusedEntries, fusedList.data(), (long long)fusedList.size(), s.stream) ||
                upload(l.sepEntries, sepList.data(), (long long)sepList.size(), s.stream))
                return LBM3_E_HIP;
            l.nFusedEntries = (int)fusedList.size();
            l.nSepEntries = (int)sepList.size();
            HIPCHK(hipMemsetAsync(openOf.p, 0xFF, sizeof(int) * (size_t)l.N, s.stream));
            launch_scatter_entries(l.openCell.p, l.fusedEntries.p, l.nFusedEntries, openOf.p, s.stream);
        }
    }
    launch_fast_topo(topo_of(l), l.nRows, l.wallMap.p, fuse ? openOf.p : nullptr, cand, l.cellRow.p, l.rowTab.p, s.stream);
    HIPCHK(hipGetLastError());
    l.nOpenGroups = 0;
    // the rotor cells in the bulk kernel (the kernel takes open cells or rotor
    // cells, not both: open cells then stay in groups)
    l.rotorInBulk = cand && tune.rotorInBulk && !wide_of(s, l);
    int G = tune.openGroup ? tune.openGroup : open_group_cells((int)storage_bytes(s.storage));
    if (G == 1 && l.rotorInBulk) G = open_group_cells((int)storage_bytes(s.storage));
    l.openInBulk = fuse && G == 1;   // the bulk kernel completes and steps the open cells
    l.laneRot = l.openInBulk && tune.openSplit == 3;
    // the bulk kernel's open cells but those on the x faces, which stay in
    // groups of the open-cell kernel (one x-face cell per row end would hold a
    // bulk wave for one lane; eight in a group share one wave's condition code)
    const bool xGroups = l.openInBulk && tune.openSplit == 2;
    if (xGroups) G = open_group_cells((int)storage_bytes(s.storage));
    l.openGroupCells = G;
    if (fuse && (!l.openInBulk || xGroups)) {
        // aligned groups of cells holding open cells, sorted by the boundary
        // condition (normal and record) of their first open cell, then by group
        std::vector<int> cell((size_t)l.nOpen);
        std::vector<uint32_t> meta((size_t)l.nOpen);
        HIPCHK(hipMemcpyAsync(cell.data(), l.openCell.p, sizeof(int) * cell.size(), hipMemcpyDeviceToHost, s.stream));
        HIPCHK(hipMemcpyAsync(meta.data(), l.openMeta.p, sizeof(uint32_t) * meta.size(), hipMemcpyDeviceToHost, s.stream));
        HIPCHK(hipStreamSynchronize(s.stream));
        std::vector<char> inKernel((size_t)l.nOpen, 1);   // entries the open-cell kernel completes
        if (l.nSepEntries) {
            std::vector<int> sep((size_t)l.nSepEntries);
            HIPCHK(hipMemcpy(sep.data(), l.sepEntries.p, sizeof(int) * sep.size(), hipMemcpyDeviceToHost));
            for (int x : sep) inKernel[(size_t)x] = 0;
        }
        if (xGroups)
            for (int x = 0; x < l.nOpen; ++x) inKernel[(size_t)x] = LBM3_BT_NORMAL[meta[(size_t)x] & 31u][0] != 0;
        std::vector<std::pair<int, int>> first((size_t)(l.N / G + 1), {-1, 0});   // {first open cell, key}
        for (int x = 0; x < l.nOpen; ++x) {
            if (!inKernel[(size_t)x]) continue;
            const int g = cell[(size_t)x] / G;
            if (first[(size_t)g].first < 0 || cell[(size_t)x] < first[(size_t)g].first)
                first[(size_t)g] = {cell[(size_t)x], int(meta[(size_t)x] & ~kOpenTrackBit)};
        }
        std::vector<std::pair<int, int>> order;
        for (size_t g = 0; g < first.size(); ++g)
            if (first[g].first >= 0) order.push_back({first[g].second, (int)g});
        std::sort(order.begin(), order.end());
        std::vector<int> groups;
        for (const auto &o : order) groups.push_back(o.second);
        l.nOpenGroups = (int)groups.size();
        if (upload(l.openGroups, groups.data(), (long long)groups.size(), s.stream)) return LBM3_E_HIP;
        launch_mark_groups(l.openGroups.p, l.nOpenGroups, G, l.N, l.cellRow.p, s.stream);
        HIPCHK(hipGetLastError());
    }
    if (cand && !l.rotorInBulk) {
        // the cells with record -4, in cell order (coalesced rows)
        std::vector<int2> rec((size_t)l.N);
        HIPCHK(hipMemcpyAsync(rec.data(), l.cellRow.p, sizeof(int2) * rec.size(), hipMemcpyDeviceToHost, s.stream));
        HIPCHK(hipStreamSynchronize(s.stream));
        std::vector<int> cells;
        for (int c = 0; c < l.N; ++c)
            if (rec[(size_t)c].x == -4) cells.push_back(c);
        l.rotorCellCount = (int)cells.size();
        if (upload(l.rotorCells, cells.data(), (long long)cells.size(), s.stream)) return LBM3_E_HIP;
    }
    if (const int rc = refresh_bulk_mask(s, l)) return rc;
    if (xGroups) {
        // the grouped cells leave the bulk kernel: skip bits set, open bits clear
        launch_group_bits(l.openGroups.p, l.nOpenGroups, G, l.bulkSkip.p, l.openBits.p, s.stream);
        HIPCHK(hipGetLastError());
    }
    HIPCHK(hipStreamSynchronize(s.stream));
    l.fusedOpen = fuse;
    return prepare_images(s, l);
}

// rotor descriptors of a level to the device; the cell records follow at the next run
int upload_rotors(Sim &s, int level)
{
    Level &l = s.L[level];
    std::vector<RotorDev> h;
    for (const Level::Rotor &r : l.rotors) h.push_back(r.dev);
    if (h.empty()) l.rotorDev.release();
    else if (upload(l.rotorDev, h.data(), (long long)h.size(), s.stream)) return LBM3_E_HIP;
    HIPCHK(hipStreamSynchronize(s.stream));
    l.openFusionChecked = false;
    return 0;
}

// apply a pending open boundary condition in place (before anything reads the level's state)
template <class S> static void settle_typed(Sim &s, Level &l)
{
    OpenArgs<S> o = open_args<S>(s, l, l.info.iterationsFinished - 1);
    if (l.fusedOpen && l.nSepEntries) {   // the x-face entries completed in their own step
        o.list = l.fusedEntries.p;
        o.count = l.nFusedEntries;
    }
    launch_open<S>(o, l.info.esotwistFlipper != 0, s.stream);
}

template <class S> static void periodic_typed(Sim &s, Level &l, bool flip)
{
    launch_periodic<S>(reinterpret_cast<S *>(l.f.p), topo_of(l), l.nPeriodic, l.perIndex.p, l.perSource.p, flip, s.stream);
}

// the periodic copy of ghosts that were stepped from their source cells
static int settle_ghosts(Sim &s, Level &l)
{
    if (!l.ghostsStale) return 0;
    l.ghostsStale = false;
    const bool flip = l.info.esotwistFlipper != 0;
    switch (s.storage) {
    case LBM3_STORE_F16: periodic_typed<__half>(s, l, flip); break;
    case LBM3_STORE_BF16: periodic_typed<__hip_bfloat16>(s, l, flip); break;
    case LBM3_STORE_F16C: periodic_typed<f16c>(s, l, flip); break;
    case LBM3_STORE_F64: periodic_typed<double>(s, l, flip); break;
    default: periodic_typed<float>(s, l, flip); break;
    }
    return check_hip(hipGetLastError(), "periodic ghost copy");
}

// The end of every call that steps: a caller who holds a level's populations
// (lbm3_device_array) finds the ghosts copied, as after every step before the
// bulk kernel stepped them, and the next step takes what that caller wrote there.
static int settle_shared(Sim &s)
{
    for (int L = 0; L < s.levels; ++L)
        if (s.L[L].shared)
            if (const int rc = settle_ghosts(s, s.L[L])) return rc;
    return 0;
}

// A condition is pending after a fused step and after a checkpoint load that
// saved one; it is applied here whether or not the level currently fuses.
// Ghosts that lag behind their sources are copied too: what follows reads the
// level's whole state.
static int settle_open(Sim &s, int L)
{
    Level &l = s.L[L];
    if (const int rc = settle_ghosts(s, l)) return rc;
    if (l.openSettled || l.nOpen == 0) {
        l.openSettled = true;
        return 0;
    }
    switch (s.storage) {
    case LBM3_STORE_F16: settle_typed<__half>(s, l); break;
    case LBM3_STORE_BF16: settle_typed<__hip_bfloat16>(s, l); break;
    case LBM3_STORE_F16C: settle_typed<f16c>(s, l); break;
    case LBM3_STORE_F64: settle_typed<double>(s, l); break;
    default: settle_typed<float>(s, l); break;
    }
    l.openSettled = true;
    return check_hip(hipGetLastError(), "open boundary settle");
}

template <class S> static void step_level(Sim &s, int level)
{
    Level &l = s.L[level];
    const int overlap = tune_of(s, l).overlap;
    const bool flip = l.info.esotwistFlipper != 0;
    const bool timed = s.timing && level == 0;
    if (timed) {
        if (s.evUsed >= (int)s.ev.size()) {
            std::array<hipEvent_t, 3> e{};
            for (auto &x : e) (void)hipEventCreate(&x);
            s.ev.push_back(e);
        }
        (void)hipEventRecord(s.ev[s.evUsed][0], s.stream);
    }
    StepArgs<S> a = step_args<S>(s, l);
    if (!l.rotors.empty()) {
        // advance the rotors (updateGrid.h:36-49); the frame's cosine and sine of
        // this step once per rotor, in the compute type
        using T = typename StoreTraits<S>::compute;
        constexpr double twoPi = 6.283185307179586476925286766559;
        for (size_t r = 0; r < l.rotors.size(); ++r) {
            Level::Rotor &Rt = l.rotors[r];
            Rt.radiansElapsed = std::fmod(Rt.radiansElapsed + (double)l.info.dtPhys * (double)Rt.dev.radiansPerSecond, twoPi);
            if (Rt.radiansElapsed < 0.0) Rt.radiansElapsed += twoPi;
            if (Rt.radiansElapsed >= twoPi) Rt.radiansElapsed = 0.0;
            if (sizeof(T) == sizeof(double)) {
                a.rotorCS[2 * r] = std::cos(Rt.radiansElapsed);
                a.rotorCS[2 * r + 1] = std::sin(Rt.radiansElapsed);
            } else {
                a.rotorCS[2 * r] = (double)std::cos((float)Rt.radiansElapsed);
                a.rotorCS[2 * r + 1] = (double)std::sin((float)Rt.radiansElapsed);
            }
        }
        a.rotors = l.rotorDev.p;
        a.nRotors = (int)l.rotors.size();
        a.trackRotor = s.C.trackRotorForce;
        a.rotorCells = l.rotorCells.p;
        a.rotorCellCount = l.rotorCellCount;
    }
    if (l.fusedOpen) {
        // open cells have their own kernel, which first applies the previous
        // step's boundary condition when it is still pending
        const OpenArgs<S> o = open_args<S>(s, l, l.info.iterationsFinished - 1);
        a.open = {l.openGroups.p, l.nOpenGroups, l.openSettled ? 0 : 1, o.meta, o.records, o.dRhoRef, o.uNormalRef, o.dRhoCum,
                  o.uNormalCum, o.iterationsFinished, o.scale, l.openGroupCells};
    }
    // the values a replayed graph reads from device memory instead
    StepParam prm{};
    prm.iter = l.info.iterationsFinished - 1;
    prm.iterNow = l.info.iterationsFinished;
    prm.pending = l.fusedOpen && !l.openSettled ? 1 : 0;
    for (int r = 0; r < 2 * LBM3_MAX_ROTORS; ++r) prm.cs[r] = a.rotorCS[r];
    if (s.dryRun) {
        // bookkeeping only: the state a launch would leave
        s.dryRun->push_back(prm);
        l.info.esotwistFlipper = flip ? 0 : 1;
        if (l.fusedOpen) l.openSettled = false;
        l.info.iterationsSinceTrackerReset++;
        l.info.iterationsFinished++;
        return;
    }
    const StepParam *slot = s.captureTable ? s.captureTable + s.captureSlot++ : nullptr;
    a.param = slot;
    // The step after an initialisation, an upload or a read of the whole state
    // takes the ghosts as they are: a caller may have written them.  A captured
    // step keeps the copy, so that every replay is the same.
    const bool images = l.imagesReady && !slot;
    if (images && l.ghostsStale) a.fast.images = images_of(l);
    // side-stream choice 3: the wall-adjacent cells in blocks ahead of the bulk
    // blocks of one launch (not with rotated lanes or 64-bit offsets)
    const bool walls = overlap == 3 && l.W > 0 && !a.laneRot && !wide_level<S>(l.N);
    a.wallBlocks = walls ? (int)((l.W + 255) / 256) : 0;
    if (timed || !overlap || ((l.W == 0 || walls) && a.open.count == 0 && a.rotorCellCount == 0)) {
        // in order on one stream, so that each kernel's events bracket it alone
        launch_collide_stream<S>(a, flip, s.stream);
        if (timed) (void)hipEventRecord(s.ev[s.evUsed][1], s.stream);
        if (!walls) launch_collide_wall<S>(a, flip, s.stream);
        launch_open_cells<S>(a, flip, s.stream);
        launch_rotor_cells<S>(a, flip, s.stream);
        if (timed) {
            (void)hipEventRecord(s.ev[s.evUsed][2], s.stream);
            s.evUsed++;
        }
    } else {
        // the kernels touch disjoint cells: run the small, latency-bound wall and
        // open-cell kernels on the second stream beside the bulk kernel, the
        // rotor cells (often the larger part of a rotor's level) on a third
        (void)hipEventRecord(s.fork, s.stream);
        (void)hipStreamWaitEvent(s.aux, s.fork, 0);
        const bool third = a.rotorCellCount > 0 && s.aux2;
        if (third) {
            (void)hipStreamWaitEvent(s.aux2, s.fork, 0);
            launch_rotor_cells<S>(a, flip, s.aux2);
            (void)hipEventRecord(s.join2, s.aux2);
        }
        if (!walls) launch_collide_wall<S>(a, flip, s.aux);
        launch_open_cells<S>(a, flip, s.aux);
        if (!third) launch_rotor_cells<S>(a, flip, s.aux);
        (void)hipEventRecord(s.join, s.aux);
        launch_collide_stream<S>(a, flip, s.stream);
        (void)hipStreamWaitEvent(s.stream, s.join, 0);
        if (third) (void)hipStreamWaitEvent(s.stream, s.join2, 0);
    }
    const bool nflip = !flip;
    l.info.esotwistFlipper = nflip ? 1 : 0;
    if (l.fusedOpen) {
        l.openSettled = false;   // this step's boundary condition is applied by the next step's open-cell kernel
        if (l.nSepEntries) {     // except on the x faces: completed now
            OpenArgs<S> o = open_args<S>(s, l, l.info.iterationsFinished);
            o.param = slot;
            o.list = l.sepEntries.p;
            o.count = l.nSepEntries;
            launch_open<S>(o, nflip, s.stream);
        }
    } else {
        OpenArgs<S> o = open_args<S>(s, l, l.info.iterationsFinished);
        o.param = slot;
        launch_open<S>(o, nflip, s.stream);
    }
    if (images) l.ghostsStale = true;
    else periodic_typed<S>(s, l, nflip);
    l.info.iterationsSinceTrackerReset++;
    l.info.iterationsFinished++;
}

static void step_level_any(Sim &s, int level)
{
    switch (s.storage) {
    case LBM3_STORE_F16: step_level<__half>(s, level); break;
    case LBM3_STORE_BF16: step_level<__hip_bfloat16>(s, level); break;
    case LBM3_STORE_F16C: step_level<f16c>(s, level); break;
    case LBM3_STORE_F64: step_level<double>(s, level); break;
    default: step_level<float>(s, level); break;
    }
}

void update_interface(Sim &s, int coarse);    // interface.hip

// updateAllGrids (updateGrid.h:388-397): the level's step, two sub-steps of
// every finer level, the interface transfer.  With Sim::Tune::overlap 2 the
// finer levels run on their own stream beside this level's step: they depend
// on this stream's earlier work (the last transfer), and the transfer waits
// for them.  s.stream is the current level's stream throughout.
static void update_all(Sim &s, int level)
{
    const bool fork = !s.dryRun && tune_of(s, s.L[level]).levelStreams() && level + 1 < s.levels && s.levelStream[level + 1];
    const hipStream_t own = s.stream;
    if (fork) {
        (void)hipEventRecord(s.levelFork[level + 1], own);
        (void)hipStreamWaitEvent(s.levelStream[level + 1], s.levelFork[level + 1], 0);
    }
    step_level_any(s, level);
    if (level < s.levels - 1) {
        if (fork) s.stream = s.levelStream[level + 1];
        for (int i = 0; i < 2; ++i) update_all(s, level + 1);
        if (fork) {
            (void)hipEventRecord(s.levelJoin[level + 1], s.stream);
            s.stream = own;
            (void)hipStreamWaitEvent(own, s.levelJoin[level + 1], 0);
        }
        if (!s.dryRun) update_interface(s, level);
    }
}

template <class S> static int init_level(Sim &s, int level, const float *fieldsDev)
{
    Level &l = s.L[level];
    InitDesc d{};
    d.kind = fieldsDev ? 2 : s.C.init.kind;
    d.dRho = s.C.init.dRho; d.ux = s.C.init.ux; d.uy = s.C.init.uy; d.uz = s.C.init.uz;
    d.u0 = s.C.init.u0; d.length = s.C.init.length; d.pressure = s.C.init.pressure;
    d.profile = s.C.init.profile;
    d.fields = fieldsDev;
    const bool flip = l.info.esotwistFlipper != 0;
    l.openSettled = true;
    l.ghostsStale = false;
    launch_init<S>(reinterpret_cast<S *>(l.f.p), topo_of(l), d, l.geom, s.codec, flip, s.stream);
    launch_open_ref_init<S>(open_args<S>(s, l, l.info.iterationsFinished), l.info.cellCountX, l.info.cellCountY, l.info.cellCountZ, flip, s.stream);
    return check_hip(hipGetLastError(), "init kernels");
}

static int init_level_any(Sim &s, int level, const float *fieldsDev)
{
    DBuf<float> hooked;
    if (!fieldsDev && s.hooks.initial_condition) {
        if (const int rc = hook_initial_fields(s, level, hooked)) return rc;
        fieldsDev = hooked.p;
    }
    switch (s.storage) {
    case LBM3_STORE_F16: return init_level<__half>(s, level, fieldsDev);
    case LBM3_STORE_BF16: return init_level<__hip_bfloat16>(s, level, fieldsDev);
    case LBM3_STORE_F16C: return init_level<f16c>(s, level, fieldsDev);
    case LBM3_STORE_F64: return init_level<double>(s, level, fieldsDev);
    default: return init_level<float>(s, level, fieldsDev);
    }
}

static int check_level(Sim &s, int level)
{
    if (level < 0 || level >= s.levels || !s.L[level].built) return set_error(LBM3_E_STATE, "level not built");
    return 0;
}

// every level a sub-cycled update touches is built, and every interface it runs is checked
static int prepare_open_fusion(Sim &s, int L);

int prepare_interface(Sim &s, int coarse);    // interface.hip: neighbour tables of the transfer lists

static int check_run(Sim &s, int from)
{
    for (int L = from; L < s.levels; ++L) {
        if (const int rc = check_level(s, L)) return rc;
        if (L + 1 < s.levels && !s.L[L].interfaceChecked)
            return set_error(LBM3_E_STATE, "interface lists of a level are not checked against the finer level");
    }
    for (int L = from; L < s.levels; ++L)
        if (!s.L[L].openFusionChecked)
            if (const int rc = prepare_open_fusion(s, L)) return rc;
    for (int L = from; L + 1 < s.levels; ++L)
        if (const int rc = prepare_interface(s, L)) return rc;
    return 0;
}

template <class T> int collide_cells(T *f, int n, const lbm3_bc *bc, T nu)
{
    if (!f || !bc || n < 0) return set_error(LBM3_E_ARG, "bad collide arguments");
    DBuf<T> d;
    HIPCHK(d.alloc(27LL * n));
    HIPCHK(hipMemcpy(d.p, f, sizeof(T) * 27 * (size_t)n, hipMemcpyHostToDevice));
    const Relax<T> R = make_relax<T>(nu, T(bc->nuMultiplier), T(bc->collisionLimiter), T(bc->gx), T(bc->gy), T(bc->gz));
    launch_collide_batch<T>(d.p, n, R, nullptr);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpy(f, d.p, sizeof(T) * 27 * (size_t)n, hipMemcpyDeviceToHost));
    return 0;
}

} // namespace lbm3

using namespace lbm3;

// one level's cells on a section plane into the image
template <class S> static void cut_level(Sim &s, int L, const CutLevel &d, float *img)
{
    Level &l = s.L[L];
    launch_section_cut<S>(reinterpret_cast<const S *>(l.f.p), topo_of(l), l.wallMap.p, s.codec, l.info.esotwistFlipper != 0,
                          d, img, s.stream);
}

// checkpoint file: magic, {version, storage, levels}, fluid updates, then per
// level a CheckpointLevel, the level's lbm3_info, the buffers checkpoint_buffers
// names (raw device bytes) and each rotor's angle
static const char kCheckpointMagic[8] = {'L', 'B', 'M', '3', 'C', 'K', 'P', 'T'};
static constexpr int kCheckpointVersion = 1;
struct CheckpointLevel {
    long long N, W, nOpen, nRotors;
    int openSettled;
    int split;          // a pending condition covers the open-cell kernel's entries only (x faces completed)
};

static CheckpointLevel checkpoint_level(const Level &l)
{
    return {l.N, l.W, l.nOpen, (long long)l.rotors.size(), l.openSettled ? 1 : 0, l.fusedOpen && l.nSepEntries ? 1 : 0};
}

// the device state a time step changes: populations, open-boundary reference
// states and statistics, wall and rotor force accumulators
static std::vector<std::pair<void *, size_t>> checkpoint_buffers(Level &l, int storage)
{
    std::vector<std::pair<void *, size_t>> b;
    b.push_back({l.f.p, (size_t)l.f.n});
    b.push_back({l.openRefs.p, 2 * (size_t)l.nOpen * compute_bytes(storage)});
    b.push_back({l.openCum.p, sizeof(double) * 2 * (size_t)l.nOpen});
    b.push_back({l.gWall.p, sizeof(double) * (size_t)l.gWall.n});
    for (auto &r : l.rotors) b.push_back({r.g.p, sizeof(double) * (size_t)r.g.n});
    return b;
}

static constexpr size_t kStageBytes = size_t(64) << 20;

static int dump_device(FILE *fp, const void *dev, size_t bytes, std::vector<unsigned char> &stage, hipStream_t st, bool &ok)
{
    stage.resize(std::min(bytes, kStageBytes));
    for (size_t o = 0; ok && o < bytes; o += kStageBytes) {
        const size_t n = std::min(kStageBytes, bytes - o);
        HIPCHK(hipMemcpyAsync(stage.data(), static_cast<const unsigned char *>(dev) + o, n, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        ok = fwrite(stage.data(), 1, n, fp) == n;
    }
    return 0;
}

static int load_device(FILE *fp, void *dev, size_t bytes, std::vector<unsigned char> &stage, hipStream_t st, bool &ok)
{
    stage.resize(std::min(bytes, kStageBytes));
    for (size_t o = 0; ok && o < bytes; o += kStageBytes) {
        const size_t n = std::min(kStageBytes, bytes - o);
        ok = fread(stage.data(), 1, n, fp) == n;
        if (!ok) break;
        HIPCHK(hipMemcpyAsync(static_cast<unsigned char *>(dev) + o, stage.data(), n, hipMemcpyHostToDevice, st));
        HIPCHK(hipStreamSynchronize(st));
    }
    return 0;
}

extern "C" {

const char *lbm3_last_error(void) { return g_error.c_str(); }

int lbm3_device_info(char *name, int nameLen, long long *hbmBytes, int *cuCount)
{
    hipDeviceProp_t p;
    HIPCHK(hipGetDeviceProperties(&p, 0));
    if (name && nameLen > 0) snprintf(name, (size_t)nameLen, "%s %s", p.name, p.gcnArchName);
    if (hbmBytes) *hbmBytes = (long long)p.totalGlobalMem;
    if (cuCount) *cuCount = p.multiProcessorCount;
    return 0;
}

int lbm3_sim_create(const lbm3_case *c, int storage, lbm3_sim **out)
{
    if (!c || !out) return set_error(LBM3_E_ARG, "null argument");
    if (c->gridLevelCount < 1 || c->gridLevelCount > LBM3_MAX_LEVELS) return set_error(LBM3_E_ARG, "gridLevelCount out of range");
    if (storage < LBM3_STORE_F32 || storage > LBM3_STORE_F16C) return set_error(LBM3_E_ARG, "unknown storage");
    lbm3_sim *h = new (std::nothrow) lbm3_sim();
    if (!h) return set_error(LBM3_E_MEMORY, "host allocation");
    h->s.C = *c;
    h->s.storage = storage;
    h->s.levels = c->gridLevelCount;
    h->s.codec = make_codec(*c, storage);
    int rc = check_hip(hipStreamCreateWithFlags(&h->s.stream, hipStreamNonBlocking), "stream");
    if (!rc) rc = check_hip(hipStreamCreateWithFlags(&h->s.aux, hipStreamNonBlocking), "stream");
    if (!rc) rc = check_hip(hipEventCreateWithFlags(&h->s.fork, hipEventDisableTiming), "event");
    if (!rc) rc = check_hip(hipEventCreateWithFlags(&h->s.join, hipEventDisableTiming), "event");
    if (!rc) rc = check_hip(hipStreamCreateWithFlags(&h->s.aux2, hipStreamNonBlocking), "stream");
    if (!rc) rc = check_hip(hipEventCreateWithFlags(&h->s.join2, hipEventDisableTiming), "event");
    for (int L = 1; L < h->s.levels && !rc; ++L) {
        rc = check_hip(hipStreamCreateWithFlags(&h->s.levelStream[L], hipStreamNonBlocking), "stream");
        if (!rc) rc = check_hip(hipEventCreateWithFlags(&h->s.levelFork[L], hipEventDisableTiming), "event");
        if (!rc) rc = check_hip(hipEventCreateWithFlags(&h->s.levelJoin[L], hipEventDisableTiming), "event");
    }
    if (rc) {
        for (int L = 1; L < LBM3_MAX_LEVELS; ++L) {
            if (h->s.levelJoin[L]) (void)hipEventDestroy(h->s.levelJoin[L]);
            if (h->s.levelFork[L]) (void)hipEventDestroy(h->s.levelFork[L]);
            if (h->s.levelStream[L]) (void)hipStreamDestroy(h->s.levelStream[L]);
        }
        if (h->s.join2) (void)hipEventDestroy(h->s.join2);
        if (h->s.aux2) (void)hipStreamDestroy(h->s.aux2);
        if (h->s.join) (void)hipEventDestroy(h->s.join);
        if (h->s.fork) (void)hipEventDestroy(h->s.fork);
        if (h->s.aux) (void)hipStreamDestroy(h->s.aux);
        if (h->s.stream) (void)hipStreamDestroy(h->s.stream);
        delete h;
        return rc;
    }
    *out = h;
    return 0;
}

int lbm3_sim_destroy(lbm3_sim *h)
{
    if (!h) return 0;
    (void)hipStreamSynchronize(h->s.stream);
    (void)hipStreamSynchronize(h->s.aux);
    (void)hipStreamSynchronize(h->s.aux2);
    (void)hipEventDestroy(h->s.join2);
    (void)hipStreamDestroy(h->s.aux2);
    for (int L = 1; L < LBM3_MAX_LEVELS; ++L) {
        if (h->s.levelStream[L]) {
            (void)hipStreamSynchronize(h->s.levelStream[L]);
            (void)hipStreamDestroy(h->s.levelStream[L]);
        }
        if (h->s.levelFork[L]) (void)hipEventDestroy(h->s.levelFork[L]);
        if (h->s.levelJoin[L]) (void)hipEventDestroy(h->s.levelJoin[L]);
    }
    for (auto &e3 : h->s.ev)
        for (auto e : e3) (void)hipEventDestroy(e);
    (void)hipEventDestroy(h->s.fork);
    (void)hipEventDestroy(h->s.join);
    (void)hipStreamDestroy(h->s.aux);
    (void)hipStreamDestroy(h->s.stream);
    delete h;
    return 0;
}

// every index the kernels follow must stay inside its array: checked on the
// host before anything reaches the device
static int validate_level(const lbm3_level_arrays &a)
{
    const long long N = a.info.cellCount, R = a.nRows, W = a.W;
    auto bad = [](const char *what) { return set_error(LBM3_E_ARG, std::string("import: ") + what); };
    if (N <= 0 || R <= 0 || W < 0 || a.nOpenIDs < 0 || a.nPeriodic < 0) return bad("negative or empty sizes");
    if (!a.shifter || !a.rowI || !a.rowJ || !a.rowK || !a.rowJPlus || !a.rowKPlus || !a.rowJKPlus || !a.wallMap)
        return bad("missing topology array");
    if (W > 0 && (!a.wallIndex || !a.wallData || !a.linkLength)) return bad("missing wall arrays");
    if (a.nOpenIDs > 0 && !a.openCount) return bad("missing open-boundary counts");
    if (a.nPeriodic > 0 && (!a.periodicIndex || !a.periodicSource)) return bad("missing periodic arrays");
    // rows are numbered in the order of their first cells (the bulk kernel relies
    // on it) and hold consecutive cells: a cell with a negative shifter is at that
    // offset from the last row head before it (gridBuilderFunctions.h:1107-1125)
    long long nextRow = 0, head = -1;
    std::vector<long long> rowLen((size_t)R, 0);
    for (long long c = 0; c < N; ++c) {
        const int sh = a.shifter[c];
        if (sh >= 0) {
            if (sh >= R) return bad("shifter row out of range");
            if (sh != nextRow) return bad("rows not numbered in the order of their first cells");
            ++nextRow;
            head = c;
        } else if (head < 0 || c + sh != head) {
            return bad("shifter offset does not reach its row head");
        }
        ++rowLen[(size_t)a.shifter[head]];
        const int wm = a.wallMap[c];
        if (wm < -3 || wm >= W) return bad("wallMap out of range");
    }
    if (nextRow != R) return bad("a row without a first cell");
    // the decode adds a cell's offset in its row to the neighbour rows' first
    // cells (cellFunctions.h:41-46): every cell of the row must land inside the level
    for (long long r = 0; r < R; ++r) {
        const long long last = rowLen[(size_t)r] - 1;
        if (a.rowJPlus[r] < 0 || a.rowJPlus[r] + last >= N || a.rowKPlus[r] < 0 || a.rowKPlus[r] + last >= N ||
            a.rowJKPlus[r] < 0 || a.rowJKPlus[r] + last >= N)
            return bad("row neighbour out of range");
    }
    for (long long w = 0; w < W; ++w)
        if (a.wallIndex[w] < 0 || a.wallIndex[w] >= N || a.wallMap[a.wallIndex[w]] != w) return bad("wallIndex inconsistent with wallMap");
    long long nOpen = 0;
    for (int b = 0; b < a.nOpenIDs; ++b) {
        if (a.openCount[b] < 0) return bad("negative open count");
        nOpen += a.openCount[b];
    }
    if (nOpen > 0 && (!a.openIndex || !a.openSource)) return bad("missing open-boundary cell lists");
    for (long long x = 0; x < nOpen; ++x)
        if (a.openIndex[x] < 0 || a.openIndex[x] >= N || a.openSource[x] < 0 || a.openSource[x] >= N) return bad("open cell out of range");
    for (long long x = 0; x < a.nPeriodic; ++x)
        if (a.periodicIndex[x] < 0 || a.periodicIndex[x] >= N || a.periodicSource[x] < 0 || a.periodicSource[x] >= N)
            return bad("periodic cell out of range");
    if (a.f2cCount < 0 || a.c2fCount < 0 || a.leftoverCount < 0) return bad("negative interface count");
    if ((a.f2cCount && (!a.f2cIndex || !a.f2cChild)) || (a.c2fCount && (!a.c2fIndex || !a.c2fChild)) ||
        (a.leftoverCount && (!a.leftoverIndex || !a.leftoverParent || !a.leftoverNbrI || !a.leftoverNbrJ || !a.leftoverNbrK)))
        return bad("missing interface arrays");
    for (long long x = 0; x < a.f2cCount; ++x)
        if (a.f2cIndex[x] < 0 || a.f2cIndex[x] >= N) return bad("F->C cell out of range");
    for (long long x = 0; x < a.c2fCount; ++x)
        if (a.c2fIndex[x] < 0 || a.c2fIndex[x] >= N) return bad("C->F cell out of range");
    auto signedCell = [N](int c) { const long long v = c < 0 ? -(long long)c - 1 : c; return v >= 0 && v < N; };
    for (long long x = 0; x < a.leftoverCount; ++x)
        if (a.leftoverParent[x] < 0 || a.leftoverParent[x] >= N || !signedCell(a.leftoverNbrI[x]) ||
            !signedCell(a.leftoverNbrJ[x]) || !signedCell(a.leftoverNbrK[x]))
            return bad("leftover cell out of range");
    return 0;
}

int lbm3_validate_level(const lbm3_level_arrays *a)
{
    if (!a) return set_error(LBM3_E_ARG, "null argument");
    return validate_level(*a);
}

// fine-level cells named by a coarse level's interface lists must exist
static int check_fine_refs(Level &coarse, long long nFine)
{
    for (const int c : coarse.fineRefs)
        if (c < 0 || c >= nFine) return set_error(LBM3_E_ARG, "import: interface list names a fine cell out of range");
    coarse.interfaceChecked = true;
    return 0;
}

int lbm3_import_level(lbm3_sim *h, int level, const lbm3_level_arrays *a)
{
    if (!h || !a || level < 0 || level >= h->s.levels) return set_error(LBM3_E_ARG, "bad import arguments");
    Sim &s = h->s;
    Level &l = s.L[level];
    hipStream_t st = s.stream;
    if (const int rc = validate_level(*a)) return rc;
    if (s.hooks.open_bc || s.hooks.local_bc)
        return set_error(LBM3_E_STATE, "imported levels take the case's rule tables, not hook callbacks");
    l.openBC.clear();                 // records of the rule table
    l.info = a->info;
    l.N = a->info.cellCount;
    l.nRows = a->nRows;
    l.W = a->W;
    l.wallCount = a->wallCount;
    if (upload(l.shifter, a->shifter, l.N, st) || upload(l.ri, a->rowI, l.nRows, st) || upload(l.rj, a->rowJ, l.nRows, st) ||
        upload(l.rk, a->rowK, l.nRows, st) || upload(l.rjp, a->rowJPlus, l.nRows, st) || upload(l.rkp, a->rowKPlus, l.nRows, st) ||
        upload(l.rjkp, a->rowJKPlus, l.nRows, st) || upload(l.wallMap, a->wallMap, l.N, st) ||
        upload(l.wallIndex, a->wallIndex, l.W, st) || upload(l.wallData, a->wallData, l.W, st) ||
        upload(l.linkLength, a->linkLength, 7LL * l.W, st))
        return LBM3_E_HIP;
    // open boundary: concatenate BCIDs, derive normal index and rule per cell on the host
    l.nOpenIDs = a->nOpenIDs;
    l.openCount.assign(a->openCount, a->openCount + a->nOpenIDs);
    l.nOpen = 0;
    for (int b = 0; b < a->nOpenIDs; ++b) l.nOpen += a->openCount[b];
    std::vector<uint32_t> meta(l.nOpen);
    for (int x = 0; x < l.nOpen; ++x) {
        const int cell = a->openIndex[x];
        const int shift = a->shifter[cell];
        const int row = shift >= 0 ? shift : a->shifter[cell + shift];
        const int back = shift >= 0 ? 0 : -shift;
        const int i = a->rowI[row] + back, j = a->rowJ[row], k = a->rowK[row];
        const lbm3_info &I = a->info;
        const int nx = i == 0 ? -1 : (i == I.cellCountX - 1 ? 1 : 0);
        const int ny = j == 0 ? -1 : (j == I.cellCountY - 1 ? 1 : 0);
        const int nz = k == 0 ? -1 : (k == I.cellCountZ - 1 ? 1 : 0);
        const int rule = open_rule(s.C, level, I.cellCountX, I.cellCountY, I.cellCountZ, i, j, k);
        const int wm = a->wallMap[cell];
        bool track = wm != -2;
        if (wm >= 0 && (a->wallData[wm] & 1u)) track = false;
        meta[x] = open_meta(normal_index(nx, ny, nz), rule, track);
    }
    if (upload(l.openCell, a->openIndex, l.nOpen, st) || upload(l.openSource, a->openSource, l.nOpen, st) ||
        upload(l.openMeta, meta.data(), l.nOpen, st))
        return LBM3_E_HIP;
    l.nPeriodic = a->nPeriodic;
    if (upload(l.perIndex, a->periodicIndex, l.nPeriodic, st) || upload(l.perSource, a->periodicSource, l.nPeriodic, st))
        return LBM3_E_HIP;
    // interface lists towards the finer level; their fine-level indices are checked
    // when that level arrives (or now, if it is already there)
    l.F2C.interfaceCount = a->f2cCount;
    l.C2F.interfaceCount = a->c2fCount;
    l.C2F.leftoverCount = a->leftoverCount;
    if (upload(l.F2C.index, a->f2cIndex, a->f2cCount, st) || upload(l.F2C.childMap, a->f2cChild, a->f2cCount, st) ||
        upload(l.C2F.index, a->c2fIndex, a->c2fCount, st) || upload(l.C2F.childMap, a->c2fChild, a->c2fCount, st) ||
        upload(l.C2F.leftoverIndex, a->leftoverIndex, a->leftoverCount, st) ||
        upload(l.C2F.leftoverParent, a->leftoverParent, a->leftoverCount, st) ||
        upload(l.C2F.leftoverNbrI, a->leftoverNbrI, a->leftoverCount, st) ||
        upload(l.C2F.leftoverNbrJ, a->leftoverNbrJ, a->leftoverCount, st) ||
        upload(l.C2F.leftoverNbrK, a->leftoverNbrK, a->leftoverCount, st))
        return LBM3_E_HIP;
    l.fineRefs.clear();
    l.fineRefs.insert(l.fineRefs.end(), a->f2cChild, a->f2cChild + a->f2cCount);
    l.fineRefs.insert(l.fineRefs.end(), a->c2fChild, a->c2fChild + a->c2fCount);
    l.fineRefs.insert(l.fineRefs.end(), a->leftoverIndex, a->leftoverIndex + a->leftoverCount);
    l.interfaceChecked = l.fineRefs.empty();
    if (level + 1 < s.levels && s.L[level + 1].built && check_fine_refs(l, s.L[level + 1].N)) return LBM3_E_ARG;
    if (level > 0 && s.L[level - 1].built && check_fine_refs(s.L[level - 1], l.N)) return LBM3_E_ARG;
    const int rc = finish_level_setup(s, level);
    if (rc) return rc;
    HIPCHK(hipStreamSynchronize(st));
    return 0;
}

int lbm3_apply_initial_condition(lbm3_sim *h, int level)
{
    if (!h) return set_error(LBM3_E_ARG, "null sim");
    if (const int rc = check_level(h->s, level)) return rc;
    return init_level_any(h->s, level, nullptr);
}

int lbm3_apply_initial_fields(lbm3_sim *h, int level, const float *fields4)
{
    if (!h || !fields4) return set_error(LBM3_E_ARG, "null argument");
    if (const int rc = check_level(h->s, level)) return rc;
    DBuf<float> d;
    if (upload(d, fields4, 4LL * h->s.L[level].N, h->s.stream)) return LBM3_E_HIP;
    const int rc = init_level_any(h->s, level, d.p);
    HIPCHK(hipStreamSynchronize(h->s.stream));
    return rc;
}

int lbm3_update_single_grid(lbm3_sim *h, int level)
{
    if (!h) return set_error(LBM3_E_ARG, "null sim");
    if (const int rc = check_level(h->s, level)) return rc;
    if (!h->s.L[level].openFusionChecked)
        if (const int rc = prepare_open_fusion(h->s, level)) return rc;
    step_level_any(h->s, level);
    if (const int rc = settle_shared(h->s)) return rc;
    return check_hip(hipGetLastError(), "updateSingleGrid launch");
}

int lbm3_update_all_grids(lbm3_sim *h, int level)
{
    if (!h) return set_error(LBM3_E_ARG, "null sim");
    if (const int rc = check_run(h->s, level)) return rc;
    update_all(h->s, level);
    if (const int rc = settle_shared(h->s)) return rc;
    return check_hip(hipGetLastError(), "updateAllGrids launch");
}

static int finite_state(Sim &s);
static int mass_sums(Sim &s, double *out2);

int lbm3_run(lbm3_sim *h, int steps)
{
    if (!h || steps < 0) return set_error(LBM3_E_ARG, "bad run arguments");
    Sim &s = h->s;
    if (const int rc = check_run(s, 0)) return rc;
    for (int t = 0; t < steps; ++t) {
        update_all(s, 0);
        // divergence watchdog: every `watchdog` coarse steps and after the last one
        if (s.watchdog > 0 && ((s.L[0].info.iterationsFinished % s.watchdog) == 0 || t == steps - 1))
            if (const int rc = finite_state(s)) return rc;
    }
    if (const int rc = settle_shared(s)) return rc;
    return check_hip(hipGetLastError(), "run launch");
}

int lbm3_set_watchdog(lbm3_sim *h, int period)
{
    if (!h || period < 0) return set_error(LBM3_E_ARG, "bad watchdog period");
    h->s.watchdog = period;
    return 0;
}

} // extern "C"

namespace lbm3 {

// the time-step state of every level, kept on the device so that timing runs
// can be undone: the buffers a checkpoint holds, the levels' step counters and
// parities, rotor angles and the pending-condition flags
struct Snapshot {
    std::vector<DBuf<unsigned char>> bufs;
    std::vector<lbm3_info> infos;
    std::vector<std::vector<double>> angles;
    std::vector<char> settled;
};

static int take_snapshot(Sim &s, Snapshot &z)
{
    z = Snapshot{};
    for (int L = 0; L < s.levels; ++L) {
        Level &l = s.L[L];
        if (const int rc = settle_ghosts(s, l)) return rc;
        for (const auto &b : checkpoint_buffers(l, s.storage)) {
            z.bufs.emplace_back();
            if (b.second == 0 || !b.first) continue;
            HIPCHK(z.bufs.back().alloc((long long)b.second));
            HIPCHK(hipMemcpyAsync(z.bufs.back().p, b.first, b.second, hipMemcpyDeviceToDevice, s.stream));
        }
        z.infos.push_back(l.info);
        std::vector<double> a;
        for (const auto &r : l.rotors) a.push_back(r.radiansElapsed);
        z.angles.push_back(a);
        z.settled.push_back(l.openSettled ? 1 : 0);
    }
    return check_hip(hipStreamSynchronize(s.stream), "snapshot");
}

static int restore_snapshot(Sim &s, Snapshot &z)
{
    HIPCHK(hipStreamSynchronize(s.aux));
    HIPCHK(hipStreamSynchronize(s.aux2));
    size_t k = 0;
    for (int L = 0; L < s.levels; ++L) {
        Level &l = s.L[L];
        for (const auto &b : checkpoint_buffers(l, s.storage)) {
            DBuf<unsigned char> &d = z.bufs[k++];
            if (b.second == 0 || !b.first) continue;
            HIPCHK(hipMemcpyAsync(b.first, d.p, b.second, hipMemcpyDeviceToDevice, s.stream));
        }
        l.info.iterationsFinished = z.infos[(size_t)L].iterationsFinished;
        l.info.iterationsSinceTrackerReset = z.infos[(size_t)L].iterationsSinceTrackerReset;
        l.info.esotwistFlipper = z.infos[(size_t)L].esotwistFlipper;
        for (size_t r = 0; r < l.rotors.size(); ++r) l.rotors[r].radiansElapsed = z.angles[(size_t)L][r];
        l.openSettled = z.settled[(size_t)L] != 0;
        l.ghostsStale = false;
    }
    return check_hip(hipStreamSynchronize(s.stream), "snapshot restore");
}

// the open-cell layout a set of launch choices gives: group width and split
static bool same_open_layout(const Sim &s, const Sim::Tune &a, const Sim::Tune &b)
{
    const int g = open_group_cells((int)storage_bytes(s.storage));
    return (a.openGroup ? a.openGroup : g) == (b.openGroup ? b.openGroup : g) && a.openSplit == b.openSplit &&
           a.rotorInBulk == b.rotorInBulk;
}

// build every level's open-cell groups and rotor-cell records again for the
// current Sim::Tune layout
static int regroup(Sim &s)
{
    for (int L = 0; L < s.levels; ++L) {
        Level &l = s.L[L];
        if (!(l.fusedOpen || !l.rotors.empty()) || !l.built) continue;
        if (const int rc = settle_open(s, L)) return rc;
        l.openFusionChecked = false;
        if (const int rc = prepare_open_fusion(s, L)) return rc;
    }
    return 0;
}

} // namespace lbm3

extern "C" {

int lbm3_autotune(lbm3_sim *h, int steps, double *out, int cap, int *nOut)
{
    if (!h || steps <= 0 || (cap > 0 && !out)) return set_error(LBM3_E_ARG, "bad autotune arguments");
    Sim &s = h->s;
    if (const int rc = check_run(s, 0)) return rc;
    // the state as it is, a pending open condition included: restored in the
    // layout it was taken in, so that an unchanged layout continues bit for bit
    Snapshot z;
    if (const int rc = take_snapshot(s, z)) return rc;
    bool fused = false, rotors = false;
    for (int L = 0; L < s.levels; ++L) {
        fused = fused || s.L[L].fusedOpen;
        rotors = rotors || !s.L[L].rotors.empty();
    }
    const int storageGroup = open_group_cells((int)storage_bytes(s.storage));
    // (group width, x-face choice) layouts of the open cells
    std::vector<std::pair<int, int>> open = {{storageGroup, 0}};
    if (fused) {
        open.push_back({storageGroup == 8 ? 16 : 8, 0});
        open.push_back({1, 0});                     // the open cells in the bulk kernel
        open.push_back({1, 2});                     // ... but those on the x faces, in groups
        open.push_back({1, 3});                     // ... a row's two x-face cells in one wave
        open.push_back({storageGroup, 1});
        open.push_back({storageGroup == 8 ? 16 : 8, 1});
    }
    struct Layout { int group, split, rotor; };
    std::vector<Layout> groups;
    for (int r = 0; r < (rotors ? 2 : 1); ++r)
        for (const auto &o : open) groups.push_back({o.first, o.second, r});
    const int ldsChoices[4] = {0, 24576, 40960, 65536};
    const Sim::Tune start = s.tune;
    const bool startChosen = s.tuneChosen;
    // candidate 0: every level's own choices (tune_of), which no single set of
    // choices gives on several levels: three-level sphere 340 us per coarse step
    // against 368 for the best single set
    struct Cand { Sim::Tune t; bool chosen; double ms; };
    std::vector<Cand> cands;
    auto layout = [&](bool chosen, const Sim::Tune &t) {
        s.tuneChosen = chosen;
        s.tune = t;
        return tune_of(s, s.L[0]);
    };
    double bestMs = 1e300;
    int rows = 0;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    int rc = 0;
    // `steps` steps of the choices in use, after one untimed step, ms per step
    auto timed = [&](double &per) {
        update_all(s, 0);
        if (const int e = check_hip(hipEventRecord(e0, s.stream), "event")) return e;
        for (int k = 0; k < steps; ++k) update_all(s, 0);
        if (const int e = check_hip(hipEventRecord(e1, s.stream), "event")) return e;
        if (const int e = check_hip(hipEventSynchronize(e1), "autotune step")) return e;
        float ms = 0.f;
        if (const int e = check_hip(hipEventElapsedTime(&ms, e0, e1), "event time")) return e;
        per = (double)ms / steps;
        return 0;
    };
    {
        Cand own{start, false, 0.0};
        const Sim::Tune was = tune_of(s, s.L[0]);
        if (!same_open_layout(s, was, layout(false, start))) rc = regroup(s);
        if (!rc) rc = timed(own.ms);
        cands.push_back(own);
    }
    s.tuneChosen = true;
    s.tune = Sim::Tune{};
    for (const Layout &gs : groups) {
        if (rc) break;
        const int g = gs.group;
        s.tune.openGroup = g;
        s.tune.openSplit = gs.split;
        s.tune.rotorInBulk = gs.rotor;
        if ((rc = regroup(s))) break;
        for (int lds : ldsChoices)
            for (int remap = 0; remap < 4 && !rc; ++remap)
                for (int overlap = 3; overlap >= 0 && !rc; --overlap) {
                    if (overlap == 2 && s.levels == 1) continue;   // no finer levels to run beside
                    s.tune.bulkLds = lds;
                    s.tune.xcdRemap = remap;
                    s.tune.overlap = overlap;
                    double per = 0.0;
                    if ((rc = timed(per))) break;
                    if (rows < cap) {
                        double *o = out + 7 * (size_t)rows;
                        o[0] = lds; o[1] = remap; o[2] = overlap; o[3] = g; o[4] = gs.split; o[5] = gs.rotor; o[6] = per;
                    }
                    ++rows;
                    cands.push_back({s.tune, true, per});
                }
        if (rc) break;
    }
    // The fastest few candidates are timed again, in turns over three rounds,
    // and the best of each candidate's rounds decides: a single noisy timing
    // in the sweep (a launch that met another's traffic in the cache, a clock
    // change) does not pick the configuration alone.
    // Candidate 0 is always among them and wins ties.
    int best = 0;
    if (!rc) {
        std::stable_sort(cands.begin() + 1, cands.end(), [](const Cand &a, const Cand &b) { return a.ms < b.ms; });
        const int K = (int)std::min<size_t>(7, cands.size());
        std::vector<double> again(K, 1e300);
        for (int round = 0; round < 3 && !rc; ++round)
            for (int i = 0; i < K && !rc; ++i) {
                const Sim::Tune was = tune_of(s, s.L[0]);
                if (!same_open_layout(s, was, layout(cands[i].chosen, cands[i].t)) && (rc = regroup(s))) break;
                double per = 0.0;
                if (!(rc = timed(per))) again[i] = std::min(again[i], per);
            }
        for (int i = 0; i < K; ++i)
            if (again[i] < bestMs) { bestMs = again[i]; best = i; }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    const Sim::Tune was = layout(startChosen, start);
    const int rg = regroup(s);
    const int rs = restore_snapshot(s, z);
    if (rc) return rc;
    if (rg) return rg;
    if (rs) return rs;
    if (nOut) *nOut = rows;
    // another open-cell layout: the pending condition is completed in the old
    // one first (regroup), which rounds it to the storage type once
    return same_open_layout(s, was, layout(cands[best].chosen, cands[best].t)) ? 0 : regroup(s);
}

// level 0's choices, as lbm3_get_tune reports them: by its cells' records, which
// the first step makes
static int reported_tune(Sim &s, int (&t6)[6])
{
    Level &l = s.L[0];
    if (!s.tuneChosen && l.built && !l.openFusionChecked)
        if (const int rc = prepare_open_fusion(s, 0)) return rc;
    const Sim::Tune t = tune_of(s, l);
    t6[0] = t.bulkLds; t6[1] = t.xcdRemap; t6[2] = t.overlap;
    t6[3] = t.openGroup ? t.openGroup : open_group_cells((int)storage_bytes(s.storage));
    t6[4] = t.openSplit;
    t6[5] = t.rotorInBulk;
    return 0;
}

int lbm3_get_tune(lbm3_sim *h, int *out6)
{
    if (!h || !out6) return set_error(LBM3_E_ARG, "null argument");
    int t[6];
    if (const int rc = reported_tune(h->s, t)) return rc;
    memcpy(out6, t, sizeof t);
    return 0;
}

int lbm3_set_tune(lbm3_sim *h, const int *in6)
{
    if (!h || !in6) return set_error(LBM3_E_ARG, "null argument");
    if (in6[0] < 0 || in6[0] > 65536 || in6[1] < 0 || in6[1] > 3 || in6[2] < 0 || in6[2] > 3 ||
        (in6[3] != 1 && in6[3] != 8 && in6[3] != 16) ||
        in6[4] < 0 || in6[4] > 3 || in6[5] < 0 || in6[5] > 1)
        return set_error(LBM3_E_ARG, "bulk LDS in 0..65536 bytes, block order 0..3, side streams 0..3, open groups of 1 (in the bulk "
                                     "kernel), 8 or 16 cells, x-face choice 0..3, rotor cells 0..1");
    Sim &s = h->s;
    if (s.timing) return set_error(LBM3_E_STATE, "launch choices changed during a timed run");
    if (!s.tuneChosen) {
        // what lbm3_get_tune reports leaves every level its own choices
        int now[6];
        if (const int rc = reported_tune(s, now)) return rc;
        if (memcmp(now, in6, sizeof now) == 0) return 0;
    }
    const Sim::Tune was = tune_of(s, s.L[0]);
    s.tuneChosen = true;
    s.tune = Sim::Tune{};
    s.tune.bulkLds = in6[0];
    s.tune.xcdRemap = in6[1];
    s.tune.overlap = in6[2];
    s.tune.openGroup = in6[3];
    s.tune.openSplit = in6[4];
    s.tune.rotorInBulk = in6[5];
    // only a new layout of the open or rotor cells rebuilds the records, which
    // completes a pending open condition first (regroup)
    return same_open_layout(s, was, s.tune) ? 0 : regroup(s);
}

int lbm3_run_graph(lbm3_sim *h, int steps)
{
    if (!h || steps < 0) return set_error(LBM3_E_ARG, "bad run arguments");
    Sim &s = h->s;
    if (const int rc = check_run(s, 0)) return rc;
    if (s.timing) return set_error(LBM3_E_STATE, "graph replay during a timed run");
    for (int L = 0; L < s.levels; ++L)
        if (const int rc = settle_ghosts(s, s.L[L])) return rc;
    if (steps >= 2) {
        // Two coarse steps bring every level's esotwist parity back, so one
        // captured pair replays with the same kernel arguments.  What changes
        // from pair to pair -- the iteration an open-boundary condition belongs
        // to, whether a deferred one is pending, the rotors' angles -- the
        // kernels read from a device table with one slot per level step,
        // refilled before each replay from a dry run of the host bookkeeping.
        struct Host {
            lbm3_info info;
            bool settled;
            std::vector<double> angles;
        };
        auto save = [&]() {
            std::vector<Host> v((size_t)s.levels);
            for (int L = 0; L < s.levels; ++L) {
                v[(size_t)L] = {s.L[L].info, s.L[L].openSettled, {}};
                for (const auto &r : s.L[L].rotors) v[(size_t)L].angles.push_back(r.radiansElapsed);
            }
            return v;
        };
        auto load_host = [&](const std::vector<Host> &v) {
            for (int L = 0; L < s.levels; ++L) {
                s.L[L].info = v[(size_t)L].info;
                s.L[L].openSettled = v[(size_t)L].settled;
                for (size_t r = 0; r < s.L[L].rotors.size(); ++r) s.L[L].rotors[r].radiansElapsed = v[(size_t)L].angles[r];
            }
        };
        long long slots = 0;
        for (int L = 0; L < s.levels; ++L) slots += 2LL << L;
        DBuf<StepParam> table;
        HIPCHK(table.alloc(slots));
        const std::vector<Host> before = save();
        hipGraph_t graph = nullptr;
        HIPCHK(hipStreamBeginCapture(s.stream, hipStreamCaptureModeThreadLocal));
        s.captureTable = table.p;
        s.captureSlot = 0;
        update_all(s, 0);
        update_all(s, 0);
        s.captureTable = nullptr;
        const hipError_t ec = hipStreamEndCapture(s.stream, &graph);
        const int captured = s.captureSlot;
        load_host(before);                    // nothing ran yet
        if (ec != hipSuccess) {
            if (graph) (void)hipGraphDestroy(graph);
            return check_hip(ec, "step capture");
        }
        if (captured != slots) {
            (void)hipGraphDestroy(graph);
            return set_error(LBM3_E_STATE, "step capture used an unexpected number of level steps");
        }
        hipGraphExec_t exec = nullptr;
        hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        // pinned staging of the table, two buffers used in turn: a buffer is
        // refilled only after the copy that last read it has completed
        StepParam *stage[2] = {nullptr, nullptr};
        hipEvent_t copied[2] = {nullptr, nullptr};
        for (int b = 0; b < 2 && e == hipSuccess; ++b) {
            e = hipHostMalloc((void **)&stage[b], sizeof(StepParam) * (size_t)slots, hipHostMallocDefault);
            if (e == hipSuccess) e = hipEventCreateWithFlags(&copied[b], hipEventDisableTiming);
        }
        std::vector<StepParam> params;
        for (int k = 0; e == hipSuccess && k < steps / 2; ++k) {
            params.clear();
            s.dryRun = &params;
            update_all(s, 0);
            update_all(s, 0);
            s.dryRun = nullptr;
            const int b = k & 1;
            if (k >= 2) e = hipEventSynchronize(copied[b]);
            if (e != hipSuccess) break;
            memcpy(stage[b], params.data(), sizeof(StepParam) * params.size());
            e = hipMemcpyAsync(table.p, stage[b], sizeof(StepParam) * params.size(), hipMemcpyHostToDevice, s.stream);
            if (e == hipSuccess) e = hipEventRecord(copied[b], s.stream);
            if (e == hipSuccess) e = hipGraphLaunch(exec, s.stream);
        }
        s.dryRun = nullptr;
        const hipError_t es = hipStreamSynchronize(s.stream);   // the graph is released after its last replay
        for (int b = 0; b < 2; ++b) {
            if (stage[b]) (void)hipHostFree(stage[b]);
            if (copied[b]) (void)hipEventDestroy(copied[b]);
        }
        if (exec) (void)hipGraphExecDestroy(exec);
        (void)hipGraphDestroy(graph);
        if (e != hipSuccess) return check_hip(e, "step graph replay");
        if (es != hipSuccess) return check_hip(es, "step graph replay");
    }
    if (steps % 2) update_all(s, 0);
    if (const int rc = settle_shared(s)) return rc;
    return check_hip(hipGetLastError(), "graph run");
}

int lbm3_synchronize(lbm3_sim *h)
{
    if (!h) return set_error(LBM3_E_ARG, "null sim");
    return check_hip(hipStreamSynchronize(h->s.stream), "synchronize");
}

int lbm3_run_timed(lbm3_sim *h, int steps, int kernelEvents, double *out)
{
    if (!h || !out || steps <= 0) return set_error(LBM3_E_ARG, "bad timed-run arguments");
    Sim &s = h->s;
    if (const int rc = check_run(s, 0)) return rc;
    hipEvent_t a, b;
    HIPCHK(hipEventCreate(&a));
    HIPCHK(hipEventCreate(&b));
    s.timing = kernelEvents != 0;
    s.evUsed = 0;
    HIPCHK(hipEventRecord(a, s.stream));
    for (int t = 0; t < steps; ++t) update_all(s, 0);
    s.timing = false;
    if (const int rc = settle_shared(s)) return rc;
    HIPCHK(hipEventRecord(b, s.stream));
    HIPCHK(hipEventSynchronize(b));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, a, b));
    double bulk = 0.0, wall = 0.0;
    for (int e = 0; e < s.evUsed; ++e) {
        float k = 0.f, w = 0.f;
        HIPCHK(hipEventElapsedTime(&k, s.ev[e][0], s.ev[e][1]));
        HIPCHK(hipEventElapsedTime(&w, s.ev[e][1], s.ev[e][2]));
        bulk += k;
        wall += w;
    }
    out[0] = ms;
    out[1] = bulk;
    out[2] = s.evUsed;
    out[3] = wall;
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return check_hip(hipGetLastError(), "timed run");
}

int lbm3_get_info(lbm3_sim *h, int level, lbm3_info *out)
{
    if (!h || !out || level < 0 || level >= h->s.levels) return set_error(LBM3_E_ARG, "bad info arguments");
    *out = h->s.L[level].info;
    return 0;
}

int lbm3_level_count(lbm3_sim *h) { return h ? h->s.levels : 0; }

int lbm3_download_macros(lbm3_sim *h, int level, void *out)
{
    if (!h || !out) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    if (const int rc = check_level(s, level)) return rc;
    if (const int rc = settle_open(s, level)) return rc;
    Level &l = s.L[level];
    const size_t cb = compute_bytes(s.storage);
    // fields of up to 64 MiB are made in a buffer that the simulation keeps: an
    // allocation and its release, which waits for the device, cost a 32^3 box
    // more than the fields themselves
    const long long bytes = 4LL * l.N * (long long)cb;
    // (one call at a time; a second thread's waits for it)
    std::unique_lock<std::mutex> kept(s.keptLock, std::defer_lock);
    DBuf<unsigned char> own;
    if (bytes <= (64LL << 20)) kept.lock();
    DBuf<unsigned char> &d = kept.owns_lock() ? s.fields : own;
    if (d.n < bytes) HIPCHK(d.alloc(bytes));
    const bool flip = l.info.esotwistFlipper != 0;
    const Topology t = topo_of(l);
    switch (s.storage) {
    case LBM3_STORE_F16: launch_macros<__half>(reinterpret_cast<__half *>(l.f.p), t, reinterpret_cast<float *>(d.p), s.codec, flip, s.stream); break;
    case LBM3_STORE_BF16: launch_macros<__hip_bfloat16>(reinterpret_cast<__hip_bfloat16 *>(l.f.p), t, reinterpret_cast<float *>(d.p), s.codec, flip, s.stream); break;
    case LBM3_STORE_F16C: launch_macros<f16c>(reinterpret_cast<f16c *>(l.f.p), t, reinterpret_cast<float *>(d.p), s.codec, flip, s.stream); break;
    case LBM3_STORE_F64: launch_macros<double>(reinterpret_cast<double *>(l.f.p), t, reinterpret_cast<double *>(d.p), s.codec, flip, s.stream); break;
    default: launch_macros<float>(reinterpret_cast<float *>(l.f.p), t, reinterpret_cast<float *>(d.p), s.codec, flip, s.stream); break;
    }
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, d.p, 4 * (size_t)l.N * cb, hipMemcpyDeviceToHost, s.stream));
    HIPCHK(hipStreamSynchronize(s.stream));
    return 0;
}

int lbm3_download_populations(lbm3_sim *h, int level, void *out, long long bytes)
{
    if (!h || !out) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    if (const int rc = check_level(s, level)) return rc;
    if (const int rc = settle_open(s, level)) return rc;
    Level &l = s.L[level];
    const long long es = storage_bytes(s.storage), n = 27LL * l.N * es;
    if (bytes < n) return set_error(LBM3_E_ARG, "buffer too small");
    DBuf<unsigned char> d;
    HIPCHK(d.alloc(n > 0 ? n : 1));
    launch_relayout(l.f.p, d.p, l.N, int(es), true, s.stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, d.p, (size_t)n, hipMemcpyDeviceToHost, s.stream));
    HIPCHK(hipStreamSynchronize(s.stream));
    return 0;
}

int lbm3_upload_populations(lbm3_sim *h, int level, const void *in, long long bytes)
{
    if (!h || !in) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    if (const int rc = check_level(s, level)) return rc;
    Level &l = s.L[level];
    const long long es = storage_bytes(s.storage), n = 27LL * l.N * es;
    if (bytes != n) return set_error(LBM3_E_ARG, "size mismatch");
    DBuf<unsigned char> d;
    HIPCHK(d.alloc(n > 0 ? n : 1));
    HIPCHK(hipMemcpyAsync(d.p, in, (size_t)n, hipMemcpyHostToDevice, s.stream));
    launch_relayout(d.p, l.f.p, l.N, int(es), false, s.stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(s.stream));
    s.L[level].openSettled = true;   // an uploaded state is complete
    s.L[level].ghostsStale = false;
    return 0;
}

// the device buffer of a named per-level array: false if the name is not one
static bool level_buffer(Level &l, const char *name, const void *&src, long long &n, size_t &es)
{
#define ARR(nm, buf, cnt) else if (!strcmp(name, nm)) { src = (buf).p; n = (cnt); es = sizeof(*(buf).p); }
    if (false) {}
    ARR("shifter", l.shifter, l.N) ARR("rowI", l.ri, l.nRows) ARR("rowJ", l.rj, l.nRows) ARR("rowK", l.rk, l.nRows)
    ARR("rowJPlus", l.rjp, l.nRows) ARR("rowKPlus", l.rkp, l.nRows) ARR("rowJKPlus", l.rjkp, l.nRows)
    ARR("wallMap", l.wallMap, l.N) ARR("wallIndex", l.wallIndex, l.W) ARR("wallData", l.wallData, l.W)
    ARR("linkLength", l.linkLength, 7LL * l.W) ARR("periodicIndex", l.perIndex, l.nPeriodic)
    ARR("periodicSource", l.perSource, l.nPeriodic) ARR("openIndex", l.openCell, l.nOpen)
    ARR("openSource", l.openSource, l.nOpen) ARR("wallForce", l.gWall, 3LL * l.W)
    else return false;
#undef ARR
    return true;
}

int lbm3_device_array(lbm3_sim *h, int level, const char *name, void **ptr, long long *count)
{
    if (!h || !name || !ptr || !count || level < 0 || level >= h->s.levels) return set_error(LBM3_E_ARG, "bad array arguments");
    Sim &s = h->s;
    Level &l = s.L[level];
    if (!l.built) return set_error(LBM3_E_STATE, "level not built");
    if (!strcmp(name, "f")) {
        // the ghost copy is waited for: a caller that synchronized after its run
        // may read on a stream of its own at once
        const bool wait = l.ghostsStale;
        if (const int rc = settle_open(s, level)) return rc;
        if (wait) HIPCHK(hipStreamSynchronize(s.stream));
        l.shared = true;
        *ptr = l.f.p;
        *count = 27LL * padded_cells(l.N);
        return 0;
    }
    const void *src = nullptr;
    long long n = 0;
    size_t es = 4;
    if (!level_buffer(l, name, src, n, es)) return set_error(LBM3_E_ARG, std::string("unknown array ") + name);
    *ptr = const_cast<void *>(src);
    *count = n;
    return 0;
}

int lbm3_population_layout(lbm3_sim *h, int *tile, int *bytes)
{
    if (!h || !tile || !bytes) return set_error(LBM3_E_ARG, "null argument");
    *tile = LBM3_TILE;
    *bytes = (int)storage_bytes(h->s.storage);
    return 0;
}

int lbm3_download_array(lbm3_sim *h, int level, const char *name, void *out, long long capacity, long long *count)
{
    if (!h || !name || !count || level < 0 || level >= h->s.levels) return set_error(LBM3_E_ARG, "bad array arguments");
    Sim &s = h->s;
    Level &l = s.L[level];
    const void *src = nullptr;
    long long n = -1;
    size_t es = 4;
#define ARR(nm, buf, cnt) else if (!strcmp(name, nm)) { src = (buf).p; n = (cnt); es = sizeof(*(buf).p); }
    if (false) {}
    ARR("shifter", l.shifter, l.N) ARR("rowI", l.ri, l.nRows) ARR("rowJ", l.rj, l.nRows) ARR("rowK", l.rk, l.nRows)
    ARR("rowJPlus", l.rjp, l.nRows) ARR("rowKPlus", l.rkp, l.nRows) ARR("rowJKPlus", l.rjkp, l.nRows)
    ARR("wallMap", l.wallMap, l.N) ARR("wallIndex", l.wallIndex, l.W) ARR("wallData", l.wallData, l.W)
    ARR("cellRow", l.cellRow, l.N)
    ARR("bulkSkip", l.bulkSkip, (l.N + 63) / 64) ARR("openBits", l.openBits, l.openInBulk ? (l.N + 63) / 64 : 0)
    ARR("rotorBits", l.rotorBits, l.rotorInBulk ? (l.N + 63) / 64 : 0)
    ARR("imageSources", l.imageSources, l.imagesReady ? (l.N + 63) / 64 : 0)
    ARR("linkLength", l.linkLength, 7LL * l.W) ARR("periodicIndex", l.perIndex, l.nPeriodic)
    ARR("periodicSource", l.perSource, l.nPeriodic) ARR("openIndex", l.openCell, l.nOpen)
    ARR("openSource", l.openSource, l.nOpen) ARR("openMeta", l.openMeta, l.nOpen)
    ARR("wallForce", l.gWall, 3LL * l.W) ARR("rayHitScan", l.rayHitScan, l.rayHitScan.n) ARR("rayMap", l.rayMap, l.rayMap.n)
    ARR("f2cIndex", l.F2C.index, l.F2C.interfaceCount) ARR("f2cChild", l.F2C.childMap, l.F2C.interfaceCount)
    ARR("c2fIndex", l.C2F.index, l.C2F.interfaceCount) ARR("c2fChild", l.C2F.childMap, l.C2F.interfaceCount)
    ARR("leftoverIndex", l.C2F.leftoverIndex, l.C2F.leftoverCount)
    ARR("leftoverParent", l.C2F.leftoverParent, l.C2F.leftoverCount)
    ARR("leftoverNbrI", l.C2F.leftoverNbrI, l.C2F.leftoverCount)
    ARR("leftoverNbrJ", l.C2F.leftoverNbrJ, l.C2F.leftoverCount)
    ARR("leftoverNbrK", l.C2F.leftoverNbrK, l.C2F.leftoverCount)
#undef ARR
    else if (!strcmp(name, "openCount")) {
        *count = l.nOpenIDs;
        if (out) {
            if (capacity < l.nOpenIDs) return set_error(LBM3_E_ARG, "buffer too small");
            memcpy(out, l.openCount.data(), sizeof(int) * (size_t)l.nOpenIDs);
        }
        return 0;
    } else if (!strncmp(name, "rotor", 5) && name[5] >= '0' && name[5] <= '9') {
        const int r = name[5] - '0';
        if (r >= (int)l.rotors.size()) return set_error(LBM3_E_ARG, "no such rotor");
        Level::Rotor &R = l.rotors[r];
        const char *f = name + 6;
        if (!strcmp(f, "Map")) { src = R.rotorMap.p; n = R.blockCount; }
        else if (!strcmp(f, "Index")) { src = R.index.p; n = R.dev.nonZero; }
        else if (!strcmp(f, "Interp")) { src = R.interp.p; n = 64LL * R.dev.nonZero; }
        else if (!strcmp(f, "Force")) { src = R.g.p; n = 81LL * R.dev.nonZero; es = 8; }
        else return set_error(LBM3_E_ARG, "unknown rotor array");
    } else if (!strncmp(name, "stl", 3) && name[3] >= '0' && name[3] <= '9' && !strcmp(name + 4, "EdgeCount")) {
        // shared-edge counts of a static body of the last build (host copy; any level)
        const size_t b = (size_t)(name[3] - '0');
        if (b >= s.stlEdges.size()) return set_error(LBM3_E_ARG, "no such STL body");
        const std::vector<int> &e = s.stlEdges[b];
        *count = (long long)e.size();
        if (out) {
            if (capacity < (long long)e.size()) return set_error(LBM3_E_ARG, "buffer too small");
            memcpy(out, e.data(), sizeof(int) * e.size());
        }
        return 0;
    } else if (!strcmp(name, "openRefs")) {
        if (l.built)
            if (const int rc = settle_open(s, level)) return rc;
        src = l.openRefs.p;
        es = compute_bytes(s.storage);
        n = 2LL * (l.nOpen > 0 ? l.nOpen : 1);
    } else return set_error(LBM3_E_ARG, std::string("unknown array ") + name);
    *count = n;
    if (!out || n <= 0 || !src) return 0;
    if (capacity < n) return set_error(LBM3_E_ARG, "buffer too small");
    HIPCHK(hipStreamSynchronize(s.stream));
    HIPCHK(hipMemcpy(out, src, es * (size_t)n, hipMemcpyDeviceToHost));
    return 0;
}

int lbm3_kinetic_energy(lbm3_sim *h, double *out)
{
    if (!h || !out) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    double total = 0.0;
    for (int level = 0; level < s.levels; ++level) {
        if (const int rc = check_level(s, level)) return rc;
        if (const int rc = settle_open(s, level)) return rc;
        Level &l = s.L[level];
        const long long nb = (l.N + 255) / 256;
        if (s.partial.n < nb) HIPCHK(s.partial.alloc(nb));
        if (!s.scalar.p) HIPCHK(s.scalar.alloc(8));
        const bool flip = l.info.esotwistFlipper != 0;
        const Topology t = topo_of(l);
        switch (s.storage) {
        case LBM3_STORE_F16: launch_kinetic_energy<__half>(reinterpret_cast<__half *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream); break;
        case LBM3_STORE_BF16: launch_kinetic_energy<__hip_bfloat16>(reinterpret_cast<__hip_bfloat16 *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream); break;
        case LBM3_STORE_F16C: launch_kinetic_energy<f16c>(reinterpret_cast<f16c *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream); break;
        case LBM3_STORE_F64: launch_kinetic_energy<double>(reinterpret_cast<double *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream); break;
        default: launch_kinetic_energy<float>(reinterpret_cast<float *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream); break;
        }
        HIPCHK(hipGetLastError());
        double v = 0.0;
        HIPCHK(hipMemcpyAsync(&v, s.scalar.p, sizeof(double), hipMemcpyDeviceToHost, s.stream));
        HIPCHK(hipStreamSynchronize(s.stream));
        total += v / (double)(1LL << (3 * level));
    }
    *out = total;
    return 0;
}

// the mass sum over every level is finite exactly when no counted cell holds
// a NaN or infinite population
static int finite_state(Sim &s)
{
    double m[2] = {0.0, 0.0};
    if (const int rc = mass_sums(s, m)) return rc;
    if (!std::isfinite(m[0]))
        return set_error(LBM3_E_DIVERGED, "non-finite populations after coarse step " +
                                              std::to_string(s.L[0].info.iterationsFinished));
    return 0;
}

int lbm3_mass(lbm3_sim *h, double *out2)
{
    if (!h || !out2) return set_error(LBM3_E_ARG, "null argument");
    return mass_sums(h->s, out2);
}

static int mass_sums(Sim &s, double *out2)
{
    for (int level = 0; level < s.levels; ++level) {
        if (const int rc = check_level(s, level)) return rc;
        if (const int rc = settle_open(s, level)) return rc;
        Level &l = s.L[level];
        const long long nb = (l.N + 255) / 256;
        if (s.partial.n < 2 * nb) HIPCHK(s.partial.alloc(2 * nb));
        if (!s.scalar.p) HIPCHK(s.scalar.alloc(8));
        const bool flip = l.info.esotwistFlipper != 0;
        const Topology t = topo_of(l);
        const double w = (double)(1LL << (3 * level));
        const bool acc = level > 0;
        switch (s.storage) {
        case LBM3_STORE_F16: launch_mass<__half>(reinterpret_cast<__half *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream, w, acc); break;
        case LBM3_STORE_BF16: launch_mass<__hip_bfloat16>(reinterpret_cast<__hip_bfloat16 *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream, w, acc); break;
        case LBM3_STORE_F16C: launch_mass<f16c>(reinterpret_cast<f16c *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream, w, acc); break;
        case LBM3_STORE_F64: launch_mass<double>(reinterpret_cast<double *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream, w, acc); break;
        default: launch_mass<float>(reinterpret_cast<float *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.partial.p, s.scalar.p, s.codec, flip, s.stream, w, acc); break;
        }
        HIPCHK(hipGetLastError());
    }
    HIPCHK(hipMemcpyAsync(out2, s.scalar.p, 2 * sizeof(double), hipMemcpyDeviceToHost, s.stream));
    HIPCHK(hipStreamSynchronize(s.stream));
    return 0;
}

int lbm3_wall_forces(lbm3_sim *h, int level, const double *origin, int nBodies, double *out)
{
    if (!h || !out || nBodies <= 0 || nBodies > LBM3_MAX_BODIES) return set_error(LBM3_E_ARG, "bad force arguments");
    Sim &s = h->s;
    if (const int rc = check_level(s, level)) return rc;
    Level &l = s.L[level];
    for (int i = 0; i < 6 * nBodies; ++i) out[i] = 0.0;
    if (l.W == 0) return 0;
    const long long nb = (l.W + 255) / 256;
    DBuf<double> part;
    HIPCHK(part.alloc(nb * 6 * nBodies));
    const double o[3] = {origin ? origin[0] : 0.0, origin ? origin[1] : 0.0, origin ? origin[2] : 0.0};
    launch_wall_force(l.gWall.p, l.W, l.wallData.p, l.wallIndex.p, topo_of(l), l.geom, o, nBodies, part.p, s.stream);
    HIPCHK(hipGetLastError());
    std::vector<double> host((size_t)(nb * 6 * nBodies));
    HIPCHK(hipMemcpyAsync(host.data(), part.p, sizeof(double) * host.size(), hipMemcpyDeviceToHost, s.stream));
    HIPCHK(hipStreamSynchronize(s.stream));
    for (long long b = 0; b < nb; ++b)
        for (int i = 0; i < 6 * nBodies; ++i) out[i] += host[(size_t)(b * 6 * nBodies + i)];
    return 0;
}

int lbm3_reset_wall_forces(lbm3_sim *h)
{
    if (!h) return set_error(LBM3_E_ARG, "null sim");
    for (int level = 0; level < h->s.levels; ++level) {
        Level &l = h->s.L[level];
        if (l.gWall.p) HIPCHK(hipMemsetAsync(l.gWall.p, 0, sizeof(double) * (size_t)l.gWall.n, h->s.stream));
        for (Level::Rotor &r : l.rotors)
            if (r.g.p) HIPCHK(hipMemsetAsync(r.g.p, 0, sizeof(double) * (size_t)r.g.n, h->s.stream));
    }
    return 0;
}

int lbm3_open_boundary_stats(lbm3_sim *h, int openBCID, double *out)
{
    if (!h || !out) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    if (!s.C.trackOpenBoundaries) return set_error(LBM3_E_ARG, "the case does not track open boundaries");
    double area = 0.0, sum[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    bool found = false;
    for (int level = 0; level < s.levels; ++level) {
        if (const int rc = check_level(s, level)) return rc;
        Level &l = s.L[level];
        if (openBCID < 0 || openBCID >= l.nOpenIDs) continue;
        found = true;
        if (const int rc = settle_open(s, level)) return rc;
        if (l.info.iterationsSinceTrackerReset <= 0) return set_error(LBM3_E_ARG, "no time step since the last reset");
        int start = 0;
        for (int b = 0; b < openBCID; ++b) start += l.openCount[b];
        const int count = l.openCount[openBCID];
        const long long nb = (count + 255) / 256;
        if (s.partial.n < 7 * nb) HIPCHK(s.partial.alloc(7 * nb));
        const long long stride = l.nOpen > 0 ? l.nOpen : 1;
        const int blocks = launch_open_stats(l.openCum.p, l.openCum.p + stride, l.openMeta.p, start, count,
                                             1.0 / double(l.info.iterationsSinceTrackerReset), s.partial.p, s.stream);
        HIPCHK(hipGetLastError());
        std::vector<double> part(7 * (size_t)blocks);
        if (blocks > 0)
            HIPCHK(hipMemcpyAsync(part.data(), s.partial.p, sizeof(double) * part.size(), hipMemcpyDeviceToHost, s.stream));
        HIPCHK(hipStreamSynchronize(s.stream));
        double v[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int b = 0; b < blocks; ++b)
            for (int k = 0; k < 7; ++k) v[k] += part[7 * (size_t)b + k];
        // physical units (trackerFunctions.h:172-192, cellFunctions.h:288-294)
        const double dx = double(l.info.res) / 1000.0, cellArea = dx * dx;
        const double vel = dx / double(l.info.dtPhys), rho = double(s.C.rhoPhys);
        const double pres = rho * vel * vel / 3.0;       // dRho -> pressure: rho_phys c_s^2
        sum[0] += v[0] * cellArea * vel;
        sum[1] += v[1] * cellArea * vel * rho;
        sum[2] += v[2] * cellArea * vel * vel * rho;
        sum[3] += v[3] * pres * cellArea;
        sum[4] += v[4] * pres * cellArea * vel;
        sum[5] += v[5] * cellArea * vel * vel * vel * rho;
        area += v[6] * cellArea;
    }
    if (!found) return set_error(LBM3_E_ARG, "no such open boundary");
    out[0] = area;
    out[1] = sum[0] / area;
    out[2] = sum[1];
    out[3] = sum[2];
    out[4] = sum[3] / area;
    out[5] = sum[4];
    out[6] = sum[5];
    return 0;
}

int lbm3_reset_open_boundary_stats(lbm3_sim *h)
{
    if (!h) return set_error(LBM3_E_ARG, "null sim");
    Sim &s = h->s;
    for (int level = 0; level < s.levels; ++level) {
        if (const int rc = check_level(s, level)) return rc;
        if (const int rc = settle_open(s, level)) return rc;   // the last step's condition belongs to the old window
        Level &l = s.L[level];
        if (l.openCum.p) HIPCHK(hipMemsetAsync(l.openCum.p, 0, sizeof(double) * (size_t)l.openCum.n, s.stream));
        l.info.iterationsSinceTrackerReset = 0;
    }
    return 0;
}

// The image of a section through every level before unit conversion
// (exportSectionCutPlotGeneral / getFlowReportGeneral, exportSectionCutPlot.h:11-290,
// flowReportFunctions.h:11-264): the plane at `cut` along its normal, cropped to
// `bounds` (all zero or null: the whole grid), at the finest level whose image
// fits 16 M pixels.  With img null only the size is computed.
struct SectionImage {
    int H = 0, V = 0, imageLevel = 0;
    CutUnits units{};
};

static int section_image(Sim &s, int plane, float cut, const lbm3_bounds *bounds, SectionImage &out, DBuf<float> *img)
{
    if (plane < LBM3_PLANE_XY || plane > LBM3_PLANE_ZX) return set_error(LBM3_E_ARG, "unknown section plane");
    for (int L = 0; L < s.levels; ++L)
        if (const int rc = check_level(s, L)) return rc;
    const int finest = s.levels - 1;
    const lbm3_info &F = s.L[finest].info;
    auto origin = [plane](const lbm3_info &I) { return plane == LBM3_PLANE_XY ? I.oz : (plane == LBM3_PLANE_ZY ? I.ox : I.oy); };
    auto normalCount = [plane](const lbm3_info &I) {
        return plane == LBM3_PLANE_XY ? I.cellCountZ : (plane == LBM3_PLANE_ZY ? I.cellCountX : I.cellCountY);
    };
    // the cut plane on the finest level (getIJKCellIndexFromXYZ, cellFunctions.h:96-101)
    const int cutIndex = (int)((cut - origin(F)) / F.res + 0.5f);
    if (cutIndex < 0 || cutIndex >= normalCount(F)) return set_error(LBM3_E_ARG, "section cut outside the finest grid");
    const double cutPos = double(origin(F)) + double(cutIndex) * double(F.res);
    // crop to the bounds (exportSectionCutPlot.h:33-55)
    int i0 = 0, i1 = F.cellCountX, j0 = 0, j1 = F.cellCountY, k0 = 0, k1 = F.cellCountZ;
    if (bounds && (bounds->xMin != 0.f || bounds->xMax != 0.f || bounds->yMin != 0.f || bounds->yMax != 0.f ||
                   bounds->zMin != 0.f || bounds->zMax != 0.f)) {
        const float xMin = F.ox - 0.5f * F.res, xMax = F.ox + F.res * (F.cellCountX - 0.5f);
        const float yMin = F.oy - 0.5f * F.res, yMax = F.oy + F.res * (F.cellCountY - 0.5f);
        const float zMin = F.oz - 0.5f * F.res, zMax = F.oz + F.res * (F.cellCountZ - 0.5f);
        i0 = std::max(0, (int)ceilf((bounds->xMin - xMin) / F.res));
        i1 = std::min(F.cellCountX, F.cellCountX - (int)ceilf((xMax - bounds->xMax) / F.res));
        j0 = std::max(0, (int)ceilf((bounds->yMin - yMin) / F.res));
        j1 = std::min(F.cellCountY, F.cellCountY - (int)ceilf((yMax - bounds->yMax) / F.res));
        k0 = std::max(0, (int)ceilf((bounds->zMin - zMin) / F.res));
        k1 = std::min(F.cellCountZ, F.cellCountZ - (int)ceilf((zMax - bounds->zMax) / F.res));
    }
    // the finest level whose image fits the pixel limit (:57-76)
    int H, V, h0, v0;
    if (plane == LBM3_PLANE_XY) { H = i1 - i0; V = j1 - j0; h0 = i0; v0 = j0; }
    else if (plane == LBM3_PLANE_ZY) { H = k1 - k0; V = j1 - j0; h0 = k0; v0 = j0; }
    else { H = k1 - k0; V = i1 - i0; h0 = k0; v0 = i0; }
    int imageLevel = finest;
    while ((long long)H * V > 16000000LL && imageLevel > 0) {
        --imageLevel;
        H /= 2; h0 /= 2;
        V /= 2; v0 /= 2;
    }
    if (H <= 0 || V <= 0 || (long long)H * V > 16000000LL) return set_error(LBM3_E_ARG, "section image empty or too large");
    out.H = H;
    out.V = V;
    out.imageLevel = imageLevel;
    out.units = CutUnits{};
    out.units.plane = plane;
    out.units.rhoPhys = s.C.rhoPhys;
    for (int L = 0; L < s.levels; ++L) {
        out.units.res[L] = s.L[L].info.res;
        out.units.dt[L] = s.L[L].info.dtPhys;
    }
    if (!img) return 0;
    const long long pixels = (long long)H * V;
    HIPCHK(img->alloc(6 * pixels));
    launch_cut_clear(img->p, pixels, s.stream);
    for (int L = 0; L < s.levels; ++L) {
        if (const int rc = settle_open(s, L)) return rc;
        const lbm3_info &I = s.L[L].info;
        if (I.cellCount <= 0 || normalCount(I) <= 0 || I.res <= 0.f) continue;
        double ni = (cutPos - double(origin(I))) / double(I.res);
        ni = std::min(std::max(ni, 0.0), double(normalCount(I) - 1));
        CutLevel d{};
        d.plane = plane;
        d.lower = (int)std::floor(ni);
        d.alpha = (float)(ni - d.lower);
        d.interpolate = d.alpha > 0.f;
        d.down = L > imageLevel ? 1 << (L - imageLevel) : 1;
        d.up = L < imageLevel ? 1 << (imageLevel - L) : 1;
        d.pixH = H;
        d.pixV = V;
        d.startH = h0;
        d.startV = v0;
        d.gridID = L;
        switch (s.storage) {
        case LBM3_STORE_F16: cut_level<__half>(s, L, d, img->p); break;
        case LBM3_STORE_BF16: cut_level<__hip_bfloat16>(s, L, d, img->p); break;
        case LBM3_STORE_F16C: cut_level<f16c>(s, L, d, img->p); break;
        case LBM3_STORE_F64: cut_level<double>(s, L, d, img->p); break;
        default: cut_level<float>(s, L, d, img->p); break;
        }
        HIPCHK(hipGetLastError());
    }
    return 0;
}

int lbm3_section_cut(lbm3_sim *h, int plane, float cut, const lbm3_bounds *bounds, float *out, long long capacity, int *dims)
{
    if (!h || !dims) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    SectionImage si;
    if (const int rc = section_image(s, plane, cut, bounds, si, nullptr)) return rc;
    dims[0] = si.V;
    dims[1] = si.H;
    if (!out) return 0;
    const long long pixels = (long long)si.H * si.V;
    if (capacity < 6 * pixels) return set_error(LBM3_E_ARG, "buffer too small for the section image");
    DBuf<float> img;
    if (const int rc = section_image(s, plane, cut, bounds, si, &img)) return rc;
    launch_cut_finish(img.p, pixels, si.units, s.stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(out, img.p, sizeof(float) * 6 * (size_t)pixels, hipMemcpyDeviceToHost, s.stream));
    HIPCHK(hipStreamSynchronize(s.stream));
    return 0;
}

int lbm3_save_checkpoint(lbm3_sim *h, const char *path)
{
    if (!h || !path) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    for (int L = 0; L < s.levels; ++L)
        if (const int rc = check_level(s, L)) return rc;
    for (int L = 0; L < s.levels; ++L)
        if (const int rc = settle_ghosts(s, s.L[L])) return rc;
    HIPCHK(hipStreamSynchronize(s.stream));
    FILE *fp = fopen(path, "wb");
    if (!fp) return set_error(LBM3_E_ARG, std::string("cannot open checkpoint file: ") + path);
    std::vector<unsigned char> stage;
    bool ok = fwrite(kCheckpointMagic, 1, 8, fp) == 8;
    const int head[3] = {kCheckpointVersion, s.storage, s.levels};
    ok = ok && fwrite(head, sizeof head, 1, fp) == 1 && fwrite(&s.fluidUpdates, sizeof s.fluidUpdates, 1, fp) == 1;
    int rc = 0;
    for (int L = 0; ok && !rc && L < s.levels; ++L) {
        Level &l = s.L[L];
        const CheckpointLevel d = checkpoint_level(l);
        ok = fwrite(&d, sizeof d, 1, fp) == 1 && fwrite(&l.info, sizeof l.info, 1, fp) == 1;
        for (const auto &b : checkpoint_buffers(l, s.storage))
            if (ok && !rc) rc = dump_device(fp, b.first, b.second, stage, s.stream, ok);
        for (const auto &r : l.rotors)
            ok = ok && fwrite(&r.radiansElapsed, sizeof r.radiansElapsed, 1, fp) == 1;
    }
    ok = (fclose(fp) == 0) && ok;
    if (rc) return rc;
    return ok ? 0 : set_error(LBM3_E_ARG, std::string("failed writing checkpoint file: ") + path);
}

int lbm3_load_checkpoint(lbm3_sim *h, const char *path)
{
    if (!h || !path) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    for (int L = 0; L < s.levels; ++L)
        if (const int rc = check_level(s, L)) return rc;
    FILE *fp = fopen(path, "rb");
    if (!fp) return set_error(LBM3_E_ARG, std::string("cannot open checkpoint file: ") + path);
    auto fail = [&](const char *why) {
        fclose(fp);
        return set_error(LBM3_E_ARG, std::string("checkpoint ") + path + ": " + why);
    };
    char magic[8];
    int head[3];
    long long updates = 0;
    if (fread(magic, 1, 8, fp) != 8 || memcmp(magic, kCheckpointMagic, 8) != 0) return fail("not a checkpoint file");
    if (fread(head, sizeof head, 1, fp) != 1 || fread(&updates, sizeof updates, 1, fp) != 1) return fail("truncated header");
    if (head[0] != kCheckpointVersion) return fail("unsupported version");
    if (head[1] != s.storage) return fail("population storage differs from the simulation's");
    if (head[2] != s.levels) return fail("level count differs from the simulation's");
    // read and check every level's shape before anything on the device changes
    std::vector<lbm3_info> infos((size_t)s.levels);
    std::vector<long> at((size_t)s.levels);
    std::vector<char> settled((size_t)s.levels), split((size_t)s.levels);
    for (int L = 0; L < s.levels; ++L) {
        Level &l = s.L[L];
        CheckpointLevel d;
        if (fread(&d, sizeof d, 1, fp) != 1 || fread(&infos[(size_t)L], sizeof(lbm3_info), 1, fp) != 1)
            return fail("truncated level record");
        const CheckpointLevel e = checkpoint_level(l);
        const lbm3_info &I = infos[(size_t)L];
        if (d.N != e.N || d.W != e.W || d.nOpen != e.nOpen || d.nRotors != e.nRotors || I.cellCount != l.info.cellCount ||
            I.cellCountX != l.info.cellCountX || I.cellCountY != l.info.cellCountY || I.cellCountZ != l.info.cellCountZ ||
            I.gridID != l.info.gridID || I.res != l.info.res || I.ox != l.info.ox || I.oy != l.info.oy || I.oz != l.info.oz ||
            I.dtPhys != l.info.dtPhys || I.nu != l.info.nu)
            return fail("grid differs from the simulation's");
        at[(size_t)L] = ftell(fp);
        long skip = 0;
        for (const auto &b : checkpoint_buffers(l, s.storage)) skip += (long)b.second;
        skip += (long)(sizeof(double) * l.rotors.size());
        if (fseek(fp, skip, SEEK_CUR) != 0) return fail("seek failed");
        settled[(size_t)L] = d.openSettled != 0;
        split[(size_t)L] = d.split != 0;
    }
    // the file ends where the last level's data ends (a short file changes nothing)
    const long end = ftell(fp);
    if (fseek(fp, 0, SEEK_END) != 0 || ftell(fp) != end) return fail("file size does not match its records");
    // decide each level's open-cell fusion now, as the saved simulation had at
    // its first run: a condition saved as pending is then completed by the next
    // step's open-cell kernel exactly as it would have been there
    for (int L = 0; L < s.levels; ++L)
        if (!s.L[L].openFusionChecked) {
            s.L[L].openSettled = true;       // the state the load replaces needs no completion
            if (const int rc = prepare_open_fusion(s, L)) { fclose(fp); return rc; }
        }
    // a condition saved as pending covers the entries the saving simulation
    // left to its open-cell kernel: group the levels the same way
    for (int L = 0; L < s.levels; ++L) {
        Level &l = s.L[L];
        if (settled[(size_t)L] || !l.fusedOpen || split[(size_t)L] == (l.nSepEntries > 0)) continue;
        if (const int rc = settle_open(s, L)) { fclose(fp); return rc; }
        (s.tuneChosen ? s.tune.openSplit : s.ownSplit) = split[(size_t)L] ? 1 : 0;
        l.openFusionChecked = false;
        if (const int rc = prepare_open_fusion(s, L)) { fclose(fp); return rc; }
    }
    std::vector<unsigned char> stage;
    for (int L = 0; L < s.levels; ++L) {
        Level &l = s.L[L];
        if (fseek(fp, at[(size_t)L], SEEK_SET) != 0) return fail("seek failed");
        bool ok = true;
        for (const auto &b : checkpoint_buffers(l, s.storage)) {
            const int rc = load_device(fp, b.first, b.second, stage, s.stream, ok);
            if (rc) { fclose(fp); return rc; }
            if (!ok) return fail("truncated level data");
        }
        for (auto &r : l.rotors)
            if (fread(&r.radiansElapsed, sizeof r.radiansElapsed, 1, fp) != 1) return fail("truncated rotor state");
        // the step state of the level's info; the rest comes from the case it was built from
        l.info.iterationsFinished = infos[(size_t)L].iterationsFinished;
        l.info.iterationsSinceTrackerReset = infos[(size_t)L].iterationsSinceTrackerReset;
        l.info.esotwistFlipper = infos[(size_t)L].esotwistFlipper;
        l.openSettled = settled[(size_t)L] != 0;
        l.ghostsStale = false;
    }
    fclose(fp);
    s.fluidUpdates = updates;
    return check_hip(hipStreamSynchronize(s.stream), "checkpoint upload");
}

int lbm3_export_vtk(lbm3_sim *h, const char *path)
{
    if (!h || !path) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    long long total = 0;
    for (int L = 0; L < s.levels; ++L) {
        if (const int rc = check_level(s, L)) return rc;
        if (const int rc = settle_open(s, L)) return rc;
        total += s.L[L].N;
    }
    // the nine fields per cell, level by level (exportVTK.h:33-112)
    std::vector<std::vector<float>> fields((size_t)s.levels);
    for (int L = 0; L < s.levels; ++L) {
        Level &l = s.L[L];
        DBuf<float> d;
        HIPCHK(d.alloc(9LL * (l.N > 0 ? l.N : 1)));
        const bool flip = l.info.esotwistFlipper != 0;
        const Topology t = topo_of(l);
        switch (s.storage) {
        case LBM3_STORE_F16: launch_vtk_fields<__half>(reinterpret_cast<const __half *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.codec, flip, l.geom, s.C.rhoPhys, d.p, s.stream); break;
        case LBM3_STORE_BF16: launch_vtk_fields<__hip_bfloat16>(reinterpret_cast<const __hip_bfloat16 *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.codec, flip, l.geom, s.C.rhoPhys, d.p, s.stream); break;
        case LBM3_STORE_F16C: launch_vtk_fields<f16c>(reinterpret_cast<const f16c *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.codec, flip, l.geom, s.C.rhoPhys, d.p, s.stream); break;
        case LBM3_STORE_F64: launch_vtk_fields<double>(reinterpret_cast<const double *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.codec, flip, l.geom, s.C.rhoPhys, d.p, s.stream); break;
        default: launch_vtk_fields<float>(reinterpret_cast<const float *>(l.f.p), t, l.wallMap.p, l.wallData.p, s.codec, flip, l.geom, s.C.rhoPhys, d.p, s.stream); break;
        }
        HIPCHK(hipGetLastError());
        fields[(size_t)L].resize(9 * (size_t)l.N);
        if (l.N > 0)
            HIPCHK(hipMemcpyAsync(fields[(size_t)L].data(), d.p, sizeof(float) * fields[(size_t)L].size(), hipMemcpyDeviceToHost,
                                  s.stream));
        HIPCHK(hipStreamSynchronize(s.stream));
    }
    // legacy ASCII polydata, one vertex per stored cell (exportVTK.h:118-156)
    FILE *fp = fopen(path, "w");
    if (!fp) return set_error(LBM3_E_ARG, std::string("cannot open VTK file: ") + path);
    auto fl = [](float v) {
        char b[32];
        snprintf(b, sizeof b, "%.9g", (double)v);
        return std::string(b);
    };
    std::string o;
    o.reserve(1 << 20);
    auto flush = [&](bool force) {
        if (force || o.size() > (1u << 20)) { fwrite(o.data(), 1, o.size(), fp); o.clear(); }
    };
    o += "# vtk DataFile Version 3.0\nLBM snapshot; coordinates in mm; grid count " + std::to_string(s.levels) + "\n";
    o += "ASCII\nDATASET POLYDATA\nPOINTS " + std::to_string(total) + " float\n";
    auto each = [&](int field, auto &&emit) {
        for (int L = 0; L < s.levels; ++L) {
            const long long N = s.L[L].N;
            const float *F = fields[(size_t)L].data() + (size_t)field * (size_t)N;
            for (long long c = 0; c < N; ++c) { emit(L, F, c); flush(false); }
        }
    };
    for (int L = 0; L < s.levels; ++L) {
        const long long N = s.L[L].N;
        const float *F = fields[(size_t)L].data();
        for (long long c = 0; c < N; ++c) {
            o += fl(F[c]) + ' ' + fl(F[N + c]) + ' ' + fl(F[2 * N + c]) + '\n';
            flush(false);
        }
    }
    o += "VERTICES " + std::to_string(total) + ' ' + std::to_string(2 * total) + '\n';
    for (long long c = 0; c < total; ++c) { o += "1 " + std::to_string(c) + '\n'; flush(false); }
    o += "POINT_DATA " + std::to_string(total) + "\nSCALARS wall int 1\nLOOKUP_TABLE default\n";
    each(3, [&](int, const float *F, long long c) { o += std::to_string((int)F[c]) + '\n'; });
    o += "VECTORS velocity_m_s float\n";
    for (int L = 0; L < s.levels; ++L) {
        const long long N = s.L[L].N;
        const float *F = fields[(size_t)L].data();
        for (long long c = 0; c < N; ++c) {
            o += fl(F[4 * N + c]) + ' ' + fl(F[5 * N + c]) + ' ' + fl(F[6 * N + c]) + '\n';
            flush(false);
        }
    }
    o += "SCALARS pressure_Pa float 1\nLOOKUP_TABLE default\n";
    each(7, [&](int, const float *F, long long c) { o += fl(F[c]) + '\n'; });
    o += "SCALARS grid_id int 1\nLOOKUP_TABLE default\n";
    each(0, [&](int L, const float *, long long) { o += std::to_string((int)s.L[L].info.gridID) + '\n'; });
    o += "SCALARS grid_resolution_mm float 1\nLOOKUP_TABLE default\n";
    each(0, [&](int L, const float *, long long) { o += fl(s.L[L].info.res) + '\n'; });
    o += "SCALARS interface_overlap int 1\nLOOKUP_TABLE default\n";
    each(8, [&](int, const float *F, long long c) { o += std::to_string((int)F[c]) + '\n'; });
    flush(true);
    const bool ok = fclose(fp) == 0;
    return ok ? 0 : set_error(LBM3_E_ARG, std::string("failed writing VTK file: ") + path);
}

int lbm3_flow_report(lbm3_sim *h, int plane, float cut, const lbm3_bounds *bounds, double *out7)
{
    if (!h || !out7) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    SectionImage si;
    DBuf<float> img;
    if (const int rc = section_image(s, plane, cut, bounds, si, &img)) return rc;
    const long long pixels = (long long)si.H * si.V;
    std::vector<float> host((size_t)(6 * pixels));
    HIPCHK(hipMemcpyAsync(host.data(), img.p, sizeof(float) * host.size(), hipMemcpyDeviceToHost, s.stream));
    HIPCHK(hipStreamSynchronize(s.stream));
    // the reduction over the fluid pixels (flowReportFunctions.h:266-297), FP64 sums
    double velocity = 0.0, densityVelocity = 0.0, momentum = 0.0, dRhoSum = 0.0, kinetic = 0.0;
    long long count = 0;
    for (long long p = 0; p < pixels; ++p) {
        const float *v = &host[(size_t)(6 * p)];
        if (!(v[4] < 0.5f)) continue;
        const double d = v[0];
        const double u = plane == LBM3_PLANE_XY ? v[3] : (plane == LBM3_PLANE_ZY ? v[1] : v[2]);
        const double rhoU = (1.0 + d) * u;
        velocity += u;
        densityVelocity += d * u;
        momentum += rhoU * std::fabs(u);
        dRhoSum += d;
        kinetic += 0.5 * rhoU * u * u;
        ++count;
    }
    for (int k = 0; k < 7; ++k) out7[k] = 0.0;
    if (count == 0) return 0;
    // units of the image level (:299-335): pixels of equal area
    const lbm3_info &R = s.L[si.imageLevel].info;
    const double px = double(R.res) / 1000.0, area = px * px, vel = px / double(R.dtPhys);
    const double pres = double(s.C.rhoPhys) * vel * vel / 3.0;
    const double massFlux = double(s.C.rhoPhys) * area * vel;
    out7[0] = velocity / double(count) * vel;                   // area-averaged normal velocity [m/s]
    out7[1] = (velocity + densityVelocity) * massFlux;          // mass flow [kg/s]
    out7[2] = momentum * massFlux * vel;                        // momentum thrust [N]
    out7[3] = dRhoSum / double(count) * pres;                   // area-averaged pressure [Pa]
    out7[4] = densityVelocity * area * pres * vel;              // pressure power [W]
    out7[5] = kinetic * massFlux * vel * vel;                   // normal kinetic power [W]
    out7[6] = double(count) * double(R.res) * double(R.res);    // area [mm^2]
    return 0;
}

int lbm3_update_tracker(lbm3_sim *h, double *walls, int nWalls, double *rotors, int nRotors, double *open, int nOpen)
{
    if (!h) return set_error(LBM3_E_ARG, "null sim");
    if (nWalls < 0 || nWalls > LBM3_MAX_BODIES || nRotors < 0 || nRotors > LBM3_MAX_ROTORS || nOpen < 0)
        return set_error(LBM3_E_ARG, "bad tracker sizes");
    if ((nWalls && !walls) || (nRotors && !rotors) || (nOpen && !open)) return set_error(LBM3_E_ARG, "null tracker output");
    Sim &s = h->s;
    for (int L = 0; L < s.levels; ++L) {
        if (const int rc = check_level(s, L)) return rc;
        if (s.L[L].info.iterationsSinceTrackerReset <= 0) return set_error(LBM3_E_ARG, "no time step since the last reset");
    }
    for (int i = 0; i < 6 * nWalls; ++i) walls[i] = 0.0;
    for (int i = 0; i < 6 * nRotors; ++i) rotors[i] = 0.0;
    const double zero[3] = {0.0, 0.0, 0.0};
    for (int L = 0; L < s.levels; ++L) {
        const lbm3_info &I = s.L[L].info;
        // time average over the period, then physical units (convertToPhysicalForce,
        // cellFunctions.h:296-301); torques about the origin come in N mm -> N m
        const double dx = double(I.res) / 1000.0;
        const double f = double(s.C.rhoPhys) * dx * dx * dx * dx / (double(I.dtPhys) * double(I.dtPhys)) /
                         double(I.iterationsSinceTrackerReset);
        double tmp[6 * LBM3_MAX_BODIES];
        if (nWalls && s.C.trackWallForce) {
            if (const int rc = lbm3_wall_forces(h, L, zero, nWalls, tmp)) return rc;
            for (int b = 0; b < nWalls; ++b)
                for (int k = 0; k < 6; ++k) walls[6 * b + k] += tmp[6 * b + k] * f * (k < 3 ? 1.0 : 0.001);
        }
        for (int r = 0; r < nRotors && s.C.trackRotorForce; ++r) {
            if (r >= (int)s.L[L].rotors.size()) continue;
            if (const int rc = lbm3_rotor_forces(h, L, r, tmp)) return rc;
            for (int k = 0; k < 6; ++k) rotors[6 * r + k] += tmp[k] * f * (k < 3 ? 1.0 : 0.001);
        }
    }
    for (int b = 0; b < nOpen; ++b)
        if (const int rc = lbm3_open_boundary_stats(h, b, open + 7 * b)) return rc;
    // the reset at the end of updateTracker (trackerFunctions.h:476-486)
    if (const int rc = lbm3_reset_wall_forces(h)) return rc;
    return lbm3_reset_open_boundary_stats(h);
}

static int check_rotor(lbm3_sim *h, int level, int rotor)
{
    if (!h) return set_error(LBM3_E_ARG, "null sim");
    if (const int rc = check_level(h->s, level)) return rc;
    if (rotor < 0 || rotor >= (int)h->s.L[level].rotors.size()) return set_error(LBM3_E_ARG, "no such rotor on this level");
    return 0;
}

int lbm3_set_rotor(lbm3_sim *h, int level, int rotor, float radiansPerSecond, int axis, float ox, float oy, float oz)
{
    if (const int rc = check_rotor(h, level, rotor)) return rc;
    if (axis < LBM3_AXIS_NONE || axis > LBM3_AXIS_Z) return set_error(LBM3_E_ARG, "bad rotor axis");
    RotorDev &d = h->s.L[level].rotors[rotor].dev;
    d.radiansPerSecond = radiansPerSecond;
    d.axis = axis;
    d.ox = ox; d.oy = oy; d.oz = oz;
    return upload_rotors(h->s, level);
}

int lbm3_rotor_info(lbm3_sim *h, int level, int rotor, double *out)
{
    if (const int rc = check_rotor(h, level, rotor)) return rc;
    if (!out) return set_error(LBM3_E_ARG, "null argument");
    const Level::Rotor &R = h->s.L[level].rotors[rotor];
    const RotorDev &d = R.dev;
    const double v[12] = {d.res, d.xMin, d.yMin, d.zMin, d.xMax, d.yMax, d.zMax, (double)d.cx, (double)d.cy, (double)d.cz,
                          R.radiansElapsed, (double)d.nonZero};
    memcpy(out, v, sizeof v);
    return 0;
}

int lbm3_rotor_forces(lbm3_sim *h, int level, int rotor, double *out)
{
    if (const int rc = check_rotor(h, level, rotor)) return rc;
    if (!out) return set_error(LBM3_E_ARG, "null argument");
    Sim &s = h->s;
    const Level::Rotor &R = s.L[level].rotors[rotor];
    const RotorDev &d = R.dev;
    for (int i = 0; i < 6; ++i) out[i] = 0.0;
    const int nz = d.nonZero;
    if (nz == 0) return 0;
    const int nb = rotor_force_blocks(nz);
    // a buffer of its own: another thread may be in a sum that uses `partial`
    std::lock_guard<std::mutex> kept(s.keptLock);
    if (s.rotorSums.n < 6LL * nb) HIPCHK(s.rotorSums.alloc(6LL * nb));
    launch_rotor_force(d, R.index.p, s.rotorSums.p, s.stream);
    HIPCHK(hipGetLastError());
    std::vector<double> host((size_t)nb * 6);
    HIPCHK(hipMemcpyAsync(host.data(), s.rotorSums.p, sizeof(double) * host.size(), hipMemcpyDeviceToHost, s.stream));
    HIPCHK(hipStreamSynchronize(s.stream));
    for (int b = 0; b < nb; ++b)
        for (int k = 0; k < 6; ++k) out[k] += host[(size_t)b * 6 + k];
    return 0;
}

int lbm3_copy_probe(long long bytes, int reps, double *msPerCopy)
{
    if (bytes <= 0 || reps <= 0 || !msPerCopy) return set_error(LBM3_E_ARG, "bad probe arguments");
    DBuf<unsigned char> a, b;
    HIPCHK(a.alloc(bytes));
    HIPCHK(b.alloc(bytes));
    HIPCHK(hipMemset(a.p, 1, (size_t)bytes));
    hipEvent_t e0, e1;
    HIPCHK(hipEventCreate(&e0));
    HIPCHK(hipEventCreate(&e1));
    launch_copy(a.p, b.p, bytes, nullptr);
    HIPCHK(hipEventRecord(e0, nullptr));
    for (int r = 0; r < reps; ++r) launch_copy(a.p, b.p, bytes, nullptr);
    HIPCHK(hipEventRecord(e1, nullptr));
    HIPCHK(hipEventSynchronize(e1));
    float ms = 0.f;
    HIPCHK(hipEventElapsedTime(&ms, e0, e1));
    *msPerCopy = ms / reps;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return check_hip(hipGetLastError(), "copy probe");
}

int lbm3_collide_cells_f32(float *f, int n, const lbm3_bc *bc, float nu) { return collide_cells<float>(f, n, bc, nu); }
int lbm3_collide_cells_f64(double *f, int n, const lbm3_bc *bc, double nu) { return collide_cells<double>(f, n, bc, nu); }

} // extern "C"
