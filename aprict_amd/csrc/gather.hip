// gather.hip -- matched adjoint of the Siddon forward projector for views
// whose detector v axis is parallel to z and whose u axis has no z component
// (circular and helical scans with upright panels), computed as a gather over
// voxels: no atomics, every voxel sum accumulated in FP64 registers.
//
// Geometry.  For such a view all rays through detector (sub-)column q lie in
// one vertical plane through the source: they share their x-y line, and
// along that line, parametrised by the horizontal distance h from the source,
// ray t has height z_t(h) = sz + h * dz_t / l, where dz_t is the height of
// its detector point above the source and l the horizontal source-pixel
// distance.  Order the rays by height (dz_t = dz0 + t dzs, dzs > 0).  The
// column's line crosses x-y cell (i, j) over [h_a, h_b]; the Siddon length of
// ray t in voxel (i, j, k) is sec_t times the measure of the h in [h_a, h_b]
// where k <= z_t(h) < k + 1.  With
//     F_t(k) = |{h in [h_a, h_b] : z_t(h) < k}|   and
//     G(k)   = sum_t yhat_t F_t(k),   yhat_t = y_t sec_t,
// the adjoint's contribution of the column to voxel k is G(k+1) - G(k).
// A ray is below plane k at h where t < kappa(h) = ((k - sz) l / h - dz0) / dzs.
// At the chord's far end h_b the first u = int(kappa) + 1 rays are.  Above the
// source (k > sz) rays rise: those u are below the plane all along the chord, and
// ray u, if it crosses the plane within the chord, is below it up to there.
// At or below the source they fall: of those u, ray u - 1 may be above the plane
// up to its crossing.  With P the exclusive prefix sum of yhat over t and x' the
// part of the chord before the crossing, both read
//     G(k) = dh (P[u] + x' (P[u'] - P[u])),   u' = u + 1 or u - 1,
// dh = h_b - h_a.  The other rays do not cross the plane within the chord when
// the rays of a column are further apart in z than one of them climbs within a
// cell; (cell, column) pairs where that is not certain go on along the rows until
// a ray does not cross.
//
// A pre-pass (k_gather_prep) writes, per view and sub-column, the FP64
// prefix sums P of the sec-weighted sinogram column (in z order), the
// column's x-y crossing constants (the forward's col_setup, so the cell
// boundaries along h are the forward's own FP32 values) and, per view, the
// reciprocal heights 1/dz_t, each at the entry u' that its crossing reads.  The
// main kernel (k_gather_adjoint) gives each workgroup (8 waves) a tile of 8 x 8
// x-y cells and 64 or 128 planes or of 8 x 4 cells and 192; each wave owns the
// cells of one x, each lane one boundary per 64 in z.  The work comes in items, a
// view and a group of the columns crossing the tile: while the workgroup
// works on one item, the next one's prefix window is loaded straight into
// the other of two LDS buffers (16-byte loads).  Per item each wave derives
// its (cell, column) pairs one per lane, then for every pair every lane
// evaluates G at its boundaries: the row (one FP64 FMA, the integer conversion,
// a clamp, addresses), three LDS reads, and five FP64 operations, of which the
// crossing is one FMA in units of the chord, clamped to [0, 1] by its clamp
// modifier.  The voxel values are differences of neighbouring boundaries, scaled
// and added to the volume once at the end.  Tiles run in blocks of 4 x 8, so that
// the workgroups on one XCD at one time share their views' prefix windows through
// its L2.  A volume with too few tiles to fill the GPU gets its views split
// between workgroups, whose FP64 partial sums k_gather_combine adds in order.
//
// Precision: the sums P and the accumulators are FP64 in units of a cell's chord, so
// a voxel keeps about 2^-53 of the rows below it in its columns, whatever their
// distance: half of the rows at 1 and half at 1e-8, 1000 voxels from the source, dim
// voxels are off by 1.3e-7 of their own terms.  (The same evaluation once per cell
// face, of chords measured from the source, reads 16 bytes instead of 24 and needs 7
// instructions instead of 11, but lost 1.5e-4 there: its sums are 1000 times as large.
// It took 128 ms at 512^3 x 720 views of 768^2, this form 118.)  The row and the crossing
// of a plane are formed in FP64 from the FP32 cell boundaries, the forward's own.  A row
// of rays that neither rise nor fall (row_flat) counts as a falling one, below the planes
// at its height: a ray in a z plane belongs to the voxel below, as in the forward.
#include <algorithm>
#include <mutex>

#include "column.h"
#include "gather.h"

namespace {

constexpr int kXcdG = 8;
constexpr int kGRowMax = 2048;     // rows of a window (at most)
constexpr int kGMaxCols = 16;      // columns staged at once
constexpr int kGW = 8;             // waves of a workgroup: one per cell of a tile along x
// cells of a tile along y (a wave's): 8 on tiles of 64 or 128 planes, 4 on taller ones
constexpr int g_cells(int kJ) { return kJ <= 2 ? 8 : 4; }

// Bytes of an LDS window buffer (two per workgroup): two workgroups share a CU, or (kTall)
// one takes it, for detectors whose rows would leave the others only a few columns at a time.
constexpr int g_win_bytes(bool kTall) { return kTall ? 57344 : 28672; }

// per-(view, sub-column) record
struct GCol {
    float r[2], c[2], P0[2];   // x-y crossing parameters along h - hc (col_setup)
    int32_t sg[2], ifix[2];
    float hs, hd;              // source and pixel along h - hc (hd <= hs: no ray meets the chunk)
    double l, hc;              // horizontal source-pixel distance, closest approach to the chunk centre
    double lods;               // l / dzs
    float pad[2];
};
static_assert(sizeof(GCol) == 80, "GCol layout");

__host__ __device__ inline size_t g_align(size_t x) { return (x + 255) & ~size_t(255); }

// A row before the first ray and rows past the last one are padded (P: 0 and the total,
// 1/dz: 0) far enough that the window loads (whole 256-byte chunks up to the one with row
// NT + 2) stay inside the row: kGPad >= 32 + 3.
constexpr uint32_t kGPad = 40;

struct GLayout {
    size_t views, count, cols, pref, iz, total;
    uint32_t cs;   // entries per column of P and per view of 1/dz: NT + kGPad
};

__host__ __device__ inline GLayout g_layout(uint32_t V, uint32_t NQ, uint32_t NT) {
    GLayout L;
    L.cs = NT + kGPad;
    L.views = 0;
    L.count = g_align((size_t)V * sizeof(GView));
    L.cols = L.count + 256;
    // one spare record: the record loads copy whole 256-byte chunks
    L.pref = L.cols + g_align(((size_t)V * NQ + 4) * sizeof(GCol));
    L.iz = L.pref + g_align((size_t)V * NQ * L.cs * sizeof(double));
    L.total = L.iz + g_align((size_t)V * L.cs * sizeof(double));
    return L;
}

// Room for partial sums behind the tables, offered to split the views of a
// volume with few tiles between workgroups: twice the tables, at most 64 MiB,
// none for a handful of views.
inline uint64_t g_partial_bytes(uint32_t V, uint64_t tables) {
    return V < 16 ? 0 : (tables < (32ull << 20) ? 2 * tables : (64ull << 20));
}

struct GCfg {
    uint32_t V, nu, nv, ssu, ssv, NQ, NT, cs;
    int64_t s0, s1, s2;   // sinogram element strides
};

// 1 / x for a nonzero finite x: the hardware reciprocal and two Newton steps
// (about 1e-16 relative)
__device__ __forceinline__ double g_rcp64(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = fma(fma(-x, y, 1.0), y, y);
    return fma(fma(-x, y, 1.0), y, y);
}

// v moved between lanes by a DPP control, 0 where no lane's value arrives
template <int kCtrl, int kRows>
__device__ __forceinline__ double g_dpp(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, kRows, 0xF, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, kRows, 0xF, false);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// inclusive sums over the lanes in order (all 64 active): within rows of 16 by shifts
// of 1, 2, 4 and 8, then row 0's and row 2's last sum to the next row, then that of
// lane 31 to the upper half.  Register moves: with six exchanges through LDS the
// pre-pass took 27.8 us for 90 views of 96^2, not 24.6, and 4.4 ms for 720 of 768^2, not 3.4.
__device__ __forceinline__ double g_scan(double v) {
    v += g_dpp<0x111, 0xF>(v);   // row_shr:1
    v += g_dpp<0x112, 0xF>(v);
    v += g_dpp<0x114, 0xF>(v);
    v += g_dpp<0x118, 0xF>(v);
    v += g_dpp<0x142, 0xA>(v);   // row_bcast:15, rows 1 and 3
    v += g_dpp<0x143, 0xC>(v);   // row_bcast:31, rows 2 and 3
    return v;
}

// ---------------------------------------------------------------------------
// pre-pass: one wave per (view, sub-column)
// ---------------------------------------------------------------------------
template <typename Tp>
__global__ __launch_bounds__(256) void k_gather_prep(RayCfg rc, GCfg gc, const ap_proj_spec* __restrict__ specs,
                                                     const Tp* __restrict__ sino, GView* __restrict__ gviews,
                                                     GCol* __restrict__ gcols, double* __restrict__ pref,
                                                     double* __restrict__ izt) {
    const int lane = threadIdx.x & 63;
    const uint64_t w = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= (uint64_t)gc.V * gc.NQ) return;
    const uint32_t p = (uint32_t)(w / gc.NQ), q = (uint32_t)(w % gc.NQ);
    GView gv;
    const bool ok = gather_view(rc, specs, p, gc.ssu, gc.ssv, gc.NT, gv);
    if (!ok) {
        if (q == 0 && lane == 0) gviews[p] = gv;
        return;
    }
    const ViewRays vr = make_view_rays(rc, specs, p);
    const uint32_t j = q / gc.ssu;
    const float ju = (float)j + sub_offset_g(q % gc.ssu, gc.ssu);
    Col2D C;
    const bool hit = col_setup(vr, rc.lo, rc.hi, ju, C);
    double* P = pref + (size_t)w * gc.cs;
    const uint32_t NT = gc.NT;
    double carry = 0.0;
    // rows in z order, 64 at a time (coalesced): inclusive wave scan plus the
    // running total of the previous chunks; P[t] is the exclusive prefix
    if (lane == 0) P[0] = 0.0;
    for (uint32_t t0 = 0; t0 + 1 < gc.cs; t0 += 64) {
        const uint32_t t = t0 + (uint32_t)lane;
        double yv = 0.0;
        if (hit && t < NT) {
            const uint32_t sr = gv.flip ? NT - 1 - t : t;
            const uint32_t k = sr / gc.ssv;
            const float kv = (float)k + sub_offset_g(sr % gc.ssv, gc.ssv);
            const double m = fma((double)kv, C.z.dm, C.z.m0);
            const float mf = (float)m;
            const float y = to_f32(sino[(int64_t)p * gc.s0 + (int64_t)j * gc.s1 + (int64_t)k * gc.s2]);
            yv = (double)(y * __builtin_amdgcn_sqrtf(__builtin_fmaf(mf, mf, 1.f)));
        }
        // exclusive sums from the lane below (the inclusive one minus the row's own
        // term would round once more)
        const double incl = g_scan(yv), below = __shfl_up(incl, 1, 64);
        if (t + 1 < gc.cs) P[t + 1] = carry + (lane ? below : 0.0);
        carry += __shfl(incl, 63, 64);
    }
    if (lane == 0) {
        GCol g;
        for (int a = 0; a < 2; a++) {
            g.r[a] = hit ? C.r[a] : 0.f;
            g.c[a] = hit ? C.c[a] : 0.f;
            g.P0[a] = hit ? C.P0[a] : 0.f;
            g.sg[a] = hit ? C.sg[a] : 0;
            g.ifix[a] = hit ? C.ifix[a] : 0;
        }
        g.hs = hit ? C.hs : 0.f;
        g.hd = hit ? C.hd : 0.f;   // hd <= hs: empty
        const double qx = vr.Q00[0] + (double)ju * vr.U[0] - vr.S[0];
        const double qy = vr.Q00[1] + (double)ju * vr.U[1] - vr.S[1];
        const double l = hit ? sqrt(qx * qx + qy * qy) : 1.0;
        g.l = l;
        g.hc = hit ? C.z.hc : 0.0;
        g.pad[0] = g.pad[1] = 0.f;
        g.lods = l / (fabs(vr.V[2]) / (double)gc.ssv);
        gcols[w] = g;
    }
    // once per view: the number of rows whose ray does not rise (dz <= 0: those before the
    // first rising one, since dz grows along the z order), and 1/dz, at the entry of P
    // that the evaluation of a crossing reads beside the plane's own, u': a falling ray t's at
    // t + 1 (the sum without it), a rising ray's at t + 2 (the sum with it).
    if (q == 0) {
        auto height = [&](uint32_t t) -> double { return gather_height(vr, gv.flip, NT, gc.ssv, t); };
        uint32_t nfall = 0;
        for (uint32_t b = 0; b < NT; b += 64) {
            const uint32_t t = b + (uint32_t)lane;
            nfall += (uint32_t)__popcll(__ballot(t < NT && ((int)t == gv.flat || !(height(min(t, NT - 1)) > 0.0))));
        }
        for (uint32_t r = (uint32_t)lane; r < gc.cs; r += 64) {
            const uint32_t t = r <= nfall ? r - 1 : r - 2;   // the ray of entry r (r = 0 and the gap: none)
            double v = 0.0;
            if (r > 0 && r != nfall + 1 && t < NT) {
                // a flat row crosses no plane: at that of the source's own height, 0 says so
                const double dz = height(t);
                v = (int)t != gv.flat && dz != 0.0 ? 1.0 / dz : 0.0;
            }
            izt[(size_t)p * gc.cs + r] = v;
        }
        if (lane == 0) gviews[p] = gv;
    }
}

// ---------------------------------------------------------------------------
// main kernel
// ---------------------------------------------------------------------------
// Tiles are taken in blocks of kSTX x kSTY (x, y) tiles of one z layer: the
// workgroups that run at the same time on one XCD cover a compact block of
// cells, whose views' prefix windows they share through that XCD's L2.
constexpr uint32_t kSTX = 4, kSTY = 8, kST = kSTX * kSTY;

struct GTile {
    uint32_t ntx, nty, ntz;   // tiles along x, y, z
    uint32_t nsx, nsy;        // tile blocks along x, y
    uint32_t total, per_xcd;  // block slots (ntz nsx nsy kST slices), slots per XCD
    uint32_t slices, vps;     // view slices, views per slice (the last ones may have fewer or none)
};

// integer part of x >= 0 (0 or less for x < 0), saturating: one instruction
__device__ __forceinline__ int cvt_int(double x) {
    int r;
    asm("v_cvt_i32_f64 %0, %1" : "=v"(r) : "v"(x));
    return r;
}
// x clamped to [1, hi]
__device__ __forceinline__ int g_row(int x, int hi) {
    int r;
    asm("v_med3_i32 %0, %1, 1, %2" : "=v"(r) : "v"(x), "s"(hi));
    return r;
}
__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }

__device__ __forceinline__ double g_dbl(float lo, float hi) {
    return __longlong_as_double((long long)(((uint64_t)__float_as_uint(hi) << 32) | __float_as_uint(lo)));
}

// prefix window of one view for the tile (views taken 64 at a time, one per lane)
struct GWin {
    int qlo, qhi, tlo, W;   // columns [qlo, qhi], rows tlo .. tlo + W - 1 of P (qlo > qhi: nothing)
    float mg;               // slack of the corner projections, in columns
    int ncg;                // columns per staging group
};

// a view's parameters, as wave-uniform values
struct GVu {
    float sz, sx, sy;
    float ax, ay, bx, by;
    float szlo;   // the source height is sz + szlo (FP64 crossings use both)
    double kb;    // 2 + kappa of the plane through the source: 2 - dz0 / dzs
};

// One workgroup of kGW waves of kC cells each per tile of 8 x kC cells and 64 kJ planes.
// What bounds it: latency and vector issue together.  A pair is a chain of LDS reads (its
// record, then P and 1 / dz at the rows) and about 11 instructions per 64 boundaries; a
// setup pass of about 150 serves a wave's 6 to 12 pairs of a view.  8 waves of 8 cells in
// two workgroups a CU on tiles of 128 planes, against 16 waves of 4 cells in one workgroup
// on 256 planes: half the setup passes, and barriers that stop half the CU (with 14
// instructions per 64 boundaries: 512^3, 720 views of 768^2, 139 against 151 ms; a helical
// gradient step at 161 x 149 x 127, 211 views of 230 x 170, 3.45 and 4.16 ms; 64^3, 90 views
// of 96^2, 101 and 120 us).  One form for both sides of the source, whose row of the other
// side is a lane's constant away, instead of one each by selects: 139 -> 126 ms, 3.45 ->
// 3.19, 101 -> 97 us.  Flat rows among the falling ones instead of a sum of their own, looked
// for at every pair: 126 -> 118 ms, 3.19 -> 3.00, 97 -> 94 us.
template <typename Tv, typename Tm, int kJ, bool kTall>
__global__ __launch_bounds__(kGW * 64, kTall ? 2 : 4) void k_gather_adjoint(
    RayCfg rc, GCfg gc, GTile tl, const GView* __restrict__ gviews, const GCol* __restrict__ gcols,
    const double* __restrict__ pref, const double* __restrict__ izt, double scale, Tv* __restrict__ vol,
    int64_t vsx, int64_t vsy, int64_t vsz, const Tm* __restrict__ mult, int64_t msx, int64_t msy, int64_t msz,
    double* __restrict__ partial, uint32_t* __restrict__ left) {
    constexpr int kGWin = g_win_bytes(kTall);
    constexpr int kC = g_cells(kJ), kNQc = (kGW + 1) * (kC + 1);
    // Two staging buffers: while the workgroup works on one (view, column group)
    // item from one buffer, the next item's window is loaded into the other.
    // A buffer holds the item's window -- rows tlo .. tlo + Wp - 1 of 1/dz, then
    // the same rows of P for each column of the group --, the group's column
    // records and the projections of the tile's cell corners.
    struct GBuf {
        double win[kGWin / 8];
        GCol cols[kGMaxCols];
        float qc[(kNQc + 3) & ~3];
    };
    __shared__ __align__(16) GBuf Buf0;
    __shared__ __align__(16) GBuf Buf1;
    __shared__ GWin Win[64];
    // the batch's view parameters, one 32-byte record per view: sz, sx, sy, szlo,
    // ax, ay, bx, by -- read from LDS at the start of a step, so that no step waits
    // on a global load of its view record
    __shared__ __align__(16) float Vw[64 * 8];
    __shared__ double Vk[64];   // the views' kb
    // per-wave (cell, column) pair records of the setup pass, one per lane: l / dh, H,
    // alpha_b (FP64), dh = h_b - h_a and the column's byte offset in the window.  (As
    // scalars from the lanes they cost 12 instructions a pair more, and operations with
    // two scalar operands a move each: 155 against 140 ms at 512^3 x 720, 768^2.)
    __shared__ __align__(16) double Rec[kGW * 64 * 4];
    // the lane from the hardware's count, not from the thread index, which would stay in
    // a register of its own; the wave as a scalar: its cells are scalars then
    const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (left) {
        // number of views this kernel does not take (for the general adjoint's early
        // exit); where it takes none (tilted panels) there is nothing to add, and the
        // partial sums are not read
        if (blockIdx.x == 0 && wave == 0) {
            uint32_t n = 0;
            for (uint32_t p = 0; p < gc.V; p += 64)
                n += (uint32_t)__popcll(__ballot(p + lane < gc.V && !gviews[min(p + lane, gc.V - 1)].ok));
            if (lane == 0) *left = n;
        }
        bool any = false;
        for (uint32_t p = 0; p < gc.V && !any; p += 64)
            any = __ballot(p + lane < gc.V && gviews[min(p + lane, gc.V - 1)].ok) != 0;
        if (!any) return;
    }
    const uint32_t L = blockIdx.x;
    const uint32_t logical = (L % kXcdG) * tl.per_xcd + L / kXcdG;
    if (logical >= tl.total) return;
    const uint32_t per_layer = tl.nsx * tl.nsy * kST;
    const uint32_t slice = logical / (per_layer * tl.ntz), lrem = logical % (per_layer * tl.ntz);
    const uint32_t tz = lrem / per_layer, r = lrem % per_layer;
    const uint32_t st = r / kST, w = r % kST;
    const uint32_t tx = (st % tl.nsx) * kSTX + w % kSTX, ty = (st / tl.nsx) * kSTY + w / kSTX;
    if (tx >= tl.ntx || ty >= tl.nty) return;   // a slot of a block past the edge
    const int X0 = rc.lo[0] + (int)tx * kGW, Y0 = rc.lo[1] + (int)ty * kC;
    const int X1 = min(X0 + kGW, rc.hi[0]), Y1 = min(Y0 + kC, rc.hi[1]);
    const int z0 = rc.lo[2] + (int)tz * 64 * kJ;
    const int z1 = min(z0 + 64 * kJ, rc.hi[2]);
    const uint32_t pbeg = slice * tl.vps, pend = min(gc.V, pbeg + tl.vps);
    const int NT = (int)gc.NT;
    double acc[kC][kJ];
#pragma unroll
    for (int i = 0; i < kC; i++)
#pragma unroll
        for (int j = 0; j < kJ; j++) acc[i][j] = 0.0;
    double topacc = 0.0;   // G at z1 of this lane's setup cell (cell si)

    // load item (view p, columns g0 .. g0 + ng - 1) into buffer B: 1/dz and P
    // rows in 1 KB pieces (16 bytes per lane, straight into LDS), the last piece
    // of each row set with only the lanes it needs
    auto stage = [&](uint32_t p, const GWin& wn, const GVu& g, int g0, int ng, GBuf& B) {
        // the cell corners' projections (column coordinate), written before the
        // loads into LDS are issued (no wait on them)
        const int tid = wave * 64 + lane;
        if (tid < kNQc) {
            const int cx = tid % (kGW + 1), cy = tid / (kGW + 1);
            const float dx = (float)min(X0 + cx, rc.hi[0]) - g.sx;
            const float dy = (float)min(Y0 + cy, rc.hi[1]) - g.sy;
            B.qc[tid] = -(g.ax * dy - g.ay * dx) * frcp(g.bx * dy - g.by * dx);
        }
        const int Wp = (wn.W + 31) & ~31;
        const int bytes = Wp * 8;                  // per row set (a multiple of 256)
        const int npc = (bytes + 1023) / 1024;     // pieces per row set
        const int lastl = (bytes - (npc - 1) * 1024) / 16;   // lanes of the last piece
        // the lane's byte offsets, opaque to the compiler so that the 64-bit
        // staging addresses are formed here, not held in registers across items
        uint32_t l16 = (uint32_t)lane * 16, l4 = (uint32_t)lane * 4;
        asm volatile("" : "+v"(l16), "+v"(l4));
        char* dst0 = reinterpret_cast<char*>(B.win);
        const char* izp = reinterpret_cast<const char*>(izt + (uint64_t)p * gc.cs + wn.tlo) + l16;
        const char* colp = reinterpret_cast<const char*>(pref + ((uint64_t)p * gc.NQ + g0) * gc.cs + wn.tlo) + l16;
        // row set 0: 1/dz; row set c + 1: P of column g0 + c
        for (int e = wave; e < (ng + 1) * npc; e += kGW) {
            const int c = e / npc, i = e - c * npc;
            const char* src = c == 0 ? izp + i * 1024 : colp + (uint64_t)(c - 1) * gc.cs * 8 + i * 1024;
            if (i + 1 < npc || lane < lastl)
                __builtin_amdgcn_global_load_lds(src, dst0 + c * bytes + i * 1024, 16, 0, 0);
        }
        // the group's column records (80 B each)
        for (int ch = wave; ch * 64 < ng * 20; ch += kGW) {
            const char* src = reinterpret_cast<const char*>(gcols + (uint64_t)p * gc.NQ + g0) + ch * 256 + l4;
            __builtin_amdgcn_global_load_lds(src, reinterpret_cast<char*>(B.cols) + ch * 256, 4, 0, 0);
        }
    };

    // the setup and main passes of item (p, g0 .. g1) from buffer B
    auto work = [&](const GWin& wn, const GVu& g, int g0, int g1, const GBuf& B) {
        const int W = wn.W;
        const int Wp = (W + 31) & ~31;
        // kz = k - sz of the lane's boundaries in FP64 with sz to FP64 precision (sz + szlo):
        // a ray nearly parallel to the planes crosses plane k at kz l / dz, so an FP32 sz
        // would move its crossing by up to 1e-5 l / dz voxels.
        double kz[kJ];
        int other[kJ];   // bytes from the P of the plane's row to that of the ray's other side
#pragma unroll
        for (int jj = 0; jj < kJ; jj++) {
            kz[jj] = ((double)(z0 + lane + 64 * jj) - (double)g.sz) - (double)g.szlo;
            other[jj] = kz[jj] > 0.0 ? 8 : -8;
        }
        const double kz1 = ((double)z1 - (double)g.sz) - (double)g.szlo;
        const int other1 = kz1 > 0.0 ? 8 : -8;
        const float kzspan = fmaxf(fabsf((float)z0 - g.sz), fabsf((float)z1 - g.sz));
        const double kb = g.kb - (double)wn.tlo;   // row of kz = 0 in the window, before its integer part
        const char* Pb = reinterpret_cast<const char*>(B.win);   // 1/dz rows at 0, column c at (c + 1) Wp 8
        auto at = [&](int o) -> double { return *reinterpret_cast<const double*>(Pb + o); };
        // bytes of the plane's row: P there holds the rays below it at the chord's far end
        auto row = [&](double kz_, double al) -> int { return g_row(cvt_int(fma(kz_, al, kb)), W - 2) * 8; };
        // x': the part of the chord before the ray with 1/dz iz crosses the plane
        auto part = [&](double kz_, double iz, double rl_, double h_) -> double {
            return __builtin_fmin(__builtin_fmax(fma(kz_ * iz, rl_, -h_), 0.0), 1.0);
        };
        // G(k) of one (cell, column) pair at a boundary, added to a: dh (P + x' (P' - P))
        auto eval = [&](double& a, double kz_, int oth, double al, double dh_, double rl_, double h_, int pbb) {
            const int u = row(kz_, al), v = u + oth;
            const double P0 = at(pbb + u), P1 = at(pbb + v), iz = at(v);
            a = fma(dh_, fma(part(kz_, iz, rl_, h_), P1 - P0, P0), a);
        };
        // the same with every ray that crosses the plane within the chord: from the row on
        // towards the chord's near end, until one does not
        auto eval_multi = [&](double& a, double kz_, int oth, double al, double dh_, double rl_, double h_, int pbb) {
            int u = row(kz_, al);
            double G = at(pbb + u);
            for (int v = u + oth; v >= 0 && v < W * 8; u = v, v += oth) {
                const double x = part(kz_, at(v), rl_, h_);
                if (x == 0.0) break;
                G = fma(x, at(pbb + v) - at(pbb + u), G);
            }
            a = fma(dh_, G, a);
        };
        // this lane's setup slot: cell si of the wave, candidate column q of the cell; from
        // an opaque copy of the lane, so that they are not kept in registers across the items
        int ln = lane;
        asm volatile("" : "+v"(ln));
        constexpr int kSlots = 64 / kC;
        const int si = ln % kC;
        const int s_ci = X0 + wave, s_cj = Y0 + si;
        int qa, qb;
        {
            const float* Q = B.qc + si * (kGW + 1) + wave;   // the cell's corners
            const float c00 = Q[0], c10 = Q[1], c01 = Q[kGW + 1], c11 = Q[kGW + 2];
            const float cmin = fminf(fminf(c00, c10), fminf(c01, c11));
            const float cmax = fmaxf(fmaxf(c00, c10), fmaxf(c01, c11));
            qa = max(g0, (int)ceilf(fmaxf(cmin - wn.mg, -1e9f)));
            qb = s_ci < X1 && s_cj < Y1 ? min(g1, (int)floorf(fminf(cmax + wn.mg, 1e9f))) : -1;
        }
        int q = qa + ln / kC;
        do {
            // ---- setup pass: lane (si, slot) takes candidate column q of its cell ----
            float dh = 0.f;
            double al = 0.0, rlq = 0.0, hq = 0.0;
            int pb_ = 0;
            bool valid = false, multi = false;
            if (q <= qb) {
                // the column record, all 80 bytes in one block of reads with one wait
                // (read field by field, its reads sit in the branches below, each with
                // its own wait)
                const uint32_t ca =
                    (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)(const char*)&B.cols[q - g0];
                float4 a0, a1, a2, a3, a4;
                asm volatile(
                    "ds_read_b128 %0, %5\n\t"
                    "ds_read_b128 %1, %5 offset:16\n\t"
                    "ds_read_b128 %2, %5 offset:32\n\t"
                    "ds_read_b128 %3, %5 offset:48\n\t"
                    "ds_read_b128 %4, %5 offset:64\n\t"
                    "s_waitcnt lgkmcnt(0)"
                    : "=&v"(a0), "=&v"(a1), "=&v"(a2), "=&v"(a3), "=&v"(a4)   // none shares the address register
                    : "v"(ca)
                    : "memory");
                // GCol: r[2] c[2] | P0[2] sg[2] | ifix[2] hs hd | l hc | lods pad
                const float Gr[2] = {a0.x, a0.y}, Gc[2] = {a0.z, a0.w}, GP0[2] = {a1.x, a1.y};
                const int Gsg[2] = {__float_as_int(a1.z), __float_as_int(a1.w)};
                const int Gif[2] = {__float_as_int(a2.x), __float_as_int(a2.y)};
                float h0 = a2.z, h1 = a2.w;
                const double Gl = g_dbl(a3.x, a3.y), Ghc = g_dbl(a3.z, a3.w), Glods = g_dbl(a4.x, a4.y);
                const int blo[2] = {s_ci, s_cj}, bhi[2] = {s_ci + 1, s_cj + 1};
#pragma unroll
                for (int a = 0; a < 2; a++) {
                    if (Gsg[a] == 0) {
                        if (Gif[a] != blo[a]) h1 = -AP_BIG;
                        continue;
                    }
                    const float ein = (float)(Gsg[a] > 0 ? blo[a] : bhi[a]) - GP0[a];
                    const float eout = (float)(Gsg[a] > 0 ? bhi[a] : blo[a]) - GP0[a];
                    h0 = fmaxf(h0, tcross(ein, Gr[a], Gc[a]));
                    h1 = fminf(h1, tcross(eout, Gr[a], Gc[a]));
                }
                if (h0 < h1) {
                    valid = true;
                    dh = h1 - h0;
                    const double ha = (double)h0 + Ghc, hb = (double)h1 + Ghc;   // from the source
                    al = Glods * g_rcp64(hb);
                    // the crossing in units of the chord: x' = (k - sz) / dz_t * l / dh - H,
                    // H = h_a / dh.  A chord too short to divide by keeps x' = 0, an error of
                    // at most dh yhat_t.
                    if (dh > 1e-20f) {
                        const double rd = g_rcp64((double)dh);
                        rlq = Gl * rd;
                        hq = ha * rd;
                    }
                    pb_ = (q - g0 + 1) * Wp * 8;
                    // |kappa_a - kappa_b| = |k - sz| |alpha_a - alpha_b| rays straddle plane k
                    // in the cell, within one: more than one needs the general evaluation
                    multi = kzspan * (float)(Glods * g_rcp64(ha) - al) >= 0.99f;
                    // G at z1
                    if (multi)
                        eval_multi(topacc, kz1, other1, al, (double)dh, rlq, hq, pb_);
                    else
                        eval(topacc, kz1, other1, al, (double)dh, rlq, hq, pb_);
                }
            }
            {
                double* R = Rec + (wave * 64 + lane) * 4;
                R[0] = rlq;
                R[1] = hq;
                R[2] = al;
                R[3] = g_dbl(dh, __int_as_float(pb_));
            }
            const uint64_t mvalid = __ballot(valid), mmulti = __ballot(multi);
            // ---- main pass: every lane, every pair of cell i ----
            constexpr uint64_t kCm = [] {
                uint64_t m = 0;
                for (int c = 0; c < kSlots; c++) m |= 1ull << (c * kC);
                return m;
            }();
#pragma unroll
            for (int i = 0; i < kC; i++) {
                uint64_t m = mvalid & (kCm << i);
                while (m) {
                    const int src = __builtin_ctzll(m);
                    m &= m - 1;
                    // the pair's record, read by every lane at one address (a broadcast).  The
                    // read is written out, with its wait in the same block, so that the
                    // compiler does not also wait for the next item's window loads
                    const uint32_t ra =
                        (uint32_t)(uintptr_t)(__attribute__((address_space(3))) double*)(Rec + (wave * 64 + src) * 4);
                    float4 q0, q1;
                    asm volatile(
                        "ds_read_b128 %0, %2\n\t"
                        "ds_read_b128 %1, %2 offset:16\n\t"
                        "s_waitcnt lgkmcnt(0)"
                        : "=&v"(q0), "=&v"(q1)   // early clobber: no output shares the address register
                        : "v"(ra)
                        : "memory");
                    const double rl = g_dbl(q0.x, q0.y), rh = g_dbl(q0.z, q0.w), ral = g_dbl(q1.x, q1.y);
                    const double rdhd = (double)q1.z;
                    const int rpb = __float_as_int(q1.w);
                    if ((mmulti >> src) & 1) {
                        for (int jj = 0; jj < kJ; jj++)
                            eval_multi(acc[i][jj], kz[jj], other[jj], ral, rdhd, rl, rh, rpb);
                    } else {
#pragma unroll
                        for (int jj = 0; jj < kJ; jj++)
                            eval(acc[i][jj], kz[jj], other[jj], ral, rdhd, rl, rh, rpb);
                    }
                }
            }
            q += kSlots;
        } while (__ballot(q <= qb) != 0);
    };

    // a window record read as wave-uniform values (scalar registers), so that the
    // view records read with them are scalar loads: a vector load in the work
    // phase would wait for the in-flight staging loads (one in-order counter)
    auto win_at = [&](int idx) -> GWin {
        const GWin w = Win[idx];
        GWin u;
        u.qlo = __builtin_amdgcn_readfirstlane(w.qlo);
        u.qhi = __builtin_amdgcn_readfirstlane(w.qhi);
        u.tlo = __builtin_amdgcn_readfirstlane(w.tlo);
        u.W = __builtin_amdgcn_readfirstlane(w.W);
        u.mg = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(w.mg)));
        u.ncg = __builtin_amdgcn_readfirstlane(w.ncg);
        return u;
    };

    // view record idx of the batch, read as wave-uniform values
    auto vw_at = [&](int idx) -> GVu {
        const uint32_t va = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)(Vw + idx * 8);
        const uint32_t vk = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) double*)(Vk + idx);
        float4 v0, v1;
        float2 v2;
        asm volatile(
            "ds_read2_b64 %0, %3 offset1:1\n\t"
            "ds_read2_b64 %1, %3 offset0:2 offset1:3\n\t"
            "ds_read_b64 %2, %4\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v0), "=&v"(v1), "=&v"(v2)   // early clobber: no output shares an address register
            : "v"(va), "v"(vk)
            : "memory");
        auto u = [](float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); };
        GVu g;
        g.sz = u(v0.x);
        g.sx = u(v0.y);
        g.sy = u(v0.z);
        g.ax = u(v1.x);
        g.ay = u(v1.y);
        g.bx = u(v1.z);
        g.by = u(v1.w);
        g.kb = g_dbl(u(v2.x), u(v2.y));
        g.szlo = u(v0.w);
        return g;
    };

    for (uint32_t pb = pbeg; pb < pend; pb += 64) {
        // ---- windows and view records of views pb .. pb + 63, one per lane of wave 0 ----
        __syncthreads();   // the previous batch's readers of Win and Vw are done
        if (wave == 0) {
            GWin wn;
            wn.qlo = 0; wn.qhi = -1; wn.tlo = 0; wn.W = 2; wn.mg = 0.f; wn.ncg = 1;
            const uint32_t p = pb + (uint32_t)lane;
            float4 v0 = make_float4(0.f, 0.f, 0.f, 0.f), v1 = v0;
            double kb = 0.0;
            if (p < pend && gviews[p].ok) {
                const GView g = gviews[p];
                v0 = make_float4(g.sz, g.sx, g.sy, g.szlo);
                v1 = make_float4(g.ax, g.ay, g.bx, g.by);
                kb = g.kb;
                float qmin = AP_BIG, qmax = -AP_BIG, dmax = 0.f;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float x = (float)((q & 1) ? X1 : X0), y = (float)((q & 2) ? Y1 : Y0);
                    const float dx = x - g.sx, dy = y - g.sy;
                    const float qc = -(g.ax * dy - g.ay * dx) * frcp(g.bx * dy - g.by * dx);
                    qmin = fminf(qmin, qc);
                    qmax = fmaxf(qmax, qc);
                    dmax = fmaxf(dmax, dx * dx + dy * dy);
                }
                // horizontal distances: nearest point of the tile box, farthest corner
                const float ex = fmaxf(fmaxf((float)X0 - g.sx, g.sx - (float)X1), 0.f);
                const float ey = fmaxf(fmaxf((float)Y0 - g.sy, g.sy - (float)Y1), 0.f);
                const float hmin = fmaxf(__builtin_amdgcn_sqrtf(ex * ex + ey * ey) * 0.999f, 1e-3f);
                const float hmax = __builtin_amdgcn_sqrtf(dmax) * 1.001f;
                // source-pixel distance over the window's columns
                auto lcol = [&](float q) {
                    const float x = g.ax + q * g.bx, y = g.ay + q * g.by;
                    return __builtin_amdgcn_sqrtf(x * x + y * y);
                };
                // Slack of the corner projections, in columns: the FP32 error of a
                // projection (a few ulp of source-pixel distance over column step) and of a
                // crossing's position (1e-3 voxel)
                const float ibn = __builtin_amdgcn_rsqf(g.bx * g.bx + g.by * g.by);
                const float le = fmaxf(lcol(qmin), lcol(qmax));
                const float mg = 0.01f + 2e-6f * le * ibn + 1e-3f * ibn * le * frcp(hmin);
                const int qlo = max(0, (int)floorf(fmaxf(qmin - mg, -1e9f)));
                const int qhi = min((int)gc.NQ - 1, (int)ceilf(fminf(qmax + mg, 1e9f)));
                if (qlo <= qhi) {
                    const float bb = g.bx * g.bx + g.by * g.by;
                    const float qv = fminf(fmaxf(-(g.ax * g.bx + g.ay * g.by) * frcp(bb), (float)qlo), (float)qhi);
                    const float la = lcol((float)qlo), lb = lcol((float)qhi), lv = lcol(qv);
                    const float lmin = fminf(fminf(la, lb), lv) * 0.999f, lmax = fmaxf(la, lb) * 1.001f;
                    const float rmin = lmin * frcp(hmax), rmax = lmax * frcp(hmin);
                    const float kz0 = (float)z0 - g.sz, kz1 = (float)z1 - g.sz;
                    const float k00 = kz0 * rmin, k01 = kz0 * rmax, k10 = kz1 * rmin, k11 = kz1 * rmax;
                    const float ids = frcp(g.dzs);
                    const float kmn = (fminf(fminf(k00, k01), fminf(k10, k11)) - g.dz0) * ids;
                    const float kmx = (fmaxf(fmaxf(k00, k01), fmaxf(k10, k11)) - g.dz0) * ids;
                    // rows int(kappa) + 2 and their neighbours, one more of slack each side
                    const int tlo = (int)fminf(fmaxf(floorf(kmn), 0.f), (float)NT);
                    const int thi = (int)fminf(fmaxf(floorf(kmx) + 4.f, 2.f), (float)(NT + 2));
                    wn.qlo = qlo;
                    wn.qhi = qhi;
                    wn.tlo = tlo;
                    wn.W = thi - tlo + 1;
                    wn.mg = mg;
                    // columns per group: the window holds Wp rows of 1/dz and of P per column
                    const int Wp = (wn.W + 31) & ~31;
                    wn.ncg = min(kGMaxCols, kGWin / (Wp * 8) - 1);
                }
            }
            Win[lane] = wn;
            reinterpret_cast<float4*>(Vw)[lane * 2] = v0;
            reinterpret_cast<float4*>(Vw)[lane * 2 + 1] = v1;
            Vk[lane] = kb;
        }
        __syncthreads();
        const uint32_t pe = min(pend, pb + 64);
        // the batch's items (view, column group) in order, the next one loading
        // while the current one is worked on
        uint32_t p = pb;
        GWin wn = win_at(0);
        while (p < pe && wn.qlo > wn.qhi) {   // the first view that meets the tile
            p++;
            if (p < pe) wn = win_at((int)(p - pb));
        }
        if (p >= pe) continue;
        int g0 = wn.qlo;
        GVu vw = vw_at((int)(p - pb));
        stage(p, wn, vw, g0, min(wn.qhi, g0 + wn.ncg - 1) - g0 + 1, Buf0);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        // one item: stage the next into Bn, work on this one from Bc.  Two named
        // buffers (not one indexed array) let the compiler see that the work's LDS
        // reads do not touch the loads in flight, so it does not wait for them.
        auto step = [&](GBuf& Bc, GBuf& Bn) {
            const int g1 = min(wn.qhi, g0 + wn.ncg - 1);
            // the next item: the view's next group, else the next view that meets the tile
            uint32_t pn = p;
            int gn = g1 + 1;
            GWin wnn = wn;
            if (gn > wn.qhi) {
                pn = p + 1;
                if (pn < pe) wnn = win_at((int)(pn - pb));
                while (pn < pe && wnn.qlo > wnn.qhi) {
                    pn++;
                    if (pn < pe) wnn = win_at((int)(pn - pb));
                }
                gn = wnn.qlo;
            }
            GVu vwn = vw;
            if (pn != p && pn < pe) vwn = vw_at((int)(pn - pb));
            if (pn < pe) stage(pn, wnn, vwn, gn, min(wnn.qhi, gn + wnn.ncg - 1) - gn + 1, Bn);
            work(wn, vw, g0, g1, Bc);
            __builtin_amdgcn_s_waitcnt(0);   // this wave's loads of the next item have landed
            __syncthreads();                 // all have, and the current buffer's readers are done
            p = pn;
            g0 = gn;
            wn = wnn;
            vw = vwn;
        };
        while (p < pe) {
            step(Buf0, Buf1);
            if (p >= pe) break;
            step(Buf1, Buf0);
        }
    }
    // ---- G at z1 per cell: sum over the lanes of the cell's setup slots ----
    for (int o = kC; o < 64; o <<= 1) topacc += __shfl_xor(topacc, o, 64);
    // ---- voxel values: differences of neighbouring boundaries ----
#pragma unroll
    for (int i = 0; i < kC; i++) {
        const double top = __shfl(topacc, i, 64);
        const int gi = X0 + wave, gj = Y0 + i;
        if (gi >= X1 || gj >= Y1) continue;
#pragma unroll
        for (int jj = 0; jj < kJ; jj++) {
            const int k = z0 + lane + 64 * jj;
            double nxt = __shfl_down(acc[i][jj], 1, 64);
            if (jj + 1 < kJ) {
                const double n0 = __shfl(acc[i][jj + 1], 0, 64);
                if (lane == 63) nxt = n0;
            }
            if (k + 1 == z1) nxt = top;
            if (k < z1) {
                const double d = nxt - acc[i][jj];
                if (partial) {
                    const uint64_t nx = (uint64_t)(rc.hi[0] - rc.lo[0]), ny = (uint64_t)(rc.hi[1] - rc.lo[1]);
                    const uint64_t nz = (uint64_t)(rc.hi[2] - rc.lo[2]);
                    partial[((slice * nx + (uint64_t)(gi - rc.lo[0])) * ny + (uint64_t)(gj - rc.lo[1])) * nz +
                            (uint64_t)(k - rc.lo[2])] = d;
                } else {
                    const float v = (float)(d * scale);
                    const int64_t ov = (int64_t)gi * vsx + (int64_t)gj * vsy + (int64_t)k * vsz;
                    const float mv =
                        mult ? to_f32(mult[(int64_t)gi * msx + (int64_t)gj * msy + (int64_t)k * msz]) : 1.f;
                    vol[ov] = from_f32<Tv>(__builtin_fmaf(mv, v, to_f32(vol[ov])));
                }
            }
        }
    }
}

// Adds the view slices' partial sums, in order, into the volume.
template <typename Tv, typename Tm>
__global__ __launch_bounds__(256) void k_gather_combine(RayCfg rc, uint32_t slices, const double* __restrict__ partial,
                                                        double scale, Tv* __restrict__ vol, int64_t vsx, int64_t vsy,
                                                        int64_t vsz, const Tm* __restrict__ mult, int64_t msx,
                                                        int64_t msy, int64_t msz, uint32_t V, const uint32_t* left) {
    if (left && *left == V) return;   // no view was the gather's: the partial sums were not written
    const uint32_t nx = (uint32_t)(rc.hi[0] - rc.lo[0]), ny = (uint32_t)(rc.hi[1] - rc.lo[1]);
    const uint32_t nz = (uint32_t)(rc.hi[2] - rc.lo[2]);
    const uint64_t n = (uint64_t)nx * ny * nz;
    for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (uint64_t)gridDim.x * 256) {
        double v = 0.0;
        for (uint32_t s = 0; s < slices; s++) v += partial[s * n + e];
        const uint32_t k = (uint32_t)(e % nz), ij = (uint32_t)(e / nz);
        const int64_t gi = rc.lo[0] + (int64_t)(ij / ny), gj = rc.lo[1] + (int64_t)(ij % ny), gk = rc.lo[2] + (int64_t)k;
        const int64_t ov = gi * vsx + gj * vsy + gk * vsz;
        const float mv = mult ? to_f32(mult[gi * msx + gj * msy + gk * msz]) : 1.f;
        vol[ov] = from_f32<Tv>(__builtin_fmaf(mv, (float)(v * scale), to_f32(vol[ov])));
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
uint64_t gather_workspace_bytes(uint32_t V, uint32_t nu, uint32_t nv, uint32_t ssu, uint32_t ssv) {
    if (V == 0 || nu == 0 || nv == 0) return 0;
    return (uint64_t)g_layout(V, nu * ssu, nv * ssv).total;
}

uint64_t gather_partial_bytes(uint32_t V, uint64_t tables) { return g_partial_bytes(V, tables); }

bool gather_supported(uint32_t nv, uint32_t ssv) {
    return (uint64_t)nv * ssv + 34 <= (uint64_t)kGRowMax;
}

int32_t launch_gather_adjoint(const RayCfg& rc, uint32_t V, uint32_t nu, uint32_t nv, int64_t s0, int64_t s1,
                              int64_t s2, uint32_t ssu, uint32_t ssv, double scale, const ap_proj_spec* specs,
                              const ap_array3* vol_desc, void* vol, int32_t mdt, const int64_t* ms,
                              const void* mult, int32_t sino_dtype, const void* sino, void* workspace,
                              uint64_t ws_bytes, hipStream_t s, const uint32_t** left) {
    if (!gather_supported(nv, ssv)) return AP_ERR_UNSUPPORTED;
    GCfg gc;
    gc.V = V;
    gc.nu = nu;
    gc.nv = nv;
    gc.ssu = ssu;
    gc.ssv = ssv;
    gc.NQ = nu * ssu;
    gc.NT = nv * ssv;
    gc.s0 = s0;
    gc.s1 = s1;
    gc.s2 = s2;
    const GLayout L = g_layout(V, gc.NQ, gc.NT);
    gc.cs = L.cs;
    if (!workspace || ws_bytes < L.total || ((uintptr_t)workspace & 255)) return AP_ERR_UNSUPPORTED;
    char* ws = (char*)workspace;
    GView* gviews = (GView*)(ws + L.views);
    GCol* gcols = (GCol*)(ws + L.cols);
    double* pref = (double*)(ws + L.pref);
    double* izt = (double*)(ws + L.iz);
    const uint64_t nwave = (uint64_t)V * gc.NQ;
    if ((nwave + 3) / 4 >= (1ull << 31)) return AP_ERR_UNSUPPORTED;
    int32_t st = dispatch_dtype(sino_dtype, [&](auto tp) -> int32_t {
        using Tp = decltype(tp);
        if constexpr (std::is_same<Tp, double>::value || std::is_same<Tp, bf16_t>::value) {
            return ap_fail(AP_ERR_UNSUPPORTED, "sinogram dtype must be F32 or F16");
        } else {
            hipLaunchKernelGGL(k_gather_prep<Tp>, dim3((uint32_t)((nwave + 3) / 4)), dim3(256), 0, s, rc, gc, specs,
                               (const Tp*)sino, gviews, gcols, pref, izt);
            return ap_check_launch("gather_prep");
        }
    });
    if (st) return st;
    uint32_t* cnt = nullptr;
    if (left) {
        cnt = (uint32_t*)(ws + L.count);
        *left = cnt;
    }
    // Tiles of 64, 128 or 192 planes: 192 where one such layer holds the volume (160 x 160 x
    // 150, 180 views of 240 x 220: 1.91 ms, two layers of 128 planes 2.41), 128 above that
    // (512^3: 118 ms, layers of 256 planes 128; 128 x 128 x 320: 0.99 and 1.17).  64 where the
    // rows of a taller tile, estimated as the detector's in proportion to its share of the
    // volume's height and a quarter more, would leave a window fewer than four columns (100 x
    // 100 x 200 from 1000 rows: 1.57 ms, 128 planes 1.70); and one workgroup per CU with larger
    // windows where even those do.
    const uint32_t nz = (uint32_t)(rc.hi[2] - rc.lo[2]);
    auto crowded = [&](uint32_t j) {
        const double rows = 32.0 + 1.25 * gc.NT * std::min(1.0, 64.0 * j / nz);
        return rows * 5 * sizeof(double) > g_win_bytes(false) ||
               (gc.NT + 34) * 2 * sizeof(double) > (size_t)g_win_bytes(false);   // 1 / dz and one whole column
    };
    uint32_t kj = nz > 192 ? 2 : (nz + 63) / 64;
    if (crowded(kj)) kj = 1;
    const bool tall = crowded(kj);
    GTile tl;
    const uint32_t tw = kGW, th = (uint32_t)g_cells((int)kj);
    tl.ntx = ((uint32_t)(rc.hi[0] - rc.lo[0]) + tw - 1) / tw;
    tl.nty = ((uint32_t)(rc.hi[1] - rc.lo[1]) + th - 1) / th;
    tl.ntz = (nz + 64 * kj - 1) / (64 * kj);
    tl.nsx = (tl.ntx + kSTX - 1) / kSTX;
    tl.nsy = (tl.nty + kSTY - 1) / kSTY;
    // Views split between workgroups where the tiles do not fill the GPU's slots
    // evenly: the fewest slices whose last round is nearly full, within the
    // scratch behind the tables and at least 8 views each.
    const uint64_t tiles = (uint64_t)tl.ntx * tl.nty * tl.ntz;
    const uint64_t nvox = (uint64_t)(rc.hi[0] - rc.lo[0]) * (uint64_t)(rc.hi[1] - rc.lo[1]) * nz;
    const uint64_t slots = tall ? 256 : 512;
    uint32_t slices = 1;
    {
        const uint64_t fit = (ws_bytes - L.total) / (nvox * sizeof(double));
        const uint64_t most = std::min<uint64_t>(std::min<uint64_t>(fit, V / 8), 32);
        auto used = [&](uint64_t n) {   // share of the rounds' slots that have work
            const uint64_t b = tiles * n;
            return (double)b / (double)((b + slots - 1) / slots * slots);
        };
        double best = used(1);
        for (uint64_t n = 2; n <= most && best < 0.9; n++)
            if (used(n) > best + 0.03) {
                best = used(n);
                slices = (uint32_t)n;
            }
    }
    tl.vps = (V + slices - 1) / slices;
    tl.slices = slices;
    double* partial = slices > 1 ? (double*)(ws + L.total) : nullptr;
    const uint64_t total = (uint64_t)tl.nsx * tl.nsy * kST * tl.ntz * slices;
    if (total >= (1ull << 31)) return ap_fail(AP_ERR_INVALID, "too many tiles");
    tl.total = (uint32_t)total;
    tl.per_xcd = (tl.total + kXcdG - 1) / kXcdG;
    dim3 grid(tl.per_xcd * kXcdG);
    return dispatch_dtype(vol_desc->dtype, [&](auto tv) -> int32_t {
        using Tv = decltype(tv);
        return dispatch_dtype(mdt, [&](auto tm) -> int32_t {
            using Tm = decltype(tm);
            if constexpr (std::is_same<Tv, double>::value || std::is_same<Tm, double>::value) {
                return ap_fail(AP_ERR_UNSUPPORTED, "unsupported dtype combination");
            } else {
                auto launch = [&](auto kern) {
                    hipLaunchKernelGGL(kern, grid, dim3(kGW * 64), 0, s, rc, gc, tl, gviews, gcols, pref, izt, scale,
                                       (Tv*)vol, vol_desc->strides[0], vol_desc->strides[1], vol_desc->strides[2],
                                       (const Tm*)mult, ms[0], ms[1], ms[2], partial, cnt);
                };
                if (tall) launch(k_gather_adjoint<Tv, Tm, 1, true>);
                else if (kj == 1) launch(k_gather_adjoint<Tv, Tm, 1, false>);
                else if (kj == 2) launch(k_gather_adjoint<Tv, Tm, 2, false>);
                else launch(k_gather_adjoint<Tv, Tm, 3, false>);
                int32_t e = ap_check_launch("gather_adjoint");
                if (e || !partial) return e;
                hipLaunchKernelGGL((k_gather_combine<Tv, Tm>), dim3((uint32_t)std::min<uint64_t>((nvox + 255) / 256, 8192)),
                                   dim3(256), 0, s, rc, slices, partial, scale, (Tv*)vol, vol_desc->strides[0],
                                   vol_desc->strides[1], vol_desc->strides[2], (const Tm*)mult, ms[0], ms[1], ms[2], V, cnt);
                return ap_check_launch("gather_combine");
            }
        });
    });
}

// ---------------------------------------------------------------------------
// allocation-free entry point
// ---------------------------------------------------------------------------
namespace {

// The gather's workspace for callers that cannot allocate: 64 MiB per GPU,
// held from the first call on that GPU until the process ends.  Host code
// must not pass the symbol itself to a kernel or a copy (it names a host-side
// stand-in); the device address of each GPU's copy comes from
// hipGetSymbolAddress with that GPU current.
constexpr uint64_t kNoAllocBytes = 64ull << 20;
__device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

int32_t scratch_address(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return ap_fail(AP_ERR_HIP, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return ap_fail(AP_ERR_UNSUPPORTED, "device %d beyond %d", dev, kMaxDevices);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return ap_fail(AP_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return AP_OK;
}

}  // namespace

extern "C" int32_t ap_backproject_matched_noalloc(const ap_config_cb_project* cfg, const ap_proj_spec* specs,
                                                  uint32_t num_projs, const ap_vol_tex_chunk_spec* chunk,
                                                  const ap_array3* vol_desc, void* vol, const ap_array3* mult_desc,
                                                  const void* multiplier, const ap_array3* sino_desc,
                                                  const void* sino, float alpha, void* stream) {
    AP_REQUIRE(cfg && sino_desc, "NULL config or sinogram descriptor");
    AP_REQUIRE(cfg->ssu >= 1 && cfg->ssv >= 1, "ssu and ssv must be >= 1");
    const uint32_t nu = sino_desc->shape[1], nv = sino_desc->shape[2];
    if (gather_supported(nv, cfg->ssv) && num_projs > 0 && nu > 0 && nv > 0) {
        const uint64_t one = gather_workspace_bytes(1, nu, nv, cfg->ssu, cfg->ssv);
        if (one > kNoAllocBytes)
            return ap_fail(AP_ERR_UNSUPPORTED,
                           "one view of this detector (%u x %u, ss %u x %u) needs %llu bytes of scratch; the "
                           "allocation-free adjoint holds %llu (use ap_backproject_matched with a workspace)",
                           nu, nv, cfg->ssu, cfg->ssv, (unsigned long long)one,
                           (unsigned long long)kNoAllocBytes);
    }
    void* ws = nullptr;
    int32_t st = scratch_address(&ws);
    if (st) return st;
    return ap_backproject_matched(cfg, specs, num_projs, chunk, vol_desc, vol, mult_desc, multiplier, sino_desc,
                                  sino, alpha, ws, kNoAllocBytes, stream);
}
