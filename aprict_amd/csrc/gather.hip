// gather.hip -- matched adjoint of the Siddon forward projector for views
// whose detector v axis is parallel to z and whose u axis has no z component
// (circular and helical scans with upright panels), computed as a gather over
// cell faces: no atomics, every voxel sum accumulated in FP64 registers.
//
// Geometry.  For such a view all rays through detector (sub-)column q lie in
// one vertical plane through the source: they share their x-y line, and
// along that line, parametrised by the horizontal distance h from the source,
// ray t has height z_t(h) = sz + h * dz_t / l, where dz_t is the height of
// its detector point above the source and l the horizontal source-pixel
// distance.  Order the rays by height (dz_t = dz0 + t dzs, dzs > 0).  The
// column's line crosses x-y cell (i, j) over [h_a, h_b]; the Siddon length of
// ray t in voxel (i, j, k) is sec_t times the measure of the h in [h_a, h_b]
// where k <= z_t(h) < k + 1.  With yhat_t = y_t sec_t and
//     I(h; k) = sum_t yhat_t |{h' in [0, h] : z_t(h') < k}|
// the column adds G(k+1) - G(k) to voxel k, G(k) = I(h_b; k) - I(h_a; k).
// The first difference is over the two planes of the voxel, the second over
// the two faces of the cell that the line crosses: a flux through the faces.
// A face between two cells gives the same I to both, with opposite signs, so
// I is evaluated once per (face, column) and accumulated per face.
//
// I in closed form.  Ray t crosses plane k at h_t = kz l / dz_t, kz = k - sz.
// Above the source (kz > 0) falling rays are below the plane everywhere and a
// rising ray up to h_t; below it (kz <= 0) rising rays nowhere and a falling
// ray beyond h_t.  Up to terms that do not depend on h (they cancel between
// the two faces) both sides read
//     I(h; k) = h P[tau] + kz S[tau],   tau = #{t : z_t(h) < k},
// with P[tau] = sum_{t < tau} yhat_t and, over the rays on the plane's side,
//     S[tau] =  l sum_{t >= tau} yhat_t / dz_t   (kz > 0, rising rays)
//     S[tau] = -l sum_{t <  tau} yhat_t / dz_t   (kz <= 0, falling rays).
// Each sum runs from the steepest ray inwards, so no near-horizontal ray's
// 1 / dz enters a plane that the ray does not reach.  The row of (P, S) pairs
// holds the falling rows 0 .. t0 and then the rising ones t0 .. NT one place
// further (t0: rows that do not rise), so tau + (kz > 0) is the row to read.
// tau is the integer part of a linear function of k, and I is continuous
// where it steps, so its rounding does not matter.  A (sub-)detector finer or
// coarser than the voxels makes no difference to the evaluation.
//
// A pre-pass (k_gather_prep) writes, per view and sub-column, the (P, S)
// pairs of the sec-weighted sinogram column in z order and the column's x-y
// crossing constants (the forward's col_setup, so the face crossings along h
// are the forward's own FP32 values).  The main kernel (k_gather_adjoint)
// gives each workgroup (8 waves) a tile of 8x8 x-y cells and 64*kJ planes;
// each wave owns 18 of its 144 faces, each lane one plane per 64 in z.  The
// work comes in items, a view and a group of the columns crossing the tile:
// while the workgroup works on one item, the next one's window of pairs is
// loaded straight into the other of two LDS buffers (16-byte loads).  Per
// item each wave finds its (face, column) crossings one per lane -- the
// forward's own order of the crossings decides which face a column takes, so
// every column enters and leaves each cell it visits exactly once -- then for
// every crossing every lane evaluates I at its planes: the row (one FP64 FMA,
// the integer conversion, a clamp, an address), one 16-byte LDS read and two
// FP64 FMAs.  At the end the faces' sums meet in LDS and every voxel takes
// the differences.  Tiles run in blocks of 4x8, so that the workgroups on one
// XCD at one time share their views' windows through its L2.  A volume with
// too few tiles to fill the GPU gets its views split between workgroups,
// whose FP64 partial sums k_gather_combine adds in order.
//
// Precision: P, S and the accumulators are FP64.  The face sums reach h P
// (about 1e3 rows times 1e3 voxels) over all views, 1e-16 of which is far
// below the FP32 rounding of the terms.  A ray lying in a z plane (the
// forward's horizontal rows, row_flat) belongs to the voxel below the
// plane, as in the forward; such rays are kept out of P and S and added
// separately.  (With such a row left in, tau and the row's crossing, both what
// rounding leaves of 0, would disagree by the row's whole length.)
#include <algorithm>
#include <mutex>

#include "column.h"
#include "gather.h"

namespace {

constexpr int kXcdG = 8;
constexpr int kGMaxCols = 16;      // columns staged at once
constexpr int kGRowMax = 2048;     // rows of a window (at most)
constexpr int kGW = 8;             // waves per workgroup
constexpr int kGT = 8;             // cells per tile side
constexpr int kGN = kGT + 1;       // planes per tile side
constexpr int kGFaces = 2 * kGT * kGN;      // 144 faces: x-faces, then y-faces
constexpr int kGF = kGFaces / kGW;          // 18 per wave
static_assert(kGF * kGW == kGFaces, "faces divide between the waves");

// bytes of an LDS window buffer (two per workgroup): 72 KB for tall tiles; half
// of that where a tile is at most 128 planes tall, so that two workgroups share a CU
constexpr int g_win_bytes(int kJ) { return kJ <= 2 ? 36864 : 73728; }

// per-(view, sub-column) record
struct GCol {
    float r[2], c[2], P0[2];   // x-y crossing parameters along h - hc (col_setup)
    int32_t sg[2], ifix[2];
    float hs, hd;              // source and pixel along h - hc (hd <= hs: no ray meets the chunk)
    double hc;                 // closest approach to the chunk centre
    double lods;               // l / dzs
    float yh;                  // value of the column's rays lying in a z plane (sec = 1), 0 if none
    int32_t ifixh;             // the voxel row they belong to
    float pad[2];
};
static_assert(sizeof(GCol) == 80, "GCol layout");

__host__ __device__ inline size_t g_align(size_t x) { return (x + 255) & ~size_t(255); }

struct GLayout {
    size_t views, count, cols, pref, total;
    uint32_t cs;   // (P, S) pairs per column: NT + 2, whole 128-byte lines
};

__host__ __device__ inline GLayout g_layout(uint32_t V, uint32_t NQ, uint32_t NT) {
    GLayout L;
    L.cs = (NT + 2 + 7) & ~7u;
    L.views = 0;
    L.count = g_align((size_t)V * sizeof(GView));
    L.cols = L.count + 256;
    // spare records: the record loads copy whole 256-byte chunks
    L.pref = L.cols + g_align(((size_t)V * NQ + 4) * sizeof(GCol));
    L.total = L.pref + g_align((size_t)V * NQ * L.cs * sizeof(double2));
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
                                                     GCol* __restrict__ gcols, double2* __restrict__ pref) {
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
    const double qx = vr.Q00[0] + (double)ju * vr.U[0] - vr.S[0];
    const double qy = vr.Q00[1] + (double)ju * vr.U[1] - vr.S[1];
    const double l = hit ? sqrt(qx * qx + qy * qy) : 1.0;
    double2* P = pref + (size_t)w * gc.cs;
    const uint32_t NT = gc.NT;
    // height of row t (z order) above the source, and its sinogram row
    auto row = [&](uint32_t t, float& kv, uint32_t& k) -> double {
        const uint32_t sr = gv.flip ? NT - 1 - t : t;
        k = sr / gc.ssv;
        kv = (float)k + sub_offset_g(sr % gc.ssv, gc.ssv);
        return vr.Q00[2] + (double)kv * vr.V[2] - vr.S[2];
    };
    auto scan = [](double v) -> double { return g_scan(v); };
    // yhat of row t, 0 for a row lying in its z plane (the forward's horizontal
    // row, lane_setup), whose value goes to yh
    double yh = 0.0;
    int ifixh = INT32_MIN;
    auto yhat = [&](float kv, uint32_t k, bool flat) -> double {
        const double m = fma((double)kv, C.z.dm, C.z.m0);
        const float mf = (float)m;
        const float y = to_f32(sino[(int64_t)p * gc.s0 + (int64_t)j * gc.s1 + (int64_t)k * gc.s2]);
        if (row_flat(mf)) {
            if (flat) {
                yh += (double)y;
                ifixh = (int)ceil(flat_height(C.z.zc)) - 1;
            }
            return 0.0;
        }
        return (double)(y * __builtin_amdgcn_sqrtf(__builtin_fmaf(mf, mf, 1.f)));
    };
    // Upwards, 64 rows at a time (coalesced): exclusive prefixes P of every row
    // and, for the rows up to the first rising one, S = -l sum yhat / dz.  The
    // rising rows' P is kept by writing it now; their S follows downwards.
    double cp = 0.0, cn = 0.0;
    uint32_t nfall = 0;
    for (uint32_t b = 0; b <= NT; b += 64) {
        const uint32_t t = b + (uint32_t)lane;
        double yv = 0.0, sv = 0.0;
        bool fall = false;
        if (t < NT) {
            float kv;
            uint32_t k;
            const double dz = row(t, kv, k);
            fall = !(dz > 0.0);
            if (hit) yv = yhat(kv, k, true);
            if (fall && yv != 0.0) sv = -yv * l * g_rcp64(dz);
        }
        // rows of the falling side: 0 .. t0 (t0 included: every falling ray below)
        const uint64_t mf = __ballot(fall);
        nfall += (uint32_t)__popcll(mf);
        // exclusive sums from the lane below (the inclusive one minus the row's own
        // term would lose the others where a near-horizontal ray's 1 / dz is huge)
        const double ip = scan(yv), in_ = scan(sv);
        const double ep = __shfl_up(ip, 1, 64), en = __shfl_up(in_, 1, 64);
        const double Pt = cp + (lane ? ep : 0.0);
        if (t <= NT) {
            if (t <= nfall) P[t] = make_double2(Pt, cn + (lane ? en : 0.0));
            if (!fall) P[t + 1].x = Pt;
        }
        cp += __shfl(ip, 63, 64);
        cn += __shfl(in_, 63, 64);
    }
    // Downwards over the rising rows: S[t] = l sum_{t' >= t} yhat / dz, row t + 1.
    // Where every row rises (falls), the planes below (above) the source read one
    // constant row, whose S cancels: row 0 (NT + 1) then repeats its neighbour, so
    // that a row clamped to the table's end reads the right pair on either side.
    double cr = 0.0;
    for (int b = (int)(NT & ~63u); b >= 0 && b + 63 >= (int)nfall; b -= 64) {
        const uint32_t t = (uint32_t)(b + 63 - lane);   // lane 0 holds the highest row
        double sv = 0.0;
        if (t < NT && t >= nfall) {
            float kv;
            uint32_t k;
            const double dz = row(t, kv, k);
            const double yv = hit ? yhat(kv, k, false) : 0.0;
            if (yv != 0.0) sv = yv * l * g_rcp64(dz);
        }
        const double is = scan(sv);
        if (t <= NT && t >= nfall) {
            P[t + 1].y = nfall == NT ? cn : cr + is;
            if (nfall == 0 && t == 0) P[0].y = cr + is;
        }
        cr += __shfl(is, 63, 64);
    }
    // the horizontal rows of the column (at most one in practice; summed)
    for (int o = 32; o > 0; o >>= 1) {
        yh += __shfl_xor(yh, o, 64);
        ifixh = max(ifixh, __shfl_xor(ifixh, o, 64));
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
        g.hc = hit ? C.z.hc : 0.0;
        g.lods = l / (fabs(vr.V[2]) / (double)gc.ssv);
        g.yh = (float)yh;
        g.ifixh = ifixh == INT32_MIN ? 0 : ifixh;
        g.pad[0] = g.pad[1] = 0.f;
        gcols[w] = g;
        if (q == 0) {
            gv.t0 = (int32_t)nfall;
            gviews[p] = gv;
        }
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
    uint32_t slices, vps;     // view slices, views per slice (a multiple of 1; the last may be short)
};

__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }

// prefix window of one view for the tile (views taken 64 at a time, one per lane)
struct GWin {
    int qlo, qhi, tlo, W;   // columns [qlo, qhi], rows tlo .. tlo + W - 1 of the pairs (qlo > qhi: nothing)
    float mg;               // slack of the corner projections, in columns
    int ncg;                // columns per staging group
};

// a view's parameters, as wave-uniform values
struct GVu {
    float sz, sx, sy;
    int t0;
    float ax, ay, bx, by;
    double kb;    // tau + 1/2 at kz = 0: -dz0 / dzs + 1/2
    float szlo;   // the source height is sz + szlo
};

// a wave's share of an item's loads: every kGW-th column
struct GStage {
    const char* src;   // the column's pairs, at the first row still to load
    char* dst;
    int W;             // rows still to load (<= 0: none)
    int Wc, more;      // rows of a column, columns after this one
    const char* rec;   // 256 bytes of the column records, and whether it loads them
    char* rdst;
    int ch;
};

__device__ __forceinline__ float g_uni(float x) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}
__device__ __forceinline__ double g_lane(double x, int src) {
    const uint64_t b = (uint64_t)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), src);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// nearest integer of x, |x| < 2^31: the low word of x + 1.5 2^52
__device__ __forceinline__ int g_nearest(double x) {
    return (int)(uint32_t)(uint64_t)__double_as_longlong(x + 6755399441055744.0);
}
// x + 1 in the lanes of `mask`, x elsewhere; clamped to [0, hi]: the mask is a carry
// in scalar registers, and each step one instruction
__device__ __forceinline__ int g_row(int x, uint64_t mask, int hi) {
    int r;
    asm("v_addc_co_u32_e64 %0, vcc, %1, 0, %2\n\tv_med3_i32 %0, %0, 0, %3"
        : "=&v"(r)
        : "v"(x), "s"(mask), "s"(hi)
        : "vcc");
    return r;
}
__device__ __forceinline__ double g_dbl(float lo, float hi) {
    return __longlong_as_double((long long)(((uint64_t)__float_as_uint(hi) << 32) | __float_as_uint(lo)));
}
// 16 bytes per address from LDS, all reads issued before the one wait
__device__ __forceinline__ void g_read(const uint32_t (&a)[1], float4 (&v)[1]) {
    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v[0]) : "v"(a[0]) : "memory");
}
__device__ __forceinline__ void g_read(const uint32_t (&a)[2], float4 (&v)[2]) {
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1])
                 : "v"(a[0]), "v"(a[1])
                 : "memory");
}
__device__ __forceinline__ void g_read(const uint32_t (&a)[3], float4 (&v)[3]) {
    asm volatile("ds_read_b128 %0, %3\n\tds_read_b128 %1, %4\n\tds_read_b128 %2, %5\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2])
                 : "v"(a[0]), "v"(a[1]), "v"(a[2])
                 : "memory");
}
__device__ __forceinline__ void g_read(const uint32_t (&a)[4], float4 (&v)[4]) {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
                 : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3])
                 : "memory");
}

// What bounds it: the LDS reads of the pairs (16 bytes per lane and evaluation, plus
// bank conflicts where the rows are closer than the planes), then the latency of the
// setup pass.  8 waves of 18 faces against 16 waves of 9: half the setup passes for
// the same evaluations, at the same time (129.9 and 125.7 ms at 512^3 x 720, 768^2;
// 3.27 and 3.71 ms for a helical gradient step at 161x149x127).  512^3: 137.9 -> 127 ms
// against evaluating every (cell, column) pair; 64^3 x 90, 96^2: 0.541 -> 0.08 ms.
template <typename Tv, typename Tm, int kJ>
__global__ __launch_bounds__(kGW * 64, kJ <= 2 ? 4 : 2) void k_gather_adjoint(
    RayCfg rc, GCfg gc, GTile tl, const GView* __restrict__ gviews, const GCol* __restrict__ gcols,
    const double2* __restrict__ pref, double scale, Tv* __restrict__ vol, int64_t vsx, int64_t vsy, int64_t vsz,
    const Tm* __restrict__ mult, int64_t msx, int64_t msy, int64_t msz, double* __restrict__ partial,
    uint32_t* __restrict__ left) {
    constexpr int kWin = g_win_bytes(kJ);
    constexpr int kNQc = kGN * kGN;
    // Two staging buffers: while the workgroup works on one (view, column group)
    // item from one buffer, the next item's window is loaded into the other.
    // A buffer holds the rows tlo .. tlo + W - 1 of (P, S) for each column of the
    // group, the group's column records and the projections of the tile's cell
    // corners.
    // The work phase reads them with written-out LDS reads and their waits: the
    // compiler would also wait for the loads in flight into the other buffer.
    struct GBuf {
        double2 win[kWin / 16];
        GCol cols[kGMaxCols];
        float qc[(kNQc + 3) & ~3];
    };
    __shared__ __align__(16) GBuf Bufs[2];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)(char*)&Bufs[0];
    __shared__ GWin Win[64];
    // the batch's view parameters: sz, sx, sy, t0 (bits), ax, ay, bx, by, then
    // kb (FP64), szlo -- read from LDS at the start of a step, so that no step
    // waits on a global load of its view record
    __shared__ __align__(16) float Vw[64 * 8];
    __shared__ __align__(16) double Vk[64 * 2];
    // the lane from the hardware's count, not from the thread index, which would stay
    // in a register of its own; the wave as a scalar: staging addresses are scalars
    const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (left && blockIdx.x == 0 && wave == 0) {
        // number of views this kernel does not take (for the general adjoint's early exit)
        uint32_t n = 0;
        for (uint32_t p = 0; p < gc.V; p += 64)
            n += (uint32_t)__popcll(__ballot(p + lane < gc.V && !gviews[min(p + lane, gc.V - 1)].ok));
        if (lane == 0) *left = n;
    }
    // no view is this kernel's (tilted panels): nothing to add, and no partial sums are read
    if (left) {
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
    const uint32_t pbeg = slice * tl.vps, pend = min(gc.V, pbeg + tl.vps);
    const int X0 = rc.lo[0] + (int)tx * kGT, Y0 = rc.lo[1] + (int)ty * kGT;
    const int X1 = min(X0 + kGT, rc.hi[0]), Y1 = min(Y0 + kGT, rc.hi[1]);
    const int z0 = rc.lo[2] + (int)tz * 64 * kJ;
    const int z1 = min(z0 + 64 * kJ, rc.hi[2]);
    const int NT = (int)gc.NT;
    // this lane's setup slot: face fi of the wave, candidate slot ss of the face.
    // Faces are dealt to the waves in turn, so each wave has x- and y-faces of
    // every part of the tile.
    constexpr int kSlots = 64 / kGF;   // 3
    // packed: corner index (y major) | plane << 8 | cell << 16 | y-face << 24 | in the tile << 25
    uint32_t face;
    {
        const int fi = lane % kGF, fid = wave + kGW * fi;
        const bool y = fid >= kGFaces / 2;
        const int fr = y ? fid - kGFaces / 2 : fid, pl = fr % kGN, ce = fr / kGN;
        const int gx = X0 + (y ? ce : pl), gy = Y0 + (y ? pl : ce);
        const bool ok = lane < kSlots * kGF && (y ? (gx < X1 && gy <= Y1) : (gx <= X1 && gy < Y1));
        face = (uint32_t)((y ? pl * kGN + ce : ce * kGN + pl) | (pl << 8) | (ce << 16) | ((y ? 1 : 0) << 24) |
                          ((ok ? 1 : 0) << 25));
    }
    double acc[kGF][kJ];
#pragma unroll
    for (int i = 0; i < kGF; i++)
#pragma unroll
        for (int j = 0; j < kJ; j++) acc[i][j] = 0.0;
    double topacc = 0.0;   // the face's sum at plane z1, over this lane's candidates

    // Loading item (view p, columns g0 .. g0 + ng - 1) into a buffer: the cell
    // corners' projections at once; then the column records and each wave's columns
    // in 1 KB pieces (16 bytes per lane, straight into LDS), the last piece with
    // only the lanes it needs.  The pieces are issued between the faces of the
    // current item: issued all at once they fill the memory pipeline, and the
    // waves stand in the issue until the first ones return.  None is issued before the
    // setup pass, whose reloads of spilled registers would wait for it.
    auto stage_begin = [&](uint32_t p, const GWin& wn, const GVu& g, int g0, int ng, int buf) -> GStage {
        GBuf& B = Bufs[buf];
        uint32_t l1 = (uint32_t)lane;
        asm volatile("" : "+v"(l1));
        const uint32_t t = l1 + (uint32_t)wave * 64;
        if (t < (uint32_t)kNQc) {
            const int cx = (int)(t % kGN), cy = (int)(t / kGN);
            const float dx = (float)min(X0 + cx, rc.hi[0]) - g.sx;
            const float dy = (float)min(Y0 + cy, rc.hi[1]) - g.sy;
            B.qc[t] = -(g.ax * dy - g.ay * dx) * frcp(g.bx * dy - g.by * dx);
        }
        GStage st;
        // the group's column records (80 B each), by the waves from the last one (the
        // first ones have the columns)
        st.ch = (kGW - 1 - wave) * 64 < ng * 20 ? kGW - 1 - wave : -1;
        st.rec = reinterpret_cast<const char*>(gcols + (uint64_t)p * gc.NQ + g0) + st.ch * 256;
        st.rdst = reinterpret_cast<char*>(B.cols) + st.ch * 256;
        st.src = reinterpret_cast<const char*>(pref + ((uint64_t)p * gc.NQ + g0 + wave) * gc.cs + wn.tlo);
        st.dst = reinterpret_cast<char*>(B.win) + wave * wn.W * 16;
        st.Wc = wn.W;
        st.W = wave < ng ? wn.W : 0;
        st.more = (ng - 1 - wave) / kGW;   // not read where W is 0
        return st;
    };
    auto stage_records = [&](GStage& st) {
        if (st.ch >= 0) {
            uint32_t l4 = (uint32_t)lane * 4;
            asm volatile("" : "+v"(l4));
            __builtin_amdgcn_global_load_lds(st.rec + l4, st.rdst, 4, 0, 0);
            st.ch = -1;
        }
    };
    auto stage_piece = [&](GStage& st) {
        if (st.W > 0) {
            uint32_t l16 = (uint32_t)lane * 16;
            asm volatile("" : "+v"(l16));
            if (lane < st.W) __builtin_amdgcn_global_load_lds(st.src + l16, st.dst, 16, 0, 0);
            st.src += 1024;
            st.dst += 1024;
            st.W -= 64;
            if (st.W <= 0 && st.more > 0) {   // the wave's next column
                st.more--;
                const int done = st.Wc - st.W;
                st.src += (int64_t)gc.cs * (16 * kGW) - done * 16;
                st.dst += st.Wc * (16 * kGW) - done * 16;
                st.W = st.Wc;
            }
        }
    };

    // the setup and main passes of item (p, g0 .. g1) from buffer B
    auto work = [&](const GWin& wn, const GVu& g, int g0, int g1, int buf, GStage& next) {
        const int W = wn.W;
        const uint32_t bwin = lds0 + (uint32_t)buf * (uint32_t)sizeof(GBuf);
        const uint32_t bcol = bwin + (uint32_t)offsetof(GBuf, cols), bqc = bwin + (uint32_t)offsetof(GBuf, qc);
        // The accumulators and one pass take nearly all registers: what can be derived
        // from one value is, from an opaque copy of it, so that the compiler does not
        // keep the derived ones across the items (spilled, they would be reloaded with
        // a wait for every load in flight).
        uint32_t fc = face;
        int kf = z0 + lane;
        asm volatile("" : "+v"(fc), "+v"(kf));
        // kz = k - sz of the lane's first plane, in FP64 with sz to FP64 precision (sz +
        // szlo): a ray nearly parallel to the planes crosses plane k at kz l / dz.  Where
        // a plane goes through the source all planes are moved up by less than any
        // crossing resolves: the tau of kz = 0 is then t0, whatever the rounding of kappa.
        double kz0 = ((double)kf - (double)g.sz) - (double)g.szlo;
        kz0 += kz0 == rint(kz0) ? 0x1p-40 : 0.0;
        const double kb = g.kb - (double)wn.tlo;   // tau + 1/2 of kz = 0, as a window row
        // candidate columns of the lane's face
        const bool fy = (fc >> 24) & 1u, fval = (fc >> 25) & 1u;
        int qa, qb;
        {
            const uint32_t ca = bqc + (fc & 255u) * 4;
            float c0, c1;
            asm volatile(
                "ds_read_b32 %0, %2\n\t"
                "ds_read_b32 %1, %3\n\t"
                "s_waitcnt lgkmcnt(0)"
                : "=&v"(c0), "=&v"(c1)
                : "v"(ca), "v"(ca + (fy ? 4u : (uint32_t)kGN * 4u))
                : "memory");
            qa = max(g0, (int)ceilf(fmaxf(fminf(c0, c1) - wn.mg, -1e9f)));
            qb = fval ? min(g1, (int)floorf(fminf(fmaxf(c0, c1) + wn.mg, 1e9f))) : -1;
        }
        int q = qa + lane / kGF;
        do {
            // ---- setup pass: lane (fi, ss) takes candidate column q of its face ----
            asm volatile("" : "+v"(fc));
            double sh = 0.0, al = 0.0;    // signed h, kappa slope
            int off = 0, flat = 0;
            bool pos = false, neg = false;
            if (q <= qb) {
                // the column record, all 80 bytes in one block of reads with one wait
                // the column record's fields of the face's axis (f: its plane) and of the
                // other one (o: its cell), in one block of reads with one wait
                const uint32_t ca = bcol + (uint32_t)(q - g0) * (uint32_t)sizeof(GCol);
                const uint32_t caf = ca + (fy ? 4u : 0u), cao = ca + (fy ? 0u : 4u);
                float2 rcf, rco, psf, pso, hsd, yhi;
                float ifof;
                float4 hl;
                // GCol: r[2] c[2] | P0[2] sg[2] | ifix[2] hs hd | hc lods | yh ifixh pad
                asm volatile(
                    "ds_read2_b32 %0, %8 offset0:0 offset1:2\n\t"
                    "ds_read2_b32 %1, %9 offset0:0 offset1:2\n\t"
                    "ds_read2_b32 %2, %8 offset0:4 offset1:6\n\t"
                    "ds_read2_b32 %3, %9 offset0:4 offset1:6\n\t"
                    "ds_read_b32 %4, %9 offset:32\n\t"
                    "ds_read_b64 %5, %10 offset:40\n\t"
                    "ds_read_b128 %6, %10 offset:48\n\t"
                    "ds_read_b64 %7, %10 offset:64\n\t"
                    "s_waitcnt lgkmcnt(0)"
                    : "=&v"(rcf), "=&v"(rco), "=&v"(psf), "=&v"(pso), "=&v"(ifof), "=&v"(hsd), "=&v"(hl), "=&v"(yhi)
                    : "v"(caf), "v"(cao), "v"(ca)
                    : "memory");
                const float rf = rcf.x, ro = rco.x, cf = rcf.y, co = rco.y, pf = psf.x, po = pso.x;
                const int sgf = __float_as_int(psf.y), sgo = __float_as_int(pso.y), ifo = __float_as_int(ifof);
                const int ipf = (int)((fc >> 8) & 255u) + (fy ? Y0 : X0);
                const int ipo = (int)((fc >> 16) & 255u) + (fy ? X0 : Y0);
                const float hf = tcross((float)ipf - pf, rf, cf);
                const float ha = tcross((float)ipo - po, ro, co), hb = tcross((float)(ipo + 1) - po, ro, co);
                const float hin = sgo > 0 ? ha : hb, hout = sgo > 0 ? hb : ha;
                // the forward's order of the crossings: x before y where they are equal
                const bool in = sgo == 0 ? ifo == ipo
                                         : (fy ? (hin <= hf && hf < hout) : (hin < hf && hf <= hout));
                if (sgf != 0 && in && hsd.x < hsd.y) {
                    pos = sgf > 0;
                    neg = !pos;
                    const double hc = g_dbl(hl.x, hl.y), lods = g_dbl(hl.z, hl.w);
                    const double h = (double)fminf(fmaxf(hf, hsd.x), hsd.y) + hc;
                    al = lods * g_rcp64(fmax(h, 1e-6));
                    sh = pos ? h : -h;
                    off = (int)bwin + (q - g0) * W * 16;
                    flat = yhi.x != 0.f ? 1 : 0;
                    // plane z1 (row by its own side)
                    const double kz1 = kz0 + (double)(z1 - kf);
                    const int row = min(max(g_nearest(fma(kz1, al, kb)) + (kz1 > 0.0 ? 1 : 0), 0), W - 1);
                    float4 b0;
                    asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                                 : "=&v"(b0)
                                 : "v"((uint32_t)(off + row * 16))
                                 : "memory");
                    topacc = fma(sh, g_dbl(b0.x, b0.y), topacc);
                    topacc = fma(pos ? kz1 : -kz1, g_dbl(b0.z, b0.w), topacc);
                    if (flat && z1 > __float_as_int(yhi.y)) topacc = fma(sh, (double)yhi.x, topacc);
                }
            }
            const uint64_t mpos = __ballot(pos), mneg = __ballot(neg), mflat = __ballot(flat != 0);
            // ---- main pass: every lane, every crossing of face i ----
            // kz of the lane's planes, and the lanes whose planes lie above the source
            double kz[kJ];
            uint64_t above[kJ];
            {
                double k0 = kz0;
                asm volatile("" : "+v"(k0));
#pragma unroll
                for (int jj = 0; jj < kJ; jj++) {
                    kz[jj] = jj == 0 ? k0 : k0 + (double)(64 * jj);
                    above[jj] = __ballot(kz[jj] > 0.0);
                }
            }
            auto event = [&](double (&a)[kJ], int src, auto sgn) {
                constexpr bool kNeg = decltype(sgn)::value;
                const double esh = g_lane(sh, src), eal = g_lane(al, src);
                const int eoff = __builtin_amdgcn_readlane(off, src);
                uint32_t ra[kJ];
#pragma unroll
                for (int jj = 0; jj < kJ; jj++) {
                    const int row = g_row(g_nearest(fma(kz[jj], eal, kb)), above[jj], W - 1);
                    ra[jj] = (uint32_t)(eoff + row * 16);
                }
                float4 ps[kJ];
                g_read(ra, ps);
#pragma unroll
                for (int jj = 0; jj < kJ; jj++) {
                    a[jj] = fma(esh, g_dbl(ps[jj].x, ps[jj].y), a[jj]);
                    a[jj] = fma(kNeg ? -kz[jj] : kz[jj], g_dbl(ps[jj].z, ps[jj].w), a[jj]);
                }
                if ((mflat >> src) & 1) {
                    // the column's rays lying in a z plane: their voxel row is below the plane
                    const uint32_t ga = bcol + (uint32_t)((eoff - (int)bwin) / (W * 16)) * (uint32_t)sizeof(GCol) +
                                        (uint32_t)offsetof(GCol, yh);
                    float2 gy2;
                    asm volatile("ds_read_b64 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(gy2) : "v"(ga) : "memory");
                    const double ryh = esh * (double)gy2.x;
                    const int rif = __float_as_int(gy2.y);
#pragma unroll
                    for (int jj = 0; jj < kJ; jj++)
                        if (kf + 64 * jj > rif) a[jj] += ryh;
                }
            };
            constexpr uint64_t kFm = [] {
                uint64_t m = 0;
                for (int s = 0; s < kSlots; s++) m |= 1ull << (s * kGF);
                return m;
            }();
#pragma unroll
            for (int i = 0; i < kGF; i++) {
                if (i == 0) stage_records(next);
                stage_piece(next);
                uint64_t m = mpos & (kFm << i);
                while (m) {
                    const int src = __builtin_ctzll(m);
                    m &= m - 1;
                    event(acc[i], src, std::false_type{});
                }
                m = mneg & (kFm << i);
                while (m) {
                    const int src = __builtin_ctzll(m);
                    m &= m - 1;
                    event(acc[i], src, std::true_type{});
                }
            }
            q += kSlots;
        } while (__ballot(q <= qb) != 0);
    };

    // a window record read as wave-uniform values (scalar registers)
    auto win_at = [&](int idx) -> GWin {
        const GWin w = Win[idx];
        GWin u;
        u.qlo = __builtin_amdgcn_readfirstlane(w.qlo);
        u.qhi = __builtin_amdgcn_readfirstlane(w.qhi);
        u.tlo = __builtin_amdgcn_readfirstlane(w.tlo);
        u.W = __builtin_amdgcn_readfirstlane(w.W);
        u.mg = g_uni(w.mg);
        u.ncg = __builtin_amdgcn_readfirstlane(w.ncg);
        return u;
    };

    // view record idx of the batch, read as wave-uniform values
    auto vw_at = [&](int idx) -> GVu {
        const uint32_t va = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)(Vw + idx * 8);
        const uint32_t vk = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) double*)(Vk + idx * 2);
        float4 v0, v1, v2;
        asm volatile(
            "ds_read2_b64 %0, %3 offset1:1\n\t"
            "ds_read2_b64 %1, %3 offset0:2 offset1:3\n\t"
            "ds_read2_b64 %2, %4 offset1:1\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v0), "=&v"(v1), "=&v"(v2)   // early clobber: no output shares an address register
            : "v"(va), "v"(vk)
            : "memory");
        GVu g;
        g.sz = g_uni(v0.x);
        g.sx = g_uni(v0.y);
        g.sy = g_uni(v0.z);
        g.t0 = __builtin_amdgcn_readfirstlane(__float_as_int(v0.w));
        g.ax = g_uni(v1.x);
        g.ay = g_uni(v1.y);
        g.bx = g_uni(v1.z);
        g.by = g_uni(v1.w);
        const uint32_t klo = (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(v2.x));
        const uint32_t khi = (uint32_t)__builtin_amdgcn_readfirstlane(__float_as_int(v2.y));
        g.kb = __longlong_as_double((long long)(((uint64_t)khi << 32) | klo));
        g.szlo = g_uni(v2.z);
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
            float szlo = 0.f;
            double kb = 0.0;
            if (p < pend && gviews[p].ok) {
                const GView g = gviews[p];
                v0 = make_float4(g.sz, g.sx, g.sy, __int_as_float(g.t0));
                v1 = make_float4(g.ax, g.ay, g.bx, g.by);
                szlo = g.szlo;
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
                // crossing's position (1e-3 voxel).  Every column that crosses a face must
                // be among its candidates: a column taken into a cell and not out of it
                // would leave all of I there.
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
                    const float kz0 = (float)z0 - g.sz, kzt = (float)z1 - g.sz;
                    const float k00 = kz0 * rmin, k01 = kz0 * rmax, k10 = kzt * rmin, k11 = kzt * rmax;
                    const float ids = frcp(g.dzs);
                    const float kmn = (fminf(fminf(k00, k01), fminf(k10, k11)) - g.dz0) * ids;
                    const float kmx = (fmaxf(fmaxf(k00, k01), fmaxf(k10, k11)) - g.dz0) * ids;
                    // rows tau + (kz > 0), tau = ceil(kappa): one row of slack each side
                    const int tlo = (int)fminf(fmaxf(floorf(kmn) - 1.f, 0.f), (float)(NT + 1));
                    const int thi = (int)fminf(fmaxf(ceilf(kmx) + 3.f, 0.f), (float)(NT + 1));
                    wn.qlo = qlo;
                    wn.qhi = qhi;
                    wn.tlo = tlo;
                    wn.W = thi - tlo + 1;
                    wn.mg = mg;
                    wn.ncg = min(kGMaxCols, kWin / (wn.W * 16));
                }
            }
            Win[lane] = wn;
            reinterpret_cast<float4*>(Vw)[lane * 2] = v0;
            reinterpret_cast<float4*>(Vw)[lane * 2 + 1] = v1;
            Vk[lane * 2] = kb;
            reinterpret_cast<float*>(Vk)[lane * 4 + 2] = szlo;
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
        int cur = 0;
        GStage st = stage_begin(p, wn, vw, g0, min(wn.qhi, g0 + wn.ncg - 1) - g0 + 1, 0);
        stage_records(st);
        while (st.W > 0) stage_piece(st);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        do {
            // stage the next item into the other buffer, work on this one
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
            st.W = 0;
            st.ch = -1;
            if (pn < pe) st = stage_begin(pn, wnn, vwn, gn, min(wnn.qhi, gn + wnn.ncg - 1) - gn + 1, cur ^ 1);
            work(wn, vw, g0, g1, cur, st);
            while (st.W > 0) stage_piece(st);
            __builtin_amdgcn_s_waitcnt(0);   // this wave's loads of the next item have landed
            __syncthreads();                 // all have, and the current buffer's readers are done
            p = pn;
            g0 = gn;
            wn = wnn;
            vw = vwn;
            cur ^= 1;
        } while (p < pe);
    }
    // ---- the faces' sums at z1: over the lanes of the face's setup slots ----
    double top = 0.0;
    for (int s = 0; s < kSlots; s++) top += __shfl(topacc, s * kGF + lane % kGF, 64);   // lane i: face i
    // ---- voxel values: outflow minus inflow of a cell, plane k + 1 minus plane k ----
    // per 64 planes the faces' plane differences go through LDS, kEp planes at a time
    constexpr int kEp = kWin / 8 / kGFaces >= 64 ? 64 : 32;
    static_assert(kEp * 8 * kGFaces <= kWin, "a round of face differences fits a window buffer");
    double* D = reinterpret_cast<double*>(Bufs[0].win);
#pragma unroll
    for (int jj = 0; jj < kJ; jj++) {
        const int kl = z0 + lane + 64 * jj;
        double d[kGF];
#pragma unroll
        for (int i = 0; i < kGF; i++) {
            double nxt = __shfl_down(acc[i][jj], 1, 64);
            if (jj + 1 < kJ) {
                const double n0 = __shfl(acc[i][jj + 1 < kJ ? jj + 1 : jj], 0, 64);
                if (lane == 63) nxt = n0;
            }
            const double tp = __shfl(top, i, 64);
            if (kl + 1 == z1) nxt = tp;
            d[i] = nxt - acc[i][jj];
        }
#pragma unroll
        for (int rr = 0; rr < 64 / kEp; rr++) {
            __syncthreads();
            if (lane / kEp == rr) {
#pragma unroll
                for (int i = 0; i < kGF; i++) D[(wave + kGW * i) * kEp + lane % kEp] = d[i];
            }
            __syncthreads();
            for (int o = wave * 64 + lane; o < kGT * kGT * kEp; o += kGW * 64) {
                const int c = o / kEp, kk = o % kEp;
                const int cx = c % kGT, cy = c / kGT;
                const int k = z0 + 64 * jj + rr * kEp + kk;
                if (X0 + cx >= X1 || Y0 + cy >= Y1 || k >= z1) continue;
                const double* Fx = D + (cy * kGN + cx) * kEp + kk;
                const double* Fy = D + (kGFaces / 2 + cx * kGN + cy) * kEp + kk;
                const double v = (Fx[kEp] - Fx[0]) + (Fy[kEp] - Fy[0]);
                const int gi = X0 + cx, gj = Y0 + cy;
                if (partial) {
                    const uint64_t ny = (uint64_t)(rc.hi[1] - rc.lo[1]), nz = (uint64_t)(rc.hi[2] - rc.lo[2]);
                    const uint64_t nx = (uint64_t)(rc.hi[0] - rc.lo[0]);
                    partial[((slice * nx + (uint64_t)(gi - rc.lo[0])) * ny + (uint64_t)(gj - rc.lo[1])) * nz +
                            (uint64_t)(k - rc.lo[2])] = v;
                    continue;
                }
                const float vf = (float)(v * scale);
                const int64_t ov = (int64_t)gi * vsx + (int64_t)gj * vsy + (int64_t)k * vsz;
                const float mv =
                    mult ? to_f32(mult[(int64_t)gi * msx + (int64_t)gj * msy + (int64_t)k * msz]) : 1.f;
                vol[ov] = from_f32<Tv>(__builtin_fmaf(mv, vf, to_f32(vol[ov])));
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
    double2* pref = (double2*)(ws + L.pref);
    const uint64_t nwave = (uint64_t)V * gc.NQ;
    if ((nwave + 3) / 4 >= (1ull << 31)) return AP_ERR_UNSUPPORTED;
    int32_t st = dispatch_dtype(sino_dtype, [&](auto tp) -> int32_t {
        using Tp = decltype(tp);
        if constexpr (std::is_same<Tp, double>::value || std::is_same<Tp, bf16_t>::value) {
            return ap_fail(AP_ERR_UNSUPPORTED, "sinogram dtype must be F32 or F16");
        } else {
            hipLaunchKernelGGL(k_gather_prep<Tp>, dim3((uint32_t)((nwave + 3) / 4)), dim3(256), 0, s, rc, gc, specs,
                               (const Tp*)sino, gviews, gcols, pref);
            return ap_check_launch("gather_prep");
        }
    });
    if (st) return st;
    uint32_t* cnt = nullptr;
    if (left) {
        cnt = (uint32_t*)(ws + L.count);
        *left = cnt;
    }
    // tiles as tall as the volume needs: ceil(nz / 256) layers of the smallest
    // multiple of 64 planes that covers it
    const uint32_t nz = (uint32_t)(rc.hi[2] - rc.lo[2]);
    const uint32_t layers = (nz + 255) / 256;
    const uint32_t kj = (nz + layers * 64 - 1) / (layers * 64);
    GTile tl;
    tl.ntx = (uint32_t)(rc.hi[0] - rc.lo[0] + kGT - 1) / kGT;
    tl.nty = (uint32_t)(rc.hi[1] - rc.lo[1] + kGT - 1) / kGT;
    tl.ntz = (nz + 64 * kj - 1) / (64 * kj);
    tl.nsx = (tl.ntx + kSTX - 1) / kSTX;
    tl.nsy = (tl.nty + kSTY - 1) / kSTY;
    // Views split between workgroups where the tiles do not fill the GPU's slots
    // evenly: the fewest slices whose last round is nearly full, within the
    // scratch behind the tables and at least 8 views each.
    const uint64_t tiles = (uint64_t)tl.ntx * tl.nty * tl.ntz;
    const uint64_t nvox = (uint64_t)(rc.hi[0] - rc.lo[0]) * (uint64_t)(rc.hi[1] - rc.lo[1]) * nz;
    const uint64_t slots = kj <= 2 ? 512 : 256;
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
                    hipLaunchKernelGGL(kern, grid, dim3(kGW * 64), 0, s, rc, gc, tl, gviews, gcols, pref, scale,
                                       (Tv*)vol, vol_desc->strides[0], vol_desc->strides[1], vol_desc->strides[2],
                                       (const Tm*)mult, ms[0], ms[1], ms[2], partial, cnt);
                };
                if (kj == 1) launch(k_gather_adjoint<Tv, Tm, 1>);
                else if (kj == 2) launch(k_gather_adjoint<Tv, Tm, 2>);
                else if (kj == 3) launch(k_gather_adjoint<Tv, Tm, 3>);
                else launch(k_gather_adjoint<Tv, Tm, 4>);
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

// The gather's workspace for callers that cannot allocate: 132 MiB per GPU,
// held from the first call on that GPU until the process ends.  Host code
// must not pass the symbol itself to a kernel or a copy (it names a host-side
// stand-in); the device address of each GPU's copy comes from
// hipGetSymbolAddress with that GPU current.
constexpr uint64_t kNoAllocBytes = 132ull << 20;
// A call is refused when 8 bytes per sub-ray of one view (with 40 rows of
// padding per column) and the view's records exceed 64 MiB; the (P, S) pairs
// take at most twice that, so every other view fits.
constexpr uint64_t kNoAllocView = 64ull << 20;
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
        const uint64_t nq = (uint64_t)nu * cfg->ssu, nt = (uint64_t)nv * cfg->ssv;
        const uint64_t one = 512 + g_align((nq + 4) * sizeof(GCol)) + g_align(nq * (nt + 40) * 8) + g_align((nt + 40) * 8);
        if (one > kNoAllocView)
            return ap_fail(AP_ERR_UNSUPPORTED,
                           "one view of this detector (%u x %u, ss %u x %u) needs %llu bytes of prefix sums; the "
                           "allocation-free adjoint holds %llu (use ap_backproject_matched with a workspace)",
                           nu, nv, cfg->ssu, cfg->ssv, (unsigned long long)one,
                           (unsigned long long)kNoAllocView);
    }
    void* ws = nullptr;
    int32_t st = scratch_address(&ws);
    if (st) return st;
    return ap_backproject_matched(cfg, specs, num_projs, chunk, vol_desc, vol, mult_desc, multiplier, sino_desc,
                                  sino, alpha, ws, kNoAllocBytes, stream);
}
