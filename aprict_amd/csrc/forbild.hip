// forbild.hip -- analytic FORBILD primitives on the GPU: exact last-wins line
// integrals (ap_project_forbild), point-sampling voxeliser
// (ap_voxelise_forbild) and per-shape bounding boxes (ap_forbild_bboxes).
//
// Every primitive is reduced once per block to an affine map M (in FP64)
// sending it onto a reference shape -- the cube [-1,1]^3, the unit ball, the
// unit-radius cylinder |z| <= h, or the truncated cone |z| <= h,
// x^2 + y^2 <= (ca + cb z)^2 -- and M applied to the view's source and pixel
// vectors, so a ray needs six FMAs and one quadratic or slab solve per shape.  Ray-primitive parameters are FP64
// (grazing rays cancel catastrophically in FP32); the compositing sweep and
// accumulation are FP32/FP64 as the output dtype requires.
//
// Semantics: cuda/structs/cu/FORBILD_{Box,Sphere,Ellipsoid,Ellipsoid_free,
// Cylinder,Cylinder_x,Cylinder_y,Cylinder_z,Ellipt_Cyl,Ellipt_Cyl_x,
// Ellipt_Cyl_y,Ellipt_Cyl_z,Cone,Cone_x,Cone_y,Cone_z,ClipAxisSpec}.cu
// (intervals / membership; a cone's radius runs linearly from r1 at -l/2 to
// r2 at +l/2 along its axis),
// FORBILD_Shape.cu:474-540 (last shape wins), CB_project_texture_chunked.cu
// :421-593 (sub-pixels, multiply_before_adding, overflow counter).
#include <algorithm>

#include "ap_common.h"

namespace {

enum PrimClass : int { kNone = 0, kCube = 1, kBall = 2, kCyl = 3, kCone = 4 };

struct Prim {
    double M[9];      // rows of the map r -> M (r - c)
    double c[3];
    double h;         // cylinder / cone half length
    double ca, cb;    // cone radius ca + cb z in the cone frame
    double cr;        // cone: max(|r1|, |r2|)
    float clip_ax[3][3];
    float clip_d[3];
    int clip_mode[3];
    float rho;
    int cls;
    float bc[3], br;    // bounding sphere for culling; radius inf or NaN (degenerate shape): never culled
};

// Radius of a sphere about c holding the primitive: |M^-1 l| <= sigma_max(M^-1) |l|
// for the local point l, |l| <= lr (the local shape's radius), and sigma_max^2 =
// lambda_max((M^-1)^T M^-1) <= its largest absolute row sum (Gershgorin; exact
// when the frame is orthonormal, since the matrix is then diagonal).
__device__ void set_bound(Prim& P, double lr) {
    const double* m = P.M;
    const double c00 = m[4] * m[8] - m[5] * m[7], c01 = m[5] * m[6] - m[3] * m[8], c02 = m[3] * m[7] - m[4] * m[6];
    const double det = m[0] * c00 + m[1] * c01 + m[2] * c02;
    const double id = 1.0 / det;
    // A = M^-1 = adj(M) / det
    const double A[9] = {c00 * id, (m[2] * m[7] - m[1] * m[8]) * id, (m[1] * m[5] - m[2] * m[4]) * id,
                         c01 * id, (m[0] * m[8] - m[2] * m[6]) * id, (m[2] * m[3] - m[0] * m[5]) * id,
                         c02 * id, (m[1] * m[6] - m[0] * m[7]) * id, (m[0] * m[4] - m[1] * m[3]) * id};
    double lam = 0.0;
    for (int i = 0; i < 3; i++) {
        double row = 0.0;
        for (int j = 0; j < 3; j++)
            row += fabs(A[i] * A[j] + A[3 + i] * A[3 + j] + A[6 + i] * A[6 + j]);
        lam = fmax(lam, row);
    }
    const double r = sqrt(lam) * lr * (1.0 + 1e-6);
    P.bc[0] = (float)P.c[0];
    P.bc[1] = (float)P.c[1];
    P.bc[2] = (float)P.c[2];
    P.br = (float)r;
}

__device__ __forceinline__ d3 unit_of(ap_fvec3 a) {
    d3 v = fv(a);
    return v * (1.0 / sqrt(dot(v, v)));
}

__device__ void make_prim(const ap_forbild_shape& s, Prim& P) {
    d3 ex = mkd3(1, 0, 0), ey = mkd3(0, 1, 0), ez = mkd3(0, 0, 1);
    double sx = 1, sy = 1, sz = 1;
    P.h = 0;
    P.ca = P.cb = P.cr = 0;
    P.cls = kNone;
    switch (s.type) {
    case 1: P.cls = kCube; sx = 2.0 / s.dx; sy = 2.0 / s.dy; sz = 2.0 / s.dz; break;
    case 10: P.cls = kBall; sx = 1.0 / s.dx; sy = 1.0 / s.dy; sz = 1.0 / s.dz; break;
    case 11:
        P.cls = kBall;
        ex = unit_of(s.a_x); ey = unit_of(s.a_y); ez = unit_of(s.a_z);
        sx = 1.0 / s.dx; sy = 1.0 / s.dy; sz = 1.0 / s.dz;
        break;
    case 13: P.cls = kBall; sx = sy = sz = 1.0 / s.r; break;
    case 6: case 7: case 8: case 9: {
        P.cls = kCyl;
        d3 ax = s.type == 6 ? unit_of(s.axis)
              : s.type == 7 ? mkd3(1, 0, 0) : s.type == 8 ? mkd3(0, 1, 0) : mkd3(0, 0, 1);
        d3 t = fabs(ax.x) < 0.9 ? mkd3(1, 0, 0) : mkd3(0, 1, 0);
        d3 e1 = cross(ax, t);
        e1 = e1 * (1.0 / sqrt(dot(e1, e1)));
        ex = e1; ey = cross(ax, e1); ez = ax;
        sx = sy = 1.0 / s.r; sz = 1.0;
        P.h = 0.5 * (double)s.l;
        break;
    }
    case 2: case 3: case 4: case 5: {
        P.cls = kCone;
        d3 ax = s.type == 2 ? unit_of(s.axis)
              : s.type == 3 ? mkd3(1, 0, 0) : s.type == 4 ? mkd3(0, 1, 0) : mkd3(0, 0, 1);
        d3 t = fabs(ax.x) < 0.9 ? mkd3(1, 0, 0) : mkd3(0, 1, 0);
        d3 e1 = cross(ax, t);
        e1 = e1 * (1.0 / sqrt(dot(e1, e1)));
        ex = e1; ey = cross(ax, e1); ez = ax;
        P.h = 0.5 * (double)s.l;
        P.ca = 0.5 * ((double)s.r1 + (double)s.r2);
        P.cb = ((double)s.r2 - (double)s.r1) / (double)s.l;
        P.cr = fmax(fabs((double)s.r1), fabs((double)s.r2));
        break;
    }
    case 12: case 14: case 15: case 16:
        P.cls = kCyl;
        if (s.type == 12) { ex = unit_of(s.a_x); ey = unit_of(s.a_y); ez = unit_of(s.axis); }
        else if (s.type == 14) { ex = mkd3(0, 1, 0); ey = mkd3(0, 0, 1); ez = mkd3(1, 0, 0); }
        else if (s.type == 15) { ex = mkd3(0, 0, 1); ey = mkd3(1, 0, 0); ez = mkd3(0, 1, 0); }
        sx = 1.0 / s.dx; sy = 1.0 / s.dy; sz = 1.0;
        P.h = 0.5 * (double)s.l;
        break;
    default: break;
    }
    P.M[0] = ex.x * sx; P.M[1] = ex.y * sx; P.M[2] = ex.z * sx;
    P.M[3] = ey.x * sy; P.M[4] = ey.y * sy; P.M[5] = ey.z * sy;
    P.M[6] = ez.x * sz; P.M[7] = ez.y * sz; P.M[8] = ez.z * sz;
    P.c[0] = s.x; P.c[1] = s.y; P.c[2] = s.z;
    const ap_forbild_clip* cs[3] = {&s.cas1, &s.cas2, &s.cas3};
    for (int i = 0; i < 3; i++) {
        P.clip_ax[i][0] = cs[i]->axis.x;
        P.clip_ax[i][1] = cs[i]->axis.y;
        P.clip_ax[i][2] = cs[i]->axis.z;
        P.clip_d[i] = cs[i]->dotprod;
        P.clip_mode[i] = cs[i]->mode;
    }
    P.rho = s.rho;
    // local radius: unit cube corner, unit ball, unit disk x [-h, h], cone of radius cr x [-h, h]
    const double lr = P.cls == kCube ? sqrt(3.0)
                    : P.cls == kBall ? 1.0
                    : P.cls == kCyl  ? sqrt(1.0 + P.h * P.h)
                    : P.cls == kCone ? sqrt(P.cr * P.cr + P.h * P.h) : 0.0;
    set_bound(P, lr);
}

// 1 / x for a nonzero finite x: the hardware reciprocal refined by two Newton
// steps (error about 1e-16 relative; an IEEE division is ten instructions)
__device__ __forceinline__ double rcp64(double x) {
    double y = __builtin_amdgcn_rcp(x);
    double e = fma(-x, y, 1.0);
    y = fma(y, e, y);
    e = fma(-x, y, 1.0);
    return fma(y, e, y);
}

// stable roots of A t^2 + 2 B t + C = 0; false if no real interval
__device__ __forceinline__ bool quad_roots(double A, double B, double C, double& t0, double& t1) {
    if (A == 0.0) return false;
    const double disc = B * B - A * C;
    if (!(disc > 0.0)) return false;
    const double sq = sqrt(disc);
    const double q = B > 0.0 ? -(B + sq) : -(B - sq);
    const double r1 = q * rcp64(A), r2 = q != 0.0 ? C * rcp64(q) : -r1;
    t0 = fmin(r1, r2);
    t1 = fmax(r1, r2);
    return true;
}

// A primitive as the rays of one view see it: the source in the local frame, and the
// local direction and the clip planes' rates as linear functions of the pixel
// coordinates (a, b) along U and V.  A ray takes six FMAs for its direction
// instead of the 3 x 3 map, and none for its origin.
struct RayPrim {
    double ls[3];                  // M (S - c)
    double l0[3], lu[3], lv[3];    // local direction l0 + a lu + b lv
    double cs[3];                  // clip planes, kept side <= 0: cs + t (c0 + a cu + b cv)
    double c0[3], cu[3], cv[3];
    double h, ca, cb;              // as in Prim
    double C;                      // constant term of the quadratic
    float bv[3], br;               // bounding sphere: centre relative to the source, radius
    float rho, cr;                 // cr: largest radius of a cone, else 1
    int cls, nclip;
    int pad;                       // 66 words: lanes reading a primitive each meet every bank twice
};
static_assert(sizeof(RayPrim) == 264, "RayPrim layout");

__device__ void make_ray_prim(const Prim& P, const ViewGeom& g, RayPrim& R) {
    const d3 s = g.S - mkd3(P.c[0], P.c[1], P.c[2]), d = g.D - g.S;
    for (int i = 0; i < 3; i++) {
        const d3 m = mkd3(P.M[3 * i], P.M[3 * i + 1], P.M[3 * i + 2]);
        R.ls[i] = dot(m, s);
        R.l0[i] = dot(m, d);
        R.lu[i] = dot(m, g.U);
        R.lv[i] = dot(m, g.V);
    }
    R.nclip = 0;
    for (int i = 0; i < 3; i++) {
        if (P.clip_mode[i] == 0) continue;
        const double sg = P.clip_mode[i] == 2 ? -1.0 : 1.0;
        const d3 n = mkd3(P.clip_ax[i][0], P.clip_ax[i][1], P.clip_ax[i][2]) * sg;
        const int k = R.nclip++;
        R.cs[k] = dot(n, g.S) - sg * (double)P.clip_d[i];
        R.c0[k] = dot(n, d);
        R.cu[k] = dot(n, g.U);
        R.cv[k] = dot(n, g.V);
    }
    R.h = P.h;
    R.ca = P.ca;
    R.cb = P.cb;
    const double g0 = P.cls == kCone ? P.ca + P.cb * R.ls[2] : 1.0;
    R.C = R.ls[0] * R.ls[0] + R.ls[1] * R.ls[1] + (P.cls == kBall ? R.ls[2] * R.ls[2] : 0.0) - g0 * g0;
    R.bv[0] = (float)(P.c[0] - g.S.x);
    R.bv[1] = (float)(P.c[1] - g.S.y);
    R.bv[2] = (float)(P.c[2] - g.S.z);
    R.br = P.br;
    R.rho = P.rho;
    R.cr = P.cls == kCone ? (float)P.cr : 1.f;
    R.cls = P.cls;
    R.pad = 0;
}

// Parametric interval (within [0,1]) of the ray through pixel coordinates (a, b)
// inside the primitive, which is the same for the whole wave
__device__ __forceinline__ bool prim_interval(const RayPrim& P, double a, double b, double& ta, double& tb) {
    ta = 0.0;
    tb = 1.0;
    const int nclip = __builtin_amdgcn_readfirstlane(P.nclip);
    for (int i = 0; i < nclip; i++) {
        const double s0 = P.cs[i], sd = fma(a, P.cu[i], fma(b, P.cv[i], P.c0[i]));
        if (sd == 0.0) {
            if (s0 > 0.0) return false;
        } else {
            const double t = -s0 * rcp64(sd);
            if (sd > 0.0) tb = fmin(tb, t); else ta = fmax(ta, t);
        }
    }
    if (!(tb > ta)) return false;
    const double ls[3] = {P.ls[0], P.ls[1], P.ls[2]};
    const double ld[3] = {fma(a, P.lu[0], fma(b, P.lv[0], P.l0[0])), fma(a, P.lu[1], fma(b, P.lv[1], P.l0[1])),
                          fma(a, P.lu[2], fma(b, P.lv[2], P.l0[2]))};
    double t0, t1;
    switch (__builtin_amdgcn_readfirstlane(P.cls)) {
    case kCube:
        for (int a = 0; a < 3; a++) {
            if (ld[a] == 0.0) {
                if (fabs(ls[a]) > 1.0) return false;
                continue;
            }
            const double inv = rcp64(ld[a]);
            const double x0 = (-1.0 - ls[a]) * inv, x1 = (1.0 - ls[a]) * inv;
            ta = fmax(ta, fmin(x0, x1));
            tb = fmin(tb, fmax(x0, x1));
        }
        break;
    case kBall:
        if (!quad_roots(ld[0] * ld[0] + ld[1] * ld[1] + ld[2] * ld[2],
                        ls[0] * ld[0] + ls[1] * ld[1] + ls[2] * ld[2], P.C, t0, t1))
            return false;
        ta = fmax(ta, t0);
        tb = fmin(tb, t1);
        break;
    case kCyl: {
        if (ld[2] == 0.0) {
            if (fabs(ls[2]) > P.h) return false;
        } else {
            const double inv = rcp64(ld[2]);
            const double x0 = (-P.h - ls[2]) * inv, x1 = (P.h - ls[2]) * inv;
            ta = fmax(ta, fmin(x0, x1));
            tb = fmin(tb, fmax(x0, x1));
        }
        const double A = ld[0] * ld[0] + ld[1] * ld[1];
        const double C = P.C;
        if (A == 0.0) {
            if (C > 0.0) return false;
        } else {
            if (!quad_roots(A, ls[0] * ld[0] + ls[1] * ld[1], C, t0, t1)) return false;
            ta = fmax(ta, t0);
            tb = fmin(tb, t1);
        }
        break;
    }
    case kCone: {
        // axial slab |z| <= h
        if (ld[2] == 0.0) {
            if (fabs(ls[2]) > P.h) return false;
        } else {
            const double inv = rcp64(ld[2]);
            const double x0 = (-P.h - ls[2]) * inv, x1 = (P.h - ls[2]) * inv;
            ta = fmax(ta, fmin(x0, x1));
            tb = fmin(tb, fmax(x0, x1));
        }
        if (!(tb > ta)) return false;
        // f(t) = x^2 + y^2 - (ca + cb z)^2 = A t^2 + 2 B t + C.  Inside the slab
        // only the nappe with ca + cb z >= 0 exists and the truncated cone is
        // convex, so {f <= 0} meets [ta, tb] in one interval.
        const double g0 = P.ca + P.cb * ls[2], gd = P.cb * ld[2];
        const double A = ld[0] * ld[0] + ld[1] * ld[1] - gd * gd;
        const double B = ls[0] * ld[0] + ls[1] * ld[1] - g0 * gd;
        const double C = P.C;
        if (A == 0.0) {
            if (B == 0.0) {
                if (C > 0.0) return false;
            } else if (B > 0.0) {
                tb = fmin(tb, -C * rcp64(2.0 * B));
            } else {
                ta = fmax(ta, -C * rcp64(2.0 * B));
            }
        } else if (A > 0.0) {
            if (!quad_roots(A, B, C, t0, t1)) return false;
            ta = fmax(ta, t0);
            tb = fmin(tb, t1);
        } else if (quad_roots(A, B, C, t0, t1)) {
            // f <= 0 outside (t0, t1): keep the piece on the real nappe
            const double la = ta, lb = fmin(tb, t0), ra = fmax(ta, t1), rb = tb;
            const bool left = lb > la, right = rb > ra;
            if (left && right) {
                const double zl = ls[2] + 0.5 * (la + lb) * ld[2];
                if (P.ca + P.cb * zl >= 0.0) tb = lb;
                else ta = ra;
            } else if (left) {
                tb = lb;
            } else if (right) {
                ta = ra;
            } else {
                return false;
            }
        }   // A < 0 without real roots: f < 0 on the whole line
        break;
    }
    default:
        return false;
    }
    return tb > ta;
}

__device__ bool prim_contains(const Prim& P, const d3& p) {
    for (int i = 0; i < 3; i++) {
        if (P.clip_mode[i] == 0) continue;
        const double dp = (double)P.clip_ax[i][0] * p.x + (double)P.clip_ax[i][1] * p.y +
                          (double)P.clip_ax[i][2] * p.z;
        if (P.clip_mode[i] == 1 && !(dp <= (double)P.clip_d[i])) return false;
        if (P.clip_mode[i] == 2 && !(dp > (double)P.clip_d[i])) return false;
    }
    const double r0 = p.x - P.c[0], r1 = p.y - P.c[1], r2 = p.z - P.c[2];
    const double a = P.M[0] * r0 + P.M[1] * r1 + P.M[2] * r2;
    const double b = P.M[3] * r0 + P.M[4] * r1 + P.M[5] * r2;
    const double e = P.M[6] * r0 + P.M[7] * r1 + P.M[8] * r2;
    switch (P.cls) {
    case kCube: return fabs(a) <= 1.0 && fabs(b) <= 1.0 && fabs(e) <= 1.0;
    case kBall: return a * a + b * b + e * e <= 1.0;
    case kCyl: return fabs(e) <= P.h && a * a + b * b <= 1.0;
    case kCone: {
        const double g = P.ca + P.cb * e;
        return fabs(e) <= P.h && a * a + b * b <= g * g;
    }
    default: return false;
    }
}

constexpr int kProjThreads = 256;  // 4 waves share the staged shapes
constexpr int kShapeBatch = 64;    // shapes staged in LDS at a time
constexpr int kUnion = 8;          // disjoint covered pieces kept per ray in registers
constexpr int kManyPieces = 64;    // and in memory, for the rays that need more, before the exact fallback
constexpr uint32_t kRefMaxIntersections = 1000;   // reference's overflow threshold

// Last-wins compositing (FORBILD_Shape.cu:474-540): the density at a point is
// that of the highest-index shape containing it, so the integral is
//   sum_q rho_q |I_q \ (union of I_q' for q' > q)|.
// Shapes are visited from the last to the first; the union of the intervals
// seen so far is kept as at most kUnion disjoint pieces in registers (empty
// pieces are [3, 2]).  Adding an interval I: its covered length is the sum of
// its overlaps with the pieces; then every piece it overlaps or touches is
// absorbed into it (one pass suffices: the pieces are disjoint, so a piece
// that meets the grown interval meets I itself) and the result takes a free
// piece.  Returns false when no piece is free.
struct Union {
    double a[kUnion], b[kUnion];
};

__device__ __forceinline__ void union_clear(Union& U) {
#pragma unroll
    for (int i = 0; i < kUnion; i++) {
        U.a[i] = 3.0;
        U.b[i] = 2.0;
    }
}

// used: pieces that any ray of the wave has used (wave-uniform); those behind it are
// empty in every ray
__device__ __forceinline__ bool union_add(Union& U, int used, double ta, double tb, double& uncovered,
                                          bool& grew) {
    double cov = 0.0, na = ta, nb = tb;
    bool placed = false;
#pragma unroll
    for (int i = 0; i < kUnion; i++) {
        if (i >= used) break;
        cov += fmax(0.0, fmin(tb, U.b[i]) - fmax(ta, U.a[i]));
        if (U.a[i] <= nb && U.b[i] >= na) {
            na = fmin(na, U.a[i]);
            nb = fmax(nb, U.b[i]);
            U.a[i] = 3.0;
            U.b[i] = 2.0;
        }
    }
    uncovered = (tb - ta) - cov;
#pragma unroll
    for (int i = 0; i < kUnion; i++) {
        if (i > used) break;
        if (!placed && U.a[i] > U.b[i]) {
            U.a[i] = na;
            U.b[i] = nb;
            placed = true;
            grew = i == used;
        }
    }
    return placed;
}

// Exact last-wins integral recomputed from global memory at every event; for
// rays whose covered set has more than kManyPieces pieces
__device__ __noinline__ double last_wins_exact(const ap_forbild_shape* __restrict__ shapes, uint32_t K,
                                               const ap_proj_spec* __restrict__ specs, uint32_t p, double a,
                                               double b) {
    const ViewGeom g = load_view(specs, p);
    double val = 0.0, prog = -1.0;
    for (uint32_t guard = 0; guard < 4 * K + 4; guard++) {
        int top = -1;
        double topb = 0.0, nxt = 2.0;
        float toprho = 0.f;
        for (int q = (int)K - 1; q >= 0; q--) {
            Prim P;
            RayPrim R;
            make_prim(shapes[q], P);
            make_ray_prim(P, g, R);
            double ta, tb;
            if (!prim_interval(R, a, b, ta, tb)) continue;
            if (top < 0 && ta <= prog && prog < tb) {
                top = q; topb = tb; toprho = P.rho;
            } else if (top < 0 && ta > prog && ta < nxt) {
                nxt = ta;   // candidate next start (no cover yet)
            }
        }
        if (top >= 0) {
            double e = topb;
            for (int q = (int)K - 1; q > top; q--) {
                Prim P;
                RayPrim R;
                make_prim(shapes[q], P);
                make_ray_prim(P, g, R);
                double ta, tb;
                if (prim_interval(R, a, b, ta, tb) && ta > prog && ta < e) e = ta;
            }
            val += (e - prog) * (double)toprho;
            prog = e;
        } else {
            if (nxt >= 2.0) break;
            prog = nxt;
        }
    }
    return val;
}

// The cone of a wave's rays: unit axis, sine and cosine of the half-angle; no cull
// where a corner is not well within 60 degrees of the axis.
struct RayCone {
    float ax[3], sa, ca;   // ca = 0: no cull
};

__device__ __forceinline__ RayCone ray_cone(const ViewGeom& g, double a, double b, double half) {
    RayCone c;
    const d3 d = g.D - g.S + g.U * a + g.V * b;
    const float dx = (float)d.x, dy = (float)d.y, dz = (float)d.z;
    const float il = 1.f / sqrtf(dx * dx + dy * dy + dz * dz);
    c.ax[0] = dx * il;
    c.ax[1] = dy * il;
    c.ax[2] = dz * il;
    float s2 = 0.f;
    bool ok = true;
    for (int q = 0; q < 4; q++) {
        const d3 e = d + g.U * ((q & 1) ? half : -half) + g.V * ((q & 2) ? half : -half);
        const float ex = (float)e.x, ey = (float)e.y, ez = (float)e.z;
        const float al = ex * c.ax[0] + ey * c.ax[1] + ez * c.ax[2], ee = ex * ex + ey * ey + ez * ez;
        // perpendicular part from its components: the difference ee - al^2 would cancel
        const float px = ex - al * c.ax[0], py = ey - al * c.ax[1], pz = ez - al * c.ax[2];
        s2 = fmaxf(s2, (px * px + py * py + pz * pz) / ee);
        ok = ok && al > 0.5f * sqrtf(ee);
    }
    c.sa = sqrtf(s2) * 1.001f + 1e-5f;   // margins for the FP32 directions
    c.ca = ok && c.sa < 0.85f ? sqrtf(1.f - c.sa * c.sa) : 0.f;   // 0 also where a value is NaN
    return c;
}

// Whether the sphere may meet the cone: the distance of its centre from the cone's
// nearest side, perp cos - along sin, is a lower bound of the distance to every ray.
// An infinite or NaN radius (degenerate shape) always may.
__device__ __forceinline__ bool cone_meets(const RayCone& c, const RayPrim& P) {
    const float al = P.bv[0] * c.ax[0] + P.bv[1] * c.ax[1] + P.bv[2] * c.ax[2];
    const float px = P.bv[0] - al * c.ax[0], py = P.bv[1] - al * c.ax[1], pz = P.bv[2] - al * c.ax[2];
    const float dist = sqrtf(px * px + py * py + pz * pz) * c.ca - al * c.sa;
    return c.ca == 0.f || !(dist > P.br * 1.0001f + 1e-5f * fabsf(al));
}

// Staging and the exact fallback are calls: inlined, their FP64 temporaries are
// spilled around the ray loop's (187 registers at 5 waves per SIMD; none of the ray
// loop's otherwise).
__device__ __noinline__ void stage_prim(const ap_forbild_shape* __restrict__ shape,
                                        const ap_proj_spec* __restrict__ specs, uint32_t p, RayPrim* out) {
    Prim P;
    make_prim(*shape, P);
    make_ray_prim(P, load_view(specs, p), *out);
}

// Whether a ray of the wave's tile may meet the primitive itself: the interval of the
// tile's central ray (a, b) in the primitive grown by how far the other rays, within
// `half` pixels of it along U and V, are from it.  FP32 with margins of 1e-5 of what
// cancels; a NaN keeps the primitive.
__device__ __forceinline__ bool tile_meets(const RayPrim& P, double a, double b, float half) {
    float ta = 0.f, tb = 1.f;
    // keeps c + t r <= 0
    auto below = [&](float c, float r) {
        const float t = -c / r;
        if (r > 0.f) tb = fminf(tb, t);
        if (r < 0.f) ta = fmaxf(ta, t);
        if (r == 0.f && c > 0.f) tb = -1.f;
    };
    auto at = [&](const double* c0, const double* cu, const double* cv, int i, float& e) {
        e = half * (fabsf((float)cu[i]) + fabsf((float)cv[i]));
        return (float)fma(a, cu[i], fma(b, cv[i], c0[i]));
    };
    for (int i = 0; i < 3; i++) {
        if (i >= P.nclip) break;
        float e;
        const float c = (float)P.cs[i], r = at(P.c0, P.cu, P.cv, i, e);
        below(c - 1e-5f * (fabsf(c) + fabsf(r)), r - e);
    }
    float l[3], d[3], e[3];
    for (int i = 0; i < 3; i++) {
        l[i] = (float)P.ls[i];
        d[i] = at(P.l0, P.lu, P.lv, i, e[i]);
    }
    // |l + t d| <= lim + t e
    auto slab = [&](int i, float lim) {
        const float m = lim * (1.f + 1e-5f) + 1e-5f * (fabsf(l[i]) + fabsf(d[i]));
        below(l[i] - m, d[i] - e[i]);
        below(-l[i] - m, -d[i] - e[i]);
    };
    if (P.cls == kCube)
        for (int i = 0; i < 3; i++) slab(i, 1.f);
    if (P.cls == kCyl || P.cls == kCone) slab(2, fabsf((float)P.h));
    if (P.cls != kCube) {
        if (P.cls != kBall) l[2] = d[2] = e[2] = 0.f;   // distance from the axis
        const float dd = d[0] * d[0] + d[1] * d[1] + d[2] * d[2];
        const float tc = -(l[0] * d[0] + l[1] * d[1] + l[2] * d[2]) / dd;
        const float px = l[0] + tc * d[0], py = l[1] + tc * d[1], pz = l[2] + tc * d[2];
        const float ll = fabsf(l[0]) + fabsf(l[1]) + fabsf(l[2]);
        const float R = P.cr * (1.f + 1e-5f) + e[0] + e[1] + e[2] + 1e-5f * ll;
        if (dd > 1e-6f * ll * ll) {   // else along the axis: no bound from it
            if (px * px + py * py + pz * pz > R * R) tb = -1.f;
            const float w = R / sqrtf(dd) + 1e-5f;
            ta = fmaxf(ta, tc - w);
            tb = fminf(tb, tc + w);
        }
    }
    return !(tb + 1e-5f < ta - 1e-5f);
}

__device__ __forceinline__ RayCone cone_of_lane(const RayCone& c, int lane) {
    auto get = [&](float x) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), lane)); };
    return RayCone{{get(c.ax[0]), get(c.ax[1]), get(c.ax[2])}, get(c.sa), get(c.ca)};
}

// A ray whose covered set needs more than 8 pieces is taken again with up to 64 in
// memory: 479 shapes of the head phantom, 90 views of 200^2 with 2 x 2 rays, 105 -> 4.9 ms
// against the exact recomputation for each of them.
// What bounds it: the FP64 intersection chains of the shapes that a tile may meet
// (about 100 instructions each), then the tests that find them.  A wave takes tiles of
// 8 x 8 pixels, narrow enough that a shape's test pays for most of the 64 rays (64
// pixels in a row met several times as many shapes); which shapes are tested is found
// once per tile, a shape per lane, first against the cone of the tile's rays, then
// against the tile's central ray with the primitive grown by the tile.  A tile that
// meets no shape neither reads nor writes the sinogram.  The shapes are reduced to what
// the view's rays need once per workgroup, for up to 32 tiles.
// 40 primitives x 720 x 512^2: 16.0 ms with a sphere test per ray and 256 pixels in a
// row, 7.3 ms with the cone alone, 2.45 ms with both; 32 views of 101 x 71, 114 -> 78 us.
// 5 waves per SIMD (96 registers, no spills in the ray loop) 2.46 ms, 6 2.8-3.2, 7 2.54.
struct ForbildTiles {
    uint32_t nk, total, per_block;   // tiles along v, tiles of a view, tiles of a workgroup
};

constexpr int kTile = 16, kWaveTile = 8;   // pixels of a workgroup's and a wave's tile side

// kOne: one ray per pixel.  kBatches: more shapes than LDS holds at once, staged again for
// every ray; a workgroup's waves then all walk every tile.
template <typename Tp, bool kOne, bool kBatches>
__global__ __launch_bounds__(kProjThreads, 5) void k_project_forbild(
    float mba, int additive, uint32_t ssu, uint32_t ssv, const ap_proj_spec* __restrict__ specs,
    const ap_forbild_shape* __restrict__ shapes, uint32_t K, ForbildTiles tm, uint32_t nu, uint32_t nv,
    int64_t s0, int64_t s1, int64_t s2, Tp* __restrict__ sino, uint32_t* __restrict__ oom) {
    __shared__ RayPrim prims[kShapeBatch];   // one view's
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const uint32_t p = blockIdx.y;
    const ViewGeom g = load_view(specs, p);
    if constexpr (kOne) ssu = ssv = 1;
    if constexpr (!kBatches) {
        if (threadIdx.x < K) stage_prim(shapes + threadIdx.x, specs, p, prims + threadIdx.x);
        __syncthreads();
    }
    // the cones of all the wave's tiles at once, one tile per lane
    // workgroups go to the XCDs in turn: turned by the view, so that no XCD gets the
    // same part of every detector (an object covers its middle)
    const uint32_t t0 = (blockIdx.x + blockIdx.y) % gridDim.x * tm.per_block, t1 = min(t0 + tm.per_block, tm.total);
    const int ju = (wave >> 1) * kWaveTile, ku = (wave & 1) * kWaveTile;
    RayCone cones;
    {
        const uint32_t t = min(t0 + (uint32_t)lane, tm.total - 1);
        cones = ray_cone(g, (double)((t / tm.nk) * kTile + ju) + 0.5 * (kWaveTile - 1) - 0.5 * (double)(g.nu - 1),
                         (double)((t % tm.nk) * kTile + ku) + 0.5 * (kWaveTile - 1) - 0.5 * (double)(g.nv - 1),
                         0.5 * kWaveTile);
    }
    const bool skip_empty = fabsf(mba) < __builtin_inff();   // 0 * mba is then 0
    for (uint32_t t = t0; t < t1; t++) {
        const RayCone cone = cone_of_lane(cones, (int)(t - t0));
        const uint32_t jt = (t / tm.nk) * kTile + ju, kt = (t % tm.nk) * kTile + ku;
        // the staged shapes that the tile's rays may meet, one per lane
        auto meets = [&](uint32_t nb) {
            const RayPrim& P = prims[min(lane, (int)nb - 1)];
            bool may = lane < (int)nb && cone_meets(cone, P);
            if (may)
                may = tile_meets(P, (double)jt + 0.5 * (kWaveTile - 1) - 0.5 * (double)(g.nu - 1),
                                 (double)kt + 0.5 * (kWaveTile - 1) - 0.5 * (double)(g.nv - 1), 0.5f * kWaveTile);
            return __ballot(may);
        };
        uint64_t first = 0;
        if constexpr (!kBatches) {
            if (K > 0) first = meets(K);
            if (first == 0 && skip_empty) continue;
        }
        // calls f(primitive, whether the ray takes part) for the shapes that the tile may
        // meet, from the last shape down; the whole wave takes every one of them
        auto each_shape = [&](bool want, auto&& f) {
            for (uint32_t end = K; end > 0;) {
                const uint32_t nb = min((uint32_t)kShapeBatch, end);
                end -= nb;
                if constexpr (kBatches) {
                    __syncthreads();
                    if (threadIdx.x < nb) stage_prim(shapes + end + threadIdx.x, specs, p, prims + threadIdx.x);
                    __syncthreads();
                }
                uint64_t mask = kBatches ? meets(nb) : first;
                while (mask) {
                    const int q = 63 - (int)__builtin_clzll(mask);
                    mask ^= 1ull << q;
                    f(prims[q], want);
                }
            }
        };
        const uint32_t j = jt + (lane >> 3), k = kt + (lane & 7);
        const bool in = j < nu && k < nv;
        const int64_t o = (int64_t)p * s0 + (int64_t)j * s1 + (int64_t)k * s2;
        const Tp base = in ? sino[o] : Tp(0);
        double tot = 0.0;
        bool overflow = false;
        for (uint32_t su = 0; su < ssu; su++) {
            double accu = 0.0;
            for (uint32_t sv = 0; sv < ssv; sv++) {
                const double a = (double)j - 0.5 + ((double)su + 0.5) / ssu - 0.5 * (double)(g.nu - 1);
                const double b = (double)k - 0.5 + ((double)sv + 0.5) / ssv - 0.5 * (double)(g.nv - 1);
                const d3 d = g.D - g.S + g.U * a + g.V * b;
                const double len = sqrt(dot(d, d));
                const bool live = in && len > 0.0;
                uint32_t nhit = 0;
                bool spill = false;
                double val = 0.0;
                Union U;
                union_clear(U);
                int used = 0;
                each_shape(live, [&](const RayPrim& P, bool want) {
                    double ta, tb;
                    bool hit = want && !spill && prim_interval(P, a, b, ta, tb);
                    // more than the reference's limit of intersections: flag
                    // it and ignore the rest (the reference drops the
                    // highest-index ones, this loop the lowest)
                    if (hit && ++nhit > kRefMaxIntersections) {
                        overflow = true;
                        hit = false;
                    }
                    bool grew = false;
                    if (hit) {
                        const double rho = (double)P.rho;
                        double un = tb - ta;
                        if (!additive) spill = !union_add(U, used, ta, tb, un, grew);
                        val += un * rho;   // a spilled ray's value is recomputed
                    }
                    used += __ballot(grew) != 0;
                });
                const bool again = kBatches ? __syncthreads_or(spill) != 0 : __ballot(spill) != 0;
                if (again) {
                    // the same with the pieces in memory, for the rays that need more of them
                    double pa[kManyPieces], pb[kManyPieces];
                    int n = 0;
                    bool over = false;
                    if (spill) val = 0.0;
                    each_shape(spill, [&](const RayPrim& P, bool want) {
                        double ta, tb;
                        if (!(want && !over && prim_interval(P, a, b, ta, tb))) return;
                        double un = tb - ta, na = ta, nb = tb;
                        int m = 0;
                        for (int i = 0; i < n; i++) {
                            const double ua = pa[i], ub = pb[i];
                            un -= fmax(0.0, fmin(tb, ub) - fmax(ta, ua));
                            if (ua <= nb && ub >= na) {
                                na = fmin(na, ua);
                                nb = fmax(nb, ub);
                            } else {
                                pa[m] = ua;
                                pb[m++] = ub;
                            }
                        }
                        over = m == kManyPieces;
                        if (over) return;
                        pa[m] = na;
                        pb[m] = nb;
                        n = m + 1;
                        val += un * (double)P.rho;
                    });
                    if (over) val = last_wins_exact(shapes, K, specs, p, a, b);
                }
                accu += val * len;
            }
            tot += accu / ssv;
        }
        tot /= ssu;
        if (!in) continue;
        if (overflow && oom) atomicAdd(oom, 1u);
        sino[o] = (Tp)((double)base + (double)mba * tot);
    }
}

template <typename Tv>
__global__ __launch_bounds__(256) void k_voxelise(
    const ap_forbild_shape* __restrict__ shapes, uint32_t K, double vw, double tpx, double tpy,
    double tpz, uint32_t ox, uint32_t oy, uint32_t oz, uint32_t cx, uint32_t cy, uint32_t cz,
    Tv* __restrict__ vol, int64_t v0, int64_t v1, int64_t v2, uint32_t ss) {
    __shared__ Prim prims[kShapeBatch];
    const uint32_t k = blockIdx.x * 64 + threadIdx.x;
    const uint32_t j = blockIdx.y * 4 + threadIdx.y;
    const uint32_t i = blockIdx.z;
    const bool in = k < cz && j < cy && i < cx;
    const uint32_t gi = i + ox, gj = j + oy, gk = k + oz;
    const int tid = threadIdx.y * 64 + threadIdx.x;
    const uint32_t npt = ss * ss * ss;
    // per sub-point value of the last containing shape; ss <= 4 => <= 64 points
    float val[64];
    for (uint32_t q = 0; q < npt && q < 64; q++) val[q] = 0.f;
    float val1 = 0.f;   // the one point of ss == 1, kept in a register
    // voxel centre in FP32 for the bounding-sphere cull; every sub-point lies
    // within the voxel's half-diagonal of it
    const float cf[3] = {(float)(tpx + (gi + 0.5) * vw), (float)(tpy + (gj + 0.5) * vw),
                         (float)(tpz + (gk + 0.5) * vw)};
    const float reach = (float)(0.8660254037844386 * vw);
    for (uint32_t k0 = 0; k0 < K; k0 += kShapeBatch) {
        const uint32_t nb = min((uint32_t)kShapeBatch, K - k0);
        __syncthreads();
        if (tid < (int)nb) make_prim(shapes[k0 + tid], prims[tid]);
        __syncthreads();
        if (!in) continue;
        for (uint32_t s = 0; s < nb; s++) {
            const Prim& P = prims[s];
            // outside the bounding sphere grown by the half-diagonal, with a
            // margin for the FP32 centre (shapes are visited in order, so the
            // last containing shape still wins)
            const float dx = cf[0] - P.bc[0], dy = cf[1] - P.bc[1], dz = cf[2] - P.bc[2];
            const float rr = P.br * 1.0001f + reach + 1e-3f;
            if (dx * dx + dy * dy + dz * dz > rr * rr) continue;
            if (ss == 1) {
                if (prim_contains(P, mkd3(tpx + (gi + 0.5) * vw, tpy + (gj + 0.5) * vw, tpz + (gk + 0.5) * vw)))
                    val1 = P.rho;
                continue;
            }
            for (uint32_t a = 0, q = 0; a < ss; a++)
                for (uint32_t b = 0; b < ss; b++)
                    for (uint32_t e = 0; e < ss; e++, q++) {
                        const double fx = ((double)a - 0.5 * (ss - 1.0)) / ss;
                        const double fy = ((double)b - 0.5 * (ss - 1.0)) / ss;
                        const double fz = ((double)e - 0.5 * (ss - 1.0)) / ss;
                        const d3 pnt = mkd3(tpx + (gi + 0.5 + fx) * vw, tpy + (gj + 0.5 + fy) * vw,
                                            tpz + (gk + 0.5 + fz) * vw);
                        if (prim_contains(P, pnt)) val[q] = P.rho;
                    }
        }
    }
    if (!in) return;
    float tot = val1;
    if (ss != 1) {
        tot = 0.f;
        for (uint32_t q = 0; q < npt; q++) tot += val[q];
        tot /= (float)npt;
    }
    const int64_t o = (int64_t)gi * v0 + (int64_t)gj * v1 + (int64_t)gk * v2;
    vol[o] = from_f32<Tv>(to_f32(vol[o]) + tot);
}

__global__ void k_bboxes(const ap_forbild_shape* __restrict__ shapes, uint32_t K, float* out) {
    const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= K) return;
    Prim P;
    make_prim(shapes[q], P);
    // extent of the reference shape mapped back: r = c + M^-1 y.  For the
    // unit reference shapes, half-extent along world axis w is
    //   cube: sum_a |Minv[w][a]|, ball: |Minv row w|_2,
    //   cylinder: |(Minv[w][0],Minv[w][1])|_2 + h |Minv[w][2]|.
    const double* M = P.M;
    const double det = M[0] * (M[4] * M[8] - M[5] * M[7]) - M[1] * (M[3] * M[8] - M[5] * M[6]) +
                       M[2] * (M[3] * M[7] - M[4] * M[6]);
    double Mi[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (det != 0.0) {
        const double id = 1.0 / det;
        Mi[0] = (M[4] * M[8] - M[5] * M[7]) * id;
        Mi[1] = (M[2] * M[7] - M[1] * M[8]) * id;
        Mi[2] = (M[1] * M[5] - M[2] * M[4]) * id;
        Mi[3] = (M[5] * M[6] - M[3] * M[8]) * id;
        Mi[4] = (M[0] * M[8] - M[2] * M[6]) * id;
        Mi[5] = (M[2] * M[3] - M[0] * M[5]) * id;
        Mi[6] = (M[3] * M[7] - M[4] * M[6]) * id;
        Mi[7] = (M[1] * M[6] - M[0] * M[7]) * id;
        Mi[8] = (M[0] * M[4] - M[1] * M[3]) * id;
    }
    for (int w = 0; w < 3; w++) {
        const double a = Mi[3 * w], b = Mi[3 * w + 1], e = Mi[3 * w + 2];
        double h;
        if (P.cls == kCube) h = fabs(a) + fabs(b) + fabs(e);
        else if (P.cls == kBall) h = sqrt(a * a + b * b + e * e);
        else if (P.cls == kCyl) h = sqrt(a * a + b * b) + P.h * fabs(e);
        else if (P.cls == kCone) h = P.cr * sqrt(a * a + b * b) + P.h * fabs(e);
        else h = 0.0;
        out[6 * q + w] = (float)(P.c[w] - h);
        out[6 * q + 3 + w] = (float)(P.c[w] + h);
    }
}

int32_t check_shapes(const ap_forbild_shape* shapes, uint32_t K) {
    if (K > 0 && !shapes) return ap_fail(AP_ERR_INVALID, "shapes is NULL");
    return AP_OK;
}

}  // namespace

extern "C" int32_t ap_project_forbild(const ap_config_cb_project_forbild* cfg,
                                      const ap_proj_spec* specs, uint32_t num_projs,
                                      const ap_forbild_shape* shapes, uint32_t num_shapes,
                                      const ap_array3* sino_desc, void* sino,
                                      uint32_t* out_of_mem_count, void* stream) {
    AP_REQUIRE(cfg && specs, "NULL config or specs");
    AP_REQUIRE(cfg->ssu >= 1 && cfg->ssv >= 1, "ssu and ssv must be >= 1");
    int32_t st = check_shapes(shapes, num_shapes);
    if (st) return st;
    if ((st = ap_check_array3(sino_desc, sino, "sino", false, false, true))) return st;
    AP_REQUIRE(sino_desc->shape[0] == num_projs, "sino has %u views, num_projs=%u",
               sino_desc->shape[0], num_projs);
    const uint32_t nu = sino_desc->shape[1], nv = sino_desc->shape[2];
    if (num_projs == 0 || nu == 0 || nv == 0) return AP_OK;
    AP_REQUIRE(num_projs <= 65535u, "at most 65535 views per call");
    const uint64_t npix = (uint64_t)nu * nv;
    AP_REQUIRE(npix < (1ull << 31), "detector too large");
    ForbildTiles tm;
    tm.nk = (nv + kTile - 1) / kTile;
    tm.total = ((nu + kTile - 1) / kTile) * tm.nk;
    // Staging the shapes takes a workgroup about 13 us: as many tiles as leave 4096
    // workgroups (three rounds of the GPU), at most 32 (at most 64: one lane each).
    // 40 primitives x 720 x 512^2: 4 tiles 3.85 ms, 16 2.74, 32 2.45, 64 2.45; scans of
    // 80-430 pixels and 30-440 views: 1024 workgroups 73-563 us, 4096 78-387, 8192 80-366.
    tm.per_block = (uint32_t)std::min<uint64_t>(
        32, std::max<uint64_t>(1, (uint64_t)tm.total * num_projs / 4096));
    dim3 grid((tm.total + tm.per_block - 1) / tm.per_block, num_projs, 1);
    hipStream_t s = (hipStream_t)stream;
    const bool one = cfg->ssu == 1 && cfg->ssv == 1, batches = num_shapes > (uint32_t)kShapeBatch;
    auto launch = [&](auto tp) {
        using Tp = decltype(tp);
        auto kern = batches ? (one ? k_project_forbild<Tp, true, true> : k_project_forbild<Tp, false, true>)
                            : (one ? k_project_forbild<Tp, true, false> : k_project_forbild<Tp, false, false>);
        hipLaunchKernelGGL(kern, grid, dim3(kProjThreads), 0, s, cfg->multiply_before_adding,
                           (int)cfg->overlap_addition, cfg->ssu, cfg->ssv, specs, shapes, num_shapes, tm, nu, nv,
                           sino_desc->strides[0], sino_desc->strides[1], sino_desc->strides[2], (Tp*)sino,
                           out_of_mem_count);
    };
    if (sino_desc->dtype == AP_F32) {
        launch(float{});
    } else if (sino_desc->dtype == AP_F64) {
        launch(double{});
    } else {
        return ap_fail(AP_ERR_UNSUPPORTED, "FORBILD sinogram must be F32 or F64");
    }
    return ap_check_launch("project_forbild");
}

extern "C" int32_t ap_voxelise_forbild(const ap_forbild_shape* shapes, uint32_t num_shapes,
                                       const ap_vol_tex_chunk_spec* chunk,
                                       const ap_array3* vol_desc, void* vol,
                                       uint32_t supersample, void* stream) {
    AP_REQUIRE(chunk, "chunk is NULL");
    AP_REQUIRE(supersample >= 1 && supersample <= 4, "supersample must be in 1..4");
    AP_REQUIRE(chunk->voxwid > 0.f, "voxwid must be positive");
    int32_t st = check_shapes(shapes, num_shapes);
    if (st) return st;
    if ((st = ap_check_array3(vol_desc, vol, "volume", true, true, false))) return st;
    const uint32_t off[3] = {chunk->offsets.x, chunk->offsets.y, chunk->offsets.z};
    const uint32_t shp[3] = {chunk->shape.x, chunk->shape.y, chunk->shape.z};
    for (int a = 0; a < 3; a++)
        AP_REQUIRE((uint64_t)off[a] + shp[a] <= vol_desc->shape[a], "chunk exceeds the volume");
    if (shp[0] == 0 || shp[1] == 0 || shp[2] == 0) return AP_OK;
    AP_REQUIRE(shp[0] <= 65535u, "chunk x extent above 65535");
    dim3 grid((shp[2] + 63) / 64, (shp[1] + 3) / 4, shp[0]);
    hipStream_t s = (hipStream_t)stream;
    return dispatch_dtype(vol_desc->dtype, [&](auto tv) -> int32_t {
        using Tv = decltype(tv);
        if constexpr (std::is_same<Tv, double>::value) {
            return ap_fail(AP_ERR_UNSUPPORTED, "float64 volumes are not supported");
        } else {
            hipLaunchKernelGGL(k_voxelise<Tv>, grid, dim3(64, 4, 1), 0, s, shapes, num_shapes,
                               (double)chunk->voxwid, (double)chunk->texpos.x, (double)chunk->texpos.y,
                               (double)chunk->texpos.z, off[0], off[1], off[2], shp[0], shp[1], shp[2],
                               (Tv*)vol, vol_desc->strides[0], vol_desc->strides[1],
                               vol_desc->strides[2], supersample);
            return ap_check_launch("voxelise_forbild");
        }
    });
}

extern "C" int32_t ap_forbild_bboxes(const ap_forbild_shape* shapes, uint32_t num_shapes,
                                     float* bboxes, void* stream) {
    int32_t st = check_shapes(shapes, num_shapes);
    if (st) return st;
    AP_REQUIRE(num_shapes == 0 || bboxes, "bboxes is NULL");
    if (num_shapes == 0) return AP_OK;
    hipLaunchKernelGGL(k_bboxes, dim3((num_shapes + 127) / 128), dim3(128), 0, (hipStream_t)stream,
                       shapes, num_shapes, bboxes);
    return ap_check_launch("forbild_bboxes");
}
