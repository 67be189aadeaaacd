// Device-side data layout and the pixel/strip footprint weight shared by every
// projector kernel.  Forward and adjoint evaluate a weight through the same inline
// functions on the same float inputs (per-ray table entries + integer pixel
// coordinates), so A and A^T are bitwise transposes of each other.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ctprj {

// Margin (pixels) added to every support bound.  Bounds only select candidates: the
// weight itself is exactly 0 outside the footprint, so a margin never changes a result.
constexpr float kSupportMargin = 0.02f;

// Word 3 of a raw (stride 0) buffer resource on the gfx9 family, gfx950 included: 32-bit
// data format, identity component selects.  Loads beyond num_records return 0.
constexpr int kBufferWord3 = 0x00020000;

// Symmetry group of a slice's view set used by the symmetric kernels (SliceDesc::sym).
// R rotates the pixel grid by 90 degrees, M reflects it in the x axis; element
// e = k + 4m is R^k M^m.  The group is the largest whose view maps are integral:
//   D4 (all eight elements) when prjFull % 4 == 0,
//   V4 = {1, R^2, M, R^2 M} when prjFull is even,
//   Z2 = {1, R^2 M} (theta -> -theta) for any prjFull.
enum : int { kGrpNone = 0, kGrpD4 = 1, kGrpV4 = 2, kGrpZ2 = 3 };

// View-row table of the symmetric slices: entry e of a canonical view locates the sinogram
// row of view e a0 as (byte offset of the row) | kRowFlip (bins read at 2pC - b) or
// kRowNone (view beyond np, e outside the slice's group, a reflection on a mirror view).
constexpr int kRowFlip = 1, kRowNone = 2;

// Element sets of a group as bit masks over e, and its canonical view range.
struct GroupMasks {
    unsigned all;        // the group's elements
    unsigned rot;        // its rotations
    unsigned fold;       // adjoint elements of a half-turn parallel scan
    int q;               // canonical views 0 <= a0 <= prjFull/q; mirror views a0 = 0, prjFull/q
    int order;           // number of elements
};

__host__ __device__ constexpr GroupMasks group_masks(int grp)
{
    // D4 fold set {1, R, M, R^3 M} maps (0, 45) degrees into [0, 180); V4's {1, M} maps
    // (0, 90) into [0, 180).  On a mirror view its rotations and its reflections each
    // reach every view once, too.  Z2 never folds (prjFull odd).
    return grp == kGrpD4   ? GroupMasks{0xFFu, 0x0Fu, 0x93u, 8, 8}
           : grp == kGrpV4 ? GroupMasks{0x55u, 0x05u, 0x11u, 4, 4}
           : grp == kGrpZ2 ? GroupMasks{0x41u, 0x01u, 0x00u, 2, 2}
                           : GroupMasks{0x01u, 0x01u, 0x00u, 1, 1};
}

// One slice of a plan.  Offsets are element offsets into the packed arrays.
struct SliceDesc {
    int n, W, np, fan;     // image edge, bins per view, views, 1 = fan beam
    int sym, fold;         // symmetry group (kGrp*); parallel beam folded over 180 deg
    int P, ncanon;         // prjFull; canonical views held in the view / ray tables
    int H;                 // (n-1)/2: pixel coordinates run over [-H, H]
    int half;              // n/2: coordinate -> index offset
    int pC;                // W/2: index of the bin at t = 0
    int blo, bhi;          // bins that carry rays: [pC-(W-1)/2, pC+(W-1)/2]
    float dSize, invDSize; // detector pitch
    float d, invd;         // source distance (fan), 0 for parallel
    float hbd;             // half beam width on the detector: dSize*effectiveRate/2
    float inver;           // 1/effectiveRate (outputs are divided by it)
    float fbp_scale;       // PI/np/dSize^2 (prj/cpuPrj.c:161,304)
    long long img_off, sino_off, view_off, ray_off;
    // symmetric slices: first entry of the view-row table; orbit image and orbit sinogram
    // (offsets into the workspaces of the slice's chunk, elements per row of one plane)
    long long tab_off, orb_off, os_off;
    int orb_pitch, os_pitch;
    // groups of four into which a plan of its own shape cuts a forward item's rows and a tile's
    // views: by this slice alone, so that its sums are the same whatever else the plan holds
    int fgroups, agroups;
};

// Per-ray footprint constants.  Parallel beam: one entry per view (dc unused, the bin
// position is (b-pC)*dSize).  Fan beam: one entry per (view, bin).
struct __attribute__((aligned(16))) Ray {
    float cosR, sinR;  // unit normal of the ray line: dist = x*cosR + y*sinR - dc
    float dc;          // offset of the ray line from the rotation centre
    float hbc;         // half strip width at the isocentre, perpendicular to the ray
    // the pixel's footprint on the detector normal, a trapezoid of plateau half width
    // b1 = (max - min)/2 between ramps of width s = min(|cosR|, |sinR|), s and b1 taken as at
    // least 2^-24 and 2^-25
    float is;          // 1/s
    float c2;          // (b1 + s)/s
    float ib;          // 1/(2 b1)
    float a;           // share of one ramp in the footprint's area, s/2 / (s + 2 b1)
};

// x clamped to [0, 1]: the clamp modifier of the instruction that forms x.
__device__ __forceinline__ float sat(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, 1.0f); }

// Area of overlap of the unit pixel centred `dist` from the ray line with the strip of
// half width hb (prj/utils.h:12-92 computes the same area by a 20-way case split).  The
// integral of the pixel's footprint over [-hb - |dist|, hb - |dist|] is, with
// q = hb - |dist|, p = hb + |dist| and every ramp and the plateau measured in its own width,
//   ramps    t(q)^2 + (1 - t(-q)^2) - t(-p)^2,  t(u) = sat(u/s + (b1 + s)/s)
//   plateau  D = sat(q/(2 b1) + 1/2) - sat(-p/(2 b1) + 1/2)
//   area     a (ramps) + (1 - 2a) D.
// gfx950 issues a wave's fma, add and mul in 2 cycles but a med3, min or max in 4, and a
// clamp to [0, 1] is free: 13 such instructions, 26 cycles, where the difference of the
// cumulative integral at both ends, with six med3, took 68.  Error against 64 bits over all
// angles: 2.1e-8 rms at hb = 0.5 (that form: 3.0e-8) and smaller than its at every hb from
// 0.15 to 4.  Small areas at the strip's edge keep their relative accuracy, and outside the
// footprint the area is exactly 0.  Evaluated at |dist| like the reference (the footprint is
// symmetric), which makes the float result of the pixel reflected through the ray identical
// bit for bit.
__device__ __forceinline__ float strip_area(float dist, float hb, const Ray& r)
{
    const float ad = fabsf(dist), q = hb - ad, p = hb + ad;
    const float t1 = sat(fmaf(q, r.is, r.c2)), t3 = sat(fmaf(-q, r.is, r.c2));
    const float t4 = sat(fmaf(-p, r.is, r.c2));
    const float D = sat(fmaf(q, r.ib, 0.5f)) - sat(fmaf(-p, r.ib, 0.5f));
    const float ramps = fmaf(-t4, t4, fmaf(t1, t1, fmaf(-t3, t3, 1.0f)));
    return fmaf(r.a, fmaf(-2.0f, D, ramps), D);
}

// Whether that overlap is a non-zero FP32 number when it is formed as the difference of
// the footprint's cumulative integral at the strip's two edges (the count of A's entries).
__device__ __forceinline__ bool strip_hits(float dist, float hb, const Ray& r)
{
    const float c = fabsf(r.cosR), n = fabsf(r.sinR);
    const float s = fminf(c, n), b1 = 0.5f * (fmaxf(c, n) - s), b2 = b1 + s;
    const float k = s > 0.0f ? 0.5f / s : 0.0f, ad = fabsf(dist);
    auto upto = [&](float u) {
        const float u1 = __builtin_amdgcn_fmed3f(u + b2, 0.0f, s);
        const float u2 = __builtin_amdgcn_fmed3f(u + b1, 0.0f, b1 + b1);
        const float u3 = __builtin_amdgcn_fmed3f(u - b1, 0.0f, s);
        return (u2 + u3) + k * ((u1 - u3) * (u1 + u3));
    };
    return upto(hb - ad) != upto(-hb - ad);
}

// Hardware reciprocal (about 1 ulp): used only where a result selects candidates and
// is padded by kSupportMargin, never in a weight.
__device__ __forceinline__ float fast_rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// Signed distance of pixel (x, y) from the ray line.
__device__ __forceinline__ float ray_dist(float x, float y, float cosR, float sinR, float dc)
{
    return fmaf(x, cosR, fmaf(y, sinR, -dc));
}

// Fan beam: strip width at the pixel relative to the isocentre width,
// 1 + (x sinT - y cosT)/d (prj/cpuPrj.c:549, 254); along an image row all but one
// operation are the row's.
__device__ __forceinline__ float fan_depth_scale(float x, float y, float cosT, float sinT,
                                                 float invd)
{
    return fmaf(x, sinT * invd, fmaf(-y, cosT * invd, 1.0f));
}

// Candidate range along a row (or column) of the walk: the pixels whose footprint can
// meet the strip, |dist| < b2 + hb(x, y), solved as two linear inequalities in the
// inner coordinate u for the walk coordinate v:
//   u in [min(U(v)*iu, L(v)*il), max(...)],  U(v) = U0 - v*U1,  L(v) = L0 - v*L1.
struct RowBounds {
    float U0, U1, L0, L1, iu, il;
};

__device__ __forceinline__ RowBounds row_bounds(const Ray& r, float cT, float sT, float invd,
                                                bool rowmode)
{
    RowBounds rb;
    const float b2 = 0.5f * (fabsf(r.cosR) + fabsf(r.sinR));
    const float m = kSupportMargin;
    const float al = r.hbc * sT * invd;  // d(hb)/dx
    const float be = r.hbc * cT * invd;  // -d(hb)/dy
    rb.U0 = r.dc + b2 + r.hbc + m;
    rb.L0 = r.dc - b2 - r.hbc - m;
    if (rowmode) {  // u = x, v = y
        rb.U1 = r.sinR + be;
        rb.L1 = r.sinR - be;
        rb.iu = 1.0f / (r.cosR - al);
        rb.il = 1.0f / (r.cosR + al);
    } else {        // u = y, v = x
        rb.U1 = r.cosR - al;
        rb.L1 = r.cosR + al;
        rb.iu = 1.0f / (r.sinR + be);
        rb.il = 1.0f / (r.sinR - be);
    }
    return rb;
}

__device__ __forceinline__ void row_range(const RowBounds& rb, float v, int H, int& lo, int& hi)
{
    const float ua = fmaf(-v, rb.U1, rb.U0) * rb.iu;
    const float ub = fmaf(-v, rb.L1, rb.L0) * rb.il;
    const float fH = (float)H;
    lo = (int)ceilf(fmaxf(fminf(ua, ub), -fH - 1.0f));
    hi = (int)floorf(fminf(fmaxf(ua, ub), fH + 1.0f));
    lo = max(lo, -H);
    hi = min(hi, H);
}

// Compensated accumulation of a partial sum (Kahan): keeps the long sums over rows /
// views at FP32 rounding of the result instead of growing with the term count.
struct KahanAcc {
    float s = 0.0f, c = 0.0f;
    __device__ __forceinline__ void add(float v)
    {
        const float y = v - c;
        const float t = s + y;
        c = (t - s) - y;
        s = t;
    }
};

}  // namespace ctprj
