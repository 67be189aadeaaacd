// Symmetric projector kernels for gfx950.
//
// The view set of a scan over a full (or half) turn is closed under a symmetry group of
// the pixel grid.  With P = prjFull,
//   R  (rotate +90):          pixel (x, y) -> (-y, x),  ray (a, b) -> (a + P/4, b)
//   M  (reflect in the x axis): pixel (x, y) -> (x, -y), ray (a, b) -> (P/2 - a, 2pC - b)
// (views mod P; prj/cpuPrj.c:401-460 writes the same eight images for P % 4 == 0).
// Element e = k + 4m is R^k M^m.  A slice uses the largest group whose view maps are
// integral: D4 (all eight) for P % 4 == 0, V4 = {1, R^2, M, R^2 M} for even P, and
// Z2 = {1, R^2 M} (theta -> -theta) otherwise.  Every weight is evaluated once, for a
// canonical view a0 in [0, P/q] (q = 8, 4, 2), and reused for the group's images:
//   A[(g a0, g b), g p] = W(a0, b, p)  for g in the group,
// which fixes the float value of every matrix entry, so forward and adjoint stay
// bitwise transposes.  Canonical views on a mirror line (a0 = 0, a0 = P/q) use the
// rotations only, otherwise each view would be counted twice.
// Parallel beam over half a turn (np <= P/2, "fold"; D4 and V4): ray (a + P/2, b) is ray
// (a, 2pC - b); the adjoint uses a half set of elements that maps the canonical range
// into [0, 180) and folds, the forward takes half the detector with all the images.
// |dist| in the weight makes W(a0, b, p) == W(a0, 2pC - b, R^2 p) exactly.
#include "ctprj_internal.h"
#include <type_traits>

#include "bhc_device.h"

namespace ctprj {

// (k, m) action on pixel coordinates: reflect first, then rotate k times.
__device__ __forceinline__ void apply_px(int k, int m, int x, int y, int& ox, int& oy)
{
    if (m) y = -y;
    switch (k & 3) {
        case 0: ox = x; oy = y; break;
        case 1: ox = -y; oy = x; break;
        case 2: ox = -x; oy = -y; break;
        default: ox = y; oy = -x; break;
    }
}

// (k, m) action on (canonical view a0, bin b) -> (view, sign, offset): bin = off + sign*b.
// 4 v = (+-4 a0) + (k + 2m) P, a multiple of 4 for every element of the slice's group.
// Views beyond np read a zero row (the caller checks v < np).
__device__ __forceinline__ int map_view(const SliceDesc& S, int k, int m, int a0, int& sign,
                                        int& off)
{
    const int P = S.P;
    // a0 <= P/2, so v starts in [-P/2, 7P/2): reduce mod P without a division
    int v = ((m ? -4 * a0 : 4 * a0) + ((k + 2 * m) & 3) * P) >> 2;
    if (v < 0) v += P;
    if (v >= 2 * P) v -= 2 * P;
    if (v >= P) v -= P;
    sign = m ? -1 : 1;
    off = m ? 2 * S.pC : 0;
    if (S.fold && 2 * v >= P) {
        v -= P >> 1;
        sign = -sign;
        off = 2 * S.pC - off;
    }
    return v;
}

// Per canonical view, what the candidate bins of a pixel need (wave-uniform values).  With
// the pixel's centre at (oc, qe) across and along the central ray and
// rho = (|cos| + |sin|) / 2 half the pixel's extent in any direction, the strips that meet
// the pixel, |dist| < b2 + hb in the weight's terms, are those of the bins at t between
//   parallel: oc -+ (rho + hbd);   fan: (d (oc -+ rho) -+ hbd qe) / (qe +- rho),
// hbd being half the strip's width on the detector (fan: the ray at t has
// dist = (d oc - t qe) / sqrt(d^2 + t^2), and its footprint is at most
// (d m + t n) / (2 sqrt(d^2 + t^2)) wide, |m|, |n| <= 2 rho), and kSupportMargin px more are
// taken.  The sign before rho in the fan's denominator is the numerator's on the left, its
// opposite on the right: the smaller (larger) of two ratios of linear functions of the
// pixel, so over a square of pixels the extreme bounds are those of its corner pixels.
template <bool FAN>
struct BinBounds {
    float cT, sT, rho, d, hbd, scale, left, right;
    int blo, bhi;

    // last: the last bin of the lane's pixels (below the first: none)
    __device__ __forceinline__ BinBounds(const SliceDesc& S, float c, float s, const Ray& r, int last)
        : cT(c), sT(s), d(S.d), hbd(S.hbd), scale(S.invDSize), blo(S.blo), bhi(last)
    {
        rho = 0.5f * (fabsf(c) + fabsf(s));
        const float m = FAN ? kSupportMargin * S.dSize : rho + r.hbc + kSupportMargin;
        left = (float)S.pC - m * S.invDSize;
        right = (float)S.pC + m * S.invDSize;
    }
    __device__ __forceinline__ void operator()(float fx, float fy, int& lo, int& hi) const
    {
        const float oc = fmaf(fx, cT, fy * sT);
        float l = oc, h = oc;
        if (FAN) {
            const float qe = fmaf(fx, sT, fmaf(-fy, cT, d)), hq = hbd * qe;
            const float a = fmaf(d, oc - rho, -hq), b = fmaf(d, oc + rho, hq);
            l = a * fast_rcp(qe + copysignf(rho, a));
            h = b * fast_rcp(qe - copysignf(rho, b));
        }
        lo = max((int)ceilf(fmaf(l, scale, left)), blo);
        hi = min((int)fmaf(h, scale, right), bhi);  // towards 0: at least the last bin
    }
};

// The sum of a RedJob by one wave: lane l adds in[l], in[l + 64], ... in order, then a
// butterfly over the lanes; the order is fixed, so every caller gets the same value.
__device__ __forceinline__ void wave_sum_job(const RedJob& job)
{
    const int lane = (int)threadIdx.x & 63;
    double acc = 0.0;
    for (long long q = lane; q < job.n; q += 64) acc += job.in[q];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) *job.out = acc;
}

__global__ __launch_bounds__(64) void k_wave_sum(const RedJob job) { wave_sum_job(job); }

void launch_wave_sum(const RedJob& job, hipStream_t st)
{
    hipLaunchKernelGGL(k_wave_sum, dim3(1), dim3(64), 0, st, job);
}

// ------------------------------------------------------------------ forward ---

// Rows are summed in plain FP32 over blocks of kRowBlock rows, and the block sums are
// added with compensation: the long sum over rows stays at FP32 rounding of the result
// while the compensation costs a quarter of a per-row update.
constexpr int kRowBlock = 4;

// Raw buffer view of `bytes` bytes from a wave-uniform base: loads take a wave-uniform
// byte offset in an SGPR and a 32-bit per-lane byte offset, and return 0 past the end.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const float* base, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, bytes,
                                             kBufferWord3);
}

__device__ __forceinline__ float4 ldb128(__amdgpu_buffer_rsrc_t r, int voff, int soff)
{
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
    return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]),
                       __uint_as_float(v[3]));
}

// Orders this wave's LDS writes before its later reads (and reads before later writes).
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Wave minimum of lo and maximum of hi: prefix reductions inside each row of 16 lanes
// (DPP row shifts; lanes with no source read the operation's identity, which lets the
// compiler fold each shift into the min / max), then the four rows' last lanes.  The
// two chains are interleaved so that each DPP read finds its operand already written.
__device__ __forceinline__ void wave_range_i32(int lo, int hi, int& wlo, int& whi)
{
    lo = min(lo, __builtin_amdgcn_update_dpp(INT_MAX, lo, 0x111, 0xf, 0xf, false));
    hi = max(hi, __builtin_amdgcn_update_dpp(INT_MIN, hi, 0x111, 0xf, 0xf, false));
    lo = min(lo, __builtin_amdgcn_update_dpp(INT_MAX, lo, 0x112, 0xf, 0xf, false));
    hi = max(hi, __builtin_amdgcn_update_dpp(INT_MIN, hi, 0x112, 0xf, 0xf, false));
    lo = min(lo, __builtin_amdgcn_update_dpp(INT_MAX, lo, 0x114, 0xf, 0xf, false));
    hi = max(hi, __builtin_amdgcn_update_dpp(INT_MIN, hi, 0x114, 0xf, 0xf, false));
    lo = min(lo, __builtin_amdgcn_update_dpp(INT_MAX, lo, 0x118, 0xf, 0xf, false));
    hi = max(hi, __builtin_amdgcn_update_dpp(INT_MIN, hi, 0x118, 0xf, 0xf, false));
    const int a = __builtin_amdgcn_readlane(lo, 15), b = __builtin_amdgcn_readlane(lo, 31);
    const int c = __builtin_amdgcn_readlane(lo, 47), d = __builtin_amdgcn_readlane(lo, 63);
    const int e = __builtin_amdgcn_readlane(hi, 15), f = __builtin_amdgcn_readlane(hi, 31);
    const int g = __builtin_amdgcn_readlane(hi, 47), h = __builtin_amdgcn_readlane(hi, 63);
    wlo = min(min(a, b), min(c, d));
    whi = max(max(e, f), max(g, h));
}

// ------------------------------------------------------------ orbit image ---
//
// The forward reads its pixels from the orbit image: for every pixel p of the walk, the
// group's values img[g p] side by side, so that a ray's step to the next pixel is one
// contiguous read for all the images instead of one read per image.  Rows are walk rows
// v, columns u in [-H, H] (orb_pitch of them).  One row holds, for each u,
//   D4: plane 0 = elements 0..3, plane 1 = elements 4..7 (orb_pitch float4 each),
//   V4: elements 0, 2, 4, 6 (float4),   Z2: elements 0, 6 (float2).
// Rows mode (v = y, u = x) comes first, then, for V4 and Z2, columns mode (v = x, u = y)
// of the canonical views steeper than 45 degrees.  Rows v < 0 are not stored where an
// element of the group maps v to -v and keeps u (all but Z2's rows mode): there the
// values at -v are those at v with the slots exchanged (neg_xor), and the forward
// exchanges its sums once, where the walk crosses v = 0.  The orbit image of a slice
// takes 4 n^2 floats (Z2: 3 n^2).
template <int GRP>
struct Orbit {
    static constexpr int N = group_masks(GRP).order;
    static constexpr int kPlane = N >= 4 ? 4 : 2;  // floats of one pixel in one plane
    // pixels of a row that a wave stages at once, and the 16-byte loads per lane it takes
    static constexpr int kPixels = 128;
    static constexpr int kLoads = kPixels * N / 256;
    __host__ __device__ static constexpr int elem(int s)
    {
        return GRP == kGrpD4 ? s : GRP == kGrpV4 ? 2 * s : 6 * s;
    }
    __host__ __device__ static constexpr int slot(int e)
    {
        return GRP == kGrpD4 ? e : GRP == kGrpV4 ? e >> 1 : (e != 0);
    }
    // slot s at walk row -v is slot s ^ neg_xor at v; 0: the rows v < 0 are stored
    __host__ __device__ static constexpr int neg_xor(bool cols)
    {
        return GRP == kGrpD4 ? 4 : GRP == kGrpV4 ? (cols ? 3 : 2) : (cols ? 1 : 0);
    }
};

// Walk row v of the orbit image of S (floats from the slice's base).
template <int GRP, bool COLS>
__device__ __forceinline__ const float* orbit_row(const SliceDesc& S, const float* orb, int v)
{
    using O = Orbit<GRP>;
    const int rec = O::N * S.orb_pitch;
    const float* base = orb + S.orb_off;
    if (COLS) base += (long long)(O::neg_xor(false) ? S.H + 1 : 2 * S.H + 1) * rec;
    return base + (long long)(O::neg_xor(COLS) ? abs(v) : v + S.H) * rec;
}

// One 32 x 32 tile of the orbit image per work-group: item (slice, first stored row, first
// column; pad = 1: columns mode).  Images whose u runs along image columns are read
// straight, the others through an LDS transpose, so every read and write is coalesced.
// Bound by its writes (16 n^2 bytes): one extra pass over a small array, 11 us at 1024^2.
template <int GRP, bool COLS>
__device__ __forceinline__ void orbit_tile(const SliceDesc& S, int r0, int u0,
                                           const float* __restrict__ img,
                                           float* __restrict__ orb, float (*tile)[32][33])
{
    using O = Orbit<GRP>;
    constexpr int neg = O::neg_xor(COLS);
    const int H = S.H, tx = (int)threadIdx.x & 31, ty = (int)threadIdx.x >> 5;
    const float* src = img + S.img_off + (long long)S.half * S.n + S.half;
    const int v0 = neg ? r0 : r0 - H;
    // u is a row index of the source where the element's rotation (and the walk) swap axes
    constexpr auto swapped = [](int e) constexpr { return ((e & 1) != 0) != COLS; };
#pragma unroll
    for (int s = 0; s < O::N; ++s) {
        const int e = O::elem(s);
        if (!swapped(e)) continue;
#pragma unroll
        for (int k = 0; k < 32; k += 8) {
            const int v = v0 + tx, u = u0 - H + ty + k;
            int x, y;
            apply_px(e & 3, e >> 2, COLS ? v : u, COLS ? u : v, x, y);
            if (v <= H && u <= H) tile[s >> (O::N == 8 ? 1 : 0)][ty + k][tx] = src[(long long)y * S.n + x];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 32; k += 8) {
        const int v = v0 + ty + k, u = u0 - H + tx;
        if (v > H || u > H) continue;
        float q[O::N];
#pragma unroll
        for (int s = 0; s < O::N; ++s) {
            const int e = O::elem(s);
            if (swapped(e)) q[s] = tile[s >> (O::N == 8 ? 1 : 0)][tx][ty + k];
            else {
                int x, y;
                apply_px(e & 3, e >> 2, COLS ? v : u, COLS ? u : v, x, y);
                q[s] = src[(long long)y * S.n + x];
            }
        }
        float* out = const_cast<float*>(orbit_row<GRP, COLS>(S, orb, v));
        const int c = u + H;
        if constexpr (O::N == 2) {
            reinterpret_cast<float2*>(out)[c] = make_float2(q[0], q[1]);
        } else {
#pragma unroll
            for (int p = 0; p < O::N / 4; ++p)
                reinterpret_cast<float4*>(out)[p * S.orb_pitch + c] =
                    make_float4(q[4 * p], q[4 * p + 1], q[4 * p + 2], q[4 * p + 3]);
        }
    }
}

__global__ __launch_bounds__(256) void k_orbit_image(const SliceDesc* __restrict__ slices,
                                                     const AdjItem* __restrict__ items,
                                                     const float* __restrict__ img,
                                                     float* __restrict__ orb)
{
    __shared__ float tile[4][32][33];
    const AdjItem it = items[blockIdx.x];
    const SliceDesc S = slices[it.slice];
    // uniform over the work-group
    if (S.sym == kGrpD4) orbit_tile<kGrpD4, false>(S, it.row0, it.col0, img, orb, tile);
    else if (S.sym == kGrpV4 && !it.pad) orbit_tile<kGrpV4, false>(S, it.row0, it.col0, img, orb, tile);
    else if (S.sym == kGrpV4) orbit_tile<kGrpV4, true>(S, it.row0, it.col0, img, orb, tile);
    else if (!it.pad) orbit_tile<kGrpZ2, false>(S, it.row0, it.col0, img, orb, tile);
    else orbit_tile<kGrpZ2, true>(S, it.row0, it.col0, img, orb, tile);
}

void launch_orbit_image(int nitems, const SliceDesc* desc, const AdjItem* items, const float* img,
                        float* orb, hipStream_t st)
{
    if (nitems > 0)
        hipLaunchKernelGGL(k_orbit_image, dim3(nitems), dim3(256), 0, st, desc, items, img, orb);
}

// ------------------------------------------------------------------ ray walk ---

// One canonical ray per lane against the group's images of the pixels it meets, over the
// walk rows [vlo, vhi].  Rows mode walks v = y with u = x inside, columns mode (canonical
// views steeper than 45 degrees) v = x with u = y.  The wave stages the orbit-image row
// that its 64 neighbouring rays cross in LDS (one 16-byte load per lane brings 64 16-byte
// units; the next row is loaded while this one is summed), and every lane then reads its
// own pixels [lo, hi] there.  Read straight from memory, a row took eight 16-byte loads
// per lane (one per image) and the vector-memory unit, at about 16 cycles a load, bounded
// the kernel; now three loads serve the wave's row.
// The staged columns start at the first pixel of an end lane (the rays of a wave are
// ordered).  Waves for which that does not hold over all of their rows, or whose rays
// cross more than kPixels pixels of a row (coarse detectors), go another way:
//   V4, Z2  each lane reads its own pixels straight from the orbit image, one load a pixel:
//       hardly a pixel is shared between lanes, and a row staged in pieces leaves the lanes
//       of the other pieces idle.  Forward, us, staged piece by piece with every load waited
//       for / so: 1024^2 fan of 181 views, pitch 4: 342 / 181, pitch 7: 595 / 286; 512^2, pitch
//       2.5: 90 / 59; 1024^2 parallel of 181, pitch 2: 160 / 113.
//   D4  two loads a pixel, 64 lines each, would bound the walk (512^2 fan of 720 views, pitch 4:
//       205); the wave forms its true range of pixels and stages it piece by piece, the next
//       piece or row being on its way: 138 / 125 there, 1024^2 fan of 180 views, pitch 3: 208 / 190.
template <bool FAN, int GRP, bool COLS>
__device__ __forceinline__ void fwd_sym_rows(const SliceDesc& S, const Ray& r, float cT, float sT,
                                             const float* __restrict__ orb, int vlo, int vhi,
                                             KahanAcc* acc, float4* __restrict__ st)
{
    using O = Orbit<GRP>;
    constexpr int N = O::N, CH = O::kPixels, neg = O::neg_xor(COLS);
    const int lane = (int)threadIdx.x & 63, H = S.H;
    if (vlo > vhi) return;  // uniform over the wave
    const float fH = (float)H, qs = sT * S.invd, qc = cT * S.invd;
    // The pixels of walk row v that the lane's ray meets are u in [lo, hi] (bounds as in
    // row_range) between two lines in v, (ua + v ub) and (la + v lb).
    const RowBounds rb = row_bounds(r, cT, sT, FAN ? S.invd : 0.0f, !COLS);
    const float ua = rb.U0 * rb.iu, ub = -rb.U1 * rb.iu, la = rb.L0 * rb.il, lb = -rb.L1 * rb.il;
    // Regular waves: at the first and the last row, and hence (all are linear in v) at every
    // row between, each lane's lines keep their order, no lane starts more than a pixel
    // before the end lane `edge` that starts first at both, and all end within the staged
    // pixels.
    const float fa = (float)vlo, fb = (float)vhi;
    const float ea = fmaf(fa, ub, ua), eb = fmaf(fb, ub, ua);
    const float ga = fmaf(fa, lb, la), gb = fmaf(fb, lb, la);
    const bool left = ga + gb <= ea + eb;  // the second line is the left one
    const float La = left ? ga : ea, Lb = left ? gb : eb, Ra = left ? ea : ga, Rb = left ? eb : gb;
    auto lane_f = [](float x, int l) {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
    };
    const int edge = lane_f(La, 0) + lane_f(Lb, 0) <= lane_f(La, 63) + lane_f(Lb, 63) ? 0 : 63;
    const float sa = lane_f(La, edge), sb = lane_f(Lb, edge);
    // (the image's width bounds the pixels, too)
    auto within = [&](float px) { return (Ra - sa < px && Rb - sb < px) || 2.0f * fH < px; };
    const bool regular = __all(La <= Ra && Lb <= Rb && La >= sa - 0.9f && Lb >= sb - 0.9f &&
                               within((float)(CH - 3)));
    const bool wide = !__all(within(61.0f));
    const float l0 = left ? la : ua, l1 = left ? lb : ub, r0 = left ? ua : la, r1 = left ? ub : lb;
    // the lane's pixels of row fv
    auto row_range = [&](float fv, float& lo, float& hi) {
        const float e = fmaf(fv, l1, l0), f = fmaf(fv, r1, r0);
        if (regular) {
            lo = fmaxf(ceilf(e), -fH);
            hi = fminf(f, fH);
        } else {
            lo = fmaxf(ceilf(fminf(e, f)), -fH);
            hi = fminf(fmaxf(e, f), fH);
        }
    };
    float part[N];
#pragma unroll
    for (int s = 0; s < N; ++s) part[s] = 0.0f;
    // the weight at pixel fu of a row of rowd, rowq (of fv in columns mode)
    auto weight = [&](float fu, float fv, float rowd, float rowq) {
        // ray_dist and fan_depth_scale at (x, y) = (fu, fv), columns mode (fv, fu)
        const float dist = COLS ? fmaf(fv, r.cosR, fmaf(fu, r.sinR, -r.dc)) : fmaf(fu, r.cosR, rowd);
        const float qd = COLS ? fmaf(fv, qs, fmaf(-fu, qc, 1.0f)) : fmaf(fu, qs, rowq);
        return strip_area(dist, FAN ? r.hbc * qd : r.hbc, r);
    };
    auto flush = [&]() {
#pragma unroll
        for (int s = 0; s < N; ++s) {
            acc[s].add(part[s]);
            part[s] = 0.0f;
        }
    };
    // 16-byte unit 64 j + lane of a staged row: pixel unit % CH of plane unit / CH; units
    // past a narrow wave's pixels are not read (offsets beyond the row load as 0)
    int voff[O::kLoads];
#pragma unroll
    for (int j = 0; j < O::kLoads; ++j) {
        const int unit = 64 * j + lane;
        voff[j] = N == 8 && unit >= CH ? (S.orb_pitch + unit - CH) * 16 : unit * 16;
        if (N >= 4 && (j & 1) && !wide) voff[j] = 0x7ffffff0;
    }
    // rows v < 0 first, then v >= 0: the sums are held by the slots of the current sign
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        const int va = half ? max(vlo, 0) : vlo, vb = half ? vhi : min(vhi, -1);
        const float* row = va <= vb ? orbit_row<GRP, COLS>(S, orb, va) : nullptr;
        const long long step = neg && !half ? -(long long)N * S.orb_pitch : N * S.orb_pitch;
        float fv = (float)va, lo, hi;
        if (va <= vb && (regular || N == 8)) {
            // the first staged column of row fv, and (D4's irregular waves) the wave's last pixel
            int c0, last = INT_MIN;
            auto column = [&]() {
                if (N < 8 || regular) {
                    // one pixel of slack; a row that no lane meets takes any column, so that
                    // its load stays inside
                    c0 = min(max(__builtin_amdgcn_readlane((int)fminf(lo, fH), edge) - 1, -H), H);
                } else {
                    const bool any = lo <= hi;
                    wave_range_i32(any ? (int)lo : INT_MAX, any ? (int)hi : INT_MIN, c0, last);
                    c0 = min(c0, H);
                }
            };
            auto load = [&](int c0, float4* g) {
                const __amdgpu_buffer_rsrc_t R = row_rsrc(row, N * S.orb_pitch * 4);
#pragma unroll
                for (int j = 0; j < O::kLoads; ++j) g[j] = ldb128(R, voff[j], (c0 + H) * O::kPlane * 4);
            };
            float4 g[O::kLoads];
            row_range(fv, lo, hi);
            column();
            load(c0, g);
#pragma unroll 1
            for (int v = va; v <= vb;) {
                const int vend = min(v + kRowBlock - 1, vb);
#pragma unroll 1
                for (; v <= vend;) {
                    wave_lds_sync();  // the previous row's reads are done
#pragma unroll
                    for (int j = 0; j < O::kLoads; ++j) st[64 * j + lane] = g[j];
                    wave_lds_sync();  // staged values visible to every lane
                    const float pv = fv;
                    float plo = lo, phi = hi;
                    int at = (int)fminf(lo, fH) - c0;
                    bool more = false;  // (wave-uniform) pixels of this row past the staged ones
                    if (N == 8 && !regular) {
                        phi = fminf(hi, (float)(c0 + CH - 1));
                        more = c0 + CH <= last;
                    }
                    if (more) {
                        c0 += CH;
                        lo = fmaxf(lo, (float)c0);
                        load(c0, g);
                    } else {
                        if (v < vb) {
                            fv += 1.0f;
                            row += step;
                            row_range(fv, lo, hi);
                            column();
                            load(c0, g);
                        }
                        ++v;
                    }
                    const float rowd = COLS ? 0.0f : fmaf(pv, r.sinR, -r.dc);
                    const float rowq = FAN && !COLS ? fmaf(-pv, qc, 1.0f) : 0.0f;
                    for (float fu = plo; fu <= phi; fu += 1.0f, ++at) {
                        float q[N];
                        if constexpr (N == 2) {
                            const float2 a = reinterpret_cast<const float2*>(st)[at];
                            q[0] = a.x;
                            q[1] = a.y;
                        } else {
#pragma unroll
                            for (int p = 0; p < N / 4; ++p) {
                                const float4 a = st[p * CH + at];
                                q[4 * p] = a.x;
                                q[4 * p + 1] = a.y;
                                q[4 * p + 2] = a.z;
                                q[4 * p + 3] = a.w;
                            }
                        }
                        const float w = weight(fu, pv, rowd, rowq);
#pragma unroll
                        for (int s = 0; s < N; ++s) part[s] = fmaf(w, q[s], part[s]);
                    }
                }
                flush();
            }
        } else if (N < 8 && va <= vb) {
            // straight from memory, a pixel (and, at its end, the next row's first) ahead
            auto load = [&](int at, float* q) {  // past the row's end: 0, or the next plane's
                const __amdgpu_buffer_rsrc_t R = row_rsrc(row, N * S.orb_pitch * 4);
                if constexpr (N == 2) {
                    const auto a = __builtin_amdgcn_raw_buffer_load_b64(R, at, 0, 0);
                    q[0] = __uint_as_float(a[0]);
                    q[1] = __uint_as_float(a[1]);
                } else {
#pragma unroll
                    for (int p = 0; p < N / 4; ++p) {
                        const float4 a = ldb128(R, at, p * S.orb_pitch * 16);
                        q[4 * p] = a.x;
                        q[4 * p + 1] = a.y;
                        q[4 * p + 2] = a.z;
                        q[4 * p + 3] = a.w;
                    }
                }
            };
            float q[N];
            auto begin = [&](int& at) {
                row_range(fv, lo, hi);
                at = (int)(fminf(lo, fH) + fH) * (O::kPlane * 4);
                load(at, q);
            };
            int at;
            begin(at);
#pragma unroll 1
            for (int v = va; v <= vb;) {
                const int vend = min(v + kRowBlock - 1, vb);
#pragma unroll 1
                for (; v <= vend; ++v) {
                    const float rowd = COLS ? 0.0f : fmaf(fv, r.sinR, -r.dc);
                    const float rowq = FAN && !COLS ? fmaf(-fv, qc, 1.0f) : 0.0f;
                    for (float fu = lo; fu <= hi; fu += 1.0f) {
                        float next[N];
                        at += O::kPlane * 4;
                        load(at, next);
                        const float w = weight(fu, fv, rowd, rowq);
#pragma unroll
                        for (int s = 0; s < N; ++s) part[s] = fmaf(w, q[s], part[s]);
#pragma unroll
                        for (int s = 0; s < N; ++s) q[s] = next[s];
                    }
                    if (v < vb) {
                        fv += 1.0f;
                        row += step;
                        begin(at);
                    }
                }
                flush();
            }
        }
        if (neg && half == 0)
#pragma unroll
            for (int s = 0; s < N; ++s)
                if (s < (s ^ neg)) {
                    const KahanAcc t = acc[s];
                    acc[s] = acc[s ^ neg];
                    acc[s ^ neg] = t;
                }
    }
}

// The walk of four canonical views at once: the work-group's four waves take the same 64
// bins of neighbouring views, whose rays cross nearly the same pixels of a row.  kRows rows
// of the orbit image, kUnits 16-byte units of each plane, are staged for all four in one of
// two buffers (each wave brings one plane of one row, kChunks loads of 64 units as far as
// the rays need them), the next rows' loads being on their way while these are summed: one
// barrier per kRows rows.
// Staging per wave, the vector memory unit (three 16-byte loads a row under D4, about 16
// cycles each), LDS (three writes and the reads) and VALU were each busy two thirds of the
// time; a row now takes one load and one write a wave, and VALU issue bounds the walk.
// Forward of 32 x 512^2 parallel 3350 -> 2420 us, 769^2 fan of odd views 352 -> 247, 1024^2
// fan 175 -> 155, 16 ragged slices 1230 -> 985.  Five waves per SIMD under D4 (96 VGPRs, 4
// spilled outside the pixel loop) against four: 8 x 512^2 607 us against 667; 1024^2 fan 183
// against 203, which is why the sums' LDS is kept below the sixth granule step (kLdsSums).
template <int GRP>
struct ViewStage {
    using O = Orbit<GRP>;
    static constexpr int kPlanes = O::N == 8 ? 2 : 1;
    static constexpr int kRows = 4 / kPlanes;
    static constexpr int kChunks = O::N == 2 ? 2 : 3;
    static constexpr int kUnits = 64 * kChunks;           // of one plane of a row
    static constexpr int kUnitPixels = O::N == 2 ? 2 : 1;
    static constexpr int kPixels = kUnits * kUnitPixels;
    static constexpr int kBuffer = kRows * kPlanes * kUnits;
    // the rows that fwd_sym_rows stages for each wave fit, too
    static constexpr int kStage = 2 * kBuffer > 4 * O::kLoads * 64 ? 2 * kBuffer : 4 * O::kLoads * 64;
    // the first so many of a wave's sums over segments wait in LDS: under D4, whose registers
    // are all taken, seven, which with the stage leave room for five work-groups a compute
    // unit (25 of 128 granules of 1280 B each; eight take 26)
    static constexpr int kLdsSums = O::N == 8 ? 7 : 0;
};

__device__ __forceinline__ float wave_min(float x)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x = fminf(x, __shfl_xor(x, off, 64));
    return x;
}

// As fwd_sym_rows, for the four waves of a work-group (every one calls it with the same
// rows, and with the same slice, bins and walk).  A wave without a view (!active) helps to
// stage and sums nothing.  The rows are vlo..vhi in segments of `per` rows: after each,
// done(acc, flip, neg) takes the sums that fwd_sym_rows gives for that segment alone, with
// flip still in the slots of the rows v < 0 (s ^ neg for s), and clears them.
// What the staged columns must hold: the lanes' lines in v are straight, so their smallest
// start lies above its chord over [vlo, vhi] and their largest end below its own, and both
// chords are known from the two end rows.  Work-groups whose lanes' lines change order or
// leave more than kPixels between the chords walk each wave by itself.
template <bool FAN, int GRP, bool COLS, class Done>
__device__ __forceinline__ void fwd_view_rows(const SliceDesc& S, const Ray& r, float cT, float sT,
                                              const float* __restrict__ orb, int vlo, int vhi,
                                              int per, bool active, int wave,
                                              float4* __restrict__ st, float (*ends)[4], Done done)
{
    using O = Orbit<GRP>;
    using V = ViewStage<GRP>;
    constexpr int N = O::N, R = V::kRows, neg = O::neg_xor(COLS);
    const int lane = (int)threadIdx.x & 63, H = S.H;
    if (vlo > vhi) return;  // uniform over the work-group
    const float fH = (float)H, qs = sT * S.invd, qc = cT * S.invd;
    const RowBounds rb = row_bounds(r, cT, sT, FAN ? S.invd : 0.0f, !COLS);
    const float ua = rb.U0 * rb.iu, ub = -rb.U1 * rb.iu, la = rb.L0 * rb.il, lb = -rb.L1 * rb.il;
    const float fa = (float)vlo, fb = (float)vhi;
    const float ea = fmaf(fa, ub, ua), eb = fmaf(fb, ub, ua);
    const float ga = fmaf(fa, lb, la), gb = fmaf(fb, lb, la);
    const bool left = ga + gb <= ea + eb;  // the second line is the left one
    float lo_a = left ? ga : ea, lo_b = left ? gb : eb, hi_a = left ? ea : ga, hi_b = left ? eb : gb;
    const bool ordered = __all(lo_a <= hi_a && lo_b <= hi_b);
    lo_a = wave_min(lo_a);
    lo_b = wave_min(lo_b);
    hi_a = -wave_min(-hi_a);
    hi_b = -wave_min(-hi_b);
    if (lane == 0) {
        ends[wave][0] = lo_a;
        ends[wave][1] = lo_b;
        ends[wave][2] = ordered ? hi_a : INFINITY;
        ends[wave][3] = hi_b;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        lo_a = fminf(lo_a, ends[w][0]);
        lo_b = fminf(lo_b, ends[w][1]);
        hi_a = fmaxf(hi_a, ends[w][2]);
        hi_b = fmaxf(hi_b, ends[w][3]);
    }
    __syncthreads();  // read: `ends` may share its place with the sums
    KahanAcc acc[N];
    // first staged column of the rows v..v + R - 1: c + (v - vlo) slope, less a pixel of slack
    const float slope = vhi > vlo ? (lo_b - lo_a) / (float)(vhi - vlo) : 0.0f;
    const float c = lo_a - 1.0f + fminf(0.0f, slope * (float)(R - 1));
    const float span = fmaxf(hi_a - lo_a, hi_b - lo_b) + fabsf(slope) * (float)(R - 1) + 3.0f;
    // (the image's width bounds the pixels, too); unordered lanes have left span = inf
    const float px = fminf(span, 2.0f * fH + 2.0f);
    const bool fits = span < INFINITY && px < (float)(V::kPixels - 1);
    if (!__builtin_amdgcn_readfirstlane((int)fits)) {
        for (int v = vlo; v <= vhi; v += per) {
            fwd_sym_rows<FAN, GRP, COLS>(S, r, cT, sT, orb, v, min(v + per - 1, vhi), acc,
                                         st + wave * O::kLoads * 64);
            done(acc, false, std::integral_constant<int, neg>{});
        }
        return;
    }
    const int chunks = __builtin_amdgcn_readfirstlane((int)px + 1 + 64 * V::kUnitPixels) /
                       (64 * V::kUnitPixels);
    const float none = 1e30f;  // beyond any pixel
    const float l0 = !active ? none : (left ? la : ua), l1 = !active ? 0.0f : (left ? lb : ub);
    const float r0 = !active ? -none : (left ? ua : la), r1 = !active ? 0.0f : (left ? ub : lb);
    const int my_row = wave / V::kPlanes, my_plane = wave % V::kPlanes;
    float4* const mine = st + wave * V::kUnits + lane;
    auto column = [&](int v) {
        const int k = (int)floorf(fmaf((float)(v - vlo), slope, c));
        return __builtin_amdgcn_readfirstlane(min(max(k, -H), H));
    };
    auto load = [&](int v, int vb, int c0, float4* g) {
        const __amdgpu_buffer_rsrc_t B =
            row_rsrc(orbit_row<GRP, COLS>(S, orb, min(v + my_row, vb)), N * S.orb_pitch * 4);
#pragma unroll
        for (int k = 0; k < V::kChunks; ++k)
            if (k < chunks)
                g[k] = ldb128(B, (my_plane * S.orb_pitch + 64 * k + lane) * 16, (c0 + H) * O::kPlane * 4);
    };
    auto store = [&](int buf, const float4* g) {
#pragma unroll
        for (int k = 0; k < V::kChunks; ++k)
            if (k < chunks) mine[buf * V::kBuffer + 64 * k] = g[k];
    };
    float part[N];
#pragma unroll
    for (int s = 0; s < N; ++s) part[s] = 0.0f;
    auto flush = [&]() {
#pragma unroll
        for (int s = 0; s < N; ++s) {
            acc[s].add(part[s]);
            part[s] = 0.0f;
        }
    };
    int buf = 0, seg_end = min(vlo + per - 1, vhi);
    // rows v < 0 first, then v >= 0: the sums are held by the slots of the current sign
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
        const int va = half ? max(vlo, 0) : vlo, vb = half ? vhi : min(vhi, -1);
        if (va <= vb) {
            int block = va + kRowBlock - 1;  // the block's last row
            float4 g[V::kChunks] = {};
            int c0 = column(va);
            load(va, vb, c0, g);
            store(buf, g);
            __syncthreads();
#pragma unroll 1
            for (int v = va; v <= vb; v += R) {
                const int now = c0, last = min(v + R - 1, vb);
                const bool more = v + R <= vb;
                if (more) {
                    c0 = column(v + R);
                    load(v + R, vb, c0, g);
                }
                const float4* row = st + buf * V::kBuffer;
#pragma unroll 1
                for (int y = v; y <= last; ++y, row += V::kPlanes * V::kUnits) {
                    const float fv = (float)y;
                    const float lo = fmaxf(ceilf(fmaf(fv, l1, l0)), -fH);
                    const float hi = fminf(fmaf(fv, r1, r0), fH);
                    const float rowd = COLS ? 0.0f : fmaf(fv, r.sinR, -r.dc);
                    const float rowq = FAN && !COLS ? fmaf(-fv, qc, 1.0f) : 0.0f;
                    // (the byte offset of the pixel is kept, not its index: one add a pixel less; lanes
                    // without pixels may have any)
                    int at = ((int)fminf(lo, fH) - now) * (O::kPlane * 4) + (int)((const char*)row - (const char*)st);
                    for (float fu = lo; fu <= hi; fu += 1.0f, at += O::kPlane * 4) {
                        const char* px = (const char*)st + at;
                        float q[N];
                        if constexpr (N == 2) {
                            const float2 a = *reinterpret_cast<const float2*>(px);
                            q[0] = a.x;
                            q[1] = a.y;
                        } else {
#pragma unroll
                            for (int p = 0; p < V::kPlanes; ++p) {
                                const float4 a = reinterpret_cast<const float4*>(px)[p * V::kUnits];
                                q[4 * p] = a.x;
                                q[4 * p + 1] = a.y;
                                q[4 * p + 2] = a.z;
                                q[4 * p + 3] = a.w;
                            }
                        }
                        // ray_dist and fan_depth_scale at (x, y) = (fu, fv), columns mode (fv, fu)
                        const float dist = COLS ? fmaf(fv, r.cosR, fmaf(fu, r.sinR, -r.dc))
                                                : fmaf(fu, r.cosR, rowd);
                        const float qd = COLS ? fmaf(fv, qs, fmaf(-fu, qc, 1.0f)) : fmaf(fu, qs, rowq);
                        const float w = strip_area(dist, FAN ? r.hbc * qd : r.hbc, r);
#pragma unroll
                        for (int s = 0; s < N; ++s) part[s] = fmaf(w, q[s], part[s]);
                    }
                    if (y == min(min(block, seg_end), vb)) {
                        flush();
                        block = y + kRowBlock;
                        if (y == seg_end) {
                            done(acc, neg && !half, std::integral_constant<int, neg>{});
                            seg_end = min(seg_end + per, vhi);
                        }
                    }
                }
                if (more) store(buf ^ 1, g);
                __syncthreads();
                buf ^= 1;
            }
        }
        if (neg && half == 0)
#pragma unroll
            for (int s = 0; s < N; ++s)
                if (s < (s ^ neg)) {
                    const KahanAcc t = acc[s];
                    acc[s] = acc[s ^ neg];
                    acc[s ^ neg] = t;
                }
    }
}

// Kernel argument of the forward launches: empty, or (BHC) the beam-hardening ray pass
// fused into the final store (ctprj_bhc_grad_alpha): every sinogram entry is stored
// once, as w of bhc_ray at Ts times its ray sum, and its FP64 NLL term goes into the
// storing work-group's partial at partials[part_off + work-group].
template <bool BHC>
struct FwdBhc {};
template <>
struct FwdBhc<true> : BhcStore {};

// Sum of v over the work-group (a multiple of 64 threads, at most 16 waves): a butterfly
// over each wave's lanes, then the waves' sums in wave order; every thread must call it.
__device__ __forceinline__ double group_sum(double v)
{
    __shared__ double sh[16];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    const int wave = (int)threadIdx.x >> 6, nw = (int)blockDim.x >> 6;
    __syncthreads();  // an earlier call's reads are done
    if ((threadIdx.x & 63) == 0) sh[wave] = v;
    __syncthreads();
    double r = sh[0];
    for (int w = 1; w < nw; ++w) r += sh[w];
    return r;
}

// The sum t of image e of canonical ray (it, lane) written to its view g_e a0; with BHC
// the entry's w instead, and the NLL term is returned (0 where nothing is stored).
template <bool BHC>
__device__ __forceinline__ double fwd_sym_store(const SliceDesc& S, const FwdItem& it, int a0,
                                                int e, int lane, float t, float* __restrict__ sino,
                                                const FwdBhc<BHC>& B)
{
    const int b = it.bin0 + lane;
    const int bmax = S.fold ? S.pC : S.bhi;
    const bool active = b >= S.blo && b <= bmax;
    float* out = sino + S.sino_off;
    int sg, off;
    const int v = map_view(S, e & 3, e >> 2, a0, sg, off);
    if (v >= S.np) return 0.0;
    // folded scans: images e and e ^ 2 (R^2 apart) meet at the centre bin, whose two sums
    // are equal up to rounding, and both reach bin 0 of an even detector; one writer
    // (k < 2) keeps the result deterministic and counts each entry once
    if (S.fold && (e & 2) && (b == S.pC || b < S.blo)) return 0.0;
    long long idx;
    float val = t;
    if (b < S.blo) {  // even detector: bin 0 carries no ray
        idx = (long long)v * S.W;
        val = 0.0f;
    } else if (active) {
        idx = (long long)v * S.W + off + sg * b;
    } else {
        return 0.0;
    }
    if constexpr (!BHC) {
        out[idx] = val;
        return 0.0;
    } else {
        float w, hw;
        const double f = bhc_ray<false>(B.P, B.Ts * val, B.Imea[S.sino_off + idx], B.Ts, &w, &hw);
        out[idx] = w;
        return f;
    }
}

// One canonical ray run over the group's images.  The image rows are cut into
// nsplit * SEG segments: this work-group walks segments split * SEG + wave.  nsplit == 1
// writes the sinogram; otherwise the work-group's sums go to part[e * 64 + lane] for
// k_forward_sym_combine.  Lanes past the detector's ends repeat the nearest ray and are
// not stored; on a mirror view the rotations alone are.
template <bool FAN, bool COLS, int SEG, int GRP, bool BHC>
__device__ __forceinline__ void fwd_sym_run(const SliceDesc& S, const FwdItem& it, float cT,
                                            float sT, int a0, unsigned mask,
                                            const Ray* __restrict__ rays,
                                            const float* __restrict__ orb,
                                            float* __restrict__ sino, float (*red)[8][64],
                                            int split, int nsplit, float* __restrict__ part,
                                            float (*tb)[64], float4* __restrict__ stage)
{
    using O = Orbit<GRP>;
    // the wave index is uniform over the wave: the row loop then runs on scalar registers
    const int lane = (int)threadIdx.x & 63;
    const int seg = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int b = min(max(it.bin0 + lane, S.blo), S.fold ? S.pC : S.bhi);
    KahanAcc acc[O::N];
    {
        Ray r;
        if (FAN) r = rays[S.ray_off + (long long)it.view * S.W + b];
        else {
            r = rays[S.ray_off + it.view];
            r.dc = (float)(b - S.pC) * S.dSize;
        }
        const int nrow = 2 * S.H + 1, nseg = SEG * nsplit, per = (nrow + nseg - 1) / nseg;
        const int vlo = -S.H + (split * SEG + seg) * per, vhi = min(S.H, vlo + per - 1);
        fwd_sym_rows<FAN, GRP, COLS>(S, r, cT, sT, orb, vlo, vhi, acc,
                                     stage + seg * O::kLoads * 64);
    }
    if (SEG > 1) {
#pragma unroll
        for (int s = 0; s < O::N; ++s) red[seg][O::elem(s)][lane] = acc[s].s * S.inver;
        __syncthreads();
    }
    // wave w finalises the images e = w (mod SEG): the sum of the waves' partials in wave
    // order, more than four as groups of four.  BHC: the sums wait in tb[e][lane] for the
    // kernel's one fused store loop (a single inlined copy of the spectrum sums)
#pragma unroll
    for (int s = 0; s < O::N; ++s) {
        const int e = O::elem(s);
        if (!(mask >> e & 1u) || (SEG > 1 && e % SEG != seg)) continue;
        float t = acc[s].s * S.inver;
        if (SEG > 1) {
            t = red[0][e][lane];
#pragma unroll
            for (int q = 1; q < (SEG > 4 ? 4 : SEG); ++q) t += red[q][e][lane];
        }
#pragma unroll
        for (int k = 4; k < SEG; k += 4) {  // as work-groups of four waves are added
            float u = red[k][e][lane];
#pragma unroll
            for (int q = k + 1; q < k + 4; ++q) u += red[q][e][lane];
            t += u;
        }
        if (part) part[e * 64 + lane] = t;
        else if (BHC) tb[e][lane] = t;
        else fwd_sym_store<false>(S, it, a0, e, lane, t, sino, FwdBhc<false>{});
    }
}

// Work-group -> (split, item): the first nitems work-groups take split 0 of every item,
// the next nitems split 1, and so on.
__device__ __forceinline__ void split_item(int nitems, int& split, int& idx)
{
    split = __builtin_amdgcn_readfirstlane((int)blockIdx.x / nitems);
    idx = (int)blockIdx.x - split * nitems;
}

// One work item: (slice, canonical view index, first bin of 64) of a slice under group
// GRP (one launch per group keeps each variant's registers to its own images).  SEG
// waves share the 64 rays, each walking 1/SEG of the work-group's image rows, and then
// share the final sums; with nsplit > 1, nsplit work-groups share the rows of an item
// and leave their sums in part (512 floats per work-group) for k_forward_sym_combine.
// capped: a slice's items take its own number (fgroups) of the nsplit work-groups, the others
// end.
template <int SEG, int GRP, bool BHC>
__global__ __launch_bounds__(64 * SEG) void k_forward_sym(const SliceDesc* __restrict__ slices,
                                                          const FwdItem* __restrict__ items,
                                                          const float4* __restrict__ views,
                                                          const Ray* __restrict__ rays,
                                                          const float* __restrict__ orb,
                                                          float* __restrict__ sino, int nitems,
                                                          int nsplit, bool capped,
                                                          float* __restrict__ part,
                                                          const FwdBhc<BHC> B)
{
    __shared__ float red[SEG > 1 ? SEG : 1][8][64];
    __shared__ float4 stage[SEG * Orbit<GRP>::kLoads * 64 + 1];  // + 1: read past a row's end, unused
    int split, idx;
    split_item(nitems, split, idx);
    const FwdItem it = items[idx];
    if (it.slice < 0) {  // uniform over the work-group: a padding item
        if constexpr (BHC)
            if (!part && threadIdx.x == 0) B.partials[B.part_off + blockIdx.x] = 0.0;
        return;
    }
    const SliceDesc S = slices[it.slice];
    if (capped) nsplit = min(nsplit, S.fgroups);
    if (split >= nsplit) return;  // uniform over the work-group
    const float4 T = views[S.view_off + it.view];
    const int a0 = __float_as_int(T.z);
    constexpr GroupMasks GM = group_masks(GRP);
    const unsigned mask = (a0 == 0 || GM.q * a0 == S.P) ? GM.rot : GM.all;
    float* mine = part ? part + (long long)blockIdx.x * 512 : nullptr;
    __shared__ float tb[BHC ? 8 : 1][64];  // BHC: each lane's final sums, by image
    // D4's canonical views lie in [0, 45] degrees and always walk rows; V4's reach 90 and
    // Z2's 180 degrees, and the steep ones walk columns.  (fan, walk) are uniform over the
    // work-group: the barrier inside is reached by all of its waves
    const bool cols = GRP != kGrpD4 && fabsf(T.x) < fabsf(T.y);
#define CTPRJ_RUN(FAN, COLS)                                                                      \
    fwd_sym_run<FAN, COLS, SEG, GRP, BHC>(S, it, T.x, T.y, a0, mask, rays, orb, sino, red, split, \
                                          nsplit, mine, tb, stage)
    if (GRP != kGrpD4 && cols) {
        if (S.fan) CTPRJ_RUN(true, GRP != kGrpD4);
        else CTPRJ_RUN(false, GRP != kGrpD4);
    } else {
        if (S.fan) CTPRJ_RUN(true, false);
        else CTPRJ_RUN(false, false);
    }
#undef CTPRJ_RUN
    if constexpr (BHC) {
        if (!mine) {  // uniform: the fused store of this lane's images, then the NLL partial
            const int lane = (int)threadIdx.x & 63;
            const int seg = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
            double f = 0.0;
            // each lane reads back only its own entries: no barrier
#pragma unroll 1
            for (int e = seg; e < 8; e += SEG)
                if (mask >> e & 1u) f += fwd_sym_store<true>(S, it, a0, e, lane, tb[e][lane], sino, B);
            const double tot = group_sum(f);
            if (threadIdx.x == 0) B.partials[B.part_off + blockIdx.x] = tot;
        }
    }
}

// Four neighbouring canonical views (four consecutive items: one slice, one walk, the same
// bins; the first is there unless all are padding), one wave each: see fwd_view_rows.  The
// rows are cut into the 4 x groups segments of k_forward_sym with four waves (groups = 0: the
// slice's own fgroups) and a wave adds them as that kernel and its second launch do, so both
// give the same bits; the level says what a work-group takes:
//   0  one segment (nsplit = 4 x groups);  m >= 1  m groups of four segments (nsplit = groups /
//   m, upwards): unless there is one group only, every segment's or group's sums go to part for
//   k_forward_sym_combine;
//   -1  all of them: where there is more than one group, the groups' sum waits in the item's
//   place of part, read and written once a group.
template <int GRP, bool BHC>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(GRP == kGrpD4 ? 5 : GRP == kGrpV4 ? 6 : 8)))
void k_forward_views(const SliceDesc* __restrict__ slices,
                                                       const FwdItem* __restrict__ items,
                                                       const float4* __restrict__ views,
                                                       const Ray* __restrict__ rays,
                                                       const float* __restrict__ orb,
                                                       float* __restrict__ sino, int nitems,
                                                       int nsplit, int level, int groups,
                                                       bool parts, float* __restrict__ part,
                                                       const FwdBhc<BHC> B)
{
    using O = Orbit<GRP>;
    using V = ViewStage<GRP>;
    constexpr int N = O::N;
    // the staged rows, then the waves' sums by slot (or, + 1, what is read past a row's end);
    // the sums' place holds the walks' ends first
    constexpr int kSums = V::kLdsSums ? 4 * V::kLdsSums * 64 / 4 : 4;
    __shared__ float4 stage[V::kStage + kSums];
    float(*const ends)[4] = reinterpret_cast<float(*)[4]>(stage + V::kStage);
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int split, quad;
    split_item(nitems / 4, split, quad);
    const FwdItem lead = items[4 * quad];
    if (lead.slice < 0) {  // uniform over the work-group: padding items
        if constexpr (BHC)
            if (!parts && threadIdx.x < 4) B.partials[B.part_off + 4 * quad + threadIdx.x] = 0.0;
        return;
    }
    FwdItem it = items[4 * quad + wave];
    const bool active = it.slice >= 0;
    if (!active) it = lead;
    const SliceDesc S = slices[lead.slice];
    if (groups == 0) groups = S.fgroups;
    const int nseg = level < 0 ? 4 * groups : level == 0 ? 1 : 4 * level, seg0 = split * nseg;
    if (seg0 >= 4 * groups) return;  // uniform over the work-group
    const float4 T = views[S.view_off + it.view];
    const int a0 = __float_as_int(T.z);
    constexpr GroupMasks GM = group_masks(GRP);
    const unsigned mask = !active ? 0u : (a0 == 0 || GM.q * a0 == S.P) ? GM.rot : GM.all;
    const int b = min(max(it.bin0 + lane, S.blo), S.fold ? S.pC : S.bhi);
    // this wave's sums by slot
    float reg[N];
    // (the places are formed anew where they are used: no register holds them over the walk)
    auto here = [&]() {
        int l = (int)threadIdx.x;
        asm("" : "+v"(l));
        return l & 63;
    };
    auto lds = [&](int s) -> float& {
        return reinterpret_cast<float*>(stage + V::kStage)[(wave * V::kLdsSums + s) * 64 + here()];
    };
    auto get = [&](int s) -> float { return s < V::kLdsSums ? lds(s) : reg[s]; };
    auto set = [&](int s, float t) { if (s < V::kLdsSums) lds(s) = t; else reg[s] = t; };
    // the sums of segment or group g of the item in part, or (g = 0) their total
    auto slot = [&](int g, int s) -> float& {
        return part[((long long)g * nitems + 4 * quad + wave) * 512 + O::elem(s) * 64 + here()];
    };
    const bool total = level < 0 && groups > 1;
    int next = level == 0 ? split : level * split;  // part's next segment or group
    {
        Ray r;
        if (S.fan) r = rays[S.ray_off + (long long)it.view * S.W + b];
        else {
            r = rays[S.ray_off + it.view];
            r.dc = (float)(b - S.pC) * S.dSize;
        }
        const int nrow = 2 * S.H + 1;
        const int per = __builtin_amdgcn_readfirstlane((nrow + 4 * groups - 1) / (4 * groups));
        const int vlo = -S.H + seg0 * per, vhi = min(S.H, vlo + nseg * per - 1);
        const bool cols = GRP != kGrpD4 && lead.pad;  // the walk, uniform over the work-group
        int segs = 0;  // finished
        bool clear = true;
        auto done = [&](KahanAcc* acc, bool flip, auto neg) {
            // (flip: the slots of the rows v < 0)
            float in[N];
#pragma unroll
            for (int s = 0; s < N; ++s) {
                in[s] = acc[s].s * S.inver;
                acc[s] = KahanAcc{};
            }
#pragma unroll
            for (int s = 0; s < N; ++s) {
                const float v = flip ? in[s ^ decltype(neg)::value] : in[s];
                set(s, clear ? v : get(s) + v);
            }
            ++segs;
            clear = false;
            if (level == 0 || segs % 4 == 0 || vlo + segs * per > vhi) {  // (the last one)
                if (parts) {
#pragma unroll
                    for (int s = 0; s < N; ++s) slot(next, s) = get(s);
                    ++next;
                    clear = true;
                } else if (total) {
#pragma unroll
                    for (int s = 0; s < N; ++s) {
                        const float t = get(s);
                        float& u = slot(0, s);
                        u = segs <= 4 ? t : u + t;
                    }
                    clear = true;
                }
            }
        };
#define CTPRJ_RUN(FAN, COLS)                                                                    \
    fwd_view_rows<FAN, GRP, COLS>(S, r, T.x, T.y, orb, vlo, vhi, per, active, wave, stage, ends, \
                                  done)
        if (GRP != kGrpD4 && cols) {
            if (S.fan) CTPRJ_RUN(true, GRP != kGrpD4);
            else CTPRJ_RUN(false, GRP != kGrpD4);
        } else {
            if (S.fan) CTPRJ_RUN(true, false);
            else CTPRJ_RUN(false, false);
        }
#undef CTPRJ_RUN
    }
    if (parts) {  // segments or groups past the last row
        const int end = level == 0 ? split + 1 : min(level * (split + 1), groups);
        for (; next < end; ++next)
#pragma unroll
            for (int s = 0; s < N; ++s) slot(next, s) = 0.0f;
        return;
    }
    if (total)
#pragma unroll
        for (int s = 0; s < N; ++s) set(s, slot(0, s));
    if constexpr (!BHC) {
#pragma unroll
        for (int s = 0; s < O::N; ++s)
            if (mask >> O::elem(s) & 1u)
                fwd_sym_store<false>(S, it, a0, O::elem(s), lane, get(s), sino, B);
    } else {
        // each lane's sums wait in LDS for one fused store loop (a single inlined copy of the
        // spectrum sums); each lane reads back only its own entries
        float(*tb)[64] = reinterpret_cast<float(*)[64]>(stage) + 8 * wave;
        __syncthreads();  // every wave's rows are read
#pragma unroll
        for (int s = 0; s < O::N; ++s) tb[O::elem(s)][lane] = get(s);
        double f = 0.0;
#pragma unroll 1
        for (int e = 0; e < 8; ++e)
            if (mask >> e & 1u) f += fwd_sym_store<true>(S, it, a0, e, lane, tb[e][lane], sino, B);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) f += __shfl_xor(f, off, 64);
        if (lane == 0) B.partials[B.part_off + 4 * quad + wave] = f;
    }
}

// The nsplit partial sums of each canonical ray and image of an item, added in split
// order (fine: by groups of four) and written like the one-work-group path (512 threads:
// image e = thread / 64 of ray lane = thread % 64).
template <int GRP, bool BHC, bool CAPPED>
__global__ __launch_bounds__(512) void k_forward_sym_combine(const SliceDesc* __restrict__ slices,
                                                             const FwdItem* __restrict__ items,
                                                             const float4* __restrict__ views,
                                                             int nitems, int nsplit, bool fine,
                                                             const float* __restrict__ part,
                                                             float* __restrict__ sino,
                                                             const FwdBhc<BHC> B)
{
    const FwdItem it = items[blockIdx.x];
    if (it.slice < 0) {  // uniform: a padding item
        if constexpr (BHC)
            if (threadIdx.x == 0) B.partials[B.part_off + blockIdx.x] = 0.0;
        return;
    }
    const SliceDesc S = slices[it.slice];
    if (CAPPED) nsplit = min(nsplit, fine ? 4 * S.fgroups : S.fgroups);
    const int a0 = __float_as_int(views[S.view_off + it.view].z);
    constexpr GroupMasks GM = group_masks(GRP);
    const unsigned mask = (a0 == 0 || GM.q * a0 == S.P) ? GM.rot : GM.all;
    const int e = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    double f = 0.0;
    if (mask >> e & 1u) {
        const float* p = part + (long long)blockIdx.x * 512 + threadIdx.x;
        const long long step = nitems * 512LL;
        float t = 0.0f;
        if (fine) {
            for (int k = 0; k < nsplit; k += 4, p += 4 * step) {
                const float u = ((p[0] + p[step]) + p[2 * step]) + p[3 * step];
                t = k ? t + u : u;
            }
        } else {
            t = p[0];
            for (int k = 1; k < nsplit; ++k) t += p[k * step];
        }
        f = fwd_sym_store<BHC>(S, it, a0, e, lane, t, sino, B);
    }
    if constexpr (BHC) {  // the work-group's NLL partial (every thread takes part)
        const double tot = group_sum(f);
        if (threadIdx.x == 0) B.partials[B.part_off + blockIdx.x] = tot;
    }
}

// ------------------------------------------------------------------ adjoint ---
//
// The adjoint reads its bins from the orbit sinogram: for every canonical view a0 and bin
// b, the values of the group's rays g (a0, b) side by side (element e in slot e; a half-turn
// scan's folded views at their reflected bin; 0 for views beyond np, bins that carry no
// ray, and, on a mirror view, the reflections).  Orbit pixel h q0 under group element g'
// reads ray h g' (a0, b), so for a fixed g' the eight pixels of an orbit read the same
// entry with its slots permuted by the product h g', known at compile time.  One row
// holds, for each bin, D4: plane 0 = elements 0..3, plane 1 = elements 4..7 (os_pitch
// float4 each), V4: elements 0, 2, 4, 6 (float4), Z2: elements 0, 6 (float2).

// Element product h g' = (k1, m1) (k2, m2), R^k M^m each.
__host__ __device__ constexpr int elem_mul(int h, int e2)
{
    const int k1 = h & 3, m1 = h >> 2, k2 = e2 & 3, m2 = e2 >> 2;
    return ((k1 + (m1 ? -k2 : k2)) & 3) + 4 * (m1 ^ m2);
}

// Rows of the orbit sinogram: item (slice, canonical view), 256 bins per work-group.
// tab: 8 entries per canonical view, the sinogram row of element e (byte offset | kRowFlip,
// or kRowNone).  The values are stored divided by the effectiveRate.
template <int GRP>
__device__ __forceinline__ void orbit_sino_bin(const SliceDesc& S, int i, int b,
                                               const int* __restrict__ tab,
                                               const float* __restrict__ sino,
                                               float* __restrict__ os)
{
    using O = Orbit<GRP>;
    const int* t = tab + S.tab_off + (long long)i * 8;
    const float* in = sino + S.sino_off;
    const bool ray = b >= S.blo && b <= S.bhi;
    float q[O::N];
#pragma unroll
    for (int s = 0; s < O::N; ++s) {
        const int r = t[O::elem(s)];
        q[s] = 0.0f;
        if (ray && !(r & kRowNone))
            q[s] = S.inver * in[((r & ~(kRowFlip | kRowNone)) >> 2) + ((r & kRowFlip) ? 2 * S.pC - b : b)];
    }
    float* out = os + S.os_off + (long long)i * (O::N * S.os_pitch);
    if constexpr (O::N == 2) {
        reinterpret_cast<float2*>(out)[b] = make_float2(q[0], q[1]);
    } else {
#pragma unroll
        for (int p = 0; p < O::N / 4; ++p)
            reinterpret_cast<float4*>(out)[p * S.os_pitch + b] =
                make_float4(q[4 * p], q[4 * p + 1], q[4 * p + 2], q[4 * p + 3]);
    }
}

__global__ __launch_bounds__(256) void k_orbit_sino(const SliceDesc* __restrict__ slices,
                                                    const int2* __restrict__ items,
                                                    const int* __restrict__ tab,
                                                    const float* __restrict__ sino,
                                                    float* __restrict__ os)
{
    const int2 it = items[blockIdx.x];
    const SliceDesc S = slices[it.x];
    const int b = (int)(blockIdx.y * 256 + threadIdx.x);
    if (b >= S.W) return;
    if (S.sym == kGrpD4) orbit_sino_bin<kGrpD4>(S, it.y, b, tab, sino, os);
    else if (S.sym == kGrpV4) orbit_sino_bin<kGrpV4>(S, it.y, b, tab, sino, os);
    else orbit_sino_bin<kGrpZ2>(S, it.y, b, tab, sino, os);
}

void launch_orbit_sino(int nitems, int max_W, const SliceDesc* desc, const int2* items,
                       const int* tab, const float* sino, float* os, hipStream_t st)
{
    if (nitems > 0)
        hipLaunchKernelGGL(k_orbit_sino, dim3(nitems, (max_W + 255) / 256), dim3(256), 0, st, desc,
                           items, tab, sino, os);
}

// Bins a wave stages at once per (canonical view, element): every pixel of an 8 x 8 tile
// reads bins within about 11 pixels' shadow of each other.
constexpr int kStageBins = 32;

// One wave's LDS area, addressed by one offset 16 k for bin k: its orbit values at val[k]
// (and val[kStageBins + k], D4's plane 1), and (fan beam) its ray record at ray[k] and
// ray[kStageBins + k].
struct AdjStage {
    float4 val[64];
    float4 ray[64];
};

// Canonical views i = i0, i0 + step, ... for the orbit of (x0, y0) under group GRP: for
// each view and each element g' the wave stages the bins that its 64 orbit pixels can
// read (one load per lane for the values, one for the fan-beam ray records; the next
// element's are loaded while this one's are summed), and every lane sums its own candidate
// bins from LDS, in increasing order: the weight W(a0, b, g'^-1 q0) is formed once and
// serves every pixel of the orbit.  On a mirror view the reflected rays' zeros leave
// rotations g' paired with rotation pixels and reflections with reflected ones, so every
// entry has the forward's key.  A folded scan takes the half set of elements that maps the
// canonical range into [0, 180).  The staged range starts at the smallest first bin of the
// tile's corner pixels (the extremes, see BinBounds); should a lane's bins lie outside,
// the wave takes the true range, piece by piece where it is wider than kStageBins.  COMPACT
// (see adj_compact): they cannot, and the check, the pieces and their bounds are left out,
// about 7 of 130 instructions an element: adjoint of 8 x 512^2 parallel 473 -> 440 us.
// The fan beam keeps them: without, 512^2 took 47.3 us against 46.1 and 512^2 of odd views 118
// against 112.
// Bound by VALU issue (4 cycles a wave instruction): what is not a weight or an update is
// kept to the candidate bounds (about 25 instructions per element) and the loop's two.
// DIRECT: os is the sinogram itself and tab the view-row table; a staged value is then
// gathered from the rows of its slots' elements, one 4-byte load each, instead of read from
// the orbit sinogram with one 16-byte load.
template <bool FAN, bool FBP, int GRP, bool FOLD, bool DIRECT, bool COMPACT>
__device__ __forceinline__ void adj_sym_pixel(const SliceDesc& S, const float4* __restrict__ views,
                                              const Ray* __restrict__ rays,
                                              const float* __restrict__ os,
                                              const int* __restrict__ tab, int lane, int x0,
                                              int y0, bool valid, int i0, int step,
                                              KahanAcc* acc, AdjStage* __restrict__ st)
{
    using O = Orbit<GRP>;
    constexpr int N = O::N, CH = kStageBins;
    constexpr GroupMasks G = group_masks(GRP);
    constexpr unsigned GSET = FOLD ? G.fold : G.all;
    const float gx = (float)x0, gy = (float)y0;
    // lane's part of a staged piece, bytes from the first bin's: values, ray records
    const int voff = N == 8 && lane >= CH ? (S.os_pitch + lane - CH) * 16 : lane * O::kPlane * 4;
    const int roff = (lane & (CH - 1)) * (int)sizeof(Ray) + (lane >= CH ? 16 : 0);
    const int rec = N * S.os_pitch, last_bin = valid ? S.bhi : INT_MIN;
    for (int i = i0; i < S.ncanon; i += step) {
        const float4 T = views[S.view_off + i];
        const float* osrow = DIRECT ? os + S.sino_off : os + S.os_off + (long long)i * rec;
        const __amdgpu_buffer_rsrc_t RV = row_rsrc(osrow, DIRECT ? S.np * S.W * 4 : rec * 4);
        // DIRECT: the lane's slots read bin c0 + lane (reflected rows: 2 pC less it) of their rows
        // at byte at0 + dir * c0; rows without an entry lie past the end and read as 0
        int at0[O::kPlane], dir[O::kPlane];
        if constexpr (DIRECT) {
            const int* t = tab + S.tab_off + (long long)i * 8 + (N == 8 && lane >= CH ? 4 : 0);
            const int k = N == 8 ? lane & (CH - 1) : lane;
#pragma unroll
            for (int q = 0; q < O::kPlane; ++q) {
                const int r = t[N == 8 ? q : O::elem(q)];
                const bool none = r & kRowNone, flip = r & kRowFlip;
                at0[q] = none ? 0x7ffffff0 : (r & ~(kRowFlip | kRowNone)) + 4 * (flip ? 2 * S.pC - k : k);
                dir[q] = none ? 0 : flip ? -4 : 4;
            }
        }
        const Ray* rview = rays + S.ray_off + (FAN ? (long long)i * S.W : i);
        const __amdgpu_buffer_rsrc_t RR = row_rsrc(reinterpret_cast<const float*>(rview),
                                                   FAN ? S.W * (int)sizeof(Ray) : 0);
        const Ray r0 = rview[0];  // parallel beam: the view's ray constants
        const BinBounds<FAN> bounds(S, T.x, T.y, r0, last_bin);
        float vpart[N];  // this view's sums; compensated once per view
#pragma unroll
        for (int s = 0; s < N; ++s) vpart[s] = 0.0f;
        // the pixel g'^-1 q0: (R^k M)^-1 = R^k M, (R^k)^-1 = R^-k
        auto pixel = [&](int e2, float& fx, float& fy) {
            const float y = (e2 >> 2) ? -gy : gy;
            switch ((e2 >> 2) ? (e2 & 3) : (-e2 & 3)) {
                case 0: fx = gx; fy = y; break;
                case 1: fx = -y; fy = gx; break;
                case 2: fx = -gx; fy = -y; break;
                default: fx = y; fy = -gx; break;
            }
        };
        // the lane's candidate bins under element e2, and the wave's first
        auto range = [&](int e2, int& blo, int& bhi, int& c0) {
            float fx, fy;
            pixel(e2, fx, fy);
            bounds(fx, fy, blo, bhi);
            c0 = min(min(__builtin_amdgcn_readlane(blo, 0), __builtin_amdgcn_readlane(blo, 7)),
                     min(__builtin_amdgcn_readlane(blo, 56), __builtin_amdgcn_readlane(blo, 63)));
            // (no candidates: any bin, so that the load stays inside)
            c0 = __builtin_amdgcn_readfirstlane(min(c0, S.bhi));
        };
        auto load = [&](int c0, float4& val, float4& ray) {
            if constexpr (DIRECT) {
                float* v = &val.x;
#pragma unroll
                for (int q = 0; q < O::kPlane; ++q)
                    v[q] = __uint_as_float(
                        __builtin_amdgcn_raw_buffer_load_b32(RV, at0[q] + dir[q] * c0, 0, 0));
            } else if constexpr (N == 2) {
                const auto v = __builtin_amdgcn_raw_buffer_load_b64(RV, voff, c0 * 8, 0);
                val.x = __uint_as_float(v[0]);
                val.y = __uint_as_float(v[1]);
            } else {
                val = ldb128(RV, voff, c0 * 16);
            }
            if (FAN) ray = ldb128(RR, roff, c0 * (int)sizeof(Ray));
        };
        auto stage = [&](float4 val, const float4& ray) {
            if constexpr (DIRECT) {  // (the orbit sinogram holds the values divided by the rate)
                val.x *= S.inver;
                val.y *= S.inver;
                if constexpr (N > 2) {
                    val.z *= S.inver;
                    val.w *= S.inver;
                }
            }
            wave_lds_sync();  // the previous piece's reads are done
            if constexpr (N == 2) *reinterpret_cast<float2*>(&st->val[lane]) = make_float2(val.x, val.y);
            else st->val[lane] = val;
            if (FAN) st->ray[lane] = ray;
            wave_lds_sync();  // staged values visible to every lane
        };
        // bins blo..bhi, staged from c0 on
        auto sum = [&](auto e2c, int blo, int bhi, int c0) {
            constexpr int e2 = decltype(e2c)::value;
            if (blo > bhi) return;
            float fx, fy;
            pixel(e2, fx, fy);
            const float qd = FAN ? fan_depth_scale(fx, fy, T.x, T.y, S.invd) : 1.0f;
            // FBP fan weight d^2/qe^2 (prj/cpuPrj.c:258), folded into each weight
            const float fw = (FBP && FAN) ? 1.0f / (qd * qd) : 1.0f;
            const float4* at = st->val + (blo - c0);
            const float4* const end = st->val + (bhi - c0);
            float fb = (float)(blo - S.pC);  // parallel beam
            do {
                Ray r = r0;
                if (FAN) {
                    const float4 a = at[64], c = at[64 + CH];
                    r = Ray{a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
                } else {
                    r.dc = fb * S.dSize;
                    fb += 1.0f;
                }
                const float4 va = at[0], vb = at[N == 8 ? CH : 0];
                const float q[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
                const float dist = ray_dist(fx, fy, r.cosR, r.sinR, r.dc);
                float w = strip_area(dist, FAN ? r.hbc * qd : r.hbc, r);
                if (FBP && FAN) w *= fw;
#pragma unroll
                for (int s = 0; s < N; ++s)
                    vpart[s] = fmaf(w, q[O::slot(elem_mul(O::elem(s), e2))], vpart[s]);
            } while (++at <= end);
        };
        int blo, bhi, c0;
        float4 val{}, ray{};
        range(0, blo, bhi, c0);  // element 0 is in every set
        load(c0, val, ray);
        // element E2, the first piece of the next element of the set on its way meanwhile
#define CTPRJ_E(E2)                                                                          \
    if constexpr ((GSET >> E2) & 1u) {                                                       \
        constexpr unsigned rest = GSET & ~((2u << E2) - 1u);                                 \
        constexpr int NX = rest ? __builtin_ctz(rest) : 0;                                   \
        const int l = blo, h = bhi;                                                          \
        int p = c0, last = c0;                                                               \
        stage(val, ray);                                                                     \
        if (rest) {                                                                          \
            range(NX, blo, bhi, c0);                                                         \
            load(c0, val, ray);                                                              \
        }                                                                                    \
        if constexpr (COMPACT) {                                                             \
            sum(std::integral_constant<int, E2>{}, l, h, p);                                 \
        } else {                                                                             \
            if (__any(l <= h && (l < p || h >= p + CH))) {                                   \
                wave_range_i32(l <= h ? l : INT_MAX, l <= h ? h : INT_MIN, p, last);         \
                float4 v2{}, r2{};                                                           \
                load(p, v2, r2);                                                             \
                stage(v2, r2);                                                               \
            }                                                                                \
            for (;;) {                                                                       \
                sum(std::integral_constant<int, E2>{}, max(l, p), min(h, p + CH - 1), p);    \
                p += CH;                                                                     \
                if (p > last) break;                                                         \
                float4 v2{}, r2{};                                                           \
                load(p, v2, r2);                                                             \
                stage(v2, r2);                                                               \
            }                                                                                \
        }                                                                                    \
    }
        CTPRJ_E(0) CTPRJ_E(1) CTPRJ_E(2) CTPRJ_E(3) CTPRJ_E(4) CTPRJ_E(5) CTPRJ_E(6) CTPRJ_E(7)
#undef CTPRJ_E
#pragma unroll
        for (int s = 0; s < N; ++s) acc[s].add(vpart[s]);
    }
}

// Even n: row 0 and column 0 lie outside the pixel grid the projector reads; the adjoint
// writes them as 0 (prj/cpuPrj.c:713-716).  The work-group that stores a slice's marked
// tile (AdjItem.pad) does it; no orbit pixel lies there.
__device__ __forceinline__ void sym_zero_border(const SliceDesc& S, float* __restrict__ img)
{
    float* out = img + S.img_off;
    for (int i = threadIdx.x; i < S.n; i += blockDim.x) {
        out[i] = 0.0f;
        out[(long long)i * S.n] = 0.0f;
    }
}

// Orbit base pixels of a work item: an 8x8 tile of the fundamental domain of the group,
//   D4: 0 <= y0 <= x0 <= H,  V4: 0 <= x0, y0 <= H,  Z2: 0 <= x0 <= H, -H <= y0 <= H
// (tiles start inside it; the upper ends are checked here).
template <int GRP>
__device__ __forceinline__ bool adj_sym_base(const SliceDesc& S, const AdjItem& it, int lane,
                                             int& x0, int& y0)
{
    x0 = it.col0 + (lane & 7);
    y0 = it.row0 + (lane >> 3);
    return x0 <= S.H && y0 <= (GRP == kGrpD4 ? x0 : S.H);
}

// The sum t of orbit image h of (x0, y0) written to the image, unless an earlier element
// (in element order) reaches the same pixel: each distinct orbit pixel is written once.
template <bool FBP, int GRP>
__device__ __forceinline__ void adj_sym_store(const SliceDesc& S, int x0, int y0, int h, float t,
                                              float* __restrict__ img)
{
    constexpr GroupMasks G = group_masks(GRP);
    int ox, oy;
    apply_px(h & 3, h >> 2, x0, y0, ox, oy);
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        if (g >= h) break;
        if (!(G.all >> g & 1u)) continue;
        int gx, gy;
        apply_px(g & 3, g >> 2, x0, y0, gx, gy);
        if (gx == ox && gy == oy) return;
    }
    img[S.img_off + (long long)(oy + S.half) * S.n + ox + S.half] = FBP ? t * S.fbp_scale : t;
}

// Parallel beam: whether the bins that the pixels of any tile can read lie within one staged
// piece from its corners' first bin on, at any view.  The first bin is a sum of rounded
// monotone terms of the pixel, so no pixel's lies before the corners'; the pixels are 7 sqrt(2)
// < 9.91 apart, a pixel's footprint is sqrt(2) wide at most, and the strip and the margins
// come to it; two bins are rounding at both ends.
__device__ __forceinline__ bool adj_compact(const SliceDesc& S)
{
    return (9.91f + 1.42f + 2.0f * (S.hbd + kSupportMargin)) * 1.001f * S.invDSize + 2.0f <
           (float)kStageBins;
}

// The canonical views are cut into groups * SEG strided sets: set g * SEG + w, wave w's in
// group g, holds i = g * SEG + w + j * groups * SEG.  A work-group takes the groups first..last
// (more than one: SEG = 4 only), the waves' sums of a group being added in wave order (eight
// waves: as two groups of four) and the groups in theirs, here or, with part, one group's
// sums to part[h * 64 + lane], in k_adjoint_sym_combine: who adds changes no bit.
template <bool FAN, bool FBP, int SEG, int GRP, bool DIRECT>
__device__ __forceinline__ void adj_sym_tile(const SliceDesc& S, const AdjItem& it,
                                             const float4* __restrict__ views,
                                             const Ray* __restrict__ rays,
                                             const float* __restrict__ os,
                                             const int* __restrict__ tab,
                                             float* __restrict__ img,
                                             float (*red)[SEG][Orbit<GRP>::N][64],
                                             float (*tot)[64], int groups, int first, int last,
                                             float* __restrict__ part, AdjStage* __restrict__ stage)
{
    using O = Orbit<GRP>;
    // the wave index is uniform over the wave: the view loop then runs on scalar registers
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    constexpr bool kPar = !FAN, kFold = kPar && GRP != kGrpZ2;
#define CTPRJ_RUN(FOLD, COMPACT)                                                               \
    adj_sym_pixel<FAN, FBP, GRP, FOLD, DIRECT, COMPACT>(S, views, rays, os, tab, lane, x0, y0, \
                                                        valid, i0, step, acc, stage + wave)
    const int step = SEG * groups;
    if (!part && it.pad) sym_zero_border(S, img);
    if (SEG != 4) last = first;
#pragma unroll 1
    for (int g = first; g <= last; ++g) {
        // (formed anew for every group: kept from one to the next, what the walk derives from
        // the lane and its pixel takes 20 registers, a wave per SIMD)
        int lane = (int)threadIdx.x & 63, x0, y0;
        if (SEG == 4) asm("" : "+v"(lane));
        const bool valid = adj_sym_base<GRP>(S, it, lane, x0, y0);
        KahanAcc acc[O::N];
        const int i0 = g * SEG + wave;
        if (kPar && adj_compact(S)) {  // uniform over the launch's work-groups of the slice
            if (kFold && S.fold) CTPRJ_RUN(kFold, kPar);
            else CTPRJ_RUN(false, kPar);
        } else {
            if (kFold && S.fold) CTPRJ_RUN(kFold, false);
            else CTPRJ_RUN(false, false);
        }
        // (two buffers: a wave that is a group ahead does not disturb the sums below)
        auto* const r = red[SEG == 4 ? (g - first) & 1 : 0];
        if (SEG > 1) {
#pragma unroll
            for (int s = 0; s < O::N; ++s) r[wave][s][lane] = acc[s].s;
            __syncthreads();
        }
        // wave w finalises the elements h = w (mod SEG)
#pragma unroll
        for (int s = 0; s < O::N; ++s) {
            const int h = O::elem(s);
            if (SEG > 1 && h % SEG != wave) continue;
            float t = acc[s].s;
            if (SEG > 1) {
                t = r[0][s][lane];
#pragma unroll
                for (int q = 1; q < (SEG > 4 ? 4 : SEG); ++q) t += r[q][s][lane];
            }
            if (SEG > 4) {
                float u = r[SEG > 4 ? 4 : 0][s][lane];
#pragma unroll
                for (int q = 5; q < SEG; ++q) u += r[q][s][lane];
                t += u;
            }
            if (SEG == 4 && g > first) t = tot[s][lane] + t;
            if (SEG == 4 && g < last) tot[s][lane] = t;  // (its own lanes read it)
            else if (!valid) continue;
            else if (part) part[h * 64 + lane] = t;
            else adj_sym_store<FBP, GRP>(S, x0, y0, h, t, img);
        }
    }
#undef CTPRJ_RUN
}

// One launch per symmetry group; SEG waves split the canonical views and then share the final
// sums; with nsplit > 1, nsplit work-groups share the views of a tile, one group of sets each,
// and leave their sums in part (512 floats per work-group) for k_adjoint_sym_combine.  capped:
// a slice's views are cut into its own number of groups of four (agroups); one work-group
// takes them all (SEG = 4, or the two of SEG = 8) or up to nsplit do, the others end.
template <bool FBP, int SEG, int GRP, bool DIRECT>
__global__ __launch_bounds__(64 * SEG) void k_adjoint_sym(const SliceDesc* __restrict__ slices,
                                                          const AdjItem* __restrict__ items,
                                                          const float4* __restrict__ views,
                                                          const Ray* __restrict__ rays,
                                                          const float* __restrict__ os,
                                                          const int* __restrict__ tab,
                                                          float* __restrict__ img, int nitems,
                                                          int nsplit, bool capped,
                                                          float* __restrict__ part,
                                                          const RedJob job)
{
    __shared__ float red[SEG == 4 ? 2 : 1][SEG][Orbit<GRP>::N][64];
    __shared__ float tot[SEG == 4 ? Orbit<GRP>::N : 1][64];
    __shared__ AdjStage stage[SEG];
    if (job.out && blockIdx.x == 0 && threadIdx.x < 64) wave_sum_job(job);  // on the side
    int split, idx;
    split_item(nitems, split, idx);
    const AdjItem it = items[idx];
    if (it.slice < 0) return;  // uniform over the work-group
    const SliceDesc S = slices[it.slice];
    const int groups = capped && SEG == 4 ? S.agroups : nsplit;
    if (split >= groups) return;  // uniform over the work-group
    const int last = nsplit > 1 ? split : groups - 1;
    float* mine = part ? part + (long long)blockIdx.x * 512 : nullptr;
    if (S.fan)
        adj_sym_tile<true, FBP, SEG, GRP, DIRECT>(S, it, views, rays, os, tab, img, red, tot, groups,
                                                  split, last, mine, stage);
    else
        adj_sym_tile<false, FBP, SEG, GRP, DIRECT>(S, it, views, rays, os, tab, img, red, tot, groups,
                                                   split, last, mine, stage);
}

// The nsplit partial sums of each orbit image of a tile, added in split order and
// written like the one-work-group path (512 threads: orbit image h = thread / 64 of base
// pixel lane = thread % 64).
template <bool FBP, int GRP, bool CAPPED>
__global__ __launch_bounds__(512) void k_adjoint_sym_combine(const SliceDesc* __restrict__ slices,
                                                             const AdjItem* __restrict__ items,
                                                             int nitems, int nsplit,
                                                             const float* __restrict__ part,
                                                             float* __restrict__ img)
{
    const AdjItem it = items[blockIdx.x];
    if (it.slice < 0) return;
    const SliceDesc S = slices[it.slice];
    if (CAPPED) nsplit = min(nsplit, S.agroups);
    constexpr GroupMasks G = group_masks(GRP);
    if (it.pad) sym_zero_border(S, img);
    const int h = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    int x0, y0;
    if (!(G.all >> h & 1u) || !adj_sym_base<GRP>(S, it, lane, x0, y0)) return;
    const float* p = part + (long long)blockIdx.x * 512 + threadIdx.x;
    float t = p[0];
    for (int k = 1; k < nsplit; ++k) t += p[(long long)k * nitems * 512];
    adj_sym_store<FBP, GRP>(S, x0, y0, h, t, img);
}


// ----------------------------------------------------------------- launchers ---

template <int GRP, bool BHC>
static void launch_forward_sym_g(int seg, bool views4, int level, int nsplit,
                                 bool capped, float* part,
                                 int nitems,
                                 const SliceDesc* desc, const FwdItem* items, const float4* views,
                                 const Ray* rays, const float* orb, float* sino,
                                 const FwdBhc<BHC>& B, hipStream_t st)
{
    float* pp = nsplit > 1 ? part : nullptr;
    // work-groups per item of k_forward_views
    const int nwg = level < 0 ? 1 : level == 0 ? nsplit : (nsplit + level - 1) / level;
    const dim3 grid((unsigned)nitems * (unsigned)nsplit);
#define CTPRJ_LAUNCH(SEG)                                                                       \
    hipLaunchKernelGGL((k_forward_sym<SEG, GRP, BHC>), grid, dim3(64 * SEG), 0, st, desc, items, \
                       views, rays, orb, sino, nitems, nsplit, capped, pp, B)
    if (views4)
        hipLaunchKernelGGL((k_forward_views<GRP, BHC>),
                           dim3((unsigned)(nitems / 4) * (unsigned)nwg), dim3(256), 0, st, desc,
                           items, views, rays, orb, sino, nitems, nwg, level, capped ? 0 : nsplit,
                           pp != nullptr, part, B);
    else switch (seg) {
        case 1: CTPRJ_LAUNCH(1); break;
        case 2: CTPRJ_LAUNCH(2); break;
        case 4: CTPRJ_LAUNCH(4); break;
        case 8: CTPRJ_LAUNCH(8); break;
        default: CTPRJ_LAUNCH(16); break;
    }
#undef CTPRJ_LAUNCH
    if (!pp) return;
    auto* combine = capped ? k_forward_sym_combine<GRP, BHC, true> : k_forward_sym_combine<GRP, BHC, false>;
    hipLaunchKernelGGL(combine, dim3((unsigned)nitems), dim3(512), 0, st, desc, items, views, nitems,
                       nsplit, views4 && level == 0, pp, sino, B);
}

template <bool BHC>
static void launch_forward_sym_b(int grp, int seg, bool views4, int level, int nsplit,
                                 bool capped,
                                 float* part, int nitems,
                                 const SliceDesc* desc, const FwdItem* items, const float4* views,
                                 const Ray* rays, const float* orb, float* sino,
                                 const FwdBhc<BHC>& B, hipStream_t st)
{
    if (grp == kGrpD4)
        launch_forward_sym_g<kGrpD4, BHC>(seg, views4, level, nsplit, capped, part, nitems, desc, items,
                                          views, rays, orb, sino, B, st);
    else if (grp == kGrpV4)
        launch_forward_sym_g<kGrpV4, BHC>(seg, views4, level, nsplit, capped, part, nitems, desc, items,
                                          views, rays, orb, sino, B, st);
    else
        launch_forward_sym_g<kGrpZ2, BHC>(seg, views4, level, nsplit, capped, part, nitems, desc, items,
                                          views, rays, orb, sino, B, st);
}

void launch_forward_sym(int grp, int seg, bool views4, int level, int nsplit,
                                 bool capped, float* part,
                        int nitems,
                        const SliceDesc* desc, const FwdItem* items, const float4* views,
                        const Ray* rays, const float* orb, float* sino, const BhcStore* bhc,
                        hipStream_t st)
{
    if (bhc) {
        FwdBhc<true> B;
        static_cast<BhcStore&>(B) = *bhc;
        launch_forward_sym_b<true>(grp, seg, views4, level, nsplit, capped, part, nitems, desc, items,
                                   views, rays, orb, sino, B, st);
    } else {
        launch_forward_sym_b<false>(grp, seg, views4, level, nsplit, capped, part, nitems, desc, items,
                                    views, rays, orb, sino, FwdBhc<false>{}, st);
    }
}

template <bool FBP, int GRP>
static void launch_adjoint_sym_t(int seg, int nsplit, bool capped, float* part, int nitems,
                                 const SliceDesc* desc, const AdjItem* items, const float4* views,
                                 const Ray* rays, const float* os, const int* direct, float* img,
                                 const RedJob& job, hipStream_t st)
{
    float* pp = nsplit > 1 ? part : nullptr;
    const dim3 grid((unsigned)nitems * (unsigned)nsplit);
#define CTPRJ_LAUNCH(SEG)                                                                      \
    hipLaunchKernelGGL((direct ? k_adjoint_sym<FBP, SEG, GRP, true>                            \
                               : k_adjoint_sym<FBP, SEG, GRP, false>),                         \
                       grid, dim3(64 * SEG), 0, st, desc, items, views, rays, os, direct, img, \
                       nitems, nsplit, capped, pp, job)
    switch (seg) {
        case 1: CTPRJ_LAUNCH(1); break;
        case 2: CTPRJ_LAUNCH(2); break;
        case 4: CTPRJ_LAUNCH(4); break;
        default: CTPRJ_LAUNCH(8); break;
    }
#undef CTPRJ_LAUNCH
    if (!pp) return;
    auto* combine = capped ? k_adjoint_sym_combine<FBP, GRP, true> : k_adjoint_sym_combine<FBP, GRP, false>;
    hipLaunchKernelGGL(combine, dim3((unsigned)nitems), dim3(512), 0, st, desc, items, nitems, nsplit,
                       pp, img);
}

template <bool FBP>
static void launch_adjoint_sym_f(int grp, int seg, int nsplit, bool capped, float* part, int nitems,
                                 const SliceDesc* desc, const AdjItem* items, const float4* views,
                                 const Ray* rays, const float* os, const int* direct, float* img,
                                 const RedJob& job, hipStream_t st)
{
    if (grp == kGrpD4)
        launch_adjoint_sym_t<FBP, kGrpD4>(seg, nsplit, capped, part, nitems, desc, items, views, rays, os,
                                          direct, img, job, st);
    else if (grp == kGrpV4)
        launch_adjoint_sym_t<FBP, kGrpV4>(seg, nsplit, capped, part, nitems, desc, items, views, rays, os,
                                          direct, img, job, st);
    else
        launch_adjoint_sym_t<FBP, kGrpZ2>(seg, nsplit, capped, part, nitems, desc, items, views, rays, os,
                                          direct, img, job, st);
}

void launch_adjoint_sym(bool fbp, int grp, int seg, int nsplit, bool capped, float* part,
                        int nitems,
                        const SliceDesc* desc, const AdjItem* items, const float4* views,
                        const Ray* rays, const float* os, const int* direct, float* img,
                        const RedJob& job, hipStream_t st)
{
    if (fbp)
        launch_adjoint_sym_f<true>(grp, seg, nsplit, capped, part, nitems, desc, items, views, rays, os,
                                   direct, img, job, st);
    else
        launch_adjoint_sym_f<false>(grp, seg, nsplit, capped, part, nitems, desc, items, views, rays, os,
                                    direct, img, job, st);
}

}  // namespace ctprj
