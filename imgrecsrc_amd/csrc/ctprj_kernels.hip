// Projector kernels for gfx950: ray-driven forward gather, pixel-driven adjoint gather,
// FBP ramp filter, ray-table construction and image transpose.
//
// Work decomposition (all slices of a plan in one launch each):
//   forward : one work item = (slice, view, run of consecutive bins); one thread per
//             ray.  Views closer to the x axis (|cos| >= |sin|) walk image rows and
//             gather along the row; the others walk the rows of the transposed image,
//             so every gather is along a contiguous row.  Consecutive bins of a view are
//             adjacent lanes: neighbouring lanes read neighbouring pixels and the
//             sinogram store is one coalesced run per wave.
//   adjoint : one work item = (slice, pixel tile); one thread per pixel, gathering
//             over every view and the bins whose strip meets the pixel.  No atomics.
//
// Reference semantics: prj/cpuPrj.c:319-616 (forward), :46-317 (adjoint), :718-784 (FBP).
#include "ctprj_internal.h"

namespace ctprj {

// ------------------------------------------------------------------ ray table ---

// views[v] = (cosT, sinT, 0, 0); bins[b] = (cosB, sinB, d*t/sqrt(d^2+t^2), beamWidth*cosB)
// for fan slices (host-computed in the reference's float expressions).
__global__ void k_build_rays(const SliceDesc* __restrict__ slices, int nslices,
                             const float4* __restrict__ views, const float4* __restrict__ bins,
                             const long long* __restrict__ bin_off,
                             const long long* __restrict__ ray_prefix, Ray* __restrict__ rays)
{
    const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= ray_prefix[nslices]) return;
    int lo = 0, hi = nslices - 1;  // slice owning gid: last prefix <= gid
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (ray_prefix[mid] <= gid) lo = mid; else hi = mid - 1;
    }
    const SliceDesc S = slices[lo];
    const long long local = gid - ray_prefix[lo];
    Ray r;
    if (S.fan) {
        const int v = (int)(local / S.W), b = (int)(local % S.W);
        const float4 T = views[S.view_off + v];
        const float4 B = bins[bin_off[lo] + b];
        // prj/cpuPrj.c:505-506; explicit roundings, no contraction
        r.cosR = __fsub_rn(__fmul_rn(B.x, T.x), __fmul_rn(B.y, T.y));
        r.sinR = __fadd_rn(__fmul_rn(B.y, T.x), __fmul_rn(B.x, T.y));
        r.dc = B.z;
        r.hbc = 0.5f * B.w;
    } else {
        const float4 T = views[S.view_off + local];
        r.cosR = T.x;
        r.sinR = T.y;
        r.dc = 0.0f;
        r.hbc = S.hbd;
    }
    const double c = fabs((double)r.cosR), s = fabs((double)r.sinR);
    const double ramp = fmax(fmin(c, s), 0x1p-24), b1 = fmax(0.5 * (fmax(c, s) - ramp), 0x1p-25);
    r.is = (float)(1.0 / ramp);
    r.c2 = (float)((b1 + ramp) / ramp);
    r.ib = (float)(0.5 / b1);
    r.a = (float)(0.5 * ramp / (ramp + 2.0 * b1));
    rays[S.ray_off + local] = r;
}

// -------------------------------------------------------------------- transpose ---

// out[j][i] = in[i][j] for every slice; 32x32 tiles through LDS.
__global__ __launch_bounds__(256) void k_transpose(const SliceDesc* __restrict__ slices,
                                                   const AdjItem* __restrict__ items,
                                                   const float* __restrict__ in,
                                                   float* __restrict__ out)
{
    __shared__ float tile[32][33];
    const AdjItem it = items[blockIdx.x];
    const SliceDesc S = slices[it.slice];
    const float* src = in + S.img_off;
    float* dst = out + S.img_off;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
    for (int k = 0; k < 32; k += 8) {
        const int r = it.row0 + ty + k, c = it.col0 + tx;
        if (r < S.n && c < S.n) tile[ty + k][tx] = src[(long long)r * S.n + c];
    }
    __syncthreads();
    for (int k = 0; k < 32; k += 8) {
        const int r = it.col0 + ty + k, c = it.row0 + tx;
        if (r < S.n && c < S.n) dst[(long long)r * S.n + c] = tile[tx][ty + k];
    }
}

// ---------------------------------------------------------------------- forward ---

template <bool FAN, bool COUNT>
__device__ __forceinline__ float forward_ray(const SliceDesc& S, const Ray& r, float cT, float sT,
                                             const float* __restrict__ img,
                                             const float* __restrict__ imgT)
{
    const bool rowmode = fabsf(cT) >= fabsf(sT);
    const RowBounds rb = row_bounds(r, cT, sT, FAN ? S.invd : 0.0f, rowmode);
    const int H = S.H, n = S.n, half = S.half;
    const float* base = (rowmode ? img : imgT) + S.img_off;
    // plain sums over blocks of 4 rows, compensated across blocks
    KahanAcc acc;
    float part = 0.0f;
    for (int v = -H; v <= H; ++v) {
        int lo, hi;
        row_range(rb, (float)v, H, lo, hi);
        const float* row = base + (long long)(v + half) * n + half;
        for (int u = lo; u <= hi; ++u) {
            const float x = rowmode ? (float)u : (float)v;
            const float y = rowmode ? (float)v : (float)u;
            const float dist = ray_dist(x, y, r.cosR, r.sinR, r.dc);
            if (COUNT) {
                const float qd = fmaf(fmaf(x, sT, -(y * cT)), S.invd, 1.0f);
                part += strip_hits(dist, FAN ? r.hbc * qd : r.hbc, r) ? 1.0f : 0.0f;
            } else {
                const float qd = FAN ? fan_depth_scale(x, y, cT, sT, S.invd) : 1.0f;
                part = fmaf(strip_area(dist, FAN ? r.hbc * qd : r.hbc, r), row[u], part);
            }
        }
        if (((v + H) & 3) == 3 || v == H) {
            acc.add(part);
            part = 0.0f;
        }
    }
    return COUNT ? acc.s : acc.s * S.inver;
}

template <bool COUNT>
__global__ __launch_bounds__(256) void k_forward(const SliceDesc* __restrict__ slices,
                                                 const FwdItem* __restrict__ items,
                                                 const float4* __restrict__ views,
                                                 const Ray* __restrict__ rays,
                                                 const float* __restrict__ img,
                                                 const float* __restrict__ imgT,
                                                 float* __restrict__ sino)
{
    const FwdItem it = items[blockIdx.x];
    if (it.slice < 0) return;
    const SliceDesc S = slices[it.slice];
    const int b = it.bin0 + (int)threadIdx.x;
    if (b >= S.W) return;
    float* out = sino + S.sino_off + (long long)it.view * S.W + b;
    if (b < S.blo || b > S.bhi) {  // even detector: bin 0 carries no ray
        *out = 0.0f;
        return;
    }
    const float4 T = views[S.view_off + it.view];
    float val;
    if (S.fan) {
        const Ray r = rays[S.ray_off + (long long)it.view * S.W + b];
        val = forward_ray<true, COUNT>(S, r, T.x, T.y, img, imgT);
    } else {
        Ray r = rays[S.ray_off + it.view];
        r.dc = (float)(b - S.pC) * S.dSize;
        val = forward_ray<false, COUNT>(S, r, T.x, T.y, img, imgT);
    }
    *out = val;
}

// ---------------------------------------------------------------------- adjoint ---

template <bool FAN, bool FBP>
__device__ __forceinline__ float adjoint_pixel(const SliceDesc& S, int x, int y,
                                               const float4* __restrict__ views,
                                               const Ray* __restrict__ rays,
                                               const float* __restrict__ sino)
{
    const float fx = (float)x, fy = (float)y;
    const float* srow = sino + S.sino_off;
    // plain sums over blocks of 4 views, compensated across blocks
    KahanAcc acc;
    float vsum = 0.0f;
    for (int a = 0; a < S.np; ++a, srow += S.W) {
        const float4 T = views[S.view_off + a];
        const float cT = T.x, sT = T.y;
        int blo, bhi;
        float qd = 1.0f;
        if (FAN) {
            // perspective shadow of the pixel on the virtual detector (4 corners)
            const float oc = fmaf(fx, cT, fy * sT);
            const float qe = fmaf(fx, sT, fmaf(-fy, cT, S.d));
            const float hc = 0.5f * (cT + sT), hd = 0.5f * (cT - sT);
            // corners (x-.5,y-.5),(x+.5,y-.5),(x+.5,y+.5),(x-.5,y+.5)
            const float t0 = S.d * (oc - hc) * fast_rcp(qe + hd);
            const float t1 = S.d * (oc + hd) * fast_rcp(qe + hc);
            const float t2 = S.d * (oc + hc) * fast_rcp(qe - hd);
            const float t3 = S.d * (oc - hd) * fast_rcp(qe - hc);
            const float tl = fminf(fminf(t0, t1), fminf(t2, t3));
            const float tr = fmaxf(fmaxf(t0, t1), fmaxf(t2, t3));
            const float m = S.hbd + kSupportMargin * S.dSize;
            blo = (int)ceilf((tl - m) * S.invDSize + (float)S.pC);
            bhi = (int)floorf((tr + m) * S.invDSize + (float)S.pC);
            qd = fan_depth_scale(fx, fy, cT, sT, S.invd);
        } else {
            const Ray r = rays[S.ray_off + a];
            const float center = fmaf(fx, cT, fy * sT);
            const float ext = 0.5f * (fabsf(cT) + fabsf(sT)) + r.hbc + kSupportMargin;
            blo = (int)ceilf((center - ext) * S.invDSize + (float)S.pC);
            bhi = (int)floorf((center + ext) * S.invDSize + (float)S.pC);
        }
        blo = max(blo, S.blo);
        bhi = min(bhi, S.bhi);
        float part = 0.0f;
        if (FAN) {
            const Ray* rr = rays + S.ray_off + (long long)a * S.W;
            for (int b = blo; b <= bhi; ++b) {
                const Ray r = rr[b];
                const float dist = ray_dist(fx, fy, r.cosR, r.sinR, r.dc);
                const float w = strip_area(dist, r.hbc * qd, r);
                part = fmaf(w, srow[b], part);
            }
            if (FBP) part *= 1.0f / (qd * qd);  // d^2/qe^2, prj/cpuPrj.c:258
        } else {
            const Ray r = rays[S.ray_off + a];
            for (int b = blo; b <= bhi; ++b) {
                const float dc = (float)(b - S.pC) * S.dSize;
                const float dist = ray_dist(fx, fy, r.cosR, r.sinR, dc);
                const float w = strip_area(dist, r.hbc, r);
                part = fmaf(w, srow[b], part);
            }
        }
        vsum += part;
        if ((a & 3) == 3 || a == S.np - 1) {
            acc.add(vsum);
            vsum = 0.0f;
        }
    }
    return acc.s;
}

template <int TILE, bool FBP>
__global__ __launch_bounds__(TILE* TILE) void k_adjoint(const SliceDesc* __restrict__ slices,
                                                        const AdjItem* __restrict__ items,
                                                        const float4* __restrict__ views,
                                                        const Ray* __restrict__ rays,
                                                        const float* __restrict__ sino,
                                                        float* __restrict__ img)
{
    const AdjItem it = items[blockIdx.x];
    if (it.slice < 0) return;
    const SliceDesc S = slices[it.slice];
    const int row = it.row0 + (int)threadIdx.x / TILE;
    const int col = it.col0 + (int)threadIdx.x % TILE;
    if (row >= S.n || col >= S.n) return;
    const int x = col - S.half, y = row - S.half;
    float val = 0.0f;
    // even n: row 0 and column 0 stay 0
    if (x >= -S.H && x <= S.H && y >= -S.H && y <= S.H) {
        if (S.fan) val = adjoint_pixel<true, FBP>(S, x, y, views, rays, sino);
        else val = adjoint_pixel<false, FBP>(S, x, y, views, rays, sino);
        val *= FBP ? S.fbp_scale * S.inver : S.inver;
    }
    img[S.img_off + (long long)row * S.n + col] = val;
}

// --------------------------------------------------------------------------- FBP ---

// Fan cosine pre-weight (prj/cpuPrj.c:737-751) and Hann-windowed ramp filter
// (prj/utils.h:94-151).  The FFT filter of the reference is a circular convolution over 2W
// samples of the zero-padded view with g = 0.5 h + 0.25 h(.-1) + 0.25 h(.+1), h the periodic
// Ram-Lak kernel; g is tabulated on the host (2W floats per slice at kern_off).
// out[i] = sum_j v[j] g[(i-j) mod 2W]: a product with a Toeplitz matrix.
//
// A work-group forms 256 outputs of four views; its eight waves split the taps j of each
// chunk, and a lane keeps 4 outputs x 4 views: per 8 taps it reads 12 values of g (three
// 16-byte reads, each serving up to 16 products) and 8 x 4 samples (broadcast) for 128 FMAs.
// One view per work-group with an LDS read of g and of v per product was bound by those
// reads: 360 views of 729 bins 73 us, now 18.  Products are summed in runs of kFbpRun taps
// and the runs, and then the eight waves, with compensation.
constexpr int kFbpViews = kFbpItemViews, kFbpOuts = 256, kFbpWaves = 8, kFbpRun = 64;
constexpr int kFbpChunk = 1024;  // taps staged at once: a multiple of 8 taps per wave

__global__ __launch_bounds__(64 * kFbpWaves) void k_fbp_filter(
    const SliceDesc* __restrict__ slices, const int2* __restrict__ items,
    const float* __restrict__ kern, const long long* __restrict__ kern_off,
    const float* __restrict__ preweight, const long long* __restrict__ prew_off,
    const float* __restrict__ sino, float* __restrict__ out)
{
    __shared__ float4 v[kFbpChunk];                   // v[tap]: the four views' samples
    __shared__ __attribute__((aligned(16))) float g[kFbpChunk + kFbpOuts];
    __shared__ float red[kFbpWaves][kFbpViews][kFbpOuts];
    const int2 it = items[blockIdx.x];
    const SliceDesc S = slices[it.x];
    const int W = S.W, L = 2 * W, i0 = (int)blockIdx.y * kFbpOuts;
    if (i0 >= W) return;  // uniform over the work-group
    const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
    const float* src = sino + S.sino_off + (long long)it.y * W;
    const float* pw = preweight + prew_off[it.x];
    const float* kk = kern + kern_off[it.x];
    const int nview = min(kFbpViews, S.np - it.y);
    KahanAcc acc[kFbpViews][4];
    for (int j0 = 0; j0 < W; j0 += kFbpChunk) {
        // taps of this chunk, a multiple of 8 per wave; samples past W are 0
        const int taps = min(kFbpChunk, (W - j0 + 8 * kFbpWaves - 1) / (8 * kFbpWaves) * (8 * kFbpWaves));
        __syncthreads();  // the previous chunk's reads are done
        for (int j = t; j < taps; j += 64 * kFbpWaves) {
            float q[kFbpViews];
            const bool in = j0 + j < W;
            const float w = in && S.fan ? pw[j0 + j] : 1.0f;
#pragma unroll
            for (int a = 0; a < kFbpViews; ++a)
                q[a] = in && a < nview ? src[(long long)a * W + j0 + j] * w : 0.0f;
            v[j] = make_float4(q[0], q[1], q[2], q[3]);
        }
        // g[x] is the kernel at i - j = x + i0 - j0 - taps (0 where no output needs it)
        for (int x = t; x < taps + kFbpOuts; x += 64 * kFbpWaves) {
            const int k = x + i0 - j0 - taps;
            g[x] = k > -W && k < W ? kk[k < 0 ? k + L : k] : 0.0f;
        }
        __syncthreads();
        const int per = taps / kFbpWaves, ja = wave * per, jb = ja + per;
        for (int jr = ja; jr < jb; jr += kFbpRun) {
            float part[kFbpViews][4] = {};
            for (int j = jr; j < min(jb, jr + kFbpRun); j += 8) {
                // outputs i0 + 4 lane + r, taps j0 + j + s: kernel value r - s + 8 of the window
                const float4* w4 = reinterpret_cast<const float4*>(g + 4 * lane - j + taps - 8);
                const float4 wa = w4[0], wb = w4[1], wc = w4[2];
                const float w[12] = {wa.x, wa.y, wa.z, wa.w, wb.x, wb.y,
                                     wb.z, wb.w, wc.x, wc.y, wc.z, wc.w};
#pragma unroll
                for (int s = 0; s < 8; ++s) {
                    const float4 q = v[j + s];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        part[0][r] = fmaf(q.x, w[r - s + 8], part[0][r]);
                        part[1][r] = fmaf(q.y, w[r - s + 8], part[1][r]);
                        part[2][r] = fmaf(q.z, w[r - s + 8], part[2][r]);
                        part[3][r] = fmaf(q.w, w[r - s + 8], part[3][r]);
                    }
                }
            }
#pragma unroll
            for (int a = 0; a < kFbpViews; ++a)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[a][r].add(part[a][r]);
        }
    }
#pragma unroll
    for (int a = 0; a < kFbpViews; ++a)
        *reinterpret_cast<float4*>(&red[wave][a][4 * lane]) =
            make_float4(acc[a][0].s, acc[a][1].s, acc[a][2].s, acc[a][3].s);
    __syncthreads();
    for (int x = t; x < kFbpViews * kFbpOuts; x += 64 * kFbpWaves) {
        const int a = x / kFbpOuts, i = x % kFbpOuts;
        if (a >= nview || i0 + i >= W) continue;
        KahanAcc sum;
#pragma unroll
        for (int w = 0; w < kFbpWaves; ++w) sum.add(red[w][a][i]);
        out[S.sino_off + (long long)(it.y + a) * W + i0 + i] = sum.s;
    }
}

// ---------------------------------------------------------------------- helpers ---

__global__ void k_scale(float* __restrict__ p, long long n, float s)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] *= s;
}

// -------------------------------------------------------------------- launchers ---

void launch_build_rays(const SliceDesc* desc, int nslices, const float4* views,
                       const float4* bins, const long long* bin_off, const long long* ray_prefix,
                       Ray* rays, long long nray, hipStream_t st)
{
    const int threads = 256;
    const long long blocks = (nray + threads - 1) / threads;
    if (blocks > 0)
        hipLaunchKernelGGL(k_build_rays, dim3((unsigned)blocks), dim3(threads), 0, st, desc,
                           nslices, views, bins, bin_off, ray_prefix, rays);
}

void launch_transpose(int nitems, const SliceDesc* desc, const AdjItem* items, const float* in,
                      float* out, hipStream_t st)
{
    if (nitems > 0)
        hipLaunchKernelGGL(k_transpose, dim3(nitems), dim3(256), 0, st, desc, items, in, out);
}

void launch_forward_kernel(bool count, int block, int nitems, const SliceDesc* desc,
                           const FwdItem* items, const float4* views, const Ray* rays,
                           const float* img, const float* imgT, float* sino, hipStream_t st)
{
    if (count)
        hipLaunchKernelGGL(k_forward<true>, dim3(nitems), dim3(block), 0, st, desc, items,
                           views, rays, img, imgT, sino);
    else
        hipLaunchKernelGGL(k_forward<false>, dim3(nitems), dim3(block), 0, st, desc, items,
                           views, rays, img, imgT, sino);
}

void launch_adjoint_kernel(int tile, bool fbp, int nitems, const SliceDesc* desc,
                           const AdjItem* items, const float4* views, const Ray* rays,
                           const float* sino, float* img, hipStream_t st)
{
    if (tile == 8) {
        if (fbp)
            hipLaunchKernelGGL((k_adjoint<8, true>), dim3(nitems), dim3(64), 0, st, desc, items,
                               views, rays, sino, img);
        else
            hipLaunchKernelGGL((k_adjoint<8, false>), dim3(nitems), dim3(64), 0, st, desc, items,
                               views, rays, sino, img);
    } else {
        if (fbp)
            hipLaunchKernelGGL((k_adjoint<16, true>), dim3(nitems), dim3(256), 0, st, desc, items,
                               views, rays, sino, img);
        else
            hipLaunchKernelGGL((k_adjoint<16, false>), dim3(nitems), dim3(256), 0, st, desc,
                               items, views, rays, sino, img);
    }
}

void launch_fbp_filter(int nitems, int max_W, const SliceDesc* desc, const int2* items,
                       const float* kern, const long long* kern_off, const float* prew,
                       const long long* prew_off, const float* sino, float* out, hipStream_t st)
{
    hipLaunchKernelGGL(k_fbp_filter, dim3(nitems, (max_W + kFbpOuts - 1) / kFbpOuts),
                       dim3(64 * kFbpWaves), 0, st, desc, items, kern, kern_off, prew, prew_off,
                       sino, out);
}

void launch_scale(float* p, long long n, float s, hipStream_t st)
{
    const long long blocks = (n + 255) / 256;
    if (blocks > 0) hipLaunchKernelGGL(k_scale, dim3((unsigned)blocks), dim3(256), 0, st, p, n, s);
}

}  // namespace ctprj
