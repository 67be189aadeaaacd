// Total-variation proximal step on gfx950: argmin 0.5||D - X||^2 + lambda TV(D) over
// D >= 0 by the fast gradient projection on the dual (utils/denoise_bound_mod.m, as
// utils/TV.m:56-80 calls it), isotropic or l1 TV (utils/tlv.m), and the TV value.
//
// One iteration is one launch over the pixels: the primal step (C = X - lambda
// Lforward(R), D = max(C, 0), with the FP64 partial sums of ||D - Dold||^2, ||D||^2,
// ||C - D||^2 and ||C||^2) at a pixel and its lower and right neighbours, and the pixel's
// dual step (P = proj(R + Ltrans(D)/(8 lambda)), then the momentum
// R = P + (tk - 1)(P - Pold)/tkp1, into the other of two R buffers).  Every work-group first
// adds the previous iteration's partial sums for itself, in one fixed order, and so knows
// the stopping test's and the momentum restart's outcome without a launch in between.  The
// dual fields P1 (vertical differences, rows 0..m-2) and P2 (horizontal, columns 0..n-2)
// are stored padded to m x n.  The host reads the state once per eight iterations, from
// host memory that a one-work-group launch writes, with the next eight already queued.  All arithmetic is FP64 in the
// reference's order; images are FP32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <new>
#include <vector>

#include "ctprj_internal.h"

namespace ctprj {

constexpr int kTvBlock = 256;
// Work-groups of an iteration, at most: every one of them reads all the partial sums (32 B
// each), which 1024 keep at 32 MB a launch from L2; larger images give a group several runs
// of kTvBlock pixels.  24 iterations at 512^2, 800^2 and 2048^2: 310, 434 and 1949 us with
// 1024, 262, 409 and 1950 with 512, 250, 439 and 1999 with 256.  (The line was drawn when the
// sums took three times the shuffles and few groups lost: 392, 600, 2357 with 1024 against 401,
// 728, 3489 with 512.)
constexpr long long kTvGroups = 1024;

// Sum of four values over the work-group, the same in every thread: each wave's lanes by
// a butterfly, then the waves in order.
__device__ __forceinline__ void tv_group_sum4(double v[4])
{
    __shared__ double sh[kTvBlock / 64][4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] += __shfl_xor(v[k], off, 64);
    const int wave = (int)threadIdx.x >> 6;
    __syncthreads();  // an earlier call's reads are done
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < 4; ++k) sh[wave][k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v[k] = sh[0][k];
#pragma unroll
        for (int w = 1; w < kTvBlock / 64; ++w) v[k] += sh[w][k];
    }
}

__device__ __forceinline__ void tv_block_sum4(double v[4], double* part)
{
    tv_group_sum4(v);
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < 4; ++k) part[4 * (long long)blockIdx.x + k] = v[k];
}

// The work-group's sums of four values as an iteration keeps them: sum k of group b at
// part[k nblk + b].  A wave's lanes halve the values they hold with the first two exchanges
// (lane l ends with value l / 16, summed over lanes of equal l % 16 first), 14 shuffled words
// where a butterfly of all four takes 48: LDS, which carries the shuffles, is a good part of a
// small iteration's time.
__device__ __forceinline__ void tv_store_sum4(const double v[4], double* part, long long nblk)
{
    __shared__ double sh[kTvBlock / 64][4];
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    const bool hi = lane & 32, up = lane & 16;
    const double a0 = hi ? v[2] : v[0], a1 = hi ? v[3] : v[1];
    const double b0 = hi ? v[0] : v[2], b1 = hi ? v[1] : v[3];
    const double c0 = a0 + __shfl_xor(b0, 32, 64), c1 = a1 + __shfl_xor(b1, 32, 64);
    double s = (up ? c1 : c0) + __shfl_xor(up ? c0 : c1, 16, 64);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((lane & 15) == 0) sh[wave][lane >> 4] = s;
    __syncthreads();
    if (threadIdx.x < 4) {
        double t = sh[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < kTvBlock / 64; ++w) t += sh[w][threadIdx.x];
        part[threadIdx.x * nblk + blockIdx.x] = t;
    }
}

// Those sums over all groups, the same in every thread: wave k adds value k.
__device__ __forceinline__ void tv_total4(const double* __restrict__ part, long long nblk, double a[4])
{
    static_assert(kTvBlock == 256, "a wave per value");
    __shared__ double sh[4];
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    const double* p = part + wave * nblk;
    double s = 0.0;
#pragma unroll 4
    for (int b = lane; b < (int)nblk; b += 64) s += p[b];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    if (lane == 0) sh[wave] = s;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] = sh[k];
}

// FGP loop state (utils/denoise_bound_mod.m:95-150) before an iteration; launches queued
// after the stop do nothing.
struct TvCtl {
    double t;     // tk of the next iteration (the last tkp1, or 1 after a restart)
    double fval;  // objective of the last iteration
    int i, count, done, pad;
};

// tkp1 from tk (utils/denoise_bound_mod.m:117), the same expression wherever it is formed
__device__ __forceinline__ double tv_next_t(double tk) { return (1.0 + sqrt(1.0 + 4.0 * tk * tk)) / 2.0; }

// End of an iteration (utils/denoise_bound_mod.m:146-150): re = ||D - Dold|| / ||D||
// counts towards the stop below epsilon, fval = -||C - D||^2 + ||C||^2, a rising fval
// restarts the momentum (tkp1 = 1); stop after maxIter iterations or 5 in a row below
// epsilon.  The per-group partials are summed in a fixed order; every thread of the
// work-group gets the state.
__device__ __forceinline__ TvCtl tv_advance(TvCtl c, const double* __restrict__ part,
                                            long long nblk, double epsilon, int maxIter)
{
    if (c.done) return c;  // uniform
    double a[4];
    tv_total4(part, nblk, a);
    const double re = sqrt(a[0]) / sqrt(a[1]);
    const double fval = -a[2] + a[3];
    const double tkp1 = tv_next_t(c.t);
    c.count = (re < epsilon) ? c.count + 1 : 0;
    c.t = (fval > c.fval) ? 1.0 : tkp1;
    c.fval = fval;
    c.i += 1;
    c.done = c.i >= maxIter || c.count >= 5;
    return c;
}

// What an iteration reads at pixel t = (i, j) of its image: X and R at the pixel, its lower
// and right neighbours and what their differences take (zero outside the image), D and P.
struct TvPix {
    int i, j;
    double x, xd, xr;              // X at t, t + n, t + 1
    double r1, r1u, r1d, r1r, r1q;  // R1 at t, t - n, t + n, t + 1, t + 1 - n
    double r2, r2l, r2r, r2d, r2q;  // R2 at t, t - 1, t + 1, t + n, t + n - 1
    double d, p1, p2;
};

__device__ __forceinline__ TvPix tv_load(const double* __restrict__ X, const double* D,
                                         const double* P1, const double* P2,
                                         const double* __restrict__ R1,
                                         const double* __restrict__ R2, long long t, int m, int n)
{
    TvPix q;
    const unsigned row = (unsigned)t / (unsigned)n;  // fewer than 2^31 pixels
    q.j = (int)((unsigned)t - row * (unsigned)n);
    q.i = (int)(row % (unsigned)m);
    const bool up = q.i > 0, left = q.j > 0, down = q.i < m - 1, right = q.j < n - 1;
    q.x = X[t];
    q.xd = down ? X[t + n] : 0.0;
    q.xr = right ? X[t + 1] : 0.0;
    q.r1 = R1[t];
    q.r1u = up ? R1[t - n] : 0.0;
    q.r1d = down ? R1[t + n] : 0.0;
    q.r1r = right ? R1[t + 1] : 0.0;
    q.r1q = right && up ? R1[t + 1 - n] : 0.0;
    q.r2 = R2[t];
    q.r2l = left ? R2[t - 1] : 0.0;
    q.r2r = right ? R2[t + 1] : 0.0;
    q.r2d = down ? R2[t + n] : 0.0;
    q.r2q = down && left ? R2[t + n - 1] : 0.0;
    q.d = D[t];
    q.p1 = P1[t];
    q.p2 = P2[t];
    return q;
}

// C = X - lambda Lforward(R) (utils/Lforward.m) from X and R1, R2 at the pixel and at the
// upper and left ones; R1 is zero on the last row and R2 on the last column.
__device__ __forceinline__ double tv_primal(double x, double r1, double r1u, double r2, double r2l,
                                            double lam)
{
    return __dsub_rn(x, __dmul_rn(lam, (r1 - r1u) + (r2 - r2l)));
}

// Iteration c0's state says (utils/denoise_bound_mod.m:118-144 with utils/Lforward.m and
// utils/Ltrans.m).  first: that state is complete; otherwise it is the previous
// iteration's, whose partial sums are in part0.  Group 0 keeps the new state in c1.
// Bound by the chain state -> partial sums -> pixels -> partial sums at small images, by the
// 88 B a pixel moves at large ones; so a group's first pixels are requested before the sums
// are added: 24 iterations with their launches take 300 us at 512^2 and 1.95 ms at 2048^2, and
// took 595 and 2.6 as primal, dual and control launches; without the early request 40 us more
// at 512^2.
__global__ __launch_bounds__(kTvBlock) void k_tv_iter(
    const double* __restrict__ X, double* __restrict__ D, double* __restrict__ P1,
    double* __restrict__ P2, const double* __restrict__ R1, const double* __restrict__ R2,
    double* __restrict__ N1, double* __restrict__ N2, int m, int n, long long total,
    long long chunk, double lam, int iso, double epsilon, int maxIter, int first,
    const double* __restrict__ part0, double* __restrict__ part1, const TvCtl* __restrict__ c0,
    TvCtl* __restrict__ c1)
{
    const long long end = min(total, (blockIdx.x + 1) * chunk);
    long long t = blockIdx.x * chunk + threadIdx.x;
    TvPix q = {};
    if (t < end) q = tv_load(X, D, P1, P2, R1, R2, t, m, n);
    TvCtl c = *c0;
    if (!first) c = tv_advance(c, part0, gridDim.x, epsilon, maxIter);
    if (c1 != c0 && blockIdx.x == 0 && threadIdx.x == 0) *c1 = c;
    if (c.done) return;  // uniform
    const double tk = c.t, tkp1 = tv_next_t(tk), l8 = 8.0 * lam;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    while (t < end) {
        const bool has1 = q.i < m - 1, has2 = q.j < n - 1;
        const double cc = tv_primal(q.x, q.r1, q.r1u, q.r2, q.r2l, lam);
        const double d = fmax(cc, 0.0);
        const double e = d - q.d, f = cc - d;
        D[t] = d;
        v[0] += e * e;
        v[1] += d * d;
        v[2] += f * f;
        v[3] += cc * cc;
        double p1 = 0.0, p2 = 0.0;
        if (has1)
            p1 = q.r1 + (d - fmax(tv_primal(q.xd, q.r1d, q.r1, q.r2d, q.r2q, lam), 0.0)) / l8;
        if (has2)
            p2 = q.r2 + (d - fmax(tv_primal(q.xr, q.r1r, q.r1q, q.r2r, q.r2, lam), 0.0)) / l8;
        if (iso) {
            // (inside the unit ball the divisor is 1)
            const double s = fmax(__dadd_rn(__dmul_rn(p1, p1), __dmul_rn(p2, p2)), 1.0);
            if (s > 1.0) {
                const double a = sqrt(s);
                p1 = p1 / a;
                p2 = p2 / a;
            }
        } else {
            p1 = fmax(fmin(p1, 1.0), -1.0);
            p2 = fmax(fmin(p2, 1.0), -1.0);
        }
        // (zero on the last row and on the last column)
        P1[t] = p1;
        N1[t] = p1 + (tk - 1.0) * (p1 - q.p1) / tkp1;
        P2[t] = p2;
        N2[t] = p2 + (tk - 1.0) * (p2 - q.p2) / tkp1;
        t += kTvBlock;
        if (t < end) q = tv_load(X, D, P1, P2, R1, R2, t, m, n);
    }
    tv_store_sum4(v, part1, gridDim.x);
}

// The state after an iteration, into c1 and host memory.
__global__ __launch_bounds__(kTvBlock) void k_tv_state(const double* __restrict__ part,
                                                       long long nblk, double epsilon,
                                                       int maxIter, const TvCtl* __restrict__ c0,
                                                       TvCtl* __restrict__ c1, TvCtl* host)
{
    const TvCtl c = tv_advance(*c0, part, nblk, epsilon, maxIter);
    if (threadIdx.x != 0) return;
    *c1 = c;
    *host = c;
}

// Support mask (utils/maskFunc.m): pixels where mask is 0 are zero; NULL keeps all.
__device__ __forceinline__ double tv_masked(const float* mask, long long i, double v)
{
    return (!mask || mask[i] != 0.0f) ? v : 0.0;
}

// TV of FP32 images (utils/tlv.m): iso sum sqrt(P1^2 + P2^2), l1 sum |P1| + |P2|
__global__ __launch_bounds__(kTvBlock) void k_tv_value(const float* __restrict__ X, int m, int n,
                                                       long long total, int iso,
                                                       const float* __restrict__ mask,
                                                       double* __restrict__ part)
{
    const long long t = (long long)blockIdx.x * kTvBlock + threadIdx.x;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (t < total) {
        const int j = (int)(t % n);
        const int i = (int)((t / n) % m);
        const double x = tv_masked(mask, t, X[t]);
        const double p1 = i < m - 1 ? x - tv_masked(mask, t + n, X[t + n]) : 0.0;
        const double p2 = j < n - 1 ? x - tv_masked(mask, t + 1, X[t + 1]) : 0.0;
        v[0] = iso ? sqrt(p1 * p1 + p2 * p2) : fabs(p1) + fabs(p2);
    }
    tv_block_sum4(v, part);
}

// The input image and D = 0, P = proj(Ltrans(0)) = 0, R = P, and the loop state: tk = 1, no
// iteration yet (utils/denoise_bound_mod.m:60-86)
__global__ void k_tv_in(const float* __restrict__ in, double* __restrict__ X,
                        double* __restrict__ D, double* __restrict__ P1, double* __restrict__ P2,
                        double* __restrict__ R1, double* __restrict__ R2, long long n,
                        const float* __restrict__ mask, TvCtl* __restrict__ c)
{
    const long long i = (long long)blockIdx.x * kTvBlock + threadIdx.x;
    if (i < n) {
        X[i] = tv_masked(mask, i, (double)in[i]);
        D[i] = P1[i] = P2[i] = R1[i] = R2[i] = 0.0;
    }
    if (i == 0) *c = TvCtl{1.0, INFINITY, 0, 0, 0, 0};
}

__global__ void k_tv_out(const double* __restrict__ in, float* __restrict__ out, long long n,
                         const float* __restrict__ mask)
{
    const long long i = (long long)blockIdx.x * kTvBlock + threadIdx.x;
    if (i < n) out[i] = (float)tv_masked(mask, i, in[i]);
}

}  // namespace ctprj

using namespace ctprj;

struct ctprj_tv {
    int rows = 0, cols = 0, batch = 0, iso = 1;
    long long n = 0, blocks = 0;
    double *d_X = nullptr, *d_D = nullptr, *d_P1 = nullptr, *d_P2 = nullptr, *d_part = nullptr;
    double *d_R1[2] = {nullptr, nullptr}, *d_R2[2] = {nullptr, nullptr};  // by parity of the iteration
    double* d_sums = nullptr;  // partial sums of an iteration, by its parity
    TvCtl* d_ctl = nullptr;    // the FGP loop's state, by the iteration's parity
    TvCtl* h_ctl = nullptr;    // ... as the host reads it (pinned), by the batch's parity
    hipEvent_t ev[2] = {nullptr, nullptr};  // the batch's state is written
    float* d_mask = nullptr;  // support (NULL: every pixel)
    std::vector<double> part;
    ~ctprj_tv()
    {
        for (void* p : {(void*)d_X, (void*)d_D, (void*)d_P1, (void*)d_P2, (void*)d_R1[0],
                        (void*)d_R1[1], (void*)d_R2[0], (void*)d_R2[1], (void*)d_part,
                        (void*)d_sums, (void*)d_ctl, (void*)d_mask})
            if (p) (void)hipFree(p);
        if (h_ctl) (void)hipHostFree(h_ctl);
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    }
};

long long ctprj::tv_elems(const ctprj_tv* w) { return w ? w->n : 0; }

extern "C" int ctprj_tv_create(int rows, int cols, int batch, int iso, ctprj_tv** out)
{
    if (!out) return fail(CTPRJ_EINVAL, "tv_create: NULL argument");
    *out = nullptr;
    if (rows < 2 || cols < 2 || batch < 1)
        return fail(CTPRJ_EINVAL, "tv_create: bad sizes (%d x %d x %d)", rows, cols, batch);
    const long long n = (long long)rows * cols * batch;
    if (n >= (1LL << 31)) return fail(CTPRJ_EINVAL, "tv_create: %lld elements is too many", n);
    ctprj_tv* w = new (std::nothrow) ctprj_tv();
    if (!w) return fail(CTPRJ_ENOMEM, "host allocation");
    w->rows = rows;
    w->cols = cols;
    w->batch = batch;
    w->iso = iso ? 1 : 0;
    w->n = n;
    w->blocks = (n + kTvBlock - 1) / kTvBlock;
    w->part.assign((size_t)4 * w->blocks, 0.0);
    hipError_t e = hipSuccess;
    for (double** p : {&w->d_X, &w->d_D, &w->d_P1, &w->d_P2, &w->d_R1[0], &w->d_R1[1], &w->d_R2[0],
                       &w->d_R2[1]})
        if (e == hipSuccess) e = hipMalloc((void**)p, sizeof(double) * (size_t)n);
    if (e == hipSuccess) e = hipMalloc((void**)&w->d_part, sizeof(double) * 4 * (size_t)w->blocks);
    if (e == hipSuccess) e = hipMalloc((void**)&w->d_sums, sizeof(double) * 8 * kTvGroups);
    if (e == hipSuccess) e = hipMalloc((void**)&w->d_ctl, 2 * sizeof(TvCtl));
    if (e == hipSuccess) e = hipHostMalloc((void**)&w->h_ctl, 2 * sizeof(TvCtl), hipHostMallocDefault);
    for (hipEvent_t& v : w->ev)
        if (e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
    if (e != hipSuccess) {
        delete w;
        return fail(CTPRJ_ENOMEM, "tv workspace: %s", hipGetErrorString(e));
    }
    *out = w;
    return 0;
}

extern "C" int ctprj_tv_set_mask(ctprj_tv* w, const float* d_mask)
{
    if (!w) return fail(CTPRJ_EINVAL, "tv_set_mask: NULL context");
    if (w->d_mask) (void)hipFree(w->d_mask);
    w->d_mask = nullptr;
    if (!d_mask) return 0;
    const size_t bytes = sizeof(float) * (size_t)w->n;
    hipError_t e = hipMalloc((void**)&w->d_mask, bytes);
    if (e == hipSuccess) e = hipMemcpy(w->d_mask, d_mask, bytes, hipMemcpyDeviceToDevice);
    return e == hipSuccess ? 0 : hip_fail(e, "tv mask");
}

extern "C" int ctprj_tv_destroy(ctprj_tv* w)
{
    delete w;
    return 0;
}

long long ctprj::tv_value_parts(const ctprj_tv* w) { return 4 * w->blocks; }

int ctprj::tv_value_queue(ctprj_tv* w, const float* d_x, double* d_part, hipStream_t st)
{
    hipLaunchKernelGGL(k_tv_value, dim3((unsigned)w->blocks), dim3(kTvBlock), 0, st, d_x, w->rows,
                       w->cols, w->n, w->iso, w->d_mask, d_part);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : hip_fail(e, "tv value launch");
}

double ctprj::tv_value_total(const ctprj_tv* w, const double* part)
{
    double s = 0.0;
    for (long long b = 0; b < w->blocks; ++b) s += part[4 * b];
    return s;
}

extern "C" int ctprj_tv_value(ctprj_tv* w, const float* d_x, double* tv, void* stream)
{
    if (!w || !d_x || !tv) return fail(CTPRJ_EINVAL, "tv_value: NULL argument");
    hipStream_t st = (hipStream_t)stream;
    int rc = tv_value_queue(w, d_x, w->d_part, st);
    if (rc) return rc;
    hipError_t e = hipMemcpyAsync(w->part.data(), w->d_part, sizeof(double) * 4 * w->blocks,
                                  hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return hip_fail(e, "tv value");
    *tv = tv_value_total(w, w->part.data());
    return 0;
}

extern "C" int ctprj_tv_denoise(ctprj_tv* w, const float* d_x, double lambda, double epsilon,
                                int maxIter, float* d_out, int* iterations, void* stream)
{
    if (!w || !d_x || !d_out) return fail(CTPRJ_EINVAL, "tv_denoise: NULL argument");
    if (!(lambda > 0.0) || !std::isfinite(lambda) || !std::isfinite(epsilon) || maxIter < 0)
        return fail(CTPRJ_EINVAL, "tv_denoise: lambda must be > 0, epsilon finite, maxIter >= 0");
    hipStream_t st = (hipStream_t)stream;
    hipStreamCaptureStatus cap;
    hipError_t ce = hipStreamIsCapturing(st, &cap);
    if (ce == hipSuccess && cap != hipStreamCaptureStatusNone) ce = hipErrorStreamCaptureUnsupported;
    if (ce != hipSuccess) return hip_fail(ce, "tv_denoise");  // the host reads the state
    const long long n = w->n;
    const unsigned g = (unsigned)w->blocks;
    // a group's pixels: a multiple of kTvBlock, kTvGroups groups at most
    const long long chunk = (w->blocks + kTvGroups - 1) / kTvGroups * kTvBlock;
    const unsigned groups = (unsigned)((n + chunk - 1) / chunk);
    TvCtl* C = w->d_ctl;
    hipLaunchKernelGGL(k_tv_in, dim3(g), dim3(kTvBlock), 0, st, d_x, w->d_X, w->d_D, w->d_P1,
                       w->d_P2, w->d_R1[0], w->d_R2[0], n, w->d_mask, C);
    // Iterations in batches of kTvBatch.  The host waits for a batch's state only when the
    // next batch (or the output) is queued: with a wait between them the GPU stood still for
    // about 30 us a batch, more than the launches of a batch past the stop take (8 x 2.5 us).
    // 24 iterations at 512^2: 32 us less.
    constexpr int kTvBatch = 8;
    int it = 0, batches = 0;
    auto queue = [&]() -> int {
        const int stop = it + std::min(kTvBatch, maxIter - it);
        for (const int begin = it; it < stop; ++it) {
            const int a = it & 1, first = it == begin;
            hipLaunchKernelGGL(k_tv_iter, dim3(groups), dim3(kTvBlock), 0, st, w->d_X, w->d_D,
                               w->d_P1, w->d_P2, w->d_R1[a], w->d_R2[a], w->d_R1[1 - a],
                               w->d_R2[1 - a], w->rows, w->cols, n, chunk, lambda, w->iso,
                               epsilon, maxIter, first, w->d_sums + 4 * kTvGroups * (1 - a),
                               w->d_sums + 4 * kTvGroups * a, first ? C + a : C + 1 - a, C + a);
        }
        const int a = (it - 1) & 1, slot = batches++ & 1;
        hipLaunchKernelGGL(k_tv_state, dim3(1), dim3(kTvBlock), 0, st,
                           w->d_sums + 4 * kTvGroups * a, (long long)groups, epsilon, maxIter,
                           C + a, C + 1 - a, w->h_ctl + slot);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(w->ev[slot], st);
        return e == hipSuccess ? 0 : hip_fail(e, "tv iteration launch");
    };
    auto output = [&]() -> int {
        hipLaunchKernelGGL(k_tv_out, dim3(g), dim3(kTvBlock), 0, st, w->d_D, d_out, n, w->d_mask);
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? 0 : hip_fail(e, "tv output");
    };
    int rc = 0, itr = 0;
    bool done = maxIter <= 0, out = false;
    if (!done && (rc = queue())) return rc;
    while (!done) {
        const int seen = batches - 1;
        out = it >= maxIter;
        if ((rc = out ? output() : queue())) return rc;
        const hipError_t e = hipEventSynchronize(w->ev[seen & 1]);
        if (e != hipSuccess) return hip_fail(e, "tv state");
        done = w->h_ctl[seen & 1].done != 0;
        itr = w->h_ctl[seen & 1].i;
        if (!done && out) return fail(CTPRJ_EHIP, "tv_denoise: the loop state did not stop");
    }
    if (iterations) *iterations = itr;
    return out ? 0 : output();
}
