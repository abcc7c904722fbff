// Mip-Splatting's 3D filter size per Gaussian (metal_gauss/mipfilter.py:29-73).
//
//   dist  = min over the views that see the Gaussian of its camera depth
//   size  = dist / focal * sqrt(0.2),  focal = max over views of (fx, fy)
//
// A view sees a Gaussian when z > near and the projected centre lies inside
// the frame widened by `margin` on every side. A Gaussian no view sees gets
// the largest distance any seen Gaussian got; if none is seen, every distance
// is 1.
//
// Three launches: the distances over all views (a workgroup takes a run of
// Gaussians, its waves a share of the views each), the seen maximum (integer
// atomics on an order-preserving encoding of the float, one per workgroup of
// a small grid), and a finishing pass that fills the unseen and scales. The
// O(N V) pass reads each mean once; vector issue bounds it.
#include "mg_common.h"

namespace mg {

constexpr int kMipThreads = 256;
constexpr int kViewChunk = 256;
// Per view: R (9, row-major), t (3), fx, fy, cx, cy, then the frame with its
// margin as four bounds u_lo, u_hi, v_lo, v_hi (-margin W, (1 + margin) W,
// -margin H, (1 + margin) H), formed on the host in double and rounded once,
// as the reference's comparisons against Python floats round them.
constexpr int kViewFloats = 20;

// Float -> int32 with the same order (negative floats flipped).
__device__ __forceinline__ int32_t f32_order(float f) {
    const int32_t i = __float_as_int(f);
    return i ^ ((i >> 31) & 0x7fffffff);
}
__device__ __forceinline__ float f32_unorder(int32_t i) {
    return __int_as_float(i ^ ((i >> 31) & 0x7fffffff));
}

constexpr int32_t kNoneSeen = INT32_MIN;

// Whether view P (kViewFloats floats) sees the point whose camera depth is z:
// the reference's expressions, two IEEE divisions.
__device__ __forceinline__ bool mip_inview(const float *__restrict__ P, float mx, float my,
                                           float mz, float z) {
    const float px = P[0] * mx + P[1] * my + P[2] * mz + P[9];
    const float py = P[3] * mx + P[4] * my + P[5] * mz + P[10];
    const float zc = fmaxf(z, 1e-6f);
    const float u = P[12] * px / zc + P[14];
    const float w = P[13] * py / zc + P[15];
    return (u > P[16]) && (u < P[17]) && (w > P[18]) && (w < P[19]);
}

// A view as the walk uses it. With c the frame's centre and h its half width
// (margin included), u lies inside the frame exactly where
// |fx px + (cx - c) z| < h z, and fx px + (cx - c) z is one affine form of the
// point: three such forms (z, ex, ey) and no division decide a pair, unless
// max(|ex| - hx z, |ey| - hy z) lies within `slack` of 0, where rounding could
// decide otherwise than mip_inview; those pairs (about one in 10^5) ask
// mip_inview. slack = e1 |m|_1 + e2 is 64 units of rounding of every term that
// enters either expression (their own errors add up to under 20), infinite
// where a term is not finite or z may lie below the depth clamp.
struct __align__(16) MipView {
    float z[4], ex[4], ey[4];
    float hx, hy, e1, e2;
};

__device__ __forceinline__ MipView mip_view(const float *__restrict__ P, float near_p) {
    MipView v;
    const double fx = P[12], fy = P[13];
    const double ox = P[14] - 0.5 * ((double)P[16] + P[17]);
    const double oy = P[15] - 0.5 * ((double)P[18] + P[19]);
    double sx = 0.0, sy = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float r0 = k < 3 ? P[k] : P[9], r1 = k < 3 ? P[3 + k] : P[10];
        const float r2 = k < 3 ? P[6 + k] : P[11];
        v.z[k] = r2;
        v.ex[k] = (float)(fx * r0 + ox * r2);
        v.ey[k] = (float)(fy * r1 + oy * r2);
        const double ax = fabs(fx * r0) + fabs(ox * r2), ay = fabs(fy * r1) + fabs(oy * r2);
        if (k < 3) {
            sx += ax;
            sy += ay;
        } else {
            const double bound = fabs((double)P[14]) + fabs((double)P[15]) +
                                 fabs((double)P[16]) + fabs((double)P[17]) +
                                 fabs((double)P[18]) + fabs((double)P[19]);
            constexpr double kUnits = 64.0 / 16777216.0;
            const double r2max = fmax(fmax(fabs((double)P[6]), fabs((double)P[7])),
                                      fabs((double)P[8]));
            const float e1 = (float)(kUnits * (sx + sy + bound * r2max));
            const float e2 = (float)(kUnits * (ax + ay + bound * fabs((double)r2)));
            const bool plain = near_p >= 1e-6f && isfinite(e1) && isfinite(e2);
            v.e1 = plain ? e1 : 0.0f;
            v.e2 = plain ? e2 : __builtin_inff();
        }
    }
    v.hx = (float)(0.5 * ((double)P[17] - P[16]));
    v.hy = (float)(0.5 * ((double)P[19] - P[18]));
    return v;
}

// One workgroup per 64 * kPer Gaussians, lane l holding Gaussians l, 64 + l,
// ... of the run; wave w takes views w, w + 4, ... and the waves' minima meet
// in LDS. Splitting the views over the waves rather than the Gaussians keeps
// every CU busy down to some 10^4 Gaussians; kPer Gaussians a lane share a
// view's four LDS reads. A pair costs about 20 vector instructions (62 with
// the divisions); with the atomics of the old pass gone too, 1M Gaussians x
// 100 views take 63 us (256 before).
constexpr int kMipWaves = kMipThreads / 64;

template <int kPer>
__global__ __launch_bounds__(kMipThreads) void mip_dist_kernel(
    const float *__restrict__ means, int64_t N, const float *__restrict__ views, int32_t V,
    float near_p, float *__restrict__ dist, int32_t *seen_max) {
    __shared__ MipView s_v[kViewChunk];
    __shared__ float s_d[kMipWaves][64 * kPer];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (blockIdx.x == 0 && threadIdx.x == 0) *seen_max = kNoneSeen;
    const int64_t g0 = (int64_t)blockIdx.x * (64 * kPer) + lane;
    float mx[kPer], my[kPer], mz[kPer], m1[kPer], d[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int64_t g = min(g0 + 64 * i, N - 1);
        mx[i] = means[3 * g];
        my[i] = means[3 * g + 1];
        mz[i] = means[3 * g + 2];
        m1[i] = fabsf(mx[i]) + fabsf(my[i]) + fabsf(mz[i]);
        d[i] = __builtin_inff();
    }
    for (int v0 = 0; v0 < V; v0 += kViewChunk) {
        const int nv = min(kViewChunk, V - v0);
        __syncthreads();
        if ((int)threadIdx.x < nv)
            s_v[threadIdx.x] = mip_view(views + (int64_t)(v0 + threadIdx.x) * kViewFloats, near_p);
        __syncthreads();
        for (int k = wave; k < nv; k += kMipWaves) {
            const MipView v = s_v[k];
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const float z = v.z[0] * mx[i] + v.z[1] * my[i] + v.z[2] * mz[i] + v.z[3];
                const float ex = fmaf(v.ex[0], mx[i],
                                      fmaf(v.ex[1], my[i], fmaf(v.ex[2], mz[i], v.ex[3])));
                const float ey = fmaf(v.ey[0], mx[i],
                                      fmaf(v.ey[1], my[i], fmaf(v.ey[2], mz[i], v.ey[3])));
                const float out = fmaxf(fmaf(-v.hx, z, fabsf(ex)), fmaf(-v.hy, z, fabsf(ey)));
                const float slack = fmaf(v.e1, m1[i], v.e2);
                const bool nearer = z > near_p && z < d[i];
                bool in = out < -slack;
                // Neither certainly inside nor certainly outside (NaN too).
                const bool unsure = nearer && !in && !(out > slack);
                if (ballot(unsure) != 0)
                    in = unsure ? mip_inview(views + (int64_t)(v0 + k) * kViewFloats, mx[i], my[i],
                                             mz[i], z)
                                : in;
                d[i] = nearer && in ? z : d[i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < kPer; ++i) s_d[wave][64 * i + lane] = d[i];
    __syncthreads();
    for (int j = threadIdx.x; j < 64 * kPer; j += kMipThreads) {
        float m = s_d[0][j];
#pragma unroll
        for (int w = 1; w < kMipWaves; ++w) m = fminf(m, s_d[w][j]);
        const int64_t g = (int64_t)blockIdx.x * (64 * kPer) + j;
        if (g < N) dist[g] = m;
    }
}

// The largest seen distance. One same-address atomic costs about 12 ns at the
// memory side whoever issues it, so a small grid issues one per workgroup
// (one per wave of the distance pass were 188 us at 1M Gaussians).
constexpr int kMaxBlocks = 128;

__global__ __launch_bounds__(kMipThreads) void mip_max_kernel(const float *__restrict__ dist,
                                                              int64_t N, int32_t *seen_max) {
    __shared__ int32_t s_m[kMipWaves];
    int32_t m = kNoneSeen;
    for (int64_t g = (int64_t)blockIdx.x * kMipThreads + threadIdx.x; g < N;
         g += (int64_t)gridDim.x * kMipThreads) {
        const float d = dist[g];
        m = max(m, d != __builtin_inff() ? f32_order(d) : kNoneSeen);
    }
    for (int o = 32; o >= 1; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kMipWaves; ++w) m = max(m, s_m[w]);
        if (m != kNoneSeen) atomicMax(seen_max, m);
    }
}

__global__ __launch_bounds__(kMipThreads) void mip_finish_kernel(float *dist, int64_t N,
                                                                 const int32_t *seen_max,
                                                                 float focal) {
    const int64_t g = (int64_t)blockIdx.x * kMipThreads + threadIdx.x;
    if (g >= N) return;
    const int32_t m = *seen_max;
    float d = dist[g];
    if (m == kNoneSeen) d = 1.0f;
    else if (d == __builtin_inff()) d = f32_unorder(m);
    // (dist / focal) * sqrt(0.2), rounded as mipfilter.py:73 rounds it.
    dist[g] = (d / focal) * 0.4472135954999579f;
}

}  // namespace mg

using namespace mg;

extern "C" {

int32_t mg_compute_3d_filter(int64_t N, const float *means, int32_t n_views, const float *views,
                             float focal, float near_plane, float *filter_3d, int32_t *scratch,
                             mg_stream_t stream) {
    MG_REQUIRE(N >= 0, "mg_compute_3d_filter: N = %lld", (long long)N);
    MG_REQUIRE(n_views >= 0, "mg_compute_3d_filter: %d views", n_views);
    if (N == 0) return MG_OK;
    MG_REQUIRE(means && filter_3d && scratch, "mg_compute_3d_filter: null pointer");
    MG_REQUIRE(n_views == 0 || views, "mg_compute_3d_filter: null views");
    // mipfilter.py:71-72: a non-positive focal length falls back to 1.
    const float f = focal > 0.0f ? focal : 1.0f;
    hipStream_t s = as_stream(stream);
    const unsigned blocks = (unsigned)ceil_div(N, kMipThreads);
    TimedScope ts("compute_3d_filter", s);
    // Four Gaussians a lane where that still leaves about three workgroups
    // per CU, one below.
    if (N >= 4 * 64 * 768)
        mip_dist_kernel<4><<<(unsigned)ceil_div(N, 256), kMipThreads, 0, s>>>(
            means, N, views, n_views, near_plane, filter_3d, scratch);
    else
        mip_dist_kernel<1><<<(unsigned)ceil_div(N, 64), kMipThreads, 0, s>>>(
            means, N, views, n_views, near_plane, filter_3d, scratch);
    MG_LAUNCHED("mip_dist_kernel");
    mip_max_kernel<<<(unsigned)min(ceil_div(N, kMipThreads), (int64_t)kMaxBlocks), kMipThreads, 0,
                     s>>>(filter_3d, N, scratch);
    MG_LAUNCHED("mip_max_kernel");
    mip_finish_kernel<<<blocks, kMipThreads, 0, s>>>(filter_3d, N, scratch, f);
    MG_LAUNCHED("mip_finish_kernel");
    return MG_OK;
}

}  // extern "C"
