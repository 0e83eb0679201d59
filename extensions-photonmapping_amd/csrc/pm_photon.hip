// pm_photon.hip -- photon emission and diffuse continuation rays for photon
// paths (the caller side of the trace: emission -> trace -> bounce -> trace
// ...).
//
// The reference has no photon tracer despite its name; its only secondary
// rays are the reflection continuations of the shading loop
// (Raytracer.cu:219-256, ColorKernels.h:43-78).  Emission samples the light
// triangles by area (emit_kernel below).  The bounce makes one
// cosine-weighted diffuse continuation per surviving hit:
//   origin    = o + t d + offset * n   (n: geometric normal facing the ray)
//   direction = cosine-weighted about n (Malley: uniform disk, lifted)
// with PCG32 (O'Neill 2014) stream (seed, purpose 6, source ray index), and
// a stable compaction (survivor counts per wave) so the output order is the
// input order.
#include "pm_device.h"
#include "pm_internal.h"

namespace pmkd {

namespace {

constexpr int TB = 256;
constexpr int BW = TB / 64;
static_assert(BW == 4, "a block's wave counts are one int4");

// The bounce is two launches.  Each wave of the grid owns `span` consecutive
// rays: alive_kernel counts its survivors, bounce_kernel adds up the counts
// before its own (at most BOUNCE_BLOCKS records, the most the device holds at
// once, so this stays a few loads a thread at any n) and writes its survivors
// from there on.  It is bound by its bytes: hits twice, a survivor's ray,
// triangle and 36 bytes out, the triangles' gathers costing whole lines.  A flag
// and an offset per ray, scanned by kernels of their own, were 32 bytes a ray
// more and four launches: hits spread over 1,000,000 triangles, 0.3M / 2.4M / 4M
// / 16M rays 46 / 177 / 276 / 984 -> 42 / 163 / 250 / 927 us.
constexpr int BOUNCE_BLOCKS = 2048;

// hits[i]'s id where ray i survives, -1 where not
__device__ __forceinline__ int survivor(int id, long long i, int n, int absorb_from) {
    return i < n && id >= 0 && id < absorb_from ? id : -1;
}

__global__ __launch_bounds__(TB) void alive_kernel(const pm_hit *__restrict__ hits, int n, int absorb_from,
                                                   int span, int *__restrict__ counts) {
    const int lane = threadIdx.x & 63, wave = (blockIdx.x * TB + threadIdx.x) >> 6;
    const long long first = (long long)wave * span + lane;
    int c = 0;
#pragma unroll 4
    for (int k = 0; k < span; k += 64) {
        const long long i = first + k;
        const int id = hits[i < n ? i : n - 1].id;
        c += __popcll(__ballot(survivor(id, i, n, absorb_from) >= 0));
    }
    if (lane == 0) counts[wave] = c;
}

__global__ __launch_bounds__(TB) void bounce_kernel(
    const float4 *__restrict__ P0, const float4 *__restrict__ P1, const float4 *__restrict__ P2,
    const float4 *__restrict__ org, const float4 *__restrict__ dir, const pm_hit *__restrict__ hits,
    int n, int absorb_from, int span, const int4 *__restrict__ counts, int *__restrict__ total,
    int *__restrict__ out_count, unsigned long long seed, float offset, float4 *__restrict__ out_org,
    float4 *__restrict__ out_dir, int *__restrict__ out_src) {
    __shared__ int part[BW];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const long long first = (long long)(blockIdx.x * BW + w) * span + lane;
    pm_hit next = hits[first < n ? first : n - 1];
    // survivors before this wave's rays
    const int4 own = counts[blockIdx.x];
    int before = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += TB) {
        const int4 c = counts[b];
        before += c.x + c.y + c.z + c.w;
    }
    for (int m = 32; m; m >>= 1) before += __shfl_xor(before, m);
    if (lane == 0) part[w] = before;
    __syncthreads();
    int j0 = part[0] + part[1] + part[2] + part[3];
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        const int sum = j0 + own.x + own.y + own.z + own.w;
        *total = sum;
        if (out_count) *out_count = sum;
    }
    j0 += (w > 0 ? own.x : 0) + (w > 1 ? own.y : 0) + (w > 2 ? own.z : 0);
    const unsigned long long below = lane ? ~0ull >> (64 - lane) : 0ull;
    for (int k = 0; k < span; k += 64) {
        const long long i = first + k;
        const pm_hit h = next;
        const long long in = i + 64;
        if (k + 64 < span) next = hits[in < n ? in : n - 1];
        const bool alive = survivor(h.id, i, n, absorb_from) >= 0;
        const unsigned long long mask = __ballot(alive);
        const int j = j0 + __popcll(mask & below);
        j0 += __popcll(mask);
        if (!alive) continue;
        const f3 v0 = mk3(P0[h.id]), v1 = mk3(P1[h.id]), v2 = mk3(P2[h.id]);
        f3 nrm = normalize3(cross3(sub3(v1, v0), sub3(v2, v0)));
        const f3 o = mk3(org[i]), d = mk3(dir[i]);
        if (dot3(nrm, d) > 0.0f) nrm = {-nrm.x, -nrm.y, -nrm.z};
        const f3 pos = {o.x + h.t * d.x + offset * nrm.x, o.y + h.t * d.y + offset * nrm.y,
                        o.z + h.t * d.z + offset * nrm.z};
        Pcg rng(seed, (6ull << 40) | (unsigned long long)i);
        const float u1 = rng.uniform(), u2 = rng.uniform();
        const f3 nd = cosine_dir(nrm, u1, u2);
        out_org[j] = make_float4(pos.x, pos.y, pos.z, 1.0f);
        out_dir[j] = make_float4(nd.x, nd.y, nd.z, 0.0f);
        if (out_src) out_src[j] = (int)i;
    }
}

__global__ void clear_count_kernel(int *out) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *out = 0;
}

// Emission: the running FP32 sum of the light triangles' areas
// (tri_area, ascending), one thread: cdf[k] = area_0 + ... + area_k.
__global__ void light_cdf_kernel(const float4 *__restrict__ L0, const float4 *__restrict__ L1,
                                 const float4 *__restrict__ L2, int m, float *__restrict__ cdf) {
    if (threadIdx.x | blockIdx.x) return;
    float acc = 0.0f;
    for (int k = 0; k < m; ++k) {
        acc += tri_area(mk3(L0[k]), mk3(L1[k]), mk3(L2[k]));
        cdf[k] = acc;
    }
}

// One photon per thread, PCG32 stream (seed, purpose 5, photon index):
//   u0 picks light k, the first with u0 * total < cdf[k] (the last if none);
//   (u1, u2) a uniform point of that triangle,
//     p = (1 - s) v0 + s (1 - u2) v1 + s u2 v2 with s = sqrt(u1);
//   (u3, u4) a cosine-weighted direction about n = normalize(e1 x e2);
// the origin is p + offset * n.
__global__ __launch_bounds__(TB) void emit_kernel(const float4 *__restrict__ L0, const float4 *__restrict__ L1,
                                                  const float4 *__restrict__ L2, int m,
                                                  const float *__restrict__ cdf, int n, unsigned long long seed,
                                                  float offset, float4 *__restrict__ out_org,
                                                  float4 *__restrict__ out_dir) {
    const int i = blockIdx.x * TB + threadIdx.x;
    if (i >= n) return;
    Pcg rng(seed, (5ull << 40) | (unsigned long long)i);
    const float u0 = rng.uniform(), u1 = rng.uniform(), u2 = rng.uniform();
    const float u3 = rng.uniform(), u4 = rng.uniform();
    const float target = u0 * cdf[m - 1];
    int lo = 0, hi = m - 1;            // first k with target < cdf[k]; m - 1 if none
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (target < cdf[mid]) hi = mid; else lo = mid + 1;
    }
    const f3 v0 = mk3(L0[lo]), v1 = mk3(L1[lo]), v2 = mk3(L2[lo]);
    const float s = sqrtf(u1);
    const float a = 1.0f - s, b = s * (1.0f - u2), c = s * u2;
    const f3 nrm = normalize3(cross3(sub3(v1, v0), sub3(v2, v0)));
    const f3 p = {a * v0.x + b * v1.x + c * v2.x, a * v0.y + b * v1.y + c * v2.y, a * v0.z + b * v1.z + c * v2.z};
    const f3 d = cosine_dir(nrm, u3, u4);
    out_org[i] = make_float4(p.x + offset * nrm.x, p.y + offset * nrm.y, p.z + offset * nrm.z, 1.0f);
    out_dir[i] = make_float4(d.x, d.y, d.z, 0.0f);
}

}  // namespace

void photon_emit(pm_ctx *ctx, const float4 *l0, const float4 *l1, const float4 *l2, int m, int n,
                 unsigned long long seed, float offset, float4 *out_org, float4 *out_dir, hipStream_t s) {
    if (n == 0) return;
    BuildScratch &sc = ctx->scratch;
    sc.light_cdf.reserve((size_t)m, s);
    light_cdf_kernel<<<1, 64, 0, s>>>(l0, l1, l2, m, sc.light_cdf.ptr);
    PM_LAUNCH_CHECK();
    emit_kernel<<<(n + TB - 1) / TB, TB, 0, s>>>(l0, l1, l2, m, sc.light_cdf.ptr, n, seed, offset, out_org,
                                                 out_dir);
    PM_LAUNCH_CHECK();
}

int photon_bounce(pm_ctx *ctx, const float4 *org, const float4 *dir, const pm_hit *hits, int n,
                  int absorb_from, unsigned long long seed, float offset, float4 *out_org,
                  float4 *out_dir, int *out_src, int *out_count, hipStream_t s) {
    if (n == 0) {
        if (out_count) {
            clear_count_kernel<<<1, 64, 0, s>>>(out_count);
            PM_LAUNCH_CHECK();
        }
        PM_HIP(hipStreamSynchronize(s));
        return 0;
    }
    BuildScratch &sc = ctx->scratch;
    const int iters = (int)(((long long)n + (long long)BOUNCE_BLOCKS * TB - 1) / ((long long)BOUNCE_BLOCKS * TB));
    const int span = 64 * iters;
    const int blocks = (int)(((long long)n + (long long)BW * span - 1) / ((long long)BW * span));
    sc.bounce_counts.reserve((size_t)BW * blocks + 1, s);
    int *const counts = sc.bounce_counts.ptr, *const total = counts + BW * blocks;
    alive_kernel<<<blocks, TB, 0, s>>>(hits, n, absorb_from, span, counts);
    PM_LAUNCH_CHECK();
    bounce_kernel<<<blocks, TB, 0, s>>>(ctx->p0, ctx->p1, ctx->p2, org, dir, hits, n, absorb_from, span,
                                        reinterpret_cast<const int4 *>(counts), total, out_count, seed, offset,
                                        out_org, out_dir, out_src);
    PM_LAUNCH_CHECK();
    sc.host.ensure(8);
    PM_HIP(hipMemcpyAsync(sc.host.ptr, total, sizeof(int), hipMemcpyDeviceToHost, s));
    PM_HIP(hipStreamSynchronize(s));
    return sc.host.ptr[0];
}

}  // namespace pmkd
