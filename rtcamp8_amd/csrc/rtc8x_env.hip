// rtc8x_env.hip -- environment importance sampling set-up: the hierarchical importance map
// (computeFirstMipOfEnvIBLImportanceMap / computeMipOfImportanceMap, renderer/gpu_kernels/
// compute_light_probs.cu:161-211, driven as renderer/renderer_scene.h:990-1069) and the two-level
// alias tables over texels (built in FP64 on the device, Vose's method).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "rtc8x_common.hpp"
#include "rtc8x_device.hpp"

namespace rtc8x {
namespace dev {

// mip 0 = luminance * (pi/2) * sin(pi (y + 1/2) / H) inside the image, 0 in the power-of-two padding.
__global__ void env_mip0_kernel(const float* __restrict__ texels, uint32_t w, uint32_t h, uint32_t dim_x, uint32_t dim_y,
                                float* __restrict__ mip0)
{
    uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= dim_x || y >= dim_y) return;
    float importance = 0.0f;
    if (x < w && y < h) {
        const float4 t = *reinterpret_cast<const float4*>(texels + ((size_t)y * w + x) * 4);
        float correction = RTC8X_PI_F / 2.0f * rtc8x_sinf(RTC8X_PI_F * ((float)y + 0.5f) / (float)h);
        importance = luminance(RGB{t.x, t.y, t.z}) * correction;
    }
    mip0[(size_t)y * dim_x + x] = importance;
}

// 2x2 box reduction (sum of ul, ur, ll, lr, then * 1/4); the 1x1 top level sets the integral.
__global__ void env_mip_kernel(const float* __restrict__ src, uint32_t sdx, uint32_t sdy, float* __restrict__ dst,
                               uint32_t ddx, uint32_t ddy, int top, float top_scale, float* __restrict__ integral)
{
    uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t y = blockIdx.y * blockDim.y + threadIdx.y;
    uint32_t ulx = 2 * x, uly = 2 * y;
    float sum = 0.0f;
    sum += (ulx < sdx && uly < sdy) ? src[(size_t)uly * sdx + ulx] : 0.0f;
    sum += (ulx + 1 < sdx && uly < sdy) ? src[(size_t)uly * sdx + ulx + 1] : 0.0f;
    sum += (ulx < sdx && uly + 1 < sdy) ? src[(size_t)(uly + 1) * sdx + ulx] : 0.0f;
    sum += (ulx + 1 < sdx && uly + 1 < sdy) ? src[(size_t)(uly + 1) * sdx + ulx + 1] : 0.0f;
    if (x < ddx && y < ddy) {
        sum *= 0.25f;
        dst[(size_t)y * ddx + x] = sum;
        if (top) *integral = sum * top_scale;
    }
}

__device__ __forceinline__ double lane_value(double v, uint32_t lane)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, (int)lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), (int)lane);
    return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}

// The sum of the n numbers m[0..n) in order: every lane adds the same ones, taken 64 to an LDS read.
template <typename T>
__device__ __forceinline__ double ordered_sum(const T* m, uint32_t n)
{
    const uint32_t lane = threadIdx.x & 63u;
    double sum = 0.0;
    for (uint32_t x0 = 0; x0 < n; x0 += 64) {
        const double v = x0 + lane < n ? (double)m[x0 + lane] : 0.0;
        const uint32_t e = min(64u, n - x0);
        for (uint32_t k = 0; k < e; ++k) sum += lane_value(v, k);
    }
    return sum;
}

// Vose's alias method in FP64 over the n weights in LDS (n <= 16,384), one wavefront per table;
// prob_to_pick_first stored as float.  The method keeps the entries below and above the mean on two stacks, in
// index order, and pairs their tops: the large one fills the small one up, and once it falls below the mean
// itself it is the next small one.  So the small entries come in descending order, with a spent large one in
// between, and the large ones in descending order: two streams, which the wavefront reads from `stack` (the
// small ones from its start, the large ones from its end) 64 at a time, one per lane, with their weights.  The
// pairing itself is a serial chain of two FP64 additions per entry, the same in every lane; an entry's result
// stays in its lane until the next 64 are read.
//
// On the host the 1,601 tables of a 3200 x 1600 sky, with the copies of its weights and tables, took 52 ms of
// an animated sky's 55 ms keyframe; here the chains run side by side, in 0.7 ms.
template <typename T>
__device__ __forceinline__ void alias_table(const T* m, uint16_t* stack, uint32_t n, double total,
                                            rtc8x_alias_entry* __restrict__ out)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t before = (1ull << lane) - 1ull;
    auto weight = [&](uint32_t i) -> double { return total > 0.0 ? (double)m[i] * (double)n / total : 1.0; };
    uint32_t ns = 0, nl = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
        const uint32_t i = i0 + lane;
        const bool is_small = i < n && weight(i) < 1.0, is_large = i < n && !is_small;
        const uint64_t bs = __ballot(is_small), bl = __ballot(is_large);
        if (is_small) stack[ns + (uint32_t)__popcll(bs & before)] = (uint16_t)i;
        if (is_large) stack[n - 1u - (nl + (uint32_t)__popcll(bl & before))] = (uint16_t)i;
        ns += (uint32_t)__popcll(bs);
        nl += (uint32_t)__popcll(bl);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // a stream's 64 entries: this lane's index and weight, and its result (what is never paired picks itself)
    struct Stream {
        uint32_t i, second;
        double w;
        float first;
        bool have;
    };
    auto flush = [&](const Stream& t) {
        if (t.have) out[t.i] = rtc8x_alias_entry{t.second, t.first};
    };
    auto read = [&](Stream& t, uint32_t left, bool large) {  // `left` entries of the stream are not yet read
        t.have = lane < left;
        t.i = t.have ? stack[large ? n - left + lane : left - 1u - lane] : 0u;
        t.w = t.have ? weight(t.i) : 1.0;
        t.second = t.i;
        t.first = 1.0f;
    };
    Stream s, l;
    uint32_t ks = 0, kl = 0;
    read(s, ns, false);
    read(l, nl, true);
    if (nl > 0) {
        uint32_t li = (uint32_t)__builtin_amdgcn_readlane((int)l.i, 0);
        double wl = lane_value(l.w, 0);
        bool more = true;
        while (more && ns > 0) {
            if (lane == ks) {
                s.second = li;
                s.first = (float)s.w;
            }
            wl = (wl + lane_value(s.w, ks)) - 1.0;
            ks++;
            ns--;
            if (ks == 64) {
                flush(s);
                read(s, ns, false);
                ks = 0;
            }
            while (wl < 1.0) {
                // the large entry is spent: the next one fills it up
                const double ws = wl;
                nl--;
                if (nl == 0) {
                    more = false;
                    break;
                }
                const uint32_t kn = kl + 1u;
                if (kn < 64u) {
                    li = (uint32_t)__builtin_amdgcn_readlane((int)l.i, (int)kn);
                    wl = lane_value(l.w, kn);
                    if (lane == kl) {
                        l.second = li;
                        l.first = (float)ws;
                    }
                    kl = kn;
                } else {
                    Stream t;
                    read(t, nl, true);
                    li = (uint32_t)__builtin_amdgcn_readlane((int)t.i, 0);
                    wl = lane_value(t.w, 0);
                    if (lane == 63u) {
                        l.second = li;
                        l.first = (float)ws;
                    }
                    flush(l);
                    l = t;
                    kl = 0;
                }
                wl = (wl + ws) - 1.0;
            }
        }
    }
    // the rest of both streams: this lane's entries, then those not yet read
    flush(s);
    flush(l);
    const uint32_t small_read = ks < ns + ks ? min(64u - ks, ns) : 0u;
    for (uint32_t k = lane; k < ns - small_read; k += 64) {
        const uint32_t i = stack[k];
        out[i] = rtc8x_alias_entry{i, 1.0f};
    }
    const uint32_t large_read = min(64u - kl, nl);
    for (uint32_t k = lane; k < nl - large_read; k += 64) {
        const uint32_t i = stack[n - 1u - k];
        out[i] = rtc8x_alias_entry{i, 1.0f};
    }
}

// One wavefront per texture row: its weights (mip 0 of the importance map) and their sum in texel order.
__global__ __launch_bounds__(64) void row_weights_kernel(const float* __restrict__ mip0, uint32_t w, uint32_t dim_x,
                                                         float* __restrict__ weights, double* __restrict__ row_sums)
{
    const uint32_t y = blockIdx.x, lane = threadIdx.x;
    for (uint32_t x = lane; x < w; x += 64) weights[(size_t)y * w + x] = mip0[(size_t)y * dim_x + x];
    const double sum = ordered_sum(mip0 + (size_t)y * dim_x, w);
    if (lane == 0) row_sums[y] = sum;
}

// One wavefront per alias table: block 0 the table over the rows (and the sum of the row sums in order), block
// y + 1 that of row y, so that the marginal's chain runs beside the rows'.
__global__ __launch_bounds__(64) void alias_kernel(const float* __restrict__ weights, const double* __restrict__ row_sums,
                                                   uint32_t w, uint32_t h, double* __restrict__ integral,
                                                   rtc8x_alias_entry* __restrict__ rows, rtc8x_alias_entry* __restrict__ cols)
{
    extern __shared__ double lds[];
    const uint32_t lane = threadIdx.x;
    if (blockIdx.x == 0) {
        for (uint32_t y = lane; y < h; y += 64) lds[y] = row_sums[y];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const double sum = ordered_sum(lds, h);
        if (lane == 0) *integral = sum;
        alias_table(lds, reinterpret_cast<uint16_t*>(lds + h), h, sum, rows);
        return;
    }
    const size_t y = blockIdx.x - 1u;
    float* const m = reinterpret_cast<float*>(lds);
    for (uint32_t x = lane; x < w; x += 64) m[x] = weights[y * w + x];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    alias_table(m, reinterpret_cast<uint16_t*>(m + w), w, row_sums[y], cols + y * w);
}

}  // namespace dev
}  // namespace rtc8x

using namespace rtc8x;

namespace {

uint32_t next_pow2(uint32_t x)
{
    uint32_t p = 1;
    while (p < x) p <<= 1;
    return p;
}

uint32_t pow2_exponent(uint32_t x)  // nextPowOf2Exponent (common/common_shared.h:129-133)
{
    if (x == 0) return 0;
    uint32_t e = 0;
    while ((1u << e) < x) ++e;
    return e;
}

}  // namespace

extern "C" rtc8x_status rtc8x_env_release(rtc8x_env_light* env)
try {
    RTC8X_REQUIRE(env != nullptr, "rtc8x_env_release: env is NULL");
    const void* ptrs[] = {env->mips, env->alias_rows, env->alias_cols, env->alias_weights};
    for (const void* p : ptrs)
        if (p) RTC8X_HIP(hipFree(const_cast<void*>(p)));
    env->mips = nullptr;
    env->alias_rows = nullptr;
    env->alias_cols = nullptr;
    env->alias_weights = nullptr;
    env->num_mip_levels = 0;
    env->map_integral = 0.0f;
    env->alias_integral = 0.0f;
    return RTC8X_OK;
}
RTC8X_CATCH_ALL("rtc8x_env_release")

extern "C" rtc8x_status rtc8x_env_build_sampler(rtc8x_env_light* env, void* stream)
try {
    RTC8X_REQUIRE(env != nullptr, "rtc8x_env_build_sampler: env is NULL");
    if (env->kind != RTC8X_ENV_LATLONG) return RTC8X_OK;
    RTC8X_REQUIRE(env->texels && env->width > 0 && env->height > 0 && env->width <= 16384 && env->height <= 16384,
                  "rtc8x_env_build_sampler: bad texture");
    hipStream_t s = (hipStream_t)stream;
    const uint32_t w = env->width, h = env->height;
    // map dimensions (compute_light_probs.cu:166-167)
    const uint32_t dim_x = next_pow2(w);
    const uint32_t dim_y = std::max(next_pow2(h), dim_x >> 1);
    RTC8X_REQUIRE(dim_x == dim_y || dim_x == 2 * dim_y, "rtc8x_env_build_sampler: map %ux%u must be 1:1 or 2:1", dim_x, dim_y);
    const uint32_t nlev = pow2_exponent(dim_x) + 1;
    size_t total = 0;
    std::vector<size_t> offs(nlev);
    for (uint32_t l = 0; l < nlev; ++l) {
        offs[l] = total;
        total += (size_t)std::max(dim_x >> l, 1u) * std::max(dim_y >> l, 1u);
    }
    // every device table is freed again unless the whole set-up succeeds
    struct Owned {
        void* p = nullptr;
        ~Owned()
        {
            if (p) (void)hipFree(p);
        }
        void* release()
        {
            void* r = p;
            p = nullptr;
            return r;
        }
    } o_mips, o_sums, o_rows, o_cols, o_weights;
    RTC8X_HIP(hipMalloc(&o_mips.p, total * sizeof(float)));
    RTC8X_HIP(hipMalloc(&o_sums.p, (h + 2) * sizeof(double)));
    RTC8X_HIP(hipMalloc(&o_rows.p, h * sizeof(rtc8x_alias_entry)));
    RTC8X_HIP(hipMalloc(&o_cols.p, (size_t)w * h * sizeof(rtc8x_alias_entry)));
    RTC8X_HIP(hipMalloc(&o_weights.p, (size_t)w * h * sizeof(float)));
    float* const mips = (float*)o_mips.p;
    double* const row_sums = (double*)o_sums.p;          // h row sums, then the two integrals
    double* const d_alias_integral = row_sums + h;
    float* const d_integral = (float*)(row_sums + h + 1);
    RTC8X_HIP(hipMemsetAsync(d_alias_integral, 0, 2 * sizeof(double), s));
    {
        dim3 blk(32, 8), grd((dim_x + 31) / 32, (dim_y + 7) / 8);
        hipLaunchKernelGGL(dev::env_mip0_kernel, grd, blk, 0, s, env->texels, w, h, dim_x, dim_y, mips);
        RTC8X_HIP(hipGetLastError());
    }
    for (uint32_t l = 1; l < nlev; ++l) {
        uint32_t sdx = std::max(dim_x >> (l - 1), 1u), sdy = std::max(dim_y >> (l - 1), 1u);
        uint32_t ddx = std::max(dim_x >> l, 1u), ddy = std::max(dim_y >> l, 1u);
        int top = (l == nlev - 1) ? 1 : 0;
        float top_scale = (float)(1u << (2 * (nlev - 1)));
        dim3 blk(16, 16), grd((ddx + 15) / 16, (ddy + 15) / 16);
        hipLaunchKernelGGL(dev::env_mip_kernel, grd, blk, 0, s, mips + offs[l - 1], sdx, sdy, mips + offs[l], ddx, ddy,
                           top, top_scale, d_integral);
        RTC8X_HIP(hipGetLastError());
    }
    // alias tables from the mip-0 weights (image region): at most 16,384 entries, 160 KB of LDS
    hipLaunchKernelGGL(dev::row_weights_kernel, dim3(h), dim3(64), 0, s, (const float*)mips, w, dim_x, (float*)o_weights.p,
                       row_sums);
    RTC8X_HIP(hipGetLastError());
    hipLaunchKernelGGL(dev::alias_kernel, dim3(h + 1), dim3(64), std::max(w * 6u, h * 10u), s, (const float*)o_weights.p,
                       (const double*)row_sums, w, h, d_alias_integral, (rtc8x_alias_entry*)o_rows.p,
                       (rtc8x_alias_entry*)o_cols.p);
    RTC8X_HIP(hipGetLastError());
    double integrals[2];
    RTC8X_HIP(hipMemcpyAsync(integrals, d_alias_integral, sizeof(integrals), hipMemcpyDeviceToHost, s));
    float top_texel = 0.0f;
    if (nlev == 1) RTC8X_HIP(hipMemcpyAsync(&top_texel, mips, sizeof(float), hipMemcpyDeviceToHost, s));
    RTC8X_HIP(hipStreamSynchronize(s));
    const double integral = integrals[0];
    float map_integral;
    std::memcpy(&map_integral, &integrals[1], sizeof(float));
    if (nlev == 1) map_integral = top_texel;
    RTC8X_REQUIRE(integral > 0.0, "rtc8x_env_build_sampler: environment is black");
    env->map_dim_x = dim_x;
    env->map_dim_y = dim_y;
    env->num_mip_levels = nlev;
    env->mips = (const float*)o_mips.release();
    env->map_integral = map_integral;
    env->alias_integral = (float)integral;
    env->alias_rows = (const rtc8x_alias_entry*)o_rows.release();
    env->alias_cols = (const rtc8x_alias_entry*)o_cols.release();
    env->alias_weights = (const float*)o_weights.release();
    return RTC8X_OK;
}
RTC8X_CATCH_ALL("rtc8x_env_build_sampler")
