// pga_loss.hip - the centre/size MSE of instances against targets and its
// gradient in one pass (gfx950).
//
// For instance i with model rows 0..2 (m, 3x4) the centre is column 3 and
// the size is the column norms of the 3x3 part:
//   c_i = (m[0][3], m[1][3], m[2][3]),  s_ij = |m[:, j]|,  j = 0..2,
//   loss = wc * sum_i |c_i - tc_i|^2 + ws * sum_i |s_i - ts_i|^2,
//   dloss/dm[r][3] = 2 wc (c_ir - tc_ir),
//   dloss/dm[r][j] = 2 ws (s_ij - ts_ij) m[r][j] / s_ij   (0 where s_ij = 0).
// 48 bytes of the instance and 24 of the targets are read, the 64-byte
// gradient row is written (column 12..15 zero): HBM bounds it. A wave takes 64
// instances at a time and moves rows and targets through LDS, so that every
// access to memory is a run of consecutive words; a lane's own 16-byte
// accesses at a stride of 64 bytes leave partly written lines. The loss is
// summed per workgroup in FP64 and added once per workgroup, and there are at
// most kBlocksMax of them: additions to one address sustain about 8e7 a
// second, so one for every 256 instances took longer than the traffic. 4.9M
// instances: 327 us with a thread per instance, 220 with fewer additions, 200
// (3.7 TB/s) with the rows through LDS as well; 0.3M: 30, 30 and 16 us.
// The reverse pass then reads the gradient rows as dL/dinstance.
#include <hip/hip_runtime.h>

#include "../../include/pga.h"

namespace pgaloss {

constexpr int kBlock = 512;
constexpr int kWaves = kBlock / 64;
constexpr uint32_t kBlocksMax = 512;      // two workgroups of 8 waves per compute unit

typedef float f4 __attribute__((ext_vector_type(4)));

// word k of record r in a wave's staging area: rotated by r / 4, so that
// neither side of the copy meets LDS bank conflicts
__device__ __forceinline__ uint32_t at(uint32_t r, uint32_t k) { return r * 4u + ((k + (r >> 2)) & 3u); }

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ void __launch_bounds__(kBlock) k_center_size_mse(const f4* __restrict__ inst,
                                                             const float* __restrict__ tc,
                                                             const float* __restrict__ ts, uint64_t n, float wc,
                                                             float ws, f4* __restrict__ grad,
                                                             double* __restrict__ loss) {
    __shared__ double part[kWaves];
    __shared__ f4 rows[kWaves][256];
    __shared__ float targets[kWaves][2][192];
    const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
    f4* S = rows[w];
    double l = 0.0;
    const uint64_t stride = (uint64_t)gridDim.x * kBlock;
    f4 v[4];
    float x[3], y[3];
    // the next tile's loads are in flight while this one is computed
    auto fetch = [&](uint64_t base) {
        const uint32_t cnt = base >= n ? 0u : (n - base < 64u ? (uint32_t)(n - base) : 64u);
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            const uint32_t q = lane + 64u * u;
            if (q < cnt * 4u) v[u] = inst[base * 4u + q];
        }
#pragma unroll
        for (uint32_t u = 0; u < 3u; ++u) {
            const uint32_t q = lane + 64u * u;
            if (q < cnt * 3u) {
                x[u] = tc[base * 3u + q];
                y[u] = ts[base * 3u + q];
            }
        }
    };
    fetch(((uint64_t)blockIdx.x * kWaves + w) * 64u);
    for (uint64_t base = ((uint64_t)blockIdx.x * kWaves + w) * 64u; base < n; base += stride) {
        const uint32_t cnt = n - base < 64u ? (uint32_t)(n - base) : 64u;
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            const uint32_t q = lane + 64u * u;
            S[at(q >> 2, q & 3u)] = v[u];
        }
#pragma unroll
        for (uint32_t u = 0; u < 3u; ++u) {
            targets[w][0][lane + 64u * u] = x[u];
            targets[w][1][lane + 64u * u] = y[u];
        }
        wave_sync();
        fetch(base + stride);
        if (lane < cnt) {
            const f4 r0 = S[at(lane, 0u)], r1 = S[at(lane, 1u)], r2 = S[at(lane, 2u)];
            const float m[12] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w};
            float g[12];
            float lc = 0.0f, lsz = 0.0f;
#pragma unroll
            for (int r = 0; r < 3; ++r) {           // centre: column 3
                const float d = m[r * 4 + 3] - targets[w][0][lane * 3u + r];
                lc += d * d;
                g[r * 4 + 3] = 2.0f * wc * d;
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {           // size: norm of column j
                const float a = m[j], b = m[4 + j], c = m[8 + j];
                const float s = sqrtf(a * a + b * b + c * c);
                const float d = s - targets[w][1][lane * 3u + j];
                lsz += d * d;
                const float k = s > 0.0f ? 2.0f * ws * d / s : 0.0f;
                g[j] = k * a;
                g[4 + j] = k * b;
                g[8 + j] = k * c;
            }
            // the lane's record is its own: written in place
            S[at(lane, 0u)] = f4{g[0], g[1], g[2], g[3]};
            S[at(lane, 1u)] = f4{g[4], g[5], g[6], g[7]};
            S[at(lane, 2u)] = f4{g[8], g[9], g[10], g[11]};
            S[at(lane, 3u)] = f4{0.0f, 0.0f, 0.0f, 0.0f};
            l += (double)wc * (double)lc + (double)ws * (double)lsz;
        }
        wave_sync();
#pragma unroll
        for (uint32_t u = 0; u < 4u; ++u) {
            const uint32_t q = lane + 64u * u;
            if (q < cnt * 4u) __builtin_nontemporal_store(S[at(q >> 2, q & 3u)], grad + base * 4u + q);
        }
        wave_sync();
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) l += __shfl_xor(l, d);
    if (lane == 0u) part[w] = l;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
#pragma unroll
        for (int k = 0; k < kWaves; ++k) t += part[k];
        if (t != 0.0) atomicAdd(loss, t);
    }
}

} // namespace pgaloss

extern "C" {

// Declared in include/pga.h.
PGA_API pga_status pga_center_size_mse(const float* instances, const float* target_centers,
                                       const float* target_sizes, uint64_t count, float weight_centers,
                                       float weight_sizes, float* dl_dinstances, double* loss, void* stream) {
    if (count == 0u) return PGA_OK;
    if (!instances || !target_centers || !target_sizes || !dl_dinstances || !loss) return PGA_ERR_INVALID_ARG;
    if ((((uintptr_t)instances) | ((uintptr_t)dl_dinstances)) & 15u) return PGA_ERR_INVALID_ARG;
    uint64_t blocks = (count + pgaloss::kBlock - 1u) / pgaloss::kBlock;
    if (blocks > 0x7FFFFFFFull) return PGA_ERR_INVALID_ARG;
    if (blocks > pgaloss::kBlocksMax) blocks = pgaloss::kBlocksMax;
    hipLaunchKernelGGL(pgaloss::k_center_size_mse, dim3((uint32_t)blocks), dim3(pgaloss::kBlock), 0,
                       (hipStream_t)stream, reinterpret_cast<const pgaloss::f4*>(instances), target_centers,
                       target_sizes, count, weight_centers, weight_sizes, reinterpret_cast<pgaloss::f4*>(dl_dinstances),
                       loss);
    return hipGetLastError() == hipSuccess ? PGA_OK : PGA_ERR_HIP;
}

} // extern "C"
