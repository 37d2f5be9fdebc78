// The brute-force pair term and the workgroup-cooperative sum over affecting bodies, shared by the
// single brute force (bf.hip) and the batched ensemble (batch.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pnb {

// a_i += d * (mu * rsq(r2)^3) for one affecting body q and R affected bodies per lane.
// MASK: a pair at zero distance adds nothing. SELF: body `self + 64 r` of the affecting array is
// affected body r itself and adds nothing (whatever its term would be); j is q's index.
// SEQ: keeps the terms and their reciprocal square roots in source order (scheduling barriers).
// Left alone, the compiler interleaves the terms of several bodies; one after the other they issue
// 10-20 % faster once a SIMD holds about four wavefronts to fill the gaps (262,144 x 65,536, one body
// per lane from scalar loads: 3.90 -> 4.21 T pairs/s; the cooperative sums 2.6 -> 3.1), and slower
// with fewer (65,536 x 4,096 in two wavefronts per SIMD 26 -> 35 us).
template <int R, bool MASK, bool SELF = false, bool SEQ = false>
__device__ __forceinline__ void bf_body(const float4 q, const float (&xi)[R], const float (&yi)[R],
                                        const float (&zi)[R], float eps2, float (&px)[R],
                                        float (&py)[R], float (&pz)[R], uint32_t j = 0,
                                        uint32_t self = 0, uint32_t stride = 64) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float dx = q.x - xi[r];
        const float dy = q.y - yi[r];
        const float dz = q.z - zi[r];
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
        if (SEQ) __builtin_amdgcn_sched_barrier(0);
        float inv = __builtin_amdgcn_rsqf(r2);
        if (SEQ) __builtin_amdgcn_sched_barrier(0);
        if (MASK) inv = (r2 > 0.0f) ? inv : 0.0f;
        if (SELF) inv = (j != self + uint32_t(r) * stride) ? inv : 0.0f;
        const float s = (q.w * inv) * (inv * inv);
        px[r] = fmaf(dx, s, px[r]);
        py[r] = fmaf(dy, s, py[r]);
        pz[r] = fmaf(dz, s, pz[r]);
        if (SEQ) __builtin_amdgcn_sched_barrier(0);
    }
}

// Four bodies; aligned as the arrays are (a slice of a tensor, an ensemble's system), not as its size is.
typedef float f32x16_t __attribute__((ext_vector_type(16), aligned(16)));
static_assert(alignof(f32x16_t) == alignof(float4), "read at any body of an array");

// T affecting bodies at a wave-uniform address, four per scalar load, the next four requested before
// the present four are summed: one by one, each body is five scalar instructions, a load and a wait.
// For sums of few wavefronts (4,096 x 60,000 91 -> 82 us, 4,096 x 4,096 10.8 -> 10.1); where a SIMD
// holds eight the waits cost nothing and this form is slower (1,048,576 x 65,536 18.7 -> 19.0 ms
// on one card).
template <int T, int R, bool MASK, bool SEQ>
__device__ __forceinline__ void bf_tile(const float4* __restrict__ q, const float (&xi)[R],
                                        const float (&yi)[R], const float (&zi)[R], float eps2,
                                        float (&px)[R], float (&py)[R], float (&pz)[R]) {
    const f32x16_t* g = reinterpret_cast<const f32x16_t*>(q);
    f32x16_t a = g[0];
    const auto four = [&](const f32x16_t& v) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            bf_body<R, MASK, false, SEQ>(make_float4(v[4 * u], v[4 * u + 1], v[4 * u + 2], v[4 * u + 3]),
                                         xi, yi, zi, eps2, px, py, pz);
    };
    // (the empty asm statements wait for a group where it is first needed, before the next is asked for)
#pragma unroll 1
    for (int j = 0; j < T; j += 8) {
        asm volatile("" ::"s"(a));
        __builtin_amdgcn_sched_barrier(0);
        const f32x16_t b = g[j / 4 + 1];
        __builtin_amdgcn_sched_barrier(0);
        four(a);
        asm volatile("" ::"s"(b));
        __builtin_amdgcn_sched_barrier(0);
        a = g[j + 8 < T ? j / 4 + 2 : 0];
        __builtin_amdgcn_sched_barrier(0);
        four(b);
    }
}

// Any number of affecting bodies at a wave-uniform address: eight at a time, then the rest requested
// together (one by one each waits for its load: a step of 2,000 x 250 bodies 13.4 us so, 11.6 now).
template <int R, bool MASK, bool SELF, bool SEQ>
__device__ __forceinline__ void bf_span(const float4* __restrict__ q, uint32_t cnt, const float (&xi)[R],
                                        const float (&yi)[R], const float (&zi)[R], float eps2,
                                        float (&px)[R], float (&py)[R], float (&pz)[R],
                                        uint32_t j0 = 0, uint32_t self = 0) {
    uint32_t j = 0;
    for (; j + 8 <= cnt; j += 8) {
        float4 b[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) b[u] = q[j + u];
        if (SEQ) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
            bf_body<R, MASK, SELF, SEQ>(b[u], xi, yi, zi, eps2, px, py, pz, j0 + j + u, self);
    }
    if (j < cnt) {
        float4 b[7];
#pragma unroll
        for (uint32_t u = 0; u < 7; ++u) b[u] = q[min(j + u, cnt - 1)];
#pragma unroll
        for (uint32_t u = 0; u < 7; ++u)
            if (j + u < cnt) bf_body<R, MASK, SELF, SEQ>(b[u], xi, yi, zi, eps2, px, py, pz, j0 + j + u, self);
    }
}

__device__ __forceinline__ void kahan_add(float& sum, float& comp, float v) {
    const float y = v - comp;
    const float t = sum + y;
    comp = (t - sum) - y;
    sum = t;
}

// Shared memory of coop_sum for a workgroup of W wavefronts: every wavefront's sums over its
// latest tile, and the running compensated sums of each group of J wavefronts (J >= 2).
template <int R, int W>
struct CoopLds {
    float part[W][3 * R][64];
    float sum[W / 2][3 * R][2][64];
};

// One affected tile of 64 R bodies summed by J wavefronts together (J a power of two, 1 <= J <= W,
// the same in every wavefront of the workgroup; wavefronts g J .. g J + J - 1 form group g).
// The affecting range [jb, je) is taken in tiles of T bodies, J tiles a round, one per wavefront,
// each read with wave-uniform addresses (scalar loads). A tile's sum is plain FP32; the J sums of
// a round go through LDS into the group's compensated sums in tile order, so the result is the
// one a single wavefront gets from the same tiles in order, whatever J is. Folding is spread over
// the group (wavefront k takes components k, k + J, ...), so a round costs two barriers and
// a few LDS reads for 256 x R pair terms per lane.
// Every wavefront of the workgroup calls it the same number of times with the same range (idle
// groups pass live = false); `ax, ay, az` come back complete in every wavefront of the group.
// Why the split: one wavefront issues about one instruction per 4.8 cycles however idle its CU is,
// so a tile of affected bodies walked by one wavefront takes m x R x 13 x 4.8 cycles (1.7 ms for
// 16,384 affecting bodies and R = 4); J wavefronts divide that by J without another pass over
// memory.
template <int R, bool MASK, bool SELF, int T, int W>
__device__ __forceinline__ void coop_sum(CoopLds<R, W>& lds, const float4* __restrict__ afg,
                                         uint32_t jb, uint32_t je, int J, int wave, bool live,
                                         float eps2, uint32_t self, const float (&xi)[R],
                                         const float (&yi)[R], const float (&zi)[R],
                                         float (&ax)[R], float (&ay)[R], float (&az)[R]) {
    const int lane = threadIdx.x & 63;
    const int slot = wave & (J - 1), g0 = wave - slot, g = g0 / J;
    const uint32_t own = SELF ? uint32_t(__builtin_amdgcn_readfirstlane(int(self))) : 0u;
    float cx[R], cy[R], cz[R];
#pragma unroll
    for (int r = 0; r < R; ++r) ax[r] = ay[r] = az[r] = cx[r] = cy[r] = cz[r] = 0.0f;
    if (J > 1) {
        for (int c = slot; c < 3 * R; c += J) lds.sum[g][c][0][lane] = lds.sum[g][c][1][lane] = 0.0f;
        __syncthreads();
    }
    const uint32_t span = uint32_t(T) * uint32_t(J);
    for (uint32_t base = jb; base < je; base += span) {
        const uint32_t j0 = base + uint32_t(T) * uint32_t(slot);
        float px[R], py[R], pz[R];
#pragma unroll
        for (int r = 0; r < R; ++r) px[r] = py[r] = pz[r] = 0.0f;
        if (live && j0 < je) {
            const float4* q = afg + j0;
            const uint32_t cnt = min(uint32_t(T), je - j0);
            if (SELF && j0 < own + 64 * R && own < j0 + cnt) {  // only here can a pair be a body with itself
                bf_span<R, MASK, true, true>(q, cnt, xi, yi, zi, eps2, px, py, pz, j0, self);
            } else if (cnt == uint32_t(T)) {
                bf_tile<T, R, MASK, true>(q, xi, yi, zi, eps2, px, py, pz);
            } else {
                bf_span<R, MASK, false, true>(q, cnt, xi, yi, zi, eps2, px, py, pz);
            }
        }
        if (J == 1) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                kahan_add(ax[r], cx[r], px[r]);
                kahan_add(ay[r], cy[r], py[r]);
                kahan_add(az[r], cz[r], pz[r]);
            }
            continue;
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            lds.part[wave][3 * r][lane] = px[r];
            lds.part[wave][3 * r + 1][lane] = py[r];
            lds.part[wave][3 * r + 2][lane] = pz[r];
        }
        __syncthreads();
        const int tiles = int(min(uint32_t(J), (je - base + uint32_t(T) - 1) / uint32_t(T)));
        for (int c = slot; c < 3 * R; c += J) {
            float s = lds.sum[g][c][0][lane], k = lds.sum[g][c][1][lane];
            for (int t = 0; t < tiles; ++t) kahan_add(s, k, lds.part[g0 + t][c][lane]);
            lds.sum[g][c][0][lane] = s;
            lds.sum[g][c][1][lane] = k;
        }
        __syncthreads();
    }
    if (J > 1) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            ax[r] = lds.sum[g][3 * r][0][lane];
            ay[r] = lds.sum[g][3 * r + 1][0][lane];
            az[r] = lds.sum[g][3 * r + 2][0][lane];
        }
        __syncthreads();  // the sums are read before the next call clears them
    }
}

}  // namespace pnb
