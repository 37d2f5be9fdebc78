// Brute-force gravitational acceleration on gfx950, and the FP64 direct sum used as the accuracy reference.
//
// Replaces the reference's wgpu brute force (particular/src/gpu/bruteforce_shared.wgsl:8-31 and
// particular/src/gpu/mod.rs:179-208) with its own design for CDNA4:
//  * each lane owns R affected particles: one by default, its terms kept in source order (bf_body), more
//    by a tuning entry (register blocking: one affecting body fetched per wave feeds R chains);
//  * affecting bodies are shared by the whole workgroup, either staged tile by tile in LDS and
//    read back as broadcasts (variant 0) or read straight from memory with wave-uniform addresses,
//    which the compiler turns into scalar loads into SGPRs (variant 1);
//  * the pair term uses the hardware reciprocal square root (v_rsq_f32),
//    a_i += d * (mu * rsq(r2)^3), r2 = |d|^2 + eps^2;
//  * sums are plain FP32 within a tile of BF_TILE affecting bodies and Kahan-compensated across
//    tiles, so the error does not grow with the affecting count;
//  * the affecting range is split over several workgroups (j_split) whose partial sums are reduced
//    in a fixed order, so results do not depend on scheduling;
//  * sums too small to fill the chip so (coop_pays) are taken by workgroups of sixteen wavefronts
//    per 64 affected bodies that share the affecting ones tile by tile (bf_coop_kernel).
// Pair semantics follow particular/src/gravity/impls/mod.rs:151-166: with `checked` a pair at
// zero unsoftened distance contributes nothing; with softening > 0 that pair contributes
// d * finite = 0 anyway, so only checked && softening == 0 needs the explicit mask.
#include "bf_common.hpp"
#include "bf_shape.hpp"
#include "pnb_internal.hpp"

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

namespace pnb {

struct BfTuneEntry {
    size_t n_min;
    int variant, per_lane, j_split;
};
struct BfTune {
    std::vector<BfTuneEntry> entries;
};

void bf_tune_free(BfTune* t) { delete t; }

// grid.x: affected tiles of BF_BLOCK * R particles; grid.y: affecting ranges of j_chunk bodies.
// With gridDim.y == 1 the result goes to `out`, else to partial[blockIdx.y * n + i].
// VAR 0: LDS tile; 1: wave-uniform global reads (scalar loads). SELF: aff and afg are one array and
// a body's pair with itself adds nothing; only the tiles that meet the workgroup's own bodies test
// for it.
template <int R, bool MASK, int VAR, bool SELF = false>
__global__ __launch_bounds__(BF_BLOCK) void bf_kernel(const float4* __restrict__ aff, uint32_t n,
                                                      const float4* __restrict__ afg, uint32_t m,
                                                      uint32_t j_chunk, float eps2,
                                                      float4* __restrict__ out) {
    constexpr bool LDS = VAR == 0;
    __shared__ float4 tile[LDS ? BF_TILE : 1];
    const uint32_t jb = blockIdx.y * j_chunk;
    const uint32_t je = min(m, jb + j_chunk);
    const uint32_t i0 = blockIdx.x * (BF_BLOCK * R) + threadIdx.x;

    float xi[R], yi[R], zi[R], ax[R], ay[R], az[R], cx[R], cy[R], cz[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t i = i0 + r * BF_BLOCK;
        const float4 p = aff[i < n ? i : n - 1];
        xi[r] = p.x; yi[r] = p.y; zi[r] = p.z;
        ax[r] = ay[r] = az[r] = 0.0f;
        cx[r] = cy[r] = cz[r] = 0.0f;
    }

    for (uint32_t j0 = jb; j0 < je; j0 += BF_TILE) {
        const uint32_t cnt = min(uint32_t(BF_TILE), je - j0);
        if (LDS) {
            __syncthreads();
            if (threadIdx.x < cnt) tile[threadIdx.x] = afg[j0 + threadIdx.x];
            __syncthreads();
        }
        float px[R], py[R], pz[R];
#pragma unroll
        for (int r = 0; r < R; ++r) px[r] = py[r] = pz[r] = 0.0f;
        const uint32_t own = blockIdx.x * uint32_t(BF_BLOCK * R);
        if (SELF && j0 < own + BF_BLOCK * R && own < j0 + cnt) {
            for (uint32_t j = 0; j < cnt; ++j)
                bf_body<R, MASK, true>(LDS ? tile[j] : afg[j0 + j], xi, yi, zi, eps2, px, py, pz, j0 + j, i0, BF_BLOCK);
        } else if (cnt == BF_TILE) {
#pragma unroll 8
            for (int j = 0; j < BF_TILE; ++j)
                bf_body<R, MASK, false, R == 1>(LDS ? tile[j] : afg[j0 + j], xi, yi, zi, eps2, px, py, pz);
        } else if (LDS) {
            for (uint32_t j = 0; j < cnt; ++j) bf_body<R, MASK>(tile[j], xi, yi, zi, eps2, px, py, pz);
        } else {
            bf_span<R, MASK, false, R == 1>(afg + j0, cnt, xi, yi, zi, eps2, px, py, pz);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            kahan_add(ax[r], cx[r], px[r]);
            kahan_add(ay[r], cy[r], py[r]);
            kahan_add(az[r], cz[r], pz[r]);
        }
    }

    float4* dst = out + size_t(blockIdx.y) * n;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t i = i0 + r * BF_BLOCK;
        if (i < n) dst[i] = make_float4(ax[r], ay[r], az[r], 0.0f);
    }
}

// Small and middle affected counts: one workgroup of COOP_WAVES wavefronts per 64 affected bodies
// (and per affecting range, grid.y), the wavefronts sharing the affecting bodies tile by tile
// (coop_sum). One wavefront per affected tile would leave SIMDs idle there, and each wavefront is bound
// by its own issue rate; coop_pays holds the sizes.
template <bool MASK, bool SELF, int T>
__global__ __launch_bounds__(64 * COOP_WAVES) void bf_coop_kernel(const float4* __restrict__ aff,
                                                                  uint32_t n,
                                                                  const float4* __restrict__ afg,
                                                                  uint32_t m, uint32_t j_chunk,
                                                                  float eps2,
                                                                  float4* __restrict__ out) {
    __shared__ CoopLds<1, COOP_WAVES> lds;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    const uint32_t i = blockIdx.x * 64 + (threadIdx.x & 63);
    const uint32_t jb = blockIdx.y * j_chunk, je = min(m, jb + j_chunk);
    const float4 p = aff[i < n ? i : n - 1];
    const float xi[1] = {p.x}, yi[1] = {p.y}, zi[1] = {p.z};
    float ax[1], ay[1], az[1];
    asm volatile("" : "+v"(eps2));  // a scalar operand halves an instruction's rate
    coop_sum<1, MASK, SELF, T, COOP_WAVES>(lds, afg, jb, je, COOP_WAVES, wave, true, eps2, i, xi, yi,
                                           zi, ax, ay, az);
    if (wave == 0 && i < n)
        out[size_t(blockIdx.y) * n + i] = make_float4(ax[0], ay[0], az[0], 0.0f);
}

// Fixed-order compensated reduction of j_split partial sums.
__global__ void bf_reduce_kernel(const float4* __restrict__ partial, uint32_t n, uint32_t splits,
                                 float4* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float ax = 0, ay = 0, az = 0, cx = 0, cy = 0, cz = 0;
#pragma unroll 8
    for (uint32_t s = 0; s < splits; ++s) {
        const float4 p = partial[size_t(s) * n + i];
        kahan_add(ax, cx, p.x);
        kahan_add(ay, cy, p.y);
        kahan_add(az, cz, p.z);
    }
    out[i] = make_float4(ax, ay, az, 0.0f);
}

__global__ void fill_zero_kernel(float4* __restrict__ out, size_t n) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) out[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

using BfKernel = void (*)(const float4*, uint32_t, const float4*, uint32_t, uint32_t, float, float4*);

template <bool MASK, int VAR>
static BfKernel pick_r(int r) {
    switch (r) {
        case 1: return bf_kernel<1, MASK, VAR>;
        case 2: return bf_kernel<2, MASK, VAR>;
        case 4: return bf_kernel<4, MASK, VAR>;
        default: return bf_kernel<8, MASK, VAR>;
    }
}

template <int VAR>
static BfKernel pick_mask(int r, bool mask) {
    return mask ? pick_r<true, VAR>(r) : pick_r<false, VAR>(r);
}

template <bool SELF>
static BfKernel pick_coop(bool mask, int tile) {
    switch (tile) {
        case 64: return mask ? bf_coop_kernel<true, SELF, 64> : bf_coop_kernel<false, SELF, 64>;
        case 128: return mask ? bf_coop_kernel<true, SELF, 128> : bf_coop_kernel<false, SELF, 128>;
        default: return mask ? bf_coop_kernel<true, SELF, 256> : bf_coop_kernel<false, SELF, 256>;
    }
}

static size_t cu_count(const pnb_ctx* c) { return c->cu_count > 0 ? size_t(c->cu_count) : 256; }

static BfShape choose_shape(pnb_ctx* c, size_t n, size_t m) {
    if (c->bf_tune) {
        const BfTuneEntry* best = nullptr;
        for (const auto& e : c->bf_tune->entries)
            if (e.n_min <= n && (!best || e.n_min > best->n_min)) best = &e;
        if (best) return {best->variant, best->per_lane, best->j_split};
    }
    return default_shape(cu_count(c), n, m);
}

static BfPlan plan(pnb_ctx* c, size_t n, size_t m) { return plan_for(choose_shape(c, n, m), m); }

// Allocates in `scratch` what bf_launch(n, m) will need of it, so that a later launch inside a graph
// capture allocates nothing.
int bf_prepare(pnb_ctx* c, size_t n, size_t m, DevBuf& scratch) {
    if (n == 0 || m == 0) return PNB_OK;
    const BfPlan p = plan(c, n, m);
    if (p.splits > 1) PNB_HIP(c, scratch.ensure(size_t(p.splits) * n * sizeof(float4)));
    return PNB_OK;
}

// Scratch of the allocation-free entry point (pnb_bf_accel_f32_dev_noalloc): the partial sums of
// the affecting split, splits * n records. 256 MiB: the default shapes need at most
// 256 * CUs * BF_BLOCK records (16,777,216 on 256 CUs). Every GPU the library runs on holds its
// own copy until the process ends; every call on that GPU shares it.
constexpr size_t BF_SCRATCH_RECORDS = size_t(1) << 24;
static __device__ __align__(256) float4 scratch[BF_SCRATCH_RECORDS];
constexpr int BF_SCRATCH_DEVICES = 64;
static float4* g_scratch_dev[BF_SCRATCH_DEVICES];  // device address of `scratch` per device
static std::mutex g_scratch_mu;

// Once per device, with that device current (called by pnb_create): the device address of
// `scratch`. In host code the array's name is a host-side stand-in, not a device address.
int bf_noalloc_init(pnb_ctx* c) {
    if (c->device < 0 || c->device >= BF_SCRATCH_DEVICES) return PNB_OK;  // entry point refuses
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[c->device]) {
        void* ptr = nullptr;
        PNB_HIP(c, hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        g_scratch_dev[c->device] = static_cast<float4*>(ptr);
    }
    c->noalloc_scratch = g_scratch_dev[c->device];
    return PNB_OK;
}

// The launch itself, with the split's partial sums in `partial` (at least splits * n records;
// unused when the plan has one split). No allocation.
static int bf_launch_with(pnb_ctx* c, const BfPlan& p, const float4* affected, size_t n,
                          const float4* affecting, size_t m, float softening, int checked,
                          float4* out, float4* partial, bool self = false) {
    const BfShape sh = p.shape;
    const bool mask = checked && softening == 0.0f;
    const bool coop = sh.variant == BF_COOP;
    BfKernel k;
    if (coop) k = self ? pick_coop<true>(mask, p.tile) : pick_coop<false>(mask, p.tile);
    else if (self && sh.variant == 0) k = mask ? bf_kernel<1, true, 0, true> : bf_kernel<1, false, 0, true>;
    else if (self) k = mask ? bf_kernel<1, true, 1, true> : bf_kernel<1, false, 1, true>;
    else k = sh.variant == 0 ? pick_mask<0>(sh.per_lane, mask) : pick_mask<1>(sh.per_lane, mask);
    const float eps2 = softening * softening;
    const uint32_t splits = p.splits, chunk = p.chunk;
    const unsigned block = bf_block(sh);
    dim3 grid(bf_grid_x(sh, n), splits);
    float4* dst = splits > 1 ? partial : out;
    return timed(c, PNB_PROF_BF, [&]() -> int {
        k<<<grid, block, 0, c->stream>>>(affected, uint32_t(n), affecting, uint32_t(m), chunk,
                                            eps2, dst);
        PNB_CHECK_LAUNCH(c);
        if (splits > 1) {
            bf_reduce_kernel<<<div_up(n, 256), 256, 0, c->stream>>>(dst, uint32_t(n), splits, out);
            PNB_CHECK_LAUNCH(c);
        }
        return PNB_OK;
    });
}

// The sum over all other bodies of one set, for sizes where the pair kernel cannot fill the chip
// (pairs.hip): a body's term with itself is left out by index, whatever the softening. The split's
// partial sums are kept in the pair kernel's scratch, so that a pair sum frees no memory that an
// f32 brute force captured in a graph goes on using (DevBuf::ensure frees what it outgrows).
int bf_self_launch(pnb_ctx* c, const float4* p, size_t n, float softening, int checked, float4* out) {
    const BfPlan pl = plan_for(default_shape(cu_count(c), n, n), n);
    if (pl.splits > 1) {
        const size_t need = size_t(pl.splits) * n * sizeof(float4);
        if (c->capturing && c->pairs_part.cap < need)
            return fail(c, PNB_E_STATE, "brute-force scratch not prepared before graph capture");
        PNB_HIP(c, c->pairs_part.ensure(need));
    }
    return bf_launch_with(c, pl, p, n, p, n, softening, checked, out, c->pairs_part.as<float4>(), true);
}

int bf_launch(pnb_ctx* c, const float4* affected, size_t n, const float4* affecting, size_t m,
              float softening, int checked, float4* out, DevBuf* scratch) {
    if (n == 0) return PNB_OK;
    if (n > 0x7fffffffu || m > 0x7fffffffu)
        return fail(c, PNB_E_ARG, "brute force supports at most 2^31-1 particles per side");
    if (m == 0) {
        fill_zero_kernel<<<div_up(n, 256), 256, 0, c->stream>>>(out, n);
        PNB_CHECK_LAUNCH(c);
        return PNB_OK;
    }
    const BfPlan p = plan(c, n, m);
    DevBuf& part = scratch ? *scratch : c->bf_partial;
    if (p.splits > 1) {
        const size_t need = size_t(p.splits) * n * sizeof(float4);
        if (c->capturing && part.cap < need)
            return fail(c, PNB_E_STATE, "brute-force scratch not prepared before graph capture");
        PNB_HIP(c, part.ensure(need));
    }
    return bf_launch_with(c, p, affected, n, affecting, m, softening, checked, out, part.as<float4>());
}

// ---- FP64 direct sum: one workgroup per affected particle, fixed-order tree reduction --------

constexpr int DF_BLOCK = 256;

__global__ __launch_bounds__(DF_BLOCK) void direct_f64_kernel(const float4* __restrict__ aff,
                                                               const float4* __restrict__ afg,
                                                               uint32_t m, double eps2,
                                                               double* __restrict__ out3) {
    const uint32_t i = blockIdx.x;
    const float4 p = aff[i];
    const double x = p.x, y = p.y, z = p.z;
    double sx = 0, sy = 0, sz = 0;
    for (uint32_t j = threadIdx.x; j < m; j += DF_BLOCK) {
        const float4 q = afg[j];
        const double dx = double(q.x) - x, dy = double(q.y) - y, dz = double(q.z) - z;
        const double r2 = dx * dx + dy * dy + dz * dz;
        if (r2 == 0.0) continue;
        const double rs = r2 + eps2;
        const double s = double(q.w) / (rs * sqrt(rs));
        sx += dx * s; sy += dy * s; sz += dz * s;
    }
    __shared__ double red[3][DF_BLOCK];
    red[0][threadIdx.x] = sx;
    red[1][threadIdx.x] = sy;
    red[2][threadIdx.x] = sz;
    __syncthreads();
    for (int w = DF_BLOCK / 2; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            for (int k = 0; k < 3; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out3[3 * size_t(i)] = red[0][0];
        out3[3 * size_t(i) + 1] = red[1][0];
        out3[3 * size_t(i) + 2] = red[2][0];
    }
}

// ---- FP64 brute force (glam::DVec3 / f64: particular/src/gravity/impls/glam.rs:234) ------------
// The reference's scalar kernel in FP64 (impls/mod.rs:151-166). A workgroup of W wavefronts (plan64)
// holds 64 affected bodies; the affecting range is split over grid.y and, inside a
// workgroup, over its wavefronts (scalar loads), whose sums are added in wavefront order, and the
// grid.y partial sums in order by bf64_reduce_kernel. checked: zero distance contributes nothing.

// mu r2^(-3/2). From the estimate y = v_rsq_f64(r2) (about 1e-8 relative, here cut to 26 bits, so that
// y^2 is exact) and e = 1 - r2 y^2, r2^(-3/2) = y^3 (1 - e)^(-3/2), the binomial series to second order
// (the third is 1e-22). The cube is corrected, not the root, whose error cubing would triple: three
// roundings, as an IEEE root, product and division have. y^2 takes the correction: it stays finite where
// the result overflows, which has to give infinity.
// An infinite r2 (y = 0) gives 0; with ZERO, a vanishing r2 infinity, as a division by it does.
// c1, c2: 3/2 and 15/8, held by the caller in vector registers (a literal is moved there for every term).
template <bool ZERO>
__device__ __forceinline__ double cubed64(double mu, double r2, double c1, double c2) {
    const double y = __longlong_as_double(__double_as_longlong(__builtin_amdgcn_rsq(r2)) & ~0x7ffffffll);
    const double y2 = y * y;
    double r = fmin(r2, 1.7976931348623157e308);
    if (ZERO) r = fmax(r, 4.9406564584124654e-324);
    const double e = fma(-r, y2, 1.0);
    return (mu * y) * fma(y2 * e, fma(e, c2, c1), y2);
}

// One lane's share, bodies jb .. je of afg. CHECK tests the unsoftened distance; ZERO as above.
template <bool CHECK, bool ZERO>
__device__ __forceinline__ double3 sum64(const double4 p, const double4* __restrict__ afg, uint32_t jb,
                                         uint32_t je, double eps2) {
    double ax = 0.0, ay = 0.0, az = 0.0, c1 = 1.5, c2 = 1.875;
    asm volatile("" : "+v"(c1), "+v"(c2));
#pragma unroll 4
    for (uint32_t j = jb; j < je; ++j) {
        const double4 q = afg[j];  // wave-uniform: a scalar load
        const double dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
        const double d2 = fma(dx, dx, fma(dy, dy, CHECK ? dz * dz : fma(dz, dz, eps2)));
        double s = cubed64<ZERO>(q.w, CHECK ? d2 + eps2 : d2, c1, c2);
        if (CHECK) s = d2 == 0.0 ? 0.0 : s;
        ax = fma(dx, s, ax);
        ay = fma(dy, s, ay);
        az = fma(dz, s, az);
    }
    return make_double3(ax, ay, az);
}

// Unchecked sums, and checked ones with a softening whose square is normal (there a pair at zero distance
// adds d s = 0 by itself unless s overflows, and an infinite mu must not reach its own body), are taken
// without test or clamp, and again with them where they come out NaN: 40,000 x 40,000 bodies 963 us,
// with the test in every term 1,095, with the clamp 1,005.
constexpr int BF64_UNCHECKED = 0, BF64_CHECKED = 1, BF64_SOFTENED = 2;

template <int MODE, int W>
__global__ __launch_bounds__(64 * W) void bf64_kernel(
    const double4* __restrict__ aff, uint32_t n, const double4* __restrict__ afg, uint32_t m,
    uint32_t j_chunk, double eps2, double4* __restrict__ out) {
    __shared__ double part[W][3][64];
    const int wave = W > 1 ? __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)) : 0;
    const int lane = threadIdx.x & 63;
    const uint32_t i = blockIdx.x * 64 + lane;
    const double4 p = aff[i < n ? i : n - 1];
    const uint32_t b0 = blockIdx.y * j_chunk, b1 = min(m, b0 + j_chunk);
    const uint32_t per = (b1 - b0 + W - 1) / W;
    const uint32_t jb = min(b1, b0 + wave * per), je = min(b1, jb + per);
    double3 a = sum64<MODE == BF64_CHECKED, false>(p, afg, jb, je, eps2);
    if (MODE != BF64_CHECKED) {
        const bool again = isnan(a.x) || isnan(a.y) || isnan(a.z);
        if (__ballot(again)) {
            const double3 b = sum64<MODE == BF64_SOFTENED, MODE == BF64_UNCHECKED>(p, afg, jb, je, eps2);
            if (again) a = b;
        }
    }
    if (W > 1) {
        part[wave][0][lane] = a.x;
        part[wave][1][lane] = a.y;
        part[wave][2][lane] = a.z;
        __syncthreads();
        if (wave != 0) return;
        for (int w = 1; w < W; ++w) {
            a.x += part[w][0][lane];
            a.y += part[w][1][lane];
            a.z += part[w][2][lane];
        }
    }
    if (i < n) out[size_t(blockIdx.y) * n + i] = make_double4(a.x, a.y, a.z, 0.0);
}

__global__ __launch_bounds__(64) void bf64_reduce_kernel(const double4* __restrict__ partial,
                                                         uint32_t n, uint32_t splits,
                                                         double4* __restrict__ out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double ax = 0.0, ay = 0.0, az = 0.0;
#pragma unroll 8
    for (uint32_t s = 0; s < splits; ++s) {
        const double4 p = partial[size_t(s) * n + i];
        ax += p.x;
        ay += p.y;
        az += p.z;
    }
    out[i] = make_double4(ax, ay, az, 0.0);
}

// Both sides of a sum over host arrays. A set on itself, or on its own first m bodies, passes one
// pointer twice and is uploaded once.
static int upload_sides(pnb_ctx* c, const void* affected, size_t n, const void* affecting, size_t m,
                        size_t record) {
    if (affecting == affected) return stage_in(c, c->h_affected, affected, std::max(n, m) * record);
    if (int rc = stage_in(c, c->h_affected, affected, n * record)) return rc;
    return stage_in(c, c->h_affecting, affecting, m * record, 1);
}

}  // namespace pnb

using namespace pnb;

extern "C" {

int pnb_bf_accel_f32_dev(pnb_ctx* c, const float* affected, size_t n, const float* affecting,
                         size_t m, float softening, int checked, float* out) {
    if (!c) return PNB_E_ARG;
    if ((n && (!affected || !out)) || (m && !affecting))
        return fail(c, PNB_E_ARG, "null pointer with non-zero length");
    if (!(softening >= 0.0f)) return fail(c, PNB_E_ARG, "softening must be >= 0");
    if (int rc = activate(c)) return rc;
    return bf_launch(c, reinterpret_cast<const float4*>(affected), n,
                     reinterpret_cast<const float4*>(affecting), m, softening, checked,
                     reinterpret_cast<float4*>(out));
}

int pnb_bf_accel_f32_dev_noalloc(pnb_ctx* c, const float* affected, size_t n,
                                 const float* affecting, size_t m, float softening, int checked,
                                 float* out) {
    if (!c) return PNB_E_ARG;
    if ((n && (!affected || !out)) || (m && !affecting))
        return fail(c, PNB_E_ARG, "null pointer with non-zero length");
    if (!(softening >= 0.0f)) return fail(c, PNB_E_ARG, "softening must be >= 0");
    if (n == 0) return PNB_OK;
    if (n > 0x7fffffffu || m > 0x7fffffffu)
        return fail(c, PNB_E_ARG, "brute force supports at most 2^31-1 particles per side");
    if (!c->noalloc_scratch)
        return fail(c, PNB_E_STATE, "no allocation-free scratch on device %d", c->device);
    if (int rc = activate(c)) return rc;
    float4* o = reinterpret_cast<float4*>(out);
    if (m == 0) {
        fill_zero_kernel<<<div_up(n, 256), 256, 0, c->stream>>>(o, n);
        PNB_CHECK_LAUNCH(c);
        return PNB_OK;
    }
    const BfPlan p = plan(c, n, m);
    if (p.splits > 1 && size_t(p.splits) * n > BF_SCRATCH_RECORDS)
        return fail(c, PNB_E_ARG,
                    "the allocation-free brute force holds %zu partial sums; %u affecting ranges "
                    "x %zu affected need %zu",
                    BF_SCRATCH_RECORDS, p.splits, n, size_t(p.splits) * n);
    return bf_launch_with(c, p, reinterpret_cast<const float4*>(affected), n,
                          reinterpret_cast<const float4*>(affecting), m, softening, checked, o,
                          c->noalloc_scratch);
}

int pnb_bf_accel_f32(pnb_ctx* c, const float* affected, size_t n, const float* affecting,
                     size_t m, float softening, int checked, float* out) {
    if (!c) return PNB_E_ARG;
    if ((n && (!affected || !out)) || (m && !affecting))
        return fail(c, PNB_E_ARG, "null pointer with non-zero length");
    if (!(softening >= 0.0f)) return fail(c, PNB_E_ARG, "softening must be >= 0");
    if (n == 0) return PNB_OK;
    if (int rc = activate(c)) return rc;
    void* o;
    if (int rc = upload_sides(c, affected, n, affecting, m, sizeof(float4))) return rc;
    if (int rc = stage_out(c, c->h_out, n * sizeof(float4), &o)) return rc;
    const DevBuf& b = affecting == affected ? c->h_affected : c->h_affecting;
    if (int rc = bf_launch(c, c->h_affected.as<float4>(), n, b.as<float4>(), m, softening, checked,
                           static_cast<float4*>(o)))
        return rc;
    return stage_done(c, out, o, n * sizeof(float4));
}

int pnb_reordered_bf_accel_f32_dev(pnb_ctx* c, const float* particles, size_t n, float softening,
                                   int checked, float* out) {
    if (!c) return PNB_E_ARG;
    if (n && (!particles || !out)) return fail(c, PNB_E_ARG, "null pointer with non-zero length");
    if (!(softening >= 0.0f)) return fail(c, PNB_E_ARG, "softening must be >= 0");
    if (n == 0) return PNB_OK;
    if (int rc = activate(c)) return rc;
    PNB_HIP(c, c->split_tmp.ensure(n * sizeof(float4)));
    uint32_t m = 0;
    const float4* p = reinterpret_cast<const float4*>(particles);
    if (int rc = split_affecting(c, p, n, c->split_tmp.as<float4>(), &m)) return rc;
    return bf_launch(c, p, n, c->split_tmp.as<float4>(), m, softening, checked,
                     reinterpret_cast<float4*>(out));
}

int pnb_reordered_bf_accel_f32(pnb_ctx* c, const float* particles, size_t n, float softening,
                               int checked, float* out) {
    if (!c) return PNB_E_ARG;
    if (n && (!particles || !out)) return fail(c, PNB_E_ARG, "null pointer with non-zero length");
    if (!(softening >= 0.0f)) return fail(c, PNB_E_ARG, "softening must be >= 0");
    if (n == 0) return PNB_OK;
    if (int rc = activate(c)) return rc;
    void* o;
    if (int rc = stage_in(c, c->h_affected, particles, n * sizeof(float4))) return rc;
    if (int rc = stage_out(c, c->h_out, n * sizeof(float4), &o)) return rc;
    if (int rc = pnb_reordered_bf_accel_f32_dev(c, c->h_affected.as<float>(), n, softening,
                                                checked, static_cast<float*>(o)))
        return rc;
    return stage_done(c, out, o, n * sizeof(float4));
}

int pnb_bf_set_tuning(pnb_ctx* c, size_t n_min, int variant, int per_lane, int j_split) {
    if (!c) return PNB_E_ARG;
    if (variant < 0 || variant > 1 ||
        (per_lane != 1 && per_lane != 2 && per_lane != 4 && per_lane != 8) || j_split < 1 ||
        j_split > 64)
        return fail(c, PNB_E_ARG, "invalid brute-force shape");
    if (!c->bf_tune) c->bf_tune = new BfTune();
    auto& v = c->bf_tune->entries;
    v.erase(std::remove_if(v.begin(), v.end(), [&](const BfTuneEntry& e) { return e.n_min == n_min; }),
            v.end());
    v.push_back({n_min, variant, per_lane, j_split});
    return PNB_OK;
}

int pnb_bf_clear_tuning(pnb_ctx* c) {
    if (!c) return PNB_E_ARG;
    if (c->bf_tune) c->bf_tune->entries.clear();
    return PNB_OK;
}

int pnb_direct_f64_dev(pnb_ctx* c, const float* affected, size_t n, const float* affecting,
                       size_t m, double softening, double* out3) {
    if (!c) return PNB_E_ARG;
    if ((n && (!affected || !out3)) || (m && !affecting))
        return fail(c, PNB_E_ARG, "null pointer with non-zero length");
    if (n == 0) return PNB_OK;
    if (n > 0x7fffffffu || m > 0x7fffffffu) return fail(c, PNB_E_ARG, "too many particles");
    if (int rc = activate(c)) return rc;
    direct_f64_kernel<<<unsigned(n), DF_BLOCK, 0, c->stream>>>(
        reinterpret_cast<const float4*>(affected), reinterpret_cast<const float4*>(affecting),
        uint32_t(m), softening * softening, out3);
    PNB_CHECK_LAUNCH(c);
    return PNB_OK;
}

int pnb_bf_accel_f64_dev(pnb_ctx* c, const double* affected, size_t n, const double* affecting,
                         size_t m, double softening, int checked, double* out) {
    if (!c) return PNB_E_ARG;
    if ((n && (!affected || !out)) || (m && !affecting))
        return fail(c, PNB_E_ARG, "null pointer with non-zero length");
    if (!(softening >= 0.0)) return fail(c, PNB_E_ARG, "softening must be >= 0");
    if (n == 0) return PNB_OK;
    if (n > 0x7fffffffu || m > 0x7fffffffu) return fail(c, PNB_E_ARG, "too many particles");
    if (int rc = activate(c)) return rc;
    Bf64Plan p = plan64(cu_count(c), n, m);
    double4* o = reinterpret_cast<double4*>(out);
    double4* dst = o;
    // Inside a caller's capture one range and no scratch: nothing can be allocated there, and a later
    // call that needs more would free the memory that the graph goes on using.
    if (p.splits > 1 && stream_capturing(c)) p = {BF64_WAVES, 1, uint32_t(m)};
    if (p.splits > 1) {
        PNB_HIP(c, c->bf64_partial.ensure(p.splits * n * sizeof(double4)));
        dst = c->bf64_partial.as<double4>();
    }
    const double eps2 = softening * softening;
    const auto pick = [&](auto w) {
        constexpr int W = decltype(w)::value;
        return !checked         ? bf64_kernel<BF64_UNCHECKED, W>
               : eps2 < 1e-300 ? bf64_kernel<BF64_CHECKED, W>
                                : bf64_kernel<BF64_SOFTENED, W>;
    };
    const auto k = p.waves == 1 ? pick(std::integral_constant<int, 1>{})
                                : pick(std::integral_constant<int, BF64_WAVES>{});
    const double4* aff = reinterpret_cast<const double4*>(affected);
    for (size_t i = 0; i < n; i += BF64_SLICE) {  // one launch but for more than 2^28 bodies, never split
        const size_t cnt = std::min(n - i, BF64_SLICE);
        k<<<dim3(div_up(cnt, 64), unsigned(p.splits)), 64 * p.waves, 0, c->stream>>>(
            aff + i, uint32_t(cnt), reinterpret_cast<const double4*>(affecting), uint32_t(m), p.chunk, eps2,
            dst + i);
        PNB_CHECK_LAUNCH(c);
    }
    if (p.splits > 1) {
        bf64_reduce_kernel<<<div_up(n, 64), 64, 0, c->stream>>>(dst, uint32_t(n), uint32_t(p.splits), o);
        PNB_CHECK_LAUNCH(c);
    }
    return PNB_OK;
}

int pnb_bf_accel_f64(pnb_ctx* c, const double* affected, size_t n, const double* affecting,
                     size_t m, double softening, int checked, double* out) {
    if (!c) return PNB_E_ARG;
    if ((n && (!affected || !out)) || (m && !affecting))
        return fail(c, PNB_E_ARG, "null pointer with non-zero length");
    if (n == 0) return PNB_OK;
    if (int rc = activate(c)) return rc;
    void* o;
    if (int rc = upload_sides(c, affected, n, affecting, m, sizeof(double4))) return rc;
    if (int rc = stage_out(c, c->h_out, n * sizeof(double4), &o)) return rc;
    const DevBuf& b = affecting == affected ? c->h_affected : c->h_affecting;
    if (int rc = pnb_bf_accel_f64_dev(c, c->h_affected.as<double>(), n, b.as<double>(), m, softening,
                                      checked, static_cast<double*>(o)))
        return rc;
    return stage_done(c, out, o, n * sizeof(double4));
}

}  // extern "C"
