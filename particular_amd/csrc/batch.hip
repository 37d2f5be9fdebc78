// Batched ensemble: many independent systems of uneven sizes stepped together.
//
// Every system is its own Between(system, system) brute force (all bodies massive within a
// system), integrated with kick-drift-kick leapfrog in FP64 like the single-system loop. The force
// pass of a step is ONE persistent launch: a few workgroups per CU that pull work items (system,
// tiles of 64 affected bodies) from a queue until it is empty, the wavefronts of a workgroup
// sharing an item's affecting bodies (coop_sum), which they read with wave-uniform addresses
// (scalar loads). Items are ordered by decreasing cost (system size x bodies per lane), so large
// systems start first and small ones fill the tail. Tuning entries that ask for more than one
// body per lane take the queue by single wavefronts, which need no barriers. The per-lane
// arithmetic and summation order are those of the brute-force kernel either way (FP32 tiles of 256
// bodies, Kahan across tiles). A step is enqueue-only and can be captured into a hipGraph (the queue
// counter is cleared by a kernel, not a memset).
#include "bf_common.hpp"
#include "pnb_internal.hpp"

#include <algorithm>
#include <vector>

namespace pnb {

constexpr int BT_TILE = 256;

struct BatchItem {
    uint32_t off;  // first particle of the system
    uint32_t n;    // system size
    uint32_t i0;   // first affected body of the tile, relative to the system
    uint32_t r;    // affected bodies per lane (1, 2, 4 or 8)
};

struct BatchState {
    size_t total = 0, systems = 0;
    float softening = 0.f;
    int checked = 1;
    std::vector<int64_t> offsets;
    std::vector<std::pair<size_t, int>> tuning;  // (n_min, per_lane)
    bool items_dirty = true;
    int waves = 0;  // wavefronts of a workgroup that shares an item (bt_coop_kernel); 0: items for wavefronts
    size_t n_items = 0;
    unsigned long long interactions = 0;
    DevBuf x, v, shadow, acc, items, queue, stage;
    hipGraphExec_t exec = nullptr;
    hipGraph_t graph = nullptr;
    size_t graph_steps = 0;
    double graph_dt = 0.0;
    hipStream_t graph_stream = nullptr;
    void drop_graph() {
        if (exec) hipGraphExecDestroy(exec);
        if (graph) hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
        graph_steps = 0;
    }
};

void batch_free(BatchState* s) {
    if (!s) return;
    s->drop_graph();
    for (DevBuf* b : {&s->x, &s->v, &s->shadow, &s->acc, &s->items, &s->queue, &s->stage}) b->release();
    delete s;
}

template <int R, bool MASK>
__device__ __forceinline__ void bt_tile(const float4* __restrict__ sh, const BatchItem w, float eps2,
                                        float4* __restrict__ acc) {
    const uint32_t lane = threadIdx.x & 63;
    const float4* sys = sh + w.off;
    float xi[R], yi[R], zi[R], ax[R], ay[R], az[R], cx[R], cy[R], cz[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t i = w.i0 + r * 64 + lane;
        const float4 p = sys[i < w.n ? i : w.n - 1];
        xi[r] = p.x; yi[r] = p.y; zi[r] = p.z;
        ax[r] = ay[r] = az[r] = cx[r] = cy[r] = cz[r] = 0.f;
    }
    for (uint32_t j0 = 0; j0 < w.n; j0 += BT_TILE) {
        const uint32_t cnt = min(uint32_t(BT_TILE), w.n - j0);
        float px[R], py[R], pz[R];
#pragma unroll
        for (int r = 0; r < R; ++r) px[r] = py[r] = pz[r] = 0.f;
        for (uint32_t j = 0; j < cnt; ++j) {
            bf_body<R, MASK>(sys[j0 + j], xi, yi, zi, eps2, px, py, pz);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            kahan_add(ax[r], cx[r], px[r]);
            kahan_add(ay[r], cy[r], py[r]);
            kahan_add(az[r], cz[r], pz[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t i = w.i0 + r * 64 + lane;
        if (i < w.n) acc[w.off + i] = make_float4(ax[r], ay[r], az[r], 0.f);
    }
}

template <bool MASK>
__global__ __launch_bounds__(256) void bt_force_kernel(const BatchItem* __restrict__ items,
                                                       uint32_t n_items,
                                                       uint32_t* __restrict__ queue,
                                                       const float4* __restrict__ sh, float eps2,
                                                       float4* __restrict__ acc) {
    const uint32_t lane = threadIdx.x & 63;
    while (true) {
        uint32_t it = 0;
        if (lane == 0) it = atomicAdd(queue, 1u);
        it = __builtin_amdgcn_readfirstlane(it);
        if (it >= n_items) break;
        const BatchItem w = items[it];
        switch (w.r) {
            case 8: bt_tile<8, MASK>(sh, w, eps2, acc); break;
            case 4: bt_tile<4, MASK>(sh, w, eps2, acc); break;
            case 2: bt_tile<2, MASK>(sh, w, eps2, acc); break;
            default: bt_tile<1, MASK>(sh, w, eps2, acc); break;
        }
    }
}

// The same queue taken by workgroups, one body per lane: W wavefronts share an item, J of them its
// affecting bodies (coop_sum; the same tiles summed in the same order, so the same bits) and, in
// systems with fewer than W tiles of affecting bodies, the others neighbouring affected tiles: an item
// covers W / J tiles of 64 bodies.
template <int W>
static __host__ __device__ inline int bt_share(uint32_t n) {  // wavefronts per affected tile
    int j = 1;
    while (j < W && uint32_t(j) * BT_TILE < n) j <<= 1;
    return j;
}

template <int W, bool MASK>
__global__ __launch_bounds__(64 * W) void bt_coop_kernel(const BatchItem* __restrict__ items,
                                                         uint32_t n_items,
                                                         uint32_t* __restrict__ queue,
                                                         const float4* __restrict__ sh, float eps2,
                                                         float4* __restrict__ acc) {
    __shared__ CoopLds<1, W> lds;
    __shared__ uint32_t next;
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    asm volatile("" : "+v"(eps2));  // a scalar operand halves an instruction's rate
    while (true) {
        if (threadIdx.x == 0) next = atomicAdd(queue, 1u);
        __syncthreads();
        const uint32_t it = __builtin_amdgcn_readfirstlane(next);
        __syncthreads();  // everyone has read it before the next round's write
        if (it >= n_items) break;
        const BatchItem w = items[it];
        const float4* sys = sh + w.off;
        const int J = bt_share<W>(w.n);
        const uint32_t i0 = w.i0 + uint32_t(wave / J) * 64, i = i0 + (threadIdx.x & 63);
        const float4 p = sys[i < w.n ? i : w.n - 1];
        const float xi[1] = {p.x}, yi[1] = {p.y}, zi[1] = {p.z};
        float ax[1], ay[1], az[1];
        coop_sum<1, MASK, false, BT_TILE, W>(lds, sys, 0, w.n, J, wave, i0 < w.n, eps2, 0, xi, yi, zi, ax,
                                             ay, az);
        if (wave % J == 0 && i < w.n) acc[w.off + i] = make_float4(ax[0], ay[0], az[0], 0.f);
    }
}

__global__ void bt_queue_reset_kernel(uint32_t* q) { *q = 0u; }

__global__ void bt_pack_kernel(const double* __restrict__ x3, const double* __restrict__ v3,
                               const float* __restrict__ mu, size_t n, double4* __restrict__ x,
                               double4* __restrict__ v, float4* __restrict__ sh) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    x[i] = make_double4(x3[3 * i], x3[3 * i + 1], x3[3 * i + 2], 0.0);
    v[i] = make_double4(v3[3 * i], v3[3 * i + 1], v3[3 * i + 2], 0.0);
    sh[i] = make_float4(float(x3[3 * i]), float(x3[3 * i + 1]), float(x3[3 * i + 2]), mu[i]);
}

// A step's drift with the half kick before it and, TWO, the previous step's last half kick (the
// same two additions to v, from the same a); also resets the queue for the step's force launch.
template <bool TWO>
__global__ void bt_kick_drift_kernel(double4* __restrict__ x, double4* __restrict__ v,
                                     const float4* __restrict__ acc, float4* __restrict__ sh,
                                     size_t n, double h, double dt, uint32_t* __restrict__ queue) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (i == 0) *queue = 0u;
    const float4 a = acc[i];
    double4 vi = v[i];
    vi.x += double(a.x) * h;
    vi.y += double(a.y) * h;
    vi.z += double(a.z) * h;
    if (TWO) {
        vi.x += double(a.x) * h;
        vi.y += double(a.y) * h;
        vi.z += double(a.z) * h;
    }
    double4 xi = x[i];
    xi.x += vi.x * dt;
    xi.y += vi.y * dt;
    xi.z += vi.z * dt;
    v[i] = vi;
    x[i] = xi;
    sh[i] = make_float4(float(xi.x), float(xi.y), float(xi.z), sh[i].w);
}

__global__ void bt_kick_kernel(double4* __restrict__ v, const float4* __restrict__ acc, size_t n,
                               double h) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 a = acc[i];
    double4 vi = v[i];
    vi.x += double(a.x) * h;
    vi.y += double(a.y) * h;
    vi.z += double(a.z) * h;
    v[i] = vi;
}

__global__ void bt_unpack_kernel(const double4* __restrict__ x, const double4* __restrict__ v,
                                 size_t n, double* __restrict__ out) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double4 a = x[i], b = v[i];
    out[3 * i] = a.x; out[3 * i + 1] = a.y; out[3 * i + 2] = a.z;
    out[3 * (n + i)] = b.x; out[3 * (n + i) + 1] = b.y; out[3 * (n + i) + 2] = b.z;
}

// A tuning entry's bodies per lane for systems of n bodies, 0 without one.
static int tuned_per_lane(const BatchState* s, size_t n) {
    int r = 0;
    size_t best = 0;
    for (const auto& t : s->tuning)
        if (t.first <= n && (r == 0 || t.first >= best)) {
            best = t.first;
            r = t.second;
        }
    return r;
}

// The queue's items. Untuned, and tuned to one body per lane throughout, workgroups share them, one body
// per lane; otherwise an item is 64 bodies times its system's tuning entry (one without an entry).
static int build_items(pnb_ctx* c, BatchState* s) {
    std::vector<BatchItem> items;
    s->interactions = 0;
    // Workgroups share the items unless a tuning entry asks for more bodies per lane, of eight
    // wavefronts, or of sixteen while eight make at most two items per CU. Eight steps and the
    // state's read, wavefronts with four bodies per lane / workgroups of 8 / of 16 (ms): one system of
    // 16,384 bodies 23.9 / 1.44 / 0.92; four 25.6 / 2.88 / 3.41; sizes log-uniform in 64 .. 500: 16
    // systems 1.03 / 0.25 / 0.23, 2,000 3.18 / 2.23 / 2.39; in 64 .. 16,384: 128 systems 30.6 / 8.64 /
    // 10.9, 1,024 79.2 / 67.9 / 86.7. Two bodies per lane in workgroups of 8: 2.41, 4.24, 0.29, 2.27,
    // 9.39, 70.5 (larger items leave a longer tail).
    s->waves = 8;
    for (size_t k = 0; k < s->systems && s->waves; ++k)
        if (tuned_per_lane(s, size_t(s->offsets[k + 1] - s->offsets[k])) > 1) s->waves = 0;
    if (s->waves) {
        size_t count = 0;
        for (size_t k = 0; k < s->systems; ++k) {
            const uint32_t n = uint32_t(s->offsets[k + 1] - s->offsets[k]);
            count += div_up(n, 64 * (8 / bt_share<8>(n)));
        }
        if (count <= 2 * size_t(std::max(1, c->cu_count))) s->waves = 16;
    }
    for (size_t k = 0; k < s->systems; ++k) {
        const uint32_t off = uint32_t(s->offsets[k]);
        const uint32_t n = uint32_t(s->offsets[k + 1] - s->offsets[k]);
        if (n == 0) continue;
        s->interactions += (unsigned long long)n * n;
        const uint32_t r = uint32_t(std::max(1, tuned_per_lane(s, n)));
        const uint32_t tile = s->waves == 16  ? 64 * (16 / bt_share<16>(n))
                              : s->waves == 8 ? 64 * (8 / bt_share<8>(n))
                                              : 64 * r;
        for (uint32_t i0 = 0; i0 < n; i0 += tile) items.push_back({off, n, i0, r});
    }
    std::stable_sort(items.begin(), items.end(), [](const BatchItem& a, const BatchItem& b) {
        return uint64_t(a.n) * a.r > uint64_t(b.n) * b.r;
    });
    s->n_items = items.size();
    PNB_HIP(c, s->items.ensure(std::max<size_t>(1, items.size()) * sizeof(BatchItem)));
    if (!items.empty())
        PNB_HIP(c, hipMemcpyAsync(s->items.ptr, items.data(), items.size() * sizeof(BatchItem),
                                  hipMemcpyHostToDevice, c->stream));
    PNB_HIP(c, hipStreamSynchronize(c->stream));
    s->items_dirty = false;
    return PNB_OK;
}

// The queue has to be 0 (bt_queue_reset_kernel, bt_kick_drift_kernel).
static int force(pnb_ctx* c, BatchState* s) {
    const bool mask = s->checked && s->softening == 0.0f;
    const float eps2 = s->softening * s->softening;
    auto k = s->waves == 0   ? (mask ? bt_force_kernel<true> : bt_force_kernel<false>)
             : s->waves == 8 ? (mask ? bt_coop_kernel<8, true> : bt_coop_kernel<8, false>)
                             : (mask ? bt_coop_kernel<16, true> : bt_coop_kernel<16, false>);
    const unsigned block = s->waves ? 64 * s->waves : 256;
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k, int(block), 0) != hipSuccess || occ < 1) occ = 2;
    const unsigned grid = unsigned(std::max(1, c->cu_count) * occ);
    return timed(c, PNB_PROF_BATCH, [&]() -> int {
        k<<<grid, block, 0, c->stream>>>(s->items.as<BatchItem>(), uint32_t(s->n_items),
                                         s->queue.as<uint32_t>(), s->shadow.as<float4>(), eps2,
                                         s->acc.as<float4>());
        PNB_CHECK_LAUNCH(c);
        return PNB_OK;
    });
}

static int enqueue(pnb_ctx* c, BatchState* s, size_t steps, double dt) {
    const unsigned g = div_up(s->total, 256);
    const double h = 0.5 * dt;
    for (size_t k = 0; k < steps; ++k) {
        (k == 0 ? bt_kick_drift_kernel<false> : bt_kick_drift_kernel<true>)<<<g, 256, 0, c->stream>>>(
            s->x.as<double4>(), s->v.as<double4>(), s->acc.as<float4>(), s->shadow.as<float4>(),
            s->total, h, dt, s->queue.as<uint32_t>());
        PNB_CHECK_LAUNCH(c);
        if (int rc = force(c, s)) return rc;
    }
    if (steps) {
        bt_kick_kernel<<<g, 256, 0, c->stream>>>(s->v.as<double4>(), s->acc.as<float4>(), s->total, h);
        PNB_CHECK_LAUNCH(c);
    }
    return PNB_OK;
}

}  // namespace pnb

using namespace pnb;

extern "C" {

int pnb_batch_set_tuning(pnb_ctx* c, size_t n_min, int per_lane) {
    if (!c) return PNB_E_ARG;
    if (per_lane != 1 && per_lane != 2 && per_lane != 4 && per_lane != 8)
        return fail(c, PNB_E_ARG, "per_lane must be 1, 2, 4 or 8");
    if (!c->batch) c->batch = new BatchState();
    auto& t = c->batch->tuning;
    t.erase(std::remove_if(t.begin(), t.end(), [&](const std::pair<size_t, int>& e) { return e.first == n_min; }),
            t.end());
    t.emplace_back(n_min, per_lane);
    c->batch->items_dirty = true;
    c->batch->drop_graph();
    return PNB_OK;
}

int pnb_batch_init(pnb_ctx* c, const double* pos3, const double* vel3, const float* mu,
                   const int64_t* offsets, size_t num_systems, float softening, int checked) {
    if (!c) return PNB_E_ARG;
    if (!offsets || num_systems == 0) return fail(c, PNB_E_ARG, "no systems");
    if (!(softening >= 0.0f)) return fail(c, PNB_E_ARG, "softening must be >= 0");
    for (size_t k = 0; k < num_systems; ++k)
        if (offsets[k + 1] < offsets[k] || offsets[0] != 0)
            return fail(c, PNB_E_ARG, "offsets must start at 0 and be non-decreasing");
    const size_t total = size_t(offsets[num_systems]);
    if (total == 0 || !pos3 || !vel3 || !mu) return fail(c, PNB_E_ARG, "no particles");
    if (total > 0x7fffffffu) return fail(c, PNB_E_ARG, "too many particles");
    if (int rc = activate(c)) return rc;
    if (!c->batch) c->batch = new BatchState();
    BatchState* s = c->batch;
    s->drop_graph();
    s->total = total;
    s->systems = num_systems;
    s->softening = softening;
    s->checked = checked;
    s->offsets.assign(offsets, offsets + num_systems + 1);
    PNB_HIP(c, s->x.ensure(total * sizeof(double4)));
    PNB_HIP(c, s->v.ensure(total * sizeof(double4)));
    PNB_HIP(c, s->shadow.ensure(total * sizeof(float4)));
    PNB_HIP(c, s->acc.ensure(total * sizeof(float4)));
    PNB_HIP(c, s->queue.ensure(sizeof(uint32_t)));
    PNB_HIP(c, s->stage.ensure(total * (6 * sizeof(double) + sizeof(float))));
    double* dx = s->stage.as<double>();
    double* dv = dx + 3 * total;
    float* dm = reinterpret_cast<float*>(dv + 3 * total);
    PNB_HIP(c, hipMemcpyAsync(dx, pos3, 3 * total * sizeof(double), hipMemcpyHostToDevice, c->stream));
    PNB_HIP(c, hipMemcpyAsync(dv, vel3, 3 * total * sizeof(double), hipMemcpyHostToDevice, c->stream));
    PNB_HIP(c, hipMemcpyAsync(dm, mu, total * sizeof(float), hipMemcpyHostToDevice, c->stream));
    bt_pack_kernel<<<div_up(total, 256), 256, 0, c->stream>>>(dx, dv, dm, total, s->x.as<double4>(),
                                                              s->v.as<double4>(), s->shadow.as<float4>());
    PNB_CHECK_LAUNCH(c);
    if (int rc = build_items(c, s)) return rc;
    bt_queue_reset_kernel<<<1, 1, 0, c->stream>>>(s->queue.as<uint32_t>());
    PNB_CHECK_LAUNCH(c);
    if (int rc = force(c, s)) return rc;
    PNB_HIP(c, hipStreamSynchronize(c->stream));
    return PNB_OK;
}

int pnb_batch_run(pnb_ctx* c, size_t steps, double dt, int use_graph) {
    if (!c) return PNB_E_ARG;
    BatchState* s = c->batch;
    if (!s || s->total == 0) return fail(c, PNB_E_STATE, "pnb_batch_init has not been called");
    if (steps == 0) return PNB_OK;
    if (int rc = activate(c)) return rc;
    if (s->items_dirty)
        if (int rc = build_items(c, s)) return rc;
    if (!use_graph) return enqueue(c, s, steps, dt);
    if (!c->stream) return fail(c, PNB_E_STATE, "graph capture needs a non-null stream");
    if (!s->exec || s->graph_steps != steps || s->graph_dt != dt || s->graph_stream != c->stream) {
        s->drop_graph();
        PNB_HIP(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        c->capturing = true;
        int rc = enqueue(c, s, steps, dt);
        c->capturing = false;
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(c->stream, &g);
        if (rc) {
            if (g) hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess) return hip_fail(c, e, "hipStreamEndCapture", __FILE__, __LINE__);
        s->graph = g;
        PNB_HIP(c, hipGraphInstantiate(&s->exec, g, nullptr, nullptr, 0));
        s->graph_steps = steps;
        s->graph_dt = dt;
        s->graph_stream = c->stream;
    }
    PNB_HIP(c, hipGraphLaunch(s->exec, c->stream));
    return PNB_OK;
}

int pnb_batch_read(pnb_ctx* c, double* pos3, double* vel3, float* acc4) {
    if (!c) return PNB_E_ARG;
    BatchState* s = c->batch;
    if (!s || s->total == 0) return fail(c, PNB_E_STATE, "pnb_batch_init has not been called");
    if (int rc = activate(c)) return rc;
    const size_t n = s->total;
    double* st = s->stage.as<double>();
    bt_unpack_kernel<<<div_up(n, 256), 256, 0, c->stream>>>(s->x.as<double4>(), s->v.as<double4>(), n, st);
    PNB_CHECK_LAUNCH(c);
    return stage_fetch(c, {{pos3, st, 24 * n}, {vel3, st + 3 * n, 24 * n}, {acc4, s->acc.ptr, 16 * n}});
}

int pnb_batch_info(pnb_ctx* c, size_t* particles, size_t* items,
                   unsigned long long* interactions_per_step) {
    if (!c) return PNB_E_ARG;
    BatchState* s = c->batch;
    if (!s || s->total == 0) return fail(c, PNB_E_STATE, "pnb_batch_init has not been called");
    if (particles) *particles = s->total;
    if (items) *items = s->n_items;
    if (interactions_per_step) *interactions_per_step = s->interactions;
    return PNB_OK;
}

}  // extern "C"
