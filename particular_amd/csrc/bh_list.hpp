// Barnes-Hut walk over batches of nodes, included by bh.hip (which defines the records).
//
// The stackless walk (bh_walk_kernel) visits one node per step, and every step waits for a record
// whose address the previous step decided: with few wavefronts per CU its time is that latency
// times the steps (1,100 steps of 0.17 us for 4,096 bodies). Here a wavefront keeps the nodes still
// to be visited as a sequence in LDS, in pre-order, and handles its first 64 at once, one node per
// lane: all 64 records arrive together, nodes are decided for the whole group of particles from its
// bounding box, and an opened node is replaced in place by its children (from a child table
// the bottom-up pass writes), so some 15-60 rounds replace 400-2,200 steps. Nodes at the front of
// the sequence that nobody opens are then summed by the group's particles, in sequence order: every
// particle adds exactly the nodes of its own pre-order traversal, in that order, with the
// same arithmetic as the stackless walk, so the plain walk's results are the same bits.
//
// Decisions are the reference's exactly: f32 rounding is monotonic, so with the box's nearest and
// farthest coordinate differences in place of a particle's the criterion's rounded value bounds
// every particle's from below and above; nodes the bounds do not decide are tested particle by
// particle (the lanes of a ballot), which splits the group: the particles that accept the node
// sum it, its children carry the mask of those that opened it.
//
// L particles per wavefront (4 or 16): Q = 64 / L nodes are tested or evaluated at once, each by
// its own L lanes; the terms then go through LDS to lanes that hold one component of one
// particle's sum each and add them in order.
#pragma once

// Sequence entries per wavefront. A sequence that would outgrow them expands fewer nodes at a time;
// when not even the first fits, its subtree is walked node by node.
constexpr int LIST_CAP = 1024;
constexpr uint32_t LIST_FINAL = 0x80000000u;  // entry state: summed when it reaches the front
constexpr uint32_t LIST_NODE = (1u << 27) - 1;  // trees of 2^27 nodes or more are not walked here

template <int L>
struct ListEntry;
template <>
struct ListEntry<16> {  // node | final, mask
    uint2 e[LIST_CAP];
    __device__ void put(int at, uint32_t k, uint32_t m) { e[at] = make_uint2(k, m); }
    __device__ void get(int at, uint32_t& k, uint32_t& m) const { k = e[at].x; m = e[at].y; }
};
template <>
struct ListEntry<4> {  // node | mask << 27 | final
    uint32_t e[LIST_CAP];
    __device__ void put(int at, uint32_t k, uint32_t m) { e[at] = k | (m << 27); }
    __device__ void get(int at, uint32_t& k, uint32_t& m) const {
        const uint32_t v = e[at];
        k = v & (LIST_FINAL | LIST_NODE);
        m = (v >> 27) & 15u;
    }
};

template <int L, int U>
struct ListLds {
    ListEntry<L> seq;     // the sequence: its front is the last entry
    float4 rec[64];       // the window's records: centre of mass and mass
    float w2[64];
    float4 ev[64];        // the nodes to sum, compact
    uint32_t ev_mask[64];
    uint32_t pos[64];     // window positions of the nodes to test; the summed nodes' indices
    uint32_t res[64];     // their accepting masks | opening masks << 16
    float4 term[U][64];   // U Q nodes' terms
};
// A term that is not to be added: a signaling NaN, which no arithmetic result is.
constexpr uint32_t LIST_SKIP = 0x7fa00001u;

// Inclusive sum over the wavefront's lanes (DPP shifts within rows, then row broadcasts).
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
    return v;
}

// The learned correction of an accepted internal node added to (vx, vy, vz), and its factor of
// the direction term: the formulas of bh_walk_kernel. oh: MODE WALK_OCT's entry.
template <bool OCT>
__device__ __forceinline__ float corrected_terms(float dx, float dy, float dz, float s, float inv2,
                                                 float w2, uint32_t h0, uint32_t h1, uint32_t h2,
                                                 const float* o, bool octupole, float& vx, float& vy,
                                                 float& vz) {
    const float q[6] = {half_lo(h0), half_hi(h0), half_lo(h1), half_hi(h1), half_lo(h2), half_hi(h2)};
    const float qx = fmaf(q[4], dz, fmaf(q[3], dy, fmaf(q[0], dx, 0.f)));
    const float qy = fmaf(q[5], dz, fmaf(q[1], dy, fmaf(q[3], dx, 0.f)));
    const float qz = fmaf(q[2], dz, fmaf(q[5], dy, fmaf(q[4], dx, 0.f)));
    const float dqd = dx * qx + dy * qy + dz * qz;
    const float s5 = s * (w2 * inv2);
    const float s5u = s5 * inv2;
    float st = fmaf(s5u, 2.5f * dqd, s);
    vx = fmaf(-s5, qx, vx);
    vy = fmaf(-s5, qy, vy);
    vz = fmaf(-s5, qz, vz);
    if (OCT && octupole) {
        const float ta = dx * dx - dz * dz, tb = dy * dy - dz * dz;
        const float pxy = dx * dy, pxz = dx * dz, pyz = dy * dz;
        const float p2xy = pxy + pxy;
        const float fx = fmaf(o[0], ta, fmaf(o[1], tb, fmaf(o[2], p2xy, fmaf(o[6], pxz, o[7] * pyz))));
        const float fy = fmaf(o[2], ta, fmaf(o[3], tb, fmaf(o[1], p2xy, fmaf(o[7], pxz, o[8] * pyz))));
        const float fz = fmaf(o[4], ta, fmaf(o[5], tb, fmaf(o[7], pxy, fmaf(o[9], pxz, o[10] * pyz))));
        const float gdd = dx * fx + dy * fy + dz * fz;
        st = fmaf(-7.f * s5u * inv2, gdd, st);
        const float s7x3 = 3.f * s5u;
        vx = fmaf(s7x3, fx, vx);
        vy = fmaf(s7x3, fy, vy);
        vz = fmaf(s7x3, fz, vz);
    }
    return st;
}

// One workgroup (a wavefront) per L consecutive particles in walk order. kids: per internal node its
// children's indices, their number less one in the first one's top bits. dd: as in bh_walk_kernel.
template <int MODE, int L>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void bh_list_kernel(const NodeRec* __restrict__ nodes,
                                                     const uint4* __restrict__ kids, uint32_t total,
                                                     const float4* __restrict__ pts,
                                                     const uint32_t* __restrict__ perm, uint32_t n,
                                                     float theta2, float eps2,
                                                     float4* __restrict__ out,
                                                     BhInfo* __restrict__ info,
                                                     const QuadH* __restrict__ qh,
                                                     const OctH* __restrict__ oh, int dd) {
    constexpr bool QUAD = MODE == WALK_QUAD || MODE == WALK_OCT;
    constexpr bool OCT = MODE == WALK_OCT;
    constexpr int Q = 64 / L;  // nodes evaluated at once
    constexpr int U = QUAD || L == 16 ? 2 : 1;  // batches of Q nodes summed together
    constexpr uint32_t FULL = (1u << L) - 1;
    __shared__ ListLds<L, QUAD ? 1 : U> lds;
    const int lane = threadIdx.x, sub = lane & (L - 1), slot = lane / L;
    const int comp = (lane / L) & 3, row = lane & ~(L - 1);
    const uint32_t i = blockIdx.x * L + sub;
    const bool valid = i < n;
    if (dd) {
        if (info->flags) {
            if (valid && slot == 0) out[perm ? perm[i] : i] = make_float4(NAN, NAN, NAN, 0.f);
            return;
        }
        total = info->total;
    }
    const float4 p = pts[valid ? i : n - 1];
    // the group's box (lanes without a particle hold a copy of the last one)
    float lx = p.x, ly = p.y, lz = p.z, hx = p.x, hy = p.y, hz = p.z;
#pragma unroll
    for (int o = 1; o < L; o <<= 1) {
        lx = fminf(lx, __shfl_xor(lx, o, 64));
        ly = fminf(ly, __shfl_xor(ly, o, 64));
        lz = fminf(lz, __shfl_xor(lz, o, 64));
        hx = fmaxf(hx, __shfl_xor(hx, o, 64));
        hy = fmaxf(hy, __shfl_xor(hy, o, 64));
        hz = fmaxf(hz, __shfl_xor(hz, o, 64));
    }
    const uint64_t valid_all = __builtin_amdgcn_ballot_w64(valid);
    const uint32_t everyone = uint32_t(valid_all) & FULL;
    const uint64_t below = (uint64_t(1) << lane) - 1;

    // plain: component `comp` of particle `sub` in (ax, cx), in 4 L lanes (the others hold copies;
    // component 3 is not used); corrected: the slot's share of all three.
    float ax = 0.f, ay = 0.f, az = 0.f, cx = 0.f, cy = 0.f, cz = 0.f;
    float px = 0.f, py = 0.f, pz = 0.f;  // corrected: partial sums
    uint32_t steps = 0, accepted = 0;    // wave-uniform

    // Sums U x Q nodes, in order, Q at a time (one per slot): com and mass in c, internal width^2 (or
    // < 0) in w2, index k; take: this lane's particle accepts it. U independent terms per lane keep
    // a lone wavefront issuing (one at a time took 380 cycles per node).
    auto add_terms = [&](auto u_const, const auto& c, const auto& w2, const auto& k, const auto& take) {
        constexpr int U = decltype(u_const)::value;  // at most the kernel's
        float dx[U], dy[U], dz[U], inv[U], s[U];
        uint64_t act[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            dx[u] = sub_rn(c[u].x, p.x);
            dy[u] = sub_rn(c[u].y, p.y);
            dz[u] = sub_rn(c[u].z, p.z);
            const float d2 = norm2_ref(dx[u], dy[u], dz[u]);
            act[u] = __builtin_amdgcn_ballot_w64(take[u]) & __builtin_amdgcn_ballot_w64(d2 != 0.0f);
            inv[u] = __builtin_amdgcn_rsqf(add_rn(d2, eps2));
            s[u] = (c[u].w * inv[u]) * (inv[u] * inv[u]);
            accepted += uint32_t(__popcll(act[u]));
        }
        if constexpr (QUAD) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (!__builtin_amdgcn_inverse_ballot_w64(act[u])) continue;
                float st = s[u];
                if (w2[u] >= 0.0f) {
                    if constexpr (OCT) {
                        const OctH oe = oh[k[u]];
                        const uint32_t* hq = reinterpret_cast<const uint32_t*>(oe.q);
                        st = corrected_terms<true>(dx[u], dy[u], dz[u], s[u], inv[u] * inv[u], w2[u], hq[0],
                                                   hq[1], hq[2], oe.o, oe.flag != 0, px, py, pz);
                    } else {
                        const uint4 h = *reinterpret_cast<const uint4*>(qh + k[u]);
                        st = corrected_terms<false>(dx[u], dy[u], dz[u], s[u], inv[u] * inv[u], w2[u], h.x,
                                                    h.y, h.z, nullptr, false, px, py, pz);
                    }
                }
                px = fmaf(dx[u], st, px);
                py = fmaf(dy[u], st, py);
                pz = fmaf(dz[u], st, pz);
            }
            steps += U;
            if ((steps & (PART_STEPS - 1)) < U) fold_partial(ax, ay, az, cx, cy, cz, px, py, pz);
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u)
                lds.term[u][lane] =
                    make_float4(dx[u], dy[u], dz[u],
                                __builtin_amdgcn_inverse_ballot_w64(act[u]) ? s[u]
                                                                            : __uint_as_float(LIST_SKIP));
            wave_lds_sync();
            const float* t4 = reinterpret_cast<const float*>(&lds.term[0][sub]);
            float d[U * Q], m[U * Q];
#pragma unroll
            for (int q = 0; q < U * Q; ++q) {
                d[q] = t4[q * L * 4 + comp];
                m[q] = t4[q * L * 4 + 3];
            }
#pragma unroll
            for (int q = 0; q < U * Q; ++q) {
                const bool add = __float_as_uint(m[q]) != LIST_SKIP;
                const float y = fmaf(d[q], m[q], -cx);
                const float t = ax + y;
                const float e = (t - ax) - y;
                cx = add ? e : cx;
                ax = add ? t : ax;
            }
            wave_lds_sync();
            steps += U * Q;
        }
    };

    int size = 0;  // entries of the sequence
    if (total > 0) {
        if (lane == 0) lds.seq.put(0, 0u, everyone);
        size = 1;
    }
    wave_lds_sync();
    // The window: the sequence's first entries, one per lane, with their records and children. The
    // next one is requested before the front is summed, which hides its latency.
    int w = 0;
    bool have = false, fin = false;
    uint32_t k = 0, mine = 0;
    NodeRec r{};
    uint4 ka = make_uint4(0, 0, 0, 0), kb = ka;
    auto load_window = [&]() {
        w = min(64, size);
        have = lane < w;
        mine = 0;
        fin = false;
        if (have) {
            lds.seq.get(size - 1 - lane, k, mine);
            fin = (k & LIST_FINAL) != 0;
            k &= LIST_NODE;
            r = nodes[k];
            if (!fin) {
                ka = kids[2 * size_t(k)];
                kb = kids[2 * size_t(k) + 1];
            }
        }
    };
    load_window();
    while (size > 0) {
        lds.rec[lane] = make_float4(r.cx, r.cy, r.cz, r.mass);
        lds.w2[lane] = r.w2;
        // decided by the box: nobody opens it, or everybody does
        const float nx = fmaxf(0.f, fmaxf(sub_rn(lx, r.cx), sub_rn(r.cx, hx)));
        const float ny = fmaxf(0.f, fmaxf(sub_rn(ly, r.cy), sub_rn(r.cy, hy)));
        const float nz = fmaxf(0.f, fmaxf(sub_rn(lz, r.cz), sub_rn(r.cz, hz)));
        const float fx = fmaxf(sub_rn(r.cx, lx), sub_rn(hx, r.cx));
        const float fy = fmaxf(sub_rn(r.cy, ly), sub_rn(hy, r.cy));
        const float fz = fmaxf(sub_rn(r.cz, lz), sub_rn(hz, r.cz));
        const float near2 = norm2_ref(nx, ny, nz), far2 = norm2_ref(fx, fy, fz);
        const bool leaf = r.w2 < 0.0f;
        uint32_t acc = 0, open = 0;  // the particles that sum this node, and those that need its children
        bool mixed = false;
        if (have) {
            if (fin || leaf || !(mul_rn(theta2, near2) < r.w2)) acc = mine;
            else if (near2 > 0.0f && mul_rn(theta2, far2) < r.w2) open = mine;
            else mixed = true;
        }
        const uint64_t todo = __builtin_amdgcn_ballot_w64(mixed);
        if (todo) {  // particle by particle, Q nodes at a time
            const int count = __popcll(todo);
            if (mixed) lds.pos[__popcll(todo & below)] = uint32_t(lane);
            wave_lds_sync();
            for (int t0 = 0; t0 < count; t0 += 2 * Q) {
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int t = t0 + u * Q + slot;
                    const uint32_t at = lds.pos[t < count ? t : 0];
                    const float4 c = lds.rec[at];
                    const float d2 = norm2_ref(sub_rn(c.x, p.x), sub_rn(c.y, p.y), sub_rn(c.z, p.z));
                    const uint64_t far = __builtin_amdgcn_ballot_w64(d2 != 0.0f);
                    const uint64_t crit =
                        __builtin_amdgcn_fcmpf(mul_rn(theta2, d2), lds.w2[at], 4 /*olt*/);
                    if (t < count && sub == 0)
                        lds.res[at] = (uint32_t((far & ~crit) >> row) & FULL) |
                                      ((uint32_t((far & crit) >> row) & FULL) << 16);
                }
            }
            wave_lds_sync();
            if (mixed) {
                const uint32_t both = lds.res[lane];
                acc = both & mine;
                open = (both >> 16) & mine;
            }
        }
        // what replaces each entry: itself as final (acc), then its children (open)
        int nch = open ? 1 + int(ka.x >> 28) : 0;
        ka.x &= LIST_NODE;
        int cnt = (acc ? 1 : 0) + nch;
        int incl = wave_scan(cnt);
        bool pending = false;  // no room to replace it yet: it stays as it was
        const uint64_t over =
            __builtin_amdgcn_ballot_w64(have && size - w + incl + (w - 1 - lane) > LIST_CAP);
        if (over) {
            pending = have && !fin && lane >= __builtin_ctzll(over);
            if (pending) {
                nch = 0;
                cnt = 1;
            }
            incl = wave_scan(cnt);
        }
        // the front: every entry up to the first that still has children to come
        const uint64_t waits = __builtin_amdgcn_ballot_w64(have && (nch > 0 || pending));
        const int first = waits ? __builtin_ctzll(waits) : 64;
        const bool emit = acc && !pending && lane <= first;
        const uint64_t emits = __builtin_amdgcn_ballot_w64(emit);
        const int n_emit = __popcll(emits);
        if (emit) {
            const int at = __popcll(emits & below);
            lds.ev[at] = make_float4(r.cx, r.cy, r.cz, r.mass);
            lds.ev_mask[at] = acc;
            if (QUAD) {
                lds.pos[at] = k;
                lds.w2[at] = r.w2;  // the window's widths are no longer needed
            }
        }
        wave_lds_sync();
        const bool stuck = __builtin_amdgcn_readfirstlane(int(pending)) != 0;
        // write the rest back, the first remaining entry on top
        const int base = size - w;
        if (waits) {
            const int a0 = int((emits >> first) & 1u);  // the first waiting entry's own part is summed now
            const int start = __builtin_amdgcn_readlane(incl - cnt, first) + a0;
            const int rest = __builtin_amdgcn_readlane(incl, w - 1) - start;
            size = base + rest;
            if (have && lane >= first) {
                int at = size - 1 - (incl - cnt - start);
                if (lane == first && a0) at = size - 1;
                if (pending) {
                    lds.seq.put(at, k, mine);
                } else {
                    if (acc && !emit) {
                        lds.seq.put(at, k | LIST_FINAL, acc);
                        --at;
                    }
                    if (nch) {
                        const uint32_t ch[8] = {ka.x, ka.y, ka.z, ka.w, kb.x, kb.y, kb.z, kb.w};
#pragma unroll
                        for (int c = 0; c < 8; ++c)
                            if (c < nch) lds.seq.put(at - c, ch[c], open);
                    }
                }
            }
        } else {
            size = base;
        }
        uint32_t k0 = 0, end = 0, m0 = 0;
        if (stuck) {
            k0 = uint32_t(__builtin_amdgcn_readlane(int(k), 0));
            end = uint32_t(__builtin_amdgcn_readlane(int(r.skip), 0));
            m0 = uint32_t(__builtin_amdgcn_readlane(int(mine), 0));
            --size;
        }
        wave_lds_sync();
        load_window();
        // sum the front
        for (int e0 = 0; e0 < n_emit; e0 += U * Q) {
            float4 c[U];
            float w2[U];
            uint32_t kk[U];
            bool take[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int e = e0 + u * Q + slot, at = min(e, n_emit - 1);
                c[u] = lds.ev[at];
                take[u] = e < n_emit && ((lds.ev_mask[at] >> sub) & 1u);
                w2[u] = QUAD ? lds.w2[at] : 0.f;
                kk[u] = QUAD ? lds.pos[at] : 0u;
            }
            add_terms(std::integral_constant<int, U>{}, c, w2, kk, take);
        }
        if (stuck) {
            // not even the first entry fits: its subtree node by node, every lane from its mask
            uint32_t resume = ((m0 >> sub) & 1u) ? k0 : end;
            uint32_t c0 = k0;
            while (c0 < end) {
                const NodeRec nr = nodes[c0];
                const float d2 = norm2_ref(sub_rn(nr.cx, p.x), sub_rn(nr.cy, p.y), sub_rn(nr.cz, p.z));
                const bool active = c0 >= resume, nonzero = d2 != 0.0f;
                const bool crit = mul_rn(theta2, d2) < nr.w2;
                const bool o = active && nonzero && crit;
                const float4 c[1] = {make_float4(nr.cx, nr.cy, nr.cz, nr.mass)};
                const float w2[1] = {nr.w2};
                const uint32_t kk[1] = {c0};
                const bool take[1] = {active && nonzero && !crit && slot == 0};
                add_terms(std::integral_constant<int, 1>{}, c, w2, kk, take);
                if (!o) resume = max(resume, nr.skip);
                c0 = __builtin_amdgcn_ballot_w64(o) ? c0 + 1 : nr.skip;
            }
        }
        wave_lds_sync();
    }
    if constexpr (QUAD) {
        fold_partial(ax, ay, az, cx, cy, cz, px, py, pz);
#pragma unroll
        for (int o = L; o < 64; o <<= 1) {  // the slots' shares
            ax += __shfl_xor(ax, o, 64);
            ay += __shfl_xor(ay, o, 64);
            az += __shfl_xor(az, o, 64);
        }
    }
    if (valid) {
        const size_t at = perm ? perm[i] : i;
        if constexpr (QUAD) {
            if (slot == 0) out[at] = make_float4(ax, ay, az, 0.f);
        } else if (slot < 4) {
            reinterpret_cast<float*>(out + at)[slot] = slot < 3 ? ax : 0.f;
        }
    }
    if (lane == 0) {
        atomicAdd(&info->steps, (unsigned long long)steps);
        atomicAdd(&info->accepted, (unsigned long long)accepted);
    }
}
