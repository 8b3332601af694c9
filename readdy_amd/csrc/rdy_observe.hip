// Device observables.
//
// Radial distribution (RadialDistribution::evaluate, readdy/main/model/observables/
// RadialDistribution.cpp:75-124).  The reference loops over every ordered pair of particles on the
// host (O(N^2)); here each "from" particle visits the cells within the largest border of its own
// cell (per axis ceil(r_max / cell size) cells, the de-duplicated stencil of the cell list), so the
// work is O(N * density * r_max^3).  Counts are integers, binned exactly as the reference bins them:
// dist = sqrt(distSquared(from, to)) with the minimum image, bin = upper_bound(borders, dist) - 1,
// nothing counted at or beyond the last border.  The normalisation (shell volume, number of "from"
// particles, particleToDensity) is applied by the caller, in FP64, as the reference does.
#pragma once

#include "rdy_step.hip"

namespace rdy {

constexpr uint32_t RDF_MAX_BORDERS = 4097;  // 4096 bins: one LDS histogram per block

__device__ __forceinline__ bool in_mask(const uint32_t *mask, uint32_t t) { return (mask[t >> 5] >> (t & 31u)) & 1u; }

// std::upper_bound over borders[0 .. nb): the first index whose border exceeds dist (nb if none)
__device__ __forceinline__ uint32_t upper_bound_border(const double *b, uint32_t nb, double dist) {
    uint32_t lo = 0, hi = nb;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (dist < b[mid]) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

// Pairs by bricks.  A block stages a brick of cells and the halo that the last border reaches into LDS once, in FP32
// positions local to the brick; a wave takes 64 of the brick's "from" records, a lane each, and a share of the rows
// of cells around them (runs of staged records).  A pair's bin comes from its FP32 distance, except within the
// FP32 rounding bound of a border, where the FP64 expression of the general kernel decides: the counts are the same.
// The bin search starts from a table of RDF_LUT equal steps of the distance.  Blocks are persistent: a histogram in
// LDS is added to the result once a block.  (A thread a record that reads its candidates from the bins, FP64 and a
// binary search each, took 8.4 ms for 1,000,000 particles, 100 bins to 5.0, 343 cells a particle; this 1.4 ms, of
// which 0.5 stages.  Bound by vector issue and LDS latency: gathering the pairs in a ring and counting them 64 at a
// time costs more than the idle lanes of counting in place, 1.9 ms.)
constexpr uint32_t RDF_LUT = 1024, RDF_BATCH = 4, RDF_SHARES = 16, RDF_STATIC_LDS = 64;

struct RdfPlan {
    uint32_t e[3], nb[3];   // cells of a brick, bricks an axis
    int32_t rad[3];         // cells of halo
    uint32_t max_states, max_own, max_halo;
    uint32_t n_bricks, n_blocks;
};

__host__ __device__ inline size_t rdf_smem_bytes(uint32_t nb, const RdfPlan &p) {
    const size_t fixed = 16 * ((size_t)p.max_states + RDF_BATCH) + 4 * (size_t)p.max_states + 4 * (size_t)p.max_own +
                         8 * (size_t)nb + 12 + 4 * (size_t)RDF_LUT + 2 * ((size_t)p.max_halo + 1);
    return (fixed + 15) & ~(size_t)15;
}

__device__ __forceinline__ uint32_t rdf_brick_of(const RdfPlan &p, uint32_t x, uint32_t y, uint32_t z) {
    return ((x / p.e[0]) * p.nb[1] + y / p.e[1]) * p.nb[2] + z / p.e[2];
}

// distSquared(from, to): the difference to - from, minimum image per axis; its bin (0 or nb: none)
__device__ __forceinline__ uint32_t rdf_bin(const RepGeom &geo, const State &me, const State &o, const double *borders,
                                            uint32_t nb) {
    const double dx = min_image(o.x - me.x, geo.box[0], geo.pbc[0]);
    const double dy = min_image(o.y - me.y, geo.box[1], geo.pbc[1]);
    const double dz = min_image(o.z - me.z, geo.box[2], geo.pbc[2]);
    return upper_bound_border(borders, nb, sqrt(dist2(dx, dy, dz)));
}

// Requires (host): borders finite, the last one positive; periodic axes of at least 2 rad + 2 cells (then a pair
// within the last border is adjacent through one image only, and no other image of it is staged).  Bricks whose halo
// outgrows max_states are flagged in full[] (and counted) for k_rdf.
__global__ __launch_bounds__(256) void k_rdf_bricks(Grid cur, const ReplicaDev *reps, uint32_t r, uint32_t cap, RdfPlan p,
                                                    const double *borders, uint32_t nb, const uint32_t *from_mask,
                                                    const uint32_t *to_mask, unsigned long long *counts,
                                                    unsigned long long *n_from, uint32_t *outside, uint32_t outside_cap,
                                                    uint32_t *n_outside, uint32_t *n_full, uint32_t *full) {
    extern __shared__ char smem[];
    float4 *P = (float4 *)smem;                      // x, y, z, 0 ("to" records) or infinity
    uint32_t *slot = (uint32_t *)(P + p.max_states + RDF_BATCH);
    uint32_t *own = slot + p.max_states;             // "from" records: staged record << 16 | halo cell
    float *fb = (float *)(own + p.max_own) + 1;   // borders, between two infinities
    uint32_t *hist = (uint32_t *)(fb + nb + 1);      // by upper bound: 0 and nb are pairs of no bin
    uint32_t *lut = hist + nb + 1;                   // upper bounds of each step's edges
    uint16_t *hstart = (uint16_t *)(lut + RDF_LUT);
    __shared__ uint32_t sums[4], n_own, n_mine, froms;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wid = tid >> 6;
    const RepGeom geo = load_geom(reps[r]);
    const double rmax_d = borders[nb - 1];
    const float rmax = (float)rmax_d;
    for (uint32_t k = tid; k < nb; k += 256) fb[k] = (float)borders[k];
    for (uint32_t k = tid; k <= nb; k += 256) hist[k] = 0u;
    if (tid == 0) {
        fb[-1] = -__builtin_inff();
        fb[nb] = __builtin_inff();
        froms = 0u;
    }
    __syncthreads();
    for (uint32_t k = tid; k < RDF_LUT; k += 256) {
        uint32_t u[2];
        for (int side = 0; side < 2; ++side) {
            const float edge = rmax * ((float)(k + side) / (float)RDF_LUT);
            uint32_t lo = 0, hi = nb;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (edge < fb[mid]) hi = mid;
                else lo = mid + 1;
            }
            u[side] = lo;
        }
        lut[k] = u[0] | u[1] << 16;
    }
    const uint32_t H[3] = {p.e[0] + 2u * (uint32_t)p.rad[0], p.e[1] + 2u * (uint32_t)p.rad[1], p.e[2] + 2u * (uint32_t)p.rad[2]};
    float M = rmax;
#pragma unroll
    for (int a = 0; a < 3; ++a) M = fmaxf(M, (float)H[a] * (float)geo.cs[a]);
    // FP32 rounding of local positions below M (2^-24 M an axis and record), of a difference, the root and the borders:
    // below 8 2^-24 M in the distance
    const float margin = 16.0f * M * 1.1920929e-07f;
    const float far2 = (rmax + margin) * (rmax + margin) * (1.0f + 1.0e-6f), scale = (float)RDF_LUT / rmax;
    const uint32_t nh = H[0] * H[1] * H[2], per = (nh + 255) / 256;
    uint32_t counted = 0;  // bound on what a histogram entry holds
    for (uint32_t b = blockIdx.x; b < p.n_bricks; b += gridDim.x) {  // block-uniform
        const uint32_t bi[3] = {b / (p.nb[1] * p.nb[2]), (b / p.nb[2]) % p.nb[1], b % p.nb[2]};
        int32_t o[3], len[3];
        double org[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            o[a] = (int32_t)(bi[a] * p.e[a]);
            len[a] = min((int32_t)p.e[a], geo.dims[a] - o[a]);
            org[a] = -.5 * geo.box[a] + ((double)o[a] + .5 * p.e[a]) * geo.cs[a];
        }
        // fn(halo cell, its cell or 0xFFFFFFFF (beyond an open wall, or a short brick's end), the brick's own, its
        // image) for the thread's cells
        auto for_cells = [&](auto &&fn) {
            uint32_t c = tid * per;
            uint32_t h[3] = {c / (H[1] * H[2]), (c / H[2]) % H[1], c % H[2]};
            for (const uint32_t c1 = min(nh, c + per); c < c1; ++c) {
                int32_t q[3], img[3];
                bool valid = true, mine = true;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const int32_t k = (int32_t)h[a] - p.rad[a], x = o[a] + k;
                    const bool lo = x < 0, hi = x >= geo.dims[a];
                    valid = valid && k < len[a] + p.rad[a] && (geo.pbc[a] || !(lo || hi));
                    mine = mine && k >= 0 && k < len[a];
                    img[a] = lo ? -1 : (hi ? 1 : 0);
                    q[a] = x + (lo ? geo.dims[a] : 0) - (hi ? geo.dims[a] : 0);
                }
                fn(c, valid ? geo.cell_base + ((uint32_t)q[0] * (uint32_t)geo.dims[1] + (uint32_t)q[1]) * (uint32_t)geo.dims[2] +
                                  (uint32_t)q[2]
                            : 0xFFFFFFFFu,
                   mine, img);
                if (++h[2] == H[2]) {
                    h[2] = 0;
                    if (++h[1] == H[1]) {
                        h[1] = 0;
                        ++h[0];
                    }
                }
            }
        };
        __syncthreads();  // the last brick's records are read; the tables are written
        if (tid == 0) n_own = n_mine = 0u;
        __syncthreads();
        uint32_t sum = 0, sum_mine = 0;
        for_cells([&](uint32_t, uint32_t cell, bool mine, const int32_t *) {
            if (cell == 0xFFFFFFFFu) return;
            const uint32_t k = cur.counts[cell];
            sum += k;
            if (mine) sum_mine += k;
        });
        if (sum_mine) atomicAdd(&n_mine, sum_mine);
        const uint32_t incl = wave_inclusive_sum(sum);
        if (lane == 63) sums[wid] = incl;
        __syncthreads();
        uint32_t off = incl - sum, total = 0;
#pragma unroll
        for (uint32_t w = 0; w < 4; ++w) {
            if (w < wid) off += sums[w];
            total += sums[w];
        }
        if (total > p.max_states || n_mine > p.max_own) {  // block-uniform
            if (tid == 0) {
                atomicAdd(n_full, 1u);
                atomicOr(&full[b >> 5], 1u << (b & 31u));
            }
            continue;
        }
        for_cells([&](uint32_t c, uint32_t cell, bool mine, const int32_t *img) {
            hstart[c] = (uint16_t)off;
            if (cell == 0xFFFFFFFFu) return;
            const double sx = (double)img[0] * geo.box[0] - org[0], sy = (double)img[1] * geo.box[1] - org[1],
                         sz = (double)img[2] * geo.box[2] - org[2];
            const uint32_t end = off + cur.counts[cell];
            cell_records4(cur, cap, cell, [&](uint32_t s, const State &st) {
                if (off >= end) return;
                const bool in = !(st.tw & (TW_DEAD | TW_OUTSIDE));
                P[off] = make_float4((float)(st.x + sx), (float)(st.y + sy), (float)(st.z + sz),
                                     in && in_mask(to_mask, tw_type(st.tw)) ? 0.f : __builtin_inff());
                slot[off] = s;
                if (mine && !(st.tw & TW_DEAD)) {
                    const bool from = in_mask(from_mask, tw_type(st.tw));
                    if (from) atomicAdd(&froms, 1u);
                    if (!in) {
                        const uint32_t k = atomicAdd(n_outside, 1u);
                        if (k < outside_cap) outside[k] = s;
                    } else if (from) {
                        own[atomicAdd(&n_own, 1u)] = off << 16 | c;
                    }
                }
                ++off;
            });
            for (; off < end; ++off) P[off] = make_float4(0.f, 0.f, 0.f, __builtin_inff());  // a truncated overflow
        });
        if (tid == 255) hstart[nh] = (uint16_t)total;
        __syncthreads();
        const uint32_t no = n_own;
        if ((unsigned long long)counted + (unsigned long long)no * total > 0xFFFFFFFFull) {  // block-uniform
            for (uint32_t k = tid + 1; k < nb; k += 256) {
                if (hist[k]) atomicAdd(&counts[k - 1], (unsigned long long)hist[k]);
                hist[k] = 0u;
            }
            counted = 0;
            __syncthreads();
        }
        counted += no * total;
        const uint32_t row = (uint32_t)(2 * p.rad[1] + 1), n_rows = (uint32_t)(2 * p.rad[0] + 1) * row;
        // a lane takes one of `shares` shares of a record's rows, the shares of all records dealt to the waves 64 at
        // a time (whole records in rounds of 64 left most lanes idle in every second brick's last round)
        const uint32_t shares = min(RDF_SHARES, n_rows);
        for (uint32_t i0 = wid * 64; i0 < shares * no; i0 += 256) {  // wave-uniform
            const uint32_t i = i0 + lane;
            const bool have = i < shares * no;
            const uint32_t share = have ? i / no : 0u, ow = have ? own[i - share * no] : 0u, j = ow >> 16, hc = ow & 0xFFFFu;
            const float4 a = P[j];
            for (uint32_t k0 = 0; k0 < n_rows; k0 += shares) {
                const uint32_t k = k0 + share;
                const int32_t dx = (int32_t)(k / row) - p.rad[0], dy = (int32_t)(k % row) - p.rad[1];
                const int32_t mid = (int32_t)hc + (dx * (int32_t)H[1] + dy) * (int32_t)H[2];
                const bool walk = have && k < n_rows;
                uint32_t t = walk ? hstart[mid - p.rad[2]] : 0u;
                const uint32_t t1 = walk ? hstart[mid + p.rad[2] + 1] : 0u;
                for (; t < t1; t += RDF_BATCH) {
                    float d[RDF_BATCH];
                    uint32_t lo[RDF_BATCH], hi[RDF_BATCH];
                    float4 c[RDF_BATCH];
#pragma unroll
                    for (uint32_t u = 0; u < RDF_BATCH; ++u) c[u] = P[t + u];  // (P is padded by a batch)
#pragma unroll
                    for (uint32_t u = 0; u < RDF_BATCH; ++u) {
                        const float ex = c[u].x - a.x, ey = c[u].y - a.y, ez = c[u].z - a.z;
                        const float d2 = fmaf(ex, ex, fmaf(ey, ey, fmaf(ez, ez, c[u].w)));
                        const bool hit = t + u < t1 && d2 <= far2 && t + u != j;
                        d[u] = hit ? __builtin_amdgcn_sqrtf(d2) : -1.0f;  // (within 1 ulp)
                        const uint32_t step = min((uint32_t)(fmaxf(d[u], 0.0f) * scale), RDF_LUT - 1);
                        const uint32_t l = lut[step];
                        lo[u] = l & 0xFFFFu;
                        hi[u] = l >> 16;
                    }
#pragma unroll
                    for (uint32_t u = 0; u < RDF_BATCH; ++u) {
                        if (d[u] < 0.0f) continue;
                        while (lo[u] < hi[u]) {
                            const uint32_t m = (lo[u] + hi[u]) >> 1;
                            if (d[u] < fb[m]) hi[u] = m;
                            else lo[u] = m + 1;
                        }
                        // within the rounding bound of a border (or of several); fb is padded by infinities
                        if (fb[lo[u]] - d[u] < margin || d[u] - fb[(int32_t)lo[u] - 1] < margin)
                            lo[u] = rdf_bin(geo, cur.bins[slot[j]], cur.bins[slot[t + u]], borders, nb);
                        atomicAdd(&hist[lo[u]], 1u);
                    }
                }
            }
        }
    }
    __syncthreads();
    if (tid == 0 && froms) atomicAdd(n_from, (unsigned long long)froms);
    for (uint32_t k = tid + 1; k < nb; k += 256)
        if (hist[k]) atomicAdd(&counts[k - 1], (unsigned long long)hist[k]);
}

// One thread per live record of the work list; only: those of the flagged bricks of plan p that k_rdf_bricks left
// (they count as "from" and outside records here), null: all.  Records of replica r whose type is in from_mask are
// counted into *n_from; those inside the box count their pairs with the in-box "to" records of the
// stencil of radius rad[a] cells; records outside the box (never binned as neighbours) are listed
// for k_rdf_outside.  Per-block histogram in LDS, added to counts[nb - 1] (64-bit) at the end.
__global__ __launch_bounds__(256) void k_rdf(Grid cur, const ReplicaDev *reps, uint32_t r, uint32_t cap,
                                             const double *borders, uint32_t nb, const uint32_t *from_mask,
                                             const uint32_t *to_mask, int rad0, int rad1, int rad2,
                                             unsigned long long *counts, unsigned long long *n_from,
                                             uint32_t *outside, uint32_t outside_cap, uint32_t *n_outside,
                                             uint32_t max_wl, RdfPlan p, const uint32_t *only) {
    __shared__ double sb[RDF_MAX_BORDERS];
    __shared__ uint32_t hist[RDF_MAX_BORDERS - 1];
    for (uint32_t k = threadIdx.x; k < nb; k += blockDim.x) sb[k] = borders[k];
    for (uint32_t k = threadIdx.x; k + 1 < nb; k += blockDim.x) hist[k] = 0u;
    __syncthreads();
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t n = *cur.wl_count;
    n = n < max_wl ? n : max_wl;
    bool from = false;
    if (i < n) {
        const uint32_t s = cur.wl[i];
        const State me = cur.bins[s];
        bool listed = !(me.tw & TW_DEAD) && tw_replica(me.tw) == r;
        if (listed && only) {
            const uint32_t cl = cell_of_slot(cur, s, cap) - reps[r].cell_base;
            const uint32_t nz = (uint32_t)reps[r].dims[2], ny = (uint32_t)reps[r].dims[1];
            const uint32_t b = rdf_brick_of(p, cl / (nz * ny), (cl / nz) % ny, cl % nz);
            listed = only[b >> 5] >> (b & 31u) & 1u;
        }
        if (listed) {
            from = in_mask(from_mask, tw_type(me.tw));
            if (me.tw & TW_OUTSIDE) {
                const uint32_t p = atomicAdd(n_outside, 1u);
                if (p < outside_cap) outside[p] = s;
            } else if (from) {
                const RepGeom geo = load_geom(reps[r]);
                const uint32_t cl = cell_of_slot(cur, s, cap) - geo.cell_base;
                const int nz = geo.dims[2], ny = geo.dims[1];
                const int c[3] = {(int)(cl / (uint32_t)(nz * ny)), (int)((cl / (uint32_t)nz) % (uint32_t)ny),
                                  (int)(cl % (uint32_t)nz)};
                const int rad[3] = {rad0, rad1, rad2};
                int cnt[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) cnt[a] = axis_count(c[a], geo.dims[a], geo.pbc[a], rad[a]);
                for (int ka = 0; ka < cnt[0]; ++ka) {
                    const int x = axis_elem(ka, c[0], geo.dims[0], geo.pbc[0], rad[0]);
                    for (int kb = 0; kb < cnt[1]; ++kb) {
                        const int y = axis_elem(kb, c[1], geo.dims[1], geo.pbc[1], rad[1]);
                        const uint32_t row = geo.cell_base + ((uint32_t)x * (uint32_t)ny + (uint32_t)y) * (uint32_t)nz;
                        for (int kc = 0; kc < cnt[2]; ++kc) {
                            const uint32_t cell = row + (uint32_t)axis_elem(kc, c[2], nz, geo.pbc[2], rad[2]);
                            cell_records(cur, cap, cell, [&](uint32_t s2) {
                                if (s2 == s) return;
                                const State o = cur.bins[s2];
                                if ((o.tw & (TW_DEAD | TW_OUTSIDE)) || !in_mask(to_mask, tw_type(o.tw))) return;
                                const uint32_t u = rdf_bin(geo, me, o, sb, nb);
                                if (u > 0 && u < nb) atomicAdd(&hist[u - 1], 1u);
                            });
                        }
                    }
                }
            }
        }
    }
    const unsigned long long fm = __ballot(from);
    if ((threadIdx.x & 63u) == 0u && fm) atomicAdd(n_from, (unsigned long long)__popcll(fm));
    __syncthreads();
    for (uint32_t k = threadIdx.x; k + 1 < nb; k += blockDim.x)
        if (hist[k]) atomicAdd(&counts[k], (unsigned long long)hist[k]);
}

// The pairs that involve a record outside the box: thread (o, i) pairs listed record o with work-list
// record i of the replica; o -> i when o is "from" and i is "to", i -> o when i is an in-box "from"
// record and o is "to" (a pair of two outside records is counted from each side by its own row).
__global__ __launch_bounds__(256) void k_rdf_outside(Grid cur, const ReplicaDev *reps, uint32_t r,
                                                     const double *borders, uint32_t nb, const uint32_t *from_mask,
                                                     const uint32_t *to_mask, unsigned long long *counts,
                                                     const uint32_t *outside, const uint32_t *n_outside,
                                                     uint32_t max_wl) {
    uint32_t n = *cur.wl_count;
    n = n < max_wl ? n : max_wl;
    const uint32_t no = *n_outside;
    const unsigned long long idx = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (n == 0 || idx >= (unsigned long long)no * n) return;
    const uint32_t s = outside[idx / n], s2 = cur.wl[idx % n];
    if (s2 == s) return;
    const State a = cur.bins[s], b = cur.bins[s2];
    if ((b.tw & TW_DEAD) || tw_replica(b.tw) != r) return;
    const RepGeom geo = load_geom(reps[r]);
    auto count = [&](const State &f, const State &t) {
        const double dx = min_image(t.x - f.x, geo.box[0], geo.pbc[0]);
        const double dy = min_image(t.y - f.y, geo.box[1], geo.pbc[1]);
        const double dz = min_image(t.z - f.z, geo.box[2], geo.pbc[2]);
        const uint32_t u = upper_bound_border(borders, nb, sqrt(dist2(dx, dy, dz)));
        if (u > 0 && u < nb) atomicAdd(&counts[u - 1], 1ull);
    };
    if (in_mask(from_mask, tw_type(a.tw)) && in_mask(to_mask, tw_type(b.tw))) count(a, b);
    if (!(b.tw & TW_OUTSIDE) && in_mask(from_mask, tw_type(b.tw)) && in_mask(to_mask, tw_type(a.tw))) count(b, a);
}

// HistogramAlongAxis as the CPU kernel evaluates it (kernels/cpu/src/observables/CPUObservables.cpp:
// 85-136): each live record of replica r whose type is in mask adds one to bin u - 1, u =
// upper_bound(borders, position[axis]), when 1 <= u < nb - 1 (the CPU kernel compares u with the bin
// count, so the last bin stays empty).  One thread per work-list record, per-block LDS histogram.
__global__ __launch_bounds__(256) void k_hist_axis(Grid cur, uint32_t r, const double *borders, uint32_t nb,
                                                   const uint32_t *mask, int axis, unsigned long long *counts,
                                                   uint32_t max_wl) {
    __shared__ double sb[RDF_MAX_BORDERS];
    __shared__ uint32_t hist[RDF_MAX_BORDERS - 1];
    for (uint32_t k = threadIdx.x; k < nb; k += blockDim.x) sb[k] = borders[k];
    for (uint32_t k = threadIdx.x; k + 1 < nb; k += blockDim.x) hist[k] = 0u;
    __syncthreads();
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t n = *cur.wl_count;
    n = n < max_wl ? n : max_wl;
    if (i < n) {
        const State me = cur.bins[cur.wl[i]];
        if (!(me.tw & TW_DEAD) && tw_replica(me.tw) == r && in_mask(mask, tw_type(me.tw))) {
            const double x = axis == 0 ? me.x : (axis == 1 ? me.y : me.z);
            const uint32_t u = upper_bound_border(sb, nb, x);
            if (u >= 1u && u + 1u < nb) atomicAdd(&hist[u - 1], 1u);
        }
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k + 1 < nb; k += blockDim.x)
        if (hist[k]) atomicAdd(&counts[k], (unsigned long long)hist[k]);
}

}  // namespace rdy
