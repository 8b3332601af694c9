// LDS-staged stencil kernels: one workgroup per brick of cells.
//
// A brick is a box of cells of one replica.  Its workgroup copies the brick plus a halo of
// `radius` cells (periodic images wrapped, non-periodic ones clipped) from the cell bins into LDS
// once, packs every cell's members contiguously (z-fastest, so the z-neighbours of a cell form one
// contiguous run), and walks the (2r+1)^3 stencil of every particle of the brick against LDS.
// Each staged record carries an FP32 position in the brick's local frame with periodic images
// already shifted, used as a conservative prefilter: a candidate is dropped in FP32 only when it
// is farther than the cutoff by more than the FP32 rounding bound, so the exact pair set is
// unchanged.  The exact work (FP64 min-image displacement, the reference gate d2 < rc^2, the pair
// math, the reaction draws) runs on the survivors only, and not per lane: each wave streams its
// survivors through rings in LDS and evaluates them 64 at a time with every lane busy, because a
// per-lane evaluation would make the whole wave execute the exact branch whenever any one lane
// had a survivor (almost always).  Forces are gathered per particle as 64-bit fixed-point sums
// (LDS atomics; integer addition is order-free, so the result stays deterministic).
// A brick whose halo holds more particles than the LDS budget takes a slow path that reads
// neighbours straight from the bins.
//
// Four consecutive records of one z-row of cells share a quad of lanes and their candidates: the quad
// walks the rows of cells around them four candidates at a time, and the matrix cores form the 4 x 4
// squared distances (mfma_pipeline).
//
// Per axis a brick is either in halo mode (extent e, halo r on both sides; the axis has at least 2r + 1
// cells when it is periodic, so the cells of a stencil are distinct; when e + 2r exceeds the axis, halo
// cells repeat cells of the brick at another image) or in whole-axis mode (a periodic axis of at most
// 2r cells: the brick spans it, no halo; neighbour coordinates wrap inside the brick), which also
// reproduces the de-duplicated adjacency of small grids (CellLinkedList.cpp:74-137).
#pragma once

#include "rdy_kernels.hip"

#include <type_traits>

namespace rdy {

struct BrickDev {
    int32_t o[3];    // origin cell
    int32_t e[3];    // extent in cells
    int32_t h[3];    // halo width (0 in whole-axis mode)
    uint32_t r;      // replica
    uint32_t whole;  // bit a: axis a spans the grid
    // ceil(2^32 / d) for d = H1 * H2, H2 and e1 (H = e + 2h; 0 when d == 1): exact n / d as a high
    // multiply for n, d < 2^16
    uint32_t m_hh, m_h2, m_e1;
    // the replica's grid, so that the halo's cells are known before the replica's record arrives
    uint32_t cell_base;
    int32_t dims[3];
    uint32_t pbc;    // bit a: the replica's axis a is periodic
    uint32_t pad;
};
static_assert(sizeof(BrickDev) == 80, "brick record size");

constexpr int BRICK_THREADS = 256;
constexpr int BRICK_WAVES = BRICK_THREADS / 64;
constexpr uint32_t BATCH = 2;       // candidates a lane takes from its current run per iteration (general walk)
constexpr uint32_t RING = 256;      // per-wave ring of its survivors (power of two, >= 63 + 64 * BATCH)
constexpr uint32_t QRING = 128;     // per-wave ring of harvested pairs of the matrix-core walk
constexpr uint32_t ORING = 128;     // and of its sifted pairs (>= 63 + 64)
constexpr uint32_t QSTEPS = 8;      // its steps between two harvests: 8 x 4 result bits fill a word
constexpr size_t WAVE_RING_BYTES = 4 * QRING + 4 * ORING + 2 * 16 * QSTEPS;  // two rings and the steps' candidates
static_assert(WAVE_RING_BYTES >= 4 * RING, "or the general walk's ring");
constexpr float FAR_POS = 1.0e18f, FAR_SQ = 1.0e36f;  // a record that is no neighbour lies here
constexpr uint32_t NO_ENTRY = 0xFFFFFFFFu;  // an idle lane's entry in the last batch of the ring

__host__ __device__ inline uint32_t div_magic(uint32_t d) {
    return d > 1 ? (uint32_t)((0x100000000ull + d - 1) / d) : 0u;
}
__device__ __forceinline__ uint32_t fdiv(uint32_t n, uint32_t m) { return m ? __umulhi(n, m) : n; }

struct Halo {  // halo box of a brick, z fastest: hc = (hx * H1 + hy) * H2 + hz
    uint32_t H0, H1, H2, HH, nh, m_hh, m_h2;
    __device__ __forceinline__ void decode(uint32_t hc, uint32_t &hx, uint32_t &hy, uint32_t &hz) const {
        hx = fdiv(hc, m_hh);
        const uint32_t rem = hc - hx * HH;
        hy = fdiv(rem, m_h2);
        hz = rem - hy * H2;
    }
};

__device__ __forceinline__ Halo make_halo(const BrickDev &B) {
    Halo s;
    s.H0 = (uint32_t)(B.e[0] + 2 * B.h[0]);
    s.H1 = (uint32_t)(B.e[1] + 2 * B.h[1]);
    s.H2 = (uint32_t)(B.e[2] + 2 * B.h[2]);
    s.HH = s.H1 * s.H2;
    s.nh = s.H0 * s.HH;
    s.m_hh = B.m_hh;
    s.m_h2 = B.m_h2;
    return s;
}

struct BrickSmem {  // carved out of dynamic LDS
    float4 *P;         // [max_states + 1] local-frame FP32 position, w = its square; the last one is far away
    uint32_t *slot;    // [max_states] bin slot (the FP64 record is read from the bins when needed)
    uint16_t *hstart;  // [max_halo + 1] (at most 60000 records are staged)
    uint16_t *hc_of;   // [max_states]
    uint8_t *typ;      // [max_states] species (below MAX_STAGED_TYPES), TYP_OUTSIDE, TYP_DEAD
    char *rings;       // [BRICK_WAVES][WAVE_RING_BYTES]
    uint32_t far;      // index of the far record
};
// A flagged record (typ >= TYP_OUTSIDE) is no neighbour: the matrix-core walk refuses it by its distance, the general
// walk by the flag; a table of the types is indexed by typ & TYP_MASK wherever a flagged record can come.
constexpr uint8_t TYP_OUTSIDE = 0x40, TYP_DEAD = 0x80, TYP_MASK = 0x0F;

__device__ __forceinline__ BrickSmem carve(char *base, uint32_t max_states, uint32_t max_halo) {
    BrickSmem m;
    char *p = base;
    m.P = (float4 *)p;
    p += sizeof(float4) * (max_states + 1);
    m.slot = (uint32_t *)p;
    p += 4 * max_states;
    m.hstart = (uint16_t *)p;
    p += 2 * (max_halo + 1);
    m.hc_of = (uint16_t *)p;
    p += 2 * max_states;
    m.typ = (uint8_t *)p;
    p += max_states;
    p = base + ((p - base + 15) & ~(ptrdiff_t)15);
    m.rings = p;
    m.far = max_states;
    return m;
}

__host__ __device__ inline size_t brick_smem_bytes(uint32_t max_states, uint32_t max_halo) {
    const size_t fixed = sizeof(float4) * ((size_t)max_states + 1) + (4 + 2 + 1) * (size_t)max_states +
                         2 * ((size_t)max_halo + 1);
    return ((fixed + 15) & ~(size_t)15) + BRICK_WAVES * WAVE_RING_BYTES;
}

// Kernel arguments and records that a kernel only reads, through the constant address space: they come in
// scalar loads, and laundering the pointer makes a part of a kernel load what it needs where it needs it.  (Kept in
// registers from the start, a walk's arguments, geometry and tables exceed the scalar registers: 1441 of the 5976
// vector instructions of k_brick_step moved spilled ones.)
template <class T>
__device__ __forceinline__ const T &read_only(const T *p) {
    typedef const __attribute__((address_space(4))) T *C;
    C c = (C)p;
    asm volatile("" : "+s"(c));
    return *(const T *)c;
}

// the kernel's arguments: its one by-value argument, the first of the kernarg segment
template <class T>
__device__ __forceinline__ const T &kernel_args() {
    typedef const __attribute__((address_space(4))) T *C;
    C c = (C)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(c));
    return *(const T *)c;
}

struct Frame {       // local frame of a brick
    double org[3];   // real coordinate of local 0
    float L[3];      // box lengths (FP32) for whole-axis min image
    uint32_t whole;
    float margin;    // 16 * 2^-23 * largest local coordinate (FP32 rounding bound, 4x safety)
    float expand;    // bound on the rounding of |a|^2 + |b|^2 - 2 ab against |a - b|^2 (mfma_pipeline)
};

__device__ __forceinline__ Frame make_frame(const BrickDev &B, const RepGeom &geo) {
    Frame f;
    float M = 0.f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const bool w = B.whole & (1u << a);
        f.org[a] = w ? -.5 * geo.box[a] : (-.5 * geo.box[a] + (double)B.o[a] * geo.cs[a]);
        f.L[a] = (float)geo.box[a];
        const float ext = w ? (float)geo.box[a] : (float)((B.e[a] + 2 * B.h[a]) * geo.cs[a]);
        M = fmaxf(M, ext);
    }
    f.whole = B.whole;
    f.margin = 16.0f * M * 1.1920929e-07f;
    // |p|^2 <= 3 M^2 = S for every local position p.  With u = 2^-24: the squares carry 3 u S each, each of the
    // four accumulations rounds a partial sum of at most 4 S, each product at most 2 S: below 40 u S = 2.4e-6 S
    f.expand = 3.0e-5f * M * M;
    return f;
}

// prefilter threshold: cutoff^2 widened by the FP32 rounding bound (negative: nothing to find)
__device__ __forceinline__ float prefilter_thr(float cut2_f, bool any, float margin) {
    return any ? cut2_f * (1.0f + 3.0e-6f) + 2.0f * sqrtf(cut2_f) * margin + margin * margin : -1.0f;
}

// Staging a brick.  A thread owns a chunk of consecutive halo cells: it reads their counters (one global round
// trip, issued from the brick record alone, so that they travel with the replica's record), and a block scan
// places every cell's records: their bin slots are listed in LDS.  Then the records are dealt out evenly over
// the threads (the second round trip).  (Requesting a chunk's records before the scan saved a tenth of the
// staging's latency, and its idle slots cost more instructions than that.)
constexpr uint32_t STAGE_CELLS = 4;   // cells of a thread at a time
constexpr uint32_t STAGE_UNROLL = 4;  // records of a thread in flight

struct HaloCells {  // a thread's cells (registers): global cell and records
    uint32_t cl[STAGE_CELLS], n[STAGE_CELLS];
};

__device__ __forceinline__ uint32_t cells_per_thread(const Halo &Hs) { return (Hs.nh + BRICK_THREADS - 1) / BRICK_THREADS; }

// halo cells c0 .. c0 + count - 1 (count <= STAGE_CELLS); clear: the counters of the brick's own cells among them are
// cleared in this buffer (null: none)
__device__ __forceinline__ HaloCells load_halo_cells(const uint32_t *counts, uint32_t *clear, const BrickDev &B,
                                                     const Halo &Hs, uint32_t c0, uint32_t count) {
    HaloCells h;
    uint32_t hh[3];
    Hs.decode(c0, hh[0], hh[1], hh[2]);
#pragma unroll
    for (uint32_t u = 0; u < STAGE_CELLS; ++u) {
        h.cl[u] = h.n[u] = 0;
        if (u < count && c0 + u < Hs.nh) {
            int32_t c[3];
            bool own = true, valid = true;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int32_t x = B.o[a] - B.h[a] + (int32_t)hh[a];
                const bool lo = x < 0, hi = x >= B.dims[a];  // |overhang| <= r < dims
                valid = valid && ((B.pbc >> a & 1u) || !(lo || hi));
                c[a] = x + (lo ? B.dims[a] : 0) - (hi ? B.dims[a] : 0);
                own = own && hh[a] - (uint32_t)B.h[a] < (uint32_t)B.e[a];
            }
            const uint32_t cl =
                B.cell_base + ((uint32_t)c[0] * (uint32_t)B.dims[1] + (uint32_t)c[1]) * (uint32_t)B.dims[2] + (uint32_t)c[2];
            if (valid) {
                h.cl[u] = cl;
                h.n[u] = counts[cl];
            }
            if (clear && own) clear[cl] = 0u;
        }
        if (++hh[2] == Hs.H2) {
            hh[2] = 0;
            if (++hh[1] == Hs.H1) {
                hh[1] = 0;
                ++hh[0];
            }
        }
    }
    return h;
}

// inclusive sum over the lanes of a wave (DPP row shifts and row broadcasts: no LDS round trips)
__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true);  // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true);  // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true);  // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
    return v;
}

// stages buffer g around brick B into LDS; returns the number of staged records, or UINT32_MAX if
// they do not fit (the caller then takes the slow path).  h: load_halo_cells of the thread's cells
// (only used when a thread has at most STAGE_CELLS).
__device__ __forceinline__ uint32_t stage_brick(const Grid &g, const BrickDev &B, const RepGeom &geo, const Frame &F, uint32_t cap,
                                const BrickSmem &m, uint32_t max_states, const Halo &Hs, HaloCells h) {
    __shared__ uint32_t wave_sums[BRICK_WAVES];
    const uint32_t tid = threadIdx.x, nh = Hs.nh, per = cells_per_thread(Hs), c0 = tid * per;
    uint32_t off = 0, total = 0;
    auto place = [&](uint32_t sum) {  // off = records before this thread's, total = all
        const uint32_t incl = wave_inclusive_sum(sum), wid = tid / 64;
        if (__lane_id() == 63) wave_sums[wid] = incl;
        __syncthreads();
        off = incl - sum;
        total = 0;
#pragma unroll
        for (uint32_t w = 0; w < BRICK_WAVES; ++w) {
            const uint32_t ws = wave_sums[w];
            if (w < wid) off += ws;
            total += ws;
        }
    };
    if (per > STAGE_CELLS) {  // a large halo: its counters are read twice
        uint32_t sum = 0;
        for (uint32_t u = 0; u < per; u += STAGE_CELLS) {
            const HaloCells q = load_halo_cells(g.counts, nullptr, B, Hs, c0 + u, min(per - u, STAGE_CELLS));
            sum += q.n[0] + q.n[1] + q.n[2] + q.n[3];
        }
        place(sum);
    }
    if (per <= STAGE_CELLS) place(h.n[0] + h.n[1] + h.n[2] + h.n[3]);
    if (total > max_states) return 0xFFFFFFFFu;  // block-uniform
    for (uint32_t u0 = 0; u0 < per; u0 += STAGE_CELLS) {  // once, but for large halos
        if (per > STAGE_CELLS) h = load_halo_cells(g.counts, nullptr, B, Hs, c0 + u0, min(per - u0, STAGE_CELLS));
#pragma unroll
        for (uint32_t u = 0; u < STAGE_CELLS; ++u) {
            const uint32_t hc = c0 + u0 + u;
            if (u0 + u >= per || hc >= nh) break;
            m.hstart[hc] = (uint16_t)off;
            for (uint32_t k = 0; k < h.n[u]; ++k) {
                uint32_t s = h.cl[u] * cap + k;
                if (k >= cap) {
                    // the (k - cap)-th overflow record of a crowded cell (rare); beyond a truncated overflow
                    // list the counter runs ahead of the records: a dead placeholder
                    uint32_t no = *g.ovf_count;
                    no = no < g.ovf_cap ? no : g.ovf_cap;
                    s = 0xFFFFFFFFu;
                    for (uint32_t o = 0, seen = 0; o < no; ++o)
                        if (g.ovf_cell[o] == h.cl[u] && seen++ == k - cap) {
                            s = g.nbin + o;
                            break;
                        }
                }
                m.slot[off + k] = s;
                m.hc_of[off + k] = (uint16_t)hc;
            }
            off += h.n[u];
        }
    }
    __syncthreads();
    bool edge = false;  // some halo cell lies across a boundary (block-uniform)
    for (int a = 0; a < 3; ++a) edge = edge || B.o[a] < B.h[a] || B.o[a] + B.e[a] + B.h[a] > B.dims[a];
    auto put = [&](uint32_t j, const State &st) {
        double lx = st.x - F.org[0], ly = st.y - F.org[1], lz = st.z - F.org[2];
        if (edge) {  // unwraps halo images into the local frame (a whole axis has none)
            uint32_t hh[3];
            Hs.decode(m.hc_of[j], hh[0], hh[1], hh[2]);
            double shift[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const int32_t u = B.o[a] - B.h[a] + (int32_t)hh[a];
                shift[a] = u < 0 ? -geo.box[a] : (u >= B.dims[a] ? geo.box[a] : 0.0);
            }
            lx += shift[0];
            ly += shift[1];
            lz += shift[2];
        }
        const float fx = (float)lx, fy = (float)ly, fz = (float)lz;
        // a dead or outside record is never a neighbour: it fails every distance test
        const bool dead = (st.tw & TW_DEAD) != 0u, gone = dead || (st.tw & TW_OUTSIDE) != 0u;
        m.P[j] = gone ? make_float4(FAR_POS, 0.f, 0.f, FAR_SQ) : make_float4(fx, fy, fz, prefilter_d2(fx, fy, fz));
        m.typ[j] = (uint8_t)(tw_type(st.tw) | (gone ? TYP_OUTSIDE : 0u) | (dead ? TYP_DEAD : 0u));
    };
    for (uint32_t j0 = 0; j0 < total; j0 += STAGE_UNROLL * BRICK_THREADS) {
        State st[STAGE_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < STAGE_UNROLL; ++u) {
            const uint32_t j = j0 + u * BRICK_THREADS + tid;
            if (j < total) {
                const uint32_t s = m.slot[j];
                st[u].tw = TW_DEAD;
                if (s != 0xFFFFFFFFu) st[u] = g.bins[s];
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < STAGE_UNROLL; ++u) {
            const uint32_t j = j0 + u * BRICK_THREADS + tid;
            if (j < total) put(j, st[u]);
        }
    }
    if (tid == 0) {
        m.hstart[nh] = (uint16_t)total;
        m.P[m.far] = make_float4(0.f, 0.f, 0.f, FAR_SQ);
    }
    __syncthreads();
    return total;
}

// The quads q0 .. q0 + 15 of the brick's own records, listed in the wave's own array (first record | number << 16):
// the own records of a row of cells are consecutive, and each row is dealt into quads.  Returns the number of
// quads of the brick.  Every wave lists its own, a row a lane.
__device__ __forceinline__ uint32_t wave_quads(const BrickSmem &m, const BrickDev &B, const Halo &Hs, uint32_t *quads,
                                               uint32_t q0) {
    const uint32_t lane = __lane_id(), rows = (uint32_t)(B.e[0] * B.e[1]);
    uint32_t n_quads = 0;
    for (uint32_t r0 = 0; r0 < rows; r0 += 64) {  // wave-uniform
        const uint32_t row = r0 + lane;
        uint32_t a = 0, n = 0;
        if (row < rows) {
            const uint32_t x = fdiv(row, B.m_e1), y = row - x * (uint32_t)B.e[1];
            const uint32_t hc = (x + (uint32_t)B.h[0]) * Hs.HH + (y + (uint32_t)B.h[1]) * Hs.H2 + (uint32_t)B.h[2];
            a = m.hstart[hc];
            n = m.hstart[hc + (uint32_t)B.e[2]] - a;
        }
        const uint32_t nq = (n + 3) / 4, incl = wave_inclusive_sum(nq);
        const uint32_t at = n_quads + incl - nq - q0;  // (wraps below q0)
        for (uint32_t k = 0; k < nq; ++k)
            if (at + k < 16u) quads[at + k] = (a + 4 * k) | (min(n - 4 * k, 4u) << 16);
        n_quads += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
    }
    return n_quads;
}

// The owner of this lane: the wave's quads (wave_quads from q0 on) take its lanes four by four.
// j: the owner's staged record, t: its species and flags (valid: there is one, and it lives).
struct OwnerLane {
    uint32_t j, t;
    bool valid;
};
__device__ __forceinline__ OwnerLane owner_lane(const BrickSmem &m, const uint32_t *quads, uint32_t q0, uint32_t n_quads) {
    const uint32_t lane = __lane_id();
    OwnerLane o{0, 0, false};
    if (q0 + lane / 4 < n_quads) {
        const uint32_t e = quads[lane / 4], k = lane & 3u, n = e >> 16;
        o.j = (e & 0xFFFFu) + min(k, n - 1u);  // an idle lane repeats the quad's last record (its cell)
        o.t = m.typ[o.j];
        o.valid = k < n && !(o.t & TYP_DEAD);
    }
    return o;
}

// ---- stencil walkers: visit the staged records of the (2r+1)^3 stencil of halo cell hc as
// contiguous runs [q, qe) -------------------------------------------------------------------------
struct WalkCtx {
    Halo Hs;
    uint32_t whole;
    int32_t dims[3];
    int radius;
    int32_t h[3];       // halo widths
    float cs[3], inv_cs[3];
};

__device__ __forceinline__ WalkCtx make_walk(const BrickDev &B, const RepGeom &geo, const Halo &Hs, int radius) {
    WalkCtx c;
    c.Hs = Hs;
    c.whole = B.whole;
    c.dims[0] = geo.dims[0];
    c.dims[1] = geo.dims[1];
    c.dims[2] = geo.dims[2];
    c.radius = radius;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        c.h[a] = B.h[a];
        c.cs[a] = (float)geo.cs[a];
        c.inv_cs[a] = __builtin_amdgcn_rcpf(c.cs[a]);  // (1 ulp; the reaches carry more slack)
    }
    return c;
}

// general case: per axis the offsets -r..r (halo mode) or all cells (whole-axis mode); z is one run
struct Walk {
    int nx, ny, nz;  // cells an axis
    int bx, by, bz;  // the first ones
    int ia, ib;
    uint32_t q, qe;

    __device__ __forceinline__ static void axis(const WalkCtx &c, int a, uint32_t hcoord, int &n, int &base) {
        const bool whole = c.whole >> a & 1u;
        n = whole ? c.dims[a] : 2 * c.radius + 1;
        base = whole ? 0 : (int)hcoord - c.radius;
    }
    __device__ __forceinline__ void range(const WalkCtx &c, const uint16_t *hs) {
        const uint32_t z0 = ((uint32_t)(bx + ia) * c.Hs.H1 + (uint32_t)(by + ib)) * c.Hs.H2 + (uint32_t)bz;
        q = hs[z0];
        qe = hs[z0 + (uint32_t)nz];
    }
    __device__ __forceinline__ bool begin(const WalkCtx &c, uint32_t hc, const uint16_t *hs) {
        uint32_t hx, hy, hz;
        c.Hs.decode(hc, hx, hy, hz);
        axis(c, 0, hx, nx, bx);
        axis(c, 1, hy, ny, by);
        axis(c, 2, hz, nz, bz);
        ia = ib = 0;
        range(c, hs);
        return q < qe || advance(c, hs);
    }
    __device__ __forceinline__ bool advance(const WalkCtx &c, const uint16_t *hs) {
        do {
            if (++ib >= ny) {
                ib = 0;
                if (++ia >= nx) return false;
            }
            range(c, hs);
        } while (q >= qe);
        return true;
    }
};

// makes LDS writes of this wave visible to its other lanes (and orders the compiler's accesses)
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The general walk (bricks with a whole-axis axis).
// Streams candidate pairs through the wave's ring: every active lane walks the stencil of its own
// staged record (halo cell hc), taking up to BATCH candidates of its current run per iteration (independent LDS reads), and offers each to keep(q, P[q]); survivors are
// appended as (lane << 16 | q) and evaluated by eval(entry) 64 at a time with all lanes of the
// wave.  A lane's survivors of one iteration take consecutive ring places after those of the lower
// lanes (one prefix over the lanes' survivor counts per iteration).  The last, partial batch too runs
// eval on every lane, idle lanes with NO_ENTRY (so that eval may read other lanes' registers).  Must
// be called by all 64 lanes of a wave (wave-uniform control flow around it).
template <class Keep, class Eval>
__device__ __forceinline__ void pair_pipeline(const WalkCtx &c, const uint16_t *hs, const float4 *P, uint32_t *ring,
                                              bool active, uint32_t hc, Keep &&keep, Eval &&eval) {
    static_assert(BATCH <= 7, "survivor counts are ranked as three bit planes");
    const uint32_t lane = __lane_id();
    Walk w;
    w.q = w.qe = 0;
    bool more = false;
    if (active) more = w.begin(c, hc, hs);
    uint32_t head = 0, tail = 0;  // wave-uniform
    while (__ballot(more)) {
        uint32_t q0 = 0, nq = 0;
        if (more) {
            q0 = w.q;
            nq = min(w.qe - w.q, BATCH);
            w.q += nq;
            if (w.q >= w.qe) more = w.advance(c, hs);
        }
        // candidates q0 .. q0 + nq - 1; reads past the batch repeat its last record (masked out)
        const uint32_t last = nq ? q0 + nq - 1u : q0;
        float4 pq[BATCH];  // the batch's records first (independent LDS reads), then the tests
#pragma unroll
        for (uint32_t i = 0; i < BATCH; ++i) pq[i] = P[min(q0 + i, last)];
        uint32_t bits = 0;
#pragma unroll
        for (uint32_t i = 0; i < BATCH; ++i) bits |= (keep(min(q0 + i, last), pq[i]) & (i < nq)) ? (1u << i) : 0u;
        const uint32_t cnt = (uint32_t)__popc(bits);
        const unsigned long long b0 = __ballot(cnt & 1u), b1 = __ballot(cnt & 2u), b2 = __ballot(cnt & 4u);
        uint32_t pos = tail + rank_in_mask(b0) + 2u * rank_in_mask(b1) + 4u * rank_in_mask(b2);
        tail += (uint32_t)__popcll(b0) + 2u * (uint32_t)__popcll(b1) + 4u * (uint32_t)__popcll(b2);
        while (bits) {  // at most BATCH passes, usually one
            const uint32_t i = (uint32_t)__ffs(bits) - 1u;
            bits &= bits - 1u;
            ring[pos & (RING - 1)] = (lane << 16) | (q0 + i);
            ++pos;
        }
        while (tail - head >= 64) {
            wave_lds_sync();
            eval(ring[(head + lane) & (RING - 1)]);
            head += 64;
            wave_lds_sync();
        }
    }
    if (tail != head) {
        wave_lds_sync();
        eval(lane < tail - head ? ring[(head + lane) & (RING - 1)] : NO_ENTRY);
        wave_lds_sync();
    }
}

// exchanges within a quad of lanes (DPP quad_perm) and broadcasts of one of its lanes
template <int CTRL>
__device__ __forceinline__ int quad_perm(int v) {
    return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xF, 0xF, true);
}
__device__ __forceinline__ int quad_min(int v) {
    v = min(v, quad_perm<0xB1>(v));  // lanes 1 0 3 2
    return min(v, quad_perm<0x4E>(v));  // lanes 2 3 0 1
}
__device__ __forceinline__ int quad_max(int v) {
    v = max(v, quad_perm<0xB1>(v));
    return max(v, quad_perm<0x4E>(v));
}
template <int LANE>
__device__ __forceinline__ float quad_bcast(float v) {
    return __int_as_float(quad_perm<LANE * 0x55>(__float_as_int(v)));
}

// The walk of bricks in halo mode on every axis.  A quad of lanes holds up to four consecutive records of one
// row of cells (halo cell hc, local position p, reach; active: the lane's record looks for neighbours).  The
// cells that any of them reaches form rows (2r + 1 by 2r + 1 at most, pruned by the records' positions) of one
// z-range, each row one contiguous run of staged records.  Each step the quad takes four candidates, one a lane,
// and the matrix cores form the 4 x 4 values |a|^2 + |b|^2 - 2 ab - threshold(a) (v_mfma_f32_4x4x1, sixteen
// quads at once, K = x, y, z, 1; the owners' |a|^2 - threshold is the accumulator's start): lane l gets its
// candidate against the quad's four records, and keeps the four signs as bits.  Every QSTEPS steps the wave
// harvests the set bits into a ring of (owner lane << 16 | candidate) entries; these pass filter(entry) 64 at a
// time (the pair's own threshold, and not the record itself), and the survivors eval(entry) 64 at a time with
// all lanes of the wave (the last batch's idle lanes with NO_ENTRY, so that eval may read other lanes'
// registers); after(done) runs once a turn of the loop, at last until it returns false.  Must be called by all 64
// lanes of a wave.
// A lane used to test its own candidates one by one, about 36 vector instructions each with the ring
// bookkeeping (1900 of the 3400 of a wave of 49 records at 1,000,000 particles; the whole wave now takes 2550 for up
// to 64).  The kernel went from 169 to 137 us there.
template <class Filter, class Eval, class After>
__device__ __forceinline__ void mfma_pipeline(const WalkCtx &c, const uint16_t *hs, const float4 *P, uint32_t far,
                                              char *wave_lds, bool active, uint32_t hc, const float4 &p, float reach,
                                              float expand, Filter &&filter, Eval &&eval, After &&after) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    const uint32_t lane = __lane_id();
    uint32_t *ring = (uint32_t *)wave_lds, *out = ring + QRING;
    uint16_t *cand = (uint16_t *)(out + ORING);
    // the owner's side
    const float own_far = active ? p.w - (reach * reach * (1.0f + 1.0e-6f) + expand) : FAR_SQ;
    const float ax = active ? -2.0f * p.x : 0.f, ay = active ? -2.0f * p.y : 0.f, az = active ? -2.0f * p.z : 0.f;
    const f4 start = {quad_bcast<0>(own_far), quad_bcast<1>(own_far), quad_bcast<2>(own_far), quad_bcast<3>(own_far)};
    // the cells within reach of the quad's records: offsets in x and y from its row, halo cells in z
    uint32_t hh[3];
    c.Hs.decode(hc, hh[0], hh[1], hh[2]);
    const float pp[3] = {p.x, p.y, p.z};
    int lo[3], hi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float u = pp[a] - (float)((int)hh[a] - c.h[a]) * c.cs[a];  // position inside its cell
        // clamped in FP32 first (a huge reach selects the full stencil)
        const int l = min(0, (int)fmaxf(floorf((u - reach) * c.inv_cs[a]), -(float)c.radius));
        const int h = max(0, (int)fminf(floorf((u + reach) * c.inv_cs[a]), (float)c.radius));
        const int at = a == 2 ? (int)hh[2] : 0;
        lo[a] = quad_min(active ? at + l : 0x7FFFFF);
        hi[a] = quad_max(active ? at + h : -0x7FFFFF);
    }
    const bool any = hi[2] >= lo[2];  // the quad has an active record
    const uint32_t ny = (uint32_t)(hi[1] - lo[1] + 1), nz = (uint32_t)(hi[2] - lo[2] + 1);
    uint32_t left = any ? (uint32_t)(hi[0] - lo[0] + 1) * ny : 0u;  // rows of the quad not yet begun
    const uint32_t x_step = c.Hs.HH - (ny - 1u) * c.Hs.H2;
    uint32_t cur = any ? (uint32_t)((int)(hc - hh[2]) + lo[0] * (int)c.Hs.HH + lo[1] * (int)c.Hs.H2 + lo[2]) : 0u;
    uint32_t iy = ny;
    // The quads of a wave go through their rows together (a row's steps are those of the longest run of the
    // sixteen), which leaves a step little more than its products; rows of their own cost a step three times
    // the vector instructions and saved a fifth of the steps.  The next row's bounds are read ahead.
    uint32_t nq = left ? hs[cur] : 0u, nqe = left ? hs[cur + nz] : 0u;
    uint32_t q = 0, qe = 0;  // this lane's candidate and the end of the run
    bool more = __ballot(left != 0u) != 0ull;  // rows left
    // One loop with one copy of the filter and of the evaluation: walk until QSTEPS steps are done, harvest until the
    // ring holds a batch, sift a batch, evaluate a batch.
    uint32_t head = 0, tail = 0, ohead = 0, otail = 0;  // wave-uniform
    uint32_t bits = 0, n = 0;                           // pending result bits, tests of the last walk
    while (true) {
        if (!__ballot(bits != 0u)) {
            uint32_t s = 0;
            while (s < QSTEPS) {
                const bool in = q < qe;
                if (!__ballot(in)) {  // the next row
                    if (!more) break;
                    q = nq + (lane & 3u);
                    qe = nqe;
                    left = left ? left - 1u : 0u;
                    const bool turn = --iy == 0u;
                    cur += turn ? x_step : c.Hs.H2;
                    iy = turn ? ny : iy;
                    nq = left ? hs[cur] : 0u;
                    nqe = left ? hs[cur + nz] : 0u;
                    more = __ballot(left != 0u) != 0ull;
                    continue;
                }
                const uint32_t idx = in ? q : far;
                const float4 b = P[idx];
                cand[s * 16u + lane / 4] = (uint16_t)(q - (lane & 3u));  // the quad's first (one value, one place)
                q += 4;
                f4 d = __builtin_amdgcn_mfma_f32_4x4x1f32(ax, b.x, start, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_4x4x1f32(ay, b.y, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_4x4x1f32(az, b.z, d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_4x4x1f32(1.0f, b.w, d, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(d[r]), 31);
                ++s;
            }
            n = 4 * s;
        }
        // harvest: bit n - 1 - t is test t = 4 step + owner.  A lane's entries take consecutive places after those of
        // the lower lanes; when they do not fit, one from each lane as long as the ring is short of a batch.
        auto entry_of = [&]() -> uint32_t {  // the lowest pending bit's
            const uint32_t t = n - 1u - (uint32_t)__builtin_ctz(bits);
            bits &= bits - 1u;
            return (((lane & 60u) | (t & 3u)) << 16) | (cand[(t >> 2) * 16u + lane / 4] + (lane & 3u));
        };
        unsigned long long mk = __ballot(bits != 0u);
        if (mk && tail - head < 64) {
            const uint32_t cnt = (uint32_t)__popc(bits), incl = wave_inclusive_sum(cnt);
            const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            if (tail - head + all <= QRING) {
                uint32_t at = tail + incl - cnt;
                while (bits) ring[at++ & (QRING - 1)] = entry_of();
                tail += all;
                mk = 0ull;
            } else {
                while (mk && tail - head < 64) {
                    if (bits) {
                        const uint32_t at = tail + rank_in_mask(mk);
                        ring[at & (QRING - 1)] = entry_of();
                    }
                    tail += (uint32_t)__popcll(mk);
                    mk = __ballot(bits != 0u);
                }
            }
        }
        const bool last = !more && !mk && !__ballot(q < qe);
        if (tail - head >= 64 || (last && tail != head)) {
            const uint32_t k = min(64u, tail - head);
            wave_lds_sync();
            const uint32_t ent = ring[(head + lane) & (QRING - 1)];
            const bool ok = lane < k && filter(ent);
            const unsigned long long om = __ballot(ok);
            if (ok) out[(otail + rank_in_mask(om)) & (ORING - 1)] = ent;
            otail += (uint32_t)__popcll(om);
            head += k;
        }
        const bool flush = last && tail == head;
        if (otail - ohead >= 64 || (flush && otail != ohead)) {
            wave_lds_sync();
            eval(lane < otail - ohead ? out[(ohead + lane) & (ORING - 1)] : NO_ENTRY);
            ohead += min(64u, otail - ohead);
            wave_lds_sync();
        }
        const bool done = flush && otail == ohead;
        if (!after(done) && done) break;
    }
}

struct NoAfter {
    __device__ __forceinline__ bool operator()(bool) const { return false; }
};

// ---- per-block type tables, carved from dynamic LDS ahead of the staged records -----------------
// Staged bricks need n_types <= MAX_STAGED_TYPES (larger type counts take the slow path).
constexpr uint32_t MAX_STAGED_TYPES = 16;

__host__ __device__ inline size_t align16(size_t v) { return (v + 15) & ~(size_t)15; }

// bytes of the force tables for nt types and np potentials
__host__ __device__ inline size_t force_table_bytes(uint32_t nt, uint32_t np) {
    const size_t n2 = (size_t)nt * nt;
    return align16(sizeof(PairIdx) * n2) + align16(sizeof(PotDev) * np) + align16(4 * n2) + align16(4 * nt);
}

// bytes of the table region for nt types and np potentials: the force tables followed by the
// search tables (the fused forces + search kernel holds both; the others use one of them)
__host__ __device__ inline size_t table_bytes(uint32_t nt, uint32_t np) {
    const size_t n2 = (size_t)nt * nt;
    return force_table_bytes(nt, np) + align16(sizeof(RxPairIdx) * n2) + align16(4 * n2) + 2 * align16(4 * nt);
}

struct ForceTables {
    PairIdx *pidx;  // [nt * nt]
    PotDev *pots;   // [n_pots]
    float *thr;     // [nt * nt] prefilter thresholds
    float *reach;   // [nt] largest cutoff of the type's row plus rounding slack (< 0: no potentials)
};

struct SearchTables {
    RxPairIdx *o2;  // [nt * nt]
    float *thr;     // [nt * nt]
    float *reach;   // [nt] (< 0: no pair reactions)
    uint32_t *o1;   // [nt] order-1 reactions of the type: first entry of the list | number << 16 (the fused walk)
};

// reach of a type from the FP32 squared cutoffs of its row, widened like the prefilter
__device__ __forceinline__ float reach_of(float max_cut2_f, bool any, float margin) {
    return any ? sqrtf(max_cut2_f) * (1.0f + 1.0e-6f) + 2.0f * margin : -1.0f;
}

__device__ __forceinline__ ForceTables load_force_tables(char *base, const Tables &T, float margin) {
    const uint32_t nt = T.n_types, n2 = nt * nt;
    ForceTables t;
    char *p = base;
    t.pidx = (PairIdx *)p;
    p += align16(sizeof(PairIdx) * n2);
    t.pots = (PotDev *)p;
    p += align16(sizeof(PotDev) * T.n_pots);
    t.thr = (float *)p;
    p += align16(4 * n2);
    t.reach = (float *)p;
    for (uint32_t k = threadIdx.x; k < n2; k += BRICK_THREADS) {
        const PairIdx pi = T.pidx[k];
        t.pidx[k] = pi;
        t.thr[k] = prefilter_thr(pi.maxcut2_f, pi.count != 0, margin);
    }
    for (uint32_t k = threadIdx.x; k < T.n_pots; k += BRICK_THREADS) t.pots[k] = T.pots[k];
    if (threadIdx.x < nt) {
        float m2 = 0.f;
        bool any = false;
        for (uint32_t u = 0; u < nt; ++u) {
            const PairIdx pi = T.pidx[threadIdx.x * nt + u];
            if (pi.count) {
                any = true;
                m2 = fmaxf(m2, pi.maxcut2_f);
            }
        }
        t.reach[threadIdx.x] = reach_of(m2, any, margin);
    }
    __syncthreads();
    return t;
}

__device__ __forceinline__ SearchTables load_search_tables(char *base, const Tables &T, float margin) {
    const uint32_t nt = T.n_types, n2 = nt * nt;
    SearchTables t;
    char *p = base;
    t.o2 = (RxPairIdx *)p;
    p += align16(sizeof(RxPairIdx) * n2);
    t.thr = (float *)p;
    p += align16(4 * n2);
    t.reach = (float *)p;
    for (uint32_t k = threadIdx.x; k < n2; k += BRICK_THREADS) {
        const RxPairIdx pi = T.o2idx[k];
        t.o2[k] = pi;
        t.thr[k] = prefilter_thr(pi.maxr2_f, pi.count != 0, margin);
    }
    if (threadIdx.x < nt) {
        float m2 = 0.f;
        bool any = false;
        for (uint32_t u = 0; u < nt; ++u) {
            const RxPairIdx pi = T.o2idx[threadIdx.x * nt + u];
            if (pi.count) {
                any = true;
                m2 = fmaxf(m2, pi.maxr2_f);
            }
        }
        t.reach[threadIdx.x] = reach_of(m2, any, margin);
    }
    __syncthreads();
    return t;
}


// FP32 min image of a local-frame displacement on whole-axis axes (halo axes need none)
__device__ __forceinline__ void frame_min_image(uint32_t whole, const float *L, float &dx, float &dy, float &dz) {
    if (whole & 1u) dx = dx > .5f * L[0] ? dx - L[0] : (dx <= -.5f * L[0] ? dx + L[0] : dx);
    if (whole & 2u) dy = dy > .5f * L[1] ? dy - L[1] : (dy <= -.5f * L[1] ? dy + L[1] : dy);
    if (whole & 4u) dz = dz > .5f * L[2] ? dz - L[2] : (dz <= -.5f * L[2] ? dz + L[2] : dz);
}

// the pair sum reading neighbours from the bins (slow path for bricks that do not fit in LDS)
__device__ __forceinline__ void global_forces(const Grid &cur, const RepGeom &geo, uint32_t cap, int radius,
                                              const Tables &T, uint32_t s, const State &me, long long &fx,
                                              long long &fy, long long &fz, long long &e, long long *vir = nullptr) {
    const PairIdx *prow = T.pidx + (size_t)tw_type(me.tw) * T.n_types;
    const uint32_t cl = cell_of_slot(cur, s, cap) - geo.cell_base;
    for_each_stencil_slot(geo, cur, cap, radius, cl, [&](uint32_t s2) {
        if (s2 == s) return;
        const State o = cur.bins[s2];
        if (o.tw & (TW_DEAD | TW_OUTSIDE)) return;
        const PairIdx pi = prow[tw_type(o.tw)];
        if (pi.count == 0) return;
        const double dx = min_image(o.x - me.x, geo.box[0], geo.pbc[0]);
        const double dy = min_image(o.y - me.y, geo.box[1], geo.pbc[1]);
        const double dz = min_image(o.z - me.z, geo.box[2], geo.pbc[2]);
        const double d2 = dist2(dx, dy, dz);
        long long px, py, pz, pe;
        if (!pair_fixed(T.pots, pi, dx, dy, dz, d2, px, py, pz, pe)) return;
        fx += px;
        fy += py;
        fz += pz;
        e += pe;
        if (vir) pair_virial(T.pots, pi, dx, dy, dz, d2, vir);
    });
}

// block-wide sum of a fixed-point energy, one atomic per block
__device__ __forceinline__ void block_add_energy(ReplicaDev *reps, uint32_t r, long long e) {
    __shared__ long long s_e[BRICK_THREADS / 64];
    for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off);
    if (__lane_id() == 0) s_e[threadIdx.x / 64] = e;
    __syncthreads();
    if (threadIdx.x == 0) {
        long long t = 0;
        for (int w = 0; w < BRICK_THREADS / 64; ++w) t += s_e[w];
        if (t != 0) atomicAdd(&reps[r].energy, (unsigned long long)t);
    }
    __syncthreads();  // s_e may be written again by a following call
}

// block-wide sums of the nine fixed-point virial components, one atomic each per block
__device__ __forceinline__ void block_add_virial(unsigned long long *virial, uint32_t r, const long long v[9]) {
    __shared__ long long s_v[9][BRICK_THREADS / 64];
#pragma unroll
    for (int c = 0; c < 9; ++c) {
        long long x = v[c];
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
        if (__lane_id() == 0) s_v[c][threadIdx.x / 64] = x;
    }
    __syncthreads();
    if (threadIdx.x < 9) {
        long long t = 0;
        for (int w = 0; w < BRICK_THREADS / 64; ++w) t += s_v[threadIdx.x][w];
        if (t != 0) atomicAdd(&virial[9ull * r + threadIdx.x], (unsigned long long)t);
    }
    __syncthreads();
}

// one particle: bonded force, optional force output, integration and re-binning
template <int MODE>
__device__ __forceinline__ void finish_particle(const Grid &nxt, const ReplicaDev &R, const RepGeom &geo,
                                                const Tables &T, const Topo &topo, uint32_t cap, double dt,
                                                const double *noise, double *force_out, uint32_t s, State me,
                                                bool do_forces, long long fx, long long fy, long long fz,
                                                uint32_t *err) {
    if (do_forces && (me.tw & TW_TOPO) && topo.fb) {
        long long *fb = topo.fb + 3ull * (R.topo_base + me.h);
        fx += fb[0];
        fy += fb[1];
        fz += fb[2];
        fb[0] = 0;
        fb[1] = 0;
        fb[2] = 0;
    }
    if (do_forces && (fixed_saturated(fx) || fixed_saturated(fy) || fixed_saturated(fz)))
        atomicAdd(&err[ERR_FORCE_RANGE], 1u);
    const double Fx = (double)fx * FORCE_INV, Fy = (double)fy * FORCE_INV, Fz = (double)fz * FORCE_INV;
    if (MODE != MODE_REBIN && force_out && do_forces) {
        force_out[3ull * s] = Fx;
        force_out[3ull * s + 1] = Fy;
        force_out[3ull * s + 2] = Fz;
    }
    if (MODE == MODE_FORCES) return;
    State nw = me;
    nw.tw &= ~TW_NEW;
    if (MODE == MODE_STEP && R.active) {
        double xi[3];
        bd_noise(noise, me.h, R.step, R.seed, xi);
        const double Fv[3] = {Fx, Fy, Fz};
        double p[3] = {me.x, me.y, me.z};
        em_move(T, tw_type(me.tw), dt, Fv, xi, geo.box, geo.pbc, p, err);
        nw.x = p[0];
        nw.y = p[1];
        nw.z = p[2];
    }
    const uint32_t slot = bin_insert(nxt, geo, cap, nw, err, false, 0);
    if (slot != 0xFFFFFFFFu && (me.tw & TW_TOPO) && topo.loc) topo.loc[R.topo_base + me.h] = slot;
}

// the ci-th of the brick's own cells
__device__ __forceinline__ uint32_t own_cell(const BrickDev &B, uint32_t ci) {
    const uint32_t lz = ci % B.e[2], ly = (ci / B.e[2]) % B.e[1], lx = ci / (B.e[2] * B.e[1]);
    return B.cell_base + ((uint32_t)(B.o[0] + lx) * (uint32_t)B.dims[1] + (uint32_t)(B.o[1] + ly)) * (uint32_t)B.dims[2] +
           (uint32_t)(B.o[2] + lz);
}

// fn(cell) for the brick's own cells, spread over the block's threads
template <class Fn>
__device__ __forceinline__ void for_each_own_cell(const BrickDev &B, Fn &&fn) {
    const uint32_t ncell = (uint32_t)(B.e[0] * B.e[1] * B.e[2]);
    for (uint32_t ci = threadIdx.x; ci < ncell; ci += BRICK_THREADS) fn(own_cell(B, ci));
}

// What a staging capacity of max_states records leaves to the bin-reading path, a wave a brick: full[0] bricks, and
// full[1 + r] records of replica r in them.
__global__ void __launch_bounds__(BRICK_THREADS) k_brick_fill(const uint32_t *counts, const BrickDev *bricks, uint32_t nb,
                                                              uint32_t max_states, uint32_t *full) {
    const uint32_t b = blockIdx.x * BRICK_WAVES + threadIdx.x / 64;
    if (b >= nb) return;
    const BrickDev &B = bricks[b];
    const Halo Hs = make_halo(B);
    uint32_t sum = 0, own = 0;
    for (uint32_t c = __lane_id(); c < Hs.nh; c += 64) sum += load_halo_cells(counts, nullptr, B, Hs, c, 1).n[0];
    sum = (uint32_t)__builtin_amdgcn_readlane((int)wave_inclusive_sum(sum), 63);
    if (sum <= max_states) return;  // wave-uniform
    const uint32_t n_cells = (uint32_t)(B.e[0] * B.e[1] * B.e[2]);
    for (uint32_t ci = __lane_id(); ci < n_cells; ci += 64) own += counts[own_cell(B, ci)];
    own = wave_inclusive_sum(own);
    if (__lane_id() == 63) {
        atomicAdd(&full[0], 1u);
        atomicAdd(&full[1 + B.r], own);
    }
}

// visits the records of the brick's own cells straight from the bins: fn(slot, state), a slot a thread (a cell a
// thread left most of the block idle)
template <class Fn>
__device__ __forceinline__ void for_each_own_record(const Grid &cur, const BrickDev &B, uint32_t cap, Fn &&fn) {
    const uint32_t n_slots = (uint32_t)(B.e[0] * B.e[1] * B.e[2]) * cap;
    for (uint32_t i = threadIdx.x; i < n_slots; i += BRICK_THREADS) {
        const uint32_t cell = own_cell(B, i / cap), k = i % cap, n = cur.counts[cell];
        if (k < n) fn(cell * cap + k, cur.bins[cell * cap + k]);
        if (k == 0 && n > cap) {
            uint32_t no = *cur.ovf_count;
            no = no < cur.ovf_cap ? no : cur.ovf_cap;
            uint32_t seen = 0;
            for (uint32_t o = 0; o < no && seen < n - cap; ++o)
                if (cur.ovf_cell[o] == cell) {
                    ++seen;
                    fn(cur.nbin + o, cur.bins[cur.nbin + o]);
                }
        }
    }
}

struct ForceWave {  // per-wave LDS of k_brick
    unsigned long long acc[3][64];  // fixed-point force of the wave's 64 particles
    uint32_t quads[16];             // its quads (wave_quads)
    uint16_t j[64];                 // the particles' staged records
};

struct StepWave : ForceWave {  // per-wave LDS of k_brick_step
    uint32_t draw[128];        // its reaction candidates (entries of the pairs' kind)
};
constexpr uint32_t NO_PARTNER = 0xFFFFu;  // an order-1 candidate's entry

// Bricks whose halo does not fit in LDS are listed for a second kernel that reads neighbours
// straight from the bins.  list: [0] count, [1] blocks of the second kernel done, [2..] bricks.
__device__ __forceinline__ void list_slow_brick(uint32_t *list, uint32_t b, uint32_t *err) {
    if (threadIdx.x == 0) {
        list[2 + atomicAdd(&list[0], 1u)] = b;
        atomicAdd(&err[STAT_SLOW_BRICKS], 1u);
    }
}

// count of listed bricks; with none listed the second kernel's blocks exit at once (and nothing
// needs clearing)
__device__ __forceinline__ uint32_t slow_count(const uint32_t *list) {
    return __atomic_load_n(list, __ATOMIC_RELAXED);
}

// the last block of the second kernel clears the list for the next launch (every block has read
// the nonzero count before it counts itself done)
__device__ __forceinline__ void release_slow_list(uint32_t *list) {
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        if (atomicAdd(&list[1], 1u) == gridDim.x - 1) {
            list[0] = 0u;
            list[1] = 0u;
            __threadfence();
        }
    }
}

// forces (+ Euler-Maruyama + re-bin) of every particle of one brick; MODE as in k_fused.
// AH: the launch covers bricks brick0.. that are in halo mode on every axis (else: none is).
template <int MODE, bool AH>
__global__ __launch_bounds__(BRICK_THREADS) void k_brick(Grid cur, Grid nxt, Grid clear, ReplicaDev *reps, Tables T, Topo topo,
                                                         const BrickDev *bricks, uint32_t brick0, uint32_t cap,
                                                         int radius, double dt,
                                                         const double *noise, double *force_out, uint32_t max_states,
                                                         uint32_t max_halo, uint32_t smem_bytes, uint32_t *slow,
                                                         uint32_t *err, unsigned long long *virial) {
    extern __shared__ __align__(16) char smem[];
    __shared__ ForceWave wave_lds[BRICK_WAVES];
    const uint32_t bidx = brick0 + xcd_block(blockIdx.x, gridDim.x);
    const BrickDev B = bricks[bidx];
    const ReplicaDev &R = reps[B.r];
    if (MODE == MODE_REBIN) {  // the buffer after the target is cleared for the re-binning (or walk) that follows
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *nxt.wl_count = 0u;
            *clear.ovf_count = 0u;
        }
        for_each_own_cell(B, [&](uint32_t cell) { clear.counts[cell] = 0u; });
    }
    if (!R.in_use) return;
    if (MODE != MODE_FORCES) virial = nullptr;
    long long vir[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    const RepGeom geo = load_geom(R);
    const bool forces_on = MODE == MODE_FORCES || (MODE == MODE_STEP && R.active);
    if (!forces_on) {
        // re-bin only (neighbour-list update, or a replica whose step budget is spent): no staging
        for_each_own_record(cur, B, cap, [&](uint32_t s, const State &me) {
            if (!(me.tw & TW_DEAD))
                finish_particle<MODE_REBIN>(nxt, R, geo, T, topo, cap, dt, noise, force_out, s, me, false, 0, 0, 0,
                                            err);
        });
        return;
    }
    long long e_blk = 0;
    uint32_t total = 0xFFFFFFFFu;
    const uint32_t nt = T.n_types;
    BrickSmem m;
    ForceTables ft;
    const Frame F = make_frame(B, geo);
    const Halo Hs = make_halo(B);
    if (nt <= MAX_STAGED_TYPES) {
        if (table_bytes(nt, T.n_pots) + brick_smem_bytes(max_states, max_halo) > smem_bytes) {  // block-uniform
            if (threadIdx.x == 0) atomicAdd(&err[ERR_LDS_LAYOUT], 1u);
            return;
        }
        ft = load_force_tables(smem, T, F.margin);
        m = carve(smem + table_bytes(nt, T.n_pots), max_states, max_halo);
        total = stage_brick(cur, B, geo, F, cap, m, max_states, Hs,
                            load_halo_cells(cur.counts, nullptr, B, Hs, threadIdx.x * cells_per_thread(Hs),
                                            min(cells_per_thread(Hs), STAGE_CELLS)));
    }
    if (total != 0xFFFFFFFFu) {
        const WalkCtx wc = make_walk(B, geo, Hs, radius);
        if (AH != (wc.whole == 0)) {  // launch and brick disagree (host invariant): refuse the brick
            if (threadIdx.x == 0) atomicAdd(&err[ERR_LDS_LAYOUT], 1u);
            return;
        }
        ForceWave &W = wave_lds[threadIdx.x / 64];
        const uint32_t lane = __lane_id();
        // the exact pair force of a survivor (entry = owner lane << 16 | staged neighbour)
        auto eval = [&](uint32_t ent) {
            if (ent == NO_ENTRY) return;
            const uint32_t ol = ent >> 16, q = ent & 0xFFFFu;
            const State me = cur.bins[m.slot[W.j[ol]]];
            const State o = cur.bins[m.slot[q]];
            const PairIdx pi = ft.pidx[tw_type(me.tw) * nt + tw_type(o.tw)];
            // CPUCalculateForces.cpp:226-259: x_ij = shortestDifference(x_i, x_j), gate d2 < rc^2
            const double ddx = min_image(o.x - me.x, geo.box[0], geo.pbc[0]);
            const double ddy = min_image(o.y - me.y, geo.box[1], geo.pbc[1]);
            const double ddz = min_image(o.z - me.z, geo.box[2], geo.pbc[2]);
            const double d2 = dist2(ddx, ddy, ddz);
            long long px, py, pz, pe;
            bool saturated;
            if (!pair_fixed(ft.pots, pi, ddx, ddy, ddz, d2, px, py, pz, pe, &saturated)) return;
            if (saturated) atomicAdd(&err[ERR_FORCE_RANGE], 1u);
            atomicAdd(&W.acc[0][ol], (unsigned long long)px);
            atomicAdd(&W.acc[1][ol], (unsigned long long)py);
            atomicAdd(&W.acc[2][ol], (unsigned long long)pz);
            e_blk += pe;
            if (virial) pair_virial(ft.pots, pi, ddx, ddy, ddz, d2, vir);
        };
        auto rounds = [&]() {
            for (uint32_t q0 = threadIdx.x / 64 * 16;; q0 += BRICK_THREADS / 4) {  // wave-uniform
                const uint32_t n_quads = wave_quads(m, B, Hs, W.quads, q0);
                if (q0 >= n_quads) break;
                wave_lds_sync();
                const OwnerLane ow = owner_lane(m, W.quads, q0, n_quads);
                const uint32_t j = ow.j;
                const bool valid = ow.valid;
                State me{};
                uint32_t sj = 0;
                if (valid) {
                    sj = m.slot[j];
                    me = cur.bins[sj];
                }
                W.j[lane] = (uint16_t)j;
                W.acc[0][lane] = 0ull;
                W.acc[1][lane] = 0ull;
                W.acc[2][lane] = 0ull;
                wave_lds_sync();
                const float4 pj = m.P[j];
                const uint32_t t = ow.t & TYP_MASK;
                const float reach = ft.reach[t];
                const bool active = valid && !(ow.t & TYP_OUTSIDE) && reach >= 0.f;
                char *wave_ring = m.rings + (threadIdx.x / 64) * WAVE_RING_BYTES;
                if constexpr (AH) {
                    auto filter = [&](uint32_t ent) -> bool {
                        const uint32_t q = ent & 0xFFFFu, jo = W.j[ent >> 16];
                        const float4 a = m.P[jo], b = m.P[q];
                        return (q != jo) &
                               (prefilter_d2(b.x - a.x, b.y - a.y, b.z - a.z) < ft.thr[m.typ[jo] * nt + m.typ[q]]);
                    };
                    mfma_pipeline(wc, m.hstart, m.P, m.far, wave_ring, active, m.hc_of[j], pj, reach, F.expand, filter,
                                  eval, NoAfter{});
                } else {
                    const float *thr_row = ft.thr + t * nt;
                    // prefilter, branch-free: one LDS read of the candidate, one of the threshold
                    auto keep = [&](uint32_t q, const float4 &pq) -> bool {
                        const uint32_t tq = m.typ[q];
                        float dx = pq.x - pj.x, dy = pq.y - pj.y, dz = pq.z - pj.z;
                        frame_min_image(F.whole, F.L, dx, dy, dz);
                        return (q != j) & (tq < TYP_OUTSIDE) & (prefilter_d2(dx, dy, dz) < thr_row[tq & TYP_MASK]);
                    };
                    pair_pipeline(wc, m.hstart, m.P, (uint32_t *)wave_ring, active, m.hc_of[j], keep, eval);
                }
                wave_lds_sync();
                if (valid)
                    finish_particle<MODE>(nxt, R, geo, T, topo, cap, dt, noise, force_out, sj, me, true,
                                          (long long)W.acc[0][lane], (long long)W.acc[1][lane],
                                          (long long)W.acc[2][lane], err);
                wave_lds_sync();
            }
        };
        rounds();
        block_add_energy(reps, B.r, e_blk);
        if (virial) block_add_virial(virial, B.r, vir);
    } else {
        list_slow_brick(slow, bidx, err);
    }
}

// the listed bricks of k_brick, neighbours read straight from the bins
template <int MODE>
__global__ __launch_bounds__(BRICK_THREADS) void k_brick_slow(Grid cur, Grid nxt, ReplicaDev *reps, Tables T,
                                                              Topo topo, const BrickDev *bricks, uint32_t cap,
                                                              int radius, double dt, const double *noise,
                                                              double *force_out, uint32_t *slow, uint32_t *err,
                                                              unsigned long long *virial) {
    const uint32_t n = slow_count(slow);
    if (n == 0) return;  // grid-uniform
    if (MODE != MODE_FORCES) virial = nullptr;
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {  // block-uniform
        const BrickDev B = bricks[slow[2 + i]];
        const ReplicaDev &R = reps[B.r];
        const RepGeom geo = load_geom(R);
        long long e_blk = 0;
        long long vir[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        for_each_own_record(cur, B, cap, [&](uint32_t s, const State &me) {
            if (me.tw & TW_DEAD) return;
            long long fx = 0, fy = 0, fz = 0, e = 0;
            if (!(me.tw & TW_OUTSIDE))
                global_forces(cur, geo, cap, radius, T, s, me, fx, fy, fz, e, virial ? vir : nullptr);
            e_blk += e;
            finish_particle<MODE>(nxt, R, geo, T, topo, cap, dt, noise, force_out, s, me, true, fx, fy, fz, err);
        });
        block_add_energy(reps, B.r, e_blk);
        if (virial) block_add_virial(virial, B.r, vir);
    }
    release_slow_list(slow);
}

struct SearchWave {  // per-wave LDS of k_brick_search
    uint32_t quads[16];
    uint16_t j[64];  // staged records of the wave's 64 particles
};

// reaction candidate search of one brick on the current buffer (see search_one for the rules)
template <bool AH>
__global__ __launch_bounds__(BRICK_THREADS) void k_brick_search(Grid cur, ReplicaDev *reps, Tables T,
                                                                const BrickDev *bricks, uint32_t brick0,
                                                                uint32_t cap,
                                                                int radius, int handler, Event *events,
                                                                uint32_t *ev_count, uint32_t max_states,
                                                                uint32_t max_halo, uint32_t smem_bytes, uint32_t *slow,
                                                                uint32_t *err) {
    extern __shared__ __align__(16) char smem[];
    __shared__ SearchWave wave_lds[BRICK_WAVES];
    const uint32_t bidx = brick0 + xcd_block(blockIdx.x, gridDim.x);
    const BrickDev B = bricks[bidx];
    const ReplicaDev &R = reps[B.r];
    const RepGeom geo = load_geom(R);
    if (replica_handler(R, handler) > 1 || !R.in_use || !R.active) return;
    const uint32_t nt = T.n_types;
    if (!T.has_o2 && T.o1idx[nt] == 0) return;  // no reactions
    const Frame F = make_frame(B, geo);
    const Halo Hs = make_halo(B);
    uint32_t total = 0xFFFFFFFFu;
    BrickSmem m;
    SearchTables st;
    if (nt <= MAX_STAGED_TYPES) {
        if (table_bytes(nt, T.n_pots) + brick_smem_bytes(max_states, max_halo) > smem_bytes) {  // block-uniform
            if (threadIdx.x == 0) atomicAdd(&err[ERR_LDS_LAYOUT], 1u);
            return;
        }
        st = load_search_tables(smem, T, F.margin);
        m = carve(smem + table_bytes(nt, T.n_pots), max_states, max_halo);
        total = stage_brick(cur, B, geo, F, cap, m, max_states, Hs,
                            load_halo_cells(cur.counts, nullptr, B, Hs, threadIdx.x * cells_per_thread(Hs),
                                            min(cells_per_thread(Hs), STAGE_CELLS)));
    }
    if (total == 0xFFFFFFFFu) {
        list_slow_brick(slow, bidx, err);
        return;
    }
    const uint32_t r = B.r, step = R.step;
    const uint64_t seed = R.seed;
    auto emit = [&](uint32_t rx, uint32_t s1, uint32_t s2, uint32_t h1, uint32_t h2, unsigned long long key) {
        uint32_t p = atomicAdd(&ev_count[r], 1u);
        if (p < R.ev_cap) {
            Event ev;
            ev.key = key;
            ev.s1 = s1;
            ev.s2 = s2;
            ev.h1 = h1;
            ev.h2 = h2;
            ev.rx = rx;
            ev.pad = 0;
            events[R.ev_base + p] = ev;
        } else {
            atomicAdd(&err[ERR_EVENT_OVERFLOW], 1u);
        }
    };
    const WalkCtx wc = make_walk(B, geo, Hs, radius);
    if (AH != (wc.whole == 0)) {  // launch and brick disagree (host invariant): refuse the brick
        if (threadIdx.x == 0) atomicAdd(&err[ERR_LDS_LAYOUT], 1u);
        return;
    }
    SearchWave &W = wave_lds[threadIdx.x / 64];
    const uint32_t lane = __lane_id();
    // the exact test and draws of a surviving pair (entry = owner lane << 16 | staged neighbour)
    auto eval = [&](uint32_t ent) {
        if (ent == NO_ENTRY) return;
        const uint32_t ol = ent >> 16, q = ent & 0xFFFFu;
        const uint32_t s1 = m.slot[W.j[ol]], s2 = m.slot[q];
        const State me = cur.bins[s1];
        const State o = cur.bins[s2];
        const uint32_t mh = me.h, t = tw_type(me.tw);
        const RxPairIdx pi = st.o2[t * nt + tw_type(o.tw)];
        // distSquared(neighbor.pos, entry.pos) (CPUUncontrolledApproximation.cpp:108)
        const double ddx = min_image(me.x - o.x, geo.box[0], geo.pbc[0]);
        const double ddy = min_image(me.y - o.y, geo.box[1], geo.pbc[1]);
        const double ddz = min_image(me.z - o.z, geo.box[2], geo.pbc[2]);
        const double d2 = dist2(ddx, ddy, ddz);
        const uint32_t lo = mh < o.h ? mh : o.h, hi = mh < o.h ? o.h : mh;
        for (uint32_t p = 0; p < pi.count; ++p) {
            const uint32_t rx = T.o2list[pi.start + p];
            const RxDev X = T.rx[rx];
            if (!(X.rate > 0 && d2 < X.educt_dist2)) continue;
            uint32_t x4[4];
            philox(lo, step, 2u | (rx << 8), hi, seed, x4);
            if (!(u53(x4[0], x4[1]) < X.p_accept)) continue;
            // entry1: the educt of type educts[0]; equal educt types: the lower handle
            const bool me_first = (X.educts[0] != X.educts[1]) ? (t == X.educts[0]) : (mh < o.h);
            if (me_first) emit(rx, s1, s2, mh, o.h, event_words(x4));
            else emit(rx, s2, s1, o.h, mh, event_words(x4));
        }
    };
    auto rounds = [&]() {
        for (uint32_t q0 = threadIdx.x / 64 * 16;; q0 += BRICK_THREADS / 4) {  // wave-uniform
            const uint32_t n_quads = wave_quads(m, B, Hs, W.quads, q0);
            if (q0 >= n_quads) break;
            wave_lds_sync();
            const OwnerLane ow = owner_lane(m, W.quads, q0, n_quads);
            const uint32_t j = ow.j;
            const bool valid = ow.valid;
            State me{};
            uint32_t sj = 0;
            if (valid) {
                sj = m.slot[j];
                me = cur.bins[sj];
            }
            const uint32_t t = tw_type(me.tw);
            if (valid) {  // order 1 (CPUUncontrolledApproximation.cpp:81-95)
                for (uint32_t k = T.o1idx[t]; k < T.o1idx[t + 1]; ++k) {
                    const uint32_t rx = T.o1list[k];
                    const RxDev X = T.rx[rx];
                    if (!(X.rate > 0)) continue;
                    uint32_t x4[4];
                    philox(me.h, step, 1u | (rx << 8), 0u, seed, x4);
                    if (!(u53(x4[0], x4[1]) < X.p_accept)) continue;
                    emit(rx, sj, sj, me.h, me.h, event_words(x4));
                }
            }
            if (!T.has_o2) continue;  // block-uniform
            W.j[lane] = (uint16_t)j;
            wave_lds_sync();
            const float4 pj = m.P[j];
            const float reach = st.reach[t];
            const bool active = valid && !(me.tw & TW_OUTSIDE) && reach >= 0.f;
            char *wave_ring = m.rings + (threadIdx.x / 64) * WAVE_RING_BYTES;
            // each unordered pair once: the lower type finds it; equal types: the lower bin slot
            // (which also excludes the particle itself); branch-free
            if constexpr (AH) {
                auto filter = [&](uint32_t ent) -> bool {
                    const uint32_t q = ent & 0xFFFFu, ol = ent >> 16, jo = W.j[ol];
                    const float4 a = m.P[jo], b = m.P[q];
                    const uint32_t t1 = m.typ[jo], t2 = m.typ[q];
                    return ((t2 > t1) | ((t2 == t1) & (m.slot[q] > m.slot[W.j[ol]]))) &
                           (prefilter_d2(b.x - a.x, b.y - a.y, b.z - a.z) < st.thr[t1 * nt + t2]);
                };
                mfma_pipeline(wc, m.hstart, m.P, m.far, wave_ring, active, m.hc_of[j], pj, reach, F.expand, filter, eval,
                              NoAfter{});
            } else {
                const float *thr_row = st.thr + t * nt;
                auto keep = [&](uint32_t q, const float4 &pq) -> bool {
                    const uint32_t tq = m.typ[q], t2 = tq & TYP_MASK;
                    float dx = pq.x - pj.x, dy = pq.y - pj.y, dz = pq.z - pj.z;
                    frame_min_image(F.whole, F.L, dx, dy, dz);
                    const float d2p = prefilter_d2(dx, dy, dz);
                    const float thr = thr_row[t2];
                    const uint32_t sq = m.slot[q];
                    return ((t2 > t) | ((t2 == t) & (sq > sj))) & (tq < TYP_OUTSIDE) & (d2p < thr);
                };
                pair_pipeline(wc, m.hstart, m.P, (uint32_t *)wave_ring, active, m.hc_of[j], keep, eval);
            }
            wave_lds_sync();
        }
    };
    rounds();
}

// the listed bricks of k_brick_search, searched straight from the bins
__global__ __launch_bounds__(BRICK_THREADS) void k_brick_search_slow(Grid cur, ReplicaDev *reps, Tables T,
                                                                     const BrickDev *bricks, uint32_t cap, int radius,
                                                                     Event *events, uint32_t *ev_count,
                                                                     uint32_t *slow, uint32_t *err) {
    const uint32_t n = slow_count(slow);
    if (n == 0) return;  // grid-uniform
    for (uint32_t i = blockIdx.x; i < n; i += gridDim.x) {
        const BrickDev B = bricks[slow[2 + i]];
        for_each_own_record(cur, B, cap, [&](uint32_t s, const State &me) {
            if (!(me.tw & TW_DEAD))
                search_one(cur, reps, T, cap, radius, 0, events, ev_count, nullptr, 0, s, me, err);
        });
    }
    release_slow_list(slow);
}

}  // namespace rdy
