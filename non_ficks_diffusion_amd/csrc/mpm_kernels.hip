// gfx950 kernels of the MPM snow substep, for a batch of scenes.
//
// Layout in HBM:
//   particles  field-major FP32 arrays (X[D], V[D], F[D*D], Jp, m, V0) of
//              capacity pcap, double buffered, with a scene id per particle;
//              after binning they are grouped by home block (so by scene,
//              then block, then cell) and every block's particles are one
//              contiguous range.
//   grid       block-sparse: each scene's padded domain is cut into 4^3
//              (3D) or 8^2 (2D) node blocks; the scenes' dense slot tables
//              are concatenated and map block coordinates to a compacted
//              ordinal; every node channel is an array of ordinal*64 + local
//              node entries.  Scene parameters are looked up per block.
//   tiles      per active block, the (B+2)^D node tile (block plus a
//              one-node halo) of each scattered channel.
// Block kernels (P2G, force, CG operator, G2P) run one work-group per
// active block.  A block's particles touch only its nodes and the one-node
// halo, so scatters accumulate into LDS tiles and the work-group writes
// the whole tile to the tile buffer with plain stores; the next node kernel
// sums, for every node, the (at most 2^D) tiles that cover it in a fixed
// order.  There are no global atomics on the scatter path, and the
// cross-block sum is deterministic.  Gathers load the tile once from the
// 3^D neighbour blocks.  Node kernels run one wave per block.  Reductions sum a
// scene's partials in a fixed order: G2P's max speed in a kernel of one
// work-group per scene, the CG's dot products and norms within the launch that
// forms them (k_cg_node, k_cg_solve).
#include "mpm_kernels.h"
#include <algorithm>

namespace mpm {

template <int D>
struct PF {
    // MAT: the particle's material entry (int bits); J holds the density of EOS particles
    static constexpr int X = 0, V = D, F = 2 * D, J = 2 * D + D * D, M = J + 1, VOL = J + 2, MAT = J + 3, N = J + 4;
};

// Work-groups are dispatched round-robin over the 8 XCDs (work-group w runs
// on XCD w % 8).  Block loops give each XCD one contiguous eighth of the
// active blocks, so every XCD has work whatever the block count, and
// neighbouring blocks (which share halo nodes) meet in the same L2.
// Requires gridDim.x % 8 == 0.
struct XcdRange {
    int first, end, step;
};
__device__ inline XcdRange xcd_blocks(int n) {
    const int x = (int)(blockIdx.x & 7), k = (int)(blockIdx.x >> 3);
    const int lo = (int)(((int64_t)n * x) >> 3), hi = (int)(((int64_t)n * (x + 1)) >> 3);
    return {lo + k, hi, (int)(gridDim.x >> 3)};
}
// Node loops: one wave per block (lane = node), over the same per-XCD block
// range as the block kernels, so a node kernel reads the tiles its XCD's
// block kernel wrote.
__device__ inline XcdRange xcd_wave_blocks(int n) {
    constexpr int W = WG / 64;
    const int x = (int)(blockIdx.x & 7), k = (int)(blockIdx.x >> 3);
    const int lo = (int)(((int64_t)n * x) >> 3), hi = (int)(((int64_t)n * (x + 1)) >> 3);
    return {lo + k * W + (int)(threadIdx.x >> 6), hi, (int)(gridDim.x >> 3) * W};
}

// Accesses of data that work-groups on different XCDs exchange inside one
// kernel: relaxed atomics at device scope, so that a load never hits a stale
// line of its XCD's L2 and a store reaches memory without a write-back of the
// whole cache (a release fence at device scope is one per work-group).
__device__ inline float ld_agent(const float* a) { return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline double ld_agent(const double* a) { return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline int ld_agent(const int* a) { return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void st_agent(float* a, float v) { __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void st_agent(double* a, double v) { __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void st_agent(int* a, int v) { __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline int add_agent(int* a, int v) { return __hip_atomic_fetch_add(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <bool AGENT, class T>
__device__ inline T ld(const T* a) {
    if constexpr (AGENT) return ld_agent(a);
    else return *a;
}
template <bool AGENT, class T>
__device__ inline void st(T* a, T v) {
    if constexpr (AGENT) st_agent(a, v);
    else *a = v;
}

// A place for a partial of k_cg_solve that has not been written: a NaN no
// arithmetic yields.
constexpr unsigned long long CG_EMPTY = 0x7ff8c0dec0dec0deull;
// The same for a float that is its own flag; what is stored there goes through
// `flagged`.
constexpr unsigned CG_EMPTY_FLOAT = 0x7fc0dec0u;
__device__ inline bool is_empty(float v) { return __float_as_uint(v) == CG_EMPTY_FLOAT; }
__device__ inline float flagged(float v) { return v == v ? v : __uint_as_float(0x7fc00000u); }
// k_cg_solve's force tile of block b in an iteration of parity k
template <int D>
__device__ inline float* cg_tile(const KP& p, int k, int b) {
    return p.cg_tiles + ((int64_t)(k & 1) * min(p.bcap, CG_RESIDENT) + b) * (D * Dims<D>::TN);
}

// Active block b holds no particles (a halo block of its neighbours).
__device__ inline bool block_empty(const KP& p, int b) { return p.block_pstart[b + 1] == p.block_pstart[b]; }

// Scene of a global slot (slot ranges of an arena are not in scene order).
__device__ inline int scene_of_slot(const KP& p, int slot) { return p.slot_scene[slot]; }

template <int D>
__device__ inline void slot_coords(int slot, int nb, int* b) {
    if constexpr (D == 3) {
        b[2] = slot % nb;
        b[1] = (slot / nb) % nb;
        b[0] = slot / (nb * nb);
    } else {
        b[1] = slot % nb;
        b[0] = slot / nb;
    }
}

// Coordinates of active block b in its scene's slot grid (written by
// k_block_setup; a load instead of the slot index's divisions).
template <int D>
__device__ inline void block_coords(const KP& p, int b, int* bb) {
#pragma unroll
    for (int a = 0; a < D; ++a) bb[a] = p.block_org[b * 3 + a];
}

template <int D>
__device__ inline void local_coords(int l, int* lc) {
    if constexpr (D == 3) { lc[0] = l >> 4; lc[1] = (l >> 2) & 3; lc[2] = l & 3; }
    else { lc[0] = l >> 3; lc[1] = l & 7; }
}

// tile index -> (neighbour ordinal in 0..3^D-1, local node in 0..63, tile coords)
template <int D>
__device__ inline void tile_map(int t, int& nbr, int& local, int* tc) {
    using Dm = Dims<D>;
    constexpr int TE = Dm::TE, B = Dm::B;
    if constexpr (D == 3) {
        tc[0] = t / (TE * TE);
        tc[1] = (t / TE) % TE;
        tc[2] = t % TE;
    } else {
        tc[0] = t / TE;
        tc[1] = t % TE;
    }
    nbr = 0;
    local = 0;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        const int o = tc[a] == 0 ? 0 : (tc[a] == TE - 1 ? 2 : 1);
        const int l = tc[a] - 1 - B * (o - 1);
        nbr = nbr * 3 + o;
        local = local * B + l;
    }
}

// stencil offsets of node s (last axis fastest) -> LDS tile index of that node for local cell l
template <int D>
__device__ inline int tile_index(const int* l, int s, int* off) {
    using Dm = Dims<D>;
    if constexpr (D == 3) {
        off[0] = s / 9;
        off[1] = (s / 3) % 3;
        off[2] = s % 3;
        return (l[0] + off[0]) * Dm::LX + (l[1] + off[1]) * Dm::LY + (l[2] + off[2]);
    } else {
        off[0] = s / 3;
        off[1] = s % 3;
        return (l[0] + off[0]) * Dm::LX + (l[1] + off[1]);
    }
}

// LDS index of tile node tc (tile coordinates 0..TE-1)
template <int D>
__device__ inline int lds_index(const int* tc) {
    using Dm = Dims<D>;
    if constexpr (D == 3) return tc[0] * Dm::LX + tc[1] * Dm::LY + tc[2];
    else return tc[0] * Dm::LX + tc[1];
}

// Weight (Tools/Influence_Iterator.h:85-90): left-to-right product over axes.
template <int D>
__device__ inline float stencil_weight(const float (*w)[3], const int* off) {
#pragma clang fp contract(off)
    float r = w[0][off[0]];
#pragma unroll
    for (int a = 1; a < D; ++a) r = r * w[a][off[a]];
    return r;
}
// Weight_Gradient (Tools/Influence_Iterator.h:92-99)
template <int D>
__device__ inline void stencil_grad(const float (*w)[3], const float (*dw)[3], const int* off, float* g) {
#pragma clang fp contract(off)
#pragma unroll
    for (int i = 0; i < D; ++i) {
        float r = (i == 0) ? dw[0][off[0]] : w[0][off[0]];
#pragma unroll
        for (int j = 1; j < D; ++j) r = r * ((i == j) ? dw[j][off[j]] : w[j][off[j]]);
        g[i] = r;
    }
}

// Weights of particle i and its cell relative to block bb.  Returns false
// (and the caller skips the particle) when the cell is not inside the block,
// which can only happen if particles moved after the last binning; no tile
// index outside [0, B+1]^D is ever formed.
template <int D>
__device__ inline bool particle_weights(const KP& p, const SceneParams& sc, int i, const int* bb, float (*w)[3],
                                        float (*dw)[3], int* l, float* X) {
    constexpr int B = Dims<D>::B;
    bool ok = true;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        X[a] = p.pcur[(PF<D>::X + a) * p.pcap + i];
        int c;
        bspline_weights(X[a], sc.dx, sc.inv_dx, c, w[a], dw[a]);
        l[a] = c + B - B * bb[a];
        ok = ok && l[a] >= 0 && l[a] < B;
    }
    return ok;
}

// Sum, for node n, of channel c over every tile covering it, in a fixed
// order.  Blocks without particles write no tile (their contribution is
// zero) and are absent from the tile neighbour table.  With crop_ghost_x, nodes whose x index is outside [0, counts-1]
// receive nothing (the reference's slab crop,
// Tools/Cropped_Influence_Iterator.h:31-42).
// tile_of(o): entry o of that table for the node's block.  WAIT: the tiles
// (k_cg_solve's) are written meanwhile, a value is there once it is not empty.
template <int D, int C, bool AGENT, bool WAIT, class TileOf>
__device__ inline void gather_tiles(const KP& p, const SceneParams& sc, int n, const float* tiles, TileOf&& tile_of, float* out) {
    using Dm = Dims<D>;
    constexpr int B = Dm::B, TE = Dm::TE, TN = Dm::TN;
    const int b = n >> 6;
    int lc[D];
    local_coords<D>(n & 63, lc);
    // per axis: option 0 is the node's own block; a node on a block face
    // also lies in the face neighbour's tile (option 1)
    int od1[D], td0[D], td1[D], face = 0;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        td0[a] = lc[a] + 1;
        face |= (lc[a] == 0 || lc[a] == B - 1) ? 1 << (D - 1 - a) : 0;
        od1[a] = lc[a] == 0 ? 0 : 2;
        td1[a] = lc[a] == 0 ? TE - 1 : 0;
    }
    // every candidate tile's neighbour entry, then every tile value, is
    // loaded before the first sum (no load waits on another candidate's);
    // candidate m takes option 1 on the axes of its set bits, and the sum
    // runs over the candidates in lexicographic option order
    constexpr int NC = 1 << D;
    int blk[NC];
#pragma unroll
    for (int m = 0; m < NC; ++m) {
        int o = 0;
#pragma unroll
        for (int a = 0; a < D; ++a) o = o * 3 + (((m >> (D - 1 - a)) & 1) ? od1[a] : 1);
        const int e = tile_of(o);  // o is an entry of the table whether or not it is used
        blk[m] = (m & ~face) == 0 ? e : -1;
    }
    // a candidate on the node's faces loads even where its block wrote no
    // tile (from block 0's slot, in bounds, and not summed), so that no sum
    // shares its load's condition and none is scheduled ahead of the loads
    float v[NC][C];
    bool waiting;
    do {
#pragma unroll
        for (int m = 0; m < NC; ++m) {
            int t = 0;
#pragma unroll
            for (int a = 0; a < D; ++a) t = t * TE + (((m >> (D - 1 - a)) & 1) ? td1[a] : td0[a]);
#pragma unroll
            for (int c = 0; c < C; ++c) v[m][c] = 0.0f;
            if ((m & ~face) == 0) {
                const float* src = tiles + (int64_t)max(blk[m], 0) * C * TN + t;
#pragma unroll
                for (int c = 0; c < C; ++c) v[m][c] = ld<AGENT>(src + c * TN);
            }
        }
        waiting = false;
        if (WAIT) {
#pragma unroll
            for (int m = 0; m < NC; ++m)
#pragma unroll
                for (int c = 0; c < C; ++c) waiting |= blk[m] >= 0 && is_empty(v[m][c]);
        }
        // (a short rest: polling without one slowed the stores it waits for)
        if (WAIT && __any(waiting)) __builtin_amdgcn_s_sleep(4);
    } while (WAIT && __any(waiting));
    // the crop test's loads go out with the tile loads (a cropped node sums
    // nothing)
    bool keep = true;
    {
        const int crop = sc.crop_ghost_x, counts = sc.counts;
        int bb[D];
        block_coords<D>(p, b, bb);
        const int ix = B * bb[0] + lc[0] - B;
        keep = (crop == 0) | ((ix >= 0) & (ix <= counts - 1));
    }
#pragma unroll
    for (int c = 0; c < C; ++c) out[c] = 0.0f;
#pragma unroll
    for (int m = 0; m < NC; ++m)
        if (keep && blk[m] >= 0) {
#pragma unroll
            for (int c = 0; c < C; ++c) out[c] += v[m][c];
        }
}
template <int D, int C, bool AGENT = false>
__device__ inline void gather_node_tiles(const KP& p, const SceneParams& sc, int n, float* out) {
    const int* nbr = p.block_tnbr + (int64_t)(n >> 6) * Dims<D>::NBR;
    gather_tiles<D, C, AGENT, false>(p, sc, n, p.tiles, [&](int o) { return nbr[o]; }, out);
}

__device__ inline bool inside_plane(const SceneParams& sc, int id, const float* x, int D) {
    float s = 0.0f;
    for (int a = 0; a < D; ++a) s += (x[a] - sc.ps[id][a]) * sc.pn[id][a];
    return s < 0.0f;
}

template <int D>
__device__ inline void node_center(const KP& p, const SceneParams& sc, int n, float* x) {
    constexpr int B = Dims<D>::B;
    int bb[D], lc[D];
    block_coords<D>(p, n >> 6, bb);
    local_coords<D>(n & 63, lc);
#pragma unroll
    for (int a = 0; a < D; ++a) {
        const int i = B * bb[a] + lc[a] - B;
        x[a] = ((float)i + 0.5f) * sc.dx;
    }
}

// ============================================================================
// Binning: key = global slot*64 + cell of the home cell, rank within the
// cell, activation marks of the home block's 3^D neighbourhood.  Empty and
// removed entries carry key -1.
// ============================================================================
template <int D>
__global__ __launch_bounds__(WG) void k_bin(KP p) {
    constexpr int B = Dims<D>::B;
    const int n = p.ctr->n_live;
    const int lane = threadIdx.x & 63;
    // whole waves iterate together so the ballots below are convergent
    for (int base = blockIdx.x * WG + (threadIdx.x & ~63); base < n; base += gridDim.x * WG) {
        const int i = base + lane;
        // the key, scene and position load together (a lane past the end
        // reads the last particle and is not valid), then the scene's
        // parameters (scene 0's for a lane that is not live); no branch
        // separates them, so no load waits on another
        const int ic = min(i, n - 1);
        const int key0 = p.keycur[ic], si0 = p.scur[ic];
        float X[D];
#pragma unroll
        for (int a = 0; a < D; ++a) X[a] = p.pcur[(PF<D>::X + a) * p.pcap + ic];
        const bool live = i < n && key0 >= 0;
        const int si = live ? si0 : 0;
        const SceneParams& sc = p.scn[si];
        const float inv_dx = sc.inv_dx;
        const int counts = sc.counts, nb = sc.nb, slot_base = sc.slot_base;
        bool finite = true;
#pragma unroll
        for (int a = 0; a < D; ++a) finite = finite & (bool)isfinite(X[a]);
        int c[D];
        bool valid = live && finite;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            c[a] = finite ? cell_of(X[a], inv_dx) : -1;
            valid = valid & (c[a] >= 0) & (c[a] <= counts - 1);
        }
        if (live && !valid) {
            p.keycur[i] = -1;
            if (!finite) atomicOr(&p.sst[si].nonfinite, 1);
        }
        int slot = -1, key = -1;
        if (valid) {
            int local = 0, cell = 0;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                local = local * nb + (c[a] + B) / B;
                cell = cell * B + (c[a] + B) % B;
            }
            slot = slot_base + local;
            key = slot * 64 + cell;
        }
        // wave-aggregated atomics: one per distinct (block, cell) for the rank in
        // the cell, one per distinct block for the block total.  The groups are
        // found first (ballots only), then every group's first lane adds its
        // group's size at once, so a wave waits for one round of atomics.
        int leader = 0, in_group = 0, group_size = 0;
        unsigned long long todo = __ballot(valid);
        while (todo) {
            const int l = __ffsll((long long)todo) - 1;
            const int lkey = __shfl(key, l);
            const unsigned long long grp = __ballot(valid && key == lkey);
            if (valid && key == lkey) {
                leader = l;
                in_group = __popcll(grp & ((1ull << lane) - 1ull));
            }
            if (lane == l) group_size = __popcll(grp);
            todo &= ~grp;
        }
        int r0 = 0;
        if (valid && lane == leader) r0 = atomicAdd(&p.cell_count[key], group_size);
        const int rank = __shfl(r0, leader) + in_group;
        todo = __ballot(valid);
        while (todo) {
            const int leader = __ffsll((long long)todo) - 1;
            const int lslot = __shfl(slot, leader);
            const unsigned long long grp = __ballot(valid && slot == lslot);
            if (lane == leader) atomicAdd(&p.slot_count[lslot], __popcll(grp));
            todo &= ~grp;
        }
        if (valid) {
            p.prank[i] = rank;
            p.keycur[i] = key;
            int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
#pragma unroll
            for (int a = 0; a < D; ++a) { lo[a] = (c[a] + B - 1) / B; hi[a] = (c[a] + B + 1) / B; }
            const int sb = slot_base;
            if constexpr (D == 3) {
                for (int x = lo[0]; x <= hi[0]; ++x)
                    for (int y = lo[1]; y <= hi[1]; ++y)
                        for (int z = lo[2]; z <= hi[2]; ++z) p.slot_touched[sb + (x * nb + y) * nb + z] = 1;
            } else {
                for (int x = lo[0]; x <= hi[0]; ++x)
                    for (int y = lo[1]; y <= hi[1]; ++y) p.slot_touched[sb + x * nb + y] = 1;
            }
        }
    }
}

// exclusive scan of one int per thread over the work-group
__device__ inline int wg_exclusive_scan(int v, int& total) {
    __shared__ int wsum[WG / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    __syncthreads();
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int before = 0;
    total = 0;
#pragma unroll
    for (int k = 0; k < WG / 64; ++k) {
        if (k < wave) before += wsum[k];
        total += wsum[k];
    }
    return before + x - v;
}

// Slots scanned: [0, slot_hw) -- an arena keeps its scenes' ranges low.
__device__ inline int scanned_slots(const KP& p) { return min(p.nslots, p.ctr->slot_hw); }

// A thread's SCAN_PER_THREAD consecutive slots from `base`: marks and particle
// counts, one int4 each where all of them are below ns (base is a multiple
// of 4 and the arrays are 256-byte aligned), zeros past ns.
__device__ inline void load_slots(const KP& p, int base, int ns, int* act, int* cnt) {
    static_assert(SCAN_PER_THREAD == 4, "one int4 per array");
    if (base + SCAN_PER_THREAD <= ns) {
        const int4 a = *reinterpret_cast<const int4*>(p.slot_touched + base);
        const int4 c = *reinterpret_cast<const int4*>(p.slot_count + base);
        act[0] = a.x; act[1] = a.y; act[2] = a.z; act[3] = a.w;
        cnt[0] = c.x; cnt[1] = c.y; cnt[2] = c.z; cnt[3] = c.w;
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_PER_THREAD; ++k) {
            const int s = base + k;
            act[k] = s < ns ? p.slot_touched[s] : 0;
            cnt[k] = s < ns ? p.slot_count[s] : 0;
        }
    }
}

// The scan's totals: active blocks and particles (one thread).
__device__ inline void record_totals(const KP& p, int ta, int tc) {
    p.ctr->n_prev = p.ctr->n_live;
    if (ta > p.bcap) {
        // the substep becomes a no-op: particles keep their order and state
        p.ctr->overflow = 1;
        p.ctr->nblocks = 0;
    } else {
        p.ctr->overflow = 0;  // a binning that fits clears an earlier overflow
        p.ctr->n_live = tc;
        p.ctr->nblocks = ta;
        p.block_pstart[ta] = tc;
    }
}

// The slots of load_slots, ra blocks and rc particles before them (moved past
// them): their blocks and active indices, and the binning's marks cleared.
__device__ inline void apply_scan(const KP& p, int base, int ns, const int* act, const int* cnt, int& ra, int& rc, bool overflow) {
    // after an overflow no block is set up, so the binning's cell counters of
    // the touched slots are cleared here instead of by the block set-up
    int sact[SCAN_PER_THREAD];
#pragma unroll
    for (int k = 0; k < SCAN_PER_THREAD; ++k) {
        const int s = base + k;
        sact[k] = act[k] ? ra : -1;
        if (act[k] && s < ns) {
            if (ra < p.bcap) {
                p.block_slot[ra] = s;
                p.block_pstart[ra] = rc;
            }
            if (overflow)
                for (int cell = 0; cell < 64; ++cell) p.cell_count[s * 64 + cell] = 0;
        }
        ra += act[k];
        rc += cnt[k];
    }
    if (base + SCAN_PER_THREAD <= ns) {
        *reinterpret_cast<int4*>(p.slot_active + base) = make_int4(sact[0], sact[1], sact[2], sact[3]);
        *reinterpret_cast<int4*>(p.slot_touched + base) = make_int4(0, 0, 0, 0);
        *reinterpret_cast<int4*>(p.slot_count + base) = make_int4(0, 0, 0, 0);
    } else {
#pragma unroll
        for (int k = 0; k < SCAN_PER_THREAD; ++k) {
            const int s = base + k;
            if (s < ns) {
                p.slot_active[s] = sact[k];
                p.slot_touched[s] = 0;
                p.slot_count[s] = 0;
            }
        }
    }
}

__global__ __launch_bounds__(WG) void k_scan_reduce(KP p) {
    const int ns = scanned_slots(p);
    if ((int64_t)blockIdx.x * SCAN_TILE >= ns) {  // beyond the scanned slots: empty part
        if (threadIdx.x == 0) {
            p.scan_part[blockIdx.x] = 0;
            p.scan_part[p.nparts + blockIdx.x] = 0;
        }
        return;
    }
    const int base = blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_PER_THREAD;
    int at[SCAN_PER_THREAD], ct[SCAN_PER_THREAD];
    load_slots(p, base, ns, at, ct);
    int act = 0, cnt = 0;
#pragma unroll
    for (int k = 0; k < SCAN_PER_THREAD; ++k) {
        act += at[k] != 0;
        cnt += ct[k];
    }
    int ta, tc;
    wg_exclusive_scan(act, ta);
    wg_exclusive_scan(cnt, tc);
    if (threadIdx.x == 0) {
        p.scan_part[blockIdx.x] = ta;
        p.scan_part[p.nparts + blockIdx.x] = tc;
    }
}

__global__ __launch_bounds__(WG) void k_scan_top(KP p) {
    // one work-group: exclusive scan of nparts block totals (two arrays)
    const int per = (p.nparts + WG - 1) / WG;
    const int b0 = threadIdx.x * per;
    int sa = 0, sc = 0;
    for (int k = 0; k < per; ++k) {
        const int j = b0 + k;
        if (j < p.nparts) { sa += p.scan_part[j]; sc += p.scan_part[p.nparts + j]; }
    }
    int ta, tc;
    const int ea = wg_exclusive_scan(sa, ta);
    const int ec = wg_exclusive_scan(sc, tc);
    int ra = ea, rc = ec;
    for (int k = 0; k < per; ++k) {
        const int j = b0 + k;
        if (j < p.nparts) {
            const int va = p.scan_part[j], vc = p.scan_part[p.nparts + j];
            p.scan_part[j] = ra;
            p.scan_part[p.nparts + j] = rc;
            ra += va;
            rc += vc;
        }
    }
    if (threadIdx.x == 0) record_totals(p, ta, tc);
}

__global__ __launch_bounds__(WG) void k_scan_apply(KP p) {
    const int ns = scanned_slots(p);
    if ((int64_t)blockIdx.x * SCAN_TILE >= ns) return;
    const int base = blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_PER_THREAD;
    int act[SCAN_PER_THREAD], cnt[SCAN_PER_THREAD];
    load_slots(p, base, ns, act, cnt);
    int sa = 0, sc = 0;
#pragma unroll
    for (int k = 0; k < SCAN_PER_THREAD; ++k) {
        act[k] = act[k] != 0;
        sa += act[k];
        sc += cnt[k];
    }
    int ta, tc;
    int ra = wg_exclusive_scan(sa, ta) + p.scan_part[blockIdx.x];
    int rc = wg_exclusive_scan(sc, tc) + p.scan_part[p.nparts + blockIdx.x];
    apply_scan(p, base, ns, act, cnt, ra, rc, p.ctr->overflow != 0);
}

// The whole scan in one work-group of SCAN_ONE threads, Q times
// SCAN_PER_THREAD consecutive slots each, for up to 8,192 slots (grids of up to
// 68 cells an axis in 3D).  Bound by latency: three launches of 2.9 to 4.5 us
// there do almost nothing, this one takes 4.5 us (1,331 slots) and 4.6 us (6,859);
// with 16 slots a thread (13,824) it took 11.8 us, as long as the three.
constexpr int SCAN_ONE = 1024;
template <int Q>
__global__ __launch_bounds__(SCAN_ONE) void k_scan_one(KP p) {
    __shared__ int wa[SCAN_ONE / 64], wc[SCAN_ONE / 64];
    const int ns = scanned_slots(p), lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int base = (int)threadIdx.x * Q * SCAN_PER_THREAD;
    int act[Q][SCAN_PER_THREAD], cnt[Q][SCAN_PER_THREAD], sa = 0, sc = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q) load_slots(p, base + q * SCAN_PER_THREAD, ns, act[q], cnt[q]);
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < SCAN_PER_THREAD; ++k) {
            act[q][k] = act[q][k] != 0;
            sa += act[q][k];
            sc += cnt[q][k];
        }
    // inclusive over the wave, then the waves before
    int ia = sa, ic = sc;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int ua = __shfl_up(ia, off), uc = __shfl_up(ic, off);
        if (lane >= off) {
            ia += ua;
            ic += uc;
        }
    }
    if (lane == 63) {
        wa[wv] = ia;
        wc[wv] = ic;
    }
    __syncthreads();
    int ra = ia - sa, rc = ic - sc, ta = 0, tc = 0;
#pragma unroll
    for (int w = 0; w < SCAN_ONE / 64; ++w) {
        if (w < wv) {
            ra += wa[w];
            rc += wc[w];
        }
        ta += wa[w];
        tc += wc[w];
    }
    if (threadIdx.x == 0) record_totals(p, ta, tc);
#pragma unroll
    for (int q = 0; q < Q; ++q) apply_scan(p, base + q * SCAN_PER_THREAD, ns, act[q], cnt[q], ra, rc, ta > p.bcap);
}

// Per active block (one wave, lane = cell): its scene, the neighbour table
// (inside the scene's slot range), and the cell ranges -- an exclusive scan
// of the block's 64 cell counts -- after which the cell counters are
// cleared for the next binning.
template <int D>
__global__ __launch_bounds__(WG) void k_block_setup(KP p) {
    using Dm = Dims<D>;
    const int nblocks = p.ctr->nblocks;
    const int group = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int b = blockIdx.x * (WG / 64) + group; b < nblocks; b += gridDim.x * (WG / 64)) {
        const int slot = p.block_slot[b];
        const int si = scene_of_slot(p, slot);
        const SceneParams& sc = p.scn[si];
        if (lane == 0) p.block_scene[b] = si;
        if (lane < Dm::NBR) {
            int bb[D];
            slot_coords<D>(slot - sc.slot_base, sc.nb, bb);
            if (lane < D) p.block_org[b * 3 + lane] = bb[lane];
            int o[3];
            if constexpr (D == 3) { o[0] = lane / 9; o[1] = (lane / 3) % 3; o[2] = lane % 3; }
            else { o[0] = lane / 3; o[1] = lane % 3; }
            int s = 0;
            bool in = true;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const int c = bb[a] + o[a] - 1;
                in = in && c >= 0 && c < sc.nb;
                s = s * sc.nb + c;
            }
            const int act = in ? p.slot_active[sc.slot_base + s] : -1;
            p.block_nbr[b * Dm::NBR + lane] = act;
            // tiles exist only for blocks that hold particles
            p.block_tnbr[b * Dm::NBR + lane] = (act >= 0 && p.block_pstart[act + 1] > p.block_pstart[act]) ? act : -1;
        }
        const int cnt = p.cell_count[slot * 64 + lane];
        int x = cnt;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(x, off);
            if (lane >= off) x += y;
        }
        const int start = p.block_pstart[b] + x - cnt;
        p.cell_start[b * 65 + lane] = start;
        if (lane == 63) p.cell_start[b * 65 + 64] = start + cnt;
        int full = cnt;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) full = max(full, __shfl_xor(full, off));
        if (lane == 0) p.block_full[b] = full;
        p.cell_count[slot * 64 + lane] = 0;
    }
}

// Per scene: its active block range and particle range (active blocks are
// in slot order, so each scene's blocks are contiguous).
__device__ inline void scene_ranges(const KP& p, int bid) {
    const int si = bid * WG + (int)threadIdx.x;
    if (si >= p.nscenes) return;
    const int nb = p.ctr->nblocks;
    auto lower = [&](int slot) {
        int lo = 0, hi = nb;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (p.block_slot[mid] < slot) lo = mid + 1;
            else hi = mid;
        }
        return lo;
    };
    const SceneParams& sc = p.scn[si];
    const int b0 = lower(sc.slot_base), b1 = lower(sc.slot_base + sc.nslots);
    SceneState& st = p.sst[si];
    st.block_begin = b0;
    st.block_end = b1;
    st.pbegin = nb > 0 ? p.block_pstart[b0] : 0;
    st.pend = nb > 0 ? p.block_pstart[b1] : 0;
}

// One work-group per XCD range of the active blocks (the ranges of
// xcd_blocks) and per key: the range's blocks by descending particle count
// (bucketed by eight; work-groups 0-7) and by descending count of their
// fullest cell (work-groups 8-15), each a counting sort whose order within
// a bucket is that of the LDS atomics.  The CG operator's time per block
// follows its fullest cell (its lane-per-cell passes are as many as that
// cell's particles); P2G, the constitutive/force kernel and G2P measured
// fastest in particle-count order.  Block loops that follow the hardware's
// dispatch order then start the long blocks first and leave short ones for
// the tail.  Only which work-group computes a block changes, never a
// block's result.
__device__ inline void block_order(const KP& p, int bid) {
    constexpr int NBK = WG;  // buckets, one per thread for the scan
    __shared__ int hist[NBK];
    const int n = p.ctr->nblocks, x = bid & 7, by_cell = bid >> 3;
    const int lo = (int)(((int64_t)n * x) >> 3), hi = (int)(((int64_t)n * (x + 1)) >> 3);
    int* order = p.block_order + (by_cell ? p.bcap : 0);
    auto key = [&](int b) {  // the longest first
        const int w = by_cell ? p.block_full[b] : (p.block_pstart[b + 1] - p.block_pstart[b]) >> 3;
        return NBK - 1 - min(NBK - 1, w);
    };
    hist[threadIdx.x] = 0;
    __syncthreads();
    for (int b = lo + (int)threadIdx.x; b < hi; b += WG) atomicAdd(&hist[key(b)], 1);
    __syncthreads();
    int total;
    const int off = wg_exclusive_scan(hist[threadIdx.x], total);
    __syncthreads();
    hist[threadIdx.x] = off;
    __syncthreads();
    for (int b = lo + (int)threadIdx.x; b < hi; b += WG) order[lo + atomicAdd(&hist[key(b)], 1)] = b;
}

// scatter into (block, cell) order
// The binning ranks come from atomics, so the order they give within a cell
// depends on arrival.  Each particle writes its index into its cell's range
// at that rank; k_reorder then places it by the number of indices in the
// range below its own, which orders every cell by the particles' previous
// positions (a stable sort by cell) and makes the layout, and every sum over
// a cell's particles, the same from run to run.
__device__ inline void cell_order(const KP& p, int bid, int nbid) {
    if (p.ctr->overflow != 0) return;
    const int n = p.ctr->n_prev;
    for (int i = bid * WG + (int)threadIdx.x; i < n; i += nbid * WG) {
        const int key = p.keycur[i];
        if (key < 0) continue;
        p.cell_order[p.cell_start[p.slot_active[key >> 6] * 65 + (key & 63)] + p.prank[i]] = i;
    }
}

// The three set-up steps that follow the block set-up and do not depend on
// one another, in one launch: work-groups 0-15 sort the blocks (the XCD of
// work-group w is w mod 8, as for the block kernels), the next ceil(scenes /
// WG) find the scenes' ranges, the rest scatter the particles' indices into
// their cells.
constexpr int ORDER_GROUPS = 16;
__global__ __launch_bounds__(WG) void k_setup_order(KP p) {
    const int sr = (p.nscenes + WG - 1) / WG;
    const int bid = (int)blockIdx.x;
    if (bid < ORDER_GROUPS) block_order(p, bid);
    else if (bid < ORDER_GROUPS + sr) scene_ranges(p, bid - ORDER_GROUPS);
    else cell_order(p, bid - ORDER_GROUPS - sr, (int)gridDim.x - ORDER_GROUPS - sr);
}

template <int D>
__global__ __launch_bounds__(WG) void k_reorder(KP p) {
    const int n = p.ctr->n_prev;
    const bool overflow = p.ctr->overflow != 0;
    for (int i = blockIdx.x * WG + threadIdx.x; i < n; i += gridDim.x * WG) {
        // the particle's state loads with its key, before the destination is
        // known (the buffers may alias as far as the compiler knows, so a load
        // after a store would wait for it).  Only a placed particle (a live key
        // and no overflow) reads the cell tables; a removed one (key < 0) or an
        // identity copy reads cell 0's bounds (the table always has them: slot
        // tables hold -1, and after an overflow indices past the capacity, so
        // they are not read for these) and a removed one stores nothing.
        const int key = p.keycur[i];
        float v[PF<D>::N];
#pragma unroll
        for (int f = 0; f < PF<D>::N; ++f) v[f] = p.pcur[f * p.pcap + i];
        const int id = p.idcur[i], si = p.scur[i];
        const bool live = overflow || key >= 0;
        const bool placed = !overflow && key >= 0;
        const int cs = placed ? p.slot_active[key >> 6] * 65 + (key & 63) : 0;
        const int start = p.cell_start[cs], end = p.cell_start[cs + 1];
        // rank: indices of the cell below i, eight loads in flight at a time
        // (an index past the range reads its last entry and is not counted)
        constexpr int U = 8;
        int rank = 0;
        if (placed) {
            for (int j0 = start; j0 < end; j0 += U) {
                int e[U];
#pragma unroll
                for (int u = 0; u < U; ++u) e[u] = p.cell_order[min(j0 + u, end - 1)];
#pragma unroll
                for (int u = 0; u < U; ++u) rank += (j0 + u < end && e[u] < i) ? 1 : 0;
            }
        }
        // overflow: identity copy, the buffer swap leaves the state unchanged
        const int dest = overflow ? i : start + rank;
        if (!live) continue;
#pragma unroll
        for (int f = 0; f < PF<D>::N; ++f) p.palt[f * p.pcap + dest] = v[f];
        p.idalt[dest] = id;
        p.salt[dest] = si;
        p.keyalt[dest] = overflow ? key : 0;
    }
}

// Block kernels run NW waves per active block.  In scatter kernels lane c of
// every wave owns cell c of the block (particles are in (block, cell) order,
// cell ranges in cell_start) and wave w takes the cell's particles w, w+NW,
// ...  All particles of a lane share one 3^D stencil and, for a fixed stencil
// offset, the 64 lanes of a wave address 64 distinct tile nodes.  Each wave
// therefore scatters into its own LDS tile with plain read-add-write steps
// (one stencil node per step; LDS operations of a wave execute in order), and
// the NW wave tiles are summed when the block's tile is stored.  No LDS or
// global atomics are used.
constexpr int NW = 4;
constexpr int BWG = 64 * NW;

// Compiler-only memory barrier between two read-add-write steps of a wave
// scatter: a lane's step s+1 may read the node another lane wrote in step s,
// so no LDS access may move across it (a wave's LDS operations execute in
// issue order).
#define MPM_STEP_FENCE() __asm__ __volatile__("" ::: "memory")

// Sum of the NW wave tiles (C channels each, LDS layout) of block b into
// its tile slot (compact layout, node (x,y,z) at (x*TE + y)*TE + z).
template <int D, int C>
__device__ inline void store_wave_tiles(const KP& p, int b, const float* lds) {
    constexpr int TN = Dims<D>::TN, LTN = Dims<D>::LTN;
    float* dst = p.tiles + (int64_t)b * C * TN;
    for (int t = threadIdx.x; t < C * TN; t += BWG) {
        const int c = t / TN;
        int nb, local, tc[D];
        tile_map<D>(t - c * TN, nb, local, tc);
        const int li = c * LTN + lds_index<D>(tc);
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += lds[w * C * LTN + li];
        dst[t] = v;
    }
}

// The record of an EOS particle: its CG force V0 K gamma rho^(gamma-1)
// (grad w . u) grad w (MPM_CG_System.h:169-174, 205-207) is A = c tr(T) I,
// taking the reference's matrix-plus-scalar as adding to the diagonal.  In
// the record's layout: U = I, every entry of the diagonal block c, no pair
// blocks (2D: c at (00,00), (00,11), (11,11)).
template <int D>
__device__ inline void store_operator_eos(const KP& p, int i, float c, const float* xo);

// ============================================================================
// Linearised force operator per particle.  MPM_CG_System::Force
// (MPM_CG_System.h:150-215) maps the node field u to forces through
//   T = sum_i grad w_ip (x) u_i,  dF = T^T F,  A = V0 F dP(dF)^T,
//   q_i += A^T grad w_ip.
// T -> A is linear and fixed for the whole solve, so it is evaluated once
// per substep as a D^2 x D^2 matrix (columns = A of the unit T's), which is
// symmetric (dP is the Hessian of the energy: V0 dP(dF):dF' = V0 dP(dF'):dF)
// and is stored after the particle's stencil offsets as its upper triangle.
// One CG application then costs D^4 multiply-adds per particle instead of
// re-deriving the stress state, and reads one contiguous record.
// ============================================================================
template <int D> struct OpRec;
// 3D: x[3] (the stencil offsets of the particle's position in its binned
// cell, in cells), q[4] (unit quaternion of U), the singular values S[3] and the
// four scalars A = 2 mu V0, B = lambda V0 (J - 1), P = B J, Q = lambda V0 J^2
// from which the 3x3 block on the diagonal entries and the three 2x2 pair
// blocks follow, pad 2 (64 B: four float4).
template <> struct OpRec<3> { static constexpr int W = 16; };  // 4 x float4
// 2D: x[2] (stencil offsets), the full symmetric 4x4 operator (upper triangle, 10).
template <> struct OpRec<2> { static constexpr int L = 10, W = 12; };  // 3 x float4
static_assert(OpRec<3>::W == op_record_floats(3) && OpRec<2>::W == op_record_floats(2), "operator record size");

template <int D>
__device__ constexpr int op_index(int r, int c) {
    // upper triangle, row-major, of a D^2 x D^2 matrix (r <= c)
    return r * D * D - (r * (r - 1)) / 2 + (c - r);
}

// A = V0 F dP(T^T F)^T, the reference's per-particle force map
template <int D>
__device__ inline void force_map(const StressState<D>& st, float V0, const float* T, float* A) {
    constexpr int DD = D * D;
    float dF[DD];
#pragma unroll
    for (int r = 0; r < D; ++r)
#pragma unroll
        for (int cc = 0; cc < D; ++cc) {
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < D; ++k) s += T[k * D + r] * st.F[k * D + cc];
            dF[r * D + cc] = s;
        }
    float dP[DD];
    dP_of<D>(st, dF, dP);
#pragma unroll
    for (int r = 0; r < D; ++r)
#pragma unroll
        for (int cc = 0; cc < D; ++cc) {
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < D; ++k) s += st.F[r * D + k] * dP[cc * D + k];
            A[r * D + cc] = s * V0;
        }
}

// rotation matrix (row-major) <-> unit quaternion (w, x, y, z)
__device__ inline void quat_of(const float* U, float* q) {
    const float tr = U[0] + U[4] + U[8];
    float w, x, y, z;
    if (tr > 0.0f) {
        const float s = 2.0f * sqrtf(tr + 1.0f);
        w = 0.25f * s; x = (U[7] - U[5]) / s; y = (U[2] - U[6]) / s; z = (U[3] - U[1]) / s;
    } else if (U[0] > U[4] && U[0] > U[8]) {
        const float s = 2.0f * sqrtf(1.0f + U[0] - U[4] - U[8]);
        w = (U[7] - U[5]) / s; x = 0.25f * s; y = (U[1] + U[3]) / s; z = (U[2] + U[6]) / s;
    } else if (U[4] > U[8]) {
        const float s = 2.0f * sqrtf(1.0f + U[4] - U[0] - U[8]);
        w = (U[2] - U[6]) / s; x = (U[1] + U[3]) / s; y = 0.25f * s; z = (U[5] + U[7]) / s;
    } else {
        const float s = 2.0f * sqrtf(1.0f + U[8] - U[0] - U[4]);
        w = (U[3] - U[1]) / s; x = (U[2] + U[6]) / s; y = (U[5] + U[7]) / s; z = 0.25f * s;
    }
    const float n = 1.0f / sqrtf(w * w + x * x + y * y + z * z);
    q[0] = w * n; q[1] = x * n; q[2] = y * n; q[3] = z * n;
}
// The operator's and the solve's arithmetic is compiled into several kernels and
// forms: products and sums fuse as written (contract(on), and fmaf where the order
// matters) and not as each one's code around them happens to allow, so that a
// form and its fallback round alike.
#pragma clang fp contract(on)
// Which product of a rotation's sums of two is rounded on its own: the launched
// operator and the one-launch solve with one and with two blocks to a work-group
// each came to differ in this, and keep it, so that a scene's results stay what
// they were.  (The solve's fallback, ROUND_EITHER, is told whose it is.)
enum Rounding { ROUND_LAUNCHED, ROUND_ONE, ROUND_TWO, ROUND_EITHER };
template <int R>
__device__ inline void rot_of(const float* q, bool two, float* U) {
    constexpr bool SOLVE = R != ROUND_LAUNCHED;
    const float w = q[0], x = q[1], y = q[2], z = q[3];
    const bool xy = R == ROUND_TWO || (R == ROUND_EITHER && two);
    const float a = xy ? x : y, b = xy ? y : x;
    U[0] = fmaf(-2.0f, SOLVE ? fmaf(y, y, z * z) : fmaf(z, z, y * y), 1.0f);
    U[1] = 2.0f * fmaf(x, y, -(w * z));
    U[2] = 2.0f * fmaf(x, z, w * y);
    U[3] = 2.0f * fmaf(x, y, w * z);
    U[4] = fmaf(-2.0f, SOLVE ? fmaf(x, x, z * z) : fmaf(z, z, x * x), 1.0f);
    U[5] = 2.0f * (SOLVE ? fmaf(-w, x, y * z) : fmaf(y, z, -(w * x)));
    U[6] = 2.0f * fmaf(x, z, -(w * y));
    U[7] = 2.0f * (SOLVE ? fmaf(w, x, y * z) : fmaf(y, z, w * x));
    U[8] = fmaf(-2.0f, fmaf(a, a, b * b), 1.0f);
}

// Ahat = U^T A U (3x3)
__device__ inline void rotate_in(const float* U, const float* A, float* out) {
    float t[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) t[i * 3 + j] = A[i * 3 + 0] * U[0 * 3 + j] + A[i * 3 + 1] * U[1 * 3 + j] + A[i * 3 + 2] * U[2 * 3 + j];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) out[i * 3 + j] = U[0 * 3 + i] * t[0 * 3 + j] + U[1 * 3 + i] * t[1 * 3 + j] + U[2 * 3 + i] * t[2 * 3 + j];
}
// A = U Ahat U^T (3x3)
__device__ inline void rotate_out(const float* U, const float* Ah, float* out) {
    float t[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const float u0 = U[i * 3], u1 = U[i * 3 + 1], a0 = Ah[j], a1 = Ah[3 + j];
            t[i * 3 + j] = fmaf(U[i * 3 + 2], Ah[6 + j], j == 0 ? fmaf(u1, a1, u0 * a0) : fmaf(u0, a0, u1 * a1));
        }
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) out[i * 3 + j] = t[i * 3 + 0] * U[j * 3 + 0] + t[i * 3 + 1] * U[j * 3 + 1] + t[i * 3 + 2] * U[j * 3 + 2];
}

#pragma clang fp contract(fast)

// The record of particle i.  3D: in the frame of U (F = U S V^T, R = U V^T)
// the reference's force map T -> A = V0 F dP(T^T F)^T of fixed-corotated
// snow (MPM_CG_System.h:176-210, dP of MPM_Constitutive_Model.cpp) decouples:
// with T^ = U^T T U, dF^ = T^T S, the rotation term W^_ij = (dF^_ij -
// dF^_ji) / (s_i + s_j) and the derivative of cof(S), A^ = U^T A U = V0 S dP^T
// is a 3x3 block on the diagonal entries,
//   V0 (2 mu s_a^2 [c == a] + lambda J^2 + lambda J (J - 1) [c != a])
//   = diag(A s_a^2 - P) + (P + Q) 1 1^T,
// plus per off-diagonal pair (lo, hi), with s = s_lo + s_hi and k the third
// index, the symmetric block
//   [[A s_lo^2 (s - 1) / s,  s_lo s_hi (A / s - B s_k)],
//    [         ...,          A s_hi^2 (s - 1) / s   ]],
// where A = 2 mu V0, B = lambda V0 (J - 1), P = B J, Q = lambda V0 J^2.  The
// record holds S and these four scalars (formed in FP64, stored in FP32);
// apply_operator forms the block entries from them.
template <int D>
__device__ inline void store_operator(const KP& p, int i, const StressState<D>& st, float V0, const float* xo,
                                      const float* U, const double* S) {
    constexpr int DD = D * D;
    float rec[OpRec<D>::W];
#pragma unroll
    for (int k = 0; k < OpRec<D>::W; ++k) rec[k] = 0.0f;
#pragma unroll
    for (int a = 0; a < D; ++a) rec[a] = xo[a];
    if constexpr (D == 3) {
        quat_of(U, rec + 3);
        const double v0 = (double)V0, mu = (double)st.mu, lam = (double)st.lambda;
        const double J = S[0] * S[1] * S[2];
        const double B = lam * v0 * (J - 1.0);
        rec[7] = (float)S[0];
        rec[8] = (float)S[1];
        rec[9] = (float)S[2];
        rec[10] = (float)(2.0 * mu * v0);
        rec[11] = (float)B;
        rec[12] = (float)(B * J);
        rec[13] = (float)(lam * v0 * J * J);
    } else {
        float L[DD][DD];
#pragma unroll
        for (int j = 0; j < DD; ++j) {
            float T[DD], A[DD];
#pragma unroll
            for (int k = 0; k < DD; ++k) T[k] = k == j ? 1.0f : 0.0f;
            force_map<D>(st, V0, T, A);
#pragma unroll
            for (int r = 0; r < DD; ++r) L[r][j] = A[r];
        }
#pragma unroll
        for (int r = 0; r < DD; ++r)
#pragma unroll
            for (int c = r; c < DD; ++c) rec[D + op_index<D>(r, c)] = 0.5f * (L[r][c] + L[c][r]);
    }
    float4* dst = reinterpret_cast<float4*>(p.pop + (int64_t)i * OpRec<D>::W);
#pragma unroll
    for (int k = 0; k < OpRec<D>::W / 4; ++k) dst[k] = make_float4(rec[4 * k], rec[4 * k + 1], rec[4 * k + 2], rec[4 * k + 3]);
}

#pragma clang fp contract(on)
// The 2x2 block of pair (lo, hi) with third index k applied to
// (Th_lo,hi, Th_hi,lo).  FIRST: the pair (0, 1).
template <bool FIRST>
__device__ inline void apply_pair(float A, float B, float slo, float shi, float sk, float tlh, float thl, float& alh,
                                  float& ahl) {
    const float sm = slo + shi;
    const float inv = __builtin_amdgcn_rcpf(sm);
    const float g = A * (sm - 1.0f) * inv;
    const float a = g * slo * slo, c = g * shi * shi;
    const float b = slo * shi * fmaf(A, inv, -(B * sk));
    alh = FIRST ? fmaf(b, thl, a * tlh) : fmaf(a, tlh, b * thl);
    ahl = fmaf(b, tlh, c * thl);
}

// A = scale L T from a particle's operator record (in registers)
template <int D, int R>
__device__ inline void apply_operator(const float* rec, float scale, bool two, const float* T, float* A) {
    constexpr int DD = D * D;
    if constexpr (D == 3) {
        const float s0 = rec[7], s1 = rec[8], s2 = rec[9];
        const float a2 = scale * rec[10], bl = scale * rec[11], pj = scale * rec[12], kappa = fmaf(scale, rec[13], pj);
        float U[9], Th[9], Ah[9];
        rot_of<R>(rec + 3, two, U);
        rotate_in(U, T, Th);
        const float tr = kappa * (Th[0] + Th[4] + Th[8]);
        Ah[0] = fmaf(fmaf(a2 * s0, s0, -pj), Th[0], tr);
        Ah[4] = fmaf(fmaf(a2 * s1, s1, -pj), Th[4], tr);
        Ah[8] = fmaf(fmaf(a2 * s2, s2, -pj), Th[8], tr);
        apply_pair<true>(a2, bl, s0, s1, s2, Th[1], Th[3], Ah[1], Ah[3]);
        apply_pair<false>(a2, bl, s0, s2, s1, Th[2], Th[6], Ah[2], Ah[6]);
        apply_pair<false>(a2, bl, s1, s2, s0, Th[5], Th[7], Ah[5], Ah[7]);
        rotate_out(U, Ah, A);
    } else {
        const float* tri = rec + D;
#pragma unroll
        for (int r = 0; r < DD; ++r) A[r] = 0.0f;
#pragma unroll
        for (int r = 0; r < DD; ++r)
#pragma unroll
            for (int c = r; c < DD; ++c) {
                const float v = tri[op_index<D>(r, c)];
                A[r] += v * T[c];
                if (c != r) A[c] += v * T[r];
            }
#pragma unroll
        for (int r = 0; r < DD; ++r) A[r] *= scale;
    }
}

#pragma clang fp contract(fast)

template <int D>
__device__ inline void store_operator_eos(const KP& p, int i, float c, const float* xo) {
    float rec[OpRec<D>::W];
#pragma unroll
    for (int k = 0; k < OpRec<D>::W; ++k) rec[k] = 0.0f;
#pragma unroll
    for (int a = 0; a < D; ++a) rec[a] = xo[a];
    if constexpr (D == 3) {
        // U = I, S = (1, 1, 1), A = B = P = 0, Q = c: every entry of the
        // diagonal block c, empty pair blocks
        rec[3] = 1.0f;
        rec[7] = rec[8] = rec[9] = 1.0f;
        rec[13] = c;
    } else {
        rec[D + op_index<D>(0, 0)] = c;
        rec[D + op_index<D>(0, 3)] = c;
        rec[D + op_index<D>(3, 3)] = c;
    }
    float4* dst = reinterpret_cast<float4*>(p.pop + (int64_t)i * OpRec<D>::W);
#pragma unroll
    for (int k = 0; k < OpRec<D>::W / 4; ++k) dst[k] = make_float4(rec[4 * k], rec[4 * k + 1], rec[4 * k + 2], rec[4 * k + 3]);
}

#pragma clang fp contract(on)
// ---------------------------------------------------------------------------
// The CG operator's stencil in difference form.  Per axis the weights of the
// three stencil nodes sum to one, so a field in a cell is
//   u = u1 + w0 (u0 - u1) + w2 (u2 - u1),   u' = w0' (u0 - u1) + w2' (u2 - u1):
// the middle node's weight and derivative drop out.  The differences are
// formed once per cell (two operations a node triple) and shared by its
// particles; a particle's gradient then takes 180 operations in 3D instead
// of 270.  Forces go back through the transpose, moments of the functions
// {w0, 1, w2}.  The outer weights keep their own products, so a node that
// carries only a sliver of a particle's weight (and of its mass) gets its
// force to the same relative accuracy as node by node; a power basis loses
// that to cancellation (measured: CG solves stall on light nodes).
// ---------------------------------------------------------------------------
template <int D>
struct CellStencil {
    static constexpr int NC = D == 3 ? 27 : 9;    // functions of a cell
    static constexpr int MID = NC / 2;            // the constant: no gradient needs it
    static constexpr int ROWS = D * (NC - 1);     // coefficient rows of a block, [channel][function][cell]
    static constexpr int PACK = D == 3 ? 20 : 12;  // floats of a packed particle: A, w0, w2, d0
    __device__ static constexpr int row(int cc, int n) { return cc * (NC - 1) + (n < MID ? n : n - 1); }
};

// node values -> differences along one axis (u1 stays)
__device__ inline void diff_of_nodes(float& u0, const float& u1, float& u2) {
    u0 -= u1;
    u2 -= u1;
}
// its transpose: moments -> node contributions along one axis
__device__ inline void nodes_of_moments(const float& m0, float& m1, const float& m2) { m1 -= m0 + m2; }

// Coefficients of channel array u (an LDS tile) for the cell whose stencil
// corner has tile index `base`.
template <int D>
__device__ inline void cell_coefficients(const float* u, int base, float* c) {
    constexpr int LX = Dims<D>::LX, LY = Dims<D>::LY;
    if constexpr (D == 3) {
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                float* r = c + (i * 3 + j) * 3;
#pragma unroll
                for (int k = 0; k < 3; ++k) r[k] = u[base + i * LX + j * LY + k];
                diff_of_nodes(r[0], r[1], r[2]);
            }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k) diff_of_nodes(c[i * 9 + k], c[i * 9 + 3 + k], c[i * 9 + 6 + k]);
#pragma unroll
        for (int k = 0; k < 9; ++k) diff_of_nodes(c[k], c[9 + k], c[18 + k]);
    } else {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
#pragma unroll
            for (int k = 0; k < 3; ++k) c[i * 3 + k] = u[base + i * LX + k];
            diff_of_nodes(c[i * 3], c[i * 3 + 1], c[i * 3 + 2]);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) diff_of_nodes(c[k], c[3 + k], c[6 + k]);
    }
}

// A particle's outer weights and their derivatives (in cells; the operator
// scales its result by inv_dx twice) per axis, the weights operation for
// operation as in bspline_from_offset.
template <int D>
struct OuterWeights {
    float w0[D], w2[D], d0[D], d2[D];
    __device__ explicit OuterWeights(const float* xo) {
#pragma unroll
        for (int a = 0; a < D; ++a) {
#pragma clang fp contract(off)
            float x = xo[a];
            w0[a] = fabsf(0.5f * x * x - 1.5f * x + 1.125f);
            d0[a] = x - 1.5f;
            x -= 2.0f;
            w2[a] = fabsf(0.5f * x * x + 1.5f * x + 1.125f);
            d2[a] = x + 1.5f;
        }
    }
};

// T[r][cc] = d_r of channel cc at a particle of cell `cell` (per cell), from
// the block's coefficient rows in LDS: particles of one cell read the same
// words (broadcast), neighbouring cells neighbouring banks.
template <int D>
__device__ inline void stencil_gradient(const OuterWeights<D>& g, const float* coef, int cell, float* T) {
    using CS = CellStencil<D>;
    auto val = [](float w0, float w2, float c0, float c1, float c2) { return fmaf(w2, c2, fmaf(w0, c0, c1)); };
    auto der = [](float d0, float d2, float c0, float c2) { return fmaf(d2, c2, d0 * c0); };
#pragma unroll
    for (int cc = 0; cc < D; ++cc) {
        auto c = [&](int n) { return coef[CS::row(cc, n) * 64 + cell]; };
        if constexpr (D == 3) {
            float v[3], dy[3], dz[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                float z[3], s[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const int n = (i * 3 + j) * 3;
                    const bool mid = i == 1 && j == 1;  // its value meets no derivative
                    const float k0 = c(n), k1 = mid ? 0.0f : c(n + 1), k2 = c(n + 2);
                    z[j] = mid ? 0.0f : val(g.w0[2], g.w2[2], k0, k1, k2);
                    s[j] = der(g.d0[2], g.d2[2], k0, k2);
                }
                v[i] = i == 1 ? 0.0f : val(g.w0[1], g.w2[1], z[0], z[1], z[2]);
                dy[i] = der(g.d0[1], g.d2[1], z[0], z[2]);
                dz[i] = val(g.w0[1], g.w2[1], s[0], s[1], s[2]);
            }
            T[0 * 3 + cc] = der(g.d0[0], g.d2[0], v[0], v[2]);
            T[1 * 3 + cc] = val(g.w0[0], g.w2[0], dy[0], dy[1], dy[2]);
            T[2 * 3 + cc] = val(g.w0[0], g.w2[0], dz[0], dz[1], dz[2]);
        } else {
            float v[3], dy[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const int n = i * 3;
                const float k0 = c(n), k2 = c(n + 2);
                v[i] = i == 1 ? 0.0f : val(g.w0[1], g.w2[1], k0, c(n + 1), k2);
                dy[i] = der(g.d0[1], g.d2[1], k0, k2);
            }
            T[0 * 2 + cc] = der(g.d0[0], g.d2[0], v[0], v[2]);
            T[1 * 2 + cc] = val(g.w0[0], g.w2[0], dy[0], dy[1], dy[2]);
        }
    }
}

// A particle as the scatter reads it: the outer weights and w0' per axis
// (w2' = w0' + 1 exactly, offsets lie in [1/2, 3/2)) and the columns of its
// force map A, so that the wave of channel cc reads three (2D: two) float4:
//   3D: w0[3] d0x | w2[3] d0y | A[.][0] d0z | A[.][1] d0z | A[.][2] d0z
//   2D: w0[2] w2[2] | A[.][0] d0[2] | A[.][1] d0[2]
template <int D>
__device__ inline void pack_particle(const OuterWeights<D>& g, const float* A, float* pack) {
    float4* q = reinterpret_cast<float4*>(pack);
    if constexpr (D == 3) {
        q[0] = make_float4(g.w0[0], g.w0[1], g.w0[2], g.d0[0]);
        q[1] = make_float4(g.w2[0], g.w2[1], g.w2[2], g.d0[1]);
#pragma unroll
        for (int cc = 0; cc < 3; ++cc) q[2 + cc] = make_float4(A[cc], A[3 + cc], A[6 + cc], g.d0[2]);
    } else {
        q[0] = make_float4(g.w0[0], g.w0[1], g.w2[0], g.w2[1]);
#pragma unroll
        for (int cc = 0; cc < 2; ++cc) q[1 + cc] = make_float4(A[cc], A[2 + cc], g.d0[0], g.d0[1]);
    }
}
template <int D>
struct PackedForce {
    float4 q[D == 3 ? 3 : 2];
    // pack: the particle's words; cpack: the same shifted by the channel's four
    __device__ void load(const float* pack, const float* cpack) {
        q[0] = reinterpret_cast<const float4*>(pack)[0];
        if constexpr (D == 3) {
            q[1] = reinterpret_cast<const float4*>(pack)[1];
            q[2] = reinterpret_cast<const float4*>(cpack)[2];
        } else {
            q[1] = reinterpret_cast<const float4*>(cpack)[1];
        }
    }
};

// One packed particle's force on channel cc: M += sum_r A[r][cc] d_r of every
// function (the transpose of stencil_gradient; the constant's moment stays 0).
template <int D>
__device__ inline void add_force_moments(const PackedForce<D>& f4, float* M) {
    if constexpr (D == 3) {
        const float4 p = f4.q[0], r = f4.q[1], a = f4.q[2];
        const float d2x = p.w + 1.0f, d2y = r.w + 1.0f, d2z = a.w + 1.0f;
        const float e[3] = {p.w * a.x, 0.0f, d2x * a.x};
        const float f[3] = {p.x * a.y, a.y, r.x * a.y};
        const float h[3] = {p.x * a.z, a.z, r.x * a.z};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const float y[3] = {i == 1 ? r.w * f[i] : fmaf(p.y, e[i], r.w * f[i]), e[i],
                                i == 1 ? d2y * f[i] : fmaf(r.y, e[i], d2y * f[i])};
            const float z[3] = {p.y * h[i], h[i], r.y * h[i]};
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                float* k = M + (i * 3 + j) * 3;
                if (i != 1 || j != 1) {
                    k[0] = fmaf(a.w, z[j], fmaf(p.z, y[j], k[0]));
                    if (i == 1) k[1] = fmaf(j == 0 ? r.w : d2y, f[1], k[1]);
                    else if (j == 1) k[1] = fmaf(i == 0 ? p.w : d2x, a.x, k[1]);
                    else k[1] += y[j];
                    k[2] = fmaf(d2z, z[j], fmaf(r.z, y[j], k[2]));
                } else {
                    k[0] = fmaf(a.w, z[j], k[0]);
                    k[2] = fmaf(d2z, z[j], k[2]);
                }
            }
        }
    } else {
        const float4 p = f4.q[0], a = f4.q[1];
        const float d2x = a.z + 1.0f, d2y = a.w + 1.0f;
        const float e[3] = {a.z * a.x, 0.0f, d2x * a.x};
        const float f[3] = {p.x * a.y, a.y, p.z * a.y};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            float* k = M + i * 3;
            if (i != 1) {
                k[0] = fmaf(a.w, f[i], fmaf(p.y, e[i], k[0]));
                k[1] = fmaf(i == 0 ? a.z : d2x, a.x, k[1]);
                k[2] = fmaf(d2y, f[i], fmaf(p.w, e[i], k[2]));
            } else {
                k[0] = fmaf(a.w, f[i], k[0]);
                k[2] = fmaf(d2y, f[i], k[2]);
            }
        }
    }
}

// The value of lane P0..P3 of each group of four lanes (DPP quad_perm).
template <int P0, int P1, int P2, int P3>
__device__ inline float quad_perm(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), P0 | (P1 << 2) | (P2 << 4) | (P3 << 6), 0xf, 0xf, true));
}

// A cell's moments of one channel into its node contributions (the transposed
// transform), in place.
template <int D>
__device__ inline void nodes_of_cell(float* M) {
    if constexpr (D == 3) {
#pragma unroll
        for (int k = 0; k < 9; ++k) nodes_of_moments(M[k], M[9 + k], M[18 + k]);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int k = 0; k < 3; ++k) nodes_of_moments(M[i * 9 + k], M[i * 9 + 3 + k], M[i * 9 + 6 + k]);
#pragma unroll
        for (int r = 0; r < 9; ++r) nodes_of_moments(M[r * 3], M[r * 3 + 1], M[r * 3 + 2]);
    } else {
#pragma unroll
        for (int k = 0; k < 3; ++k) nodes_of_moments(M[k], M[3 + k], M[6 + k]);
#pragma unroll
        for (int r = 0; r < 3; ++r) nodes_of_moments(M[r * 3], M[r * 3 + 1], M[r * 3 + 2]);
    }
}

// Adds one channel's node contributions M of all cells (lane = cell) to the
// channel's LDS tile q in ordered read-add-writes in which the lanes' nodes
// are distinct (the fence keeps the steps in order: a step may read a node
// that another lane wrote in the step before).  3D: the four cells of a row in
// z are neighbouring lanes, so their three planes are summed across the lanes
// first (lane z keeps node z, lanes 2 and 3 also nodes 4 and 5), nine steps
// instead of 27.
template <int D>
__device__ inline void add_cell_nodes(const float* M, int base, int lane, float* q) {
    constexpr int LX = Dims<D>::LX, LY = Dims<D>::LY;
    if constexpr (D == 3) {
        const int lz = lane & 3;
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const float* n = M + r * 3;
            const float up1 = quad_perm<0, 0, 1, 2>(n[1]), up2 = quad_perm<0, 1, 0, 1>(n[2]);
            const float last = quad_perm<3, 3, 3, 3>(n[1]);
            const float s0 = n[0] + (lz >= 1 ? up1 : 0.0f) + (lz >= 2 ? up2 : 0.0f);
            const float s1 = n[2] + (lz == 2 ? last : 0.0f);
            float* d = q + base + (r / 3) * LX + (r % 3) * LY;
            const float o0 = d[0], o1 = d[2];
            d[0] = o0 + s0;
            if (lz >= 2) d[2] = o1 + s1;
            MPM_STEP_FENCE();
        }
    } else {
#pragma unroll
        for (int n = 0; n < 9; ++n) {
            q[base + (n / 3) * LX + n % 3] += M[n];
            MPM_STEP_FENCE();
        }
    }
}

#pragma clang fp contract(fast)

// Weights of particle i; false if it is not in cell l of block bb (only after
// particles moved without re-binning: the particle is skipped).
template <int D>
__device__ inline bool cell_particle(const KP& p, const SceneParams& sc, int i, const int* bb, const int* l,
                                     float (*w)[3], float (*dw)[3], float* X) {
    int lp[D];
    if (!particle_weights<D>(p, sc, i, bb, w, dw, lp, X)) return false;
    bool same = true;
#pragma unroll
    for (int a = 0; a < D; ++a) same = same && lp[a] == l[a];
    return same;
}

// ============================================================================
// P2G (Rasterize, MPM_Example.cpp:520-537): m_i += w m_p, (mv)_i += w m_p V_p.
// Lane c runs the particles of cell c, summing the cell's 3^D-node contribution
// in registers (the particles of a cell share its stencil), then adds it to the
// wave's LDS tile in 3^D ordered read-add-write steps (lanes hold distinct
// cells).  LDS traffic is one stencil per cell instead of one per particle.
// One wave per block (the waves of a work-group take different blocks and share
// nothing); SPLIT: a work-group per block, its waves taking every NW-th
// particle of a cell, where there are too few blocks to fill the chip and the
// fullest cell's particles, one after another, are the time.  Up to
// P2G_SPLIT_BLOCKS active blocks, read here, so that launched and replayed
// substeps agree: 3.8k particles in 72 blocks 24.5 us whole, 13.5 split, 200k in
// 805 22.9 and 15.0, 390k in 1,415 24.3 and 22.9, 390k in 1,576 24.6 and 21.6, 1.0M
// in 986 56 and 40; but 1.0k in 1,869 11.4 and 15.8, 320k in 2,724 25.7 and 29.9,
// 1.0M in 3,347 33.2 and 39.7, 200k scattered over 20,490 56 and 140 (four tiles of
// which most of the nodes are empty).
// ============================================================================
constexpr int P2G_SPLIT_BLOCKS = 1536;
template <int D, bool SPLIT>
__device__ inline void p2g_blocks(const KP& p, float (*tile_all)[(D + 1) * Dims<D>::LTN]) {
    using Dm = Dims<D>;
    constexpr int LTN = Dm::LTN, C = D + 1, TN = Dm::TN, LX = Dm::LX, LY = Dm::LY;
    constexpr int NS = D == 3 ? 27 : 9, EACH = SPLIT ? NW : 1;
    const int c = threadIdx.x & 63, first = SPLIT ? (int)(threadIdx.x >> 6) : 0;
    float* mine = tile_all[threadIdx.x >> 6];
    int l[D];
    local_coords<D>(c, l);
    int base;  // tile index of this cell's stencil corner
    {
        int off0[D];
        base = tile_index<D>(l, 0, off0);
    }
    const XcdRange xr = SPLIT ? xcd_blocks(p.ctr->nblocks) : xcd_wave_blocks(p.ctr->nblocks);
    for (int kb = xr.first; kb < xr.end; kb += xr.step) {
        // one scene: heavy blocks first within the XCD's range; batches keep
        // slot order, measured faster there (small blocks of many scenes, and
        // neighbouring waves share a scene in slot order)
        const int b = p.nscenes > 1 ? kb : p.block_order[kb];
        const SceneParams& sc = p.scn[p.block_scene[b]];
        if (!sc.active || block_empty(p, b)) continue;
        for (int t = c; t < C * LTN; t += 64) mine[t] = 0.0f;
        int bb[D];
        block_coords<D>(p, b, bb);
        float acc[NS][C];
#pragma unroll
        for (int n = 0; n < NS; ++n)
#pragma unroll
            for (int ch = 0; ch < C; ++ch) acc[n][ch] = 0.0f;
        const int i0 = p.cell_start[b * 65 + c] + first, i1 = p.cell_start[b * 65 + c + 1];
        for (int i = i0; i < i1; i += EACH) {
            float w[D][3], dw[D][3], X[D];
            if (!cell_particle<D>(p, sc, i, bb, l, w, dw, X)) continue;
            float mv[C];
            mv[0] = p.pcur[PF<D>::M * p.pcap + i];
#pragma unroll
            for (int a = 0; a < D; ++a) mv[1 + a] = mv[0] * p.pcur[(PF<D>::V + a) * p.pcap + i];
            if constexpr (D == 3) {
#pragma unroll
                for (int ii = 0; ii < 3; ++ii)
#pragma unroll
                    for (int jj = 0; jj < 3; ++jj) {
                        const float wij = w[0][ii] * w[1][jj];
#pragma unroll
                        for (int kk = 0; kk < 3; ++kk) {
                            const float wt = wij * w[2][kk];
#pragma unroll
                            for (int ch = 0; ch < C; ++ch) acc[(ii * 3 + jj) * 3 + kk][ch] += wt * mv[ch];
                        }
                    }
            } else {
#pragma unroll
                for (int ii = 0; ii < 3; ++ii)
#pragma unroll
                    for (int jj = 0; jj < 3; ++jj) {
                        const float wt = w[0][ii] * w[1][jj];
#pragma unroll
                        for (int ch = 0; ch < C; ++ch) acc[ii * 3 + jj][ch] += wt * mv[ch];
                    }
            }
        }
        MPM_STEP_FENCE();
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            const int t = D == 3 ? base + (n / 9) * LX + ((n / 3) % 3) * LY + n % 3 : base + (n / 3) * LX + n % 3;
#pragma unroll
            for (int ch = 0; ch < C; ++ch) mine[ch * LTN + t] += acc[n][ch];
            MPM_STEP_FENCE();
        }
        if (SPLIT) {
            __syncthreads();
            store_wave_tiles<D, C>(p, b, tile_all[0]);
            __syncthreads();
            continue;
        }
        float* dst = p.tiles + (int64_t)b * C * TN;
        for (int t = c; t < C * TN; t += 64) {
            const int cc = t / TN;
            int nb, local, tc[D];
            tile_map<D>(t - cc * TN, nb, local, tc);
            dst[t] = mine[cc * LTN + lds_index<D>(tc)];
        }
        MPM_STEP_FENCE();
    }
}
template <int D>
__global__ __launch_bounds__(BWG) void k_p2g(KP p) {
    __shared__ float tile_all[NW][(D + 1) * Dims<D>::LTN];
    if (p.ctr->nblocks <= P2G_SPLIT_BLOCKS) p2g_blocks<D, true>(p, tile_all);
    else p2g_blocks<D, false>(p, tile_all);
}

// Tile sum of P2G + Flag_Setup_Helper (Flag_Setup_Helper.h:25-35) +
// Velocity_Normalization_Helper (Velocity_Normalization_Helper.h:39-52)
template <int D>
__global__ __launch_bounds__(WG) void k_normalize(KP p) {
    const XcdRange r = xcd_wave_blocks(p.ctr->nblocks);
    const int lane = threadIdx.x & 63;
    for (int b = r.first; b < r.end; b += r.step) {
        const SceneParams& sc = p.scn[p.block_scene[b]];
        if (!sc.active) continue;
        const int n = b * 64 + lane;
        float v[D + 1];
        gather_node_tiles<D, D + 1>(p, sc, n, v);
        const float m = v[0];
        const bool interior = m > 0.0f;
        p.g_m[n] = m;
        p.g_flags[n] = interior ? MPM_FLAG_INTERIOR_DEV : 0u;
        const float inv = interior ? 1.0f / m : 0.0f;
#pragma unroll
        for (int a = 0; a < D; ++a) p.g_v[a * p.gcap + n] = interior ? v[1 + a] * inv : v[1 + a];
    }
}

// gather of `nch` grid channel arrays into an LDS tile
template <int D, int NCH>
__device__ inline void gather_tile(const KP& p, const int* nbr, float (*tile)[Dims<D>::LTN], const float* const* src) {
    constexpr int TN = Dims<D>::TN;
    for (int t = threadIdx.x; t < TN; t += (int)blockDim.x) {
        int nb, local, tc[D];
        tile_map<D>(t, nb, local, tc);
        const int blk = nbr[nb];
        const int li = lds_index<D>(tc);
#pragma unroll
        for (int c = 0; c < NCH; ++c) tile[c][li] = blk >= 0 ? src[c][(int64_t)blk * 64 + local] : 0.0f;
    }
}

// Process_Waiting_Particles (MPM_Example.cpp:827-840): V0 = m / (sum w m_i / dx^d)
template <int D>
__global__ __launch_bounds__(BWG) void k_init_volume(KP p) {
    using Dm = Dims<D>;
    constexpr int LTN = Dm::LTN, NBR = Dm::NBR;
    __shared__ float tile[1][LTN];
    __shared__ int nbr[NBR];
    const int nblocks = p.ctr->nblocks;
    const XcdRange xr = xcd_blocks(nblocks);
    for (int kb = xr.first; kb < xr.end; kb += xr.step) {
        const int b = p.block_order[kb];  // heavy blocks first within the XCD's range
        const SceneParams& sc = p.scn[p.block_scene[b]];
        if (!sc.waiting || block_empty(p, b)) continue;
        float vol = 1.0f;
        for (int a = 0; a < D; ++a) vol *= sc.dx;
        const float inv_vol = 1.0f / vol;
        if (threadIdx.x < NBR) nbr[threadIdx.x] = p.block_nbr[b * NBR + threadIdx.x];
        int bb[D];
        block_coords<D>(p, b, bb);
        __syncthreads();
        const float* src[1] = {p.g_m};
        gather_tile<D, 1>(p, nbr, tile, src);
        __syncthreads();
        const int i1 = p.block_pstart[b + 1];
        for (int i = p.block_pstart[b] + (int)threadIdx.x; i < i1; i += BWG) {
            // the waiting particles are those without a volume yet (new or emitted)
            if (p.pcur[PF<D>::VOL * p.pcap + i] != 0.0f) continue;
            float w[D][3], dw[D][3], X[D];
            int l[D];
            if (!particle_weights<D>(p, sc, i, bb, w, dw, l, X)) continue;
            float rho = 0.0f;
#pragma unroll
            for (int s = 0; s < Dm::ST; ++s) {
                int off[D];
                const int t = tile_index<D>(l, s, off);
                rho += stencil_weight<D>(w, off) * tile[0][t];
            }
            rho *= inv_vol;
            p.pcur[PF<D>::VOL * p.pcap + i] = p.pcur[PF<D>::M * p.pcap + i] / rho;
        }
        __syncthreads();
    }
}

// ============================================================================
// Explicit force of one particle, added to its cell's 3^D nodes:
// f_i += g m w_i - A grad w_i, A = V0 P F^T (MPM_Example.cpp:774-784).  The
// sums over all but the last axis are shared by the three nodes along it.
template <int D>
__device__ inline void add_explicit_force(const SceneParams& sc, const float (*w)[3], const float (*dw)[3], const float* A,
                                          float m, float (*acc)[D]) {
    float gm[D];
#pragma unroll
    for (int a = 0; a < D; ++a) gm[a] = sc.gravity[a] * m;
#pragma unroll
    for (int r = 0; r < (D == 3 ? 9 : 3); ++r) {
        const int i = D == 3 ? r / 3 : r, j = r % 3;
        const float wr = D == 3 ? w[0][i] * w[1][j] : w[0][i];
        const float gx = D == 3 ? dw[0][i] * w[1][j] : dw[0][i], gy = D == 3 ? w[0][i] * dw[1][j] : 0.0f;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            float even = gm[a] * wr - A[a * D] * gx;
            if (D == 3) even -= A[a * D + 1] * gy;
            const float odd = A[a * D + D - 1] * wr;
#pragma unroll
            for (int k = 0; k < 3; ++k) acc[r * 3 + k][a] += even * w[D - 1][k] - odd * dw[D - 1][k];
        }
    }
}

// Constitutive update (MPM_Example.cpp:563-571) of particle i of material
// mat (CONST: plasticity, F, Jp and the CG operator record) and its stress
// term A of the explicit force (FORCE: f_i -= A grad w_i with A = V0 P F^T,
// MPM_Example.cpp:757-784); an EOS particle has no constitutive model and its
// term is A = -(V0/rho) K rho^(gamma-1) I (MPM_Example.cpp:774-782).
// ============================================================================
// The operator record's position: particle i's stencil offsets, the same
// arithmetic as the weights of its binned cell (binning and the record are
// formed from the same position, and particles do not move between them).
template <int D>
__device__ inline void particle_offsets(const KP& p, const SceneParams& sc, int i, float* xo) {
#pragma unroll
    for (int a = 0; a < D; ++a) {
        int c;
        xo[a] = stencil_offset(p.pcur[(PF<D>::X + a) * p.pcap + i], sc.dx, sc.inv_dx, c);
    }
}

template <int D, bool CONST, bool FORCE>
__device__ __forceinline__ void particle_stress(const KP& p, const SceneParams& sc, const Material& mat, int i,
                                                float* A) {
    constexpr int DD = D * D;
    float Jp = p.pcur[PF<D>::J * p.pcap + i];
    const float V0 = p.pcur[PF<D>::VOL * p.pcap + i];
    if (mat.eos) {
        // EOS fluid (Jp slot = density): no constitutive model
        const float rg = powf(Jp, mat.gamma - 1.0f);
        if (CONST) {
            float xo[D];
            particle_offsets<D>(p, sc, i, xo);
            store_operator_eos<D>(p, i, V0 * mat.K * mat.gamma * rg, xo);
            if (!FORCE) {
#pragma unroll
                for (int k = 0; k < DD; ++k) p.rcache[k * p.pcap + i] = (k % (D + 1) == 0) ? 1.0f : 0.0f;
            }
        }
        // f += (V0/rho) K rho^(gamma-1) grad w
        const float coeff = V0 / Jp * mat.K * rg;
#pragma unroll
        for (int k = 0; k < DD; ++k) A[k] = (k % (D + 1) == 0) ? -coeff : 0.0f;
    } else {
        float F[DD], R[DD];
#pragma unroll
        for (int k = 0; k < DD; ++k) F[k] = p.pcur[(PF<D>::F + k) * p.pcap + i];
        if (CONST) {
            float U[DD];
            double Sv[D];
            plasticity<D>(F, Jp, R, mat, U, Sv);
#pragma unroll
            for (int k = 0; k < DD; ++k) {
                p.pcur[(PF<D>::F + k) * p.pcap + i] = F[k];
                // R is read back only by the staged explicit force
                if (!FORCE) p.rcache[k * p.pcap + i] = R[k];
            }
            p.pcur[PF<D>::J * p.pcap + i] = Jp;
            StressState<D> so;
            stress_state<D>(F, R, Jp, mat, so);
            float xo[D];
            particle_offsets<D>(p, sc, i, xo);
            store_operator<D>(p, i, so, V0, xo, U, Sv);
        } else {
#pragma unroll
            for (int k = 0; k < DD; ++k) R[k] = p.rcache[k * p.pcap + i];
        }
        if (FORCE) {
            StressState<D> st;
            stress_state<D>(F, R, Jp, mat, st);
            float P[DD];
            first_pk<D>(st, P);
            // V0 P F^T
#pragma unroll
            for (int r = 0; r < D; ++r)
#pragma unroll
                for (int cc = 0; cc < D; ++cc) {
                    float s = 0.0f;
#pragma unroll
                    for (int k = 0; k < D; ++k) s += P[r * D + k] * F[cc * D + k];
                    A[r * D + cc] = s * V0;
                }
        }
    }
}

// One work-group per block, its particles in chunks of PF_CHUNK (a full
// block of 8 per cell is one chunk).  Each chunk is first updated a particle
// per thread in storage order (coalesced loads and stores; a wave past the
// block's last particle skips its part), one pass per entry of the scene's
// material table, each pass taking the particles of that entry (a single
// pass without a check in a one-material scene): the material's parameters
// stay scalar operands.  With FORCE the chunk's stress terms go to LDS and
// are then summed cell by cell (lane = cell, waves interleave a cell's
// particles) in registers and added to the wave tiles once per chunk.  Bound by
// the FP64 SVD.  Against adding every particle to the tile (81 ordered
// read-add-writes each): avalanche of 1.0M particles 138 -> 129 us, two balls of
// 243k 57.6 -> 52.2, twelve scenes 103 -> 96, fluid of 20k 42 -> 29, balls of
// 3.8k 26.7 -> 22.3.  Loading the next particle ahead takes the kernel over 168
// registers, to two waves a SIMD (1.0M: 160 us).
constexpr int PF_CHUNK = 2 * BWG;
template <int D, bool CONST, bool FORCE>
__global__ __launch_bounds__(BWG) void k_particle_force(KP p) {
    using Dm = Dims<D>;
    constexpr int LTN = Dm::LTN, DD = D * D, ST = Dm::ST;
    __shared__ __align__(16) float tile[NW * D * LTN];
    __shared__ float stress[DD][PF_CHUNK];
    const int nblocks = p.ctr->nblocks;
    const int c = threadIdx.x & 63, wv = threadIdx.x >> 6;
    float* mine = tile + wv * D * LTN;
    int l[D], off0[D];
    local_coords<D>(c, l);
    const int base = tile_index<D>(l, 0, off0);  // cell c's stencil corner
    const XcdRange xr = xcd_blocks(nblocks);
    for (int kb = xr.first; kb < xr.end; kb += xr.step) {
        const int b = p.block_order[kb];  // heavy blocks first within the XCD's range
        const SceneParams& sc = p.scn[p.block_scene[b]];
        if (!sc.active || block_empty(p, b)) continue;
        int bb[D];
        slot_coords<D>(p.block_slot[b] - sc.slot_base, sc.nb, bb);  // computed: the loaded form costs occupancy here
        if (FORCE)
            for (int t = threadIdx.x; t < NW * D * LTN; t += BWG) tile[t] = 0.0f;
        const int p0 = p.block_pstart[b], p1 = p.block_pstart[b + 1];
        const int c0 = p.cell_start[b * 65 + c], c1 = p.cell_start[b * 65 + c + 1];
        const int nmat = sc.nmat;
        for (int chunk = p0; chunk < p1; chunk += PF_CHUNK) {
            for (int half = 0; half < PF_CHUNK; half += BWG) {
                const int t = half + (int)threadIdx.x, i = chunk + t;
                if (chunk + half + (int)(threadIdx.x & ~63u) >= p1) continue;  // the wave's part is past the block
                for (int u = 0; u < nmat; ++u) {
                    if (i < p1 && (nmat == 1 || __float_as_int(p.pcur[PF<D>::MAT * p.pcap + i]) == u)) {
                        float A[DD];
                        particle_stress<D, CONST, FORCE>(p, sc, sc.mats[u], i, A);
                        if (FORCE) {
#pragma unroll
                            for (int k = 0; k < DD; ++k) stress[k][t] = A[k];
                        }
                    }
                }
            }
            if (FORCE) {
                __syncthreads();  // the chunk's stress terms (and, first, the zeroed tiles)
                const int lo = max(c0, chunk), hi = min(c1, chunk + PF_CHUNK);
                float acc[ST][D];
#pragma unroll
                for (int n = 0; n < ST; ++n)
#pragma unroll
                    for (int a = 0; a < D; ++a) acc[n][a] = 0.0f;
                for (int j = lo + wv; j < hi; j += NW) {
                    float w[D][3], dw[D][3], X[D];
                    if (!cell_particle<D>(p, sc, j, bb, l, w, dw, X)) continue;
                    float A[DD];
#pragma unroll
                    for (int k = 0; k < DD; ++k) A[k] = stress[k][j - chunk];
                    add_explicit_force<D>(sc, w, dw, A, p.pcur[PF<D>::M * p.pcap + j], acc);
                }
                // (lanes hold distinct cells: at one node of the stencil no two write the same place)
#pragma unroll
                for (int n = 0; n < ST; ++n) {
                    const int t = D == 3 ? base + (n / 9) * Dm::LX + ((n / 3) % 3) * Dm::LY + n % 3 : base + (n / 3) * Dm::LX + n % 3;
#pragma unroll
                    for (int a = 0; a < D; ++a) mine[a * LTN + t] += acc[n][a];
                    MPM_STEP_FENCE();
                }
                __syncthreads();  // before the next chunk overwrites the stress terms
            }
        }
        if (FORCE) {
            store_wave_tiles<D, D>(p, b, tile);
            __syncthreads();
        }
    }
}

// ============================================================================
// Grid update: tile sum of the force, Explicit_Force_Helper (v* = v + dt f/m),
// plane collision (Grid_Based_Collision_Helper.h:57-85) and the CG set-up
// (MPM_RHS_Helper, Reset_Solver_Channels: r = b = v*, s = 0).
// WRITE_F keeps the force in g_q for inspection.
// ============================================================================
template <int D, bool FORCE, bool COLL, bool CGINIT, bool WRITE_F>
__global__ __launch_bounds__(WG) void k_grid_update(KP p) {
    if (CGINIT) {
        // a new solve for every scene; one at rest or without blocks is done
        if (blockIdx.x == 0) {
            __shared__ int rest;
            if (threadIdx.x == 0) rest = 0;
            __syncthreads();
            for (int si = threadIdx.x; si < p.nscenes; si += WG) {
                CGState& cg = p.cg[si];
                const int idle = !p.scn[si].active || p.sst[si].block_end <= p.sst[si].block_begin ? 1 : 0;
                cg.iter = 0;
                cg.arrived = 0;
                cg.done = cg.closed = cg.converged = idle;
                cg.multiplies = p.one_active ? 0 : idle;
                cg.rho_hist[0] = cg.rho_hist[1] = 0.0;
                cg.alpha = cg.beta = cg.conv = cg.rr = cg.sq = 0.0;
                if (idle) atomicAdd(&rest, 1);
            }
            __syncthreads();
            if (threadIdx.x == 0) {
                p.ctr->cg_ndone = rest;
                p.ctr->cg_iters = 0;
                p.ctr->door = 0;
                p.ctr->group = 0;
            }
        }
        // k_cg_solve's places for partials (both parities) and its counted waits
        if (p.one_launch)
            for (int i = blockIdx.x * WG + threadIdx.x; i < max(2 * CG_RESIDENT, CG_WAIT_INTS); i += gridDim.x * WG) {
                const double empty = __longlong_as_double((long long)CG_EMPTY);
                if (i < 2 * CG_RESIDENT) p.bsum[i] = p.bmax[i] = p.bsq[i] = empty;
                if (i < CG_WAIT_INTS) p.cg_waits[i] = 0;
            }
    }
    const XcdRange r = xcd_wave_blocks(p.ctr->nblocks);
    const int lane = threadIdx.x & 63;
    for (int b = r.first; b < r.end; b += r.step) {
        const SceneParams& sc = p.scn[p.block_scene[b]];
        if (!sc.active) continue;
        const int n = b * 64 + lane;
        const float dt = sc.dt;
        const bool interior = (p.g_flags[n] & MPM_FLAG_INTERIOR_DEV) != 0;
        float vs[D];
        if (FORCE) {
            float f[D];
            gather_node_tiles<D, D>(p, sc, n, f);
            if (WRITE_F) {
#pragma unroll
                for (int a = 0; a < D; ++a) p.g_q[a * p.gcap + n] = f[a];
            }
            if (interior) {
                const float dtm = dt / p.g_m[n];
#pragma unroll
                for (int a = 0; a < D; ++a) vs[a] = p.g_v[a * p.gcap + n] + dtm * f[a];
            } else {
#pragma unroll
                for (int a = 0; a < D; ++a) vs[a] = 0.0f;
            }
        } else {
#pragma unroll
            for (int a = 0; a < D; ++a) vs[a] = p.g_vs[a * p.gcap + n];
        }
        if (COLL && interior) {
            float x[D];
            node_center<D>(p, sc, n, x);
            for (int id = 0; id < sc.nplanes; ++id) {
                if (!inside_plane(sc, id, x, D)) continue;
                float proj = 0.0f;
#pragma unroll
                for (int a = 0; a < D; ++a) proj += vs[a] * sc.pn[id][a];
                if (proj < 0.0f) {
#pragma unroll
                    for (int a = 0; a < D; ++a) vs[a] -= sc.pn[id][a] * proj;
                    float nrm = 0.0f;
#pragma unroll
                    for (int a = 0; a < D; ++a) nrm += vs[a] * vs[a];
                    nrm = sqrtf(nrm);
                    const float mu = sc.pmu[id];
                    if (-proj * mu < nrm) {
#pragma unroll
                        for (int a = 0; a < D; ++a) vs[a] += vs[a] / nrm * proj * mu;
                    } else {
#pragma unroll
                        for (int a = 0; a < D; ++a) vs[a] = 0.0f;
                    }
                }
            }
        }
        if (FORCE || COLL) {
#pragma unroll
            for (int a = 0; a < D; ++a) p.g_vs[a * p.gcap + n] = vs[a];
        }
        if (CGINIT) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                p.g_r[a * p.gcap + n] = interior ? vs[a] : 0.0f;
                p.g_s[a * p.gcap + n] = p.one_launch ? __uint_as_float(CG_EMPTY_FLOAT) : 0.0f;
            }
            if (p.one_launch && (n >> 6) < min(p.bcap, CG_RESIDENT))
                for (int i = n & 63; i < D * Dims<D>::TN; i += 64)
                    cg_tile<D>(p, 0, n >> 6)[i] = cg_tile<D>(p, 1, n >> 6)[i] = __uint_as_float(CG_EMPTY_FLOAT);
        }
    }
}

#pragma clang fp contract(on)
// ============================================================================
// CG (Apply_Force's solve, MPM_Example.cpp:700-711) for every scene of the
// batch at once: Hestenes-Stiefel CG in the M inner product with a restart
// at iteration 0.  Launch order per solve:
//   grid_update<CGINIT>, cg_force<RESTART>, cg_node<RESTART>,
//   then for k = 0, 1, ...: cg_force(k), cg_node(k).
// A scene whose solve is finished is skipped by every kernel; when all are,
// the kernels return at once.
// ============================================================================

// s = r (k = 0) or r + beta s
__device__ inline float cg_direction(float r, float s, float beta, int k) {
    return k == 0 ? r : fmaf(beta, s, r);
}

// The node pass's work-groups: NGB blocks, a wave each.  What they exchange:
//   bsq   the runs' partials of s.q,
//   bsum  the runs' partials of r.r and max |r|^2, in pairs,
//   bmax  for scenes of many runs the sums over chunks of CG_CHUNK_RUNS of
//         them, s.q and then the pairs, a copy per XCD.
constexpr int NGW = 512;
static_assert(NGW == 64 * NGB, "a wave per block");
constexpr int CG_NODE_GROUPS = 768;  // three of 512 threads a CU: all fit at once
constexpr int CG_DIRECT_RUNS = 192;  // (scenes of up to so many runs are summed directly)

// LDS of the CG operator's work-group of NT threads:
//   coef  the block's coefficient rows, later the node contributions of every
//         part (27 x 64 x channels a part, running on into pack);
//   pack  the packed particles of a chunk (and a few words past them, read
//         ahead and unused), before that the node tile the coefficients come
//         from;
//   tile  the force tile, and before it the counting sort's histogram;
//   cell  the cell of every particle of the chunk;
//   perm  the block's cells by descending particle count.
template <int D, int NT>
struct OperatorLds {
    using CS = CellStencil<D>;
    static constexpr int LTN = Dims<D>::LTN;
    static constexpr int TASKS = D * 64;         // cells and channels of a block
    static constexpr int PARTS = NT / TASKS;     // lanes that share a task's particles
    static constexpr int COEF = CS::ROWS * 64;
    static constexpr int PACKED = CS::PACK * (NT + PARTS);
    static constexpr int NODES = CS::NC * TASKS * PARTS;
    // the force tile sits past the packed particles' place or the node
    // contributions, whichever ends last -- inside pack where that has room
    static constexpr int TILE = NODES > COEF + 1024 ? NODES : COEF + 1024;
    static constexpr int WORDS = TILE + D * LTN > COEF + PACKED ? TILE + D * LTN : COEF + PACKED;
    static_assert(D * LTN <= 1024 && COEF % 4 == 0 && TILE % 4 == 0, "aliases");
    float coef[WORDS];
    unsigned char cell[NT];
    unsigned char perm[64];
    __device__ float* pack() { return coef + COEF; }
    __device__ float* tile() { return coef + TILE; }
};

// perm: the cells by descending count n (lane = cell) -- a counting sort by
// one wave; the order among equal counts follows the LDS atomics and decides
// only which lane sums a cell, never its sum.
__device__ inline void sort_cells(int n, int lane, int* hist, unsigned char* perm) {
    const int key = 63 - min(n, 63);
    hist[lane] = 0;
    MPM_STEP_FENCE();
    atomicAdd(&hist[key], 1);
    MPM_STEP_FENCE();
    const int h = hist[lane];
    int x = h;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    hist[lane] = x - h;
    MPM_STEP_FENCE();
    perm[atomicAdd(&hist[key], 1)] = (unsigned char)lane;
}

// One block of the operator by one work-group (every thread makes every call;
// all trip counts are uniform): open, then any number of apply.
//
// Particles are taken twice.  Storage order, one per lane, for the gather and
// the force map (about 415 operations): every lane is filled whatever the
// counts of the cells.  For the scatter a lane takes one cell and channel (a
// part of its particles in work-groups of more lanes than tasks) and keeps the
// 26 moments in registers, so nothing is read, added and written back per
// particle and only these 70 operations wait for the fullest cell of the
// wave; the cells are dealt to the waves by descending count, so that a
// wave's cells are alike.
template <int D, int NT, int R>
struct BlockOperator {
    using CS = CellStencil<D>;
    using Dm = Dims<D>;
    using L = OperatorLds<D, NT>;
    static constexpr int LTN = Dm::LTN, TN = Dm::TN, NBR = Dm::NBR, W = OpRec<D>::W, DD = D * D;
    static constexpr int PARTS = L::PARTS, TASKS = L::TASKS, LAST = NT / 64 - 1;
    static_assert(TN <= NT && D <= LAST, "thread roles");

    const KP& p;
    L& S;
    const float4* rec4;
    float4 next[W / 4];
    int b, tid, lane, wv, p0, p1, c0, c1, base;
    int chunks;  // particle p0 + t chunks + c sits at place t of chunk c
    int li, node;  // tile node tid: its LDS index and grid node (-1: none)

    const bool two;  // (ROUND_EITHER)

    __device__ BlockOperator(const KP& kp, L& lds, bool round_two = false)
        : p(kp), S(lds), rec4(reinterpret_cast<const float4*>(kp.pop)), tid(threadIdx.x), lane(tid & 63), wv(tid >> 6), two(round_two) {
        int l[D], off0[D];
        local_coords<D>(lane, l);
        base = tile_index<D>(l, 0, off0);  // cell `lane`'s stencil corner
    }
    // A block of more than NT particles is taken in chunks of every chunks-th
    // one, so that each chunk holds a like part of every cell: in consecutive
    // chunks most cells would have none, and their lanes nothing to sum.
    __device__ void load_records(int c) {
        const int64_t i = min(p0 + tid * chunks + c, p1 - 1);
#pragma unroll
        for (int k = 0; k < W / 4; ++k) next[k] = rec4[i * (W / 4) + k];
    }
    // the first place of chunk c whose particle is m or later
    __device__ int place(int m, int c) const {
        const unsigned d = (unsigned)max(m - p0 - c, 0);
        return chunks == 1 ? (int)d : (int)((d + (unsigned)chunks - 1u) / (unsigned)chunks);
    }
    __device__ void mark_cells(int c) {
        for (int t = place(c0, c), e = place(c1, c); t < e; ++t) S.cell[t] = (unsigned char)lane;
    }
    // Block bi: its ranges, the tile node of this thread, the order of its
    // cells and the first chunk's records (in flight).
    __device__ void open(int bi) {
        b = bi;
        p0 = p.block_pstart[b];
        p1 = p.block_pstart[b + 1];
        c0 = p.cell_start[b * 65 + lane];
        c1 = p.cell_start[b * 65 + lane + 1];
        chunks = max(1, (p1 - p0 + NT - 1) / NT);
        if (p1 > p0) load_records(0);
        li = 0;
        node = -1;
        if (tid < TN) {
            int nb, local, tc[D];
            tile_map<D>(tid, nb, local, tc);
            li = lds_index<D>(tc);
            const int blk = p.block_nbr[(int64_t)b * NBR + nb];
            node = blk >= 0 ? blk * 64 + local : -1;
        }
        if (wv == LAST) {
            sort_cells(c1 - c0, lane, reinterpret_cast<int*>(S.tile()), S.perm);
            mark_cells(0);
        }
    }
    // The operator of node values u (channels of tile node tid): leaves the
    // block's force tile in S.tile().  `again`: not the first apply since open.
    __device__ void apply(float inv_dx, const float* u, bool again) {
        float* pack = S.pack();
        if (tid < TN) {
#pragma unroll
            for (int a = 0; a < D; ++a) pack[a * LTN + li] = u[a];
        }
        if (again && wv == LAST && chunks > 1) mark_cells(0);
        __syncthreads();
        if (wv < D) {
            float c[CS::NC];
            cell_coefficients<D>(pack + wv * LTN, base, c);
#pragma unroll
            for (int n = 0; n < CS::NC; ++n)
                if (n != CS::MID) S.coef[CS::row(0, n) * 64 + wv * (CS::NC - 1) * 64 + lane] = c[n];
        }
        __syncthreads();
        // the lane's cell, channel and part of the scatter
        const int part = tid / TASKS, task = tid - part * TASKS;
        const bool scatter = part < PARTS;
        const int ch = task % D, mine = S.perm[task / D];
        const int m0 = p.cell_start[b * 65 + mine], m1 = scatter ? p.cell_start[b * 65 + mine + 1] : m0;
        float m[CS::NC];
#pragma unroll
        for (int n = 0; n < CS::NC; ++n) m[n] = 0.0f;
        const float scale = inv_dx * inv_dx;
        for (int c = 0; c < chunks; ++c) {
            if (p0 + tid * chunks + c < p1) {
                float rec[W];
#pragma unroll
                for (int k = 0; k < W / 4; ++k) {
                    rec[4 * k] = next[k].x;
                    rec[4 * k + 1] = next[k].y;
                    rec[4 * k + 2] = next[k].z;
                    rec[4 * k + 3] = next[k].w;
                }
                const OuterWeights<D> g(rec);
                float T[DD], A[DD];  // A = V0 F dP(T^T F)^T
                stencil_gradient<D>(g, S.coef, S.cell[tid], T);
                apply_operator<D, R>(rec, scale, two, T, A);
                pack_particle<D>(g, A, pack + tid * CS::PACK);
            }
            __syncthreads();
            if (c + 1 < chunks) {
                load_records(c + 1);
                if (wv == LAST) mark_cells(c + 1);
            }
            // the next particle's words load while the current one is added
            int j = place(m0, c) + part;
            const int end = place(m1, c);
            if (j < end) {
                const float *a = pack + j * CS::PACK, *ac = a + ch * 4;
                PackedForce<D> f0, f1;
                f0.load(a, ac);
                for (;;) {
                    a += CS::PACK * PARTS;
                    ac += CS::PACK * PARTS;
                    f1.load(a, ac);
                    add_force_moments<D>(f0, m);
                    j += PARTS;
                    if (j >= end) break;
                    a += CS::PACK * PARTS;
                    ac += CS::PACK * PARTS;
                    f0.load(a, ac);
                    add_force_moments<D>(f1, m);
                    j += PARTS;
                    if (j >= end) break;
                }
            }
            __syncthreads();
        }
        // every part's node contributions, then the force tile in cell order
        if (scatter) {
            nodes_of_cell<D>(m);
#pragma unroll
            for (int n = 0; n < CS::NC; ++n) S.coef[(part * CS::NC + n) * TASKS + ch * 64 + mine] = m[n];
        }
        if (wv == LAST)
            for (int t = lane; t < D * LTN; t += 64) S.tile()[t] = 0.0f;
        __syncthreads();
        if (wv < D) {
            const float* q = S.coef + wv * 64 + lane;
#pragma unroll
            for (int n = 0; n < CS::NC; ++n) m[n] = q[n * TASKS];
#pragma unroll 1
            for (int k = 1; k < PARTS; ++k) {
                q += CS::NC * TASKS;
#pragma unroll
                for (int n = 0; n < CS::NC; ++n) m[n] += q[n * TASKS];
            }
            add_cell_nodes<D>(m, base, lane, S.tile() + wv * LTN);
        }
        __syncthreads();
    }
    // The force tile to its place in memory (AGENT: other work-groups of this
    // kernel read it, FLAG: as values that are their own flags).
    template <bool AGENT, bool FLAG = false>
    __device__ void store(float* tile) {
        if (tid < TN) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const float f = S.tile()[a * LTN + li];
                st<AGENT>(tile + tid + a * TN, FLAG ? flagged(f) : f);
            }
        }
    }
};

// load(a, n): channel a of node n
template <int D, int NT, int R, bool AGENT, class Load>
__device__ inline void operator_block(const KP& p, int b, float inv_dx, bool two, OperatorLds<D, NT>& S, Load&& load) {
    BlockOperator<D, NT, R> op(p, S, two);
    op.open(b);
    float u[D];
#pragma unroll
    for (int a = 0; a < D; ++a) u[a] = 0.0f;
    if (op.node >= 0) {
#pragma unroll
        for (int a = 0; a < D; ++a) u[a] = load(a, op.node);
    }
    op.apply(inv_dx, u, false);
    op.template store<AGENT>(p.tiles + (int64_t)b * D * Dims<D>::TN);
    __syncthreads();
}

// MPM_CG_System::Force (MPM_CG_System.h:150-215) with the linearised operator
// record: T = sum_i grad w_ip (x) u_i;  A = L T;  q_i += A^T grad w_ip.
// RESTART applies it to v* (the initial guess); otherwise to the search
// direction of iteration k, s = r + beta s, formed while gathering.
//
// Bound by VALU issue in large scenes, by one block's chain of phases in small
// ones.  Per launch, against one lane per cell for everything (nodes read per
// particle, 81 LDS read-add-writes per particle): avalanche of 1.0M particles
// in 256^3 mid-slide 57 -> 49 us with chunks of consecutive particles, 42 with
// chunks that hold a part of every cell (32.9M, 19.9M, 16.7M VALU wave
// instructions); two balls of 243k 24.4, 20.0, 16.6; 3.8k particles 24.0, 13.2,
// 11.0.  One wave per block with the moments of its cells in registers (255
// VGPRs, two waves a SIMD) took 61 us: everything then waits for the fullest
// cell, which holds two to three times the mean.
//
// It also readies what the node pass after it exchanges: empty places for the
// partials, open doors, and which scenes are still live.
template <int D, bool RESTART>
__global__ __launch_bounds__(BWG, 4) void k_cg_force(KP p) {
    __shared__ __align__(16) OperatorLds<D, BWG> S;
    const int live = p.nscenes - p.ctr->cg_ndone;
    if (blockIdx.x == 0) {
        for (int si = threadIdx.x; si < p.nscenes; si += BWG) p.cg[si].closed = p.cg[si].done;
        if (threadIdx.x < 8) p.ctr->doors[threadIdx.x][0] = 0;
        if (threadIdx.x == 0) {
            p.ctr->live = live;
            p.ctr->again = 0;
        }
    }
    if (live <= 0) return;
    const int ng = cg_groups(p.ctr->nblocks), places = cg_places(ng, p.nscenes), chunks = 24 * cg_chunk_places(ng);
    for (int i = (int)blockIdx.x * BWG + (int)threadIdx.x; i < max(2 * places, chunks); i += (int)gridDim.x * BWG) {
        const double empty = __longlong_as_double((long long)CG_EMPTY);
        if (i < places) p.bsq[i] = empty;
        if (i < 2 * places) p.bsum[i] = empty;
        if (i < chunks) p.bmax[i] = empty;
    }
    const XcdRange xr = xcd_blocks(p.ctr->nblocks);
    for (int kb = xr.first; kb < xr.end; kb += xr.step) {
        const int b = p.block_order[p.bcap + kb];  // the fullest cells first within the XCD's range
        const int si = p.nscenes == 1 ? 0 : p.block_scene[b];
        const SceneParams& sc = p.scn[si];
        if (!sc.active || (p.nscenes > 1 && p.cg[si].done) || block_empty(p, b)) continue;
        operator_block<D, BWG, ROUND_LAUNCHED, false>(p, b, sc.inv_dx, false, S, [&](int a, int64_t n) {
            return RESTART ? p.g_vs[a * p.gcap + n] : p.g_s[a * p.gcap + n];
        });
    }
}

// Project (Project_Helper.h:30-45): zero at nodes inside a plane
template <int D>
__device__ inline bool project_zero(const KP& p, const SceneParams& sc, int n) {
    if (sc.project_mode != 0 || sc.nplanes == 0) return false;
    float x[D];
    node_center<D>(p, sc, n, x);
    for (int id = 0; id < sc.nplanes; ++id)
        if (inside_plane(sc, id, x, D)) return true;
    return false;
}

// sum and max over a wave; result valid in every lane
__device__ inline void wave_reduce2(double& sum, double& mx) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        sum += __shfl_xor(sum, off);
        mx = fmax(mx, __shfl_xor(mx, off));
    }
}

// Sum / max of `count` partials starting at `first`, in await_partials' order (a
// lane adds every 64th, then the lanes are added); the result is in every
// thread.  buf: 2 NT doubles of LDS.
template <int NT>
__device__ inline void reduce_range(const double* sums, const double* maxs, int first, int count, double* buf, double& sum,
                                    double& mx) {
    constexpr int U = 4;  // independent loads in flight per thread
    const int tid = (int)threadIdx.x, lane = tid & 63;
    sum = 0.0;
    mx = 0.0;
    __syncthreads();
    for (int base = 0; base < count; base += U * NT) {
        // the round's loads all go out before its first add (an index past
        // the range reads the range's last entry and is not added)
        double vs[U], vm[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = min(base + u * NT + tid, count - 1);
            vs[u] = ld_agent(sums + first + j);
            vm[u] = maxs ? ld_agent(maxs + first + j) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (base + u * NT >= count) break;
            const bool in = base + u * NT + tid < count;
            buf[tid] = in ? vs[u] : 0.0;
            buf[NT + tid] = in ? vm[u] : 0.0;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < NT / 64; ++w) {
                sum += buf[w * 64 + lane];
                mx = fmax(mx, buf[NT + w * 64 + lane]);
            }
            __syncthreads();
        }
    }
    wave_reduce2(sum, mx);
}

// Convergence test of iteration k (Convergence_Norm, MPM_CG_System.h:241-249:
// L-inf over nodes of |r|) on r.r and max |r|^2, and beta = rho_k / rho_{k-1}.
// A scene is done when the test passes (after cg_min iterations) or at its
// cap cg_max.  `record`: this thread writes the scene's state.
// The scene's inputs of the test, read in one go (before the partial
// reduction, so that their loads overlap it).
struct CGTestIn {
    double rho_prev, tol;
    int cg_min, cg_max;
    bool empty;
};
__device__ inline CGTestIn cg_test_in(const KP& p, int si, int k) {
    const SceneParams& sc = p.scn[si];
    CGTestIn in;
    in.rho_prev = ld_agent(&p.cg[si].rho_hist[(k + 1) & 1]);
    in.tol = sc.cg_tol;
    in.cg_min = sc.cg_min;
    in.cg_max = sc.cg_max;
    const int active = sc.active, b0 = p.sst[si].block_begin, b1 = p.sst[si].block_end;
    in.empty = (active == 0) | (b1 <= b0);
    return in;
}

__device__ inline bool cg_test(const KP& p, int si, int k, double rr, double mx, bool record, float& beta_f,
                               const CGTestIn& in) {
    CGState& cg = p.cg[si];
    const double conv = sqrt(mx);
    const bool pass = conv <= in.tol && (k >= in.cg_min || conv < (double)FLT_EPSILON);
    const bool done = pass || k >= in.cg_max || in.empty;
    const double beta = k == 0 ? 0.0 : rr / in.rho_prev;
    if (record) {
        if (k == 0) cg.multiplies = 1;  // the restart Multiply
        cg.iter = k;
        cg.conv = conv;
        cg.rr = rr;
        if (done) {
            cg.converged = (pass || in.empty) ? 1 : 0;
            st_agent(&cg.done, 1);
            atomicMax(&p.ctr->cg_iters, k);
            atomicAdd(&p.ctr->cg_ndone, 1);
        } else {
            st_agent(&cg.beta, beta);
            st_agent(&cg.rho_hist[k & 1], rr);
        }
    }
    beta_f = (float)beta;
    return done;
}

// ---- what work-groups of one launch exchange ---------------------------------
constexpr int CG_DOOR_CLOSED = 1 << 30;

// A value that is the same in every lane, in scalar registers.
__device__ inline double scalar(double v) {
    const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v)), hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
    return __hiloint2double(hi, lo);
}
// Every store of this wave has reached memory.
__device__ inline void drain_stores() { __asm__ __volatile__("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }

// ---- a partial that is its own flag -----------------------------------------
__device__ inline void put_partial(double* a, double v) {
    if (!(v == v)) v = __longlong_as_double(0x7ff8000000000000ll);
    st_agent(a, v);
}
__device__ inline void clear_partial(double* a) { st_agent(a, __longlong_as_double((long long)CG_EMPTY)); }
// The node values of one lane of a wave that holds a block.
template <int D, bool AGENT>
struct NodeRows {
    float x[D], r[D], s[D], q[D], m;
    bool interior;
    __device__ void load(const KP& p, int n) {
        interior = (p.g_flags[n] & MPM_FLAG_INTERIOR_DEV) != 0;
        m = p.g_m[n];
#pragma unroll
        for (int a = 0; a < D; ++a) {
            s[a] = ld<AGENT>(p.g_s + a * p.gcap + n);
            q[a] = p.g_q[a * p.gcap + n];
            x[a] = p.g_vs[a * p.gcap + n];
            r[a] = ld<AGENT>(p.g_r + a * p.gcap + n);
        }
    }
    // the block's r.r (M-weighted) and max |r|^2
    __device__ void residual(double& sum, double& mx) {
        sum = 0.0;
        mx = 0.0;
        if (interior) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                sum += (double)r[a] * ((double)r[a] * (double)m);
                mx += (double)r[a] * (double)r[a];
            }
        }
        wave_reduce2(sum, mx);
    }
    // x += alpha s, r -= alpha q on block b; its r.r and max |r|^2
    __device__ void step(const KP& p, int n, float alpha, double& sum, double& mx) {
        if (interior) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                p.g_vs[a * p.gcap + n] = alpha * s[a] + x[a];
                r[a] = -alpha * q[a] + r[a];
                st<AGENT>(p.g_r + a * p.gcap + n, r[a]);
            }
        }
        residual(sum, mx);
    }
};

// r = b - q, Project(r) at node n; r holds b (0 outside the interior)
template <int D>
__device__ inline void cg_restart_residual(const KP& p, const SceneParams& sc, int n, bool interior, const float* q, float* r) {
    if (interior) {
#pragma unroll
        for (int a = 0; a < D; ++a) r[a] = r[a] - q[a];
    }
    if (project_zero<D>(p, sc, n)) {
#pragma unroll
        for (int a = 0; a < D; ++a) r[a] = 0.0f;
    }
}

// CG restart of block b: q = dt^2/m q + x (Multiply_Helper), r = b - q,
// Project(r); the block's r.r (M-weighted) and max |r|^2.  STORE: q, r and s = 0
// are stored, otherwise nothing is.
template <int D, bool AGENT, bool STORE>
__device__ inline void cg_restart_block(const KP& p, const SceneParams& sc, int b, int lane, float* q, double& sum, double& mx) {
    const int n = b * 64 + lane;
    const float sds = sc.dt * sc.dt;
    const bool interior = (p.g_flags[n] & MPM_FLAG_INTERIOR_DEV) != 0;
    float rv[D];
    gather_node_tiles<D, D, AGENT>(p, sc, n, q);
#pragma unroll
    for (int a = 0; a < D; ++a) rv[a] = p.g_r[a * p.gcap + n];
    const float mn = p.g_m[n];
    if (interior) {
        const float cm = sds / mn;
#pragma unroll
        for (int a = 0; a < D; ++a) q[a] = cm * q[a] + p.g_vs[a * p.gcap + n];
    }
    cg_restart_residual<D>(p, sc, n, interior, q, rv);
    if (STORE) {
#pragma unroll
        for (int a = 0; a < D; ++a) {
            st<AGENT>(p.g_r + a * p.gcap + n, rv[a]);
            st<AGENT>(p.g_s + a * p.gcap + n, 0.0f);
            p.g_q[a * p.gcap + n] = q[a];
        }
    }
    sum = 0.0;
    mx = 0.0;
    if (interior) {
#pragma unroll
        for (int a = 0; a < D; ++a) {
            sum += (double)rv[a] * ((double)rv[a] * (double)mn);
            mx += (double)rv[a] * (double)rv[a];
        }
    }
    wave_reduce2(sum, mx);
}

// Tile sum of the operator, q = dt^2/m q + s, Project(q) on block b; the
// block's s.q.  FORM: this iteration's s = r + beta s is formed and stored first
// (interior nodes), and q is stored.
template <int D, bool FORM, bool AGENT>
__device__ inline void cg_product_block(const KP& p, const SceneParams& sc, int b, int lane, float beta, int k, float* q, double& sum) {
    const float sds = sc.dt * sc.dt;
    const int n = b * 64 + lane;
    const bool interior = (p.g_flags[n] & MPM_FLAG_INTERIOR_DEV) != 0;
    float sv[D], rv[D];
    // s, r and m load alongside the flags and the tile gather (every node of
    // an active block has them; only interior ones use them)
    const float mn = p.g_m[n];
#pragma unroll
    for (int a = 0; a < D; ++a) {
        sv[a] = ld<AGENT>(p.g_s + a * p.gcap + n);
        if (FORM) rv[a] = ld<AGENT>(p.g_r + a * p.gcap + n);
    }
    gather_node_tiles<D, D, AGENT>(p, sc, n, q);
    if (interior) {
        const float cm = sds / mn;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            if (FORM) {
                sv[a] = cg_direction(rv[a], sv[a], beta, k);
                st<AGENT>(p.g_s + a * p.gcap + n, sv[a]);
            }
            q[a] = cm * q[a] + sv[a];
        }
    }
    if (project_zero<D>(p, sc, n)) {
#pragma unroll
        for (int a = 0; a < D; ++a) q[a] = 0.0f;
    }
    if (FORM) {
#pragma unroll
        for (int a = 0; a < D; ++a) p.g_q[a * p.gcap + n] = q[a];
    }
    sum = 0.0;
    double mx = 0.0;
    if (interior) {
        const double m = (double)mn;
#pragma unroll
        for (int a = 0; a < D; ++a) sum += (double)sv[a] * ((double)q[a] * m);
    }
    wave_reduce2(sum, mx);
}

// alpha = rho_k / s.q
__device__ inline double cg_alpha(double rho, double sq) { return sq != 0.0 ? rho / sq : (double)FLT_MAX; }
__device__ inline void cg_record_alpha(CGState& cg, double sq, double alpha) {
    cg.sq = sq;
    cg.alpha = alpha;
    cg.multiplies += 1;
}

// ---- the node pass -----------------------------------------------------------
// Everything of an iteration but the operator, in one launch: q = A s and s.q;
// alpha, x and r, r.r; the convergence test, beta and s.  Its work-groups
// exchange the two sums inside the launch.
//
// Groups of NGB consecutive blocks, a wave each.  A run is the part of one
// scene's blocks in one group: its partial is the sum over them in block
// order, formed and read by the wave of its first block.  A partial's place is
// its own flag: it holds CG_EMPTY until the partial is there, the operator
// launch before empties it.  A scene of many runs is summed in chunks first, by
// the wave of a chunk's first run: everybody reading everybody's partials was
// most of the pass (420 work-groups: 3 and 5 us for the two sums).  The order
// of every sum is fixed, so the result depends neither on the grid nor on who
// computes a group.
//
// Work-groups wait for one another, so all that take part have to be running.
// Each takes a ticket at its XCD's door when it starts.  Before anything is
// changed that the pass reads, every one waits until all tickets are out; one
// that has waited for too long while some are missing closes the doors.  Then
// those that hold a ticket wait for one another, share all groups by ticket and
// start again (the partials that are there already are the same), and those
// that come later leave.  They may come when the others have long finished, so
// nothing is stored before the ticket is known; and a block that one ticket
// holder has begun may end with another, on an XCD whose stores are not ordered
// with the first one's, so what is stored before all are settled (q) is the
// same whoever stores it.  (A door is one word: tickets taken, and once it is
// closed a bit and how many had been taken by then.  The first door to close
// does so while one of its tickets is missing, so that nobody ever sees all of
// them taken; the others follow.)
//
// Bound by latency: the gather of the tiles (2.4 to 3.5 us), two sums that each
// take two or three memory round trips, the start and end of a launch.  Per
// iteration, against three launches for one scene (s; q and s.q; x, r and r.r,
// each reducing the partials of the one before) and four for a batch: avalanche
// of 1.0M particles (3,360 blocks) 18.6 -> 17.0 us, of 2.0M (6,500) 24.1 ->
// 22.2, two balls of 243k (1,100) 14.1 -> 10.9, twelve scenes (2,000 blocks)
// 18.9 -> 13.4; and a captured substep holds half the launches.  Work-groups
// of 256 threads take 18.0, of 1024 15.9 us on the first, 11.4 and 12.9 on the
// third.
// Waits until the doors are settled: 0 if all have come that own groups of the
// ng, else the number of those that have, all of them here now, and `rank`
// among them of the one with `ticket`.  (One wave.)
__device__ inline int cg_settle(const KP& p, int ng, long long t0, int ticket, int lane, int& rank) {
    int* const word = p.ctr->doors[lane & 7];
    const auto close = [&](int v) {
        return __hip_atomic_compare_exchange_strong(word, &v, v | v << 16 | CG_DOOR_CLOSED, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT);
    };
    const int x = lane & 7;
    const int most = min((int)(gridDim.x >> 3), (int)(((int64_t)ng * (x + 1)) >> 3) - (int)(((int64_t)ng * x) >> 3));
    int v;
    for (;;) {
        v = ld_agent(word);
        if (__any(v >= CG_DOOR_CLOSED)) break;
        const unsigned long long missing = __ballot(v < most);
        if (missing == 0) return 0;
        if (wall_clock64() - t0 >= p.door_ticks && __any(lane == __ffsll(missing) - 1 && close(v))) break;
        __builtin_amdgcn_s_sleep(1);
    }
    while ((v = ld_agent(word)) < CG_DOOR_CLOSED)
        if (lane < 8) (void)close(v);
    const int taken = (v & ~CG_DOOR_CLOSED) >> 16;
    int group = 0;
    rank = ticket;
#pragma unroll
    for (int y = 0; y < 8; ++y) {
        const int t = __shfl(taken, y);
        if (y < (int)(blockIdx.x & 7)) rank += t;
        group += t;
    }
    if (lane == 0) {
        add_agent(&p.ctr->again, 1);
        while (ld_agent(&p.ctr->again) < group) __builtin_amdgcn_s_sleep(1);
    }
    return group;
}

// A partial, W = 1 or 2 values: sums are added, the second is a maximum.
template <int W>
__device__ inline void put_values(double* at, const double* v) {
#pragma unroll
    for (int w = 0; w < W; ++w) put_partial(at + w, v[w]);
}
// Waits for `count` partials, the i-th at(i), and reduces them; one wave, result
// in every lane.  `late` is asked while it waits: nonzero ends the wait and is
// returned.
template <int W, int U, class At, class F>
__device__ inline int await_values(At&& at, int count, int lane, double* v, F&& late) {
#pragma unroll
    for (int w = 0; w < W; ++w) v[w] = 0.0;
    for (int base = 0; base < count; base += U * 64) {
        double u[U][W];
#pragma unroll
        for (int j = 0; j < U; ++j)
#pragma unroll
            for (int w = 0; w < W; ++w)
                u[j][w] = base + j * 64 + lane < count ? __longlong_as_double((long long)CG_EMPTY) : 0.0;
        for (;;) {
            bool waiting = false;
#pragma unroll
            for (int j = 0; j < U; ++j) {
                if (base + j * 64 >= count) break;
                const double* from = at(base + j * 64 + lane);
#pragma unroll
                for (int w = 0; w < W; ++w)
                    if ((unsigned long long)__double_as_longlong(u[j][w]) == CG_EMPTY) u[j][w] = ld_agent(from + w);
            }
#pragma unroll
            for (int j = 0; j < U; ++j)
#pragma unroll
                for (int w = 0; w < W; ++w) waiting |= (unsigned long long)__double_as_longlong(u[j][w]) == CG_EMPTY;
            if (!__any(waiting)) break;
            if (const int group = late()) return group;
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            v[0] += u[j][0];
            if (W > 1) v[W - 1] = fmax(v[W - 1], u[j][W - 1]);
        }
    }
    double mx = W > 1 ? v[W - 1] : 0.0;
    wave_reduce2(v[0], mx);
    if (W > 1) v[W - 1] = mx;
    return 0;
}

template <int D, bool RESTART>
__global__ __launch_bounds__(NGW, 6) void k_cg_node(KP p, int k) {
    __shared__ double ws[NGB], wm[NGB];  // a block's partials
    __shared__ float sh_alpha[NGB], sh_beta[NGB];
    __shared__ int sh_fin[NGB], sh_ticket, sh_group, sh_rank;
    if (p.ctr->live == 0) return;
    const long long t0 = wall_clock64();
    const int n = p.ctr->nblocks, ng = cg_groups(n), cp = cg_chunk_places(ng);
    const XcdRange xr = xcd_blocks(ng);
    if (xr.first >= xr.end) return;
    int ticket = 0;
    if (threadIdx.x == 0) ticket = add_agent(p.ctr->doors[blockIdx.x & 7], 1);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool batch = p.nscenes > 1;
    // the wave's block in group g (b < 0: none), its scene's blocks [b0, b1),
    // its run's first wave and number, its scene's number of runs
    int b, si, b0, b1, head, run, runs;
    const auto take = [&](int g) {
        b = g * NGB + wv;
        si = 0;
        b0 = 0;
        b1 = n;
        if (b < n && batch) {
            si = p.block_scene[b];
            b0 = p.sst[si].block_begin;
            b1 = p.sst[si].block_end;
        }
        if (b >= n || p.cg[si].closed) b = -1;
        head = max(b0 - g * NGB, 0);
        run = g - b0 / NGB;
        runs = (b1 - 1) / NGB - b0 / NGB + 1;
    };
    const auto place = [&](int i) { return i == 0 ? ng + si : b0 / NGB + i; };
    const auto chunk_place = [&](int c) { return b0 / NGB / (CG_CHUNK_RUNS / 2) + c; };
    // the run's partial, the chunk's sum (from the wave of the first run), and
    // the scene's
    const auto publish = [&](auto width, double* sums, int g) {
        constexpr int W = decltype(width)::value;
        const int len = min(b1, (g + 1) * NGB) - b;
        double v[2] = {0.0, 0.0};
        for (int w = 0; w < len; ++w) {
            v[0] += ws[wv + w];
            v[1] = fmax(v[1], wm[wv + w]);
        }
        if (lane == 0) put_values<W>(sums + W * place(run), v);
    };
    const auto lead = [&](auto width, const double* sums, double* chunks, auto&& late) {
        constexpr int W = decltype(width)::value;
        if (runs <= CG_DIRECT_RUNS || run % CG_CHUNK_RUNS != 0) return 0;
        double c[W];
        const int group = await_values<W, 1>([&](int i) { return sums + W * place(run + i); }, min(CG_CHUNK_RUNS, runs - run), lane,
                                             c, late);
        if (group == 0 && lane < 8) put_values<W>(chunks + W * (lane * cp + chunk_place(run / CG_CHUNK_RUNS)), c);
        return group;
    };
    const auto total = [&](auto width, const double* sums, const double* chunks, double* t, auto&& late) {
        constexpr int W = decltype(width)::value;
        if (runs <= CG_DIRECT_RUNS)
            return await_values<W, CG_DIRECT_RUNS / 64>([&](int i) { return sums + W * place(i); }, runs, lane, t, late);
        const double* copy = chunks + W * (int)(blockIdx.x & 7) * cp;
        return await_values<W, 1>([&](int i) { return copy + W * chunk_place(i); }, (runs + CG_CHUNK_RUNS - 1) / CG_CHUNK_RUNS, lane,
                                  t, late);
    };
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using First = std::integral_constant<int, RESTART ? 2 : 1>;  // the launch's first sum: s.q, at the restart r.r
    double* const rr_chunks = p.bmax + 8 * cp;
    double* const first_sums = RESTART ? p.bsum : p.bsq;
    double* const first_chunks = RESTART ? rr_chunks : p.bmax;
    const auto never = [] { return 0; };

    int first = xr.first, step = xr.step, end = xr.end;
    NodeRows<D, false> v;
    double t[2];  // the scene's sum (a run's first wave)
    for (bool settled = false;; settled = true) {
        // q and s.q (restart: q and r.r)
        for (int g = first; g < end; g += step) {
            take(g);
            float q[D];
            if (b >= 0) {
                const SceneParams& sc = p.scn[si];
                double sum, mx = 0.0;
                if (RESTART) cg_restart_block<D, false, false>(p, sc, b, lane, q, sum, mx);
                else cg_product_block<D, false, false>(p, sc, b, lane, 0.0f, k, q, sum);
                if (lane == 0) {
                    ws[wv] = sum;
                    wm[wv] = mx;
                }
            }
            if (threadIdx.x == 0) {
                sh_ticket = ticket;
                sh_group = 0;
            }
            __syncthreads();
            if (sh_ticket >= CG_DOOR_CLOSED) return;
            if (b >= 0) {
#pragma unroll
                for (int a = 0; a < D; ++a) p.g_q[a * p.gcap + b * 64 + lane] = q[a];
            }
            if (b >= 0 && wv == head) publish(First{}, first_sums, g);
            __syncthreads();
        }
        // The sum of one scene is complete only if everybody has come: it
        // settles the doors by itself, and they are looked at when it is late.
        // In a batch the last wave settles them while the sums are awaited.
        const auto settle = [&] {
            int rank;
            const int group = cg_settle(p, ng, t0, sh_ticket, lane, rank);
            if (group != 0 && lane == 0) {
                sh_rank = rank;
                __hip_atomic_store(&sh_group, group, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            return group;
        };
        const auto late = [&] {
            if (settled) return 0;
            if (batch) return __hip_atomic_load(&sh_group, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            return wall_clock64() - t0 < p.door_ticks ? 0 : settle();
        };
        int group = batch && !settled && wv == NGB - 1 ? settle() : 0;
        for (int g = first; g < end && group == 0; g += step) {
            if (first + step < end) take(g);
            if (b >= 0 && wv == head) group = lead(First{}, first_sums, first_chunks, late);
        }
        if (first + step < end) take(first);
        if (b >= 0) {
            v.load(p, b * 64 + lane);
            if (wv == head && group == 0) (void)total(First{}, first_sums, first_chunks, t, late);
        }
        __syncthreads();
        if (sh_group == 0) break;
        first = sh_rank;
        step = sh_group;
        end = ng;
        __syncthreads();
    }
    const bool several = first + step < end;
    if (!RESTART) {
        // alpha, x and r, r.r
        for (int g = first; g < end; g += step) {
            if (g != first) {
                take(g);
                if (b >= 0) {
                    v.load(p, b * 64 + lane);
                    if (wv == head) (void)total(One{}, p.bsq, p.bmax, t, never);
                }
            }
            if (b >= 0 && wv == head && lane == 0) {
                const double alpha = cg_alpha(p.cg[si].rho_hist[k & 1], t[0]);
                if (b == b0) cg_record_alpha(p.cg[si], t[0], alpha);
                sh_alpha[wv] = (float)alpha;
            }
            __syncthreads();
            if (b >= 0) {
                double sum, mx;
                v.step(p, b * 64 + lane, sh_alpha[head], sum, mx);
                if (lane == 0) {
                    ws[wv] = sum;
                    wm[wv] = mx;
                }
            }
            __syncthreads();
            if (b >= 0 && wv == head) publish(Two{}, p.bsum, g);
        }
        for (int g = first; g < end; g += step) {
            if (several) take(g);
            if (b >= 0 && wv == head) (void)lead(Two{}, p.bsum, rr_chunks, never);
        }
    }
    // convergence test of the next iteration, beta and s
    const int kn = RESTART ? 0 : k + 1;
    for (int g = first; g < end; g += step) {
        if (several) {
            take(g);
            if (b >= 0) v.load(p, b * 64 + lane);
        }
        if (b >= 0 && wv == head) {
            const CGTestIn in = cg_test_in(p, si, kn);
            if (!RESTART || g != first) (void)total(Two{}, p.bsum, rr_chunks, t, never);
            float beta;
            const bool fin = cg_test(p, si, kn, t[0], t[1], b == b0 && lane == 0, beta, in);
            if (lane == 0) {
                sh_beta[wv] = beta;
                sh_fin[wv] = fin ? 1 : 0;
            }
        }
        __syncthreads();
        if (b >= 0 && RESTART) {
            cg_restart_residual<D>(p, p.scn[si], b * 64 + lane, v.interior, v.q, v.r);
#pragma unroll
            for (int a = 0; a < D; ++a) {
                p.g_r[a * p.gcap + b * 64 + lane] = v.r[a];
                p.g_s[a * p.gcap + b * 64 + lane] = sh_fin[head] ? 0.0f : v.r[a];  // (done: no direction was taken)
            }
        } else if (b >= 0 && !sh_fin[head] && v.interior) {
#pragma unroll
            for (int a = 0; a < D; ++a)
                p.g_s[a * p.gcap + b * 64 + lane] = cg_direction(v.r[a], v.s[a], sh_beta[head], kn);
        }
        if (several) __syncthreads();
    }
}

// The CG's done poll: the eight ints from Counters::nblocks to cg_iters into
// the host's pinned poll slot.
__global__ __launch_bounds__(64) void k_poll(KP p, int* dst) {
    const int t = (int)threadIdx.x;
    if (t < 8) dst[t] = (&p.ctr->nblocks)[t];
}

// The overflow flag and the bits of every scene's max |V|^2, likewise: the
// host's dt rule reads them after every substep of a launched frame.
__global__ __launch_bounds__(WG) void k_read_speeds(KP p, int* dst) {
    if (threadIdx.x == 0) dst[0] = p.ctr->overflow;
    for (int s = (int)threadIdx.x; s < p.nscenes; s += WG) dst[1 + s] = (int)p.sst[s].max_v2;
}

// ============================================================================
// The whole CG solve of every scene in one launch, for scenes too small to
// fill the chip: there a launch's work is a few microseconds, and the launches
// of an iteration cost more than it.  The iterations and a block's arithmetic are
// those of the launched kernels; a scene's sums run over a partial per block, in
// the order of await_partials whichever form is taken.
//
// Work-groups share the blocks and wait for one another.  No wait depends on a
// work-group that might not run: they enter through a door (cg_enter) that the
// first of them closes as soon as all that are needed have come, or at the
// wait limit; those that come later leave, and whoever is inside is running until
// the kernel ends.  The results do not depend on how many they are.  What
// work-groups exchange goes through device-scope accesses.
//
// All inside (the usual case, at most CG_RESIDENT blocks): one block each, or
// two, their nodes' m, x, r and s and their tiles' s in LDS for the whole solve
// (a halo node's s = r + beta s follows from r alone, so only r and the force
// tiles travel).  An iteration waits three times: for the neighbours' force
// tiles, for the scene's partials of s.q and, with r of the tile's nodes, for
// those of r.r.  Everything that travels is its own flag: a place holds a bit
// pattern that no value has until it is written, and its owner puts the pattern
// back once every reader is known to have passed.  Stores to two places are not
// ordered, so a wave that polls for the place's next value has to know something
// that the owner published behind a wait for the emptying store; those waits
// are the drains before every s.q:
//   tiles, s.q  two places each, by parity of the iteration.  Those of k - 1 are
//         emptied in iteration k before its s.q; the next values in their places
//         are polled in k + 1, behind the test of r.r k, which follows s.q k.
//   r.r   two places.  r.r k - 1 is emptied in iteration k behind the sum of s.q
//         k, so before s.q k + 1, which all that poll for r.r k + 1 have seen.
//   r     three places: a tile's waves poll for r k as soon as their operator of
//         k is stored, when all they know is r.r k - 1 (its test opened iteration
//         k), and so s.q k - 1.  The place's last value r k - 3 was emptied in
//         iteration k - 2, before s.q k - 1.  (Of two places, r k - 2 would be
//         emptied in k - 1 behind its s.q: nothing they know follows that.)
// Otherwise: work-group r of G takes blocks [r n / G, (r + 1) n / G) and counts
// itself in at its scenes' counters before each wait.
//
// Bound by the latency of an iteration's chain (gather, operator phases, three
// exchanges of a store and a load that has to find it).  Two balls of 3.8k
// particles, captured, a frame: 18.1 ms with launched kernels, 7.7 resident with
// a flag per force tile and r waited for before r.r goes out (stores drained,
// then the flag, then the values: three round trips for one), 6.9 now; 2D scene
// of 3.0k 18.3 -> 17.0, twelve scenes of 48k 19.3 -> 18.6, and the disk of 512
// 0.77 -> 0.74 ms for four substeps.
// ============================================================================
// The work-group's rank among those inside and their number (at most `most`
// come), false if the door is closed.
__device__ inline bool cg_enter(const KP& p, int most, int& rank, int& group) {
    __shared__ int sh[2];
    if (threadIdx.x == 0) {
        const int ticket = add_agent(&p.ctr->door, 1);
        int g = 0;
        if (ticket == 0) {
            const long long t0 = wall_clock64();
            while (ld_agent(&p.ctr->door) < most && wall_clock64() - t0 < p.door_ticks) __builtin_amdgcn_s_sleep(1);
            g = __hip_atomic_fetch_or(&p.ctr->door, CG_DOOR_CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            st_agent(&p.ctr->group, g);
        } else if (ticket < CG_DOOR_CLOSED) {
            while ((g = ld_agent(&p.ctr->group)) == 0) __builtin_amdgcn_s_sleep(1);
        }
        sh[0] = ticket;
        sh[1] = g;
    }
    __syncthreads();
    rank = sh[0];
    group = sh[1];
    return group != 0;
}

// The same value, not known to be: what is computed from it stays inside the
// loop instead of holding registers across it.
__device__ inline int opaque(int v) {
    __asm__ __volatile__("" : "+v"(v));
    return v;
}

// Waits for the count (<= MOST) partials at sums (and maxs), and sums (takes
// the largest of) them in a fixed order; one wave, result in every lane.
template <int MOST>
__device__ inline void await_partials(const double* sums, const double* maxs, int count, int lane, double& sum, double& mx) {
    constexpr int U = MOST / 64;
    double vs[U], vm[U];
    bool waiting;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        vs[u] = u * 64 + lane < count ? __longlong_as_double((long long)CG_EMPTY) : 0.0;
        vm[u] = maxs ? vs[u] : 0.0;
    }
    do {
        waiting = false;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u * 64 >= count) break;
            if ((unsigned long long)__double_as_longlong(vs[u]) == CG_EMPTY) vs[u] = ld_agent(sums + u * 64 + lane);
            if (maxs && (unsigned long long)__double_as_longlong(vm[u]) == CG_EMPTY) vm[u] = ld_agent(maxs + u * 64 + lane);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            waiting |= (unsigned long long)__double_as_longlong(vs[u]) == CG_EMPTY ||
                       (unsigned long long)__double_as_longlong(vm[u]) == CG_EMPTY;
    } while (__any(waiting));
    sum = 0.0;
    mx = 0.0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        sum += vs[u];
        mx = fmax(mx, vm[u]);
    }
    wave_reduce2(sum, mx);
}

// Work-group of k_cg_solve: one operator launch of blocks that find the chip
// empty takes 13.2 us with 256 threads a block (56 blocks), 8.9 with 512, 10.2
// with 1024 (102 dense blocks: 31.5, 17.0, 14.3); 512 lets two share a CU.
constexpr int CGW = 512;
// K blocks' part of their scenes' solves (every thread of the work-group);
// a negative one is none.
template <int D, int K>
__device__ inline void cg_solve_resident(const KP& p, int blk0, int blk1, OperatorLds<D, CGW>& S) {
    constexpr int TN = Dims<D>::TN, NBR = Dims<D>::NBR, MOST = K * CG_GROUPS;
    // the wave of block j's nodes: NODES + j, after those with tile nodes
    constexpr int NODES = (TN + 63) / 64;
    static_assert(NODES + K < CGW / 64, "wave roles");
    // by parity of the iteration: in a block without particles no other barrier
    // keeps a wave from writing the next ones before every wave has read these
    __shared__ float sh_beta[2][K];
    __shared__ int sh_done[2][K];
    __shared__ int tnbr[K][NBR];
    // the node state lives in LDS: registers held across the operator would
    // spill (x, r, s of the blocks' nodes and the tiles' s)
    __shared__ float nx[K][D][64], nr[K][D][64], ns[K][D][64], nm[K][64], ts[K][D][TN];
    // the wave's number as a scalar: its block's and scene's data stay scalar
    const int lane0 = threadIdx.x & 63, nw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) - NODES;
    BlockOperator<D, CGW, K == 1 ? ROUND_ONE : ROUND_TWO> op(p, S);
    // wave NODES + j: the nodes of block j; tile threads: their node's s in
    // every tile.  full, done: a bit per block.
    unsigned long long interiors = 0, zeros = 0;  // a bit per lane (scalar)
    int b = -1, si = 0, b0 = 0, nb = 0;
    unsigned full = 0, done = 0;
    for (int j = 0; j < K; ++j) {
        const int bj = j == 0 ? blk0 : blk1;
        const int sj = bj >= 0 ? p.block_scene[bj] : 0;
        if (bj < 0 || !p.scn[sj].active) {
            done |= 1u << j;
            continue;
        }
        if (!block_empty(p, bj)) full |= 1u << j;
        if (nw == j) {
            b = bj;
            si = sj;
        }
    }
    constexpr unsigned ALL = (1u << K) - 1u;
    if (done == ALL) return;
    if (K == 1 && full) op.open(blk0);
    const SceneParams& sc = p.scn[si];
    // r of iteration k travels in g_s, g_r or the first words of the tiles (idle
    // here, and more than the nodes), in turn from k = -1; `turn` is that of r k
    // (offsets: a choice between pointers became a table in scratch)
    static_assert((D + 1) * TN >= D * 64, "a block's tile place holds its nodes' r");
    const int64_t to_r = (int64_t)(reinterpret_cast<uintptr_t>(p.g_r) - reinterpret_cast<uintptr_t>(p.g_s)) / (int64_t)sizeof(float);
    const int64_t to_t = (int64_t)(reinterpret_cast<uintptr_t>(p.tiles) - reinterpret_cast<uintptr_t>(p.g_s)) / (int64_t)sizeof(float);
    const auto r_place = [&](int t) { return p.g_s + (t == 0 ? 0 : t == 1 ? to_r : to_t); };
    int turn = 0;
    if (b >= 0) {
        const int lane = lane0, n = b * 64 + lane;
        b0 = p.sst[si].block_begin;
        nb = p.sst[si].block_end - b0;
        interiors = __ballot((p.g_flags[n] & MPM_FLAG_INTERIOR_DEV) != 0);
        nm[nw][lane] = p.g_m[n];
        zeros = __ballot(project_zero<D>(p, sc, n));
        if (lane < NBR) tnbr[nw][lane] = p.block_tnbr[(int64_t)b * NBR + lane];
#pragma unroll
        for (int a = 0; a < D; ++a) {
            nx[nw][a][lane] = p.g_vs[a * p.gcap + n];
            nr[nw][a][lane] = p.g_r[a * p.gcap + n];
            ns[nw][a][lane] = 0.0f;
            st_agent(r_place(1) + a * p.gcap + n, __uint_as_float(CG_EMPTY_FLOAT));
            st_agent(r_place(2) + a * p.gcap + n, __uint_as_float(CG_EMPTY_FLOAT));
        }
    }
    // iteration -1 is the restart: the operator on x, r = b - A x
    double rho = 0.0;
    for (int k = -1;; ++k, turn = turn == 2 ? 0 : turn + 1) {
        const int par = (k & 1) * CG_RESIDENT, before = turn == 0 ? 2 : turn - 1;
        const int lane = opaque(lane0), n = b * 64 + lane;
        op.tid = opaque(op.tid);
        // r of tile node `node`
        float rn[D];
        const auto await_r = [&](int node) {
            bool waiting;
            do {
                waiting = false;
#pragma unroll
                for (int a = 0; a < D; ++a) rn[a] = ld_agent(r_place(before) + a * p.gcap + node);
#pragma unroll
                for (int a = 0; a < D; ++a) waiting |= is_empty(rn[a]);
                if (waiting) __builtin_amdgcn_s_sleep(4);
            } while (waiting);
        };
        if (k >= 0) {
            if (b >= 0 && !((done >> nw) & 1u)) {
                // convergence test and beta on the scene's r.r
                double rr, mx;
                await_partials<MOST>(p.bsum + par + b0, p.bmax + par + b0, nb, lane, rr, mx);
                // every reader of the s.q partials of iteration k - 1 has passed
                if (lane == 0) clear_partial(p.bsq + (CG_RESIDENT - par) + b);
                const CGTestIn in{rho, sc.cg_tol, sc.cg_min, sc.cg_max, false};
                float beta;
                const bool fin = cg_test(p, si, k, rr, mx, b == b0 && lane == 0, beta, in);
                rho = scalar(rr);
                if (lane == 0) {
                    sh_beta[k & 1][nw] = beta;
                    sh_done[k & 1][nw] = fin ? 1 : 0;
                }
            } else if (K == 1 && full && op.node >= 0) {
                await_r(op.node);  // meanwhile
            }
            __syncthreads();
            for (int j = 0; j < K; ++j)
                if (!((done >> j) & 1u) && sh_done[k & 1][j]) done |= 1u << j;
            if (done == ALL) break;
        }
#pragma unroll 1
        for (int j = 0; j < K; ++j) {
            if (!((full & ~done) >> j & 1u)) continue;
            const int bj = j == 0 ? blk0 : blk1;
            if (K > 1) op.open(bj);
            op.node = opaque(op.node);
            // s = r + beta s of the tile's nodes
            float u[D];
#pragma unroll
            for (int a = 0; a < D; ++a) u[a] = 0.0f;
            if (op.node >= 0) {
                if (K > 1 && k >= 0) await_r(op.node);
#pragma unroll
                for (int a = 0; a < D; ++a) {
                    if (k < 0) {
                        u[a] = p.g_vs[a * p.gcap + op.node];
                        ts[j][a][op.tid] = 0.0f;
                    } else {
                        u[a] = cg_direction(rn[a], ts[j][a][op.tid], sh_beta[k & 1][j], k);
                        ts[j][a][op.tid] = u[a];
                    }
                }
            }
            // every reader of the tile of iteration k - 1 has passed
            if (k >= 0 && op.tid < TN) {
#pragma unroll
                for (int a = 0; a < D; ++a) st_agent(cg_tile<D>(p, k - 1, bj) + op.tid + a * TN, __uint_as_float(CG_EMPTY_FLOAT));
            }
            op.apply(p.scn[p.block_scene[bj]].inv_dx, u, K == 1 && k >= 0);
            drain_stores();  // places emptied in this iteration: before its s.q is out
            op.template store<true, true>(cg_tile<D>(p, k, bj));
            __syncthreads();
            if (K == 1) op.load_records(0);  // for the next time
        }
        if (b < 0 || ((done >> nw) & 1u)) continue;
        // the neighbours' tiles, and this block's nodes
        const bool interior = (interiors >> lane) & 1, zero = (zeros >> lane) & 1;
        float q[D], r[D];
        gather_tiles<D, D, true, true>(p, sc, n, cg_tile<D>(p, k, 0), [&](int o) { return tnbr[nw][o]; }, q);
        const double m = (double)nm[nw][lane];
        const float cm = sc.dt * sc.dt / nm[nw][lane];
        double sum = 0.0, mx = 0.0;
        if (k < 0) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                r[a] = nr[nw][a][lane];
                if (interior) {
                    q[a] = cm * q[a] + nx[nw][a][lane];
                    r[a] = r[a] - q[a];
                }
                if (zero) r[a] = 0.0f;
            }
            drain_stores();  // the places emptied above: r 0 is polled by waves that know no more than r.r -1
        } else {
            const float beta = sh_beta[k & 1][nw];
            float s[D];
#pragma unroll
            for (int a = 0; a < D; ++a) {
                s[a] = ns[nw][a][lane];
                if (interior) {
                    s[a] = cg_direction(nr[nw][a][lane], s[a], beta, k);
                    ns[nw][a][lane] = s[a];
                    q[a] = cm * q[a] + s[a];
                }
                if (zero) q[a] = 0.0f;
                if (interior) sum += (double)s[a] * ((double)q[a] * m);
            }
            double sq;
            wave_reduce2(sum, mx);
            drain_stores();
            if (lane == 0) put_partial(p.bsq + par + b, sum);
            await_partials<MOST>(p.bsq + par + b0, nullptr, nb, lane, sq, mx);
            // every reader of this iteration's r.r partials and of r of
            // iteration k - 1 has passed
            if (lane == 0) {
                clear_partial(p.bsum + par + b);
                clear_partial(p.bmax + par + b);
            }
#pragma unroll
            for (int a = 0; a < D; ++a) st_agent(r_place(before) + a * p.gcap + n, __uint_as_float(CG_EMPTY_FLOAT));
            const double alpha_d = cg_alpha(rho, sq);
            if (b == b0 && lane == 0) cg_record_alpha(p.cg[si], sq, alpha_d);
            const float alpha = (float)alpha_d;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                r[a] = nr[nw][a][lane];
                if (interior) {
                    nx[nw][a][lane] = alpha * s[a] + nx[nw][a][lane];
                    r[a] = -alpha * q[a] + r[a];
                }
            }
        }
        // r and its partials
        sum = 0.0;
        mx = 0.0;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            st_agent(r_place(turn) + a * p.gcap + n, flagged(r[a]));
            if (interior) {
                sum += (double)r[a] * ((double)r[a] * m);
                mx += (double)r[a] * (double)r[a];
            }
            nr[nw][a][lane] = r[a];
            p.g_q[a * p.gcap + n] = q[a];
        }
        wave_reduce2(sum, mx);
        if (lane == 0) {
            put_partial(p.bsum + (CG_RESIDENT - par) + b, sum);
            put_partial(p.bmax + (CG_RESIDENT - par) + b, mx);
        }
    }
    if (b >= 0) {
        const int lane = lane0, n = b * 64 + lane;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            p.g_vs[a * p.gcap + n] = nx[nw][a][lane];
            p.g_r[a * p.gcap + n] = flagged(nr[nw][a][lane]);
            p.g_s[a * p.gcap + n] = flagged(ns[nw][a][lane]);
        }
    }
}

// ---- fewer work-groups than blocks -------------------------------------------
// The work-group that owns block b of n when g (<= n) share them.
__device__ inline int cg_owner(int b, int n, int g) { return (int)((((int64_t)b + 1) * g - 1) / n); }

// A run is the part of one scene's blocks that a work-group owns.  f(si, e,
// r, b): run r of scene si is blocks [b, e).
template <class F>
__device__ inline void for_runs(const KP& p, int w0, int w1, F&& f) {
    int r = 0;
    for (int b = w0; b < w1; ++r) {
        const int si = p.block_scene[b], e = min(w1, p.sst[si].block_end);
        f(si, e, r, b);
        b = e;
    }
}

// Waits until every work-group that owns blocks of the scenes still running
// here (runs not in `done`) has come; `phase` counts the waits from 1.  A scene of
// many owners is counted in eighths, the last of each counts at one place, the
// last there gives the go-aheads: with all 512 adding to and polling one counter a
// wait took some 20 us (one scene of 1,260 blocks: a substep of 25 iterations 2.05
// ms, in eighths 1.10; of 1,650: 3.1 and 1.7).
__device__ inline void cg_wait(const KP& p, int w0, int w1, int n, int g, unsigned long long done, int phase) {
    drain_stores();  // before the work-group is counted
    __syncthreads();
    if (threadIdx.x == 0) {
        const int me = cg_owner(w0, n, g);
        // f(first owner, owners) of every scene that is waited for
        const auto for_scenes = [&](auto&& f) {
            for_runs(p, w0, w1, [&](int si, int, int r, int) {
                if ((done >> r) & 1) return;
                const int o0 = cg_owner(p.sst[si].block_begin, n, g);
                f(si, o0, cg_owner(p.sst[si].block_end - 1, n, g) - o0 + 1);
            });
        };
        // (scenes of more than CG_WAIT_FLAT owners begin at least as many apart)
        const auto set = [&](int o0) { return p.cg_waits + o0 / CG_WAIT_FLAT * CG_WAIT_SET; };
        for_scenes([&](int si, int o0, int owners) {
            if (owners <= CG_WAIT_FLAT) {
                add_agent(&p.cg[si].arrived, 1);
                return;
            }
            int* const w = set(o0);
            const int x = (me - o0) & 7;
            if (add_agent(w + x * CG_WAIT_LINE, 1) != (owners - x + 7) / 8 * phase - 1) return;
            if (add_agent(w + 8 * CG_WAIT_LINE, 1) != 8 * phase - 1) return;
            for (int q = 0; q < 8; ++q) st_agent(w + (9 + q) * CG_WAIT_LINE, phase);
        });
        for_scenes([&](int si, int o0, int owners) {
            if (owners <= CG_WAIT_FLAT) {
                while (ld_agent(&p.cg[si].arrived) < owners * phase) __builtin_amdgcn_s_sleep(1);
            } else {
                while (ld_agent(set(o0) + (9 + ((me - o0) & 7)) * CG_WAIT_LINE) < phase) __builtin_amdgcn_s_sleep(1);
            }
        });
    }
    __syncthreads();
    __asm__ __volatile__("" ::: "memory");
}

static_assert(CG_SOLVE_MAX_SCENES <= 64, "a work-group holds at most that many runs, a bit each");
// Blocks [w0, w1) of n, work-groups g.
template <int D>
__device__ inline void cg_solve_shared(const KP& p, int w0, int w1, int n, int g, OperatorLds<D, CGW>& S) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned long long done = 0, all = 0;
    for_runs(p, w0, w1, [&](int si, int, int r, int) {
        all |= 1ull << r;
        if (!p.scn[si].active) done |= 1ull << r;
    });
    if (done == all) return;
    int phase = 0;
    for (int k = -1;; ++k) {
        // convergence test and beta of every scene, then its operator
        // (iteration -1: the restart, the operator on x, r = b - A x)
        for_runs(p, w0, w1, [&](int si, int e, int r, int b) {
            if ((done >> r) & 1) return;
            float beta = 0.0f;
            if (k >= 0) {
                const int b0 = p.sst[si].block_begin, b1 = p.sst[si].block_end;
                const CGTestIn in = cg_test_in(p, si, k);
                double rr, mx;
                reduce_range<CGW>(p.bsum, p.bmax, b0, b1 - b0, reinterpret_cast<double*>(S.coef), rr, mx);
                if (cg_test(p, si, k, rr, mx, b == b0 && threadIdx.x == 0, beta, in)) {
                    done |= 1ull << r;
                    return;
                }
            }
            for (; b < e; ++b)
                if (!block_empty(p, b))
                    operator_block<D, CGW, ROUND_EITHER, true>(p, b, p.scn[si].inv_dx, n > CG_GROUPS, S, [&](int a, int64_t nd) {
                        return k < 0 ? p.g_vs[a * p.gcap + nd]
                                     : cg_direction(ld_agent(p.g_r + a * p.gcap + nd), ld_agent(p.g_s + a * p.gcap + nd), beta, k);
                    });
        });
        if (k < 0) {
            cg_wait(p, w0, w1, n, g, done, ++phase);
            for_runs(p, w0, w1, [&](int si, int e, int r, int b) {
                if ((done >> r) & 1) return;
                for (b += wv; b < e; b += CGW / 64) {
                    float q[D];
                    double sum, mx;
                    cg_restart_block<D, true, true>(p, p.scn[si], b, lane, q, sum, mx);
                    if (lane == 0) {
                        st_agent(p.bsum + b, sum);
                        st_agent(p.bmax + b, mx);
                    }
                }
            });
            cg_wait(p, w0, w1, n, g, done, ++phase);
            continue;
        }
        if (done == all) return;
        cg_wait(p, w0, w1, n, g, done, ++phase);
        // q = A s and s itself, s.q
        for_runs(p, w0, w1, [&](int si, int e, int r, int b) {
            if ((done >> r) & 1) return;
            const float beta = (float)ld_agent(&p.cg[si].beta);
            for (b += wv; b < e; b += CGW / 64) {
                float q[D];
                double sum;
                cg_product_block<D, true, true>(p, p.scn[si], b, lane, beta, k, q, sum);
                if (lane == 0) st_agent(p.bsq + b, sum);
            }
        });
        cg_wait(p, w0, w1, n, g, done, ++phase);
        // alpha, x and r, r.r
        for_runs(p, w0, w1, [&](int si, int e, int r, int b) {
            if ((done >> r) & 1) return;
            const int b0 = p.sst[si].block_begin, b1 = p.sst[si].block_end;
            const double rho = ld_agent(&p.cg[si].rho_hist[k & 1]);
            double sq, unused;
            reduce_range<CGW>(p.bsq, nullptr, b0, b1 - b0, reinterpret_cast<double*>(S.coef), sq, unused);
            const double alpha = cg_alpha(rho, sq);
            if (b == b0 && threadIdx.x == 0) cg_record_alpha(p.cg[si], sq, alpha);
            for (b += wv; b < e; b += CGW / 64) {
                double sum, mx;
                NodeRows<D, true> v;
                v.load(p, b * 64 + lane);
                v.step(p, b * 64 + lane, (float)alpha, sum, mx);
                if (lane == 0) {
                    st_agent(p.bsum + b, sum);
                    st_agent(p.bmax + b, mx);
                }
            }
        });
        cg_wait(p, w0, w1, n, g, done, ++phase);
    }
}

// One resident block a work-group up to CG_GROUPS blocks; above, up to
// CG_RESIDENT, two, heaviest with lightest within an XCD's range of the block
// order, so that a block of particles is paired with a halo block wherever
// there are as many.
template <int D>
__global__ __launch_bounds__(CGW, 4) void k_cg_solve(KP p) {
    __shared__ __align__(16) OperatorLds<D, CGW> S;
    const int n = p.ctr->nblocks, bid = (int)blockIdx.x;
    const bool pairs = n > CG_GROUPS && n <= CG_RESIDENT;
    int blk0 = bid, blk1 = -1, most = min(n, CG_GROUPS);
    bool mine = bid < most;
    if (pairs) {
        const auto lo = [&](int x) { return (int)(((int64_t)n * x) >> 3); };
        most = 0;
        for (int x = 0; x < 8; ++x) most += (lo(x + 1) - lo(x) + 1) / 2;
        const int i = lo(bid & 7) + (bid >> 3), e = lo((bid & 7) + 1) - 1 - (bid >> 3);
        mine = i <= e;
        blk0 = mine ? p.block_order[p.bcap + i] : -1;
        blk1 = i < e ? p.block_order[p.bcap + e] : -1;
    }
    if (!mine) return;
    int rank, group;
    if (!cg_enter(p, most, rank, group)) return;
    if (group == most && n <= CG_GROUPS) {
        cg_solve_resident<D, 1>(p, blk0, -1, S);
    } else if (group == most && pairs) {
        cg_solve_resident<D, 2>(p, blk0, blk1, S);
    } else {
        const int g = min(group, n);
        if (rank >= g) return;
        const int w0 = (int)((int64_t)rank * n / g), w1 = (int)((int64_t)(rank + 1) * n / g);
        cg_solve_shared<D>(p, w0, w1, n, g, S);
    }
}

#pragma clang fp contract(fast)

// ============================================================================
// G2P (MPM_Example.cpp:631-660): PIC/FLIP velocity, F and X update, removal
// ============================================================================
template <int D>
__global__ __launch_bounds__(BWG) void k_g2p(KP p) {
    using Dm = Dims<D>;
    constexpr int LTN = Dm::LTN, NBR = Dm::NBR, DD = D * D;
    __shared__ float vt[2 * D][LTN];
    __shared__ int nbr[NBR];
    __shared__ unsigned wbest[NW];
    __shared__ int wrem[NW];
    const int nblocks = p.ctr->nblocks;
    const XcdRange xr = xcd_blocks(nblocks);
    for (int kb = xr.first; kb < xr.end; kb += xr.step) {
        const int b = p.block_order[kb];  // heavy blocks first within the XCD's range
        const SceneParams& sc = p.scn[p.block_scene[b]];
        if (!sc.active) continue;
        if (block_empty(p, b)) {  // no particles: empty partials for the scene's reduction
            if (threadIdx.x == 0) {
                p.bu[b] = 0u;
                p.bu[p.bcap + b] = 0u;
            }
            continue;
        }
        const float dt = sc.dt, flip = sc.flip;
        const float lo = 0.0f + 0.5f * sc.dx, hi = 1.0f - 0.5f * sc.dx;
        unsigned best = 0u;
        int removed = 0;
        if (threadIdx.x < NBR) nbr[threadIdx.x] = p.block_nbr[b * NBR + threadIdx.x];
        int bb[D];
        block_coords<D>(p, b, bb);
        // the first particle's position and velocity load while the tile is gathered
        const int i0 = p.block_pstart[b] + (int)threadIdx.x, i1 = p.block_pstart[b + 1];
        float nX[D], nV[D];
        auto load = [&](int i) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                nX[a] = p.pcur[(PF<D>::X + a) * p.pcap + i];
                nV[a] = p.pcur[(PF<D>::V + a) * p.pcap + i];
            }
        };
        if (i0 < i1) load(i0);
        __syncthreads();
        const float* src[2 * D];
#pragma unroll
        for (int a = 0; a < D; ++a) {
            src[a] = p.g_vs + a * p.gcap;
            src[D + a] = p.g_v + a * p.gcap;
        }
        gather_tile<D, 2 * D>(p, nbr, vt, src);
        __syncthreads();
        for (int i = i0; i < i1; i += BWG) {
            float w[D][3], dw[D][3], X[D], V0[D];
            int l[D];
#pragma unroll
            for (int a = 0; a < D; ++a) {
                X[a] = nX[a];
                V0[a] = nV[a];
            }
            if (i + BWG < i1) load(i + BWG);
            bool in_block = true;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                int cl;
                bspline_weights(X[a], sc.dx, sc.inv_dx, cl, w[a], dw[a]);
                l[a] = cl + Dm::B - Dm::B * bb[a];
                in_block = in_block && l[a] >= 0 && l[a] < Dm::B;
            }
            if (!in_block) continue;
            float vpic[D], vflip[D], G[DD];
#pragma unroll
            for (int a = 0; a < D; ++a) {
                vpic[a] = 0.0f;
                vflip[a] = V0[a];
            }
#pragma unroll
            for (int k = 0; k < DD; ++k) G[k] = 0.0f;
#pragma unroll
            for (int s = 0; s < Dm::ST; ++s) {
                int off[D];
                const int t = tile_index<D>(l, s, off);
                const float wt = stencil_weight<D>(w, off);
                if (wt > 0.0f) {
                    float g[D];
                    stencil_grad<D>(w, dw, off, g);
#pragma unroll
                    for (int a = 0; a < D; ++a) {
                        const float vs = vt[a][t], v = vt[D + a][t];
                        vpic[a] += wt * vs;
                        vflip[a] += wt * (vs - v);
#pragma unroll
                        for (int cc = 0; cc < D; ++cc) G[a * D + cc] += vs * g[cc];
                    }
                }
            }
            const int mid = sc.nmat > 1 ? __float_as_int(p.pcur[PF<D>::MAT * p.pcap + i]) : 0;
            if (sc.mats[mid].eos) {
                // EOS: density /= 1 + dt tr(grad v) (MPM_Example.cpp:646); F unchanged
                float tr = 0.0f;
#pragma unroll
                for (int a = 0; a < D; ++a) tr += G[a * D + a];
                p.pcur[PF<D>::J * p.pcap + i] = p.pcur[PF<D>::J * p.pcap + i] / (1.0f + dt * tr);
            } else {
                float F[DD];
#pragma unroll
                for (int k = 0; k < DD; ++k) F[k] = p.pcur[(PF<D>::F + k) * p.pcap + i];
#pragma unroll
                for (int r = 0; r < D; ++r)
#pragma unroll
                    for (int cc = 0; cc < D; ++cc) {
                        float s = 0.0f;
#pragma unroll
                        for (int k = 0; k < D; ++k) s += (dt * G[r * D + k]) * F[k * D + cc];
                        p.pcur[(PF<D>::F + r * D + cc) * p.pcap + i] = F[r * D + cc] + s;
                    }
            }
            bool inside = true, finite = true;
            float v2 = 0.0f;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const float V = vflip[a] * flip + vpic[a] * (1.0f - flip);
                const float Xn = X[a] + vpic[a] * dt;
                p.pcur[(PF<D>::V + a) * p.pcap + i] = V;
                p.pcur[(PF<D>::X + a) * p.pcap + i] = Xn;
                inside = inside && Xn >= lo && Xn <= hi;
                finite = finite && isfinite(V) && isfinite(Xn);
                v2 += V * V;
            }
            // a NaN/Inf state leaves the domain test false (removal, as in the
            // reference) and flags the scene for the caller
            if (!finite) atomicOr(&p.sst[p.block_scene[b]].nonfinite, 1);
            if (!inside) {
                p.keycur[i] = -1;
                ++removed;
            } else {
                best = max(best, __float_as_uint(v2));
            }
        }
        // per-block partials (plain stores); k_g2p_reduce folds each scene's
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            best = max(best, (unsigned)__shfl_xor((int)best, off));
            removed += __shfl_xor(removed, off);
        }
        if ((threadIdx.x & 63) == 0) {
            wbest[threadIdx.x >> 6] = best;
            wrem[threadIdx.x >> 6] = removed;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned bm = 0u;
            int rm = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                bm = max(bm, wbest[w]);
                rm += wrem[w];
            }
            p.bu[b] = bm;
            p.bu[p.bcap + b] = (unsigned)rm;
        }
        __syncthreads();
    }
}

// One work-group per scene: max speed and removal count of the last G2P, in
// a fixed order (MPM_Example::Max_Particle_Velocity, MPM_Example.cpp:375-387).
// Scenes that did not advance keep their values.
__global__ __launch_bounds__(WG) void k_g2p_reduce(KP p) {
    const int si = blockIdx.x;
    if (si == 0 && threadIdx.x == 0 && p.blocks_out) *p.blocks_out = p.ctr->nblocks;
    if (!p.scn[si].active) return;
    const int b0 = p.sst[si].block_begin, b1 = p.sst[si].block_end;
    constexpr int U = 8;
    unsigned ba[U], ra[U];
#pragma unroll
    for (int u = 0; u < U; ++u) { ba[u] = 0u; ra[u] = 0u; }
    for (int base = b0 + (int)threadIdx.x; base < b1; base += U * WG) {
        // the chunk's loads all go out before the first use (a block past the
        // range reads the range's last one and is not counted)
        unsigned bv[U], rv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int b = min(base + u * WG, b1 - 1);
            bv[u] = p.bu[b];
            rv[u] = p.bu[p.bcap + b];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (base + u * WG < b1) {
                ba[u] = max(ba[u], bv[u]);
                ra[u] += rv[u];
            }
    }
    unsigned best = 0u, removed = 0u;
#pragma unroll
    for (int u = 0; u < U; ++u) { best = max(best, ba[u]); removed += ra[u]; }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        best = max(best, (unsigned)__shfl_xor((int)best, off));
        removed += (unsigned)__shfl_xor((int)removed, off);
    }
    __shared__ unsigned sb[WG / 64], sr[WG / 64];
    if ((threadIdx.x & 63) == 0) {
        sb[threadIdx.x >> 6] = best;
        sr[threadIdx.x >> 6] = removed;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < WG / 64; ++w) {
            best = max(best, sb[w]);
            removed += sr[w];
        }
        p.sst[si].max_v2 = best;
        p.sst[si].n_removed = (int)removed;
    }
}

// Max |V|^2 per scene over the particle buffer (before the first binning):
// one atomic per distinct scene in a wave.
template <int D>
__global__ __launch_bounds__(WG) void k_max_speed(KP p) {
    const int n = p.ctr->n_live;
    const int lane = threadIdx.x & 63;
    for (int base = blockIdx.x * WG + (threadIdx.x & ~63); base < n; base += gridDim.x * WG) {
        const int i = base + lane;
        const bool valid = i < n && p.keycur[i] >= 0;
        unsigned v2b = 0u;
        int si = -1;
        if (valid) {
            si = p.scur[i];
            float v2 = 0.0f;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const float v = p.pcur[(PF<D>::V + a) * p.pcap + i];
                v2 += v * v;
            }
            v2b = __float_as_uint(v2);
        }
        unsigned long long todo = __ballot(valid);
        while (todo) {
            const int leader = __ffsll((long long)todo) - 1;
            const int ls = __shfl(si, leader);
            const unsigned long long grp = __ballot(valid && si == ls);
            unsigned m = (valid && si == ls) ? v2b : 0u;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, off));
            if (lane == leader && m) atomicMax(&p.sst[ls].max_v2, m);
            todo &= ~grp;
        }
    }
}

// ============================================================================
// Download: the live particles of one scene by id, particle-major as the
// caller's arrays are.  Every id finds its particle (k_pack_mark), the ids that
// found one are numbered by a scan over tiles of PACK_TILE ids (k_pack_count,
// k_pack_top), and each particle is written at its number (k_pack_write).
// Bound by the copy to the host, then by the gathers of k_pack_write, whose
// particles are in cell order (most of its loads take a line each).  A download
// of 1.0M particles, host copy included: 180 -> 7.3 ms, 2M: 370 -> 18, 20k: 1.3
// -> 0.25, against copying the fields and sorting and transposing on the host.
// ============================================================================
constexpr int PACK_PER_THREAD = 4, PACK_TILE = WG * PACK_PER_THREAD;
__global__ __launch_bounds__(WG) void k_pack_clear(PackArgs a) {
    for (int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x; i < a.nid; i += (int64_t)gridDim.x * WG) a.inv[i] = -1;
}
__global__ __launch_bounds__(WG) void k_pack_mark(KP p, PackArgs a) {
    for (int64_t i = a.first + (int64_t)blockIdx.x * WG + threadIdx.x; i < a.last; i += (int64_t)gridDim.x * WG) {
        const int id = p.idcur[i];
        if (p.keycur[i] >= 0 && p.scur[i] == a.scene && id >= 0 && id < a.nid) a.inv[id] = (int)i;
    }
}
__global__ __launch_bounds__(WG) void k_pack_count(PackArgs a) {
    const int64_t base = (int64_t)blockIdx.x * PACK_TILE + threadIdx.x * PACK_PER_THREAD;
    int c = 0;
#pragma unroll
    for (int k = 0; k < PACK_PER_THREAD; ++k) c += base + k < a.nid && a.inv[base + k] >= 0 ? 1 : 0;
    int total;
    wg_exclusive_scan(c, total);
    if (threadIdx.x == 0) a.part[blockIdx.x] = total;
}
// one work-group: exclusive scan of the tiles' counts, their total behind them
__global__ __launch_bounds__(WG) void k_pack_top(PackArgs a, int tiles) {
    const int per = (tiles + WG - 1) / WG;
    const int64_t t0 = (int64_t)threadIdx.x * per;
    int sum = 0;
    for (int k = 0; k < per; ++k)
        if (t0 + k < tiles) sum += a.part[t0 + k];
    int total;
    int run = wg_exclusive_scan(sum, total);
    for (int k = 0; k < per; ++k)
        if (t0 + k < tiles) {
            const int c = a.part[t0 + k];
            a.part[t0 + k] = run;
            run += c;
        }
    if (threadIdx.x == 0) a.part[tiles] = total;
}
template <int D>
__global__ __launch_bounds__(WG) void k_pack_write(KP p, PackArgs a) {
    const int64_t base = (int64_t)blockIdx.x * PACK_TILE + threadIdx.x * PACK_PER_THREAD;
    int from[PACK_PER_THREAD], c = 0;
#pragma unroll
    for (int k = 0; k < PACK_PER_THREAD; ++k) {
        from[k] = base + k < a.nid ? a.inv[base + k] : -1;
        c += from[k] >= 0 ? 1 : 0;
    }
    int total;
    int64_t to = wg_exclusive_scan(c, total) + a.part[blockIdx.x];
#pragma unroll
    for (int k = 0; k < PACK_PER_THREAD; ++k) {
        if (from[k] < 0) continue;
        float f[PF<D>::N];
#pragma unroll
        for (int q = 0; q < PF<D>::N; ++q) f[q] = p.pcur[q * p.pcap + from[k]];
        if (a.x) {
#pragma unroll
            for (int q = 0; q < D; ++q) a.x[to * D + q] = f[PF<D>::X + q];
        }
        if (a.v) {
#pragma unroll
            for (int q = 0; q < D; ++q) a.v[to * D + q] = f[PF<D>::V + q];
        }
        if (a.F) {
#pragma unroll
            for (int q = 0; q < D * D; ++q) a.F[to * D * D + q] = f[PF<D>::F + q];
        }
        if (a.Jp) a.Jp[to] = f[PF<D>::J];
        if (a.mass) a.mass[to] = f[PF<D>::M];
        if (a.volume) a.volume[to] = f[PF<D>::VOL];
        if (a.material) a.material[to] = __float_as_int(f[PF<D>::MAT]);
        if (a.ids) a.ids[to] = (int)(base + k);
        ++to;
    }
}

// dt and activity of scenes [first, first + n) for the next substep
__global__ __launch_bounds__(WG) void k_set_step(KP p, StepArgs a) {
    const int i = blockIdx.x * WG + threadIdx.x;
    if (i >= a.n) return;
    SceneParams& sc = p.scn[a.first + i];
    const float dt = a.dt[i];
    sc.dt = dt > 0.0f ? dt : 0.0f;
    sc.active = (a.force_active || dt > 0.0f) ? 1 : 0;
    if (a.clear_waiting) sc.waiting = 0;
}

// Process_Waiting_Particles ran for every waiting scene: clear the flags.
// After a binning over the block capacity no block was set up and the
// waiting particles have no volume yet: they keep waiting.
__global__ __launch_bounds__(WG) void k_clear_waiting(KP p) {
    const int i = blockIdx.x * WG + threadIdx.x;
    if (i < p.nscenes && !p.ctr->overflow) p.scn[i].waiting = 0;
}

// Removes every particle of scene `scene` (key -1: the next binning drops it).
__global__ __launch_bounds__(WG) void k_remove_scene(KP p, int scene) {
    const int n = p.ctr->n_live;
    for (int i = blockIdx.x * WG + threadIdx.x; i < n; i += gridDim.x * WG)
        if (p.scur[i] == scene) p.keycur[i] = -1;
}

// The same from a device array of nscenes dts (replayed graphs: the host
// copies the substep's dts into `dt` before each replay).
__global__ __launch_bounds__(WG) void k_set_step_dev(KP p, const float* dt) {
    const int i = blockIdx.x * WG + threadIdx.x;
    if (i >= p.nscenes) return;
    SceneParams& sc = p.scn[i];
    const float d = dt[i];
    sc.dt = d > 0.0f ? d : 0.0f;
    sc.active = d > 0.0f ? 1 : 0;
}

// The dt of the next substep of every scene in the device frame loop: the
// reference's rule (MPM_Driver.cpp:55-80) on the scene's max |V| from its last
// G2P (MPM_Example::Max_Particle_Velocity), in the same float operations as
// the host loop, so both take the same dts: dt = clamp(cfl dx / max(vmax,
// 1e-2), min_dt, max_dt); the last substep of the frame takes what remains
// when that is under 1.001 dt, and the one before half of it when it is
// under 2 dt.  A scene at its frame end gets dt 0 (it idles).  One work-group.
__global__ __launch_bounds__(WG) void k_frame_dt(KP p, FrameState* f, float* dt_out) {
#pragma clang fp contract(off)
    int done = 0;
    for (int s = threadIdx.x; s < p.nscenes; s += WG) {
        FrameState st = f[s];
        float d = 0.0f;
        if (!st.done) {
            const float v2 = __uint_as_float(p.sst[s].max_v2);
            const float vmax = (float)sqrt((double)v2);  // the correctly rounded float sqrt
            const float vfloor = vmax < 1e-2f ? 1e-2f : vmax;
            const float cfl_dt = st.cfl * st.dx / vfloor;
            const float capped = cfl_dt < st.max_dt ? cfl_dt : st.max_dt;
            d = st.min_dt < capped ? capped : st.min_dt;
            bool last = false;
            const float rem = st.target - st.time;
            if (rem < d * 1.001f) {
                d = rem;
                last = true;
            } else if (rem < 2.0f * d) {
                d = rem * 0.5f;
            }
            if (!(d > 0.0f)) {
                st.done = 1;
                d = 0.0f;
            } else {
                st.time += d;
                st.steps += 1;
                st.last_dt = d;
                if (last) st.done = 1;
            }
            f[s] = st;
        }
        dt_out[s] = d;
        done += st.done ? 1 : 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) done += __shfl_xor(done, off);
    __shared__ int wsum[WG / 64];
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = done;
    __syncthreads();
    if (threadIdx.x == 0) {
        int total = 0;
#pragma unroll
        for (int w = 0; w < WG / 64; ++w) total += wsum[w];
        p.ctr->frame_ndone = total;
    }
}

// ============================================================================
// Allocation-free substep: the scene table, the counters and the binning's
// slot and cell counters of the static scratch start over at every call (the
// scratch keeps the last call's contents), and the caller's particle-major
// arrays become binning's field-major input; afterwards every binned
// particle goes back to the caller's arrays at its original index.
// ============================================================================
template <int D>
__global__ __launch_bounds__(WG) void k_noalloc_load(KP p, SceneParams sp, NoallocIn a) {
    const int gid = blockIdx.x * WG + threadIdx.x, stride = gridDim.x * WG;
    if (gid == 0) {
        p.scn[0] = sp;
        Counters c{};
        c.n_live = a.n;
        c.n_prev = a.n;
        c.slot_hw = p.nslots;
        *p.ctr = c;
        p.sst[0] = SceneState{};
        a.d_dt[0] = a.dt;
    }
    for (int s = gid; s < p.nslots; s += stride) {
        p.slot_count[s] = 0;
        p.slot_touched[s] = 0;
        a.slot_scene[s] = 0;
    }
    for (int64_t k = gid; k < (int64_t)p.nslots * 64; k += stride) p.cell_count[k] = 0;
    const Material& mat = sp.mats[0];
    for (int i = gid; i < a.n; i += stride) {
#pragma unroll
        for (int c = 0; c < D; ++c) {
            p.pcur[(PF<D>::X + c) * p.pcap + i] = a.x[(int64_t)i * D + c];
            p.pcur[(PF<D>::V + c) * p.pcap + i] = a.v[(int64_t)i * D + c];
        }
#pragma unroll
        for (int k = 0; k < D * D; ++k)
            p.pcur[(PF<D>::F + k) * p.pcap + i] = a.F ? a.F[(int64_t)i * D * D + k] : (k % (D + 1) == 0 ? 1.0f : 0.0f);
        p.pcur[PF<D>::J * p.pcap + i] = a.Jp ? a.Jp[i] : (mat.eos ? mat.rho0 : 1.0f);
        p.pcur[PF<D>::M * p.pcap + i] = a.mass[i];
        p.pcur[PF<D>::VOL * p.pcap + i] = a.volume[i];
        p.pcur[PF<D>::MAT * p.pcap + i] = __int_as_float(0);
        p.idcur[i] = i;
        p.keycur[i] = 0;
        p.scur[i] = 0;
        a.valid[i] = 0;
    }
}

template <int D>
__global__ __launch_bounds__(WG) void k_noalloc_store(KP p, NoallocOut o) {
    const int n = p.ctr->n_live;  // binned particles (dropped ones keep valid = 0)
    for (int j = blockIdx.x * WG + threadIdx.x; j < n; j += gridDim.x * WG) {
        const int64_t i = p.idcur[j];
        o.valid[i] = p.keycur[j] >= 0 ? 1 : 0;
#pragma unroll
        for (int c = 0; c < D; ++c) {
            o.x[i * D + c] = p.pcur[(PF<D>::X + c) * p.pcap + j];
            o.v[i * D + c] = p.pcur[(PF<D>::V + c) * p.pcap + j];
        }
        if (o.F) {
#pragma unroll
            for (int k = 0; k < D * D; ++k) o.F[i * D * D + k] = p.pcur[(PF<D>::F + k) * p.pcap + j];
        }
        if (o.Jp) o.Jp[i] = p.pcur[PF<D>::J * p.pcap + j];
        o.volume[i] = p.pcur[PF<D>::VOL * p.pcap + j];
    }
}

// ============================================================================
// launchers
// ============================================================================
template <int D> void launch_noalloc_load(const KP& p, hipStream_t s, int grid, const SceneParams& sp, const NoallocIn& a) {
    hipLaunchKernelGGL(k_noalloc_load<D>, dim3(grid), dim3(WG), 0, s, p, sp, a);
}
template <int D> void launch_noalloc_store(const KP& p, hipStream_t s, int grid, const NoallocOut& o) {
    hipLaunchKernelGGL(k_noalloc_store<D>, dim3(grid), dim3(WG), 0, s, p, o);
}
template void launch_noalloc_load<2>(const KP&, hipStream_t, int, const SceneParams&, const NoallocIn&);
template void launch_noalloc_load<3>(const KP&, hipStream_t, int, const SceneParams&, const NoallocIn&);
template void launch_noalloc_store<2>(const KP&, hipStream_t, int, const NoallocOut&);
template void launch_noalloc_store<3>(const KP&, hipStream_t, int, const NoallocOut&);
void launch_set_step(const KP& p, hipStream_t s, const StepArgs& a) {
    hipLaunchKernelGGL(k_set_step, dim3((a.n + WG - 1) / WG), dim3(WG), 0, s, p, a);
}
void launch_set_step_dev(const KP& p, hipStream_t s, const float* dt) {
    hipLaunchKernelGGL(k_set_step_dev, dim3((p.nscenes + WG - 1) / WG), dim3(WG), 0, s, p, dt);
}
void launch_frame_dt(const KP& p, hipStream_t s, FrameState* f, float* dt) {
    hipLaunchKernelGGL(k_frame_dt, dim3(1), dim3(WG), 0, s, p, f, dt);
}
void launch_clear_waiting(const KP& p, hipStream_t s) {
    hipLaunchKernelGGL(k_clear_waiting, dim3((p.nscenes + WG - 1) / WG), dim3(WG), 0, s, p);
}
void launch_remove_scene(const KP& p, hipStream_t s, int grid, int scene) {
    hipLaunchKernelGGL(k_remove_scene, dim3(grid), dim3(WG), 0, s, p, scene);
}
template <int D> void launch_bin(const KP& p, hipStream_t s, int grid) { hipLaunchKernelGGL(k_bin<D>, dim3(grid), dim3(WG), 0, s, p); }

// Streaming copy of n4 float4 (the measured bandwidth roof): one float4
// per thread over a grid that covers the buffer (on MI355X this form beat
// grid-stride loops with four loads in flight, 6.2 against 4.3-4.9 TB/s).
__global__ __launch_bounds__(WG) void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, int64_t n4) {
    const int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x;
    if (i < n4) dst[i] = src[i];
}
void launch_copy(const float4* src, float4* dst, int64_t n4, hipStream_t s) {
    hipLaunchKernelGGL(k_copy, dim3((unsigned)((n4 + WG - 1) / WG)), dim3(WG), 0, s, src, dst, n4);
}
void launch_scan(const KP& p, hipStream_t s) {
    constexpr int EACH = SCAN_ONE * SCAN_PER_THREAD;
    if (p.nslots <= EACH) {
        hipLaunchKernelGGL(k_scan_one<1>, dim3(1), dim3(SCAN_ONE), 0, s, p);
    } else if (p.nslots <= 2 * EACH) {
        hipLaunchKernelGGL(k_scan_one<2>, dim3(1), dim3(SCAN_ONE), 0, s, p);
    } else {
        hipLaunchKernelGGL(k_scan_reduce, dim3(p.nparts), dim3(WG), 0, s, p);
        hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(WG), 0, s, p);
        hipLaunchKernelGGL(k_scan_apply, dim3(p.nparts), dim3(WG), 0, s, p);
    }
}
template <int D> void launch_block_setup(const KP& p, hipStream_t s, int grid) { hipLaunchKernelGGL(k_block_setup<D>, dim3(grid), dim3(WG), 0, s, p); }
void launch_setup_order(const KP& p, hipStream_t s, int cell_groups) {
    const int grid = ORDER_GROUPS + (p.nscenes + WG - 1) / WG + cell_groups;
    hipLaunchKernelGGL(k_setup_order, dim3(grid), dim3(WG), 0, s, p);
}
int pack_tiles(int64_t nid) { return (int)((nid + PACK_TILE - 1) / PACK_TILE); }
void launch_pack_count(const KP& p, hipStream_t s, const PackArgs& a) {
    const auto groups = [](int64_t n) { return dim3((unsigned)std::min<int64_t>(std::max<int64_t>((n + WG - 1) / WG, 1), 8192)); };
    const int tiles = pack_tiles(a.nid);
    hipLaunchKernelGGL(k_pack_clear, groups(a.nid), dim3(WG), 0, s, a);
    hipLaunchKernelGGL(k_pack_mark, groups(a.last - a.first), dim3(WG), 0, s, p, a);
    hipLaunchKernelGGL(k_pack_count, dim3(tiles), dim3(WG), 0, s, a);
    hipLaunchKernelGGL(k_pack_top, dim3(1), dim3(WG), 0, s, a, tiles);
}
template <int D> void launch_pack_write(const KP& p, hipStream_t s, const PackArgs& a) {
    hipLaunchKernelGGL(k_pack_write<D>, dim3(pack_tiles(a.nid)), dim3(WG), 0, s, p, a);
}
template void launch_pack_write<2>(const KP&, hipStream_t, const PackArgs&);
template void launch_pack_write<3>(const KP&, hipStream_t, const PackArgs&);
void launch_read_speeds(const KP& p, hipStream_t s, int* dst) { hipLaunchKernelGGL(k_read_speeds, dim3(1), dim3(WG), 0, s, p, dst); }
void launch_poll(const KP& p, hipStream_t s, int* dst) { hipLaunchKernelGGL(k_poll, dim3(1), dim3(64), 0, s, p, dst); }
template <int D> void launch_reorder(const KP& p, hipStream_t s, int grid) { hipLaunchKernelGGL(k_reorder<D>, dim3(grid), dim3(WG), 0, s, p); }
template <int D> void launch_p2g(const KP& p, hipStream_t s, int grid) {
    hipLaunchKernelGGL(k_p2g<D>, dim3(grid), dim3(BWG), 0, s, p);
}
template <int D> void launch_normalize(const KP& p, hipStream_t s, int grid) { hipLaunchKernelGGL(k_normalize<D>, dim3(grid), dim3(WG), 0, s, p); }
template <int D> void launch_init_volume(const KP& p, hipStream_t s, int grid) { hipLaunchKernelGGL(k_init_volume<D>, dim3(grid), dim3(BWG), 0, s, p); }
template <int D> void launch_particle_force(const KP& p, hipStream_t s, int grid, bool constitutive, bool force) {
    if (constitutive && force) hipLaunchKernelGGL((k_particle_force<D, true, true>), dim3(grid), dim3(BWG), 0, s, p);
    else if (constitutive) hipLaunchKernelGGL((k_particle_force<D, true, false>), dim3(grid), dim3(BWG), 0, s, p);
    else if (force) hipLaunchKernelGGL((k_particle_force<D, false, true>), dim3(grid), dim3(BWG), 0, s, p);
}
template <int D> void launch_grid_update(const KP& p, hipStream_t s, int grid, bool force, bool collision, bool cg_init, bool write_f) {
    if (force && collision && !cg_init && !write_f) hipLaunchKernelGGL((k_grid_update<D, true, true, false, false>), dim3(grid), dim3(WG), 0, s, p);
    else if (force && !collision && !cg_init && write_f) hipLaunchKernelGGL((k_grid_update<D, true, false, false, true>), dim3(grid), dim3(WG), 0, s, p);
    else if (force && !collision && !cg_init) hipLaunchKernelGGL((k_grid_update<D, true, false, false, false>), dim3(grid), dim3(WG), 0, s, p);
    else if (!force && collision && !cg_init) hipLaunchKernelGGL((k_grid_update<D, false, true, false, false>), dim3(grid), dim3(WG), 0, s, p);
    else if (!force && !collision && cg_init) hipLaunchKernelGGL((k_grid_update<D, false, false, true, false>), dim3(grid), dim3(WG), 0, s, p);
    else hipLaunchKernelGGL((k_grid_update<D, true, true, true, false>), dim3(grid), dim3(WG), 0, s, p);
}
template <int D> void launch_cg_force(const KP& p, hipStream_t s, int grid, bool restart) {
    if (restart) hipLaunchKernelGGL((k_cg_force<D, true>), dim3(grid), dim3(BWG), 0, s, p);
    else hipLaunchKernelGGL((k_cg_force<D, false>), dim3(grid), dim3(BWG), 0, s, p);
}
template <int D> void launch_cg_node(const KP& p, hipStream_t s, int blocks, int k, bool restart) {
    const int grid = std::min(CG_NODE_GROUPS, ((blocks + NGB - 1) / NGB + 7) / 8 * 8);
    if (restart) hipLaunchKernelGGL((k_cg_node<D, true>), dim3(grid), dim3(NGW), 0, s, p, 0);
    else hipLaunchKernelGGL((k_cg_node<D, false>), dim3(grid), dim3(NGW), 0, s, p, k);
}
template <int D> void launch_cg_solve(const KP& p, hipStream_t s) {
    hipLaunchKernelGGL((k_cg_solve<D>), dim3(CG_GROUPS), dim3(CGW), 0, s, p);
}
template <int D> void launch_g2p(const KP& p, hipStream_t s, int grid) {
    hipLaunchKernelGGL(k_g2p<D>, dim3(grid), dim3(BWG), 0, s, p);
    hipLaunchKernelGGL(k_g2p_reduce, dim3(p.nscenes), dim3(WG), 0, s, p);
}
template <int D> void launch_max_speed(const KP& p, hipStream_t s, int grid) { hipLaunchKernelGGL(k_max_speed<D>, dim3(grid), dim3(WG), 0, s, p); }

#define MPM_INSTANTIATE(D)                                                                    \
    template void launch_bin<D>(const KP&, hipStream_t, int);                                 \
    template void launch_block_setup<D>(const KP&, hipStream_t, int);                         \
    template void launch_reorder<D>(const KP&, hipStream_t, int);                             \
    template void launch_p2g<D>(const KP&, hipStream_t, int);                                 \
    template void launch_normalize<D>(const KP&, hipStream_t, int);                           \
    template void launch_init_volume<D>(const KP&, hipStream_t, int);                         \
    template void launch_particle_force<D>(const KP&, hipStream_t, int, bool, bool);          \
    template void launch_grid_update<D>(const KP&, hipStream_t, int, bool, bool, bool, bool); \
    template void launch_cg_force<D>(const KP&, hipStream_t, int, bool);                      \
    template void launch_cg_node<D>(const KP&, hipStream_t, int, int, bool);                  \
    template void launch_cg_solve<D>(const KP&, hipStream_t);                                 \
    template void launch_g2p<D>(const KP&, hipStream_t, int);                                 \
    template void launch_max_speed<D>(const KP&, hipStream_t, int);
MPM_INSTANTIATE(2)
MPM_INSTANTIATE(3)

}  // namespace mpm
