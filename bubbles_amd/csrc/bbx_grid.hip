// bbx_grid.hip -- neighbour-grid build on gfx950.
//
// Replaces the reference's per-cell linked-list redistribution
// (UpdateGridDistributionKernel / SwapGridStatesKernel / UpdateParticlesBuckets,
// src/equations/sph_equations3.cpp:487-539 over src/core/grid.h:389-500,422-447)
// with a counting sort into cell-contiguous storage:
//
//   1. hash      one thread per particle: FP64 cell hash, sort key, atomic count
//                (and the key into its cell's bin)
//   2. scan      exclusive prefix sum of the cell counts (wave64 shuffles + LDS)
//   3. scatter   place each particle in its cell's segment (arrival order; not
//                where there are bins)
//   4. rank+move rank every particle inside its cell by key and move x, v
//   5. buckets   per particle, walk the 27 cells in (y,x,z) order, apply the
//                reference's FP64 cutoff, keep the first 100 -- fused with the
//                density sum over the same members
//
// Reference chain order is reproduced by the key: a full distribution orders
// each cell by particle id (DistributeByParticle); an incremental one
// (DistributeToCellOpt) concatenates the 27 neighbour cells' old chains in
// (y,x,z) order, i.e. key = (direction of the old cell seen from the new cell,
// old storage slot), since storage is the old chain order.
#include <algorithm>

#include "bbx_mlp_device.h"
#include "bbx_tile.h"

namespace bbx {

// ---------------------------------------------------------------------------
// fills and scan
// ---------------------------------------------------------------------------
__global__ void k_fill_int(int *__restrict__ p, int value, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

int launch_fill_int(bbx_solver *s, int *p, int value, size_t n) {
    if (n == 0) return BBX_OK;
    size_t blocks = (n + kBlock - 1) / kBlock;
    k_fill_int<<<dim3((unsigned)blocks), dim3(kBlock), 0, s->stream>>>(p, value, n);
    BBX_HIP_CHECK(hipGetLastError());
    return BBX_OK;
}

// A new solver's per-particle fields at zero, every slot in no chain and no
// tile staged: one launch for what were eleven clears and two uploads.
__global__ void __launch_bounds__(kBlock) k_init_fields(size_t n, int none, float4 *__restrict__ force,
                                                        float4 *__restrict__ fp, float4 *__restrict__ xstar,
                                                        float4 *__restrict__ xq, float *__restrict__ rho,
                                                        float *__restrict__ pres, float *__restrict__ rho_star,
                                                        float *__restrict__ feat, int *__restrict__ nbr_cnt,
                                                        int *__restrict__ cell, int *__restrict__ home,
                                                        int *__restrict__ tab, size_t ntab) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ntab) tab[i] = 0;
    if (i >= n) return;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    force[i] = zero;
    fp[i] = zero;
    xstar[i] = zero;
    xq[i] = zero;
    rho[i] = 0.f;
    pres[i] = 0.f;
    rho_star[i] = 0.f;
    for (int f = 0; f < BBX_NFEAT; f++) feat[(size_t)f * n + i] = 0.f;
    nbr_cnt[i] = 0;
    cell[i] = none;
    home[i] = none;
}

int launch_init_fields(bbx_solver *s) {
    const size_t n = (size_t)s->stride, ntab = (size_t)s->ntiles * kTabIntsHost;
    const size_t blocks = ((n > ntab ? n : ntab) + kBlock - 1) / kBlock;
    k_init_fields<<<dim3((unsigned)blocks), dim3(kBlock), 0, s->stream>>>(
        n, (int)s->grid.total, s->force, s->fp, s->xstar, s->xq, s->rho, s->pres, s->rho_star, s->feat, s->nbr_cnt,
        s->cellA, s->home, s->tile_tab, ntab);
    BBX_HIP_CHECK(hipGetLastError());
    return BBX_OK;
}

// Block-wide exclusive scan of kScanItems items per thread.  Each workgroup
// scans kBlock*kScanItems elements and writes its total to block_sums.
__global__ void __launch_bounds__(kBlock) k_scan_block(const int *__restrict__ in,
                                                       int *__restrict__ out,
                                                       int *__restrict__ block_sums, size_t n) {
    __shared__ int wave_tot[kBlock / 64];
    const size_t base = (size_t)blockIdx.x * kBlock * kScanItems + (size_t)threadIdx.x * kScanItems;
    int v[kScanItems];
    int sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        size_t i = base + k;
        v[k] = i < n ? in[i] : 0;
        sum += v[k];
    }
    // inclusive scan of thread sums inside the wave
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int incl = sum;
    for (int off = 1; off < 64; off <<= 1) {
        int o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    if (lane == 63) wave_tot[wave] = incl;
    __syncthreads();
    int wave_off = 0;
    for (int w = 0; w < wave; w++) wave_off += wave_tot[w];
    int run = wave_off + incl - sum;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        size_t i = base + k;
        if (i < n) out[i] = run;
        run += v[k];
    }
    if (threadIdx.x == kBlock - 1) {
        int tot = 0;
        for (int w = 0; w < kBlock / 64; w++) tot += wave_tot[w];
        block_sums[blockIdx.x] = tot;
    }
}

__global__ void k_scan_add(int *__restrict__ out, const int *__restrict__ block_off, size_t n) {
    const size_t per = (size_t)kBlock * kScanItems;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] += block_off[i / per];
}

// Second pass of a scan over at most kScanFuseBlocks first-pass blocks:
// workgroup w adds to its kBlock * kScanItems elements (those of first-pass
// block w) the sum of the first-pass totals before it, which it reduces
// itself, so the totals need no scan of their own.
constexpr int kScanFuseBlocks = 4 * kBlock;
__global__ void __launch_bounds__(kBlock) k_scan_add_reduce(int *__restrict__ out,
                                                            const int *__restrict__ block_sums, size_t n) {
    __shared__ int wave_tot[kBlock / 64];
    __shared__ int offset;
    const int w = (int)blockIdx.x;
    int part = 0;
    for (int t = (int)threadIdx.x; t < w; t += kBlock) part += block_sums[t];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
    if (lane == 0) wave_tot[wave] = part;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int k = 0; k < kBlock / 64; k++) tot += wave_tot[k];
        offset = tot;
    }
    __syncthreads();
    const int add = offset;
    const size_t base = (size_t)w * kBlock * kScanItems;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        const size_t i = base + (size_t)k * kBlock + threadIdx.x;
        if (i < n) out[i] += add;
    }
}

// The whole scan in one launch for few blocks: every workgroup sums what
// lies before its own elements itself (at most 30k ints) instead of a second
// launch that adds block totals (4.0 + 3.0 us for 9k cells, 4.5 now).
constexpr int kScanOneLaunch = 16;  // blocks
__global__ void __launch_bounds__(kBlock) k_scan_small(const int *__restrict__ in, int *__restrict__ out, size_t n) {
    __shared__ int before[kBlock / 64], wave_tot[kBlock / 64];
    const size_t base = (size_t)blockIdx.x * kBlock * kScanItems;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int v[kScanItems], sum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        const size_t i = base + (size_t)threadIdx.x * kScanItems + k;
        v[k] = i < n ? in[i] : 0;
        sum += v[k];
    }
    int part = 0;
    const int4 *in4 = reinterpret_cast<const int4 *>(in);  // base is a multiple of 4
    const int lim = (int)(base / 4);
    for (int t = (int)threadIdx.x; t < lim; t += 8 * kBlock) {
        int4 q[8];
#pragma unroll
        for (int k = 0; k < 8; k++) q[k] = in4[min(t + k * kBlock, lim - 1)];
#pragma unroll
        for (int k = 0; k < 8; k++) part += t + k * kBlock < lim ? q[k].x + q[k].y + q[k].z + q[k].w : 0;
    }
    for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
    int incl = sum;
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(incl, off, 64);
        if (lane >= off) incl += o;
    }
    if (lane == 63) wave_tot[wave] = incl;
    if (lane == 0) before[wave] = part;
    __syncthreads();
    int run = incl - sum;
    for (int w = 0; w < kBlock / 64; w++) run += before[w] + (w < wave ? wave_tot[w] : 0);
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        const size_t i = base + (size_t)threadIdx.x * kScanItems + k;
        if (i < n) out[i] = run;
        run += v[k];
    }
}

// Exclusive scan, recursive over block totals.  Needs scan_tmp sized by
// scan_scratch_elems(n).
static size_t blocks_for(size_t n) { return (n + (size_t)kBlock * kScanItems - 1) / ((size_t)kBlock * kScanItems); }

size_t scan_scratch_elems(size_t n) {
    size_t total = 0;
    while (n > 1) {
        size_t b = blocks_for(n);
        total += 2 * b;
        n = b;
    }
    return total + 2;
}

static int scan_rec(bbx_solver *s, const int *in, int *out, size_t n, int *tmp) {
    size_t b = blocks_for(n);
    int *sums = tmp;
    int *sums_scanned = tmp + b;
    k_scan_block<<<dim3((unsigned)b), dim3(kBlock), 0, s->stream>>>(in, out, sums, n);
    BBX_HIP_CHECK(hipGetLastError());
    if (b > 1 && b <= (size_t)kScanFuseBlocks) {
        k_scan_add_reduce<<<dim3((unsigned)b), dim3(kBlock), 0, s->stream>>>(out, sums, n);
        BBX_HIP_CHECK(hipGetLastError());
    } else if (b > 1) {
        BBX_CHECK(scan_rec(s, sums, sums_scanned, b, tmp + 2 * b));
        size_t blocks = (n + kBlock - 1) / kBlock;
        k_scan_add<<<dim3((unsigned)blocks), dim3(kBlock), 0, s->stream>>>(out, sums_scanned, n);
        BBX_HIP_CHECK(hipGetLastError());
    }
    return BBX_OK;
}

int launch_scan(bbx_solver *s, const int *in, int *out, size_t n) {
    if (n == 0) return BBX_OK;
    const size_t b = blocks_for(n);
    if (b <= (size_t)kScanOneLaunch) {
        k_scan_small<<<dim3((unsigned)b), dim3(kBlock), 0, s->stream>>>(in, out, n);
        BBX_HIP_CHECK(hipGetLastError());
        return BBX_OK;
    }
    if (scan_scratch_elems(n) > s->scan_tmp_elems) return fail(BBX_E_RANGE, "scan scratch too small");
    return scan_rec(s, in, out, n, s->scan_tmp);
}

// ---------------------------------------------------------------------------
// 1. hash + key + count
// ---------------------------------------------------------------------------
// Full mode (flag set, or first distribution): key = particle id.
// Incremental mode: key = (27-neighbour direction index of the old cell as
// seen from the new cell, old slot); a particle whose cell moved by more than
// one in any axis, or that was in no chain, stays in no chain (the reference
// only looks at the 27 neighbours' chains).
// Append mode (append_from >= 0, after new particles were placed in slots
// append_from..n-1): every old particle keeps its chain and place (key = old
// slot), every new one joins the chain of the cell it hashes into, after the
// old members in the order added (DistributeByParticleList + AddToChain,
// src/core/grid.h:358-387,128-140).
//
// With kBins (see distribute_grid) the key also goes into its cell's bin at
// its arrival slot, so that the particle's rank can be counted from the bin
// and neither a scatter into cell segments nor its index is needed.  The keys
// behind a full bin go into blocks of as many.  How many a cell needs is not
// known yet, so they are found by hashing (cell, number of the block): whoever
// comes first enters it into the table, whose slot is the block.  An entry
// carries the pass number, so that those of earlier passes need no clearing.
// Particles in no chain, which may be many, are listed by arrival.
constexpr int kBinCap = 32;
constexpr int kTagPassBits = 13, kTagCellBits = 28;
struct BinKeys {
    unsigned long long *__restrict__ bin;  // [cells][kBinCap]
    unsigned long long *tag;               // [nblk] pass | number | cell
    unsigned long long *__restrict__ more; // [nblk][kBinCap]
    int *__restrict__ none;                // [n] particles in no chain
    unsigned nblk;                         // more than a pass can need: a block's cell has 32 others, and a full bin
    unsigned pass;

    __device__ __forceinline__ unsigned long long want(int cell, unsigned block) const {
        return ((unsigned long long)pass << (64 - kTagPassBits)) | ((unsigned long long)block << kTagCellBits) | (unsigned)cell;
    }
    __device__ __forceinline__ unsigned home(int cell, unsigned block) const {
        unsigned h = (unsigned)cell * 0x9E3779B1u + block * 0x85EBCA77u;
        h ^= h >> 15;
        return __umulhi(h * 0x2C1B3C6Du, nblk);
    }
    __device__ __forceinline__ unsigned after(unsigned h) const { return h + 1 < nblk ? h + 1 : 0u; }
    // The block, entered if it is new.  The table is never full and a block
    // that is read has been entered, so both searches end at it; the bound on
    // their steps only says that they end.
    __device__ __forceinline__ unsigned enter(int cell, unsigned block) const {
        const unsigned long long w = want(cell, block);
        unsigned h = home(cell, block);
        for (unsigned k = 0; k < nblk; k++, h = after(h)) {
            unsigned long long v = __hip_atomic_load(&tag[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (v != w && (unsigned)(v >> (64 - kTagPassBits)) != pass) {
                const unsigned long long old = atomicCAS(&tag[h], v, w);
                v = old == v ? w : old;  // an entry changes once in a pass
            }
            if (v == w) break;
        }
        return h;
    }
    // a block that an earlier launch entered, given what its home holds
    __device__ __forceinline__ unsigned find(int cell, unsigned block, unsigned long long at_home) const {
        const unsigned long long w = want(cell, block);
        unsigned h = home(cell, block);
        unsigned long long v = at_home;
        for (unsigned k = 0; v != w && k < nblk; k++, v = tag[h]) h = after(h);
        return h;
    }
};
template <bool kBins>
__global__ void __launch_bounds__(kBlock) k_hash(SimConst c, const float4 *__restrict__ pos,
                                                 const int *__restrict__ cell_old,
                                                 const int *__restrict__ flag, int force_full,
                                                 int append_from,
                                                 int *__restrict__ newc, int *__restrict__ hcell,
                                                 unsigned long long *__restrict__ key,
                                                 int *__restrict__ count,
                                                 int *__restrict__ rank_tmp, BinKeys bk) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int none = (int)c.g.total;
    const bool valid = s < c.n;
    // the wave stays whole for the aggregated count below
    const float4 p = valid ? pos[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    int u[3], bad = 0;
    int cid = hash_cell(c.g, p, u, &bad);
    bool full = append_from < 0 && (force_full || (*flag != 0));
    int nc;
    unsigned long long k;
    if (append_from >= 0) {
        k = (unsigned long long)s;
        if (s < append_from)
            nc = valid ? cell_old[s] : none;
        else
            nc = bad ? none : cid;
    } else if (full) {
        nc = bad ? none : cid;
        k = (unsigned long long)(unsigned)pid_of(p);
    } else {
        const int co = valid ? cell_old[s] : none;
        nc = none;
        k = (unsigned long long)s;
        if (!bad && co != none) {
            int uo[3];
            unlinear(c.g, co, uo);
            int dx = uo[0] - u[0], dy = uo[1] - u[1], dz = uo[2] - u[2];
            if (dx >= -1 && dx <= 1 && dy >= -1 && dy <= 1 && dz >= -1 && dz <= 1) {
                nc = cid;
                unsigned d = (unsigned)((dy + 1) * 9 + (dx + 1) * 3 + (dz + 1));
                k = ((unsigned long long)d << 32) | (unsigned long long)(unsigned)s;
            }
        }
    }
    // Storage is sorted by cell, so lanes with the same new cell mostly form
    // runs: one atomic per run reserves its slots (the order inside a cell
    // is set later by the key, not by arrival).
    const int lane = threadIdx.x & 63;
    const int cellv = valid ? nc : -1;
    const int prev = __shfl_up(cellv, 1, 64);
    const bool head = lane == 0 || prev != cellv;
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
    const int head_lane = 63 - __builtin_clzll(heads & upto);
    const unsigned long long after = heads & ~upto;
    const int next_head = after ? __builtin_ctzll(after) : 64;
    int base = 0;
    if (head && valid) base = atomicAdd(&count[nc], next_head - lane);
    base = __shfl(base, head_lane, 64);
    const int slot = base + (lane - head_lane);
    unsigned block = 0u;
    if constexpr (kBins) {
        // the first lane of a run that is in a block enters it for the others
        const bool over = valid && nc != none && slot >= kBinCap;
        if (__any(over)) {
            const int first = max(lane - slot % kBinCap, head_lane);
            if (over && lane == first) block = bk.enter(nc, (unsigned)(slot / kBinCap - 1));
            block = (unsigned)__shfl((int)block, first, 64);
        }
    }
    if (!valid) return;
    newc[s] = nc;
    // a point outside the grid has no home cell: its bucket stays empty
    hcell[s] = bad ? -1 : cid;
    key[s] = k;
    if constexpr (kBins) {
        if (nc == none)
            bk.none[slot] = s;
        else if (slot < kBinCap)
            bk.bin[(size_t)nc * kBinCap + slot] = k;
        else
            bk.more[(size_t)block * kBinCap + slot % kBinCap] = k;
    } else {
        rank_tmp[s] = slot;
    }
}

size_t grid_bin_words(size_t cells) { return cells * kBinCap; }
// the table of blocks, then the blocks (see BinKeys)
static size_t bin_blocks(size_t stride) { return stride / (kBinCap / 2) + 64; }
size_t grid_block_words(size_t stride) { return bin_blocks(stride) * (kBinCap + 1); }

// What the pass reports and leaves behind, done by the last launch that may
// (thread t of all): statistics, the higher-level flag, the cell counts back
// at zero for the next pass, and `clear` (a substep's step block behind its
// counters), which took a launch of their own (4.2 us at 1M).
struct PassEnd {
    int *__restrict__ count;
    size_t cells;
    int *__restrict__ flag;
    int force_full, append;
    int *__restrict__ counters;
    int *__restrict__ clear;
    size_t clear_n;
};
__device__ __forceinline__ void end_pass(const SimConst &c, const PassEnd &e, const int *__restrict__ start, size_t t) {
    if (t == 0) {
        e.counters[CNT_OVERFLOW] = 0;
        e.counters[CNT_LOST] = c.n - start[c.g.total];
        if (!e.append) {  // an append leaves the higher-level flag to the next substep
            e.counters[CNT_FULL] = (e.force_full || *e.flag) ? 1 : 0;
            *e.flag = 0;  // ResetHigherLevel
        } else {
            e.counters[CNT_FULL] = 0;
        }
    }
    if (t < e.cells) e.count[t] = 0;
    if (t < e.clear_n) e.clear[t] = 0;
}

// ---------------------------------------------------------------------------
// 3. scatter into cell segments (arrival order); the cell counts have been
// read for the last time, so the pass ends here
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kBlock) k_scatter(SimConst c, const int *__restrict__ newc,
                                                    const int *__restrict__ rank_tmp,
                                                    const int *__restrict__ start,
                                                    int *__restrict__ tmp_idx, PassEnd end) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    end_pass(c, end, start, t);
    if (t < (size_t)c.n) tmp_idx[start[newc[t]] + rank_tmp[t]] = (int)t;
}

// ---------------------------------------------------------------------------
// 4. rank inside the cell by key and move the particle state
// ---------------------------------------------------------------------------
// Keys are unique inside a cell (particle id, or (direction, old slot), or
// old slot), so rank = number of smaller keys in the cell is a permutation
// of the cell's segment at every occupancy.  A workgroup whose particles all
// lie in one crowded cell stages the cell's keys through LDS a workgroup-
// width chunk at a time (every lane then reads the same LDS word: a
// broadcast); any other workgroup compares against global memory.
constexpr int kRankLds = 512;  // cells above this use the LDS chunks when uniform
__global__ void __launch_bounds__(kBlock) k_rank_move(SimConst c, const int *__restrict__ tmp_idx,
                                                      const int *__restrict__ newc,
                                                      const int *__restrict__ hcell,
                                                      const unsigned long long *__restrict__ key,
                                                      const int *__restrict__ start,
                                                      const float4 *__restrict__ pos_in,
                                                      const float4 *__restrict__ vel_in,
                                                      float4 *__restrict__ pos_out,
                                                      float4 *__restrict__ vel_out,
                                                      int *__restrict__ cell_out,
                                                      int *__restrict__ home_out) {
    __shared__ unsigned long long skey[kBlock];
    __shared__ int cell0;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = t < c.n;
    const int s = valid ? tmp_idx[t] : 0;
    const int cc = valid ? newc[s] : -1;
    const unsigned long long k = valid ? key[s] : 0ull;
    const int b = valid ? start[cc] : 0;
    const int total = (int)c.g.total;  // start[total]: the particles in no chain, up to n
    const int e = valid ? (cc < total ? start[cc + 1] : c.n) : 0;
    // thread 0 is valid in every launched workgroup (the grid is ceil(n / kBlock))
    if (threadIdx.x == 0) cell0 = cc;
    // Thread t holds the key of storage slot t, so the keys of the cell
    // members inside this workgroup's slots come from LDS; only members in
    // neighbouring workgroups' slots are read from global memory.
    const int blk0 = (int)(blockIdx.x * blockDim.x);
    skey[threadIdx.x] = k;
    __syncthreads();
    const bool uniform = __syncthreads_and(!valid || cc == cell0) != 0;
    const int c0 = cell0;
    const int bb = uniform ? start[c0] : 0;
    const int ee = uniform ? (c0 < total ? start[c0 + 1] : c.n) : 0;
    int rank = 0;
    if (uniform && ee - bb > kRankLds) {
        // every valid thread has [b, e) == [bb, ee); the trip count and the
        // barriers are the same for the whole workgroup
        for (int q0 = bb; q0 < ee; q0 += kBlock) {
            const int q = q0 + (int)threadIdx.x;
            if (q < ee) skey[threadIdx.x] = key[tmp_idx[q]];
            __syncthreads();
            if (valid) {
                const int m = min(kBlock, ee - q0);
                for (int u = 0; u < m; u++) rank += skey[u] < k ? 1 : 0;
            }
            __syncthreads();
        }
    } else if (valid) {
        for (int q = b; q < e; q++) {
            const int u = q - blk0;
            const unsigned long long kq = (u >= 0 && u < kBlock) ? skey[u] : key[tmp_idx[q]];
            rank += kq < k ? 1 : 0;
        }
    }
    if (!valid) return;
    const int dest = b + rank;
    pos_out[dest] = pos_in[s];
    vel_out[dest] = vel_in[s];
    cell_out[dest] = cc;
    home_out[dest] = hcell[s];
}

// How many of the keys behind a full bin are smaller (whole waves; cnt > kBinCap
// where there are any).  A wave of one cell -- storage is sorted, so all but the
// first pass over a very crowded cell -- reads two blocks at a time, a key a
// lane, the next two while it compares these; otherwise each lane streams its
// own cell's.  Hash and rank from the bins / hash, scatter and rank through the
// index (us), storage sorted: 10,000 particles in cells of 33 17.7 / 21.8, of 100
// 19.4 / 33.5, of 1,000 57 / 196, of 10,000 177 / 172; 1M in cells of 100 67 / 98.
// Shuffled: 10,000 in cells of 100 37 / 44, of 1,000 120 / 229; 1M in cells of
// 100 382 / 216.
__device__ __forceinline__ int smaller_behind_bin(const BinKeys &bk, int cell, int cnt, unsigned long long k, bool valid) {
    int rank = 0;
    const int lane = threadIdx.x & 63;
    const int cell0 = __builtin_amdgcn_readfirstlane(cell), cnt0 = __builtin_amdgcn_readfirstlane(cnt);
    if (__all(!valid || (cell == cell0 && cnt == cnt0))) {
        const int at = lane % kBinCap, half = lane / kBinCap;
        auto load = [&](int w0) {
            const int w = w0 + half;
            if (kBinCap * (w + 1) + at >= cnt0) return ~0ull;
            const unsigned h = bk.find(cell0, (unsigned)w, bk.tag[bk.home(cell0, (unsigned)w)]);
            return bk.more[(size_t)h * kBinCap + at];
        };
        unsigned long long v = load(0);
        for (int w0 = 0; kBinCap * (w0 + 1) < cnt0; w0 += 64 / kBinCap) {
            const unsigned long long next = load(w0 + 64 / kBinCap);
            const int lo = (int)(unsigned)v, hi = (int)(unsigned)(v >> 32);
            const int hi0 = __builtin_amdgcn_readfirstlane(hi);
            if (__all(hi == hi0)) {  // ids, or slots of one direction
                int below = 0;
#pragma unroll
                for (int u = 0; u < 64; u++) below += (unsigned)__builtin_amdgcn_readlane(lo, u) < (unsigned)k ? 1 : 0;
                rank += (unsigned)hi0 == (unsigned)(k >> 32) ? below : ((unsigned)hi0 < (unsigned)(k >> 32) ? 64 : 0);
            } else {
#pragma unroll
                for (int u = 0; u < 64; u++) {
                    const unsigned long long key =
                        ((unsigned long long)(unsigned)__builtin_amdgcn_readlane(hi, u) << 32) | (unsigned)__builtin_amdgcn_readlane(lo, u);
                    rank += key < k ? 1 : 0;
                }
            }
            v = next;
        }
        return rank;
    }
    const unsigned blocks = cnt > kBinCap ? (unsigned)(cnt - 1) / kBinCap : 0u;
    unsigned long long at_home = blocks ? bk.tag[bk.home(cell, 0)] : 0ull;
    for (unsigned w = 0; w < blocks; w++) {
        const unsigned h = bk.find(cell, w, at_home);
        if (w + 1 < blocks) at_home = bk.tag[bk.home(cell, w + 1)];
        const ulonglong2 *more = reinterpret_cast<const ulonglong2 *>(bk.more + (size_t)h * kBinCap);
        const int m = min(kBinCap, cnt - kBinCap * (int)(w + 1));
        constexpr int kAhead = kBinCap / 4;  // pairs of keys in flight
        for (int u0 = 0; 2 * u0 < m; u0 += kAhead) {
            ulonglong2 q[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; u++) q[u] = more[u0 + u];
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                rank += 2 * (u0 + u) < m && q[u].x < k ? 1 : 0;
                rank += 2 * (u0 + u) + 1 < m && q[u].y < k ? 1 : 0;
            }
        }
    }
    return rank;
}

// 3 and 4 from the bins: a particle's rank is the number of smaller keys in
// its cell's bin, eight of them (a cell of ordinary density) requested beside
// its other data, and in the blocks behind a full bin.  Workgroups of
// particles in no chain read those through LDS as k_rank_move does.
__global__ void __launch_bounds__(kBlock) k_rank_bins(SimConst c, const int *__restrict__ newc,
                                                      const int *__restrict__ hcell,
                                                      const unsigned long long *__restrict__ key,
                                                      const int *__restrict__ start, BinKeys bk,
                                                      const float4 *__restrict__ pos_in,
                                                      const float4 *__restrict__ vel_in,
                                                      float4 *__restrict__ pos_out,
                                                      float4 *__restrict__ vel_out,
                                                      int *__restrict__ cell_out,
                                                      int *__restrict__ home_out, PassEnd end) {
    __shared__ unsigned long long skey[kBlock];
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    end_pass(c, end, start, t);
    if ((size_t)blockIdx.x * blockDim.x >= (size_t)c.n) return;  // whole workgroups
    const bool valid = t < (size_t)c.n;
    const int total = (int)c.g.total;  // start[total]: the particles in no chain, up to n
    int cc = 0, home = -1, b = 0, cnt = 0, rank = 0;
    unsigned long long k = 0ull;
    float4 p{}, v{};
    bool lost = false;
    if (valid) {
        cc = newc[t];
        k = key[t];
        p = pos_in[t];
        v = vel_in[t];
        home = hcell[t];
        lost = cc == total;
        b = start[cc];
        if (!lost) {
            const ulonglong2 *bin = reinterpret_cast<const ulonglong2 *>(bk.bin + (size_t)cc * kBinCap);
            constexpr int kFirst = 4;  // pairs of keys
            ulonglong2 q[kFirst];
#pragma unroll
            for (int u = 0; u < kFirst; u++) q[u] = bin[u];
            cnt = start[cc + 1] - b;
#pragma unroll
            for (int u = 0; u < kFirst; u++) {
                rank += 2 * u < cnt && q[u].x < k ? 1 : 0;
                rank += 2 * u + 1 < cnt && q[u].y < k ? 1 : 0;
            }
            const int binned = min(cnt, kBinCap);
            for (int u = kFirst; 2 * u < binned; u++) {
                const ulonglong2 w = bin[u];
                rank += w.x < k ? 1 : 0;
                rank += 2 * u + 1 < binned && w.y < k ? 1 : 0;
            }
        }
    }
    if (__any(cnt > kBinCap)) rank += smaller_behind_bin(bk, cc, cnt, k, valid);
    if (__syncthreads_or(lost)) {
        const int lost_n = c.n - start[total];
        for (int q0 = 0; q0 < lost_n; q0 += kBlock) {
            const int q = q0 + (int)threadIdx.x;
            if (q < lost_n) skey[threadIdx.x] = key[bk.none[q]];
            __syncthreads();
            if (lost) {
                const int m = min(kBlock, lost_n - q0);
                for (int u = 0; u < m; u++) rank += skey[u] < k ? 1 : 0;
            }
            __syncthreads();
        }
    }
    if (!valid) return;
    const int dest = b + rank;
    pos_out[dest] = p;
    vel_out[dest] = v;
    cell_out[dest] = cc;
    home_out[dest] = home;
}

// ---------------------------------------------------------------------------
// 5. tile tables: one wave per tile of kBlock particles
// ---------------------------------------------------------------------------
// The tile's home cells span [cmin, cmax]; its nine neighbour rows become at
// most nine merged storage intervals (tab_row, tab_merge).  Every gather of
// the substep reads this table.  Storage is sorted by cell up to
// start[total], so for a tile of chained particles cmin and cmax are the
// homes of its first and last ones.  Behind them lie the particles in no
// chain in no order: outside the grid (home -1, no neighbours), or inside it
// after a jump that an incremental pass does not follow.  The latter look
// for neighbours from homes anywhere and are no candidates themselves, so
// that their own positions are in no interval: their tiles are not staged.
// A tile with any particle in no chain takes a wave reduction.  The row
// ranges of lanes 0-8 are gathered by shuffles and merged by lane 0.
// (one wave; lane 0's table is complete when the wave has synchronised)
__device__ __forceinline__ void tile_table(const SimConst &c, const int *__restrict__ home,
                                           const int *__restrict__ start, int tile, int lane, TileTab &tt) {
    const int t0 = tile * kBlock, t1 = min(t0 + kBlock, c.n) - 1;
    const int chained = start[c.g.total];
    int lo = home[t0], hi = home[t1], cap = c.tile_cap;
    if (t1 >= chained) {
        lo = 0x7fffffff;
        hi = -1;
        bool astray = false;
#pragma unroll
        for (int k = 0; k < kBlock / 64; k++) {
            const int i = t0 + k * 64 + lane;
            const int hc = i < c.n ? home[i] : -1;
            if (hc >= 0) {
                lo = min(lo, hc);
                hi = max(hi, hc);
                astray = astray || i >= chained;
            }
        }
        lo = wave_min_i32(lo);
        hi = wave_max_i32(hi);
        if (__any(astray)) cap = -1;  // no total is within it
    }
    int a = -1, b = -1;
    if (lane < 9) tab_row(c.g, hi >= 0 ? lo : 0, hi, start, lane, a, b);
    int ra[9], rb[9];
#pragma unroll
    for (int r = 0; r < 9; r++) {
        ra[r] = __shfl(a, r, 64);
        rb[r] = __shfl(b, r, 64);
    }
    if (lane == 0 && !tab_merge_ordered(ra, rb, cap, tt)) tab_merge(ra, rb, cap, tt);
}

constexpr int kTabWaves = kBlock / 64;
__global__ void __launch_bounds__(kBlock) k_tile_tables(SimConst c, const int *__restrict__ home,
                                                        const int *__restrict__ start, int ntiles,
                                                        int *__restrict__ tile_tab) {
    __shared__ TileTab tt[kTabWaves];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tile = blockIdx.x * kTabWaves + w;  // wave-uniform
    if (tile >= ntiles) return;
    tile_table(c, home, start, tile, lane, tt[w]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (lane < kTabWords) tile_tab[(size_t)tile * kTabInts + lane] = reinterpret_cast<const int *>(&tt[w])[lane];
}

// ---------------------------------------------------------------------------
// 5. buckets + density (+ Tait pressure for SPH)
// ---------------------------------------------------------------------------
// ComputeDensityFor (src/equations/sph_equations3.cpp:25-58) sums poly6 over
// the bucket in bucket order; the sum runs as the bucket is built.
// The tile's candidate intervals are staged in LDS; the bucket of a staged
// tile is written as LDS-local indices (nbr16), otherwise as storage indices
// (nbr32).  Candidates are visited in the reference's order: neighbour cells
// y outer, x, z inner (src/core/grid.h:568-591), each cell in chain order.
// The learned warm start fused into the bucket kernel (kFeat > 0): the
// features of include/bbx_features.h come from the finished bucket, the
// density and the particle's own state, so they need nothing another
// particle computes in this launch.  kFeat == 2 then infers the network on
// the workgroup's 256 particles and starts the substep from its pressures.
struct WarmIn {
    float4 *__restrict__ vr;              // (v, 1 / rho) for the viscosity gather
    StepConst st;
    const float4 *__restrict__ vel;       // own velocity, w = previous converged pressure
    int store_feat;                       // write the features to feat
    float *__restrict__ feat;             // [16][stride]
    const float *__restrict__ P;          // network parameters (kFeat == 2)
    float *__restrict__ pwarm;            // network pressure
    float *__restrict__ rho_star;         // rho* = rho at k = 0
    float4 *__restrict__ xq;              // (x, q): q = p0 / rho^2 (kFeat == 2), p / rho^2 (SPH), else 0
};

// Acceptance mask of the candidates of one row (bit t: candidate t; len <=
// 64): staged at `row` in LDS (with slack slots behind) or from storage index
// a on.  Eight at a time with no branches.  The FP32 test uses
// t = |pi - pj|^2 - band_c (the offset folded into the first FMA): t < 0
// accepts; a candidate with |t| <= band_w (rare) makes the lane re-test its
// row with the reference's FP64 rule.  The sign bits of a group enter a
// 64-bit shift register {hi, lo} at its top.
template <bool kStaged>
__device__ __forceinline__ unsigned long long row_mask(const SimConst &c, float4 pi, const float4 *row,
                                                       const float4 *__restrict__ pos, int a, int len) {
    unsigned lo = 0u, hi = 0u;
    float bdist = 3.4e38f;
    int t0 = 0;
    // Two groups of four per step: the second group's loads are in flight
    // while the first group's arithmetic runs (one step of a row reads up to
    // seven candidates past its end: slack slots when staged, clamped
    // otherwise; their bits are cleared below).
    for (; t0 < len; t0 += 8) {
        float4 pc[8];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            if (kStaged)
                pc[q] = lds_slot(row + t0 + q);
            else
                pc[q] = pos[min(a + t0 + q, c.n - 1)];
        }
        float tq[8];
#pragma unroll
        for (int q = 0; q < 8; q++) tq[q] = cut_offset(pi, pc[q], c.band_c);
#pragma unroll
        for (int q = 0; q < 8; q += 2) bdist = fminf(fminf(bdist, fabsf(tq[q])), fabsf(tq[q + 1]));
        unsigned byte = __float_as_uint(tq[7]) >> 31;  // bit q: candidate t0 + q
#pragma unroll
        for (int q = 6; q >= 0; q--) byte = __builtin_amdgcn_alignbit(byte, __float_as_uint(tq[q]), 31);
        lo = __builtin_amdgcn_alignbit(hi, lo, 8);
        hi = __builtin_amdgcn_alignbit(byte, hi, 8);
    }
    // t0 = 8 * steps; candidate t sits at bit 64 - t0 + t
    unsigned long long m = ((unsigned long long)hi << 32) | lo;
    m = t0 > 0 ? m >> (64 - t0) : 0ull;
    if (len < 64) m &= (1ull << len) - 1ull;
    if (bdist <= c.band_w) {
        // candidates inside the band: the exact FP64 rule
        for (int t = 0; t < len; t++) {
            const float4 pj = kStaged ? lds_slot(row + t) : pos[a + t];
            if (fabsf(cut_offset(pi, pj, c.band_c)) <= c.band_w) {
                const unsigned long long bit = 1ull << t;
                m = within_std_fp64(pi, pj, c.h2d) ? (m | bit) : (m & ~bit);
            }
        }
    }
    return m;
}

// ComputePressureValue (src/equations/sph_equations3.cpp:7-18)
__device__ __forceinline__ float tait_pressure(const SimConst &c, float d) {
    float p = c.eos_scale / c.eos_exp * (powf(d / c.rho0, c.eos_exp) - 1.f);
    if (p < 0.f) p *= c.nps;
    return p;
}

// A bucket as it is emitted.  The current quad of entries.  Staged: a 64-bit
// shift register of 16-bit entries held as two words (entry k of the quad
// ends in bits 16k..16k+15); global: four 32-bit entries.
template <bool kStaged>
struct BucketWriter {
    unsigned short *__restrict__ nbr16;
    int *__restrict__ nbr32;
    int stride, i;
    int cnt = 0, dropped = 0;
    unsigned qlo = 0u, qhi = 0u;
    int e0 = 0, e1 = 0, e2 = 0, e3 = 0;

    __device__ __forceinline__ BucketWriter(unsigned short *n16, int *n32, int str, int at)
        : nbr16(n16), nbr32(n32), stride(str), i(at) {}
    __device__ __forceinline__ void store_quad(int nfill) {  // nfill = entries in the quad
        const size_t at = (size_t)((cnt - 1) >> 2) * stride + i;
        if (kStaged) {
            unsigned long long q = ((unsigned long long)qhi << 32) | qlo;
            if (nfill < 4) {  // a partial quad moves down to slot 0
                q >>= 16 * (4 - nfill);
                q |= (kFarEntry * 0x0001000100010001ull) << (16 * nfill);
            }
            reinterpret_cast<uint2 *>(nbr16)[at] = make_uint2((unsigned)q, (unsigned)(q >> 32));
        } else {
            int4 v = make_int4(e0, e1, e2, e3);
            if (nfill == 3) v = make_int4(e1, e2, e3, 0);
            else if (nfill == 2) v = make_int4(e2, e3, 0, 0);
            else if (nfill == 1) v = make_int4(e3, 0, 0, 0);
            reinterpret_cast<int4 *>(nbr32)[at] = v;
        }
    }
    // append accepted candidate j (storage index; LDS index j + sh) to the
    // bucket (emit: up to the cap).  Only the index is handled here: the
    // emission loops run as long as the wave's longest cell, so the density
    // sum runs afterwards over the finished bucket, one uniform pass.
    __device__ __forceinline__ void append(int j, int sh) {
        if (kStaged) {  // the entry is the candidate's LDS byte offset
            qlo = __builtin_amdgcn_alignbit(qhi, qlo, 16);
            qhi = __builtin_amdgcn_alignbit((unsigned)(j + sh) << kSlotShift, qhi, 16);
        } else {
            e0 = e1;
            e1 = e2;
            e2 = e3;
            e3 = j;
        }
        cnt++;
        if ((cnt & 3) == 0) store_quad(4);
    }
    __device__ __forceinline__ void emit(int j, int sh) {
        if (cnt >= kBucket)
            dropped++;
        else
            append(j, sh);
    }
    __device__ __forceinline__ void finish() {
        if (cnt & 3) store_quad(cnt & 3);
    }
};

// The bucket cell by cell, in the reference's order and with its cap.
// sh[r]: LDS index - storage index of row r (zero when not staged).
template <bool kStaged>
__device__ __forceinline__ void walk_cells(const SimConst &c, float4 pi, const int (&u)[3],
                                           const int *__restrict__ start, const float4 *sx,
                                           const float4 *__restrict__ pos, const int *sh, BucketWriter<kStaged> &bw) {
    const int nx = c.g.n[0], ny = c.g.n[1], nz = c.g.n[2];
    for (int dy = 0; dy < 3; dy++)
        for (int dx = 0; dx < 3; dx++) {
            const int x = u[0] + dx - 1;
            if (x < 0 || x >= nx) continue;
            for (int dz = 0; dz < 3; dz++) {
                const int yy = u[1] + dy - 1, zz = u[2] + dz - 1;
                if (yy < 0 || yy >= ny || zz < 0 || zz >= nz) continue;
                const int cell = x + yy * nx + zz * nx * ny;
                const int sr = sh[dz * 3 + dy];
                const int e = start[cell + 1];
                for (int j = start[cell]; j < e; j++) {
                    const float4 pj = kStaged ? lds_slot(sx + j + sr) : pos[j];
                    if (in_bucket(c, pi, pj)) bw.emit(j, sr);
                }
            }
        }
}

// The features of particle i from its bucket's sums.
__device__ __forceinline__ void finish_features(const SimConst &c, const WarmIn &wi, int i, float4 pi, float di,
                                                int cnt, float m1, float m2, float m3, float cx, float cy, float cz,
                                                float *fv) {
    const float4 vi = wi.vel[i];
    const float inv = 1.f / (cnt > 1 ? (float)(cnt - 1) : 1.f);
    float wall = 3.4e38f;
    const float p3[3] = {pi.x, pi.y, pi.z};
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float lo = p3[a] - (c.tank_c[a] - c.tank_h[a]);
        const float hi = (c.tank_c[a] + c.tank_h[a]) - p3[a];
        wall = fminf(wall, fminf(lo, hi));
    }
    const float vs = wi.st.dt * c.inv_h;
    const float s1 = c.inv_h * inv, s2 = s1 * c.inv_h, s3 = s2 * c.inv_h;
    cx *= c.inv_h;
    cy *= c.inv_h;
    cz *= c.inv_h;
    fv[BBX_F_DENSITY_ERR] = di / c.rho0 - 1.f;
    fv[BBX_F_RESERVED1] = 0.f;
    fv[BBX_F_COUNT] = (float)cnt;
    fv[BBX_F_M1] = m1 * s1;
    fv[BBX_F_M2] = m2 * s2;
    fv[BBX_F_M3] = m3 * s3;
    fv[BBX_F_CX] = cx * inv;
    fv[BBX_F_CY] = cy * inv;
    fv[BBX_F_CZ] = cz * inv;
    fv[BBX_F_CNORM] = sqrtf(fmaf(cz, cz, fmaf(cy, cy, cx * cx))) * inv;
    fv[BBX_F_PPREV] = wi.st.delta != 0.f ? vi.w / (wi.st.delta * c.rho0) : 0.f;
    fv[BBX_F_VY] = vi.y * vs;
    fv[BBX_F_VNORM] = sqrtf(vi.x * vi.x + vi.y * vi.y + vi.z * vi.z) * vs;
    fv[BBX_F_RESERVED2] = 0.f;
    fv[BBX_F_RESERVED3] = 0.f;
    fv[BBX_F_WALL] = fminf(fmaxf(wall * c.inv_h, 0.f), 4.f);
}

// Network pressures of a workgroup's kRows particles (thread t < kRows holds
// particle t's features): the feature rows go through LDS (over the staged
// candidates, which every thread has finished with) into the MFMA layout;
// the waves share the rows in 16-sample tiles.
// Returns the kRows pressures in LDS; the whole workgroup calls.
template <int kRows>
__device__ __forceinline__ const float *infer_block(const WarmIn &wi, float4 *sx, int row, bool valid,
                                                    const float *fv) {
    constexpr int kRow = BBX_NFEAT + 1;  // padded feature row
    constexpr int kTiles = kRows * 4 / kBlock;  // 16-sample tiles per wave
    constexpr int kT = kTiles > 1 ? 2 : 1;
    float *lf = reinterpret_cast<float *>(sx);  // feature rows
    float *lp = lf + kRows * kRow;              // warm-start pressures
    float *lb = lp + kRows;                     // b1 | b2 | w3
    unsigned short *lw = reinterpret_cast<unsigned short *>(lb + 3 * kH);  // BF16 weights of both layers
    static_assert((kRows * (kRow + 1) + 3 * kH) * 4 + kLdsWeights * 2 <= (int)sizeof(float4) * kTileCap &&
                      (kRows * (kRow + 1) + 3 * kH) % 4 == 0,
                  "warm-start LDS layout over the staged candidates");
    __syncthreads();
    if (row >= 0) {
#pragma unroll
        for (int f = 0; f < BBX_NFEAT; f++) lf[row * kRow + f] = valid ? fv[f] : 0.f;
    }
    stage_infer_weights(wi.P, lw, lb, (int)threadIdx.x, kBlock);
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int qq = lane >> 4, jj = lane & 15;
    bf16x4 w1[4], w2[4][4];
    load_weight_operands_lds(lw, lane, w1, w2);
    float mean[4], istd[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
        mean[v] = wi.P[OFF_MEAN + 4 * qq + v];
        istd[v] = wi.P[OFF_ISTD + 4 * qq + v];
    }
    const float b3 = wi.P[OFF_B3], oscale = wi.P[OFF_OSCALE], alpha = wi.P[OFF_ALPHA];
    const float pcap = wi.P[OFF_PCAP], resid = wi.P[OFF_RESID];
#pragma unroll
    for (int part = 0; part < kTiles / kT; part++) {  // pairs of tiles keep the registers below 128
        float xv[kT][4];
#pragma unroll
        for (int t = 0; t < kT; t++) {
            const int smp = (wv * kTiles + kT * part + t) * 16 + jj;
#pragma unroll
            for (int v = 0; v < 4; v++) xv[t][v] = lf[smp * kRow + 4 * qq + v];
        }
        float yn[kT];
        forward_infer_tiles<kT>(w1, w2, lb, lb + kH, lb + 2 * kH, b3, xv, mean, istd, qq, yn);
        if (lane < 16) {
#pragma unroll
            for (int t = 0; t < kT; t++) {
                const int smp = (wv * kTiles + kT * part + t) * 16 + jj;
                // the same expression as the standalone inference kernel
                float y = yn[t] * oscale;
                if (resid != 0.f) y += resid * lf[smp * kRow + BBX_F_PPREV];
                y = alpha * fminf(fmaxf(y, 0.f), pcap);
                lp[smp] = y * wi.st.warm_scale;
            }
        }
    }
    __syncthreads();
    return lp;
}

// PredictVelocityAndPositionFor at k = 0 (src/equations/pcisph_equations3.cpp:3-28)
// with the network's pressure p instead of 0: rho* = rho, p = p0
__device__ __forceinline__ void warm_start_one(const WarmIn &wi, int i, float4 pi, float di, float p,
                                               float *__restrict__ pres) {
    const float d2 = di * di;
    pres[i] = p;
    wi.pwarm[i] = p;
    wi.rho_star[i] = di;
    wi.xq[i] = make_float4(pi.x, pi.y, pi.z, (fabsf(d2) < 1e-8f) ? 0.f : p / d2);
}

// Up to kOwnTables particles -- four workgroups on every CU, all resident at
// once -- the tables cost one workgroup's latency instead of a launch; above,
// every round of workgroups would pay it.  Bucket kernel + table kernel / with
// own tables (us): 30.5 + 5.6 / 31.8 at 94k, 65.5 + 5.4 / 66.9 at 255k,
// 178.0 + 6.0 / 186.4 at 1M, 224.4 + 6.0 / 235.9 there with the network.
constexpr int kOwnTables = 4 * 256 * kBlock;
// kOwnTab: the first wave makes the tile's table here, beside the row-bound
// loads, instead of a launch before this one.
template <bool kPressure, int kFeat, bool kOwnTab>
__global__ void __launch_bounds__(kBlock) k_buckets_density(SimConst c,
                                                            const float4 *__restrict__ pos,
                                                            const int *__restrict__ home,
                                                            const int *__restrict__ start,
                                                            unsigned short *__restrict__ nbr16,
                                                            int *__restrict__ nbr32,
                                                            int *__restrict__ nbr_cnt,
                                                            float *__restrict__ rho,
                                                            float *__restrict__ pres,
                                                            int *__restrict__ tile_tab,
                                                            int *__restrict__ counters,
                                                            WarmIn wi) {
    // staged candidate positions (16-byte LDS DMA); eight slack slots let
    // the candidate test read whole groups of four, and the group after
    // them, past the end of a row
    __shared__ float4 sx[kTileCap + 8];
    __shared__ TileTab tt;
    const int tile = tile_of_block();
    // The tile table is read first, into each wave's lanes: the staging
    // below then waits for nothing but it, not for the row bounds requested
    // in between, and needs no workgroup barrier (the LDS copy that the rest
    // of the kernel reads is visible after the barrier behind the staging).
    const int tw = kOwnTab ? 0 : tab_load_wave(tile_tab + (size_t)tile * kTabInts);
    const int i = tile * kBlock + threadIdx.x;
    const bool valid = i < c.n;
    const int hc = valid ? home[i] : -1;
    // The particle's position and its nine row bounds do not depend on the
    // tile table or the staging: they are requested first.  Row r =
    // (dz+1)*3 + (dy+1): the cells x-1, x, x+1 of a row are contiguous in
    // storage; A[r] = storage start of cell x-1, and O[r] packs the offsets
    // of cells x-1 (zero), x, x+1 and of the row end as bytes 0-3 (rows
    // outside the grid are empty).  A row of at most 64 candidates whose cells hold at most 32
    // each is "narrow": it is tested into a bit mask; otherwise the particle
    // walks cell by cell.
    const int nx = c.g.n[0], ny = c.g.n[1], nz = c.g.n[2], nxy = nx * ny;
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
    int u[3] = {0, 0, 0};
    int A[9];
    unsigned O[9];
    bool narrow = true;
#pragma unroll
    for (int r = 0; r < 9; r++) {
        A[r] = 0;
        O[r] = 0u;
    }
    if (valid) pi = pos[i];
    // All 36 row-bound loads are issued before any is used (indices clamped
    // into start[0 .. total]; rows outside the grid and cells past the x
    // bounds read a valid word and ignore it), and the staging is issued
    // behind them, so the latencies overlap instead of following one another
    // row by row.
    int b[9][4];
    if (hc >= 0) {
        unlinear_fast(c.g, c.inv_nx, c.inv_nxy, hc, u);
        const int last = (int)c.g.total;
#pragma unroll
        for (int r = 0; r < 9; r++) {
            const int yy = u[1] + (r % 3) - 1, zz = u[2] + (r / 3) - 1;
            const bool in = yy >= 0 && yy < ny && zz >= 0 && zz < nz;
            const int cx = in ? u[0] + yy * nx + zz * nxy : 0;
#pragma unroll
            for (int q = 0; q < 4; q++) b[r][q] = start[min(max(cx - 1 + q, 0), last)];
        }
    }
    bool staged;
    if constexpr (kOwnTab) {
        if (threadIdx.x < 64) tile_table(c, home, start, tile, (int)threadIdx.x, tt);
        __syncthreads();
        staged = tt.staged != 0;
        if (staged) tab_stage_dma(tt, [&](int j, int e) { lds_dma16(pos + j, sx + e); });
        tab_store(tile_tab + (size_t)tile * kTabInts, tt);
    } else {
        if (threadIdx.x < kTabWords) reinterpret_cast<int *>(&tt)[threadIdx.x] = tw;
        staged = tab_word(tw, 1) != 0;
        if (staged) tab_stage_dma_wave(tw, [&](int j, int e) { lds_dma16(pos + j, sx + e); });
    }
    if (hc >= 0) {
#pragma unroll
        for (int r = 0; r < 9; r++) {
            const int yy = u[1] + (r % 3) - 1, zz = u[2] + (r / 3) - 1;
            if (yy >= 0 && yy < ny && zz >= 0 && zz < nz) {
                const int b1 = b[r][1], b2 = b[r][2];
                const int b0 = u[0] > 0 ? b[r][0] : b1;
                const int b3 = u[0] + 1 < nx ? b[r][3] : b2;
                A[r] = b0;
                O[r] = ((unsigned)(b1 - b0) << 8) | ((unsigned)(b2 - b0) << 16) | ((unsigned)(b3 - b0) << 24);
                narrow = narrow && (b3 - b0 <= c.row_max) && (b1 - b0 <= 32) && (b2 - b1 <= 32) &&
                         (b3 - b2 <= 32);
            }
        }
    }
    lds_dma_wait();
    __syncthreads();
    if (kFeat != 2 && !valid) return;  // the inference below needs the whole block at its barriers
    float fv[kFeat ? BBX_NFEAT : 1];
    float di = 0.f;
    // The particle's work is instantiated once for LDS-staged and once for
    // global-memory tiles, so no load selects between the two address spaces
    // (that would compile to a slower generic load).
    auto per_particle = [&](auto staged_tag) {
        constexpr bool kStaged = decltype(staged_tag)::value;
        float sum = 0.f, comp = 0.f;
        float m1 = 0.f, m2 = 0.f, m3 = 0.f, cx = 0.f, cy = 0.f, cz = 0.f;  // features
        BucketWriter<kStaged> bw{nbr16, nbr32, c.stride, i};
        if (hc >= 0) {
            int sh[9];
#pragma unroll
            for (int r = 0; r < 9; r++) sh[r] = kStaged ? tt.rdelta[r] : 0;
            bool emitted = false;
            if (narrow) {
                // Pass 1: each row's candidates into an acceptance mask
                unsigned long long M[9];
                int total = 0;
#pragma unroll
                for (int r = 0; r < 9; r++) {
                    const unsigned long long m =
                        row_mask<kStaged>(c, pi, sx + A[r] + sh[r], pos, A[r], (int)(O[r] >> 24));
                    M[r] = m;
                    total += __popcll(m);
                }
                // Pass 2: emit in the reference's order, cells (y, x, z), chain
                // order inside each cell.  x runs as a loop with its cell bounds
                // selected, which keeps the kernel's code (nine emission sites
                // instead of 27) small.  A narrow row's cells hold <= 32
                // candidates, so each cell's bits fit one 32-bit word.  The
                // bucket cap cannot bind here (a lane over it takes the
                // cell-by-cell path below, which truncates).
                if (total <= kBucket) {
                    emitted = true;
#pragma unroll
                    for (int dy = 0; dy < 3; dy++)
#pragma unroll 1
                        for (int dx = 0; dx < 3; dx++)
#pragma unroll
                            for (int dz = 0; dz < 3; dz++) {
                                const int r = dz * 3 + dy;
                                const int lo = (int)__builtin_amdgcn_ubfe(O[r], 8 * dx, 8);
                                const int hi = (int)__builtin_amdgcn_ubfe(O[r], 8 * dx + 8, 8);
                                const int w = hi - lo;
                                if (w <= 0) continue;
                                unsigned m = (unsigned)(M[r] >> lo);
                                if (w < 32) m = __builtin_amdgcn_ubfe(m, 0, w);
                                while (m) {
                                    const int b = __builtin_ctz(m);
                                    m &= m - 1u;
                                    bw.append(A[r] + lo + b, sh[r]);
                                }
                            }
                }
            }
            // a wide row, a crowded cell or a bucket over the cap
            if (!emitted) walk_cells<kStaged>(c, pi, u, start, sx, pos, sh, bw);
        }
        bw.finish();
        const int cnt = bw.cnt;
        // ComputeDensityFor over the bucket in bucket order, read back from
        // the table this lane has just written (its own quads: no other lane
        // or wave writes them, and no earlier load in this kernel cached them)
        __builtin_amdgcn_s_waitcnt(0);
        // The particle's own index (its LDS slot in the centre row: a staged
        // tile's particles with neighbours are all candidates).  Dead
        // entries of the last quad read the particle itself: its staged copy
        // is its position bit for bit, so they add exact zeros to the
        // feature sums below, as the particle's own entry does, and only
        // the density masks them.
        const int self = kStaged ? (i + tt.rdelta[4]) << kSlotShift : i;
        for_each_neighbour_dead<kNbrDepth>(nbr16, nbr32, kStaged, i, cnt, c.stride, [&](int j, bool live) {
            const float4 pj = kStaged ? lds_at(sx, j) : pos[j];
            const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const float d2 = dx * dx + dy * dy + dz * dz;
            const float w = poly6_w_member(c, d2);
            kahan_add(sum, comp, live ? w : 0.f);  // a dead entry adds an exact zero
            if constexpr (kFeat > 0) {
                // distance moments r, r^2, r^3 and the centroid offset over
                // the members (powers of 1/h applied once afterwards)
                const float r = fast_sqrt(d2);
                m1 += r;
                m2 += d2;
                m3 = fmaf(r, d2, m3);
                cx -= dx;
                cy -= dy;
                cz -= dz;
            }
        }, self);
        nbr_cnt[i] = cnt;
        di = sum * c.mass;
        rho[i] = di;
        if constexpr (kFeat > 0) {
            finish_features(c, wi, i, pi, di, cnt, m1, m2, m3, cx, cy, cz, fv);
            if (kFeat == 1 || wi.store_feat) {
                const size_t S = (size_t)c.stride;
#pragma unroll
                for (int f = 0; f < BBX_NFEAT; f++) wi.feat[(size_t)f * S + i] = fv[f];
            }
        }
        float p = 0.f;
        if (kPressure) {
            p = tait_pressure(c, di);
            pres[i] = p;
        }
        // the positions of the pressure-force gather; q follows
        if (kFeat != 2) wi.xq[i] = make_float4(pi.x, pi.y, pi.z, kPressure ? p / (di * di) : 0.f);
        const float4 vo = wi.vel[i];
        wi.vr[i] = make_float4(vo.x, vo.y, vo.z, fast_rcp(di));
        if (bw.dropped) atomicAdd(&counters[CNT_OVERFLOW], bw.dropped);
    };
    if (valid) with_staging(staged, per_particle);
    if constexpr (kFeat == 2) {
        const float *lp = infer_block<kBlock>(wi, sx, (int)threadIdx.x, valid, fv);
        if (valid) warm_start_one(wi, i, pi, di, lp[threadIdx.x], pres);
    }
}

// The same with four lanes per particle and four workgroups per tile, for
// sets that leave the chip idle otherwise: the kernel above is one long chain
// per lane (nine rows of tests, the emission, the sum), 26 us for 2k
// particles however few tiles there are.  Each lane of a particle takes rows
// lane, lane + 4, lane + 8; the lanes exchange the cells' counts, so that
// each knows where its entries go, and emit into LDS; then each evaluates
// (and writes out) every fourth quad.  A workgroup stages its tile's candidates
// like the others, so tile tables and entries are the same.  A particle with
// a crowded row or more neighbours than the cap is walked cell by cell by its
// first lane.
//
// Used up to kSmallSet.  Measured (us, one lane per particle / four): 25.2 / 12.9
// at 2k, 27.2 / 15.0 at 16k, 30.2 / 25.6 at 35k, 28.6 / 27.1 at 49k, 29.0 / 28.7
// at 58k, 29.0 / 30.8 at 65k, 31.8 / 40.0 at 94k, 66.9 / 121.8 at 255k, where
// the chip is full and the four workgroups' staging and the longer emission
// count.
constexpr int kSplitLanes = 4;
constexpr int kSplitRows = kBlock / kSplitLanes;  // particles per workgroup
constexpr int kSplitMax = kBucket;                // bucket entries held in LDS
constexpr int kSplitStride = kSplitMax / 2 + 1;   // words per particle (odd: its lanes spread over the banks)

// value of lane k of the own group of four / of the lane across the mask
template <int k>
__device__ __forceinline__ int quad_lane(int v) {
    return __builtin_amdgcn_mov_dpp(v, k * 0x55, 0xf, 0xf, true);
}
__device__ __forceinline__ int quad_xor1(int v) { return __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, true); }
__device__ __forceinline__ int quad_xor2(int v) { return __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, true); }
template <int k>
__device__ __forceinline__ float quad_lane_f(float v) {
    return __int_as_float(quad_lane<k>(__float_as_int(v)));
}

template <bool kPressure, int kFeat>
__global__ void __launch_bounds__(kBlock) k_buckets_density_split(SimConst c,
                                                                  const float4 *__restrict__ pos,
                                                                  const int *__restrict__ home,
                                                                  const int *__restrict__ start,
                                                                  unsigned short *__restrict__ nbr16,
                                                                  int *__restrict__ nbr32,
                                                                  int *__restrict__ nbr_cnt,
                                                                  float *__restrict__ rho,
                                                                  float *__restrict__ pres,
                                                                  int *__restrict__ tile_tab,
                                                                  int *__restrict__ counters,
                                                                  WarmIn wi) {
    __shared__ float4 sx[kTileCap + 8];
    __shared__ unsigned ent[kSplitRows][kSplitStride];  // buckets of a staged tile, two entries a word
    __shared__ TileTab tt;
    const int unit = tile_of_block();
    const int tile = unit / kSplitLanes, part = unit % kSplitLanes;
    const int pl = threadIdx.x / kSplitLanes, sub = threadIdx.x % kSplitLanes;
    const int i = tile * kBlock + part * kSplitRows + pl;
    const bool valid = i < c.n;
    const int hc = valid ? home[i] : -1;
    const int nx = c.g.n[0], ny = c.g.n[1], nz = c.g.n[2], nxy = nx * ny;
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid) pi = pos[i];
    int u[3] = {0, 0, 0};
    // slot k holds row r = sub + 4k (k < 3, r < 9): bounds as in the kernel above
    int A[3] = {0, 0, 0};
    unsigned O[3] = {0u, 0u, 0u};
    int b[3][4];
    int wide = 0;
    if (hc >= 0) {
        unlinear_fast(c.g, c.inv_nx, c.inv_nxy, hc, u);
        const int last = (int)c.g.total;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const int r = sub + 4 * k;
            const int yy = u[1] + (r % 3) - 1, zz = u[2] + (r / 3) - 1;
            const bool in = r < 9 && yy >= 0 && yy < ny && zz >= 0 && zz < nz;
            const int cx = in ? u[0] + yy * nx + zz * nxy : 0;
#pragma unroll
            for (int q = 0; q < 4; q++) b[k][q] = start[min(max(cx - 1 + q, 0), last)];
        }
    }
    // The tile's table, by the first wave while the loads above are under way
    // (a kernel of its own takes 4.9 us); the later gathers read it from the
    // first part's copy.
    if (threadIdx.x < 64) tile_table(c, home, start, tile, (int)threadIdx.x, tt);
    __syncthreads();
    const bool staged = tt.staged != 0;
    if (staged) tab_stage_dma(tt, [&](int j, int e) { lds_dma16(pos + j, sx + e); });
    if (part == 0) tab_store(tile_tab + (size_t)tile * kTabInts, tt);
    if (hc >= 0) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const int r = sub + 4 * k;
            const int yy = u[1] + (r % 3) - 1, zz = u[2] + (r / 3) - 1;
            if (r < 9 && yy >= 0 && yy < ny && zz >= 0 && zz < nz) {
                const int b1 = b[k][1], b2 = b[k][2];
                const int b0 = u[0] > 0 ? b[k][0] : b1;
                const int b3 = u[0] + 1 < nx ? b[k][3] : b2;
                A[k] = b0;
                O[k] = ((unsigned)(b1 - b0) << 8) | ((unsigned)(b2 - b0) << 16) | ((unsigned)(b3 - b0) << 24);
                wide |= b3 - b0 > c.row_max || b1 - b0 > 32 || b2 - b1 > 32 || b3 - b2 > 32;
            }
        }
    }
    wide |= quad_xor1(wide);
    wide |= quad_xor2(wide);
    lds_dma_wait();
    __syncthreads();
    if (kFeat != 2 && !valid) return;  // the inference below needs the whole block at its barriers
    float fv[kFeat ? BBX_NFEAT : 1];
    float di = 0.f;
    // an unstaged tile's buckets: storage indices, in the candidates' place
    static_assert(kSplitRows * (kSplitMax + 1) * sizeof(int) <= sizeof(sx), "unstaged buckets in LDS");
    int *const far = reinterpret_cast<int *>(sx) + pl * (kSplitMax + 1);
    auto per_particle = [&](auto staged_tag) {
        constexpr bool kStaged = decltype(staged_tag)::value;
        int cnt = 0, dropped = 0;
        bool in_lds = false;
        if (hc >= 0 && !wide) {
            // acceptance masks and the accepted candidates of each cell, a byte a cell
            unsigned long long M[3];
            int P[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const int r = sub + 4 * k;
                M[k] = row_mask<kStaged>(c, pi, sx + A[k] + (kStaged && r < 9 ? tt.rdelta[r] : 0), pos, A[k], (int)(O[k] >> 24));
                const int b1 = (O[k] >> 8) & 0xff, b2 = (O[k] >> 16) & 0xff;
                // b1 <= 32 and b2 <= 64; a shift by 64 is not defined
                const unsigned long long from2 = b2 < 64 ? M[k] >> b2 : 0ull;
                const int c0 = __popcll(M[k] & ((1ull << b1) - 1ull)), c2 = __popcll(from2);
                P[k] = c0 | (__popcll(M[k]) - c0 - c2) << 8 | c2 << 16;
            }
            // every row's counts; r = dz * 3 + dy
            const int R[9] = {quad_lane<0>(P[0]), quad_lane<1>(P[0]), quad_lane<2>(P[0]),
                              quad_lane<3>(P[0]), quad_lane<0>(P[1]), quad_lane<1>(P[1]),
                              quad_lane<2>(P[1]), quad_lane<3>(P[1]), quad_lane<0>(P[2])};
            // the bucket's order is cells (y, x, z): where each row's three
            // cells begin, a byte a cell (read only where the total is within
            // the cap, so that every sum fits)
            int at[9], total = 0;
#pragma unroll
            for (int dy = 0; dy < 3; dy++) {
                const int S = R[dy] + R[3 + dy] + R[6 + dy];
                const int X = total * 0x010101 + ((S << 8) & 0xffff00) + ((S << 16) & 0xff0000);
                at[dy] = X;
                at[3 + dy] = X + R[dy];
                at[6 + dy] = X + R[dy] + R[3 + dy];
                total += (S & 0xff) + ((S >> 8) & 0xff) + ((S >> 16) & 0xff);
            }
            if (total <= kSplitMax) {
                in_lds = true;
                cnt = total;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    const int lo = sub & 1 ? at[min(4 * k + 1, 8)] : at[4 * k], hi = sub & 1 ? at[min(4 * k + 3, 8)] : at[min(4 * k + 2, 8)];
                    int to = sub & 2 ? hi : lo;
                    const int r = sub + 4 * k;
                    const int slot0 = A[k] + (kStaged && r < 9 ? tt.rdelta[r] : 0);
                    const int b1 = (O[k] >> 8) & 0xff, b2 = (O[k] >> 16) & 0xff;
                    unsigned long long m = M[k];
                    while (m) {
                        const int t = __builtin_ctzll(m);
                        m &= m - 1ull;
                        const int sh = t < b1 ? 0 : (t < b2 ? 8 : 16);
                        if (kStaged)
                            reinterpret_cast<unsigned short *>(ent[pl])[(to >> sh) & 0xff] =
                                (unsigned short)((slot0 + t) << kSlotShift);
                        else
                            far[(to >> sh) & 0xff] = slot0 + t;
                        to += 1 << sh;
                    }
                }
            }
        }
        if (!in_lds && sub == 0) {
            int sh[9];
#pragma unroll
            for (int r = 0; r < 9; r++) sh[r] = kStaged ? tt.rdelta[r] : 0;
            BucketWriter<kStaged> bw{nbr16, nbr32, c.stride, i};
            if (hc >= 0) walk_cells<kStaged>(c, pi, u, start, sx, pos, sh, bw);
            bw.finish();
            cnt = bw.cnt;
            dropped = bw.dropped;
        }
        cnt = quad_lane<0>(cnt);
        // the wave's entries are in LDS, its stores in the cache below
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // density (and features) over quads sub, sub + 4, ... of the bucket;
        // dead entries read the particle itself, as in the kernel above
        float sum = 0.f, comp = 0.f;
        float m1 = 0.f, m2 = 0.f, m3 = 0.f, cx = 0.f, cy = 0.f, cz = 0.f;
        const int self = kStaged ? (i + tt.rdelta[4]) << kSlotShift : i;
        for (int q0 = 0; 4 * q0 < cnt; q0 += kSplitLanes) {
            const int q = q0 + sub, rem = cnt - 4 * q;
            int4 e = make_int4(self, self, self, self);
            if (rem <= 0) {
                // a lane past the last quad adds zeros below
            } else if (in_lds) {  // unused slots of the last quad as in BucketWriter
                if (kStaged) {
                    constexpr unsigned kTop = kFarEntry << 16;
                    unsigned w0 = ent[pl][2 * q], w1 = ent[pl][2 * q + 1];
                    w0 = rem > 1 ? w0 : (w0 & 0xffffu) | kTop;
                    w1 = rem > 3 ? w1 : (rem > 2 ? w1 & 0xffffu : kFarEntry) | kTop;
                    reinterpret_cast<uint2 *>(nbr16)[(size_t)q * c.stride + i] = make_uint2(w0, w1);
                    e = quad_unpack(make_int4((int)w0, (int)w1, 0, 0), true);
                } else {
                    const int *f = far + 4 * q;
                    e = make_int4(f[0], rem > 1 ? f[1] : 0, rem > 2 ? f[2] : 0, rem > 3 ? f[3] : 0);
                    reinterpret_cast<int4 *>(nbr32)[(size_t)q * c.stride + i] = e;
                }
            } else {
                e = quad_unpack(nbr_quad(nbr16, nbr32, kStaged, i, c.stride, q), kStaged);
            }
            const int j4[4] = {e.x, rem > 1 ? e.y : self, rem > 2 ? e.z : self, rem > 3 ? e.w : self};
            float w[4], d2[4], dx[4], dy[4], dz[4];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float4 pj = kStaged ? lds_at(sx, j4[v]) : pos[j4[v]];
                dx[v] = pi.x - pj.x;
                dy[v] = pi.y - pj.y;
                dz[v] = pi.z - pj.z;
                d2[v] = dx[v] * dx[v] + dy[v] * dy[v] + dz[v] * dz[v];
                const float m = poly6_w_member(c, d2[v]);
                w[v] = v < rem ? m : 0.f;  // a dead entry adds an exact zero
            }
            // The terms are the lanes'; the sums run in bucket order, each
            // lane the same one, so that they are those of the kernel above
            // bit for bit.
            auto add_quad = [&](auto lane) {
                constexpr int L = decltype(lane)::value;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    kahan_add(sum, comp, quad_lane_f<L>(w[v]));
                    if constexpr (kFeat > 0) {
                        const float dd = quad_lane_f<L>(d2[v]), r = fast_sqrt(dd);
                        m1 += r;
                        m2 += dd;
                        m3 = fmaf(r, dd, m3);
                        cx -= quad_lane_f<L>(dx[v]);
                        cy -= quad_lane_f<L>(dy[v]);
                        cz -= quad_lane_f<L>(dz[v]);
                    }
                }
            };
            add_quad(std::integral_constant<int, 0>{});
            add_quad(std::integral_constant<int, 1>{});
            add_quad(std::integral_constant<int, 2>{});
            add_quad(std::integral_constant<int, 3>{});
        }
        di = sum * c.mass;
        if (sub == 0) {
            nbr_cnt[i] = cnt;
            rho[i] = di;
            if constexpr (kFeat > 0) {
                finish_features(c, wi, i, pi, di, cnt, m1, m2, m3, cx, cy, cz, fv);
                if (kFeat == 1 || wi.store_feat) {
                    const size_t S = (size_t)c.stride;
#pragma unroll
                    for (int f = 0; f < BBX_NFEAT; f++) wi.feat[(size_t)f * S + i] = fv[f];
                }
            }
            float p = 0.f;
            if (kPressure) {
                p = tait_pressure(c, di);
                pres[i] = p;
            }
            if (kFeat != 2) wi.xq[i] = make_float4(pi.x, pi.y, pi.z, kPressure ? p / (di * di) : 0.f);
            const float4 vo = wi.vel[i];
            wi.vr[i] = make_float4(vo.x, vo.y, vo.z, fast_rcp(di));
            if (dropped) atomicAdd(&counters[CNT_OVERFLOW], dropped);
        }
    };
    if (valid) with_staging(staged, per_particle);
    if constexpr (kFeat == 2) {
        const float *lp = infer_block<kSplitRows>(wi, sx, sub == 0 ? pl : -1, valid, fv);
        if (valid && sub == 0) warm_start_one(wi, i, pi, di, lp[pl], pres);
    }
}

// density over the existing buckets (after an upload of positions)
__global__ void __launch_bounds__(kBlock) k_density(SimConst c, const float4 *__restrict__ pos,
                                                    const unsigned short *__restrict__ nbr16,
                                                    const int *__restrict__ nbr32,
                                                    const int *__restrict__ nbr_cnt,
                                                    const int *__restrict__ tile_tab,
                                                    float *__restrict__ rho) {
    __shared__ float4 sx[kFarSlot + 1];
    __shared__ TileTab tt;
    const int tile = tile_of_block();
    tab_load_shared(tile_tab + (size_t)tile * kTabInts, tt);
    if (threadIdx.x == 0) sx[kFarSlot] = far_particle(0.f);
    __syncthreads();
    const bool staged = tt.staged != 0;
    if (staged) tab_stage(tt, sx, [&](int j) { return pos[j]; });
    __syncthreads();
    const int i = tile * kBlock + threadIdx.x;
    if (i >= c.n) return;
    const float4 pi = pos[i];
    float sum = 0.f, comp = 0.f;
    const int cnt = nbr_cnt[i];
    with_staging(staged, [&](auto tag) {
        constexpr bool kS = decltype(tag)::value;
        for_each_neighbour<2>(nbr16, nbr32, kS, i, cnt, c.stride, [&](int j, bool live) {
            const float4 pj = kS ? lds_at(sx, j) : pos[j];
            float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            const float w = poly6_w(c, dx * dx + dy * dy + dz * dz);
            kahan_add(sum, comp, live ? w : 0.f);  // a dead entry adds an exact zero
        });
    });
    rho[i] = sum * c.mass;
}

static unsigned nblocks(int n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// UpdateGridDistribution: full or incremental chain update, then buckets.
int distribute_grid(bbx_solver *s, bool force_full, int append_from, int *clear, size_t clear_n) {
    SimConst &c = s->sc;
    const int n = s->n;
    const size_t cells = (size_t)c.g.total + 1;
    if (n == 0) {
        BBX_CHECK(launch_fill_int(s, s->counters, 0, CNT_N));
        return clear_n ? launch_fill_int(s, clear, 0, clear_n) : BBX_OK;
    }
    // From the bins where the solver has them (grids of up to kBinCells cells,
    // or one per particle): one launch less, and no index to follow.  Scatter
    // and rank through the index / rank from the bins (us): 2.6 + 5.3 / 3.4
    // at 2k, 2.4 + 5.7 / 4.2 at 16k, 2.8 + 7.2 / 4.4 at 94k, 3.1 + 9.4 / 7.1 at
    // 255k, 5.3 + 20.0 / 21.3 at 1M (where the hash gains 1.8).  A grid with
    // many more cells than particles would pay for its bins in memory.
    const bool bins = s->bins != nullptr;
    // the pass leaves the counts at zero; not so before the first one, or
    // behind one that did not get that far
    if (!s->counts_clear) BBX_CHECK(launch_fill_int(s, s->cell_count, 0, cells));
    s->counts_clear = false;
    BinKeys bk{};
    if (bins) {
        const size_t nblk = bin_blocks((size_t)s->stride);
        if (s->bin_pass == 0 || s->bin_pass + 1 == 1u << kTagPassBits) {  // the table holds nothing yet, or any pass
            BBX_CHECK(launch_fill_int(s, reinterpret_cast<int *>(s->blocks), 0, 2 * nblk));
            s->bin_pass = 0;
        }
        bk = BinKeys{s->bins, s->blocks, s->blocks + nblk, s->tmp_idx, (unsigned)nblk, ++s->bin_pass};
    }
    const PassEnd end{s->cell_count, cells, s->flag, force_full ? 1 : 0, append_from >= 0 ? 1 : 0, s->counters,
                      clear, clear_n};
    const unsigned end_blocks = (unsigned)((std::max({(size_t)n, cells, clear_n}) + kBlock - 1) / kBlock);
    {
        BBX_PROF_BEGIN("grid_hash");
        (bins ? k_hash<true> : k_hash<false>)<<<nblocks(n), kBlock, 0, s->stream>>>(
            c, s->posA, s->cellA, s->flag, force_full ? 1 : 0, append_from, s->newc, s->hash_tmp, s->key,
            s->cell_count, s->rank_tmp, bk);
        BBX_HIP_CHECK(hipGetLastError());
        BBX_PROF_END();
    }
    {
        BBX_PROF_BEGIN("grid_scan");
        BBX_CHECK(launch_scan(s, s->cell_count, s->cell_start, cells));
        BBX_PROF_END();
    }
    if (!bins) {
        BBX_PROF_BEGIN("grid_scatter");
        k_scatter<<<end_blocks, kBlock, 0, s->stream>>>(c, s->newc, s->rank_tmp, s->cell_start, s->tmp_idx, end);
        BBX_HIP_CHECK(hipGetLastError());
        BBX_PROF_END();
    }
    {
        BBX_PROF_BEGIN("grid_rank_move");
        if (bins) {
            k_rank_bins<<<end_blocks, kBlock, 0, s->stream>>>(c, s->newc, s->hash_tmp, s->key, s->cell_start, bk,
                                                              s->posA, s->velA, s->posB, s->velB, s->cellB, s->home,
                                                              end);
        } else {
            k_rank_move<<<nblocks(n), kBlock, 0, s->stream>>>(c, s->tmp_idx, s->newc,
                                                              s->hash_tmp, s->key, s->cell_start,
                                                              s->posA, s->velA, s->posB,
                                                              s->velB, s->cellB, s->home);
        }
        BBX_HIP_CHECK(hipGetLastError());
        s->counts_clear = true;
        BBX_PROF_END();
    }
    std::swap(s->posA, s->posB);
    std::swap(s->velA, s->velB);
    std::swap(s->cellA, s->cellB);
    return BBX_OK;
}

int build_buckets(bbx_solver *s, bool with_pressure, int feat_mode, const StepConst *st) {
    if (feat_mode && (with_pressure || !st))
        return fail(BBX_E_INVALID, "warm-start features need a PCISPH bucket build and step constants");
    if (feat_mode == 2 && !s->mlp) return fail(BBX_E_INVALID, "no MLP attached");
    SimConst &c = s->sc;
    const int n = s->n;
    if (n > 0) {
        if (n > kOwnTables) {  // smaller sets' bucket kernels make their own
            BBX_PROF_BEGIN("tile_tables");
            k_tile_tables<<<(unsigned)((s->ntiles + kTabWaves - 1) / kTabWaves), kBlock, 0, s->stream>>>(
                c, s->home, s->cell_start, s->ntiles, s->tile_tab);
            BBX_HIP_CHECK(hipGetLastError());
            BBX_PROF_END();
        }
        WarmIn wi{};
        if (st) wi.st = *st;
        wi.vel = s->velA;
        wi.vr = s->vr ? s->vr : s->velB;  // velB is free until the integration writes it
        wi.store_feat = s->keep_features;
        wi.feat = s->feat;
        wi.P = feat_mode == 2 ? mlp_params_device(s->mlp) : nullptr;
        wi.pwarm = s->pwarm;
        wi.rho_star = s->rho_star;
        wi.xq = s->xq;
        BBX_PROF_BEGIN(feat_mode == 2 ? "buckets_density_warm"
                                      : (feat_mode == 1 ? "buckets_density_features" : "buckets_density"));
#define BBX_BUCKETS(P, F)                                                                                     \
    if (n <= kSmallSet)                                                                                       \
        k_buckets_density_split<P, F><<<nblocks(n) * kSplitLanes, kBlock, 0, s->stream>>>(                    \
            c, s->posA, s->home, s->cell_start, s->nbr16, s->nbr32, s->nbr_cnt, s->rho, s->pres, s->tile_tab, \
            s->counters, wi);                                                                                 \
    else                                                                                                      \
        (n <= kOwnTables ? k_buckets_density<P, F, true> : k_buckets_density<P, F, false>)                    \
            <<<nblocks(n), kBlock, 0, s->stream>>>(                                                           \
            c, s->posA, s->home, s->cell_start, s->nbr16, s->nbr32, s->nbr_cnt, s->rho, s->pres, s->tile_tab, \
            s->counters, wi)
        if (with_pressure) {
            BBX_BUCKETS(true, 0);
        } else if (feat_mode == 2) {
            BBX_BUCKETS(false, 2);
        } else if (feat_mode == 1) {
            BBX_BUCKETS(false, 1);
        } else {
            BBX_BUCKETS(false, 0);
        }
#undef BBX_BUCKETS
        BBX_HIP_CHECK(hipGetLastError());
        BBX_PROF_END();
    }
    return BBX_OK;
}

int distribute(bbx_solver *s, bool force_full, bool buckets, bool with_pressure, int append_from,
               int feat_mode, const StepConst *st) {
    if (feat_mode && !buckets) return fail(BBX_E_INVALID, "warm-start features need a bucket build");
    BBX_CHECK(distribute_grid(s, force_full, append_from));
    return buckets ? build_buckets(s, with_pressure, feat_mode, st) : BBX_OK;
}

int run_density_only(bbx_solver *s) {
    if (s->n == 0) return BBX_OK;
    BBX_PROF_BEGIN("density");
    k_density<<<nblocks(s->n), kBlock, 0, s->stream>>>(s->sc, s->posA, s->nbr16, s->nbr32, s->nbr_cnt,
                                                        s->tile_tab, s->rho);
    BBX_HIP_CHECK(hipGetLastError());
    BBX_PROF_END();
    return BBX_OK;
}

}  // namespace bbx
