// route.hip -- token-to-expert permutation on one GPU (the intra-GPU form of
// the reference's EP dispatch metadata: route_build_body, src/prologue.cuh:
// 126-226; publish_counts_body :230-256; task_setup_body :269-498).
//
// P = tokens * topk (token, k) pairs.  Up to kRouteOneP pairs one workgroup does
// it all (route_one); above, three stream-ordered kernels (two where route_scan
// builds the histograms itself):
//   1. route_hist:    per chunk of pairs, an LDS histogram over experts.
//   2. route_scan:    one workgroup; per expert the exclusive prefix over chunks,
//                     the capped count, the exclusive prefix over experts
//                     (slot offsets), the work-item list (expert, first row),
//                     the big GEMMs' XCD unit ranges and the ticket order
//                     of L1's tail queues.
//   3. route_scatter: per chunk, a stable rank of every pair among the pairs of
//                     the same expert (wave ballots over the expert-id bits +
//                     an LDS prefix across waves), giving the canonical slot
//                     order = ascending pair index.  Writes perm[slot] and
//                     pair_pos[pair].
// Pairs whose id is outside [0, E) or whose rank is >= slot_capacity get
// pair_pos = -1 (reference: dropped at route_build_body, prologue.cuh:150-175).
#include "mm_kernels.h"

namespace mm {

__global__ void __launch_bounds__(kRouteThreads)
route_hist_kernel(const int64_t* __restrict__ topk_idx, int P, int E, int chunk,
                  int* __restrict__ chunk_hist) {
    __shared__ int hist[kMaxExperts];
    for (int i = threadIdx.x; i < E; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    const int base = blockIdx.x * chunk;
    const int end = min(base + chunk, P);
    for (int p = base + threadIdx.x; p < end; p += blockDim.x) {
        const int64_t e = topk_idx[p];
        if (e >= 0 && e < E) atomicAdd(&hist[(int)e], 1);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < E; i += blockDim.x)
        chunk_hist[(size_t)blockIdx.x * E + i] = hist[i];
}

// Block-wide exclusive scan of one int4 per thread, component by component
// (blockDim = kScanThreads); *total: the sums.
__device__ int4 block_exclusive_scan4(int4 v, int4* smem, int4* total) {
    constexpr int kWaves = kScanThreads / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto wave_scan = [&](int4 x, int n) {   // inclusive, over the first n lanes
        for (int d = 1; d < n; d <<= 1) {
            const int4 y = make_int4(__shfl_up(x.x, d, 64), __shfl_up(x.y, d, 64),
                                     __shfl_up(x.z, d, 64), __shfl_up(x.w, d, 64));
            if (lane >= d) {
                x.x += y.x;
                x.y += y.y;
                x.z += y.z;
                x.w += y.w;
            }
        }
        return x;
    };
    const int4 x = wave_scan(v, 64);
    if (lane == 63) smem[wave] = x;
    __syncthreads();
    const int4 t = wave_scan(smem[lane & (kWaves - 1)], kWaves);   // the waves' running sums
    const int prev = wave > 0 ? wave - 1 : 0, on = wave > 0;
    *total = make_int4(__shfl(t.x, kWaves - 1, 64), __shfl(t.y, kWaves - 1, 64),
                       __shfl(t.z, kWaves - 1, 64), __shfl(t.w, kWaves - 1, 64));
    return make_int4(on * __shfl(t.x, prev, 64) + x.x - v.x, on * __shfl(t.y, prev, 64) + x.y - v.y,
                     on * __shfl(t.z, prev, 64) + x.z - v.z, on * __shfl(t.w, prev, 64) + x.w - v.w);
}

// LDS of route_finish.
struct RouteSmem {
    int4 waves[kScanThreads / 64];
    int cuts[9];                       // the L1 XCD unit ranges
    int rows;                          // rows of the largest work item
    int ioff[kMaxExperts + 1];         // first item of each expert (+ the item count)
    int cnt[kMaxExperts];              // routed rows of each expert
    int off[kMaxExperts];              // first slot of each expert
    int cost[kMaxExperts];             // modelled cost of the experts before it
    uint8_t tnt[8][kQueueTail];        // token tiles of L1's tail units
};

struct RouteOut {
    int* counts;
    int* offsets;
    int* items;
    int* status;
};

// Everything the routing derives from the experts' pair counts: called by all
// kScanThreads threads of one workgroup, thread e holding expert e's pairs
// `run` (E <= kMaxExperts = kScanThreads).  The four running sums it needs
// (pairs, routed rows, items, modelled cost) follow from `run` alone, so one
// scan makes them all (measured on MI355X at T = 1, one scan each, thread 0
// summing the waves, and a 64-bit division for each XCD cut: routing 11.4 us in
// two launches, 6.5 in one with this).
__device__ void route_finish(RouteSmem& sh, int run, int P, int E, int cap, int m_tile,
                             int max_items, int nb1, int nb2, const RouteOut& o) {
    const int e = threadIdx.x;
    const int cnt = min(run, cap);   // 0 for e >= E
    if (e < E) {
        o.counts[e] = cnt;
        sh.cnt[e] = cnt;
    }
    // the status word of this launch (only this kernel sets its error bits;
    // thread 0 clears it before its own atomicOr below)
    if (e == 0) {
        o.status[0] = 0;
        sh.rows = 0;
    }
    // Work items: the expert's rows split evenly into ceil(cnt / m_tile)
    // items of at most m_tile rows (no item re-streams the expert's weights
    // for a small remainder).  The items of one expert then have equal token
    // tile counts, so the units that read one weight block run in lockstep
    // and all but the first take it from L2.  (Measured on MI355X at T =
    // 8192: splitting at 16-row multiples instead ran 2% less MFMA work but
    // its unequal items drifted apart; L1 fetched 9.30 vs 7.33 GB and the
    // layer took 4908-4943 vs 4841-4854 us.)  Record: (expert, first slot,
    // end slot, index within the expert | item count of the expert << 16),
    // the slots absolute (the expert's offset included), so that a GEMM unit
    // needs no offsets[] load after its item.
    const int nm = (cnt + m_tile - 1) / m_tile;
    const int sz = nm > 0 ? (cnt + nm - 1) / nm : 0;
    // XCD ranges of the big GEMMs' units (nb blocks per item; an expert's
    // nb * nm units are contiguous in the kernels' numbering).  Modelled cost
    // of one of the expert's units per k-step, in token-tile MFMA times:
    // max(9, 2 + token tiles of its largest item) -- the fixed per-step work
    // (barrier, conversions, operand reads) is worth ~2 token tiles and the
    // weight stream at the full-chip HBM rate ~9 (measured on MI355X: a
    // k-step costs ~0.33 us + 0.137 us per token tile without weight loads,
    // and a weight block's k-step streams in ~1.23 us).  XCD x starts where
    // the running cost crosses x/8 of the total (the same expert for L1 and
    // L2, whose costs differ by the factor nb); each range is then clamped to
    // its share of the grid, nb * max_items + 8 workgroups.  (The constants were
    // fitted before big_step spread its loads, on the bf16 path; the fp8 path
    // uses them too.)
    // An expert whose items big_unit runs as fewer units of up to 17 token tiles
    // is planned as its items here and in the tail order below: two units of
    // 9 tiles, say, for one of 17 and an empty one.  Planned as they run (measured on
    // MI355X, as it is vs the order alone vs the cuts as well, all even): T =
    // 8192 4168 vs 4173 vs 4167 us, Zipf(1.1) 4387 vs 4394 vs 4384, Zipf(1.1) T =
    // 2048 1834 vs 1837 vs 1831; fp8 path T = 8192 2876 vs 2871 vs 2880, Zipf(1.1)
    // 3098 vs 3096 vs 3086.
    const int uc = max(9, 2 + min((sz + 15) >> 4, kBigMaxTiles));
    const int w = nm * uc;
    __syncthreads();   // sh.rows
    if (sz > 0) atomicMax(&sh.rows, sz);   // ordered before the read by the scan's barrier
    int4 tot;
    const int4 pre = block_exclusive_scan4(make_int4(run, cnt, nm, w), sh.waves, &tot);
    // valid: pairs with an id in [0, E) before the slot cap (the rest of P had
    // ids outside [0, E))
    const int off = pre.y, ioff = pre.z, wpre = pre.w;
    const int valid = tot.x, slots = tot.y, nitems = tot.z, wtot = tot.w;
    if (e < E) {
        o.offsets[e] = off;
        sh.off[e] = off;
    }
    if (e == 0) o.offsets[E] = slots;
    for (int j = 0; j < nm; ++j) {
        const int it = ioff + j;
        if (it < max_items) {
            const int m0 = j * sz;
            reinterpret_cast<int4*>(o.items)[it] =
                make_int4(e, off + m0, off + min(cnt, m0 + sz), j | (nm << 16));
        }
    }
    if (threadIdx.x < 2 * kQueueInts) o.status[kQueueL1 + threadIdx.x] = 0;   // tail queues
    // per-item L1 ready counters of the fused L1 -> L2 launch (after the table)
    for (int i = threadIdx.x; i < max_items; i += kScanThreads) o.items[4 * max_items + i] = 0;
    if (e == 0) {
        o.status[1] = min(nitems, max_items);
        o.status[2] = slots;
        o.status[3] = valid - slots;   // pairs dropped by the slot capacity
        o.status[4] = P - valid;       // pairs whose expert id is outside [0, E)
        o.status[kStatusMaxRows] = sh.rows;
        if (nitems > max_items) atomicOr(&o.status[0], kStatusItemOverflow);
    }
    if (e < E) {
        sh.cost[e] = wpre;
        sh.ioff[e] = ioff;
    }
    if (e == 0) sh.ioff[E] = nitems;
    __syncthreads();
    // One thread per cut (XCD x of L1: threads 0-7, of L2: 8-15) finds the
    // expert that its target cost falls in: the last one whose running cost is
    // not above it (never an empty one: the next expert's is the same).
    if (e < 16) {
        const int g = e >> 3, x = e & 7, nb = g == 0 ? nb1 : nb2;
        const int n = min(nitems, max_items), units = nb * n, share = (nb * max_items + 8) / 8;
        // a target past the last complete expert (item overflow) cuts at the end
        int v = units;
        if (nitems <= max_items && n > 0) {
            const int64_t t = (int64_t)wtot * nb * x / 8;
            int lo = 0, hi = E - 1;
            while (lo < hi) {
                const int m = (lo + hi + 1) >> 1;
                if ((int64_t)sh.cost[m] * nb <= t) lo = m; else hi = m - 1;
            }
            const int c = sh.cnt[lo], cn = (c + m_tile - 1) / m_tile;
            const int cz = (c + cn - 1) / cn;
            const int ucl = max(9, 2 + min((cz + 15) >> 4, kBigMaxTiles));
            // below nb * nm * ucl of one expert: 32 bits
            v = nb * sh.ioff[lo] + (int)((uint32_t)(t - (int64_t)sh.cost[lo] * nb) / (uint32_t)ucl);
        }
        int* cuts = o.status + (g == 0 ? kCutsL1 : kCutsL2);
        int prev = 0, mine = 0;
#pragma unroll
        for (int y = 1; y < 8; ++y) {
            int c = __shfl(v, 8 * g + y, 64);
            c = min(max(c, prev), prev + share);
            c = max(c, units - (8 - y) * share);
            if (y == x) mine = c;
            prev = c;
        }
        cuts[x] = mine;
        if (x == 0) cuts[8] = units;
        if (g == 0) {
            sh.cuts[x] = mine;
            if (x == 0) sh.cuts[8] = units;
        }
    }
    // Ticket order of L1's tail queues (the last t = min(range, kQueueTail)
    // units of each XCD range; only a range of more than 2 * kQueueTail units
    // reads it): by the token tiles of the unit's item, descending, ties in unit
    // order, so that the units of heavy items do not start after light ones at
    // the end of the kernel (units of 17 tiles rank as their items, above).
    // Tail unit i of XCD x
    // is unit cuts[x + 1] - t + i; L1 runs ticket k as tail unit order[k]
    // (gemm_big.hip: claim_tail_unit).  One thread per tail slot finds its
    // unit's expert by binary search over the item offsets.  Only when some
    // item holds more than kTailOrderRows rows (skewed routing, T = 8192):
    // below, the units differ by a few token tiles at most, and the order is
    // the identity.  (Measured on MI355X: a loop over the 8 tails in every
    // expert thread added 10.6 us to this one-workgroup kernel; L2's tails
    // gained nothing from the order and keep ticket order.)
    uint8_t* order = reinterpret_cast<uint8_t*>(o.status + kTailOrdL1);
    __syncthreads();   // sh.cuts, and sh.rows of every expert
    if (sh.rows > kTailOrderRows) {   // uniform over the workgroup
        if (threadIdx.x < 8 * kQueueTail) {
            const int x = threadIdx.x / kQueueTail, i = threadIdx.x % kQueueTail;
            const int lo = sh.cuts[x], hi = sh.cuts[x + 1], t = min(hi - lo, kQueueTail);
            if (i < t) {
                const int u = hi - t + i, im = u / nb1;
                int a = 0, b = E - 1;   // the last expert whose first item is <= im
                while (a < b) {
                    const int m = (a + b + 1) >> 1;
                    if (sh.ioff[m] <= im) a = m; else b = m - 1;
                }
                const int n = max(sh.ioff[a + 1] - sh.ioff[a], 1), c = sh.cnt[a];
                const int z = (c + n - 1) / n, j = (u - nb1 * sh.ioff[a]) % n;
                sh.tnt[x][i] = (uint8_t)min((min(c, (j + 1) * z) - j * z + 15) >> 4, kBigMaxTiles);
            }
        }
        __syncthreads();
        if (threadIdx.x < 8 * kQueueTail) {
            const int x = threadIdx.x / kQueueTail, i = threadIdx.x % kQueueTail;
            const int t = min(sh.cuts[x + 1] - sh.cuts[x], kQueueTail);
            if (i < t) {
                const int v = sh.tnt[x][i];
                int r = 0;
                for (int k = 0; k < t; ++k) {
                    const int w = sh.tnt[x][k];
                    r += (w > v) || (w == v && k < i);
                }
                order[kQueueTail * x + r] = (uint8_t)i;
            }
        }
    } else if (threadIdx.x < 8 * kQueueTail) {
        order[threadIdx.x] = (uint8_t)(threadIdx.x % kQueueTail);
    }
}

__global__ void __launch_bounds__(kScanThreads)
route_scan_kernel(const int64_t* __restrict__ topk_idx, int P, int chunk,
                  int* __restrict__ chunk_hist, int nchunks, int E, int cap, int m_tile,
                  int max_items, int nb1, int nb2, int* __restrict__ counts,
                  int* __restrict__ offsets, int* __restrict__ items, int* __restrict__ status) {
    __shared__ RouteSmem sh;
    __shared__ int lh[kFusedHist];   // [chunk][expert] when topk_idx is given
    // Small launches (topk_idx given, nchunks * E <= kFusedHist): the chunk
    // histograms of route_hist_kernel, built here in LDS, 8 pairs' loads in
    // flight per thread.
    const bool fused = topk_idx != nullptr;
    if (fused) {
        for (int i = threadIdx.x; i < nchunks * E; i += kScanThreads) lh[i] = 0;
        __syncthreads();
        for (int p0 = threadIdx.x; p0 < P; p0 += 8 * kScanThreads) {
            int64_t ev[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int p = p0 + u * kScanThreads;
                ev[u] = p < P ? topk_idx[p] : -1;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int p = p0 + u * kScanThreads;
                if (ev[u] >= 0 && ev[u] < E) atomicAdd(&lh[(p / chunk) * E + (int)ev[u]], 1);
            }
        }
        __syncthreads();
    }
    // E <= kMaxExperts = kScanThreads: one expert per thread.
    const int e = threadIdx.x;
    int run = 0;
    if (e < E) {
        // exclusive prefix over chunks (uncapped rank base), 8 chunks' loads
        // in flight at a time
        for (int c0 = 0; c0 < nchunks; c0 += 8) {
            int h[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                h[u] = c0 + u >= nchunks ? 0
                       : fused           ? lh[(c0 + u) * E + e]
                                         : chunk_hist[(size_t)(c0 + u) * E + e];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (c0 + u < nchunks) {
                    chunk_hist[(size_t)(c0 + u) * E + e] = run;
                    run += h[u];
                }
        }
    }
    route_finish(sh, run, P, E, cap, m_tile, max_items, nb1, nb2,
                 RouteOut{counts, offsets, items, status});
}

// The whole routing in one workgroup, for at most kRouteOneSegs segments x
// experts counters and kRouteOneRounds rounds: a segment is 64 consecutive
// pairs, one per lane of a wave.  Every wave ranks its pairs within the
// segment (ballots over the expert-id bits) and counts them per expert in
// LDS; thread e then runs over the segments for expert e's running counts, and
// a pair's slot is its expert's offset + the count before its segment + its
// rank.  The pairs are read once and stay in registers.
// Latency-bound: one launch instead of two or three (measured on MI355X, all
// routing kernels, E = 256: T = 1 11.4 -> 6.5 us, T = 13 11.9 -> 7.3, T = 512
// 15.6 -> 14.2).  Workgroups after the first fold bf16 activations (x8 groups
// of 8 values), a launch of its own otherwise.
__global__ void __launch_bounds__(kScanThreads)
route_one_kernel(const int64_t* __restrict__ topk_idx, int P, int E, int nbits, int cap,
                 int m_tile, int max_items, int nb1, int nb2, int* __restrict__ counts,
                 int* __restrict__ offsets, int* __restrict__ items, int* __restrict__ status,
                 uint32_t* __restrict__ perm, int* __restrict__ pair_pos,
                 const uint16_t* __restrict__ x, size_t x8, uint8_t* __restrict__ xq,
                 uint8_t* __restrict__ xq_sf) {
    if (blockIdx.x > 0) {   // the fold of bf16 activations, next to the routing
        quant_act8(x, (size_t)(blockIdx.x - 1) * kScanThreads + threadIdx.x, x8, xq, xq_sf);
        return;
    }
    __shared__ RouteSmem sh;
    __shared__ __align__(16) uint16_t seg[kRouteOneSegs];   // [segment][expert]
    constexpr int kWaves = kScanThreads / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nseg = (P + 63) >> 6;
    int64_t ev[kRouteOneRounds];
#pragma unroll
    for (int r = 0; r < kRouteOneRounds; ++r) {
        const int p = r * kScanThreads + threadIdx.x;
        ev[r] = p < P ? topk_idx[p] : -1;
    }
    for (int i = threadIdx.x * 8; i < nseg * E; i += kScanThreads * 8)   // E * nseg <= kRouteOneSegs
        *reinterpret_cast<v4i*>(&seg[i]) = v4i{0, 0, 0, 0};
    __syncthreads();
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int rank[kRouteOneRounds];
#pragma unroll
    for (int r = 0; r < kRouteOneRounds; ++r) {
        if (r * kScanThreads + wave * 64 >= P) break;   // uniform over the wave
        const bool ok = ev[r] >= 0 && ev[r] < E;
        const int e = ok ? (int)ev[r] : 0;
        // lanes holding the same expert id: AND of per-bit ballots
        uint64_t m = __ballot(ok);
        for (int b = 0; b < nbits; ++b) {
            const uint64_t bb = __ballot(ok && ((e >> b) & 1));
            m &= ((e >> b) & 1) ? bb : ~bb;
        }
        rank[r] = __popcll(m & lt_mask);
        if (ok && rank[r] == 0) seg[(r * kWaves + wave) * E + e] = (uint16_t)__popcll(m);
    }
    __syncthreads();
    int run = 0;
    if ((int)threadIdx.x < E) {
        // 8 segments' counts in flight at a time
        for (int s0 = 0; s0 < nseg; s0 += 8) {
            int h[8];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                h[u] = s0 + u < nseg ? seg[(s0 + u) * E + threadIdx.x] : 0;
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (s0 + u < nseg) {
                    seg[(s0 + u) * E + threadIdx.x] = (uint16_t)run;
                    run += h[u];
                }
        }
    }
    route_finish(sh, run, P, E, cap, m_tile, max_items, nb1, nb2,
                 RouteOut{counts, offsets, items, status});
    // sh.cnt, sh.off and seg were written before route_finish's barriers
#pragma unroll
    for (int r = 0; r < kRouteOneRounds; ++r) {
        const int p = r * kScanThreads + threadIdx.x;
        if (p >= P) break;
        int pos = -1;
        if (ev[r] >= 0 && ev[r] < E) {
            const int e = (int)ev[r];
            const int k = seg[(r * kWaves + wave) * E + e] + rank[r];
            if (k < sh.cnt[e]) {
                pos = sh.off[e] + k;
                perm[pos] = (uint32_t)p;
            }
        }
        pair_pos[p] = pos;
    }
}

__global__ void __launch_bounds__(kRouteThreads)
route_scatter_kernel(const int64_t* __restrict__ topk_idx, int P, int E, int nbits, int chunk,
                     const int* __restrict__ chunk_hist, const int* __restrict__ counts,
                     const int* __restrict__ offsets, uint32_t* __restrict__ perm,
                     int* __restrict__ pair_pos) {
    constexpr int kWaves = kRouteThreads / 64;
    __shared__ int run[kMaxExperts];
    __shared__ int cntw[kWaves][kMaxExperts];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < E; i += blockDim.x) {
        run[i] = chunk_hist[(size_t)blockIdx.x * E + i];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) cntw[w][i] = 0;
    }
    __syncthreads();
    const int base = blockIdx.x * chunk;
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int r0 = base; r0 < min(base + chunk, P); r0 += kRouteThreads) {
        const int p = r0 + threadIdx.x;
        const bool in = p < P;
        const int64_t e64 = in ? topk_idx[p] : -1;
        const bool ok = e64 >= 0 && e64 < E;
        const int e = ok ? (int)e64 : 0;
        // lanes holding the same expert id: AND of per-bit ballots
        uint64_t m = __ballot(ok);
        for (int b = 0; b < nbits; ++b) {
            const uint64_t bb = __ballot(ok && ((e >> b) & 1));
            m &= ((e >> b) & 1) ? bb : ~bb;
        }
        const int rank = __popcll(m & lt_mask);
        const int wcnt = __popcll(m);
        if (ok && rank == 0) cntw[wave][e] = wcnt;
        __syncthreads();
        if (ok) {
            int pre = run[e];
            for (int w = 0; w < wave; ++w) pre += cntw[w][e];
            const int r = pre + rank;
            if (r < counts[e]) {
                const int pos = offsets[e] + r;
                perm[pos] = (uint32_t)p;
                pair_pos[p] = pos;
            } else {
                pair_pos[p] = -1;
            }
        } else if (in) {
            pair_pos[p] = -1;
        }
        __syncthreads();
        if (ok && rank == 0) {
            atomicAdd(&run[e], wcnt);
            cntw[wave][e] = 0;
        }
        __syncthreads();
    }
}

// DISPATCH pool (diagnostic / parity): pool[slot][:] = x[perm[slot] / topk][:],
// 16 bytes per thread.
__global__ void __launch_bounds__(256)
dispatch_gather_kernel(const uint8_t* __restrict__ x, int H, int topk,
                       const uint32_t* __restrict__ perm, const int* __restrict__ status,
                       uint8_t* __restrict__ pool) {
    const int slot = blockIdx.x;
    if (slot >= status[2]) return;
    const size_t tok = perm[slot] / (uint32_t)topk;
    const v4i* src = reinterpret_cast<const v4i*>(x + tok * H);
    v4i* dst = reinterpret_cast<v4i*>(pool + (size_t)slot * H);
    for (int c = threadIdx.x; c < H / 16; c += blockDim.x) dst[c] = src[c];
}

}  // namespace mm
