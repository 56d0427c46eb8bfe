// Leafwise and levelwise grow loops on the device.
//
// Both reuse the depthwise data plane (partition count/scan/scatter, histogram units,
// fixed-order completion, node finder) and add their own control kernels:
//   levelwise (ObliviousGrower::grow, src/grower_impl.hpp:598-734): one split per level
//     chosen over the whole frontier (k_find_level + k_level_pick), broadcast to every
//     node, empty children kept;
//   leafwise (LeafwiseGrower::grow, src/grower_impl.hpp:743-862): a device-resident
//     candidate pool replaces the host max-heap; every round pops the best leaf (gain,
//     then lowest node id), partitions it, builds the smaller child, subtracts in place
//     and scores both children.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "bh_common.hpp"
#include "kernels.hpp"
#include "kernels_ext.hpp"
#include "bh_device.hpp"
#include "bh_find.hpp"

namespace bh {

namespace {

__device__ __forceinline__ double l1_thr(double g, double l1)
{
    if (g > l1) return g - l1;
    if (g < -l1) return g + l1;
    return 0.0;
}
__device__ __forceinline__ double score_of(double g, double h, double l1, double l2)
{
    double const t = l1_thr(g, l1);
    double const d = h + l2;
    return d > 0.0 ? (t * t) / d : 0.0;
}
__device__ __forceinline__ float leaf_weight(double g, double h, double l1, double l2)
{
    double const d = h + l2;
    double const w = d > 0.0 ? -l1_thr(g, l1) / d : 0.0;
    return static_cast<float>(w);
}
__device__ __forceinline__ float node_value(NodeInfo const &n, GrowCfg const &c, double const *scales)
{
    if (c.mono) // write_leaf's bounded weight (src/step/primitives.hpp:42-50)
        return c.quantized ? fd_leaf_value(n.id, static_cast<double>(n.itg) * scales[0],
                                           static_cast<double>(n.ith) * scales[1], c)
                           : fd_leaf_value(n.id, n.tg, n.th, c);
    if (c.quantized)
        return leaf_weight(static_cast<double>(n.itg) * scales[0], static_cast<double>(n.ith) * scales[1], c.l1,
                           c.l2);
    return leaf_weight(n.tg, n.th, c.l1, c.l2);
}
__device__ __forceinline__ void put_leaf(DevNode *tree, u32 id, float v)
{
    DevNode n = tree[id];
    n.feature = -1;
    n.bin = n.default_left = n.left = n.right = 0;
    n.value = v;
    tree[id] = n;
}

// Node totals of a frontier (Histogram::totals, include/bonsai/histogram.hpp:76-87)
// from the first selected feature's cells (include/bonsai/split.hpp:36-53) when no
// parent split supplied them.  One workgroup per node.
template <bool Q>
__global__ __launch_bounds__(64) void k_totals(NodeInfo *__restrict__ front, TreeCtl const *__restrict__ ctl,
                                               void const *__restrict__ hist, u16 const *__restrict__ n_bins, u32 F,
                                               u32 SB, u8 const *__restrict__ fmask, u32 local)
{
    u32 const i = blockIdx.x;
    if (i >= ctl->n_front || ctl->done) return;
    NodeInfo nd = front[i];
    if (nd.totals_ready) return;
    if (local && nd.cnt == 0) { // no cells
        if (threadIdx.x == 0) {
            nd.itg = nd.ith = 0;
            nd.tg = nd.th = 0.0F;
            nd.totals_ready = 1;
            front[i] = nd;
        }
        return;
    }
    size_t const nc = static_cast<size_t>(F) * SB;
    u32 f0 = 0;
    if (fmask)
        while (f0 + 1u < F && !fmask[f0]) ++f0;
    u32 const nb0 = n_bins[f0];
    size_t const off = static_cast<size_t>(f0) * SB;
    if (Q) {
        i64 const *c = reinterpret_cast<i64 const *>(hist) + (static_cast<size_t>(nd.slot) * nc + off) * 2;
        i64 g = 0, h = 0;
        for (u32 b = threadIdx.x; b < nb0; b += 64) {
            g += c[2 * b];
            h += c[2 * b + 1];
        }
        for (int o = 32; o > 0; o >>= 1) {
            g += __shfl_xor(g, o);
            h += __shfl_xor(h, o);
        }
        if (threadIdx.x == 0) {
            nd.itg = g;
            nd.ith = h;
            nd.totals_ready = 1;
            front[i] = nd;
        }
    } else if (threadIdx.x == 0) {
        float2 const *c = reinterpret_cast<float2 const *>(hist) + static_cast<size_t>(nd.slot) * nc + off;
        double g = 0.0, h = 0.0;
        u32 b = 0;
        for (; b + 8 <= nb0; b += 8) {
            float2 v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = c[b + k];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                g += v[k].x;
                h += v[k].y;
            }
        }
        for (; b < nb0; ++b) {
            g += c[b].x;
            h += c[b].y;
        }
        nd.tg = static_cast<float>(g);
        nd.th = static_cast<float>(h);
        nd.totals_ready = 1;
        front[i] = nd;
    }
}

// ---------------------------------------------------------------------------------
// Level (oblivious) finder: HistogramLevelSplitFinder::find (src/split.cpp:164-235,
// :350-372).  One workgroup per feature.  Frontier nodes are taken in tiles: the tile's
// prefix sums (fill_prefix: double running sums stored as float, or exact integers) go
// to LDS, every (node, bin, direction) child score is computed in parallel, and each
// (bin, direction) candidate adds the tile's scores to its running sum in node order; an
// infeasible node contributes its parent score.
//
// FP64 bound at deep levels (two divisions per candidate and node; 512 nodes of 2,000
// features x 64 bins: 720 us when every candidate's thread also ran its divisions in node
// order, 550 so).  Where every cell comes from the nodes' own rows (local: a grower's level, not a
// caller's step over histograms it may have summed elsewhere), a node without rows adds
// exactly 0 to every sum and is left out.  A feature whose missing cells are all empty
// scans one direction (the other's sums are the same).
// ---------------------------------------------------------------------------------
constexpr u32 kLevelTile = 8;
constexpr u32 kLevelMaxNodes = 1024; // split levels of a levelwise tree (max_depth <= 11)
// LDS bytes per bin: the tile's prefix cells and both directions' scores.
constexpr u32 level_lds_per_bin(bool q) { return kLevelTile * ((q ? 16u : 8u) + 16u); }

template <bool Q>
__global__ __launch_bounds__(256) void k_find_level(NodeInfo const *__restrict__ front,
                                                    TreeCtl const *__restrict__ ctl, void const *__restrict__ hist,
                                                    u16 const *__restrict__ n_bins, u32 F, u32 SB, GrowCfg cfg,
                                                    double const *__restrict__ scales, SplitRec *__restrict__ fbest,
                                                    u32 local)
{
    typedef typename CellT<Q>::T Cell;
    extern __shared__ __align__(16) unsigned char smem[];
    u32 const f = blockIdx.x;
    if (f >= F) return;
    if (ctl->done) return;
    u32 const P = ctl->n_front;
    u32 const nb = (cfg.fmask && !cfg.fmask[f]) ? 0u : n_bins[f]; // unselected: no cut
    u32 const ncut = nb >= 2 ? nb - 2 : 0;
    SplitRec best{};
    best.default_left = 1;
    if (ncut == 0 || P == 0) {
        if (threadIdx.x == 0) fbest[f] = best;
        return;
    }
    Cell *s_pre = reinterpret_cast<Cell *>(smem);                       // [kLevelTile][SB] prefix over the cut bins
    double *s_cs = reinterpret_cast<double *>(s_pre + kLevelTile * SB); // [kLevelTile][candidates]
    __shared__ double s_ps[kLevelTile], s_rg[kLevelTile], s_rh[kLevelTile], s_mg[kLevelTile], s_mh[kLevelTile];
    __shared__ i64 s_itg[kLevelTile], s_ith[kLevelTile], s_img[kLevelTile], s_imh[kLevelTile];
    __shared__ double s_sum_parent;
    __shared__ u32 s_nonempty, s_live, s_wave[4];
    __shared__ u16 s_list[kLevelMaxNodes];
    size_t const nc = static_cast<size_t>(F) * SB;
    Cell const *cells = reinterpret_cast<Cell const *>(hist) + static_cast<size_t>(f) * SB;
    double const sg = Q ? scales[0] : 0.0, sh = Q ? scales[1] : 0.0;
    u32 const lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) {
        s_sum_parent = 0.0;
        s_nonempty = 0;
        s_live = 0;
    }
    __syncthreads();
    // The nodes with rows, in order, and whether any has a missing cell.
    for (u32 p0 = 0; p0 < P; p0 += blockDim.x) {
        u32 const p = p0 + threadIdx.x;
        NodeInfo nd{};
        if (p < P) nd = front[p];
        bool const live = p < P && (!local || nd.cnt != 0);
        u64 const bal = __ballot(live);
        if (lane == 0) s_wave[wave] = static_cast<u32>(__popcll(bal));
        __syncthreads();
        u32 at = s_live + static_cast<u32>(__popcll(bal & ((1ull << lane) - 1ull)));
        for (u32 w = 0; w < wave; ++w) at += s_wave[w];
        if (live) {
            if (local) s_list[at] = static_cast<u16>(p);
            Cell const m = cells[static_cast<size_t>(nd.slot) * nc + nb - 1u];
            if (m.x != 0 || m.y != 0) atomicOr(&s_nonempty, 1u);
        }
        __syncthreads();
        if (threadIdx.x == 0) s_live += s_wave[0] + s_wave[1] + s_wave[2] + s_wave[3];
        __syncthreads();
    }
    u32 const n_live = s_live;
    auto node_at = [&](u32 i) { return local ? static_cast<u32>(s_list[i]) : i; };
    // candidate c: bin c, missing left (one direction) or bin c / 2, missing left first
    bool const one_dir = s_nonempty == 0;
    u32 const ncand = one_dir ? ncut : 2u * ncut;
    double acc[2] = {0.0, 0.0}; // candidates threadIdx.x and + 256 (ncut <= 254)
    for (u32 p0 = 0; p0 < n_live; p0 += kLevelTile) {
        u32 const tn = min(kLevelTile, n_live - p0);
        if (Q) {
            // exact integers: a wave scans a node's cells in parallel
            for (u32 t = wave; t < tn; t += 4u) {
                i64 const *c = reinterpret_cast<i64 const *>(cells + static_cast<size_t>(front[node_at(p0 + t)].slot) * nc);
                i64 *out = reinterpret_cast<i64 *>(s_pre + t * SB);
                i64 g0 = 0, h0 = 0;
                for (u32 b0 = 0; b0 < ncut; b0 += 64u) {
                    u32 const b = b0 + lane;
                    i64 g = b < ncut ? c[2 * b] : 0, h = b < ncut ? c[2 * b + 1] : 0;
                    for (int o = 1; o < 64; o <<= 1) {
                        i64 const ug = __shfl_up(g, o), uh = __shfl_up(h, o);
                        if (static_cast<int>(lane) >= o) {
                            g += ug;
                            h += uh;
                        }
                    }
                    if (b < ncut) {
                        out[2 * b] = g0 + g;
                        out[2 * b + 1] = h0 + h;
                    }
                    g0 += __shfl(g, 63);
                    h0 += __shfl(h, 63);
                }
            }
        } else {
            // coalesced into LDS, then a thread per node sums in bin order
            for (u32 k = threadIdx.x; k < tn * ncut; k += blockDim.x) {
                u32 const t = k / ncut, b = k - t * ncut;
                s_pre[t * SB + b] = cells[static_cast<size_t>(front[node_at(p0 + t)].slot) * nc + b];
            }
            __syncthreads();
            if (threadIdx.x < tn) {
                float2 *c = reinterpret_cast<float2 *>(s_pre + threadIdx.x * SB);
                double g = 0.0, h = 0.0;
                for (u32 b = 0; b < ncut; ++b) {
                    g = g + c[b].x;
                    h = h + c[b].y;
                    c[b] = make_float2(static_cast<float>(g), static_cast<float>(h));
                }
            }
        }
        if (threadIdx.x < tn) {
            u32 const t = threadIdx.x;
            NodeInfo const nd = front[node_at(p0 + t)];
            Cell const m = cells[static_cast<size_t>(nd.slot) * nc + nb - 1u];
            if (Q) {
                s_img[t] = static_cast<i64>(m.x);
                s_imh[t] = static_cast<i64>(m.y);
                s_itg[t] = nd.itg;
                s_ith[t] = nd.ith;
                s_ps[t] = score_of(static_cast<double>(nd.itg) * sg, static_cast<double>(nd.ith) * sh, cfg.l1, cfg.l2);
            } else {
                s_mg[t] = m.x;
                s_mh[t] = m.y;
                s_ps[t] = score_of(nd.tg, nd.th, cfg.l1, cfg.l2);
                s_rg[t] = static_cast<double>(nd.tg) - m.x;
                s_rh[t] = static_cast<double>(nd.th) - m.y;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0)
            for (u32 k = 0; k < tn; ++k) s_sum_parent += s_ps[k];
        for (u32 i = threadIdx.x; i < tn * ncand; i += blockDim.x) {
            u32 const p = i / ncand, k = i - p * ncand;
            u32 const b = one_dir ? k : k >> 1;
            bool const dl = one_dir || (k & 1u) == 0;
            double cs;
            bool ok;
            if (Q) {
                i64 const *pq = reinterpret_cast<i64 const *>(s_pre + p * SB + b);
                i64 const lg = pq[0], lh = pq[1];
                i64 const mg = s_img[p], mh = s_imh[p];
                i64 const hL = lh + (dl ? mh : 0);
                i64 const hR = ((s_ith[p] - mh) - lh) + (!dl ? mh : 0);
                i64 const gL = lg + (dl ? mg : 0);
                i64 const gR = ((s_itg[p] - mg) - lg) + (!dl ? mg : 0);
                double const dhL = static_cast<double>(hL) * sh, dhR = static_cast<double>(hR) * sh;
                ok = !(dhL < cfg.min_child_hess || dhR < cfg.min_child_hess);
                cs = ok ? score_of(static_cast<double>(gL) * sg, dhL, cfg.l1, cfg.l2) +
                              score_of(static_cast<double>(gR) * sg, dhR, cfg.l1, cfg.l2)
                        : 0.0;
            } else {
                float2 const lp = reinterpret_cast<float2 const *>(s_pre)[p * SB + b];
                double const lg = lp.x, lh = lp.y;
                double const mg = s_mg[p], mh = s_mh[p];
                double const right_g = s_rg[p] - lg, right_h = s_rh[p] - lh;
                double const gL = lg + (dl ? mg : 0.0), hL = lh + (dl ? mh : 0.0);
                double const gR = right_g + (!dl ? mg : 0.0), hR = right_h + (!dl ? mh : 0.0);
                ok = !(hL < cfg.min_child_hess || hR < cfg.min_child_hess);
                cs = ok ? score_of(gL, hL, cfg.l1, cfg.l2) + score_of(gR, hR, cfg.l1, cfg.l2) : 0.0;
            }
            s_cs[i] = ok ? cs : s_ps[p];
        }
        __syncthreads();
        for (u32 s = 0; s < 2; ++s) {
            u32 const k = threadIdx.x + s * blockDim.x;
            if (k >= ncand) continue;
            double sum = acc[s];
            for (u32 p = 0; p < tn; ++p) sum += s_cs[p * ncand + k];
            acc[s] = sum;
        }
        __syncthreads();
    }
    // Per-feature winner: max gain, earliest (bin, dl=true first).
    __shared__ double s_g[256];
    __shared__ u32 s_k[256];
    double bg = 0.0;
    u32 bk = kNone;
    double const sp = s_sum_parent;
    for (u32 s = 0; s < 2; ++s) {
        u32 const c = threadIdx.x + s * blockDim.x;
        if (c >= ncand) continue;
        u32 const k = one_dir ? 2u * c : c; // bin << 1 | missing right
        double const gain = acc[s] - sp;
        if (!(gain > 0.0 && gain >= cfg.min_gain)) continue;
        if (gain > bg || (gain == bg && k < bk)) {
            bg = gain;
            bk = k;
        }
    }
    s_g[threadIdx.x] = bg;
    s_k[threadIdx.x] = bk;
    __syncthreads();
    for (u32 st = blockDim.x / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) {
            double const og = s_g[threadIdx.x + st];
            u32 const ok = s_k[threadIdx.x + st];
            if (ok != kNone &&
                (s_k[threadIdx.x] == kNone || og > s_g[threadIdx.x] || (og == s_g[threadIdx.x] && ok < s_k[threadIdx.x]))) {
                s_g[threadIdx.x] = og;
                s_k[threadIdx.x] = ok;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (s_k[0] != kNone) {
            best.gain = s_g[0];
            best.feature = f;
            best.bin = s_k[0] >> 1;
            best.default_left = (s_k[0] & 1u) == 0 ? 1u : 0u;
            best.valid = 1;
        }
        fbest[f] = best;
    }
}

// reduce_in_feature_order (src/split.cpp:240-253) + the level's bookkeeping
// (src/grower_impl.hpp:633-645): record the split or stop growth.
__global__ __launch_bounds__(256) void k_level_pick(SplitRec const *__restrict__ fbest, u32 F,
                                                    TreeCtl *__restrict__ ctl, u32 *__restrict__ level_splits,
                                                    float *__restrict__ level_gains, SplitRec *__restrict__ pick)
{
    if (ctl->done) return;
    __shared__ double s_g[256];
    __shared__ u32 s_f[256];
    double bg = 0.0;
    u32 bf = kNone;
    for (u32 f = threadIdx.x; f < F; f += blockDim.x) {
        SplitRec const c = fbest[f];
        if (c.valid && (c.gain > bg || bf == kNone || (c.gain == bg && f < bf))) {
            if (bf == kNone || c.gain > bg || (c.gain == bg && f < bf)) {
                bg = c.gain;
                bf = f;
            }
        }
    }
    s_g[threadIdx.x] = bg;
    s_f[threadIdx.x] = bf;
    __syncthreads();
    for (u32 st = blockDim.x / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) {
            double const og = s_g[threadIdx.x + st];
            u32 const of = s_f[threadIdx.x + st];
            if (of != kNone &&
                (s_f[threadIdx.x] == kNone || og > s_g[threadIdx.x] || (og == s_g[threadIdx.x] && of < s_f[threadIdx.x]))) {
                s_g[threadIdx.x] = og;
                s_f[threadIdx.x] = of;
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        u32 const d = ctl->oblivious_depth;
        if (s_f[0] == kNone) {
            ctl->done = 1;
            SplitRec z{};
            pick[0] = z;
            return;
        }
        SplitRec const s = fbest[s_f[0]];
        pick[0] = s;
        level_splits[3 * d] = s.feature;
        level_splits[3 * d + 1] = s.bin;
        level_splits[3 * d + 2] = s.default_left;
        level_gains[d] = static_cast<float>(s.gain);
        ctl->oblivious_depth = d + 1;
    }
}

// Broadcast the level split to every frontier node: one partition op per node (empty
// nodes included), the node's child sums under the split (for leaves made at the last
// level), and the partition units.
template <bool Q>
__global__ __launch_bounds__(1024) void k_plan_oblivious(NodeInfo const *__restrict__ front,
                                                         TreeCtl *__restrict__ ctl, SplitRec const *__restrict__ pick,
                                                         void const *__restrict__ hist, u16 const *__restrict__ n_bins,
                                                         u32 F, u32 SB, SplitRec *__restrict__ splits,
                                                         PartOp *__restrict__ ops, PartChunk *__restrict__ pch, u32 dst,
                                                         u32 is_last, u32 chunk_rows, u32 local)
{
    __shared__ u32 scratch[1024];
    __shared__ u32 s_chunks;
    if (ctl->done) {
        if (threadIdx.x == 0) {
            ctl->n_ops = 0;
            ctl->n_part_chunks = 0;
        }
        return;
    }
    SplitRec const s = pick[0];
    u32 const P = ctl->n_front;
    u32 const nb = n_bins[s.feature];
    bool const dl = s.default_left != 0;
    size_t const nc = static_cast<size_t>(F) * SB;
    if (threadIdx.x == 0) s_chunks = 0;
    __syncthreads();
    for (u32 t0 = 0; t0 < P; t0 += blockDim.x) {
        u32 const i = t0 + threadIdx.x;
        bool const in = i < P;
        u32 nch = 0;
        NodeInfo nd{};
        if (in) {
            nd = front[i];
            nch = (nd.cnt + chunk_rows - 1) / chunk_rows;
        }
        u32 ctot;
        u32 const cfirst = block_exscan(nch, scratch, &ctot) + s_chunks;
        if (in) {
            SplitRec r = s;
            if (!is_last) {
                // child sums are only read for leaves made at the last level
            } else if (local && nd.cnt == 0) { // no cells: every sum is zero
                r.gL = r.hL = r.gR = r.hR = 0.0;
                r.igL = r.ihL = r.igR = r.ihR = 0;
            } else if (Q) {
                i64 const *c = reinterpret_cast<i64 const *>(hist) +
                               (static_cast<size_t>(nd.slot) * nc + static_cast<size_t>(s.feature) * SB) * 2;
                i64 lg = 0, lh = 0;
                for (u32 b = 0; b <= s.bin; ++b) {
                    lg += c[2 * b];
                    lh += c[2 * b + 1];
                }
                i64 const mg = c[2 * (nb - 1)], mh = c[2 * (nb - 1) + 1];
                r.igL = lg + (dl ? mg : 0);
                r.ihL = lh + (dl ? mh : 0);
                r.igR = ((nd.itg - mg) - lg) + (!dl ? mg : 0);
                r.ihR = ((nd.ith - mh) - lh) + (!dl ? mh : 0);
            } else {
                float2 const *c = reinterpret_cast<float2 const *>(hist) + static_cast<size_t>(nd.slot) * nc +
                                  static_cast<size_t>(s.feature) * SB;
                double g = 0.0, h = 0.0;
                for (u32 b = 0; b <= s.bin; ++b) {
                    g = g + c[b].x;
                    h = h + c[b].y;
                }
                double const lg = static_cast<float>(g), lh = static_cast<float>(h);
                double const mg = c[nb - 1].x, mh = c[nb - 1].y;
                double const rg = static_cast<double>(nd.tg) - mg, rh = static_cast<double>(nd.th) - mh;
                r.gL = lg + (dl ? mg : 0.0);
                r.hL = lh + (dl ? mh : 0.0);
                r.gR = (rg - lg) + (!dl ? mg : 0.0);
                r.hR = (rh - lh) + (!dl ? mh : 0.0);
            }
            splits[i] = r;
            PartOp op{};
            op.parent = i;
            op.feature = s.feature;
            op.bin = s.bin;
            op.default_left = s.default_left;
            op.last_bin = nb - 1u;
            op.off = nd.off;
            op.cnt = nd.cnt;
            op.src = nd.src;
            op.dst = dst;
            op.chunk_first = cfirst;
            op.chunk_count = nch;
            op.alive = 1;
            ops[i] = op;
        }
        __syncthreads();
        if (threadIdx.x == 0) s_chunks += ctot;
        __syncthreads();
    }
    u32 const n_ch = s_chunks;
    for (u32 c = threadIdx.x; c < n_ch; c += blockDim.x) {
        u32 lo = 0, hi = P;
        while (hi - lo > 1) {
            u32 const mid = (lo + hi) >> 1;
            if (ops[mid].chunk_first <= c) lo = mid;
            else hi = mid;
        }
        PartOp const op = ops[lo];
        u32 const k = c - op.chunk_first;
        PartChunk pc;
        pc.op = lo;
        pc.begin = k * chunk_rows;
        pc.end = min(op.cnt, (k + 1) * chunk_rows);
        pc.left_before = 0;
        pch[c] = pc;
    }
    if (threadIdx.x == 0) {
        ctl->n_ops = P;
        ctl->n_part_chunks = n_ch;
    }
}

// Level swap for the oblivious loop: a stopped tree keeps its frontier (copied into
// the buffer the next level reads).
__global__ __launch_bounds__(256) void k_next_level_obl(TreeCtl *__restrict__ ctl, NodeInfo const *__restrict__ cur,
                                                        NodeInfo *__restrict__ nxt)
{
    bool const done = ctl->done != 0;
    u32 const P = ctl->n_front;
    if (done)
        for (u32 i = threadIdx.x; i < P; i += blockDim.x) nxt[i] = cur[i];
    __syncthreads();
    if (threadIdx.x == 0) {
        if (!done) ctl->n_front = ctl->next_front;
        ctl->depth += 1;
    }
}

// The finished oblivious tree as a perfect dense tree (ObliviousTree ->
// dense_equivalent, src/tree.cpp:21-50): internal node i at level lvl(i) carries that
// level's split, children 2i+1 / 2i+2, leaves 2^D-1 .. in leaf-table order, covers
// aggregated bottom-up.
template <bool Q>
__global__ __launch_bounds__(1024) void k_oblivious_tree(NodeInfo const *__restrict__ front,
                                                         TreeCtl *__restrict__ ctl, u32 const *__restrict__ level_splits,
                                                         float const *__restrict__ level_gains, DevNode *__restrict__ tree,
                                                         GrowCfg cfg, double const *__restrict__ scales)
{
    u32 const D = ctl->oblivious_depth;
    u32 const n_int = (1u << D) - 1u, n_leaf = 1u << D;
    for (u32 j = threadIdx.x; j < n_leaf; j += blockDim.x) {
        NodeInfo const nd = front[j];
        DevNode n{};
        n.feature = -1;
        n.value = node_value(nd, cfg, scales);
        n.cover = static_cast<float>(nd.cnt);
        tree[n_int + j] = n;
    }
    __syncthreads();
    // Internal nodes level by level from the bottom.
    for (int lvl = static_cast<int>(D) - 1; lvl >= 0; --lvl) {
        u32 const first = (1u << lvl) - 1u, count = 1u << lvl;
        for (u32 k = threadIdx.x; k < count; k += blockDim.x) {
            u32 const i = first + k;
            DevNode n{};
            n.feature = static_cast<int32_t>(level_splits[3 * lvl]);
            n.bin = level_splits[3 * lvl + 1];
            n.default_left = level_splits[3 * lvl + 2];
            n.left = 2 * i + 1;
            n.right = 2 * i + 2;
            n.gain = level_gains[lvl];
            n.cover = tree[2 * i + 1].cover + tree[2 * i + 2].cover;
            tree[i] = n;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) ctl->n_nodes = n_int + n_leaf;
}

// ---------------------------------------------------------------------------------
// Leafwise rounds.
//
// Growth pops the pool's best leaf (gain, ties to the lower node id), and each pop needs
// its children's splits before the next one is known: as one leaf a round that is five
// launches of mostly idle chip, 254 times for 255 leaves (57 us a round, nearly all
// launch and latency).  A round here expands up to kLwBatch leaves: the one the pops wait
// for and the best of the others, children of expanded but not yet popped leaves
// included; what is expanded early is popped later without a round of its own.  Pops and
// node ids follow the one-leaf order exactly, and a leaf expanded but never popped stays
// the leaf it is (its rows only moved inside their segment).  255 leaves take 33 rounds on
// the logistic table (of 32 possible), 31 take 7; 16M x 28, 255
// leaves, 3 trees: 44.5 -> 22.2 ms; 1M x 28 FP32, 31 leaves, 10 trees: 23.9 -> 13.1 ms.
//
// NodeInfo::id is the leaf's record here: a child may be searched before its node id is
// known, and monotone boxes and interaction paths are kept by it.  1M x 28 quantized, 255
// leaves, monotone: 2.9 ms a tree; with one leaf a round, as ids would need, 12.4.
// ---------------------------------------------------------------------------------
// Rows per partition chunk of a leaf of `rows` rows: about kLwChunkTarget chunks,
// multiples of 256 rows, kLwMinChunk..kPartChunk, and at most cap (the chunk of wide
// rows).
__device__ __forceinline__ u32 lw_chunk_rows(u32 rows, u32 cap)
{
    u32 const per = ((rows + kLwChunkTarget - 1u) / kLwChunkTarget + 255u) & ~255u;
    return min(cap, min(kPartChunk, max(kLwMinChunk, per)));
}

// Rows per histogram unit of a built node of `rows` rows: at most `target` units of
// kLwMinUnit..kHistChunk rows (multiples of 256); target 0 keeps kHistChunk.  FP32 sums
// run in ascending rows within a unit and over units in order, so this rule is part of
// the FP32 leafwise summation order (the oracle restates it).
__device__ __forceinline__ u32 lw_unit_rows(u32 rows, u32 target)
{
    if (target == 0) return kHistChunk;
    u32 const per = ((rows + target - 1u) / target + 255u) & ~255u;
    return min(kHistChunk, max(kLwMinUnit, per));
}

// Upper bound of a built node's unit count over all its row counts up to `rows`.
__device__ __forceinline__ u32 lw_unit_bound(u32 rows, u32 target)
{
    u32 const whole = (rows + kHistChunk - 1u) / kHistChunk;
    return max(whole, min(target, (rows + kLwMinUnit - 1u) / kLwMinUnit));
}

enum : u32 { kLwPlain = 0, kLwExpanded = 1, kLwDemoted = 2 };

// Argmax over an LDS list (value, then lower key: a total order, so the butterfly is
// exact) by one wave; every lane receives the index.
__device__ __forceinline__ u32 lw_argmax(double const *val, u32 const *key, u32 n)
{
    double bg = 0.0;
    u32 bid = kNone, bix = kNone;
    for (u32 k = threadIdx.x & 63u; k < n; k += 64u)
        if (bix == kNone || val[k] > bg || (val[k] == bg && key[k] < bid)) {
            bg = val[k];
            bid = key[k];
            bix = k;
        }
    for (int o = 32; o > 0; o >>= 1) {
        double const og = __shfl_xor(bg, o);
        u32 const oid = __shfl_xor(bid, o), oix = __shfl_xor(bix, o);
        if (oix != kNone && (bix == kNone || og > bg || (og == bg && oid < bid))) {
            bg = og;
            bid = oid;
            bix = oix;
        }
    }
    return bix;
}
// One wave's LDS writes before its next reads.
__device__ __forceinline__ void lw_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One expanded split of a round on its way to its children.
struct LwSplit {
    u32 rec;             // its record
    u32 demoted, leaves; // one side has no rows; the children sit at max_depth
    u32 nL, cnt, off, dst, slot, left_id, depth;
    u32 urows, units, small_cnt, small_off, left_small;
    u32 fresh, fin, part_first, unit_first; // from lw_place
};

__device__ __forceinline__ void lw_measure(LwSplit &x, u32 nL, GrowCfg const &cfg, u32 unit_target)
{
    u32 const nR = x.cnt - nL;
    x.nL = nL;
    x.demoted = (nL == 0) != (nR == 0) ? 1u : 0u;
    x.leaves = static_cast<int>(x.depth) + 1 >= cfg.max_depth ? 1u : 0u;
    x.left_small = nL <= nR ? 1u : 0u;
    x.small_cnt = x.left_small ? nL : nR;
    x.small_off = x.left_small ? x.off : x.off + nL;
    x.urows = lw_unit_rows(x.small_cnt, unit_target);
    x.units = x.demoted || x.leaves ? 0u : (x.small_cnt + x.urows - 1) / x.urows;
}

// Slots, finish ops, units and partials of the round's splits, in order (one thread);
// fresh: the top kLwBatch free slots, top first.
__device__ __forceinline__ void lw_place(LwSplit *x, u32 n, u32 const *fresh, u32 *free_slots, LwCtl *lw, TreeCtl *ctl)
{
    u32 fin = 0, units = 0, parts = 0;
    for (u32 j = 0; j < n; ++j) {
        if (x[j].demoted || x[j].leaves) continue;
        x[j].fresh = fresh[fin];
        x[j].fin = fin++;
        x[j].unit_first = units;
        x[j].part_first = parts;
        units += x[j].units;
        parts += x[j].units > 1 ? x[j].units : 0u;
    }
    u32 nf = lw->n_free - fin;
    for (u32 j = 0; j < n; ++j)
        if (x[j].demoted || x[j].leaves) free_slots[nf++] = x[j].slot;
    lw->n_free = nf;
    ctl->n_front = 2u * n;
    ctl->n_finish = fin;
    ctl->n_hist_chunks = units;
}

// The round's children (commit_pop, src/grower_impl.hpp:370-400): the larger keeps the
// parent's histogram slot (completed in place), the smaller gets the fresh one and the
// histogram units.  Children at max_depth only need totals, from the split's sums, as do
// all quantized ones (exact integers).
template <bool Q>
__device__ __forceinline__ void lw_children(LwSplit const *xs, u32 n, LwCtl *lw, LwRec *recs, NodeInfo *kids,
                                            FinishOp *fops, HistChunk *hch)
{
    if (threadIdx.x < n) {
        u32 const j = threadIdx.x;
        LwSplit const x = xs[j];
        SplitRec const s = recs[x.rec].split;
        NodeInfo L{}, R{};
        L.id = x.left_id;
        R.id = x.left_id + 1u;
        L.off = x.off;
        L.cnt = x.nL;
        R.off = x.off + x.nL;
        R.cnt = x.cnt - x.nL;
        L.src = R.src = x.dst;
        L.depth = R.depth = x.depth + 1u;
        if (Q || x.leaves) {
            L.totals_ready = R.totals_ready = 1;
            if (Q) {
                L.itg = s.igL;
                L.ith = s.ihL;
                R.itg = s.igR;
                R.ith = s.ihR;
            } else {
                L.tg = static_cast<float>(s.gL);
                L.th = static_cast<float>(s.hL);
                R.tg = static_cast<float>(s.gR);
                R.th = static_cast<float>(s.hR);
            }
        }
        if (x.demoted || x.leaves) {
            L.slot = R.slot = kNone;
        } else {
            L.slot = x.left_small ? x.fresh : x.slot;
            R.slot = x.left_small ? x.slot : x.fresh;
            FinishOp fo{};
            fo.small_slot = x.fresh;
            fo.large_slot = x.slot;
            fo.parent_slot = x.slot;
            fo.part_first = x.part_first;
            fo.part_count = x.units > 1 ? x.units : 0;
            fo.empty = x.small_cnt == 0;
            fops[x.fin] = fo;
        }
        kids[2 * j] = L;
        kids[2 * j + 1] = R;
        lw->batch[j] = x.rec;
        lw->demoted[j] = x.demoted;
    }
    for (u32 j = 0; j < n; ++j) {
        u32 const units = xs[j].units;
        for (u32 k = threadIdx.x; k < units; k += blockDim.x) {
            HistChunk hc{};
            hc.slot = xs[j].fresh;
            hc.src = xs[j].dst;
            hc.begin = xs[j].small_off + k * xs[j].urows;
            hc.end = xs[j].small_off + min(xs[j].small_cnt, (k + 1) * xs[j].urows);
            hc.part = units > 1 ? xs[j].part_first + k : kNone;
            hch[xs[j].unit_first + k] = hc;
        }
    }
}

// A record's meta word: bits 0..1 the state, bit 2 a valid split, then the unit bound of
// the child it would build.  Quantized splits whose children need no histogram are born
// expanded (at max_depth) or demoted (one side without rows).
constexpr u32 kLwValid = 4u;
template <bool COUNTED> __device__ __forceinline__ u32 lw_meta(LwRec const &c, GrowCfg const &cfg, u32 unit_target)
{
    if (!c.split.valid) return kLwExpanded;
    u32 const nL = c.split.n_left, nR = c.node.cnt - nL;
    u32 state = kLwPlain;
    if (COUNTED && (nL == 0) != (nR == 0)) state = kLwDemoted;
    else if (COUNTED && static_cast<int>(c.node.depth) + 1 >= cfg.max_depth) state = kLwExpanded;
    return state | kLwValid | lw_unit_bound(COUNTED ? min(nL, nR) : c.node.cnt / 2u, unit_target) << 3;
}
__device__ __forceinline__ bool lw_listed(u32 meta) { return (meta & 7u) == (kLwPlain | kLwValid); }

// Round start: the last round's children become records, then leaves are popped while
// the best one is expanded (max gain, ties to the lower node id; the reference's
// gain_less, src/grower_impl.hpp:763-770), each committing its split
// (commit_split_node, :188-210) and queueing its children (:404-428), until the pool is
// empty, the leaf budget is spent or the best leaf has no children yet.  Then the round's
// leaves are chosen and their partition ops emitted, in chunks sized to each leaf.
// COUNTED (quantized): a split carries its child row counts, so the children, their slots
// and the histogram units are set here, the scatter takes each chunk's prefix from the
// chunk counts, and a split whose children need no histogram (at max_depth, the last one
// of the budget, demoted) takes no round at all.  Runs as its own one-block kernel for the
// first round and in the last workgroup of every round's split find for the next; any
// workgroup size that is a multiple of 64.  Bound by latency, so the pops and the choice
// run in one wave over what they need of every record in LDS, and the popped nodes, the
// ops and the children are then written in parallel.
template <bool COUNTED>
__device__ __forceinline__ void lw_select_round(TreeCtl *__restrict__ ctl, LwCtl *__restrict__ lw, LwLists const &ls,
                                                NodeInfo *__restrict__ kids, SplitRec const *__restrict__ kid_splits,
                                                DevNode *__restrict__ tree, PartOp *__restrict__ ops,
                                                PartChunk *__restrict__ pch, HistChunk *__restrict__ hch,
                                                u16 const *__restrict__ n_bins, FinishOp *__restrict__ fops,
                                                GrowCfg const &cfg, double const *__restrict__ scales)
{
    __shared__ double s_pg[kLwPoolCap], s_lv[kLwListCap], s_gain[kLwRecCap];
    __shared__ u32 s_pid[kLwPoolCap], s_prec[kLwPoolCap], s_lrec[kLwListCap];
    __shared__ u32 s_link[kLwRecCap], s_meta[kLwRecCap], s_pop_rec[kLwPoolCap], s_pop_id[kLwPoolCap];
    __shared__ LwSplit s_x[kLwBatch];
    __shared__ u32 s_nl, s_np, s_free, s_act, s_pops, s_n, s_sel[kLwBatch], s_fresh[kLwBatch];
    __shared__ u32 s_chunk[kLwBatch + 1], s_crow[kLwBatch], s_deep;
    if (ctl->done) return; // every work list is empty
    u32 const nb = lw->n_batch, r0 = lw->n_rec, np0 = lw->n_pool, nl0 = lw->n_list;
    if (threadIdx.x == 0) {
        s_nl = nl0;
        s_free = lw->n_free;
        s_deep = ctl->max_depth_seen;
    }
    for (u32 k = threadIdx.x; k < np0; k += blockDim.x) {
        s_pg[k] = ls.pool_gain[k];
        s_pid[k] = ls.pool_id[k];
        s_prec[k] = ls.pool_rec[k];
    }
    for (u32 k = threadIdx.x; k < nl0; k += blockDim.x) {
        s_lv[k] = ls.list_prio[k];
        s_lrec[k] = ls.list_rec[k];
    }
    for (u32 k = threadIdx.x; k < r0; k += blockDim.x) {
        s_gain[k] = ls.gain[k];
        s_link[k] = ls.link[k];
        s_meta[k] = ls.meta[k];
    }
    __syncthreads();
    // The round's children.
    if (threadIdx.x < 2u * nb) {
        u32 const j = threadIdx.x >> 1, e = threadIdx.x & 1u, p = lw->batch[j], r = r0 + threadIdx.x;
        bool const gone = lw->demoted[j] != 0;
        if (e == 0) {
            s_link[p] = ls.link[p] = r;
            s_meta[p] = ls.meta[p] = (s_meta[p] & ~3u) | (gone ? kLwDemoted : kLwExpanded);
        }
        u32 meta = 0;
        double gain = 0.0;
        if (!gone) {
            LwRec &par = ls.recs[p];
            LwRec c{};
            c.node = kids[threadIdx.x];
            c.split = kid_splits[threadIdx.x];
            c.value = node_value(c.node, cfg, scales);
            c.prio = min(par.prio, c.split.gain);
            gain = c.split.gain;
            meta = lw_meta<COUNTED>(c, cfg, ls.unit_target);
            if (lw_listed(meta)) {
                u32 const k = atomicAdd(&s_nl, 1u);
                s_lv[k] = c.prio;
                s_lrec[k] = r;
            } else if (c.node.slot != kNone) {
                ls.free_slots[atomicAdd(&s_free, 1u)] = c.node.slot;
            }
            ls.recs[r] = c;
            par.kval[e] = c.value;
            par.kcnt[e] = c.node.cnt;
        }
        s_gain[r] = ls.gain[r] = gain;
        s_link[r] = ls.link[r] = kNone;
        s_meta[r] = ls.meta[r] = meta;
    }
    __syncthreads();
    // Pops, then the round's leaves: one wave, on LDS alone.
    u32 const max_leaves = static_cast<u32>(cfg.max_leaves), limit = max_leaves + 7u; // pops of one tree
    u32 const n_nodes = ctl->n_nodes;
    if (threadIdx.x < 64u) {
        u32 const lane = threadIdx.x;
        u32 np = np0, live = ctl->live, ahead = lw->n_ahead, k = 0, act, block = 0;
        u32 const pops = lw->pops;
        for (;;) {
            act = 2; // the tree is complete
            if (np == 0 || live >= max_leaves || pops + k >= limit) break;
            u32 const ix = lw_argmax(s_pg, s_pid, np);
            u32 const r = s_prec[ix], id = s_pid[ix], meta = s_meta[r], link = s_link[r], lid = n_nodes + 2u * k;
            act = 1; // waits for this leaf's children
            block = r;
            if ((meta & 3u) == kLwPlain && !(COUNTED && live + 1u >= max_leaves)) break;
            np -= 1;
            double const lg = s_pg[np];
            u32 const li = s_pid[np], lr = s_prec[np];
            lw_wave_sync();
            if (lane == 0) {
                s_pop_rec[k] = r;
                s_pop_id[k] = id;
                s_pg[ix] = lg;
                s_pid[ix] = li;
                s_prec[ix] = lr;
            }
            ++k;
            if (link != kNone) ahead -= 1;
            if ((meta & 3u) != kLwDemoted) {
                live += 1;
                if (link != kNone)
                    for (u32 e = 0; e < 2; ++e)
                        if (s_meta[link + e] & kLwValid) {
                            if (lane == 0) {
                                s_pg[np] = s_gain[link + e];
                                s_pid[np] = lid + e;
                                s_prec[np] = link + e;
                            }
                            np += 1;
                        }
            }
            lw_wave_sync();
        }
        u32 n = 0, nl = s_nl;
        if (act == 1) {
            // The leaf the pops wait for, then the best others, while their partials fit
            // and children are expected to be asked for.
            u32 const left = max_leaves - live;
            u32 kmax = min(kLwBatch, max(1u, COUNTED ? left - 1u : left)), parts = 0;
            kmax = max(1u, min(kmax, kLwAhead - min(kLwAhead, ahead)));
            while (n < kmax && nl > 0) {
                u32 ix = kNone;
                if (n == 0) {
                    for (u32 q = lane; q < nl; q += 64u)
                        if (s_lrec[q] == block) ix = q;
                    for (int o = 32; o > 0; o >>= 1) ix = min(ix, static_cast<u32>(__shfl_xor(ix, o)));
                } else {
                    ix = lw_argmax(s_lv, s_lrec, nl);
                }
                u32 const r = s_lrec[ix], ub = s_meta[r] >> 3;
                if (n > 0 && parts + ub > ls.max_parts) break;
                parts += ub;
                nl -= 1;
                double const lv = s_lv[nl];
                u32 const lr = s_lrec[nl];
                lw_wave_sync();
                if (lane == 0) {
                    s_sel[n] = r;
                    s_lv[ix] = lv;
                    s_lrec[ix] = lr;
                }
                lw_wave_sync();
                ++n;
            }
        }
        if (lane == 0) {
            ctl->live = live;
            ctl->n_nodes = n_nodes + 2u * k;
            lw->pops = pops + k;
            lw->n_ahead = ahead + n;
            lw->n_rec = r0 + 2u * nb;
            lw->n_batch = n;
            lw->n_pool = np;
            lw->n_list = nl;
            s_np = np;
            s_nl = nl;
            s_act = act;
            s_pops = k;
            s_n = n;
        }
    }
    __syncthreads();
    // The popped leaves' splits in the tree (commit_split_node, :188-210): children first,
    // since a child may have been popped as well.
    u32 const n_pops = s_pops;
    for (u32 k = threadIdx.x; k < n_pops; k += blockDim.x) {
        u32 const lid = n_nodes + 2u * k, rid = lid + 1u, r = s_pop_rec[k];
        LwRec const &c = ls.recs[r];
        DevNode l{}, rr{};
        l.feature = rr.feature = -1;
        if ((s_meta[r] & 3u) != kLwDemoted) {
            atomicMax(&s_deep, c.node.depth + 1u);
            if (COUNTED && s_link[r] == kNone) { // never expanded: leaves from the split's sums
                double const gl = static_cast<double>(c.split.igL) * scales[0],
                             hl = static_cast<double>(c.split.ihL) * scales[1],
                             gr = static_cast<double>(c.split.igR) * scales[0],
                             hr = static_cast<double>(c.split.ihR) * scales[1];
                if (cfg.mono) {
                    double llo, lhi, rlo, rhi;
                    fd_child_bounds(cfg, scales, r, c.split, llo, lhi, rlo, rhi);
                    l.value = static_cast<float>(fd_bounded_weight(gl, hl, cfg.l1, cfg.l2, llo, lhi));
                    rr.value = static_cast<float>(fd_bounded_weight(gr, hr, cfg.l1, cfg.l2, rlo, rhi));
                } else {
                    l.value = leaf_weight(gl, hl, cfg.l1, cfg.l2);
                    rr.value = leaf_weight(gr, hr, cfg.l1, cfg.l2);
                }
                l.cover = static_cast<float>(c.split.n_left);
                rr.cover = static_cast<float>(c.node.cnt - c.split.n_left);
            } else {
                l.value = c.kval[0];
                rr.value = c.kval[1];
                l.cover = static_cast<float>(c.kcnt[0]);
                rr.cover = static_cast<float>(c.kcnt[1]);
            }
        }
        tree[lid] = l;
        tree[rid] = rr;
    }
    __syncthreads();
    for (u32 k = threadIdx.x; k < n_pops; k += blockDim.x) {
        u32 const lid = n_nodes + 2u * k, r = s_pop_rec[k];
        LwRec const &c = ls.recs[r];
        DevNode pn{};
        pn.cover = static_cast<float>(c.node.cnt);
        if ((s_meta[r] & 3u) == kLwDemoted) {
            pn.feature = -1;
            pn.value = c.value;
        } else {
            pn.feature = static_cast<int32_t>(c.split.feature);
            pn.bin = c.split.bin;
            pn.default_left = c.split.default_left;
            pn.left = lid;
            pn.right = lid + 1u;
            pn.gain = static_cast<float>(c.split.gain);
        }
        tree[s_pop_id[k]] = pn;
    }
    if (threadIdx.x == 0) ctl->max_depth_seen = s_deep;
    u32 const n = s_n;
    if (s_act == 2u) {
        if (threadIdx.x == 0) {
            ctl->done = 1;
            ctl->n_ops = 0;
            ctl->n_part_chunks = 0;
            ctl->n_front = 0;
            ctl->n_finish = 0;
            ctl->n_hist_chunks = 0;
        }
        return;
    }
    for (u32 k = threadIdx.x; k < s_np; k += blockDim.x) {
        ls.pool_gain[k] = s_pg[k];
        ls.pool_id[k] = s_pid[k];
        ls.pool_rec[k] = s_prec[k];
    }
    for (u32 k = threadIdx.x; k < s_nl; k += blockDim.x) {
        ls.list_prio[k] = s_lv[k];
        ls.list_rec[k] = s_lrec[k];
    }
    if (threadIdx.x < n) {
        u32 const j = threadIdx.x, r = s_sel[j];
        NodeInfo const nd = ls.recs[r].node;
        SplitRec const s = ls.recs[r].split;
        LwSplit x{};
        x.rec = r;
        x.cnt = nd.cnt;
        x.off = nd.off;
        x.dst = nd.src == 0 ? 1u : 0u;
        x.slot = nd.slot;
        x.depth = nd.depth;
        x.left_id = r0 + 2u * nb + 2u * j; // its children's records (NodeInfo::id here)
        if (COUNTED) {
            lw_measure(x, s.n_left, cfg, ls.unit_target);
            s_fresh[j] = ls.free_slots[s_free - 1u - j];
        }
        s_x[j] = x;
        s_crow[j] = lw_chunk_rows(nd.cnt, ls.chunk_cap);
        s_chunk[j] = (nd.cnt + s_crow[j] - 1u) / s_crow[j];
        fd_propagate_bounds(cfg, scales, r, s, x.left_id, x.left_id + 1u);
        fd_propagate_path(cfg, r, s.feature, x.left_id, x.left_id + 1u);
        PartOp op{};
        op.parent = r;
        op.feature = s.feature;
        op.bin = s.bin;
        op.default_left = s.default_left;
        op.last_bin = static_cast<u32>(n_bins[s.feature]) - 1u;
        op.off = nd.off;
        op.cnt = nd.cnt;
        op.src = nd.src;
        op.dst = x.dst;
        op.chunk_count = s_chunk[j];
        op.left_id = x.left_id;
        op.n_left = COUNTED ? x.nL : 0u;
        op.alive = 1;
        ops[j] = op;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        u32 c = 0;
        for (u32 j = 0; j < n; ++j) {
            u32 const k = s_chunk[j];
            s_chunk[j] = c;
            c += k;
        }
        s_chunk[n] = c;
        lw->n_free = s_free;
        if (COUNTED) lw_place(s_x, n, s_fresh, ls.free_slots, lw, ctl);
        ctl->n_ops = n;
        ctl->n_part_chunks = c;
    }
    __syncthreads();
    if (threadIdx.x < n) ops[threadIdx.x].chunk_first = s_chunk[threadIdx.x];
    for (u32 j = 0; j < n; ++j)
        for (u32 k = threadIdx.x; k < s_chunk[j + 1] - s_chunk[j]; k += blockDim.x) {
            PartChunk pc;
            pc.op = j;
            pc.begin = k * s_crow[j];
            pc.end = min(s_x[j].cnt, (k + 1) * s_crow[j]);
            pc.left_before = 0;
            pch[s_chunk[j] + k] = pc;
        }
    if (COUNTED) lw_children<true>(s_x, n, lw, ls.recs, kids, fops, hch);
}

template <bool COUNTED>
__global__ __launch_bounds__(256) void k_lw_select(TreeCtl *__restrict__ ctl, LwCtl *__restrict__ lw, LwLists ls,
                                                   NodeInfo *__restrict__ kids,
                                                   SplitRec const *__restrict__ kid_splits, DevNode *__restrict__ tree,
                                                   PartOp *__restrict__ ops, PartChunk *__restrict__ pch,
                                                   HistChunk *__restrict__ hch, u16 const *__restrict__ n_bins,
                                                   FinishOp *__restrict__ fops, GrowCfg cfg,
                                                   double const *__restrict__ scales)
{
    lw_select_round<COUNTED>(ctl, lw, ls, kids, kid_splits, tree, ops, pch, hch, n_bins, fops, cfg, scales);
}

// Split find of a round's children (k_find's body) whose last workgroup to finish -- all
// others have stopped reading anything the select writes -- starts the next round and,
// when the host waits for it, reports whether the tree is complete.
struct LwNext {
    LwLists ls;
    DevNode *tree;
    PartOp *ops;
    PartChunk *pch;
    HistChunk *hch;
    FinishOp *fops;
    u32 *report; // pinned host memory, or null
};

template <bool Q, bool COUNTED, bool CON>
__global__ __launch_bounds__(kFindThreads) void k_lw_find(NodeInfo *__restrict__ kids, TreeCtl *__restrict__ ctl,
                                                        LwCtl *__restrict__ lw, void const *__restrict__ hist,
                                                        u16 const *__restrict__ n_bins, u32 F, u32 SB, GrowCfg cfg,
                                                        double const *__restrict__ scales,
                                                        SplitRec *__restrict__ splits, SplitRec *__restrict__ part,
                                                        u32 *__restrict__ done, u32 const *__restrict__ cnt, LwNext nx)
{
    __shared__ u32 s_last_wg;
    find_node<Q, CON, kLwFindTile>(kids, ctl, hist, n_bins, F, SB, cfg, scales, splits, 0u, 0u, part, done, cnt);
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        s_last_wg = atomicAdd(&lw->grid_done, 1u) == gridDim.x * gridDim.y - 1u ? 1u : 0u;
    }
    __syncthreads();
    if (!s_last_wg) return;
    if (threadIdx.x == 0) lw->grid_done = 0u;
    __threadfence();
    __syncthreads();
    lw_select_round<COUNTED>(ctl, lw, nx.ls, kids, splits, nx.tree, nx.ops, nx.pch, nx.hch, n_bins, nx.fops, cfg,
                             scales);
    if (nx.report && threadIdx.x == 0) {
        *nx.report = ctl->done;
        __threadfence_system();
    }
}

// Round middle of the FP32 grower: left counts from the chunk prefixes, then the
// children and their histogram units.
template <bool Q>
__global__ __launch_bounds__(1024) void k_lw_scan(PartOp *__restrict__ ops, PartChunk *__restrict__ pch,
                                                  u32 const *__restrict__ chunk_left, TreeCtl *__restrict__ ctl,
                                                  LwCtl *__restrict__ lw, LwLists ls, NodeInfo *__restrict__ kids,
                                                  HistChunk *__restrict__ hch, FinishOp *__restrict__ fops,
                                                  GrowCfg cfg)
{
    __shared__ u32 scratch[1024];
    __shared__ u32 s_run, s_base[kLwBatch + 1], s_fresh[kLwBatch];
    __shared__ LwSplit s_x[kLwBatch];
    u32 const n = ctl->n_ops;
    if (n == 0) return;
    u32 const n_ch = ctl->n_part_chunks;
    if (threadIdx.x == 0) s_run = 0;
    __syncthreads();
    for (u32 t0 = 0; t0 < n_ch; t0 += blockDim.x) {
        u32 const c = t0 + threadIdx.x;
        u32 const v = c < n_ch ? chunk_left[c] : 0u;
        u32 tot;
        u32 const pre = block_exscan(v, scratch, &tot) + s_run;
        if (c < n_ch) {
            u32 const j = pch[c].op;
            pch[c].left_before = pre;
            if (c == ops[j].chunk_first) s_base[j] = pre;
        }
        __syncthreads();
        if (threadIdx.x == 0) s_run += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) s_base[n] = s_run;
    __syncthreads();
    for (u32 c = threadIdx.x; c < n_ch; c += blockDim.x) pch[c].left_before -= s_base[pch[c].op];
    if (threadIdx.x < n) {
        PartOp op = ops[threadIdx.x];
        LwSplit x{};
        x.rec = op.parent;
        x.cnt = op.cnt;
        x.off = op.off;
        x.dst = op.dst;
        x.left_id = op.left_id;
        x.slot = ls.recs[x.rec].node.slot;
        x.depth = ls.recs[x.rec].node.depth;
        lw_measure(x, s_base[threadIdx.x + 1] - s_base[threadIdx.x], cfg, ls.unit_target);
        op.n_left = x.nL;
        op.alive = x.demoted ? 0u : 1u;
        ops[threadIdx.x] = op;
        s_x[threadIdx.x] = x;
        s_fresh[threadIdx.x] = ls.free_slots[lw->n_free - 1u - threadIdx.x];
    }
    __syncthreads();
    if (threadIdx.x == 0) lw_place(s_x, n, s_fresh, ls.free_slots, lw, ctl);
    __syncthreads();
    lw_children<Q>(s_x, n, lw, ls.recs, kids, fops, hch);
}

// The root's split joins the pool (or the root becomes a leaf).
template <bool COUNTED>
__global__ void k_lw_push_root(LwCtl *__restrict__ lw, LwLists ls, NodeInfo const *__restrict__ kids,
                               SplitRec const *__restrict__ splits, DevNode *__restrict__ tree, GrowCfg cfg,
                               double const *__restrict__ scales)
{
    if (threadIdx.x != 0) return;
    LwRec c{};
    c.node = kids[0];
    c.split = splits[0];
    c.value = node_value(c.node, cfg, scales);
    c.prio = c.split.gain;
    if (!c.split.valid || cfg.max_depth <= 0) {
        put_leaf(tree, c.node.id, c.value);
        return;
    }
    u32 const meta = lw_meta<COUNTED>(c, cfg, ls.unit_target);
    ls.recs[0] = c;
    ls.pool_gain[0] = ls.gain[0] = c.split.gain;
    ls.pool_id[0] = ls.pool_rec[0] = 0;
    ls.link[0] = kNone;
    ls.meta[0] = meta;
    lw->n_rec = lw->n_pool = 1;
    if (lw_listed(meta)) {
        ls.list_prio[0] = c.prio;
        ls.list_rec[0] = 0;
        lw->n_list = 1;
    } else {
        ls.free_slots[lw->n_free++] = c.node.slot;
    }
}

// Leafwise tree start: root frontier (slot 0), free list 1.., pool empty.
__global__ __launch_bounds__(256) void k_lw_begin(TreeCtl *__restrict__ ctl, LwCtl *__restrict__ lw,
                                                  NodeInfo *__restrict__ kids, DevNode *__restrict__ tree,
                                                  HistChunk *__restrict__ hch, FinishOp *__restrict__ fops,
                                                  u32 *__restrict__ free_slots, u32 n_slots, RootSel root,
                                                  u32 unit_target)
{
    u32 const n_rows = root.n_from_ctl ? ctl->root_n : root.n;
    u32 const urows = lw_unit_rows(n_rows, unit_target);
    u32 const n_units = (n_rows + urows - 1) / urows;
    u32 const multi = n_units > 1;
    for (u32 k = threadIdx.x; k < n_units; k += blockDim.x) {
        HistChunk hc{};
        hc.slot = 0;
        hc.src = root.src;
        hc.begin = k * urows;
        hc.end = min(n_rows, (k + 1) * urows);
        hc.part = multi ? k : kNone;
        hch[k] = hc;
    }
    for (u32 k = threadIdx.x; k + 1 < n_slots; k += blockDim.x) free_slots[k] = n_slots - 1 - k;
    if (threadIdx.x == 0) {
        NodeInfo rn{};
        rn.cnt = n_rows;
        rn.src = root.src;
        rn.slot = 0;
        kids[0] = rn;
        DevNode r{};
        r.feature = -1;
        r.cover = static_cast<float>(n_rows);
        tree[0] = r;
        FinishOp fo{};
        fo.small_slot = 0;
        fo.large_slot = kNone;
        fo.part_count = multi ? n_units : 0;
        fo.empty = n_rows == 0;
        fops[0] = fo;
        ctl->n_front = 1;
        ctl->n_nodes = 1;
        ctl->n_ops = 0;
        ctl->n_part_chunks = 0;
        ctl->n_hist_chunks = n_units;
        ctl->n_finish = 1;
        ctl->done = 0;
        ctl->live = 1;
        ctl->max_depth_seen = 0;
        lw->n_pool = lw->n_list = lw->n_rec = lw->n_batch = 0;
        lw->pops = lw->n_ahead = 0;
        lw->n_free = n_slots - 1;
        lw->grid_done = 0;
    }
}

__global__ void k_obl_begin(TreeCtl *ctl)
{
    if (threadIdx.x == 0) {
        ctl->done = 0;
        ctl->oblivious_depth = 0;
    }
}

} // namespace

hipError_t ext_alloc(ExtState &s, bh_fit_config const &f, u32 F, u32 hist_slots)
{
    s.n_features = F;
    hipError_t e;
    if (f.grower == BH_LEAFWISE) {
        if ((e = hipMalloc(&s.ls.recs, sizeof(LwRec) * kLwRecCap)) != hipSuccess) return e;
        if ((e = hipMalloc(&s.ls.pool_gain, sizeof(double) * (kLwPoolCap + kLwListCap + kLwRecCap))) != hipSuccess)
            return e;
        if ((e = hipMalloc(&s.ls.pool_id, sizeof(u32) * (2u * kLwPoolCap + kLwListCap + 2u * kLwRecCap))) != hipSuccess)
            return e;
        s.ls.list_prio = s.ls.pool_gain + kLwPoolCap;
        s.ls.gain = s.ls.list_prio + kLwListCap;
        s.ls.pool_rec = s.ls.pool_id + kLwPoolCap;
        s.ls.list_rec = s.ls.pool_rec + kLwPoolCap;
        s.ls.link = s.ls.list_rec + kLwListCap;
        s.ls.meta = s.ls.link + kLwRecCap;
        if ((e = hipMalloc(&s.ls.free_slots, sizeof(u32) * (hist_slots + 4))) != hipSuccess) return e;
        if ((e = hipMalloc(&s.lw, sizeof(LwCtl))) != hipSuccess) return e;
        if ((e = hipHostMalloc(reinterpret_cast<void **>(&s.report), sizeof(u32), hipHostMallocDefault)) != hipSuccess)
            return e;
    }
    if (f.grower == BH_LEVELWISE) {
        if ((e = hipMalloc(&s.feat_best, sizeof(SplitRec) * (F + 2))) != hipSuccess) return e;
        if ((e = hipMalloc(&s.level_splits, sizeof(u32) * 3 * 16)) != hipSuccess) return e;
        if ((e = hipMalloc(&s.level_gains, sizeof(float) * 16)) != hipSuccess) return e;
    }
    s.hist_slots = hist_slots;
    return hipSuccess;
}

void ext_free(ExtState &s)
{
    void *p[] = {s.ls.recs, s.ls.pool_gain, s.ls.pool_id, s.ls.free_slots, s.lw, s.feat_best, s.level_splits,
                 s.level_gains};
    for (void *q : p)
        if (q) (void)hipFree(q);
    if (s.report) (void)hipHostFree(s.report);
    s = ExtState{};
}

// The leafwise finders use the device's full per-workgroup LDS like k_find.
hipError_t ext_set_limits()
{
    int dev = 0, max_shared = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&max_shared, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess) return e;
    void const *fns[] = {reinterpret_cast<void const *>(&k_lw_find<true, true, false>),
                         reinterpret_cast<void const *>(&k_lw_find<false, false, false>),
                         reinterpret_cast<void const *>(&k_lw_find<true, true, true>),
                         reinterpret_cast<void const *>(&k_lw_find<false, false, true>)};
    for (void const *fn : fns) {
        hipFuncAttributes a{};
        if (hipFuncGetAttributes(&a, fn) != hipSuccess) continue;
        int const dyn = max_shared - static_cast<int>(a.sharedSizeBytes);
        if (dyn > 0) (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, dyn);
    }
    (void)hipGetLastError();
    return hipSuccess;
}

// ObliviousGrower::grow as a launch sequence (fixed shape: every level is enqueued, a
// stopped tree turns the remaining levels into no-ops).
void enqueue_levelwise(ExtState &s, hipStream_t st, bool q, GrowView const &v)
{
    u32 const D = static_cast<u32>(v.fc.max_depth);
    u32 const gh_bytes = q ? 4 : 8;
    SplitRec *pick = s.feat_best + v.F; // one spare record after the per-feature bests
    launch_tree_begin(st, v.ctl, v.front[0], v.tree, v.hch, v.fops, v.root);
    hipLaunchKernelGGL(k_obl_begin, dim3(1), dim3(64), 0, st, v.ctl);
    launch_hist(st, q, v.hch, v.ctl, v.work[0], v.work[1], v.plane0, v.gh[0], v.gh[1], v.gh[2], v.Fs, v.F, v.SB,
                v.fsl, v.waves, std::max(1u, std::min(v.max_hch, 4096u)), v.partials, v.hist[0], v.fx);
    launch_finish(st, q, v.fops, v.ctl, v.partials, v.hist[1], v.hist[0], v.F * v.SB, 1, nullptr, nullptr, false,
                  hist_transpose_F(q, v.Fs, v.F));
    size_t const lds_level = static_cast<size_t>(v.SB) * level_lds_per_bin(q);
    for (u32 d = 0; d < D; ++d) {
        NodeInfo *cur = v.front[d & 1u], *nxt = v.front[(d + 1) & 1u];
        void *hcur = v.hist[d & 1u], *hnext = v.hist[(d + 1) & 1u];
        u32 const width = 1u << d;
        bool const last = d + 1 == D;
        if (q)
            hipLaunchKernelGGL(k_totals<true>, dim3(width), dim3(64), 0, st, cur, v.ctl, hcur, v.d_nbins, v.F, v.SB,
                               v.gc.fmask, 1u);
        else
            hipLaunchKernelGGL(k_totals<false>, dim3(width), dim3(64), 0, st, cur, v.ctl, hcur, v.d_nbins, v.F, v.SB,
                               v.gc.fmask, 1u);
        if (q)
            hipLaunchKernelGGL(k_find_level<true>, dim3(v.F), dim3(256), lds_level, st, cur, v.ctl, hcur, v.d_nbins, v.F,
                               v.SB, v.gc, v.scales, s.feat_best, 1u);
        else
            hipLaunchKernelGGL(k_find_level<false>, dim3(v.F), dim3(256), lds_level, st, cur, v.ctl, hcur, v.d_nbins,
                               v.F, v.SB, v.gc, v.scales, s.feat_best, 1u);
        hipLaunchKernelGGL(k_level_pick, dim3(1), dim3(256), 0, st, s.feat_best, v.F, v.ctl, s.level_splits,
                           s.level_gains, pick);
        if (q)
            hipLaunchKernelGGL(k_plan_oblivious<true>, dim3(1), dim3(1024), 0, st, cur, v.ctl, pick, hcur, v.d_nbins,
                               v.F, v.SB, v.splits, v.ops, v.pch, d & 1u, last ? 1u : 0u, part_chunk_rows(v.Fs, v.N), 1u);
        else
            hipLaunchKernelGGL(k_plan_oblivious<false>, dim3(1), dim3(1024), 0, st, cur, v.ctl, pick, hcur,
                               v.d_nbins, v.F, v.SB, v.splits, v.ops, v.pch, d & 1u, last ? 1u : 0u,
                               part_chunk_rows(v.Fs, v.N), 1u);
        launch_part_count(st, v.pch, v.ops, v.ctl, v.work[0], v.work[1], v.plane0, v.Fs, v.chunk_left,
                          std::max(1u, std::min(v.max_pch, tuning().part_grid)));
        launch_part_scan(st, q, v.ops, v.pch, v.chunk_left, v.ctl, cur, nxt, v.splits, v.tree, v.hch, v.fops, v.gc,
                         v.scales, last ? 1u : 0u, 1u, v.Fs > 64 ? 1u : 0u);
        if (!last) {
            launch_part_scatter(st, v.pch, v.ops, v.ctl, v.work[0], v.work[1], v.plane0, v.gh[0], v.gh[1], v.gh[2],
                                v.work[0], v.work[1], const_cast<void *>(v.gh[0]), const_cast<void *>(v.gh[1]), v.Fs,
                                gh_bytes, std::max(1u, std::min(v.max_pch, tuning().part_grid)));
            launch_hist(st, q, v.hch, v.ctl, v.work[0], v.work[1], v.plane0, v.gh[0], v.gh[1], v.gh[2], v.Fs, v.F,
                        v.SB, v.fsl, v.waves, std::max(1u, std::min(v.max_hch, 4096u)), v.partials, hnext, v.fx,
                        nullptr, nullptr, false, hcur);
            launch_finish(st, q, v.fops, v.ctl, v.partials, hcur, hnext, v.F * v.SB, std::min(width, v.max_ops),
                          nullptr, nullptr, false, hist_transpose_F(q, v.Fs, v.F));
        }
        hipLaunchKernelGGL(k_next_level_obl, dim3(1), dim3(256), 0, st, v.ctl, cur, nxt);
        if (v.host_sync) (void)hipStreamSynchronize(st);
    }
    if (q)
        hipLaunchKernelGGL(k_oblivious_tree<true>, dim3(1), dim3(1024), 0, st, v.front[D & 1u], v.ctl, s.level_splits,
                           s.level_gains, v.tree, v.gc, v.scales);
    else
        hipLaunchKernelGGL(k_oblivious_tree<false>, dim3(1), dim3(1024), 0, st, v.front[D & 1u], v.ctl,
                           s.level_splits, s.level_gains, v.tree, v.gc, v.scales);
}

// find_level_split as one step over a frontier the host laid out (front[0 .. n) with
// ctl->n_front = n): node totals, the per-feature level scan, the pick (pick[0], valid
// = 0 when no split is feasible), and every node's child sums under the pick in
// v.splits[i] (k_plan_oblivious's last-level arm; its partition ops are not used).
void launch_level_find_step(ExtState &s, hipStream_t st, bool q, GrowView const &v, NodeInfo *front, u32 n,
                            void const *hist, SplitRec *pick)
{
    size_t const lds_level = static_cast<size_t>(v.SB) * level_lds_per_bin(q);
    hipLaunchKernelGGL(k_obl_begin, dim3(1), dim3(64), 0, st, v.ctl);
    if (q) {
        hipLaunchKernelGGL(k_totals<true>, dim3(n), dim3(64), 0, st, front, v.ctl, hist, v.d_nbins, v.F, v.SB,
                           v.gc.fmask, 0u);
        hipLaunchKernelGGL(k_find_level<true>, dim3(v.F), dim3(256), lds_level, st, front, v.ctl, hist, v.d_nbins,
                           v.F, v.SB, v.gc, v.scales, s.feat_best, 0u);
    } else {
        hipLaunchKernelGGL(k_totals<false>, dim3(n), dim3(64), 0, st, front, v.ctl, hist, v.d_nbins, v.F, v.SB,
                           v.gc.fmask, 0u);
        hipLaunchKernelGGL(k_find_level<false>, dim3(v.F), dim3(256), lds_level, st, front, v.ctl, hist, v.d_nbins,
                           v.F, v.SB, v.gc, v.scales, s.feat_best, 0u);
    }
    hipLaunchKernelGGL(k_level_pick, dim3(1), dim3(256), 0, st, s.feat_best, v.F, v.ctl, s.level_splits, s.level_gains,
                       pick);
    if (q)
        hipLaunchKernelGGL(k_plan_oblivious<true>, dim3(1), dim3(1024), 0, st, front, v.ctl, pick, hist, v.d_nbins, v.F,
                           v.SB, v.splits, v.ops, v.pch, 0u, 1u, part_chunk_rows(v.Fs, v.N), 0u);
    else
        hipLaunchKernelGGL(k_plan_oblivious<false>, dim3(1), dim3(1024), 0, st, front, v.ctl, pick, hist, v.d_nbins,
                           v.F, v.SB, v.splits, v.ops, v.pch, 0u, 1u, part_chunk_rows(v.Fs, v.N), 0u);
}

template <bool Q, bool COUNTED>
static void launch_lw_find(hipStream_t st, GrowView const &v, LwCtl *lw, u32 *cnt, LwNext const &nx)
{
    size_t const lds = static_cast<size_t>(kLwFindTile) * v.SB * (Q ? (cnt ? 36 : 32) : 24);
    dim3 const grid(find_blocks_per_node(v.F, kLwFindTile), 2u * kLwBatch);
    bool const con = v.gc.fmask || v.gc.mono || v.gc.n_groups;
    auto const fn = con ? &k_lw_find<Q, COUNTED, true> : &k_lw_find<Q, COUNTED, false>;
    hipLaunchKernelGGL(fn, grid, dim3(kFindThreads), lds, st, v.front[0], v.ctl, lw, v.hist[0], v.d_nbins, v.F, v.SB,
                       v.gc, v.scales, v.splits, v.fscr.part, v.fscr.done, cnt, nx);
}

static LwLists lw_lists(ExtState const &s, GrowView const &v)
{
    LwLists ls = s.ls;
    ls.unit_target = v.lw_units;
    ls.chunk_cap = part_chunk_rows(v.Fs, v.N);
    ls.max_parts = v.lw_parts;
    return ls;
}

u32 lw_head_rounds(GrowView const &v)
{
    u32 const L = static_cast<u32>(v.fc.max_leaves);
    return std::min(L + 7u, (L - 1u + kLwBatch - 1u) / kLwBatch + 4u);
}

// `rounds` rounds; the last one's find reports to the host whether the tree is complete.
// A complete tree turns rounds into no-ops.
void enqueue_leafwise_rounds(ExtState &s, hipStream_t st, bool q, GrowView const &v, u32 rounds)
{
    u32 const gh_bytes = q ? 4 : 8;
    LwCtl *lw = s.lw;
    NodeInfo *kids = v.front[0];
    void *pool = v.hist[0];
    u32 *cnt = q ? v.cnt : nullptr;
    LwLists const ls = lw_lists(s, v);
    u32 const pgrid = std::max(1u, std::min(v.lw_pch, tuning().part_grid));
    u32 const hgrid = std::max(1u, std::min(v.lw_parts, 4096u));
    for (u32 r = 0; r < rounds; ++r) {
        launch_part_count(st, v.pch, v.ops, v.ctl, v.work[0], v.work[1], v.plane0, v.Fs, v.chunk_left, pgrid);
        if (!q)
            hipLaunchKernelGGL(k_lw_scan<false>, dim3(1), dim3(1024), 0, st, v.ops, v.pch, v.chunk_left, v.ctl, lw, ls,
                               kids, v.hch, v.fops, v.gc);
        launch_part_scatter(st, v.pch, v.ops, v.ctl, v.work[0], v.work[1], v.plane0, v.gh[0], v.gh[1], v.gh[2],
                            v.work[0], v.work[1], const_cast<void *>(v.gh[0]), const_cast<void *>(v.gh[1]), v.Fs,
                            gh_bytes, pgrid, q ? v.chunk_left : nullptr);
        launch_hist(st, q, v.hch, v.ctl, v.work[0], v.work[1], v.plane0, v.gh[0], v.gh[1], v.gh[2], v.Fs, v.F, v.SB,
                    v.fsl, v.waves, hgrid, v.partials, pool, v.fx, cnt);
        launch_finish(st, q, v.fops, v.ctl, v.partials, pool, pool, v.F * v.SB, kLwBatch, cnt, cnt, false,
                      hist_transpose_F(q, v.Fs, v.F));
        LwNext const nx{ls, v.tree, v.ops, v.pch, v.hch, v.fops, r + 1 == rounds ? s.report : nullptr};
        if (q) launch_lw_find<true, true>(st, v, lw, cnt, nx);
        else launch_lw_find<false, false>(st, v, lw, cnt, nx);
        if (v.host_sync) (void)hipStreamSynchronize(st);
    }
}

// LeafwiseGrower::grow as a launch sequence: the root, then lw_head_rounds rounds.  More
// may be needed (a chain of leaves each the next best): the caller looks at *s.report
// and adds kLwMoreRounds at a time until the tree is complete.
void enqueue_leafwise(ExtState &s, hipStream_t st, bool q, GrowView const &v)
{
    LwCtl *lw = s.lw;
    NodeInfo *kids = v.front[0];
    void *pool = v.hist[0];
    // Quantized: count cells beside the histogram pool give every split its child row
    // counts (the counted round); FP32: the chunk counts are scanned on the device.
    u32 *cnt = q ? v.cnt : nullptr;
    LwLists const ls = lw_lists(s, v);
    u32 const hgrid = std::max(1u, std::min(v.max_hch, 4096u));
    hipLaunchKernelGGL(k_lw_begin, dim3(1), dim3(256), 0, st, v.ctl, lw, kids, v.tree, v.hch, v.fops, ls.free_slots,
                       s.hist_slots, v.root, v.lw_units);
    launch_hist(st, q, v.hch, v.ctl, v.work[0], v.work[1], v.plane0, v.gh[0], v.gh[1], v.gh[2], v.Fs, v.F, v.SB,
                v.fsl, v.waves, hgrid, v.partials, pool, v.fx, cnt);
    launch_finish(st, q, v.fops, v.ctl, v.partials, pool, pool, v.F * v.SB, 1, cnt, cnt, false,
                      hist_transpose_F(q, v.Fs, v.F));
    launch_find(st, q, kids, v.ctl, pool, v.d_nbins, v.F, v.SB, v.gc, v.scales, v.splits, 2, 0, 0, v.fscr, cnt);
    // The first round's select is a kernel of its own; every later one runs in the last
    // workgroup of the previous round's split find.
    if (q) {
        hipLaunchKernelGGL(k_lw_push_root<true>, dim3(1), dim3(64), 0, st, lw, ls, kids, v.splits, v.tree, v.gc,
                           v.scales);
        hipLaunchKernelGGL(k_lw_select<true>, dim3(1), dim3(256), 0, st, v.ctl, lw, ls, kids, v.splits, v.tree, v.ops,
                           v.pch, v.hch, v.d_nbins, v.fops, v.gc, v.scales);
    } else {
        hipLaunchKernelGGL(k_lw_push_root<false>, dim3(1), dim3(64), 0, st, lw, ls, kids, v.splits, v.tree, v.gc,
                           v.scales);
        hipLaunchKernelGGL(k_lw_select<false>, dim3(1), dim3(256), 0, st, v.ctl, lw, ls, kids, v.splits, v.tree, v.ops,
                           v.pch, v.hch, v.d_nbins, v.fops, v.gc, v.scales);
    }
    enqueue_leafwise_rounds(s, st, q, v, lw_head_rounds(v));
}

} // namespace bh
