// Predict / TreeSHAP plans and the continuous-batching serving loop (H15, H16, cfg4).
//
// A bh_predictor holds one ensemble resident in HBM, packed for each kernel:
//   walk nodes (8 B each) for the bin-space walk of few rows, and LDS tiles of 4-byte nodes
//   for the walk of many,
//   step streams (32 B slots) of whole trees and of their subtrees for TreeSHAP, or leaf
//   paths (8 B elements, 12 B heads) where the ensemble does not fit the tree form.
// Its device data is immutable after creation, so serving streams share it; the buffers of
// small host calls are taken by one call at a time.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/bonsai_hip.h"
#include "bh_common.hpp"

using namespace bh;

namespace {

} // namespace

// The engine's thread-local error slot (bh_last_error).
void bh_set_error(std::string const &m);

namespace {

int sfail(int code, std::string const &m)
{
    bh_set_error(m);
    return code;
}
#define SHIP(expr)                                                                          \
    do {                                                                                    \
        hipError_t const e_ = (expr);                                                       \
        if (e_ != hipSuccess) return sfail(-1, std::string("hip: ") + #expr + ": " + hipGetErrorString(e_)); \
    } while (0)

// Predict walk node: internal {feature, bin, default_left, left, right}; leaf
// {0xFFFF, value}.  Child ids are local to the tree.
struct PNode {
    u16 feature;
    u8 bin;
    u8 dl;
    union {
        struct {
            u16 left, right;
        } c;
        float value;
    } u;
};
static_assert(sizeof(PNode) == 8, "PNode");

// TreeSHAP packed path element / head (src/shap_paths.cpp:33-110 layout).
struct SElem {
    u16 feature; // bit 15: the missing bin satisfies
    u8 lo, hi;
    float z;
};
struct SHead {
    u32 first;
    u16 n;
    u16 klass;
    float value;
};
static_assert(sizeof(SElem) == 8 && sizeof(SHead) == 12, "shap layout");

constexpr int kMaxPath = 16;

// ---------------------------------------------------------------------------------
// Predict: init + lr * sum_t leaf_t(row), the tree sum in tree order, multiply then
// add each rounded (predict_walk_kernel, src/cuda/predict.cu:50-85; host
// predict_at_binned, include/bonsai/booster.hpp:831-846).
//
// Small batches (and any ensemble): a workgroup takes a few rows, its threads walk (row,
// tree) pairs of one tree tile from global memory into LDS, then one thread per row adds
// the tile in tree order.  Latency bound: the walk's dependent node loads and the ordered
// float sum (about 3 us per 1,000 trees); one row per workgroup while the rows alone do
// not fill the chip (walk_shape).
// ---------------------------------------------------------------------------------

__global__ __launch_bounds__(1024) void k_predict_direct(u8 const *__restrict__ bins, u64 n, u64 stride, u32 F,
                                                         u32 rows, u32 tile, PNode const *__restrict__ nodes,
                                                         u32 const *__restrict__ roots, u32 n_trees,
                                                         u16 const *__restrict__ last, float lr, float init,
                                                         float *__restrict__ out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    float *s_val = reinterpret_cast<float *>(smem);                  // [rows][tile]
    u16 *s_last = reinterpret_cast<u16 *>(s_val + rows * tile);      // [F]
    u8 *s_rows = reinterpret_cast<u8 *>(s_last + F);                         // [rows][F]
    u64 const r0 = static_cast<u64>(blockIdx.x) * rows;
    u32 const nr = static_cast<u32>(min<u64>(rows, n - r0));
    for (u32 k = threadIdx.x; k < nr * F; k += blockDim.x) {
        u32 const rr = k / F, f = k - rr * F;
        s_rows[k] = bins[(r0 + rr) * stride + f];
    }
    for (u32 f = threadIdx.x; f < F; f += blockDim.x) s_last[f] = last[f];
    __syncthreads();
    float acc = 0.0F;
    for (u32 t0 = 0; t0 < n_trees; t0 += tile) {
        u32 const tt = min(tile, n_trees - t0);
        for (u32 k = threadIdx.x; k < nr * tt; k += blockDim.x) {
            u32 const rr = k / tt, t = k - rr * tt;
            PNode const *tn = nodes + roots[t0 + t];
            u8 const *row = s_rows + rr * F;
            PNode nd = tn[0];
            while (nd.feature != 0xFFFFu) {
                u32 const b = row[nd.feature];
                bool const left = b == s_last[nd.feature] ? (nd.dl != 0) : (b <= nd.bin);
                nd = tn[left ? nd.u.c.left : nd.u.c.right];
            }
            s_val[rr * tile + t] = nd.u.value;
        }
        __syncthreads();
        if (threadIdx.x < nr) {
            float const *v = s_val + threadIdx.x * tile;
            u32 t = 0;
            for (; t + 16 <= tt; t += 16) {
                float4 q[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) q[k] = reinterpret_cast<float4 const *>(v + t)[k];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    acc += q[k].x;
                    acc += q[k].y;
                    acc += q[k].z;
                    acc += q[k].w;
                }
            }
            for (; t < tt; ++t) acc += v[t];
        }
        __syncthreads();
    }
    if (threadIdx.x < nr) out[r0 + threadIdx.x] = __fadd_rn(init, __fmul_rn(lr, acc));
}

// Larger batches: one row per lane, trees walked from LDS.  The ensemble is laid out in
// tiles of at most kTileNodes 4-byte nodes (and their values); a workgroup keeps ROWS rows
// in LDS and streams the tiles through it, the next tile's loads in flight in registers.
// A leaf is a node whose comparison always holds and whose left child is itself, so a
// walk is a fixed number of steps (the deepest of its trees): one random 4-byte read of
// a node, one random byte of the row and seven vector instructions.  LDS bound: about 11
// clocks per wave step.  With fewer than 1,024 rows the workgroup's 16 waves split each
// tile's trees, leave the values in LDS and the first waves add them in tree order.
// A row's bins are stored shifted, the missing bin as 0, others as bin + 1: with d = 1
// where the missing bin goes right, the row goes left when (shifted - d) as unsigned is
// at most bin + 1 - d.
constexpr u32 kTileNodes = 8192;
constexpr u32 kTileThreads = 1024;
// node: feature | bin + 1 - d (at most 255) << 8 | left child's index in the tile << 16 | d << 31
constexpr u32 tile_row_stride(u32 F) { return ((F + 3u) / 4u | 1u) * 4u; } // odd dwords: lanes' rows spread over banks

struct TileTree {
    u32 root; // index in the tile | levels << 16
};
struct Tile {
    u32 off, count; // first word of its nodes (count of them, then count values), count a multiple of 4
    u32 tree0, n_trees;
};

template <int G> __device__ __forceinline__ void tile_walk(u32 const *s_nodes, u32 count, u8 const *row,
                                                           TileTree const *__restrict__ tt, float (&v)[G])
{
    u32 at[G], steps = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
        u32 const r = __builtin_amdgcn_readfirstlane(tt[g].root);
        at[g] = r & 0xFFFFu;
        steps = max(steps, r >> 16);
    }
    for (u32 k = 0; k < steps; ++k) {
        u32 nd[G], b[G];
#pragma unroll
        for (int g = 0; g < G; ++g) nd[g] = s_nodes[at[g]];
#pragma unroll
        for (int g = 0; g < G; ++g) b[g] = row[nd[g] & 0xFFu];
#pragma unroll
        for (int g = 0; g < G; ++g)
            at[g] = (nd[g] >> 16 & 0x7FFFu) + (b[g] - (nd[g] >> 31) <= (nd[g] >> 8 & 0xFFu) ? 0u : 1u);
    }
#pragma unroll
    for (int g = 0; g < G; ++g) v[g] = reinterpret_cast<float const *>(s_nodes + count)[at[g]];
}

template <u32 ROWS>
__global__ __launch_bounds__(kTileThreads) void k_predict_tile(u8 const *__restrict__ bins, u64 n, u64 stride, u32 F,
                                                               u32 const *__restrict__ words,
                                                               Tile const *__restrict__ tiles, u32 n_tiles,
                                                               TileTree const *__restrict__ trees,
                                                               u16 const *__restrict__ last, float lr, float init,
                                                               float *__restrict__ out)
{
    constexpr u32 S = kTileThreads / ROWS; // waves of one row group that split a tile's trees
    constexpr u32 NW = 2 * kTileNodes / 4 / kTileThreads; // 16-byte words of a tile per thread
    extern __shared__ __align__(16) unsigned char smem[];
    u32 *s_nodes = reinterpret_cast<u32 *>(smem);                       // 2 * kTileNodes: nodes, then values
    float *s_out = reinterpret_cast<float *>(s_nodes + 2 * kTileNodes); // S > 1: [2][S * 4][ROWS]
    u8 *s_rows = reinterpret_cast<u8 *>(s_out + (S > 1 ? 2 * S * 4 * ROWS : 0)); // [ROWS][RS]
    u32 const RS = tile_row_stride(F);
    u64 const r0 = static_cast<u64>(blockIdx.x) * ROWS;
    u32 const nr = static_cast<u32>(min<u64>(ROWS, n - r0));
    uint4 pf[NW];
    auto fetch = [&](Tile const &t) {
        uint4 const *src = reinterpret_cast<uint4 const *>(words + t.off);
#pragma unroll
        for (u32 k = 0; k < NW; ++k) {
            u32 const i = threadIdx.x + k * kTileThreads;
            pf[k] = i < t.count / 2u ? src[i] : make_uint4(0, 0, 0, 0);
        }
    };
    Tile tile = tiles[0];
    fetch(tile);
    for (u32 k = threadIdx.x; k < ROWS * F; k += kTileThreads) {
        u32 const rr = k / F, f = k - rr * F;
        u32 const b = rr < nr ? bins[(r0 + rr) * stride + f] : 0u;
        s_rows[rr * RS + f] = static_cast<u8>(b == last[f] ? 0u : min(b + 1u, 255u));
    }
    u32 const rr = threadIdx.x % ROWS;
    u32 const s = __builtin_amdgcn_readfirstlane(threadIdx.x / ROWS);
    u8 const *row = s_rows + rr * RS;
    float acc = 0.0F;
    u32 buf = 0;
    for (u32 i = 0; i < n_tiles; ++i) {
        __syncthreads(); // the previous tile is walked
#pragma unroll
        for (u32 k = 0; k < NW; ++k) {
            u32 const w = threadIdx.x + k * kTileThreads;
            if (w < tile.count / 2u) reinterpret_cast<uint4 *>(s_nodes)[w] = pf[k];
        }
        u32 const count = tile.count, t0 = tile.tree0, t1 = tile.tree0 + tile.n_trees;
        if (i + 1 < n_tiles) {
            tile = tiles[i + 1];
            fetch(tile);
        }
        __syncthreads();
        if constexpr (S == 1) {
            u32 t = t0;
            for (; t + 4 <= t1; t += 4) {
                float v[4];
                tile_walk<4>(s_nodes, count, row, trees + t, v);
                acc += v[0];
                acc += v[1];
                acc += v[2];
                acc += v[3];
            }
            for (; t < t1; ++t) {
                float v[1];
                tile_walk<1>(s_nodes, count, row, trees + t, v);
                acc += v[0];
            }
        } else {
            // g trees per wave and round; a round's values are added while the next is
            // walked into the other buffer
            u32 const g = t1 - t0 >= 4u * S ? 4u : (t1 - t0 >= 2u * S ? 2u : 1u);
            for (u32 t = t0; t < t1; t += g * S) {
                float *o = s_out + buf * (S * 4 * ROWS);
                u32 const mine = t + s * g, end = min(t1, mine + g);
                if (mine + 4 <= end) {
                    float v[4];
                    tile_walk<4>(s_nodes, count, row, trees + mine, v);
#pragma unroll
                    for (u32 k = 0; k < 4; ++k) o[(s * g + k) * ROWS + rr] = v[k];
                } else if (mine + 2 == end) {
                    float v[2];
                    tile_walk<2>(s_nodes, count, row, trees + mine, v);
                    o[s * g * ROWS + rr] = v[0];
                    o[(s * g + 1) * ROWS + rr] = v[1];
                } else {
                    for (u32 k = mine; k < end; ++k) {
                        float v[1];
                        tile_walk<1>(s_nodes, count, row, trees + k, v);
                        o[(k - t) * ROWS + rr] = v[0];
                    }
                }
                __syncthreads();
                if (s == 0) {
                    u32 const m = min(g * S, t1 - t);
                    for (u32 k = 0; k < m; ++k) acc += o[k * ROWS + rr];
                }
                buf ^= 1u;
            }
        }
    }
    if (s == 0 && rr < nr) out[r0 + rr] = __fadd_rn(init, __fmul_rn(lr, acc));
}

// ---------------------------------------------------------------------------------
// TreeSHAP, packed closed form (eval_shap_paths, src/shap_paths.cpp:196-278):
//   P(t) = prod_j (z_j + o_j t);  unsatisfied element: -value * sum_i w_i [t^i] P;
//   satisfied element: value * (1 - z) * sum_i w_i [t^i] (P / (t + z)).
// Paths are packed in groups of 64, element j of the group's paths stored contiguously
// ([group][j][lane]), so one coalesced load gives every lane its path's element.  A
// workgroup serves kShapRows rows: each lane loads a path once and applies it to all of
// them.  Contributions are accumulated as 64-bit fixed point (value x scale, scale from
// the ensemble's leaf magnitudes) with LDS integer atomics: exact and order-free, so a
// row's result does not depend on the order of the adds or on what shares its batch.
// ---------------------------------------------------------------------------------
constexpr u32 kShapRows = 32;
// A launch with fewer row blocks than this splits each block's path groups over more
// workgroups, so small batches still spread over the chip.
constexpr u32 kShapFillBlocks = 2048;

// φ of one cell from its 64-bit fixed-point sum.
__device__ __forceinline__ double shap_from_fixed(unsigned long long v, double scale, float lr)
{
    return static_cast<double>(static_cast<long long>(v)) / scale * static_cast<double>(lr);
}

// Serves the ensembles the tree form (below) does not take.  KM: compile-time bound on the
// path length (8 or 16), so every per-path array lives in registers.
template <int KM>
__global__ __launch_bounds__(256) void k_shap(u8 const *__restrict__ bins, u64 n, u64 stride, u32 F,
                                              SElem const *__restrict__ elems, SHead const *__restrict__ heads,
                                              u32 n_groups, u32 K, float const *__restrict__ weights,
                                              u16 const *__restrict__ last, float lr, double bias, double scale,
                                              double *__restrict__ out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned long long *s_phi = reinterpret_cast<unsigned long long *>(smem); // [kShapRows][F] fixed point
    u8 *s_row = reinterpret_cast<u8 *>(s_phi + kShapRows * F);                 // [kShapRows][F]
    u64 const r0 = static_cast<u64>(blockIdx.x) * kShapRows;
    if (r0 >= n) return;
    u32 const nr = static_cast<u32>(min<u64>(kShapRows, n - r0));
    for (u32 k = threadIdx.x; k < kShapRows * F; k += blockDim.x) s_phi[k] = 0ull;
    for (u32 k = threadIdx.x; k < nr * F; k += blockDim.x) {
        u32 const rr = k / F, f = k - rr * F;
        s_row[k] = bins[(r0 + rr) * stride + f];
    }
    __syncthreads();
    // gridDim.y workgroups share a row block, each taking every gridDim.y-th set of
    // NW path groups.
    u32 const wave = threadIdx.x >> 6, lane = threadIdx.x & 63u, NW = blockDim.x >> 6;
    for (u32 g = blockIdx.y * NW + wave; g < n_groups; g += NW * gridDim.y) {
        SHead const hd = heads[static_cast<size_t>(g) * 64u + lane];
        u32 const nel = hd.n;
        // The group's longest path (wave-uniform): the 16-slot body skips element slots past
        // it; the 8-slot one runs them all (its branches would cost a quarter more).
        u32 nmax = nel;
        for (int o = 32; o > 0; o >>= 1) nmax = max(nmax, static_cast<u32>(__shfl_xor(static_cast<int>(nmax), o)));
        nmax = __builtin_amdgcn_readfirstlane(nmax);
        if (nmax == 0) continue;
        // Slots past a lane's path hold a neutral element: z = 1 and never satisfied
        // (lo > hi, a missing bin no byte equals), so it multiplies P(t) by exactly 1 and
        // its deflation terms are exact zeros (P's coefficients past the path are 0, as
        // are its weights).  No per-lane guard is needed until the contribution's add.
        u32 feat[KM], lo[KM], hi[KM], lst[KM];
        bool miss[KM];
        float z[KM], wl[KM], vz[KM];
        float const *w = weights + (nel - 1) * nel / 2;
        // The leaf value in fixed-point units, rounded once to float: each contribution
        // is then a float product of the path's float polynomial terms, rounded to the
        // 64-bit accumulator's integer grid (|value| * scale <= 2^59).
        float const vs = static_cast<float>(static_cast<double>(hd.value) * scale);
#pragma unroll
        for (int j = 0; j < KM; ++j) {
            feat[j] = 0;
            lo[j] = 1;
            hi[j] = 0;
            lst[j] = 0xFFFFFFFFu;
            miss[j] = false;
            z[j] = 1.0F;
            wl[j] = 0.0F;
            vz[j] = 0.0F;
            if (static_cast<u32>(j) < nel) {
                SElem const e = elems[(static_cast<size_t>(g) * K + j) * 64u + lane];
                feat[j] = e.feature & 0x7FFFu;
                miss[j] = (e.feature & 0x8000u) != 0;
                lo[j] = e.lo;
                hi[j] = e.hi;
                lst[j] = last[feat[j]]; // the element's missing bin, read once per path
                z[j] = e.z;
                wl[j] = w[j];
                vz[j] = vs * (1.0F - e.z); // a satisfied element's factor before its sum
            }
        }
        // Lanes start on different rows, so one atomic instruction spreads over the
        // rows' accumulators instead of piling onto one row's few features.
        u32 rr = lane % nr;
        for (u32 r = 0; r < nr; ++r, rr = rr + 1 == nr ? 0u : rr + 1) {
            u8 const *row = s_row + rr * F;
            unsigned long long *phi = s_phi + rr * F;
            float poly[KM + 1];
            bool sat[KM];
#pragma unroll
            for (int j = 0; j <= KM; ++j) poly[j] = j == 0 ? 1.0F : 0.0F;
#pragma unroll
            for (int j = 0; j < KM; ++j) {
                sat[j] = false;
                if (KM <= 8 || static_cast<u32>(j) < nmax) {
                    u32 const b = row[feat[j]];
                    bool const one = b == lst[j] ? miss[j] : (b >= lo[j] && b <= hi[j]);
                    sat[j] = one;
                    // multiply by (z + o t)
                    float const zj = z[j];
#pragma unroll
                    for (int i = KM; i >= 1; --i)
                        if (i <= j + 1) poly[i] = __builtin_fmaf(zj, poly[i], one ? poly[i - 1] : 0.0F);
                    poly[0] *= zj;
                }
            }
            float unsat = 0.0F;
#pragma unroll
            for (int i = 0; i < KM; ++i) unsat = __builtin_fmaf(wl[i], poly[i], unsat); // wl[i] = 0 beyond the path
            float const nu = -vs * unsat;
#pragma unroll
            for (int k = 0; k < KM; ++k) {
                if (KM <= 8 || static_cast<u32>(k) < nmax) {
                    // synthetic division by (t + z_k), from the top: deflated[i] =
                    // P[i+1] - z_k deflated[i+1], zero above the path's degree; used only
                    // where element k is satisfied (P then holds the factor t + z_k)
                    float const nzk = -z[k];
                    float sdef = 0.0F, prev = 0.0F;
#pragma unroll
                    for (int i = KM - 1; i >= 0; --i) {
                        if (KM <= 8 || static_cast<u32>(i) < nmax) {
                            prev = __builtin_fmaf(nzk, prev, poly[i + 1]);
                            sdef = __builtin_fmaf(wl[i], prev, sdef);
                        }
                    }
                    float const c = sat[k] ? vz[k] * sdef : nu;
                    if (static_cast<u32>(k) < nel)
                        atomicAdd(phi + feat[k], static_cast<unsigned long long>(__float2ll_rn(c)));
                }
            }
        }
    }
    __syncthreads();
    if (gridDim.y > 1) {
        // Path groups split over workgroups: the block's fixed-point sums go into the
        // zeroed output cells with 64-bit integer atomics (exact in any order), and
        // k_shap_to_double converts them once every workgroup has added its share.
        unsigned long long *acc = reinterpret_cast<unsigned long long *>(out);
        for (u32 k = threadIdx.x; k < nr * F; k += blockDim.x) {
            u32 const rr = k / F, f = k - rr * F;
            if (s_phi[k] != 0ull) atomicAdd(acc + (r0 + rr) * (F + 1) + f, s_phi[k]);
        }
        return;
    }
    for (u32 k = threadIdx.x; k < nr * F; k += blockDim.x) {
        u32 const rr = k / F, f = k - rr * F;
        out[(r0 + rr) * (F + 1) + f] = shap_from_fixed(s_phi[k], scale, lr);
    }
    for (u32 rr = threadIdx.x; rr < nr; rr += blockDim.x) out[(r0 + rr) * (F + 1) + F] = bias;
}

// ---------------------------------------------------------------------------------
// TreeSHAP, tree form: one row per lane, a wave walks whole trees.
//
// The closed form's sum over coefficients is an integral: w_i = 1 / (n C(n-1, i)) is
// the Beta integral of x^i (1-x)^(n-1-i) over [0, 1], so element k's term is
//   value (o_k - z_k) * integral of prod_{j != k} (z_j (1-x) + o_j x) dx,
// a polynomial of degree n - 1 that M >= n/2 Gauss-Legendre nodes x_q integrate exactly.
// At a fixed x_q the paths' products factor over the tree's edges, so they are formed
// once per edge and shared by every path through it (the edge-sharing of Linear
// TreeSHAP, Yu et al. 2022, at quadrature points instead of in coefficient form).  For
// an internal node whose child c holds the cover fraction z_c and s_c = 1 on the row's
// side, with T_q the product above the node and H_q(c) the values below c:
//   M = sum_c z_c H(c), S = sum_c s_c H(c), d = S - M,
//   H(node) = M + k_q d,  T(c) = T(node) (z_c + k_q (s_c - z_c)),
//   phi[feature] += sum_q T_q(node) l_q d_q,
// k_q = x_q and l_q = 1 when no edge above splits on the node's feature.  When one does,
// its edge carries the merged fraction z' and satisfaction o' of that feature: o' = 0
// turns k and l into 0, o' = 1 gives k_q = x_q / a, l_q = z' / a^2, a = z' + x_q (1 - z').
// Nodes past 1/2 use 1 - k_q, which floats hold more exactly: H = S - (1 - k) d,
// T(c) = T(node) (s_c - (1 - k) (s_c - z_c)); the weights carry a common factor that
// makes them nearly exact in float (tree_quad), so neither adds a systematic error.
//
// Lanes are rows and a wave's control flow and node records are uniform.  Bound by vector
// issue: 14,900 wave instructions per 255-node tree and 64 rows (about 58 a node, against
// some 265 a path of the packed form) at 4 clocks each are 6.2 of the 7.6 ms that 16,384
// rows of 1,000 such trees take (packed form 28.4 ms).  Contributions go through float to
// 64-bit fixed point and into LDS with conflict-free integer atomics: exact in any order, so
// a row's result depends neither on the batch nor on how trees are dealt to waves and
// workgroups.  The grid is never coarser than the packed form's (tree_grid): where the
// largest leaf stands among many (Sum |leaf| of some 2^11 of it) one FP64 add against
// 1.5 * 2^52 rounds to it, otherwise (WIDE: few trees, or one leaf far above the rest) a
// conversion of the whole 64 bits does, which takes the batch above 5% longer (8.0 ms).
// ---------------------------------------------------------------------------------
// A tree is stored as the steps of its depth-first walk, read as one sequential stream:
//   block    a subtree of at most three levels, as seven nodes in one straight run of
//            instructions (a shallower leaf becomes nodes that split it into itself)
//   enter    a node above the blocks: its decision, T of the child walked first
//   turn     its left child is done: keep its value, T of the right child
//   combine  its right child is done (or is a leaf): the node's value and contribution
// so one product T and one left value per level above the blocks stay in registers.  A wave holds 64 consecutive
// 32-byte slots of the stream in registers, one per lane (the next 64 in flight), and
// broadcasts the words a step needs with v_readlane.  A node with a same-feature edge
// above has its k and l in slots after the step's own; a step never crosses a group of
// 64 slots (kTSkip pads).
// ---------------------------------------------------------------------------------
struct TSlot {
    u32 w[8];
};
// Words of a step.  op: kind | level << 2 | dup bit of node i << (8 + i).
// lv: level of the same-feature edge above node i << 4 i.  Splits: byte offset of the
// bin column (shifted plane where the missing bin goes left) | first bin going right << 16.
enum : u32 {
    kTEnter = 0, kTTurn = 1, kTCombine = 2, kTBlock = 3, kTSkip = 15,
    kTLeafL = 0x10000u, kTLeafR = 0x20000u, // enter / combine: that child is a leaf
    kTOnlyL = 0x40000u, kTOnlyR = 0x80000u, // enter: the way down to a share goes there only
    kTHeldL = 0x100000u, kTHeldR = 0x200000u, // with kTLeaf: a share's value, kept in LDS
    kTwOp = 0, kTwLv = 1, kTwSplit = 2,
    kTwZl = 3, kTwZr = 4, kTwVl = 5, kTwVr = 6,          // enter, turn, combine
    kTwZ = 9, kTwMean = 15, kTwLeaf = 19, kTwBlock = 27, // block: z of 3 nodes, means of 4, 8 leaves
};
constexpr u32 kTBlockLevels = 3;
constexpr u32 tree_dup_slots(u32 m) { return (2u * m + 7u) / 8u; }
constexpr u32 tree_step_slots(u32 kind) { return kind == kTBlock ? (kTwBlock + 7u) / 8u : 1u; }
constexpr u32 kTreeShapRows = 64; // rows of a workgroup, one per lane
// Four waves a workgroup, three workgroups a CU (168 registers a lane; with 512-thread
// workgroups and two waves per SIMD the batch above takes 9.0 ms); deep trees keep more
// levels in registers and run one.
constexpr u32 kTreeShapThreads = 256;
constexpr u32 tree_shap_waves(u32 upper) { return upper <= 5u ? 3u : 1u; }
constexpr u32 kTreeShapMaxM = 6;      // quadrature nodes: paths of up to 12 features
constexpr u32 kTreeShapMaxDepth = 12;
// LDS of a workgroup: 64-bit sums, bins, and bins with the missing bin moved to 0.
constexpr size_t tree_shap_lds(u32 F) { return static_cast<size_t>(kTreeShapRows) * F * 10u; }

// Quadrature of M nodes, ascending: y = x for the first half, 1 - x past 1/2; weights
// times a common factor.
struct TQuad {
    float y[kTreeShapMaxM], w[kTreeShapMaxM];
};

// A row's arithmetic at a split, and at the seven of a block; D reads the running step's
// words (word, dup_word), the row's bin and its sum of the column a split names (bin_at,
// phi_at).  WIDE: contributions of up to 63 bits (tree_grid).
template <class D, int M, bool WIDE> struct ShapRow {
    typedef float V[M];
    u32 op;              // the running step's first word
    V y;                 // quadrature nodes (TQuad)
    u32 sat;             // bit l: the row satisfies the merged feature of the edge below level l

    __device__ __forceinline__ D const &d() const { return static_cast<D const &>(*this); }
    __device__ __forceinline__ float fword(u32 j) const { return __uint_as_float(d().word(j)); }
    static __device__ __forceinline__ float keep(float v, u32 m) { return __uint_as_float(__float_as_uint(v) & m); }
    static __device__ __forceinline__ float pick(u32 m, float a, float b)
    {
        return __uint_as_float((__float_as_uint(a) & m) | (__float_as_uint(b) & ~m));
    }

    __device__ __forceinline__ u32 goes_left(u32 split) const
    {
        return d().bin_at(split & 0xFFFFu) < split >> 16 ? ~0u : 0u;
    }

    __device__ __forceinline__ void add(u32 split, float c)
    {
        unsigned long long q;
        if (WIDE) { // round(c) as hi * 2^32 + lo, exactly
            double const v = __builtin_rintf(c), hi = __builtin_floor(v * 0x1p-32);
            u32 const lo = static_cast<u32>(__builtin_fma(hi, -0x1p32, v));
            q = static_cast<unsigned long long>(static_cast<u32>(static_cast<int>(hi))) << 32 | lo;
        } else { // |c| < 2^51: the sum's low 52 bits hold round(c) beside 1.5 * 2^52's own
            double const v = static_cast<double>(c) + 6755399441055744.0;
            q = static_cast<unsigned long long>(__double_as_longlong(v)) - 0x4338000000000000ull;
        }
        atomicAdd(d().phi_at(split & 0xFFFFu), q);
    }

    static constexpr bool past_half(int q) { return 2 * q >= M + (M & 1); }
    // value at k_q between a (k = 0) and b (k = 1), slope = b - a
    static __device__ __forceinline__ float mix(int q, float k, float slope, float a, float b)
    {
        return past_half(q) ? __builtin_fmaf(-k, slope, b) : __builtin_fmaf(k, slope, a);
    }

    // A node's same-feature edge above: none, or where its constants are.  Lane masks are
    // words and constants are read before use: selects of bools would become branches.
    struct Dup {
        bool is;
        u32 slot, level;
    };
    // all ones where the row satisfies the merged feature of that edge
    __device__ __forceinline__ u32 dup_sat(Dup const &u) const
    {
        return static_cast<u32>(__builtin_amdgcn_sbfe(static_cast<int>(sat), u.level, 1u));
    }
    // its k_q (or 1 - k_q) there, else k_q = 0
    __device__ __forceinline__ float dup_k(Dup const &u, int q, u32 o) const
    {
        u32 const k = d().dup_word(q, u.slot);
        return __uint_as_float(past_half(q) ? (k & o) | (0x3F800000u & ~o) : k & o);
    }
    __device__ __forceinline__ float dup_l(Dup const &u, int q) const { return __uint_as_float(d().dup_word(M + q, u.slot)); }

    // A node's k_q (1 - k_q past the half) for every row.
    __device__ __forceinline__ void consts(V &k, Dup const &u) const
    {
        if (u.is) {
            u32 const o = dup_sat(u);
#pragma unroll
            for (int q = 0; q < M; ++q) k[q] = dup_k(u, q, o);
        } else {
#pragma unroll
            for (int q = 0; q < M; ++q) k[q] = y[q];
        }
    }

    // T of the child taken by the rows of m, with cover fraction zc
    static __device__ __forceinline__ void descend(V const &Tn, V &Tc, V const &k, u32 m, float zc)
    {
        float const sc = keep(1.0F, m);
        float const e = sc - zc;
#pragma unroll
        for (int q = 0; q < M; ++q) Tc[q] = Tn[q] * mix(q, k[q], e, zc, sc);
    }
    // the edge to that child at `level`: what same-feature nodes below it test
    __device__ __forceinline__ void mark(u32 m, u32 level, Dup const &u)
    {
        if (u.is) m &= dup_sat(u);
        u32 const bit = 1u << level;
        sat = (m & bit) | (sat & ~bit);
    }

    // Value and contribution of a node from its children's values.
    __device__ __forceinline__ void join(V const &Tn, V const &k, V const &L, V const &R, V &out, u32 m, float zl,
                                         float zr, u32 split, Dup const &u)
    {
        V d;
#pragma unroll
        for (int q = 0; q < M; ++q) {
            float const mean = __builtin_fmaf(zr, R[q], zl * L[q]);
            float const S = pick(m, L[q], R[q]);
            d[q] = S - mean;
            out[q] = mix(q, k[q], d[q], mean, S);
        }
        float c = 0.0F;
        if (u.is) {
#pragma unroll
            for (int q = 0; q < M; ++q) c = __builtin_fmaf(Tn[q] * dup_l(u, q), d[q], c);
            c = keep(c, dup_sat(u));
        } else {
#pragma unroll
            for (int q = 0; q < M; ++q) c = __builtin_fmaf(Tn[q], d[q], c);
        }
        add(split, c);
    }

    // Value and contribution of a node whose children are leaves, below the edge of the
    // rows of em (fraction ze) of a node with product Tn and constants k: without a
    // same-feature edge above, its product is only needed summed over q, which is
    // ze a0 + e a1 with a0 = sum Tn_q, a1 = sum Tn_q k_q.
    __device__ __forceinline__ void leaves(V const &Tn, V const &k, float a0, float a1, u32 em, float ze, V &out,
                                           u32 m, float vl, float vr, float mean, u32 split, Dup const &u)
    {
        float const S = pick(m, vl, vr);
        float const d = S - mean;
        float t;
        if (u.is) {
            V Tc;
            descend(Tn, Tc, k, em, ze);
            u32 const o = dup_sat(u);
            t = 0.0F;
#pragma unroll
            for (int q = 0; q < M; ++q) {
                t = __builtin_fmaf(Tc[q], dup_l(u, q), t);
                out[q] = mix(q, dup_k(u, q, o), d, mean, S);
            }
            t = keep(t, o);
        } else {
            t = __builtin_fmaf(ze, a0 - a1, keep(a1, em));
#pragma unroll
            for (int q = 0; q < M; ++q) out[q] = mix(q, y[q], d, mean, S);
        }
        add(split, t * d);
    }

    // Seven nodes in preorder (r; a, a0, a1; b, b0, b1) below the product Tr.
    __device__ __forceinline__ void block(V const &Tr, V &H, u32 level)
    {
        u32 const lv = d().word(kTwLv);
        u32 split[7], m[7];
        Dup u[7];
        u32 slot = tree_step_slots(kTBlock);
#pragma unroll
        for (int i = 0; i < 7; ++i) {
            split[i] = d().word(kTwSplit + i);
            m[i] = goes_left(split[i]);
            u[i] = Dup{(op >> (8 + i) & 1u) != 0, slot, lv >> (4 * i) & 15u};
            slot += u[i].is ? tree_dup_slots(M) : 0u;
        }
        float z[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) z[i] = fword(kTwZ + i);
        V kr, ka, Ta, H0, H1, Ha;
        consts(kr, u[0]);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            int const n = 1 + 3 * s; // a, then b
            u32 const me = s ? ~m[0] : m[0];
            descend(Tr, Ta, kr, me, z[s]);
            mark(me, level, u[0]);
            consts(ka, u[n]);
            float a0 = 0.0F, a1 = 0.0F;
#pragma unroll
            for (int q = 0; q < M; ++q) {
                a0 += Ta[q];
                a1 = past_half(q) ? a1 + __builtin_fmaf(-ka[q], Ta[q], Ta[q]) : __builtin_fmaf(ka[q], Ta[q], a1);
            }
            mark(m[n], level + 1u, u[n]);
            leaves(Ta, ka, a0, a1, m[n], z[2 + 2 * s], H0, m[n + 1], fword(kTwLeaf + 4 * s), fword(kTwLeaf + 4 * s + 1),
                   fword(kTwMean + 2 * s), split[n + 1], u[n + 1]);
            mark(~m[n], level + 1u, u[n]);
            leaves(Ta, ka, a0, a1, ~m[n], z[3 + 2 * s], H1, m[n + 2], fword(kTwLeaf + 4 * s + 2),
                   fword(kTwLeaf + 4 * s + 3), fword(kTwMean + 2 * s + 1), split[n + 2], u[n + 2]);
            join(Ta, ka, H0, H1, s ? H : Ha, m[n], z[2 + 2 * s], z[3 + 2 * s], split[n], u[n]);
        }
        join(Tr, kr, Ha, H, H, m[0], z[0], z[1], split[0], u[0]);
    }
};

// A wave's walk.  U: levels above the blocks.  AT: the walk may start below a tree's root
// (levels come from the steps) and meet shares' values.
template <int M, int U, bool WIDE, bool AT = false>
struct TreeShap : ShapRow<TreeShap<M, U, WIDE, AT>, M, WIDE> {
    using Row = ShapRow<TreeShap<M, U, WIDE, AT>, M, WIDE>;
    using typename Row::Dup;
    using typename Row::V;
    using Row::fword;
    using Row::op; // uniform
    u8 const *bins;      // LDS: this lane's column of the bins
    unsigned char *phi;  // LDS: this lane's column of the sums
    u32 plane;           // bytes of one plane of bins
    TSlot const *ahead;  // this lane's slot of the group after the next
    uint4 nx0, nx1;      // its slot of the next group, in flight
    u32 cur[8];          // its slot of the current group
    u32 at;              // the running step's slot in it (uniform)
    float *held;         // AT: LDS, this lane's column of the shares' values [share][M][64]

    __device__ __forceinline__ u32 bin_at(u32 col) const { return bins[col]; }
    __device__ __forceinline__ unsigned long long *phi_at(u32 col) const
    {
        return reinterpret_cast<unsigned long long *>(phi + min(col, col - plane) * 8u);
    }
    __device__ __forceinline__ void load()
    {
        uint4 const *p = reinterpret_cast<uint4 const *>(ahead);
        nx0 = p[0];
        nx1 = p[1];
        ahead += 64;
    }
    __device__ __forceinline__ void shift()
    {
        cur[0] = nx0.x;
        cur[1] = nx0.y;
        cur[2] = nx0.z;
        cur[3] = nx0.w;
        cur[4] = nx1.x;
        cur[5] = nx1.y;
        cur[6] = nx1.z;
        cur[7] = nx1.w;
        load(); // whole groups of 64 slots are allocated, and two past the last
    }
    // The step at `at`: a skip or the group's end moves on to the next group.
    __device__ __forceinline__ void fetch()
    {
        op = at < 64u ? __builtin_amdgcn_readlane(cur[kTwOp], at & 63u) : kTSkip << 2;
        if ((op >> 2 & 15u) == kTSkip) {
            shift();
            at = 0;
            op = __builtin_amdgcn_readlane(cur[kTwOp], 0);
        }
    }
    __device__ __forceinline__ void advance(u32 slots)
    {
        at += slots + __popc(op >> 8 & 0x7Fu) * tree_dup_slots(M);
    }

    // word j (a constant) of the slots from `slot` after the step's first
    __device__ __forceinline__ u32 word(u32 j, u32 slot = 0) const
    {
        return __builtin_amdgcn_readlane(cur[j & 7u], at + slot + (j >> 3));
    }
    __device__ __forceinline__ u32 dup_word(u32 j, u32 slot) const { return word(j, slot); }

    // The subtree whose first step is fetched, at level L below the product Tn.  Each
    // level is one copy of this code: its two children are two trips of a loop.
    template <int L> __device__ __forceinline__ void walk(V const &Tn, V &H)
    {
        if (L == U || (op & 3u) == kTBlock) {
            this->block(Tn, H, level_of<L>());
            advance(tree_step_slots(kTBlock));
            return;
        }
        if constexpr (L < U) {
            u32 const m = this->goes_left(word(kTwSplit));
            V HL;
#pragma clang loop unroll(disable)
            for (u32 side = 0; side < 2u; ++side) {
                if (op & (kTLeafL << side)) {
                    float const v = side ? fword(kTwVr) : fword(kTwVl);
                    if (AT && (op & (kTHeldL << side))) {
                        float const *h = held + static_cast<u32>(v) * (M * 64u);
#pragma unroll
                        for (int q = 0; q < M; ++q) H[q] = h[q * 64];
                    } else {
#pragma unroll
                        for (int q = 0; q < M; ++q) H[q] = v;
                    }
                } else {
                    V Tc;
                    V k;
                    u32 const me = side ? ~m : m;
                    this->consts(k, dup_of<L>());
                    Row::descend(Tn, Tc, k, me, side ? fword(kTwZr) : fword(kTwZl));
                    this->mark(me, level_of<L>(), dup_of<L>());
                    advance(1);
                    fetch();
                    walk<L + 1>(Tc, H);
                    fetch();
                }
                if (side == 0) {
#pragma unroll
                    for (int q = 0; q < M; ++q) HL[q] = H[q];
                }
            }
            V k;
            this->consts(k, dup_of<L>());
            this->join(Tn, k, HL, H, H, m, fword(kTwZl), fword(kTwZr), word(kTwSplit), dup_of<L>());
            advance(1);
        }
    }
    template <int L> __device__ __forceinline__ Dup dup_of() const
    {
        return Dup{(AT || L > 0) && (op & 0x100u) != 0, 1u, word(kTwLv)};
    }
    template <int L> __device__ __forceinline__ u32 level_of() const { return AT ? op >> 2 & 15u : L; }

    // Starts reading at slot pc.
    __device__ __forceinline__ void seek(TSlot const *slots, u32 pc)
    {
        ahead = slots + (pc & ~63u) + (threadIdx.x & 63u);
        load();
        shift();
        at = pc & 63u;
        this->sat = 0;
    }
    // The way from a tree's root down to the share whose steps follow.
    __device__ __forceinline__ void go_down(V &T)
    {
        while ((op & 3u) == kTEnter && (op & (kTOnlyL | kTOnlyR))) {
            bool const right = (op & kTOnlyR) != 0;
            u32 const m = this->goes_left(word(kTwSplit)), me = right ? ~m : m;
            V k, Tc;
            this->consts(k, dup_of<0>());
            Row::descend(T, Tc, k, me, right ? fword(kTwZr) : fword(kTwZl));
            this->mark(me, level_of<0>(), dup_of<0>());
#pragma unroll
            for (int q = 0; q < M; ++q) T[q] = Tc[q];
            advance(1);
            fetch();
        }
    }
};

// Deep trees (past kSplitAbove levels), few row blocks x trees.  A walk is one serial chain
// (0.27 us a split), so a batch with fewer of them than the chip has room for waves waits
// for one tree's: 280 us at depth 10 whatever the batch.  Here a workgroup takes one tree of
// a row block: its 8 waves walk the tree's shares (the subtrees below a cut, each with the
// product T carried down to it), leave their values in LDS, and the first wave walks the
// splits above the cut over them.  Every split's arithmetic is the walk's own, so a row's
// bits are the same either way.  128 rows x 100 depth-10 trees 283 -> 76 us, 64 rows x 100
// of depth 12 1,170 -> 250.  Shallower trees' few rows take k_shap_lanes at less (depth 8,
// 256 rows x 100 trees: 33 us, 54 so).
constexpr u32 kSplitAbove = 8;
struct SplitTree {
    u32 share0, n_shares, top; // first share, shares, first slot of the steps above (kNone: none)
    u32 pad;
};
constexpr u32 kSplitThreads = 512;   // 16 waves a workgroup spill (128 registers): a sixth slower at depth 8
constexpr u32 kSplitLevels = 6; // cut at most this far below the root (TreePacker::cut_of)
template <int M, bool WIDE>
__global__ __launch_bounds__(kSplitThreads) void k_shap_split(u8 const *__restrict__ bins, u64 n, u64 stride, u32 F,
                                                             u16 const *__restrict__ last,
                                                             TSlot const *__restrict__ slots,
                                                             u32 const *__restrict__ first,
                                                             SplitTree const *__restrict__ trees, u32 n_trees,
                                                             TQuad quad, double *__restrict__ out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned long long *s_phi = reinterpret_cast<unsigned long long *>(smem); // [F][64] fixed point
    float *s_held = reinterpret_cast<float *>(s_phi + kTreeShapRows * F);      // [shares][M][64]
    constexpr u32 nw = kSplitThreads / 64u;
    u64 const r0 = static_cast<u64>(blockIdx.x) * kTreeShapRows;
    u32 const nr = static_cast<u32>(min<u64>(kTreeShapRows, n - r0));
    u32 const plane = kTreeShapRows * F;
    u32 held = 0;
    for (u32 t = blockIdx.y; t < n_trees; t += gridDim.y) held = max(held, trees[t].n_shares);
    u8 *s_bins = reinterpret_cast<u8 *>(s_held + held * M * 64u); // [2][F][64]
    for (u32 k = threadIdx.x; k < plane; k += kSplitThreads) {
        u32 const rr = k / F, f = k - rr * F;
        u32 const b = rr < nr ? bins[(r0 + rr) * stride + f] : 0u;
        s_phi[k] = 0ull;
        s_bins[f * kTreeShapRows + rr] = static_cast<u8>(b);
        s_bins[plane + f * kTreeShapRows + rr] = static_cast<u8>(b == last[f] ? 0u : min(b + 1u, 255u));
    }
    __syncthreads();
    u32 const lane = threadIdx.x & 63u;
    u32 const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    auto begin = [&](auto &w, float(&T)[M]) {
        w.bins = s_bins + lane;
        w.phi = reinterpret_cast<unsigned char *>(s_phi + lane);
        w.plane = plane;
        w.held = s_held + lane;
#pragma unroll
        for (int q = 0; q < M; ++q) {
            w.y[q] = quad.y[q];
            T[q] = quad.w[q];
        }
    };
    for (u32 t = blockIdx.y; t < n_trees; t += gridDim.y) {
        SplitTree const tr = trees[t];
        for (u32 j = wave; j < tr.n_shares; j += nw) {
            TreeShap<M, 3, WIDE, true> w;
            float T[M], H[M];
            begin(w, T);
            w.seek(slots, __builtin_amdgcn_readfirstlane(first[tr.share0 + j]));
            w.fetch();
            w.go_down(T);
            w.template walk<0>(T, H);
#pragma unroll
            for (int q = 0; q < M; ++q) w.held[(j * M + q) * 64u] = H[q];
        }
        __syncthreads();
        if (wave == 0 && tr.top != kNone) {
            TreeShap<M, kSplitLevels, WIDE, true> w;
            float T[M], H[M];
            begin(w, T);
            w.seek(slots, __builtin_amdgcn_readfirstlane(tr.top));
            w.fetch();
            w.template walk<0>(T, H);
        }
        __syncthreads();
    }
    // Trees of one row block meet in the zeroed output cells, as shares of k_shap_tree do.
    unsigned long long *acc = reinterpret_cast<unsigned long long *>(out);
    for (u32 k = threadIdx.x; k < nr * F; k += kSplitThreads) {
        u32 const rr = k / F, f = k - rr * F;
        unsigned long long const v = s_phi[f * kTreeShapRows + rr];
        if (v != 0ull) atomicAdd(acc + (r0 + rr) * (F + 1) + f, v);
    }
}

// A handful of rows.  In a walk a row has one lane of 64, and its splits are one chain.  Here
// a lane takes one block of a tree for one row: it forms the products T down its own way
// from the root, runs the block, and the blocks' values are joined level by level through
// LDS, every split by the lane of the first block below it.  A split's arithmetic is the
// walk's own (ShapRow), so a row's bits are the same either way.  A workgroup's lanes are the
// rows of `per` trees' blocks at a time.  Bound by latency (records from L2, a barrier a
// level) with few lanes, by its instructions with many: the way down is taken again for
// every block.  One row x 20 trees: depth 8 28 (k_shap_split) -> 14 us, depth 10 74 -> 20,
// 5 of depth 12 245 -> 21; 16 rows x 1,000 depth-8 trees 78 (k_shap_tree) -> 35.
constexpr u32 lane_threads(u32 m) { return m <= 5u ? 1024u : 512u; } // of a workgroup at most
// Four waves a SIMD (a few spills with 5 nodes): 64 rows x 100 depth-10 trees 82 -> 73 us,
// one row 17.4 -> 19.4; with 6 nodes they would cost more than they give.
constexpr u32 lane_waves(u32 m) { return m <= 5u ? 4u : 3u; }
constexpr u32 kLaneLevels = kTreeShapMaxDepth - kTBlockLevels; // splits above a block at most
struct alignas(16) LaneUnit {
    u32 block, info;            // the block's slot; splits above | right turns << 4 | own splits << 13
    u32 node[kLaneLevels];      // by level: the split's step (kTEnter)
    u32 other[kLaneLevels];     // own splits: the unit that owns the other child, kNone: a leaf
};

template <int M, bool WIDE> struct LaneShap : ShapRow<LaneShap<M, WIDE>, M, WIDE> {
    u8 const *bins;      // LDS: [2][F][rows], this lane's row
    unsigned char *phi;  // LDS: [F][rows], this lane's row
    u32 plane, rs;       // bytes of a plane of bins in the steps' columns; log2 of the rows
    TSlot const *step, *next;
    uint4 nx0, nx1;
    u32 cur[8 * tree_step_slots(kTBlock)]; // its words (of a split: the first slot's)

    __device__ __forceinline__ u32 word(u32 j) const { return cur[j]; }
    __device__ __forceinline__ u32 dup_word(u32 j, u32 slot) const { return step[slot + (j >> 3)].w[j & 7u]; }
    __device__ __forceinline__ u32 bin_at(u32 col) const { return bins[col / kTreeShapRows << rs]; }
    __device__ __forceinline__ unsigned long long *phi_at(u32 col) const
    {
        return reinterpret_cast<unsigned long long *>(phi) + (min(col, col - plane) / kTreeShapRows << rs);
    }
    // A step's first slot into flight (fetch), then it is the running step (take); rest():
    // a block's other slots.
    __device__ __forceinline__ void fetch(TSlot const *s)
    {
        next = s;
        nx0 = reinterpret_cast<uint4 const *>(s)[0];
        nx1 = reinterpret_cast<uint4 const *>(s)[1];
    }
    __device__ __forceinline__ void put(u32 k, uint4 const &v)
    {
        cur[4 * k] = v.x;
        cur[4 * k + 1] = v.y;
        cur[4 * k + 2] = v.z;
        cur[4 * k + 3] = v.w;
    }
    __device__ __forceinline__ void take()
    {
        step = next;
        put(0, nx0);
        put(1, nx1);
        this->op = cur[kTwOp];
    }
    __device__ __forceinline__ void rest()
    {
#pragma unroll
        for (u32 k = 2; k < 2u * tree_step_slots(kTBlock); ++k) put(k, reinterpret_cast<uint4 const *>(step)[k]);
    }
};

template <int M, int U, bool WIDE>
__global__ __launch_bounds__(lane_threads(M), lane_waves(M)) void k_shap_lanes(
    u8 const *__restrict__ bins, u64 n, u64 stride, u32 F, u16 const *__restrict__ last,
    TSlot const *__restrict__ slots, LaneUnit const *__restrict__ units, u32 const *__restrict__ first, u32 n_trees,
    u32 per, u32 rs, u32 upper, TQuad quad, float lr, double bias, double scale, double *__restrict__ out)
{
    typedef float V[M];
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned long long *s_phi = reinterpret_cast<unsigned long long *>(smem); // [F][rows] fixed point
    float *s_held = reinterpret_cast<float *>(s_phi + (F << rs));              // [2][M][threads] values
    u32 const threads = blockDim.x, rows = 1u << rs;
    u8 *s_bins = reinterpret_cast<u8 *>(s_held + 2u * M * threads);            // [2][F][rows]
    u64 const r0 = static_cast<u64>(blockIdx.x) << rs;
    u32 const nr = static_cast<u32>(min<u64>(rows, n - r0));
    for (u32 k = threadIdx.x; k < F << rs; k += threads) {
        u32 const rr = k / F, f = k - rr * F;
        u32 const b = rr < nr ? bins[(r0 + rr) * stride + f] : 0u;
        s_phi[k] = 0ull;
        s_bins[(f << rs) + rr] = static_cast<u8>(b);
        s_bins[((F + f) << rs) + rr] = static_cast<u8>(b == last[f] ? 0u : min(b + 1u, 255u));
    }
    __syncthreads();
    u32 const rr = threadIdx.x & (rows - 1u), unit = threadIdx.x >> rs;
    LaneShap<M, WIDE> w;
    w.bins = s_bins + rr;
    w.phi = reinterpret_cast<unsigned char *>(s_phi + rr);
    w.plane = kTreeShapRows * F;
    w.rs = rs;
#pragma unroll
    for (int q = 0; q < M; ++q) w.y[q] = quad.y[q];
    u32 const chunks = (n_trees + per - 1u) / per;
    u32 buf = 0;
    for (u32 c = blockIdx.y; c < chunks; c += gridDim.y) {
        u32 const u0 = first[c * per], u1 = first[min(n_trees, (c + 1u) * per)];
        bool const live = rr < nr && unit < u1 - u0;
        V Ts[U], H; // products at the splits above; the value of the child last joined
        u32 info = 0u, len = 0u, node[U]; // the steps down to the block
        if (live) {
            LaneUnit const *un = units + u0 + unit;
            info = un->info;
            len = info & 15u;
#pragma unroll
            for (int L = 0; L < U; ++L) node[L] = un->node[L];
            u32 const block = un->block;
            w.fetch(slots + (len ? node[0] : block));
            V T;
            w.sat = 0;
#pragma unroll
            for (int q = 0; q < M; ++q) T[q] = quad.w[q];
#pragma unroll
            for (int L = 0; L < U; ++L)
                if (L < static_cast<int>(len)) {
                    w.take();
                    w.fetch(slots + (L + 1 < U && L + 1 < static_cast<int>(len) ? node[L + 1] : block));
                    typename LaneShap<M, WIDE>::Dup const u{L > 0 && (w.op & 0x100u) != 0, 1u, w.word(kTwLv)};
                    bool const right = (info >> (4 + L) & 1u) != 0;
                    u32 const m = w.goes_left(w.word(kTwSplit)), me = right ? ~m : m;
                    V k, Tc;
                    w.consts(k, u);
                    w.descend(T, Tc, k, me, right ? w.fword(kTwZr) : w.fword(kTwZl));
                    w.mark(me, L, u);
#pragma unroll
                    for (int q = 0; q < M; ++q) {
                        Ts[L][q] = T[q];
                        T[q] = Tc[q];
                    }
                }
            w.take();
            w.rest();
            w.block(T, H, len);
        }
#pragma unroll
        for (int L = U - 1; L >= 0; --L) {
            if (L >= static_cast<int>(upper)) continue;
            bool const own = (info >> (13 + L) & 1u) != 0;
            u32 other = kNone;
            if (own) {
                w.fetch(slots + node[L]);
                other = units[u0 + unit].other[L];
            }
            float *held = s_held + buf * M * threads;
            buf ^= 1u; // the next level writes beside what this one still reads
            if (live) {
#pragma unroll
                for (int q = 0; q < M; ++q) held[q * threads + threadIdx.x] = H[q];
            }
            __syncthreads();
            if (own) {
                w.take();
                typename LaneShap<M, WIDE>::Dup const u{L > 0 && (w.op & 0x100u) != 0, 1u, w.word(kTwLv)};
                bool const right = (info >> (4 + L) & 1u) != 0;
                u32 const at = ((other - u0) << rs) + rr;
                float const leaf = right ? w.fword(kTwVl) : w.fword(kTwVr);
                V k, HL, HR;
#pragma unroll
                for (int q = 0; q < M; ++q) {
                    float const x = other == kNone ? leaf : held[q * threads + at];
                    HL[q] = right ? x : H[q];
                    HR[q] = right ? H[q] : x;
                }
                w.consts(k, u);
                w.join(Ts[L], k, HL, HR, H, w.goes_left(w.word(kTwSplit)), w.fword(kTwZl), w.fword(kTwZr),
                       w.word(kTwSplit), u);
            }
        }
    }
    __syncthreads();
    if (gridDim.y > 1) {
        // Trees of one row block meet in the zeroed output cells, as k_shap_tree's do.
        unsigned long long *acc = reinterpret_cast<unsigned long long *>(out);
        for (u32 k = threadIdx.x; k < nr * F; k += threads) {
            u32 const r = k / F, f = k - r * F;
            unsigned long long const v = s_phi[(f << rs) + r];
            if (v != 0ull) atomicAdd(acc + (r0 + r) * (F + 1) + f, v);
        }
        return;
    }
    for (u32 k = threadIdx.x; k < nr * (F + 1); k += threads) {
        u32 const r = k / (F + 1), f = k - r * (F + 1);
        out[(r0 + r) * (F + 1) + f] = f == F ? bias : shap_from_fixed(s_phi[(f << rs) + r], scale, lr);
    }
}

// gridDim.y workgroups share a row block; each of their waves walks a run of trees.
template <int M, int U, bool WIDE>
__global__ __launch_bounds__(kTreeShapThreads, tree_shap_waves(U)) void k_shap_tree(
    u8 const *__restrict__ bins, u64 n, u64 stride, u32 F, u16 const *__restrict__ last,
    TSlot const *__restrict__ slots, u32 const *__restrict__ first, u32 n_trees, TQuad quad, float lr, double bias,
    double scale, double *__restrict__ out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned long long *s_phi = reinterpret_cast<unsigned long long *>(smem); // [F][64] fixed point
    u8 *s_bins = reinterpret_cast<u8 *>(s_phi + kTreeShapRows * F);            // [2][F][64]
    constexpr u32 threads = kTreeShapThreads, nw = threads / 64u;
    u64 const r0 = static_cast<u64>(blockIdx.x) * kTreeShapRows;
    u32 const nr = static_cast<u32>(min<u64>(kTreeShapRows, n - r0));
    u32 const plane = kTreeShapRows * F;
    for (u32 k = threadIdx.x; k < plane; k += threads) {
        u32 const rr = k / F, f = k - rr * F;
        u32 const b = rr < nr ? bins[(r0 + rr) * stride + f] : 0u;
        s_phi[k] = 0ull;
        s_bins[f * kTreeShapRows + rr] = static_cast<u8>(b);
        s_bins[plane + f * kTreeShapRows + rr] = static_cast<u8>(b == last[f] ? 0u : min(b + 1u, 255u));
    }
    __syncthreads();
    u32 const lane = threadIdx.x & 63u;
    u32 const wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    TreeShap<M, U, WIDE> w;
    w.bins = s_bins + lane;
    w.phi = reinterpret_cast<unsigned char *>(s_phi + lane);
    w.plane = plane;
    w.sat = 0;
    float T[M];
#pragma unroll
    for (int q = 0; q < M; ++q) {
        w.y[q] = quad.y[q];
        T[q] = quad.w[q];
    }
    u32 const wi = blockIdx.y * nw + wave, waves = gridDim.y * nw;
    u32 const per = n_trees / waves, more = n_trees - per * waves;
    u32 const t0 = wi * per + min(wi, more), t1 = t0 + per + (wi < more ? 1u : 0u);
    if (t0 < t1) {
        u32 const pc = __builtin_amdgcn_readfirstlane(first[t0]);
        w.ahead = slots + (pc & ~63u) + lane;
        w.load();
        w.shift();
        w.at = pc & 63u;
        for (u32 t = t0; t < t1; ++t) {
            float H[M];
            w.fetch();
            w.template walk<0>(T, H);
        }
    }
    __syncthreads();
    if (gridDim.y > 1) {
        // Shares of one row block meet in the zeroed output cells (exact in any order);
        // k_shap_to_double converts them once every workgroup has added its own.
        unsigned long long *acc = reinterpret_cast<unsigned long long *>(out);
        for (u32 k = threadIdx.x; k < nr * F; k += threads) {
            u32 const rr = k / F, f = k - rr * F;
            unsigned long long const v = s_phi[f * kTreeShapRows + rr];
            if (v != 0ull) atomicAdd(acc + (r0 + rr) * (F + 1) + f, v);
        }
        return;
    }
    for (u32 k = threadIdx.x; k < nr * (F + 1); k += threads) {
        u32 const rr = k / (F + 1), f = k - rr * (F + 1);
        out[(r0 + rr) * (F + 1) + f] = f == F ? bias : shap_from_fixed(s_phi[f * kTreeShapRows + rr], scale, lr);
    }
}

// Split launches: the output cells start at zero (a fill kernel, so the sequence stays
// capturable in a graph) ...
__global__ __launch_bounds__(256) void k_shap_zero(unsigned long long *__restrict__ acc, u64 cells)
{
    for (u64 i = blockIdx.x * 256ull + threadIdx.x; i < cells; i += static_cast<u64>(gridDim.x) * 256ull) acc[i] = 0ull;
}

// ... and end as doubles, each cell converted in place by the thread that reads it.
__global__ __launch_bounds__(256) void k_shap_to_double(double *__restrict__ out, u64 n, u32 F, float lr, double bias,
                                                        double scale)
{
    u64 const cells = n * (F + 1);
    for (u64 i = blockIdx.x * 256ull + threadIdx.x; i < cells; i += static_cast<u64>(gridDim.x) * 256ull) {
        u32 const f = static_cast<u32>(i % (F + 1));
        if (f == F) {
            out[i] = bias;
        } else {
            unsigned long long const v = reinterpret_cast<unsigned long long const *>(out)[i];
            out[i] = shap_from_fixed(v, scale, lr);
        }
    }
}

// Tiles of an ensemble (k_predict_tile); false when a tree or the features do not fit.
bool pack_tiles(bh_node const *nodes, uint32_t const *offsets, u32 n_trees, u32 F,
                std::vector<u32> &words, std::vector<Tile> &tiles, std::vector<TileTree> &trees)
{
    if (F > 256u || n_trees == 0) return false;
    std::vector<u32> nd, order; // the open tile's nodes; a tree's node ids, siblings adjacent
    std::vector<float> val;
    auto close = [&] {
        if (tiles.empty() || tiles.back().count != 0) return;
        while (nd.size() & 3u) {
            nd.push_back(0u);
            val.push_back(0.0F);
        }
        Tile &t = tiles.back();
        t.off = static_cast<u32>(words.size());
        t.count = static_cast<u32>(nd.size());
        t.n_trees = static_cast<u32>(trees.size()) - t.tree0;
        words.insert(words.end(), nd.begin(), nd.end());
        words.resize(words.size() + val.size());
        std::memcpy(words.data() + t.off + t.count, val.data(), val.size() * sizeof(float));
        nd.clear();
        val.clear();
    };
    for (u32 k = 0; k < n_trees; ++k) {
        bh_node const *t = nodes + offsets[k];
        order.assign(1, 0u);
        u32 levels = 0;
        for (size_t i = 0, end = 1; i < order.size();) { // breadth first, level by level
            for (; i < end; ++i)
                if (t[order[i]].feature >= 0) {
                    order.push_back(t[order[i]].left);
                    order.push_back(t[order[i]].right);
                    if (order.size() > kTileNodes) return false;
                }
            if (order.size() > end) ++levels;
            end = order.size();
        }
        if (tiles.empty() || nd.size() + order.size() > kTileNodes) {
            close();
            tiles.push_back(Tile{0u, 0u, static_cast<u32>(trees.size()), 0u});
        }
        u32 const base = static_cast<u32>(nd.size());
        trees.push_back(TileTree{base | levels << 16});
        u32 child = base + 1u;
        for (size_t i = 0; i < order.size(); ++i) {
            bh_node const &n = t[order[i]];
            if (n.feature < 0) {
                nd.push_back(255u << 8 | (base + static_cast<u32>(i)) << 16);
                val.push_back(n.value);
                continue;
            }
            u32 const d = n.default_left ? 0u : 1u;
            nd.push_back(static_cast<u32>(n.feature) | std::min(255u, n.bin + 1u - d) << 8 | child << 16 | d << 31);
            val.push_back(0.0F);
            child += 2u;
        }
    }
    close();
    return true;
}

struct ActiveElem {
    u32 feature;
    int lo, hi;
    bool missing_ok;
    double zero;
};

// pack_shap_paths (src/shap_paths.cpp:57-163): every root-to-leaf path, repeated
// features merged into one interval, zero fractions multiplied along the path.
void pack_paths(bh_node const *t, u16 const *last, u32 id, std::vector<ActiveElem> &act, std::vector<SElem> &el,
                std::vector<SHead> &hd, size_t &max_len)
{
    bh_node const &nd = t[id];
    if (nd.feature < 0) {
        SHead h{};
        h.first = static_cast<u32>(el.size());
        h.n = static_cast<u16>(act.size());
        h.value = nd.value;
        hd.push_back(h);
        for (auto const &a : act) {
            int lo = a.lo, hi = a.hi;
            if (hi < lo) {
                lo = 1;
                hi = 0;
            }
            SElem e{};
            e.feature = static_cast<u16>(a.feature | (a.missing_ok ? 0x8000u : 0u));
            e.lo = static_cast<u8>(lo);
            e.hi = static_cast<u8>(hi);
            e.z = static_cast<float>(a.zero);
            el.push_back(e);
        }
        max_len = std::max(max_len, act.size());
        return;
    }
    u32 const f = static_cast<u32>(nd.feature);
    int const split = static_cast<int>(nd.bin), lb = static_cast<int>(last[f]);
    double const cover = nd.cover;
    auto frac = [&](u32 c) { return cover > 0.0 ? static_cast<double>(t[c].cover) / cover : 0.0; };
    size_t idx = act.size();
    for (size_t k = 0; k < act.size(); ++k)
        if (act[k].feature == f) {
            idx = k;
            break;
        }
    bool const fresh = idx == act.size();
    if (fresh) act.push_back({f, 0, lb - 1, true, 1.0});
    ActiveElem const saved = act[idx];
    act[idx].hi = std::min(saved.hi, split);
    act[idx].missing_ok = saved.missing_ok && nd.default_left != 0;
    act[idx].zero = saved.zero * frac(nd.left);
    pack_paths(t, last, nd.left, act, el, hd, max_len);
    act[idx].lo = std::max(saved.lo, split + 1);
    act[idx].hi = saved.hi;
    act[idx].missing_ok = saved.missing_ok && nd.default_left == 0;
    act[idx].zero = saved.zero * frac(nd.right);
    pack_paths(t, last, nd.right, act, el, hd, max_len);
    if (fresh) act.pop_back();
    else act[idx] = saved;
}

// Levels of splits below every node of a tree, and the most distinct features on a path
// (seen: per feature, its splits on the way; distinct: the features among them).
u32 tree_levels(bh_node const *t, u32 id, std::vector<u32> &levels, std::vector<u32> &seen, size_t distinct,
                size_t &max_len)
{
    bh_node const &nd = t[id];
    if (nd.feature < 0) {
        max_len = std::max(max_len, distinct);
        return 0;
    }
    u32 &on_path = seen[static_cast<u32>(nd.feature)];
    distinct += on_path++ == 0 ? 1u : 0u;
    u32 const l = tree_levels(t, nd.left, levels, seen, distinct, max_len);
    u32 const r = tree_levels(t, nd.right, levels, seen, distinct, max_len);
    --on_path;
    return levels[id] = 1u + std::max(l, r);
}

struct GaussRule { // m nodes on [0, 1], ascending
    u32 m;
    double x[kTreeShapMaxM], w[kTreeShapMaxM];
};
bool past_half(u32 i, u32 m) { return 2u * i >= m + (m & 1u); }

// Tree-form steps of an ensemble (TSlot stream).
struct TreePacker {
    bh_node const *t = nullptr;   // current tree
    u32 const *levels = nullptr;  // and its nodes' levels of splits below
    u16 const *last;
    u32 F;
    double scale;
    GaussRule rule;
    std::vector<TSlot> out;
    std::vector<std::pair<u32, u32>> spans; // of every node walked: its subtree's slots in out
    std::vector<LaneUnit> units;     // k_shap_lanes: the blocks, in the walk's order
    std::vector<std::pair<u32, u32>> down; // (step, side) of the splits above the walk
    struct Edge { // on the way down: feature, level and merged cover fraction of its latest edge
        u32 feature, level;
        double z;
    };
    std::vector<Edge> above;

    // What the kernel reads of one node; a leaf taken as a node splits into itself.
    struct Node {
        u32 split = 0, level = 0; // level: of the same-feature edge above
        bool dup = false, leaf = false;
        double z = 1.0;           // and its merged fraction
        float k[kTreeShapMaxM], l[kTreeShapMaxM]; // then its k_q (1 - k_q past the half) and l_q
        double zl = 0.5, zr = 0.5, value = 0.0;
    };
    Node node(u32 id) const
    {
        bh_node const &nd = t[id];
        Node r;
        if (nd.feature < 0) {
            r.leaf = true;
            r.value = static_cast<double>(nd.value) * scale;
            return r;
        }
        u32 const f = static_cast<u32>(nd.feature), lb = last[f];
        // rows go left below the bound on the plane where the missing bin sorts last
        // (bound bin + 1) or first (bin + 2); a split past the missing bin takes every
        // other row left
        u32 const bin = std::min<u32>(nd.bin + 1u, lb);
        r.split = nd.default_left ? (F + f) * kTreeShapRows | (bin + 1u) << 16 : f * kTreeShapRows | bin << 16;
        double const cover = nd.cover;
        r.zl = cover > 0.0 ? static_cast<double>(t[nd.left].cover) / cover : 0.0;
        r.zr = cover > 0.0 ? static_cast<double>(t[nd.right].cover) / cover : 0.0;
        for (size_t k = above.size(); k-- > 0;)
            if (above[k].feature == f) {
                r.dup = true;
                r.level = above[k].level;
                r.z = above[k].z;
                for (u32 q = 0; q < rule.m; ++q) {
                    double const x = rule.x[q], inv = 1.0 / (r.z + x * (1.0 - r.z)), zi = r.z * inv;
                    r.k[q] = static_cast<float>(past_half(q, rule.m) ? zi * (1.0 - x) : x * inv);
                    r.l[q] = static_cast<float>(zi * inv);
                }
                break;
            }
        return r;
    }
    static void put(TSlot *s, u32 word, float v) { std::memcpy(&s[word / 8u].w[word % 8u], &v, sizeof(v)); }
    static void put(TSlot *s, u32 word, double v) { put(s, word, static_cast<float>(v)); }

    // Room for a step of `need` slots inside a group; returns its first slot.
    size_t room(u32 need)
    {
        while ((out.size() & 63u) + need > 64u) {
            TSlot skip{};
            skip.w[kTwOp] = kTSkip << 2;
            out.push_back(skip);
        }
        size_t const at = out.size();
        out.resize(at + need);
        return at;
    }

    // Room for a step and the constants of its n nodes; returns its first slot.
    size_t open(u32 kind, Node const *nodes, u32 n)
    {
        u32 const ds = tree_dup_slots(rule.m);
        u32 need = tree_step_slots(kind);
        for (u32 i = 0; i < n; ++i) need += nodes[i].dup ? ds : 0u;
        size_t const at = room(need);
        size_t o = at + tree_step_slots(kind);
        for (u32 i = 0; i < n; ++i) {
            if (!nodes[i].dup) continue;
            auto *const to = reinterpret_cast<unsigned char *>(out.data() + o);
            std::memcpy(to, nodes[i].k, rule.m * sizeof(float));
            std::memcpy(to + rule.m * sizeof(float), nodes[i].l, rule.m * sizeof(float));
            o += ds;
        }
        return at;
    }

    size_t step(u32 kind, u32 level, Node const &nd, u32 flags, double vl, double vr)
    {
        size_t const at = open(kind, &nd, 1);
        TSlot *s = &out[at];
        s->w[kTwOp] = kind | level << 2 | (nd.dup ? 0x100u : 0u) | flags;
        s->w[kTwLv] = nd.level;
        s->w[kTwSplit] = nd.split;
        put(s, kTwZl, nd.zl);
        put(s, kTwZr, nd.zr);
        put(s, kTwVl, vl);
        put(s, kTwVr, vr);
        return at;
    }

    // Nodes of a block in preorder: `depth` more levels below id.
    void collect(u32 id, u32 level, u32 depth, Node *&nodes, double *&leaf)
    {
        Node const nd = node(id);
        if (depth == 0) {
            *leaf++ = nd.value;
            return;
        }
        *nodes++ = nd;
        bool const self = nd.leaf; // its two children are itself
        for (u32 side = 0; side < 2; ++side) {
            if (!self) above.push_back({static_cast<u32>(t[id].feature), level, nd.z * (side ? nd.zr : nd.zl)});
            collect(self ? id : (side ? t[id].right : t[id].left), level + 1, depth - 1, nodes, leaf);
            if (!self) above.pop_back();
        }
    }

    size_t block(u32 id, u32 level)
    {
        Node nd[7], *np = nd;
        double leaf[8], *lp = leaf;
        collect(id, level, kTBlockLevels, np, lp);
        size_t const at = open(kTBlock, nd, 7);
        TSlot *s = &out[at];
        u32 op = kTBlock | level << 2, lv = 0;
        for (u32 i = 0; i < 7; ++i) {
            op |= nd[i].dup ? 0x100u << i : 0u;
            lv |= nd[i].level << (4 * i);
            s[(kTwSplit + i) / 8].w[(kTwSplit + i) % 8] = nd[i].split;
        }
        s->w[kTwOp] = op;
        s->w[kTwLv] = lv;
        static const u32 inner[3] = {0, 1, 4}, low[4] = {2, 3, 5, 6};
        for (u32 i = 0; i < 3; ++i) {
            put(s, kTwZ + 2 * i, nd[inner[i]].zl);
            put(s, kTwZ + 2 * i + 1, nd[inner[i]].zr);
        }
        for (u32 i = 0; i < 4; ++i) {
            put(s, kTwMean + i, nd[low[i]].zl * leaf[2 * i] + nd[low[i]].zr * leaf[2 * i + 1]);
            put(s, kTwLeaf + 2 * i, leaf[2 * i]);
            put(s, kTwLeaf + 2 * i + 1, leaf[2 * i + 1]);
        }
        return at;
    }

    // Returns the first unit below id, which owns it.
    u32 walk(u32 id, u32 level)
    {
        u32 const begin = static_cast<u32>(out.size());
        u32 const own = levels[id] <= kTBlockLevels ? leaf_block(id, level) : inner(id, level);
        spans[id] = {begin, static_cast<u32>(out.size())};
        return own;
    }
    u32 leaf_block(u32 id, u32 level)
    {
        LaneUnit u{};
        u.block = static_cast<u32>(block(id, level));
        u.info = level;
        for (u32 l = 0; l < level; ++l) {
            u.node[l] = down[l].first;
            u.info |= down[l].second << (4 + l);
        }
        units.push_back(u);
        return static_cast<u32>(units.size() - 1);
    }
    u32 inner(u32 id, u32 level)
    {
        bh_node const &n = t[id];
        Node const nd = node(id);
        bool const ll = t[n.left].feature < 0, rl = t[n.right].feature < 0;
        double const vl = ll ? static_cast<double>(t[n.left].value) * scale : 0.0;
        double const vr = rl ? static_cast<double>(t[n.right].value) * scale : 0.0;
        u32 const flags = (ll ? kTLeafL : 0u) | (rl ? kTLeafR : 0u);
        u32 const at = static_cast<u32>(step(kTEnter, level, nd, flags, vl, vr));
        u32 kid[2] = {kNone, kNone};
        for (u32 side = 0; side < 2; ++side) {
            if (side ? rl : ll) continue;
            if (side && !ll) step(kTTurn, level, nd, flags, vl, vr);
            above.push_back({static_cast<u32>(n.feature), level, nd.z * (side ? nd.zr : nd.zl)});
            down.push_back({at, side});
            kid[side] = walk(side ? n.right : n.left, level + 1);
            down.pop_back();
            above.pop_back();
        }
        step(kTCombine, level, nd, flags, vl, vr);
        u32 const own = ll ? kid[1] : kid[0];
        units[own].info |= 1u << (13 + level);
        units[own].other[level] = ll ? kNone : kid[1];
        return own;
    }

    // Appends a walked subtree's steps again, in a third of the time packing them takes.
    void copy_steps(u32 id)
    {
        for (u32 at = spans[id].first; at < spans[id].second;) {
            u32 const op = out[at].w[kTwOp];
            if ((op >> 2 & 15u) == kTSkip) {
                ++at;
                continue;
            }
            u32 const need = tree_step_slots(op & 3u) + static_cast<u32>(__builtin_popcount(op >> 8 & 0x7Fu)) * tree_dup_slots(rule.m);
            size_t const to = room(need);
            std::copy_n(out.begin() + at, need, out.begin() + static_cast<std::ptrdiff_t>(to));
            at += need;
        }
    }

    // The split form (k_shap_split): every subtree at depth `cut`, or shallower of at most a
    // block's levels, is a share: the steps down to it, then its own walk's.
    std::vector<u32> first;          // first slot of every share
    std::vector<std::pair<u32, u32>> way; // (node, side) from the root
    static u32 cut_of(u32 deepest) { return std::min(deepest - kTBlockLevels, std::max(4u, deepest / 2u)); }
    bool is_share(u32 id, u32 level, u32 cut) const { return level == cut || levels[id] <= kTBlockLevels; }
    void go_down(u32 id, u32 level)
    {
        if (level == way.size()) {
            copy_steps(id);
            return;
        }
        u32 const side = way[level].second;
        bh_node const &n = t[way[level].first];
        Node const nd = node(way[level].first);
        step(kTEnter, level, nd, side ? kTOnlyR : kTOnlyL, 0.0, 0.0);
        above.push_back({static_cast<u32>(n.feature), level, nd.z * (side ? nd.zr : nd.zl)});
        go_down(id, level + 1);
        above.pop_back();
    }
    void shares(u32 id, u32 level, u32 cut)
    {
        if (is_share(id, level, cut)) {
            first.push_back(static_cast<u32>(out.size()));
            go_down(id, 0);
            return;
        }
        for (u32 side = 0; side < 2; ++side) {
            u32 const kid = side ? t[id].right : t[id].left;
            if (t[kid].feature < 0) continue;
            way.push_back({id, side});
            shares(kid, level + 1, cut);
            way.pop_back();
        }
    }
    // The steps above the shares, which come in the same order.
    void top(u32 id, u32 level, u32 cut, u32 &share)
    {
        bh_node const &n = t[id];
        Node const nd = node(id);
        u32 const kids[2] = {n.left, n.right};
        u32 flags = 0;
        double v[2] = {0.0, 0.0};
        u32 next = share; // index of the side's first share
        for (u32 side = 0; side < 2; ++side) {
            if (t[kids[side]].feature < 0) {
                flags |= kTLeafL << side;
                v[side] = static_cast<double>(t[kids[side]].value) * scale;
            } else if (is_share(kids[side], level + 1, cut)) {
                flags |= (kTLeafL | kTHeldL) << side;
                v[side] = next++;
            } else if (side == 0) {
                next += count(kids[0], level + 1, cut);
            }
        }
        bool const ll = (flags & kTLeafL) != 0, rl = (flags & kTLeafR) != 0;
        if (!ll || !rl) step(kTEnter, level, nd, flags, v[0], v[1]);
        if (flags & kTHeldL) ++share;
        for (u32 side = 0; side < 2; ++side) {
            if (side ? rl : ll) continue;
            if (side && !ll) step(kTTurn, level, nd, flags, v[0], v[1]);
            above.push_back({static_cast<u32>(n.feature), level, nd.z * (side ? nd.zr : nd.zl)});
            top(kids[side], level + 1, cut, share);
            above.pop_back();
        }
        if (flags & kTHeldR) ++share;
        step(kTCombine, level, nd, flags, v[0], v[1]);
    }
    u32 count(u32 id, u32 level, u32 cut) const
    {
        if (t[id].feature < 0) return 0;
        if (is_share(id, level, cut)) return 1;
        return count(t[id].left, level + 1, cut) + count(t[id].right, level + 1, cut);
    }
};

// Gauss-Legendre nodes on [0, 1], ascending (Newton's method on the Legendre polynomial),
// and their weights times a common factor `g` searched so that every weight lands
// within 2^-29 of a float (or the nearest found): a weight's rounding would be the same
// relative error in every contribution.
GaussRule gauss_legendre(u32 m)
{
    GaussRule r{};
    r.m = m;
    for (u32 i = 0; i < m; ++i) {
        double x = std::cos(3.14159265358979323846 * (m - 1 - i + 0.75) / (m + 0.5)), d = 1.0;
        for (int it = 0; it < 60; ++it) {
            double p0 = 1.0, p1 = x;
            for (u32 k = 2; k <= m; ++k) {
                double const p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
                p0 = p1;
                p1 = p2;
            }
            d = m * (x * p1 - p0) / (x * x - 1.0);
            x -= p1 / d;
        }
        r.x[i] = 0.5 * (1.0 + x);
        r.w[i] = 1.0 / ((1.0 - x * x) * d * d);
    }
    return r;
}
TQuad tree_quad(GaussRule const &r, double &g)
{
    u32 const m = r.m;
    TQuad q{};
    for (u32 i = 0; i < m; ++i) q.y[i] = static_cast<float>(past_half(i, m) ? 1.0 - r.x[i] : r.x[i]);
    double best = 1.0;
    g = 1.0;
    for (u32 k = 0; k < 200000 && best > 0x1p-29; ++k) {
        double const c = 1.0 + k * 0x1p-18;
        double worst = 0.0;
        for (u32 i = 0; i < (m + 1) / 2; ++i) { // the rule is symmetric
            double const v = r.w[i] * c;
            worst = std::max(worst, std::fabs(static_cast<double>(static_cast<float>(v)) - v) / v);
        }
        if (worst < best) {
            best = worst;
            g = c;
        }
    }
    for (u32 i = 0; i < m; ++i) q.w[i] = static_cast<float>(r.w[std::min(i, m - 1 - i)] * g);
    return q;
}

// Leaf magnitudes of an ensemble.
struct LeafStats {
    std::vector<double> top; // the largest of every tree
    double sum = 0.0;        // of all
    bool finite = true;      // with one leaf that is not, every contribution is NaN
    bool covers = true;      // every node's children hold fractions of it that sum to 1 at most
};

// log2 of the tree form's fixed-point scale.  The packed form's grid is 2^61 / (4 Sum |leaf|),
// the next power of two at least what 63-bit contributions take (wide).  The 52-bit add takes
// contributions below 2^51: each is at most 4 max |leaf| of its tree, and one level's of a
// tree together too, if the covers are proper; it serves where its grid is as fine.
int tree_grid(LeafStats const &s, u32 deepest, bool &wide)
{
    double top = 0.0, tops = 0.0;
    for (double v : s.top) {
        top = std::max(top, v);
        tops += v;
    }
    wide = false;
    if (!s.finite || s.sum <= 0.0) return 0;
    int e_all = 0, e_top = 0, e_tops = 0;
    (void)std::frexp(s.sum, &e_all);
    (void)std::frexp(top, &e_top);
    (void)std::frexp(tops * std::max(1u, deepest), &e_tops);
    int const narrow = std::min(48 - e_top, 60 - e_tops);
    wide = !s.covers || narrow < 60 - e_all;
    return wide ? 60 - e_all : narrow;
}

// tree_expected_value (src/shap.cpp:246-292): cover-weighted mean of the leaves.
double expected_value(bh_node const *t, u32 id)
{
    bh_node const &nd = t[id];
    if (nd.feature < 0) return nd.value;
    double const cover = nd.cover;
    if (cover <= 0.0) return 0.0;
    return (static_cast<double>(t[nd.left].cover) * expected_value(t, nd.left) +
            static_cast<double>(t[nd.right].cover) * expected_value(t, nd.right)) /
           cover;
}

} // namespace

struct bh_predictor {
    int device = 0;
    u32 n_trees = 0, F = 0;
    float lr = 0.0F, init = 0.0F;
    double shap_bias = 0.0;
    u32 n_heads = 0, max_len = 0;
    u32 n_groups = 0;          // TreeSHAP path groups of 64
    double shap_scale = 1.0;   // fixed-point scale of the TreeSHAP accumulators
    // tree-form TreeSHAP (tree_m quadrature nodes; 0: the packed form serves the ensemble)
    u32 tree_m = 0, tree_depth = 0, n_ttrees = 0, max_shares = 0; // max_shares 0: no split form
    u32 max_units = 1;         // blocks of a tree at most
    double tree_scale = 1.0;   // its fixed-point scale, times the weights' common factor
    bool tree_wide = false;    // TreeShap's WIDE
    TQuad quad{};
    TSlot *d_tslots = nullptr;
    u32 *d_tfirst = nullptr;
    u32 *d_sfirst = nullptr;
    SplitTree *d_split = nullptr;
    LaneUnit *d_units = nullptr;
    u32 *d_ufirst = nullptr;
    PNode *d_nodes = nullptr;
    u32 *d_roots = nullptr;
    // tile form (n_tiles 0: the ensemble does not fit it)
    u32 n_tiles = 0;
    double mean_levels = 0.0;  // splits above a leaf if the mean tree were full
    u32 *d_words = nullptr;
    Tile *d_tiles = nullptr;
    TileTree *d_ttrees = nullptr;
    u16 *d_last = nullptr;
    SElem *d_elems = nullptr;
    SHead *d_heads = nullptr;
    float *d_w = nullptr;
    std::vector<void *> owned; // the allocations they lie in (Upload)
    hipStream_t stream = nullptr;
    // Buffers of small host calls (SmallCall): one call at a time.
    std::mutex ws_busy;
    unsigned char *ws_host = nullptr, *ws_dev = nullptr; // kWsBytes each, pinned and device
};

namespace {

constexpr size_t kPredLdsMax = 160u * 1024u;

// Microseconds of a batch served from tiles, and the rows a workgroup takes: one workgroup
// per CU (LDS), so rounds of 256 of them; a round costs a tile's barriers and loads and its
// trees' walks (1,000 depth-8 trees, 63 tiles: 145, 235 and 595 us with 64, 256 and 1,024
// rows; 20 of depth 12, a tile each: 39, 45 and 50).
struct TileShape {
    double us;
    u32 rows;
};
size_t tile_lds(bh_predictor const *p, u32 rows)
{
    u32 const split = kTileThreads / rows;
    return static_cast<size_t>(2u * kTileNodes * 4u) + (split > 1 ? 2u * split * 4u * rows * 4u : 0u) +
           rows * tile_row_stride(p->F);
}
TileShape tile_shape(bh_predictor const *p, u64 n)
{
    static const struct {
        u32 rows;
        double tile, tree;
    } shapes[] = {{64, 1.9, 0.045}, {256, 2.2, 0.1}, {1024, 2.4, 0.44}};
    TileShape best{1e300, 0u};
    for (auto const &q : shapes) {
        u64 const rounds = ((n + q.rows - 1) / q.rows + 255) / 256;
        double const us = static_cast<double>(rounds) * (p->n_tiles * q.tile + p->n_trees * q.tree);
        if (us < best.us && tile_lds(p, q.rows) <= kPredLdsMax) best = TileShape{us, q.rows};
    }
    return best;
}

// Walking from memory costs about 6 ps a level, tree and row (2 to 7 over 1 to 100 trees of
// 3 to 13 levels, 2,048 to 65,536 rows), 9 with kManyTrees (a row's ordered sum is long), so
// tiles serve from where their rounds cost less: 1,000 depth-8 trees from 2,300 rows (146 us),
// 20 of depth 12 (39 us from tiles, 20 walked at 16,384 rows) from 32,000; and never an
// ensemble they do not hold.
constexpr u32 kManyTrees = 500;
bool served_from_tiles(bh_predictor const *p, u64 n)
{
    double const per = p->n_trees >= kManyTrees ? 9e-6 : 6e-6;
    return p->n_tiles && static_cast<double>(n) * p->n_trees * p->mean_levels * per > tile_shape(p, n).us;
}

// Rows of a workgroup, trees whose values wait in its LDS and its threads at most.  Of many
// trees, rows a lane each (64) share a tree's nodes, and few values a row keep workgroups on
// a CU while one thread a row adds: 1,000 depth-8 trees, 300 features: 65,536 rows 4,483 ->
// 2,202 us against 8 rows and 1,024 trees, 4,096 rows (16 and 256) 299 -> 232; fewer rows
// have the chip to fill first, and of 100 trees 8 rows take as long or less.  A tile of the
// trees there are: 262,144 rows of 4 depth-13 trees 470 -> 104 us.
struct WalkShape {
    u32 rows, tile, threads;
};
WalkShape walk_shape(u64 n, u32 n_trees, u32 F)
{
    u32 const lanes = 64u / std::min(64u, std::max(1u, n_trees)); // rows that fill a wave
    WalkShape w{static_cast<u32>(std::min<u64>(8u, std::max<u64>(lanes, n / 1024))), 1024u, 1024u};
    if (n >= 16384 && n_trees >= kManyTrees) w = WalkShape{64u, 64u, 256u};
    else if (n >= 2560 && n_trees >= kManyTrees) w = WalkShape{16u, 256u, 256u};
    w.tile = std::min(w.tile, (std::max(1u, n_trees) + 15u) / 16u * 16u); // float4 reads of a row's values
    while (w.rows > 1 && static_cast<size_t>(w.rows) * (w.tile * sizeof(float) + F) > kPredLdsMax / 4) w.rows /= 2;
    // A thread a walk; with few trees 256 to load the rows while the chip has room for them
    // (4 depth-13 trees, 300 features: 16,384 rows 12.7 -> 10.2 us, but 200,000 80.7 -> 118.6).
    u32 const walks = w.rows * std::min(w.tile, std::max(1u, n_trees));
    u32 const load = n / w.rows <= 4096u ? std::min(256u, w.rows * F) : 64u;
    w.threads = std::min(w.threads, (std::max(walks, load) + 63u) / 64u * 64u);
    return w;
}

int launch_predict(bh_predictor *p, u8 const *d_bins, u64 n, u64 stride, float *d_out, hipStream_t s)
{
    if (n == 0) return 0;
    if (served_from_tiles(p, n)) {
        u32 const rows = tile_shape(p, n).rows;
#define BH_PT(R)                                                                                                    \
    hipLaunchKernelGGL(k_predict_tile<R>, dim3(static_cast<u32>((n + R - 1) / R)), dim3(kTileThreads),              \
                       tile_lds(p, R), s, d_bins, n, stride, p->F, p->d_words, p->d_tiles, p->n_tiles,              \
                       p->d_ttrees, p->d_last, p->lr, p->init, d_out)
        if (rows == 64) BH_PT(64);
        else if (rows == 256) BH_PT(256);
        else BH_PT(1024);
#undef BH_PT
        SHIP(hipGetLastError());
        return 0;
    }
    WalkShape const w = walk_shape(n, p->n_trees, p->F);
    size_t const lds = static_cast<size_t>(w.rows) * (w.tile * sizeof(float) + p->F) + p->F * sizeof(u16);
    if (lds > kPredLdsMax) return sfail(1, "predict: too many features for one row in LDS");
    hipLaunchKernelGGL(k_predict_direct, dim3(static_cast<u32>((n + w.rows - 1) / w.rows)), dim3(w.threads), lds, s,
                       d_bins, n, stride, p->F, w.rows, w.tile, p->d_nodes, p->d_roots, p->n_trees, p->d_last, p->lr,
                       p->init, d_out);
    SHIP(hipGetLastError());
    return 0;
}

// Workgroups that fill the chip with tree-form waves: smaller batches split their trees.
constexpr u32 kTreeShapFill = 768;

// Row blocks x trees up to which a workgroup takes one tree (k_shap_split): two rounds of
// workgroups (depth 10, 400 walks: 148 us split, 287 whole; 1,600: 574 whole).
constexpr u64 kSplitWalks = 512;
// LDS of a k_shap_split workgroup whose trees have up to `shares` shares.
size_t split_lds(u32 F, u32 shares, u32 m) { return tree_shap_lds(F) + static_cast<size_t>(shares) * m * 64u * sizeof(float); }

// Launch of k_shap_lanes: rows and trees of a workgroup's lanes, and the workgroups that
// share the trees.  256 lanes where a tree's blocks allow it: more workgroups, and more of
// them on a CU (64 rows x 20 depth-10 trees 28 -> 20 us against 512); up to 1,024 where one
// workgroup then takes the batch and writes its output itself.
constexpr u32 kLaneFill = 1024;
struct LaneShape {
    u32 rs, per, threads, split;
    u64 blocks;
    size_t lds;
};
LaneShape lane_shape(bh_predictor const *p, u64 n)
{
    LaneShape s{};
    u32 most = (p->max_units <= 256u ? 256u : 512u) / p->max_units; // rows x trees of full lanes
    if (n * p->n_ttrees * p->max_units <= lane_threads(p->tree_m)) most = lane_threads(p->tree_m) / p->max_units;
    auto const lds = [&](u32 rs, u32 threads) {
        return (static_cast<size_t>(p->F) * 10u << rs) + 2u * p->tree_m * threads * sizeof(float);
    };
    while ((2u << s.rs) <= most && (1u << s.rs) < n && lds(s.rs + 1, 512u) <= 64u * 1024u) ++s.rs;
    s.per = std::max(1u, std::min(p->n_ttrees, most >> s.rs));
    u32 const lanes = (s.per * p->max_units) << s.rs;
    s.threads = (std::max(lanes, std::min(256u, p->F << s.rs)) + 63u) / 64u * 64u; // some to load the rows with
    s.lds = lds(s.rs, s.threads);
    s.blocks = (n + (1u << s.rs) - 1u) >> s.rs;
    s.split = static_cast<u32>(std::min<u64>((p->n_ttrees + s.per - 1u) / s.per, std::max<u64>(1, kLaneFill / s.blocks)));
    return s;
}

// Microseconds of a batch, measured over 1 to 1,000 trees of 4 to 12 levels x 1 to 1,024 rows
// of 28 and 200 features.  Several workgroups a row block (shares) zero the output, add to
// it and convert it.
double shares_us(bh_predictor const *p, u64 n, u32 shares)
{
    return shares > 1 ? 6.0 + static_cast<double>(n) * (p->F + 1) * 8.0 * (2.0 + shares) / 3e6 : 0.0;
}
// Whole walks: a wave's trees one after the other, 2.1 us a block of seven splits.
double whole_us(bh_predictor const *p, u64 n, u32 split)
{
    u64 const wgs = (n + kTreeShapRows - 1) / kTreeShapRows * split;
    u32 const cu = std::max<u32>(1u, std::min<size_t>(kTreeShapFill / 256u, 160u * 1024u / tree_shap_lds(p->F)));
    u32 const trees = (p->n_ttrees + split * (kTreeShapThreads / 64u) - 1u) / (split * (kTreeShapThreads / 64u));
    return static_cast<double>((wgs + 256u * cu - 1) / (256u * cu)) * (2.1 * p->max_units * trees + 0.08 * p->F) +
           shares_us(p, n, split);
}
// A tree a workgroup: 256 at a time.
double split_us(bh_predictor const *p, u64 n)
{
    u64 const walks = (n + kTreeShapRows - 1) / kTreeShapRows * p->n_ttrees;
    if (!p->max_shares || walks > kSplitWalks) return 1e300;
    return static_cast<double>((walks + 255) / 256) * (7.0 + 0.47 * p->max_units + 0.04 * p->F) + shares_us(p, n, 2);
}
// A lane a block and row: 8 ps and more by the levels of the way down; its rows' loads.
double lanes_us(bh_predictor const *p, u64 n, u32 upper, LaneShape const &s)
{
    double const lanes = static_cast<double>(n) * p->n_ttrees * p->max_units;
    double const per = std::max(20.0, 7.0 + 1.2 * upper * upper) * (p->tree_m <= 5 ? 1.0 : 1.3);
    double const load = 0.1 * (p->F << s.rs) / s.threads * ((s.blocks * s.split + 1023) / 1024);
    return 7.0 + 0.6 * upper + load + lanes * 1e-6 * per + shares_us(p, n, s.split);
}

// The node counts and levels the tree form's kernels are built for.
#define BH_FORMS(LAUNCH)                       \
    if (upper <= 5) {                          \
        if (p->tree_m <= 2) LAUNCH(2, 5);      \
        else if (p->tree_m == 3) LAUNCH(3, 5); \
        else LAUNCH(4, 5);                     \
    } else if (p->tree_m <= 4) {               \
        LAUNCH(4, 9);                          \
    } else if (p->tree_m == 5) {               \
        LAUNCH(5, 9);                          \
    } else {                                   \
        LAUNCH(6, 9);                          \
    }

int launch_shap_tree(bh_predictor *p, u8 const *d_bins, u64 n, u64 stride, double *d_out, hipStream_t s)
{
    u32 const blocks = static_cast<u32>((n + kTreeShapRows - 1) / kTreeShapRows);
    u32 const upper = p->tree_depth > kTBlockLevels ? p->tree_depth - kTBlockLevels : 0u;
    // Every launch gives a row the same bits: the cheapest one.
    // Whole walks: the trees of a row block over `shares` workgroups, the fewest rounds of
    // kTreeShapFill workgroups per share of the trees, then the fewest shares; or one, where
    // adding to the output costs more than that saves.
    u32 const waves = kTreeShapThreads / 64u;
    u32 const most = std::min(std::max(1u, kTreeShapFill / std::min(blocks, kTreeShapFill)) + 7u,
                              std::max(1u, (p->n_ttrees + waves - 1) / waves));
    u32 shares = 1;
    u64 rounds = (static_cast<u64>(blocks) + kTreeShapFill - 1) / kTreeShapFill;
    for (u32 k = 2; k <= most && blocks < 16u * kTreeShapFill; ++k) {
        u64 const r = (static_cast<u64>(blocks) * k + kTreeShapFill - 1) / kTreeShapFill;
        if (r * shares < rounds * k) {
            rounds = r;
            shares = k;
        }
    }
    double us = whole_us(p, n, shares);
    if (double const one = whole_us(p, n, 1); one < us) {
        us = one;
        shares = 1;
    }
    LaneShape const ls = lane_shape(p, n);
    enum { kWhole, kSplit, kLanes } form = kWhole;
    if (split_us(p, n) < us) {
        us = split_us(p, n);
        form = kSplit;
        shares = 2; // at least: the output is added to
    }
    if (p->n_ttrees && lanes_us(p, n, upper, ls) < 0.9 * us && ls.blocks <= 0x7FFFFFFFu) {
        form = kLanes;
        shares = ls.split;
    }
    u64 const cells = n * (p->F + 1);
    u32 const cgrid = static_cast<u32>(std::min<u64>((cells + 255) / 256, 4096));
    if (shares > 1) {
        hipLaunchKernelGGL(k_shap_zero, dim3(cgrid), dim3(256), 0, s, reinterpret_cast<unsigned long long *>(d_out),
                           cells);
        SHIP(hipGetLastError());
    }
    size_t const lds = tree_shap_lds(p->F);
    if (form == kLanes) {
        dim3 const grid(static_cast<u32>(ls.blocks), ls.split);
#define BH_SL(MV, UV)                                                                                              \
    hipLaunchKernelGGL((p->tree_wide ? k_shap_lanes<MV, UV, true> : k_shap_lanes<MV, UV, false>), grid,            \
                       dim3(ls.threads), ls.lds, s, d_bins, n, stride, p->F, p->d_last, p->d_tslots, p->d_units,   \
                       p->d_ufirst, p->n_ttrees, ls.per, ls.rs, upper, p->quad, p->lr, p->shap_bias,               \
                       p->tree_scale, d_out)
        BH_FORMS(BH_SL)
#undef BH_SL
    } else if (form == kSplit) {
        dim3 const grid(blocks, p->n_ttrees);
#define BH_SP(MV)                                                                                                  \
    hipLaunchKernelGGL((p->tree_wide ? k_shap_split<MV, true> : k_shap_split<MV, false>), grid,                    \
                       dim3(kSplitThreads), split_lds(p->F, p->max_shares, p->tree_m), s, d_bins, n, stride, p->F, \
                       p->d_last, p->d_tslots, p->d_sfirst, p->d_split, p->n_ttrees, p->quad, d_out)
        if (p->tree_m <= 4) BH_SP(4); // deep trees have 4 nodes at least
        else if (p->tree_m == 5) BH_SP(5);
        else BH_SP(6);
#undef BH_SP
    } else {
        dim3 const grid(blocks, shares);
#define BH_TS(MV, UV)                                                                                              \
    hipLaunchKernelGGL((p->tree_wide ? k_shap_tree<MV, UV, true> : k_shap_tree<MV, UV, false>), grid,              \
                       dim3(kTreeShapThreads), lds, s, d_bins, n, stride, p->F, p->d_last, p->d_tslots,            \
                       p->d_tfirst, p->n_ttrees, p->quad, p->lr, p->shap_bias, p->tree_scale, d_out)
        BH_FORMS(BH_TS)
#undef BH_TS
    }
    SHIP(hipGetLastError());
    if (shares > 1) {
        hipLaunchKernelGGL(k_shap_to_double, dim3(cgrid), dim3(256), 0, s, d_out, n, p->F, p->lr, p->shap_bias,
                           p->tree_scale);
        SHIP(hipGetLastError());
    }
    return 0;
}

int launch_shap(bh_predictor *p, u8 const *d_bins, u64 n, u64 stride, double *d_out, hipStream_t s)
{
    if (n == 0) return 0;
    if (p->tree_m) return launch_shap_tree(p, d_bins, n, stride, d_out, s);
    size_t const lds = static_cast<size_t>(kShapRows) * p->F * (sizeof(unsigned long long) + 1u);
    if (lds > 160u * 1024u) return sfail(1, "TreeSHAP: too many features for the LDS accumulators");
    u32 const blocks = static_cast<u32>((n + kShapRows - 1) / kShapRows);
    // Split the path groups of each row block over `split` workgroups while the row
    // blocks alone leave the chip idle; every workgroup keeps at least one group per wave.
    u32 split = 1;
    if (blocks < kShapFillBlocks)
        split = std::min((kShapFillBlocks + blocks - 1) / blocks, std::max(1u, p->n_groups / 4u));
    u64 const cells = n * (p->F + 1);
    u32 const cgrid = static_cast<u32>(std::min<u64>((cells + 255) / 256, 4096));
    if (split > 1) {
        hipLaunchKernelGGL(k_shap_zero, dim3(cgrid), dim3(256), 0, s, reinterpret_cast<unsigned long long *>(d_out),
                           cells);
        SHIP(hipGetLastError());
    }
    dim3 const grid(blocks, split);
    // Paths of at most 8 features take half the registers and a quarter of the polynomial's
    // work: 16,384 rows x 300 features, 1,000 depth-8 trees 83.9 ms (16 slots: 199.5).
    hipLaunchKernelGGL((p->max_len <= 8 ? k_shap<8> : k_shap<kMaxPath>), grid, dim3(256), lds, s, d_bins, n, stride,
                       p->F, p->d_elems, p->d_heads, p->n_groups, p->max_len, p->d_w, p->d_last, p->lr, p->shap_bias,
                       p->shap_scale, d_out);
    SHIP(hipGetLastError());
    if (split > 1) {
        hipLaunchKernelGGL(k_shap_to_double, dim3(cgrid), dim3(256), 0, s, d_out, n, p->F, p->lr, p->shap_bias,
                           p->shap_scale);
        SHIP(hipGetLastError());
    }
    return 0;
}

// A host call's buffers: allocating, copying and freeing around a kernel of some 20 us took
// about 60 us.  Calls whose rows and results fit kWsBytes take the predictor's pinned and
// device buffers (made by the first one, freed with the predictor) unless another thread's
// call holds them; then, and for larger batches, buffers are allocated for the call.
constexpr size_t kWsBytes = 1u << 20;
class SmallCall {
public:
    SmallCall(bh_predictor *p, size_t in, size_t out) : p_(p), out_((in + 255u) & ~static_cast<size_t>(255)), lock_(p->ws_busy, std::defer_lock)
    {
        if (in > kWsBytes || out > kWsBytes || out_ + out > kWsBytes || !lock_.try_lock()) return;
        if (!p->ws_host && hipHostMalloc(reinterpret_cast<void **>(&p->ws_host), kWsBytes, hipHostMallocDefault) != hipSuccess)
            p->ws_host = nullptr;
        if (!p->ws_dev && hipMalloc(&p->ws_dev, kWsBytes) != hipSuccess) p->ws_dev = nullptr;
        ready_ = p->ws_host && p->ws_dev;
        if (!ready_) (void)hipGetLastError();
    }
    bool ready() const { return ready_; }
    unsigned char *host_in() const { return p_->ws_host; }
    unsigned char *host_out() const { return p_->ws_host + out_; }
    unsigned char *dev_in() const { return p_->ws_dev; }
    unsigned char *dev_out() const { return p_->ws_dev + out_; }

private:
    bh_predictor *p_;
    size_t out_; // results' offset
    std::unique_lock<std::mutex> lock_;
    bool ready_ = false;
};

// A predictor's device data: the small arrays share one allocation and one copy (13 of each
// took 60 us of the 200 a small predictor takes to create), large ones have their own (in
// one allocation of 20 MB the first TreeSHAP pass took 12.0 ms where it takes 10.1 so).
class Upload {
public:
    template <typename T> void add(T *&dev, T const *src, size_t count)
    {
        parts_.push_back({reinterpret_cast<void **>(&dev), src, count * sizeof(T)});
    }
    // The allocations, also after an error, go to `owned`.
    hipError_t run(std::vector<void *> &owned)
    {
        std::vector<unsigned char> host;
        auto const get = [&](void **ptr, size_t bytes) {
            hipError_t const e = hipMalloc(ptr, bytes);
            if (e == hipSuccess) owned.push_back(*ptr);
            return e;
        };
        for (Part &q : parts_) {
            if (q.bytes > kLarge) {
                if (hipError_t const e = get(q.dev, q.bytes); e != hipSuccess) return e;
                if (hipError_t const e = hipMemcpy(*q.dev, q.src, q.bytes, hipMemcpyHostToDevice); e != hipSuccess) return e;
                continue;
            }
            q.at = host.size();
            host.resize(host.size() + ((std::max<size_t>(q.bytes, 16) + 255u) & ~static_cast<size_t>(255)));
            if (q.bytes) std::memcpy(host.data() + q.at, q.src, q.bytes);
        }
        void *base = nullptr;
        if (hipError_t const e = get(&base, std::max<size_t>(host.size(), 16)); e != hipSuccess) return e;
        for (Part const &q : parts_)
            if (q.bytes <= kLarge) *q.dev = static_cast<unsigned char *>(base) + q.at;
        return hipMemcpy(base, host.data(), host.size(), hipMemcpyHostToDevice);
    }

private:
    static constexpr size_t kLarge = 256u << 10;
    struct Part {
        void **dev;
        void const *src;
        size_t bytes, at = 0;
    };
    std::vector<Part> parts_;
};

// Whole words (both ends lie in buffers of kWsBytes).
__global__ void k_copy_words(u32 const *__restrict__ src, u32 *__restrict__ dst, u32 n)
{
    for (u32 i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) dst[i] = src[i];
}
void launch_copy_words(hipStream_t s, void const *src, void *dst, size_t bytes)
{
    u32 const n = static_cast<u32>((bytes + 3u) / 4u);
    hipLaunchKernelGGL(k_copy_words, dim3(std::min(256u, (n + 255u) / 256u)), dim3(256), 0, s,
                       static_cast<u32 const *>(src), static_cast<u32 *>(dst), n);
}

} // namespace

extern "C" {

int bh_predictor_create(int device, const bh_node *nodes, const uint32_t *tree_offsets, uint32_t n_trees,
                        const uint16_t *last_bin, uint32_t n_features, float learning_rate, float init_score,
                        bh_predictor **out)
{
    *out = nullptr;
    if (n_features == 0) return sfail(1, "no features");
    SHIP(hipSetDevice(device));
    auto *p = new bh_predictor();
    p->device = device;
    p->n_trees = n_trees;
    p->F = n_features;
    p->lr = learning_rate;
    p->init = init_score;
    std::vector<PNode> pn;
    std::vector<u32> roots(n_trees);
    std::vector<SElem> el;
    std::vector<SHead> hd;
    size_t max_len = 0;
    double ev_sum = 0.0;
    std::vector<std::vector<u32>> levels(n_trees);
    std::vector<u32> seen(n_features, 0u);
    u32 deepest = 0;
    LeafStats leaves;
    leaves.top.assign(n_trees, 0.0);
    for (u32 t = 0; t < n_trees; ++t) {
        bh_node const *tn = nodes + tree_offsets[t];
        u32 const end = t + 1 < n_trees ? tree_offsets[t + 1] : 0;
        // node count: walk reachable ids (covers the whole array for grown trees)
        u32 count = 0;
        std::vector<u32> stack{0};
        while (!stack.empty()) {
            u32 const i = stack.back();
            stack.pop_back();
            count = std::max(count, i + 1);
            if (tn[i].feature < 0) {
                double const a = std::fabs(static_cast<double>(tn[i].value));
                leaves.finite = leaves.finite && std::isfinite(a);
                leaves.top[t] = std::max(leaves.top[t], a);
                leaves.sum += a;
            } else {
                if (static_cast<u32>(tn[i].feature) >= n_features || tn[i].bin > 255) {
                    delete p;
                    return sfail(1, "tree node out of range (feature id or bin)");
                }
                double const c = tn[i].cover, l = tn[tn[i].left].cover, r = tn[tn[i].right].cover;
                leaves.covers = leaves.covers && (c <= 0.0 || (l >= 0.0 && r >= 0.0 && l + r <= c * 1.0001));
                stack.push_back(tn[i].left);
                stack.push_back(tn[i].right);
            }
        }
        (void)end;
        if (count > 65535) {
            delete p;
            return sfail(1, "tree larger than 65535 nodes");
        }
        roots[t] = static_cast<u32>(pn.size());
        for (u32 i = 0; i < count; ++i) {
            PNode q{};
            if (tn[i].feature < 0) {
                q.feature = 0xFFFFu;
                q.u.value = tn[i].value;
            } else {
                q.feature = static_cast<u16>(tn[i].feature);
                q.bin = static_cast<u8>(tn[i].bin);
                q.dl = static_cast<u8>(tn[i].default_left);
                q.u.c.left = static_cast<u16>(tn[i].left);
                q.u.c.right = static_cast<u16>(tn[i].right);
            }
            pn.push_back(q);
        }
        levels[t].assign(count, 0u);
        deepest = std::max(deepest, tree_levels(tn, 0, levels[t], seen, 0, max_len));
        ev_sum += expected_value(tn, 0);
    }
    if (max_len > static_cast<size_t>(kMaxPath)) {
        delete p;
        return sfail(1, "TreeSHAP paths longer than 16 features are not supported");
    }
    // bias column: sum of per-tree expected values, times lr, plus init
    // (include/bonsai/booster.hpp:902-925).
    p->shap_bias = ev_sum * static_cast<double>(learning_rate) + static_cast<double>(init_score);
    p->max_len = static_cast<u32>(std::max<size_t>(max_len, 1));
    // The tree form serves every ensemble whose trees, paths and feature count fit its
    // kernels; the packed form the rest, and deep trees on few features: past 8 levels the
    // walk runs one wave a SIMD, and paths of at most 8 features take the short body (4
    // features, 5 depth-12 trees: 16,384 rows 2,437 -> 1,645 us, 64 rows 255 -> 41).
    bool const tree_form = deepest <= kTreeShapMaxDepth && max_len <= 2 * kTreeShapMaxM &&
                           tree_shap_lds(n_features) <= 160u * 1024u && (deepest <= 8u || max_len > 8u);
    if (!tree_form) {
        std::vector<ActiveElem> act;
        size_t longest = 0;
        for (u32 t = 0; t < n_trees; ++t) pack_paths(nodes + tree_offsets[t], last_bin, 0, act, el, hd, longest);
    }
    p->n_heads = static_cast<u32>(hd.size());
    // Interleave the paths in groups of 64: element j of the group's paths contiguous.
    u32 const K = p->max_len;
    p->n_groups = (p->n_heads + 63u) / 64u;
    std::vector<SElem> el2(static_cast<size_t>(p->n_groups) * K * 64u);
    std::vector<SHead> hd2(static_cast<size_t>(p->n_groups) * 64u);
    double leaf_abs = 0.0;
    for (size_t q = 0; q < hd.size(); ++q) {
        size_t const g = q / 64u, l = q % 64u;
        hd2[g * 64u + l] = hd[q];
        hd2[g * 64u + l].first = 0;
        for (u32 j = 0; j < hd[q].n; ++j) el2[(g * K + j) * 64u + l] = el[hd[q].first + j];
        leaf_abs += std::fabs(static_cast<double>(hd[q].value));
    }
    // |one path's contribution| <= |value| * sum_i w_i C(n, i) < 4 |value| for n <= 16,
    // so every accumulator stays below 2^61 in magnitude.
    p->shap_scale = std::ldexp(1.0, 61) / std::max(4.0 * leaf_abs, 1e-300);
    el.swap(el2);
    hd.swap(hd2);
    // Permutation weights w_i = 1 / (n C(n-1, i)) (shap_path_weights, src/shap_paths.cpp:165-194).
    std::vector<float> w(kMaxPath * (kMaxPath + 1) / 2, 0.0F);
    {
        std::vector<double> binom(kMaxPath, 0.0);
        binom[0] = 1.0;
        for (size_t nn = 1; nn <= static_cast<size_t>(kMaxPath); ++nn) {
            size_t const rr = nn - 1;
            if (rr > 0) {
                binom[rr] = 0.0;
                for (size_t i = rr + 1; i-- > 1;) binom[i] += binom[i - 1];
            }
            for (size_t i = 0; i < nn; ++i)
                w[rr * nn / 2 + i] = static_cast<float>(1.0 / (static_cast<double>(nn) * binom[i]));
        }
    }
    if (n_trees) p->mean_levels = std::log2((static_cast<double>(pn.size()) / n_trees + 1.0) / 2.0);
    TreePacker pack{};
    std::vector<u32> tfirst;
    std::vector<SplitTree> split;
    std::vector<u32> ufirst; // of every tree: its first unit
    std::vector<std::vector<std::pair<u32, u32>>> spans;
    if (tree_form) {
        // kernels' node counts: 2, 3, 4 (up to 8 levels), 4, 5, 6 (more)
        u32 const m = std::max<u32>(deepest <= 8 ? 2u : 4u, (p->max_len + 1u) / 2u);
        int const bits = tree_grid(leaves, deepest, p->tree_wide);
        double const scale = std::ldexp(1.0, bits);
        pack.last = last_bin;
        pack.F = n_features;
        pack.scale = scale;
        pack.rule = gauss_legendre(m);
        u32 const cut = deepest > kSplitAbove ? TreePacker::cut_of(deepest) : 0u;
        u32 walked = 0, most = 0; // trees with splits; shares of one
        for (u32 t = 0; t < n_trees; ++t) {
            pack.t = nodes + tree_offsets[t];
            pack.levels = levels[t].data();
            if (pack.t[0].feature < 0) continue; // a single leaf has no contributions
            ++walked;
            if (cut) most = std::max(most, pack.count(0, 0, cut));
        }
        // The split form serves up to kSplitWalks trees whose shares' values fit LDS.
        if (walked <= kSplitWalks && split_lds(n_features, most, m) <= 160u * 1024u) p->max_shares = most;
        pack.out.reserve(pn.size() * (p->max_shares ? 3u : 2u) + 256u); // about 1.5 slots a node each
        for (u32 t = 0; t < n_trees; ++t) {
            pack.t = nodes + tree_offsets[t];
            pack.levels = levels[t].data();
            if (pack.t[0].feature < 0) continue;
            pack.spans.assign(levels[t].size(), {0u, 0u});
            tfirst.push_back(static_cast<u32>(pack.out.size()));
            ufirst.push_back(static_cast<u32>(pack.units.size()));
            pack.walk(0, 0);
            p->max_units = std::max(p->max_units, static_cast<u32>(pack.units.size()) - ufirst.back());
            if (p->max_shares) spans.push_back(std::move(pack.spans));
        }
        tfirst.push_back(static_cast<u32>(pack.out.size()));
        ufirst.push_back(static_cast<u32>(pack.units.size()));
        for (u32 t = 0, k = 0; p->max_shares && t < n_trees; ++t) {
            pack.t = nodes + tree_offsets[t];
            pack.levels = levels[t].data();
            if (pack.t[0].feature < 0) continue;
            pack.spans = std::move(spans[k++]);
            SplitTree st{static_cast<u32>(pack.first.size()), 0u, kNone, 0u};
            pack.shares(0, 0, cut);
            st.n_shares = static_cast<u32>(pack.first.size()) - st.share0;
            if (!pack.is_share(0, 0, cut)) {
                u32 share = 0;
                st.top = static_cast<u32>(pack.out.size());
                pack.top(0, 0, cut, share);
            }
            split.push_back(st);
        }
        pack.out.resize((pack.out.size() / 64u + 3u) * 64u); // the kernel reads whole groups, two ahead
        double g = 1.0;
        p->quad = tree_quad(pack.rule, g);
        p->tree_m = m;
        p->tree_depth = deepest;
        p->n_ttrees = static_cast<u32>(tfirst.size() - 1);
        p->tree_scale = leaves.finite ? scale * g : std::nan("");
    }
    std::vector<u32> words;
    std::vector<Tile> tiles;
    std::vector<TileTree> ttrees;
    if (pack_tiles(nodes, tree_offsets, n_trees, n_features, words, tiles, ttrees))
        p->n_tiles = static_cast<u32>(tiles.size());
    Upload up;
    up.add(p->d_nodes, pn.data(), pn.size());
    up.add(p->d_roots, roots.data(), roots.size());
    up.add(p->d_last, last_bin, n_features);
    up.add(p->d_elems, el.data(), el.size());
    up.add(p->d_heads, hd.data(), hd.size());
    up.add(p->d_w, w.data(), w.size());
    up.add(p->d_words, words.data(), words.size());
    up.add(p->d_tiles, tiles.data(), tiles.size());
    up.add(p->d_ttrees, ttrees.data(), ttrees.size());
    up.add(p->d_tslots, pack.out.data(), pack.out.size());
    up.add(p->d_tfirst, tfirst.data(), tfirst.size());
    up.add(p->d_sfirst, pack.first.data(), pack.first.size());
    up.add(p->d_split, split.data(), split.size());
    up.add(p->d_units, pack.units.data(), pack.units.size());
    up.add(p->d_ufirst, ufirst.data(), ufirst.size());
    hipError_t e = up.run(p->owned);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        bh_predictor_destroy(p);
        return sfail(-1, std::string("hip: predictor upload: ") + hipGetErrorString(e));
    }
    *out = p;
    return 0;
}

int bh_predictor_destroy(bh_predictor *p)
{
    if (!p) return 0;
    (void)hipSetDevice(p->device);
    for (void *q : p->owned) (void)hipFree(q);
    if (p->ws_dev) (void)hipFree(p->ws_dev);
    if (p->ws_host) (void)hipHostFree(p->ws_host);
    if (p->stream) (void)hipStreamDestroy(p->stream);
    delete p;
    return 0;
}

int bh_predict_device(bh_predictor *p, const uint8_t *d_bins, uint64_t n, uint64_t row_stride, float *d_out,
                      void *hip_stream)
{
    if (!p) return sfail(1, "null predictor");
    if (row_stride < p->F) return sfail(1, "row_stride < n_features");
    return launch_predict(p, d_bins, n, row_stride, d_out, static_cast<hipStream_t>(hip_stream));
}

int bh_shap_device(bh_predictor *p, const uint8_t *d_bins, uint64_t n, uint64_t row_stride, double *d_out,
                   void *hip_stream)
{
    if (!p) return sfail(1, "null predictor");
    if (row_stride < p->F) return sfail(1, "row_stride < n_features");
    return launch_shap(p, d_bins, n, row_stride, d_out, static_cast<hipStream_t>(hip_stream));
}

int bh_predict(bh_predictor *p, const uint8_t *bins, uint64_t n, uint64_t row_stride, float *out)
{
    if (!p) return sfail(1, "null predictor");
    if (row_stride < p->F) return sfail(1, "row_stride < n_features");
    if (n == 0) return 0;
    SHIP(hipSetDevice(p->device));
    if (!served_from_tiles(p, n)) {
        // the walk reads a row once and writes one value: both stay in host memory
        SmallCall c(p, n * row_stride, n * sizeof(float));
        if (c.ready()) {
            std::memcpy(c.host_in(), bins, n * row_stride);
            if (int rc = launch_predict(p, c.host_in(), n, row_stride, reinterpret_cast<float *>(c.host_out()), p->stream))
                return rc;
            SHIP(hipStreamSynchronize(p->stream));
            std::memcpy(out, c.host_out(), n * sizeof(float));
            return 0;
        }
    }
    u8 *d_bins = nullptr;
    float *d_out = nullptr;
    SHIP(hipMalloc(&d_bins, n * row_stride));
    SHIP(hipMalloc(&d_out, n * sizeof(float)));
    SHIP(hipMemcpy(d_bins, bins, n * row_stride, hipMemcpyHostToDevice));
    int rc = launch_predict(p, d_bins, n, row_stride, d_out, p->stream);
    if (rc == 0) {
        hipError_t e = hipStreamSynchronize(p->stream);
        if (e == hipSuccess) e = hipMemcpy(out, d_out, n * sizeof(float), hipMemcpyDeviceToHost);
        if (e != hipSuccess) rc = sfail(-1, std::string("hip: predict: ") + hipGetErrorString(e));
    }
    (void)hipFree(d_bins);
    (void)hipFree(d_out);
    return rc;
}

int bh_shap(bh_predictor *p, const uint8_t *bins, uint64_t n, uint64_t row_stride, double *out)
{
    if (!p) return sfail(1, "null predictor");
    if (row_stride < p->F) return sfail(1, "row_stride < n_features");
    if (n == 0) return 0;
    SHIP(hipSetDevice(p->device));
    {
        // many workgroups read a row and add to its contributions: device buffers, with the
        // copies in the stream
        size_t const nb = n * row_stride, no = n * (p->F + 1) * sizeof(double);
        SmallCall c(p, nb, no);
        if (c.ready()) {
            std::memcpy(c.host_in(), bins, nb);
            launch_copy_words(p->stream, c.host_in(), c.dev_in(), nb);
            if (int rc = launch_shap(p, c.dev_in(), n, row_stride, reinterpret_cast<double *>(c.dev_out()), p->stream))
                return rc;
            launch_copy_words(p->stream, c.dev_out(), c.host_out(), no);
            SHIP(hipGetLastError());
            SHIP(hipStreamSynchronize(p->stream));
            std::memcpy(out, c.host_out(), no);
            return 0;
        }
    }
    u8 *d_bins = nullptr;
    double *d_out = nullptr;
    SHIP(hipMalloc(&d_bins, n * row_stride));
    SHIP(hipMalloc(&d_out, n * (p->F + 1) * sizeof(double)));
    SHIP(hipMemcpy(d_bins, bins, n * row_stride, hipMemcpyHostToDevice));
    int rc = launch_shap(p, d_bins, n, row_stride, d_out, p->stream);
    if (rc == 0) {
        hipError_t e = hipStreamSynchronize(p->stream);
        if (e == hipSuccess) e = hipMemcpy(out, d_out, n * (p->F + 1) * sizeof(double), hipMemcpyDeviceToHost);
        if (e != hipSuccess) rc = sfail(-1, std::string("hip: shap: ") + hipGetErrorString(e));
    }
    (void)hipFree(d_bins);
    (void)hipFree(d_out);
    return rc;
}

} // extern "C"


// ---------------------------------------------------------------------------------
// Continuous-batching serving loop (cfg4).  Requests arrive on a clock; whenever an
// execution slot (one HIP stream with its pinned staging and device buffers) is free,
// every request that has arrived and still fits the slot's row capacity and the HBM
// budget is packed into one batch: rows H2D, predict (+ TreeSHAP), results D2H, all
// asynchronous on the slot's stream, so batches on different slots overlap on the
// device.  Each row's result depends only on that row (per-row kernels, fixed-order
// reductions), so a request's output is identical alone and in any batch.
// ---------------------------------------------------------------------------------
namespace {

struct Slot {
    hipStream_t stream = nullptr;
    hipEvent_t done = nullptr;
    hipEvent_t k0 = nullptr, k1 = nullptr; // the batch's kernels: first start, last end
    u8 *h_rows = nullptr, *d_rows = nullptr;
    float *h_pred = nullptr, *d_pred = nullptr;
    double *h_shap = nullptr, *d_shap = nullptr;
    std::vector<u32> reqs; // requests in the batch
    u64 rows = 0;
    u64 bytes = 0;
    bool busy = false;
};

} // namespace

extern "C" int bh_serve(bh_predictor *p, const uint8_t *rows, uint64_t row_stride, const uint64_t *req_offsets,
                        const double *arrival_s, uint32_t n_req, const bh_serve_config *cfg, float *pred_out,
                        double *shap_out, double *latency_ms, bh_serve_stats *stats)
{
    if (!p) return sfail(1, "null predictor");
    if (row_stride < p->F) return sfail(1, "row_stride < n_features");
    if (cfg->n_slots == 0 || cfg->max_batch_rows == 0) return sfail(1, "n_slots and max_batch_rows must be > 0");
    SHIP(hipSetDevice(p->device));
    u32 const F = p->F;
    bool const shap = cfg->do_shap != 0;
    u64 const per_row = row_stride + sizeof(float) + (shap ? (F + 1) * sizeof(double) : 0);
    for (u32 i = 0; i < n_req; ++i)
        if (req_offsets[i + 1] - req_offsets[i] > cfg->max_batch_rows)
            return sfail(1, "a request is larger than max_batch_rows");
    std::vector<Slot> slots(cfg->n_slots);
    u64 const cap = cfg->max_batch_rows;
    hipError_t e = hipSuccess;
    for (auto &s : slots) {
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&s.stream, hipStreamNonBlocking);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming);
        if (e == hipSuccess) e = hipEventCreate(&s.k0);
        if (e == hipSuccess) e = hipEventCreate(&s.k1);
        if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void **>(&s.h_rows), cap * row_stride, 0);
        if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void **>(&s.h_pred), cap * sizeof(float), 0);
        if (e == hipSuccess) e = hipMalloc(&s.d_rows, cap * row_stride);
        if (e == hipSuccess) e = hipMalloc(&s.d_pred, cap * sizeof(float));
        if (shap) {
            if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void **>(&s.h_shap), cap * (F + 1) * sizeof(double), 0);
            if (e == hipSuccess) e = hipMalloc(&s.d_shap, cap * (F + 1) * sizeof(double));
        }
    }
    auto cleanup = [&]() {
        for (auto &s : slots) {
            if (s.stream) (void)hipStreamSynchronize(s.stream);
            if (s.h_rows) (void)hipHostFree(s.h_rows);
            if (s.h_pred) (void)hipHostFree(s.h_pred);
            if (s.h_shap) (void)hipHostFree(s.h_shap);
            if (s.d_rows) (void)hipFree(s.d_rows);
            if (s.d_pred) (void)hipFree(s.d_pred);
            if (s.d_shap) (void)hipFree(s.d_shap);
            if (s.done) (void)hipEventDestroy(s.done);
            if (s.k0) (void)hipEventDestroy(s.k0);
            if (s.k1) (void)hipEventDestroy(s.k1);
            if (s.stream) (void)hipStreamDestroy(s.stream);
        }
    };
    if (e != hipSuccess) {
        cleanup();
        return sfail(-1, std::string("hip: serve buffers: ") + hipGetErrorString(e));
    }
    // Device-time intervals of every batch's kernels, from a base event on the first
    // slot's stream: they show whether batches of different slots ran on the device at
    // the same time.
    hipEvent_t base = nullptr;
    e = hipEventCreate(&base);
    if (e == hipSuccess) e = hipEventRecord(base, slots[0].stream);
    if (e == hipSuccess) e = hipEventSynchronize(base);
    if (e != hipSuccess) {
        if (base) (void)hipEventDestroy(base);
        cleanup();
        return sfail(-1, std::string("hip: serve events: ") + hipGetErrorString(e));
    }
    std::vector<std::pair<double, double>> kspans;
    using clk = std::chrono::steady_clock;
    auto const t0 = clk::now();
    auto now_s = [&]() { return std::chrono::duration<double>(clk::now() - t0).count(); };
    u32 next = 0, completed = 0, inflight = 0, max_inflight = 0;
    u64 inflight_bytes = 0, total_rows = 0;
    int rc = 0;
    while (completed < n_req && rc == 0) {
        bool progressed = false;
        // completions
        for (auto &s : slots) {
            if (!s.busy) continue;
            hipError_t const q = hipEventQuery(s.done);
            if (q == hipErrorNotReady) continue;
            if (q != hipSuccess) {
                rc = sfail(-1, std::string("hip: serve batch: ") + hipGetErrorString(q));
                break;
            }
            double const t_done = now_s();
            float a_ms = 0.0F, b_ms = 0.0F;
            if (hipEventElapsedTime(&a_ms, base, s.k0) == hipSuccess &&
                hipEventElapsedTime(&b_ms, base, s.k1) == hipSuccess)
                kspans.emplace_back(a_ms, b_ms);
            u64 pos = 0;
            for (u32 r : s.reqs) {
                u64 const a = req_offsets[r], nr = req_offsets[r + 1] - a;
                std::memcpy(pred_out + a, s.h_pred + pos, nr * sizeof(float));
                if (shap && shap_out)
                    std::memcpy(shap_out + a * (F + 1), s.h_shap + pos * (F + 1), nr * (F + 1) * sizeof(double));
                latency_ms[r] = (t_done - arrival_s[r]) * 1000.0;
                pos += nr;
                ++completed;
            }
            inflight -= static_cast<u32>(s.reqs.size());
            inflight_bytes -= s.bytes;
            s.busy = false;
            s.reqs.clear();
            progressed = true;
        }
        if (rc) break;
        // admissions: fill free slots with arrived requests
        double const t = now_s();
        for (auto &s : slots) {
            if (s.busy || next >= n_req || arrival_s[next] > t) continue;
            u64 rows_in = 0, bytes_in = 0;
            while (next < n_req && arrival_s[next] <= t) {
                u64 const nr = req_offsets[next + 1] - req_offsets[next];
                u64 const nb = nr * per_row;
                bool const first = s.reqs.empty();
                if (!first && (rows_in + nr > cap || inflight_bytes + bytes_in + nb > cfg->hbm_budget)) break;
                if (first && inflight > 0 && inflight_bytes + nb > cfg->hbm_budget) break; // wait for memory
                std::memcpy(s.h_rows + rows_in * row_stride, rows + req_offsets[next] * row_stride, nr * row_stride);
                s.reqs.push_back(next);
                rows_in += nr;
                bytes_in += nb;
                ++next;
            }
            if (s.reqs.empty()) continue;
            s.rows = rows_in;
            s.bytes = bytes_in;
            inflight += static_cast<u32>(s.reqs.size());
            inflight_bytes += bytes_in;
            max_inflight = std::max(max_inflight, inflight);
            total_rows += rows_in;
            e = hipMemcpyAsync(s.d_rows, s.h_rows, rows_in * row_stride, hipMemcpyHostToDevice, s.stream);
            if (e == hipSuccess) e = hipEventRecord(s.k0, s.stream);
            if (e == hipSuccess) {
                rc = launch_predict(p, s.d_rows, rows_in, row_stride, s.d_pred, s.stream);
                if (rc == 0 && shap) rc = launch_shap(p, s.d_rows, rows_in, row_stride, s.d_shap, s.stream);
            }
            if (rc) break;
            if (e == hipSuccess) e = hipEventRecord(s.k1, s.stream);
            if (e == hipSuccess) e = hipMemcpyAsync(s.h_pred, s.d_pred, rows_in * sizeof(float), hipMemcpyDeviceToHost, s.stream);
            if (e == hipSuccess && shap)
                e = hipMemcpyAsync(s.h_shap, s.d_shap, rows_in * (F + 1) * sizeof(double), hipMemcpyDeviceToHost, s.stream);
            if (e == hipSuccess) e = hipEventRecord(s.done, s.stream);
            if (e != hipSuccess) {
                rc = sfail(-1, std::string("hip: serve enqueue: ") + hipGetErrorString(e));
                break;
            }
            s.busy = true;
            progressed = true;
        }
        if (!progressed) std::this_thread::yield();
    }
    double const wall = now_s();
    cleanup();
    (void)hipEventDestroy(base);
    if (rc) return rc;
    // Sweep the kernel spans: time with two or more batches on the device, and the most
    // at once.
    std::vector<std::pair<double, int>> ev;
    for (auto const &k : kspans) {
        ev.emplace_back(k.first, +1);
        ev.emplace_back(k.second, -1);
    }
    std::sort(ev.begin(), ev.end(), [](auto const &x, auto const &y) {
        return x.first < y.first || (x.first == y.first && x.second < y.second);
    });
    int live = 0, peak = 0;
    double overlap = 0.0, prev = 0.0;
    for (auto const &v : ev) {
        if (live >= 2) overlap += v.first - prev;
        live += v.second;
        peak = std::max(peak, live);
        prev = v.first;
    }
    std::vector<double> lat(latency_ms, latency_ms + n_req);
    std::sort(lat.begin(), lat.end());
    auto pct = [&](double q) {
        if (lat.empty()) return 0.0;
        size_t const k = std::min(lat.size() - 1, static_cast<size_t>(std::ceil(q * lat.size())) - 1);
        return lat[k];
    };
    double mean = 0.0;
    for (double v : lat) mean += v;
    stats->wall_s = wall;
    stats->rows = total_rows;
    stats->requests = n_req;
    stats->rows_per_s = wall > 0 ? static_cast<double>(total_rows) / wall : 0.0;
    stats->p50_ms = pct(0.50);
    stats->p99_ms = pct(0.99);
    stats->mean_ms = n_req ? mean / n_req : 0.0;
    stats->max_inflight = max_inflight;
    stats->device_overlap_ms = overlap;
    stats->max_device_concurrency = static_cast<uint32_t>(peak);
    return 0;
}
