// Vamana graph construction on the device: the batched incremental builder of
// build_graph (src/build_graph.cpp:95-392), node for node and edge for edge.
//
// The reference inserts the points of a random order in batches (1, 2, 4, ... up to 2% of
// n per batch).  Every point of a batch searches the graph as it stood before the batch,
// keeps the nodes it expanded, and dedupes / prunes them to its out-list; then the
// batch's edges are mirrored into their targets' lists in batch order, and every list
// longer than the degree is pruned again.  All of it is deterministic, so the device runs
// the same steps in parallel where the reference does:
//   vb_search      a wavefront per point of the batch: the greedy beam search (beam of
//                  beam_width (dist, node) keys in registers, a per-search visited bitmap
//                  in HBM, every candidate pushed in list order under the reference's
//                  rule "size < width or dist < tail"), the expanded nodes appended to
//                  the point's visit list;
//   vb_prune       a wavefront per list: the list sorted by (dist, node) (in LDS; lists over 1024
//                  keys by a segmented radix sort before), then dedupe_and_prune
//                  (build_graph.cpp:156-208) --
//                  skip the node itself and repeated ids, then two passes (alpha 1, then
//                  alpha) keeping a candidate unless alpha * d(candidate, kept) <= its
//                  distance for a kept node;
//   vb_rev_*       the mirrored edges as 64-bit keys (target << 32 | batch position),
//                  radix-sorted, so each target's new entries arrive in the reference's
//                  append order; lists that stay within the degree get them appended,
//                  the others are gathered, sorted and pruned;
//   vb_final       a wavefront per node: the final dedupe (sort by (dist, node)) and the
//                  edge row, padded with node 0 as the reference pads.
// Distances are the reference's sequential float sums (build_graph.cpp:95-102), one lane
// per pair, so every comparison sees the reference's values.
#include "bs_hip.h"
#include "bs_device.hpp"
#include "bs_order.hpp"

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <numeric>
#include <random>
#include <string>
#include <vector>

void bs_internal_set_error(const std::string& msg);
int bs_internal_exception();

namespace bvb {

using namespace bsw;
using bsd::EMPTY_KEY;
using bsd::INVALID;

// list entries are (dist, node) keys: orderable(dist) << 32 | node
__device__ __forceinline__ uint64_t lkey(float d, uint32_t id) {
    return (static_cast<uint64_t>(bsd::orderable(d)) << 32) | id;
}
__device__ __forceinline__ float lkey_dist(uint64_t k) { return bsd::key_dist(k); }

// build_graph.cpp:95-102: sum += diff * diff in dimension order (rows are 16-B aligned)
__device__ __forceinline__ float l2_seq(const float* a, const float* b, uint32_t dim) {
    float s = 0.0f;
    uint32_t i = 0;
    for (; i + 4 <= dim; i += 4) {
        const float4 x = *reinterpret_cast<const float4*>(a + i);
        const float4 y = *reinterpret_cast<const float4*>(b + i);
        float d = x.x - y.x;
        s = s + d * d;
        d = x.y - y.y;
        s = s + d * d;
        d = x.z - y.z;
        s = s + d * d;
        d = x.w - y.w;
        s = s + d * d;
    }
    for (; i < dim; ++i) {
        const float d = a[i] - b[i];
        s = s + d * d;
    }
    return s;
}

using f32x4 = float __attribute__((ext_vector_type(4)));

struct Graph {
    const float* vecs;  // n * dstride
    uint32_t dstride, dim, deg;
    uint64_t n;
    uint32_t* lid;      // n * deg
    float* ldist;       // n * deg
    uint32_t* lcnt;     // n
};

// key of element e of the register-major beam (e uniform)
template <int TR>
__device__ __forceinline__ uint64_t beam_at(const uint64_t (&beam)[TR], uint32_t e) {
    return readlane64(bsd::beam_reg<TR>(beam, e >> 6), e & 63u);
}

// value of the lane below; lane 0 gets `first` (one DPP move)
__device__ __forceinline__ uint32_t lane_below(uint32_t v, uint32_t first) {
    constexpr int WAVE_SHR1 = 0x138;
    return static_cast<uint32_t>(
        __builtin_amdgcn_update_dpp(static_cast<int>(first), static_cast<int>(v), WAVE_SHR1, 0xF, 0xF, false));
}

// push of one candidate key (LSB 0 = unexpanded) into the sorted beam of sz <= cap keys:
// sorted insert, then truncation to cap (build_graph.cpp:45-89 BeamQueue::push)
template <int TR>
__device__ __forceinline__ void beam_insert(uint64_t (&beam)[TR], uint32_t& sz, uint32_t cap, uint64_t ck) {
    uint64_t lt[TR], carry[TR];  // lt: lanes whose key stays
#pragma unroll
    for (int r = 0; r < TR; ++r) {
        lt[r] = ballot(beam[r] < ck);
        carry[r] = r == 0 ? EMPTY_KEY : readlane64(beam[r - 1], 63);
    }
#pragma unroll
    for (int r = 0; r < TR; ++r) {
        const bool here = r == 0 || lt[r - 1] == ~0ull;  // the slot, the lowest that does not stay, is not below
        const uint64_t slot = here ? ~lt[r] & (lt[r] + 1) : 0ull;
        const uint32_t plo = lane_below(static_cast<uint32_t>(beam[r]), static_cast<uint32_t>(carry[r]));
        const uint32_t phi = lane_below(static_cast<uint32_t>(beam[r] >> 32), static_cast<uint32_t>(carry[r] >> 32));
        uint64_t v = (static_cast<uint64_t>(phi) << 32) | plo;
        v = lane_in(slot) ? ck : v;
        v = lane_in(lt[r]) ? beam[r] : v;
        if (64u * r + 64u > cap) v = 64u * r + lane_id() < cap ? v : EMPTY_KEY;
        beam[r] = v;
    }
    sz = sz + 1 < cap ? sz + 1 : cap;
}

// the first unexpanded key (EMPTY_KEY if none), its register and lane (EMPTY's mark bit is set)
template <int TR>
__device__ __forceinline__ uint64_t first_open(const uint64_t (&beam)[TR], uint32_t& pr, uint32_t& pl) {
    uint64_t mp = 0;
    pr = TR;
#pragma unroll
    for (int r = TR - 1; r >= 0; --r) {
        const uint64_t m = ballot((static_cast<uint32_t>(beam[r]) & 1u) == 0u);
        pr = m != 0 ? static_cast<uint32_t>(r) : pr;
        mp = m != 0 ? m : mp;
    }
    if (pr == static_cast<uint32_t>(TR)) return EMPTY_KEY;
    pl = static_cast<uint32_t>(__builtin_ctzll(mp));
    return readlane64(bsd::beam_reg<TR>(beam, pr), pl);
}

constexpr uint32_t VS_ROWS = 32;    // rows per tile of squared differences
constexpr uint32_t VS_S = 64 + 4;   // floats per row of a tile: 16 lanes of a b128 phase hit 16 distinct 4-bank groups

// Distances of n <= 64 rows (ids in LDS, in list order) to the target, as l2_seq sums them;
// lane j gets row j's.  Up to 32 rows x 64 dimensions at a time: loaded coalesced (16 lanes per
// row, 4 rows per load, all loads in flight together), squared where they land, and passed
// through LDS to the lane that adds its row's 64 terms in dimension order.
__device__ __forceinline__ float rows_dist(const Graph& G, const float* trow, const uint32_t* ids, uint32_t n,
                                           float* tile, float* out) {
    const uint32_t lane = lane_id(), lr = lane >> 4, lc = (lane & 15u) * 4;
    for (uint32_t g0 = 0; g0 < n; g0 += VS_ROWS) {
        const uint32_t m = std::min(VS_ROWS, n - g0);
        uint32_t id[VS_ROWS / 4];
#pragma unroll
        for (uint32_t t = 0; t < VS_ROWS / 4; ++t) id[t] = ids[g0 + std::min(4 * t + lr, m - 1)];
        float s = 0.0f;
        for (uint32_t d0 = 0; d0 < G.dstride; d0 += 64) {
            const uint32_t c = d0 + lc < G.dstride ? d0 + lc : 0u;  // columns past the row are not added
            f32x4 x[VS_ROWS / 4];
#pragma unroll
            for (uint32_t t = 0; t < VS_ROWS / 4; ++t)
                if (4 * t < m) x[t] = *reinterpret_cast<const f32x4*>(G.vecs + static_cast<uint64_t>(id[t]) * G.dstride + c);
            const f32x4 y = *reinterpret_cast<const f32x4*>(trow + c);
            wave_sync();  // the previous tile's reads are done before it is overwritten
#pragma unroll
            for (uint32_t t = 0; t < VS_ROWS / 4; ++t)
                if (4 * t < m) {
                    const f32x4 d = x[t] - y;
                    *reinterpret_cast<f32x4*>(tile + (4 * t + lr) * VS_S + lc) = d * d;
                }
            wave_sync();
            const float* mine = tile + (lane & (VS_ROWS - 1)) * VS_S;
            const uint32_t cols = std::min(64u, G.dstride - d0);  // a multiple of 16
            for (uint32_t k = 0; k < cols; k += 16) {
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) {
                    const f32x4 p = *reinterpret_cast<const f32x4*>(mine + k + 4 * i);
                    s = s + p.x;
                    s = s + p.y;
                    s = s + p.z;
                    s = s + p.w;
                }
            }
        }
        if (lane < m) out[g0 + lane] = s;
    }
    wave_sync();
    return lane < n ? out[lane] : 0.0f;
}

// The greedy search of one point (build_graph.cpp:284-312), a wavefront per point.
// out: the expanded nodes as list keys in expansion order (at most outcap; *overflow set
// beyond); vis: this search's visited bitmap (cleared by the host before the batch).
// A step is a chain of dependent round trips: the node's list, the visited words, the rows.  The
// list of the next open beam entry, the likeliest next node, is requested while the current
// node's neighbours are looked at.  (Requesting every neighbour's row beside the visited words,
// also those that turn out to be seen, was slower at any number of searches: 0.55 against 0.43 ms
// below.)  50k x 128, degree 32, beam 128: 0.84 -> 0.43 ms per batch of 1000.
template <int TR>
__global__ void __launch_bounds__(256) vb_search(const Graph G, const uint32_t* order, uint64_t start, uint64_t count,
                                                 uint32_t L, uint64_t* outk, uint32_t* outn, uint32_t outcap,
                                                 uint32_t* vis, uint64_t vis_words, uint32_t* overflow) {
    __shared__ __attribute__((aligned(16))) float tiles[4][VS_ROWS * VS_S];
    __shared__ uint32_t ids_s[4][64];
    __shared__ float dist_s[4][64];
    const uint32_t lane = lane_id(), w = uniform(threadIdx.x >> 6);
    const uint64_t j = static_cast<uint64_t>(blockIdx.x) * 4 + w;
    if (j >= count) return;
    const uint32_t target = order[start + j];
    const uint32_t ep = order[0];
    const float* trow = G.vecs + static_cast<uint64_t>(target) * G.dstride;
    uint32_t* vb = vis + j * vis_words;
    uint64_t* out = outk + j * outcap;
    uint32_t* ids = ids_s[w];
    uint64_t beam[TR];
#pragma unroll
    for (int r = 0; r < TR; ++r) beam[r] = EMPTY_KEY;
    uint32_t sz = 0;
    {
        const float d0 = l2_seq(G.vecs + static_cast<uint64_t>(ep) * G.dstride, trow, G.dim);
        beam_insert<TR>(beam, sz, L, bsd::make_key(d0, ep));
        if (lane == 0) vb[ep >> 5] |= 1u << (ep & 31u);
    }
    // entry `lane` of a node's list (an entry past its length is not used) and its length
    const uint32_t le = std::min(lane, G.deg - 1);
    uint32_t nout = 0, pre = INVALID, pre_cnt = 0, pre_nb = 0;
    for (;;) {
        // the first unexpanded entry: its key, then its mark
        uint32_t pr, pl = 0;
        const uint64_t kp = first_open<TR>(beam, pr, pl);
        if (kp == EMPTY_KEY) break;
#pragma unroll
        for (int r = 0; r < TR; ++r)
            if (pr == static_cast<uint32_t>(r)) beam[r] |= (lane == pl) ? 1ull : 0ull;
        const uint32_t cur = uniform(bsd::key_id(kp));
        if (nout == outcap) {
            if (lane == 0) atomicOr(overflow, 1u);
            break;
        }
        if (lane == 0) out[nout] = lkey(bsd::key_dist(kp), cur);
        ++nout;
        uint32_t cnt = pre_cnt, nb0 = pre_nb;
        if (cur != pre) {
            cnt = G.lcnt[cur];
            nb0 = G.lid[static_cast<uint64_t>(cur) * G.deg + le];
        }
        cnt = uniform(cnt);
        // neighbours in list order; a neighbour not visited before joins the frontier
        for (uint32_t k0 = 0; k0 < cnt; k0 += 64) {
            const uint32_t k = k0 + lane;
            uint32_t nb = nb0;
            if (k0 > 0) nb = G.lid[static_cast<uint64_t>(cur) * G.deg + std::min(k, cnt - 1)];
            uint32_t seen = 0;
            const uint32_t bit = 1u << (nb & 31u);
            if (k < cnt) seen = atomicOr(&vb[nb >> 5], bit);
            if (k0 == 0) {
                uint32_t nr, nl = 0;
                const uint64_t nk = first_open<TR>(beam, nr, nl);
                pre = INVALID;
                if (nk != EMPTY_KEY) {
                    pre = uniform(bsd::key_id(nk));
                    pre_cnt = G.lcnt[pre];
                    pre_nb = G.lid[static_cast<uint64_t>(pre) * G.deg + le];
                }
            }
            const uint64_t fm = ballot(k < cnt && (seen & bit) == 0u);
            const uint32_t n = static_cast<uint32_t>(__builtin_popcountll(fm));
            if (n == 0) continue;
            if (lane_in(fm)) ids[lanes_below(fm)] = nb;
            wave_sync();
            const float d = rows_dist(G, trow, ids, n, tiles[w], dist_s[w]);
            uint64_t m = n == 64u ? ~0ull : (1ull << n) - 1ull;
            const uint32_t id = ids[lane < n ? lane : 0u];
            const uint64_t ck = lane_in(m) ? bsd::make_key(d, id) : EMPTY_KEY;
            if (sz == L && m) {
                // a full beam's last entry only moves closer, so a candidate at or beyond it
                // now is refused at its turn as well: only the others go through the pushes
                const float dl = bsd::key_dist(beam_at<TR>(beam, L - 1));
                m &= ballot(d < dl);
            }
            while (m) {
                const uint32_t l = static_cast<uint32_t>(__builtin_ctzll(m));
                m &= m - 1;
                const uint64_t c = readlane64(ck, l);
                // push if the beam has room or the distance is below the last entry's
                bool take = sz < L;
                if (!take) take = bsd::key_dist(c) < bsd::key_dist(beam_at<TR>(beam, sz - 1));
                if (take) beam_insert<TR>(beam, sz, L, c);
            }
            wave_sync();  // ids are read before the next block writes them
        }
    }
    if (lane == 0) outn[j] = nout;
}

// A vector read through the scalar cache: its address is the same in every lane, so the values
// arrive in scalar registers and the vector unit takes them as operands.
using const_row = const __attribute__((address_space(4))) f32x4*;
__device__ __forceinline__ const_row uniform_row(const Graph& G, uint32_t id) {
    return reinterpret_cast<const_row>(reinterpret_cast<uintptr_t>(G.vecs + static_cast<uint64_t>(uniform(id)) * G.dstride));
}

// s continued over one chunk of 4 dimensions, in dimension order (l2_seq's operations; the rows'
// zero padding past dim adds exactly 0)
__device__ __forceinline__ float l2_chunk(float s, f32x4 x, f32x4 y) {
    float d = x.x - y.x;
    s = s + d * d;
    d = x.y - y.y;
    s = s + d * d;
    d = x.z - y.z;
    s = s + d * d;
    d = x.w - y.w;
    return s + d * d;
}

// The two passes of the robust prune over nu sorted, deduplicated candidates; the kept ones go
// to `kept`, their number (<= deg) is returned.  A lane owns one candidate of a block of 64 and
// the least of its distances to the nodes kept so far: a * d <= e for some kept node is a *
// (least d) <= e, since rounding is monotone (a NaN distance counts for neither).  So each kept
// node costs one round in which every lane advances its own sum, instead of one dependent
// distance per candidate; the next candidate to keep is the lowest open lane.  With D4 > 0 (rows
// of 4 D4 floats) the lane's row is held in registers and the kept row comes through
// the scalar cache: a round is 3 vector instructions per dimension and no vector load (the
// former lanes each streamed two rows of scattered 16-byte pieces per distance).  50k x 128,
// degree 32, per batch of 1000: the mirrored lists 1.51 -> 0.34 ms, the visit lists 0.47 -> 0.13 ms.
// D4 = 0: any dimension, the rows read per round, each by its lane while its candidate is not
// dominated.  Degree 32, beam 128: 50k x 200 0.15 s with every lane reading, 0.12 so; 100k x 960 1.16
// and 0.80, 1M x 960 18.4 and 9.3 (18.0 when each candidate was tested against the kept ones).
template <int D4>
__device__ __forceinline__ uint32_t robust_prune(const Graph& G, const uint64_t* keys, uint32_t nu, float alpha,
                                                 uint64_t* kept) {
    const uint32_t lane = lane_id(), nch = G.dstride / 4;
    uint32_t kc = 0;
    f32x4 row[D4 > 0 ? D4 : 1];
    const f32x4* mine = nullptr;
    uint64_t e = EMPTY_KEY;
    float least = __builtin_nanf("");
    auto dist = [&](uint32_t id) __attribute__((always_inline)) {
        const const_row k = uniform_row(G, id);
        float s = 0.0f;
        if constexpr (D4 > 0) {
#pragma unroll
            for (int c = 0; c < D4; ++c) s = l2_chunk(s, row[c], k[c]);
        } else {
            for (uint32_t c = 0; c < nch; c += 4) {  // rows are a multiple of 16 floats
                f32x4 x[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) x[t] = mine[c + t];
#pragma unroll
                for (int t = 0; t < 4; ++t) s = l2_chunk(s, x[t], k[c + t]);
            }
        }
        return s;
    };
    // the lane's least distance with a kept node counted in.  Where rows are read per round (D4 = 0),
    // a lane whose candidate is dominated already, at `stay`, reads none.
    float stay = 1.0f;
    auto count_in = [&](uint32_t id) __attribute__((always_inline)) {
        if constexpr (D4 > 0) {
            least = fminf(least, dist(id));
        } else {
            if (e != EMPTY_KEY && !(stay * least <= lkey_dist(e))) least = fminf(least, dist(id));
        }
    };
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        const float a = pass == 0 ? 1.0f : alpha;
        // a single block's distances serve the second pass too: they count until alpha dominates
        stay = nu > 64 ? a : alpha;
#pragma unroll 1
        for (uint32_t c0 = 0; c0 < nu && kc < G.deg; c0 += 64) {
            const uint32_t j = c0 + lane;
            if (pass == 0 || nu > 64) {  // a single block keeps its rows and distances for the second pass
                e = j < nu ? keys[j] : EMPTY_KEY;
                // lanes past the list take its first node
                const uint32_t id = static_cast<uint32_t>(j < nu ? e : keys[0]);
                mine = reinterpret_cast<const f32x4*>(G.vecs + static_cast<uint64_t>(id) * G.dstride);
                if constexpr (D4 > 0) {
#pragma unroll
                    for (int c = 0; c < D4; ++c) row[c] = mine[c];
                }
                least = __builtin_nanf("");
#pragma unroll 1
                for (uint32_t k = 0; k < kc; ++k) count_in(static_cast<uint32_t>(kept[k]));
            }
            uint64_t after = ~0ull;
            for (;;) {
                const uint64_t open = ballot(j < nu && !(a * least <= lkey_dist(e))) & after;
                if (!open) break;
                const uint32_t l = static_cast<uint32_t>(__builtin_ctzll(open));
                after = l == 63u ? 0ull : ~0ull << (l + 1);
                const uint64_t ek = readlane64(e, l);
                if (lane == 0) kept[kc] = ek;
                ++kc;
                wave_sync();
                if (kc == G.deg) break;
                count_in(static_cast<uint32_t>(ek));
            }
        }
    }
    return kc;
}

// dedupe_and_prune (build_graph.cpp:156-208) of one sorted list of list keys, a
// wavefront per list; the result becomes node src's list.  keys are rewritten in place
// (the deduplicated prefix).  kept: LDS, deg entries per wavefront.
template <int D4>
__device__ __forceinline__ void prune_list(const Graph& G, uint64_t* keys, uint32_t n, uint32_t src, float alpha, uint64_t* kept) {
    const uint32_t lane = lane_id();
    // dedupe: skip src and an id equal to the last kept one (in place, order kept)
    uint32_t nu = 0, last = INVALID;
    for (uint32_t i0 = 0; i0 < n; i0 += 64) {
        const uint32_t i = i0 + lane;
        const uint64_t k = i < n ? keys[i] : EMPTY_KEY;
        const uint32_t id = static_cast<uint32_t>(k);
        const bool valid = i < n && id != src;
        const uint64_t vm = ballot(valid);
        // id of the closest valid element before this lane (or the carried last)
        const uint64_t below = vm & ((1ull << lane) - 1ull);
        const uint32_t src_lane = below ? 63u - static_cast<uint32_t>(__builtin_clzll(below)) : lane;
        const uint32_t pid = static_cast<uint32_t>(
            __builtin_amdgcn_ds_bpermute(static_cast<int>(src_lane << 2), static_cast<int>(id)));
        const uint32_t prev = below ? pid : last;
        const bool keep = valid && id != prev;
        const uint64_t km = ballot(keep);
        wave_sync();
        if (keep) keys[nu + lanes_below(km)] = k;
        nu += static_cast<uint32_t>(__builtin_popcountll(km));
        if (vm) last = readlane(id, 63u - static_cast<uint32_t>(__builtin_clzll(vm)));
        wave_sync();
    }
    __threadfence_block();
    uint32_t* lid = G.lid + static_cast<uint64_t>(src) * G.deg;
    float* ld = G.ldist + static_cast<uint64_t>(src) * G.deg;
    if (nu <= G.deg) {
        for (uint32_t i = lane; i < nu; i += 64) {
            const uint64_t k = keys[i];
            lid[i] = static_cast<uint32_t>(k);
            ld[i] = lkey_dist(k);
        }
        if (lane == 0) G.lcnt[src] = nu;
        return;
    }
    const uint32_t kc = robust_prune<D4>(G, keys, nu, alpha, kept);
    for (uint32_t i = lane; i < kc; i += 64) {
        const uint64_t k = kept[i];
        lid[i] = static_cast<uint32_t>(k);
        ld[i] = lkey_dist(k);
    }
    if (lane == 0) G.lcnt[src] = kc;
}

constexpr uint32_t SORT_CAP = 1024;  // keys a wavefront sorts in its LDS slice

// n <= SORT_CAP keys sorted ascending into S (LDS): up to 64 across the lanes, more by a bitonic
// network in LDS over the next power of two, padded with EMPTY keys
__device__ __forceinline__ void sort_list(const uint64_t* keys, uint32_t n, uint64_t* S) {
    const uint32_t lane = lane_id();
    if (n <= 64) {
        const uint64_t v = bsd::sort_lanes(lane < n ? keys[lane] : EMPTY_KEY, n);
        S[lane] = v;
        wave_sync();
        return;
    }
    uint32_t N = 128;
    while (N < n) N <<= 1;
    for (uint32_t i = lane; i < N; i += 64) S[i] = i < n ? keys[i] : EMPTY_KEY;
    wave_sync();
#pragma unroll 1
    for (uint32_t k = 2; k <= N; k <<= 1) {
#pragma unroll 1
        for (uint32_t j = k >> 1; j >= 1; j >>= 1) {
            for (uint32_t i = lane; i < N / 2; i += 64) {
                const uint32_t a = ((i & ~(j - 1u)) << 1) | (i & (j - 1u));
                const uint64_t x = S[a], y = S[a + j];
                const bool sw = (a & k) == 0 ? (y < x) : (x < y);
                S[a] = sw ? y : x;
                S[a + j] = sw ? x : y;
            }
            wave_sync();
        }
    }
}

// the batch's visit lists: job j = (keys at j * outcap, outn[j] keys, order[start + j]).  SORT:
// the lists are unsorted and at most SORT_CAP keys; else sorted in memory
template <int D4, bool SORT>
__global__ void __launch_bounds__(256) vb_prune_targets(const Graph G, uint64_t* keys, const uint32_t* outn,
                                                        uint32_t outcap, const uint32_t* order, uint64_t start,
                                                        uint64_t count, float alpha) {
    __shared__ uint64_t kept_s[4][128];
    __shared__ uint64_t sort_s[SORT ? 4 : 1][SORT ? SORT_CAP : 1];
    const uint32_t w = uniform(threadIdx.x >> 6);
    const uint64_t j = static_cast<uint64_t>(blockIdx.x) * 4 + w;
    if (j >= count) return;
    const uint32_t n = uniform(outn[j]), src = uniform(order[start + j]);
    if constexpr (SORT) {
        sort_list(keys + j * outcap, n, sort_s[w]);
        prune_list<D4>(G, sort_s[w], n, src, alpha, kept_s[w]);
    } else {
        prune_list<D4>(G, keys + j * outcap, n, src, alpha, kept_s[w]);
    }
}

// segment j of the visit lists for the sort in memory: [j * outcap, j * outcap + outn[j])
__global__ void __launch_bounds__(256) vb_segments(const uint32_t* outn, uint32_t outcap, uint64_t count,
                                                   uint64_t* begin, uint64_t* end) {
    const uint64_t j = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (j >= count) return;
    begin[j] = j * outcap;
    end[j] = j * outcap + outn[j];
}

// what a batch's kernels count, read by the host once per batch
struct Counters {
    unsigned long long records, big_keys;  // mirrored edges, keys of the lists to prune
    uint32_t overflow, heads, big, longest;  // searches over their list, targets, lists to prune and the longest
};

// mirrored edges: record (j, k) of the batch -> key (target << 32 | j * deg + k), or ~0
__global__ void __launch_bounds__(256) vb_rev_keys(const Graph G, const uint32_t* order, uint64_t start,
                                                   uint64_t count, uint64_t* rk, Counters* ctr) {
    const uint64_t t = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (t >= count * G.deg) return;
    const uint64_t j = t / G.deg;
    const uint32_t k = static_cast<uint32_t>(t - j * G.deg);
    const uint32_t src = order[start + j];
    uint64_t key = ~0ull;
    if (k < G.lcnt[src]) {
        key = (static_cast<uint64_t>(G.lid[static_cast<uint64_t>(src) * G.deg + k]) << 32) | static_cast<uint32_t>(t);
        atomicAdd(&ctr->records, 1ull);
    }
    rk[t] = key;
}

// sum of v over the lanes below this one, and the wavefront's total
__device__ __forceinline__ uint32_t scan_wave(uint32_t v, uint32_t& total) {
    uint32_t x = v;
    const uint32_t lane = lane_id();
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t y = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(
            static_cast<int>(((lane - d) & 63u) << 2), static_cast<int>(x)));
        x += lane >= d ? y : 0u;
    }
    total = readlane(x, 63);
    return x - v;
}

// targets of the mirrored edges: every first record of a target registers (target, begin,
// end, 0) -- end by binary search for the next target.  A target whose list outgrows the degree
// also registers a prune job (target, offset of its old + new keys in `big`, their number), its
// index + 1 in the head's last word.  One atomic per wavefront and counter: with one per
// head, in vb_rev_apply, that kernel took 214 us per batch of 1000 points, now 7.
__global__ void __launch_bounds__(256) vb_rev_heads(const Graph G, const uint64_t* rk, uint4* heads, uint4* bigjobs,
                                                    Counters* ctr) {
    const uint32_t lane = lane_id();
    const uint64_t m = ctr->records;
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    const uint32_t dst = i < m ? static_cast<uint32_t>(rk[i] >> 32) : INVALID;
    const bool head = i < m && (i == 0 || static_cast<uint32_t>(rk[i - 1] >> 32) != dst);
    uint64_t end = 0;
    uint32_t tot = 0;
    if (head) {
        uint64_t lo = i + 1, hi = m;  // first index with a larger target: doubling steps, then halving
        for (uint64_t step = 1; lo < m; step *= 2) {
            const uint64_t at = std::min<uint64_t>(lo + step - 1, m - 1);
            if (static_cast<uint32_t>(rk[at] >> 32) != dst) {
                hi = at;
                break;
            }
            lo = at + 1;
        }
        while (lo < hi) {
            const uint64_t mid = (lo + hi) / 2;
            if (static_cast<uint32_t>(rk[mid] >> 32) == dst) lo = mid + 1;
            else hi = mid;
        }
        end = lo;
        tot = G.lcnt[dst] + static_cast<uint32_t>(end - i);
    }
    const uint64_t hm = ballot(head);
    if (!hm) return;
    const bool isbig = head && tot > G.deg;
    const uint64_t bm = ballot(isbig);
    uint32_t sum = 0;
    const uint32_t before = scan_wave(isbig ? tot : 0u, sum);
    unsigned int h0 = 0, b0 = 0;
    unsigned long long off0 = 0;
    if (lane == 0) {
        h0 = atomicAdd(&ctr->heads, static_cast<uint32_t>(__builtin_popcountll(hm)));
        if (bm) {
            b0 = atomicAdd(&ctr->big, static_cast<uint32_t>(__builtin_popcountll(bm)));
            off0 = atomicAdd(&ctr->big_keys, static_cast<unsigned long long>(sum));
        }
    }
    if (isbig && tot > 64u) atomicMax(&ctr->longest, tot);
    h0 = readlane(h0, 0);
    b0 = readlane(b0, 0);
    const uint64_t off = readlane64(off0, 0) + before;
    uint32_t job = 0;
    if (isbig) {
        job = b0 + lanes_below(bm) + 1;
        bigjobs[job - 1] = make_uint4(dst, static_cast<uint32_t>(off), static_cast<uint32_t>(off >> 32), tot);
    }
    if (head) heads[h0 + lanes_below(hm)] = make_uint4(dst, static_cast<uint32_t>(i), static_cast<uint32_t>(end), job);
}

// apply the mirrored edges of one target (a wavefront each): append when the list stays
// within the degree, else gather old + new list keys for the sort and prune
__global__ void __launch_bounds__(256) vb_rev_apply(const Graph G, const uint64_t* rk, const uint4* heads,
                                                    unsigned int nheads, const uint32_t* order, uint64_t start,
                                                    uint64_t* big, const uint4* bigjobs) {
    const uint32_t lane = lane_id();
    const uint64_t h = static_cast<uint64_t>(blockIdx.x) * 4 + uniform(threadIdx.x >> 6);
    if (h >= nheads) return;
    const uint4 hd = heads[h];
    const uint32_t dst = hd.x, b = hd.y, app = hd.z - hd.y;
    const uint32_t old = G.lcnt[dst];
    uint32_t* lid = G.lid + static_cast<uint64_t>(dst) * G.deg;
    float* ld = G.ldist + static_cast<uint64_t>(dst) * G.deg;
    auto rec = [&](uint32_t k, uint32_t& src, float& d) __attribute__((always_inline)) {
        const uint32_t t = static_cast<uint32_t>(rk[b + k]);
        const uint32_t j = t / G.deg, kk = t - j * G.deg;
        src = order[start + j];
        d = G.ldist[static_cast<uint64_t>(src) * G.deg + kk];
    };
    if (hd.w == 0) {
        for (uint32_t k = lane; k < app; k += 64) {
            uint32_t src;
            float d;
            rec(k, src, d);
            lid[old + k] = src;
            ld[old + k] = d;
        }
        if (lane == 0) G.lcnt[dst] = old + app;
        return;
    }
    const uint4 jb = bigjobs[hd.w - 1];
    const uint64_t off = (static_cast<uint64_t>(jb.z) << 32) | jb.y;
    const uint32_t tot = jb.w;
    for (uint32_t k = lane; k < tot; k += 64) {
        uint64_t key;
        if (k < old) {
            key = lkey(ld[k], lid[k]);
        } else {
            uint32_t src;
            float d;
            rec(k - old, src, d);
            key = lkey(d, src);
        }
        big[off + k] = key;
    }
}

__global__ void __launch_bounds__(256) vb_big_offsets(const uint4* bigjobs, unsigned int nbig, uint64_t* begin,
                                                      uint64_t* end) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= nbig) return;
    const uint4 jb = bigjobs[i];
    const uint64_t off = (static_cast<uint64_t>(jb.z) << 32) | jb.y;
    begin[i] = off;
    end[i] = off + jb.w;
}

template <int D4, bool SORT>
__global__ void __launch_bounds__(256) vb_prune_big(const Graph G, uint64_t* keys, const uint4* bigjobs,
                                                    unsigned int nbig, float alpha) {
    __shared__ uint64_t kept_s[4][128];
    __shared__ uint64_t sort_s[SORT ? 4 : 1][SORT ? SORT_CAP : 1];
    const uint32_t w = uniform(threadIdx.x >> 6);
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 4 + w;
    if (i >= nbig) return;
    const uint4 jb = bigjobs[i];
    const uint64_t off = (static_cast<uint64_t>(jb.z) << 32) | jb.y;
    const uint32_t n = uniform(jb.w), src = uniform(jb.x);
    if constexpr (SORT) {
        sort_list(keys + off, n, sort_s[w]);
        prune_list<D4>(G, sort_s[w], n, src, alpha, kept_s[w]);
    } else {
        prune_list<D4>(G, keys + off, n, src, alpha, kept_s[w]);
    }
}

// the final dedupe_and_prune of every node (build_graph.cpp:382-390): its list (at most
// deg <= 128 entries) sorted by (dist, node), the node itself and repeats skipped, the row
// padded with node 0
template <int TR>
__global__ void __launch_bounds__(256) vb_final(const Graph G, uint32_t* edges_out) {
    const uint32_t lane = lane_id();
    const uint64_t u = static_cast<uint64_t>(blockIdx.x) * 4 + uniform(threadIdx.x >> 6);
    if (u >= G.n) return;
    const uint32_t cnt = G.lcnt[u];
    uint64_t v[TR];
#pragma unroll
    for (int r = 0; r < TR; ++r) {
        const uint32_t e = static_cast<uint32_t>(r) * 64u + lane;
        v[r] = e < cnt ? lkey(G.ldist[u * G.deg + e], G.lid[u * G.deg + e]) : EMPTY_KEY;
    }
    bsd::bitonic_sort<TR>(v);
    uint32_t nu = 0, last = INVALID;
    uint32_t* row = edges_out + u * G.deg;
#pragma unroll
    for (int r = 0; r < TR; ++r) {
        const uint32_t id = static_cast<uint32_t>(v[r]);
        const bool valid = v[r] != EMPTY_KEY && id != static_cast<uint32_t>(u);
        const uint64_t vm = ballot(valid);
        const uint64_t below = vm & ((1ull << lane) - 1ull);
        const uint32_t src_lane = below ? 63u - static_cast<uint32_t>(__builtin_clzll(below)) : lane;
        const uint32_t pid = static_cast<uint32_t>(
            __builtin_amdgcn_ds_bpermute(static_cast<int>(src_lane << 2), static_cast<int>(id)));
        const uint32_t prev = below ? pid : last;
        const bool keep = valid && id != prev;
        const uint64_t km = ballot(keep);
        const uint32_t p = nu + lanes_below(km);
        if (keep && p < G.deg) row[p] = id;
        nu += static_cast<uint32_t>(__builtin_popcountll(km));
        if (vm) last = readlane(id, 63u - static_cast<uint32_t>(__builtin_clzll(vm)));
    }
    for (uint32_t e = nu + lane; e < G.deg; e += 64) row[e] = 0u;
}

}  // namespace bvb

namespace {

int vfail(int code, const std::string& msg) {
    bs_internal_set_error(msg);
    return code;
}

template <typename F>
hipError_t launch_tr(uint32_t TR, F&& f) {
    switch (TR) {
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 8: f(std::integral_constant<int, 8>{}); break;
    default: f(std::integral_constant<int, 16>{}); break;
    }
    return hipGetLastError();
}

// the prune instance that holds rows of dstride floats in registers (0: longer than 128)
template <typename F>
hipError_t launch_d4(uint32_t dstride, F&& f) {
    switch (dstride / 16) {
    case 1: f(std::integral_constant<int, 4>{}); break;
    case 2: f(std::integral_constant<int, 8>{}); break;
    case 3: f(std::integral_constant<int, 12>{}); break;
    case 4: f(std::integral_constant<int, 16>{}); break;
    case 5: f(std::integral_constant<int, 20>{}); break;
    case 6: f(std::integral_constant<int, 24>{}); break;
    case 7: f(std::integral_constant<int, 28>{}); break;
    case 8: f(std::integral_constant<int, 32>{}); break;
    default: f(std::integral_constant<int, 0>{}); break;
    }
    return hipGetLastError();
}

struct DevBuf {
    void* p = nullptr;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
    template <typename T>
    T* as() const {
        return static_cast<T*>(p);
    }
};

// sort_cap: the most keys a list sorted in LDS may have, at most SORT_CAP; stats (may be null): the
// longest mirrored list and the batches whose mirrored lists were sorted in memory
int build_vamana(const float* vecs, uint64_t n, uint32_t dim, uint32_t degree, uint32_t beam_width, float alpha,
                 uint32_t seed, uint32_t* edges_out, int verbose, uint32_t sort_cap, uint32_t* stats) {
    if (!vecs || !edges_out) return vfail(BS_EINVAL, "vecs and edges_out must be given");
    if (n == 0) return vfail(BS_EINVAL, "base dataset is empty");
    if (n > 0x7FFFFFFFull) return vfail(BS_EINVAL, "at most 2^31-1 points");
    if (dim == 0 || dim > 4096) return vfail(BS_EINVAL, "dim must be in 1..4096");
    if (degree == 0 || degree > 128) return vfail(BS_EINVAL, "degree must be in 1..128");
    if (beam_width == 0 || beam_width > 1024) return vfail(BS_EINVAL, "beam width must be in 1..1024");
    if (!(alpha >= 1.0f)) return vfail(BS_EINVAL, "alpha must be at least 1.0");
    const auto t0 = std::chrono::steady_clock::now();
    const uint32_t dstride = (dim + 15) & ~15u;  // rows of whole 64-byte pieces, zero-padded
    const uint32_t TR = beam_width <= 64 ? 1 : beam_width <= 128 ? 2 : beam_width <= 256 ? 4 : beam_width <= 512 ? 8 : 16;
    const uint32_t outcap = std::max<uint32_t>(1024u, 4u * beam_width);

    // insertion order (build_graph.cpp:268-272)
    std::vector<uint32_t> order(n);
    std::iota(order.begin(), order.end(), 0u);
    std::mt19937 gen(seed);
    std::shuffle(order.begin(), order.end(), gen);
    const uint64_t batch_bound = std::max<uint64_t>(1, static_cast<uint64_t>(0.02 * static_cast<double>(n)));
    const uint64_t max_batch = std::min<uint64_t>(batch_bound, n);
    // searches in flight: bounded by the visited bitmaps (at most 2 GiB)
    const uint64_t vis_words = (n + 31) / 32;
    const uint64_t slots = std::max<uint64_t>(1, std::min<uint64_t>(max_batch, (2ull << 30) / (vis_words * 4)));

    DevBuf d_vecs, d_lid, d_ld, d_lcnt, d_order, d_vis, d_outk, d_outn, d_rk, d_rks, d_heads, d_ctr, d_big, d_bigjobs, d_edges,
        d_tmp;
    // of the sorts in memory: the visit lists' (beams over 256) and the mirrored lists' (made when
    // one first passes the LDS)
    DevBuf d_outs, d_segb, d_sege, d_bigs, d_beg, d_end, d_bigtmp;
    // visit lists short enough are sorted by the kernel that prunes them
    const bool sort_here = outcap <= sort_cap;
    auto alloc = [&](DevBuf& b, size_t bytes) { return hipMalloc(&b.p, std::max<size_t>(bytes, 8)) == hipSuccess; };
    const uint64_t mrec = max_batch * degree;
    const uint64_t bigcap = mrec * (static_cast<uint64_t>(degree) + 1);
    if (!alloc(d_vecs, n * dstride * 4ull) || !alloc(d_lid, n * degree * 4ull) || !alloc(d_ld, n * degree * 4ull) ||
        !alloc(d_lcnt, n * 4ull) || !alloc(d_order, n * 4ull) || !alloc(d_vis, slots * vis_words * 4ull) ||
        !alloc(d_outk, slots * outcap * 8ull) || !alloc(d_outn, slots * 4ull) ||
        !alloc(d_rk, mrec * 8ull) || !alloc(d_rks, mrec * 8ull) || !alloc(d_heads, mrec * 16ull) ||
        !alloc(d_ctr, sizeof(bvb::Counters)) || !alloc(d_big, bigcap * 8ull) || !alloc(d_bigjobs, mrec * 16ull) ||
        !alloc(d_edges, n * degree * 4ull) ||
        (!sort_here && (!alloc(d_outs, slots * outcap * 8ull) || !alloc(d_segb, slots * 8ull) || !alloc(d_sege, slots * 8ull))))
        return vfail(BS_ENOMEM, "hipMalloc of the graph-construction buffers failed");

    hipError_t e = hipSuccess;
    if (dstride == dim) {
        e = hipMemcpy(d_vecs.p, vecs, n * dim * 4ull, hipMemcpyHostToDevice);
    } else {
        // the rows as they are, up to 256 MiB at a time, spread to their padded places by a kernel
        const uint64_t rows = std::min<uint64_t>(n, std::max<uint64_t>(1, (256ull << 20) / (dim * 4ull)));
        DevBuf stage;
        if (!alloc(stage, rows * dim * 4ull)) return vfail(BS_ENOMEM, "hipMalloc of the row staging buffer failed");
        for (uint64_t r0 = 0; e == hipSuccess && r0 < n; r0 += rows) {
            const uint64_t m = std::min(rows, n - r0);
            e = hipMemcpy(stage.p, vecs + r0 * dim, m * dim * 4ull, hipMemcpyHostToDevice);
            if (e != hipSuccess) break;
            e = bso::launch_pad_rows(stage.as<float>(), m, dim, dstride, d_vecs.as<float>() + r0 * dstride, nullptr);
        }
        if (e == hipSuccess) e = hipDeviceSynchronize();  // the staging buffer is freed
    }
    if (e == hipSuccess) e = hipMemcpy(d_order.p, order.data(), n * 4ull, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(d_lcnt.p, 0, n * 4ull);
    if (e != hipSuccess) return vfail(BS_EHIP, std::string("graph construction upload: ") + hipGetErrorString(e));

    bvb::Graph G{d_vecs.as<float>(), dstride, dim, degree, n, d_lid.as<uint32_t>(), d_ld.as<float>(),
                 d_lcnt.as<uint32_t>()};
    const uint32_t* ord = d_order.as<uint32_t>();
    bvb::Counters* ctr = d_ctr.as<bvb::Counters>();

    if (slots * outcap > 0x7FFFFFFFull || bigcap > 0x7FFFFFFFull || mrec > 0xFFFFFFFFull)
        return vfail(BS_EINVAL, "batch too large for the device sorts (n or beam width too large)");
    // hipCUB work space, sized for the larger of the two sorts
    size_t tmp_bytes = 0;
    {
        size_t b1 = 0, b2 = 0;
        if (!sort_here)
            e = hipcub::DeviceSegmentedRadixSort::SortKeys(nullptr, b1, d_outk.as<uint64_t>(), d_outs.as<uint64_t>(),
                                                           static_cast<int>(slots * outcap), static_cast<int>(slots),
                                                           d_segb.as<uint64_t>(), d_sege.as<uint64_t>());
        if (e == hipSuccess)
            e = hipcub::DeviceRadixSort::SortKeys(nullptr, b2, d_rk.as<uint64_t>(), d_rks.as<uint64_t>(),
                                                  static_cast<int>(mrec));
        if (e != hipSuccess) return vfail(BS_EHIP, std::string("sort sizing: ") + hipGetErrorString(e));
        tmp_bytes = std::max(b1, b2);
        if (!alloc(d_tmp, tmp_bytes)) return vfail(BS_ENOMEM, "hipMalloc of the sort work space failed");
    }
    size_t bigtmp_bytes = 0;

    uint64_t start = 1;
    double last_print = 0.0;
    while (start < n) {
        const uint64_t end = std::min(std::min(start * 2, start + batch_bound), n);
        e = hipMemsetAsync(ctr, 0, sizeof(bvb::Counters), nullptr);
        // 1. searches and visit-list prunes, `slots` points at a time
        for (uint64_t s0 = start; e == hipSuccess && s0 < end; s0 += slots) {
            const uint64_t cnt = std::min(slots, end - s0);
            e = hipMemsetAsync(d_vis.p, 0, cnt * vis_words * 4ull, nullptr);
            if (e != hipSuccess) break;
            const dim3 wg(static_cast<uint32_t>((cnt + 3) / 4));
            e = launch_tr(TR, [&](auto trc) {
                constexpr int T = decltype(trc)::value;
                hipLaunchKernelGGL(bvb::vb_search<T>, wg, dim3(256), 0, nullptr, G, ord, s0, cnt, beam_width,
                                   d_outk.as<uint64_t>(), d_outn.as<uint32_t>(), outcap, d_vis.as<uint32_t>(),
                                   vis_words, &ctr->overflow);
            });
            if (e == hipSuccess && !sort_here) {
                hipLaunchKernelGGL(bvb::vb_segments, dim3(static_cast<uint32_t>((cnt + 255) / 256)), dim3(256), 0, nullptr,
                                   d_outn.as<uint32_t>(), outcap, cnt, d_segb.as<uint64_t>(), d_sege.as<uint64_t>());
                e = hipGetLastError();
                if (e == hipSuccess)
                    e = hipcub::DeviceSegmentedRadixSort::SortKeys(d_tmp.p, tmp_bytes, d_outk.as<uint64_t>(),
                                                                   d_outs.as<uint64_t>(), static_cast<int>(cnt * outcap),
                                                                   static_cast<int>(cnt), d_segb.as<uint64_t>(),
                                                                   d_sege.as<uint64_t>());
            }
            if (e == hipSuccess)
                e = launch_d4(dstride, [&](auto d4) {
                    constexpr int D = decltype(d4)::value;
                    auto go = [&](auto k, uint64_t* lists) {
                        hipLaunchKernelGGL(k, wg, dim3(256), 0, nullptr, G, lists, d_outn.as<uint32_t>(), outcap, ord, s0,
                                           cnt, alpha);
                    };
                    if (sort_here) go(bvb::vb_prune_targets<D, true>, d_outk.as<uint64_t>());
                    else go(bvb::vb_prune_targets<D, false>, d_outs.as<uint64_t>());
                });
        }
        if (e != hipSuccess) break;
        // 2. mirrored edges in batch order
        const uint64_t bcnt = end - start, m = bcnt * degree;
        const dim3 mg(static_cast<uint32_t>((m + 255) / 256));
        hipLaunchKernelGGL(bvb::vb_rev_keys, mg, dim3(256), 0, nullptr, G, ord, start, bcnt, d_rk.as<uint64_t>(), ctr);
        e = hipGetLastError();
        if (e == hipSuccess)
            e = hipcub::DeviceRadixSort::SortKeys(d_tmp.p, tmp_bytes, d_rk.as<uint64_t>(), d_rks.as<uint64_t>(),
                                                  static_cast<int>(m));
        if (e == hipSuccess) {
            hipLaunchKernelGGL(bvb::vb_rev_heads, mg, dim3(256), 0, nullptr, G, d_rks.as<uint64_t>(), d_heads.as<uint4>(),
                               d_bigjobs.as<uint4>(), ctr);
            e = hipGetLastError();
        }
        // the batch's one wait for the device
        bvb::Counters c = {};
        if (e == hipSuccess) e = hipMemcpy(&c, ctr, sizeof(c), hipMemcpyDeviceToHost);
        if (e != hipSuccess) break;
        if (c.overflow) return vfail(BS_EINVAL, "a search expanded more than " + std::to_string(outcap) + " nodes");
        if (c.heads) {
            hipLaunchKernelGGL(bvb::vb_rev_apply, dim3((c.heads + 3) / 4), dim3(256), 0, nullptr, G, d_rks.as<uint64_t>(),
                               d_heads.as<uint4>(), c.heads, ord, start, d_big.as<uint64_t>(), d_bigjobs.as<uint4>());
            e = hipGetLastError();
        }
        if (e == hipSuccess && c.big) {
            const bool here = c.longest <= sort_cap;
            if (stats) {
                stats[0] = std::max(stats[0], c.longest);
                stats[1] += here ? 0u : 1u;
            }
            if (!here) {
                if (!d_bigs.p) {
                    e = hipcub::DeviceSegmentedRadixSort::SortKeys(nullptr, bigtmp_bytes, d_big.as<uint64_t>(),
                                                                   d_bigs.as<uint64_t>(), static_cast<int>(bigcap),
                                                                   static_cast<int>(mrec), d_beg.as<uint64_t>(),
                                                                   d_end.as<uint64_t>());
                    if (e != hipSuccess) break;
                    if (!alloc(d_bigs, bigcap * 8ull) || !alloc(d_beg, mrec * 8ull) || !alloc(d_end, mrec * 8ull) ||
                        !alloc(d_bigtmp, bigtmp_bytes))
                        return vfail(BS_ENOMEM, "hipMalloc of the graph-construction buffers failed");
                }
                hipLaunchKernelGGL(bvb::vb_big_offsets, dim3((c.big + 255) / 256), dim3(256), 0, nullptr,
                                   d_bigjobs.as<uint4>(), c.big, d_beg.as<uint64_t>(), d_end.as<uint64_t>());
                e = hipGetLastError();
                if (e == hipSuccess)
                    e = hipcub::DeviceSegmentedRadixSort::SortKeys(d_bigtmp.p, bigtmp_bytes, d_big.as<uint64_t>(),
                                                                   d_bigs.as<uint64_t>(), static_cast<int>(c.big_keys),
                                                                   static_cast<int>(c.big), d_beg.as<uint64_t>(),
                                                                   d_end.as<uint64_t>());
            }
            if (e == hipSuccess)
                e = launch_d4(dstride, [&](auto d4) {
                    constexpr int D = decltype(d4)::value;
                    auto go = [&](auto k, uint64_t* lists) {
                        hipLaunchKernelGGL(k, dim3((c.big + 3) / 4), dim3(256), 0, nullptr, G, lists, d_bigjobs.as<uint4>(),
                                           c.big, alpha);
                    };
                    if (here) go(bvb::vb_prune_big<D, true>, d_big.as<uint64_t>());
                    else go(bvb::vb_prune_big<D, false>, d_bigs.as<uint64_t>());
                });
        }
        if (e != hipSuccess) break;
        if (verbose) {
            e = hipDeviceSynchronize();
            const double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            if (end == n || el - last_print >= 5.0) {
                std::fprintf(stderr, "  build_graph (device): %llu / %llu points inserted, %.1fs\n",
                             static_cast<unsigned long long>(end), static_cast<unsigned long long>(n), el);
                last_print = el;
            }
        }
        start = end;
    }
    if (e == hipSuccess) {
        e = launch_tr(degree <= 64 ? 1 : 2, [&](auto trc) {
            constexpr int T = decltype(trc)::value;
            hipLaunchKernelGGL(bvb::vb_final<T>, dim3(static_cast<uint32_t>((n + 3) / 4)), dim3(256), 0, nullptr, G,
                               d_edges.as<uint32_t>());
        });
    }
    if (e == hipSuccess) e = hipMemcpy(edges_out, d_edges.p, n * degree * 4ull, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return vfail(BS_EHIP, std::string("graph construction: ") + hipGetErrorString(e));
    return BS_OK;
}
}  // namespace

extern "C" int bs_build_vamana_device(const float* vecs, uint64_t n, uint32_t dim, uint32_t degree,
                                      uint32_t beam_width, float alpha, uint32_t seed, uint32_t* edges_out,
                                      int verbose) try {
    return build_vamana(vecs, n, dim, degree, beam_width, alpha, seed, edges_out, verbose, bvb::SORT_CAP, nullptr);
} catch (...) {
    return bs_internal_exception();
}

extern "C" int bs_debug_build_vamana(const float* vecs, uint64_t n, uint32_t dim, uint32_t degree, uint32_t beam_width,
                                     float alpha, uint32_t seed, uint32_t sort_cap, uint32_t* edges_out,
                                     uint32_t* stats) try {
    if (sort_cap < 64 || sort_cap > bvb::SORT_CAP) return vfail(BS_EINVAL, "sort_cap must be in 64..1024");
    if (!stats) return vfail(BS_EINVAL, "stats must be given");
    stats[0] = stats[1] = 0;
    return build_vamana(vecs, n, dim, degree, beam_width, alpha, seed, edges_out, 0, sort_cap, stats);
} catch (...) {
    return bs_internal_exception();
}
