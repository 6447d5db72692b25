// Exact brute-force k nearest neighbours on the GPU (the ground truth the recall of a
// search is scored against).  The reference has no such tool (its ground truth comes
// from HDF5 files, script/unpack.py:56-81); this is the one dense contraction near the
// search path, so it runs on the matrix cores.
//
//   gt_split    every row scaled by a power of two and split into three fp16 planes (h + m + l =
//               the fp32 value) in the matrix cores' operand layout, and |b_j|^2 (fp64 sum,
//               rounded once)
//   gt_select   32 x 32 tiles of a_j = |b_j|^2 - 2 q.b_j from v_mfma_f32_32x32x16_f16, six
//               products of the planes; the 128 smallest (a_j, j) per (query, row split) kept
//               in HBM with a per-query threshold in registers and an LDS append buffer
//   gt_refine   merge the splits' lists, exact fp64 distances of the 128 candidates summed
//               in dimension order (the host bs_groundtruth's arithmetic), order by
//               (distance, id), and a certificate: every other row j has
//               a_j >= a_C (the 128th approximate value), and |a_j + |q|^2 - d_j| <= eps, so
//               when the k-th exact distance is below a_C + |q|^2 - eps no other row can
//               be among the k nearest.  Uncertified queries are reported, not guessed.
#include "bs_hip.h"
#include "bs_device.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

int bs_internal_vecs(bs_index idx, const float** vecs, uint32_t* dstride);
std::mutex& bs_internal_gt_mutex(bs_index idx);
hipError_t bs_internal_gt_workspace(bs_index idx, size_t bytes, char** ws);
void bs_internal_set_error(const std::string& msg);
int bs_internal_exception();

namespace bsg {

using bsd::EMPTY_KEY;
using bsd::orderable;
using bsw::ballot;
using bsw::lane_id;
using bsw::readlane;
using bsw::readlane64;
using bsw::wave_sync;

constexpr uint32_t C = 128;           // candidates kept per (query, split)
constexpr uint32_t BUF = 64;          // LDS append slots per query
constexpr uint32_t FLUSH = BUF - 32;  // a buffer is merged once it holds this many keys
constexpr uint32_t PUB = 64;          // splits whose published values bound a query's C-th value
constexpr uint32_t REFRESH = 16;      // tiles between two reads of the published values

constexpr uint32_t TS = 36;           // floats per lane of the values staged for an append (16-byte aligned)

// the place in a split's list of the value it publishes, of G = min(splits, PUB) that do
__host__ __device__ constexpr uint32_t pub_place(uint32_t nsplit) {
    const uint32_t G = nsplit < PUB ? nsplit : PUB;
    return (C + G - 1) / G;
}
// tiles of a split's priming pass (0: none), the same for all splits: one that publishes later holds
// the others up.  A sixteenth of the split, but 4 tiles where that is no more than half of it: a tile
// costs 3 us and its unfiltered rows, 32 keys for each of 64 queries to append and merge, 100.  At most
// 0, 2 (a quarter) and 4 (half) tiles in short splits: 20k x 128, 300 queries 0.89, 0.42 and 0.38 ms;
// 12k x 16, 500 queries 0.56, 0.38, 0.33; 500k x 128, 64 queries 1.20, 1.04, 0.97.
__host__ __device__ constexpr uint32_t prime_tiles(uint32_t nsplit, uint32_t tiles) {
    if (nsplit <= 1 || pub_place(nsplit) > 32u) return 0;
    const uint32_t longer = tiles / 16u < 64u ? tiles / 16u : 64u, shorter = tiles / 2u < 4u ? tiles / 2u : 4u;
    return longer > shorter ? longer : shorter;
}

// LDS of a gt_select wavefront of QB x 32 queries: append buffers, 32 lanes' values, key counts
constexpr uint32_t lds_wave(int qb) { return static_cast<uint32_t>(qb) * 32 * (BUF * 8 + 4) + 32 * TS * 4; }

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// The exponent of the power of two that brings a vector's largest magnitude into [2^14, 2^15),
// below fp16's 65504 (0 for an empty vector or one with an infinity or NaN; -113..100, so that
// the power and its reciprocal are normal numbers).
__device__ __forceinline__ int scale_exp(float largest) {
    const int e = static_cast<int>(__float_as_uint(largest) >> 23);  // biased exponent, 0 for 0 and subnormals
    return largest == 0.0f || e == 255 ? 0 : std::min(141 - e, 100);
}
__device__ __forceinline__ float exp2i(int e) { return __uint_as_float(static_cast<uint32_t>(e + 127) << 23); }

constexpr int NP = 3;  // fp16 planes of a value: h, m, l

// steps of 16 dimensions that a base tile's m and l planes are loaded ahead (a divisor of KC): as
// many as the registers hold beside the queries' planes.  10k queries, 200k x 256: 4 steps 8.9 ms,
// 8 (10 registers spilled) 9.4, 16 26.7; 5k, 200k x 200: 4 steps 4.7, 6 5.0; 10k, 500k x 128: 2
// steps 10.0, 4 9.5, 8 (6 spilled) 13.1; 200k x 96: 3 and 6 steps 4.3
constexpr int ahead(int KC) { return KC == 6 ? 3 : KC >= 8 ? 4 : KC; }

// x (already scaled) as fp16 planes: each keeps the next 11 significant bits, rounded to nearest.
// h leaves at most 2^-11 |x|, m at most the last of the 24 bits, 2^-23 |x|, and l holds that one.
// What falls below fp16's range is less than 2^-27 of the row's largest value (if the matrix unit
// takes fp16 subnormals as zero; else 2^-39).  A value that is infinite or NaN leaves a NaN, which
// makes every product with it a survivor.
__device__ __forceinline__ void split_value(float x, _Float16 (&p)[NP]) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
        p[i] = static_cast<_Float16>(x);
        x = x - static_cast<float>(p[i]);
    }
}

// Operand layout of v_mfma_f32_32x32x16_f16 (A and B alike): lane l holds row (column) l % 32
// and 8 of the 16 dimensions, 8 (l / 32) .. + 7.  Both operands are filled by the same rule, so
// the order of the dimensions inside the instruction does not matter.  A fragment is one
// operand register set of the wavefront, 64 x 16 bytes; the base's fragments are stored
// [tile of 32 rows][16 dimensions][plane], so a wavefront's load of one is 1 KB contiguous.
//
// Rows row0 .. row0 + m of the base, a wavefront per tile.  Memory bound (4 bytes read and 6
// written per value).  The norm is summed in fp64 (one rounding).  meta[j] = (|b_j|^2, -2 over
// the row's scale).
template <int KC>
__global__ void __launch_bounds__(256) gt_split(const float* vecs, uint64_t row0, uint64_t m, uint32_t dstride,
                                                uint4* frag, float2* meta, uint32_t* bmax_bits) {
    const uint32_t lane = lane_id(), half = lane >> 5, l32 = lane & 31u;
    const uint64_t tiles = (m + 31) / 32, step = static_cast<uint64_t>(gridDim.x) * 4;
    float mx = 0.0f;
    for (uint64_t t = static_cast<uint64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); t < tiles; t += step) {
        const uint64_t j = std::min<uint64_t>(t * 32 + l32, m - 1);  // the last tile's spare rows repeat its last one
        const float* row = vecs + (row0 + j) * dstride;
        f32x4 x[KC][2];
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int q = 0; q < 2; ++q) {  // loads of columns past the row read column 0
                const uint32_t d = 16u * kc + 8u * half + 4u * q;
                x[kc][q] = *reinterpret_cast<const f32x4*>(row + (d < dstride ? d : 0u));
            }
        double s = 0.0;
        float big = 0.0f;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (16u * kc + 8u * half + 4u * q >= dstride) x[kc][q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v = x[kc][q][i];
                    big = fabsf(v) > big || v != v ? (v != v ? __builtin_inff() : fabsf(v)) : big;
                    s += static_cast<double>(v) * static_cast<double>(v);
                }
            }
        big = fmaxf(big, bsw::xor_lane_f<32>(big));
        const float sc = exp2i(scale_exp(big));
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
            f16x8 p[NP];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                _Float16 v[NP];
                split_value(x[kc][i / 4][i % 4] * sc, v);
#pragma unroll
                for (int q = 0; q < NP; ++q) p[q][i] = v[q];
            }
            uint4* f = frag + ((t * KC + kc) * NP) * 64 + lane;
#pragma unroll
            for (int q = 0; q < NP; ++q) f[q * 64] = __builtin_bit_cast(uint4, p[q]);
        }
        s += __longlong_as_double(static_cast<long long>(
            bsw::xor_lane64<32>(static_cast<uint64_t>(__double_as_longlong(s)))));
        const float nj = static_cast<float>(s);
        if (half == 0) meta[t * 32 + l32] = make_float2(nj, -2.0f / sc);
        mx = fmaxf(mx, nj);
    }
    mx = bsw::wave_max(mx);  // mx >= 0, so the float order is the bit order
    if (lane == 0) atomicMax(bmax_bits, __float_as_uint(mx));
}

// D (32 x 32) element of accumulator register r in this lane: row (query) 8(r/4) + 4(lane/32)
// + r%4, column (base row) lane % 32 -- the 32 x 32 output layout of the f32 and f16
// instructions alike, checked by bs_debug_mfma32_f16 and bs_debug_mfma32.
__device__ __forceinline__ uint32_t acc_row(int r, uint32_t half) {
    return 8u * static_cast<uint32_t>(r / 4) + 4u * half + static_cast<uint32_t>(r % 4);
}

__device__ __forceinline__ float tau_of(uint32_t key_hi) {
    return key_hi == ~0u ? __builtin_inff() : bsd::key_dist(static_cast<uint64_t>(key_hi) << 32);
}

// the C smallest of the sorted beam and the sorted list whose keys are given in reverse (rev[r]
// of lane l = key C - 1 - (64 r + l)): the elementwise minimum is bitonic and holds exactly
// them, seven steps sort it
__device__ __forceinline__ void merge_lists(uint64_t (&beam)[2], const uint64_t (&rev)[2]) {
#pragma unroll
    for (int r = 0; r < 2; ++r) beam[r] = rev[r] < beam[r] ? rev[r] : beam[r];
    const uint64_t x = beam[0], y = beam[1];
    beam[0] = y < x ? y : x;
    beam[1] = y < x ? x : y;
#pragma unroll
    for (int i = 5; i >= 0; --i) {
        const uint32_t step = 1u << i;
        const uint64_t lower = bsd::lanes_bit_clear(step);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint64_t p = bsw::xor_lane64_rt(beam[r], step);
            beam[r] = bsw::lane_in(~(lower ^ ballot(p < beam[r]))) ? p : beam[r];
        }
    }
}

// v sorted over the 64 lanes, largest first
__device__ __forceinline__ uint64_t sort_descending(uint64_t v) {
#pragma unroll
    for (int ki = 1; ki <= 6; ++ki)
#pragma unroll
        for (int si = ki - 1; si >= 0; --si) {
            const uint64_t p = bsw::xor_lane64_rt(v, 1u << si);
            const uint64_t keep_max = ~(bsd::lanes_bit_clear(1u << si) ^ bsd::lanes_bit_clear(1u << ki));
            v = bsw::lane_in(keep_max ^ ballot(p < v)) ? p : v;
        }
    return v;
}

// A operands of a wavefront: block b, lane (l32, half): query q0 + 32 b + l32, dimensions
// 16 kc + 8 half + i, scaled by 2^-qe[b].  Each query has its own scale, as each row has, so what
// a query loses below fp16's range does not depend on its neighbours.  Bit i of nanq[b]: query
// 32 b + i has a NaN.
template <int KC, int QB>
__device__ __forceinline__ void load_queries(const float* queries, uint32_t dim, uint64_t nq, uint64_t q0,
                                             f16x8 (&a)[QB][KC][NP], int (&qe)[QB], uint32_t (&nanq)[QB]) {
    const uint32_t lane = lane_id(), half = lane >> 5, l32 = lane & 31u;
    float x[QB][KC][8];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
        const uint64_t qi = q0 + 32u * b + l32;
        const float* qv = queries + std::min<uint64_t>(qi, nq - 1) * dim;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int i = 0; i < 8; ++i) {  // all loads first (clamped), then the zeroing
                const uint32_t d = 16u * kc + 8u * half + i;
                x[b][kc][i] = qv[d < dim ? d : 0u];
            }
        float big = 0.0f;
        bool nan = false;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t d = 16u * kc + 8u * half + i;
                const float v = qi < nq && d < dim ? x[b][kc][i] : 0.0f;
                x[b][kc][i] = v;
                nan = nan || v != v;
                big = fabsf(v) > big || v != v ? (v != v ? __builtin_inff() : fabsf(v)) : big;
            }
        big = fmaxf(big, bsw::xor_lane_f<32>(big));
        const uint64_t nm = ballot(nan);
        nanq[b] = static_cast<uint32_t>(nm | (nm >> 32));
        const int e = scale_exp(big);
        const float sc = exp2i(e);
        qe[b] = -e;
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                _Float16 v[NP];
                split_value(x[b][kc][i] * sc, v);
#pragma unroll
                for (int p = 0; p < NP; ++p) a[b][kc][p][i] = v[p];
            }
    }
}

// A wavefront holds 32 QB queries as A operands (KC steps of 16 dimensions x 3 planes) and
// streams its split's base tiles as B operands, each operand register reloaded as soon as the
// products have read it.  a.b = (hl + lh + mm + hm + mh) + hh: the small products are summed first
// and the large ones on top, so the small ones' roundings are 2^-11 of the large ones', and
// the dropped ones (ml, lm, ll) are below 2^-32 |a||b|: the fp32 operands with all their bits.
// Against fp64 the rms error of q.b is 0.36-0.56 of the fp32 instructions' over mixture and
// unit-sphere data of 16..256 dimensions and 0.12-0.79 over wide-ranged data of 32 and more and
// values that differ in their last 12 bits, because the chain rounds 8 times less often; where one or
// two products are most of the sum and both round once, 1.0-1.27 (the matrix unit's rounding).
// Two planes and three products hold 22 to 24 of the 24 bits: 1.9-2.9 there and up to 1.27 on
// wide-ranged data.
// Six fp16 products of 16 dimensions take 192 matrix cycles, eight v_mfma_f32_32x32x2f32 512.
// 500k x 128, 10k queries: 17.1 -> 8.7 ms with the filtering below.
// Two query blocks per wavefront (dim <= 128) halve the base bytes per product.
//
// The matrix pipe and the vector unit work at the same time: while tile t's products run, tile
// t - 1's 16 QB values per lane are formed and compared, two after each step's products (two
// accumulator sets).  Only a tile with a survivor leaves that rhythm.
//
// Filtering: a query's candidates are the rows with a_j <= tau, tau = the least of
//   - this split's C-th value so far,
//   - any split's C-th value (tshare: published with an atomic minimum),
//   - the largest over G = min(splits, PUB) splits of each one's ceil(C / G)-th value: those
//     splits together hold at least C values that are no larger.
// Each bounds the query's C-th value over all rows from above, so no row among the C smallest
// is dropped.  The third keeps the survivors near C (1 + ln(n / C)) per query instead of that
// per split (500k rows in 6 splits: 917 -> 490 keys per query and split, 220 with the priming
// below).
template <int KC, int QB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
gt_select(const uint4* frag, const float2* meta, uint64_t row0, uint64_t m, const float* queries, uint32_t dim,
          uint64_t nq, uint32_t nsplit, uint32_t prime, uint32_t fresh, uint64_t* topc, uint32_t* tshare,
          uint32_t* pub) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const uint32_t lane = lane_id(), wave = bsw::uniform(threadIdx.x >> 6), half = lane >> 5, l32 = lane & 31u;
    constexpr uint32_t NQ = 32 * QB;
    const uint64_t w = static_cast<uint64_t>(blockIdx.x) * 4 + wave;
    const uint64_t nqb = (nq + NQ - 1) / NQ;
    if (w >= nqb * nsplit) return;
    // consecutive wavefronts take consecutive query blocks of the same row split, so the
    // wavefronts resident together stream the same base tiles and share them through L2
    const uint64_t qb = w % nqb;
    const uint32_t s = static_cast<uint32_t>(w / nqb);
    const uint32_t ntile = static_cast<uint32_t>((m + 31) / 32);
    // the splits share the tiles evenly: with equal shares rounded up the last ones can come out
    // empty, and a split that publishes nothing leaves the shared bound below (G values) without effect
    const uint32_t t0 = static_cast<uint32_t>(static_cast<uint64_t>(s) * ntile / nsplit);
    const uint32_t t1 = static_cast<uint32_t>((static_cast<uint64_t>(s) + 1) * ntile / nsplit);
    const uint32_t G = std::min(nsplit, PUB), mth = pub_place(nsplit);

    char* my = smem + static_cast<size_t>(wave) * lds_wave(QB);
    uint64_t* buf = reinterpret_cast<uint64_t*>(my);
    float* vals = reinterpret_cast<float*>(my + NQ * BUF * 8);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(my + NQ * BUF * 8 + 32 * TS * 4);  // keys in each query's buffer

    f16x8 a[QB][KC][NP];
    int qe[QB];
    uint32_t nanq[QB];
    load_queries<KC, QB>(queries, dim, nq, qb * NQ, a, qe, nanq);
    // the exponents by accumulator register, a byte each (a register each, 16 QB, does not fit: 10.3
    // ms for 10k queries, 500k x 128; in bytes 9.85; one scale for the wavefront's queries 9.5):
    // byte r % 4 of qep[b][r / 4] is that of query 32 b + acc_row(r, half)
    int qep[QB][4] = {};
#pragma unroll
    for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            qep[b][r / 4] |= (__builtin_amdgcn_ds_bpermute(static_cast<int>(acc_row(r, half) << 2), qe[b]) & 0xFF) << (8 * (r % 4));
    // tau: per accumulator register, the threshold of its query (a float compare passes a
    // superset of the list's key order; none passes for a query past nq).  Lane i's tq is query
    // i's.
    const uint64_t nan2 = (static_cast<uint64_t>(nanq[QB - 1]) << 32) | nanq[0];
    float tq = qb * NQ + lane < nq && lane < NQ && !bsw::lane_in(nan2) ? __builtin_inff() : -__builtin_inff();
    float tau[QB][16];
    // the bits of `bits` (below) whose query exists and has no NaN: a query with one has no
    // neighbours, and every row would survive for it
    uint32_t real = 0;
#pragma unroll
    for (int e = 0; e < 16 * QB; ++e) {
        const uint32_t i = acc_row(e % 16, half);
        real |= qb * NQ + 32u * (e / 16) + i < nq && !((nanq[e / 16] >> i) & 1u) ? 1u << e : 0u;
    }
    // queries whose list has been written to HBM (each lane re-reads only what it wrote)
    uint64_t written = fresh ? 0ull : ~0ull;

    auto spread_tau = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                tau[b][r] = __int_as_float(__builtin_amdgcn_ds_bpermute(
                    static_cast<int>((32u * b + acc_row(r, half)) << 2), __float_as_int(tq)));
    };
    // every query's threshold from what the splits have published
    auto refresh = [&]() __attribute__((always_inline)) {
        const uint64_t qi = std::min<uint64_t>(qb * NQ + (lane & (NQ - 1)), nq - 1);
        uint32_t v = 0;
        for (uint32_t g = 0; g < G; ++g)
            v = std::max(v, __hip_atomic_load(&pub[static_cast<uint64_t>(g) * nq + qi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        tq = fminf(tq, tau_of(std::min(v, tshare[qi])));
        return v != ~0u;
    };

    // merge every query buffer holding at least `need` keys into its top-C list; the next
    // buffer's list is requested before this one's is merged
    struct Row {
        uint64_t k0, k1;
        uint32_t sh, pb;
    };
    auto compact = [&](uint32_t need) __attribute__((always_inline)) {
        const uint32_t have = cnt[lane & (NQ - 1)];  // lane i: query i's
        uint64_t todo = ballot(lane < NQ && have >= need && qb * NQ + lane < nq);
        auto fetch = [&](uint32_t i, Row& x) __attribute__((always_inline)) {
            const uint64_t qi = qb * NQ + i;
            const uint64_t* top = topc + (qi * nsplit + s) * C;
            x.sh = tshare[qi];
            x.pb = lane < G ? pub[static_cast<uint64_t>(lane) * nq + qi] : 0u;
            x.k0 = x.k1 = EMPTY_KEY;
            if ((written >> i) & 1u) {
                x.k0 = top[lane];
                x.k1 = top[64 + lane];
            }
        };
        if (!todo) return;
        if (bsw::lane_in(todo)) cnt[lane] = 0u;
        Row cur;
        uint32_t i = static_cast<uint32_t>(__builtin_ctzll(todo));
        fetch(i, cur);
        while (todo) {
            todo &= todo - 1;
            Row nxt = {EMPTY_KEY, EMPTY_KEY, 0u, 0u};
            const uint32_t ni = todo ? static_cast<uint32_t>(__builtin_ctzll(todo)) : i;
            if (todo) fetch(ni, nxt);
            const uint32_t c = readlane(have, i);
            const uint64_t qi = qb * NQ + i;
            uint64_t* top = topc + (qi * nsplit + s) * C;
            uint64_t beam[2] = {cur.k0, cur.k1};
            // the list's second half against the new keys, largest first, is already bitonic
            const uint64_t rev[2] = {EMPTY_KEY, sort_descending(lane < c ? buf[i * BUF + lane] : EMPTY_KEY)};
            merge_lists(beam, rev);
            top[lane] = beam[0];
            top[64 + lane] = beam[1];
            written |= 1ull << i;
            const uint32_t last = static_cast<uint32_t>(readlane64(beam[1], 63) >> 32);
            const uint32_t mk = static_cast<uint32_t>(
                readlane64(mth > 64u ? beam[1] : beam[0], (mth - 1) & 63u) >> 32);
            if (lane == 0) {
                if (last != ~0u) atomicMin(&tshare[qi], last);
                if (s < G) atomicMin(&pub[static_cast<uint64_t>(s) * nq + qi], mk);  // primed values may be lower
            }
            uint32_t pb = lane == s ? std::min(mk, cur.pb) : cur.pb;
            pb = std::max(pb, bsw::xor_lane<1>(pb));
            pb = std::max(pb, bsw::xor_lane<2>(pb));
            pb = std::max(pb, bsw::partner<4>(pb));
            pb = std::max(pb, bsw::partner<8>(pb));
            const uint32_t all = std::max(std::max(readlane(pb, 0), readlane(pb, 16)),
                                          std::max(readlane(pb, 32), readlane(pb, 48)));
            const float nt = tau_of(std::min(std::min(last, cur.sh), all));
            tq = lane == i ? nt : tq;
            cur = nxt;
            i = ni;
        }
        spread_tau();
        wave_sync();
    };

    // The survivors (bit 16 b + r of a lane's `bits`: its value of block b, register r) into
    // their queries' buffers.  The values of 32 lanes at a time go to LDS, where each lane picks
    // its survivors one by one; a slot is an LDS counter's.  (Appending from the registers, a
    // branch and a ballot for each of the 32, took three times as long, and its code did not fit
    // the instruction cache.)  Returns whether a buffer has reached FLUSH.
    auto append = [&](uint32_t bits, const float (&av)[QB][16], uint32_t j) __attribute__((always_inline)) {
        bool full = false;
        uint64_t todo = ballot(bits != 0u);
        while (todo) {
            const uint32_t rank = bsw::lanes_below(todo);
            const uint64_t now = todo & ballot(rank < 32u);
            float* mine = vals + std::min(rank, 31u) * TS;
            uint32_t left = 0;
            if (bsw::lane_in(now)) {
#pragma unroll
                for (int b = 0; b < QB; ++b)
#pragma unroll
                    for (int r = 0; r < 16; r += 4)
                        *reinterpret_cast<f32x4*>(mine + 16 * b + r) = f32x4{av[b][r], av[b][r + 1], av[b][r + 2], av[b][r + 3]};
                left = bits;
            }
            wave_sync();
            while (ballot(left != 0u)) {
                if (left) {
                    const uint32_t e = static_cast<uint32_t>(__builtin_ctz(left));
                    left &= left - 1;
                    const uint32_t q = (e & 16u) * 2u + (e & 12u) * 2u + 4u * half + (e & 3u);  // 32 b + acc_row(r, half)
                    const uint32_t pos = __hip_atomic_fetch_add(&cnt[q], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                    float x = mine[e];
                    if (x != x) x = __builtin_nanf("");  // any NaN sorts last
                    buf[q * BUF + pos] = (static_cast<uint64_t>(orderable(x)) << 32) | j;  // pos < BUF: < FLUSH before the tile
                    full |= pos >= FLUSH - 1;
                }
            }
            todo &= ~now;
            wave_sync();
        }
        return ballot(full) != 0;
    };

    // B operands: the h planes of the whole next tile, the m and l planes of the next D steps
    constexpr int D = ahead(KC);
    f16x8 bh[KC], bml[D][2];
    auto frag_at = [&](uint32_t tile, int kc, int p) __attribute__((always_inline)) {
        return __builtin_bit_cast(f16x8, frag[((static_cast<uint64_t>(tile) * KC + kc) * NP + p) * 64 + lane]);
    };
    if (lane < NQ) cnt[lane] = 0u;
    wave_sync();

    // Tile t's products into accN (the next tile's operands requested as these are read), with
    // the previous tile's values av formed from accO on the way; returns the lane's survivors
    float av[QB][16];
    auto step = [&](uint32_t tile, uint32_t next, f32x16 (&accN)[QB], const f32x16 (&accO)[QB], float2 mo) __attribute__((always_inline)) {
        uint32_t bits = 0;
        // keeps the bytes packed: taken apart before the loop they are the 16 QB registers again
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) asm volatile("" : "+v"(qep[b][g]));
        constexpr int SMALL = 5 * QB, ALL = KC * (SMALL + QB);  // matrix instructions
        // the values screened beside instructions [m0, m1) of the tile's ALL
        auto screen = [&](int m0, int m1) __attribute__((always_inline)) {
#pragma unroll
            for (int e = 16 * QB * m0 / ALL; e < 16 * QB * m1 / ALL; ++e) {
                const int b = e / 16, r = e % 16;
                // a_j = |b_j|^2 - 2 acc / (row scale query scale): exact factors, one rounding
                const int e8 = static_cast<int>(static_cast<uint32_t>(qep[b][r / 4]) << (24 - 8 * (r % 4))) >> 24;
                av[b][r] = __builtin_amdgcn_ldexpf(accO[b][r] * mo.y, e8) + mo.x;
                bits |= !(av[b][r] > tau[b][r]) ? 1u << e : 0u;  // a NaN survives
            }
        };
#define BSG_MFMA(kc, pa, y, from)                                                                    \
    _Pragma("unroll") for (int b = 0; b < QB; ++b) accN[b] =                                          \
        __builtin_amdgcn_mfma_f32_32x32x16_f16(a[b][kc][pa], y, from, 0, 0, 0);
        const f32x16 zero = {};
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
            const f16x8 m = bml[kc % D][0], l = bml[kc % D][1];
            if (kc == 0) {
                BSG_MFMA(kc, 0, l, zero)
            } else {
                BSG_MFMA(kc, 0, l, accN[b])
            }
            BSG_MFMA(kc, 2, bh[kc], accN[b])
            BSG_MFMA(kc, 1, m, accN[b])
            BSG_MFMA(kc, 0, m, accN[b])
            BSG_MFMA(kc, 1, bh[kc], accN[b])
            const bool wraps = kc + D >= KC;
            bml[kc % D][0] = frag_at(wraps ? next : tile, (kc + D) % KC, 1);
            bml[kc % D][1] = frag_at(wraps ? next : tile, (kc + D) % KC, 2);
            screen(kc * SMALL, (kc + 1) * SMALL);
            // keep the reloads and the screening among the products: a matrix instruction, then
            // vector ones in its shadow
#pragma unroll
            for (int i = 0; i < SMALL; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
            BSG_MFMA(kc, 0, bh[kc], accN[b])
            bh[kc] = frag_at(next, kc, 0);
            screen(KC * SMALL + kc * QB, KC * SMALL + (kc + 1) * QB);
#pragma unroll
            for (int i = 0; i < QB; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#undef BSG_MFMA
        return bits;
    };
    // the survivors of `tile` (values av) appended, full buffers merged: every buffer holds <
    // FLUSH keys before the next 32 rows arrive
    auto keep = [&](uint32_t bits, uint32_t tile) __attribute__((always_inline)) {
        const uint32_t at = tile * 32u + l32;
        bits = at < m ? bits & real : 0u;  // the last tile may be partial
        if (ballot(bits != 0u) && append(bits, av, static_cast<uint32_t>(row0) + at)) compact(FLUSH);
    };
    // Priming.  A pass over the split's first `prime` tiles keeps only each lane's least value per
    // query (in tau): the mth smallest of a query's 32 lane minima is no less than the mth
    // smallest value of those rows, so it can be published as this split's mth value before any
    // list exists, and the lists then start at a threshold that admits about one row in 50
    // instead of every row.
    auto publish_minima = [&]() __attribute__((always_inline)) {
        float* st = reinterpret_cast<float*>(buf);  // no keys yet: NQ queries x TS floats
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) st[(32u * b + acc_row(r, half)) * TS + l32] = tau[b][r];
        wave_sync();
        float x[32];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(st + (lane & (NQ - 1)) * TS + 4 * i);
#pragma unroll
            for (int k = 0; k < 4; ++k) x[4 * i + k] = v[k];
        }
        wave_sync();
        // ascending bitonic network over the lane's 32 values
#pragma unroll
        for (int ki = 1; ki <= 5; ++ki)
#pragma unroll
            for (int si = ki - 1; si >= 0; --si)
#pragma unroll
                for (int i = 0; i < 32; ++i)
                    if (!(i & (1 << si))) {
                        const int o = i | (1 << si);
                        const float lo = fminf(x[i], x[o]), hi = fmaxf(x[i], x[o]);
                        x[i] = (i & (1 << ki)) ? hi : lo;
                        x[o] = (i & (1 << ki)) ? lo : hi;
                    }
        float v = x[31];
#pragma unroll
        for (int i = 0; i < 31; ++i) v = mth == static_cast<uint32_t>(i + 1) ? x[i] : v;
        if (s < G && lane < NQ && qb * NQ + lane < nq && v < __builtin_inff())
            __hip_atomic_store(&pub[static_cast<uint64_t>(s) * nq + qb * NQ + lane], static_cast<uint32_t>(orderable(v)),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the other splits reach this point at about the same time: read until all have
        // published, at most 32 times (a read is 8 us for 64 splits; a split that is not resident yet
        // never will).  Measured: one read and 20 us with every split resident.
        for (int i = 0; i < 32; ++i)
            if (ballot(!refresh() && tq != -__builtin_inff()) == 0) break;
        spread_tau();
    };
    if (t0 < t1) {
#pragma unroll
        for (int kc = 0; kc < KC; ++kc) {
            bh[kc] = frag_at(t0, kc, 0);
            if (kc < D) {
                bml[kc][0] = frag_at(t0, kc, 1);
                bml[kc][1] = frag_at(t0, kc, 2);
            }
        }
        refresh();
        spread_tau();
        if (prime) {
#pragma unroll
            for (int b = 0; b < QB; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) tau[b][r] = __builtin_inff();
        }
        // step u takes the products of tile_of(u) -- the primed tiles, then all of them, then the
        // last once more -- and the values of the one before
        const uint32_t total = prime + (t1 - t0), lastt = t1 - 1;
        auto tile_of = [&](uint32_t u) __attribute__((always_inline)) {
            return std::min(u < prime ? t0 + u : t0 + (u - prime), lastt);
        };
        auto done = [&](uint32_t bits, uint32_t u) __attribute__((always_inline)) {  // step u's values are in av
            if (u < prime) {
#pragma unroll
                for (int b = 0; b < QB; ++b)
#pragma unroll
                    for (int r = 0; r < 16; ++r) tau[b][r] = fminf(tau[b][r], av[b][r]);
                if (u + 1 == prime) publish_minima();
            } else {
                keep(bits, tile_of(u));
            }
        };
        // the pass before the first screens zeros and its result is dropped
        f32x16 acc0[QB], acc1[QB];
#pragma unroll
        for (int b = 0; b < QB; ++b) acc0[b] = acc1[b] = f32x16{};
        float2 m0 = meta[t0 * 32u + l32], m1;
        step(t0, tile_of(1), acc0, acc1, m0);
        for (uint32_t u = 1;; u += 2) {
            m1 = meta[tile_of(u) * 32u + l32];
            uint32_t bits = step(tile_of(u), tile_of(u + 1), acc1, acc0, m0);
            done(bits, u - 1);
            if (u >= total) break;
            m0 = meta[tile_of(u + 1) * 32u + l32];
            bits = step(tile_of(u + 1), tile_of(u + 2), acc0, acc1, m1);
            done(bits, u);
            if (u + 1 >= total) break;
            if (u % REFRESH == 1 && u > prime) {  // u is odd
                refresh();
                spread_tau();
            }
        }
    }
    compact(1);
    // a list with no key at all is still written
    for (uint32_t i = 0; i < NQ; ++i) {
        const uint64_t qi = qb * NQ + i;
        if (!((written >> i) & 1u) && qi < nq) {
            topc[(qi * nsplit + s) * C + lane] = EMPTY_KEY;
            topc[(qi * nsplit + s) * C + 64 + lane] = EMPTY_KEY;
        }
    }
}

// One workgroup of NW wavefronts per query: the split lists merged (a wavefront takes every
// NW-th, the NW results meet in LDS), the 128 candidates re-scored exactly in fp64, ordered,
// certified.  The candidates' rows pass through LDS: loaded coalesced (16 lanes per 64
// dimensions of a row), read back by the lane that sums the row's distance in dimension order.
// Bound by the gather of 128 rows per query: 10k queries x 128 dims 1.16 -> 0.27 ms (13 lists
// before, 6 after) against a wavefront per query that merged by ranks and whose lanes read
// their rows a word at a time.
constexpr uint32_t RF_TS = 64 + 4;  // floats per staged row: 16 lanes of a b128 phase hit 16 distinct 4-bank groups

template <int NW>
__global__ void __launch_bounds__(64 * NW) gt_refine(const float* vecs, uint32_t dstride, const float* queries,
                                                     uint32_t dim, uint32_t nsplit, const uint64_t* topc, uint32_t k,
                                                     const uint32_t* bmax_bits,
                                                     int32_t* out, uint8_t* unc, unsigned long long* n_unc) {
    static_assert(NW >= 4, "four wavefronts score the candidates");
    __shared__ __attribute__((aligned(16))) uint64_t keys[NW][C];
    __shared__ __attribute__((aligned(16))) float rows[4][32 * RF_TS];
    __shared__ float q[256];
    __shared__ double dist[C];
    __shared__ uint32_t ids[C], rank2[C];
    const uint32_t t = threadIdx.x, lane = lane_id(), wave = bsw::uniform(t >> 6);
    const uint64_t qi = blockIdx.x;
    const float* qv = queries + qi * dim;
    for (uint32_t i = t; i < dim; i += 64 * NW) q[i] = qv[i];

    const uint64_t* lists = topc + qi * nsplit * C;
    uint64_t beam[2] = {EMPTY_KEY, EMPTY_KEY};
    for (uint32_t s = wave; s < nsplit; s += NW) {
        const uint64_t rev[2] = {lists[static_cast<uint64_t>(s) * C + C - 1 - lane], lists[static_cast<uint64_t>(s) * C + 63 - lane]};
        merge_lists(beam, rev);
    }
    // pairs of results, halving: the upper wavefront leaves its list in reverse
#pragma unroll 1
    for (uint32_t h = NW / 2; h >= 1; h >>= 1) {
        if (wave >= h && wave < 2 * h) {
            keys[wave][C - 1 - lane] = beam[0];
            keys[wave][63 - lane] = beam[1];
        }
        __syncthreads();
        if (wave < h) {
            const uint64_t rev[2] = {keys[wave + h][lane], keys[wave + h][64 + lane]};
            merge_lists(beam, rev);
        }
    }
    if (wave == 0) {
        keys[0][lane] = beam[0];
        keys[0][64 + lane] = beam[1];
        ids[lane] = beam[0] == EMPTY_KEY ? 0xFFFFFFFFu : static_cast<uint32_t>(beam[0]);
        ids[64 + lane] = beam[1] == EMPTY_KEY ? 0xFFFFFFFFu : static_cast<uint32_t>(beam[1]);
    }
    if (t < C) rank2[t] = 0u;
    __syncthreads();
    const uint64_t kc = keys[0][C - 1];  // the C-th approximate key

    // exact distances, dimension order, fp64 (bs_groundtruth's l2d): wavefront w < 4 takes
    // candidates 32 w .. 32 w + 31
    if (wave < 4) {
        float* tile = rows[wave];
        const uint32_t lr = lane >> 4, lc = (lane & 15u) * 4;
        double acc = 0.0;
        for (uint32_t d0 = 0; d0 < dim; d0 += 64) {
            f32x4 v[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) {
                const uint32_t id = ids[32 * wave + 4 * i + lr];
                const float* row = vecs + static_cast<uint64_t>(id == 0xFFFFFFFFu ? 0u : id) * dstride;
                v[i] = *reinterpret_cast<const f32x4*>(row + (d0 + lc < dstride ? d0 + lc : 0u));
            }
            wave_sync();  // the previous tile's reads are done before it is overwritten
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) *reinterpret_cast<f32x4*>(tile + (4 * i + lr) * RF_TS + lc) = v[i];
            wave_sync();
            const float* mine = tile + (lane & 31u) * RF_TS;
            const uint32_t cols = dim - d0 < 64 ? dim - d0 : 64;
            for (uint32_t i = 0; i < cols; ++i) {
                const double diff = __dsub_rn(static_cast<double>(q[d0 + i]), static_cast<double>(mine[i]));
                acc = __dadd_rn(acc, __dmul_rn(diff, diff));
            }
        }
        if (lane < 32) {
            // no neighbour: an empty slot, or a row whose distance is a NaN (the select keeps every
            // row with a NaN value, which may stand for an infinity); a NaN has no rank
            const uint32_t c = 32 * wave + lane;
            const bool none = ids[c] == 0xFFFFFFFFu || acc != acc;
            dist[c] = none ? __builtin_inf() : acc;
            if (none) ids[c] = 0xFFFFFFFFu;
        }
    }
    __syncthreads();
    // rank of each candidate in (distance, id) order: thread t counts candidate t % C against
    // half of the others
    if (t < 2 * C) {
        const uint32_t c = t & (C - 1), e0 = (t / C) * (C / 2);
        const double d = dist[c];
        const uint32_t id = ids[c];
        uint32_t rank = 0;
        for (uint32_t e = e0; e < e0 + C / 2; ++e) rank += (dist[e] < d || (dist[e] == d && ids[e] < id)) ? 1u : 0u;
        if (rank) atomicAdd(&rank2[c], rank);
    }
    __syncthreads();
    if (wave != 0) return;
    // valid candidates take ranks 0..nvalid-1; the slots from nvalid to k get -1
    int32_t* o = out + qi * k;
    const uint32_t id[2] = {ids[lane], ids[64 + lane]}, rank[2] = {rank2[lane], rank2[64 + lane]};
    const double dd[2] = {dist[lane], dist[64 + lane]};
    const uint32_t nvalid = static_cast<uint32_t>(__builtin_popcountll(ballot(id[0] != 0xFFFFFFFFu)) +
                                                  __builtin_popcountll(ballot(id[1] != 0xFFFFFFFFu)));
    for (uint32_t e = nvalid + lane; e < k; e += 64) o[e] = -1;
#pragma unroll
    for (int r = 0; r < 2; ++r)
        if (id[r] != 0xFFFFFFFFu && rank[r] < k) o[rank[r]] = static_cast<int32_t>(id[r]);

    // certificate
    bool ok = true;
    if (kc != EMPTY_KEY && k <= C) {
        double dk = __builtin_inf();
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint64_t m = ballot(id[r] != 0xFFFFFFFFu && rank[r] == k - 1);
            if (m) dk = __longlong_as_double(static_cast<long long>(
                           readlane64(static_cast<uint64_t>(__double_as_longlong(dd[r])), __builtin_ctzll(m))));
        }
        double qn2 = 0.0;
        for (uint32_t i = 0; i < dim; ++i) qn2 += static_cast<double>(q[i]) * static_cast<double>(q[i]);
        const double ac = static_cast<double>(bsd::key_dist(kc));
        const double bm = __builtin_sqrt(static_cast<double>(__uint_as_float(*bmax_bits)));
        const double qb = __builtin_sqrt(qn2) + bm;
        // q.b's error, in 2^-24 |q||b|: dim roundings of the sum of the large products (dim; twice
        // that if the matrix unit truncates), 5 dim roundings of partial sums of the small ones,
        // each 2^-9 of it at most (0.02 dim), the dropped products (below 0.01), what lies below
        // fp16's range in the row and in the query (2^-27 sqrt(dim) each: below sqrt(dim) / 4
        // together).  a_j doubles it; |b_j|^2 and a_j are rounded once each.  (|q| + |b|)^2 >=
        // 4 |q||b|, so 2 (dim + 3) 2^-24 (|q| + |b|)^2 grants 8 dim + 24 of 4.1 dim + sqrt(dim) / 2
        // + 2, and 6 |b|^2 of 2.  A vector whose largest value is below 2^-86 has the largest
        // scale, 2^100: it loses 2^-113 per value.  2^-140: results below fp32's normal range.
        const double eps = 2.0 * (dim + 3) * 0x1p-24 * qb * qb +
                           2.0 * 0x1p-113 * __builtin_sqrt(static_cast<double>(dim)) * qb + 0x1p-140;
        ok = dk < ac + qn2 - eps;
    }
    if (lane == 0) {
        if (unc) unc[qi] = ok ? 0 : 1;
        if (!ok) atomicAdd(n_unc, 1ull);
    }
}

// The dot products as gt_select forms them: 32 queries against every row (out: 32 x 32 tiles),
// a wavefront per tile.  For the check of their rounding.
template <int KC>
__global__ void __launch_bounds__(64) dbg_products(const uint4* frag, const float2* meta, const float* queries,
                                                   uint32_t dim, float* out) {
    const uint32_t lane = lane_id(), half = lane >> 5, l32 = lane & 31u, t = blockIdx.x;
    f16x8 a[1][KC][NP];
    int qe[1];
    uint32_t nanq[1];
    load_queries<KC, 1>(queries, dim, 32, 0, a, qe, nanq);
    auto b = [&](int kc, int p) __attribute__((always_inline)) {
        return __builtin_bit_cast(f16x8, frag[((static_cast<uint64_t>(t) * KC + kc) * NP + p) * 64 + lane]);
    };
    f32x16 acc = {};
    auto mul = [&](int kc, int pa, int pb) __attribute__((always_inline)) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[0][kc][pa], b(kc, pb), acc, 0, 0, 0);
    };
    for (int kc = 0; kc < KC; ++kc) {
        mul(kc, 0, 2);
        mul(kc, 2, 0);
        mul(kc, 1, 1);
        mul(kc, 0, 1);
        mul(kc, 1, 0);
    }
    for (int kc = 0; kc < KC; ++kc) mul(kc, 0, 0);
    const float binv = -0.5f * meta[t * 32u + l32].y;
#pragma unroll
    for (int r = 0; r < 16; ++r) out[(static_cast<uint64_t>(acc_row(r, half)) * gridDim.x + t) * 32 + l32] =
        __builtin_amdgcn_ldexpf(acc[r] * binv, __builtin_amdgcn_ds_bpermute(static_cast<int>(acc_row(r, half) << 2), qe[0]));
}

// the same products from the fp32 instruction (lane half h: dimensions KC 8 h ..), one chain
template <int KC>
__global__ void __launch_bounds__(64) dbg_products_f32(const float* vecs, uint32_t dstride, const float* queries,
                                                       uint32_t dim, float* out) {
    const uint32_t lane = lane_id(), half = lane >> 5, l32 = lane & 31u, t = blockIdx.x;
    f32x16 acc = {};
    for (uint32_t i = 0; i < KC * 8; ++i) {
        const uint32_t d = half * KC * 8 + i;
        const float x = d < dim ? queries[l32 * dim + d] : 0.0f;
        const float y = d < dim ? vecs[(static_cast<uint64_t>(t) * 32 + l32) * dstride + d] : 0.0f;
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x, y, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) out[(static_cast<uint64_t>(acc_row(r, half)) * gridDim.x + t) * 32 + l32] = acc[r];
}

// v_mfma_f32_32x32x2f32 layout check: A 32x2, B 2x32 given row-major; D 32x32 row-major
__global__ void __launch_bounds__(64) dbg_mfma32(const float* A, const float* B, float* D) {
    const uint32_t lane = lane_id(), half = lane >> 5, l32 = lane & 31u;
    f32x16 acc = {};
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(A[l32 * 2 + half], B[half * 32 + l32], acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) D[acc_row(r, half) * 32 + l32] = acc[r];
}

// the same for v_mfma_f32_32x32x16_f16 with the operand rule of gt_split and load_queries: A 32x16,
// B 16x32
__global__ void __launch_bounds__(64) dbg_mfma32_f16(const float* A, const float* B, float* D) {
    const uint32_t lane = lane_id(), half = lane >> 5, l32 = lane & 31u;
    f16x8 a, b;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
        a[i] = static_cast<_Float16>(A[l32 * 16 + 8 * half + i]);
        b[i] = static_cast<_Float16>(B[(8 * half + i) * 32 + l32]);
    }
    f32x16 acc = {};
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 16; ++r) D[acc_row(r, half) * 32 + l32] = acc[r];
}

}  // namespace bsg

namespace {
int gfail(int code, const std::string& msg) {
    bs_internal_set_error(msg);
    return code;
}
#define GTRY(call)                                                                                    \
    do {                                                                                              \
        hipError_t e_ = (call);                                                                       \
        if (e_ != hipSuccess) return gfail(BS_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

// one workgroup of the select: KC steps of 16 dimensions, QB query blocks of 32 per wavefront
template <int KC, int QB>
hipError_t launch_select(dim3 g, hipStream_t s, const uint4* frag, const float2* meta, uint64_t row0, uint64_t m,
                         const float* q, uint32_t dim, uint64_t nq, uint32_t nsplit, uint32_t prime,
                         uint64_t* topc, uint32_t* tshare, uint32_t* pub) {
    constexpr int lds = 4 * bsg::lds_wave(QB);
    auto k = bsg::gt_select<KC, QB>;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, g, dim3(256), lds, s, frag, meta, row0, m, q, dim, nq, nsplit, prime,
                       row0 == 0 ? 1u : 0u, topc, tshare, pub);
    return hipGetLastError();
}

// steps of 16 dimensions of the instance that takes rows of dim, and f(steps, query blocks) for it
uint32_t steps_of(uint32_t dim) { return dim <= 32 ? 2 : dim <= 64 ? 4 : dim <= 96 ? 6 : dim <= 128 ? 8 : dim <= 192 ? 12 : 16; }
template <typename F>
hipError_t with_steps(uint32_t KC, F&& f) {
    std::integral_constant<int, 1> q1;
    std::integral_constant<int, 2> q2;
    switch (KC) {
    case 2: return f(std::integral_constant<int, 2>{}, q2);
    case 4: return f(std::integral_constant<int, 4>{}, q2);
    case 6: return f(std::integral_constant<int, 6>{}, q2);
    case 8: return f(std::integral_constant<int, 8>{}, q2);
    case 12: return f(std::integral_constant<int, 12>{}, q1);
    default: return f(std::integral_constant<int, 16>{}, q1);
    }
}

constexpr uint64_t REFINE_QUERIES = 1ull << 21;

// Row splits per query block: nqb * nsplit wavefronts run 4 per CU (a SIMD holds one), so the
// count is the one that fills whole rounds of them best, few rounds and few splits first (a
// split costs its query another list of 128 to fill, publish and merge).  At least 8 tiles
// per split.  A round costs 0.15 of the fill: 200k x 128, 10k queries take 4.9 ms in one round of 6
// splits, filled to 0.92, and 7.2 in two of 13, filled to 0.996 (what 0.05 would take); 33k queries 17.8
// in two rounds of 3 and 21.7 in one of 1, filled to 0.50 (0.4).  Between 640 and 20k queries the
// three weights differ nowhere else.
uint64_t pick_splits(uint64_t nqb, uint64_t tiles, uint64_t slots) {
    const uint64_t most = std::max<uint64_t>(1, std::min<uint64_t>({1024, tiles / 8, 3 * slots / nqb}));
    uint64_t best = 1;
    double score = -1e9;
    for (uint64_t s = 1; s <= most; ++s) {
        const uint64_t w = nqb * s, rounds = (w + slots - 1) / slots;
        const double fill = static_cast<double>(w) / static_cast<double>(rounds * slots) - 0.15 * static_cast<double>(rounds);
        if (fill > score + 1e-9) {
            score = fill;
            best = s;
        }
    }
    return best;
}

// How a call is cut up, and its one work buffer: planes, norms, lists, published values, counters.
struct Plan {
    uint32_t KC;   // 16-dimension steps
    uint64_t nqb;  // query blocks: 64 queries per wavefront while their operands fit beside a tile's, else 32
    uint64_t tiles, chunk, nsplit;  // tiles of the base, held as planes at a time; row splits
    uint32_t split_tiles, prime;    // tiles of the smallest split (the others have one more at most), primed ones
    uint64_t tile_bytes, o_bn, o_top, o_share, o_pub, o_cnt, need;
};
Plan make_plan(uint64_t n, uint64_t nq, uint32_t dim, uint32_t cus, uint64_t plane_bytes) {
    auto al = [](uint64_t v) { return (v + 255) & ~255ull; };
    Plan p;
    p.KC = steps_of(dim);
    const uint32_t NQ = p.KC <= 8 ? 64 : 32;
    p.nqb = (nq + NQ - 1) / NQ;
    p.tile_bytes = static_cast<uint64_t>(p.KC) * bsg::NP * 1024;
    p.tiles = (n + 31) / 32;
    p.chunk = std::max<uint64_t>(1, std::min<uint64_t>(p.tiles, plane_bytes / p.tile_bytes));
    p.nsplit = pick_splits(p.nqb, p.chunk, 4ull * cus);
    p.split_tiles = static_cast<uint32_t>(p.chunk / p.nsplit);
    p.prime = bsg::prime_tiles(static_cast<uint32_t>(p.nsplit), p.split_tiles);
    p.o_bn = al(p.chunk * p.tile_bytes);
    p.o_top = p.o_bn + al(p.chunk * 32 * 8);
    p.o_share = p.o_top + al(nq * p.nsplit * bsg::C * 8);
    p.o_pub = p.o_share + nq * 4;  // tshare and pub start as all ones together
    p.o_cnt = al(p.o_pub + std::min<uint64_t>(p.nsplit, bsg::PUB) * nq * 4);
    p.need = p.o_cnt + 256;
    return p;
}
constexpr uint64_t PLANE_BYTES = 1ull << 30;  // of planes at a time, where there is room; the lists carry over
constexpr uint64_t KEEP_BYTES = 5ull << 28;   // the largest work buffer that an index keeps

uint32_t device_cus() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        return 256;
    return static_cast<uint32_t>(cus);
}

// ws_limit: the largest work buffer that may be allocated
int groundtruth(bs_index idx, const float* d_queries, uint64_t nq, uint32_t k, int32_t* d_out, uint8_t* d_uncertified,
                hipStream_t s, uint64_t* n_uncertified, uint64_t ws_limit) {
    const float* vecs = nullptr;
    uint32_t dstride = 0;
    int rc = bs_internal_vecs(idx, &vecs, &dstride);
    if (rc) return rc;
    uint64_t n = 0;
    uint32_t dim = 0;
    rc = bs_index_info(idx, &n, &dim, nullptr, nullptr, nullptr);
    if (rc) return rc;
    if (k == 0 || k > bsg::C) return gfail(BS_EINVAL, "k must be in 1..128");
    if (dim > 256) return gfail(BS_EINVAL, "the device ground truth supports dim <= 256");
    if (nq == 0) return BS_OK;
    if (!d_queries || !d_out) return gfail(BS_EINVAL, "queries and output must be given");
    const uint32_t cus = device_cus();
    // The work buffer is the index's, kept for its next call, where it is free and not over KEEP_BYTES;
    // else this call's own.  (Memory given back is wiped by the driver at some 40 GB/s: one query on
    // 500k x 128 took 0.75 ms, but 11.0 when repeated with 450 MB allocated and freed each time.)
    // Where it does not fit, planes of half as many rows at a time, down to 8 tiles (500k x 128, 10k
    // queries: 9.7 ms with the 450 MB it takes, 9.6 with 200, 10.7 with 100, 51 with 40).
    std::unique_lock<std::mutex> lock(bs_internal_gt_mutex(idx), std::try_to_lock);
    Plan p = make_plan(n, nq, dim, cus, PLANE_BYTES);
    char* ws = nullptr;
    auto keep = [&]() { return lock.owns_lock() && p.need <= KEEP_BYTES; };
    while (p.need > ws_limit || (keep() ? bs_internal_gt_workspace(idx, p.need, &ws)
                                        : hipMalloc(reinterpret_cast<void**>(&ws), p.need)) != hipSuccess) {
        (void)hipGetLastError();
        if (p.chunk <= 8) return gfail(BS_ENOMEM, "hipMalloc of the ground-truth work buffers failed");
        p = make_plan(n, nq, dim, cus, p.chunk / 2 * p.tile_bytes);
    }
    uint4* frag = reinterpret_cast<uint4*>(ws);
    float2* meta = reinterpret_cast<float2*>(ws + p.o_bn);
    uint64_t* topc = reinterpret_cast<uint64_t*>(ws + p.o_top);
    uint32_t* tshare = reinterpret_cast<uint32_t*>(ws + p.o_share);
    uint32_t* pub = reinterpret_cast<uint32_t*>(ws + p.o_pub);
    unsigned long long* nunc = reinterpret_cast<unsigned long long*>(ws + p.o_cnt);
    uint32_t* bmax = reinterpret_cast<uint32_t*>(ws + p.o_cnt + 8);
    hipError_t e = hipMemsetAsync(nunc, 0, 16, s);
    if (e == hipSuccess) e = hipMemsetAsync(tshare, 0xFF, p.o_cnt - p.o_share, s);  // no bound published yet
    const dim3 g(static_cast<uint32_t>((p.nqb * p.nsplit + 3) / 4));
    for (uint64_t c0 = 0; e == hipSuccess && c0 < p.tiles; c0 += p.chunk) {
        const uint64_t row0 = c0 * 32, m = std::min(p.chunk * 32, n - row0), mt = (m + 31) / 32;
        const dim3 sg(static_cast<uint32_t>(std::min<uint64_t>((mt + 3) / 4, 8ull * cus)));
        auto go = [&](auto kc, auto qb) {
            constexpr int K = decltype(kc)::value;
            hipLaunchKernelGGL(bsg::gt_split<K>, sg, dim3(256), 0, s, vecs, row0, m, dstride, frag, meta, bmax);
            const hipError_t le = hipGetLastError();
            if (le != hipSuccess) return le;
            return launch_select<K, decltype(qb)::value>(g, s, frag, meta, row0, m, d_queries, dim, nq,
                                                         static_cast<uint32_t>(p.nsplit),
                                                         row0 == 0 ? p.prime : 0u, topc, tshare, pub);
        };
        e = with_steps(p.KC, go);
    }
    // a wavefront merges a list in ~0.3 us: with many splits (few queries) 16 share them.  At most
    // 2^21 queries per launch: a grid of 2^32 work-items is cut short without an error.
    for (uint64_t q0 = 0; e == hipSuccess && q0 < nq; q0 += REFINE_QUERIES) {
        const dim3 rg(static_cast<uint32_t>(std::min<uint64_t>(REFINE_QUERIES, nq - q0)));
        auto go = [&](auto kernel, uint32_t threads) {
            hipLaunchKernelGGL(kernel, rg, dim3(threads), 0, s, vecs, dstride, d_queries + q0 * dim, dim,
                               static_cast<uint32_t>(p.nsplit), topc + q0 * p.nsplit * bsg::C, k, bmax, d_out + q0 * k,
                               d_uncertified ? d_uncertified + q0 : nullptr, nunc);
        };
        if (p.nsplit > 32) go(bsg::gt_refine<16>, 1024);
        else go(bsg::gt_refine<4>, 256);
        e = hipGetLastError();
    }
    unsigned long long nu = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&nu, nunc, 8, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // nothing may still write to the buffer
    if (!keep()) (void)hipFree(ws);
    if (e != hipSuccess) return gfail(BS_EHIP, std::string("ground truth: ") + hipGetErrorString(e));
    if (n_uncertified) *n_uncertified = nu;
    return BS_OK;
}

// the same on host buffers
int groundtruth_host(bs_index idx, const float* queries, uint64_t nq, uint32_t k, int32_t* out, uint8_t* uncertified,
                     uint64_t* n_uncertified, uint64_t ws_limit) {
    if (nq == 0) {
        if (n_uncertified) *n_uncertified = 0;
        return BS_OK;
    }
    uint32_t dim = 0;
    int rc = bs_index_info(idx, nullptr, &dim, nullptr, nullptr, nullptr);
    if (rc) return rc;
    if (!queries || !out) return gfail(BS_EINVAL, "queries and output must be given");
    float* dq = nullptr;
    int32_t* dout = nullptr;
    uint8_t* dunc = nullptr;
    auto release = [&]() {
        if (dq) (void)hipFree(dq);
        if (dout) (void)hipFree(dout);
        if (dunc) (void)hipFree(dunc);
    };
    if (hipMalloc(&dq, nq * dim * 4) != hipSuccess || hipMalloc(&dout, nq * k * 4) != hipSuccess ||
        hipMalloc(&dunc, nq) != hipSuccess) {
        release();
        return gfail(BS_ENOMEM, "hipMalloc of the ground-truth buffers failed");
    }
    if (hipMemcpy(dq, queries, nq * dim * 4, hipMemcpyHostToDevice) != hipSuccess) {
        release();
        return gfail(BS_EHIP, "query upload failed");
    }
    rc = groundtruth(idx, dq, nq, k, dout, dunc, nullptr, n_uncertified, ws_limit);
    if (rc == BS_OK) {
        hipError_t e = hipMemcpy(out, dout, nq * k * 4, hipMemcpyDeviceToHost);
        if (e == hipSuccess && uncertified) e = hipMemcpy(uncertified, dunc, nq, hipMemcpyDeviceToHost);
        if (e != hipSuccess) rc = gfail(BS_EHIP, std::string("result download failed: ") + hipGetErrorString(e));
    }
    release();
    return rc;
}
}  // namespace

extern "C" int bs_index_groundtruth_device(bs_index idx, const float* d_queries, uint64_t nq, uint32_t k,
                                           int32_t* d_out, uint8_t* d_uncertified, void* stream,
                                           uint64_t* n_uncertified) try {
    return groundtruth(idx, d_queries, nq, k, d_out, d_uncertified, static_cast<hipStream_t>(stream), n_uncertified, ~0ull);
} catch (...) {
    return bs_internal_exception();
}

extern "C" int bs_index_groundtruth(bs_index idx, const float* queries, uint64_t nq, uint32_t k, int32_t* out,
                                    uint8_t* uncertified, uint64_t* n_uncertified) try {
    return groundtruth_host(idx, queries, nq, k, out, uncertified, n_uncertified, ~0ull);
} catch (...) {
    return bs_internal_exception();
}

extern "C" int bs_debug_gt_plan(uint64_t n, uint64_t nq, uint32_t dim, uint32_t out[4]) try {
    if (!out) return gfail(BS_EINVAL, "null argument");
    if (n == 0 || n > 0x7FFFFFFFull || nq == 0 || dim == 0 || dim > 256) return gfail(BS_EINVAL, "n, nq or dim out of range");
    const Plan p = make_plan(n, nq, dim, device_cus(), PLANE_BYTES);
    out[0] = static_cast<uint32_t>(p.nsplit);
    out[1] = p.split_tiles;
    out[2] = p.prime;
    out[3] = p.KC <= 8 ? 2 : 1;
    return BS_OK;
} catch (...) {
    return bs_internal_exception();
}

extern "C" int bs_debug_groundtruth(bs_index idx, const float* queries, uint64_t nq, uint32_t k, uint64_t ws_limit,
                                    int32_t* out, uint8_t* uncertified) try {
    return groundtruth_host(idx, queries, nq, k, out, uncertified, nullptr, ws_limit);
} catch (...) {
    return bs_internal_exception();
}

extern "C" int bs_debug_gt_products(const float* rows, uint32_t n, const float* queries, uint32_t dim, int fp32,
                                    float* out) try {
    if (!rows || !queries || !out) return gfail(BS_EINVAL, "null argument");
    if (n == 0 || n % 32 != 0 || n > (1u << 20)) return gfail(BS_EINVAL, "n must be a multiple of 32 up to 2^20");
    if (dim == 0 || dim > 256) return gfail(BS_EINVAL, "dim must be in 1..256");
    const uint32_t dstride = (dim + 3) & ~3u, KC = steps_of(dim);
    std::vector<float> padded(static_cast<size_t>(n) * dstride, 0.0f);
    for (uint32_t j = 0; j < n; ++j)
        std::memcpy(&padded[static_cast<size_t>(j) * dstride], rows + static_cast<size_t>(j) * dim, dim * sizeof(float));
    const size_t b_rows = padded.size() * 4, b_q = 32ull * dim * 4, b_out = 32ull * n * 4, b_meta = n * 8ull,
                 b_frag = static_cast<size_t>(n / 32) * KC * bsg::NP * 1024;
    char* ws = nullptr;
    auto al = [](size_t v) { return (v + 255) & ~static_cast<size_t>(255); };
    if (hipMalloc(reinterpret_cast<void**>(&ws), al(b_rows) + al(b_q) + al(b_out) + al(b_meta) + al(b_frag) + 4) != hipSuccess)
        return gfail(BS_ENOMEM, "hipMalloc failed");
    float* dr = reinterpret_cast<float*>(ws);
    float* dq = reinterpret_cast<float*>(ws + al(b_rows));
    float* dout = reinterpret_cast<float*>(ws + al(b_rows) + al(b_q));
    float2* meta = reinterpret_cast<float2*>(ws + al(b_rows) + al(b_q) + al(b_out));
    uint4* frag = reinterpret_cast<uint4*>(ws + al(b_rows) + al(b_q) + al(b_out) + al(b_meta));
    uint32_t* bmax = reinterpret_cast<uint32_t*>(ws + al(b_rows) + al(b_q) + al(b_out) + al(b_meta) + al(b_frag));
    hipError_t e = hipMemcpy(dr, padded.data(), b_rows, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dq, queries, b_q, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(bmax, 0, 4);
    if (e == hipSuccess)
        e = with_steps(KC, [&](auto kc, auto) {
            constexpr int K = decltype(kc)::value;
            if (fp32) {
                hipLaunchKernelGGL(bsg::dbg_products_f32<K>, dim3(n / 32), dim3(64), 0, nullptr, dr, dstride, dq, dim, dout);
            } else {
                hipLaunchKernelGGL(bsg::gt_split<K>, dim3((n / 32 + 3) / 4), dim3(256), 0, nullptr, dr, uint64_t{0}, uint64_t{n},
                                   dstride, frag, meta, bmax);
                hipLaunchKernelGGL(bsg::dbg_products<K>, dim3(n / 32), dim3(64), 0, nullptr, frag, meta, dq, dim, dout);
            }
            return hipGetLastError();
        });
    if (e == hipSuccess) e = hipMemcpy(out, dout, b_out, hipMemcpyDeviceToHost);
    (void)hipFree(ws);
    if (e != hipSuccess) return gfail(BS_EHIP, std::string("products check: ") + hipGetErrorString(e));
    return BS_OK;
} catch (...) {
    return bs_internal_exception();
}

namespace {
// one 32 x 32 product, K values per row of A and column of B
int mfma_check(void (*kernel)(const float*, const float*, float*), uint32_t K, const float* A, const float* B, float* D) {
    float *dA = nullptr, *dB = nullptr, *dD = nullptr;
    auto release = [&]() {
        if (dA) (void)hipFree(dA);
        if (dB) (void)hipFree(dB);
        if (dD) (void)hipFree(dD);
    };
    const size_t bytes = 32ull * K * 4;
    if (hipMalloc(&dA, bytes) != hipSuccess || hipMalloc(&dB, bytes) != hipSuccess || hipMalloc(&dD, 1024 * 4) != hipSuccess) {
        release();
        return gfail(BS_ENOMEM, "hipMalloc failed");
    }
    hipError_t e = hipMemcpy(dA, A, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dB, B, bytes, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(kernel, dim3(1), dim3(64), 0, nullptr, dA, dB, dD);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(D, dD, 1024 * 4, hipMemcpyDeviceToHost);
    release();
    if (e != hipSuccess) return gfail(BS_EHIP, std::string("mfma check: ") + hipGetErrorString(e));
    return BS_OK;
}
}  // namespace

extern "C" int bs_debug_mfma32(const float* A, const float* B, float* D) try {
    return mfma_check(bsg::dbg_mfma32, 2, A, B, D);
} catch (...) {
    return bs_internal_exception();
}

extern "C" int bs_debug_mfma32_f16(const float* A, const float* B, float* D) try {
    if (!A || !B || !D) return gfail(BS_EINVAL, "null argument");
    return mfma_check(bsg::dbg_mfma32_f16, 16, A, B, D);
} catch (...) {
    return bs_internal_exception();
}
