// Pippenger MSM kernels for G1/G2 on gfx950 (see msm.hpp for the design).
#include <algorithm>
#include <exception>
#include <mutex>
#include <type_traits>
#include <vector>

#include "msm_kernels.hpp"
#include "qap.hpp"
#include "scan.hpp"

namespace zk {

// window for an untuned size: the 2n GLV halves of n scalars favour about
// log2(n) - 3 bits (2^22 points: c = 19, 7 windows, measured 7% faster than 8)
int msm_default_c(size_t n) {
    int lg = ilog2(n ? n : 1);
    int c = lg - 3;
    if (c < 4) c = 4;
    if (c > 19) c = 19;
    return c;
}

// parts per bucket, a power of two: at most `threads` in all, about two entries each
static int msm_double_parts(size_t nb, size_t load, size_t threads) {
    int s = 1;
    while (s < MSM_SPLIT_MAX && nb * s * 2 <= threads && load >= (size_t)s * 4) s *= 2;
    return s;
}

int msm_default_split(size_t n, int c, bool g2, bool merged) {
    const MsmGeom g = msm_geom(n, c, g2, merged);
    // two rounds of waves at 6 (G1) and 3 (G2) waves per SIMD, i.e. three
    // and two rounds at the 4 and 2 the accumulation kernels hold (128 VGPRs;
    // 172 VGPRs and LDS); the autotuner picks the splits of a circuit's sizes
    const size_t target = (size_t)1024 * 64 * 2 * (g2 ? 3 : 6);
    const size_t nb = (size_t)g.Wr * g.K, load = 2 * n * (size_t)g.W / nb;
    // Few buckets: up to half a wave per SIMD for each of a proof's MSMs, while a
    // part keeps about two entries, as below; the chain of entries per thread set
    // the time. Proofs of 5000 constraints 531 -> 460 us, 8200 680 -> 510, 11000
    // 748 -> 547; where it comes to 4 parts (2^13 buckets, 2^14 constraints) the
    // same. A limit of 2^16 threads is the same, 2^17 slower (2^14 constraints
    // 656 -> 758 us, 8 proofs of 50021 5.5 -> 6.1 ms).
    const int s = msm_double_parts(nb, load, (size_t)1 << 15);
    if (s >= 4) return s;
    return (int)std::max<size_t>(1, std::min<size_t>(3, target / nb));
}

// Nothing else runs beside an MSM of its own, so its accumulation takes up to
// half a million threads (two rounds of the resident waves for G1, four for G2)
// while every part keeps about two entries: the chain of entries per thread,
// about 10 us each in a GPU that is not full, gets shorter, and more rounds of
// waves even out their lengths. Each part costs one addition in the tree.
// Against at most 3 threads per bucket (other limits in brackets): G1 1000
// points 0.52 -> 0.33 ms, 20000 0.48 -> 0.37, 100000 0.61 -> 0.51 (2^17 0.61,
// 2^20 0.57), 400000 and more unchanged; G2 1000 1.10 -> 0.57, 200003 1.88 ->
// 1.41 (2^18 1.62, 2^20 1.58). In proofs, where five MSMs share
// the GPU, the extra additions cost more than they give (8 proofs of 50021
// constraints 6.6 ms at 3 threads, 7.1 at 8, 8.4 at 16), but where buckets are few.
int msm_alone_split(size_t n, int c, bool g2) {
    const MsmGeom g = msm_geom(n, c, g2);
    const size_t nb = (size_t)g.Wr * g.K, load = 2 * n * (size_t)g.W / nb;
    const int s = msm_double_parts(nb, load, (size_t)1 << 19);
    return s >= 4 ? s : msm_default_split(n, c, g2);
}

MsmGeom msm_geom(size_t n, int c, bool g2, bool merged) {
    if (c <= 0) c = msm_default_c(n);
    ZK_REQUIRE(c >= 4 && c <= 22, ZK_E_ARG, "MSM window must be in [4, 22]");
    MsmGeom g;
    // W windows of the requested width at most, then the 128 bits shared
    // evenly: nlo windows of c - 1 bits, the others of c bits
    g.W = (GLV_BITS + c - 1) / c;
    c = (GLV_BITS + g.W - 1) / g.W;
    g.c = c;
    g.nlo = g.W * c - GLV_BITS;
    g.merged = merged;
    g.Wr = merged ? 1 : g.W;
    g.K = 1u << (c - 1);
    return g;
}

MsmTree msm_tree(const MsmGeom& g, bool g2, int split) {
    MsmTree t{};
    // Level 1 first where the additions, not their depth, take the time: a
    // group of lanes spends about 1.6 times the work of one thread on an
    // addition. G1, 7 sets of 2^18 buckets: tree alone 0.91 ms, segments of 4
    // 0.95 ms, of 8 0.60 ms. One set of 2^18 in batched proofs of 2^20
    // constraints (10.5 ms each): segments of 4 1.5 % faster than the tree
    // alone or segments of 8. Below that the tree alone: G1 2^15 buckets 45 us
    // against 0.44 ms for segments of 4 and a block scan, G2 2^10 0.14 against
    // 1.4 ms.
    const size_t nb = (size_t)g.Wr * g.K;
    t.l1 = nb >= (1u << 20) ? std::min(8u, g.K) : nb >= (1u << 18) ? std::min(4u, g.K) : 1u;
    uint32_t C = 1;
    t.parts = 1;
    if (t.l1 > 1) {
        t.nodes = g.K / t.l1;
        t.seg = 2 * nb / t.l1;
        C = 2;
    } else if ((split & (split - 1)) == 0) {
        t.plain = ilog2(split);
        t.nodes = g.K * (uint32_t)split;
    } else {
        t.parts = (uint32_t)split;
        t.nodes = g.K;
    }
    const int qmax = g2 ? TREE_LOG<Fq2> : TREE_LOG<Fp>;
    int rem = ilog2(t.nodes), plain = t.plain;
    do {   // at least one launch: it converts the points for the host
        const int q = std::min(rem, qmax);
        t.q[t.levels] = q;
        C += (uint32_t)std::max(0, q - plain);
        plain = std::max(0, plain - q);
        rem -= q;
        size_t& buf = t.levels & 1 ? t.node1 : t.node0;
        buf = std::max(buf, ((size_t)g.Wr * C) << rem);
        t.levels++;
    } while (rem > 0);
    t.nout = C;
    return t;
}

int msm_table_c(size_t n) {
    // relative costs: a mixed addition per entry 10 products, a bucket two
    // general additions of 14
    int best = 0;
    double best_cost = 0;
    for (int c = 11; c <= 22; c++) {
        const MsmGeom g = msm_geom(n, c, false, true);
        const double cost = 2.0 * (double)n * g.W * 10 + (double)g.K * 28;
        if (!best || cost < best_cost) {
            best = g.c;
            best_cost = cost;
        }
    }
    return best;
}

// ---------------------------------------------------------------- digits
// Signed digits of a half scalar, least significant window first, window w
// being c - 1 bits wide for w < nlo and c bits above (128 bits in all):
// v = window bits + carry; v > 2^(width-1) becomes v - 2^width with a carry
// into the next window (include/msm_g1.cuh:271-329 uses the same recoding
// with one width). The magnitude is below 2^127, so the top window's v stays
// at most 2^(width-1): no carry out. Every magnitude fits the 2^(c-1) buckets
// of a window. A negative half scalar flips the sign of every digit.
struct DigitIter {
    uint32_t s[4];
    uint32_t carry, c, left;
    bool flip;
    ZK_DEV void init(const uint4& a, int cc, int nlo) {
        s[0] = a.x; s[1] = a.y; s[2] = a.z; s[3] = a.w & 0x7fffffffu;
        flip = (a.w >> 31) != 0;
        carry = 0;
        c = (uint32_t)cc;
        left = (uint32_t)nlo;
    }
    // returns magnitude (0 = skip) and sign
    ZK_DEV uint32_t next(bool& neg) {
        const uint32_t wd = left ? c - 1 : c;
        left -= left ? 1u : 0u;
        const uint32_t mask = (1u << wd) - 1, half = 1u << (wd - 1);
        uint32_t v = (s[0] & mask) + carry;
#pragma unroll
        for (int k = 0; k < 3; k++) s[k] = __builtin_amdgcn_alignbit(s[k + 1], s[k], wd);
        s[3] >>= wd;
        if (v > half) {
            carry = 1;
            neg = !flip;
            return (mask + 1) - v;
        }
        carry = 0;
        neg = flip;
        return v;
    }
};

// ---------------------------------------------------------------- digit sort
// Two-pass LDS radix sort of the flat bucket ids b = w*Kw + |digit| - 1 of all
// nonzero digits (no global atomics; Kw = K, or 0 when all windows share one
// set of buckets). Buckets are grouped by b >> s.
// Pass A, per tile of scalars: the GLV split (glv.hpp) of every scalar k_i into
// two half scalars, half[i] = k1 for P_i and half[n + i] = k2 for lambda*P_i,
// each a 127-bit magnitude with its sign in bit 127, and an LDS histogram of
// their digits' groups into a count matrix [group][tile]; a device scan of the
// matrix gives every tile its run inside every group; the tile then writes
// (entry, b) pairs at run + LDS rank.
// Pass B, per group: LDS counts of its 2^s buckets give the bucket offsets,
// then the entries go to offset + LDS rank.
//
// The first block also clears what later kernels of the sort count into
// (SortZero): the matrix's last element, the load histograms, the chunk counters.
struct SortZero {
    uint32_t* end;
    uint32_t* hist;
    uint32_t nhist;
    uint32_t* counters;
};
__global__ void __launch_bounds__(1024) k_sort_tile_hist(const uint4* __restrict__ sc, size_t n, size_t tile, int c,
                                                         int nlo, int W, uint32_t Kw, int s, uint32_t G, uint32_t nt,
                                                         uint32_t* __restrict__ matrix, uint4* __restrict__ half,
                                                         SortZero z) {
    extern __shared__ uint32_t lh[];
    for (uint32_t k = threadIdx.x; k < G; k += blockDim.x) lh[k] = 0;
    if (blockIdx.x == 0) {
        for (uint32_t k = threadIdx.x; k < z.nhist; k += blockDim.x) z.hist[k] = 0;
        if (threadIdx.x < 16) z.counters[threadIdx.x] = 0;
        if (threadIdx.x == 0) *z.end = 0;
    }
    __syncthreads();
    const size_t i0 = (size_t)blockIdx.x * tile, i1 = i0 + tile < n ? i0 + tile : n;
    for (size_t i = i0 + threadIdx.x; i < i1; i += blockDim.x) {
        const uint4 a = sc[2 * i], b = sc[2 * i + 1];
        const uint64_t k[4] = {a.x | (uint64_t)a.y << 32, a.z | (uint64_t)a.w << 32, b.x | (uint64_t)b.y << 32,
                               b.z | (uint64_t)b.w << 32};
        uint64_t kh[2][2];
        glv::split(k, kh[0], kh[1]);
#pragma unroll 1
        for (int h = 0; h < 2; h++) {
            const uint64_t lo = h ? kh[1][0] : kh[0][0], hi = h ? kh[1][1] : kh[0][1];
            const uint4 v = make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
            half[h * n + i] = v;
            DigitIter it;
            it.init(v, c, nlo);
            for (int w = 0; w < W; w++) {
                bool ng;
                uint32_t mag = it.next(ng);
                if (mag) atomicAdd(&lh[((uint32_t)w * Kw + mag - 1) >> s], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < G; k += blockDim.x) matrix[(size_t)k * nt + blockIdx.x] = lh[k];
}

// entry of half h of scalar i in window w: slot i + w*sw (sw = n for window
// tables, else 0), half, sign
__global__ void __launch_bounds__(1024) k_sort_tile_scatter(const uint4* __restrict__ half, size_t n, size_t tile, int c,
                                                            int nlo, int W, uint32_t Kw, uint32_t sw, int s, uint32_t G,
                                                            uint32_t nt, const uint32_t* __restrict__ mscan,
                                                            const uint8_t* __restrict__ cls, uint2* __restrict__ pairs) {
    extern __shared__ uint32_t lds[];   // where this tile's next pair of each group goes
    for (uint32_t k = threadIdx.x; k < G; k += blockDim.x) lds[k] = mscan[(size_t)k * nt + blockIdx.x];
    __syncthreads();
    const size_t i0 = (size_t)blockIdx.x * tile, i1 = i0 + tile < n ? i0 + tile : n;
    for (size_t i = i0 + threadIdx.x; i < i1; i += blockDim.x) {
        const uint32_t ctag = cls ? (uint32_t)cls[i] << 30 : 0u;
#pragma unroll 1
        for (int h = 0; h < 2; h++) {
            DigitIter it;
            it.init(half[h * n + i], c, nlo);
            const uint32_t ref0 = (uint32_t)i | (h ? 0x40000000u : 0u);
            for (int w = 0; w < W; w++) {
                bool ng;
                uint32_t mag = it.next(ng);
                if (mag) {
                    const uint32_t b = (uint32_t)w * Kw + mag - 1;
                    pairs[atomicAdd(&lds[b >> s], 1u)] =
                        make_uint2((ref0 + (uint32_t)w * sw) | (ng ? 0x80000000u : 0u), b | ctag);
                }
            }
        }
    }
}

// Adds 1 to cnt[key] for every active lane; returns the count before it. Lanes
// that share the first lane's key, and then the next one's, take one atomic
// together where that saves many: the atomics of one address go one lane at a
// time, and a bit-heavy witness sends a third of all entries to one bucket.
ZK_DEV uint32_t lds_count(uint32_t* cnt, uint32_t key) {
    uint32_t pos = 0;
    bool todo = true;
#pragma unroll
    for (int round = 0; round < 2; round++) {
        if (!todo) continue;
        const uint32_t k0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)key);
        const uint64_t same = __ballot(key == k0);
        if (__popcll(same) < 8) break;
        if (key == k0) {
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
            uint32_t base = 0;
            if (rank == 0) base = atomicAdd(&cnt[k0], (uint32_t)__popcll(same));
            pos = (uint32_t)__builtin_amdgcn_readfirstlane((int)base) + rank;
            todo = false;
        }
    }
    return todo ? atomicAdd(&cnt[key], 1u) : pos;
}

// Entries of a group go to their final positions through an LDS stage of
// `stage_cap` words when the group fits (then the block writes its whole
// range with coalesced stores), else straight to global memory: scattered
// 4-byte stores into a range that other blocks do not touch.
constexpr uint32_t SORT_GROUP_LDS = 65536 - 256;   // dynamic LDS bytes of k_sort_group by default
// gfx950 gives one workgroup up to 160 KiB of LDS once the kernel asks for
// more than the default 64 KiB
constexpr uint32_t SORT_GROUP_LDS_MAX = 160 * 1024 - 1024;
// 16 waves per group: the LDS stage often leaves room for one workgroup per
// CU, whose waves then carry the pass's LDS atomics and loads alone
constexpr int SORT_GROUP_THREADS = 1024;
// pairs each thread has in flight: a heavy group has one workgroup, whose loads
// wait one after the other (245000 entries in one bucket 416 -> 179 us with
// lds_count and 4; uniform 2^22 points' pass 344 -> 320 us, 8 no better)
constexpr uint32_t SORT_UNROLL = 4;
//
// With scalar classes (cls_off non-null; the class is in bits 30..31 of a
// pair's bucket word) the entries go out class by class: one pass over the
// group's pairs per class, each bucket's cursor then standing where the next
// class starts, which cls_off records.
__global__ void __launch_bounds__(1024) k_sort_group(const uint2* __restrict__ pairs, const uint32_t* __restrict__ mscan,
                                                    uint32_t nt, int s, uint32_t nb, uint32_t stage_cap,
                                                    uint32_t* __restrict__ offsets, uint32_t* __restrict__ entries,
                                                    uint32_t* __restrict__ cls_off) {
    extern __shared__ uint32_t cnt[];   // 2^s counters, then the stage
    __shared__ uint32_t wsum[16];
    const uint32_t g = blockIdx.x, F = 1u << s, mask = F - 1;
    const uint32_t start = mscan[(size_t)g * nt], end = mscan[(size_t)(g + 1) * nt];
    for (uint32_t f = threadIdx.x; f < F; f += blockDim.x) cnt[f] = 0;
    __syncthreads();
    for (uint32_t e = start + threadIdx.x; e < end; e += SORT_UNROLL * blockDim.x) {
        uint32_t b[SORT_UNROLL];
#pragma unroll
        for (uint32_t j = 0; j < SORT_UNROLL; j++) b[j] = e + j * blockDim.x < end ? pairs[e + j * blockDim.x].y & mask : ~0u;
#pragma unroll
        for (uint32_t j = 0; j < SORT_UNROLL; j++)
            if (b[j] != ~0u) lds_count(cnt, b[j]);
    }
    __syncthreads();
    // exclusive scan of the counters: per-thread chunks, then the block scan
    const uint32_t q = (F + blockDim.x - 1) / blockDim.x, f0 = threadIdx.x * q;
    const uint32_t f1 = f0 + q < F ? f0 + q : F;
    uint32_t sum = 0;
    for (uint32_t f = f0; f < f1; f++) sum += cnt[f];
    uint32_t total;
    uint32_t run = start + block_exclusive_scan(sum, wsum, &total);
    for (uint32_t f = f0; f < f1; f++) {
        const uint32_t v = cnt[f];
        cnt[f] = run;
        run += v;
    }
    __syncthreads();
    for (uint32_t f = threadIdx.x; f < F; f += blockDim.x) {
        const uint32_t b = g * F + f;
        if (b < nb) offsets[b] = cnt[f];
    }
    if (g == gridDim.x - 1 && threadIdx.x == 0) offsets[nb] = end;
    __syncthreads();
    const bool staged = end - start <= stage_cap;
    uint32_t* stage = cnt + F;
    const int ncls = cls_off ? 4 : 1;
    for (int k = 0; k < ncls; k++) {
        if (k) {
            // every entry of classes < k is placed: cnt[f] is where class k starts
            __syncthreads();
            for (uint32_t f = threadIdx.x; f < F; f += blockDim.x) {
                const uint32_t b = g * F + f;
                if (b < nb) cls_off[3 * (size_t)b + (k - 1)] = cnt[f];
            }
            __syncthreads();
        }
        for (uint32_t e = start + threadIdx.x; e < end; e += SORT_UNROLL * blockDim.x) {
            uint2 p[SORT_UNROLL];
#pragma unroll
            for (uint32_t j = 0; j < SORT_UNROLL; j++)
                if (e + j * blockDim.x < end) p[j] = pairs[e + j * blockDim.x];
#pragma unroll
            for (uint32_t j = 0; j < SORT_UNROLL; j++) {
                if (e + j * blockDim.x >= end || (cls_off && (int)(p[j].y >> 30) != k)) continue;
                const uint32_t pos = lds_count(cnt, p[j].y & mask);
                if (staged) stage[pos - start] = p[j].x;
                else entries[pos] = p[j].x;
            }
        }
    }
    if (staged) {
        __syncthreads();
        for (uint32_t e = threadIdx.x; e < end - start; e += blockDim.x) entries[start + e] = stage[e];
    }
}

// accumulation-order key of bucket b: 0 = oversized (by the whole bucket),
// then descending length of the part the MSM reads (MsmRange over a sort with
// classes: the lanes of a wave get parts of nearly equal length), nkey-1 =
// empty
__device__ inline uint32_t load_key(const uint32_t* __restrict__ off, const uint32_t* __restrict__ cls_off, int range,
                                    uint32_t b, uint32_t lmax, int qs, uint32_t nkey) {
    uint32_t s0 = off[b], e0 = off[b + 1];
    if (e0 - s0 > lmax) return 0u;
    if (range == MSM_RANGE_A) {
        s0 = cls_off[3 * (size_t)b];
        e0 = cls_off[3 * (size_t)b + 2];
    } else if (range == MSM_RANGE_B) {
        e0 = cls_off[3 * (size_t)b + 1];
    }
    return (nkey - 1) - ((e0 - s0) >> qs);
}

// With classes (cls_off non-null) blockIdx.y = 0, 1, 2 orders the buckets by
// the length of their MSM_RANGE_A, MSM_RANGE_B and whole parts, each with its
// own nkey histogram (hist + y * nkey) and cursors; every order holds all nb
// buckets, so one exclusive scan over the three histograms gives order y its
// positions offset by y * nb.
__device__ inline int order_range(const uint32_t* cls_off) {
    return !cls_off ? MSM_RANGE_ALL : blockIdx.y == 0 ? MSM_RANGE_A : blockIdx.y == 1 ? MSM_RANGE_B : MSM_RANGE_ALL;
}

__global__ void __launch_bounds__(1024) k_load_hist(const uint32_t* __restrict__ off, const uint32_t* __restrict__ cls_off,
                                                    uint32_t nb, uint32_t lmax, int qs, uint32_t nkey,
                                                    uint32_t* __restrict__ hist) {
    extern __shared__ uint32_t lh[];
    const int range = order_range(cls_off);
    hist += (size_t)blockIdx.y * nkey;
    for (uint32_t k = threadIdx.x; k < nkey; k += blockDim.x) lh[k] = 0;
    __syncthreads();
    uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < nb) atomicAdd(&lh[load_key(off, cls_off, range, b, lmax, qs, nkey)], 1u);
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < nkey; k += blockDim.x)
        if (lh[k]) atomicAdd(&hist[k], lh[k]);
}

// each block reserves one range per key, then ranks its buckets inside it in LDS
__global__ void __launch_bounds__(1024) k_load_scatter(const uint32_t* __restrict__ off,
                                                       const uint32_t* __restrict__ cls_off, uint32_t nb,
                                                       uint32_t lmax, int qs, uint32_t nkey,
                                                       uint32_t* __restrict__ cursor, uint32_t* __restrict__ order_a,
                                                       uint32_t* __restrict__ order_b, uint32_t* __restrict__ order) {
    extern __shared__ uint32_t lh[];
    const int range = order_range(cls_off);
    cursor += (size_t)blockIdx.y * nkey;
    uint32_t* out = range == MSM_RANGE_A ? order_a : range == MSM_RANGE_B ? order_b : order;
    const uint32_t base = blockIdx.y * nb;   // the scan's offset of order y
    for (uint32_t k = threadIdx.x; k < nkey; k += blockDim.x) lh[k] = 0;
    __syncthreads();
    uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t key = 0, rank = 0;
    if (b < nb) {
        key = load_key(off, cls_off, range, b, lmax, qs, nkey);
        rank = atomicAdd(&lh[key], 1u);
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < nkey; k += blockDim.x)
        if (lh[k]) lh[k] = atomicAdd(&cursor[k], lh[k]);
    __syncthreads();
    if (b < nb) out[lh[key] + rank - base] = b;
}

// chunk list entries of oversized bucket b (k_msm_chunks, k_msm_merge)
__device__ inline void list_chunks(uint32_t b, const uint32_t* off, uint32_t* counters, ChunkRec* chunks, LargeRec* large) {
    const uint32_t s0 = off[b], e0 = off[b + 1];
    const uint32_t parts = min((e0 - s0 + CHUNK - 1) / CHUNK, CHUNK_PARTS);
    const uint32_t len = (e0 - s0 + parts - 1) / parts, nch = (e0 - s0 + len - 1) / len;
    const uint32_t first = atomicAdd(&counters[0], nch);
    for (uint32_t j = 0; j < nch; j++) {
        const uint32_t c0 = s0 + j * len;
        chunks[first + j] = {b, c0, min(len, e0 - c0), 0u};
    }
    const uint32_t li = atomicAdd(&counters[1], 1u);
    large[li] = {b, first, nch, 0u};
}

// Chunk lists of the oversized buckets (load key 0, first in the accumulation
// order): one thread per oversized bucket, grid-stride; hist[0] is their count.
__global__ void __launch_bounds__(256) k_chunk_list(const uint32_t* __restrict__ order, const uint32_t* __restrict__ off,
                                                    const uint32_t* __restrict__ hist, uint32_t* __restrict__ counters,
                                                    ChunkRec* __restrict__ chunks, LargeRec* __restrict__ large) {
    const uint32_t n_over = hist[0];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n_over; i += gridDim.x * blockDim.x)
        list_chunks(order[i], off, counters, chunks, large);
}

// The three kernels above for few buckets, in one workgroup per order: the
// histogram and its scan stay in LDS. The whole buckets' order (the last) also
// lists the chunks.
__global__ void __launch_bounds__(1024) k_order_small(const uint32_t* __restrict__ off, const uint32_t* __restrict__ cls_off,
                                                      uint32_t nb, uint32_t lmax, int qs, uint32_t nkey,
                                                      uint32_t* __restrict__ order_a, uint32_t* __restrict__ order_b,
                                                      uint32_t* __restrict__ order, uint32_t* __restrict__ counters,
                                                      ChunkRec* __restrict__ chunks, LargeRec* __restrict__ large) {
    extern __shared__ uint32_t lh[];
    __shared__ uint32_t wsum[16];
    const int range = order_range(cls_off);
    uint32_t* out = range == MSM_RANGE_A ? order_a : range == MSM_RANGE_B ? order_b : order;
    for (uint32_t k = threadIdx.x; k < nkey; k += blockDim.x) lh[k] = 0;
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < nb; b += blockDim.x)
        atomicAdd(&lh[load_key(off, cls_off, range, b, lmax, qs, nkey)], 1u);
    __syncthreads();
    const uint32_t per = (nkey + blockDim.x - 1) / blockDim.x, k0 = threadIdx.x * per;
    const uint32_t k1 = k0 + per < nkey ? k0 + per : nkey;
    uint32_t sum = 0, total;
    for (uint32_t k = k0; k < k1; k++) sum += lh[k];
    uint32_t run = block_exclusive_scan(sum, wsum, &total);
    for (uint32_t k = k0; k < k1; k++) {
        const uint32_t v = lh[k];
        lh[k] = run;
        run += v;
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < nb; b += blockDim.x) {
        const uint32_t key = load_key(off, cls_off, range, b, lmax, qs, nkey);
        out[atomicAdd(&lh[key], 1u)] = b;
        if (key == 0 && range == MSM_RANGE_ALL) list_chunks(b, off, counters, chunks, large);
    }
}

// bucket sets up to here are ordered by one workgroup per order (k_order_small):
// one launch of 4 us instead of four; at 2^15 its 32 rounds take longer than the
// launches (8 proofs of 50021 constraints 6.12 against 6.24 ms)
constexpr size_t ORDER_SMALL = 16384;

// sizes of one digit sort over n scalars at window c (shared by reserve and run)
struct SortShape {
    MsmGeom g;
    size_t n2, nb, tile, mlen, ne, max_chunks, max_large;
    size_t group_max;   // expected entries of the heaviest group (uniform scalars)
    uint32_t G, nt, lmax, nkey;
    int sh, qs;
};

static SortShape sort_shape(size_t n, int c, bool merged, size_t min_tile = 64) {
    ZK_REQUIRE(n < 0x40000000ull, ZK_E_ARG, "MSM size must be < 2^30");
    SortShape z;
    z.g = msm_geom(n, c, false, merged);
    // entries name the slot w*n + i of window w's table in 30 bits
    ZK_REQUIRE(!merged || (size_t)z.g.W * n < 0x40000000ull, ZK_E_ARG, "MSM over window tables needs W*n < 2^30");
    // the sort runs over the 2n half scalars of the GLV split
    z.n2 = 2 * n;
    z.nb = (size_t)z.g.Wr * z.g.K;
    // group size 2^s: at most 4096 groups (LDS histograms of pass A)
    z.sh = 7;
    while (((z.nb + (1ull << z.sh) - 1) >> z.sh) > 4096) z.sh++;
    z.G = (uint32_t)((z.nb + (1ull << z.sh) - 1) >> z.sh);
    // tiles of pass A: up to 2^19 scalars, powers of two from 64 (one wave) to
    // 2048 that make at most 256 tiles, since a tile's digits go through one
    // CU's LDS atomics one after the other (1000 scalars, 22 windows: one tile 39
    // + 40 us, 16 tiles 12 + 11); above, multiples of 2048, at most 512 tiles (two
    // workgroups per CU): longer runs per group and tile for the pair writes,
    // whose short runs wrote several times their bytes
    z.tile = min_tile;
    while (z.tile < 2048 && z.tile * 256 < n) z.tile *= 2;
    if (z.tile == 2048) z.tile *= std::max<size_t>(1, (n + 2048 * 512 - 1) / (2048 * 512));
    z.nt = (uint32_t)std::max<size_t>(1, (n + z.tile - 1) / z.tile);
    z.mlen = (size_t)z.G * z.nt + 1;
    z.ne = std::max<size_t>(1, (size_t)z.g.W * z.n2);
    // accumulation order. Oversized threshold: 8x the mean bucket load
    // (uniform scalars put about ne/nb entries in a bucket).
    z.lmax = std::max<uint32_t>(L_MIN_LARGE, 8u * (uint32_t)((z.ne + z.nb - 1) / z.nb));
    z.qs = 0;
    while ((z.lmax >> z.qs) + 2 > 4096) z.qs++;
    z.nkey = (z.lmax >> z.qs) + 2;
    // ceil(len / CHUNK) <= len / L_MIN_LARGE for the len > L_MIN_LARGE entries of
    // an oversized bucket
    z.max_chunks = z.ne / L_MIN_LARGE + 2;
    z.max_large = z.ne / L_MIN_LARGE + 2;
    // a window of width wd spreads the 2n digits of its halves over 2^(wd-1)
    // magnitudes; the lowest buckets carry the most: those of the narrower
    // windows, or of every window when they share one bucket set
    double per_b = 0;
    for (int w = 0; w < z.g.W; w++) {
        const int wd = w < z.g.nlo ? z.g.c - 1 : z.g.c;
        const double load = (double)z.n2 / (double)(1ull << (wd - 1));
        per_b = merged ? per_b + load : std::max(per_b, load);
    }
    z.group_max = (size_t)(per_b * (double)(1ull << z.sh));
    return z;
}

// every buffer of a sort with its size for shape z: f(buffer, bytes)
template <class S, class F>
static void sort_buffers(S& s, const SortShape& z, F&& f) {
    f(s.half, std::max<size_t>(1, z.n2) * 16);
    f(s.matrix, z.mlen * 4);
    f(s.mscan, z.mlen * 4 + (size_t)4 * (cdiv(z.mlen, SCAN_TILE) + 1));
    f(s.pairs, z.ne * 8);
    f(s.entries, z.ne * 4);
    f(s.offsets, (z.nb + 1) * 4);
    f(s.order, z.nb * 4);
    f(s.lkeys, (size_t)4 * (2 * z.nkey + cdiv(z.nkey, SCAN_TILE) + 1));
    f(s.chunks, z.max_chunks * sizeof(ChunkRec));
    f(s.large, z.max_large * sizeof(LargeRec));
    f(s.counters, (size_t)64);
}

// the buffers of a sort with scalar classes over nb buckets
template <class S, class F>
static void class_buffers(S& s, const SortShape& z, F&& f) {
    const size_t nb = z.nb, nkey = z.nkey;
    f(s.cls_off, nb * 12);
    f(s.order_a, nb * 4);
    f(s.order_b, nb * 4);
    f(s.okeys, (size_t)4 * (6 * (size_t)nkey + cdiv(3 * (size_t)nkey, SCAN_TILE) + 1));
}

static void sort_reserve(MsmSort& s, const SortShape& z) {
    sort_buffers(s, z, [](DevBuf& b, size_t n) { b.ensure(n); });
}

size_t MsmSort::reserve(size_t n_, int c, bool merged, bool with_classes) {
    const SortShape z = sort_shape(n_, c, merged);
    sort_reserve(*this, z);
    if (with_classes) class_buffers(*this, z, [](DevBuf& b, size_t n) { b.ensure(n); });
    return z.max_chunks;
}

size_t MsmSort::count_reserve(size_t n_, int c, GrowCount& gc, bool merged, bool with_classes) const {
    const SortShape z = sort_shape(n_, c, merged);
    sort_buffers(*this, z, [&](const DevBuf& b, size_t n) { gc.need(b, n); });
    if (with_classes) class_buffers(*this, z, [&](const DevBuf& b, size_t n) { gc.need(b, n); });
    return z.max_chunks;
}

void MsmSort::run(const void* d_scalars, size_t n_, int c, hipStream_t st, bool merged, const uint8_t* cls) {
    const SortShape z = sort_shape(n_, c, merged, min_tile);
    sort_reserve(*this, z);
    if (cls) class_buffers(*this, z, [](DevBuf& b, size_t n) { b.ensure(n); });
    n = n_;
    classes = cls != nullptr && n_ != 0;
    g = z.g;
    lmax = z.lmax;
    qs = z.qs;
    nkey = z.nkey;
    n_chunk_max = z.max_chunks;
    const size_t nb = z.nb, tile = z.tile, mlen = z.mlen;
    const uint32_t G = z.G, nt = z.nt;
    const int sh = z.sh;
    uint32_t* mat = matrix.as<uint32_t>();
    uint32_t* msc = mscan.as<uint32_t>();
    // accumulation orders: the whole buckets', and with classes also those of
    // the A and B parts, in one histogram, scan and scatter
    const uint32_t nord = classes ? 3 : 1;
    uint32_t* h = (classes ? okeys : lkeys).as<uint32_t>();
    if (n) {
        const unsigned threads = (unsigned)std::min<size_t>(1024, tile);
        const SortZero zero{mat + mlen - 1, h, nord * nkey, counters.as<uint32_t>()};
        k_sort_tile_hist<<<nt, threads, G * 4, st>>>((const uint4*)d_scalars, n, tile, g.c, g.nlo, g.W,
                                                     merged ? 0u : g.K, sh, G, nt, mat, half.as<uint4>(), zero);
        ZK_HIP(hipGetLastError());
        exclusive_scan(mat, msc, msc + mlen, mlen, st);
        k_sort_tile_scatter<<<nt, threads, G * 4, st>>>(half.as<uint4>(), n, tile, g.c, g.nlo, g.W, merged ? 0u : g.K,
                                                        merged ? (uint32_t)n : 0u, sh, G, nt, msc, cls,
                                                        pairs.as<uint2>());
        ZK_HIP(hipGetLastError());
    } else {
        fill_u32(mat, 0u, mlen, st);
        fill_u32(h, 0u, nord * nkey, st);
        fill_u32(counters.as<uint32_t>(), 0u, 16, st);
        exclusive_scan(mat, msc, msc + mlen, mlen, st);
    }
    // stage for the heaviest group uniform scalars give, plus a margin
    // (group sizes are sums of many digits, so larger ones are rare and take
    // the global path); above 64 KiB of LDS the kernel is allowed up to
    // 160 KiB, or keeps 64 KiB if the runtime refuses
    ZK_REQUIRE((4u << sh) < SORT_GROUP_LDS / 2, ZK_E_INTERNAL, "sort group counters exceed the LDS budget");
    const size_t want = z.group_max + z.group_max / 16 + 256;
    uint32_t lds_budget = SORT_GROUP_LDS;
    if (4 * ((1u << sh) + want) > SORT_GROUP_LDS) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(&k_sort_group), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)SORT_GROUP_LDS_MAX) == hipSuccess)
            lds_budget = SORT_GROUP_LDS_MAX;
        else
            (void)hipGetLastError();
    }
    const uint32_t stage_cap = (uint32_t)std::min<size_t>((lds_budget - (4u << sh)) / 4, want);
    k_sort_group<<<G, SORT_GROUP_THREADS, 4u * ((1u << sh) + stage_cap), st>>>(pairs.as<uint2>(), msc, nt, sh, (uint32_t)nb, stage_cap,
                                                                offsets.as<uint32_t>(), entries.as<uint32_t>(),
                                                                cls ? cls_off.as<uint32_t>() : nullptr);
    ZK_HIP(hipGetLastError());
    const uint32_t* off = offsets.as<uint32_t>();
    const uint32_t* co = classes ? cls_off.as<uint32_t>() : nullptr;
    if (nb <= ORDER_SMALL) {
        k_order_small<<<dim3(1, nord), 1024, nkey * 4, st>>>(off, co, (uint32_t)nb, lmax, qs, nkey,
                                                             order_a.as<uint32_t>(), order_b.as<uint32_t>(),
                                                             order.as<uint32_t>(), counters.as<uint32_t>(),
                                                             chunks.as<ChunkRec>(), large.as<LargeRec>());
        ZK_HIP(hipGetLastError());
        return;
    }
    const unsigned nblk_o = (unsigned)cdiv(nb, 1024);
    uint32_t* cur = h + nord * nkey;
    k_load_hist<<<dim3(nblk_o, nord), 1024, nkey * 4, st>>>(off, co, (uint32_t)nb, lmax, qs, nkey, h);
    ZK_HIP(hipGetLastError());
    exclusive_scan(h, cur, cur + nord * nkey, nord * nkey, st);
    k_load_scatter<<<dim3(nblk_o, nord), 1024, nkey * 4, st>>>(off, co, (uint32_t)nb, lmax, qs, nkey, cur,
                                                              order_a.as<uint32_t>(), order_b.as<uint32_t>(),
                                                              order.as<uint32_t>());
    ZK_HIP(hipGetLastError());
    // chunk lists of the oversized buckets (hist[0] of the whole buckets' order),
    // shared by every MSM over this sort
    k_chunk_list<<<64, 256, 0, st>>>(order.as<uint32_t>(), off, h + (nord - 1) * nkey, counters.as<uint32_t>(),
                                     chunks.as<ChunkRec>(), large.as<LargeRec>());
    ZK_HIP(hipGetLastError());
}

void msm_reserve_partials(MsmPartials& out, const MsmGeom& g, bool g2, int split) {
    out.host.ensure((size_t)g.Wr * msm_tree(g, g2, split).nout * (g2 ? 256 : 128));
}

void msm_points_to29(const void* d_points, size_t n, void* d_out, bool g2, hipStream_t st) {
    if (!n) return;
    ZK_REQUIRE(n < 0x40000000ull, ZK_E_ARG, "MSM size must be < 2^30");
    if (g2) msm_points_to29_g2(d_points, n, d_out, st);
    else msm_points_to29_g1(d_points, n, d_out, st);
}

void msm_points_table(const void* d_points, size_t n, int c, void* d_out, bool g2, hipStream_t st) {
    if (!n) return;
    const MsmGeom g = msm_geom(n, c, g2, true);
    ZK_REQUIRE((size_t)g.W * n < 0x40000000ull, ZK_E_ARG, "window tables need W*n < 2^30");
    msm_points_to29(d_points, n, d_out, g2, st);
    if (g2) msm_points_table_g2(d_points, n, g, d_out, st);
    else msm_points_table_g1(d_points, n, g, d_out, st);
}

void MsmScratch::enable_timing() {
    if (ev_acc0) return;
    ZK_HIP(hipEventCreate(&ev_acc0));
    ZK_HIP(hipEventCreate(&ev_acc1));
    ZK_HIP(hipEventCreate(&ev_end));
}

MsmScratch::~MsmScratch() {
    if (ev_acc0) (void)hipEventDestroy(ev_acc0);
    if (ev_acc1) (void)hipEventDestroy(ev_acc1);
    if (ev_end) (void)hipEventDestroy(ev_end);
}

static DevBuf MsmSort::* const SORT_BUFS[] = {
    &MsmSort::half, &MsmSort::matrix, &MsmSort::mscan, &MsmSort::pairs, &MsmSort::offsets, &MsmSort::entries,
    &MsmSort::order, &MsmSort::lkeys, &MsmSort::cls_off, &MsmSort::order_a, &MsmSort::order_b, &MsmSort::okeys,
    &MsmSort::chunks, &MsmSort::large, &MsmSort::counters};
static DevBuf MsmScratch::* const SCRATCH_BUFS[] = {&MsmScratch::buckets, &MsmScratch::seg, &MsmScratch::node0,
                                                          &MsmScratch::node1, &MsmScratch::partials};

size_t MsmSort::bytes() const {
    size_t b = 0;
    for (auto m : SORT_BUFS) b += (this->*m).bytes;
    return b;
}

size_t MsmScratch::bytes() const {
    size_t b = 0;
    for (auto m : SCRATCH_BUFS) b += (this->*m).bytes;
    return b;
}

// ---------------------------------------------------------------- workspaces
static std::mutex g_ws_mu;
// never destroyed: a program may free its contexts in exit handlers that run
// after the library's own
static std::vector<KeptWorkspace*>& workspaces() {
    static auto* v = new std::vector<KeptWorkspace*>;
    return *v;
}

KeptWorkspace::KeptWorkspace(int dev) : device(dev) {
    std::lock_guard<std::mutex> lk(g_ws_mu);
    workspaces().push_back(this);
}

KeptWorkspace::~KeptWorkspace() {
    std::lock_guard<std::mutex> lk(g_ws_mu);
    auto& v = workspaces();
    v.erase(std::find(v.begin(), v.end(), this));
}

void MsmWorkspace::release() {
    for (auto m : SORT_BUFS) (sort.*m).release();
    for (auto m : SCRATCH_BUFS) (scr.*m).release();
    p29.release();
}

WorkspaceUse::WorkspaceUse(KeptWorkspace& k, hipStream_t s) : w(&k), st(s) {
    if (!k.busy.exchange(true)) {
        kept = &k;
        return;
    }
    own = std::make_unique<MsmWorkspace>();
    w = own.get();
}

WorkspaceUse::~WorkspaceUse() {
    // a call that failed may have left work queued on the buffers
    const bool failed = std::uncaught_exceptions() > 0;
    if (failed) (void)hipStreamSynchronize(st);
    if (!kept) return;
    if (failed || kept->bytes() > MSM_KEEP_BYTES) kept->release();
    kept->held = kept->bytes();
    kept->busy = false;
}

void KeptWorkspace::take_back() {
    if (busy.exchange(true)) return;
    release();
    held = 0;
    busy = false;
}

void release_idle_workspaces(int device) {
    std::lock_guard<std::mutex> lk(g_ws_mu);
    for (KeptWorkspace* w : workspaces())
        if (device < 0 || w->device == device) w->take_back();
}

size_t idle_workspace_bytes(int device) {
    std::lock_guard<std::mutex> lk(g_ws_mu);
    size_t b = 0;
    for (const KeptWorkspace* w : workspaces())
        if ((device < 0 || w->device == device) && !w->busy) b += w->held;
    return b;
}

template <class S, class F>
static void scratch_buffers(S& q, const MsmGeom& g, size_t max_chunks, bool g2, int split, F&& f) {
    const size_t xb = g2 ? 256 : 128;
    const size_t nb = (size_t)g.Wr * g.K;
    f(q.buckets, nb * split * xb);
    const MsmTree t = msm_tree(g, g2, split);
    f(q.seg, t.seg * xb);
    f(q.node0, t.node0 * xb);
    f(q.node1, t.node1 * xb);
    f(q.partials, max_chunks * xb);
}

void MsmScratch::ensure(const MsmGeom& g, size_t max_chunks, bool g2, int split) {
    scratch_buffers(*this, g, max_chunks, g2, split, [](DevBuf& b, size_t n) { b.ensure(n); });
}

void MsmScratch::count_ensure(const MsmGeom& g, size_t max_chunks, bool g2, int split, GrowCount& gc) const {
    scratch_buffers(*this, g, max_chunks, g2, split, [&](const DevBuf& b, size_t n) { gc.need(b, n); });
}

static void check_jobs(const MsmSort& sort, const MsmJob* jobs, int count) {
    ZK_REQUIRE(count >= 1 && count <= MSM_GROUP, ZK_E_INTERNAL, "MSM group size");
    for (int j = 0; j < count; j++) {
        ZK_REQUIRE(sort.n == 0 || jobs[j].pts29, ZK_E_INTERNAL, "MSM launch without the 29-bit copy of its points");
        ZK_REQUIRE(jobs[j].range >= MSM_RANGE_ALL && jobs[j].range <= MSM_RANGE_B, ZK_E_INTERNAL, "unknown MSM entry range");
    }
}

void msm_launch_pre(const MsmSort& sort, bool g2, const MsmJob* jobs, int count, hipStream_t st, int split) {
    ZK_REQUIRE(split >= 1 && split <= MSM_SPLIT_MAX, ZK_E_ARG, "bucket split out of range");
    check_jobs(sort, jobs, count);
    if (g2) msm_launch_pre_g2(sort, jobs, count, st, split);
    else msm_launch_pre_g1(sort, jobs, count, st, split);
}

void msm_launch_main(const MsmSort& sort, bool g2, const MsmJob* jobs, int count, hipStream_t st) {
    check_jobs(sort, jobs, count);
    for (int j = 0; j < count; j++)
        ZK_REQUIRE(jobs[j].scr->split >= 1 && jobs[j].scr->split == jobs[0].scr->split, ZK_E_INTERNAL,
                   "MSM accumulation queued before its chunked path");
    if (g2) msm_launch_main_g2(sort, jobs, count, st);
    else msm_launch_main_g1(sort, jobs, count, st);
}

void msm_launch(const MsmSort& sort, bool g2, const MsmJob& job, hipStream_t st, int split) {
    msm_launch_pre(sort, g2, &job, 1, st, split);
    msm_launch_main(sort, g2, &job, 1, st);
}

// ---------------------------------------------------------------- fixed-scratch G1 MSM
// The whole device workspace of msm_g1_noalloc: allocated with the code
// object on every device the library runs on, held until the process ends.
static __device__ __align__(256) uint8_t scratch[MSM_NOALLOC_SCRATCH_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static std::mutex g_noalloc_mu;
static void* g_noalloc_ptr[NOALLOC_MAX_DEVICES] = {};
// host partials of the fixed-scratch MSM: at most W*(c + 2) XYZZ points of 128 B
static uint64_t g_noalloc_host[16384];

void msm_noalloc_setup(int device) {
    ZK_REQUIRE(device >= 0 && device < NOALLOC_MAX_DEVICES, ZK_E_ARG, "device index out of range");
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    if (g_noalloc_ptr[device]) return;
    void* ptr = nullptr;
    // the host-side name of a __device__ array is not its device address
    ZK_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_noalloc_ptr[device] = ptr;
}

zkh::Xyzz<zkh::Fp> msm_g1_noalloc(int device, const void* d_points, const void* d_scalars, size_t n, int window,
                                  hipStream_t st) {
    void* base = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_noalloc_mu);
        if (device >= 0 && device < NOALLOC_MAX_DEVICES) base = g_noalloc_ptr[device];
    }
    ZK_REQUIRE(base != nullptr, ZK_E_STATE, "fixed MSM scratch not set up on this device");
    SortShape z = sort_shape(n, window, false);
    const MsmGeom& g = z.g;
    // the same buffers the allocating path sizes, laid out in the array; fewer
    // threads per bucket, then fewer tiles, where that makes them fit
    MsmSort sort;
    MsmScratch scr;
    DevBuf p29;
    size_t need = 0;
    auto count = [&](const DevBuf&, size_t b) { need = ((need + 255) & ~(size_t)255) + b; };
    int split = msm_alone_split(n, g.c, false);
    for (;;) {
        need = 0;
        sort_buffers(sort, z, count);
        scratch_buffers(scr, g, z.max_chunks, false, split, count);
        count(p29, std::max<size_t>(n, 1) * PT29_BYTES);
        if (need <= MSM_NOALLOC_SCRATCH_BYTES) break;
        if (split > 1) {
            split = split > 4 ? split / 2 : split - 1;
        } else if (sort.min_tile < 2048) {
            sort.min_tile = 2048;
            z = sort_shape(n, window, false, sort.min_tile);
        } else {
            break;
        }
    }
    ZK_REQUIRE(need <= MSM_NOALLOC_SCRATCH_BYTES, ZK_E_ARG,
               "MSM of " + std::to_string(n) + " points at window " + std::to_string(g.c) + " needs " +
                   std::to_string(need) + " bytes of workspace; the fixed scratch holds " +
                   std::to_string(MSM_NOALLOC_SCRATCH_BYTES) + " (65536 points at the default window)");
    const size_t host_need = (size_t)g.Wr * msm_tree(g, false, split).nout * 128;
    ZK_REQUIRE(host_need <= sizeof g_noalloc_host, ZK_E_ARG, "MSM window too large for the fixed host partials");
    size_t used = 0;
    auto take = [&](DevBuf& b, size_t bytes) {
        used = (used + 255) & ~(size_t)255;
        b.borrow((char*)base + used, bytes);
        used += bytes;
    };
    sort_buffers(sort, z, take);
    scratch_buffers(scr, g, z.max_chunks, false, split, take);
    take(p29, std::max<size_t>(n, 1) * PT29_BYTES);
    MsmPartials part;
    part.ext = g_noalloc_host;
    part.ext_bytes = sizeof g_noalloc_host;
    if (n) msm_points_to29(d_points, n, p29.p, false, st);
    sort.run(d_scalars, n, window, st);
    msm_launch(sort, false, {p29.p, &scr, &part}, st, split);
    ZK_HIP(hipStreamSynchronize(st));
    return msm_finish_g1(part);
}

// ---------------------------------------------------------------- host finish
template <class HT>
static HT load_h(const uint64_t* p);
template <>
zkh::Fp load_h<zkh::Fp>(const uint64_t* p) { return zkh::Fp::from_raw(p); }
template <>
zkh::Fp2 load_h<zkh::Fp2>(const uint64_t* p) { return {zkh::Fp::from_raw(p), zkh::Fp::from_raw(p + 4)}; }

// The points of every set by their power of two (offset of the set's window
// plus the bit of the bucket index), then one Horner chain from the top.
template <class HT>
static zkh::Xyzz<HT> finish_t(const MsmPartials& p) {
    const MsmGeom& g = p.g;
    const size_t lw = sizeof(HT) / 8;  // u64 words per coordinate
    auto ld = [&](size_t i) {
        const uint64_t* q = p.data() + i * 4 * lw;
        return zkh::Xyzz<HT>{load_h<HT>(q), load_h<HT>(q + lw), load_h<HT>(q + 2 * lw), load_h<HT>(q + 3 * lw)};
    };
    const uint32_t first = p.bit0 ? 1 : 0;   // the constant's channel, the O_t after it
    std::vector<std::vector<size_t>> at(GLV_BITS + 1);
    int off = 0;
    for (int w = 0; w < g.Wr; w++) {
        at[off].push_back((size_t)w * p.nout + first);
        for (uint32_t t = first + 1; t < p.nout; t++)
            at[off + p.bit0 + (int)(t - first - 1)].push_back((size_t)w * p.nout + t);
        off += w < g.nlo ? g.c - 1 : g.c;   // widths of the windows
    }
    zkh::Xyzz<HT> total = zkh::Xyzz<HT>::infinity();
    for (int b = GLV_BITS; b >= 0; b--) {
        total = zkh::xyzz_dbl(total);
        for (size_t i : at[b]) total = zkh::xyzz_add(total, ld(i));
    }
    return total;
}

zkh::Xyzz<zkh::Fp> msm_finish_g1(const MsmPartials& p) { return finish_t<zkh::Fp>(p); }
zkh::Xyzz<zkh::Fp2> msm_finish_g2(const MsmPartials& p) { return finish_t<zkh::Fp2>(p); }

}  // namespace zk
