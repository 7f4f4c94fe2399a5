// Device code shared by the per-curve MSM translation units (msm_g1.hip,
// msm_g2.hip): constants of the bucket phase, the oversized-bucket chunk path,
// the bucket reduction, and the launch sequence of one MSM's bucket phase,
// templated on the coordinate field. msm.hip holds the digit sort and the
// host finish.
#pragma once
#include <algorithm>
#include <type_traits>

#include "coop29.hpp"
#include "curve.hpp"
#include "field29.hpp"
#include "glv.hpp"
#include "msm.hpp"

namespace zk {

constexpr uint32_t L_MIN_LARGE = 64;  // floor of the oversized-bucket threshold
constexpr uint32_t CHUNK = 512;       // entries per chunk of an oversized bucket, or more:
constexpr uint32_t CHUNK_PARTS = 1024;   // chunks per bucket at most
// the tree reduction (k_msm_tree): threads per workgroup, nodes per workgroup
// (18 KiB of LDS; one join per lane group in its first step)
constexpr int TREE_THREADS = 256;
template <class T> inline constexpr int TREE_LOG = 7;   // G1: 64 groups of 4 lanes
template <> inline constexpr int TREE_LOG<Fq2> = 6;     // 32 groups of 8 lanes
template <class T> inline constexpr int TREE_NODES = 1 << TREE_LOG<T>;

// what the MSMs of one launch do not share (MsmJob), by blockIdx.y (the tree:
// blockIdx.z)
struct MsmArgs {
    const void* pts29[MSM_GROUP];
    const uint32_t* order[MSM_GROUP];
    const uint32_t* cls_off[MSM_GROUP];   // null: whole buckets
    int range[MSM_GROUP];
    void* buckets[MSM_GROUP];
    void* partials[MSM_GROUP];
    const void* in[MSM_GROUP];            // of a reduction launch
    void* out[MSM_GROUP];
};

struct ChunkRec { uint32_t bucket, start, len, pad; };
struct LargeRec { uint32_t bucket, first, count, pad; };

// oversized-bucket threshold floor and chunk size are shared with the sort
// (msm.hip), which builds the chunk lists

// ---------------------------------------------------------------- point forms
// Buckets and the tree's nodes are in the 29-bit form (field29.hpp), in which
// the accumulation leaves its buckets; the tree's last points go to the host in
// the standard form.
template <class T> struct Red;
template <>
struct Red<Fp> {
    using Pt = Xyzz29;
    static constexpr int WORDS = 32;  // packed words per point (xyzz29_pack)
    ZK_DEV static Pt inf() { return xyzz29_inf(); }
    ZK_DEV static Pt add(const Pt& a, const Pt& b) { return f29_xyzz_add(a, b); }
    ZK_DEV static void pack(const Pt& p, uint32_t* w) { xyzz29_pack(p, w); }
    ZK_DEV static Pt unpack(const uint32_t* w) { return xyzz29_unpack(w); }
};
template <>
struct Red<Fq2> {
    using Pt = Xyzz29q;
    static constexpr int WORDS = 64;  // packed words per point (xyzz29q_pack)
    ZK_DEV static Pt inf() { return xyzz29q_inf(); }
    ZK_DEV static Pt add(const Pt& a, const Pt& b) { return f29q_xyzz_add(a, b); }
    ZK_DEV static void pack(const Pt& p, uint32_t* w) { xyzz29q_pack(p, w); }
    ZK_DEV static Pt unpack(const uint32_t* w) { return xyzz29q_unpack(w); }
};

// points of this form in memory: WORDS words each, 16-byte aligned
template <class T>
ZK_DEV typename Red<T>::Pt red_load(const void* base, size_t i) {
    const uint4* q = reinterpret_cast<const uint4*>(base) + (size_t)(Red<T>::WORDS / 4) * i;
    uint32_t w[Red<T>::WORDS];
#pragma unroll
    for (int k = 0; k < Red<T>::WORDS / 4; k++) {
        const uint4 v = q[k];
        w[4 * k] = v.x;
        w[4 * k + 1] = v.y;
        w[4 * k + 2] = v.z;
        w[4 * k + 3] = v.w;
    }
    return Red<T>::unpack(w);
}
template <class T>
ZK_DEV void red_store(void* base, size_t i, const typename Red<T>::Pt& p) {
    uint4* o = reinterpret_cast<uint4*>(base) + (size_t)(Red<T>::WORDS / 4) * i;
    uint32_t w[Red<T>::WORDS];
    Red<T>::pack(p, w);
#pragma unroll
    for (int k = 0; k < Red<T>::WORDS / 4; k++) o[k] = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
}
// ---------------------------------------------------------------- buckets
// Bucket accumulation, G1. One thread per bucket, in the sort's accumulation
// order (longest first, so a wave's lanes carry near-equal loads and the
// launch has no long tail); buckets above lmax entries go to the chunked path.
// Arithmetic in the 29-bit-limb form (field29.hpp): points come from the
// converted copy of the bases; the buckets stay in that form for the
// reduction.
// Thread tid of an accumulation launch over nb buckets, each split into
// `split` parts of consecutive entries (bucket b's parts go to slots
// b*split + h, summed by the reduction). Returns false when the thread
// has nothing to accumulate: past the end, or a bucket above lmax entries.
// Such a bucket is summed by the chunked path before this launch
// (k_msm_chunks, k_msm_merge into slot b*split); its other parts store
// infinity here. Otherwise [st, en) are the thread's entries and slot its
// bucket slot. With cls_off (a sort with scalar classes) the parts cover the
// bucket's entries of MsmRange `range` only; the chunked path reads whole
// buckets and passes over the infinite bases there.
template <class T>
ZK_DEV bool acc_range(uint32_t tid, uint32_t nb, uint32_t split, const uint32_t* __restrict__ order,
                      const uint32_t* __restrict__ offsets, const uint32_t* __restrict__ cls_off, int range,
                      uint32_t lmax, void* __restrict__ buckets, uint32_t& st, uint32_t& en, uint32_t& slot) {
    if (tid >= nb * split) return false;
    const uint32_t ob = tid / split, h = tid - ob * split;
    const uint32_t b = order[ob];
    uint32_t s0 = offsets[b], e0 = offsets[b + 1];
    slot = b * split + h;
    if (e0 - s0 > lmax) {
        if (h != 0) red_store<T>(buckets, slot, Red<T>::inf());
        return false;
    }
    if (cls_off && range == MSM_RANGE_A) {
        s0 = cls_off[3 * (size_t)b];
        e0 = cls_off[3 * (size_t)b + 2];
    } else if (cls_off && range == MSM_RANGE_B) {
        e0 = cls_off[3 * (size_t)b + 1];
    }
    const uint32_t cnt = e0 - s0;
    st = s0 + (uint32_t)(((uint64_t)cnt * h) / split);
    en = s0 + (uint32_t)(((uint64_t)cnt * (h + 1)) / split);
    return true;
}

// endomorphism constant (Montgomery, 8 x u32) as a field element
ZK_DEV Fp beta_mont(const uint32_t* c) {
    Fp b;
#pragma unroll
    for (int k = 0; k < 8; k++) b.v[k] = c[k];
    return b;
}

// ---------------------------------------------------------------- oversized buckets
// A lane's sum over entries of the 29-bit slots, by mixed additions: G1 in
// registers, G2 with three coordinates in LDS (AccLds) as in the accumulation.
// coord: coordinate q (X, Y, ZZ, ZZZ), component c, of the sum.
template <class T> struct LaneSum;
template <>
struct LaneSum<Fp> {
    static constexpr int LDS_WORDS = 1;
    Xyzz29 a;
    ZK_DEV explicit LaneSum(uint32_t*) { a = xyzz29_inf(); }
    ZK_DEV void add(const void* pts, uint32_t ref) {
        F29 x, y;
        f29_load_point(pts, ref, x, y);
        if (f29_is_zero(x) && f29_is_zero(y)) return;   // infinity
        f29_madd(a, x, ref >> 31 ? f29_neg_lazy2(y) : y, [&](F29& px, F29& py) { f29_load_signed(pts, ref, px, py); });
    }
    ZK_DEV bool inf() const { return a.inf; }
    ZK_DEV F29 coord(int q, int) const { return q == 0 ? a.X : q == 1 ? a.Y : q == 2 ? a.ZZ : a.ZZZ; }
};
template <>
struct LaneSum<Fq2> {
    static constexpr int LDS_WORDS = AccLds<64>::LDS_WORDS;
    AccLds<64> a;
    bool empty = true;
    ZK_DEV explicit LaneSum(uint32_t* lds) : a{lds + threadIdx.x, {}} {}
    ZK_DEV void add(const void* pts, uint32_t ref) {
        F29q x, y;
        f29q_load_point(pts, ref, x, y);
        if (f29_is_zero(x.c0) && f29_is_zero(x.c1) && f29_is_zero(y.c0) && f29_is_zero(y.c1)) return;
        if (ref >> 31) y = {f29_neg_lazy2(y.c0), f29_neg_lazy2(y.c1)};
        f29q_madd(a, empty, x, y, [&](F29q& px, F29q& py) { f29q_load_signed(pts, ref, px, py); });
    }
    ZK_DEV bool inf() const { return empty; }
    ZK_DEV F29 coord(int q, int c) const {
        using L = AccLds<64>;
        const F29q v = a.ld(q == 0 ? L::X : q == 1 ? L::Y : q == 2 ? L::ZZ : L::ZZZ);
        return c ? v.c1 : v.c0;
    }
};

// sum of the n = 2^k points of sh (coordinates of point i at (i*L + lane)*9, as
// in k_msm_tree) by the block's lane groups, into point 0; one barrier per level
template <class T>
ZK_DEV void tree_sum(uint32_t* sh, uint32_t n, const Coop<T>& k) {
    constexpr uint32_t L = Coop<T>::LANES;
    const uint32_t lane = threadIdx.x % L, grp = threadIdx.x / L, G = blockDim.x / L;
    auto ld = [&](uint32_t i) {
        F29 v;
#pragma unroll
        for (int l = 0; l < 9; l++) v.l[l] = sh[(i * L + lane) * 9 + l];
        return v;
    };
#pragma unroll 1
    for (uint32_t h = n / 2; h >= 1; h /= 2) {
        __syncthreads();
#pragma unroll 1
        for (uint32_t i = grp; i < h; i += G) {
            const F29 r = coop_add<T>(k, ld(i), ld(i + h));
#pragma unroll
            for (int l = 0; l < 9; l++) sh[(i * L + lane) * 9 + l] = r.l[l];
        }
    }
    __syncthreads();
}
// point 0 of sh to point i of out, packed, by the first lane group
template <class T>
ZK_DEV void store_sum(const uint32_t* sh, void* out, size_t i) {
    constexpr uint32_t L = Coop<T>::LANES;
    if (threadIdx.x >= L) return;
    const uint32_t lane = threadIdx.x;
    F29 v;
#pragma unroll
    for (int l = 0; l < 9; l++) v.l[l] = sh[lane * 9 + l];
    uint32_t w[8];
    f29_pack(f29_reduce(v), w);   // X may be above 2^256
    uint4* dst = reinterpret_cast<uint4*>(out) + (size_t)(Red<T>::WORDS / 4) * i + 2 * ((lane & 3) * (L / 4) + (lane >> 2));
    dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
    dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
}

// The chunked path of the oversized buckets: one wave per chunk, each lane
// adding every 64th entry, then a tree over the 64 sums by lane groups; then one
// workgroup per bucket adds its chunks' sums. Chunks are short (CHUNK entries, 8
// per lane, but at most CHUNK_PARTS per bucket), since a bit-heavy witness has
// one bucket with a third of the scalars and nothing else to fill the GPU:
// 700001 points, 70 % of them bits, took 0.75 + 0.09 ms in the standard form with
// 64 entries per lane, now 0.07 + 0.04 ms.
// One-wave chunk workgroups with 9 KiB of LDS (G2 18): they must find CU slots
// while other streams' accumulations hold most of the LDS, and with uniform
// scalars they have nothing to do.
constexpr int CHUNK_THREADS = 64, MERGE_THREADS = 256;
template <class T>
__global__ void __launch_bounds__(CHUNK_THREADS) k_msm_chunks(const uint32_t* __restrict__ entries,
                                                             const uint32_t* __restrict__ counters,
                                                             const ChunkRec* __restrict__ chunks, MsmArgs args) {
    constexpr int L = Coop<T>::LANES;
    const void* __restrict__ points29 = args.pts29[blockIdx.y];
    void* __restrict__ partials = args.partials[blockIdx.y];
    __shared__ uint32_t sh[CHUNK_THREADS * L * 9 > LaneSum<T>::LDS_WORDS ? CHUNK_THREADS * L * 9 : LaneSum<T>::LDS_WORDS];
    const Coop<T> k(threadIdx.x % L);
    const uint32_t nch = counters[0];
    for (uint32_t ci = blockIdx.x; ci < nch; ci += gridDim.x) {
        const ChunkRec cr = chunks[ci];
        LaneSum<T> acc(sh);
#pragma unroll 1
        for (uint32_t e = threadIdx.x; e < cr.len; e += CHUNK_THREADS) acc.add(points29, entries[cr.start + e]);
        F29 v[L];
        const bool inf = acc.inf();
#pragma unroll
        for (int j = 0; j < L; j++) v[j] = inf ? F29{} : acc.coord(j & 3, j >> 2);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < L; j++)
#pragma unroll
            for (int l = 0; l < 9; l++) sh[(threadIdx.x * L + j) * 9 + l] = v[j].l[l];
        tree_sum<T>(sh, CHUNK_THREADS, k);
        store_sum<T>(sh, partials, ci);
        __syncthreads();
    }
}

// one workgroup per oversized bucket: sum its chunk partials
template <class T>
__global__ void __launch_bounds__(MERGE_THREADS) k_msm_merge(const uint32_t* __restrict__ counters,
                                                            const LargeRec* __restrict__ large, uint32_t split,
                                                            MsmArgs args) {
    constexpr int L = Coop<T>::LANES, G = MERGE_THREADS / L;
    const void* __restrict__ partials = args.partials[blockIdx.y];
    void* __restrict__ buckets = args.buckets[blockIdx.y];
    __shared__ uint32_t sh[G * L * 9];
    const uint32_t lane = threadIdx.x % L, grp = threadIdx.x / L;
    const Coop<T> k(lane);
    const uint4* src = reinterpret_cast<const uint4*>(partials) + 2 * ((lane & 3) * (L / 4) + (lane >> 2));
    const uint32_t nl = counters[1];
    for (uint32_t li = blockIdx.x; li < nl; li += gridDim.x) {
        const LargeRec lr = large[li];
        F29 v{};
#pragma unroll 1
        for (uint32_t j = grp; j < lr.count; j += G)
            v = coop_add<T>(k, v, f29_load_packed(src + (size_t)(Red<T>::WORDS / 4) * (lr.first + j)));
#pragma unroll
        for (int l = 0; l < 9; l++) sh[(grp * L + lane) * 9 + l] = v.l[l];
        tree_sum<T>(sh, G, k);
        store_sum<T>(sh, buckets, (size_t)lr.bucket * split);
        __syncthreads();
    }
}

// ---------------------------------------------------------------- reduction
// Arithmetic in the 29-bit form. The point additions are inlined, each loop
// body holding one or two addition sites: out-of-line calls would pass the
// operands through scratch memory on every step of these chains.
//
// Level 1 of large bucket sets: thread j owns buckets [j*L1, (j+1)*L1) of one
// window; with bucket b holding digit b+1: R_j = sum B_b, T_j = sum (b - j*L1
// + 1) B_b, so the window value is sum_j (T_j + j*L1*R_j). B_b is the sum of
// the bucket's `split` slots from the accumulation. out: [W][R, T][K/L1], the
// two channels of the tree's nodes.
template <class T>
__global__ void __launch_bounds__(128) k_msm_reduce1(MsmArgs args, uint32_t K, int W, uint32_t L1,
                                                     uint32_t split) {
    using P = Red<T>;
    const void* __restrict__ buckets = args.in[blockIdx.y];
    void* __restrict__ out = args.out[blockIdx.y];
    uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t nseg = K / L1;
    if (j >= (uint32_t)W * nseg) return;
    uint32_t w = j / nseg, jj = j - w * nseg;
    size_t base = (size_t)w * K + (size_t)jj * L1;
    typename P::Pt run = P::inf(), acc = P::inf();
#pragma unroll 1
    for (int b = (int)L1 - 1; b >= 0; b--) {
#pragma unroll 1
        for (uint32_t h = 0; h < split; h++) run = P::add(run, red_load<T>(buckets, (base + b) * split + h));
        acc = P::add(acc, run);
    }
    red_store<T>(out, (size_t)w * 2 * nseg + jj, run);
    red_store<T>(out, ((size_t)w * 2 + 1) * nseg + jj, acc);
}

// Tree over the nodes of every bucket set, in groups of lanes (coop29.hpp).
// A node covers 2^j consecutive buckets and holds points by channel: 0 its
// plain sum S, then sums that only add up, among them O_t, the sum of its
// buckets whose index has bit t set. Joining a left and a right node adds
// channel by channel, and S of the right node is the new O_j: nothing but
// independent additions, 2K of them for K buckets in a depth of log2 K (a
// running sum per segment takes as many, two dependent ones per bucket), and
// no doubling on the device: the host weighs the O_t by 2^t.
//
// The workgroup (x, y) takes the 2^q nodes x * 2^q.. of channel c = y mod C of
// set y / C (input [set][c][N]), joins them in LDS and writes one node to
// [set][c][N >> q]; channel 0 also makes the O_t of the joins' bits, `plain`
// joins first being parts of one bucket (they make none), as channels C, C +
// 1, ... of the Cout output channels. Every entry may come in `parts`
// consecutive points. O_t of the node at i lies where S of its right half was
// joined, at i + 2^t. last: to the standard form, for the host.
//
// Bound by the depth of the additions (2.3 us each for a lone wave, G2 about
// 4.5 us) up to about 2^16 buckets, by instruction issue above. Measured alone,
// all launches: G1 2^15 buckets 45 us, 2^17 100 us, 2^18 in 3 parts 243 us; G2
// 10 sets of 2^12 138 us, 2^12 in 3 parts 0.14 ms. The level-1 segments with a
// suffix scan and a tree sum over one workgroup per 1024 segments that this
// replaced took 0.43, 0.52, 0.56, 1.31 and 1.42 ms.
template <class T>
__global__ void __launch_bounds__(TREE_THREADS) k_msm_tree(MsmArgs args, uint32_t N, uint32_t C, uint32_t parts,
                                                           int plain, int q, int last, uint32_t Cout) {
    constexpr int L = Coop<T>::LANES, G = TREE_THREADS / L;
    const void* __restrict__ in = args.in[blockIdx.z];
    void* __restrict__ out = args.out[blockIdx.z];
    __shared__ uint32_t sh[TREE_NODES<T> * L * 9];
    const uint32_t lane = threadIdx.x % L, grp = threadIdx.x / L;
    const Coop<T> k(lane);
    // place of this lane's coordinate in a packed point: c0 before c1
    const uint32_t word4 = 2 * ((lane & 3) * (L / 4) + (lane >> 2));
    const uint32_t set = blockIdx.y / C, c = blockIdx.y - set * C, nodes = 1u << q;
    const uint4* src = reinterpret_cast<const uint4*>(in) + word4 +
                       (size_t)(Red<T>::WORDS / 4) * parts * ((size_t)blockIdx.y * N + ((size_t)blockIdx.x << q));
    auto ld = [&](uint32_t i) {
        F29 v;
#pragma unroll
        for (int l = 0; l < 9; l++) v.l[l] = sh[(i * L + lane) * 9 + l];
        return v;
    };
    auto st = [&](uint32_t i, const F29& v) {
#pragma unroll
        for (int l = 0; l < 9; l++) sh[(i * L + lane) * 9 + l] = v.l[l];
    };
    for (uint32_t i = grp; i < nodes; i += G) {
        F29 v = f29_load_packed(src + (size_t)(Red<T>::WORDS / 4) * parts * i);
#pragma unroll 1
        for (uint32_t h = 1; h < parts; h++)
            v = coop_add<T>(k, v, f29_load_packed(src + (size_t)(Red<T>::WORDS / 4) * (parts * i + h)));
        st(i, v);
    }
#pragma unroll 1
    for (int j = 0; j < q; j++) {
        __syncthreads();
        const int lp = q - 1 - j;   // 2^lp joins
        const uint32_t bits = c == 0 && j > plain ? (uint32_t)(j - plain) : 0u;
        const uint32_t tasks = (1u + bits) << lp;
#pragma unroll 1
        for (uint32_t t = grp; t < tasks; t += G) {
            const uint32_t b = t >> lp;   // 0: S; b >= 1: O of the join plain + b - 1
            const uint32_t l = ((t & ((1u << lp) - 1)) << (j + 1)) + (b ? 1u << (plain + b - 1) : 0u);
            st(l, coop_add<T>(k, ld(l), ld(l + (1u << j))));
        }
    }
    __syncthreads();
    // outputs: the channel itself, and for channel 0 the new O_t
    const uint32_t nout = 1u + (c == 0 && q > plain ? (uint32_t)(q - plain) : 0u);
    for (uint32_t o = grp; o < nout; o += G) {
        const F29 v = ld(o ? 1u << (plain + o - 1) : 0u);
        uint32_t w[8];
        if (last) {
            const Fp s = f29_to_std(v);
#pragma unroll
            for (int i = 0; i < 8; i++) w[i] = s.v[i];
        } else {
            f29_pack(f29_reduce(v), w);   // X may be above 2^256
        }
        uint4* dst = reinterpret_cast<uint4*>(out) + word4 +
                     (size_t)(Red<T>::WORDS / 4) *
                         (((size_t)set * Cout + (o ? C + o - 1 : c)) * (N >> q) + blockIdx.x);
        dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
        dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
    }
}

// The chunked path of the oversized buckets (lists built by the sort): their
// sums land in bucket slot b*split before the accumulation. Queued ahead of
// the accumulation so that these short launches run while the GPU has room,
// instead of waiting behind the large accumulation launches of other streams;
// a few small workgroups each (grid-stride over the lists): with uniform
// scalars the lists are empty, and a launch that needs many CU slots would
// wait behind other streams' accumulations while its own stream's
// accumulation waits behind it.
template <class T>
static void launch_pre_t(const MsmSort& sort, const MsmJob* jobs, int count, hipStream_t st, int split) {
    const bool g2 = std::is_same<T, Fq2>::value;
    const MsmGeom g = msm_geom(sort.n, sort.g.c, g2, sort.g.merged);
    MsmArgs args{};
    for (int j = 0; j < count; j++) {
        MsmScratch& scr = *jobs[j].scr;
        scr.ensure(g, sort.n_chunk_max, g2, split);
        scr.split = split;
        args.pts29[j] = jobs[j].pts29;
        args.buckets[j] = scr.buckets.p;
        args.partials[j] = scr.partials.p;
    }
    k_msm_chunks<T><<<dim3(CHUNK_PARTS, count), CHUNK_THREADS, 0, st>>>(
        sort.entries.as<uint32_t>(), sort.counters.as<uint32_t>(), sort.chunks.as<ChunkRec>(), args);
    ZK_HIP(hipGetLastError());
    k_msm_merge<T><<<dim3(16, count), MERGE_THREADS, 0, st>>>(sort.counters.as<uint32_t>(), sort.large.as<LargeRec>(),
                                                              (uint32_t)split, args);
    ZK_HIP(hipGetLastError());
}

// accumulation order of the MSMs that read MsmRange `range` of the sort
inline const uint32_t* msm_range_order(const MsmSort& sort, int range) {
    const DevBuf& o = range == MSM_RANGE_A ? sort.order_a : range == MSM_RANGE_B ? sort.order_b : sort.order;
    return o.as<uint32_t>();
}

// the bucket-accumulation kernel of curve T (msm_g1.hip / msm_g2.hip)
template <class T>
void launch_accum(const MsmSort& sort, uint32_t nb, int split, const MsmArgs& args, int count, hipStream_t st);

template <class T>
static void launch_main_t(const MsmSort& sort, const MsmJob* jobs, int count, hipStream_t st) {
    const bool g2 = std::is_same<T, Fq2>::value;
    const MsmGeom g = msm_geom(sort.n, sort.g.c, g2, sort.g.merged);
    const int split = jobs[0].scr->split;
    const uint32_t nb = (uint32_t)((size_t)g.Wr * g.K);
    MsmArgs args{};
    for (int j = 0; j < count; j++) {
        const int range = sort.classes ? jobs[j].range : (int)MSM_RANGE_ALL;
        args.pts29[j] = jobs[j].pts29;
        args.order[j] = msm_range_order(sort, range);
        args.cls_off[j] = range != MSM_RANGE_ALL ? sort.cls_off.as<uint32_t>() : nullptr;
        args.range[j] = range;
        args.buckets[j] = jobs[j].scr->buckets.p;
        if (jobs[j].scr->ev_acc0) ZK_HIP(hipEventRecord(jobs[j].scr->ev_acc0, st));
    }
    launch_accum<T>(sort, nb, split, args, count, st);
    ZK_HIP(hipGetLastError());
    for (int j = 0; j < count; j++)
        if (jobs[j].scr->ev_acc1) ZK_HIP(hipEventRecord(jobs[j].scr->ev_acc1, st));
    const MsmTree t = msm_tree(g, g2, split);
    const size_t bytes = (size_t)g.Wr * t.nout * (g2 ? 256 : 128);
    for (int j = 0; j < count; j++) {
        MsmPartials& out = *jobs[j].out;
        out.g = g;
        out.g2 = g2;
        out.bit0 = ilog2(t.l1);
        out.nout = t.nout;
        if (out.ext) ZK_REQUIRE(out.ext_bytes >= bytes, ZK_E_INTERNAL, "MSM partials exceed the caller's host buffer");
        else out.host.ensure(bytes);
        args.in[j] = jobs[j].scr->buckets.p;
    }
    if (t.l1 > 1) {
        for (int j = 0; j < count; j++) args.out[j] = jobs[j].scr->seg.p;
        k_msm_reduce1<T><<<dim3(cdiv((size_t)g.Wr * (g.K / t.l1), 128), count), 128, 0, st>>>(args, g.K, g.Wr, t.l1,
                                                                                            (uint32_t)split);
        ZK_HIP(hipGetLastError());
        for (int j = 0; j < count; j++) args.in[j] = args.out[j];
    }
    uint32_t N = t.nodes, C = t.l1 > 1 ? 2 : 1, parts = t.parts;
    int plain = t.plain;
    for (int lev = 0; lev < t.levels; lev++) {
        const int q = t.q[lev], last = lev == t.levels - 1;
        const uint32_t Cout = C + (uint32_t)std::max(0, q - plain);
        // the last launch writes pinned host memory itself: a copy would be a
        // launch of its own at the end of every MSM
        for (int j = 0; j < count; j++)
            args.out[j] = last && !jobs[j].out->ext ? jobs[j].out->host.p
                                                    : (lev & 1 ? jobs[j].scr->node1 : jobs[j].scr->node0).p;
        k_msm_tree<T><<<dim3(N >> q, (unsigned)g.Wr * C, count), TREE_THREADS, 0, st>>>(args, N, C, parts, plain, q, last,
                                                                                        Cout);
        ZK_HIP(hipGetLastError());
        for (int j = 0; j < count; j++) args.in[j] = args.out[j];
        N >>= q;
        C = Cout;
        parts = 1;
        plain = std::max(0, plain - q);
    }
    for (int j = 0; j < count; j++) {
        if (jobs[j].out->ext) ZK_HIP(hipMemcpyAsync(jobs[j].out->ext, args.in[j], bytes, hipMemcpyDeviceToHost, st));
        if (jobs[j].scr->ev_end) ZK_HIP(hipEventRecord(jobs[j].scr->ev_end, st));
    }
}


// per-curve entry points, defined in msm_g1.hip and msm_g2.hip
void msm_launch_pre_g1(const MsmSort& sort, const MsmJob* jobs, int count, hipStream_t st, int split);
void msm_launch_main_g1(const MsmSort& sort, const MsmJob* jobs, int count, hipStream_t st);
void msm_points_to29_g1(const void* d_points, size_t n, void* d_out, hipStream_t st);
void msm_points_table_g1(const void* d_points, size_t n, const MsmGeom& g, void* d_out, hipStream_t st);
void msm_launch_pre_g2(const MsmSort& sort, const MsmJob* jobs, int count, hipStream_t st, int split);
void msm_launch_main_g2(const MsmSort& sort, const MsmJob* jobs, int count, hipStream_t st);
void msm_points_to29_g2(const void* d_points, size_t n, void* d_out, hipStream_t st);
void msm_points_table_g2(const void* d_points, size_t n, const MsmGeom& g, void* d_out, hipStream_t st);

}  // namespace zk
