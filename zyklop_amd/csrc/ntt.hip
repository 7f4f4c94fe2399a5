// Fr NTT kernels (design in ntt.hpp): a pass transforms units of R = 2^q points
// by a group of lanes of one wave, multiplies by the inter-pass twiddle and
// writes back; the last pass writes the digit-reversed (natural) order.
#include <vector>

#include "coop29.hpp"
#include "field.hpp"
#include "field29.hpp"
#include "host_field.hpp"
#include "ntt.hpp"

namespace zk {

constexpr int NTT_THREADS = 256;
constexpr int NTT_MAX_BATCH = 4;

struct NttPtrs {
    void* in[NTT_MAX_BATCH];
    void* out[NTT_MAX_BATCH];
};

struct NttDigits {
    int np;
    int lr[NTT_MAX_PASSES];
};

// ---- elements: 9 x 29-bit limbs in registers, 8 canonical words in memory ----
// A product by a prescaled table value keeps the standard form (field29.hpp).
ZK_DEV F29 ld29(const void* base, size_t i) {
    const uint4* p = reinterpret_cast<const uint4*>(base) + 2 * i;
    const uint4 a = p[0], b = p[1];
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    return f29_unpack(w);
}
// x normalized and below 2r
ZK_DEV void st29(void* base, size_t i, const F29& x) {
    uint32_t w[8];
    f29_pack(fr29_canon(x), w);
    uint4* p = reinterpret_cast<uint4*>(base) + 2 * i;
    p[0] = make_uint4(w[0], w[1], w[2], w[3]);
    p[1] = make_uint4(w[4], w[5], w[6], w[7]);
}
// x normalized and below 5r, not made canonical: between the passes of one
// transform, whose loads take any value that fits 8 words
ZK_DEV void st29_lazy(void* base, size_t i, const F29& x) {
    uint32_t w[8];
    f29_pack(x, w);
    uint4* p = reinterpret_cast<uint4*>(base) + 2 * i;
    p[0] = make_uint4(w[0], w[1], w[2], w[3]);
    p[1] = make_uint4(w[4], w[5], w[6], w[7]);
}
// limbs below 2^32, value below 2^261 -> normalized, below r + 2^240
ZK_DEV F29 settle29(const F29& x) { return fr29_reduce(f29_norm(x)); }

// root i of the DFTs inside a unit, w_256^i in limbs, 12 words apart
constexpr int ROOTS = 256;
static_assert(NTT_THREADS == ROOTS, "k_ntt_quad: a root a thread");
constexpr int ROOT_WORDS = 12;
ZK_DEV F29 ld_root(const void* roots, uint32_t i) {
    const uint4* p = reinterpret_cast<const uint4*>(roots) + ROOT_WORDS / 4 * i;
    const uint4 a = p[0], b = p[1];
    return F29{{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w, reinterpret_cast<const uint32_t*>(p + 2)[0]}};
}
// The same in a workgroup's LDS, limb by limb: [9][ROOTS]. For k_ntt_quad, where
// ten gathers of scattered roots a lane kept the address unit busy beside the
// twiddles and points: 2^22 points 506 -> 488 us, three arrays of 2^20 378 -> 374.
// k_ntt_lane reads them from the cache: fewer roots a lane, and the copy comes
// first in a launch that waits for nothing else (three arrays of 2^18 125 us
// from LDS, 124 from the cache).
ZK_DEV void st_root_lds(uint32_t* sh, uint32_t i, const F29& r) {
#pragma unroll
    for (int l = 0; l < 9; l++) sh[l * ROOTS + i] = r.l[l];
}
ZK_DEV F29 ld_root_lds(const uint32_t* sh, uint32_t i) {
    F29 r;
#pragma unroll
    for (int l = 0; l < 9; l++) r.l[l] = sh[l * ROOTS + i];
    return r;
}

// what a pass reads and writes: unit u of 2^q points. Passes 0..np-2, in place
// over blocks of M = R*S elements: u is the column c of block beta, points
// beta*M + b*S + c. The last pass: points of row r (unrev of u), r*R + b, to
// out[u + k*O], O = n/R.
struct NttShape {
    NttDigits dg;
    int logS;     // of a pass that is not the last
    int last;
    size_t n;
    const void* roots;   // w_256^i, i < 256 (ld_root)
    const void* tw;      // w_M^(c k), [k][c], passes but the last
    const void* pre;     // first pass: multiplies input i
    const void* post;    // last pass: multiplies output i
};
struct NttUnit {
    size_t in, in_step, out, out_step, col;
};
template <int Q>
ZK_DEV NttUnit ntt_unit(const NttShape& z, size_t u) {
    if (!z.last) {
        const size_t c = u & (((size_t)1 << z.logS) - 1), base = ((u >> z.logS) << (z.logS + Q)) + c;
        return {base, (size_t)1 << z.logS, base, (size_t)1 << z.logS, c};
    }
    size_t r = u, row = 0;
    for (int d = 0; d < z.dg.np - 1; d++) {
        const size_t digit = r & (((size_t)1 << z.dg.lr[d]) - 1);
        r >>= z.dg.lr[d];
        row = (row << z.dg.lr[d]) | digit;
    }
    return {row << Q, 1, u, z.n >> Q, 0};
}
// output k of a unit, x with limbs below 2.5 * 2^30 and value below 20r: scaled,
// then stored. Apart, so that the scaling loads of all outputs come before any
// store, which they could not pass.
ZK_DEV F29 ntt_scale(const NttShape& z, const NttUnit& t, uint32_t k, const F29& x) {
    if (!z.last) return fr29_mul(x, ld29(z.tw, ((size_t)k << z.logS) + t.col));
    if (z.post) return fr29_mul(x, ld29(z.post, t.out + k * t.out_step));
    return settle29(x);
}
ZK_DEV void ntt_store(const NttShape& z, const NttUnit& t, void* out, uint32_t k, const F29& x) {
    if (!z.last) st29_lazy(out, t.out + k * t.out_step, x);
    else st29(out, t.out + k * t.out_step, x);
}

// ---- two points per lane
// A unit's 2^q points on 2^(q-1) lanes, radix-2 DIT stages in registers; before
// stage s the lanes swap one point with lane ^ 2^(s-2), so that every lane holds
// both points of its butterfly: position bit s-1 is then the slot, bits below
// are lane bits 0..s-2. About 20 % more instructions per point than four points
// per lane (below), but half the chain per launch and twice the waves: for
// transforms that do not fill the GPU, where the chain sets the time. 2^12
// points: two launches of 9 and 7 us, against 26 + 13 + 9 us for radix-8 threads
// whose pass pairs went through 36 KiB of LDS (77 -> 45 us for the call); three
// arrays of 2^17 142 -> 89 us.
// Bounds: after stage 1 values below 3.2r, each later stage adds at most 2r
// (its b is a product, below 1.1r): below 16r after 7. Limbs grow by at most
// 2^30 a stage from 2^29; normalized after every second stage, so a product's
// operand stays below 1.5 * 2^30.
template <int BIT>
ZK_DEV void lane_swap(F29& x0, F29& x1) {
    if (BIT == 4 || BIT == 5) {
#pragma unroll
        for (int i = 0; i < 9; i++) {
            // odd rows (halves) of x0 against even ones of x1
            const auto r = BIT == 4 ? __builtin_amdgcn_permlane16_swap(x0.l[i], x1.l[i], false, false)
                                    : __builtin_amdgcn_permlane32_swap(x0.l[i], x1.l[i], false, false);
            x0.l[i] = r[0];
            x1.l[i] = r[1];
        }
        return;
    }
    const uint32_t m = 0u - (threadIdx.x >> BIT & 1u);   // lanes with the bit keep x1
    const F29 give = f29_sel(m, x0, x1);
    F29 got;
#pragma unroll
    for (int i = 0; i < 9; i++) {
        if (BIT == 0) got.l[i] = u32_quad<1, 0, 3, 2>(give.l[i]);
        if (BIT == 1) got.l[i] = u32_quad<2, 3, 0, 1>(give.l[i]);
        if (BIT == 2) got.l[i] = u32_xor4(give.l[i]);
        if (BIT == 3) got.l[i] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give.l[i], 0x128, 0xf, 0xf, true);   // row_ror:8
    }
    x0 = f29_sel(m, got, x0);
    x1 = f29_sel(m, x1, got);
}
template <int Q, int S>
struct LaneStage {
    ZK_DEV static void run(F29& x0, F29& x1, uint32_t lane, const void* roots) {
        lane_swap<S - 2>(x0, x1);
        const uint32_t p = lane & ((1u << (S - 1)) - 1);
        const F29 b = fr29_mul(x1, ld_root(roots, p << (8 - S)));
        x1 = fr29_sub(x0, b);
        x0 = f29_add(x0, b);
        if (S % 2 == 0) {
            x0 = f29_norm(x0);
            x1 = f29_norm(x1);
        }
        LaneStage<Q, S + 1>::run(x0, x1, lane, roots);
    }
};
template <int Q> struct LaneEnd {
    ZK_DEV static void run(F29&, F29&, uint32_t, const void*) {}
};
template <> struct LaneStage<1, 2> : LaneEnd<1> {};
template <> struct LaneStage<2, 3> : LaneEnd<2> {};
template <> struct LaneStage<3, 4> : LaneEnd<3> {};
template <> struct LaneStage<4, 5> : LaneEnd<4> {};
template <> struct LaneStage<5, 6> : LaneEnd<5> {};
template <> struct LaneStage<6, 7> : LaneEnd<6> {};
template <> struct LaneStage<7, 8> : LaneEnd<7> {};

template <int Q>
__global__ void __launch_bounds__(NTT_THREADS) k_ntt_lane(NttPtrs ptrs, NttShape z) {
    constexpr uint32_t LANES = 1u << (Q - 1);
    const size_t tid = (size_t)blockIdx.x * NTT_THREADS + threadIdx.x, u = tid >> (Q - 1);
    if (u >= z.n >> Q) return;   // whole units
    const uint32_t lane = (uint32_t)tid & (LANES - 1);
    const void* in = ptrs.in[blockIdx.y];
    const NttUnit t = ntt_unit<Q>(z, u);
    const uint32_t b = Q > 1 ? __brev(lane) >> (33 - Q) : 0u;
    const size_t i0 = t.in + b * t.in_step, i1 = i0 + LANES * t.in_step;
    F29 x0 = ld29(in, i0), x1 = ld29(in, i1);
    if (z.pre) {
        x0 = fr29_mul(x0, ld29(z.pre, i0));
        x1 = fr29_mul(x1, ld29(z.pre, i1));
    }
    const F29 a = x0;
    x0 = f29_add(a, x1);
    x1 = fr29_sub(a, x1);
    LaneStage<Q, 2>::run(x0, x1, lane, z.roots);
    void* out = z.last ? ptrs.out[blockIdx.y] : ptrs.in[blockIdx.y];
    x0 = ntt_scale(z, t, lane, x0);
    x1 = ntt_scale(z, t, lane + LANES, x1);
    ntt_store(z, t, out, lane, x0);
    ntt_store(z, t, out, lane + LANES, x1);
}

// ---- four points per lane
// A unit's 2^Q points on 2^(Q-2) lanes, radix-4 steps in registers (a radix-2
// one last when Q is odd). Step t transforms the top digit left, which the
// lane's four slots hold, multiplies output k_t by w^(k_t * rest) and swaps the
// slots with the two lane bits that hold the next digit. In the end the lane
// bits hold k_1, k_2, ... from the top and the slots the last digit, of output k
// = k_1 + 4 k_2 + 16 k_3 + ...
// Which lane bits: the first swap on bits 5, 4 (v_permlane32/16_swap, one
// instruction per limb for both points), then 1, 0 (DPP in a quad); 3, 2 only
// in units of 2^7 points and more. The bits left over number the wave's units.
// Bound by instruction issue: 5044 VALU instructions per lane for 2^8 points per
// unit (3336 for 2^6), 60 % of them v_mad_u64_u32: 14.1 G lane instructions for the
// 2^22 transform, 0.38 ms at the 37 T/s of its mix, 0.25 ms of them the multiplies
// (34 T/s). Four waves per SIMD (five are the same, six spill 12 %). The
// radix-8 threads before took four launches (call 617 us, now 488); eight points
// per lane with the same exchange held three waves per SIMD and 563 us. Products
// with a stored b' = floor(b 2^261 / r) instead of Montgomery's: the same time.
constexpr int quad_bit(int Q, int i) {   // lane bit of the i-th bit from the top of the unit's lane
    return Q == 8 ? 5 - i : Q == 7 ? (i < 2 ? 5 - i : i < 4 ? 3 - i : 3) : (i < 2 ? 5 - i : 3 - i);
}
template <int BIT_HI, int BIT_LO>
ZK_DEV void quad_swap(F29 (&x)[4]) {
    lane_swap<BIT_HI>(x[0], x[2]);
    lane_swap<BIT_HI>(x[1], x[3]);
    lane_swap<BIT_LO>(x[0], x[1]);
    lane_swap<BIT_LO>(x[2], x[3]);
}
// Four-point DFT, natural order in and out. Inputs normalized and below 1.2r;
// outputs below 7r, limbs below 2.5 * 2^30 (a product takes them as they are: 9
// * 2.5 * 2^59 + 9 * 2^58 and the carry stay below 2^64). The difference of two
// sums takes 4r borrowed twice (R4B).
ZK_DEV void dft4(F29 (&x)[4], const F29& w4) {
    const F29 a = f29_add(x[0], x[2]), b = f29_add(x[1], x[3]);
    const F29 c = fr29_sub(x[0], x[2]), d = fr29_mul(fr29_sub(x[1], x[3]), w4);
    x[0] = f29_add(a, b);
#pragma unroll
    for (int i = 0; i < 9; i++) x[2].l[i] = a.l[i] + fr29c::R4B[i] - b.l[i];
    x[1] = f29_add(c, d);
    x[3] = fr29_sub(c, d);
}
// step T of a unit of 2^Q points, the digit over what lies below it in the lane
template <int Q, int T>
struct QuadStep {
    ZK_DEV static void run(F29 (&x)[4], uint32_t lane, const uint32_t* roots, const F29& w4) {
        constexpr int LEFT = Q - 2 * T;   // bits below this step's digit
        dft4(x, w4);
        if constexpr (LEFT > 0) {
            const uint32_t rest = lane & ((1u << LEFT) - 1);   // of the unit's lane, its low LEFT bits
            x[0] = settle29(x[0]);
#pragma unroll
            for (uint32_t k = 1; k < 4; k++)   // w_{2^(LEFT + 2)}^(rest * k)
                x[k] = fr29_mul(x[k], ld_root_lds(roots, (rest * k) << (8 - LEFT - 2)));
            if constexpr (LEFT == 1) {
                lane_swap<quad_bit(Q, Q - 3)>(x[0], x[2]);
                lane_swap<quad_bit(Q, Q - 3)>(x[1], x[3]);
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const F29 a = x[i], b = x[i + 2];
                    x[i] = f29_add(a, b);
                    x[i + 2] = fr29_sub(a, b);
                }
            } else {
                quad_swap<quad_bit(Q, 2 * T - 2), quad_bit(Q, 2 * T - 1)>(x);
                QuadStep<Q, T + 1>::run(x, lane, roots, w4);
            }
        }
    }
};

template <int Q>
__global__ void __launch_bounds__(NTT_THREADS) __attribute__((amdgpu_waves_per_eu(4))) k_ntt_quad(NttPtrs ptrs, NttShape z) {
    constexpr int LB = Q - 2;            // lane bits of a unit
    __shared__ uint32_t roots[9 * ROOTS];
    const F29 root = ld_root(z.roots, threadIdx.x);
    const uint32_t hw = threadIdx.x & 63;
    uint32_t lane = 0, used = 0, sub = 0;   // the unit's lane; the unit in the wave
#pragma unroll
    for (int i = 0; i < LB; i++) {
        lane |= (hw >> quad_bit(Q, i) & 1u) << (LB - 1 - i);
        used |= 1u << quad_bit(Q, i);
    }
#pragma unroll
    for (int i = 0, k = 0; i < 6; i++)
        if (!(used >> i & 1u)) sub |= (hw >> i & 1u) << k++;
    const size_t u = (((size_t)blockIdx.x * (NTT_THREADS / 64) + threadIdx.x / 64) << (6 - LB)) + sub, units = z.n >> Q;
    const void* in = ptrs.in[blockIdx.y];
    const NttUnit t = ntt_unit<Q>(z, u < units ? u : units - 1);
    F29 x[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) x[i] = ld29(in, t.in + (lane + (i << LB)) * t.in_step);
    st_root_lds(roots, threadIdx.x, root);
    __syncthreads();
    if (u >= units) return;   // whole units
    if (z.pre) {
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) x[i] = fr29_mul(x[i], ld29(z.pre, t.in + (lane + (i << LB)) * t.in_step));
    }
    QuadStep<Q, 1>::run(x, lane, roots, ld_root_lds(roots, 64));
    // output of slot s: digits k_1.. from the lane's top bits, the last from the slot
    uint32_t k0 = 0;
#pragma unroll
    for (int d = 0; 2 * d + 1 < LB; d++) k0 |= (lane >> (LB - 2 - 2 * d) & 3u) << (2 * d);
    // an odd Q's radix-2 step left the low bit of its radix-4 neighbour's digit
    // in slot bit 0, its high bit in the lane's last bit, its own digit in slot bit 1
    uint32_t k[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++)
        k[i] = Q % 2 ? k0 | (2 * (lane & 1u) + (i & 1u)) << (Q - 3) | (i >> 1) << (Q - 1) : k0 | i << LB;
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = ntt_scale(z, t, k[i], x[i]);
    void* out = z.last ? ptrs.out[blockIdx.y] : ptrs.in[blockIdx.y];
#pragma unroll
    for (int i = 0; i < 4; i++) ntt_store(z, t, out, k[i], x[i]);
}

// table[i] = lo[e & 4095] * hi[e >> 12] for e = exponent(i)
//   mode 0: e = i * step (mod 2n)
//   mode 1: pass twiddle, i = k*S + c -> e = c*k*step
__global__ void k_pow_table(void* __restrict__ out, size_t count, const void* __restrict__ lo, const void* __restrict__ hi,
                            int mode, uint64_t step, int logS, uint64_t mask, const void* __restrict__ scale) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    uint64_t e;
    if (mode == 0) e = (i * step) & mask;
    else {
        uint64_t k = i >> logS, c = i & (((uint64_t)1 << logS) - 1);
        e = (c * k * step) & mask;
    }
    Fr v = load<FrCfg>(lo, e & 4095);
    if (e >> 12) v = mul<FrCfg>(v, load<FrCfg>(hi, e >> 12));
    if (scale) v = mul<FrCfg>(v, load<FrCfg>(scale, 0));
    store<FrCfg>(out, i, v);
}

// host: powers tables of g (order 2^log_ord): lo[i] = g^i (i < 4096), hi[j] = g^(4096 j)
static void host_pow_tables(const zkh::Fr& g, int log_ord, std::vector<zkh::Fr>& lo, std::vector<zkh::Fr>& hi) {
    lo.assign(4096, zkh::Fr::one());
    for (int i = 1; i < 4096; i++) lo[i] = lo[i - 1] * g;
    zkh::Fr g4096 = lo[4095] * g;
    size_t nh = log_ord > 12 ? ((size_t)1 << (log_ord - 12)) : 1;
    hi.assign(nh, zkh::Fr::one());
    for (size_t j = 1; j < nh; j++) hi[j] = hi[j - 1] * g4096;
}

static zkh::Fr root_of_unity(int log_n) {
    // w_{2^log_n} = 5^((r-1) >> log_n)
    uint64_t e[4];
    memcpy(e, zkh::FrP::M, 32);
    e[0] -= 1;
    for (int s = 0; s < log_n; s++) {
        for (int k = 0; k < 3; k++) e[k] = (e[k] >> 1) | (e[k + 1] << 63);
        e[3] >>= 1;
    }
    return zkh::Fr::from_u64(5).pow(e);
}

// Pass radices of a size-2^ln transform; returns the pass count. Up to 2^17, two
// points per lane: radices up to 2^7 of even sizes. Above, four points per lane:
// up to 2^8, even powers (radix-4 steps only) but for an odd ln's last pass.
constexpr int NTT_LANE_LOG = 17;
static int ntt_layout(int ln, int lr[NTT_MAX_PASSES]) {
    const int most = ln <= NTT_LANE_LOG ? 7 : 8, np = (ln + most - 1) / most;
    for (int j = 0; j < NTT_MAX_PASSES; j++) lr[j] = 0;
    if (ln <= NTT_LANE_LOG) {
        for (int j = 0; j < np; j++) lr[j] = ln / np + (j < ln % np);
        return np;
    }
    int rem = ln;
    for (int j = 0; j < np; j++) rem -= lr[j] = ln / (2 * np) * 2;
    for (int j = 0; rem >= 2; j++, rem -= 2) lr[j] += 2;
    lr[np - 1] += rem;
    return np;
}
// Two points per lane below 2^20 points in all, where four leave less than four
// waves per SIMD: three arrays of 2^18 125 against 130 us, one of 2^19 101
// against 107, three of 2^17 89 against 103; from 2^20 on four are faster (three
// of 2^20 374 against 415, one of 2^22 488 against 569).
static bool ntt_two_points(int ln, size_t points) {
    return ln <= NTT_LANE_LOG || (ln <= 19 && points < ((size_t)1 << 20));   // 2^20 and up have 2^8 passes
}

// entries of the concatenated pass twiddle tables (passes 0..np-2), and each pass's offset
static size_t ntt_tw_entries(int ln, int np, const int lr[NTT_MAX_PASSES], size_t* off) {
    size_t tot = 0;
    int consumed = 0;
    for (int j = 0; j < np; j++) {
        if (off) off[j] = tot;
        if (j < np - 1) tot += (size_t)1 << (ln - consumed);
        consumed += lr[j];
    }
    return tot;
}

size_t NttPlan::bytes_for(int ln) {
    int lr_[NTT_MAX_PASSES];
    const int np_ = ntt_layout(ln, lr_);
    const size_t tot = ntt_tw_entries(ln, np_, lr_, nullptr);
    return 2 * std::max<size_t>(tot, 1) * 32 + 2 * ROOTS * ROOT_WORDS * 4 + 4 * ((size_t)1 << ln) * 32;
}

void NttPlan::build(int ln, hipStream_t st) {
    ZK_REQUIRE(ln >= 1 && ln <= 27, ZK_E_ARG, "NTT size must be 2^1..2^27");
    log_n = ln;
    n = (size_t)1 << ln;
    np = ntt_layout(ln, lr);

    // base power tables for w_2n and w_2n^-1 (cover every w_M, w_R and the coset factors)
    zkh::Fr w2n = root_of_unity(ln + 1), w2n_inv = w2n.inv();
    std::vector<zkh::Fr> lo_f, hi_f, lo_i, hi_i;
    host_pow_tables(w2n, ln + 1, lo_f, hi_f);
    host_pow_tables(w2n_inv, ln + 1, lo_i, hi_i);
    DevBuf d_lo_f(4096 * 32), d_hi_f(hi_f.size() * 32), d_lo_i(4096 * 32), d_hi_i(hi_i.size() * 32), d_scale(32),
        d_s32(32);
    ZK_HIP(hipMemcpyAsync(d_lo_f.p, lo_f.data(), 4096 * 32, hipMemcpyHostToDevice, st));
    ZK_HIP(hipMemcpyAsync(d_hi_f.p, hi_f.data(), hi_f.size() * 32, hipMemcpyHostToDevice, st));
    ZK_HIP(hipMemcpyAsync(d_lo_i.p, lo_i.data(), 4096 * 32, hipMemcpyHostToDevice, st));
    ZK_HIP(hipMemcpyAsync(d_hi_i.p, hi_i.data(), hi_i.size() * 32, hipMemcpyHostToDevice, st));
    // every table value the kernels multiply by is prescaled by 2^5 (the
    // 29-bit product's R'/2^256, field29.hpp "Fr")
    const zkh::Fr s32 = zkh::Fr::from_u64(32);
    const zkh::Fr ninv = zkh::Fr::from_u64(n).inv() * s32;
    ZK_HIP(hipMemcpyAsync(d_scale.p, &ninv, 32, hipMemcpyHostToDevice, st));
    ZK_HIP(hipMemcpyAsync(d_s32.p, &s32, 32, hipMemcpyHostToDevice, st));
    const uint64_t mask2n = (2 * (uint64_t)n) - 1;

    // w_256^i for the DFTs inside a unit, forward and inverse, in limbs
    std::vector<uint32_t> limbs[2];
    for (int d = 0; d < 2; d++) {
        const zkh::Fr g = d ? root_of_unity(8).inv() : root_of_unity(8);
        zkh::Fr f = s32;
        limbs[d].assign(ROOTS * ROOT_WORDS, 0);
        for (int i = 0; i < ROOTS; i++, f = f * g)
            for (int l = 0; l < 9; l++) {
                const int k = 29 * l / 64, sh = 29 * l % 64;
                uint64_t v = f.v[k] >> sh;
                if (sh > 35 && k < 3) v |= f.v[k + 1] << (64 - sh);
                limbs[d][ROOT_WORDS * i + l] = (uint32_t)v & f29c::MASK;
            }
        DevBuf& dst = d ? roots_inv : roots_fwd;
        dst.ensure(ROOTS * ROOT_WORDS * 4);
        ZK_HIP(hipMemcpyAsync(dst.p, limbs[d].data(), ROOTS * ROOT_WORDS * 4, hipMemcpyHostToDevice, st));
    }
    // pass twiddle tables w_M^(c k), layout [k][c], for passes 0..np-2
    const size_t tot = ntt_tw_entries(ln, np, lr, tw_off);
    tw_fwd.ensure(std::max<size_t>(tot, 1) * 32);
    tw_inv.ensure(std::max<size_t>(tot, 1) * 32);
    int consumed = 0;
    for (int j = 0; j < np - 1; j++) {
        int logM = ln - consumed;
        int logS = logM - lr[j];
        uint64_t step_M = (uint64_t)1 << (ln + 1 - logM);  // w_M = w_2n^(2n/M)
        size_t cnt = (size_t)1 << logM;
        k_pow_table<<<cdiv(cnt, 256), 256, 0, st>>>((char*)tw_fwd.p + tw_off[j] * 32, cnt, d_lo_f.p, d_hi_f.p, 1, step_M,
                                                   logS, mask2n, d_s32.p);
        k_pow_table<<<cdiv(cnt, 256), 256, 0, st>>>((char*)tw_inv.p + tw_off[j] * 32, cnt, d_lo_i.p, d_hi_i.p, 1, step_M,
                                                   logS, mask2n, d_s32.p);
        consumed += lr[j];
    }
    // element-wise tables
    coset_fwd.ensure(n * 32);
    inv_coset.ensure(n * 32);
    inv_plain.ensure(n * 32);
    inv_uncoset.ensure(n * 32);
    k_pow_table<<<cdiv(n, 256), 256, 0, st>>>(coset_fwd.p, n, d_lo_f.p, d_hi_f.p, 0, 1, 0, mask2n, d_s32.p);
    k_pow_table<<<cdiv(n, 256), 256, 0, st>>>(inv_coset.p, n, d_lo_f.p, d_hi_f.p, 0, 1, 0, mask2n, d_scale.p);
    k_pow_table<<<cdiv(n, 256), 256, 0, st>>>(inv_plain.p, n, d_lo_f.p, d_hi_f.p, 0, 0, 0, mask2n, d_scale.p);
    k_pow_table<<<cdiv(n, 256), 256, 0, st>>>(inv_uncoset.p, n, d_lo_i.p, d_hi_i.p, 0, 1, 0, mask2n, d_scale.p);
    ZK_HIP(hipGetLastError());
    ZK_HIP(hipStreamSynchronize(st));  // the temporaries above are freed on return
}

template <int Q>
static void launch_lane(const NttPtrs& ptrs, int batch, const NttShape& z, hipStream_t st) {
    k_ntt_lane<Q><<<dim3(cdiv(z.n / 2, NTT_THREADS), batch), NTT_THREADS, 0, st>>>(ptrs, z);
}
template <int Q>
static void launch_quad(const NttPtrs& ptrs, int batch, const NttShape& z, hipStream_t st) {
    k_ntt_quad<Q><<<dim3(cdiv(z.n / 4, NTT_THREADS), batch), NTT_THREADS, 0, st>>>(ptrs, z);
}

void ntt_run(const NttPlan& p, void* const* in, void* const* out, int batch, bool inverse, const void* pre, const void* post,
             hipStream_t st) {
    ZK_REQUIRE(batch >= 1 && batch <= NTT_MAX_BATCH, ZK_E_ARG, "NTT batch must be 1..4");
    NttPtrs ptrs;
    for (int b = 0; b < NTT_MAX_BATCH; b++) {
        ptrs.in[b] = b < batch ? in[b] : nullptr;
        ptrs.out[b] = b < batch ? out[b] : nullptr;
        if (b < batch && p.log_n > 4) ZK_REQUIRE(in[b] != out[b], ZK_E_ARG, "NTT of more than 16 points needs distinct in/out");
    }
    NttShape z;
    z.dg.np = p.np;
    for (int j = 0; j < NTT_MAX_PASSES; j++) z.dg.lr[j] = p.lr[j];
    z.n = p.n;
    z.roots = (inverse ? p.roots_inv : p.roots_fwd).p;
    const char* tw = (const char*)(inverse ? p.tw_inv.p : p.tw_fwd.p);
    const bool lanes = ntt_two_points(p.log_n, p.n * batch);
    int consumed = 0;
    for (int j = 0; j < p.np; j++) {
        const int q = p.lr[j];
        consumed += q;
        z.last = j == p.np - 1;
        z.logS = p.log_n - consumed;
        z.tw = tw + p.tw_off[j] * 32;
        z.pre = j == 0 ? pre : nullptr;
        z.post = post;
        if (lanes) {
            switch (q) {
                case 1: launch_lane<1>(ptrs, batch, z, st); break;
                case 2: launch_lane<2>(ptrs, batch, z, st); break;
                case 3: launch_lane<3>(ptrs, batch, z, st); break;
                case 4: launch_lane<4>(ptrs, batch, z, st); break;
                case 5: launch_lane<5>(ptrs, batch, z, st); break;
                case 6: launch_lane<6>(ptrs, batch, z, st); break;
                default: launch_lane<7>(ptrs, batch, z, st); break;
            }
        } else {
            switch (q) {
                case 6: launch_quad<6>(ptrs, batch, z, st); break;
                case 7: launch_quad<7>(ptrs, batch, z, st); break;
                default: launch_quad<8>(ptrs, batch, z, st); break;
            }
        }
        ZK_HIP(hipGetLastError());
    }
}

}  // namespace zk
