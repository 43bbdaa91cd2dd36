// Negacyclic NTT / iNTT on uint64 RNS limbs for CDNA4.
//
// Transform (same convention as the reference, fntt_2d.cu / intt_2d.cu):
//   forward Cooley-Tukey, stage s (m = 2^s groups, distance t = N/2^(s+1)),
//   group i uses tw[m + i] with tw[brv(k)] = psi^k; the output is the
//   evaluation at psi^(2 brv(j) + 1) in slot j, fully reduced to [0, q).
//   inverse Gentleman-Sande with itw[brv(k)] = psi^-k, then x N^-1.
//
// Decomposition: N = N1 * 512. The first log N1 = log N - 9 stages (3 to 8) pair words
// whose indices differ by multiples of 512 (column pass): up to 5 stages a thread holds a
// whole column in registers; 6 to 8 stages take two rounds of register units with one
// exchange through LDS. The last 9 stages act on 512 contiguous words (row pass): one wave
// runs a row in three rounds of radix-8 units, 8 words per lane, and exchanges between
// rounds through LDS words of its own, so the row pass has no block barrier at all. An
// earlier split of 4 + 12 stages staged 4096-word tiles through LDS with five barriers, and
// its tile pass held 734 of a word group's 890 vector instructions; with 7 + 9 stages both
// passes stay below the memory's time (64 x 24 limbs at N = 2^16, forward: column pass 267
// -> 294 us, tile / row pass 393 -> 326 us; each moves 1.61 GB).
//
// Twiddles are 16-byte entries: the split form of a prime just below a power of two
// (FoldMod, arith.h) or (w, floor(w 2^64 / q)) of any other. A row's 511 entries lie in the
// order its lanes read them, [round 1: 7][round 2: 7][8][round 3: 7][64], so that every
// load of a wave is one contiguous run (round 3 read from a table in stage order
// spreads a load over up to 64 cache lines).
//
// Butterfly arithmetic, by prime:
//   - split form: signed unreduced words, (a + t, a - t) with |t| <= R = fold_bound, nine
//     issue slots a butterfly (a Shoup butterfly takes about 26);
//   - otherwise Harvey's lazy ranges: [0, 4q) forward, [0, 2q) inverse (primes < 2^61).
// A launch whose primes all have split forms and whose log N products fit a signed word
// runs kernels of that form alone (FAST); any other launch runs kernels that pick the form
// per limb and fold split-form words every second stage (GENERAL). Outputs are canonical
// residues, the same words in every form.
#include <algorithm>

#include <mutex>
#include <type_traits>
#include <vector>

#include "engine.h"

namespace shm {

struct LimbMap {
    uint32_t n_active;    // transformed limbs per polynomial
    uint32_t lo;          // first limb
    uint32_t skip_lo;     // limbs >= skip_lo are shifted by skip_width
    uint32_t skip_width;
    uint32_t Ql;          // limbs >= Ql use special primes nQ + (k - Ql)
    uint32_t nQ;
    uint32_t first_prime; // prime of limb k < Ql is first_prime + k
    uint64_t poly_stride; // words between polynomials
};

__device__ __forceinline__ void limb_of(const LimbMap &m, uint32_t z, uint32_t &poly, uint32_t &k,
                                        uint32_t &prime) {
    poly = z / m.n_active;
    const uint32_t j = z - poly * m.n_active;
    k = m.lo + j;
    if (k >= m.skip_lo) k += m.skip_width;
    prime = k < m.Ql ? m.first_prime + k : m.nQ + (k - m.Ql);
}

namespace {

constexpr int kRow = 512;       // words of a row: the last 9 stages
constexpr int kRowLds = 576;    // LDS words of a row: one of padding per 8 (row_slot)
constexpr int kThreads = 256;

typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
// Pointers the kernel reads out of device memory or selects between are known to
// address global memory: the cast lets their accesses use global instead of flat
// instructions (flat ones also hold the LDS wait counter).
template <typename V>
__device__ __forceinline__ __attribute__((address_space(1))) V *global_ptr(V *p) {
    return (__attribute__((address_space(1))) V *)p;
}
template <typename V>
__device__ __forceinline__ const __attribute__((address_space(1))) V *global_ptr(const V *p) {
    return (const __attribute__((address_space(1))) V *)p;
}

// Tables that no kernel writes while it reads them: wave-uniform reads through this
// pointer stay scalar loads also after the kernel's own stores.
template <typename V>
__device__ __forceinline__ const __attribute__((address_space(4))) V *table_ptr(const V *p) {
    return (const __attribute__((address_space(4))) V *)(uintptr_t)p;
}
__device__ __forceinline__ FoldMod table_fold(const FoldMod *p) {
    static_assert(sizeof(FoldMod) == 5 * sizeof(uint64_t), "FoldMod is read in words");
    uint64_t w[5];
    const auto q = table_ptr(reinterpret_cast<const uint64_t *>(p));
#pragma unroll
    for (int i = 0; i < 5; i++) w[i] = q[i];
    FoldMod f;
    __builtin_memcpy(&f, w, sizeof f);
    return f;
}

// Twiddle and constant tables of one launch (forward or inverse set).
struct NttTables {
    const DevMod *mods;
    const FoldMod *fold;              // pw = 0: the prime has no split form
    const u32x4 *col;                 // [QP][kNttCols]: twiddles 1 .. N1 - 1 of the column stages
    const u32x4 *row;                 // [QP][N / 512][512]: each row's twiddles in lane order
    const uint64_t *ninv, *ninv_s;
};

// Arithmetic of one prime. fwd / inv: one stage's butterflies on a unit of 2^R words, tw(e)
// being the entry of group i at unit stage u, e = 2^u - 1 + i.
struct HarveyK {
    uint64_t q;
    __device__ HarveyK(const NttTables &tb, uint32_t prime) : q(table_ptr(&tb.mods[prime].q)[0]) {}
    __device__ __forceinline__ const HarveyK &here() const { return *this; }
    static __device__ __forceinline__ uint64_t lo(u32x4 w) { return ((uint64_t)w.y << 32) | w.x; }
    static __device__ __forceinline__ uint64_t hi(u32x4 w) { return ((uint64_t)w.w << 32) | w.z; }
    __device__ __forceinline__ void fwd(uint64_t &a, uint64_t &b, u32x4 w) const {
        const uint64_t q2 = q << 1, s = a >= q2 ? a - q2 : a;
        const uint64_t t = mul_shoup_lazy(b, lo(w), hi(w), q);
        a = s + t;
        b = s + q2 - t;
    }
    __device__ __forceinline__ void inv(uint64_t &a, uint64_t &b, u32x4 w) const {
        const uint64_t q2 = q << 1, d = a + q2 - b, s = a + b;
        a = s >= q2 ? s - q2 : s;
        b = mul_shoup_lazy(d, lo(w), hi(w), q);
    }
    template <int R>
    __device__ __forceinline__ void after_fwd(uint64_t *, int) const {}
    template <int R>
    __device__ __forceinline__ void after_inv(uint64_t *, int) const {}
    // canonical residue of a forward word, and of x w (Shoup pair w, ws)
    __device__ __forceinline__ uint64_t canon(uint64_t v) const {
        v = v >= (q << 1) ? v - (q << 1) : v;
        return v >= q ? v - q : v;
    }
    struct Const {
        uint64_t w, ws;
    };
    __device__ __forceinline__ Const constant(uint64_t w, uint64_t ws) const { return {w, ws}; }
    __device__ __forceinline__ uint64_t mul(uint64_t x, Const c) const { return mul_shoup(x, c.w, c.ws, q); }
    __device__ __forceinline__ uint64_t sub_mul(uint64_t acc, uint64_t v, Const c) const {
        return mul_shoup(sub_mod(acc, canon(v), q), c.w, c.ws, q);
    }
    __device__ __forceinline__ uint64_t load_residue(uint64_t v, uint64_t center, const DevMod &m) const {
        uint64_t y = reduce64(v, m);
        if (center && v > center) y = sub_mod(y, reduce64(2 * center + 1, m), q);
        return y;
    }
    __device__ __forceinline__ uint64_t load_signed(uint64_t v, const DevMod &m) const {
        const bool neg = (int64_t)v < 0;
        const uint64_t y = reduce64(neg ? 0 - v : v, m);
        return neg ? neg_mod(y, q) : y;
    }
};

// SAFE folds a unit's words every second stage, so only a few products ever add up (for
// primes further below the power of two, and for limbs of GENERAL launches); otherwise the
// launcher has checked that log N of them fit.
template <bool SAFE>
struct FoldK {
    uint64_t q;
    FoldMod f;
    __device__ FoldK(const NttTables &tb, uint32_t prime)
        : q(table_ptr(&tb.mods[prime].q)[0]), f(table_fold(tb.fold + prime)) {}
    // The constants, redefined at the place of use. Their sign extensions must stand in the
    // block of the products that use them: hoisted out of a loop, a product by delta is no
    // longer seen as 32 x 32 bits and costs a multiply-add, two multiplies and two adds. In the
    // row pass that was 144 of 635 vector instructions per 8 words.
    __device__ __forceinline__ FoldK here() const {
        FoldK k = *this;
        asm volatile("" : "+s"(k.f.d4), "+s"(k.f.d));
        return k;
    }
    __device__ __forceinline__ void fwd(uint64_t &a, uint64_t &b, u32x4 w) const {
        const uint64_t t = fold_mul(b, w, f), s = a;
        a = s + t;
        b = s - t;
    }
    __device__ __forceinline__ void inv(uint64_t &a, uint64_t &b, u32x4 w) const {
        const uint64_t d = a - b;
        a = a + b;
        b = fold_mul(d, w, f);
    }
    template <int R>
    __device__ __forceinline__ void after_fwd(uint64_t *x, int u) const {
        if (SAFE && ((u & 1) || u == R - 1))
#pragma unroll
            for (int l = 0; l < (1 << R); l++) x[l] = fold_tight(x[l], f);
    }
    // sums double per stage: those of a unit's last stage (l < 2^(R-1)) come back to b bits
    template <int R>
    __device__ __forceinline__ void after_inv(uint64_t *x, int u) const {
#pragma unroll
        for (int l = 0; l < (1 << R); l++)
            if (u == 0 ? l < (1 << (R - 1)) : SAFE && (((R - 1 - u) & 1) != 0)) x[l] = fold_tight(x[l], f);
    }
    __device__ __forceinline__ uint64_t canon(uint64_t v) const { return fold_canon<SAFE>(v, q, f); }
    typedef u32x4 Const;
    __device__ __forceinline__ Const constant(uint64_t w, uint64_t ws) const { return fold_split(w, ws, q, f); }
    __device__ __forceinline__ uint64_t mul(uint64_t x, Const c) const { return fold_canon<SAFE>(fold_mul(x, c, f), q, f); }
    __device__ __forceinline__ uint64_t sub_mul(uint64_t acc, uint64_t v, Const c) const { return mul(acc - v, c); }
    // signed words need no reduction
    __device__ __forceinline__ uint64_t load_residue(uint64_t v, uint64_t center, const DevMod &) const {
        return center && v > center ? v - (2 * center + 1) : v;
    }
    __device__ __forceinline__ uint64_t load_signed(uint64_t v, const DevMod &) const { return v; }
};

template <int R, typename K, typename TW>
__device__ __forceinline__ void ct_unit(uint64_t *x, const K &kc, TW tw) {
    const K k = kc.here();
#pragma unroll
    for (int u = 0; u < R; u++) {
        const int h = 1 << (R - 1 - u);
#pragma unroll
        for (int l = 0; l < (1 << R); l++)
            if ((l & h) == 0) k.fwd(x[l], x[l + h], tw((1 << u) - 1 + (l >> (R - u))));
        k.template after_fwd<R>(x, u);
    }
}

template <int R, typename K, typename TW>
__device__ __forceinline__ void gs_unit(uint64_t *x, const K &kc, TW tw) {
    const K k = kc.here();
#pragma unroll
    for (int u = R - 1; u >= 0; u--) {
        const int h = 1 << (R - 1 - u);
#pragma unroll
        for (int l = 0; l < (1 << R); l++)
            if ((l & h) == 0) k.inv(x[l], x[l + h], tw((1 << u) - 1 + (l >> (R - u))));
        k.template after_inv<R>(x, u);
    }
}

// Extra I/O of fused variants.
//   IO_PLAIN   : in-place transform of `data`.
//   IO_REDUCE  : (phase A, forward) the input of limb k of polynomial p is
//                src[p * N + idx] reduced mod the limb's prime (a broadcast of
//                one coefficient-form limb to other primes, rns.cu:1125-1137).
//   IO_RESCALE : (phase B, forward) instead of storing v = NTT(delta), store
//                (acc - v) * qinv mod q to outs[p / ppo] + (p % ppo) L1 N + k N
//                (rns.cu:1138-1155 fused with the final NTT pass). With
//                out_packed, polynomial p reads acc at its acc_limbs stride and
//                writes out_p[p], adding onto it when bit p of acc_mask is set
//                (the ModDown combine, rns_bconv.cu:680-690 and 776-828, fused the same way).
//   IO_GATHER  : (phase B, inverse) limb k of polynomial p is read from
//                acc_p.p[p] + k N (separate input buffers) and the transform is
//                written to `data`: the gather copy fused into the first pass.
//   IO_DIGITS  : (phase B, forward) polynomial m digits + g is digit g of member m: its own
//                limbs [g alpha, (g + 1) alpha) below Ql are copied from acc_p.p[m] (copy_own)
//                or left untouched, the others transformed.
enum { IO_PLAIN = 0, IO_REDUCE = 1, IO_RESCALE = 2, IO_GATHER = 4, IO_DIGITS = 5 };

struct NttIO {
    const uint64_t *src;      // IO_REDUCE: [n_polys][N]
    const uint64_t *acc;      // IO_RESCALE: [n_polys][acc_limbs][N]
    uint64_t *const *outs;    // IO_RESCALE: output base per group of ppo polys (device array)
    uint64_t *out_single;     // IO_RESCALE: used instead of outs when outs is null
    const uint64_t *qinv;     // IO_RESCALE: per prime
    const uint64_t *qinv_s;
    uint32_t acc_limbs;
    uint32_t ppo;
    uint64_t center;          // IO_REDUCE: 0, or h = q_last >> 1: values above h stand for v - q_last
    uint32_t packed;          // IO_RESCALE: nonzero -> polynomial p reads acc_p[p], writes out_p[p]
    uint32_t out_packed;      // IO_RESCALE: nonzero -> polynomial p reads acc, writes out_p[p]
    uint64_t acc_mask;        // IO_RESCALE with out_packed: bit p set -> out_p[p] += result
    uint32_t out_limbs;       // IO_RESCALE with outs: limbs per output polynomial (0: the launch's)
    PolyPack acc_p, out_p;    // IO_RESCALE with packed / out_packed; IO_GATHER inputs in acc_p
    const uint32_t *add_perm; // IO_RESCALE with out_packed: add add_src.p[p] read through this
    PolyPack add_src;         // NTT-domain permutation instead of out_p[p] (acc_mask bit p set)
    const uint64_t *scale;    // inverse, phase A: limb k is multiplied by scale[k - scale_lo]
    const uint64_t *scale_s;  // (value, Shoup companion) instead of N^-1, unless null
    uint32_t scale_lo;
    uint32_t digits, alpha, copy_own;  // IO_DIGITS
    const uint32_t *perm;     // IO_GATHER: inputs read through this NTT-domain permutation, unless null
};

// Column pass, log N1 = RA + RB stages. A block takes C columns (consecutive words of a
// row of 512) with all their N1 words. Round 1 (RA stages) runs on register units of words
// 2^RB rows apart, its twiddles the same for every column (scalar loads); with RB > 0 the
// block then exchanges through LDS once and round 2 (RB stages) runs on 2^RB adjacent rows.
// 32 columns (16 for RB = 4) keep each access a run of 256 (128) bytes and the block at 16
// to 32 KB of LDS, five or more blocks a CU. Memory bounds the pass: 1.61 GB in 294 us (5.5
// TB/s); 64 columns and 512 threads measured 287 us forward and 324 us inverse against 294
// and 305 us.
constexpr int col_width(int ra, int rb) { return rb == 0 ? kThreads : kThreads >> rb; }

template <int RA, int RB, bool FWD, int IO, typename K>
__device__ __forceinline__ void col_pass(const K &k, uint64_t *lds, uint64_t *base, const u32x4 *__restrict__ col,
                                         uint32_t c0, const NttTables &tb, uint32_t prime, uint32_t poly, uint32_t limb,
                                         size_t N, const NttIO &io) {
    constexpr int C = col_width(RA, RB);
    constexpr int UNITS = RB == 0 ? 1 : (C << RA) / kThreads;  // round-2 units per thread
    const uint32_t cl = threadIdx.x % C, c = c0 + cl;
    const uint32_t r0 = RB == 0 ? 0 : threadIdx.x / C;         // round 1: rows r0 + l 2^RB
    auto tw1 = [&](int e) { return col[e + 1]; };
    uint64_t x[1 << RA];
    // round 2 on unit m: rows g 2^RB + l, g = threadIdx / C + m 256 / C
    auto round2 = [&](auto body) {
        if constexpr (RB > 0) {
#pragma unroll
            for (int m = 0; m < UNITS; m++) {
                const uint32_t g = threadIdx.x / C + m * (kThreads / C);
                auto tw2 = [&](int e) {
                    const int u = e >= 7 ? 3 : e >= 3 ? 2 : e >= 1 ? 1 : 0;
                    return col[(((1u << RA) + g) << u) + (uint32_t)(e - ((1 << u) - 1))];
                };
                body(g, tw2);
            }
        }
    };
    if constexpr (FWD) {
        if (IO == IO_REDUCE) {
            const DevMod m = tb.mods[prime];
            const uint64_t *src = io.src + (size_t)poly * N + c;
#pragma unroll
            for (int l = 0; l < (1 << RA); l++)
                x[l] = k.load_residue(src[(size_t)(r0 + (l << RB)) * kRow], io.center, m);
        } else {
#pragma unroll
            for (int l = 0; l < (1 << RA); l++) x[l] = base[(size_t)(r0 + (l << RB)) * kRow + c];
        }
        ct_unit<RA>(x, k, tw1);
        if constexpr (RB == 0) {
#pragma unroll
            for (int l = 0; l < (1 << RA); l++) __builtin_nontemporal_store(x[l], &base[(size_t)l * kRow + c]);
        } else {
#pragma unroll
            for (int l = 0; l < (1 << RA); l++) lds[(r0 + (l << RB)) * C + cl] = x[l];
            __syncthreads();
            round2([&](uint32_t g, auto tw2) {
                uint64_t y[1 << RB];
#pragma unroll
                for (int l = 0; l < (1 << RB); l++) y[l] = lds[((g << RB) + l) * C + cl];
                ct_unit<RB>(y, k, tw2);
                // streaming store: the row pass reads these words back long after
#pragma unroll
                for (int l = 0; l < (1 << RB); l++)
                    __builtin_nontemporal_store(y[l], &base[(size_t)((g << RB) + l) * kRow + c]);
            });
        }
    } else {
        if constexpr (RB == 0) {
#pragma unroll
            for (int l = 0; l < (1 << RA); l++) x[l] = base[(size_t)l * kRow + c];
        } else {
            round2([&](uint32_t g, auto tw2) {
                uint64_t y[1 << RB];
#pragma unroll
                for (int l = 0; l < (1 << RB); l++) y[l] = base[(size_t)((g << RB) + l) * kRow + c];
                gs_unit<RB>(y, k, tw2);
#pragma unroll
                for (int l = 0; l < (1 << RB); l++) lds[((g << RB) + l) * C + cl] = y[l];
            });
            __syncthreads();
#pragma unroll
            for (int l = 0; l < (1 << RA); l++) x[l] = lds[(r0 + (l << RB)) * C + cl];
        }
        gs_unit<RA>(x, k, tw1);
        const K kh = k.here();
        const auto ni = io.scale ? k.constant(io.scale[limb - io.scale_lo], io.scale_s[limb - io.scale_lo])
                                 : k.constant(tb.ninv[prime], tb.ninv_s[prime]);
#pragma unroll
        for (int l = 0; l < (1 << RA); l++)
            __builtin_nontemporal_store(kh.mul(x[l], ni), &base[(size_t)(r0 + (l << RB)) * kRow + c]);
    }
}

template <int RA, int RB, bool FWD, int IO, bool FAST>
__global__ __launch_bounds__(kThreads) void k_ntt_cols(uint64_t *__restrict__ data, LimbMap mp, NttTables tb, int logN,
                                                       NttIO io) {
    constexpr int C = col_width(RA, RB);
    __shared__ uint64_t lds[RB == 0 ? 1 : C << (RA + RB)];
    const size_t N = size_t(1) << logN;
    const uint32_t z = blockIdx.x / (kRow / C);
    const uint32_t c0 = (blockIdx.x % (kRow / C)) * C;
    uint32_t poly, k, prime;
    limb_of(mp, z, poly, k, prime);
    uint64_t *base = data + poly * mp.poly_stride + (size_t)k * N;
    const u32x4 *col = tb.col + (size_t)prime * kNttCols;
    if constexpr (FAST) {
        col_pass<RA, RB, FWD, IO>(FoldK<false>(tb, prime), lds, base, col, c0, tb, prime, poly, k, N, io);
    } else {
        if (tb.fold[prime].pw)
            col_pass<RA, RB, FWD, IO>(FoldK<true>(tb, prime), lds, base, col, c0, tb, prime, poly, k, N, io);
        else
            col_pass<RA, RB, FWD, IO>(HarveyK(tb, prime), lds, base, col, c0, tb, prime, poly, k, N, io);
    }
}

// Base conversion into the column stages (ConvertJob). A block keeps the source words of its
// columns in registers (A words per coefficient, 16 coefficients a thread at N = 2^16: 160 of
// its 256 VGPRs for 5 special primes) and loops over a run of output limbs: sums of split
// products, column stages, store. One exchange through LDS per limb, double-buffered, so one
// barrier; the limb's column twiddles come through LDS too, requested a limb ahead. Against a
// conversion kernel that writes every limb and a column pass that reads it back, the words
// in between (and their reduction to canonical residues) are gone: a shared-a chunk's
// conversions and forward column passes at N = 2^16 took 29.0 ms apart and take 18.3 ms
// here; one top-level rotation's 154 and 87 us. Bound by VALU issue at 2 waves per SIMD
// (8 words a thread, which halves the registers, needs a third exchange at 7 stages).
template <int RA, int RB, int A, bool FAST>
__global__ __launch_bounds__(kThreads, 2) void k_convert_cols(ConvertJob job, NttTables tb, int logN, uint32_t nQ,
                                                              uint32_t run) {
    constexpr int C = col_width(RA, RB), U = 1 << RA, N1 = 1 << (RA + RB);
    constexpr int UNITS = RB == 0 ? 1 : (C << RA) / kThreads;
    __shared__ uint64_t lds[2][RB == 0 ? 1 : C * N1];
    __shared__ __align__(16) u32x4 ltw[2][N1];
    const size_t N = size_t(1) << logN;
    const uint32_t cl = threadIdx.x % C, c = blockIdx.x * C + cl, r0 = RB == 0 ? 0 : threadIdx.x / C;
    const uint32_t poly = blockIdx.y, g = poly % job.digits, start = g * job.alpha;
    const uint32_t size = min(job.alpha, job.total - start);
    const uint64_t *src = job.src + (size_t)(poly / job.digits) * job.src_stride + (size_t)(job.src_lo + start) * N + c;
    auto prime_of = [&](uint32_t k) { return k < job.Ql ? k : nQ + (k - job.Ql); };
    // source words in halves, and each coefficient's rounding (at most A < 16) in 4 bits
    uint32_t yl[A][U], yh[A][U], r[(U + 7) / 8] = {};
    bool big = false;
    {
        uint64_t y[A][U];
        double v[U];
#pragma unroll
        for (int l = 0; l < U; l++) v[l] = 0.0;
        if (A == 1 && job.fft) {
            // rounded encoder coefficients: rows below N1 / 2 are real parts, row r + N1 / 2 the
            // imaginary part of the same entry. Those of 2^60 and more are reduced per prime.
            const double2 *fb = job.fft + (size_t)poly * (N / 2) + c;
#pragma unroll
            for (int l = 0; l < U; l++) {
                const uint32_t row = r0 + (l << RB);
                const double2 z = fb[(size_t)(row & (N1 / 2 - 1)) * kRow];
                const double t = round(row < N1 / 2 ? z.x : z.y);
                big = big || !(fabs(t) < 1152921504606846976.0);
                y[0][l] = (uint64_t)(int64_t)t;
            }
        } else
#pragma unroll
        for (int i = 0; i < A; i++) {
            if ((uint32_t)i < size) {
#pragma unroll
                for (int l = 0; l < U; l++) y[i][l] = src[(size_t)i * N + (size_t)(r0 + (l << RB)) * kRow];
            } else {
#pragma unroll
                for (int l = 0; l < U; l++) y[i][l] = 0;
            }
        }
        if (job.rounded) {
#pragma unroll
            for (int i = 0; i < A; i++) {
                if ((uint32_t)i < size) {
                    const double q = (double)table_ptr(&tb.mods[prime_of(job.src_lo + start + i)].q)[0];
#pragma unroll
                    for (int l = 0; l < U; l++) v[l] = __dadd_rn(v[l], __ddiv_rn((double)y[i][l], q));
                }
            }
#pragma unroll
            for (int l = 0; l < U; l++) r[l / 8] |= (uint32_t)(uint64_t)__dadd_rn(v[l], 0.5) << (4 * (l % 8));
            if (A == 1) {  // one source limb: the signed word itself
                const uint64_t q = table_ptr(&tb.mods[prime_of(job.src_lo + start)].q)[0];
#pragma unroll
                for (int l = 0; l < U; l++) y[0][l] -= ((r[l / 8] >> (4 * (l % 8))) & 15) ? q : 0;
            }
        }
#pragma unroll
        for (int i = 0; i < A; i++)
#pragma unroll
            for (int l = 0; l < U; l++) {
                yl[i][l] = (uint32_t)y[i][l];
                yh[i][l] = (uint32_t)(y[i][l] >> 32);
            }
    }
    const uint32_t k_end = min((blockIdx.z + 1) * run, job.n_out);
    uint64_t *out = job.out + (size_t)poly * job.out_stride + c;
    // the next limb to convert from k on (uniform over the block)
    auto next = [&](uint32_t k) {
        return job.skip_own && k >= start && k < start + size ? start + size : k;
    };
    auto tw_of = [&](uint32_t k) {
        return k < k_end && threadIdx.x < N1 ? tb.col[(size_t)prime_of(k) * kNttCols + threadIdx.x] : u32x4{0, 0, 0, 0};
    };
    uint32_t k = next(blockIdx.z * run);
    u32x4 tw_next = tw_of(k);
    // waited for here: in the loop, that wait would cover the previous limb's stores as well
    asm volatile("" : "+v"(tw_next));
    int buf = 0;
    while (k < k_end) {
        const uint32_t prime = prime_of(k), k_next = next(k + 1);
        if (threadIdx.x < N1) ltw[buf][threadIdx.x] = tw_next;
        tw_next = tw_of(k_next);
        // The halves pass through an empty statement each turn: their widening stays inside
        // the loop, next to the multiply-adds it belongs to (hoisted, it doubles the registers
        // and turns every product into a 64 x 64 one).
#pragma unroll
        for (int i = 0; i < A; i++)
#pragma unroll
            for (int l = 0; l < U; l++) asm("" : "+v"(yl[i][l]), "+v"(yh[i][l]));
#pragma unroll
        for (int l = 0; l < (U + 7) / 8; l++) asm("" : "+v"(r[l]));
        auto body = [&](const auto &kk) {
            uint64_t x[U];
            if constexpr (A == 1) {
                DevMod m{};
                if (!FAST) m = tb.mods[prime];
#pragma unroll
                for (int l = 0; l < U; l++) x[l] = kk.load_signed(((uint64_t)yh[0][l] << 32) | yl[0][l], m);
                if (big) {
                    const double2 *fb = job.fft + (size_t)poly * (N / 2) + c;
                    const DevMod mp = tb.mods[prime];
#pragma unroll 1
                    for (int l = 0; l < U; l++) {
                        const uint32_t row = r0 + (l << RB);
                        const double2 z = fb[(size_t)(row & (N1 / 2 - 1)) * kRow];
                        const uint64_t t = residue_of_rounded(round(row < N1 / 2 ? z.x : z.y), mp);
#pragma unroll
                        for (int i = 0; i < U; i++) x[i] = i == l ? t : x[i];
                    }
                }
            } else if constexpr (FAST) {
                // A is the table's number of terms. The branch on the rounding stands outside of
                // the words: inside, every word's sums were a block of their own, a serial chain.
                const auto cv = table_ptr(job.conv + ((size_t)g * job.n_out + k) * (A + 1));
                u32x4 w[A + 1];
#pragma unroll
                for (int i = 0; i <= A; i++) w[i] = cv[i];
                auto convert = [&](auto rounded) {
#pragma unroll
                    for (int l = 0; l < U; l++) {
                        ConvAcc acc{0, 0};
#pragma unroll
                        for (int i = 0; i < A; i++) conv_mac(acc, yl[i][l], yh[i][l], w[i]);
                        if (decltype(rounded)::value) {
                            const uint32_t rl = (r[l / 8] >> (4 * (l % 8))) & 15;
                            acc.H += (uint64_t)rl * w[A].x;
                            acc.L += (uint64_t)rl * w[A].y;
                        }
                        x[l] = conv_value(acc, kk.f);
                    }
                };
                if (job.rounded)
                    convert(std::true_type{});
                else
                    convert(std::false_type{});
            }
            const auto col = table_ptr(tb.col + (size_t)prime * kNttCols);
            ct_unit<RA>(x, kk, [&](int e) -> u32x4 { return col[e + 1]; });
            if constexpr (RB == 0) {
#pragma unroll
                for (int l = 0; l < U; l++) __builtin_nontemporal_store(x[l], &out[(size_t)k * N + (size_t)l * kRow]);
            } else {
#pragma unroll
                for (int l = 0; l < U; l++) lds[buf][(r0 + (l << RB)) * C + cl] = x[l];
                __syncthreads();
#pragma unroll
                for (int m = 0; m < UNITS; m++) {
                    const uint32_t u0 = threadIdx.x / C + m * (kThreads / C);
                    uint64_t z[1 << RB];
#pragma unroll
                    for (int l = 0; l < (1 << RB); l++) z[l] = lds[buf][((u0 << RB) + l) * C + cl];
                    ct_unit<RB>(z, kk, [&](int e) -> u32x4 {
                        const int u = e >= 7 ? 3 : e >= 3 ? 2 : e >= 1 ? 1 : 0;
                        return ltw[buf][(((1u << RA) + u0) << u) + (uint32_t)(e - ((1 << u) - 1))];
                    });
#pragma unroll
                    for (int l = 0; l < (1 << RB); l++)
                        __builtin_nontemporal_store(z[l], &out[(size_t)k * N + (size_t)((u0 << RB) + l) * kRow]);
                }
            }
        };
        if constexpr (FAST) {
            body(FoldK<false>(tb, prime));
        } else {
            if (tb.fold[prime].pw)
                body(FoldK<true>(tb, prime));
            else
                body(HarveyK(tb, prime));
        }
        buf ^= 1;
        k = k_next;
    }
}

// LDS word of row word i. Each round's accesses of a unit differ by constants (8 words of a
// lane lie 64, 8 or 1 apart), and lanes a row apart by 8 words fall 9 apart: 32 lanes reach
// 32 banks in every round.
__device__ __forceinline__ int row_slot(int i) { return i + (i >> 3); }

// Orders a wave's own LDS writes before its later reads of them (a wave's LDS accesses
// execute in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Unit words of a lane: round 1 lane + 64 l; round 2 64 (lane / 8) + lane % 8 + 8 l; round 3
// 8 lane + l.
struct RowWords {
    uint64_t *lds;
    int i1, i2, i3;
    __device__ RowWords(uint64_t *l, int lane)
        : lds(l), i1(row_slot(lane)), i2(row_slot(64 * (lane >> 3) + (lane & 7))), i3(9 * lane) {}
    template <int STEP>
    __device__ __forceinline__ void put(int i, const uint64_t *x) const {
#pragma unroll
        for (int l = 0; l < 8; l++) lds[i + STEP * l] = x[l];
    }
    template <int STEP>
    __device__ __forceinline__ void get(int i, uint64_t *x) const {
        wave_lds_order();
#pragma unroll
        for (int l = 0; l < 8; l++) x[l] = lds[i + STEP * l];
        wave_lds_order();
    }
};

// The forward row stages of x (words lane + 64 l); the results are left in LDS.
template <typename K, typename T1, typename T2, typename T3, typename H>
__device__ __forceinline__ void row_forward(const K &k, const RowWords &w, uint64_t (&x)[8], T1 tw1, T2 tw2, T3 tw3,
                                            H before_last) {
    ct_unit<3>(x, k, tw1);
    w.template put<72>(w.i1, x);
    w.template get<9>(w.i2, x);
    ct_unit<3>(x, k, tw2);
    w.template put<9>(w.i2, x);
    before_last();
    w.template get<1>(w.i3, x);
    ct_unit<3>(x, k, tw3);
    w.template put<1>(w.i3, x);
    wave_lds_order();
}

// Row pass: one wave per row of 512 words, 8 words per lane.
template <bool FWD, int IO, typename K>
__device__ __forceinline__ void row_pass(const K &k, uint64_t *lds, uint64_t *base, const u32x4 *w2,
                                         const u32x4 (&w3)[7], uint64_t (&x)[8], uint32_t poly, uint32_t limb,
                                         uint32_t row0, uint32_t n_active, size_t N, int lane, const NttIO &io,
                                         const typename K::Const &qi) {
    const RowWords w(lds, lane);
    auto tw1 = [&](int e) { return w2[e]; };
    auto tw2 = [&](int e) { return w2[8 + 8 * e + (lane >> 3)]; };
    auto tw3 = [&](int e) { return w3[e]; };
    auto pair_of = [&](int j) { return 2 * lane + 128 * j; };  // words i, i + 1
    if constexpr (!FWD) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            lds[row_slot(pair_of(j))] = x[2 * j];
            lds[row_slot(pair_of(j)) + 1] = x[2 * j + 1];
        }
        w.template get<1>(w.i3, x);
        gs_unit<3>(x, k, tw3);
        w.template put<1>(w.i3, x);
        w.template get<9>(w.i2, x);
        gs_unit<3>(x, k, tw2);
        w.template put<9>(w.i2, x);
        w.template get<72>(w.i1, x);
        gs_unit<3>(x, k, tw1);
#pragma unroll
        for (int l = 0; l < 8; l++) base[lane + 64 * l] = x[l];
        return;
    }
    const uint64_t *accp = nullptr;
    uint64_t *out = base;
    if (IO == IO_RESCALE) {
        accp = io.packed ? io.acc_p.p[poly] + (size_t)limb * N + row0
                         : io.acc + ((size_t)poly * io.acc_limbs + limb) * N + row0;
        if (io.packed || io.out_packed) {
            out = io.out_p.p[poly] + (size_t)limb * N + row0;
        } else {
            uint64_t *ob = io.out_single;
            if (io.outs) ob = table_ptr(io.outs)[poly / io.ppo];
            out = ob + ((size_t)(poly % io.ppo) * (io.out_limbs ? io.out_limbs : n_active) + limb) * N + row0;
        }
    }
    // rescale: the accumulator words are loaded before the last round, so they arrive during
    // it; outputs leave in 16-byte pairs
    u64x2 accv[IO == IO_RESCALE ? 4 : 1];
    row_forward(k, w, x, tw1, tw2, tw3, [&] {
        if (IO == IO_RESCALE) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                accv[j] = __builtin_nontemporal_load(global_ptr(reinterpret_cast<const u64x2 *>(accp + pair_of(j))));
        }
    });
    // words that are added on: all requested at once, since a load's wait behind a store of this
    // loop would wait for the store as well
    const bool addto = IO == IO_RESCALE && io.out_packed && poly < 64 && ((io.acc_mask >> poly) & 1);
    u64x2 ov[IO == IO_RESCALE ? 4 : 1];
    if (addto) {
        if (io.add_perm) {
            const auto src = global_ptr(io.add_src.p[poly] + (size_t)limb * N);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const auto at = global_ptr(io.add_perm + row0 + pair_of(j));
                ov[j] = u64x2{src[at[0]], src[at[1]]};
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) ov[j] = *global_ptr(reinterpret_cast<const u64x2 *>(out + pair_of(j)));
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int i = pair_of(j);
        u64x2 y = {lds[row_slot(i)], lds[row_slot(i) + 1]};
        if (IO == IO_RESCALE) {
            const K kh = k.here();
            y.x = kh.sub_mul(accv[j].x, y.x, qi);
            y.y = kh.sub_mul(accv[j].y, y.y, qi);
            if (addto) {
                y.x = add_mod(y.x, ov[j].x, k.q);
                y.y = add_mod(y.y, ov[j].y, k.q);
            }
        } else {
            y.x = k.canon(y.x);
            y.y = k.canon(y.y);
        }
        __builtin_nontemporal_store(y, global_ptr(reinterpret_cast<u64x2 *>(out + i)));
    }
}

// One wave per row and up to `chunk` polynomials of one prime: the row's twiddles are loaded
// once (round 3 into registers, rounds 1 and 2 into LDS), and the next polynomial's words are
// requested before the current one's stages. 118 VGPRs, 4 waves per SIMD: the prefetch and
// the shared twiddles (a row's twiddles are twice its data) gave more than 8 waves did.
// GENERAL launches hold both kinds of arithmetic and run 3 waves per SIMD, in blocks of 256
// threads, three of which fill it: held to 4 waves they spilled 36 to 80 registers (64 x 9 limbs
// of 50 and 60 bits at N = 2^16, forward 415 -> 269 us, inverse 333 -> 266; at N = 2^13 63 -> 38
// and 67 -> 39), and blocks of 512 leave only 2 waves (283, 275, 43 and 44).
// Work order: workgroups are dispatched to the 8 XCDs round-robin, so block
// b runs on XCD b % 8. Each XCD takes a contiguous range of blocks' row indices
// O = (limb * rows + row) * chunks + chunk: the polynomials that share one prime and row
// (hence one run of twiddles) run back to back on the same L2.
template <bool FWD, int IO, bool FAST, int NT>
__global__ __launch_bounds__(NT, FAST ? 4 : 3) void k_ntt_rows(uint64_t *__restrict__ data, LimbMap mp, NttTables tb, int logN,
                                                 NttIO io, uint32_t n_polys, uint32_t per_xcd, uint32_t chunk) {
    __shared__ uint64_t lds[NT / 64][kRowLds];
    const size_t N = size_t(1) << logN;
    const uint32_t rows = (uint32_t)(N / kRow);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t O = ((blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3)) * (NT / 64) + wave;
    if (O >= (n_polys + chunk - 1) / chunk * mp.n_active * rows) return;  // no barrier in this kernel
    const uint32_t chunks = (n_polys + chunk - 1) / chunk;
    const uint32_t ch = O % chunks, rest = O / chunks;
    const uint32_t p0 = ch * chunk, p1 = min(p0 + chunk, n_polys);
    const uint32_t row = rest % rows;
    uint32_t poly0, limb, prime;
    limb_of(mp, rest / rows, poly0, limb, prime);  // limb of the first polynomial
    const uint32_t row0 = row * kRow;
    const u32x4 *tw = tb.row + (size_t)prime * N + row0;
    auto own = [&](uint32_t p) {  // whether this limb is digit p's own
        const uint32_t lo = p % io.digits * io.alpha;
        return limb >= lo && limb < min(lo + io.alpha, mp.Ql);
    };
    auto src_of = [&](uint32_t p) -> const uint64_t * {
        if (IO == IO_DIGITS && io.copy_own && own(p)) return io.acc_p.p[p / io.digits] + (size_t)limb * N + row0;
        return IO == IO_GATHER ? io.acc_p.p[p] + (size_t)limb * N + row0
                               : data + p * mp.poly_stride + (size_t)limb * N + row0;
    };
    auto load = [&](uint64_t (&x)[8], uint32_t p) {
        if (IO == IO_DIGITS && !io.copy_own && own(p)) return;
        if (IO == IO_GATHER && io.perm) {
            const auto src = global_ptr(io.acc_p.p[p] + (size_t)limb * N);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const auto at = global_ptr(io.perm + row0 + 2 * lane + 128 * j);
                x[2 * j] = src[at[0]];
                x[2 * j + 1] = src[at[1]];
            }
            return;
        }
        const uint64_t *ld = src_of(p);
        if constexpr (FWD) {
#pragma unroll
            for (int l = 0; l < 8; l++) x[l] = __builtin_nontemporal_load(global_ptr(ld + lane + 64 * l));
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const u64x2 v = __builtin_nontemporal_load(global_ptr(reinterpret_cast<const u64x2 *>(ld + 2 * lane + 128 * j)));
                x[2 * j] = v.x;
                x[2 * j + 1] = v.y;
            }
        }
    };
    uint64_t x[8], nx[8];
    load(x, p0);
    __shared__ __align__(16) u32x4 lds2[NT / 64][64];
    u32x4 *w2 = lds2[wave];
    u32x4 w3[7];
    w2[lane] = tw[lane];
#pragma unroll
    for (int e = 0; e < 7; e++) w3[e] = tw[64 + 64 * e + lane];
    wave_lds_order();
    auto loop = [&](const auto &k) {
        const auto qi = IO == IO_RESCALE ? k.constant(table_ptr(io.qinv)[prime], table_ptr(io.qinv_s)[prime]) : k.constant(0, 0);
        // the first words and the twiddles are waited for here: in the loop, that wait would take
        // the next polynomial's words along
#pragma unroll
        for (int l = 0; l < 8; l++) asm volatile("" : "+v"(x[l]));
#pragma unroll
        for (int e = 0; e < 7; e++) asm volatile("" : "+v"(w3[e]));
        for (uint32_t p = p0; p < p1; p++) {
            if (p + 1 < p1) load(nx, p + 1);
            uint64_t *base = data + p * mp.poly_stride + (size_t)limb * N + row0;
            if (IO == IO_DIGITS && own(p)) {
                if (io.copy_own)
#pragma unroll
                    for (int l = 0; l < 8; l++) __builtin_nontemporal_store(x[l], base + lane + 64 * l);
            } else {
                row_pass<FWD, IO>(k, lds[wave], base, w2, w3, x, p, limb, row0, mp.n_active, N, lane, io, qi);
            }
            wave_lds_order();
#pragma unroll
            for (int l = 0; l < 8; l++) x[l] = nx[l];
        }
    };
    if constexpr (FAST) {
        loop(FoldK<false>(tb, prime));
    } else {
        if (tb.fold[prime].pw)
            loop(FoldK<true>(tb, prime));
        else
            loop(HarveyK(tb, prime));
    }
}

// Sums of products y a of words y < 2^(b + 1) and canonical a = ah 2^32 + al: y and
// y 2^32 mod p (2^33 delta + 2^(b + 1) < 2^63, folded to 2^53) are split at 26 bits, so a term adds two
// products to each of two sums (H 2^26 + L) and `a` needs no splitting. For a < 2^52 a term adds
// less than 2^59 + 2^47 to H and 2^58 + 2^46 to L: 16 terms fit. Two sums take 4 registers a
// word where 26-bit halves of both factors take 6, which is the third wave per SIMD of
// k_rows_mac: 560 -> 516 us for 128 masked plaintexts, 754 -> 683 us per relinearisation launch
// of a chunk of 8 shared-a refreshes.
struct RowAcc {
    uint64_t H, L;
};
struct RowWord {
    uint32_t h0, l0, h1, l1;
};
__device__ __forceinline__ RowWord row_word(uint64_t y, const FoldMod &f) {
    const uint64_t up = (uint64_t)((uint32_t)y & (2 * f.mask + 1)) << 32;
    const uint32_t hi = __builtin_amdgcn_alignbit((uint32_t)(y >> 32), (uint32_t)y, f.sh + 1);  // y >> (b - 31)
    uint64_t z = (uint64_t)hi * (2 * (uint32_t)f.d) + up;
    const uint32_t zh = (uint32_t)(z >> 32);
    z = (uint64_t)(zh >> f.sh) * (uint32_t)f.d + (((uint64_t)(zh & f.mask) << 32) | (uint32_t)z);
    const Split26 s = split26(y), t = split26(z);
    return RowWord{s.hi, s.lo, t.hi, t.lo};
}
__device__ __forceinline__ void row_mac(RowAcc &a, const RowWord &y, uint64_t x) {
    const uint32_t xl = (uint32_t)x, xh = (uint32_t)(x >> 32);
    a.H += (uint64_t)xl * y.h0;
    a.L += (uint64_t)xl * y.l0;
    a.H += (uint64_t)xh * y.h1;
    a.L += (uint64_t)xh * y.l1;
}
__device__ __forceinline__ uint64_t row_sum(const RowAcc &a, const DevMod &m) { return reduce52(Acc52{a.L, a.H, 0}, m); }

// Row stages fused with the products that consume them (MacJob): a wave takes one row of one
// limb for one group, runs the row stages of each term's polynomial and multiplies its words
// by two operand rows into split sums (RowAcc), so transformed words never reach memory. The
// next term's words and this term's operand rows are requested before the stages. Per wave 8
// KB of twiddles and 4.6 KB of exchange in LDS; 64 registers hold the sums, 3 waves per SIMD.
// Groups of one row are neighbours in launch order, so operand rows that groups share (a
// key's, or the inputs' of a product) come from L2 after the first. Bound by VALU issue where
// groups share operands (540 vector instructions per term and row of 512 words; 128 masked
// plaintexts of 24 limbs in 516 us, about 400 of them issue), by its key's and digits' bytes
// for a single rotation. Against row pass and product kernels apart at N = 2^16: one top-level
// rotation's 66 + 96 us in 95; relinearisations of 16 members, 18 per shared-a chunk, 20.7 ms
// in 12.3; the masked plaintexts 500 + 517 us in 516.
template <bool KEY>
__global__ __launch_bounds__(256, 3) void k_rows_mac(MacJob job, NttTables tb, int logN, uint32_t nQ, uint32_t per_xcd) {
    __shared__ uint64_t lds[4][kRowLds];
    __shared__ __align__(16) u32x4 ltw[4][kRow];
    const size_t N = size_t(1) << logN;
    const uint32_t rows = (uint32_t)(N / kRow);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t O = ((blockIdx.x & 7u) * per_xcd + (blockIdx.x >> 3)) * 4 + wave;
    if (O >= job.groups * job.limbs * rows) return;  // no barrier in this kernel
    const uint32_t e = O % job.groups, rest = O / job.groups, row0 = rest % rows * kRow, limb = rest / rows;
    const uint32_t prime = limb < job.Ql ? limb : nQ + (limb - job.Ql);
    const size_t at = (size_t)limb * N + row0;
    const FoldK<false> k(tb, prime);
    const RowWords w(lds[wave], lane);
    auto pair_of = [&](int j) { return 2 * lane + 128 * j; };
    auto own = [&](uint32_t t) { return KEY && limb < job.Ql && limb / job.alpha == t; };
    auto load = [&](uint64_t (&x)[8], uint32_t t) {
        if (own(t)) return;
        const uint64_t *p = job.data + (size_t)(e * job.ge + t * job.gt) * job.stride + at;
#pragma unroll
        for (int l = 0; l < 8; l++) x[l] = __builtin_nontemporal_load(global_ptr(p + lane + 64 * l));
    };
    uint64_t x[8], nx[8];
    RowAcc acc[2][8];
#pragma unroll
    for (int o = 0; o < 2; o++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[o][j] = RowAcc{0, 0};
    load(x, 0);
    const u32x4 *tw = tb.row + (size_t)prime * N + row0;
#pragma unroll
    for (int j = 0; j < 8; j++) ltw[wave][lane + 64 * j] = tw[lane + 64 * j];
    const u32x4 *lt = ltw[wave];
    u32x4 w1[7];
#pragma unroll
    for (int i = 0; i < 7; i++) {
        w1[i] = table_ptr(tw)[i];
        asm volatile("" : "+s"(w1[i]));  // loaded once
    }
    // the first words are waited for here: in the loop, that wait would take the next term's along
#pragma unroll
    for (int l = 0; l < 8; l++) asm volatile("" : "+v"(x[l]));
    for (uint32_t t = 0; t < job.terms; t++) {
        if (t + 1 < job.terms) load(nx, t + 1);
        const uint64_t *op = KEY ? job.key + (size_t)t * 2 * job.op_stride + (size_t)prime * N + row0 : job.op.p[t] + at;
        u64x2 a[2][4];
#pragma unroll
        for (int o = 0; o < 2; o++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                a[o][j] = *global_ptr(reinterpret_cast<const u64x2 *>(op + o * job.op_stride + pair_of(j)));
        u64x2 y[4];
        if (own(t)) {
            if (job.perm) {
                const auto p = global_ptr(job.op.p[e] + (size_t)limb * N);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const auto i = global_ptr(job.perm + row0 + pair_of(j));
                    y[j] = u64x2{p[i[0]], p[i[1]]};
                }
            } else {
                const uint64_t *p = job.op.p[e] + at;
#pragma unroll
                for (int j = 0; j < 4; j++) y[j] = *global_ptr(reinterpret_cast<const u64x2 *>(p + pair_of(j)));
            }
        } else {
            wave_lds_order();
            row_forward(k, w, x, [&](int i) { return w1[i]; }, [&](int i) { return lt[8 + 8 * i + (lane >> 3)]; },
                        [&](int i) { return lt[64 + 64 * i + lane]; }, [] {});
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = row_slot(pair_of(j));
                y[j] = u64x2{fold_positive(lds[wave][i], k.f), fold_positive(lds[wave][i + 1], k.f)};
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const FoldK<false> kh = k.here();
            const RowWord s0 = row_word(y[j].x, kh.f), s1 = row_word(y[j].y, kh.f);
#pragma unroll
            for (int o = 0; o < 2; o++) {
                row_mac(acc[o][2 * j], s0, a[o][j].x);
                row_mac(acc[o][2 * j + 1], s1, a[o][j].y);
            }
        }
#pragma unroll
        for (int l = 0; l < 8; l++) x[l] = nx[l];
    }
    const DevMod m = tb.mods[prime];
#pragma unroll
    for (int o = 0; o < 2; o++) {
        uint64_t *out = job.out + (size_t)(2 * e + o) * job.out_stride + at;
        const bool add_on = KEY && job.add_on && limb < job.Ql && (o == 0 || !job.perm);
        const uint64_t *add = add_on ? job.add.p[2 * e + o] + (size_t)limb * N : nullptr;
        const uint64_t pm = add_on ? job.pmod[limb] : 0, pms = add_on ? job.pmod_s[limb] : 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const auto at2 = global_ptr(reinterpret_cast<u64x2 *>(out + pair_of(j)));
            u64x2 v = {row_sum(acc[o][2 * j], m), row_sum(acc[o][2 * j + 1], m)};
            if (job.accumulate) {
                const u64x2 c = *at2;
                v = u64x2{add_mod(v.x, c.x, m.q), add_mod(v.y, c.y, m.q)};
            } else if (add_on) {
                u64x2 c;
                if (job.perm) {
                    const auto i = global_ptr(job.perm + row0 + pair_of(j));
                    c = u64x2{global_ptr(add)[i[0]], global_ptr(add)[i[1]]};
                } else {
                    c = *global_ptr(reinterpret_cast<const u64x2 *>(add + row0 + pair_of(j)));
                }
                v = u64x2{add_mod(v.x, mul_shoup(c.x, pm, pms, m.q), m.q), add_mod(v.y, mul_shoup(c.y, pm, pms, m.q), m.q)};
            }
            __builtin_nontemporal_store(v, at2);
        }
    }
}

// optional events around the row pass of the fused rescale (timing of one launch)
hipEvent_t g_rescale_tile_ev[2] = {nullptr, nullptr};

// Probe of the fused last pass (IO_RESCALE row pass of forward NTTs: the ModDown
// combine and the rescale): while on, every eager launch is bracketed by a pair of
// timing events and its algorithmic bytes are recorded.
struct FusedProbe {
    std::mutex mu;
    bool on = false;
    std::vector<hipEvent_t> ev;  // start, stop per launch of the fused last pass
    double bytes = 0.0;
    std::vector<hipEvent_t> ev_plain;  // the same for the plain forward row pass
    double bytes_plain = 0.0;
    size_t last_plain_launches = 0;
    double last_plain_ms = 0.0, last_plain_bytes = 0.0;
} g_probe;

// Whether the limb's prime has a split form, one fold of a word ends below 2q, and an input of
// magnitude `in` plus log N products (and one residue) fit a signed word.
bool forward_fits(const Context &c, uint32_t prime, uint64_t in) {
    const uint64_t q = c.q.at(prime), r = c.fold_bound.at(prime), top = (uint64_t(1) << 63) - 1 - 2 * q;
    return r != 0 && !c.fold_twice.at(prime) && in < top && r <= (top - in) / (uint64_t)c.logN;
}

template <bool FWD, int IOA, int IOB>
void launch_ntt(const Context &c, uint64_t *data, const LimbMap &mp, size_t total_limbs, hipStream_t s,
                const NttIO &io = NttIO{}, bool columns_done = false) {
    if (total_limbs == 0) return;
    if (c.N < (size_t)4096) throw InvalidArgument("NTT requires N >= 4096");
    if (total_limbs % mp.n_active != 0) throw LogicError("NTT limb count is not a multiple of the polynomial size");
    const int logN = c.logN;
    const size_t N = c.N;
    const int stages = logN - 9;                       // of the column pass
    const int unit = stages >= 7 ? 4 : 3;  // of its longest unit
    const uint32_t n_polys = (uint32_t)(total_limbs / mp.n_active);
    NttTables tb{c.mods(),
                 c.d_fold.as<FoldMod>(),
                 FWD ? c.tw_col.as<u32x4>() : c.itw_col.as<u32x4>(),
                 FWD ? c.tw_row.as<u32x4>() : c.itw_row.as<u32x4>(),
                 c.ninv.as<uint64_t>(),
                 c.ninv_s.as<uint64_t>()};
    // FAST when every prime of the launch has a split form and the signed words cannot
    // overflow: forward, input (below 4q, or a residue of another prime of the context, or an
    // encoder's coefficient) plus log N products plus the fused epilogue's operand; inverse,
    // the sums of one unit, which start from products or folded words.
    bool fast = true;
    const uint64_t q_any = *std::max_element(c.q.begin(), c.q.end());
    for (uint32_t j = 0; j < mp.n_active && fast; j++) {
        uint32_t k = mp.lo + j;
        if (k >= mp.skip_lo) k += mp.skip_width;
        const uint32_t prime = k < mp.Ql ? mp.first_prime + k : mp.nQ + (k - mp.Ql);
        const uint64_t q = c.q.at(prime), r = c.fold_bound.at(prime);
        if (FWD)
            fast = forward_fits(c, prime, IOA == IO_REDUCE ? std::max(q_any, 4 * q) : 4 * q);
        else
            fast = r != 0 && !c.fold_twice.at(prime) && r < (uint64_t(1) << (63 - std::max(unit, 3)));
    }
    // the row pass moves its words in 16-byte pairs (outs are ciphertext buffers of the pool)
    bool aligned = ((uintptr_t)data & 15) == 0 && mp.poly_stride % 2 == 0;
    if (IOB == IO_GATHER)
        for (uint32_t p = 0; p < n_polys; p++) aligned = aligned && ((uintptr_t)io.acc_p.p[p] & 15) == 0;
    if (IOB == IO_RESCALE) {
        aligned = aligned && (((uintptr_t)io.acc | (uintptr_t)io.out_single) & 15) == 0;
        for (uint32_t p = 0; p < n_polys && (io.packed || io.out_packed); p++)
            aligned = aligned && (((uintptr_t)io.out_p.p[p] | (io.packed ? (uintptr_t)io.acc_p.p[p] : 0)) & 15) == 0;
    }
    if (!aligned) throw InvalidArgument("NTT operands must be 16-byte aligned");
    const int row_threads = fast ? ks_tuning().ntt_tile_threads : 256;
    // up to 4 polynomials per wave share a row's twiddles in registers and prefetch each
    // other's words, while 8192 waves (8 per SIMD) remain: the plain forward pass of a
    // shared-a chunk's launches 96 -> 75 us (8 polynomials measured the same)
    uint32_t chunk = 1;
    while (chunk < 4 && chunk < n_polys &&
           (size_t)((n_polys + 2 * chunk - 1) / (2 * chunk)) * mp.n_active * (N / kRow) >= 8192)
        chunk *= 2;
    const size_t row_waves = (size_t)((n_polys + chunk - 1) / chunk) * mp.n_active * (N / kRow);
    const uint32_t per_xcd = (uint32_t)((row_waves + row_threads / 64 * 8 - 1) / (row_threads / 64 * 8));
    auto cols = [&]() {
#define SHM_COLS(S, RA, RB)                                                                                 \
    case S: {                                                                                               \
        const size_t grid = total_limbs * (kRow / col_width(RA, RB));                                       \
        if (grid * kThreads >> 32) throw LogicError("NTT beyond the threads of one launch");                \
        if (fast)                                                                                           \
            k_ntt_cols<RA, RB, FWD, IOA, true><<<(unsigned)grid, kThreads, 0, s>>>(data, mp, tb, logN, io); \
        else                                                                                                \
            k_ntt_cols<RA, RB, FWD, IOA, false><<<(unsigned)grid, kThreads, 0, s>>>(data, mp, tb, logN, io);\
        break;                                                                                              \
    }
        switch (stages) {
            SHM_COLS(3, 3, 0)
            SHM_COLS(4, 2, 2)
            SHM_COLS(5, 3, 2)
            SHM_COLS(6, 3, 3)
            SHM_COLS(7, 4, 3)
            SHM_COLS(8, 4, 4)
            default: throw InvalidArgument("unsupported ring degree for NTT");
        }
#undef SHM_COLS
    };
    auto rows = [&]() {
#define SHM_ROWS(F, NT) k_ntt_rows<FWD, IOB, F, NT><<<8u * per_xcd, NT, 0, s>>>(data, mp, tb, logN, io, n_polys, per_xcd, chunk)
        if (fast && row_threads == 512)
            SHM_ROWS(true, 512);
        else if (fast)
            SHM_ROWS(true, 256);
        else
            SHM_ROWS(false, 256);
#undef SHM_ROWS
    };
    if (FWD) {
        if (!columns_done) cols();
        const bool timed = IOB == IO_RESCALE && g_rescale_tile_ev[0] && g_rescale_tile_ev[1];
        if (timed) SHM_HIP(hipEventRecord(g_rescale_tile_ev[0], s));
        hipEvent_t pe[2] = {nullptr, nullptr};
        if (IOB == IO_PLAIN || IOB == IO_DIGITS) {
            std::lock_guard<std::mutex> lk(g_probe.mu);
            hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
            if (g_probe.on && hipStreamIsCapturing(s, &cs) == hipSuccess && cs == hipStreamCaptureStatusNone) {
                SHM_HIP(hipEventCreate(&pe[0]));
                SHM_HIP(hipEventCreate(&pe[1]));
                g_probe.ev_plain.push_back(pe[0]);
                g_probe.ev_plain.push_back(pe[1]);
                // the transform's algorithmic bytes: every limb read and written once (not the
                // digits' own limbs where they are neither)
                const size_t own = IOB == IO_DIGITS && !io.copy_own ? n_polys / io.digits * (size_t)mp.Ql : 0;
                g_probe.bytes_plain += 16.0 * N * (total_limbs - own);
            }
        }
        if (IOB == IO_RESCALE) {
            std::lock_guard<std::mutex> lk(g_probe.mu);
            hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
            if (g_probe.on && hipStreamIsCapturing(s, &cs) == hipSuccess && cs == hipStreamCaptureStatusNone) {
                SHM_HIP(hipEventCreate(&pe[0]));
                SHM_HIP(hipEventCreate(&pe[1]));
                g_probe.ev.push_back(pe[0]);
                g_probe.ev.push_back(pe[1]);
                // per output limb: the result written and the combined operand read
                // (plus the output read where the pass accumulates onto it); the
                // transform's intermediate written by the column pass is not counted
                size_t acc_polys = 0;
                if (io.out_packed)
                    for (uint32_t p = 0; p < n_polys && p < 64; p++) acc_polys += (io.acc_mask >> p) & 1;
                g_probe.bytes += 16.0 * N * total_limbs + 8.0 * N * mp.n_active * acc_polys;
            }
        }
        if (pe[0]) SHM_HIP(hipEventRecord(pe[0], s));
        rows();
        if (pe[1]) SHM_HIP(hipEventRecord(pe[1], s));
        if (timed) SHM_HIP(hipEventRecord(g_rescale_tile_ev[1], s));
    } else {
        rows();
        cols();
    }
    SHM_HIP(hipGetLastError());
}

// One thread per twiddle i = 1 .. N - 1 of prime blockIdx.y.
__global__ void k_ntt_tables(const uint64_t *__restrict__ tw, const DevMod *__restrict__ mods,
                             const FoldMod *__restrict__ fold, u32x4 *__restrict__ col, u32x4 *__restrict__ row,
                             uint32_t N) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, p = blockIdx.y;
    if (i == 0 || i >= N) return;
    const DevMod m = mods[p];
    const FoldMod f = fold[p];
    const uint64_t w = tw[(size_t)p * N + i], ws = shoup_companion(w, m);
    const u32x4 e = f.pw ? fold_split(w, ws, m.q, f)
                         : u32x4{(uint32_t)w, (uint32_t)(w >> 32), (uint32_t)ws, (uint32_t)(ws >> 32)};
    const uint32_t rows = N / kRow;
    if (i < rows) {
        col[(size_t)p * kNttCols + i] = e;
        return;
    }
    // row stage j = 3 round + u has rows 2^j groups: group `loc` of its row, of which unit
    // loc >> u holds entry 2^u - 1 + (loc mod 2^u)
    const int j = (31 - __clz(i)) - (31 - __clz(rows)), r = j / 3, u = j % 3;
    const uint32_t g = i - (rows << j), loc = g & ((1u << j) - 1);
    const uint32_t en = (1u << u) - 1 + (loc & ((1u << u) - 1)), un = loc >> u;
    const uint32_t at = r == 0 ? en : r == 1 ? 8 + 8 * en + un : 64 + 64 * en + un;
    row[(size_t)p * N + (size_t)(g >> j) * kRow + at] = e;
}

}  // namespace

void ntt_make_tables(const Context &c, const uint64_t *tw, DevBuf &col, DevBuf &row) {
    const size_t QP = c.nQP();
    col.alloc(QP * kNttCols * sizeof(u32x4));
    row.alloc(QP * c.N * sizeof(u32x4));
    if (c.N < 4096) return;  // the transforms refuse such rings
    k_ntt_tables<<<dim3((unsigned)((c.N + 255) / 256), (unsigned)QP), 256>>>(
        tw, c.mods(), c.d_fold.as<FoldMod>(), col.as<u32x4>(), row.as<u32x4>(), (uint32_t)c.N);
    SHM_HIP(hipGetLastError());
}

// Any number of polynomials, in launches of up to 2^33 words (64 GB): the column pass has a
// thread per 4 words of a ring of 2^13 and per 8 of the others, and of 2^32 threads and more a
// launch runs the remainder modulo 2^32, with no error.
template <bool FWD>
static void ntt_polys(const Context &c, uint64_t *data, size_t n_polys, size_t n_limbs, size_t first_prime,
                      hipStream_t s) {
    if (n_limbs == 0) return;
    LimbMap mp{(uint32_t)n_limbs, 0, 0xffffffffu, 0, 0xffffffffu, (uint32_t)c.nQ, (uint32_t)first_prime,
               (uint64_t)n_limbs * c.N};
    const size_t step = std::max<size_t>(1, (size_t(1) << 33) / (n_limbs * c.N));
    for (size_t p = 0; p < n_polys; p += step)
        launch_ntt<FWD, IO_PLAIN, IO_PLAIN>(c, data + p * n_limbs * c.N, mp, std::min(step, n_polys - p) * n_limbs, s);
}

void ntt_forward(const Context &c, uint64_t *data, size_t n_polys, size_t n_limbs, size_t first_prime,
                 hipStream_t s) {
    ntt_polys<true>(c, data, n_polys, n_limbs, first_prime, s);
}

void probe_fused_ntt_begin() {
    std::lock_guard<std::mutex> lk(g_probe.mu);
    for (hipEvent_t e : g_probe.ev) (void)hipEventDestroy(e);
    for (hipEvent_t e : g_probe.ev_plain) (void)hipEventDestroy(e);
    g_probe.ev.clear();
    g_probe.ev_plain.clear();
    g_probe.bytes = 0.0;
    g_probe.bytes_plain = 0.0;
    g_probe.on = true;
}

void probe_fused_ntt_end(size_t *launches, double *ms, double *bytes) {
    SHM_HIP(hipDeviceSynchronize());
    std::lock_guard<std::mutex> lk(g_probe.mu);
    g_probe.on = false;
    double total = 0.0;
    for (size_t i = 0; i + 1 < g_probe.ev.size(); i += 2) {
        float t = 0.0f;
        SHM_HIP(hipEventElapsedTime(&t, g_probe.ev[i], g_probe.ev[i + 1]));
        total += t;
    }
    if (launches) *launches = g_probe.ev.size() / 2;
    if (ms) *ms = total;
    if (bytes) *bytes = g_probe.bytes;
    for (hipEvent_t e : g_probe.ev) (void)hipEventDestroy(e);
    g_probe.ev.clear();
    double tp = 0.0;
    for (size_t i = 0; i + 1 < g_probe.ev_plain.size(); i += 2) {
        float t = 0.0f;
        SHM_HIP(hipEventElapsedTime(&t, g_probe.ev_plain[i], g_probe.ev_plain[i + 1]));
        tp += t;
    }
    g_probe.last_plain_launches = g_probe.ev_plain.size() / 2;
    g_probe.last_plain_ms = tp;
    g_probe.last_plain_bytes = g_probe.bytes_plain;
    for (hipEvent_t e : g_probe.ev_plain) (void)hipEventDestroy(e);
    g_probe.ev_plain.clear();
}

void probe_plain_ntt_last(size_t *launches, double *ms, double *bytes) {
    std::lock_guard<std::mutex> lk(g_probe.mu);
    if (launches) *launches = g_probe.last_plain_launches;
    if (ms) *ms = g_probe.last_plain_ms;
    if (bytes) *bytes = g_probe.last_plain_bytes;
}

void set_rescale_tile_events(hipEvent_t start, hipEvent_t stop) {
    g_rescale_tile_ev[0] = start;
    g_rescale_tile_ev[1] = stop;
}

void ntt_encoded_columns(const Context &c, const double2 *fft, uint64_t *out, size_t n_polys, size_t n_limbs,
                         hipStream_t s) {
    ConvertJob job{};
    job.fft = fft;
    job.alpha = job.total = job.digits = 1;
    job.members = (uint32_t)n_polys;
    job.out = out;
    job.out_stride = n_limbs * c.N;
    job.n_out = job.Ql = (uint32_t)n_limbs;
    convert_cols(c, job, s);
}

void ntt_forward_encoded(const Context &c, const double2 *fft, uint64_t *out, size_t n_polys, size_t n_limbs,
                         hipStream_t s) {
    ntt_encoded_columns(c, fft, out, n_polys, n_limbs, s);
    LimbMap mp{(uint32_t)n_limbs, 0, 0xffffffffu, 0, 0xffffffffu, (uint32_t)c.nQ, 0, (uint64_t)n_limbs * c.N};
    launch_ntt<true, IO_PLAIN, IO_PLAIN>(c, out, mp, n_polys * n_limbs, s, NttIO{}, true);
}

bool rows_mac_covers(const Context &c, size_t n_data, bool special, size_t terms) {
    if (terms == 0 || terms > 16) return false;
    for (size_t p = 0; p < n_data + (special ? c.nP : 0); p++) {
        const uint32_t prime = (uint32_t)(p < n_data ? p : c.nQ + (p - n_data));
        const uint64_t q = c.q.at(prime);
        if (!(q > (uint64_t(1) << 45) && q < (uint64_t(1) << 52)) || !forward_fits(c, prime, uint64_t(1) << 61)) return false;
    }
    return true;
}

void rows_mac(const Context &c, const MacJob &job, hipStream_t s) {
    NttTables tb{c.mods(), c.d_fold.as<FoldMod>(), nullptr, c.tw_row.as<u32x4>(), nullptr, nullptr};
    const size_t waves = (size_t)job.groups * job.limbs * (c.N / kRow);
    const uint32_t per_xcd = (uint32_t)((waves + 31) / 32);
    if (job.key)
        k_rows_mac<true><<<8u * per_xcd, 256, 0, s>>>(job, tb, c.logN, (uint32_t)c.nQ, per_xcd);
    else
        k_rows_mac<false><<<8u * per_xcd, 256, 0, s>>>(job, tb, c.logN, (uint32_t)c.nQ, per_xcd);
    SHM_HIP(hipGetLastError());
}

void ntt_inverse(const Context &c, uint64_t *data, size_t n_polys, size_t n_limbs, size_t first_prime,
                 hipStream_t s) {
    ntt_polys<false>(c, data, n_polys, n_limbs, first_prime, s);
}

void ntt_inverse_gather(const Context &c, const PolyPack &in, uint64_t *out, size_t n_polys, size_t n_limbs,
                        size_t first_prime, hipStream_t s) {
    if (n_polys == 0) return;
    if (n_polys > (size_t)kPolyPack) throw InvalidArgument("inverse NTT: 1..64 polynomials per batch");
    LimbMap mp{(uint32_t)n_limbs, 0, 0xffffffffu, 0, 0xffffffffu, (uint32_t)c.nQ, (uint32_t)first_prime,
               (uint64_t)n_limbs * c.N};
    NttIO io{};
    io.acc_p = in;
    launch_ntt<false, IO_PLAIN, IO_GATHER>(c, out, mp, n_polys * n_limbs, s, io);
}

void ntt_forward_qlp(const Context &c, uint64_t *data, size_t Ql, size_t lo, size_t hi, size_t skip_lo,
                     size_t skip_hi, size_t n_polys, size_t poly_stride, hipStream_t s) {
    size_t active = hi - lo;
    uint32_t sl = 0xffffffffu, sw = 0;
    if (skip_hi > skip_lo && skip_lo >= lo && skip_hi <= hi) {
        active -= skip_hi - skip_lo;
        sl = (uint32_t)skip_lo;
        sw = (uint32_t)(skip_hi - skip_lo);
    }
    LimbMap mp{(uint32_t)active, (uint32_t)lo, sl, sw, (uint32_t)Ql, (uint32_t)c.nQ, 0, (uint64_t)poly_stride};
    launch_ntt<true, IO_PLAIN, IO_PLAIN>(c, data, mp, n_polys * active, s);
}

void ntt_inverse_qlp(const Context &c, uint64_t *data, size_t Ql, size_t lo, size_t hi, size_t n_polys,
                     size_t poly_stride, hipStream_t s) {
    LimbMap mp{(uint32_t)(hi - lo), (uint32_t)lo, 0xffffffffu, 0, (uint32_t)Ql, (uint32_t)c.nQ, 0,
               (uint64_t)poly_stride};
    launch_ntt<false, IO_PLAIN, IO_PLAIN>(c, data, mp, n_polys * (hi - lo), s);
}

void rescale_ntt_fused(const Context &c, const uint64_t *last, const uint64_t *acc, size_t acc_limbs,
                       uint64_t *delta, uint64_t *const *outs, uint64_t *out_single, size_t ppo, size_t n_polys,
                       size_t L1, const uint64_t *qinv, const uint64_t *qinv_s, hipStream_t s, bool rounded) {
    LimbMap mp{(uint32_t)L1, 0, 0xffffffffu, 0, 0xffffffffu, (uint32_t)c.nQ, 0, (uint64_t)L1 * c.N};
    NttIO io{};
    io.src = last;
    io.acc = acc;
    io.outs = outs;
    io.out_single = out_single;
    io.qinv = qinv;
    io.qinv_s = qinv_s;
    io.acc_limbs = (uint32_t)acc_limbs;
    io.ppo = (uint32_t)ppo;
    io.center = rounded ? (c.q[L1] >> 1) : 0;
    launch_ntt<true, IO_REDUCE, IO_RESCALE>(c, delta, mp, n_polys * L1, s, io);
}

void rescale_ntt_fused_window(const Context &c, const uint64_t *last, const uint64_t *acc, size_t acc_limbs,
                              uint64_t *delta, uint64_t *const *outs, size_t ppo, size_t n_polys, size_t L1,
                              size_t lo, size_t n, const uint64_t *qinv, const uint64_t *qinv_s, hipStream_t s) {
    if (lo + n > L1 || n == 0) throw InvalidArgument("rescale window outside the output limbs");
    LimbMap mp{(uint32_t)n, (uint32_t)lo, 0xffffffffu, 0, 0xffffffffu, (uint32_t)c.nQ, 0, (uint64_t)L1 * c.N};
    NttIO io{};
    io.src = last;
    io.acc = acc;
    io.outs = outs;
    io.qinv = qinv;
    io.qinv_s = qinv_s;
    io.acc_limbs = (uint32_t)acc_limbs;
    io.ppo = (uint32_t)ppo;
    io.out_limbs = (uint32_t)L1;
    launch_ntt<true, IO_REDUCE, IO_RESCALE>(c, delta, mp, n_polys * n, s, io);
}

void moddown_ntt_fused(const Context &c, uint64_t *delta, const uint64_t *cx, size_t Ql, size_t cx_limbs,
                       const PolyPack &out, size_t n_polys, uint64_t acc_mask, const uint64_t *pinv,
                       const uint64_t *pinv_s, hipStream_t s, const PolyPack *add_src, const uint32_t *add_perm,
                       bool columns_done) {
    if (n_polys == 0 || n_polys > (size_t)kPolyPack) throw InvalidArgument("ModDown: 1..64 polynomials per batch");
    if ((add_src == nullptr) != (add_perm == nullptr)) throw LogicError("ModDown: permuted addend needs both parts");
    LimbMap mp{(uint32_t)Ql, 0, 0xffffffffu, 0, 0xffffffffu, (uint32_t)c.nQ, 0, (uint64_t)Ql * c.N};
    NttIO io{};
    io.acc = cx;
    io.acc_limbs = (uint32_t)cx_limbs;
    io.qinv = pinv;
    io.qinv_s = pinv_s;
    io.out_packed = 1;
    io.acc_mask = acc_mask;
    io.out_p = out;
    if (add_src) {
        io.add_src = *add_src;
        io.add_perm = add_perm;
    }
    launch_ntt<true, IO_PLAIN, IO_RESCALE>(c, delta, mp, n_polys * Ql, s, io, columns_done);
}

bool convert_covers(const Context &c, size_t terms) { return terms == 1 || (c.conv_ok && terms <= 6); }

void convert_cols(const Context &c, const ConvertJob &job, hipStream_t s) {
    if (!convert_covers(c, job.alpha)) throw LogicError("conversion outside the fused form");
    const int logN = c.logN, stages = logN - 9;
    NttTables tb{c.mods(), c.d_fold.as<FoldMod>(), c.tw_col.as<u32x4>(), nullptr, nullptr, nullptr};
    const unsigned polys = job.members * job.digits;
    // one source word: below 2^61 (2^60 from the encoder), and its transform fits or GENERAL
    // kernels fold; more: conv_ok
    bool fast = true;
    for (uint32_t k = 0; k < job.n_out && job.alpha == 1 && fast; k++)
        fast = forward_fits(c, k < job.Ql ? k : (uint32_t)c.nQ + (k - job.Ql), uint64_t(1) << (job.fft ? 60 : 61));
    auto launch = [&](auto fn, int width) {
        const unsigned blocks = (unsigned)(kRow / width) * polys;
        // a run of output limbs per block, shorter (but at least 4) where that leaves fewer
        // than 6 blocks a CU: every run reads the digit's source words again
        unsigned runs = std::max(1u, std::min((1536u + blocks - 1) / blocks, (job.n_out + 3) / 4));
        const unsigned run = (job.n_out + runs - 1) / runs;
        runs = (job.n_out + run - 1) / run;
        fn<<<dim3(kRow / width, polys, runs), kThreads, 0, s>>>(job, tb, logN, (uint32_t)c.nQ, run);
    };
#define SHM_CONV_A(RA, RB)                                                                                   \
    if (job.alpha == 1 && !fast)                                                                             \
        launch(k_convert_cols<RA, RB, 1, false>, col_width(RA, RB));                                         \
    else if (job.alpha == 1)                                                                                 \
        launch(k_convert_cols<RA, RB, 1, true>, col_width(RA, RB));                                          \
    else if (job.alpha == 2)                                                                                 \
        launch(k_convert_cols<RA, RB, 2, true>, col_width(RA, RB));                                          \
    else if (job.alpha == 3)                                                                                 \
        launch(k_convert_cols<RA, RB, 3, true>, col_width(RA, RB));                                          \
    else if (job.alpha == 4)                                                                                 \
        launch(k_convert_cols<RA, RB, 4, true>, col_width(RA, RB));                                          \
    else if (job.alpha == 5)                                                                                 \
        launch(k_convert_cols<RA, RB, 5, true>, col_width(RA, RB));                                          \
    else                                                                                                     \
        launch(k_convert_cols<RA, RB, 6, true>, col_width(RA, RB));                                          \
    break;
    switch (stages) {
        case 3: SHM_CONV_A(3, 0)
        case 4: SHM_CONV_A(2, 2)
        case 5: SHM_CONV_A(3, 2)
        case 6: SHM_CONV_A(3, 3)
        case 7: SHM_CONV_A(4, 3)
        case 8: SHM_CONV_A(4, 4)
        default: throw InvalidArgument("unsupported ring degree for NTT");
    }
#undef SHM_CONV_A
    SHM_HIP(hipGetLastError());
}

void ntt_rows_digits(const Context &c, uint64_t *d, size_t Ql, size_t beta, size_t members, const PolyPack &own,
                     bool copy_own, hipStream_t s) {
    const size_t QlP = Ql + c.nP;
    LimbMap mp{(uint32_t)QlP, 0, 0xffffffffu, 0, (uint32_t)Ql, (uint32_t)c.nQ, 0, (uint64_t)QlP * c.N};
    NttIO io{};
    io.acc_p = own;
    io.digits = (uint32_t)beta;
    io.alpha = (uint32_t)c.nP;
    io.copy_own = copy_own ? 1 : 0;
    launch_ntt<true, IO_PLAIN, IO_DIGITS>(c, d, mp, members * beta * QlP, s, io, true);
}

void ntt_inverse_gather_scaled(const Context &c, const PolyPack &in, uint64_t *out, size_t n_polys, size_t n_limbs,
                               const uint64_t *scale, const uint64_t *scale_s, hipStream_t s, const uint32_t *perm) {
    if (n_polys == 0) return;
    if (n_polys > (size_t)kPolyPack) throw InvalidArgument("inverse NTT: 1..64 polynomials per batch");
    LimbMap mp{(uint32_t)n_limbs, 0, 0xffffffffu, 0, 0xffffffffu, (uint32_t)c.nQ, 0, (uint64_t)n_limbs * c.N};
    NttIO io{};
    io.acc_p = in;
    io.perm = perm;
    io.scale = scale;
    io.scale_s = scale_s;
    launch_ntt<false, IO_PLAIN, IO_GATHER>(c, out, mp, n_polys * n_limbs, s, io);
}

void ntt_inverse_qlp_scaled(const Context &c, uint64_t *data, size_t Ql, size_t lo, size_t hi, size_t n_polys,
                            size_t poly_stride, const uint64_t *scale, const uint64_t *scale_s, hipStream_t s) {
    LimbMap mp{(uint32_t)(hi - lo), (uint32_t)lo, 0xffffffffu, 0, (uint32_t)Ql, (uint32_t)c.nQ, 0,
               (uint64_t)poly_stride};
    NttIO io{};
    io.scale = scale;
    io.scale_s = scale_s;
    io.scale_lo = (uint32_t)lo;
    launch_ntt<false, IO_PLAIN, IO_PLAIN>(c, data, mp, n_polys * (hi - lo), s, io);
}

void rescale_ntt_fused_pack(const Context &c, const uint64_t *last, const PolyPack &in, const PolyPack &out,
                            uint64_t *delta, size_t n_polys, size_t L1, const uint64_t *qinv, const uint64_t *qinv_s,
                            hipStream_t s, bool rounded) {
    if (n_polys == 0 || n_polys > (size_t)kPolyPack) throw InvalidArgument("rescale: 1..64 polynomials per batch");
    LimbMap mp{(uint32_t)L1, 0, 0xffffffffu, 0, 0xffffffffu, (uint32_t)c.nQ, 0, (uint64_t)L1 * c.N};
    NttIO io{};
    io.src = last;
    io.qinv = qinv;
    io.qinv_s = qinv_s;
    io.center = rounded ? (c.q[L1] >> 1) : 0;
    io.packed = 1;
    io.acc_p = in;
    io.out_p = out;
    launch_ntt<true, IO_REDUCE, IO_RESCALE>(c, delta, mp, n_polys * L1, s, io);
}

}  // namespace shm
