// CKKS canonical-embedding encoder/decoder (FP64), on device.
//
// Encode (ckks.cu:89-170): bit-reverse the slot vector, special inverse FFT
// (fft.cu:226-356, Gentleman-Sande stages with twiddle roots[M - psiIdx]) with
// the last stage scaled by scale/n, round half away from zero, reduce per
// prime (negative v -> q - (|v| mod q)), place coefficient ci at ci*N/(2n),
// then NTT. Decode (ckks.cu:172-246) is iNTT, CRT composition to a centred
// multi-precision integer, conversion to double by 64-bit words, the forward
// special FFT (fft.cu:88-224) and a bit reversal.
//
// This file is compiled with -ffp-contract=off: every product and sum is
// rounded separately, in the operation order written here.
#include <cmath>

#include "engine.h"

namespace shm {

namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(size_t work) {
    size_t g = (work + kBlock - 1) / kBlock;
    if (g > (1u << 20)) g = 1u << 20;
    return (unsigned)(g ? g : 1);
}

__device__ __forceinline__ uint32_t brv_bits(uint32_t x, int bits) { return bits ? (__brev(x) >> (32 - bits)) : 0; }

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    const double t0 = a.x * b.x;
    const double t1 = a.y * b.y;
    const double t2 = a.x * b.y;
    const double t3 = a.y * b.x;
    return make_double2(t0 - t1, t2 + t3);
}

// Twiddles of both special FFTs by stage: entry m + k, m = n / (2 pairs) groups, is group k's.
__global__ void k_fft_tables(const double2 *roots, const uint32_t *group, double2 *fwd, double2 *inv, uint32_t n,
                             int logn, int logRatio, uint32_t M) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0 || i >= n) return;
    const int logm = 31 - __clz(i), logPairs = logn - 1 - logm;
    const uint32_t k = i - (1u << logm);
    const uint32_t bk = logn > 1 ? brv_bits(k << logPairs, logn - 1) : 0;
    const uint32_t idx = (uint32_t)(((uint64_t)group[bk] << (logPairs + logRatio)) & (M - 1));
    fwd[i] = roots[idx];
    inv[i] = roots[M - idx];
}

// The special FFTs (forward: Cooley-Tukey from the widest pairs; inverse: Gentleman-Sande
// from adjacent ones) of n = 2^logn complex words run as two passes, like the NTT: rows of
// 512 contiguous words, one wave each, three rounds of radix-8 units in registers with
// exchanges through LDS words of the wave's own; and columns of n / 512 words, 512 apart, in
// at most two rounds of register units. Each butterfly is the one of a stage-by-stage
// transform on the same operands, so the results are the same bits. One launch per stage
// moved the vector through memory 15 times at N = 2^16: 128 vectors took 237 us, now 38 us;
// one vector's 15 launches took 37 (inverse) and 69 us (forward) of kernel time.
constexpr int kFftRow = 512;

template <bool FWD>
__device__ __forceinline__ void fft_pair(double2 &a, double2 &b, double2 w) {
    if (FWD) {
        const double2 t = cmul(b, w), s = a;
        a = make_double2(s.x + t.x, s.y + t.y);
        b = make_double2(s.x - t.x, s.y - t.y);
    } else {
        const double2 d = make_double2(a.x - b.x, a.y - b.y);
        a = make_double2(a.x + b.x, a.y + b.y);
        b = cmul(d, w);
    }
}

// R stages on the words i0 + l 2^lp, l < 2^R (bits lp .. lp + R - 1 of i0 are zero).
template <int R, bool FWD>
__device__ __forceinline__ void fft_unit(double2 *z, uint32_t i0, int lp, const double2 *__restrict__ tw, uint32_t n) {
#pragma unroll
    for (int v = 0; v < R; v++) {
        const int u = FWD ? R - 1 - v : v, h = 1 << u;
        const double2 *t = tw + (n >> (lp + u + 1)) + (i0 >> (lp + u + 1));
#pragma unroll
        for (int l = 0; l < (1 << R); l++)
            if ((l & h) == 0) fft_pair<FWD>(z[l], z[l + h], t[l >> (u + 1)]);
    }
}

// Where a row's words come from or go to besides buf: bit-reversed slot values.
enum { FFT_BUF = 0, FFT_VALUES = 1, FFT_MASK = 2 };
struct FftIO {
    const double *re, *im;   // FFT_VALUES, inverse: slot values (im may be null), nv of them, then zeros
    size_t nv;
    const double *w;         // FFT_MASK: value of vector b where mask[slot] is set, else 0
    const uint8_t *mask;
    double *out_re, *out_im; // FFT_VALUES, forward
};

__device__ __forceinline__ int fft_slot(int i) { return i + (i >> 3); }
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <bool FWD, int IO>
__global__ __launch_bounds__(64) void k_fft_rows(double2 *buf_all, const double2 *__restrict__ tw, uint32_t n, int logn,
                                                 FftIO io) {
    __shared__ double2 lds[kFftRow / 8 * 9];
    const int lane = threadIdx.x;
    const uint32_t base = blockIdx.x * kFftRow;
    double2 *buf = buf_all + (size_t)blockIdx.y * n;
    // unit words of a lane: adjacent (lp 0), 8 apart (lp 3), 64 apart (lp 6)
    const int i0 = 8 * lane, i3 = 64 * (lane >> 3) + (lane & 7), i6 = lane;
    auto put = [&](const double2 *z, int i, int step) {
#pragma unroll
        for (int l = 0; l < 8; l++) lds[fft_slot(i) + l * step] = z[l];
    };
    auto get = [&](double2 *z, int i, int step) {
        wave_order();
#pragma unroll
        for (int l = 0; l < 8; l++) z[l] = lds[fft_slot(i) + l * step];
        wave_order();
    };
    double2 z[8];
#pragma unroll
    for (int l = 0; l < 8; l++) {
        const uint32_t i = base + lane + 64 * l;
        if (!FWD && IO == FFT_VALUES) {
            const uint32_t t = brv_bits(i, logn);
            z[l] = t < io.nv ? make_double2(io.re[t], io.im ? io.im[t] : 0.0) : make_double2(0.0, 0.0);
        } else if (!FWD && IO == FFT_MASK) {
            z[l] = make_double2(io.mask[brv_bits(i, logn)] ? io.w[blockIdx.y] : 0.0, 0.0);
        } else {
            z[l] = buf[i];
        }
    }
    if (FWD) {
        fft_unit<3, true>(z, base + i6, 6, tw, n);
        put(z, i6, 72);
        get(z, i3, 9);
        fft_unit<3, true>(z, base + i3, 3, tw, n);
        put(z, i3, 9);
        get(z, i0, 1);
        fft_unit<3, true>(z, base + i0, 0, tw, n);
        put(z, i0, 1);
        get(z, i6, 72);
    } else {
        put(z, i6, 72);
        get(z, i0, 1);
        fft_unit<3, false>(z, base + i0, 0, tw, n);
        put(z, i0, 1);
        get(z, i3, 9);
        fft_unit<3, false>(z, base + i3, 3, tw, n);
        put(z, i3, 9);
        get(z, i6, 72);
        fft_unit<3, false>(z, base + i6, 6, tw, n);
    }
#pragma unroll
    for (int l = 0; l < 8; l++) {
        const uint32_t i = base + lane + 64 * l;
        if (FWD && IO == FFT_VALUES) {
            const uint32_t t = brv_bits(i, logn);
            io.out_re[t] = z[l].x;
            io.out_im[t] = z[l].y;
        } else {
            buf[i] = z[l];
        }
    }
}

// RA + RB = logn - 9 column stages; inverse: the last scales its outputs by the vector's factor.
template <int RA, int RB, bool FWD>
__global__ __launch_bounds__(kBlock) void k_fft_cols(double2 *buf_all, const double2 *__restrict__ tw, uint32_t n,
                                                     const double *fix, double fix1) {
    constexpr int C = kBlock >> RB, U = 1 << RA, V = 1 << RB, UNITS = (C << RA) / kBlock;
    __shared__ double2 lds[RB == 0 ? 1 : C << (RA + RB)];
    const uint32_t cl = threadIdx.x % C, c = blockIdx.x * C + cl, r0 = threadIdx.x / C;
    double2 *buf = buf_all + (size_t)blockIdx.y * n;
    double2 z[U];
    auto wide = [&]() { fft_unit<RA, FWD>(z, r0 * kFftRow + c, 9 + RB, tw, n); };  // rows r0 + l 2^RB
    auto narrow = [&](auto load, auto store) {                                       // rows g 2^RB + l
        if constexpr (RB > 0) {
#pragma unroll
            for (int m = 0; m < UNITS; m++) {
                const uint32_t g = threadIdx.x / C + m * (kBlock / C);
                double2 y[V];
#pragma unroll
                for (int l = 0; l < V; l++) y[l] = load((g << RB) + l);
                fft_unit<RB, FWD>(y, (g << RB) * kFftRow + c, 9, tw, n);
#pragma unroll
                for (int l = 0; l < V; l++) store((g << RB) + l, y[l]);
            }
        }
    };
    auto from_buf = [&](uint32_t r) { return buf[r * kFftRow + c]; };
    auto to_buf = [&](uint32_t r, double2 v) { buf[r * kFftRow + c] = v; };
    auto from_lds = [&](uint32_t r) { return lds[r * C + cl]; };
    auto to_lds = [&](uint32_t r, double2 v) { lds[r * C + cl] = v; };
    if constexpr (FWD) {
#pragma unroll
        for (int l = 0; l < U; l++) z[l] = from_buf(r0 + (l << RB));
        wide();
        if constexpr (RB == 0) {
#pragma unroll
            for (int l = 0; l < U; l++) to_buf(l, z[l]);
        } else {
#pragma unroll
            for (int l = 0; l < U; l++) to_lds(r0 + (l << RB), z[l]);
            __syncthreads();
            narrow(from_lds, to_buf);
        }
    } else {
        if constexpr (RB == 0) {
#pragma unroll
            for (int l = 0; l < U; l++) z[l] = from_buf(l);
        } else {
            narrow(from_buf, to_lds);
            __syncthreads();
#pragma unroll
            for (int l = 0; l < U; l++) z[l] = from_lds(r0 + (l << RB));
        }
        wide();
        const double f = fix ? fix[blockIdx.y] : fix1;
#pragma unroll
        for (int l = 0; l < U; l++)
            to_buf(r0 + (l << RB), f != 0.0 ? make_double2(z[l].x * f, z[l].y * f) : z[l]);
    }
}

template <bool FWD>
void fft_cols(const Context &c, double2 *buf, uint32_t n, int logn, size_t B, const double *fix, double fix1,
              hipStream_t s) {
    const double2 *tw = FWD ? c.enc_fwd.as<double2>() : c.enc_inv.as<double2>();
#define SHM_FFT_COLS(S, RA, RB)                                                                              \
    case S:                                                                                                  \
        k_fft_cols<RA, RB, FWD><<<dim3(kFftRow / (kBlock >> RB), (unsigned)B), kBlock, 0, s>>>(buf, tw, n, fix, \
                                                                                               fix1);        \
        break;
    switch (logn - 9) {
        SHM_FFT_COLS(2, 2, 0)
        SHM_FFT_COLS(3, 3, 0)
        SHM_FFT_COLS(4, 2, 2)
        SHM_FFT_COLS(5, 3, 2)
        SHM_FFT_COLS(6, 3, 3)
        SHM_FFT_COLS(7, 4, 3)
        default: throw InvalidArgument("NTT requires N >= 4096");
    }
#undef SHM_FFT_COLS
    SHM_HIP(hipGetLastError());
}

// Inverse special FFT of B slot vectors (io: where they come from), scaled by fix[b] or fix1.
template <int IO>
void ifft(const Context &c, double2 *buf, uint32_t n, int logn, size_t B, const FftIO &io, const double *fix,
          double fix1, hipStream_t s) {
    if (logn < 11) throw InvalidArgument("NTT requires N >= 4096");
    k_fft_rows<false, IO><<<dim3(n / kFftRow, (unsigned)B), 64, 0, s>>>(buf, c.enc_inv.as<double2>(), n, logn, io);
    fft_cols<false>(c, buf, n, logn, B, fix, fix1, s);
}

// Constant plaintext in NTT form: every slot holds [round(fl(value*scale))]_q.
__global__ void k_fill_scalar(uint64_t *pt, const DevMod *mods, double v, size_t N, size_t total) {
    for (size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x; t < total; t += (size_t)gridDim.x * blockDim.x) {
        const DevMod m = mods[t >> __builtin_ctzll(N)];
        uint64_t r = residue_of_rounded(v, m);
        pt[t] = r >= m.q ? r - m.q : r;
    }
}

// A decoded coefficient is far below Q (its scale times a message), so its centred value v
// mostly follows from its first two residues: v = x_0 + q_0 ([(x_1 - x_0) / q_0]_{q_1}),
// centred mod q_0 q_1, and every other residue either confirms it (then |v| < q_0 q_1 / 2
// and v = X mod Q, so it is the centred value) or the full composition runs. Returns
// whether it holds, with |v| in (hi, lo).
__device__ __forceinline__ bool compose_short(const uint64_t *x, const DevMod *mods, uint64_t i01, uint64_t i01_s,
                                              size_t Ql, size_t stride, size_t at, uint64_t &hi, uint64_t &lo, bool &neg) {
    if (Ql < 2) return false;
    const uint64_t q0 = mods[0].q, q1 = mods[1].q, x0 = x[at];
    const uint64_t a1 = mul_shoup(sub_mod(x[stride + at], reduce64(x0, mods[1]), q1), i01, i01_s, q1);
    lo = q0 * a1 + x0;
    hi = __umul64hi(q0, a1) + (lo < x0);
    const uint64_t plo = q0 * q1, phi = __umul64hi(q0, q1);
    const uint64_t nlo = plo - lo, nhi = phi - hi - (plo < lo);  // q_0 q_1 - v
    neg = nhi < hi || (nhi == hi && nlo < lo);
    if (neg) {
        hi = nhi;
        lo = nlo;
    }
    bool same = true;
    for (size_t i = 2; i < Ql; i++) {
        const uint64_t r = barrett128(hi, lo, mods[i]);
        same = same && (neg ? neg_mod(r, mods[i].q) : r) == x[i * stride + at];
    }
    return same;
}

// rns_base.cu:200-262 compose_kernel: CRT compose, centre, convert. consts (ComposeTable):
// Q [W], half [W], q_0^-1 mod q_1 and its Shoup companion, qhinv [Ql], qhinv_s [Ql],
// qhat [Ql][W], W = Ql <= 64 words.
// The full composition keeps W words per coefficient in scratch memory and takes Ql W
// multiply-adds of 64 bits: 829 us for N = 2^16 at 24 limbs, where the short form takes
// 11 us.
__global__ void k_compose(const uint64_t *x, double2 *buf, const DevMod *mods, const uint64_t *consts, size_t Ql,
                          size_t N, uint32_t n, size_t ratio, double inv_scale) {
    const uint64_t *Q = consts, *half = Q + Ql, *inv01 = half + Ql, *qhinv = inv01 + 2, *qhinv_s = qhinv + Ql,
                   *qhat = qhinv_s + Ql;
    for (size_t ci = blockIdx.x * (size_t)blockDim.x + threadIdx.x; ci < 2 * (size_t)n;
         ci += (size_t)gridDim.x * blockDim.x) {
        const size_t W = Ql;
        const double two64 = 18446744073709551616.0;
        uint64_t vh, vl;
        bool neg;
        if (compose_short(x, mods, inv01[0], inv01[1], Ql, N, ci * ratio, vh, vl, neg)) {
            // the same word sums as below, words that are zero (or equal Q's) left out
            double res = 0.0, sc = inv_scale;
            if (neg) {
                uint64_t borrow = 0;
                for (size_t w = 0; w < W && (w < 2 || borrow); w++, sc *= two64) {
                    const uint64_t qw = Q[w], m = w == 0 ? vl : w == 1 ? vh : 0, a = qw - m - borrow;
                    borrow = (qw < m) || (qw == m && borrow) ? 1 : 0;
                    if (a > qw) {
                        const uint64_t d = a - qw;
                        res += d ? (double)d * sc : 0.0;
                    } else {
                        const uint64_t d = qw - a;
                        res -= d ? (double)d * sc : 0.0;
                    }
                }
            } else {
                res += vl ? (double)vl * sc : 0.0;
                sc *= two64;
                res += vh ? (double)vh * sc : 0.0;
            }
            if (ci < n)
                buf[ci].x = res;
            else
                buf[ci - n].y = res;
            continue;
        }
        uint64_t acc[64];
        for (size_t w = 0; w < W; w++) acc[w] = 0;
        for (size_t i = 0; i < Ql; i++) {
            const uint64_t q = mods[i].q;
            const uint64_t prod = mul_shoup(x[i * N + ci * ratio], qhinv[i], qhinv_s[i], q);
            // acc += qhat_i * prod (multi-precision), then reduce mod Q
            uint64_t carry = 0;
            for (size_t w = 0; w < W; w++) {
                const uint64_t a = qhat[i * W + w];
                const uint64_t lo = a * prod, hi = __umul64hi(a, prod);
                uint64_t s = acc[w] + lo;
                uint64_t c1 = s < lo;
                s += carry;
                c1 += s < carry;
                acc[w] = s;
                carry = hi + c1;
            }
            bool ge = carry != 0;
            if (!ge) {
                ge = true;
                for (size_t w = W; w-- > 0;) {
                    if (acc[w] != Q[w]) {
                        ge = acc[w] > Q[w];
                        break;
                    }
                }
            }
            if (ge) {
                uint64_t borrow = 0;
                for (size_t w = 0; w < W; w++) {
                    const uint64_t a = acc[w], b = Q[w];
                    const uint64_t d = a - b - borrow;
                    borrow = (a < b) || (a == b && borrow) ? 1 : 0;
                    acc[w] = d;
                }
            }
        }
        bool upper = true;
        for (size_t w = W; w-- > 0;) {
            if (acc[w] != half[w]) {
                upper = acc[w] > half[w];
                break;
            }
        }
        double res = 0.0, sc = inv_scale;
        if (upper) {
            for (size_t w = 0; w < W; w++, sc *= two64) {
                if (acc[w] > Q[w]) {
                    const uint64_t d = acc[w] - Q[w];
                    res += d ? (double)d * sc : 0.0;
                } else {
                    const uint64_t d = Q[w] - acc[w];
                    res -= d ? (double)d * sc : 0.0;
                }
            }
        } else {
            for (size_t w = 0; w < W; w++, sc *= two64) {
                const uint64_t d = acc[w];
                res += d ? (double)d * sc : 0.0;
            }
        }
        if (ci < n)
            buf[ci].x = res;
        else
            buf[ci - n].y = res;
    }
}

int ilog2(size_t v) {
    int l = 0;
    while ((size_t(1) << l) < v) l++;
    return l;
}

// Every slot holds one complex constant (the vector(slot_count, value) the
// facade's encode(double) builds, ckks_evaluator_parallel.cuh:73-78); a constant
// vector is its own bit reversal.
__global__ void k_fill_const(double2 *buf, double2 v, uint32_t n) {
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) buf[t] = v;
}

// batch_input's interleaved column packing (Batch_encode_encrypt.cuh:26-33): plaintext
// b holds column i = col0 + b with slot num_x * k + j = X[j][k][i] (X is
// [num_x][num_row][num_col]) and zeros beyond num_x * num_row, bit-reversed.
__global__ void k_columns_load_batch(const double *X, uint32_t num_x, uint32_t num_row, uint32_t num_col,
                                     uint32_t col0, double2 *buf, uint32_t n, int logn) {
    const uint32_t b = blockIdx.y, i = col0 + b, used = num_x * num_row;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        double v = 0.0;
        if (t < used) {
            const uint32_t j = t % num_x, k = t / num_x;
            v = X[((size_t)j * num_row + k) * num_col + i];
        }
        buf[(size_t)b * n + brv_bits(t, logn)] = make_double2(v, 0.0);
    }
}

}  // namespace

void encoder_tables(Context &c) {
    const size_t n = c.N / 2, M = 2 * c.N;
    const int logn = ilog2(n);
    c.enc_fwd.alloc(n * sizeof(double2));
    c.enc_inv.alloc(n * sizeof(double2));
    k_fft_tables<<<grid_for(n), kBlock>>>(c.enc_roots.as<double2>(), c.enc_group.as<uint32_t>(),
                                          c.enc_fwd.as<double2>(), c.enc_inv.as<double2>(), (uint32_t)n, logn,
                                          ilog2(M) - logn - 2, (uint32_t)M);
    SHM_HIP(hipGetLastError());
}

void encode(const Context &c, const double *re, const double *im, size_t n_values, size_t Ql, double scale,
            uint64_t *out, hipStream_t s) {
    const size_t n = c.N / 2;
    if (n_values > n) throw InvalidArgument("values_size is too large");
    if (!(scale > 0)) throw InvalidArgument("scale out of bounds");
    const int logn = ilog2(n);
    Scratch vals(2 * std::max<size_t>(n_values, 1) * sizeof(double), s);
    Scratch buf(n * sizeof(double2), s);
    double *dre = vals.as<double>(), *dim = dre + std::max<size_t>(n_values, 1);
    if (n_values) {
        SHM_HIP(hipMemcpyAsync(dre, re, n_values * sizeof(double), hipMemcpyHostToDevice, s));
        if (im) SHM_HIP(hipMemcpyAsync(dim, im, n_values * sizeof(double), hipMemcpyHostToDevice, s));
    }
    FftIO io{};
    io.re = dre;
    io.im = im ? dim : nullptr;
    io.nv = n_values;
    ifft<FFT_VALUES>(c, buf.as<double2>(), (uint32_t)n, logn, 1, io, nullptr, scale / (double)n, s);
    ntt_forward_encoded(c, buf.as<double2>(), out, 1, Ql, s);
}

void encode_const(const Context &c, double re, double im, size_t Ql, double scale, uint64_t *out, hipStream_t s) {
    const size_t n = c.N / 2;
    if (!(scale > 0)) throw InvalidArgument("scale out of bounds");
    const int logn = ilog2(n);
    Scratch buf(n * sizeof(double2), s);
    k_fill_const<<<grid_for(n), kBlock, 0, s>>>(buf.as<double2>(), make_double2(re, im), (uint32_t)n);
    ifft<FFT_BUF>(c, buf.as<double2>(), (uint32_t)n, logn, 1, FftIO{}, nullptr, scale / (double)n, s);
    ntt_forward_encoded(c, buf.as<double2>(), out, 1, Ql, s);
}

void encode_columns_batch(const Context &c, const double *X, size_t num_x, size_t num_row, size_t num_col,
                          size_t col0, size_t B, size_t Ql, const double *fix, uint64_t *out, double2 *fftbuf,
                          hipStream_t s) {
    const size_t n = c.N / 2;
    if (B == 0) return;
    if (B > 65535) throw InvalidArgument("encode_columns_batch: at most 65535 plaintexts");
    if (num_x * num_row > n) throw InvalidArgument("batch_input: num_X * num_row exceeds the slot count");
    const int logn = ilog2(n);
    k_columns_load_batch<<<dim3(std::min<unsigned>(grid_for(n), 128u), (unsigned)B), kBlock, 0, s>>>(
        X, (uint32_t)num_x, (uint32_t)num_row, (uint32_t)num_col, (uint32_t)col0, fftbuf, (uint32_t)n, logn);
    ifft<FFT_BUF>(c, fftbuf, (uint32_t)n, logn, B, FftIO{}, fix, 0.0, s);
    SHM_HIP(hipGetLastError());
    ntt_forward_encoded(c, fftbuf, out, B, Ql, s);
}

void encode_masked_batch(const Context &c, const double *w, const double *fix, const uint8_t *mask, size_t B,
                         size_t Ql, uint64_t *out, double2 *fftbuf, hipStream_t s, bool rows) {
    const size_t n = c.N / 2;
    if (B == 0) return;
    if (B > 65535) throw InvalidArgument("encode_masked_batch: at most 65535 plaintexts");
    const int logn = ilog2(n);
    FftIO io{};
    io.w = w;
    io.mask = mask;
    ifft<FFT_MASK>(c, fftbuf, (uint32_t)n, logn, B, io, fix, 0.0, s);
    SHM_HIP(hipGetLastError());
    // decompose (round, residue per prime) fused into the NTT's column pass
    if (rows)
        ntt_forward_encoded(c, fftbuf, out, B, Ql, s);
    else
        ntt_encoded_columns(c, fftbuf, out, B, Ql, s);
}

void encode_scalar(const Context &c, double value, size_t Ql, double scale, uint64_t *out, hipStream_t s) {
    if (!(scale > 0)) throw InvalidArgument("scale out of bounds");
    const double v = round(value * scale);
    k_fill_scalar<<<grid_for(Ql * c.N), kBlock, 0, s>>>(out, c.mods(), v, c.N, Ql * c.N);
    SHM_HIP(hipGetLastError());
}

void decode(const Context &c, const uint64_t *pt, size_t Ql, double scale, double *re, double *im, size_t nout,
            hipStream_t s) {
    const size_t N = c.N, n = N / 2;
    if (Ql > 64) throw InvalidArgument("decode supports at most 64 limbs");
    const int logn = ilog2(n);
    Scratch x(Ql * N * sizeof(uint64_t), s);
    PolyPack in{};
    in.p[0] = const_cast<uint64_t *>(pt);  // read only
    ntt_inverse_gather(c, in, x.as<uint64_t>(), 1, Ql, 0, s);
    Scratch buf(n * sizeof(double2), s);  // k_compose writes every entry
    k_compose<<<(unsigned)((2 * n + 63) / 64), 64, 0, s>>>(x.as<uint64_t>(), buf.as<double2>(), c.mods(),
                                                          c.level(Ql).compose.as<uint64_t>(), Ql, N, (uint32_t)n,
                                                          N / (2 * n), 1.0 / scale);
    Scratch o(2 * n * sizeof(double), s);
    fft_cols<true>(c, buf.as<double2>(), (uint32_t)n, logn, 1, nullptr, 0.0, s);
    FftIO io{};
    io.out_re = o.as<double>();
    io.out_im = o.as<double>() + n;
    k_fft_rows<true, FFT_VALUES><<<(unsigned)(n / kFftRow), 64, 0, s>>>(buf.as<double2>(), c.enc_fwd.as<double2>(),
                                                                        (uint32_t)n, logn, io);
    SHM_HIP(hipGetLastError());
    const size_t cnt = std::min(nout, n);
    SHM_HIP(hipMemcpyAsync(re, o.as<double>(), cnt * sizeof(double), hipMemcpyDeviceToHost, s));
    if (im) SHM_HIP(hipMemcpyAsync(im, o.as<double>() + n, cnt * sizeof(double), hipMemcpyDeviceToHost, s));
    SHM_HIP(hipStreamSynchronize(s));
}

}  // namespace shm
