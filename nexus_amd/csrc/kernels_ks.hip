// Key switching on a two-pass ring (2^14 <= n <= 2^17) without a stored ModUp.
//
// The ModUp digits of a key switch are transformed, multiplied by the key and
// summed: of a stored T[output prime][digit] each word is written by the base
// conversion, read and written by each pass of the forward transform and read
// by the inner product.  Here the digits leave the column pass as doubles
// (the conversion runs in its load phase: k_modup_col in kernels_ntt.hip for
// several special primes, k_lift_col below for one), and k_row_inner runs the
// row pass of every digit of one output prime in registers and multiplies the
// result into two accumulators: T is written once and read once, a digit's own
// limbs are read where they lie (their transform is the input), and nothing
// but the accumulated inner product is written.
//
// Arithmetic as in kernels_ntt.hip: primes below 2^51 in double precision,
// larger ones in 64-bit Shoup butterflies with 128-bit sums.  Every output
// word is the residue in [0, q) of the same integer as before, so results are
// word for word those of the separate launches.
#include <algorithm>

#include "kernels.h"
#include "ntt_steps.h"
#include "prof.h"

namespace nx {

namespace {

// ---- lift of one-prime digits (one special prime) in the column pass

struct LiftColArgs {
    uint64_t *T;           // [B][nout][l][n]
    const uint64_t *coef;  // [B][l][n]
    const ulonglong2 *tw;
    const double *twd;
    const ModConst *mod;
    const double2 *qd;
    uint32_t l, nout, logn, chunk, chunks, listed;
    uint32_t list[kMaxPrimes];  // the output primes I of this launch
    uint32_t outp[kMaxPrimes];
};

// column stages of one tile on 64-bit words, values left in [0, 4q)
template <int LOGS>
__device__ __forceinline__ void col_stages_int(uint64_t *lds, const ulonglong2 *tw, uint64_t q, uint32_t N2,
                                               uint32_t col0, uint64_t *out)
{
    constexpr int CW = ColTile<LOGS>::CW;
    __syncthreads();
    int s = 0;
#pragma unroll
    for (int st = 0; st < LOGS / 3; st++) {
        fwd_step<LOGS, kCol, 3, CW>(lds, s, tw, q, 1u, col0);
        s += 3;
        __syncthreads();
    }
    fwd_step<LOGS, kCol, LOGS % 3, CW>(lds, s, tw, q, 1u, col0);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int e = threadIdx.x + k * kThreads;
        out[digit_word((uint32_t)(e / CW), col0 / CW, (uint32_t)(e % CW), N2 / CW, 11 - LOGS)] = lds[e];
    }
    __syncthreads();
}

// Workgroup (column tile, b, digit j, chunk of the listed output primes): the
// digit's coefficients are read once, and for every output prime of the chunk
// but the digit's own they are reduced, column-transformed and stored.  INT:
// the listed primes are 2^51 and above.  Below, the bound of four waves a SIMD
// costs six spilled words a lane.
template <int LOGS, bool INT>
__global__ __launch_bounds__(kThreads, INT ? 2 : 4) void k_lift_col(LiftColArgs a)
{
    using C = ColTile<LOGS>;
    static_assert(C::LDS >= 2048, "the 64-bit stages use one buffer");
    __shared__ uint64_t words[2 * C::LDS];
    const uint32_t n = 1u << a.logn;
    const uint32_t N2 = n >> LOGS;
    const uint32_t row = blockIdx.y;  // (b * l + j) * chunks + chunk
    const uint32_t bj = row / a.chunks, chunk = row - bj * a.chunks;
    const uint32_t b = bj / a.l, j = bj - b * a.l;
    const uint32_t r0 = chunk * a.chunk, r1 = min(a.listed, r0 + a.chunk);
    const uint32_t col0 = xcd_tile(blockIdx.x, gridDim.x) * C::CW;
    const int tid = threadIdx.x;
    const uint32_t at = (uint32_t)(tid / C::CW) * N2 + col0 + tid % C::CW;
    const uint64_t *src = a.coef + (uint64_t)bj * n;
    uint64_t x[8];
#pragma unroll
    for (int k = 0; k < 8; k++) x[k] = (src + C::row_step(k) * N2)[at];
    const bool small = a.mod[j].q <= (1ull << 52);  // the digit's words convert exactly
    uint32_t buf = 0;
    for (uint32_t r = r0; r < r1; r++) {
        const uint32_t I = a.list[r];
        if (I == j) continue;  // the input's own limb
        const uint32_t kp = a.outp[I];
        uint64_t *out = a.T + (((uint64_t)b * a.nout + I) * a.l + j) * n;
        if constexpr (INT) {
            const ModConst m = table_mod(a.mod, kp);
#pragma unroll
            for (int k = 0; k < 8; k++)
                words[C::row_in(tid, k) * C::CW + tid % C::CW] = x[k] >= m.q ? barrett64(x[k], m) : x[k];
            col_stages_int<LOGS>(words, a.tw + (uint64_t)kp * n, m.q, N2, col0, out);
        } else {
            double q, qinv;
            table_prime(a.qd, kp, q, qinv);
            ColTwiddles<LOGS> tw;
            tw.load_lane(a.twd + (uint64_t)kp * n);
            tw.load_uniform(a.twd + (uint64_t)kp * n);
            double v[8];
            if (small) {  // uniform
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = fp_reduce(fp_from(x[k]), q, qinv);
            } else {
                const ModConst m = table_mod(a.mod, kp);
#pragma unroll
                for (int k = 0; k < 8; k++) v[k] = fp_reduce(fp_from(barrett64(x[k], m)), q, qinv);
            }
            col_forward<LOGS, true>(v, reinterpret_cast<double *>(words) + buf * C::LDS, tw, q, qinv, (int)a.logn, N2,
                                    col0, out);
            buf ^= 1;
        }
    }
}

// ---- row pass and inner product

struct RowInnerArgs {
    uint64_t *acc;          // [B][2][nout][n] (sums of rotations: [sum[s]][2][nout][n])
    const uint64_t *T;      // [inputs][nout][digits][n]
    const uint64_t *own;    // the inputs in NTT form: [B][l][n], or ownp[b]
    const uint64_t *ownp[kMaxHoist];
    const uint64_t *key[kMaxHoist];    // per rotation; key[0] without rotations
    const uint64_t *aseed[kMaxHoist];  // non-null: the key's uniform half is regenerated (ctr_uniform)
    const uint32_t *perm[kMaxHoist];
    const ulonglong2 *tw;
    const double *twd;
    const ModConst *mod;
    const double2 *qd;
    uint32_t B, l, alpha, digits, nout, key_limbs, logn, log_cw;  // B: inputs, or sums of rotations
    uint32_t accumulate;           // the first sum is added to acc
    uint32_t sum[kMaxHoist];       // sum b: its index in acc and inputs first[b] .. first[b + 1] - 1
    uint8_t first[kMaxHoist + 1];
    uint32_t outp[kMaxPrimes];
};

// Rows of 2^LOGS words, whole rows per wave, W words a lane (4; 8 for rows of
// 512): the row stages run in steps of log2 W in registers with an exchange
// through the wave's own part of LDS between them, so no barrier is needed.
// Four words a lane hold both accumulators, the row's twiddles and the key words
// of a digit: 136 to 138 registers for rows of 256 (three waves a SIMD), 150 to
// 152 for rows of 128 (three); with rotations 166 to 168 (three) and 172 to 176
// (two).  Rows of 512 take all 256 and one wave.
// Step i (of K stages from stage s) joins 2^K positions D apart in blocks of
// S >> s: group gg = o + LPR u of a lane is block gg / D, offset gg % D.  In
// LDS position p sits at p + PAD (p / 16): blocks of four words 16 apart then
// fall on different banks.
template <int LOGS>
struct RowWave {
    static constexpr int S = 1 << LOGS;
    static constexpr int W = LOGS >= 9 ? 8 : 4;
    static constexpr int K1 = W == 8 ? 3 : 2;
    static constexpr int STEPS = (LOGS + K1 - 1) / K1;
    static constexpr int KL = LOGS - K1 * (STEPS - 1);  // stages of the last step
    static constexpr int LPR = S / W;                   // lanes per row
    static constexpr int ROWS = 64 / LPR;               // rows per wave
    static constexpr int PAD = 6;
    static constexpr int SP = S + S / 16 * PAD;
    static constexpr int LDS = ROWS * SP;
    static constexpr int R = 1 << KL;  // consecutive words a lane holds at the end
    static constexpr int G = W / R;
    static constexpr int TW = (STEPS - 1) * (W - 1) + G * (R - 1);  // twiddles of a lane
    __device__ static __forceinline__ int at(int p) { return p + PAD * (p / 16); }
    // position of word k of a lane in step i
    template <int i>
    __device__ static __forceinline__ int pos(int o, int k)
    {
        constexpr int K = i + 1 < STEPS ? K1 : KL, D = S >> (i * K1 + K), B = S >> (i * K1);
        const int gg = o + LPR * (k >> K);
        return gg / D * B + gg % D + D * (k & ((1 << K) - 1));
    }
    __device__ static __forceinline__ int out(int o, int k) { return pos<STEPS - 1>(o, k); }
};

// twiddles of one row for one lane
template <int LOGS>
struct RowTwiddles {
    using P = RowWave<LOGS>;
    double w[P::TW];
    template <int i>
    __device__ __forceinline__ void load_step(const double *tw, uint32_t mrow, int o)
    {
        constexpr int K = i + 1 < P::STEPS ? P::K1 : P::KL, D = P::S >> (i * P::K1 + K);
#pragma unroll
        for (int u = 0; u < (P::W >> K); u++)
            load_group_tw<K>(w + i * (P::W - 1) + u * ((1 << K) - 1), tw, i * P::K1, mrow,
                             (uint32_t)((o + P::LPR * u) / D));
        if constexpr (i + 1 < P::STEPS) load_step<i + 1>(tw, mrow, o);
    }
    __device__ __forceinline__ void load(const double *tw, uint32_t mrow, int o) { load_step<0>(tw, mrow, o); }
};

// Row stages of one row from step i on: v[k] at position pos<i>(o, k), out at
// P::out(o, k); lds points at the row's part.
template <int LOGS, bool LAZY, int i = 0>
__device__ __forceinline__ void row_forward(double *v, double *lds, int o, const RowTwiddles<LOGS> &t, double q,
                                            double qinv)
{
    using P = RowWave<LOGS>;
    constexpr int K = i + 1 < P::STEPS ? P::K1 : P::KL;
#pragma unroll
    for (int u = 0; u < (P::W >> K); u++)
        group_f<K, LAZY>(v + (u << K), t.w + i * (P::W - 1) + u * ((1 << K) - 1), q, qinv);
    if constexpr (i + 1 < P::STEPS) {
#pragma unroll
        for (int k = 0; k < P::W; k++) lds[P::at(P::template pos<i>(o, k))] = v[k];
        wave_sync();
#pragma unroll
        for (int k = 0; k < P::W; k++) v[k] = lds[P::at(P::template pos<i + 1>(o, k))];
        wave_sync();
        row_forward<LOGS, LAZY, i + 1>(v, lds, o, t, q, qinv);
    }
}

// the same stages on 64-bit words in [0, 4q), twiddles read as they are used
template <int K>
__device__ __forceinline__ void group_i(uint64_t *v, int s, uint32_t mrow, uint32_t block, const ulonglong2 *tw,
                                        uint64_t q)
{
    const uint64_t two_q = 2 * q;
#pragma unroll
    for (int d = 0; d < K; d++) {
        const int h = 1 << (K - 1 - d);
#pragma unroll
        for (int j = 0; j < (1 << d); j++) {
            const ulonglong2 w = tw[((uint32_t)1 << (s + d)) * mrow + (block << d) + j];
#pragma unroll
            for (int u = 0; u < h; u++) {
                const int t = j * 2 * h + u;
                const uint64_t x = v[t] >= two_q ? v[t] - two_q : v[t];
                const uint64_t y = shoup_lazy(v[t + h], w.x, w.y, q);
                v[t] = x + y;
                v[t + h] = x - y + two_q;
            }
        }
    }
}

template <int LOGS, int i = 0>
__device__ __forceinline__ void row_forward_int(uint64_t *v, uint64_t *lds, int o, uint32_t mrow,
                                                const ulonglong2 *tw, uint64_t q)
{
    using P = RowWave<LOGS>;
    constexpr int K = i + 1 < P::STEPS ? P::K1 : P::KL, D = P::S >> (i * P::K1 + K);
#pragma unroll
    for (int u = 0; u < (P::W >> K); u++)
        group_i<K>(v + (u << K), i * P::K1, mrow, (uint32_t)((o + P::LPR * u) / D), tw, q);
    if constexpr (i + 1 < P::STEPS) {
#pragma unroll
        for (int k = 0; k < P::W; k++) lds[P::at(P::template pos<i>(o, k))] = v[k];
        wave_sync();
#pragma unroll
        for (int k = 0; k < P::W; k++) v[k] = lds[P::at(P::template pos<i + 1>(o, k))];
        wave_sync();
        row_forward_int<LOGS, i + 1>(v, lds, o, mrow, tw, q);
    } else {
#pragma unroll
        for (int k = 0; k < P::W; k++) {
            uint64_t x = v[k];
            x = x >= 2 * q ? x - 2 * q : x;
            v[k] = x >= q ? x - q : x;
        }
    }
}

// words P::out(o, k) of a row, 16 bytes at a time
template <int LOGS>
__device__ __forceinline__ void load_row(uint64_t *v, const uint64_t *row, int o)
{
    using P = RowWave<LOGS>;
#pragma unroll
    for (int k = 0; k < P::W; k += 2) {
        const ulonglong2 x = *reinterpret_cast<const ulonglong2 *>(row + P::out(o, k));
        v[k] = x.x;
        v[k + 1] = x.y;
    }
}

template <int LOGS>
__device__ __forceinline__ void store_row(const uint64_t *v, uint64_t *row, int o)
{
    using P = RowWave<LOGS>;
#pragma unroll
    for (int k = 0; k < P::W; k += 2)
        *reinterpret_cast<ulonglong2 *>(row + P::out(o, k)) = make_ulonglong2(v[k], v[k + 1]);
}

// acc[b][k][I] = sum_j NTT(digit j)[I] key[j][k][I] (ROT: acc[b][k][I] (+)= the
// sum over the rotations r of sum b of sigma_r(NTT(digit j of input r))[I] key_r[j][k][I]).
// Workgroup: one output prime I and input or sum b, four waves, each of
// which owns its rows for the whole sum.  The automorphism maps rows onto rows (row and
// position in the row are the low and high bits of the bit-reversed exponent,
// and exponents are multiplied by an odd number), so a wave transforms the
// source row of its output row and gathers from LDS.
template <int LOGS, bool ROT, bool SEED>
__global__ __launch_bounds__(kThreads) void k_row_inner(RowInnerArgs a)
{
    using P = RowWave<LOGS>;
    constexpr int W = P::W;
    __shared__ uint64_t words[(kThreads / 64) * P::LDS];
    const uint32_t n = 1u << a.logn, N1 = n >> LOGS;
    const uint32_t lane = threadIdx.x % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int cc = (int)lane / P::LPR, o = (int)lane % P::LPR;
    uint64_t *wlds = words + wave * P::LDS + cc * P::SP;
    // neighbours in y: the same output prime of consecutive inputs or sums, whose
    // key words are then in this XCD's L2
    const uint32_t I = blockIdx.y / a.B, b = blockIdx.y - I * a.B;
    const uint32_t kp = a.outp[I];
    const uint32_t row = (blockIdx.x * (kThreads / 64) + wave) * P::ROWS + cc;
    const uint64_t base = (uint64_t)row * P::S;
    const ModConst m = a.mod[kp];
    const uint64_t kstride = (uint64_t)a.key_limbs * n;
    const uint64_t koff = (uint64_t)kp * n + base;
    const uint32_t own_digit = I < a.l ? I / a.alpha : ~0u;
    uint64_t *out = a.acc + (uint64_t)(ROT ? a.sum[b] : b) * 2 * a.nout * n + (uint64_t)I * n + base;
    const uint64_t poly1 = (uint64_t)a.nout * n;
    const uint32_t begin = ROT ? a.first[b] : b, end = ROT ? a.first[b + 1] : b + 1;
    const bool accumulate = ROT && a.accumulate && b == 0;

    if (m.q < kFpPrime) {
        const double q = a.qd[kp].x, qinv = a.qd[kp].y;
        const double *tw = a.twd + (uint64_t)kp * n;
        // through: the digits come unreduced and stay so, |t| <= 2^50, in the sums
        const bool through = lazy_forward(q, (int)a.logn), lazy = through || lazy_forward(q, LOGS);
        const double M = through ? kFpLazyMagic : fp_inner_magic(m.q);
        const uint32_t terms = through ? kFpLazyTerms : fp_inner_terms(m.q);
        double *lds = reinterpret_cast<double *>(wlds);
        FpSum s0[W], s1[W];
#pragma unroll
        for (int k = 0; k < W; k++) {
            s0[k].start(M);
            s1[k].start(M);
        }
        if (accumulate) {
            uint64_t v0[W], v1[W];
            load_row<LOGS>(v0, out, o);
            load_row<LOGS>(v1, out + poly1, o);
#pragma unroll
            for (int k = 0; k < W; k++) {
                s0[k].l = fp_reduce(fp_from(v0[k]), q, qinv);
                s1[k].l = fp_reduce(fp_from(v1[k]), q, qinv);
            }
        }
        uint64_t mix[W];  // the counter's half of the generator, the same for every digit
        if (SEED) {
#pragma unroll
            for (int k = 0; k < W; k++) mix[k] = ctr_mix64(koff + P::out(o, k) + 0x9e3779b97f4a7c15ull);
        }
        RowTwiddles<LOGS> w;
        if (!ROT) w.load(tw, N1 + row, o);
        uint32_t left = terms;
        for (uint32_t i = begin; i < end; i++) {
            const uint64_t *t0 = a.T + ((uint64_t)i * a.nout + I) * a.digits * n;
            const uint64_t *own = (a.own ? a.own + (uint64_t)i * a.l * n : a.ownp[i]) + (uint64_t)I * n;
            const uint64_t *key = a.key[ROT ? i : 0] + koff;
            const uint64_t *seed = a.aseed[ROT ? i : 0];
            uint32_t src[W];
            uint32_t trow = row;
            if (ROT) {
#pragma unroll
                for (int k = 0; k < W; k += 2) {
                    const uint2 p = *reinterpret_cast<const uint2 *>(a.perm[i] + base + P::out(o, k));
                    src[k] = p.x;
                    src[k + 1] = p.y;
                }
                trow = src[0] >> LOGS;
                w.load(tw, N1 + trow, o);
            }
            uint32_t tcol[W];
#pragma unroll
            for (int k = 0; k < W; k++) {
                const uint32_t x = (uint32_t)P::template pos<0>(o, k);
                tcol[k] = digit_word(trow, x >> a.log_cw, x & ((1u << a.log_cw) - 1), (uint32_t)P::S >> a.log_cw, a.log_cw);
            }
            // digit j's words as they lie: its own limb at the output positions, else doubles
            uint64_t x[W];
            auto load_digit = [&](uint32_t j) {
                if (j == own_digit) {  // uniform
                    if (ROT) {
#pragma unroll
                        for (int k = 0; k < W; k++) x[k] = own[src[k]];
                    } else {
                        load_row<LOGS>(x, own + base, o);
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < W; k++) x[k] = t0[(uint64_t)j * n + tcol[k]];
                }
            };
            load_digit(0);
            for (uint32_t j = 0; j < a.digits; j++) {
                // the key words and the next digit are asked for ahead of the
                // stages: two or three waves a SIMD do not hide the loads by themselves
                double t[W];
#pragma unroll
                for (int k = 0; k < W; k++) t[k] = j == own_digit ? fp_from(x[k]) : __longlong_as_double((long long)x[k]);
                const uint64_t *kj = key + (uint64_t)j * 2 * kstride;
                uint64_t ka[W], kb[W];
                load_row<LOGS>(ka, kj, o);
                if (!SEED) load_row<LOGS>(kb, kj + kstride, o);
                if (j + 1 < a.digits) load_digit(j + 1);
                if (j == own_digit) {
#pragma unroll
                    for (int k = 0; k < W; k++) t[k] = fp_reduce(t[k], q, qinv);
                } else {
                    if (lazy)
                        row_forward<LOGS, true>(t, lds, o, w, q, qinv);
                    else
                        row_forward<LOGS, false>(t, lds, o, w, q, qinv);
                    if (ROT) {
#pragma unroll
                        for (int k = 0; k < W; k++) lds[P::at(P::out(o, k))] = t[k];
                        wave_sync();
#pragma unroll
                        for (int k = 0; k < W; k++) t[k] = lds[P::at((int)(src[k] & (P::S - 1)))];
                        wave_sync();
                    }
                    if (lazy && !through) {  // uniform
#pragma unroll
                        for (int k = 0; k < W; k++) t[k] = fp_reduce(t[k], q, qinv);
                    }
                }
                if (left == 0) {  // uniform
#pragma unroll
                    for (int k = 0; k < W; k++) {
                        s0[k].l = s0[k].value(M, q, qinv);
                        s0[k].h = M;
                        s1[k].l = s1[k].value(M, q, qinv);
                        s1[k].h = M;
                    }
                    left = terms;
                }
                left--;
#pragma unroll
                for (int k = 0; k < W; k++) s0[k].mac(t[k], fp_from(ka[k]));
                if (SEED) {
                    const uint64_t sj = seed[j];
#pragma unroll
                    for (int k = 0; k < W; k++) kb[k] = mulhi64(ctr_mix64(sj ^ mix[k]), m.q);
                }
#pragma unroll
                for (int k = 0; k < W; k++) s1[k].mac(t[k], fp_from(kb[k]));
            }
        }
        uint64_t v0[W], v1[W];
#pragma unroll
        for (int k = 0; k < W; k++) {
            double x = s0[k].value(M, q, qinv), y = s1[k].value(M, q, qinv);
            v0[k] = fp_to(x < 0 ? x + q : x);
            v1[k] = fp_to(y < 0 ? y + q : y);
        }
        store_row<LOGS>(v0, out, o);
        store_row<LOGS>(v1, out + poly1, o);
        return;
    }

    // 64-bit words, 128-bit sums: at most 64 products below 2^122 are summed
    // between two reductions
    const ulonglong2 *tw = a.tw + (uint64_t)kp * n;
    uint64_t lo0[W] = {}, hi0[W] = {}, lo1[W] = {}, hi1[W] = {};
    if (accumulate) {
        load_row<LOGS>(lo0, out, o);
        load_row<LOGS>(lo1, out + poly1, o);
    }
    uint32_t sum = 1;
    for (uint32_t i = begin; i < end; i++) {
        const uint64_t *t0 = a.T + ((uint64_t)i * a.nout + I) * a.digits * n;
        const uint64_t *own = (a.own ? a.own + (uint64_t)i * a.l * n : a.ownp[i]) + (uint64_t)I * n;
        const uint64_t *key = a.key[ROT ? i : 0] + koff;
        const uint64_t *seed = a.aseed[ROT ? i : 0];
        uint32_t src[W];
        uint32_t mrow = N1 + row;
        if (ROT) {
#pragma unroll
            for (int k = 0; k < W; k++) src[k] = a.perm[i][base + P::out(o, k)];
            mrow = N1 + (src[0] >> LOGS);
        }
        uint32_t tcol[W];
#pragma unroll
        for (int k = 0; k < W; k++) {
            const uint32_t x = (uint32_t)P::template pos<0>(o, k);
            tcol[k] = digit_word(mrow - N1, x >> a.log_cw, x & ((1u << a.log_cw) - 1), (uint32_t)P::S >> a.log_cw, a.log_cw);
        }
        for (uint32_t j = 0; j < a.digits; j++) {
            uint64_t t[W];
            if (j == own_digit) {
                if (ROT) {
#pragma unroll
                    for (int k = 0; k < W; k++) t[k] = own[src[k]];
                } else {
                    load_row<LOGS>(t, own + base, o);
                }
            } else {
                const uint64_t *tj = t0 + (uint64_t)j * n;
#pragma unroll
                for (int k = 0; k < W; k++) t[k] = tj[tcol[k]];
                row_forward_int<LOGS>(t, wlds, o, mrow, tw, m.q);
                if (ROT) {
#pragma unroll
                    for (int k = 0; k < W; k++) wlds[P::at(P::out(o, k))] = t[k];
                    wave_sync();
#pragma unroll
                    for (int k = 0; k < W; k++) t[k] = wlds[P::at((int)(src[k] & (P::S - 1)))];
                    wave_sync();
                }
            }
            if (sum == 64) {  // uniform
#pragma unroll
                for (int k = 0; k < W; k++) {
                    lo0[k] = barrett128(hi0[k], lo0[k], m);
                    lo1[k] = barrett128(hi1[k], lo1[k], m);
                    hi0[k] = hi1[k] = 0;
                }
                sum = 1;
            }
            sum++;
            const uint64_t *kj = key + (uint64_t)j * 2 * kstride;
            uint64_t ka[W], kb[W];
            load_row<LOGS>(ka, kj, o);
            if (SEED) {
                const uint64_t sj = seed[j];
#pragma unroll
                for (int k = 0; k < W; k++) kb[k] = ctr_uniform(sj, koff + P::out(o, k), m.q);
            } else {
                load_row<LOGS>(kb, kj + kstride, o);
            }
#pragma unroll
            for (int k = 0; k < W; k++) {
                uint64_t pl = t[k] * ka[k], ph = mulhi64(t[k], ka[k]);
                lo0[k] += pl;
                hi0[k] += ph + (lo0[k] < pl);
                pl = t[k] * kb[k];
                ph = mulhi64(t[k], kb[k]);
                lo1[k] += pl;
                hi1[k] += ph + (lo1[k] < pl);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < W; k++) {
        lo0[k] = barrett128(hi0[k], lo0[k], m);
        lo1[k] = barrett128(hi1[k], lo1[k], m);
    }
    store_row<LOGS>(lo0, out, o);
    store_row<LOGS>(lo1, out + poly1, o);
}

}  // namespace

// Workgroups of k_row_inner for one output prime of one input or sum.
static uint32_t row_inner_tiles(int logn) { return (1u << logn) / (logn == 17 ? 2048u : 1024u); }

// Primes of 2^51 and above take the kernel's 64-bit form: a serial chain of digits
// with two waves a SIMD (rows of 512: one) to hide it.  It needs the device full,
// two workgroups a CU, to beat a stored ModUp, whose transforms and products
// spread over every digit; at N = 2^17 it does not where most primes are wide.
// Microseconds, stored ModUp / this one:
//   160 blocks, N = 2^14, ten primes, two of 58 bits: one input 84 / 97, a sum of 16: 356 / 504
//   320 blocks, 2^15, the same: 104 / 116, 619 / 748;  336, 2^14, 21 of 60 bits: 158 / 163, 1585 / 1715
//   640 blocks, 2^16, ten of 60 bits: 163 / 158, 1360 / 1282;  six sums at 2^15: 3261 / 2827
//   2^17: ten primes, two of 60 bits: 230 / 238, 2235 / 2071; 21 of 60 bits: 918 / 966, 24 sums of eight 135 / 147 ms
// Below 2^51 it is ahead from the smallest call on (2^14, ten primes of 46 bits: 75 / 70, 333 / 315).
bool ks_row_inner_ok(const DeviceTables &t, uint32_t alpha, const uint8_t *out_primes_host, uint32_t nout,
                     uint32_t count)
{
    if (t.logn < 14 || t.logn > 17 || t.max_bits > 61 || !(alpha == 1 || ks_modup_col_ok(t, alpha))) return false;
    uint32_t wide = 0;
    for (uint32_t I = 0; I < nout; I++) wide += t.mod_host[out_primes_host[I]] >= kFpPrime ? 1 : 0;
    if (!wide) return true;
    return row_inner_tiles(t.logn) * nout * count >= 512u && (t.logn < 17 || 2 * wide <= nout);
}

void ks_lift_col(const DeviceTables &t, uint64_t *T, const uint64_t *coef, uint32_t B, uint32_t l,
                 const uint8_t *out_primes_host, uint32_t nout, hipStream_t s)
{
    if (t.logn < 14 || t.logn > 17 || nout > (uint32_t)kMaxPrimes || !nout || !l || !B)
        throw std::invalid_argument("ks_lift_col: unsupported parameters");
    LiftColArgs a;
    a.T = T;
    a.coef = coef;
    a.tw = t.fwd;
    a.twd = t.fwd_d;
    a.mod = t.mod;
    a.qd = t.qd;
    a.l = l;
    a.nout = nout;
    a.logn = (uint32_t)t.logn;
    for (int i = 0; i < kMaxPrimes; i++) a.outp[i] = i < (int)nout ? out_primes_host[i] : 0;
    const int l1 = t.logn / 2;
    const uint32_t n = 1u << t.logn, tiles = n / 2048;
    ProfScope prof("ks_lift_col", s, 8.0 * n * B * l * (1.0 + nout) + 8.0 * (double)(1u << l1) * B * l * nout);
    for (int wide = 0; wide < 2; wide++) {  // primes below 2^51, then the others
        a.listed = 0;
        for (uint32_t I = 0; I < nout; I++)
            if ((t.mod_host[out_primes_host[I]] >= kFpPrime) == (wide != 0)) a.list[a.listed++] = I;
        if (!a.listed) continue;
        // outputs per workgroup: enough workgroups to fill the device, at least 4
        // outputs per read of the digit
        const uint32_t want = (2048u + tiles * B * l - 1) / (tiles * B * l);
        a.chunk = std::max((a.listed + want - 1) / want, std::min(4u, a.listed));
        a.chunks = (a.listed + a.chunk - 1) / a.chunk;
        const dim3 grid(tiles, B * l * a.chunks);
        if (l1 == 7 && wide)
            hipLaunchKernelGGL((k_lift_col<7, true>), grid, dim3(kThreads), 0, s, a);
        else if (l1 == 7)
            hipLaunchKernelGGL((k_lift_col<7, false>), grid, dim3(kThreads), 0, s, a);
        else if (wide)
            hipLaunchKernelGGL((k_lift_col<8, true>), grid, dim3(kThreads), 0, s, a);
        else
            hipLaunchKernelGGL((k_lift_col<8, false>), grid, dim3(kThreads), 0, s, a);
    }
}

void ks_row_inner(const DeviceTables &t, const KsRowInner &p, hipStream_t s)
{
    const bool rot = p.perms != nullptr;
    if (!p.count || (rot && (p.count > (uint32_t)kMaxHoist || !p.sum)) ||
        (p.own_list && p.count > (uint32_t)kMaxHoist) || p.nout > (uint32_t)kMaxPrimes || t.logn < 14 || t.logn > 17)
        throw std::invalid_argument("ks_row_inner: unsupported parameters");
    RowInnerArgs a;
    a.acc = p.acc;
    a.T = p.T;
    a.own = p.own_list ? nullptr : p.own;
    bool seeded = true;
    for (uint32_t i = 0; i < (uint32_t)kMaxHoist; i++) {
        a.ownp[i] = p.own_list && i < p.count ? p.own_list[i] : nullptr;
        const bool on = rot ? i < p.count : i == 0;
        a.key[i] = on ? p.keys[i] : nullptr;
        // one key for several inputs: its words come from the L2, cheaper than
        // generating half of them again for every input
        a.aseed[i] = on && p.aseeds && (rot || p.count == 1) ? p.aseeds[i] : nullptr;
        a.perm[i] = on && rot ? p.perms[i] : nullptr;
        seeded = seeded && (!on || a.aseed[i]);  // a key without seeds (uploaded): all are read in full
    }
    // runs of inputs of one sum
    a.B = rot ? 0 : p.count;
    a.accumulate = 0;
    for (uint32_t i = 0; i < (uint32_t)kMaxHoist; i++) {
        a.sum[i] = 0;
        a.first[i] = 0;
    }
    if (rot) {
        for (uint32_t i = 0; i < p.count; i++) {
            if (i && p.sum[i] == p.sum[i - 1]) continue;
            a.first[a.B] = (uint8_t)i;
            a.sum[a.B++] = p.sum[i];
        }
        a.accumulate = p.accumulate ? 1u : 0u;
    }
    a.first[rot ? a.B : 0] = (uint8_t)(rot ? p.count : 0);
    a.tw = t.fwd;
    a.twd = t.fwd_d;
    a.mod = t.mod;
    a.qd = t.qd;
    a.l = p.l;
    a.alpha = p.alpha;
    a.digits = p.digits;
    a.nout = p.nout;
    a.key_limbs = p.key_limbs;
    a.logn = (uint32_t)t.logn;
    a.log_cw = 11u - (uint32_t)(t.logn / 2);  // ColTile: 2048 words a tile
    for (int i = 0; i < kMaxPrimes; i++) a.outp[i] = i < (int)p.nout ? p.out_primes[i] : 0;
    const uint32_t n = 1u << t.logn;
    const int l2 = t.logn - t.logn / 2;
    ProfScope prof(rot ? "ks_row_inner_rot" : "ks_row_inner", s,
                   // digits, the words of each key once, permutations, results
                   (double)n * p.nout *
                       (8.0 * p.count * p.digits + (seeded ? 8.0 : 16.0) * (rot ? p.count : 1u) * p.digits +
                        (rot ? 4.0 * p.count : 0.0) + 16.0 * (a.B + a.accumulate)));
    const dim3 grid(row_inner_tiles(t.logn), p.nout * a.B);
#define NX_RI(L)                                                                             \
    if (l2 == L) {                                                                         \
        if (rot && seeded)                                                                 \
            hipLaunchKernelGGL((k_row_inner<L, true, true>), grid, dim3(kThreads), 0, s, a);   \
        else if (rot)                                                                      \
            hipLaunchKernelGGL((k_row_inner<L, true, false>), grid, dim3(kThreads), 0, s, a);  \
        else if (seeded)                                                                   \
            hipLaunchKernelGGL((k_row_inner<L, false, true>), grid, dim3(kThreads), 0, s, a);  \
        else                                                                               \
            hipLaunchKernelGGL((k_row_inner<L, false, false>), grid, dim3(kThreads), 0, s, a); \
        return;                                                                            \
    }
    NX_RI(7) NX_RI(8) NX_RI(9)
#undef NX_RI
}

}  // namespace nx
