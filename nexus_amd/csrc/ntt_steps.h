// Radix-2^K steps of the negacyclic NTT over a tile held in LDS or registers,
// shared by the transform passes (kernels_ntt.hip) and the key-switching
// kernels that run them on their own tiles (kernels_ks.hip).  See
// kernels_ntt.hip for the transform's definition and arithmetic.  Files using
// these are compiled without floating-point contraction.
#pragma once
#include "fpmod.h"
#include "modarith.h"

namespace nx {

namespace {

enum Role { kWhole = 0, kCol = 1, kRow = 2 };

constexpr int kThreads = 256;

// CW: sub-transforms per workgroup -- columns of the column pass (8 by
// default: a 16 KB tile keeps twice the workgroups of a 16-wide one resident,
// and once a batch outgrows the last-level cache the strided column reads of
// 8-wide tiles stream faster), and an upper bound on the rows of the row pass.
template <int LOGS, int ROLE, int CW>
struct Geometry {
    static constexpr int S = 1 << LOGS;
    static constexpr int ROWS = S >= 2048 ? 1 : 2048 / S;
    static constexpr int C = ROLE == kCol ? CW : (ROLE == kRow ? (ROWS < CW ? ROWS : CW) : 1);
    static constexpr int TILE = S * C;
};

// LDS address of local position `pos` of sub-transform `cc`.
template <int ROLE, int S, int C>
__device__ __forceinline__ int lds_addr(int cc, int pos)
{
    return ROLE == kCol ? pos * C + cc : cc * S + pos;
}

// Forward radix-2^K step over local stages s .. s+K-1.
template <int LOGS, int ROLE, int K, int CW, int NT = kThreads>
__device__ __forceinline__ void fwd_step(uint64_t *lds, int s, const ulonglong2 *tw, uint64_t q, uint32_t m0,
                                         uint32_t row0)
{
    using G = Geometry<LOGS, ROLE, CW>;
    constexpr int R = 1 << K;
    constexpr int GROUPS_PER = G::S / R;
    constexpr int GROUPS = G::TILE / R;
    const uint64_t two_q = 2 * q;
    const int B = G::S >> s;
    const int D = B >> K;
    for (int g = threadIdx.x; g < GROUPS; g += NT) {
        int cc, gg;
        if (ROLE == kCol) {
            cc = g % G::C;
            gg = g / G::C;
        } else {
            cc = g / GROUPS_PER;
            gg = g % GROUPS_PER;
        }
        const int blockid = gg / D;
        const int o = gg - blockid * D;
        const uint32_t mrow = (ROLE == kRow) ? (m0 + row0 + cc) : m0;
        uint64_t v[R];
        int addr[R];
#pragma unroll
        for (int t = 0; t < R; t++) {
            addr[t] = lds_addr<ROLE, G::S, G::C>(cc, blockid * B + o + t * D);
            v[t] = lds[addr[t]];
        }
#pragma unroll
        for (int d = 0; d < K; d++) {
            const int h = 1 << (K - 1 - d);
#pragma unroll
            for (int j = 0; j < (1 << d); j++) {
                const uint32_t b = (uint32_t)blockid * (1u << d) + j;
                const ulonglong2 w = tw[((uint32_t)1 << (s + d)) * mrow + b];
#pragma unroll
                for (int u = 0; u < h; u++) {
                    const int t = j * 2 * h + u;
                    uint64_t x = v[t];
                    x = x >= two_q ? x - two_q : x;
                    const uint64_t y = shoup_lazy(v[t + h], w.x, w.y, q);
                    v[t] = x + y;
                    v[t + h] = x - y + two_q;
                }
            }
        }
#pragma unroll
        for (int t = 0; t < R; t++) lds[addr[t]] = v[t];
    }
}

// Inverse radix-2^K step over local stages s .. s+K-1 (gaps 2^s .. 2^(s+K-1)).
template <int LOGS, int ROLE, int K, int CW, int NT = kThreads>
__device__ __forceinline__ void inv_step(uint64_t *lds, int s, const ulonglong2 *tw, uint64_t q, uint32_t n,
                                         uint32_t mx, uint32_t row0)
{
    using G = Geometry<LOGS, ROLE, CW>;
    constexpr int R = 1 << K;
    constexpr int GROUPS_PER = G::S / R;
    constexpr int GROUPS = G::TILE / R;
    const uint64_t two_q = 2 * q;
    const int so = 1 << s;
    for (int g = threadIdx.x; g < GROUPS; g += NT) {
        int cc, gg;
        if (ROLE == kCol) {
            cc = g % G::C;
            gg = g / G::C;
        } else {
            cc = g / GROUPS_PER;
            gg = g % GROUPS_PER;
        }
        const int o = gg & (so - 1);
        const int blockid = gg >> s;
        const int base = blockid * (so << K) + o;
        const uint32_t r = row0 + cc;
        uint64_t v[R];
        int addr[R];
#pragma unroll
        for (int t = 0; t < R; t++) {
            addr[t] = lds_addr<ROLE, G::S, G::C>(cc, base + t * so);
            v[t] = lds[addr[t]];
        }
#pragma unroll
        for (int d = 0; d < K; d++) {
            const int sd = s + d;
            const uint32_t first = n - (mx >> sd) + 1 + (ROLE == kRow ? r * ((uint32_t)G::S >> (sd + 1)) : 0u);
#pragma unroll
            for (int j = 0; j < (R >> (d + 1)); j++) {
                const uint32_t b = (uint32_t)blockid * (uint32_t)(R >> (d + 1)) + j;
                const ulonglong2 w = tw[first + b];
#pragma unroll
                for (int u = 0; u < (1 << d); u++) {
                    const int t = j * (2 << d) + u;
                    const uint64_t x = v[t], y = v[t + (1 << d)];
                    uint64_t sum = x + y;
                    v[t] = sum >= two_q ? sum - two_q : sum;
                    v[t + (1 << d)] = shoup_lazy(x - y + two_q, w.x, w.y, q);
                }
            }
        }
#pragma unroll
        for (int t = 0; t < R; t++) lds[addr[t]] = v[t];
    }
}

// Sums of the double-precision butterflies.  Twiddles are centred, |w| <= q/2,
// so the quotient of a product is off by at most 3 2^-53 |a| / 2 + 1/2 and
// |fp_mulmod(a, w)| <= q/2 + 1.5 2^-53 q |a|; it is exact while |a| < 2^53.
// Forward (v +- mulmod_f): from q/2 the bound grows to 1.19 q, 2.13 q and 3.43 q
// < 2^53 over three stages for any q < 2^51, so a step of up to three stages
// reduces once, at its end.  LAZY: q small enough for the whole pass
// (lazy_forward, lazy_inverse); nothing is reduced.
template <int K, bool LAZY>
__device__ __forceinline__ void reduce_step(double *v, double q, double qinv)
{
    if (!LAZY) {
#pragma unroll
        for (int t = 0; t < (1 << K); t++) v[t] = fp_reduce(v[t], q, qinv);
    }
}

// The butterflies of one forward radix-2^K group in registers: local stages
// s .. s+K-1 of block `blockid`, twiddle row mrow (1 for columns).
template <int K, bool LAZY>
__device__ __forceinline__ void fwd_group_f(double *v, int s, uint32_t blockid, uint32_t mrow, const double *tw,
                                            double q, double qinv)
{
#pragma unroll
    for (int d = 0; d < K; d++) {
        const int h = 1 << (K - 1 - d);
#pragma unroll
        for (int j = 0; j < (1 << d); j++) {
            const uint32_t b = blockid * (1u << d) + j;
            const double w = tw[((uint32_t)1 << (s + d)) * mrow + b];
#pragma unroll
            for (int u = 0; u < h; u++) {
                const int t = j * 2 * h + u;
                const double x = v[t];
                const double y = fp_mulmod(v[t + h], w, q, qinv);
                v[t] = x + y;
                v[t + h] = x - y;
            }
        }
        if (K > 3 && d == 1) reduce_step<K, LAZY>(v, q, qinv);  // a fourth stage would pass 2^53
    }
    reduce_step<K, LAZY>(v, q, qinv);
}

// Forward radix-2^K step in double precision (values |v| <= q/2 (1 + eps)
// between steps; LAZY: unreduced).
template <int LOGS, int ROLE, int K, int CW, bool LAZY, int NT = kThreads>
__device__ __forceinline__ void fwd_step_f(double *lds, int s, const double *tw, double q, double qinv, uint32_t m0,
                                           uint32_t row0)
{
    using G = Geometry<LOGS, ROLE, CW>;
    constexpr int R = 1 << K;
    constexpr int GROUPS_PER = G::S / R;
    constexpr int GROUPS = G::TILE / R;
    const int B = G::S >> s;
    const int D = B >> K;
    for (int g = threadIdx.x; g < GROUPS; g += NT) {
        int cc, gg;
        if (ROLE == kCol) {
            cc = g % G::C;
            gg = g / G::C;
        } else {
            cc = g / GROUPS_PER;
            gg = g % GROUPS_PER;
        }
        const int blockid = gg / D;
        const int o = gg - blockid * D;
        const uint32_t mrow = (ROLE == kRow) ? (m0 + row0 + cc) : m0;
        double v[R];
        int addr[R];
#pragma unroll
        for (int t = 0; t < R; t++) {
            addr[t] = lds_addr<ROLE, G::S, G::C>(cc, blockid * B + o + t * D);
            v[t] = lds[addr[t]];
        }
        fwd_group_f<K, LAZY>(v, s, (uint32_t)blockid, mrow, tw, q, qinv);
#pragma unroll
        for (int t = 0; t < R; t++) lds[addr[t]] = v[t];
    }
}

// Inverse radix-2^K step in double precision.  Sums double the bound (q/2 to 4 q
// <= 2^53 over three stages) and products stay below half of it, so a step
// reduces once, at its end.  LAZY: nothing is reduced.
template <int LOGS, int ROLE, int K, int CW, bool LAZY, int NT = kThreads>
__device__ __forceinline__ void inv_step_f(double *lds, int s, const double *tw, double q, double qinv, uint32_t n,
                                           uint32_t mx, uint32_t row0)
{
    using G = Geometry<LOGS, ROLE, CW>;
    constexpr int R = 1 << K;
    constexpr int GROUPS_PER = G::S / R;
    constexpr int GROUPS = G::TILE / R;
    const int so = 1 << s;
    for (int g = threadIdx.x; g < GROUPS; g += NT) {
        int cc, gg;
        if (ROLE == kCol) {
            cc = g % G::C;
            gg = g / G::C;
        } else {
            cc = g / GROUPS_PER;
            gg = g % GROUPS_PER;
        }
        const int o = gg & (so - 1);
        const int blockid = gg >> s;
        const int base = blockid * (so << K) + o;
        const uint32_t r = row0 + cc;
        double v[R];
        int addr[R];
#pragma unroll
        for (int t = 0; t < R; t++) {
            addr[t] = lds_addr<ROLE, G::S, G::C>(cc, base + t * so);
            v[t] = lds[addr[t]];
        }
#pragma unroll
        for (int d = 0; d < K; d++) {
            const int sd = s + d;
            const uint32_t first = n - (mx >> sd) + 1 + (ROLE == kRow ? r * ((uint32_t)G::S >> (sd + 1)) : 0u);
#pragma unroll
            for (int j = 0; j < (R >> (d + 1)); j++) {
                const uint32_t b = (uint32_t)blockid * (uint32_t)(R >> (d + 1)) + j;
                const double w = tw[first + b];
#pragma unroll
                for (int u = 0; u < (1 << d); u++) {
                    const int t = j * (2 << d) + u;
                    const double x = v[t], y = v[t + (1 << d)];
                    v[t] = x + y;
                    v[t + (1 << d)] = fp_mulmod(x - y, w, q, qinv);
                }
            }
            if (K > 3 && d == 1) reduce_step<K, LAZY>(v, q, qinv);
        }
        reduce_step<K, LAZY>(v, q, qinv);
#pragma unroll
        for (int t = 0; t < R; t++) lds[addr[t]] = v[t];
    }
}

// The radix steps of one pass in double precision, barrier after each.
template <int LOGS, int ROLE, bool FWD, int CW, bool LAZY, int NT = kThreads, bool R16 = false>
__device__ __forceinline__ void stages_f(double *lds, const double *tw, double q, double qinv, uint32_t n,
                                         uint32_t N1, uint32_t first)
{
    if constexpr (R16) {
        // radix-16 steps (half the LDS passes and barriers of radix-8), then
        // the remaining 1..3 stages in one step
        int s = 0;
        if (FWD) {
            const uint32_t m0 = ROLE == kRow ? N1 : 1u;
#pragma unroll
            for (int st = 0; st < LOGS / 4; st++) {
                fwd_step_f<LOGS, ROLE, 4, CW, LAZY, NT>(lds, s, tw, q, qinv, m0, first);
                s += 4;
                __syncthreads();
            }
            if constexpr (LOGS % 4 != 0) {
                fwd_step_f<LOGS, ROLE, LOGS % 4, CW, LAZY, NT>(lds, s, tw, q, qinv, m0, first);
                __syncthreads();
            }
        } else {
            const uint32_t mx = ROLE == kCol ? N1 : n;
#pragma unroll
            for (int st = 0; st < LOGS / 4; st++) {
                inv_step_f<LOGS, ROLE, 4, CW, LAZY, NT>(lds, s, tw, q, qinv, n, mx, first);
                s += 4;
                __syncthreads();
            }
            if constexpr (LOGS % 4 != 0) {
                inv_step_f<LOGS, ROLE, LOGS % 4, CW, LAZY, NT>(lds, s, tw, q, qinv, n, mx, first);
                __syncthreads();
            }
        }
        return;
    }
    int s = 0;
    if (FWD) {
        const uint32_t m0 = ROLE == kRow ? N1 : 1u;
        if constexpr (LOGS >= 3) {
#pragma unroll
            for (int st = 0; st < LOGS / 3; st++) {
                fwd_step_f<LOGS, ROLE, 3, CW, LAZY, NT>(lds, s, tw, q, qinv, m0, first);
                s += 3;
                __syncthreads();
            }
        }
        if constexpr (LOGS % 3 == 2) {
            fwd_step_f<LOGS, ROLE, 2, CW, LAZY, NT>(lds, s, tw, q, qinv, m0, first);
            __syncthreads();
        } else if constexpr (LOGS % 3 == 1) {
            fwd_step_f<LOGS, ROLE, 1, CW, LAZY, NT>(lds, s, tw, q, qinv, m0, first);
            __syncthreads();
        }
    } else {
        const uint32_t mx = ROLE == kCol ? N1 : n;
        if constexpr (LOGS >= 3) {
#pragma unroll
            for (int st = 0; st < LOGS / 3; st++) {
                inv_step_f<LOGS, ROLE, 3, CW, LAZY, NT>(lds, s, tw, q, qinv, n, mx, first);
                s += 3;
                __syncthreads();
            }
        }
        if constexpr (LOGS % 3 == 2) {
            inv_step_f<LOGS, ROLE, 2, CW, LAZY, NT>(lds, s, tw, q, qinv, n, mx, first);
            __syncthreads();
        } else if constexpr (LOGS % 3 == 1) {
            inv_step_f<LOGS, ROLE, 1, CW, LAZY, NT>(lds, s, tw, q, qinv, n, mx, first);
            __syncthreads();
        }
    }
}

// sum_k y_k f_k mod q, |r| <= q/2 (1 + eps): one output word of a base
// conversion over A inputs 0 <= y_k < p_k < 2^51 with centred factors
// |f_k| <= q/2, q < 2^51 (FpSum; at most 8 terms share a division, so the
// quotient stays below 2^53).  narrow: every p_k q < 2^97, so with s = 49 the
// terms (below 2^96) fit the accumulator and L stays below 2^51 unreduced.
// Otherwise s = 52 and four terms share an accumulator (4 2^101 <= 2^103, L <=
// 4 2^51); the two high parts, multiples of 2^52 below 2^104, add exactly.
// Eight terms take 40 (narrow) or 49 instructions, against 71 with a
// reduced product a term.
template <int A>
__device__ __forceinline__ double conv_sum(const double *y, int ystride, const double *f, double q, double qinv,
                                           bool narrow)
{
    double acc = 0.0;
#pragma unroll
    for (int k0 = 0; k0 < A; k0 += 8) {
        double r;
        if (narrow) {
            FpSum s;
            s.start(0x1.8p101);
#pragma unroll
            for (int k = k0; k < k0 + 8 && k < A; k++) s.mac(y[k * ystride], f[k]);
            const double H = s.h - 0x1.8p101;
            r = __builtin_fma(-__builtin_rint(H * qinv), q, H) + s.l;
        } else {
            FpSum s, u;
            s.start(0x1.8p104);
            u.start(0x1.8p104);
#pragma unroll
            for (int k = k0; k < k0 + 4 && k < A; k++) s.mac(y[k * ystride], f[k]);
#pragma unroll
            for (int k = k0 + 4; k < k0 + 8 && k < A; k++) u.mac(y[k * ystride], f[k]);
            const double H = (s.h - 0x1.8p104) + (u.h - 0x1.8p104);
            r = __builtin_fma(-__builtin_rint(H * qinv), q, H) + (fp_reduce(s.l, q, qinv) + fp_reduce(u.l, q, qinv));
        }
        acc = k0 ? acc + r : r;
        if (k0 + 8 < A) acc = fp_reduce(acc, q, qinv);
    }
    return fp_reduce(acc, q, qinv);
}

// the 8 words of a thread, y[A][8]; four words at a time, so that the partial sums of only those are live at once
template <int A>
__device__ __forceinline__ void conv_tile(double *cv, const double *y, const double *f, double q, double qinv,
                                          bool narrow)
{
    if (narrow) {  // uniform
#pragma unroll
        for (int k = 0; k < 8; k++) {
            cv[k] = conv_sum<A>(y + k, 8, f, q, qinv, true);
            if ((k & 3) == 3) __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int k = 0; k < 8; k++) {
            cv[k] = conv_sum<A>(y + k, 8, f, q, qinv, false);
            if (k & 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// How a column pass leaves its values: as words in [0, q) (a transform's
// intermediate), or as signed doubles for a row pass that reads them as such,
// reduced to |v| <= q/2 (1 + eps) or as the lazy stages left them.
enum ColOut { kWords = 0, kReduced = 1, kUnreduced = 2 };

template <bool LAZY, int OUT>
__device__ __forceinline__ uint64_t col_out(double x, double q, double qinv)
{
    if (LAZY && OUT != kUnreduced) x = fp_reduce(x, q, qinv);
    if (OUT != kWords) return (uint64_t)__double_as_longlong(x);
    return fp_to(x < 0 ? x + q : x);
}

// Whether `stages` forward stages from |v| <= q/2 (1 + eps) stay below 2^50
// unreduced: while |v| <= 2^50 a product is below q (1/2 + 1.5 2^-3).
__device__ __forceinline__ bool lazy_forward(double q, int stages) { return q * (0.5 + 0.6875 * stages) <= 0x1p50; }
// Whether `stages` inverse stages from |v| <= q/2 (1 + eps) stay below 2^53.
__device__ __forceinline__ bool lazy_inverse(double q, int stages) { return q * (double)(1u << stages) <= 0x1p54; }

// ---- column pass of a tile of 2048 words, 256 threads, 8 words a thread
//
// CW columns of 2^LOGS rows.  The first two stages join rows a quarter of the
// column apart: a thread holds rows g + QR t (t < 4) for two g of one column
// and runs them in registers.  After one exchange through LDS each wave owns
// one quarter of every column, and the remaining stages (3 + 3, or 3 + 2 for
// 2^7 rows) run inside the wave: one barrier a tile instead of three, the
// first five stages' twiddles are uniform (scalar loads), and loads and stores
// stay CW words wide.  Row r sits at (r + r / PB) CW in LDS, so the last
// step's reads PB rows apart fall on different banks.
template <int LOGS>
struct ColTile {
    static constexpr int CW = 2048 >> LOGS;
    static constexpr int QR = 1 << (LOGS - 2);   // rows of a quarter
    static constexpr int OL = 64 / CW;           // row groups of a wave
    static constexpr int K3 = LOGS - 5;          // stages of the last step
    static constexpr int PB = 1 << K3;
    static constexpr int LDS = ((1 << LOGS) + (1 << LOGS) / PB) * CW;
    // row of word k of a thread where the conversions leave it (row_step(k) past the first)
    __device__ static __forceinline__ int row_in(int tid, int k) { return tid / CW + row_step(k); }
    __device__ static __forceinline__ constexpr int row_step(int k) { return (256 / CW) * (k / 4) + QR * (k % 4); }
    // row of word k of a thread after the stages
    __device__ static __forceinline__ int row_out(int wave, int lane, int k)
    {
        return QR * wave + (lane / CW + OL * (k / PB)) * PB + k % PB;
    }
    __device__ static __forceinline__ int at(int row, int c) { return (row + row / PB) * CW + c; }
};

__device__ __forceinline__ void wave_sync()
{
    // a wave's LDS operations are carried out in order; only the compiler has
    // to keep them so
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void table_prime(const double2 *qd, uint32_t i, double &q, double &qinv)
{
    const double *p = reinterpret_cast<const double *>(qd);
    q = table_at(p, 2 * i);
    qinv = table_at(p, 2 * i + 1);
}

__device__ __forceinline__ ModConst table_mod(const ModConst *mod, uint32_t i)
{
    const uint64_t *p = reinterpret_cast<const uint64_t *>(mod + i);
    ModConst m;
    m.q = table_at(p, 0);
    m.ratio0 = table_at(p, 1);
    m.ratio1 = table_at(p, 2);
    m.two_q = table_at(p, 3);
    return m;
}

// 2^K-point forward butterflies (K <= 3) with the group's twiddles in
// w[(1 << d) - 1 + j]
template <int K, bool LAZY>
__device__ __forceinline__ void group_f(double *v, const double *w, double q, double qinv)
{
#pragma unroll
    for (int d = 0; d < K; d++) {
        const int h = 1 << (K - 1 - d);
#pragma unroll
        for (int j = 0; j < (1 << d); j++)
#pragma unroll
            for (int u = 0; u < h; u++) {
                const int t = j * 2 * h + u;
                const double x = v[t], y = fp_mulmod(v[t + h], w[(1 << d) - 1 + j], q, qinv);
                v[t] = x + y;
                v[t + h] = x - y;
            }
    }
    reduce_step<K, LAZY>(v, q, qinv);
}

// the same for a block that is uniform over the wave
template <int K>
__device__ __forceinline__ void uniform_group_tw(double *w, const double *tw, int s, uint32_t block)
{
#pragma unroll
    for (int d = 0; d < K; d++)
#pragma unroll
        for (int j = 0; j < (1 << d); j++) w[(1 << d) - 1 + j] = table_at(tw, ((uint32_t)1 << (s + d)) + (block << d) + j);
}

template <int K>
__device__ __forceinline__ void load_group_tw(double *w, const double *tw, int s, uint32_t mrow, uint32_t block)
{
#pragma unroll
    for (int d = 0; d < K; d++)
#pragma unroll
        for (int j = 0; j < (1 << d); j++) w[(1 << d) - 1 + j] = tw[((uint32_t)1 << (s + d)) * mrow + (block << d) + j];
}

// Word of (row, column tile, column in the tile) of a limb between a column
// pass and k_row_inner: four rows of one tile are contiguous (256 bytes at 8
// columns), so the column pass writes and the row pass, whose workgroups own
// four rows, reads whole cache lines; in the limb's own order each line is
// shared by two column tiles.
__device__ __forceinline__ uint32_t digit_word(uint32_t row, uint32_t tile, uint32_t c, uint32_t tiles, uint32_t log_cw)
{
    return (((row >> 2) * tiles + tile) << (log_cw + 2)) + ((row & 3) << log_cw) + c;
}

// Twiddles of the column stages of one prime.  The first two steps' are uniform
// over the wave (scalar loads); the last step's differ from lane to lane:
// vector loads, which return in order with the stores issued before them, so
// kernels that store one output after another ask for the next output's before
// they store the current one.
template <int LOGS>
struct ColTwiddles {
    using C = ColTile<LOGS>;
    double a[3], b[7], c[(8 / C::PB) * (C::PB - 1)];
    __device__ __forceinline__ void load_uniform(const double *tw)
    {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
        uniform_group_tw<2>(a, tw, 0, 0);
        uniform_group_tw<3>(b, tw, 2, (uint32_t)wave);
    }
    __device__ __forceinline__ void load_lane(const double *tw)
    {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), o = (int)(threadIdx.x % 64) / C::CW;
#pragma unroll
        for (int u = 0; u < 8 / C::PB; u++)
            load_group_tw<C::K3>(c + u * (C::PB - 1), tw, 5, 1, (uint32_t)(wave * (C::QR / C::PB) + o + C::OL * u));
    }
};

// The forward column stages: v[k] at ColTile::row_in (|v| <= q (1 + eps)),
// out at ColTile::row_out, stored at row N2 + col0 + column of out, or as
// doubles at digit_word.  lds: one of two buffers of ColTile::LDS words used in
// turn, so that the next tile's first exchange needs no second barrier.
template <int LOGS, bool LAZY, int OUT>
__device__ __forceinline__ void col_forward_store(double *v, double *lds, const ColTwiddles<LOGS> &tw, double q,
                                                  double qinv, uint32_t N2, uint32_t col0, uint64_t *out)
{
    using C = ColTile<LOGS>;
    const int tid = threadIdx.x;
    group_f<2, LAZY>(v, tw.a, q, qinv);
    group_f<2, LAZY>(v + 4, tw.a, q, qinv);
#pragma unroll
    for (int k = 0; k < 8; k++) lds[C::at(C::row_in(tid, k), tid % C::CW)] = v[k];
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int c = lane % C::CW, o = lane / C::CW;
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 8; t++) v[t] = lds[C::at(C::QR * wave + o + C::OL * t, c)];
    group_f<3, LAZY>(v, tw.b, q, qinv);
    wave_sync();
#pragma unroll
    for (int t = 0; t < 8; t++) lds[C::at(C::QR * wave + o + C::OL * t, c)] = v[t];
    wave_sync();
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = lds[C::at(C::row_out(wave, lane, k), c)];
#pragma unroll
    for (int u = 0; u < 8 / C::PB; u++) group_f<C::K3, LAZY>(v + u * C::PB, tw.c + u * (C::PB - 1), q, qinv);
    // one lane offset, uniform steps from word to word
    const uint32_t row0 = (uint32_t)C::row_out(wave, lane, 0), tiles = N2 / C::CW;
    const uint32_t at = OUT == kWords ? row0 * N2 + col0 + c
                                      : digit_word(row0, col0 / C::CW, (uint32_t)c, tiles, 11 - LOGS);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const uint32_t row = (uint32_t)((k / C::PB) * C::OL * C::PB + k % C::PB);  // past row0, a multiple of 4
        const uint32_t step = OUT == kWords ? row * N2 : ((row >> 2) * tiles * 4 + (row & 3)) * C::CW;
        (out + step)[at] = col_out<LAZY, OUT>(v[k], q, qinv);
    }
}

// the instance for the prime q: RAW stores doubles for a row pass of the
// remaining logn - LOGS stages that takes them as they are, else words
template <int LOGS, bool RAW>
__device__ __forceinline__ void col_forward(double *v, double *lds, const ColTwiddles<LOGS> &tw, double q, double qinv,
                                            int logn, uint32_t N2, uint32_t col0, uint64_t *out)
{
    if (RAW && lazy_forward(q, logn))  // uniform
        col_forward_store<LOGS, true, kUnreduced>(v, lds, tw, q, qinv, N2, col0, out);
    else if (lazy_forward(q, LOGS))
        col_forward_store<LOGS, true, RAW ? kReduced : kWords>(v, lds, tw, q, qinv, N2, col0, out);
    else
        col_forward_store<LOGS, false, RAW ? kReduced : kWords>(v, lds, tw, q, qinv, N2, col0, out);
}

// workgroups go to the 8 XCDs round-robin: consecutive column tiles, which
// share 128-byte lines, to workgroups of one XCD where the grid allows
__device__ __forceinline__ uint32_t xcd_tile(uint32_t block, uint32_t blocks)
{
    return (blocks & 7) == 0 ? (block & 7) * (blocks >> 3) + (block >> 3) : block;
}

}  // namespace

}  // namespace nx
