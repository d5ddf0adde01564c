// Negacyclic NTT / INTT over RNS limbs for gfx950.
//
// Transform definition (SEAL, util/ntt.cpp:241-477 and util/dwthandler.h):
//  forward: Cooley-Tukey stages m = 1, 2, ..., n/2 with gap n/(2m); butterfly
//           block i of stage m uses fwd[m + i]; natural order in, bit-reversed out.
//  inverse: Gentleman-Sande stages m = n/2, ..., 1 with gap n/(2m); block i of
//           stage m uses inv[n - 2m + 1 + i]; followed by multiplication by n^-1.
// Outputs are fully reduced, so they are bit-identical to SEAL's however the
// lazy reductions inside are scheduled.
//
// Mapping.  n <= 2^13: one workgroup holds a whole limb in LDS (a few limbs of
// 2^13: two passes, see two_passes).  n >= 2^14: the
// limb is viewed as an N1 x N2 matrix (index = t * N2 + c).  The first log2(N1)
// forward stages only pair elements of the same column c (gap >= N2), the last
// log2(N2) stages only pair elements of the same row t; the inverse runs rows
// first, then columns.  Each pass stages a tile of 8 columns or 8 contiguous
// rows (4 or 16 where the autotuner says so) through LDS and runs radix-8/4/2
// register butterflies between barriers, 256 threads (four wave64) per workgroup.  Row twiddles for row r at
// local stage s are the contiguous block fwd[2^s (N1 + r) ...].
//
// Arithmetic.  Limbs of primes q < 2^51 run in double precision, where the FMA
// is full rate: exact products (fp_mulmod, six instructions) with centred
// twiddles |w| <= q/2.  Loads are reduced to |v| <= q/2 (1 + eps); the sums of a
// step of up to three stages are reduced at its end, or not at all in a pass
// where they stay small enough (reduce_step, lazy_forward, lazy_inverse); stores
// are mapped to [0, q), so the output words equal the integer path's.  Larger
// primes use 64-bit Shoup butterflies (ten 32-bit multiplies each) on [0, 4q).
// This file is compiled without floating-point contraction.
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <stdexcept>

#include "kernels.h"
#include "ntt_steps.h"
#include "prof.h"

namespace nx {

namespace {

struct NttKArgs {
    uint64_t *data;
    uint64_t poly_stride;
    const uint64_t *src;  // input of this pass (null: in place)
    uint64_t src_poly_stride;
    uint32_t nsrcs;       // > 0: poly p of this pass reads srcs[p]
    const uint64_t *srcs[kNttSrcMax];
    double tw_bytes;      // mean twiddle bytes per entry over the batch (profiler accounting)
    uint32_t limbs;
    uint32_t logn;
    uint32_t prime_by_poly;
    uint32_t poly_period;
    const ulonglong2 *tw;
    const ModConst *mod;
    const double2 *qd;
    const ulonglong2 *ninv;
    const double *twd;    // the same twiddles as doubles
    const double *ninvd;  // n^-1 mod q as doubles
    uint32_t skip_l, skip_alpha, skipped;  // NttBatch::skip_*; skipped: limbs left out
    NttEpilogue epi;                        // applied by the forward transform's last pass
    uint32_t epi_int;                       // double-precision path: the epilogue in 64-bit integers
    const uint64_t *in;                     // NttBatch::lift / center (LOAD kLift / kCenter): the words read,
    uint64_t in_stride;                     // words from a poly's to the next one's (kCenter),
    uint32_t in_prime;                      // and their prime (kCenter)
    uint8_t prime_of[kMaxPrimes];
};

__host__ __device__ inline bool epi_on(const NttEpilogue &e) { return e.out != nullptr || e.outs[0] != nullptr; }

// NttEpilogue's store of the transform value t (in [0, q)) of poly p, limb i
// of a batch of l limbs
__device__ __forceinline__ void epi_store(const NttEpilogue &e, uint32_t p, uint32_t i, uint64_t gidx, uint64_t t,
                                          uint64_t q, uint32_t l, uint32_t n)
{
    const uint64_t off = (uint64_t)i * n + gidx;
    const ulonglong2 w = e.inv[i];
    const uint32_t ct = p / e.polys_per, k = p - ct * e.polys_per;
    const uint64_t xv = e.xs[0] ? e.xs[ct][((uint64_t)k * e.x_limbs + i) * n + gidx] : e.x[p * e.x_stride + off];
    uint64_t r = shoup(sub_mod(xv, t, q), w.x, w.y, q);
    if (e.out) {
        uint64_t *o = e.out + p * e.out_stride + off;
        if (e.accumulate == 1 || (e.accumulate == 2 && (p & 1) == 0))
            r = add_mod(e.base ? e.base[p * e.base_stride + off] : *o, r, q);
        *o = r;
        return;
    }
    const uint64_t *a0 = e.a0s[0] ? e.a0s[ct] : e.a0;
    if (a0 && k == 0) r = add_mod(r, a0[(uint64_t)i * n + e.perm[ct][gidx]], q);
    if (e.d) {
        const ulonglong2 w2 = e.inv2[i];
        r = add_mod(r, shoup(e.d[p * e.d_stride + off], w2.x, w2.y, q), q);
    }
    e.outs[ct][((uint64_t)k * l + i) * n + gidx] = r;
}

constexpr int kTuneLogNMin = 14, kTuneLogN = 4, kTuneBuckets = 9;

// epi_store in double precision (every prime of the batch below 2^51): the
// transform value t in [0, q) as a double, the Shoup constants' values (below
// q) as factors of exact products.  |x - t| < q, each product is within 1.25 q
// and a term in [0, q) is added at most twice, so the sum stays below 2^53 and
// the stored residue equals epi_store's.
__device__ __forceinline__ void epi_store_f(const NttEpilogue &e, uint32_t p, uint32_t i, uint64_t gidx, double t,
                                            double q, double qinv, uint32_t l, uint32_t n)
{
    const uint64_t off = (uint64_t)i * n + gidx;
    const uint32_t ct = p / e.polys_per, k = p - ct * e.polys_per;
    const uint64_t xv = e.xs[0] ? e.xs[ct][((uint64_t)k * e.x_limbs + i) * n + gidx] : e.x[p * e.x_stride + off];
    double r = fp_mulmod(fp_from(xv) - t, fp_from(e.inv[i].x), q, qinv);
    uint64_t *o;
    if (e.out) {
        o = e.out + p * e.out_stride + off;
        if (e.accumulate == 1 || (e.accumulate == 2 && (p & 1) == 0))
            r += fp_from(e.base ? e.base[p * e.base_stride + off] : *o);
    } else {
        const uint64_t *a0 = e.a0s[0] ? e.a0s[ct] : e.a0;
        if (a0 && k == 0) r += fp_from(a0[(uint64_t)i * n + e.perm[ct][gidx]]);
        if (e.d) r += fp_mulmod(fp_from(e.d[p * e.d_stride + off]), fp_from(e.inv2[i].x), q, qinv);
        o = e.outs[ct] + ((uint64_t)k * l + i) * n + gidx;
    }
    r = fp_reduce(r, q, qinv);
    *o = fp_to(r < 0 ? r + q : r);
}

// What the first pass of a forward transform reads (NttBatch::lift, center).
// Taking the words mod the limb's prime here saves the key switch and the
// rescale a pass that only wrote them out for this one to read back: bound by
// memory traffic on large rings (16 degree-7 products at N = 2^16 with 60-bit
// primes: 14.3 to 13.4 ms), by launches on small ones (multiply, relinearise and
// rescale at 2^13: 83 to 75 us).
enum Load { kPlain = 0, kLift = 1, kCenter = 2 };

template <int LOAD>
__device__ __forceinline__ uint64_t load_word(uint64_t v, const NttKArgs &a, const ModConst &m)
{
    if constexpr (LOAD == kLift) return v >= m.q ? barrett64(v, m) : v;
    if constexpr (LOAD == kCenter) {
        const uint64_t p = a.mod[a.in_prime].q, half = p >> 1;
        v += half;
        v = v >= p ? v - p : v;  // (x + (p - 1) / 2) mod p
        return sub_mod(barrett64(v, m), barrett64(half, m), m.q);
    }
    return v;
}

// The whole transform body of one tile in double precision: load (reduced),
// the radix steps, store in [0, q) (times n^-1 on the inverse's last pass).
//
// Lazy reduction: see reduce_step and the inverse step (ntt_steps.h).  The
// stored words are the fully reduced residues either way.
template <int LOGS, int ROLE, bool FWD, int CW, bool R16, int NT, int LOAD>
__device__ __forceinline__ void ntt_tile_f(const NttKArgs &a, uint64_t *lds_words, uint64_t *data,
                                           const uint64_t *src, uint32_t prime, uint32_t n, uint32_t N2, uint32_t N1,
                                           uint32_t first, uint32_t poly, uint32_t limb)
{
    using G = Geometry<LOGS, ROLE, CW>;
    const bool epi = FWD && ROLE != kCol && epi_on(a.epi);
    double *lds = reinterpret_cast<double *>(lds_words);
    const double q = a.qd[prime].x, qinv = a.qd[prime].y;
    const double *tw = a.twd + (uint64_t)prime * n;
    const bool lazy = FWD ? lazy_forward(q, LOGS) : lazy_inverse(q, LOGS);  // uniform: one prime per workgroup
    if constexpr (FWD && ROLE == kRow && LOGS == 8 && G::C == 8 && !R16) {
        // rows of 256, 8 rows per tile, 256 threads: each thread loads one
        // radix-8 group of the first three stages (row g / 32, positions
        // g % 32 + 32 t) and runs it in registers; one LDS pass and one barrier
        // fewer, the rest as below
        {
            const int g = threadIdx.x, cc = g / 32, o = g % 32;
            double v[8];
#pragma unroll
            for (int t = 0; t < 8; t++)
                v[t] = fp_reduce(fp_from(src[(uint64_t)(first + cc) * G::S + o + 32 * t]), q, qinv);
            if (lazy)
                fwd_group_f<3, true>(v, 0, 0, N1 + first + cc, tw, q, qinv);
            else
                fwd_group_f<3, false>(v, 0, 0, N1 + first + cc, tw, q, qinv);
#pragma unroll
            for (int t = 0; t < 8; t++) lds[cc * G::S + o + 32 * t] = v[t];
        }
        __syncthreads();
        if (lazy) {
            fwd_step_f<LOGS, ROLE, 3, CW, true>(lds, 3, tw, q, qinv, N1, first);
            __syncthreads();
            fwd_step_f<LOGS, ROLE, 2, CW, true>(lds, 6, tw, q, qinv, N1, first);
        } else {
            fwd_step_f<LOGS, ROLE, 3, CW, false>(lds, 3, tw, q, qinv, N1, first);
            __syncthreads();
            fwd_step_f<LOGS, ROLE, 2, CW, false>(lds, 6, tw, q, qinv, N1, first);
        }
        __syncthreads();
    } else {
        for (int e = threadIdx.x; e < G::TILE; e += NT) {
            uint64_t gidx;
            if (ROLE == kCol) {
                const int k = e / G::C, cc = e % G::C;
                gidx = (uint64_t)k * N2 + first + cc;
            } else if (ROLE == kRow) {
                gidx = (uint64_t)first * G::S + e;
            } else {
                gidx = e;
            }
            if constexpr (LOAD == kPlain)
                lds[e] = fp_reduce(fp_from(src[gidx]), q, qinv);
            else
                lds[e] = fp_reduce(fp_from(load_word<LOAD>(src[gidx], a, a.mod[prime])), q, qinv);
        }
        __syncthreads();
        if (lazy)
            stages_f<LOGS, ROLE, FWD, CW, true, NT, R16>(lds, tw, q, qinv, n, N1, first);
        else
            stages_f<LOGS, ROLE, FWD, CW, false, NT, R16>(lds, tw, q, qinv, n, N1, first);
    }
    const bool scale_out = !FWD && ROLE != kRow;  // the inverse's last pass
    const double ni = a.ninvd[prime];
    for (int e = threadIdx.x; e < G::TILE; e += NT) {
        uint64_t gidx;
        if (ROLE == kCol) {
            const int k = e / G::C, cc = e % G::C;
            gidx = (uint64_t)k * N2 + first + cc;
        } else if (ROLE == kRow) {
            gidx = (uint64_t)first * G::S + e;
        } else {
            gidx = e;
        }
        double v = lds[e];
        if (scale_out)
            v = fp_reduce(fp_mulmod(v, ni, q, qinv), q, qinv);
        else if (lazy)
            v = fp_reduce(v, q, qinv);
        v = v < 0 ? v + q : v;
        if (epi) {
            if (a.epi_int)
                epi_store(a.epi, poly, limb, gidx, fp_to(v), (uint64_t)q, a.limbs, n);
            else
                epi_store_f(a.epi, poly, limb, gidx, v, q, qinv, a.limbs, n);
        } else {
            data[gidx] = fp_to(v);
        }
    }
}

template <int LOGS, int ROLE, bool FWD, int CW, bool R16, int NT, int LOAD>
__device__ __forceinline__ void ntt_pass(const NttKArgs &a)
{
    using G = Geometry<LOGS, ROLE, CW>;
    __shared__ uint64_t lds[G::TILE];
    const uint32_t bidx = blockIdx.y;
    const uint32_t poly = bidx / a.limbs, limb = bidx - poly * a.limbs;
    if (a.skip_alpha) {  // uniform per workgroup, before any barrier
        const uint32_t I = poly % a.poly_period;
        if (I < a.skip_l && I / a.skip_alpha == limb) return;
    }
    const uint32_t prime =
        a.prime_by_poly ? a.prime_of[a.poly_period ? poly % a.poly_period : poly] : a.prime_of[limb];
    const uint32_t n = 1u << a.logn;
    uint64_t *data = a.data + poly * a.poly_stride + (uint64_t)limb * n;
    const uint64_t *src = a.nsrcs ? a.srcs[poly] + (uint64_t)limb * n
                                  : (a.src ? a.src + poly * a.src_poly_stride + (uint64_t)limb * n : data);
    if (LOAD == kLift) src = a.in + ((uint64_t)(poly / a.poly_period) * a.limbs + limb) * n;
    if (LOAD == kCenter) src = a.in + poly * a.in_stride;
    const ulonglong2 *tw = a.tw + (uint64_t)prime * n;
    const uint64_t q = a.mod[prime].q;
    const uint32_t N2 = ROLE == kCol ? (n >> LOGS) : (ROLE == kRow ? (uint32_t)G::S : n);
    const uint32_t N1 = n / N2;
    // Column tiles share 128-byte lines with their neighbours (CW x 8 bytes per
    // row).  Workgroups go to the 8 XCDs round-robin, so consecutive tiles are
    // given to workgroups on the same XCD (one L2) when the grid allows.
    uint32_t tile = blockIdx.x;
    if (ROLE == kCol && (gridDim.x & 7) == 0) tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const uint32_t first = tile * G::C;  // first column / row of the tile
    if (q < kFpPrime) {
        ntt_tile_f<LOGS, ROLE, FWD, CW, R16, NT, LOAD>(a, lds, data, src, prime, n, N2, N1, first, poly, limb);
        return;
    }

    // ---- load
    for (int e = threadIdx.x; e < G::TILE; e += NT) {
        uint64_t gidx;
        if (ROLE == kCol) {
            const int k = e / G::C, cc = e % G::C;
            gidx = (uint64_t)k * N2 + first + cc;
        } else if (ROLE == kRow) {
            gidx = (uint64_t)first * G::S + e;
        } else {
            gidx = e;
        }
        lds[e] = LOAD == kPlain ? src[gidx] : load_word<LOAD>(src[gidx], a, a.mod[prime]);
    }
    __syncthreads();

    if (FWD) {
        const uint32_t m0 = ROLE == kRow ? N1 : 1u;
        int s = 0;
        if constexpr (LOGS >= 3) {
#pragma unroll
            for (int st = 0; st < LOGS / 3; st++) {
                fwd_step<LOGS, ROLE, 3, CW, NT>(lds, s, tw, q, m0, first);
                s += 3;
                __syncthreads();
            }
        }
        if constexpr (LOGS % 3 == 2) {
            fwd_step<LOGS, ROLE, 2, CW, NT>(lds, s, tw, q, m0, first);
            __syncthreads();
        } else if constexpr (LOGS % 3 == 1) {
            fwd_step<LOGS, ROLE, 1, CW, NT>(lds, s, tw, q, m0, first);
            __syncthreads();
        }
    } else {
        const uint32_t mx = ROLE == kCol ? N1 : n;
        int s = 0;
        if constexpr (LOGS >= 3) {
#pragma unroll
            for (int st = 0; st < LOGS / 3; st++) {
                inv_step<LOGS, ROLE, 3, CW, NT>(lds, s, tw, q, n, mx, first);
                s += 3;
                __syncthreads();
            }
        }
        if constexpr (LOGS % 3 == 2) {
            inv_step<LOGS, ROLE, 2, CW, NT>(lds, s, tw, q, n, mx, first);
            __syncthreads();
        } else if constexpr (LOGS % 3 == 1) {
            inv_step<LOGS, ROLE, 1, CW, NT>(lds, s, tw, q, n, mx, first);
            __syncthreads();
        }
    }

    // ---- store (final reduction on the last pass)
    const bool last_pass = FWD ? (ROLE != kCol) : (ROLE != kRow);
    const bool epi = FWD && ROLE != kCol && epi_on(a.epi);
    const ulonglong2 ni = a.ninv[prime];
    for (int e = threadIdx.x; e < G::TILE; e += NT) {
        uint64_t gidx;
        if (ROLE == kCol) {
            const int k = e / G::C, cc = e % G::C;
            gidx = (uint64_t)k * N2 + first + cc;
        } else if (ROLE == kRow) {
            gidx = (uint64_t)first * G::S + e;
        } else {
            gidx = e;
        }
        uint64_t v = lds[e];
        if (last_pass) {
            if (FWD) {
                v = v >= 2 * q ? v - 2 * q : v;
                v = v >= q ? v - q : v;
            } else {
                v = shoup(v, ni.x, ni.y, q);
            }
        }
        if (epi)
            epi_store(a.epi, poly, limb, gidx, v, q, a.limbs, n);
        else
            data[gidx] = v;
    }
}

template <int LOGS, int ROLE, bool FWD, int CW, bool R16, int NT, int LOAD>
__global__ __launch_bounds__(NT) void k_ntt(NttKArgs a)
{
    ntt_pass<LOGS, ROLE, FWD, CW, R16, NT, LOAD>(a);
}

// The inverse's column pass of a tile, on the 8 words of a thread in the order the
// conversions hold them; fully reduced to [0, q).  lds: 2048 doubles that no
// other thread still reads.
template <int LOGS>
__device__ __forceinline__ void col_inverse(double *x, double *lds, const double *tw, double ninv, double q,
                                            double qinv, uint32_t n, uint32_t col0)
{
    using C = ColTile<LOGS>;
    const int tid = threadIdx.x;
#pragma unroll
    for (int k = 0; k < 8; k++) lds[C::row_in(tid, k) * C::CW + tid % C::CW] = fp_reduce(x[k], q, qinv);
    __syncthreads();
    stages_f<LOGS, kCol, false, C::CW, false, kThreads, false>(lds, tw, q, qinv, n, 1u << LOGS, col0);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const double v = fp_reduce(fp_mulmod(lds[C::row_in(tid, k) * C::CW + tid % C::CW], ninv, q, qinv), q, qinv);
        x[k] = v < 0 ? v + q : v;
    }
}

// ---- ModUp base conversion fused into the forward column pass
//
// Workgroup (tile, b, digit j, chunk): the digit's A input limbs are read once
// over the tile (8 columns x 2^LOGS rows) and their products y_k = [x_k
// Dhat_k^-1]_(q_k) kept in registers; then for each output prime I of the
// chunk (the primes outside the digit) the converted values sum_k y_k f_(k,I)
// are written to LDS and transformed by the column stages of prime I, and the
// column-transformed limb is stored into T[b][I][j].  The conversion of
// T's limb is never written and read back.  Every prime below 2^51: the
// products are the exact double-precision ones of the unfused conversion
// (k_modup_conv_a), and the column stages those of the double-precision pass,
// so the stored words equal the unfused conversion followed by the column pass.
struct ModUpColArgs {
    const double *invd, *ninvd;  // the inverse's tables (INV)
    uint64_t *T;
    const uint64_t *coef;
    const ulonglong2 *w;
    const double *convd;
    const double2 *qd;
    const double *twd;
    uint32_t l, digits, nout, key_limbs, logn, chunk, chunks;
    uint32_t outp[kMaxPrimes];  // words: uniform indices take scalar loads
};

// RAW: the values are left as doubles for k_row_inner instead of as words.
// S: the inputs of the digit at hand (A, or half of it for a short last digit).
// The order of the loop hides the latencies behind arithmetic: an output's
// twiddles are asked for before its conversion, the next output's factors
// before the current one's stages.
// INV: the inputs come from the inverse's row pass; its column pass runs here.
template <int LOGS, int A, int S, bool RAW, bool INV>
__device__ __forceinline__ void modup_tile(const ModUpColArgs &a, double *lds, uint32_t b, uint32_t j, uint32_t s,
                                           uint32_t r0, uint32_t r1)
{
    using C = ColTile<LOGS>;
    const uint32_t n = 1u << a.logn;
    const uint32_t N2 = n >> LOGS;
    const uint32_t first = j * A;
    const uint32_t col0 = xcd_tile(blockIdx.x, gridDim.x) * C::CW;
    const int tid = threadIdx.x;
    const uint32_t at = (uint32_t)(tid / C::CW) * N2 + col0 + tid % C::CW;
    // the digit's products [x Dhat^-1]_q in [0, q) (rows i >= s stay zero)
    const uint32_t base = (j * A + s - 1) * A;
    double y[S][8];
    double qmax = 0.0;
#pragma unroll
    for (int i = 0; i < S; i++) {
        const bool on = (uint32_t)i < s;
        const uint32_t p = on ? first + i : first;
        const double q = a.qd[p].x, qinv = a.qd[p].y;
        qmax = q > qmax ? q : qmax;
        const double wi = (double)a.w[base + (on ? i : 0)].x;
        const uint64_t *x = a.coef + ((uint64_t)b * a.l + p) * n;
#pragma unroll
        for (int k = 0; k < 8; k++) y[i][k] = fp_from((x + C::row_step(k) * N2)[at]);
        if (INV && on)  // uniform
            col_inverse<LOGS>(y[i], lds + (i & 1) * C::LDS, a.invd + (uint64_t)p * n, a.ninvd[p], q, qinv, n, col0);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            double v = fp_reduce(fp_mulmod(y[i][k], wi, q, qinv), q, qinv);
            v = v < 0 ? v + q : v;
            y[i][k] = on ? v : 0.0;
        }
    }
    if (INV) __syncthreads();  // the last input's buffer may be the first output's
    const double *factors = a.convd + (uint64_t)base * a.key_limbs;
    auto prime = [&](uint32_t r) { return a.outp[r < first ? r : r + s]; };
    double f[S], q, qinv;
    auto load_factors = [&](uint32_t kp) {
#pragma unroll
        for (int i = 0; i < S; i++) f[i] = table_at(factors, (uint64_t)i * a.key_limbs + kp);
        table_prime(a.qd, kp, q, qinv);
    };
    load_factors(prime(r0));
    ColTwiddles<LOGS> tw, next;
    next.load_lane(a.twd + (uint64_t)prime(r0) * n);
    uint32_t buf = 0;
    for (uint32_t r = r0; r < r1; r++, buf ^= 1) {
        const uint32_t I = r < first ? r : r + s;
        const double qc = q, qic = qinv;
        tw = next;
        tw.load_uniform(a.twd + (uint64_t)prime(r) * n);
        __builtin_amdgcn_sched_barrier(0);
        double cv[8];
        conv_tile<S>(cv, &y[0][0], f, qc, qic, qmax * qc <= 0x1p97);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t kn = prime(min(r + 1, r1 - 1));
        load_factors(kn);
        next.load_lane(a.twd + (uint64_t)kn * n);
        __builtin_amdgcn_sched_barrier(0);
        col_forward<LOGS, RAW>(cv, lds + buf * C::LDS, tw, qc, qic, (int)a.logn, N2, col0,
                               a.T + (((uint64_t)b * a.nout + I) * a.digits + j) * n);
    }
}

template <int LOGS, int A, bool RAW, bool INV>
__global__ __launch_bounds__(kThreads, A <= 9 ? 2 : 1) void k_modup_col(ModUpColArgs a)
{
    __shared__ double lds[2 * ColTile<LOGS>::LDS];
    const uint32_t row = blockIdx.y;  // (b * digits + j) * chunks + chunk
    const uint32_t bj = row / a.chunks, chunk = row - bj * a.chunks;
    const uint32_t b = bj / a.digits, j = bj - b * a.digits;
    const uint32_t s = min((uint32_t)A, a.l - j * A);
    const uint32_t count = a.nout - s;  // output primes outside the digit
    const uint32_t r0 = chunk * a.chunk;
    if (r0 >= count) return;  // uniform, before any barrier
    const uint32_t r1 = min(count, r0 + a.chunk);
    if (A > 4 && s <= A / 2)
        modup_tile<LOGS, A, A / 2, RAW, INV>(a, lds, b, j, s, r0, r1);
    else
        modup_tile<LOGS, A, A, RAW, INV>(a, lds, b, j, s, r0, r1);
}

// ---- Rescale centring fused into the forward column pass
//
// Workgroup (tile, poly p, chunk): the INTT'd last limb of poly p (prime p_l,
// [0, p_l)) is read once over the tile; each output prime q_i of the chunk
// gets (x + (p_l - 1)/2) mod p_l - (p_l - 1)/2 (SEAL's centred remainder,
// an integer of magnitude below 2^51, exact in double precision) reduced mod
// q_i, transformed by the column stages of q_i, stored into z[p][i].  The
// words equal a transform's with that load (NttBatch::center).  Every prime below
// 2^51.
struct CenterColArgs {
    uint64_t *z;
    const uint64_t *last;
    uint64_t last_stride;
    const double2 *qd;
    const double *twd;
    uint64_t p, half;
    uint32_t limbs, logn, chunk, chunks;
};

template <int LOGS>
__global__ __launch_bounds__(kThreads) void k_center_col(CenterColArgs a)
{
    using C = ColTile<LOGS>;
    __shared__ double lds[2 * C::LDS];
    const uint32_t n = 1u << a.logn;
    const uint32_t N2 = n >> LOGS;
    const uint32_t p = blockIdx.y / a.chunks, chunk = blockIdx.y - p * a.chunks;
    const uint32_t i0 = chunk * a.chunk;
    if (i0 >= a.limbs) return;  // uniform, before any barrier
    const uint32_t i1 = min(a.limbs, i0 + a.chunk);
    const uint32_t col0 = xcd_tile(blockIdx.x, gridDim.x) * C::CW;
    const int tid = threadIdx.x;
    double v[8];
    const uint32_t at = (uint32_t)(tid / C::CW) * N2 + col0 + tid % C::CW;
    const uint64_t *x = a.last + (uint64_t)p * a.last_stride;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        uint64_t u = (x + C::row_step(k) * N2)[at] + a.half;
        u = u >= a.p ? u - a.p : u;
        v[k] = fp_from(u) - fp_from(a.half);
    }
    uint32_t buf = 0;
    ColTwiddles<LOGS> tw, next;
    next.load_lane(a.twd + (uint64_t)i0 * n);
    for (uint32_t i = i0; i < i1; i++, buf ^= 1) {
        double q, qinv;
        table_prime(a.qd, i, q, qinv);
        tw = next;
        tw.load_uniform(a.twd + (uint64_t)i * n);
        double cv[8];
#pragma unroll
        for (int k = 0; k < 8; k++) cv[k] = fp_reduce(v[k], q, qinv);
        next.load_lane(a.twd + (uint64_t)min(i + 1, i1 - 1) * n);
        col_forward<LOGS, false>(cv, lds + buf * C::LDS, tw, q, qinv, (int)a.logn, N2, col0,
                                 a.z + ((uint64_t)p * a.limbs + i) * n);
    }
}

// ---- ModDown base conversion fused into the forward column pass
//
// Workgroup (tile, poly p, chunk): the A input limbs at limbs lo .. lo + A - 1
// of poly p of acc (coefficient form) are read once over the tile; per
// position v_k = [y_k w_k]_(p_k) (as k_moddown_conv_a) and the
// centring quotient r = floor(sum_k v_k / p_k + 1/2) stay in registers; each
// output prime q_i (i < lo) of the chunk gets sum_k v_k f_(k,i) - r (P mod q_i)
// in exact double-precision products, transformed by the column stages of q_i
// and stored into z[p][i].  The words equal the unfused conversion followed
// by the column pass.  Every prime below 2^51.
struct ModDownColArgs {
    const double *invd, *ninvd;  // the inverse's tables (INV)
    uint64_t *z;
    const uint64_t *acc;
    uint64_t acc_stride;
    const ulonglong2 *w;
    const double *convd;
    const double2 *qd;
    const double *twd;
    uint32_t lo, L, logn, chunk, chunks;
    uint32_t inp[kMaxPrimes];
};

template <int LOGS, int A, bool INV>
__global__ __launch_bounds__(kThreads, A <= 9 ? 2 : 1) void k_moddown_col(ModDownColArgs a)
{
    using C = ColTile<LOGS>;
    __shared__ double lds[2 * C::LDS];
    const uint32_t n = 1u << a.logn;
    const uint32_t N2 = n >> LOGS;
    const uint32_t p = blockIdx.y / a.chunks, chunk = blockIdx.y - p * a.chunks;
    const uint32_t i0 = chunk * a.chunk;
    if (i0 >= a.lo) return;  // uniform, before any barrier
    const uint32_t i1 = min(a.lo, i0 + a.chunk);
    const uint32_t col0 = xcd_tile(blockIdx.x, gridDim.x) * C::CW;
    const int tid = threadIdx.x;
    const uint32_t at = (uint32_t)(tid / C::CW) * N2 + col0 + tid % C::CW;
    const uint64_t *y = a.acc + (uint64_t)p * a.acc_stride + (uint64_t)a.lo * n;
    double v[A][8], rr[8];
    double pmax = 0.0;
#pragma unroll
    for (int k = 0; k < 8; k++) rr[k] = 0.0;
#pragma unroll
    for (int i = 0; i < A; i++) {
        const double wi = (double)a.w[i].x;
        const double pi = a.qd[a.inp[i]].x, pinv = a.qd[a.inp[i]].y;
        pmax = pi > pmax ? pi : pmax;
#pragma unroll
        for (int k = 0; k < 8; k++) v[i][k] = fp_from((y + (uint64_t)i * n + C::row_step(k) * N2)[at]);
        if (INV)
            col_inverse<LOGS>(v[i], lds + (i & 1) * C::LDS, a.invd + (uint64_t)a.inp[i] * n, a.ninvd[a.inp[i]], pi,
                              pinv, n, col0);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            double x = fp_reduce(fp_mulmod(v[i][k], wi, pi, pinv), pi, pinv);
            x = x < 0 ? x + pi : x;
            // x / p_i correctly rounded: pinv is the correctly rounded 1 / p_i, so
            // one residual step on x pinv gives the quotient a division gives
            const double d = x * pinv;
            rr[k] += __builtin_fma(__builtin_fma(-d, pi, x), pinv, d);
            v[i][k] = x;
        }
    }
#pragma unroll
    for (int k = 0; k < 8; k++) rr[k] = __builtin_floor(rr[k] + 0.5);  // <= A
    if (INV) __syncthreads();  // the last input's buffer may be the first output's
    double f[A + 1], q, qinv;
    auto load_factors = [&](uint32_t i) {
#pragma unroll
        for (int k = 0; k <= A; k++) f[k] = table_at(a.convd, (uint64_t)k * a.L + i);
        table_prime(a.qd, i, q, qinv);
    };
    load_factors(i0);
    ColTwiddles<LOGS> tw;
    uint32_t buf = 0;
    for (uint32_t i = i0; i < i1; i++, buf ^= 1) {
        const double qc = q, qic = qinv;
        tw.load_lane(a.twd + (uint64_t)i * n);
        tw.load_uniform(a.twd + (uint64_t)i * n);
        __builtin_amdgcn_sched_barrier(0);
        double cv[8];
        conv_tile<A>(cv, &v[0][0], f, qc, qic, pmax * qc <= 0x1p97);
        // - r (P mod q_i) as r times the centred q_i - P mod q_i
#pragma unroll
        for (int k = 0; k < 8; k++) cv[k] = fp_reduce(cv[k] + fp_mulmod(rr[k], f[A], qc, qic), qc, qic);
        __builtin_amdgcn_sched_barrier(0);
        load_factors(min(i + 1, i1 - 1));
        __builtin_amdgcn_sched_barrier(0);
        col_forward<LOGS, false>(cv, lds + buf * C::LDS, tw, qc, qic, (int)a.logn, N2, col0,
                                 a.z + ((uint64_t)p * a.lo + i) * n);
    }
}

// The forward column pass with 8-wide tiles held to 64 VGPRs: 8 waves per SIMD
// instead of 7 (the other passes reach 8 as they are, or would spill).
template <int LOGS, int ROLE, bool FWD, int CW, bool R16>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(8))) void k_ntt_w8(NttKArgs a)
{
    ntt_pass<LOGS, ROLE, FWD, CW, R16, kThreads, kPlain>(a);
}

template <int LOGS, int ROLE, bool FWD, int CW = 16, bool R16 = false, int LOAD = kPlain>
void launch_one(const NttKArgs &a, uint32_t batch, hipStream_t s)
{
    using G = Geometry<LOGS, ROLE, CW>;
    const uint32_t n = 1u << a.logn;
    const uint32_t tiles = ROLE == kWhole ? 1u : (n / G::TILE);
    dim3 grid(tiles, batch);
    static const char *names[2][3] = {{"ntt_inv_whole", "ntt_inv_col", "ntt_inv_row"},
                                      {"ntt_fwd_whole", "ntt_fwd_col", "ntt_fwd_row"}};
    // algorithmic bytes: each limb read + written once (16 n) plus the pass's
    // twiddle entries: {w, w'} (16 B) on the 64-bit path, w (8 B) in double
    // precision
    const double tw = ROLE == kWhole ? (double)n : (ROLE == kCol ? (double)G::S : (double)(n - n / G::S));
    // with an epilogue the last pass also reads x (and base or out) per word
    const bool epi = FWD && ROLE != kCol && epi_on(a.epi);
    const double epi_reads =
        a.epi.out ? (a.epi.accumulate ? 1.0 : 0.0) : ((a.epi.a0 || a.epi.a0s[0]) ? 0.5 : 0.0) + (a.epi.d ? 1.0 : 0.0);
    const double epi_bytes = epi ? 8.0 * n * (1.0 + epi_reads) : 0.0;
    ProfScope prof(epi ? "ntt_fwd_sub_mul" : names[FWD ? 1 : 0][ROLE], s,
                   (double)(batch - a.skipped) * (16.0 * n + a.tw_bytes * tw + epi_bytes));
    // a whole limb of 2^13 words leaves room for two workgroups on a CU: one
    // radix-8 group a thread fills it (177 limbs of 60 bits: 22.4 us, with 512
    // threads 26.3; 256 threads took 40 us for any number up to 256)
    constexpr int NT = ROLE != kWhole || LOGS < 12 ? kThreads : (LOGS == 12 ? 512 : 1024);
    if constexpr (ROLE == kCol && FWD && CW == 8 && !R16 && LOAD == kPlain)
        hipLaunchKernelGGL((k_ntt_w8<LOGS, ROLE, FWD, CW, R16>), grid, dim3(kThreads), 0, s, a);
    else
        hipLaunchKernelGGL((k_ntt<LOGS, ROLE, FWD, CW, R16, NT, LOAD>), grid, dim3(NT), 0, s, a);
}

template <bool FWD, int LOAD = kPlain>
void launch_whole(const NttKArgs &a, uint32_t batch, hipStream_t s)
{
    switch (a.logn) {
#define NX_CASE(L) \
    case L: launch_one<L, kWhole, FWD, 16, false, LOAD>(a, batch, s); break;
        NX_CASE(1) NX_CASE(2) NX_CASE(3) NX_CASE(4) NX_CASE(5) NX_CASE(6) NX_CASE(7)
        NX_CASE(8) NX_CASE(9) NX_CASE(10) NX_CASE(11) NX_CASE(12) NX_CASE(13)
#undef NX_CASE
    default: break;
    }
}

// Epilogue arithmetic of the double-precision path (0: exact double-precision
// products, 1: 64-bit integer Shoup products; the same words).  Set by the autotuner.
std::atomic<int> g_epi_int{0};

// Tile widths chosen by the autotuner: [log n - 14][pass][direction][batch bucket],
// 0 = the default (tiles of 8).  Written by ntt_set_tile, read at every launch.
std::atomic<int> g_tile[kTuneLogN][2][2][kTuneBuckets];
// Radix of the double-precision passes, same indexing: 0 = radix-8 steps, 1 =
// radix-16 steps (the integer path always takes radix 8).  Set by the autotuner.
std::atomic<int> g_radix[kTuneLogN][2][2][kTuneBuckets];

int tune_bucket(uint32_t batch)
{
    int b = 0;
    while (b + 1 < kTuneBuckets && (2u << b) <= batch) b++;
    return b;  // floor(log2(batch)), capped
}

template <int LOGS, int ROLE, bool FWD, bool R16>
void launch_width(int cw, const NttKArgs &a, uint32_t batch, hipStream_t s)
{
    if (cw == 4)
        launch_one<LOGS, ROLE, FWD, 4, R16>(a, batch, s);
    else if (cw == 8)
        launch_one<LOGS, ROLE, FWD, 8, R16>(a, batch, s);
    else
        launch_one<LOGS, ROLE, FWD, 16, R16>(a, batch, s);
}

template <int LOGS, int ROLE, bool FWD>
void launch_sized(const NttKArgs &a, uint32_t batch, hipStream_t s)
{
    int cw = 0, r16 = 0;
    const int li = (int)a.logn - kTuneLogNMin;
    if (li >= 0 && li < kTuneLogN) {
        cw = g_tile[li][ROLE == kCol ? 0 : 1][FWD ? 1 : 0][tune_bucket(batch)].load();
        r16 = g_radix[li][ROLE == kCol ? 0 : 1][FWD ? 1 : 0][tune_bucket(batch)].load();
    }
    if (!cw) cw = 8;
    if (r16)
        launch_width<LOGS, ROLE, FWD, true>(cw, a, batch, s);
    else
        launch_width<LOGS, ROLE, FWD, false>(cw, a, batch, s);
}

template <int ROLE, bool FWD>
void launch_pass(int logs, const NttKArgs &a, uint32_t batch, hipStream_t s)
{
    switch (logs) {
    case 6: launch_one<6, ROLE, FWD, 8>(a, batch, s); break;
    case 7: launch_sized<7, ROLE, FWD>(a, batch, s); break;
    case 8: launch_sized<8, ROLE, FWD>(a, batch, s); break;
    case 9: launch_sized<9, ROLE, FWD>(a, batch, s); break;
    default: break;
    }
}

// The first pass of a forward transform with a load of its own: tiles of 8, radix 8
// (the words do not depend on either).
template <int LOAD>
void launch_load_col(int logs, const NttKArgs &a, uint32_t batch, hipStream_t s)
{
    switch (logs) {
    case 6: launch_one<6, kCol, true, 8, false, LOAD>(a, batch, s); break;
    case 7: launch_one<7, kCol, true, 8, false, LOAD>(a, batch, s); break;
    case 8: launch_one<8, kCol, true, 8, false, LOAD>(a, batch, s); break;
    default: break;
    }
}

NttKArgs make_args(const DeviceTables &t, const NttBatch &b, bool fwd)
{
    NttKArgs a;
    a.data = b.data;
    a.poly_stride = b.poly_stride;
    a.src = b.src;
    a.src_poly_stride = b.src_poly_stride;
    a.nsrcs = 0;
    for (int i = 0; i < kNttSrcMax; i++) a.srcs[i] = nullptr;
    {
        // limbs whose prime takes the double-precision path read 8-byte twiddles
        const uint32_t m = b.prime_by_poly ? (b.poly_period ? b.poly_period : b.polys) : b.limbs;
        const uint32_t cnt = m < (uint32_t)kMaxPrimes ? m : (uint32_t)kMaxPrimes;
        uint32_t fp = 0;
        for (uint32_t i = 0; i < cnt; i++) fp += t.mod_host[b.prime_of[i]] < kFpPrime ? 1u : 0u;
        a.tw_bytes = cnt ? (8.0 * fp + 16.0 * (cnt - fp)) / cnt : 16.0;
    }
    if (b.src_list) {
        // a source per poly: the batch must fit the argument array
        if (b.polys > (uint32_t)kNttSrcMax) throw std::invalid_argument("ntt: too many sources in one batch");
        a.nsrcs = b.polys;
        for (uint32_t i = 0; i < b.polys; i++) a.srcs[i] = b.src_list[i];
    }
    a.epi = b.epi;
    a.epi_int = (uint32_t)g_epi_int.load();
    a.in = nullptr;
    a.in_stride = 0;
    a.in_prime = 0;
    if (!fwd) {
        a.epi.out = nullptr;
        a.epi.outs[0] = nullptr;
    }
    a.skip_l = a.skip_alpha = a.skipped = 0;
    if (b.skip_alpha && b.prime_by_poly && b.poly_period) {
        a.skip_l = b.skip_l;
        a.skip_alpha = b.skip_alpha;
        for (uint32_t I = 0; I < b.skip_l && I < b.poly_period; I++)
            if (I / b.skip_alpha < b.limbs) a.skipped += b.polys / b.poly_period;
    }
    a.limbs = b.limbs;
    a.logn = (uint32_t)t.logn;
    a.prime_by_poly = b.prime_by_poly;
    a.poly_period = b.poly_period;
    a.tw = fwd ? t.fwd : t.inv;
    a.mod = t.mod;
    a.qd = t.qd;
    a.ninv = t.ninv;
    a.twd = fwd ? t.fwd_d : t.inv_d;
    a.ninvd = t.ninv_d;
    for (int i = 0; i < kMaxPrimes; i++) a.prime_of[i] = b.prime_of[i];
    return a;
}

}  // namespace

// Split of log2(n) into column (N1) and row (N2) passes for n >= 2^14.
static inline void split_logn(int logn, int &l1, int &l2)
{
    l1 = logn / 2;
    l2 = logn - l1;
}

void ntt_set_epilogue_int(bool on) { g_epi_int.store(on ? 1 : 0); }
bool ntt_get_epilogue_int() { return g_epi_int.load() != 0; }

void ntt_set_tile(int logn, int pass, bool fwd, uint32_t batch, int width)
{
    const int li = logn - kTuneLogNMin;
    if (li < 0 || li >= kTuneLogN || pass < 0 || pass > 1) return;
    if (width != 0 && width != 4 && width != 8 && width != 16) return;
    g_tile[li][pass][fwd ? 1 : 0][tune_bucket(batch)].store(width);
}

void ntt_set_radix16(int logn, int pass, bool fwd, uint32_t batch, bool on)
{
    const int li = logn - kTuneLogNMin;
    if (li < 0 || li >= kTuneLogN || pass < 0 || pass > 1) return;
    g_radix[li][pass][fwd ? 1 : 0][tune_bucket(batch)].store(on ? 1 : 0);
}

bool ntt_get_radix16(int logn, int pass, bool fwd, uint32_t batch)
{
    const int li = logn - kTuneLogNMin;
    if (li < 0 || li >= kTuneLogN || pass < 0 || pass > 1) return false;
    return g_radix[li][pass][fwd ? 1 : 0][tune_bucket(batch)].load() != 0;
}

int ntt_get_tile(int logn, int pass, bool fwd, uint32_t batch)
{
    const int li = logn - kTuneLogNMin;
    if (li < 0 || li >= kTuneLogN || pass < 0 || pass > 1) return 0;
    return g_tile[li][pass][fwd ? 1 : 0][tune_bucket(batch)].load();
}

// Rings of 2^14 and above always run in two passes.  A limb of 2^13 words held
// by one workgroup takes its time on one CU however few limbs there are (60-bit
// primes: 17 us, 46-bit: 12.5 us for 3 to 48 limbs); cut into passes of 64 x 128
// it takes 11.6 and 9.6 us.  The two cross between 48 limbs (17.9 / 14.2 us and
// 13.3 / 11.9 us) and 96 (18.7 / 17.6, 13.8 / 15.4).  At 2^12 one workgroup is
// never behind (10.3 us against 10.1 for 3 limbs, 11.2 against 12.4 for 96).
static bool two_passes(int logn, uint32_t batch) { return logn >= 14 || (logn == 13 && batch <= 64); }

void ntt_forward(const DeviceTables &t, const NttBatch &b, hipStream_t s)
{
    const uint32_t batch = b.polys * b.limbs;
    if (!batch) return;
    NttKArgs a = make_args(t, b, true);
    const int load = b.lift ? kLift : b.center ? kCenter : kPlain;
    if (load == kLift && (!b.prime_by_poly || !b.poly_period || b.polys % b.poly_period))
        throw std::invalid_argument("ntt: a lift needs a prime per poly of a period");
    if (load != kPlain && (b.rows_only || b.src || b.src_list || b.skip_alpha))
        throw std::invalid_argument("ntt: a lift or centring is the only source of a whole transform");
    a.in = b.lift ? b.lift : b.center;
    a.in_stride = b.center_stride;
    a.in_prime = b.center_prime;
    if (!two_passes(t.logn, batch)) {
        if (load == kLift)
            launch_whole<true, kLift>(a, batch, s);
        else if (load == kCenter)
            launch_whole<true, kCenter>(a, batch, s);
        else
            launch_whole<true>(a, batch, s);
    } else {
        int l1, l2;
        split_logn(t.logn, l1, l2);
        if (load == kLift)
            launch_load_col<kLift>(l1, a, batch, s);
        else if (load == kCenter)
            launch_load_col<kCenter>(l1, a, batch, s);
        else if (!b.rows_only)
            launch_pass<kCol, true>(l1, a, batch, s);
        a.src = nullptr;  // the second pass runs in place on the output
        a.nsrcs = 0;
        launch_pass<kRow, true>(l2, a, batch, s);
    }
}

// Algorithmic double-precision operations (an FMA counts two, rint one) of the
// fused column kernels: an exact product (mul, fma, mul, rint, fma, add) is 8, a
// reduction (mul, rint, fma) 4.  A conversion to one output word is a term of
// FpSum an input (two fma, a subtraction, an addition: 6), a quotient every eight
// (conv_sum's narrow form: subtraction, mul, rint, fma, addition: 6), a sum and a
// reduction between them and a reduction at the end.  A column pass is half a
// butterfly (a product, an addition and a subtraction) per word and stage; stores
// as words reduce once more, and the inverse's takes a reduction on load and the
// reduced product with n^-1.
constexpr double kFlopsProduct = 8.0, kFlopsReduce = 4.0;
inline double conv_flops(uint32_t A)
{
    const uint32_t sums = (A + 7) / 8;
    return 6.0 * A + 6.0 * sums + (sums - 1) * (1.0 + kFlopsReduce) + kFlopsReduce;
}
inline double col_flops(int logs) { return logs * (kFlopsProduct + 2.0) / 2.0; }
// one input word: its reduced product with a constant, and the inverse's column pass
inline double input_flops(int logs, bool inverse)
{
    return kFlopsProduct + kFlopsReduce +
           (inverse ? col_flops(logs) + kFlopsReduce + kFlopsProduct + kFlopsReduce : 0.0);
}

// Fused ModUp column pass of a stored ModUp, per power-of-two bucket of the batch
// size B: 0 = on (outputs per workgroup by the default rule), -1 = off (conversion
// and column pass as separate launches), k > 0 = on with k outputs per workgroup.
// Process-wide; set by the autotuner.
static std::atomic<int> g_modup_col[kTuneBuckets];
// The same for the digits of key switches without a stored ModUp, which have no
// separate form: 0 = the default rules (the inverse's column pass included where
// ks_modup_col_inverse says so), k > 0 = k outputs per workgroup of the plain form.
static std::atomic<int> g_digits_col[kTuneBuckets];
constexpr int kColMaxA = 12;   // largest digit / special-prime count of the fused conversions

void ks_modup_col_set(uint32_t B, int mode) { g_modup_col[tune_bucket(B)].store(mode); }

void ks_digits_col_set(uint32_t B, int mode) { g_digits_col[tune_bucket(B)].store(mode); }

int ks_modup_col_get(uint32_t B) { return g_modup_col[tune_bucket(B)].load(); }

bool ks_modup_col_ok(const DeviceTables &t, uint32_t alpha)
{
    return t.max_bits <= 51 && alpha >= 2 && alpha <= kColMaxA && t.logn >= 14 && t.logn <= 17 &&
           t.modup_conv_d != nullptr;
}

// Outputs per workgroup: enough workgroups to fill the device, at least 4
// outputs per read of the digit's inputs.
static uint32_t modup_col_chunk(const DeviceTables &t, uint32_t B, uint32_t l, uint32_t alpha, uint32_t nout, int mode)
{
    const uint32_t tiles = (1u << t.logn) / 2048u, digits = (l + alpha - 1) / alpha;
    const uint32_t count = nout - std::min(alpha, l);  // most outputs of a digit (a partial digit has more)
    const uint32_t want = (2048u + tiles * B * digits - 1) / (tiles * B * digits);
    uint32_t chunk = std::max((count + want - 1) / want, std::min(4u, count));
    if (mode > 0) chunk = std::min((uint32_t)mode, count);  // 0: this rule
    return chunk;
}

// The inverse's column pass belongs in the conversion where one workgroup can
// make all outputs of a digit and there are still kInverseBlocks of them (two
// rounds of the two a CU holds): it saves a read and a write of every input.
// With the outputs cut up each part would repeat it.
// 64 fused products at 20 limbs, N = 2^16: 6.37 ms with the column pass apart,
// 5.99 with it here; with the line at 2048 workgroups and outputs cut up below
// that, 6.14.  Six sums of sixteen rotations: 4.94, 4.80 and 4.91 ms.
// Up to kInverseMaxA inputs: they are all live during the column passes, and from
// ten on the conversions have one wave a SIMD to hide those.  33 fused products
// (apart, here): ten special primes 3.45, 3.57 ms at N = 2^16 and 7.41, 7.72 at
// 2^17; eight 3.35, 3.20 and 7.06, 6.83; 33 plain ones with nine at 2^16 3.60,
// 3.50.  The ModDowns of eight and nine inputs spill (9 over columns of 2^8 40
// words, of 2^7 105), which costs what the pass saves over columns of 2^7: 1.33
// and 1.34 ms at 2^15.
constexpr uint32_t kInverseBlocks = 1024, kInverseMaxA = 9;
bool ks_modup_col_inverse(const DeviceTables &t, uint32_t B, uint32_t l, uint32_t alpha)
{
    return ks_modup_col_ok(t, alpha) && alpha <= kInverseMaxA && l >= 1 && g_digits_col[tune_bucket(B)].load() == 0 &&
           (1u << t.logn) / 2048u * B * ((l + alpha - 1) / alpha) >= kInverseBlocks;
}

void ks_modup_convert_col(const DeviceTables &t, uint64_t *T, const uint64_t *coef, const ulonglong2 *w,
                          uint32_t B, uint32_t l, uint32_t alpha, uint32_t key_limbs, const uint8_t *out_primes_host,
                          uint32_t nout, hipStream_t s, bool raw, bool inverse)
{
    if (!ks_modup_col_ok(t, alpha)) throw std::invalid_argument("ks_modup_convert_col: unsupported parameters");
    if (nout > (uint32_t)kMaxPrimes || l < 1 || nout <= alpha) throw std::invalid_argument("ks_modup_convert_col: bad sizes");
    if (inverse && (!raw || alpha > kInverseMaxA)) throw std::invalid_argument("ks_modup_convert_col: no such form");
    ModUpColArgs a;
    a.T = T;
    a.coef = coef;
    a.w = w;
    a.convd = t.modup_conv_d;
    a.qd = t.qd;
    a.twd = t.fwd_d;
    a.l = l;
    a.digits = (l + alpha - 1) / alpha;
    a.nout = nout;
    a.key_limbs = key_limbs;
    a.logn = (uint32_t)t.logn;
    for (int i = 0; i < kMaxPrimes; i++) a.outp[i] = i < (int)nout ? out_primes_host[i] : 0;
    int l1, l2;
    split_logn(t.logn, l1, l2);
    const uint32_t n = 1u << t.logn;
    const uint32_t tiles = n / 2048u;
    const int mode = (raw ? g_digits_col : g_modup_col)[tune_bucket(B)].load();
    const uint32_t chunk = inverse ? nout - 1 : modup_col_chunk(t, B, l, alpha, nout, mode);
    a.invd = t.inv_d;
    a.ninvd = t.ninv_d;
    a.chunk = chunk;
    a.chunks = (nout - 1 + chunk - 1) / chunk;  // covers a partial last digit (nout - s <= nout - 1 outputs)
    uint32_t outs = 0;
    for (uint32_t j = 0; j < a.digits; j++) outs += nout - std::min(alpha, l - j * alpha);
    ProfScope prof("ks_modup_col", s,
                   8.0 * n * ((double)B * l + (double)B * outs) +
                       8.0 * (double)(1u << l1) * B * (outs + (inverse ? l : 0u)),
                   (double)n * B * (l * input_flops(l1, inverse) +
                                    outs * (conv_flops(alpha) + col_flops(l1) + (raw ? 0.0 : kFlopsReduce))));
    const dim3 grid(tiles, B * a.digits * a.chunks);
#define NX_MC(LOGS, A)                                                                      \
    if (l1 == LOGS && alpha == A) {                                                       \
        if (raw && inverse)                                                               \
            hipLaunchKernelGGL((k_modup_col<LOGS, A, true, (A <= kInverseMaxA)>), grid, dim3(kThreads), 0, s, a); \
        else if (raw)                                                                     \
            hipLaunchKernelGGL((k_modup_col<LOGS, A, true, false>), grid, dim3(kThreads), 0, s, a);  \
        else                                                                              \
            hipLaunchKernelGGL((k_modup_col<LOGS, A, false, false>), grid, dim3(kThreads), 0, s, a); \
        return;                                                                           \
    }
    NX_MC(7, 2) NX_MC(7, 3) NX_MC(7, 4) NX_MC(7, 5) NX_MC(7, 6) NX_MC(7, 7) NX_MC(7, 8) NX_MC(7, 9) NX_MC(7, 10)
    NX_MC(7, 11) NX_MC(7, 12)
    NX_MC(8, 2) NX_MC(8, 3) NX_MC(8, 4) NX_MC(8, 5) NX_MC(8, 6) NX_MC(8, 7) NX_MC(8, 8) NX_MC(8, 9) NX_MC(8, 10)
    NX_MC(8, 11) NX_MC(8, 12)
#undef NX_MC
    throw std::invalid_argument("ks_modup_convert_col: unsupported split");
}

bool center_col_ok(const DeviceTables &t) { return t.max_bits <= 51 && t.logn >= 14 && t.logn <= 17; }

void rns_center_last_col(const DeviceTables &t, uint64_t *z, const uint64_t *last, uint64_t last_stride,
                         uint32_t last_prime, uint32_t polys, uint32_t limbs, hipStream_t s)
{
    if (!center_col_ok(t) || limbs < 1) throw std::invalid_argument("rns_center_last_col: unsupported parameters");
    CenterColArgs a;
    a.z = z;
    a.last = last;
    a.last_stride = last_stride;
    a.qd = t.qd;
    a.twd = t.fwd_d;
    a.p = t.mod_host[last_prime];
    a.half = a.p >> 1;
    a.limbs = limbs;
    a.logn = (uint32_t)t.logn;
    int l1, l2;
    split_logn(t.logn, l1, l2);
    const uint32_t n = 1u << t.logn;
    const uint32_t tiles = n / 2048u;
    const uint32_t want = (2048u + tiles * polys - 1) / (tiles * polys);
    uint32_t chunk = (limbs + want - 1) / want;
    chunk = std::max(chunk, std::min(4u, limbs));
    a.chunk = chunk;
    a.chunks = (limbs + chunk - 1) / chunk;
    ProfScope prof("rescale_col", s, 8.0 * n * polys * (1.0 + limbs) + 8.0 * (double)(1u << l1) * polys * limbs,
                   (double)n * polys * limbs * (2.0 * kFlopsReduce + col_flops(l1)));
    const dim3 grid(tiles, polys * a.chunks);
    if (l1 == 7)
        hipLaunchKernelGGL((k_center_col<7>), grid, dim3(kThreads), 0, s, a);
    else if (l1 == 8)
        hipLaunchKernelGGL((k_center_col<8>), grid, dim3(kThreads), 0, s, a);
    else
        throw std::invalid_argument("rns_center_last_col: unsupported split");
}

static std::atomic<int> g_moddown_col[kTuneBuckets];

void ks_moddown_col_set(uint32_t polys, int mode) { g_moddown_col[tune_bucket(polys)].store(mode); }

int ks_moddown_col_get(uint32_t polys) { return g_moddown_col[tune_bucket(polys)].load(); }

bool ks_moddown_col_ok(const DeviceTables &t, uint32_t A)
{
    return t.max_bits <= 51 && A >= 2 && A <= kColMaxA + 1 && t.logn >= 14 && t.logn <= 17;
}

static uint32_t moddown_col_chunk(const DeviceTables &t, uint32_t polys, uint32_t lo)
{
    const uint32_t tiles = (1u << t.logn) / 2048u;
    const uint32_t want = (2048u + tiles * polys - 1) / (tiles * polys);
    uint32_t chunk = std::max((lo + want - 1) / want, std::min(4u, lo));
    const int mode = g_moddown_col[tune_bucket(polys)].load();
    if (mode > 0) chunk = std::min((uint32_t)mode, lo);
    return chunk;
}

bool ks_moddown_col_inverse(const DeviceTables &t, uint32_t A, uint32_t polys)
{
    return A <= kInverseMaxA && g_moddown_col[tune_bucket(polys)].load() == 0 && (1u << t.logn) / 2048u * polys >= kInverseBlocks;
}

void ks_moddown_convert_col(const DeviceTables &t, uint64_t *z, const uint64_t *acc, uint64_t acc_stride,
                            const ulonglong2 *w, const double *convd, const uint8_t *in_primes_host, uint32_t A,
                            uint32_t polys, uint32_t lo, uint32_t L, hipStream_t s, bool inverse)
{
    if (!ks_moddown_col_ok(t, A) || !convd) throw std::invalid_argument("ks_moddown_convert_col: unsupported parameters");
    if (lo < 1 || lo + A > (uint32_t)kMaxPrimes) throw std::invalid_argument("ks_moddown_convert_col: bad sizes");
    if (inverse && A > kInverseMaxA) throw std::invalid_argument("ks_moddown_convert_col: no such form");
    ModDownColArgs a;
    a.z = z;
    a.acc = acc;
    a.acc_stride = acc_stride;
    a.w = w;
    a.convd = convd;
    a.qd = t.qd;
    a.twd = t.fwd_d;
    a.lo = lo;
    a.L = L;
    a.logn = (uint32_t)t.logn;
    for (int i = 0; i < kMaxPrimes; i++) a.inp[i] = i < (int)A ? in_primes_host[i] : 0;
    int l1, l2;
    split_logn(t.logn, l1, l2);
    const uint32_t n = 1u << t.logn;
    const uint32_t tiles = n / 2048u;
    const uint32_t chunk = inverse ? lo : moddown_col_chunk(t, polys, lo);
    a.invd = t.inv_d;
    a.ninvd = t.ninv_d;
    a.chunk = chunk;
    a.chunks = (lo + chunk - 1) / chunk;
    ProfScope prof("ks_moddown_col", s,
                   8.0 * n * polys * ((double)A + lo) +
                       8.0 * (double)(1u << l1) * polys * (lo + (inverse ? A : 0u)),
                   // an input's share of the quotient: x / p_k (mul, two fma) and an addition; an output's
                   // product with it, an addition and a reduction
                   (double)n * polys * (A * (input_flops(l1, inverse) + 6.0) +
                                        lo * (conv_flops(A) + kFlopsProduct + 1.0 + kFlopsReduce + col_flops(l1) +
                                              kFlopsReduce)));
    const dim3 grid(tiles, polys * a.chunks);
#define NX_MD(LOGS, AA)                                                                     \
    if (l1 == LOGS && A == AA) {                                                          \
        if (inverse)                                                                      \
            hipLaunchKernelGGL((k_moddown_col<LOGS, AA, (AA <= kInverseMaxA)>), grid, dim3(kThreads), 0, s, a); \
        else                                                                              \
            hipLaunchKernelGGL((k_moddown_col<LOGS, AA, false>), grid, dim3(kThreads), 0, s, a); \
        return;                                                                           \
    }
    NX_MD(7, 2) NX_MD(7, 3) NX_MD(7, 4) NX_MD(7, 5) NX_MD(7, 6) NX_MD(7, 7) NX_MD(7, 8) NX_MD(7, 9) NX_MD(7, 10)
    NX_MD(7, 11) NX_MD(7, 12) NX_MD(7, 13)
    NX_MD(8, 2) NX_MD(8, 3) NX_MD(8, 4) NX_MD(8, 5) NX_MD(8, 6) NX_MD(8, 7) NX_MD(8, 8) NX_MD(8, 9) NX_MD(8, 10)
    NX_MD(8, 11) NX_MD(8, 12) NX_MD(8, 13)
#undef NX_MD
    throw std::invalid_argument("ks_moddown_convert_col: unsupported split");
}

void ntt_inverse(const DeviceTables &t, const NttBatch &b, hipStream_t s)
{
    const uint32_t batch = b.polys * b.limbs;
    if (!batch) return;
    NttKArgs a = make_args(t, b, false);
    if (!two_passes(t.logn, batch)) {
        launch_whole<false>(a, batch, s);
    } else {
        int l1, l2;
        split_logn(t.logn, l1, l2);
        launch_pass<kRow, false>(l2, a, batch, s);
        if (b.rows_only) return;
        a.src = nullptr;
        a.nsrcs = 0;
        launch_pass<kCol, false>(l1, a, batch, s);
    }
}

}  // namespace nx
