// Periodic plaintexts and block mixing.
//
// A slot vector that repeats every `period` slots is a polynomial in
// X^(n / B), B = 2 period (rotation by `period` is the automorphism
// X -> X^(5^period), whose fixed ring is spanned by the powers of X^(n / B)).
// In the bit-reversed NTT order the value at position c is the evaluation at
// psi^(2 br(c) + 1), and a polynomial in X^(n / B) only sees that exponent mod
// 2B, i.e. the top log2(B) bits of c: the NTT form is constant over B blocks
// of n / B positions.  A set of such plaintexts is therefore held as
// [limb][block][entry] words, and a product W (.) x costs one word of W per
// block instead of one per position.  Limbs of primes below 2^51 hold them as
// centred doubles, |w| <= q/2.
//
// block_mix computes out[m] = sum_k W[p(m, k)] (.) in[k] for many outputs at
// once: a workgroup stages a 64-position tile of every input polynomial
// through LDS and each wave accumulates whole outputs from it, so every input
// word is read from HBM once however many outputs use it.
#include <vector>

#include "fpmod.h"
#include "kernels.h"
#include "prof.h"

namespace nx {

namespace {

constexpr int kBlock = 256;
constexpr int kTile = 64;  // positions per workgroup (one wave's lanes)

// work[e][i][c] = coef[e][i][c / stride] where c is a multiple of stride, else 0;
// flags cleared
__global__ void k_periodic_scatter(uint64_t *work, uint8_t *flags, const uint64_t *coef, uint32_t blocks,
                                   uint32_t log_stride, uint32_t n)
{
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= n) return;
    const uint64_t row = blockIdx.y;  // e * limbs + i
    const uint32_t stride = 1u << log_stride;
    work[row * n + c] = (c & (stride - 1)) ? 0 : coef[row * blocks + (c >> log_stride)];
    if (c < blocks) flags[row * blocks + c] = 0;
}

// the word held for the residue v, and back
__device__ __forceinline__ uint64_t held(uint64_t v, uint64_t q)
{
    if (q >= kFpPrime) return v;
    return (uint64_t)__double_as_longlong(v > q / 2 ? -fp_from(q - v) : fp_from(v));
}

__device__ __forceinline__ uint64_t residue(uint64_t w, uint64_t q)
{
    if (q >= kFpPrime) return w;
    const double d = __longlong_as_double((long long)w);
    return fp_to(d < 0 ? d + (double)q : d);
}

// table[i][b][e] = work[e][i][b * stride]; flags[e][i][b] = 1 where a position
// of block b differs from its first
__global__ void k_periodic_gather(uint64_t *table, uint8_t *flags, const uint64_t *work, const ModConst *mod,
                                  uint32_t limbs, uint32_t count, uint32_t blocks, uint32_t log_stride, uint32_t n)
{
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= n) return;
    const uint64_t row = blockIdx.y;  // e * limbs + i
    const uint32_t e = blockIdx.y / limbs, i = blockIdx.y - e * limbs;
    const uint32_t b = c >> log_stride;
    const uint64_t v = work[row * n + c], first = work[row * n + ((uint64_t)b << log_stride)];
    if (v != first) flags[row * blocks + b] = 1;
    if ((c & ((1u << log_stride) - 1)) == 0) table[((uint64_t)i * blocks + b) * count + e] = held(v, mod[i].q);
}

// out[i][c] = the residue of table[i][c / stride][index]
__global__ void k_periodic_expand(uint64_t *out, const uint64_t *table, const ModConst *mod, uint32_t index,
                                  uint32_t count, uint32_t blocks, uint32_t log_stride, uint32_t n)
{
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= n) return;
    const uint32_t i = blockIdx.y;
    out[(uint64_t)i * n + c] = residue(table[((uint64_t)i * blocks + (c >> log_stride)) * count + index], mod[i].q);
}

// Three-word accumulator of 64x64-bit products from four 32x32-bit products:
// lo32 + 2^32 mid + 2^64 hi.  With both factors below 2^58, 16 products keep
// every word below 2^64.
struct Acc3 {
    uint64_t lo32 = 0, mid = 0, hi = 0;
    __device__ __forceinline__ void mac(uint64_t a, uint64_t b)
    {
        const uint64_t a0 = (uint32_t)a, a1 = a >> 32, b0 = (uint32_t)b, b1 = b >> 32;
        const uint64_t p00 = a0 * b0;
        lo32 += (uint32_t)p00;
        mid += (p00 >> 32) + a0 * b1 + a1 * b0;
        hi += a1 * b1;
    }
    __device__ __forceinline__ uint64_t reduce(const ModConst &m) const
    {
        const uint64_t ml = mid << 32;
        const uint64_t l = lo32 + ml;
        const uint64_t h = hi + (mid >> 32) + (l < ml);
        return barrett128(h, l, m);
    }
};

// One (poly, limb) row and a tile of 64 positions per workgroup; LDS holds the
// tile of all K inputs and the weights of the tile's blocks.  runs[first[o] ..
// first[o + 1]) list the terms of output o as runs (k0, entry0, len, dentry):
// terms (k0 + j, entry0 + j dentry) for j < len, so the inner loop computes its
// LDS addresses instead of loading them.  FAST: every prime below 2^58
// (products folded every 16 terms through Acc3); otherwise 128-bit sums folded
// every 32 terms.  LIMBS: with both bodies in one kernel long sums below 2^51
// lose 2 % (double precision last, as here) to 5 % (first: 127 inputs to 127
// outputs, scattered, ten limbs at N = 2^16 16.5 ms, alone 15.7), so chains of one
// arithmetic have instances of their own; kWide leaves limbs below 2^51 to
// k_block_mix_quads.
enum Limbs { kEvery = 0, kSmall = 1, kWide = 2 };  // any, all below 2^51, those above
template <bool FAST, int LIMBS>
__global__ __launch_bounds__(kBlock) void k_block_mix(MixPtrs ptrs, const uint64_t *__restrict__ table,
                                                      const int4 *__restrict__ runs,
                                                      const uint32_t *__restrict__ first, const ModConst *mod,
                                                      uint32_t K, uint32_t M, uint32_t limbs, uint32_t count,
                                                      uint32_t blocks, uint32_t log_stride, uint32_t n)
{
    extern __shared__ uint64_t lds[];
    const uint32_t row = blockIdx.y;  // poly * limbs + limb
    const uint32_t limb = row % limbs;
    const uint32_t pos0 = blockIdx.x * kTile;
    const uint32_t bpt = log_stride >= 6 ? 1u : (uint32_t)kTile >> log_stride;  // blocks per tile
    const uint32_t b0 = pos0 >> log_stride;
    uint64_t *xs = lds;               // [K][64]
    uint64_t *ws = lds + K * kTile;   // [count][bpt]
    const uint64_t roff = (uint64_t)row * n + pos0;
    const ModConst m = mod[limb];
    if (LIMBS == kWide && m.q < kFpPrime) return;
    const uint32_t lane = threadIdx.x % kTile;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kTile);
    const uint32_t lb = log_stride >= 6 ? 0u : lane >> log_stride;
    if (LIMBS == kWide || (LIMBS == kEvery && m.q >= kFpPrime)) {
        {
            uint32_t k = wave;
            for (; k + 28 < K; k += 32) {
                uint64_t v[8];
#pragma unroll
                for (int u = 0; u < 8; u++) v[u] = ptrs.in[k + 4 * u][roff + lane];
#pragma unroll
                for (int u = 0; u < 8; u++) xs[(k + 4 * u) * kTile + lane] = v[u];
            }
            for (; k < K; k += 4) xs[k * kTile + lane] = ptrs.in[k][roff + lane];
        }
        for (uint32_t e = threadIdx.x; e < count * bpt; e += kBlock) {
            const uint32_t p = e / bpt, b = e - p * bpt;
            ws[e] = table[((uint64_t)limb * blocks + b0 + b) * count + p];
        }
        __syncthreads();
        for (uint32_t o = wave; o < M; o += kBlock / kTile) {
            uint64_t r = 0;
            Acc3 acc;
            uint64_t lo = 0, hi = 0;
            uint32_t cnt = 0;
            for (uint32_t ri = first[o]; ri < first[o + 1]; ri++) {
                const int4 rn = runs[ri];
                for (int j = 0; j < rn.z; j++) {
                    const uint64_t x = xs[(rn.x + j) * kTile + lane], w = ws[(rn.y + j * rn.w) * (int)bpt + lb];
                    if (FAST) {
                        acc.mac(x, w);
                        if (++cnt == 16) {
                            r = add_mod(r, acc.reduce(m), m.q);
                            acc = Acc3();
                            cnt = 0;
                        }
                    } else {
                        const uint64_t plo = x * w, phi = mulhi64(x, w);
                        lo += plo;
                        hi += phi + (lo < plo);
                        if (++cnt == 32) {
                            r = add_mod(r, barrett128(hi, lo, m), m.q);
                            lo = hi = 0;
                            cnt = 0;
                        }
                    }
                }
            }
            r = FAST ? add_mod(r, acc.reduce(m), m.q) : add_mod(r, barrett128(hi, lo, m), m.q);
            ptrs.out[o][roff + lane] = r;
        }
        return;
    }
    // double precision: the tile and the weights as doubles, one exact
    // product per term, the sum reduced every second term (|sum| < 3 q)
    double *xd = reinterpret_cast<double *>(xs), *wd = reinterpret_cast<double *>(ws);
    // wave w stages input rows w, w + 4, ...: the row (and its pointer) is
    // uniform across the wave, eight loads in flight
    {
        const uint32_t w0 = wave;
        uint32_t k = w0;
        for (; k + 28 < K; k += 32) {
            uint64_t v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = ptrs.in[k + 4 * u][roff + lane];
#pragma unroll
            for (int u = 0; u < 8; u++) xd[(k + 4 * u) * kTile + lane] = fp_from(v[u]);
        }
        for (; k < K; k += 4) xd[k * kTile + lane] = fp_from(ptrs.in[k][roff + lane]);
    }
    for (uint32_t e = threadIdx.x; e < count * bpt; e += kBlock) {
        const uint32_t p = e / bpt, b = e - p * bpt;
        wd[e] = __longlong_as_double((long long)table[((uint64_t)limb * blocks + b0 + b) * count + p]);
    }
    __syncthreads();
    const double q = (double)m.q, qinv = 1.0 / q;
    for (uint32_t o = wave; o < M; o += kBlock / kTile) {
        // two independent sums (each reduced after every second term of its
        // own) so consecutive products do not wait on one another
        double a0 = 0.0, a1 = 0.0;
        for (uint32_t ri = first[o]; ri < first[o + 1]; ri++) {
            // a run: k = k0 + j, entry = p0 + j dp for j < len (indices computed, not loaded)
            const int4 rn = runs[ri];
            const double *xp = xd + rn.x * kTile + lane;
            const int xstep = kTile, wstep = rn.w * (int)bpt;
            const double *wp = wd + rn.y * (int)bpt + lb;
            int j = 0;
            for (; j + 4 <= rn.z; j += 4) {
                a0 += fp_mulmod(xp[0], wp[0], q, qinv);
                a1 += fp_mulmod(xp[xstep], wp[wstep], q, qinv);
                a0 += fp_mulmod(xp[2 * xstep], wp[2 * wstep], q, qinv);
                a1 += fp_mulmod(xp[3 * xstep], wp[3 * wstep], q, qinv);
                a0 = fp_reduce(a0, q, qinv);
                a1 = fp_reduce(a1, q, qinv);
                xp += 4 * xstep;
                wp += 4 * wstep;
            }
            for (; j < rn.z; j++) {
                a0 = fp_reduce(a0 + fp_mulmod(xp[0], wp[0], q, qinv), q, qinv);
                xp += xstep;
                wp += wstep;
            }
        }
        double acc = fp_reduce(a0 + a1, q, qinv);
        acc = acc < 0 ? acc + q : acc;
        ptrs.out[o][roff + lane] = fp_to(acc);
    }
}

// ---- four outputs at a time (primes below 2^51, blocks of at least 64 positions)
//
// The kernel above reads an input word from LDS and a weight per product and
// is bound by those reads and by a reduced product's eight and a half
// instructions: 4.41 ms for 127 inputs and 64 outputs of 64 terms at 20 limbs,
// N = 2^16, where moving the words takes 0.9; this one takes 2.62, bound by the
// products (1.2 ms of issue) and the ragged ends of the rows.  Here a wave sums four outputs of
// one 64-position tile at a time, so that an input word read from LDS serves
// four products; the weights are the same for the whole tile and come by scalar
// loads, four consecutive entries at once; and a product is four instructions
// (FpSum, one division per sum).
//
// plan: per group of four outputs, its quad segments (kQuadWords words: k0,
// len, entries e0..e3, their common step: terms (k0 + j, e_i + j step) of all
// four outputs, len a multiple of 4) and then single segments (kSingleWords:
// k0, len, e, step, output in the group).
constexpr int kMixThreads = 512;

template <int STEP>
__device__ __forceinline__ void quad_mac(FpSum *s, const double *x, const double *w, const int *e)
{
    double wv[4][4];
#pragma unroll
    for (int o = 0; o < 4; o++)
#pragma unroll
        for (int j = 0; j < 4; j++) wv[o][j] = table_at(w, e[o] + STEP * j);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const double xv = x[j * kTile];
#pragma unroll
        for (int o = 0; o < 4; o++) s[o].mac(wv[o][j], xv);
    }
}

__global__ __launch_bounds__(kMixThreads) void k_block_mix_quads(MixPtrs ptrs, const double *__restrict__ table,
                                                                 const int32_t *__restrict__ plan,
                                                                 const ModConst *__restrict__ mod, uint32_t K,
                                                                 uint32_t M, uint32_t limbs, uint32_t count,
                                                                 uint32_t blocks, uint32_t log_stride, uint32_t n)
{
    extern __shared__ uint64_t lds[];
    const uint32_t row = blockIdx.y;  // poly * limbs + limb
    const uint32_t limb = row % limbs;
    const uint64_t qi = mod[limb].q;
    if (qi >= kFpPrime) return;  // k_block_mix
    const uint32_t pos0 = blockIdx.x * kTile;
    double *xd = reinterpret_cast<double *>(lds);  // [K][64]
    const uint64_t roff = (uint64_t)row * n + pos0;
    const uint32_t lane = threadIdx.x % kTile;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kTile);
    constexpr uint32_t kWaves = kMixThreads / kTile;
    {
        uint32_t k = wave;
        for (; k + 7 * kWaves < K; k += 8 * kWaves) {
            uint64_t v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) v[u] = ptrs.in[k + kWaves * u][roff + lane];
#pragma unroll
            for (int u = 0; u < 8; u++) xd[(k + kWaves * u) * kTile + lane] = fp_from(v[u]);
        }
        for (; k < K; k += kWaves) xd[k * kTile + lane] = fp_from(ptrs.in[k][roff + lane]);
    }
    __syncthreads();
    const double q = (double)qi, qinv = 1.0 / q;
    const double M0 = fp_inner_magic(qi);
    const uint32_t terms = fp_inner_terms(qi);  // between two folds
    const double *w = table + ((uint64_t)limb * blocks + (pos0 >> log_stride)) * count;
    const uint32_t groups = (M + 3) / 4;
    for (uint32_t g = wave; g < groups; g += kWaves) {
        FpSum s[4];
#pragma unroll
        for (int o = 0; o < 4; o++) s[o].start(M0);
        uint32_t left = terms;
        auto fold = [&] {
#pragma unroll
            for (int o = 0; o < 4; o++) {
                s[o].l = s[o].value(M0, q, qinv);
                s[o].h = M0;
            }
            left = terms;
        };
        const int32_t *d = plan + table_at(plan, 2 * g), *end = plan + table_at(plan, 2 * g + 2);
        const int32_t *singles = plan + table_at(plan, 2 * g + 1);
        for (; d < singles; d += kQuadWords) {
            const int step = table_at(d, 6);
            int e[4];
#pragma unroll
            for (int o = 0; o < 4; o++) e[o] = table_at(d, 2 + o);
            const double *x = xd + table_at(d, 0) * kTile + lane;
            for (int len = table_at(d, 1); len > 0; len -= 4) {
                if (terms >= 4) {  // uniform
                    if (left < 4) fold();
                    left -= 4;
                    if (step == 1) {
                        quad_mac<1>(s, x, w, e);
                    } else if (step == -1) {
                        quad_mac<-1>(s, x, w, e);
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; j++)
#pragma unroll
                            for (int o = 0; o < 4; o++) s[o].mac(table_at(w, e[o] + step * j), x[j * kTile]);
                    }
                } else {
#pragma unroll 1
                    for (int j = 0; j < 4; j++) {
                        if (left == 0) fold();
                        left--;
#pragma unroll
                        for (int o = 0; o < 4; o++) s[o].mac(table_at(w, e[o] + step * j), x[j * kTile]);
                    }
                }
#pragma unroll
                for (int o = 0; o < 4; o++) e[o] += 4 * step;
                x += 4 * kTile;
            }
        }
        for (; d < end; d += kSingleWords) {
            const int step = table_at(d, 3), out = table_at(d, 4);
            // a loop per output, its sum known at compile time
            auto run = [&](FpSum &sum) {
                int e = table_at(d, 2);
                const double *x = xd + table_at(d, 0) * kTile + lane;
                for (int len = table_at(d, 1); len > 0; len--) {
                    if (left == 0) fold();
                    left--;
                    sum.mac(table_at(w, e), x[0]);
                    e += step;
                    x += kTile;
                }
            };
            if (out == 0)
                run(s[0]);
            else if (out == 1)
                run(s[1]);
            else if (out == 2)
                run(s[2]);
            else
                run(s[3]);
        }
#pragma unroll
        for (int o = 0; o < 4; o++) {
            if (4 * g + o >= M) break;  // uniform
            const double v = s[o].value(M0, q, qinv);
            ptrs.out[4 * g + o][roff + lane] = fp_to(v < 0 ? v + q : v);
        }
    }
}

}  // namespace

void periodic_scatter(const DeviceTables &t, uint64_t *work, uint8_t *flags, const uint64_t *coef, uint32_t rows,
                      uint32_t blocks, hipStream_t s)
{
    const uint32_t n = 1u << t.logn;
    const uint32_t log_stride = (uint32_t)t.logn - (uint32_t)__builtin_ctz(blocks);
    hipLaunchKernelGGL(k_periodic_scatter, dim3((n + kBlock - 1) / kBlock, rows), dim3(kBlock), 0, s, work, flags,
                       coef, blocks, log_stride, n);
}

void periodic_gather(const DeviceTables &t, uint64_t *table, uint8_t *flags, const uint64_t *work, uint32_t count,
                     uint32_t limbs, uint32_t blocks, hipStream_t s)
{
    const uint32_t n = 1u << t.logn;
    const uint32_t log_stride = (uint32_t)t.logn - (uint32_t)__builtin_ctz(blocks);
    hipLaunchKernelGGL(k_periodic_gather, dim3((n + kBlock - 1) / kBlock, count * limbs), dim3(kBlock), 0, s, table,
                       flags, work, t.mod, limbs, count, blocks, log_stride, n);
}

void periodic_expand(const DeviceTables &t, uint64_t *out, const uint64_t *table, uint32_t index, uint32_t count,
                     uint32_t limbs, uint32_t blocks, hipStream_t s)
{
    const uint32_t n = 1u << t.logn;
    const uint32_t log_stride = (uint32_t)t.logn - (uint32_t)__builtin_ctz(blocks);
    hipLaunchKernelGGL(k_periodic_expand, dim3((n + kBlock - 1) / kBlock, limbs), dim3(kBlock), 0, s, out, table, t.mod,
                       index, count, blocks, log_stride, n);
}

// One list of segments per group of four outputs: where all four have a term at
// consecutive inputs with one common entry step, a quad segment (cut to a
// multiple of four terms); everything else in runs of single outputs.
//
// Empty where k_block_mix is the faster one: a wave takes four outputs here, so
// fewer than sixteen leave most of the eight waves idle, few inputs do not pay
// for the segment lists, and a single term waits for its weight.  Microseconds,
// k_block_mix / quads, ten limbs at N = 2^16 (inputs x outputs):
//   banded rows: 127x4 252 / 497, 127x12 477 / 520, 16x16 124 / 121, 127x16 604 / 556, 8x24 114 / 124
//   a quarter of the terms single: 16x24 200 / 223, 127x16 1325 / 1696, 64x32 941 / 823
//   half of them: 64x64 1989 / 2372, 127x96 8977 / 9379
//   runs of four inputs: 127x19 (three outputs without a fourth) 1768 / 2112, 127x33 3093 / 1439
std::vector<int32_t> block_mix_plan(const int32_t *index, uint32_t K, uint32_t M)
{
    const uint32_t groups = (M + 3) / 4;
    std::vector<int32_t> plan((size_t)2 * groups + 1);
    size_t quads = 0, singles = 0;  // terms that four outputs take together, terms of one
    for (uint32_t g = 0; g < groups; g++) {
        const uint32_t rows = M - 4 * g < 4 ? M - 4 * g : 4;
        auto at = [&](uint32_t o, uint32_t k) { return index[(size_t)(4 * g + o) * K + k]; };
        std::vector<char> taken((size_t)rows * K, 0);
        plan[2 * g] = (int32_t)plan.size();
        for (uint32_t k = 0; rows == 4 && k + 4 <= K;) {
            bool all = true;
            for (uint32_t o = 0; o < 4; o++) all = all && at(o, k) >= 0 && at(o, k + 1) >= 0;
            const int32_t step = at(0, k + 1) - at(0, k);
            uint32_t len = 1;
            while (all && k + len < K) {
                for (uint32_t o = 0; o < 4; o++)
                    all = all && at(o, k + len) >= 0 && at(o, k + len) == at(o, k) + (int32_t)len * step;
                len += all ? 1 : 0;
            }
            len &= ~3u;
            if (!len) {
                k++;
                continue;
            }
            const int32_t quad[kQuadWords] = {(int32_t)k, (int32_t)len, at(0, k), at(1, k), at(2, k), at(3, k), step, 0};
            plan.insert(plan.end(), quad, quad + kQuadWords);
            quads += len;
            for (uint32_t o = 0; o < 4; o++)
                for (uint32_t j = 0; j < len; j++) taken[(size_t)o * K + k + j] = 1;
            k += len;
        }
        plan[2 * g + 1] = (int32_t)plan.size();
        for (uint32_t o = 0; o < rows; o++)
            for (uint32_t k = 0; k < K;) {
                auto open = [&](uint32_t x) { return x < K && !taken[(size_t)o * K + x] && at(o, x) >= 0; };
                if (!open(k)) {
                    k++;
                    continue;
                }
                uint32_t len = 1;
                const int32_t step = open(k + 1) ? at(o, k + 1) - at(o, k) : 0;
                while (open(k + len) && at(o, k + len) == at(o, k) + (int32_t)len * step) len++;
                const int32_t single[kSingleWords] = {(int32_t)k, (int32_t)len, at(o, k), step, (int32_t)o, 0, 0, 0};
                plan.insert(plan.end(), single, single + kSingleWords);
                singles += len;
                k += len;
            }
    }
    plan[2 * groups] = (int32_t)plan.size();
    if (K < 16 || M < 16 || 8 * singles > singles + 4 * quads) plan.clear();
    return plan;
}

size_t block_mix_lds_bytes(uint32_t K, uint32_t count, uint32_t blocks, int logn)
{
    const uint32_t log_stride = (uint32_t)logn - (uint32_t)__builtin_ctz(blocks);
    const uint32_t bpt = log_stride >= 6 ? 1u : (uint32_t)kTile >> log_stride;
    return 8 * ((size_t)K * kTile + (size_t)count * bpt);
}

void block_mix(const DeviceTables &t, const MixPtrs &p, const uint64_t *table, const int32_t *terms,
               const uint32_t *first, const int32_t *plan, uint32_t K, uint32_t M, uint32_t limbs, uint32_t count,
               uint32_t blocks, hipStream_t s)
{
    const uint32_t n = 1u << t.logn;
    const uint32_t log_stride = (uint32_t)t.logn - (uint32_t)__builtin_ctz(blocks);
    const size_t lds = block_mix_lds_bytes(K, count, blocks, t.logn);
    const dim3 grid(n / kTile, 2 * limbs);
    // a tile inside one block has uniform weights: the quad kernel (where there is
    // a plan) for the limbs below 2^51, the general one for what is left
    const bool quads = plan && log_stride >= 6;
    uint32_t fp = 0;
    for (uint32_t i = 0; i < limbs; i++) fp += t.mod_host[i] < kFpPrime ? 1 : 0;
    // inputs read once, outputs written once (both polynomials of every limb)
    const double limb_bytes = 16.0 * n * ((double)K + (double)M);
    if (quads && fp) {
        ProfScope prof("block_mix_quads", s, limb_bytes * fp);
        hipLaunchKernelGGL(k_block_mix_quads, grid, dim3(kMixThreads), (size_t)K * kTile * 8, s, p,
                           reinterpret_cast<const double *>(table), plan, t.mod, K, M, limbs, count, blocks, log_stride,
                           n);
    }
    if (quads && fp == limbs) return;
    ProfScope prof("block_mix", s, limb_bytes * (quads ? limbs - fp : limbs));
    const bool fast = t.max_bits <= 58, skip = quads || !fp;
    auto *kernel = fp == limbs ? k_block_mix<true, kSmall>
                   : fast      ? (skip ? k_block_mix<true, kWide> : k_block_mix<true, kEvery>)
                               : (skip ? k_block_mix<false, kWide> : k_block_mix<false, kEvery>);
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), lds, s, p, table, reinterpret_cast<const int4 *>(terms), first,
                       t.mod, K, M, limbs, count, blocks, log_stride, n);
}

}  // namespace nx
