// Order bases of matrix power series on the device.
//
//  * lbx_order_basis_m_u32 follows OrderBasis::M_Basis (order-basis.h:346-600):
//    one workgroup runs all `order` steps.  Each step sorts the shift with the
//    reference's selection-sort swaps (:388-399), forms the discrepancy
//    (coefficient k of sigma.serie, :416-444), splits its rows into the row
//    rank profile and the rest (the rank-profile PLUQ of :470-473), subtracts
//    from every other row its combination of the pivot rows (:509-517),
//    updates degrees and shifts (:546-566) and multiplies the pivot rows by x
//    (:573-580).  Rows of sigma never move in memory: a row map carries the
//    permutations, so a swap costs one word instead of a row of every
//    coefficient.
//  * lbx_order_basis_pm_u32 follows OrderBasis::PM_Basis (order-basis.h:219-326):
//    the host recursion over device buffers, M_Basis below order 32 (:47-48,232),
//    the serie update with the library's middle product (:274) and
//    sigma = sigma2.sigma1 with its polynomial-matrix product (:297).
//
// The discrepancy's rows are eliminated in increasing row order without
// divisions: a row r' below pivot row r becomes a.r' - b.r (a the pivot entry,
// b the entry of r' in the pivot column), and each row keeps its scale and its
// coefficients over the original pivot rows, so that a row that ends at zero
// gives its combination of pivot rows after one inverse of its scale.
#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <vector>

#include "lbx_ctx.h"

// wave-wide 64-bit minimum and maximum of the device library (DPP reductions)
extern "C" __device__ __attribute__((const)) unsigned long long __ockl_wfred_min_u64(unsigned long long);
extern "C" __device__ __attribute__((const)) unsigned long long __ockl_wfred_max_u64(unsigned long long);

namespace lbx {
namespace {

constexpr int kMbThreads = 1024;
constexpr int kMbWaves = kMbThreads / 64;
constexpr int kMbMaxM = 128;  // rows of the serie (= dimension of sigma)
constexpr int kMbMaxN = 64;   // columns of the serie
constexpr size_t kMbThreshold = 32;  // MBASIS_THRESHOLD (order-basis.h:47-48)
constexpr uint64_t kShiftLimit = (uint64_t)1 << 48;  // shift packed with a 7-bit row index

// x mod p for any 64-bit x and 2 <= p < 2^32, mu = floor((2^64-1)/p):
// q = hi64(x mu) undercounts x/p by less than 3, so r < 3p.
__device__ __forceinline__ uint32_t red64(uint64_t x, uint32_t p, uint64_t mu)
{
    const uint64_t q = __umul64hi(x, mu);
    uint64_t r = x - q * p;
    if (r >= p) r -= p;
    if (r >= p) r -= p;
    return (uint32_t)r;
}

__device__ __forceinline__ uint32_t mulm(uint32_t a, uint32_t b, uint32_t p, uint64_t mu)
{
    return red64((uint64_t)a * b, p, mu);
}

__device__ uint32_t invm(uint32_t a, uint32_t p, uint64_t mu)  // a^(p-2), a != 0
{
    uint32_t r = 1, b = a;
    for (uint32_t e = p - 2; e; e >>= 1) {
        if (e & 1) r = mulm(r, b, p, mu);
        b = mulm(b, b, p, mu);
    }
    return r;
}

// Montgomery product x y 2^-32 mod p for odd p < 2^31 (pinv = -p^-1 mod 2^32):
// x y + q p < 2^63, so the quotient by 2^32 is below 2p.
__device__ __forceinline__ uint32_t mont(uint32_t x, uint32_t y, uint32_t p, uint32_t pinv)
{
    const uint64_t t = (uint64_t)x * y;
    const uint32_t q = (uint32_t)t * pinv;
    return csub((uint32_t)((t + (uint64_t)q * p) >> 32), p);
}

// Sum of products kept as a 64-bit word plus a count of wraps of 2^64.
struct Acc {
    uint64_t lo = 0;
    uint32_t wraps = 0;
    __device__ __forceinline__ void add(uint32_t a, uint32_t b)
    {
        const uint64_t t = (uint64_t)a * b, s = lo + t;
        wraps += s < t ? 1u : 0u;
        lo = s;
    }
    // r64 = 2^64 mod p
    __device__ __forceinline__ uint32_t get(uint32_t p, uint64_t mu, uint32_t r64) const
    {
        return red64((uint64_t)red64(lo, p, mu) + (uint64_t)wraps * r64, p, mu);
    }
};

__global__ void __launch_bounds__(256) gather_coeff_major(DevView v, size_t count, uint32_t *out)
{
    const size_t entries = v.rows * v.cols, total = entries * count;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (size_t)gridDim.x * 256) {
        const size_t t = i / entries, e = i - t * entries;
        out[i] = v.base[view_index(v, e, t)];
    }
}

// Sum of products for p < 2^31: products are below 2^62, and the word is
// folded at 2^62 (2^62 = f62 mod p) after every second product, so it stays
// below 2^62 + 2^33 + 2^63.
struct AccSmall {
    uint64_t v = 0;
    __device__ __forceinline__ void add2(uint32_t a0, uint32_t b0, uint32_t a1, uint32_t b1, uint32_t f62)
    {
        v += (uint64_t)a0 * b0;
        v += (uint64_t)a1 * b1;
        v = (v & (((uint64_t)1 << 62) - 1)) + (uint64_t)(uint32_t)(v >> 62) * f62;
    }
    __device__ __forceinline__ void add1(uint32_t a, uint32_t b, uint32_t f62)
    {
        v += (uint64_t)a * b;
        v = (v & (((uint64_t)1 << 62) - 1)) + (uint64_t)(uint32_t)(v >> 62) * f62;
    }
    __device__ __forceinline__ uint32_t get(uint32_t p, uint64_t mu, uint32_t) const { return red64(v, p, mu); }
};

// Any p < 2^32: a 64-bit word and a count of its wraps.
struct AccWide {
    Acc a;
    __device__ __forceinline__ void add2(uint32_t a0, uint32_t b0, uint32_t a1, uint32_t b1, uint32_t)
    {
        a.add(a0, b0);
        a.add(a1, b1);
    }
    __device__ __forceinline__ void add1(uint32_t x, uint32_t y, uint32_t) { a.add(x, y); }
    __device__ __forceinline__ uint32_t get(uint32_t p, uint64_t mu, uint32_t r64) const { return a.get(p, mu, r64); }
};

// sum_j x[j] y[j*ystride], len terms
template <typename A>
__device__ __forceinline__ void dot(A &acc, const uint32_t *x, const uint32_t *y, int ystride, int len, uint32_t f62)
{
    int j = 0;
    for (; j + 7 < len; j += 8) {  // eight terms' loads issued together
        uint32_t xv[8], yv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            xv[u] = x[j + u];
            yv[u] = y[(j + u) * ystride];
        }
#pragma unroll
        for (int u = 0; u < 8; u += 2) acc.add2(xv[u], yv[u], xv[u + 1], yv[u + 1], f62);
    }
    for (; j + 1 < len; j += 2) acc.add2(x[j], y[j * ystride], x[j + 1], y[(j + 1) * ystride], f62);
    if (j < len) acc.add1(x[j], y[j * ystride], f62);
}

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void global_cvoid;

// Copies rows of `len` words from global memory into LDS with
// global_load_lds_dword (lane i of an instruction fills LDS word base + i):
// one instruction per 64 words of a row, one row per wave in turn, and no
// register staging, so every load of the copy can be in flight at once.  The
// caller waits (s_waitcnt 0) and synchronises before reading the copy.
template <typename Src, typename Dst>
__device__ __forceinline__ void stage_rows(int nrows, int len, Src src, Dst dst, int wave, int lane)
{
    for (int r = wave; r < nrows; r += kMbWaves)
        for (int j0 = 0; j0 < len; j0 += 64)
            if (j0 + lane < len)
                __builtin_amdgcn_global_load_lds((global_cvoid *)(src(r) + j0 + lane), (lds_void *)(dst(r) + j0), 4,
                                                 0, 0);
}

constexpr int kMbStageWords = 24576;  // LDS words for staged coefficient matrices
constexpr int kMbMaxOut = 4;          // m*n <= kMbMaxOut*kMbThreads
constexpr unsigned kNone = 0xffffffffu;

// One workgroup, kMbThreads threads.  S: serie, coefficient-major
// S[(t*m + j)*n + c]; W: order+1 coefficient matrices of m x m words,
// W[(l*m + phys)*m + j], phys a physical row.  Dynamic LDS: R, Z and D
// (m x n words each) and `stage` words for staged coefficient matrices.
//
// Per step k:
//  1. the shift sort (wave 0, keys in registers, one wave-wide minimum per position);
//  2. the discrepancy: rows that were pivots at step k-1 reuse that step's
//     discrepancy row (x.sigma_t has coefficient k+1 equal to coefficient k of
//     sigma_t, order-basis.h:446-456), the others are summed over staged blocks
//     of W[l] rows and S[k-l];
//  3. elimination, one barrier per pivot: the pivot column is never written, so
//     every thread reads its row's multiplier from it, and the next pivot is
//     searched for in the same pass;
//  4. non-pivot rows -= combination . pivot rows and pivot rows times x, on
//     staged blocks of W taken from the highest coefficient down, so the
//     shifted pivot rows never overwrite a coefficient still to be read.
// MONT (odd p < 2^31): the elimination runs on Montgomery forms x 2^32 mod p,
// whose zero pattern is the same and whose ratios Z/scale are the same.
template <typename A, bool MONT>
__global__ void __launch_bounds__(kMbThreads) m_basis_kernel(const uint32_t *__restrict__ S, uint32_t *__restrict__ W,
                                                             DevView out, uint64_t *__restrict__ shift_io,
                                                             uint64_t *__restrict__ deg_out, int order, int m, int n,
                                                             int stage, int out_count, uint32_t p, uint64_t mu,
                                                             uint32_t r64, uint32_t f62, uint32_t pinv, uint32_t r2m,
                                                             uint32_t one)
{
    // one = 1 in the elimination's representation (2^32 mod p with MONT)
    auto mul = [&](uint32_t x, uint32_t y) -> uint32_t {
        if constexpr (MONT) return mont(x, y, p, pinv);
        else return mulm(x, y, p, mu);
    };
    auto amb = [&](uint32_t a, uint32_t x, uint32_t b, uint32_t y) -> uint32_t {
        const uint32_t u = mul(a, x), v = mul(b, y);
        return u >= v ? u - v : u + (p - v);
    };
    extern __shared__ uint32_t dyn[];
    uint32_t *R = dyn;              // discrepancy rows under elimination, logical order
    uint32_t *Z = dyn + m * n;      // coefficients over the pivot rows, then the combination
    uint32_t *D = dyn + 2 * m * n;  // discrepancy before elimination, by physical row
    uint32_t *ST = dyn + 3 * m * n; // staged coefficient matrices
    __shared__ uint64_t shift[kMbMaxM], degree[kMbMaxM], tmp64[kMbMaxM], tmp64b[kMbMaxM];
    __shared__ int rowmap[kMbMaxM], tmpmap[kMbMaxM], pivot_of[kMbMaxM], oldrow[kMbMaxM], comp[kMbMaxM];
    __shared__ int was_piv[kMbMaxM];  // by physical row: pivot at the previous step
    __shared__ uint32_t scale[kMbMaxM];
    __shared__ unsigned smin[3];
    __shared__ int s_maxdeg, s_nc;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t mm = (size_t)m * m, nw = (size_t)(order + 1) * mm;
    const int mn = m * n;
    for (size_t i = tid; i < nw; i += kMbThreads) W[i] = 0;
    __syncthreads();
    for (int i = tid; i < m; i += kMbThreads) {
        W[(size_t)i * m + i] = 1;
        rowmap[i] = i;
        shift[i] = shift_io[i];
        degree[i] = 0;
        was_piv[i] = 0;
    }
    if (tid == 0) s_maxdeg = 0;
    __syncthreads();

    for (int k = 0; k < order; ++k) {
        const int maxdeg = s_maxdeg, lim = k < maxdeg ? k : maxdeg;
        // ---- 1. selection sort of the shift (order-basis.h:388-399) ----
        if (wave == 0) {
            uint64_t sh0 = lane < m ? shift[lane] : 0, sh1 = lane + 64 < m ? shift[lane + 64] : 0;
            uint64_t dg0 = lane < m ? degree[lane] : 0, dg1 = lane + 64 < m ? degree[lane + 64] : 0;
            int rm0 = lane < m ? rowmap[lane] : 0, rm1 = lane + 64 < m ? rowmap[lane + 64] : 0;
            // shifts spread over less than 2^24: 32-bit keys (shift - min) << 7 | position,
            // and only the positions' origins move; the arrays are gathered once at the end
            uint64_t lo = ~(uint64_t)0, hi = 0;
            if (lane < m) { lo = sh0; hi = sh0; }
            if (lane + 64 < m) { lo = sh1 < lo ? sh1 : lo; hi = sh1 > hi ? sh1 : hi; }
            for (int off = 32; off; off >>= 1) {
                const uint64_t a = __shfl_xor(lo, off), b = __shfl_xor(hi, off);
                lo = a < lo ? a : lo;
                hi = b > hi ? b : hi;
            }
            const bool narrow = hi - lo < ((uint64_t)1 << 24);
            if (narrow) {
                uint32_t v0 = (uint32_t)(sh0 - lo), v1 = (uint32_t)(sh1 - lo);
                int o0 = lane, o1 = lane + 64;
                for (int i = 0; i < m - 1; ++i) {
                    uint32_t best = 0xffffffffu;
                    if (lane < m && lane >= i) best = v0 << 7 | (uint32_t)lane;
                    if (lane + 64 < m && lane + 64 >= i) {
                        const uint32_t c1 = v1 << 7 | (uint32_t)(lane + 64);
                        best = c1 < best ? c1 : best;
                    }
                    best = __ockl_wfred_min_u32(best);  // wave-wide minimum (DPP), uniform
                    // every remaining key holds the largest shift: each later step would
                    // pick the element already in place, so the order is final
                    if ((best >> 7) == (uint32_t)(hi - lo)) break;
                    const int im = (int)(best & 127);
                    if (im != i) {
                        const int li = i & 63, lm = im & 63;
                        const bool hi_i = i >= 64, hi_m = im >= 64;
                        // uniform lanes: read them with v_readlane
                        const uint32_t vi = (uint32_t)__builtin_amdgcn_readlane((int)(hi_i ? v1 : v0), li);
                        const uint32_t vm = best >> 7;
                        const int oi = __builtin_amdgcn_readlane(hi_i ? o1 : o0, li);
                        const int om = __builtin_amdgcn_readlane(hi_m ? o1 : o0, lm);
                        if (lane == li) {
                            if (hi_i) { v1 = vm; o1 = om; } else { v0 = vm; o0 = om; }
                        }
                        if (lane == lm) {
                            if (hi_m) { v1 = vi; o1 = oi; } else { v0 = vi; o0 = oi; }
                        }
                    }
                }
                // gather by origin (all lanes read before any lane writes)
                if (lane < m) { sh0 = shift[o0]; dg0 = degree[o0]; rm0 = rowmap[o0]; }
                if (lane + 64 < m) { sh1 = shift[o1]; dg1 = degree[o1]; rm1 = rowmap[o1]; }
            }
            for (int i = 0; !narrow && i < m - 1; ++i) {
                uint64_t best = ~(uint64_t)0;  // key = shift << 7 | position: first minimum
                if (lane < m && lane >= i) best = sh0 << 7 | (uint64_t)lane;
                if (lane + 64 < m && lane + 64 >= i) {
                    const uint64_t c1 = sh1 << 7 | (uint64_t)(lane + 64);
                    best = c1 < best ? c1 : best;
                }
                for (int off = 32; off; off >>= 1) {
                    const uint64_t o = __shfl_xor(best, off);
                    best = o < best ? o : best;
                }
                if ((best >> 7) == hi) break;  // as above: the rest is in place
                const int im = (int)(best & 127);
                if (im != i) {
                    const int li = i & 63, lm = im & 63;
                    const bool hi_i = i >= 64, hi_m = im >= 64;
                    const uint64_t si = __shfl(hi_i ? sh1 : sh0, li), sm = __shfl(hi_m ? sh1 : sh0, lm);
                    const uint64_t di = __shfl(hi_i ? dg1 : dg0, li), dm = __shfl(hi_m ? dg1 : dg0, lm);
                    const int ri = __shfl(hi_i ? rm1 : rm0, li), rmm = __shfl(hi_m ? rm1 : rm0, lm);
                    if (lane == li) {
                        if (hi_i) { sh1 = sm; dg1 = dm; rm1 = rmm; } else { sh0 = sm; dg0 = dm; rm0 = rmm; }
                    }
                    if (lane == lm) {
                        if (hi_m) { sh1 = si; dg1 = di; rm1 = ri; } else { sh0 = si; dg0 = di; rm0 = ri; }
                    }
                }
            }
            if (lane < m) { shift[lane] = sh0; degree[lane] = dg0; rowmap[lane] = rm0; }
            if (lane + 64 < m) { shift[lane + 64] = sh1; degree[lane + 64] = dg1; rowmap[lane + 64] = rm1; }
            // rows to sum: those that were not pivots at the previous step
            int base = 0;
            for (int h = 0; h < m; h += 64) {
                const int r = h + lane;
                const bool need = r < m && !was_piv[h == 0 ? rm0 : rm1];
                const uint64_t bal = __ballot(need);
                if (need) comp[base + __popcll(bal & ((1ull << lane) - 1))] = r;
                base += __popcll(bal);
            }
            if (lane == 0) s_nc = base;
        }
        __syncthreads();
        // ---- 2. discrepancy: coefficient k of sigma.serie (order-basis.h:416-456) ----
        const int nc = s_nc;
        {
            A acc[kMbMaxOut];
            const int blk = nc * m + mn;  // staged words per coefficient
            const int lb = stage / blk > 0 ? stage / blk : 1;
            for (int l0 = 0; nc && l0 <= lim; l0 += lb) {
                const int l1 = l0 + lb < lim + 1 ? l0 + lb : lim + 1;
                stage_rows(
                    (l1 - l0) * nc, m,
                    [&](int pr) {
                        const int lq = pr / nc, i = pr - lq * nc;
                        return W + ((size_t)(l0 + lq) * m + rowmap[comp[i]]) * m;
                    },
                    [&](int pr) {
                        const int lq = pr / nc, i = pr - lq * nc;
                        return ST + lq * blk + i * m;
                    },
                    wave, lane);
                // serie blocks S[k-l], rows of n words
                stage_rows(
                    (l1 - l0) * m, n,
                    [&](int pr) {
                        const int lq = pr / m, j = pr - lq * m;
                        return S + (size_t)(k - l0 - lq) * mn + j * n;
                    },
                    [&](int pr) {
                        const int lq = pr / m, j = pr - lq * m;
                        return ST + lq * blk + nc * m + j * n;
                    },
                    wave, lane);
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
#pragma unroll
                for (int t = 0; t < kMbMaxOut; ++t) {
                    const int o = tid + t * kMbThreads;
                    if (o < nc * n) {
                        const int i = o / n, c = o - i * n;
                        for (int lq = 0; lq < l1 - l0; ++lq)
                            dot(acc[t], ST + lq * blk + i * m, ST + lq * blk + nc * m + c, n, m, f62);
                    }
                }
                __syncthreads();
            }
#pragma unroll
            for (int t = 0; t < kMbMaxOut; ++t) {
                const int o = tid + t * kMbThreads;
                if (o < nc * n) {
                    const int i = o / n, c = o - i * n;
                    R[comp[i] * n + c] = acc[t].get(p, mu, r64);
                }
            }
        }
        for (int o = tid; o < mn; o += kMbThreads) {
            const int r = o / n, c = o - r * n, ph = rowmap[r];
            if (was_piv[ph]) R[o] = D[ph * n + c];
            Z[o] = 0;
        }
        for (int i = tid; i < m; i += kMbThreads) {
            scale[i] = one;
            pivot_of[i] = -1;
        }
        if (tid == 0) {
            smin[0] = kNone;
            smin[1] = kNone;
            smin[2] = kNone;
        }
        __syncthreads();
        {
            bool found = false;
            for (int r = wave; r < m; r += kMbWaves) {  // one row per wave, one lane per column
                const uint32_t v = lane < n ? R[r * n + lane] : 0u;
                if (lane < n) {
                    D[rowmap[r] * n + lane] = v;
                    if constexpr (MONT) R[r * n + lane] = mont(v, r2m, p, pinv);
                }
                const uint64_t bal = __ballot(v != 0);
                if (bal && !found) {
                    found = true;
                    if (lane == 0) atomicMin(&smin[0], (unsigned)(r << 8 | __builtin_ctzll(bal)));
                }
            }
        }
        __syncthreads();
        // ---- 3. row rank profile and combinations (the PLUQ of :470-488) ----
        int rank = 0;
        for (;;) {
            // a pivot position is encoded row << 8 | column (n <= 64): the same row-major
            // order as row * n + column, decoded without a division on the pivot's path
            const unsigned hit = smin[rank % 3];
            if (hit == kNone) break;
            const int s = (int)(hit >> 8), c0 = (int)(hit & 255u);
            const uint32_t a = R[s * n + c0], sc_s = scale[s];
            // Each row below s is the word vector [R_r | Z_r], updated as a.x - b.y
            // against [R_s | Z_s] with Z_s[rank] read as -scale_s (so that
            // Z_r[rank] = b scale_s).  Columns of earlier pivots are zero in both
            // rows and column c0 becomes a b - b a = 0; b is read by the whole wave
            // before its lanes store, and no other wave touches row r.
            const uint32_t neg_sc = p - sc_s;
            const int wdt = n + rank + 1;
            unsigned *nxt = &smin[(rank + 1) % 3];
            // Every row is updated, b = 0 included (the row and its scale are then both
            // multiplied by a, which keeps Z/scale and the zero pattern): no branch per
            // row, and two rows per pass for independent chains.  Lane j holds word j
            // and word j+64 of the pivot vector (n <= 64, so word j+64 is a combination word).
            const int j1 = lane + 64;
            const bool has0 = lane < wdt, has1 = j1 < wdt, isr0 = lane < n;
            const int zo0 = lane - n, zo1 = j1 - n;
            const uint32_t y0 = !has0 ? 0u : (isr0 ? R[s * n + lane] : (zo0 == rank ? neg_sc : Z[s * n + zo0]));
            const uint32_t y1 = !has1 ? 0u : (zo1 == rank ? neg_sc : Z[s * n + zo1]);
            auto update = [&](int r, uint32_t b) -> bool {  // returns: lane's column nonzero
                bool nz = false;
                if (has0) {
                    uint32_t *xp = isr0 ? R + r * n + lane : Z + r * n + zo0;
                    const uint32_t v = amb(a, *xp, b, y0);
                    *xp = v;
                    nz = isr0 && v != 0;
                }
                if (has1) {
                    uint32_t *xp = Z + r * n + zo1;
                    *xp = amb(a, *xp, b, y1);
                }
                return nz;
            };
            bool found = false;  // this wave's rows come in increasing order: only its first hit counts
            for (int r = s + 1 + wave; r < m; r += 2 * kMbWaves) {
                const int r2 = r + kMbWaves;
                const bool two = r2 < m;
                const uint32_t b = R[r * n + c0], b2 = two ? R[r2 * n + c0] : 0u;
                const bool nz = update(r, b);
                const bool nz2 = two && update(r2, b2);
                if (lane == 0) {
                    scale[r] = mul(a, scale[r]);
                    if (two) scale[r2] = mul(a, scale[r2]);
                }
                const uint64_t bal = __ballot(nz), bal2 = __ballot(nz2);
                if (!found && (bal || bal2)) {
                    found = true;
                    const unsigned hit = bal ? (unsigned)(r << 8 | __builtin_ctzll(bal))
                                             : (unsigned)(r2 << 8 | __builtin_ctzll(bal2));
                    if (lane == 0) atomicMin(nxt, hit);
                }
            }
            if (tid == 0) {
                pivot_of[s] = rank;
                smin[(rank + 2) % 3] = kNone;
            }
            ++rank;
            __syncthreads();
        }
        // non-pivot rows: combination = Z / scale (one inverse per row, one lane each)
        for (int r = tid; r < m; r += kMbThreads)
            if (pivot_of[r] < 0 && scale[r] != 1) scale[r] = invm(scale[r], p, mu);
        __syncthreads();
        for (int r = wave; r < m; r += kMbWaves) {
            if (pivot_of[r] >= 0 || scale[r] == 1) continue;
            const uint32_t inv = scale[r];
            if (lane < rank) Z[r * n + lane] = mulm(Z[r * n + lane], inv, p, mu);  // plain product: Z~/scale~ = Z/scale
        }
        // Qt: pivot rows first, then the others, each in increasing order; a
        // non-pivot row's place counts the non-pivot rows above it (m <= 128:
        // two waves, one ballot per 64 rows)
        static_assert(kMbMaxM <= 2 * 64 && kMbThreads >= 2 * 64, "two ballots cover every row");
        if (tid < 2 * 64) {
            const uint64_t b0 = __ballot(lane < m && pivot_of[lane] < 0);
            const uint64_t b1 = __ballot(lane + 64 < m && pivot_of[lane + 64] < 0);
            const int r = tid;
            if (r < m) {
                int pos = pivot_of[r];
                if (pos < 0) {
                    const uint64_t below = (1ull << lane) - 1;
                    pos = rank + (wave == 0 ? __popcll(b0 & below) : __popcll(b0) + __popcll(b1 & below));
                }
                oldrow[pos] = r;
                tmpmap[pos] = rowmap[r];
                tmp64[pos] = shift[r];
                tmp64b[pos] = degree[r];
                was_piv[rowmap[r]] = pivot_of[r] >= 0;
            }
        }
        __syncthreads();
        for (int i = tid; i < m; i += kMbThreads) {
            rowmap[i] = tmpmap[i];
            shift[i] = tmp64[i];
            degree[i] = tmp64b[i];
        }
        __syncthreads();
        // ---- 4. non-pivot rows -= combination . pivot rows (:509-517), pivot rows times x (:573-580) ----
        {
            const int lb = stage / (int)mm > 0 ? stage / (int)mm : 1;
            for (int l1 = lim + 1; l1 > 0;) {
                const int l0 = l1 - lb > 0 ? l1 - lb : 0;
                stage_rows(
                    (l1 - l0) * m, m,
                    [&](int pr) {
                        const int lq = pr / m, i = pr - lq * m;
                        return W + ((size_t)(l0 + lq) * m + rowmap[i]) * m;
                    },
                    [&](int pr) { return ST + pr * m; }, wave, lane);
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
                const int nrows = m - rank;
                for (int pr = wave; pr < (l1 - l0) * nrows; pr += kMbWaves) {
                    const int lq = pr / nrows, si = rank + pr - lq * nrows;
                    const uint32_t *st = ST + lq * (int)mm, *y = Z + oldrow[si] * n;
                    uint32_t *dst = W + ((size_t)(l0 + lq) * m + rowmap[si]) * m;
                    for (int j = lane; j < m; j += 64) {
                        A acc;
                        dot(acc, y, st + j, m, rank, f62);
                        const uint32_t sub = acc.get(p, mu, r64), v = st[si * m + j];
                        dst[j] = v >= sub ? v - sub : v + (p - sub);
                    }
                }
                for (int pr = wave; pr < (l1 - l0) * rank; pr += kMbWaves) {
                    const int lq = pr / rank, t = pr - lq * rank;
                    const uint32_t *src = ST + lq * (int)mm + t * m;
                    uint32_t *dst = W + ((size_t)(l0 + lq + 1) * m + rowmap[t]) * m;
                    for (int j = lane; j < m; j += 64) dst[j] = src[j];
                }
                __syncthreads();
                l1 = l0;
            }
            for (int o = tid; o < rank * m; o += kMbThreads) W[(size_t)rowmap[o / m] * m + o % m] = 0;
        }
        // ---- degrees and shifts (:546-566) ----
        if (tid == 0) {
            uint64_t dmax = 0;
            for (int i = 0; i < rank; ++i) dmax = degree[i] > dmax ? degree[i] : dmax;
            for (int i = 0; i < rank; ++i) {
                degree[i]++;
                shift[i]++;
            }
            for (int i = rank; i < m; ++i) degree[i] = degree[i] < dmax ? dmax : degree[i];
            const uint64_t md = (uint64_t)maxdeg > dmax + 1 ? (uint64_t)maxdeg : dmax + 1;
            s_maxdeg = (int)(md < (uint64_t)order ? md : (uint64_t)order);
        }
        __syncthreads();
    }
    // sigma.resize(max_degree+1), shift2 = shift (:592-597); out_count coefficients
    // written when nonzero, zero above the degree
    const int md = s_maxdeg;
    const size_t cnt = out_count ? (size_t)out_count : (size_t)md + 1;
    for (size_t o = tid; o < cnt * mm; o += kMbThreads) {
        const size_t l = o / mm, e = o - l * mm, i = e / m, j = e - i * m;
        out.base[view_index(out, e, l)] = l <= (size_t)md ? W[(l * m + rowmap[i]) * m + j] : 0u;
    }
    for (int i = tid; i < m; i += kMbThreads) shift_io[i] = shift[i];
    if (tid == 0) *deg_out = (uint64_t)md;
}

// ---------------------------------------------------------------------------
// M_Basis over several workgroups (orders up to kMcMaxOrder: the PM_Basis
// base case).  The steps follow m_basis_kernel and order-basis.h:346-600, but
// instead of summing the discrepancy from sigma and the serie at each step, the
// row operations are applied to the serie itself (the residual
// x^-k sigma.serie, whose lowest coefficient is the discrepancy) and to sigma.
// Row operations act on every column alike, so the columns are split over G
// workgroups: group g keeps cs columns of the residual serie (all
// coefficients) and cj columns of sigma in LDS, and no group needs another's
// columns except to see the discrepancies.  Those come in blocks of B steps:
// every group also holds the next B coefficients of the residual in full
// (the window), runs the B eliminations on it redundantly (so all groups take
// the same decisions), and the groups exchange the following B coefficients
// through global memory at one grid barrier per block.
//
// What bounds a step is the serial chain of pivots, so the elimination goes in
// panels of four rows:
//  * rows are held in registers, kMbPanel rows (one panel) or two panels per
//    wave, NC lanes to a row, values centred in [-h, h], h = (p-1)/2;
//  * on its turn a wave runs an in-place, division-free Gauss-Jordan
//    elimination of its panel (row operations inside the panel), which gives
//    D and H = D P_C^-1 P for the panel's pivot columns C, and publishes them;
//  * every other row takes the whole panel in one update with a single
//    reduction: x <- D x - (x_C) H off C and x_C <- (x_C) H on C.
// These are column operations on the discrepancy: they leave pivot rows with
// one nonzero entry and turn a non-pivot row into its combination of the pivot
// rows times the product of the D's, so no separate combination is carried.
// The row rank profile and the combinations do not depend on which columns
// are chosen, so the result is that of a pivot-by-pivot elimination.
//
// Per step: the elimination; then, between two barriers, one wave inverts the
// product of the D's, one sorts the shifts for the next step, and the others
// form sums over the pivot rows: for the window with the combinations still
// unscaled (one Montgomery product per entry scales the sum once the inverse
// is known), and for the group's own columns with the previous step's
// combinations, so that neither waits for the inverse; then the pivot rows
// are multiplied by x.
//
// Measured at 64 x 32, order 32, p = 998244353: 553 us per base case
// against 922 us for the form before it (discrepancies summed from sigma, a grid
// barrier per step, pivot-by-pivot elimination of [R | Z]), and PM_Basis at order
// 4096 84.6 ms against 132.4 ms (8 x 4 at order 512: 4.8 against 6.1 ms, 128 x 32
// at order 128: 3.3 against 6.7 ms).  A step takes about 39 k cycles: eight panels at
// 3.3 k each (a lone wave issues an instruction every five cycles at best, and a
// panel is some 400 of them with three LDS hand-offs), 5 k for the inverse and the
// sums, 5 k for scaling and shifting, and a quarter of the 12 k of an exchange.
constexpr int kMcMaxOrder = 32;
constexpr int kMcMaxGroups = 64;
constexpr int kMcLdsWords = 38400;  // dynamic LDS words (the static arrays take 9.3 of the other 10 KiB)
constexpr unsigned kMcSpinLimit = 1u << 24;  // polls of a wait before it reports a failure
constexpr int kMbPanel = 4;          // rows per panel
constexpr int kMcMaxBlock = 4;       // steps per exchange
constexpr int kMcSumWaves = kMbWaves - 2;  // waves 0 and 1 invert and sort meanwhile
constexpr int kMcMaxTasks = 4;       // window tiles per wave (cols_split sees to it)

// Constants of one odd prime below 2^31 for arithmetic on centred values.
struct Centred {
    uint32_t p, pinv, h, one;  // p^-1 mod 2^32, (p-1)/2, 2^32 mod p
    int32_t c8[7];             // 2^(8d) mod p, centred

    __device__ __forceinline__ int32_t from(uint32_t x) const { return (int32_t)(x > h ? x - p : x); }
    __device__ __forceinline__ uint32_t canonical(int32_t x) const
    {
        return (uint32_t)x + ((uint32_t)(x >> 31) & p);
    }
    // t 2^-32 mod p, centred, for -p <= t >> 32 < p: with m = t p^-1 mod 2^32 the low
    // words of t and m p agree, so the high words' difference is exact; h + it lies in [0, 2p)
    __device__ __forceinline__ int32_t redc(int64_t t) const
    {
        const int32_t hi = (int32_t)(t >> 32), m = (int32_t)((uint32_t)t * pinv);
        uint32_t u = (uint32_t)hi + ((uint32_t)(hi >> 31) & p) + h;
        u -= (uint32_t)mulhi_s32(m, (int32_t)p);
        return (int32_t)(csub(u, p) - h);
    }
    __device__ __forceinline__ int32_t mul(int32_t x, int32_t y) const { return redc((int64_t)x * y); }
    // x - y of centred values, centred
    __device__ __forceinline__ int32_t sub(int32_t x, int32_t y) const
    {
        const int32_t d = x - y;  // in [-(p-1), p-1]
        uint32_t u = (uint32_t)d + h;
        u += (uint32_t)((int32_t)u >> 31 & (int32_t)p) & (uint32_t)(d >> 31);
        return (int32_t)(csub(u, p) - h);
    }
};

// A wait polls kMcSpinLimit times at most, and one that gives up sets the failure
// flag: what follows works on unfinished data, and the flag alone keeps the host
// from taking its result for one.  The flag only matters once a limit ran out, so
// a wait reads it now and then.
__device__ __forceinline__ bool wait_failed(unsigned *bar)
{
    return __hip_atomic_load(bar + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}
__device__ __forceinline__ void report_wait(unsigned *bar)
{
    __hip_atomic_store(bar + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// All groups of the grid meet here: bar[0] counts arrivals and is awaited to
// reach `target`; bar[1] is set when a poll limit runs out (the host reports the
// call as failed, and later barriers no longer wait).  What the groups exchange is
// written and read with agent-scope atomics, which go past the caches, so the
// barrier only waits for the stores (no write-back or invalidation of an L2).
__device__ __forceinline__ void grid_barrier(unsigned *bar, unsigned target)
{
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_add(bar, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned polls = 0;
        while ((int)(__hip_atomic_load(bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - target) < 0) {
            if ((polls & 255) == 255 && wait_failed(bar)) break;
            if (++polls == kMcSpinLimit) {
                report_wait(bar);
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
    }
    __syncthreads();
}

// Makes a count known to the group's other waves, behind the LDS words it covers: the
// fence keeps the compiler from moving their stores past it (they are other arrays,
// which it knows), and LDS does one wave's accesses in order.
template <class T>
__device__ __forceinline__ void publish(T *count, T value)
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __hip_atomic_store(count, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// i / d for 0 <= i < 2^20, d > 0, given r = 1 / (float)d: (i + 1/2) r is at least
// 1/(2d) away from an integer, more than the products' rounding
__device__ __forceinline__ int quot(int i, float r) { return (int)(((float)i + 0.5f) * r); }

// Montgomery product of canonical words by 32-bit multiplications, whose latency is
// half that of a 64-bit multiply-add: x y - m p with m = x y p^-1 mod 2^32
__device__ __forceinline__ uint32_t mont_pos(uint32_t x, uint32_t y, const Centred &K)
{
    const uint32_t m = x * y * K.pinv, r = __umulhi(x, y) - __umulhi(m, K.p), s = r + K.p;
    return s < r ? s : r;
}

// Sums over an operation's pivot rows for a tile of 16 of its non-pivot rows and
// 16 columns, on INT8 matrix instructions: out[r] is the sum for row
// 4 (lane >> 4) + r and this lane's column, as redc returns it.  A word's four
// balanced digits are four neighbouring bytes of the inner dimension, so the words
// themselves are the A operand, and with the other word's digits in reverse,
// shifted by e bytes, one 64-deep product gives the digit products of one
// anti-diagonal for 16 pivots: seven products per 16 pivots, of which 16/28 is
// needed, against no repacking into digit planes.  The sums stay below
// 64 * 4 * 2^14, so the diagonals recombine in 64 bits without a reduction.
// x: combinations, xs words per non-pivot row (up to the next multiple of 32 pivots
// other words of the LDS may be read, and count for nothing); col: this lane's
// column of M; poff: the pivot rows' offsets (any up to that multiple).
// On 64-bit multiply-adds with four rows per thread these sums were bound by LDS
// reads (each word read once per lane that needed it).
typedef int i32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void tile_sums(int32_t (&out)[4], const int32_t *x, int xs, const int32_t *col,
                                          const int *poff, int rank, int lane, const Centred &K)
{
    i32x4 acc[7];
#pragma unroll
    for (int d = 0; d < 7; ++d) acc[d] = i32x4{0, 0, 0, 0};
    const int kg = (lane >> 4) * 4;
    const int32_t *xr = x + (lane & 15) * xs + kg;
    for (int b0 = 0; b0 < rank; b0 += 32) {
        // 32 pivots' words at a time, all loads first
        int4 po[2];
        i32x4 a[2];
        int32_t w[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) po[h] = *reinterpret_cast<const int4 *>(poff + b0 + 16 * h + kg);
#pragma unroll
        for (int h = 0; h < 2; ++h) a[h] = *reinterpret_cast<const i32x4 *>(xr + b0 + 16 * h);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            w[h][0] = col[po[h].x];
            w[h][1] = col[po[h].y];
            w[h][2] = col[po[h].z];
            w[h][3] = col[po[h].w];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            uint32_t rev[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (b0 + 16 * h + kg + j >= rank) w[h][j] = 0;  // a's words there are arbitrary
                rev[j] = __builtin_bswap32((uint32_t)w[h][j] + 0x80808080u) ^ 0x80808080u;
                a[h][j] = (int)(((uint32_t)a[h][j] + 0x80808080u) ^ 0x80808080u);
            }
#pragma unroll
            for (int d = 0; d < 7; ++d) {
                i32x4 bv;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    bv[j] = (int)(d <= 3 ? rev[j] >> (8 * (3 - d)) : rev[j] << (8 * (d - 3)));
                acc[d] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[h], bv, acc[d], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        int64_t t = 0;
#pragma unroll
        for (int d = 0; d < 7; ++d) t += (int64_t)acc[d][r] * K.c8[d];
        out[r] = K.redc(t);
    }
}

// Geometry of one launch, the same in every group.
struct ColsShape {
    int order, m, n;
    int cs, cj;  // residual serie and sigma columns per group
    int B;       // steps per block
    int rs;      // words per row of M
    int xs;      // words per row of the combinations: min(m, n) rounded up to 16, and four more
    int xm;      // their rows: m rounded up to a multiple of 16
    int xb;      // 1: combinations of two steps are kept (B > 1), 0: of one
};

// G = gridDim.x groups of kMbThreads threads.  NC lanes hold a row of the
// discrepancy (n <= NC), PPW panels per wave (m <= 64 PPW).  part: 2 x m x (B n)
// words of exchanged coefficients; bar: the grid barrier's two words, bar[0]
// at bar_base when the launch begins.  Dynamic LDS: H (a vector of four words
// per panel and lane), the combinations X of one or two steps (per non-pivot row, one word
// per pivot), the panels' diagonals, and M: per physical row the
// window (coefficient t of the block at t*n + column), the group's residual
// columns and its sigma columns.  out_count: coefficients of sigma written
// (zero above the degree); 0 writes degree+1 of them.
template <int NC, int PPW>
__global__ void __launch_bounds__(kMbThreads) m_basis_cols_kernel(DevView serie, DevView out,
                                                                  uint64_t *__restrict__ shift_io,
                                                                  uint64_t *__restrict__ deg_out, int32_t *part,
                                                                  unsigned *__restrict__ bar, unsigned bar_base,
                                                                  ColsShape C, int out_count, Centred K)
{
    constexpr int RPR = 64 / NC;             // rows per register
    constexpr int PR = kMbPanel / RPR;       // registers per panel
    constexpr int NREG = PPW * PR;
    const int order = C.order, m = C.m, n = C.n, rs = C.rs, xs = C.xs;
    const int G = gridDim.x, c0 = blockIdx.x * C.cs, j0 = blockIdx.x * C.cj;
    const int ncs = c0 < n ? (n - c0 < C.cs ? n - c0 : C.cs) : 0;  // this group's serie columns
    const int ncj = j0 < m ? (m - j0 < C.cj ? m - j0 : C.cj) : 0;  // and sigma columns
    const int tid0 = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid0 >> 6);
    const int npan = (m + kMbPanel - 1) / kMbPanel;
    const int os = C.B * n, oj = os + C.cs * order;  // columns of M: window, residual, sigma
    const uint32_t p = K.p, npinv = 0u - K.pinv;
    // The thread's index as a value the compiler cannot look through: used in each
    // phase, it keeps lane conditions from being hoisted out of the step loop,
    // where they would fill the scalar registers and spill.
    auto fresh_tid = [&]() -> int {
        int t = tid0;
        asm volatile("" : "+v"(t));
        return t;
    };

    extern __shared__ int4 dyn4[];
    int4 *H = dyn4;                              // [panel][NC]
    int32_t *X = (int32_t *)(H + npan * NC);     // [step & xb][non-pivot row][xs], a word per pivot
    int32_t *Dz = X + (1 + C.xb) * C.xm * xs;    // [panel][NC]
    int32_t *M = Dz + npan * NC;                 // [physical row][rs]
    __shared__ int4 pcol[kMbMaxM / kMbPanel];    // 4 x pivot columns of a panel, in H's slot order
    __shared__ int pbits[kMbMaxM / kMbPanel];     // its pivot rows, one bit each
    __shared__ uint32_t pdet[kMbMaxM / kMbPanel]; // its D
    __shared__ uint64_t shift[kMbMaxM], degree[kMbMaxM], tmp64[kMbMaxM], tmp64b[kMbMaxM];
    __shared__ int rowmap[2][kMbMaxM], tmpmap[kMbMaxM], qtab[kMbMaxM];
    __shared__ __align__(16) int poff[2][kMbMaxN];  // M offsets of pivot rows,
    __shared__ __align__(16) int noff[2][kMbMaxM + 16];  // and of the other rows
    __shared__ int op_rank[2], op_lim[2];
    __shared__ int bidx[kMbMaxN];      // pivot index of a column, -1 without one
    __shared__ int32_t col_e[kMbMaxN];  // product of the D's of the panels before the column's
    __shared__ uint32_t s_e;   // product of the D's of the panels booked
    __shared__ int32_t s_inv[2];
    __shared__ int s_book;     // panels booked
    __shared__ int s_maxdeg;
    __shared__ unsigned s_pub;  // panels published | rank << 8 | (rank == n) << 16

    // ---- initial state ----
    {
        const int tid = tid0;
        for (int i = tid; i < m * ncj * (order + 1); i += kMbThreads) {
            const int q = i / (order + 1), l = i - q * (order + 1), ph = q / ncj, jj = q - ph * ncj;
            M[ph * rs + oj + jj * (order + 1) + l] = (l == 0 && ph == j0 + jj) ? 1 : 0;
        }
        for (int i = tid; i < m * ncs * order; i += kMbThreads) {
            const int q = i / order, t = i - q * order, ph = q / ncs, cc = q - ph * ncs;
            M[ph * rs + os + cc * order + t] = K.from(serie.base[view_index(serie, (size_t)ph * n + c0 + cc, t)]);
        }
        const int b0 = C.B < order ? C.B : order;
        for (int i = tid; i < m * n; i += kMbThreads) {
            const int ph = i / n, c = i - ph * n;
            for (int t = 0; t < b0; ++t) M[ph * rs + t * n + c] = K.from(serie.base[view_index(serie, i, t)]);
        }
        for (int i = tid; i < m; i += kMbThreads) {
            rowmap[0][i] = i;
            shift[i] = shift_io[i];
            degree[i] = 0;
        }
        if (tid < 2 * (kMbMaxM + 16)) noff[0][tid] = 0;
        if (tid < 2 * kMbMaxN) poff[0][tid] = 0;
        if (tid < kMbMaxN) bidx[tid] = -1;
        if (tid < kMbMaxM / kMbPanel) pbits[tid] = 0;
        if (tid == 0) {
            s_maxdeg = 0;
            op_lim[0] = 0;
            s_pub = 0;
            s_book = 0;
        }
    }
    __syncthreads();

    // Selection sort of the shift (order-basis.h:388-399), one value at a time, by
    // one wave: the reference's sort places the elements of the smallest remaining
    // value in order of position, and each element it displaces follows a chain of
    // those positions, which one pass of the wave resolves.  shift, degree and
    // rmap are permuted alike.
    auto sort_rows = [&](int *rmap, int lane) {
        const uint64_t below = (1ull << lane) - 1;
        const bool v0 = lane < m, v1 = lane + 64 < m;
        uint64_t k0 = v0 ? shift[lane] : 0, k1 = v1 ? shift[lane + 64] : 0;
        int o0 = lane, o1 = lane + 64;
        for (int start = 0; start < m - 1;) {
            const bool a0 = v0 && lane >= start, a1 = v1 && lane + 64 >= start;
            uint64_t lo = ~(uint64_t)0, hi = 0;
            if (a0) { lo = k0; hi = k0; }
            if (a1) { lo = k1 < lo ? k1 : lo; hi = k1 > hi ? k1 : hi; }
            lo = __ockl_wfred_min_u64(lo);
            hi = __ockl_wfred_max_u64(hi);
            if (lo == hi) break;  // what remains holds one value: every later swap is the identity
            // the smallest value's positions q_0 < q_1 < ... (c of them): step start+j
            // swaps positions start+j and q_j, since the value's elements not yet placed
            // never move and q_j >= start+j
            const bool m0 = a0 && k0 == lo, m1 = a1 && k1 == lo;
            const uint64_t b0 = __ballot(m0), b1 = __ballot(m1);
            const int n0 = __popcll(b0), end = start + n0 + __popcll(b1);
            const int r0 = __popcll(b0 & below), r1 = n0 + __popcll(b1 & below);
            if (m0) qtab[r0] = lane;
            if (m1) qtab[r1] = lane + 64;
            __builtin_amdgcn_s_waitcnt(0);
            __builtin_amdgcn_wave_barrier();
            // destination: start+rank for the value's elements; an element displaced
            // from x in [start, end) goes to q_{x-start}, and on while that is below end
            auto dest = [&](int x, bool isv, int rk) -> int {
                if (isv) return start + rk;
                if (x < start || x >= end) return x;
                int y = qtab[x - start];
                while (y < end) y = qtab[y - start];
                return y;
            };
            const int d0 = v0 ? dest(lane, m0, r0) : lane;
            const int d1 = v1 ? dest(lane + 64, m1, r1) : lane + 64;
            __builtin_amdgcn_s_waitcnt(0);
            __builtin_amdgcn_wave_barrier();
            if (v0) { tmp64[d0] = k0; tmpmap[d0] = o0; }
            if (v1) { tmp64[d1] = k1; tmpmap[d1] = o1; }
            __builtin_amdgcn_s_waitcnt(0);
            __builtin_amdgcn_wave_barrier();
            if (v0) { k0 = tmp64[lane]; o0 = tmpmap[lane]; }
            if (v1) { k1 = tmp64[lane + 64]; o1 = tmpmap[lane + 64]; }
            __builtin_amdgcn_s_waitcnt(0);
            __builtin_amdgcn_wave_barrier();
            start = end;
        }
        // gather by origin (all lanes read before any lane writes)
        uint64_t dg0 = 0, dg1 = 0;
        int rm0 = 0, rm1 = 0;
        if (v0) { dg0 = degree[o0]; rm0 = rmap[o0]; }
        if (v1) { dg1 = degree[o1]; rm1 = rmap[o1]; }
        __builtin_amdgcn_s_waitcnt(0);
        __builtin_amdgcn_wave_barrier();
        if (v0) { shift[lane] = k0; degree[lane] = dg0; rmap[lane] = rm0; }
        if (v1) { shift[lane + 64] = k1; degree[lane + 64] = dg1; rmap[lane + 64] = rm1; }
    };
    if (wave == 1) sort_rows(rowmap[0], tid0 & 63);
    __syncthreads();
    unsigned nbar = 0;
    // without an exchange nothing else keeps group 0 from writing the shift before
    // another group has read it
    if (G > 1 && order <= C.B) grid_barrier(bar, bar_base + ++nbar * (unsigned)G);

    // Column u (-1: none) of the non-pivot rows of a tile minus the tile's sums, which
    // are of unscaled combinations: times the inverse of the D's.
    auto apply_tile = [&](const int32_t (&sum)[4], int ob, int i0, int nn, int u, int lane) {
        const int i = i0 + 4 * (lane >> 4);
        const int32_t inv = s_inv[ob];
        const int4 no = *reinterpret_cast<const int4 *>(&noff[ob][i]);
        const int off[4] = {no.x, no.y, no.z, no.w};
        int32_t old[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) old[r] = M[off[r] + (u < 0 ? 0 : u)];
#pragma unroll
        for (int r = 0; r < 4; ++r) old[r] = K.sub(old[r], K.mul(sum[r], inv));
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (u >= 0 && i + r < nn) M[off[r] + u] = old[r];
    };
    // The group's own columns under the operation of step kk: non-pivot rows -=
    // combination . pivot rows (:509-517), one tile per wave at a time, tiles
    // [t, count) by nt waves.  Residual coefficients up to kk are zero from here on;
    // sigma has op_lim+1 coefficients.
    auto own_update = [&](int kk, bool residual, int t, int nt, int lane) {
        const int ob = kk & 1, rank = __builtin_amdgcn_readfirstlane(op_rank[ob]),
                  lim = __builtin_amdgcn_readfirstlane(op_lim[ob]), nn = m - rank, len = order - kk - 1;
        const int vs = residual ? ncs * len : 0, vt = vs + ncj * (lim + 1);
        if (!rank || !nn || !vt) return;
        const int nct = (vt + 15) >> 4, ntile = nct * ((nn + 15) >> 4);
        for (int i = t, rq = 0, ct = t; i < ntile; i += nt, ct += nt) {
            while (ct >= nct) ct -= nct, ++rq;
            const int v = 16 * ct + (lane & 15), vc = v < vt ? v : 0;
            int u;
            if (vc < vs) {
                const int cc = ncs > 1 ? quot(vc, 1.0f / (float)len) : 0;
                u = os + cc * order + kk + 1 + (vc - cc * len);
            } else {
                const int jj = quot(vc - vs, 1.0f / (float)(lim + 1));
                u = oj + jj * (order + 1) + (vc - vs - jj * (lim + 1));
            }
            int32_t sum[4];
            tile_sums(sum, X + ((ob & C.xb) * C.xm + 16 * rq) * xs, xs, M + u, poff[ob], rank, lane, K);
            apply_tile(sum, ob, 16 * rq, nn, v < vt ? u : -1, lane);
        }
    };
    // Pivot rows of a step times x (:573-580): words [lo, hi) of their rows of M move up
    // by `step` words.  A wave takes rows b and b + kMbWaves and reads kShiftChunks x 64
    // words of each, from the top down, before it writes any of them, so its writes
    // reach only words already read.  What enters an own residual column is a dead
    // coefficient; sigma's columns get a zero at the bottom.
    constexpr int kShiftChunks = 2, kShiftWords = 64 * kShiftChunks;
    typedef int32_t ShiftWords[2][kShiftChunks];
    auto shift_read = [&](ShiftWords &v, const int *po, int rank, int b, int lo, int top, int step, int lane) {
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int c = 0; c < kShiftChunks; ++c) {
                const int w = top - 64 * (c + 1) + lane;
                v[r][c] = b + r * kMbWaves < rank && w >= lo ? M[po[b + r * kMbWaves] + w - step] : 0;
            }
    };
    auto shift_write = [&](const ShiftWords &v, const int *po, int rank, int b, int lo, int top, int lane) {
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int c = 0; c < kShiftChunks; ++c) {
                const int w = top - 64 * (c + 1) + lane;
                if (b + r * kMbWaves < rank && w >= lo) M[po[b + r * kMbWaves] + w] = v[r][c];
            }
    };
    auto shift_rows = [&](int kk, int lo, int hi, int step, int lane) {
        const int rank = __builtin_amdgcn_readfirstlane(op_rank[kk & 1]);
        for (int b = wave; b < rank; b += 2 * kMbWaves)
            for (int top = hi; top > lo; top -= kShiftWords) {
                ShiftWords v;
                shift_read(v, poff[kk & 1], rank, b, lo, top, step, lane);
                __builtin_amdgcn_wave_barrier();
                shift_write(v, poff[kk & 1], rank, b, lo, top, lane);
                __builtin_amdgcn_wave_barrier();
            }
    };
    const int own_lo = os + 1, own_hi = oj + ncj * (order + 1);
    auto own_zero = [&](int kk, int lane) {
        const int rank = __builtin_amdgcn_readfirstlane(op_rank[kk & 1]);
        for (int b = wave; b < rank; b += kMbWaves)
            for (int jj = lane; jj < ncj; jj += 64) M[poff[kk & 1][b] + oj + jj * (order + 1)] = 0;
    };
    auto own_shift = [&](int kk, int lane) {
        shift_rows(kk, own_lo, own_hi, 1, lane);
        own_zero(kk, lane);
    };

    for (int k0 = 0; k0 < order; k0 += C.B) {
        const int bk = order - k0 < C.B ? order - k0 : C.B;  // steps of this block
        for (int b = 0; b < bk; ++b) {
            const int k = k0 + b, kb = k & 1;
            const int *rmap = rowmap[kb];
            int32_t *Xk = X + (kb & C.xb) * C.xm * xs;
            {
                const int lane = fresh_tid() & 63, col = lane & (NC - 1), half = lane / NC;
                // ---- rows of the discrepancy in shift order ----
                int32_t x[NREG];
#pragma unroll
                for (int q = 0; q < PPW; ++q) {
                    const int r0 = (wave * PPW + q) * kMbPanel;
#pragma unroll
                    for (int g = 0; g < PR; ++g) {
                        const int r = r0 + g * RPR + half;
                        x[q * PR + g] = r < m && col < n ? M[rmap[r] * rs + b * n + col] : 0;
                    }
                }
                // ---- row rank profile and combinations (the PLUQ of :470-488) ----
                const int hb4 = (lane & ~(NC - 1)) << 2;
                int applied = 0;
                unsigned state = 0;
                uint64_t used = 0;  // columns of the panels applied
                // Wave 0, whose rows are the first to be finished, books the panels as it takes
                // them in: the places of their pivots, their columns' factors (the product of the
                // D's before them) and their rows.
                uint32_t e_run = K.one;
                int rk_run = 0;
                auto book = [&](int P, const int4 &cc, bool inc) {
                    const int bits = __builtin_amdgcn_readfirstlane(pbits[P]);
                    const uint32_t det = (uint32_t)__builtin_amdgcn_readfirstlane((int)pdet[P]);
                    if (inc && half == 0) {
                        // the row of this column's slot (slots: rows 0, 2, 1, 3 with two rows a register)
                        const int c4 = col << 2;
                        // an unused slot repeats a used one's column: its row has no bit
                        constexpr int s1 = RPR == 2 ? 2 : 1, s2 = RPR == 2 ? 1 : 2;
                        const int u = cc.x == c4 && (bits & 1)           ? 0
                                      : cc.y == c4 && (bits >> s1 & 1) ? s1
                                      : cc.z == c4 && (bits >> s2 & 1) ? s2
                                                                       : 3;
                        bidx[col] = rk_run + __popc(bits & ((1 << u) - 1));
                        col_e[col] = K.from(e_run);
                    }
                    if (lane < kMbPanel && bits >> lane & 1)
                        poff[kb][rk_run + __popc(bits & ((1 << lane) - 1))] = rmap[P * kMbPanel + lane] * rs;
                    rk_run += __popc(bits);
                    e_run = mont(e_run, det, p, npinv);
                };
                // takes every published panel in; returns whether the elimination is over
                // (no unused column left) once at least `want` panels are in.  A panel's
                // words are written before the count in s_pub and one wave's LDS accesses
                // are done in order, so words read after a count that covers them are theirs.
                auto advance = [&](int want) -> bool {
                    unsigned polls = 0;
                    for (;;) {
                        state = __hip_atomic_load(&s_pub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        __atomic_signal_fence(__ATOMIC_SEQ_CST);
                        // the next panel's words, read along with the count (by the wave whose
                        // turn is next: the others would only load the LDS)
                        int4 cc, hv;
                        int32_t dz;
                        auto fetch = [&]() {
                            cc = pcol[applied];
                            hv = H[applied * NC + col];
                            dz = Dz[applied * NC + col];
                        };
                        const bool early = applied + 1 == want && applied < npan;
                        if (early) fetch();
                        __atomic_signal_fence(__ATOMIC_SEQ_CST);
                        state = (unsigned)__builtin_amdgcn_readfirstlane((int)state);
                        const int pub = (int)(state & 255u);
                        if (!early && applied < pub) fetch();
                        while (applied < pub) {
                            // a panel without pivots has no column (-1)
                            if (__builtin_amdgcn_readfirstlane(cc.x) >= 0) {
                                const int a0 = hb4 + cc.x, a1 = hb4 + cc.y, a2 = hb4 + cc.z, a3 = hb4 + cc.w;
                                int32_t z[NREG][4];
#pragma unroll
                                for (int g = 0; g < NREG; ++g) {
                                    z[g][0] = __builtin_amdgcn_ds_bpermute(a0, x[g]);
                                    z[g][1] = __builtin_amdgcn_ds_bpermute(a1, x[g]);
                                    z[g][2] = __builtin_amdgcn_ds_bpermute(a2, x[g]);
                                    z[g][3] = __builtin_amdgcn_ds_bpermute(a3, x[g]);
                                }
                                used |= __ballot(dz == 0);
#pragma unroll
                                for (int g = 0; g < NREG; ++g) {
                                    // five products of centred values: the high word is below p in size
                                    int64_t t = (int64_t)dz * x[g], t1 = (int64_t)z[g][1] * hv.y;
                                    t += (int64_t)z[g][0] * hv.x;
                                    t1 += (int64_t)z[g][2] * hv.z;
                                    t += (int64_t)z[g][3] * hv.w;
                                    x[g] = K.redc(t + t1);
                                }
                                if (wave == 0) book(applied, cc, dz == 0);
                            }
                            if (wave == 0 && lane == 0) publish(&s_book, applied + 1);
                            if (++applied < pub) fetch();
                        }
                        if (state >> 16) return true;
                        if (pub >= want) return false;
                        if ((polls & 255) == 255 && wait_failed(bar)) return true;
                        if (++polls == kMcSpinLimit) {
                            report_wait(bar);
                            return true;
                        }
                        // the wave whose turn is next polls without a pause
                        if (pub + 1 < want) __builtin_amdgcn_s_sleep(1);
                    }
                };
                int mine = 0, found = 0;  // rows of this wave, pivots among them
                int prank[PPW], prow[PPW];  // pivots before the panel, its pivot rows
                bool over = false;
#pragma unroll
                for (int q = 0; q < PPW; ++q) {
                    const int P = wave * PPW + q, r0 = P * kMbPanel;
                    prank[q] = n;
                    prow[q] = 0;
                    if (r0 < m) mine += m - r0 < kMbPanel ? m - r0 : kMbPanel;
                    if (r0 >= m || over) continue;
                    over = advance(P);
                    if (over) continue;
                    __builtin_amdgcn_s_setprio(3);
                    // Gauss-Jordan on a canonical copy of the panel; at column c of the pivot in
                    // row u the pivot vector and row u read dcur, the other rows 0 (the panel's
                    // inverse takes the place of its pivot columns).  One wave's serial chain:
                    // what counts is the number of instructions.
                    const int rank0 = (int)(state >> 8 & 255u);
                    uint32_t y[PR];
#pragma unroll
                    for (int g = 0; g < PR; ++g) y[g] = K.canonical(x[q * PR + g]);
                    uint32_t dcur = K.one;
                    uint64_t freec = ~used;  // n <= NC, and words beyond column n are zero
                    int pc[kMbPanel] = {-1, -1, -1, -1}, c_any = -1;
                    bool inc = false;  // this lane's column is a pivot column of the panel
                    unsigned rowbits = 0;
#pragma unroll
                    for (int u = 0; u < kMbPanel; ++u) {
                        const int gu = u / RPR, hu = u % RPR;
                        uint64_t bal = __ballot(y[gu] != 0);
                        if constexpr (RPR == 2) bal = (hu ? bal >> 32 : bal & 0xffffffffu) & (uint32_t)freec;
                        else bal &= freec;
                        if (bal == 0) continue;
                        const int c = RPR == 2 ? __builtin_ctz((uint32_t)bal) : (int)__builtin_ctzll(bal);
                        uint32_t bl[PR], bh[PR];
#pragma unroll
                        for (int g = 0; g < PR; ++g) {
                            bl[g] = (uint32_t)__builtin_amdgcn_readlane((int)y[g], c);
                            bh[g] = RPR == 2 ? (uint32_t)__builtin_amdgcn_readlane((int)y[g], 32 + c) : bl[g];
                        }
                        const uint32_t a = hu ? bh[gu] : bl[gu];
                        const bool isc = col == c;
                        uint32_t yr = y[gu];
                        if constexpr (RPR == 2) {
                            // the row's half in both halves of the wave
                            const auto sw = __builtin_amdgcn_permlane32_swap(y[gu], y[gu], false, false);
                            yr = hu == 0 ? (uint32_t)sw[0] : (uint32_t)sw[1];
                        }
                        const uint32_t ny = p - (isc ? dcur : yr);
#pragma unroll
                        for (int g = 0; g < PR; ++g) {
                            uint32_t am = a, bv = bl[g], at = 0;
                            if constexpr (RPR == 2) bv = half ? bh[g] : bl[g];
                            if (g == gu) {  // the pivot row is scaled, not updated
                                const bool isp = half == hu;
                                am = isp ? dcur : a;
                                bv = isp ? 0u : bv;
                                at = isp ? dcur : 0u;
                            }
                            const uint32_t xin = isc ? at : y[g];
                            const uint64_t t = (uint64_t)am * xin + (uint64_t)bv * ny;
                            const uint32_t qq = (uint32_t)t * npinv;
                            y[g] = csub((uint32_t)((t + (uint64_t)qq * p) >> 32), p);
                        }
                        dcur = mont(dcur, a, p, npinv);
                        pc[u] = c_any = c << 2;
                        rowbits |= 1u << u;
                        inc = inc || isc;
                        freec &= ~(1ull << c);
                    }
                    const unsigned cnt = (unsigned)__popc(rowbits), rk = (unsigned)rank0 + cnt;
                    // slots of rows without a pivot: H zero, any column
#pragma unroll
                    for (int u = 0; u < kMbPanel; ++u) pc[u] = pc[u] < 0 ? c_any : pc[u];
                    int32_t hv[PR];
#pragma unroll
                    for (int g = 0; g < PR; ++g) {
                        const int32_t v = K.from(y[g]);
                        hv[g] = rowbits >> (g * RPR + half) & 1 ? (inc ? v : -v) : 0;
                    }
                    int32_t *hp = reinterpret_cast<int32_t *>(H + P * NC + col);
                    if constexpr (RPR == 2) {  // slots: rows 0, 2 of the lower half, 1, 3 of the upper
                        *reinterpret_cast<int2 *>(hp + 2 * half) = make_int2(hv[0], hv[1]);
                    } else {
                        *reinterpret_cast<int4 *>(hp) = make_int4(hv[0], hv[1], hv[2], hv[3]);
                    }
                    Dz[P * NC + col] = inc ? 0 : K.from(dcur);  // both halves write the same word
                    if (lane == 0) {
                        pcol[P] = RPR == 2 ? make_int4(pc[0], pc[2], pc[1], pc[3])
                                           : make_int4(pc[0], pc[1], pc[2], pc[3]);
                        pbits[P] = (int)rowbits;
                        pdet[P] = dcur;
                        publish(&s_pub, (unsigned)(P + 1) | rk << 8 | (rk == (unsigned)n ? 1u << 16 : 0u));
                    }
                    __atomic_signal_fence(__ATOMIC_SEQ_CST);
                    __builtin_amdgcn_s_setprio(0);
                    found += (int)cnt;
                    prank[q] = rank0;
                    prow[q] = (int)rowbits;
                }
                // the non-pivot rows take the remaining panels, and their combinations
                // (times the product of all D's) go to X
                if (wave == 0 || mine > found) advance(npan);
                if (wave == 0 && lane == 0) s_e = e_run;
                if (mine > found) {
                    // wait for the last panel's booking
                    for (unsigned polls = 0; wave != 0;) {
                        const int booked = __hip_atomic_load(&s_book, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        if (__builtin_amdgcn_readfirstlane(booked) >= applied) break;
                        if ((polls & 255) == 255 && wait_failed(bar)) break;
                        if (++polls == kMcSpinLimit) {
                            report_wait(bar);
                            break;
                        }
                    }
                    __atomic_signal_fence(__ATOMIC_SEQ_CST);
                    const int bc = col < n ? bidx[col] : -1;
                    const int32_t ce = col_e[col];
#pragma unroll
                    for (int q = 0; q < PPW; ++q)
#pragma unroll
                        for (int g = 0; g < PR; ++g) {
                            const int v = g * RPR + half, r = (wave * PPW + q) * kMbPanel + v;
                            if (r < m && !(prow[q] >> v & 1)) {
                                // its place: the rows above it less the pivots among them
                                const int i = r - prank[q] - __popc(prow[q] & ((1 << v) - 1));
                                const int32_t z = K.mul(x[q * PR + g], ce);
                                if (bc >= 0) Xk[i * xs + bc] = z;
                                if (col == 0) noff[kb][i] = rmap[r] * rs;
                            }
                        }
                }
            }
            __syncthreads();
            // ---- the inverse, the next order, and the sums over the pivot rows ----
            const int rank = __builtin_amdgcn_readfirstlane((int)(s_pub >> 8 & 255u));
            const int nn = m - rank;
            const int wc = rank && nn ? (bk - b - 1) * n : 0, w0 = (b + 1) * n;
            const int wct = (wc + 15) >> 4, wtile = wct * ((nn + 15) >> 4);
            const float rwct = 1.0f / (float)(wct ? wct : 1);
            int32_t sum[kMcMaxTasks][4];
            if (wave == 0) {
                // s^(p-2), s the product of the D's: both products of a bit in every step, so that
                // their chains overlap.  Only sums take it, and a step whose rows are all pivot
                // rows (every step of a square serie of full rank) has none.
                uint32_t v = K.one, sq = s_e;
                if (nn) {
                    for (uint32_t e = p - 2; e; e >>= 1) {
                        const uint32_t f = e & 1 ? sq : K.one;
                        v = mont_pos(v, f, K);
                        sq = mont_pos(sq, sq, K);
                    }
                }
                if (fresh_tid() == 0) {
                    s_inv[kb] = K.from(v);
                    op_rank[kb] = rank;
                }
            } else if (wave == 1) {
                // Qt: pivot rows first, then the others, each in increasing order; degrees
                // and shifts (:546-566); then the next step's order
                const int lane = fresh_tid() & 63;
                const uint64_t below = (1ull << lane) - 1;
                const uint64_t pm0 = __ballot(lane < m && pbits[lane >> 2] >> (lane & 3) & 1);
                const uint64_t pm1 = __ballot(lane + 64 < m && pbits[(lane >> 2) + 16] >> (lane & 3) & 1);
                const int maxdeg = s_maxdeg, np0 = __popcll(pm0);
                uint64_t dm = 0;
                for (int h = 0; h < m; h += 64) {
                    const int r = h + lane;
                    if (r < m && (h ? pm1 : pm0) >> lane & 1) dm = degree[r] > dm ? degree[r] : dm;
                }
                dm = __ockl_wfred_max_u64(dm);
                int *next = rowmap[kb ^ 1];
                for (int h = 0; h < m; h += 64) {
                    const int r = h + lane;
                    if (r < m) {
                        const uint64_t word = h ? pm1 : pm0;
                        const bool isp = word >> lane & 1;
                        const int bel = __popcll(word & below) + (h ? np0 : 0);
                        const int pos = isp ? bel : rank + r - bel;
                        const uint64_t d = degree[r];
                        tmp64[pos] = shift[r] + (isp ? 1 : 0);
                        tmp64b[pos] = isp ? d + 1 : (d < dm ? dm : d);
                        next[pos] = rmap[r];
                    }
                }
                __builtin_amdgcn_s_waitcnt(0);
                __builtin_amdgcn_wave_barrier();
                for (int r = lane; r < m; r += 64) {
                    shift[r] = tmp64[r];
                    degree[r] = tmp64b[r];
                }
                const uint64_t md64 = (uint64_t)maxdeg > dm + 1 ? (uint64_t)maxdeg : dm + 1;
                const int md = (int)(md64 < (uint64_t)order ? md64 : (uint64_t)order);
                if (lane == 0) s_maxdeg = md;
                __builtin_amdgcn_s_waitcnt(0);
                __builtin_amdgcn_wave_barrier();
                if (k + 1 < order) sort_rows(next, lane);
            } else {
                const int lane = fresh_tid() & 63;
#pragma unroll
                for (int q = 0; q < kMcMaxTasks; ++q) {
                    const int i = wave - 2 + q * kMcSumWaves;
                    if (i < wtile) {
                        const int rq = quot(i, rwct), w = 16 * (i - rq * wct) + (lane & 15);
                        tile_sums(sum[q], Xk + 16 * rq * xs, xs, M + w0 + (w < wc ? w : 0), poff[kb], rank, lane, K);
                    }
                }
                // the own columns' tiles begin at the waves the window leaves idle
                if (b > 0) own_update(k - 1, true, kMbWaves - 1 - wave, kMcSumWaves, lane);
            }
            __syncthreads();
            // ---- scaled sums from the window; pivot rows times x ----
            {
                const int tid = fresh_tid(), lane = tid & 63;
                const int whi = bk * n;
                if (b > 0 && rank <= 2 * kMbWaves && whi - w0 <= kShiftWords && own_hi - own_lo <= kShiftWords) {
                    // both shifts in one round of reads and one of writes
                    const int rank1 = __builtin_amdgcn_readfirstlane(op_rank[kb ^ 1]);
                    ShiftWords vw, vo;
                    if (rank1 <= 2 * kMbWaves) {
                        shift_read(vw, poff[kb], rank, wave, w0, whi, n, lane);
                        shift_read(vo, poff[kb ^ 1], rank1, wave, own_lo, own_hi, 1, lane);
                        __builtin_amdgcn_wave_barrier();
                        shift_write(vw, poff[kb], rank, wave, w0, whi, lane);
                        shift_write(vo, poff[kb ^ 1], rank1, wave, own_lo, own_hi, lane);
                        __builtin_amdgcn_wave_barrier();
                        own_zero(k - 1, lane);
                    } else {
                        shift_rows(k, w0, whi, n, lane);
                        own_shift(k - 1, lane);
                    }
                } else {
                    shift_rows(k, w0, whi, n, lane);
                    if (b > 0) own_shift(k - 1, lane);
                }
                if (wave >= 2) {
#pragma unroll
                    for (int q = 0; q < kMcMaxTasks; ++q) {
                        const int i = wave - 2 + q * kMcSumWaves;
                        if (i < wtile) {
                            const int rq = quot(i, rwct), w = 16 * (i - rq * wct) + (lane & 15);
                            apply_tile(sum[q], kb, 16 * rq, nn, w < wc ? w0 + w : -1, lane);
                        }
                    }
                }
                if (tid < kMbMaxN) bidx[tid] = -1;
                if (tid < kMbMaxM / kMbPanel) pbits[tid] = 0;
                if (tid == 0) {
                    s_pub = 0;
                    s_book = 0;
                    if (b + 1 < bk) op_lim[kb ^ 1] = k + 1 < s_maxdeg ? k + 1 : s_maxdeg;
                }
            }
            __syncthreads();
        }
        // ---- the block's last operation on the own columns ----
        const int kl = k0 + bk - 1;
        const bool more = kl + 1 < order;
        own_update(kl, more, wave, kMbWaves, fresh_tid() & 63);
        __syncthreads();
        own_shift(kl, fresh_tid() & 63);
        __syncthreads();
        if (!more) break;
        // ---- the next block's window ----
        const int tid = fresh_tid();
        const int nb = order - kl - 1 < C.B ? order - kl - 1 : C.B;  // its steps
        const int cn = ncs * nb;
        const float rcn = 1.0f / (float)(cn ? cn : 1), rcs = 1.0f / (float)(ncs ? ncs : 1);
        if (G > 1) {
            int32_t *px = part + (size_t)(nbar & 1) * m * os;
            for (int i = tid; i < m * cn; i += kMbThreads) {
                const int ph = quot(i, rcn), rem = i - ph * cn, t = quot(rem, rcs), cc = rem - t * ncs;
                __hip_atomic_store(px + ph * os + t * n + c0 + cc, M[ph * rs + os + cc * order + kl + 1 + t],
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            grid_barrier(bar, bar_base + ++nbar * (unsigned)G);
            const int wn = nb * n;
            const float rwn = 1.0f / (float)wn;
            for (int i0 = tid; i0 < m * wn; i0 += 8 * kMbThreads) {
                int32_t v[8];  // eight loads in flight
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int i = i0 + u * kMbThreads, ph = quot(i, rwn), w = i - ph * wn;
                    v[u] = i < m * wn ? __hip_atomic_load(px + ph * os + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                      : 0;
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int i = i0 + u * kMbThreads, ph = quot(i, rwn), w = i - ph * wn;
                    if (i < m * wn) M[ph * rs + w] = v[u];
                }
            }
        } else {
            for (int i = tid; i < m * cn; i += kMbThreads) {
                const int ph = quot(i, rcn), rem = i - ph * cn, t = quot(rem, rcs), cc = rem - t * ncs;
                M[ph * rs + t * n + cc] = M[ph * rs + os + cc * order + kl + 1 + t];
            }
        }
        if (tid == 0) op_lim[(kl + 1) & 1] = kl + 1 < s_maxdeg ? kl + 1 : s_maxdeg;
        __syncthreads();
    }
    // sigma.resize(max_degree+1), shift2 = shift (:592-597)
    const int md = s_maxdeg;
    const int cnt = out_count ? out_count : md + 1;
    const int *rmap = rowmap[order & 1];
    for (int o = tid0; o < m * ncj * cnt; o += kMbThreads) {
        const int q = o / cnt, l = o - q * cnt, i = q / ncj, jj = q - i * ncj;
        const uint32_t v = l <= md ? K.canonical(M[rmap[i] * rs + oj + jj * (order + 1) + l]) : 0u;
        out.base[view_index(out, (size_t)i * m + j0 + jj, l)] = v;
    }
    if (blockIdx.x == 0) {
        for (int i = tid0; i < m; i += kMbThreads) shift_io[i] = shift[i];
        if (tid0 == 0) *deg_out = (uint64_t)md;
    }
}

unsigned grid_for(size_t total)
{
    const size_t g = (total + 255) / 256;
    return (unsigned)(g < 4096 ? (g ? g : 1) : 4096);
}

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Device bytes of the buffers each recursion level keeps live (sigma1, serie2,
// sigma2 and the two degree words), summed down the deepest path.
size_t pm_level_bytes(size_t m, size_t n, size_t order)
{
    if (order <= kMbThreshold) return 0;
    const size_t o1 = order >> 1, o2 = order - o1;
    const size_t own =
        align256(m * m * (o1 + 1) * 4) + align256(m * n * o2 * 4) + align256(m * m * (o2 + 1) * 4) + align256(16);
    return own + std::max(pm_level_bytes(m, n, o1), pm_level_bytes(m, n, o2));
}

struct MbScratch {
    uint32_t *S, *W;
    int32_t *part;
    uint64_t *shift, *deg;
    unsigned *bar;  // grid barrier: arrivals, then the failure flag
    unsigned arrivals;  // of the launches queued so far
};

struct PmRun {
    lbx_ctx *ctx;
    uint32_t p;
    size_t m, n;
    int method;
    hipStream_t s;
    MbScratch mb;
    uint8_t *arena;
    size_t used, cap;

    uint32_t *take(size_t bytes)
    {
        uint32_t *q = (uint32_t *)(arena + used);
        used += align256(bytes);
        return q;
    }
};

DevView polfirst_view(uint32_t *base, size_t rows, size_t cols, size_t stor, size_t size)
{
    DevView v;
    v.base = base;
    v.layout = LBX_POLFIRST;
    v.rows = rows;
    v.cols = cols;
    v.stor = stor;
    v.shift = 0;
    v.size = size;
    return v;
}

size_t mc_lds_words(const ColsShape &C)
{
    const size_t nc = C.n <= 32 ? 32 : 64, npan = ((size_t)C.m + kMbPanel - 1) / kMbPanel;
    return npan * nc * 5 + (size_t)(1 + C.xb) * C.xm * C.xs + (size_t)C.m * C.rs;
}

// The grid of m_basis_cols_kernel must fit on the device at once: one group
// per CU (its LDS takes most of a CU's 160 KiB).
lbx_status mc_check_groups(int G)
{
    int dev = 0, cus = 0;
    LBX_TRY_HIP(hipGetDevice(&dev));
    LBX_TRY_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    return G <= cus ? LBX_OK : LBX_ERR_UNSUPPORTED;
}

// Column split of m_basis_cols_kernel over the returned number of groups, or 0
// for the one-workgroup kernel (orders above kMcMaxOrder, or no split fits).
// By default about m^2 n / 4096 groups (at most 32), so that a group's own
// columns cost no more per step than its window; more where the LDS of fewer
// groups would not hold their columns.  Blocks of kMcMaxBlock steps where they
// fit, shorter ones otherwise.  LBX_MBASIS_GROUPS=N asks for N groups, 0 for the
// one-workgroup kernel.
int cols_split(size_t m, size_t n, size_t order, ColsShape *C)
{
    if (order > (size_t)kMcMaxOrder) return 0;
    size_t target = std::min<size_t>(32, std::max<size_t>(1, m * m * n / 4096));
    if (const char *e = getenv("LBX_MBASIS_GROUPS")) {
        const long want = atol(e);
        if (want <= 0) return 0;
        target = std::min<size_t>((size_t)want, (size_t)kMcMaxGroups);
    }
    for (int B = std::min<int>(kMcMaxBlock, (int)order); B > 0; B >>= 1)
        for (size_t g = target; g <= (size_t)kMcMaxGroups; ++g) {
            C->order = (int)order;
            C->m = (int)m;
            C->n = (int)n;
            C->cs = (int)((n + g - 1) / g);
            C->cj = (int)((m + g - 1) / g);
            C->B = B;
            C->rs = (int)((size_t)B * n + C->cs * order + C->cj * (order + 1)) | 1;  // odd: rows start in distinct banks
            C->xs = (int)((std::min(m, n) + 15) & ~(size_t)15) + 4;
            C->xm = (int)((m + 15) & ~(size_t)15);
            C->xb = B > 1;
            const size_t tiles = ((size_t)(B - 1) * n + 15) / 16 * ((m + 15) / 16);
            if (mc_lds_words(*C) <= (size_t)kMcLdsWords && tiles <= (size_t)(kMcSumWaves * kMcMaxTasks))
                return (int)std::max((n + C->cs - 1) / C->cs, (m + C->cj - 1) / C->cj);
        }
    return 0;
}

// T = a_top . b_top (m x m coefficient matrices: coefficient ta of a, tb of b);
// c[.][0] -= T and c[.][P] = T.  A cyclic product mod x^P - 1 of two operands
// whose full product has P+1 coefficients holds coefficient P in coefficient
// 0; this puts it back.  With fix = false only the degree word is written.
// deg = d[0] + d[1] (the degrees of sigma2 and sigma1).
__global__ void __launch_bounds__(256) wrap_fix_kernel(DevView a, size_t ta, DevView b, size_t tb, DevView c,
                                                       size_t P, int m, uint32_t p, uint64_t mu, uint32_t r64,
                                                       bool fix, const uint64_t *d, uint64_t *deg)
{
    // one workgroup per row i of T, one thread per column j
    __shared__ uint32_t arow[kMbMaxM];
    const int i = blockIdx.x, j = threadIdx.x;
    if (i == 0 && j == 0) *deg = d[0] + d[1];
    if (!fix) return;
    if (j < m) arow[j] = a.base[view_index(a, (size_t)i * m + j, ta)];
    __syncthreads();
    if (j >= m) return;
    // the loads of column j are independent: eight in flight at a time
    Acc acc;
    int q = 0;
    for (; q + 8 <= m; q += 8) {
        uint32_t bv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) bv[u] = b.base[view_index(b, (size_t)(q + u) * m + j, tb)];
#pragma unroll
        for (int u = 0; u < 8; ++u) acc.add(arow[q + u], bv[u]);
    }
    for (; q < m; ++q) acc.add(arow[q], b.base[view_index(b, (size_t)q * m + j, tb)]);
    const uint32_t t = acc.get(p, mu, r64);
    const size_t e = (size_t)i * m + j;
    uint32_t *c0 = c.base + view_index(c, e, 0);
    const uint32_t v = *c0;
    *c0 = v >= t ? v - t : v + (p - t);
    c.base[view_index(c, e, P)] = t;
}

// M_Basis on a device view of the serie (coefficients 0..order-1) into sigma.
// The degree goes to *deg on the device; out_count coefficients of sigma are
// written (zero above the degree), or degree+1 when out_count is 0.
lbx_status run_m_basis(PmRun &R, const DevView &serie, const DevView &sigma, size_t order, uint64_t *deg,
                       size_t out_count)
{
    const size_t m = R.m, n = R.n;
    uint64_t mu = ~(uint64_t)0 / R.p;
    const uint32_t r32 = (uint32_t)(((uint64_t)1 << 32) % R.p), r64 = (uint32_t)((uint64_t)r32 * r32 % R.p);
    uint32_t f62 = (uint32_t)(((uint64_t)1 << 62) % R.p);
    const bool mont_ok = R.p < (1u << 31) && (R.p & 1);
    uint32_t pinv = 0, r2m = 0, one = 1;
    if (mont_ok) {
        pinv = 0u - inv_mod32(R.p);
        one = r32;
        r2m = r64;
    }
    ColsShape C;
    const int G = mont_ok ? cols_split(m, n, order, &C) : 0;
    if (G > 0) {
        const size_t lds = mc_lds_words(C) * 4;
        const void *kern = n <= 32 ? (m <= 64 ? (const void *)m_basis_cols_kernel<32, 1>
                                              : (const void *)m_basis_cols_kernel<32, 2>)
                                   : (m <= 64 ? (const void *)m_basis_cols_kernel<64, 1>
                                              : (const void *)m_basis_cols_kernel<64, 2>);
        LBX_TRY_HIP(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        Centred K{R.p, inv_mod32(R.p), (R.p - 1) / 2, one, {}};
        for (int d = 0; d < 7; ++d) {
            const uint32_t c = (uint32_t)(((uint64_t)1 << (8 * d)) % R.p);
            K.c8[d] = (int32_t)(c > K.h ? c - R.p : c);
        }
        DevView in = serie, out = sigma;
        uint64_t *shift_io = R.mb.shift;
        int32_t *part = R.mb.part;
        unsigned *bar = R.mb.bar, bar_base = R.mb.arrivals;
        int oc = (int)out_count;
        void *args[] = {&in, &out, &shift_io, &deg, &part, &bar, &bar_base, &C, &oc, &K};
        // Every group waits for the others at each exchange, so all G must become
        // resident.  G <= 64 groups of one CU each fit on the device together,
        // and groups still queued behind other streams' work are dispatched as
        // that work drains (the barrier's poll limit bounds the wait), so an
        // ordinary launch on the caller's stream serves.  A cooperative launch
        // would go through a queue of its own, with a cross-queue hand-off
        // before and after every base case.
        LBX_TRY(mc_check_groups(G));
        LBX_TRY_HIP(hipLaunchKernel(kern, dim3(G), dim3(kMbThreads), args, lds, R.s));
        const unsigned blocks = (unsigned)((order + C.B - 1) / C.B);
        if (G > 1) R.mb.arrivals += (unsigned)G * std::max(blocks - 1, 1u);
        return LBX_OK;
    }
    const size_t g = serie.rows * serie.cols * order;
    hipLaunchKernelGGL(gather_coeff_major, dim3(grid_for(g)), dim3(256), 0, R.s, serie, order, R.mb.S);
    LBX_TRY_HIP(hipGetLastError());
    // staged words: enough for every coefficient of a step, at most kMbStageWords
    const size_t need = std::max((order + 1) * (m * m + m * n), m * m);
    const int stage = (int)std::min(need, (size_t)kMbStageWords);
    const size_t lds = (3 * m * n + (size_t)stage) * 4;
    auto kern = mont_ok ? m_basis_kernel<AccSmall, true>
                        : (R.p < (1u << 31) ? m_basis_kernel<AccSmall, false> : m_basis_kernel<AccWide, false>);
    LBX_TRY_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(1), dim3(kMbThreads), lds, R.s, R.mb.S, R.mb.W, sigma, R.mb.shift, deg, (int)order,
                       (int)m, (int)n, stage, (int)out_count, R.p, mu, r64, f62, pinv, r2m, one);
    LBX_TRY_HIP(hipGetLastError());
    return LBX_OK;
}

unsigned log2_ceil(size_t x)
{
    unsigned L = 0;
    while (((size_t)1 << L) < x) ++L;
    return L;
}

// c = a.b on device views with the routes of lbx_polymat_mul_u32.
lbx_status product(PmRun &R, const DevView &a, const DevView &b, const DevView &c, size_t m, size_t k, size_t n)
{
    const size_t sa = a.size, sb = b.size, deg = sa + sb - 2;
    const unsigned L = log2_ceil(deg + 1);
    const bool small_p = R.p < (1u << 31);
    if (sa + sb <= 2 && small_p) return constant_product(R.ctx, R.p, a, b, c, m, k, n, R.s);
    if (small_p && (R.p - 1) % ((size_t)1 << L) == 0)
        return fft_prime_product(R.ctx, R.p, L, a, b, c, m, k, n, deg + 1, R.method, R.s);
    return mp_product(R.ctx, &R.p, 1, a, b, c, m, k, n, R.method, R.s);
}

// sigma = sigma2.sigma1 (:297) on all stored coefficients: sigma2 has o2+1 and
// sigma1 o1+1 (zero above their degrees), so sigma gets order+1 coefficients,
// zero above d1+d2, without the degrees being read back.  When order is a
// power of two and an FFT prime reaches it, the product is taken mod
// x^order - 1 (the length the true degrees would need, since d1+d2 <= order)
// and the one coefficient that wraps is put back.  *deg = d[0] + d[1].
lbx_status sigma_product(PmRun &R, uint32_t *s2, size_t o2, uint32_t *s1, size_t o1, const DevView &sigma,
                         size_t order, const uint64_t *d, uint64_t *deg)
{
    const size_t m = R.m;
    const DevView a = polfirst_view(s2, m, m, o2 + 1, o2 + 1), b = polfirst_view(s1, m, m, o1 + 1, o1 + 1);
    const unsigned Lp = log2_ceil(order);
    const size_t P = (size_t)1 << Lp;
    const uint64_t mu = ~(uint64_t)0 / R.p;
    const uint32_t r32 = (uint32_t)(((uint64_t)1 << 32) % R.p), r64 = (uint32_t)((uint64_t)r32 * r32 % R.p);
    DevView c = sigma;
    const bool wrap = P == order && R.p < (1u << 31) && (R.p - 1) % P == 0;
    if (wrap) {
        c.size = P;
        LBX_TRY(fft_prime_product(R.ctx, R.p, Lp, a, b, c, m, m, m, P, R.method, R.s));
    } else {
        c.size = order + 1;
        LBX_TRY(product(R, a, b, c, m, m, m));
    }
    hipLaunchKernelGGL(wrap_fix_kernel, dim3(wrap ? (unsigned)m : 1u), dim3(256), 0, R.s, a, o2, b, o1, sigma, P,
                       (int)m, R.p, mu, r64, wrap, d, deg);
    return from_hip(hipGetLastError());
}

// PM_Basis (:219-326) over device buffers.  sigma gets order+1 coefficients,
// zero above the degree (written to *deg on the device), except that a call
// that is one base case writes out_count of them (degree+1 when 0).
lbx_status pm_basis(PmRun &R, const DevView &serie, const DevView &sigma, size_t order, uint64_t *deg,
                    size_t out_count)
{
    if (order <= kMbThreshold) return run_m_basis(R, serie, sigma, order, deg, out_count);
    const size_t m = R.m, n = R.n, o1 = order >> 1, o2 = order - o1;
    const size_t mark = R.used;
    uint32_t *s1 = R.take(m * m * (o1 + 1) * 4), *ser2 = R.take(m * n * o2 * 4), *s2 = R.take(m * m * (o2 + 1) * 4);
    uint64_t *d12 = (uint64_t *)R.take(16);
    DevView serie1 = serie;
    serie1.size = o1;  // serie1.copy(serie, 0, ord1-1) (:258) as a view
    LBX_TRY(pm_basis(R, serie1, polfirst_view(s1, m, m, o1 + 1, o1 + 1), o1, d12, o1 + 1));
    // serie2 = coefficients ord1..order-1 of sigma1.serie: midproductgen(serie2, sigma1, serie, true,
    // ord1+1, ord1+ord2) (:274) with c.size() = ord2 > 4, the FFT middle product; sigma1 enters
    // with its o1+1 stored coefficients, zero above its degree
    const DevView a = polfirst_view(s1, m, m, o1 + 1, o1 + 1);
    DevView b = serie;
    b.size = order;
    const DevView c = polfirst_view(ser2, m, n, o2, o2);
    const MidSpec mid{true, o1 + 1};
    const unsigned L = log2_ceil(order);
    if (R.p < (1u << 31) && (R.p - 1) % ((size_t)1 << L) == 0)
        LBX_TRY(fft_prime_product(R.ctx, R.p, L, a, b, c, m, m, n, o2, R.method, R.s, &mid));
    else
        LBX_TRY(mp_product(R.ctx, &R.p, 1, a, b, c, m, m, n, R.method, R.s, &mid, L));
    LBX_TRY(pm_basis(R, polfirst_view(ser2, m, n, o2, o2), polfirst_view(s2, m, m, o2 + 1, o2 + 1), o2, d12 + 1,
                     o2 + 1));
    // sigma = sigma2.sigma1 (:297); the resize to d1+d2+1 is the caller's
    LBX_TRY(sigma_product(R, s2, o2, s1, o1, sigma, order, d12, deg));
    R.used = mark;
    return LBX_OK;
}

lbx_status order_basis(lbx_ctx *ctx, uint32_t p, lbx_polmat *sigma, const lbx_polmat *serie, size_t order,
                       size_t *shift, size_t *degree, int method, void *stream, bool divide)
{
    if (!ctx || !sigma || !serie || !shift || !degree) return LBX_ERR_INVALID_ARG;
    LBX_TRY(check_view(sigma));
    LBX_TRY(check_view(serie));
    if (p < 2 || !order || method < 0 || method > 2) return LBX_ERR_INVALID_ARG;
    const size_t m = serie->rows, n = serie->cols;
    if (sigma->rows != m || sigma->cols != m) return LBX_ERR_SIZE_MISMATCH;
    if (serie->size < order || sigma->size < order + 1) return LBX_ERR_SIZE_MISMATCH;
    if (m > (size_t)kMbMaxM || n > (size_t)kMbMaxN || m * n > (size_t)kMbMaxOut * kMbThreads)
        return LBX_ERR_UNSUPPORTED;
    // PM_Basis: the middle products and products of the recursion need
    // transforms of up to 2^ceil(log2(order+1)) points; M_Basis alone keeps
    // its sigma history (order+1 coefficient matrices) on the device
    const size_t max_order = divide ? ((size_t)1 << kMaxLog) - 1 : ((size_t)1 << kMaxLdsLog) - 1;
    if (order > max_order) return LBX_ERR_UNSUPPORTED;
    for (size_t i = 0; i < m; ++i)
        if (shift[i] >= kShiftLimit) return LBX_ERR_UNSUPPORTED;

    std::lock_guard<std::mutex> lock(ctx->mu);
    DeviceGuard guard(ctx->device);
    hipStream_t s = (hipStream_t)stream;
    StreamOrder stream_order(ctx, s);
    const size_t base_order = divide ? std::min(order, kMbThreshold) : order;
    const size_t b_S = align256(m * n * base_order * 4), b_W = align256((base_order + 1) * m * m * 4);
    const size_t b_part = align256(2 * (size_t)kMcMaxBlock * m * n * 4);
    const size_t b_sh = align256(m * 8), b_small = 256;
    const size_t arena = divide ? pm_level_bytes(m, n, order) : 0;
    void *scratch = nullptr;
    LBX_TRY(ensure(ctx, "order_basis", b_S + b_W + b_part + b_sh + 2 * b_small + arena, &scratch));
    uint8_t *base = (uint8_t *)scratch;
    PmRun R{ctx, p, m, n, method, s, {}, base + b_S + b_W + b_part + b_sh + 2 * b_small, 0, arena};
    R.mb.S = (uint32_t *)base;
    R.mb.W = (uint32_t *)(base + b_S);
    R.mb.part = (int32_t *)(base + b_S + b_W);
    R.mb.shift = (uint64_t *)(base + b_S + b_W + b_part);
    R.mb.deg = (uint64_t *)(base + b_S + b_W + b_part + b_sh);
    R.mb.bar = (unsigned *)(base + b_S + b_W + b_part + b_sh + b_small);

    Staged ss, sg;
    lbx_status st = stage_in(ctx, "stage_a", serie, 4, true, &ss, s);
    if (st == LBX_OK) st = stage_in(ctx, "stage_c", sigma, 4, true, &sg, s);
    std::vector<uint64_t> sh(shift, shift + m);
    uint64_t d = 0;
    unsigned failed = 0;
    if (st == LBX_OK) st = from_hip(hipMemcpyAsync(R.mb.shift, sh.data(), m * 8, hipMemcpyHostToDevice, s));
    if (st == LBX_OK) st = from_hip(hipMemsetAsync(R.mb.bar, 0, 8, s));
    if (st == LBX_OK) {
        const DevView dser = devview(serie, ss.dev), dsig = devview(sigma, sg.dev);
        st = divide ? pm_basis(R, dser, dsig, order, R.mb.deg, 0) : run_m_basis(R, dser, dsig, order, R.mb.deg, 0);
    }
    // the one read-back of the call: shift, degree and the grid barrier's failure flag
    if (st == LBX_OK) st = from_hip(hipMemcpyAsync(sh.data(), R.mb.shift, m * 8, hipMemcpyDeviceToHost, s));
    if (st == LBX_OK) st = from_hip(hipMemcpyAsync(&d, R.mb.deg, 8, hipMemcpyDeviceToHost, s));
    if (st == LBX_OK) st = from_hip(hipMemcpyAsync(&failed, R.mb.bar + 1, 4, hipMemcpyDeviceToHost, s));
    if (st == LBX_OK && sg.owned)
        st = device_to_host(ctx, sigma->data, sg.dev, storage_words(sigma) * 4, s);
    const lbx_status sync = from_hip(hipStreamSynchronize(s));
    if (st == LBX_OK) st = sync;
    if (st == LBX_OK && failed) st = LBX_ERR_HIP;  // a grid barrier gave up waiting
    release(ss);
    release(sg);
    if (st == LBX_OK) {
        for (size_t i = 0; i < m; ++i) shift[i] = (size_t)sh[i];
        *degree = (size_t)d;
        sigma->size = (size_t)d + 1;
    }
    return st;
}

}  // namespace
}  // namespace lbx

using namespace lbx;

extern "C" lbx_status lbx_order_basis_pm_u32(lbx_ctx *ctx, uint32_t p, lbx_polmat *sigma, const lbx_polmat *serie,
                                             size_t order, size_t *shift, size_t *degree, int method, void *stream)
{
    return guarded([&]() -> lbx_status {
        return order_basis(ctx, p, sigma, serie, order, shift, degree, method, stream, true);
    });
}

extern "C" lbx_status lbx_order_basis_m_u32(lbx_ctx *ctx, uint32_t p, lbx_polmat *sigma, const lbx_polmat *serie,
                                            size_t order, size_t *shift, size_t *degree, void *stream)
{
    return guarded([&]() -> lbx_status {
        return order_basis(ctx, p, sigma, serie, order, shift, degree, LBX_METHOD_AUTO, stream, false);
    });
}
