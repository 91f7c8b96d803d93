// Multiprecision modulus route: PolynomialMatrixFFTMulDomain<Modular<integer>>::mul
// (matpoly-mult-fft-multiprecision.inl:611-630) over ZRing<integer>::mul_crtla
// (:141-277), and the few-primes route of PolynomialMatrixThreePrimesFFTMulDomain
// (three-primes.inl:67-191) for one-word moduli that are not FFT primes for the
// length.  The reference takes the few-primes domain for p < 2^29 and the
// multiprecision one above (wordsize.inl:62-83); the product is the same either
// way, and here every one-word modulus takes the few-primes route, which needs
// no multiword arithmetic (five times faster at 64x64, degree 4095).
//
// The integer product of the [0,P) representatives has coefficients below
// bound = 2 P^2 k min(sa,sb) (:616).  It is computed modulo FFT primes
// p_i < 2^31 with 2^(lpts+1) | p_i - 1, chosen in the deterministic order of
// RandomFFTPrime::generatePrimes (random-fftprime.h:107-133) until their
// product exceeds the bound, then recombined on the device:
//   1. residue kernel: every nlimbs-word coefficient of both operands -> its
//      residue mod each p_i (signed digits times the powers of 2^32);
//   2. the products mod every p_i: three launches for all primes where the
//      plain pointwise form serves (multi.hip), one product a prime otherwise;
//   3. CRT kernel: X mod P = sum_i y_i (M/p_i mod P) - q (M mod P) with the
//      quotient q from a fixed-point sum, reduced by two quotient digits, or
//      from Garner's mixed-radix digits beyond 32 primes or 16 words.
// The reference picks ~23-bit primes for fgemm on doubles (:162-164); the
// primes here are 31-bit because every step is 32-bit integer arithmetic.
// Products are unique, so the output is identical.
#include <algorithm>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "lbx_ctx.h"
#include "mp_div.h"
#include "plan_key.h"

namespace lbx {

constexpr int kMaxPrimes = 160;
constexpr int kMaxLimbs = 64;

struct MpPlan {
    std::vector<uint32_t> primes;
    unsigned lpts = 0;
    int nlimbs = 0;
    bool reduce = false;          // few-primes plans: some prime is below the modulus
    uint32_t *d_const = nullptr;  // device constant block, layout described at MpLayout / FpLayout / ZzLayout
    size_t res_off = 0;           // word offset of the residue constants (ResidueBlock)
    size_t crt_off = 0;           // word offset of the direct recombination constants (CrtBlock), 0: none
};

namespace {

typedef std::vector<uint32_t> Limbs;

void limbs_trim(Limbs &x)
{
    while (x.size() > 1 && x.back() == 0) x.pop_back();
}

void limbs_mul_small(Limbs &x, uint32_t v)
{
    uint64_t carry = 0;
    for (auto &w : x) {
        const uint64_t t = (uint64_t)w * v + carry;
        w = (uint32_t)t;
        carry = t >> 32;
    }
    if (carry) x.push_back((uint32_t)carry);
}

Limbs limbs_mul(const Limbs &a, const Limbs &b)
{
    Limbs z(a.size() + b.size(), 0);
    for (size_t i = 0; i < a.size(); ++i) {
        uint64_t carry = 0;
        for (size_t j = 0; j < b.size(); ++j) {
            const uint64_t t = (uint64_t)a[i] * b[j] + z[i + j] + carry;
            z[i + j] = (uint32_t)t;
            carry = t >> 32;
        }
        z[i + b.size()] = (uint32_t)carry;
    }
    limbs_trim(z);
    return z;
}

int limbs_cmp(const Limbs &a, const Limbs &b)
{
    const size_t n = a.size() > b.size() ? a.size() : b.size();
    for (size_t i = n; i-- > 0;) {
        const uint32_t x = i < a.size() ? a[i] : 0, y = i < b.size() ? b[i] : 0;
        if (x != y) return x < y ? -1 : 1;
    }
    return 0;
}

int limbs_bits(const Limbs &a)
{
    for (size_t i = a.size(); i-- > 0;)
        if (a[i]) return (int)(i * 32 + 32 - __builtin_clz(a[i]));
    return 0;
}

Limbs limbs_mod(Limbs x, const Limbs &P)
{
    const int bp = limbs_bits(P);
    for (int sh = limbs_bits(x) - bp; sh >= 0; --sh) {
        Limbs t(x.size() + 1, 0);
        for (size_t i = 0; i < P.size(); ++i) {
            const size_t w = i + sh / 32;
            if (w < t.size()) t[w] |= P[i] << (sh % 32);
            if (sh % 32 && w + 1 < t.size()) t[w + 1] |= P[i] >> (32 - sh % 32);
        }
        if (limbs_cmp(x, t) >= 0) {
            uint64_t borrow = 0;
            for (size_t i = 0; i < x.size(); ++i) {
                const uint64_t d = (uint64_t)x[i] - (i < t.size() ? t[i] : 0) - borrow;
                x[i] = (uint32_t)d;
                borrow = (d >> 32) & 1;
            }
        }
    }
    limbs_trim(x);
    return x;
}

typedef unsigned __int128 u128;

uint64_t mulmod_u64(uint64_t a, uint64_t b, uint64_t n) { return (uint64_t)((u128)a * b % n); }

uint64_t powmod_u64(uint64_t a, uint64_t e, uint64_t n)
{
    uint64_t r = 1 % n;
    a %= n;
    while (e) {
        if (e & 1) r = mulmod_u64(r, a, n);
        a = mulmod_u64(a, a, n);
        e >>= 1;
    }
    return r;
}

// Miller-Rabin with the first twelve prime bases: deterministic below 2^64.
bool is_prime(uint64_t n)
{
    static const uint64_t bases[12] = {2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37};
    if (n < 2) return false;
    for (uint64_t q : bases) {
        if (n == q) return true;
        if (n % q == 0) return false;
    }
    uint64_t d = n - 1;
    int s = 0;
    while (!(d & 1)) {
        d >>= 1;
        ++s;
    }
    for (uint64_t a : bases) {
        uint64_t x = powmod_u64(a, d, n);
        if (x == 1 || x == n - 1) continue;
        bool composite = true;
        for (int r = 1; r < s && composite; ++r) {
            x = mulmod_u64(x, x, n);
            if (x == n - 1) composite = false;
        }
        if (composite) return false;
    }
    return true;
}

// random-fftprime.h:107-133 generatePrimes with compute_max_m (:161-166).
bool generate_primes(uint64_t pbound, const Limbs &prodbound, unsigned kmin, std::vector<uint32_t> &out)
{
    out.clear();
    Limbs prod{1};
    if (!kmin) ++kmin;
    const int bits = 64 - __builtin_clzll(pbound - 2);
    for (int k = bits - 1; k > (int)kmin; --k) {
        const uint64_t B = pbound - 1;
        int64_t m = (B & ((1ull << k) - 1)) ? (int64_t)(B >> k) : (int64_t)(B >> k) - 1;
        if (!(m & 1)) --m;
        for (; m > 0; m -= 2) {
            const uint64_t p = ((uint64_t)m << k) + 1;
            if (is_prime(p)) {
                if (out.size() >= (size_t)kMaxPrimes) return false;
                out.push_back((uint32_t)p);
                limbs_mul_small(prod, (uint32_t)p);
                if (limbs_cmp(prod, prodbound) > 0) return true;
            }
        }
    }
    return false;
}

// Constant block of the mixed-radix kernel (32-bit words), in plans whose
// recombination is not the direct one:
//   [0..2r^2)      Garner inverses (p_j mod p_i)^-1 and their Shoup constants, i*r+j
//   then r primes p_i and r words floor(2^32/p_i) (Shoup constant of 1)
//   then r*nlimbs  prod_{j<i} p_j mod P, then nlimbs words of P
// (the inverses first: with the primes first the kernel takes 2% more, 40 primes)
struct MpLayout {
    int r, nl;
    __host__ __device__ int inv() const { return 0; }
    __host__ __device__ int primes() const { return 2 * r * r; }
    __host__ __device__ int onep() const { return 2 * r * r + r; }
    __host__ __device__ int mi() const { return 2 * r * r + 2 * r; }
    __host__ __device__ int P() const { return mi() + r * nl; }
    __host__ __device__ int words() const { return P() + nl; }
};

// Word index of element idx (entry idx / size, coefficient idx % size) of a
// view.  A polfirst view without window (stride = size, no shift) maps idx to
// itself, which spares the per-element 64-bit division.
__device__ __forceinline__ size_t elem_index(const DevView &v, size_t idx, size_t size)
{
    if (v.layout == 0 && v.stor == size && v.shift == 0) return idx;
    const size_t e = idx / size, t = idx - e * size;
    return view_index(v, e, t);
}

// ---- residues --------------------------------------------------------------
// Residues of nl-word coefficients x (unsigned, or two's complement) modulo
// every prime, out[i][e*size + t].  x = sum_l d_l 2^(32 l), l <= nl, with signed
// digits |d_l| <= 2^31 (a carry chain once per coefficient); with the constants
// 2^(32 l) mod p centred to |c| < p/2 < 2^30 each digit is one v_mad_i64_i32 of
// magnitude at most 2^61, folded every third digit (plain_s_fold: after a fold
// |acc| < 2^60 + 2^34, and three more products stay below 2^63) and reduced
// once.  Constants of prime i, kTail + nl + 1 words: the PlainSConst of scale 1
// (c0p, c1, c1p, f60, off), p, then c_0 .. c_nl.
//
// Bound by the multiply-adds (nl + 1 and some ten more products a prime for
// each coefficient), with r words written for nl read.  The words of a group's
// coefficients are staged through LDS where they are contiguous, so the loads
// are whole lines whatever nl is.  Both operands in one launch: 2^20
// coefficients of 6 words each, 14 primes: 91 us in two launches of a Horner
// scheme with two Shoup products a word, 38 us here.
struct ResidueBlock {
    static constexpr int kTail = 7;
    int nl;
    __host__ __device__ int stride() const { return kTail + nl + 1; }
};

void residue_constants(std::vector<uint32_t> &K, const std::vector<uint32_t> &primes, int nl)
{
    for (const uint32_t p : primes) {
        const PlainSConst pc = plain_s_const(p, 1);
        const uint32_t head[ResidueBlock::kTail] = {pc.c0p, pc.c1, pc.c1p, pc.f60, (uint32_t)pc.off,
                                                    (uint32_t)(pc.off >> 32), p};
        K.insert(K.end(), head, head + ResidueBlock::kTail);
        const uint32_t r32 = (uint32_t)(((uint64_t)1 << 32) % p);
        uint32_t w = 1 % p;
        for (int l = 0; l <= nl; ++l) {
            K.push_back((uint32_t)centre(w, p));
            w = (uint32_t)((uint64_t)w * r32 % p);
        }
    }
}

struct ResidueArgs {
    DevView in[2];
    size_t total[2], size[2];
    uint32_t *out[2];
    unsigned blocks0;  // groups of the first operand
};

constexpr int kResidueStage = 8;  // widest coefficient staged through LDS

// NL > 0: nl = NL words; NL = 0: any nl <= kMaxLimbs.
template <int NL, bool SIGNED>
__global__ void __launch_bounds__(256) residue_kernel(ResidueArgs A, int any_nl, int r, const uint32_t *__restrict__ K)
{
    constexpr int NW = NL ? NL : kMaxLimbs;
    __shared__ uint32_t stage[NL ? 256 * NL : 1];
    const int nl = NL ? NL : any_nl;
    const int op = blockIdx.x < A.blocks0 ? 0 : 1;
    const DevView &in = A.in[op];
    const size_t total = A.total[op], size = A.size[op];
    const size_t idx0 = (size_t)(blockIdx.x - (op ? A.blocks0 : 0)) * 256, idx = idx0 + threadIdx.x;
    const bool contiguous = in.layout == 0 && in.stor == size && in.shift == 0;
    uint32_t w[NW];
    if (NL && contiguous) {
        const uint32_t *src = in.base + idx0 * NL;
        const unsigned words = (unsigned)(total - idx0 < 256 ? total - idx0 : 256) * NL;
        uint32_t v[NL ? NL : 1];
#pragma unroll
        for (int j = 0; j < (NL ? NL : 1); ++j) v[j] = src[min(j * 256 + threadIdx.x, words - 1)];  // issued together
#pragma unroll
        for (int j = 0; j < (NL ? NL : 1); ++j) stage[j * 256 + threadIdx.x] = v[j];
        __syncthreads();
        if (idx >= total) return;
#pragma unroll
        for (int l = 0; l < NW; ++l) w[l] = stage[threadIdx.x * NW + l];
    } else {
        if (idx >= total) return;
        const uint32_t *src = in.base + elem_index(in, idx, size) * nl;
#pragma unroll
        for (int l = 0; l < NW; ++l) w[l] = (NL || l < nl) ? src[l] : 0u;
    }
    // signed digits: w_l + carry as a signed word, carry 1 when that subtracts 2^32
    uint32_t carry = 0, top = 0;
#pragma unroll
    for (int l = 0; l < NW; ++l) {
        if (NL || l < nl) {
            if (SIGNED) top = w[l];
            w[l] += carry;
            carry = (w[l] >> 31) | (w[l] < carry ? 1u : 0u);
        }
    }
    const int32_t last = (int32_t)carry - (SIGNED ? (int32_t)(top >> 31) : 0);  // digit nl, in {-1, 0, 1}
    uint32_t *__restrict__ out = A.out[op] + idx;
    for (int i = 0; i < r; ++i, K += ResidueBlock{nl}.stride()) {
        PlainSConst pc;
        pc.c0 = 1;
        pc.c0p = K[0], pc.c1 = K[1], pc.c1p = K[2], pc.f60 = K[3];
        pc.off = ((uint64_t)K[5] << 32) | K[4];
        const uint32_t *c = K + ResidueBlock::kTail;
        int64_t acc = (int64_t)last * (int32_t)c[nl];
#pragma unroll
        for (int l = 0; l < NW; ++l) {
            if (NL || l < nl) {
                if (l % 3 == 2) acc = plain_s_fold(acc, pc);
                acc += (int64_t)(int32_t)w[l] * (int32_t)c[l];
            }
        }
        out[(size_t)i * total] = plain_s_finish(acc, K[6], pc);
    }
}

// Residues of a (ea x a.size coefficients) into ra and of b into rb.
template <bool SIGNED>
hipError_t launch_residues(const DevView &a, size_t ea, uint32_t *ra, const DevView &b, size_t eb, uint32_t *rb, int nl,
                           int r, const uint32_t *K, hipStream_t s)
{
    ResidueArgs A;
    A.in[0] = a, A.in[1] = b;
    A.size[0] = a.size, A.size[1] = b.size;
    A.total[0] = ea * a.size, A.total[1] = eb * b.size;
    A.out[0] = ra, A.out[1] = rb;
    const size_t b0 = (A.total[0] + 255) / 256, b1 = (A.total[1] + 255) / 256;
    if (b0 + b1 > 0x7fffffff) return hipErrorInvalidValue;
    A.blocks0 = (unsigned)b0;
    auto k = residue_kernel<0, SIGNED>;
    switch (nl) {
    case 1: k = residue_kernel<1, SIGNED>; break;
    case 2: k = residue_kernel<2, SIGNED>; break;
    case 3: k = residue_kernel<3, SIGNED>; break;
    case 4: k = residue_kernel<4, SIGNED>; break;
    case 5: k = residue_kernel<5, SIGNED>; break;
    case 6: k = residue_kernel<6, SIGNED>; break;
    case 7: k = residue_kernel<7, SIGNED>; break;
    case 8: k = residue_kernel<8, SIGNED>; break;
    }
    static_assert(kResidueStage == 8, "one kernel per staged width");
    hipLaunchKernelGGL(k, dim3((unsigned)(b0 + b1)), dim3(256), 0, s, A, nl, r, K);
    return hipGetLastError();
}

// Garner recombination of r residues and reduction mod P.
__global__ void __launch_bounds__(128) mp_crt_kernel(const uint32_t *__restrict__ res, size_t entries, size_t size,
                                                     const uint32_t *__restrict__ K, int r, int nl, DevView out)
{
    const size_t total = entries * size;
    const MpLayout lay{r, nl};
    for (size_t idx = (size_t)blockIdx.x * 128 + threadIdx.x; idx < total; idx += (size_t)gridDim.x * 128) {
        uint32_t v[kMaxPrimes];
        uint32_t acc[kMaxLimbs + 2];
        for (int l = 0; l < nl + 2; ++l) acc[l] = 0;
        for (int i = 0; i < r; ++i) {
            const uint32_t p = K[lay.primes() + i], onep = K[lay.onep() + i];
            uint32_t t = res[(size_t)i * total + idx];
            for (int j = 0; j < i; ++j) {
                const uint32_t vj = shoup_mul(v[j], 1u, onep, p);
                t = shoup_mul(sub_mod(t, vj, p), K[lay.inv() + 2 * (i * r + j)], K[lay.inv() + 2 * (i * r + j) + 1], p);
            }
            v[i] = t;
            // acc += v_i * (prod_{j<i} p_j mod P)
            uint64_t carry = 0;
            const uint32_t *mi = K + lay.mi() + i * nl;
            for (int l = 0; l < nl; ++l) {
                const uint64_t s = (uint64_t)mi[l] * t + acc[l] + carry;
                acc[l] = (uint32_t)s;
                carry = s >> 32;
            }
            for (int l = nl; l < nl + 2; ++l) {
                const uint64_t s = (uint64_t)acc[l] + carry;
                acc[l] = (uint32_t)s;
                carry = s >> 32;
            }
        }
        // acc < r 2^31 P <= 2^37 P: binary long division by P << sh, sh = 40..0
        const uint32_t *P = K + lay.P();
        for (int sh = 40; sh >= 0; --sh) {
            const int ws = sh >> 5, bs = sh & 31;
            uint32_t shifted[kMaxLimbs + 2];
            for (int l = 0; l < nl + 2; ++l) {
                const int src = l - ws;
                uint32_t w = 0;
                if (src >= 0 && src < nl) w = P[src] << bs;
                if (bs && src - 1 >= 0 && src - 1 < nl) w |= P[src - 1] >> (32 - bs);
                shifted[l] = w;
            }
            // P < 2^(32 nl) so P << sh (sh <= 40) fits the nl+2 words of acc
            bool ge = true;
            for (int l = nl + 1; l >= 0; --l) {
                if (acc[l] != shifted[l]) {
                    ge = acc[l] > shifted[l];
                    break;
                }
            }
            if (ge) {
                uint64_t borrow = 0;
                for (int l = 0; l < nl + 2; ++l) {
                    const uint64_t d = (uint64_t)acc[l] - shifted[l] - borrow;
                    acc[l] = (uint32_t)d;
                    borrow = (d >> 32) & 1;
                }
            }
        }
        uint32_t *dst = out.base + elem_index(out, idx, size) * nl;
        for (int l = 0; l < nl; ++l) dst[l] = acc[l];
    }
}

// ---- direct recombination ---------------------------------------------------
// X = sum_i y_i (M/p_i) - q M with y_i = r_i (M/p_i)^-1 mod p_i and q =
// floor(sum_i y_i / p_i) (or the nearest integer, for the symmetric range), M
// the product of the primes: r products a coefficient where the mixed-radix
// digits above take r (r-1) / 2 modular ones.  q comes from the fixed-point sum
// S = sum_i y_i floor(2^56 / p_i), at most r 2^31 <= 2^36 below 2^56 sum_i y_i/p_i
// for r <= 32 primes above 2^24 (so that the reciprocals are words).
//  * Modulus P: M > 2 P^2 k min(sa,sb) > 2 X, so sum_i y_i/p_i = q + X/M has its
//    fraction in [0, 1/2): adding 2^37 to S before the shift gives q exactly.
//  * Integers: |X| < bound/2, and the direct form is taken when M > bound (1 +
//    2^-16), so |X/M| < 1/2 - 2^-18: adding 2^55 rounds to the nearest q exactly.
// Other plans (more primes, smaller ones, the rare tight M) keep the kernels
// on mixed-radix digits.  Every word of the sum has a compile-time index: NW
// words, the constants padded to them.  With MOD the sum is taken against
// Q = P 2^(32 off + s), P moved to the top of NW words (sum_i y_i (M_i mod P) + q
// ((-M) mod P) < (32 (2^31 - 1) + 31) P < 2^36 P), reduced by two quotient
// digits of Knuth's division (mp_div.h) and shifted back; without, modulo
// 2^(32 NW).  The group's words leave through LDS where they are contiguous.
//
// Constants: per prime p, (M/p)^-1 mod p with its Shoup constant, floor(2^56 /
// p), NW words of M/p; then NW words of -M; then (MOD) off, s, the reciprocal of
// Q's top word (div21_inverse) and NW words of Q.
// Bound by the multiply-adds: 2047 x 1024 coefficients, 14 primes, 6 words: 140 us
// on mixed-radix digits, 45 us here (57 with the carries rebuilt from comparisons and eight words for six).
struct CrtBlock {
    static constexpr int kHead = 4;
    int r, nw;
    __host__ __device__ int prime(int i) const { return i * (kHead + nw); }
    __host__ __device__ int neg() const { return r * (kHead + nw); }
    __host__ __device__ int sh() const { return neg() + nw; }
    __host__ __device__ int Q() const { return sh() + 3; }
};
constexpr int kCrtMaxPrimes = 32;
constexpr uint32_t kCrtMinPrime = 1u << 24;

// (over[i]:sum[i]) += t * w[i] for N columns: a multiply-add each with its carry
// out, which the compiler would rebuild with comparisons.  A vector instruction may
// read a carry two wait states after the one that wrote it at the earliest, and the
// compiler does not look for that inside an asm block: the products of three or four
// columns come first, then their carries,
// with two or more instructions between;
// two columns take one s_nop.
template <int N>
__device__ __forceinline__ void mad_carry(uint64_t *sum, uint32_t *over, uint32_t t, const uint32_t *w)
{
    static_assert(N >= 2 && N <= 4, "columns of one block");
    uint64_t c0, c1, c2, c3;
    if constexpr (N == 4) {
        asm("v_mad_u64_u32 %0, %8, %12, %13, %0\n\t"
            "v_mad_u64_u32 %1, %9, %12, %14, %1\n\t"
            "v_mad_u64_u32 %2, %10, %12, %15, %2\n\t"
            "v_mad_u64_u32 %3, %11, %12, %16, %3\n\t"
            "v_addc_co_u32_e64 %4, %8, 0, %4, %8\n\t"
            "v_addc_co_u32_e64 %5, %9, 0, %5, %9\n\t"
            "v_addc_co_u32_e64 %6, %10, 0, %6, %10\n\t"
            "v_addc_co_u32_e64 %7, %11, 0, %7, %11"
            : "+&v"(sum[0]), "+&v"(sum[1]), "+&v"(sum[2]), "+&v"(sum[3]), "+&v"(over[0]), "+&v"(over[1]),
              "+&v"(over[2]), "+&v"(over[3]), "=&s"(c0), "=&s"(c1), "=&s"(c2), "=&s"(c3)
            : "v"(t), "s"(w[0]), "s"(w[1]), "s"(w[2]), "s"(w[3]));
    } else if constexpr (N == 3) {
        asm("v_mad_u64_u32 %0, %6, %9, %10, %0\n\t"
            "v_mad_u64_u32 %1, %7, %9, %11, %1\n\t"
            "v_mad_u64_u32 %2, %8, %9, %12, %2\n\t"
            "v_addc_co_u32_e64 %3, %6, 0, %3, %6\n\t"
            "v_addc_co_u32_e64 %4, %7, 0, %4, %7\n\t"
            "v_addc_co_u32_e64 %5, %8, 0, %5, %8"
            : "+&v"(sum[0]), "+&v"(sum[1]), "+&v"(sum[2]), "+&v"(over[0]), "+&v"(over[1]), "+&v"(over[2]),
              "=&s"(c0), "=&s"(c1), "=&s"(c2)
            : "v"(t), "s"(w[0]), "s"(w[1]), "s"(w[2]));
    } else {
        asm("v_mad_u64_u32 %0, %4, %6, %7, %0\n\t"
            "v_mad_u64_u32 %1, %5, %6, %8, %1\n\t"
            "s_nop 0\n\t"
            "v_addc_co_u32_e64 %2, %4, 0, %2, %4\n\t"
            "v_addc_co_u32_e64 %3, %5, 0, %3, %5"
            : "+&v"(sum[0]), "+&v"(sum[1]), "+&v"(over[0]), "+&v"(over[1]), "=&s"(c0), "=&s"(c1)
            : "v"(t), "s"(w[0]), "s"(w[1]));
    }
}

// The same for NW >= 2 columns, in blocks of four and three (and two, of 2 and 5).
template <int NW>
__device__ __forceinline__ void mad_columns(uint64_t *sum, uint32_t *over, uint32_t t, const uint32_t *w)
{
    constexpr int N = NW % 4 == 0 || NW == 7 ? 4 : (NW >= 3 ? 3 : 2);
    mad_carry<N>(sum, over, t, w);
    if constexpr (NW > N) mad_columns<NW - N>(sum + N, over + N, t, w + N);
}

template <int NW, bool MOD>
__global__ void __launch_bounds__(128) crt_direct_kernel(const uint32_t *__restrict__ res, size_t entries, size_t size,
                                                         const uint32_t *__restrict__ K, int r, int ow, DevView out)
{
    constexpr int NA = MOD ? NW + 2 : NW;
    __shared__ uint32_t stage[128 * NW];
    const size_t total = entries * size;
    const CrtBlock lay{r, NW};
    const size_t idx0 = (size_t)blockIdx.x * 128, idx = idx0 + threadIdx.x;
    const bool live = idx < total;
    const size_t at = live ? idx : total - 1;
    // column sums of the products, 64 bits and the carries out of them
    uint64_t col[NW];
    uint32_t over[NW];
#pragma unroll
    for (int l = 0; l < NW; ++l) col[l] = 0, over[l] = 0;
    uint64_t S = MOD ? (uint64_t)1 << 37 : (uint64_t)1 << 55;
    // sum += t * (NW words at w)
    const auto add = [&](uint32_t t, const uint32_t *w) { mad_columns<NW>(col, over, t, w); };
    constexpr int kAhead = 8;  // residues loaded together
    for (int i0 = 0; i0 < r; i0 += kAhead) {
        uint32_t rv[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) rv[j] = i0 + j < r ? res[(size_t)(i0 + j) * total + at] : 0u;
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            if (i0 + j < r) {
                const uint32_t *c = K + lay.prime(i0 + j);
                const uint32_t y = shoup_mul(rv[j], c[1], c[2], c[0]);
                S += (uint64_t)y * c[3];
                add(y, c + CrtBlock::kHead);
            }
        }
    }
    add((uint32_t)(S >> 56), K + lay.neg());
    // the columns as words: column l is col[l] 2^(32 l) + over[l] 2^(32 (l + 2))
    uint32_t acc[NA];
    uint64_t carry = 0;
#pragma unroll
    for (int l = 0; l < NA; ++l) {
        if (l < NW) carry += (uint32_t)col[l];
        if (l >= 1 && l - 1 < NW) carry += col[l - 1] >> 32;
        if (l >= 2) carry += over[l - 2];
        acc[l] = (uint32_t)carry;
        carry >>= 32;
    }
    if constexpr (MOD) {
        const int off = (int)K[lay.sh()], sh = (int)K[lay.sh() + 1];
        uint32_t q[NW];
#pragma unroll
        for (int l = 0; l < NW; ++l) q[l] = K[lay.Q() + l];
        knuth_rem2<NW>(acc, q, K[lay.sh() + 2]);  // Q is normalized: its top word has its top bit set
        // words off.. of acc >> sh; the words of P's leading zero limbs are zero
#pragma unroll
        for (int l = 0; l < NW; ++l)
            if (l >= off && l - off < ow)
                stage[threadIdx.x * ow + l - off] = sh ? (acc[l] >> sh) | (acc[l + 1] << (32 - sh)) : acc[l];
        for (int l = NW - off; l < ow; ++l) stage[threadIdx.x * ow + l] = 0;
    } else {
#pragma unroll
        for (int l = 0; l < NW; ++l)
            if (l < ow) stage[threadIdx.x * ow + l] = acc[l];
    }
    if (out.layout == 0 && out.stor == size && out.shift == 0) {
        __syncthreads();
        uint32_t *dst = out.base + idx0 * ow;
        const int words = (int)(total - idx0 < 128 ? total - idx0 : 128) * ow;
        for (int w = threadIdx.x; w < words; w += 128) dst[w] = stage[w];
    } else if (live) {
        uint32_t *dst = out.base + elem_index(out, idx, size) * ow;
        for (int l = 0; l < ow; ++l) dst[l] = stage[threadIdx.x * ow + l];
    }
}

// Words of the direct kernel that serves r primes and ow-word results, 0 for none.
int crt_words(const std::vector<uint32_t> &primes, int ow)
{
    if (primes.size() > (size_t)kCrtMaxPrimes || ow > 16) return 0;
    for (const uint32_t p : primes)
        if (p < kCrtMinPrime) return 0;
    return ow <= 2 ? 2 : (ow <= 8 ? ow : (ow <= 12 ? 12 : 16));
}

template <bool MOD>
hipError_t launch_crt_direct(int nw, const uint32_t *res, size_t entries, size_t size, const uint32_t *K, int r, int ow,
                             const DevView &out, hipStream_t s)
{
    const size_t grid = (entries * size + 127) / 128;
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    auto k = crt_direct_kernel<16, MOD>;
    switch (nw) {
    case 2: k = crt_direct_kernel<2, MOD>; break;
    case 3: k = crt_direct_kernel<3, MOD>; break;
    case 4: k = crt_direct_kernel<4, MOD>; break;
    case 5: k = crt_direct_kernel<5, MOD>; break;
    case 6: k = crt_direct_kernel<6, MOD>; break;
    case 7: k = crt_direct_kernel<7, MOD>; break;
    case 8: k = crt_direct_kernel<8, MOD>; break;
    case 12: k = crt_direct_kernel<12, MOD>; break;
    }
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(128), 0, s, res, entries, size, K, r, ow, out);
    return hipGetLastError();
}

// Product of the primes, and of all but prime i (i >= 0).
Limbs prime_product(const std::vector<uint32_t> &primes, int skip = -1)
{
    Limbs M{1};
    for (size_t i = 0; i < primes.size(); ++i)
        if ((int)i != skip) limbs_mul_small(M, primes[i]);
    return M;
}

// Appends a CrtBlock: word(x, dst) writes the NW words of the value x (a
// multiword integer) as the kernel's sum takes it.
template <class F, class G>
void crt_constants(std::vector<uint32_t> &K, const std::vector<uint32_t> &primes, int nw, F &&words, G &&neg_words)
{
    const CrtBlock lay{(int)primes.size(), nw};
    const size_t base = K.size();
    K.resize(base + lay.Q() + nw, 0);
    for (size_t i = 0; i < primes.size(); ++i) {
        const uint32_t p = primes[i];
        uint32_t w = 1 % p;
        for (size_t j = 0; j < primes.size(); ++j)
            if (j != i) w = (uint32_t)((uint64_t)w * (primes[j] % p) % p);
        uint32_t *c = &K[base + lay.prime((int)i)];
        c[0] = p;
        c[1] = invmod_h(w, p);
        c[2] = shoup_pre(c[1], p);
        c[3] = (uint32_t)(((uint64_t)1 << 56) / p);
        words(prime_product(primes, (int)i), c + CrtBlock::kHead);
    }
    neg_words(prime_product(primes), &K[base + lay.neg()]);
}

// ---- few-primes route (three-primes.inl:67-191) ----------------------------
// Constants of a few-primes plan, r primes, modulus p < 2^32.
struct FpLayout {
    int r;
    __host__ __device__ int primes() const { return 0; }
    __host__ __device__ int onep() const { return r; }            // Shoup constant of 1 mod p_i
    __host__ __device__ int inv() const { return 2 * r; }         // p_j^-1 mod p_i and its Shoup constant
    __host__ __device__ int beta() const { return 2 * r + 2 * r * r; }  // prod_{j<i} p_j mod p, Shoup constant
    __host__ __device__ int words() const { return beta() + 2 * r; }
};

// Mixed-radix recombination (three-primes.inl:164-181): the Garner digits v_i
// of each coefficient from its residues res[i][idx] (c_i <- (c_i - c_j) p_j^-1
// mod p_i for j < i), then c = sum_i v_i beta_i mod p with beta_i = prod_{j<i}
// p_j mod p, written to the output view.  Every value is a 32-bit word: v_i <
// p_i < 2^31 and Shoup products take any 32-bit multiplicand.  WIDE (p >= 2^31):
// the Shoup remainder x*w - q*p < 2p and the sum are held in 64 bits.  `out`
// may be res[0]'s own storage.
template <int RM, bool WIDE>
__global__ void __launch_bounds__(256) few_primes_crt_kernel(const uint32_t *res, size_t entries,
                                                             size_t size, const uint32_t *__restrict__ K, int r,
                                                             uint32_t p, DevView out)
{
    const size_t total = entries * size;
    const FpLayout lay{r};
    for (size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (size_t)gridDim.x * 256) {
        uint32_t v[RM], rv[RM];
        uint32_t acc = 0;
#pragma unroll
        for (int i = 0; i < RM; ++i) rv[i] = i < r ? res[(size_t)i * total + idx] : 0u;  // loads issued together
#pragma unroll
        for (int i = 0; i < RM; ++i) {
            if (i < r) {
                const uint32_t pi = K[lay.primes() + i], onep = K[lay.onep() + i];
                uint32_t t = rv[i];
#pragma unroll
                for (int j = 0; j < i; ++j) {
                    const uint32_t vj = shoup_mul(v[j], 1u, onep, pi);
                    t = shoup_mul(sub_mod(t, vj, pi), K[lay.inv() + 2 * (i * r + j)],
                                  K[lay.inv() + 2 * (i * r + j) + 1], pi);
                }
                v[i] = t;
                const uint32_t w = K[lay.beta() + 2 * i], wp = K[lay.beta() + 2 * i + 1];
                if constexpr (!WIDE) {
                    acc = add_mod(acc, shoup_mul(t, w, wp, p), p);
                } else {
                    uint64_t y = (uint64_t)t * w - (uint64_t)mulhi32(t, wp) * p;
                    if (y >= p) y -= p;
                    y += acc;
                    if (y >= p) y -= p;
                    acc = (uint32_t)y;
                }
            }
        }
        out.base[elem_index(out, idx, size)] = acc;
    }
}

// Residues of one-word coefficients modulo every prime of a few-primes plan,
// out[i][e*size + t] (the finit of three-primes.inl:143-146), for plans with a
// prime below the modulus.
__global__ void __launch_bounds__(256) fp_residue_kernel(DevView in, size_t entries, size_t size,
                                                         const uint32_t *__restrict__ K, int r,
                                                         uint32_t *__restrict__ out)
{
    const size_t total = entries * size;
    const FpLayout lay{r};
    for (size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x; idx < total; idx += (size_t)gridDim.x * 256) {
        const uint32_t x = in.base[elem_index(in, idx, size)];
        for (int i = 0; i < r; ++i)
            out[(size_t)i * total + idx] = shoup_mul(x, 1u, K[lay.onep() + i], K[lay.primes() + i]);
    }
}

constexpr int kFewMaxPrimes = 8;

unsigned grid_of(size_t total, unsigned block)
{
    const size_t g = (total + block - 1) / block;
    return (unsigned)(g < 8192 ? (g ? g : 1) : 8192);
}

// The r products c_i = a_i b_i mod p_i of one shape (operand i of a at the view
// a + i * astride words, b alike; c_i polfirst with sc coefficients, one after
// the other).  Where the pointwise form is the plain one on whole transforms,
// all primes go through three launches, in chunks of primes whose transforms
// fit kMultiWords words of scratch (larger products fill the chip prime by
// prime); a prime by itself otherwise.  Measured (us), one prime at a time /
// chunks of 2^24 / 2^25 / 2^26 / 2^27 words: 14 primes of 32^3 at 2^11 points
// 950 / 668 / 617 / 580 / 583; 3 primes of 16^3 at 2^11 78 / 46 / 45 / 45 / 46; 3 of
// 32^3 at 2^13 372 / 372 / 373 / 371 / 373.
constexpr size_t kMultiWords = (size_t)1 << 26;

lbx_status prime_products(lbx_ctx *ctx, const std::vector<uint32_t> &primes, const DevView &a, size_t astride,
                          const DevView &b, size_t bstride, uint32_t *c, size_t m, size_t k, size_t n, size_t sc,
                          unsigned L, int method, hipStream_t s, const MidSpec *mid)
{
    const size_t r = primes.size();
    if (choose_method(method, m, k, n, L, primes[0], r) != LBX_METHOD_PLAIN_U64 || L < 1 || L > (unsigned)kMaxLdsLog) {
        for (size_t i = 0; i < r; ++i) {
            DevView va = a, vb = b;
            va.base += i * astride;
            vb.base += i * bstride;
            const DevView vc{c + i * m * n * sc, LBX_POLFIRST, m, n, sc, 0, sc};
            if (!mid && a.size + b.size <= 2 && sc == 1)
                LBX_TRY(constant_product(ctx, primes[i], va, vb, vc, m, k, n, s));
            else
                LBX_TRY(fft_prime_product(ctx, primes[i], L, va, vb, vc, m, k, n, sc, method, s, mid));
        }
        return LBX_OK;
    }
    const size_t N = (size_t)1 << L, words = (m * k + k * n + m * n) * N;
    const size_t chunk = std::min<size_t>({std::max<size_t>(kMultiWords / words, 1), r, (size_t)kMultiPrimes});
    CtxWorkspace ws(ctx);
    MultiProduct mp{};
    mp.L = L;
    mp.m = m, mp.k = k, mp.n = n;
    mp.astride = astride, mp.bstride = bstride;
    mp.rev_a = mid && mid->small_left ? mid->hdeg : 0;
    mp.rev_b = mid && !mid->small_left ? mid->hdeg : 0;
    mp.cstride = m * n * sc;
    mp.count = sc;
    void *ahat, *bhat, *chat;
    LBX_TRY(ws.get("ahat", chunk * m * k * N * 4, &ahat));
    LBX_TRY(ws.get("bhat", chunk * k * n * N * 4, &bhat));
    LBX_TRY(ws.get("chat", chunk * m * n * N * 4, &chat));
    mp.ahat = (uint32_t *)ahat, mp.bhat = (uint32_t *)bhat, mp.chat = (uint32_t *)chat;
    for (size_t i0 = 0; i0 < r; i0 += chunk) {
        mp.r = (unsigned)std::min(chunk, r - i0);
        mp.a = a, mp.b = b;
        mp.a.base += i0 * astride;
        mp.b.base += i0 * bstride;
        mp.c = DevView{c + i0 * mp.cstride, LBX_POLFIRST, m, n, sc, 0, sc};
        for (unsigned i = 0; i < mp.r; ++i) LBX_TRY(multi_prime(mp, i, primes[i0 + i], mid, ws, s));
        LBX_TRY_HIP(launch_multi_forward(mp, s));
        LBX_TRY_HIP(launch_multi_pointwise(mp, s));
        LBX_TRY_HIP(launch_multi_inverse(mp, s));
    }
    return LBX_OK;
}

// Primes, Shoup constants of 1 and Garner inverses (p_j mod p_i)^-1 with their Shoup
// constants at 2(i r + j), j < i, of a mixed-radix recombination.
void garner_constants(std::vector<uint32_t> &K, const std::vector<uint32_t> &primes, int at_primes, int at_one,
                      int at_inv)
{
    const size_t r = primes.size();
    for (size_t i = 0; i < r; ++i) {
        const uint32_t p = primes[i];
        K[at_primes + i] = p;
        K[at_one + i] = shoup_pre(1, p);
        for (size_t j = 0; j < i; ++j) {
            const uint32_t inv = invmod_h(primes[j] % p, p);
            K[at_inv + 2 * (i * r + j)] = inv;
            K[at_inv + 2 * (i * r + j) + 1] = shoup_pre(inv, p);
        }
    }
}

lbx_status upload_plan(MpPlan *plan, const std::vector<uint32_t> &K)
{
    LBX_TRY_HIP(hipMalloc(&plan->d_const, K.size() * 4));
    const hipError_t e = hipMemcpy(plan->d_const, K.data(), K.size() * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) return LBX_OK;
    (void)hipFree(plan->d_const);
    plan->d_const = nullptr;
    return from_hip(e);
}

lbx_status get_plan(lbx_ctx *ctx, const uint32_t *Pw, int nl, size_t k, size_t minsz, unsigned lpts, MpPlan **out)
{
    const std::string key = mp_plan_key(Pw, nl, k, minsz, lpts);
    auto it = ctx->mp_plans.find(key);
    if (it != ctx->mp_plans.end()) {
        *out = it->second;
        return LBX_OK;
    }
    Limbs P(Pw, Pw + nl);
    limbs_trim(P);
    if (P.size() == 1 && P[0] < 2) return LBX_ERR_INVALID_ARG;
    Limbs bound = limbs_mul(P, P);  // :616 bound = 2 P^2 k min(sa,sb)
    limbs_mul_small(bound, 2);
    limbs_mul_small(bound, (uint32_t)k);
    limbs_mul_small(bound, (uint32_t)minsz);
    std::vector<uint32_t> primes;
    if (!generate_primes((uint64_t)1 << 31, bound, lpts, primes)) return LBX_ERR_NOT_ENOUGH_PRIMES;
    const int r = (int)primes.size(), nw = crt_words(primes, nl);
    std::vector<uint32_t> K;
    std::unique_ptr<MpPlan> plan(new MpPlan());
    plan->primes = primes;
    plan->lpts = lpts;
    plan->nlimbs = nl;
    if (!nw) {
        const MpLayout lay{r, nl};
        K.resize((size_t)lay.words(), 0);
        garner_constants(K, primes, lay.primes(), lay.onep(), lay.inv());
        Limbs M{1};
        for (int i = 0; i < r; ++i) {
            const Limbs mi = limbs_mod(M, P);
            for (int l = 0; l < nl; ++l) K[lay.mi() + i * nl + l] = l < (int)mi.size() ? mi[l] : 0;
            limbs_mul_small(M, primes[i]);
            M = limbs_mod(M, P);
        }
        for (int l = 0; l < nl; ++l) K[lay.P() + l] = Pw[l];
    }
    plan->res_off = K.size();
    residue_constants(K, primes, nl);
    if (nw) {
        // P at the top of nw words with its top bit set: Q = P 2^(32 off + sh)
        const int np = (int)P.size(), off = nw - np, sh = __builtin_clz(P.back());
        const auto place = [&](const Limbs &x, uint32_t *dst) {  // x < P: x 2^(32 off + sh) in nw words
            uint32_t prev = 0;
            for (int l = 0; l < np; ++l) {
                const uint32_t w = l < (int)x.size() ? x[l] : 0u;
                dst[off + l] = sh ? (w << sh) | prev : w;
                prev = sh ? w >> (32 - sh) : 0u;
            }
        };
        plan->crt_off = K.size();
        const CrtBlock cb{r, nw};
        crt_constants(K, primes, nw, [&](const Limbs &x, uint32_t *dst) { place(limbs_mod(x, P), dst); },
                      [&](const Limbs &x, uint32_t *dst) {  // (-M) mod P
                          const Limbs mm = limbs_mod(x, P);
                          Limbs d(np, 0);
                          uint64_t borrow = 0;
                          for (int l = 0; l < np; ++l) {
                              const uint64_t t = (uint64_t)P[l] - (l < (int)mm.size() ? mm[l] : 0) - borrow;
                              d[l] = (uint32_t)t;
                              borrow = (t >> 32) & 1;
                          }
                          place(limbs_mod(d, P), dst);
                      });
        K[plan->crt_off + cb.sh()] = (uint32_t)off;
        K[plan->crt_off + cb.sh() + 1] = (uint32_t)sh;
        place(P, &K[plan->crt_off + cb.Q()]);
        K[plan->crt_off + cb.sh() + 2] = div21_inverse(K[plan->crt_off + cb.Q() + nw - 1]);
    }
    LBX_TRY(upload_plan(plan.get(), K));
    ctx->mp_plans[key] = plan.get();
    *out = plan.release();
    return LBX_OK;
}

// Plan of the few-primes route: bound = (p-1)^2 k min(sa,sb) (three-primes.inl:75-76,
// 180-181 of mul, :225-226 of midproduct), FFT primes below 2^31 with
// 2^lpts | p_i - 1 in the order of generatePrimes until their product exceeds
// the bound (:116-121).  r = 0 (the caller then takes the multiprecision
// route) when more than kFewMaxPrimes would be needed; `reduce` when some
// p_i <= p, whose operands need the reduction of :143-146.
lbx_status get_few_plan(lbx_ctx *ctx, uint32_t p, size_t k, size_t minsz, unsigned lpts, MpPlan **out)
{
    const std::string key = few_plan_key(p, k, minsz, lpts);
    auto it = ctx->mp_plans.find(key);
    if (it != ctx->mp_plans.end()) {
        *out = it->second;
        return LBX_OK;
    }
    Limbs bound{p - 1};
    limbs_mul_small(bound, p - 1);
    limbs_mul_small(bound, (uint32_t)k);
    limbs_mul_small(bound, (uint32_t)minsz);
    std::vector<uint32_t> primes;
    if (!generate_primes((uint64_t)1 << 31, bound, lpts, primes)) return LBX_ERR_NOT_ENOUGH_PRIMES;
    std::unique_ptr<MpPlan> plan(new MpPlan());
    plan->lpts = lpts;
    plan->nlimbs = 1;
    for (uint32_t q : primes) plan->reduce = plan->reduce || q <= p;
    if ((int)primes.size() <= kFewMaxPrimes) {
        const int r = (int)primes.size();
        const FpLayout lay{r};
        std::vector<uint32_t> K((size_t)lay.words(), 0);
        garner_constants(K, primes, lay.primes(), lay.onep(), lay.inv());
        uint32_t beta = 1 % p;
        for (int i = 0; i < r; ++i) {
            const uint32_t pi = primes[i];
            K[lay.beta() + 2 * i] = beta;
            K[lay.beta() + 2 * i + 1] = shoup_pre(beta, p);
            beta = (uint32_t)((uint64_t)beta * (pi % p) % p);  // beta *= p_i (:179-180)
        }
        LBX_TRY(upload_plan(plan.get(), K));
        plan->primes = primes;
    }
    ctx->mp_plans[key] = plan.get();
    *out = plan.release();
    return LBX_OK;
}

}  // namespace

void mp_release(lbx_ctx *ctx)
{
    for (auto &kv : ctx->mp_plans) {
        if (kv.second->d_const) (void)hipFree(kv.second->d_const);
        delete kv.second;
    }
    ctx->mp_plans.clear();
}

lbx_status mp_product(lbx_ctx *ctx, const uint32_t *Pw, int nl, const DevView &a, const DevView &b, const DevView &c,
                      size_t m, size_t k, size_t n, int method, hipStream_t s, const MidSpec *mid, unsigned mid_L,
                      size_t count)
{
    // product: s = max_rowdeg+1 coefficients when given, else sa+sb-1 (mul_crtla :150-152;
    // three-primes.inl:69-73); with fewer than sa+sb-1 the cyclic product mod x^pts - 1
    const size_t sa = a.size, sb = b.size, sc = mid ? c.size : (count ? count : sa + sb - 1);
    unsigned lpts = 0;
    size_t pts = 1;
    while (pts < sc) {  // mul_crtla :151-154
        pts <<= 1;
        ++lpts;
    }
    if (mid) {  // midproduct_crtla :446-447: points from deg, not from the output size
        lpts = mid_L;
        pts = (size_t)1 << lpts;
    }
    const size_t minsz = sa < sb ? sa : sb;
    if (nl == 1 && Pw[0] >= 2) {
        // few-primes route (wordsize.inl:66-68): with every p_i > p the operands
        // are already residues mod p_i (three-primes.inl:138-142), so the
        // per-prime products read them where they are; else one pass writes
        // their residues first (:143-146)
        MpPlan *fp;
        LBX_TRY(get_few_plan(ctx, Pw[0], k, minsz, lpts, &fp));
        const int r = (int)fp->primes.size();
        if (r > 0) {
            void *ra = nullptr, *rb = nullptr, *rc;
            if (fp->reduce) {
                LBX_TRY(ensure(ctx, "mp_ra", (size_t)r * m * k * sa * 4, &ra));
                LBX_TRY(ensure(ctx, "mp_rb", (size_t)r * k * n * sb * 4, &rb));
                hipLaunchKernelGGL(fp_residue_kernel, dim3(grid_of(m * k * sa, 256)), dim3(256), 0, s, a, m * k, sa,
                                   fp->d_const, r, (uint32_t *)ra);
                LBX_TRY_HIP(hipGetLastError());
                hipLaunchKernelGGL(fp_residue_kernel, dim3(grid_of(k * n * sb, 256)), dim3(256), 0, s, b, k * n, sb,
                                   fp->d_const, r, (uint32_t *)rb);
                LBX_TRY_HIP(hipGetLastError());
            }
            LBX_TRY(ensure(ctx, "mp_rc", (size_t)r * m * n * sc * 4, &rc));
            // every prime's product reads the operands: those stored by
            // coefficient become polfirst once, for all of them (a copy that
            // there is no memory for is left to the products)
            const auto as_polfirst = [&](const DevView &v, size_t entries, const char *slot) -> DevView {
                const size_t stor = (v.size + 3) & ~(size_t)3;
                void *buf;
                if (fp->reduce || !copies_to_polfirst(v, entries, v.size, lpts, CopyUse::kSharedOperand)) return v;
                if (ensure(ctx, slot, entries * stor * 4, &buf) != LBX_OK) {
                    (void)hipGetLastError();
                    return v;
                }
                const DevView pf{(uint32_t *)buf, LBX_POLFIRST, v.rows, v.cols, stor, 0, v.size};
                return launch_copy(v, pf, entries, v.size, 0, 0, s) == hipSuccess ? pf : v;
            };
            const DevView a1 = as_polfirst(a, m * k, "mp_ra"), b1 = as_polfirst(b, k * n, "mp_rb");
            DevView va = a1, vb = b1;
            if (fp->reduce) {
                va = DevView{(uint32_t *)ra, LBX_POLFIRST, m, k, sa, 0, sa};
                vb = DevView{(uint32_t *)rb, LBX_POLFIRST, k, n, sb, 0, sb};
            }
            LBX_TRY(prime_products(ctx, fp->primes, va, fp->reduce ? m * k * sa : 0, vb, fp->reduce ? k * n * sb : 0,
                                   (uint32_t *)rc, m, k, n, sc, lpts, method, s, mid));
            // a result stored by coefficient is recombined polfirst, in the place
            // of the first prime's residues, and copied out in one pass
            DevView cv = c;
            if (copies_to_polfirst(c, m * n, sc, lpts, CopyUse::kRecombined))
                cv = DevView{(uint32_t *)rc, LBX_POLFIRST, m, n, sc, 0, sc};
            const dim3 grid(grid_of(m * n * sc, 256));
            if (Pw[0] >= (1u << 31))
                hipLaunchKernelGGL((few_primes_crt_kernel<kFewMaxPrimes, true>), grid, dim3(256), 0, s,
                                   (const uint32_t *)rc, m * n, sc, fp->d_const, r, Pw[0], cv);
            else
                hipLaunchKernelGGL((few_primes_crt_kernel<kFewMaxPrimes, false>), grid, dim3(256), 0, s,
                                   (const uint32_t *)rc, m * n, sc, fp->d_const, r, Pw[0], cv);
            LBX_TRY_HIP(hipGetLastError());
            if (cv.base != c.base) LBX_TRY_HIP(launch_copy(cv, c, m * n, sc, 0, 0, s));
            return LBX_OK;
        }
    }
    MpPlan *plan;
    LBX_TRY(get_plan(ctx, Pw, nl, k, minsz, lpts, &plan));
    const int r = (int)plan->primes.size();
    void *ra, *rb, *rc;
    LBX_TRY(ensure(ctx, "mp_ra", (size_t)r * m * k * sa * 4, &ra));
    LBX_TRY(ensure(ctx, "mp_rb", (size_t)r * k * n * sb * 4, &rb));
    LBX_TRY(ensure(ctx, "mp_rc", (size_t)r * m * n * sc * 4, &rc));
    LBX_TRY_HIP(launch_residues<false>(a, m * k, (uint32_t *)ra, b, k * n, (uint32_t *)rb, nl, r,
                                       plan->d_const + plan->res_off, s));
    const DevView va{(uint32_t *)ra, LBX_POLFIRST, m, k, sa, 0, sa}, vb{(uint32_t *)rb, LBX_POLFIRST, k, n, sb, 0, sb};
    LBX_TRY(prime_products(ctx, plan->primes, va, m * k * sa, vb, k * n * sb, (uint32_t *)rc, m, k, n, sc, lpts, method,
                           s, mid));
    if (plan->crt_off)
        return from_hip(launch_crt_direct<true>(crt_words(plan->primes, nl), (const uint32_t *)rc, m * n, sc,
                                                plan->d_const + plan->crt_off, r, nl, c, s));
    hipLaunchKernelGGL(mp_crt_kernel, dim3(grid_of(m * n * sc, 128)), dim3(128), 0, s, (const uint32_t *)rc, m * n, sc,
                       plan->d_const, r, nl, c);
    LBX_TRY_HIP(hipGetLastError());
    return LBX_OK;
}

// ---- products over the integers: PolynomialMatrixFFTMulDomain<ZRing<integer>> ----
// (matpoly-mult-fft-multiprecision.inl:43-89 with mul_crtla, :141-277).
// Coefficients are nl-word (inputs) and cl-word (output) two's complement
// integers.  As in the reference, maxA = 2^(largest bit size of a's
// coefficients), likewise maxB, and bound = 2 maxA maxB k min(sa,sb) (:78-86);
// the product is taken modulo FFT primes whose product M exceeds the bound and
// reconstructed in the symmetric range.  The primes are odd, so the mixed-radix
// digits of (M-1)/2 are all (p_i-1)/2: a value is negative (X > (M-1)/2) when
// its Garner digits, read from the most significant, first exceed them.  The
// output X - [X > (M-1)/2] M is formed modulo 2^(32 cl), which holds it.
constexpr int kZzMaxIn = 32;      // words of an input coefficient
constexpr int kZzMaxOut = 80;     // words of an output coefficient
constexpr int kZzMaxPrimes = 96;

namespace {

// Constant block of the mixed-radix kernel, in plans whose recombination is not
// the direct one: primes, Shoup constants of 1, Garner inverses (p_j mod p_i)^-1
// with their Shoup constants at 2(i r + j), then W_i = prod_{j<i} p_j mod 2^(32 cl)
// in cl words each, then M mod 2^(32 cl).
struct ZzLayout {
    int r, cl;
    __host__ __device__ int primes() const { return 0; }
    __host__ __device__ int onep() const { return r; }
    __host__ __device__ int inv() const { return 2 * r; }
    __host__ __device__ int W() const { return 2 * r + 2 * r * r; }
    __host__ __device__ int M() const { return W() + r * cl; }
    __host__ __device__ int words() const { return M() + cl; }
};

// Largest bit size of the absolute values of nl-word two's complement
// coefficients (Givaro's bitsize, 0 for 0) of both operands: group g writes the
// maximum of its share to out[g], in pinned host memory that the host reduces
// after its wait (groups [0, gridDim.x/2) the first operand, the rest the
// second).  The share of a group is a run of coefficients, so a wave reads
// 64 nl contiguous words.  One launch and one wait for both operands: 2 x 404K
// coefficients of two words took 75 us each with an atomic maximum per wave,
// 6 us for both here.
constexpr unsigned kLogmaxGroups = 256;  // groups an operand

__global__ void __launch_bounds__(256) zz_logmax_kernel(DevView a, size_t ea, DevView b, size_t eb, int nl,
                                                        unsigned *__restrict__ out)
{
    __shared__ unsigned wave_max[4];
    const unsigned half = gridDim.x / 2;
    const bool second = blockIdx.x >= half;
    const DevView &in = second ? b : a;
    const size_t size = in.size, total = (second ? eb : ea) * size;
    unsigned best = 0;
    for (size_t idx = (size_t)(blockIdx.x - (second ? half : 0)) * 256 + threadIdx.x; idx < total;
         idx += (size_t)half * 256) {
        const uint32_t *src = in.base + elem_index(in, idx, size) * nl;
        const bool neg = src[nl - 1] >> 31;
        // |x|: the words themselves, or their two's complement negation
        uint32_t carry = 1;
        unsigned bits = 0;
        for (int l = 0; l < nl; ++l) {
            uint32_t w = src[l];
            if (neg) {
                const uint32_t t = ~w + carry;
                carry = carry && t == 0;
                w = t;
            }
            if (w) bits = 32 * l + 32 - __builtin_clz(w);
        }
        best = bits > best ? bits : best;
    }
    for (int off = 32; off; off >>= 1) {
        const unsigned o = __shfl_xor(best, off);
        best = o > best ? o : best;
    }
    if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) best = wave_max[w] > best ? wave_max[w] : best;
        out[blockIdx.x] = best;
    }
}

// Garner digits of each coefficient's r residues, the sign test against the
// digits (p_i-1)/2, and X - [negative] M modulo 2^(32 cl) in cl words.
__global__ void __launch_bounds__(128) zz_crt_kernel(const uint32_t *__restrict__ res, size_t entries, size_t size,
                                                     const uint32_t *__restrict__ K, int r, int cl, DevView out)
{
    const size_t total = entries * size;
    const ZzLayout lay{r, cl};
    for (size_t idx = (size_t)blockIdx.x * 128 + threadIdx.x; idx < total; idx += (size_t)gridDim.x * 128) {
        uint32_t v[kZzMaxPrimes];
        uint32_t acc[kZzMaxOut];
        for (int l = 0; l < cl; ++l) acc[l] = 0;
        for (int i = 0; i < r; ++i) {
            const uint32_t p = K[lay.primes() + i], onep = K[lay.onep() + i];
            uint32_t t = res[(size_t)i * total + idx];
            for (int j = 0; j < i; ++j) {
                const uint32_t vj = shoup_mul(v[j], 1u, onep, p);
                t = shoup_mul(sub_mod(t, vj, p), K[lay.inv() + 2 * (i * r + j)], K[lay.inv() + 2 * (i * r + j) + 1], p);
            }
            v[i] = t;
            // acc += v_i W_i (mod 2^(32 cl))
            const uint32_t *w = K + lay.W() + i * cl;
            uint64_t carry = 0;
            for (int l = 0; l < cl; ++l) {
                const uint64_t s = (uint64_t)w[l] * t + acc[l] + carry;
                acc[l] = (uint32_t)s;
                carry = s >> 32;
            }
        }
        bool neg = false;
        for (int i = r - 1; i >= 0; --i) {
            const uint32_t h = (K[lay.primes() + i] - 1) / 2;
            if (v[i] != h) {
                neg = v[i] > h;
                break;
            }
        }
        if (neg) {
            const uint32_t *Mm = K + lay.M();
            uint64_t borrow = 0;
            for (int l = 0; l < cl; ++l) {
                const uint64_t d = (uint64_t)acc[l] - Mm[l] - borrow;
                acc[l] = (uint32_t)d;
                borrow = (d >> 32) & 1;
            }
        }
        uint32_t *dst = out.base + elem_index(out, idx, size) * cl;
        for (int l = 0; l < cl; ++l) dst[l] = acc[l];
    }
}

// Largest coefficient bit sizes of both operands.
lbx_status zz_logmax(lbx_ctx *ctx, const DevView &a, const DevView &b, int nl, unsigned *la, unsigned *lb,
                     hipStream_t s)
{
    if (!ctx->zz_bits)
        LBX_TRY_HIP(hipHostMalloc((void **)&ctx->zz_bits, 2 * kLogmaxGroups * sizeof(unsigned), hipHostMallocDefault));
    const size_t ea = a.rows * a.cols, eb = b.rows * b.cols, most = std::max(ea * a.size, eb * b.size);
    const unsigned half = (unsigned)std::min<size_t>(kLogmaxGroups, (most + 255) / 256);
    hipLaunchKernelGGL(zz_logmax_kernel, dim3(2 * half), dim3(256), 0, s, a, ea, b, eb, nl, ctx->zz_bits);
    LBX_TRY_HIP(hipGetLastError());
    LBX_TRY_HIP(hipStreamSynchronize(s));
    const unsigned *v = ctx->zz_bits;
    *la = *std::max_element(v, v + half);
    *lb = *std::max_element(v + half, v + 2 * half);
    return LBX_OK;
}

// Plan of an integer product: FFT primes whose product exceeds bound = 2 maxA
// maxB k min(sa,sb), maxA maxB = 2^lab (:78-86), and the constants for nl-word
// inputs and cl-word results.  Kept in the context by these numbers; at most
// kZzPlans of them (other data of the same program has few bit sizes).
constexpr size_t kZzPlans = 64;

lbx_status get_zz_plan(lbx_ctx *ctx, unsigned lab, size_t k, size_t minsz, unsigned lpts, int nl, int cl, MpPlan **out)
{
    const std::string prefix = kZzPlanTag, key = zz_plan_key(lab, k, minsz, lpts, nl, cl);
    const auto it = ctx->mp_plans.find(key);
    if (it != ctx->mp_plans.end()) {
        *out = it->second;
        return LBX_OK;
    }
    Limbs bound{1};
    for (unsigned i = 0; i < lab + 1; ++i) limbs_mul_small(bound, 2);
    limbs_mul_small(bound, (uint32_t)k);
    limbs_mul_small(bound, (uint32_t)minsz);
    limbs_trim(bound);
    const size_t bits = 32 * (bound.size() - 1) + 32 - __builtin_clz(bound.back());  // bound < 2^bits
    if (bits > (size_t)32 * cl) return LBX_ERR_SIZE_MISMATCH;  // bound/2 < 2^(bits-1) needs bits-1 bits and a sign
    std::vector<uint32_t> primes;
    if (!generate_primes((uint64_t)1 << 31, bound, lpts, primes) || (int)primes.size() > kZzMaxPrimes)
        return LBX_ERR_NOT_ENOUGH_PRIMES;
    const int r = (int)primes.size();
    const auto low = [&](const Limbs &x, uint32_t *dst, int n) {  // x mod 2^(32 n)
        for (int l = 0; l < n; ++l) dst[l] = l < (int)x.size() ? x[l] : 0;
    };
    // the direct form where M > bound (1 + 2^-16): M 2^16 > bound (2^16 + 1)
    Limbs lhs = prime_product(primes), rhs = bound;
    limbs_mul_small(lhs, 1u << 16);
    limbs_mul_small(rhs, (1u << 16) + 1);
    const int nw = limbs_cmp(lhs, rhs) > 0 ? crt_words(primes, cl) : 0;
    std::vector<uint32_t> K;
    std::unique_ptr<MpPlan> plan(new MpPlan());
    plan->primes = primes;
    plan->lpts = lpts;
    plan->nlimbs = nl;
    if (!nw) {
        const ZzLayout lay{r, cl};
        K.resize((size_t)lay.words(), 0);
        garner_constants(K, primes, lay.primes(), lay.onep(), lay.inv());
        Limbs W{1};  // prod_{j<i} p_j
        for (int i = 0; i < r; ++i) {
            low(W, &K[lay.W() + i * cl], cl);
            limbs_mul_small(W, primes[i]);
        }
        low(W, &K[lay.M()], cl);
    }
    plan->res_off = K.size();
    residue_constants(K, primes, nl);
    if (nw) {
        plan->crt_off = K.size();
        crt_constants(K, primes, nw, [&](const Limbs &x, uint32_t *dst) { low(x, dst, nw); },
                      [&](const Limbs &x, uint32_t *dst) {  // -M mod 2^(32 nw)
                          low(x, dst, nw);
                          uint32_t carry = 1;
                          for (int l = 0; l < nw; ++l) {
                              dst[l] = ~dst[l] + carry;
                              carry = carry && dst[l] == 0;
                          }
                      });
    }
    size_t held = 0;
    for (const auto &kv : ctx->mp_plans) held += kv.first.compare(0, prefix.size(), prefix) == 0;
    if (held >= kZzPlans) {  // their constants may be in use by work still queued
        (void)hipDeviceSynchronize();
        for (auto p = ctx->mp_plans.begin(); p != ctx->mp_plans.end();) {
            if (p->first.compare(0, prefix.size(), prefix) != 0) {
                ++p;
                continue;
            }
            (void)hipFree(p->second->d_const);
            delete p->second;
            p = ctx->mp_plans.erase(p);
        }
    }
    LBX_TRY(upload_plan(plan.get(), K));
    ctx->mp_plans[key] = plan.get();
    *out = plan.release();
    return LBX_OK;
}

}  // namespace

lbx_status zz_product(lbx_ctx *ctx, int nl, int cl, const DevView &a, const DevView &b, const DevView &c, size_t m,
                      size_t k, size_t n, size_t sc, int method, hipStream_t s)
{
    const size_t sa = a.size, sb = b.size;
    unsigned lpts = 0;
    size_t pts = 1;
    while (pts < sc) {  // mul_crtla :151-154
        pts <<= 1;
        ++lpts;
    }
    unsigned la = 0, lb = 0;
    LBX_TRY(zz_logmax(ctx, a, b, nl, &la, &lb, s));
    MpPlan *plan;
    LBX_TRY(get_zz_plan(ctx, la + lb, k, sa < sb ? sa : sb, lpts, nl, cl, &plan));
    const int r = (int)plan->primes.size();
    void *ra, *rb, *rc;
    LBX_TRY(ensure(ctx, "mp_ra", (size_t)r * m * k * sa * 4, &ra));
    LBX_TRY(ensure(ctx, "mp_rb", (size_t)r * k * n * sb * 4, &rb));
    LBX_TRY(ensure(ctx, "mp_rc", (size_t)r * m * n * sc * 4, &rc));
    LBX_TRY_HIP(launch_residues<true>(a, m * k, (uint32_t *)ra, b, k * n, (uint32_t *)rb, nl, r,
                                      plan->d_const + plan->res_off, s));
    const DevView va{(uint32_t *)ra, LBX_POLFIRST, m, k, sa, 0, sa}, vb{(uint32_t *)rb, LBX_POLFIRST, k, n, sb, 0, sb};
    LBX_TRY(prime_products(ctx, plan->primes, va, m * k * sa, vb, k * n * sb, (uint32_t *)rc, m, k, n, sc, lpts, method,
                           s, nullptr));
    if (plan->crt_off)
        return from_hip(launch_crt_direct<false>(crt_words(plan->primes, cl), (const uint32_t *)rc, m * n, sc,
                                                 plan->d_const + plan->crt_off, r, cl, c, s));
    hipLaunchKernelGGL(zz_crt_kernel, dim3(grid_of(m * n * sc, 128)), dim3(128), 0, s, (const uint32_t *)rc, m * n,
                       sc, (const uint32_t *)plan->d_const, r, cl, c);
    LBX_TRY_HIP(hipGetLastError());
    return LBX_OK;
}

}  // namespace lbx

using namespace lbx;

extern "C" lbx_status lbx_polymat_mul_mp(lbx_ctx *ctx, const uint32_t *P, int nlimbs, lbx_polmat *c,
                                         const lbx_polmat *a, const lbx_polmat *b, size_t max_rowdeg, int method,
                                         void *stream)
{
    return guarded([&]() -> lbx_status {
        if (!ctx || !P || !a || !b || !c) return LBX_ERR_INVALID_ARG;
        if (nlimbs < 1 || nlimbs > kMaxLimbs) return LBX_ERR_PRIME_TOO_LARGE;
        if (method < 0 || method > 2) return LBX_ERR_INVALID_ARG;
        LBX_TRY(check_view(a));
        LBX_TRY(check_view(b));
        LBX_TRY(check_view(c));
        bool nonzero = false, big = false;
        for (int l = 0; l < nlimbs; ++l) {
            nonzero |= P[l] != 0;
            if (l > 0) big |= P[l] != 0;
        }
        if (!nonzero || (!big && P[0] < 2)) return LBX_ERR_INVALID_ARG;
        if (a->cols != b->rows || c->rows != a->rows || c->cols != b->cols) return LBX_ERR_SIZE_MISMATCH;
        if (!a->size || !b->size) return LBX_ERR_INVALID_ARG;
        const size_t m = a->rows, k = a->cols, n = b->cols;
        const size_t sc = max_rowdeg ? max_rowdeg + 1 : a->size + b->size - 1;
        if (c->size < sc) return LBX_ERR_SIZE_MISMATCH;
        size_t pts = 1;
        while (pts < sc) pts <<= 1;
        if (a->size > pts || b->size > pts) return LBX_ERR_SIZE_MISMATCH;  // the padded copies hold pts coefficients
        if (k > 0xffffffffu || a->size > 0xffffffffu || sc > 0xffffffffu) return LBX_ERR_UNSUPPORTED;

        std::lock_guard<std::mutex> lock(ctx->mu);
        DeviceGuard guard(ctx->device);
        hipStream_t s = (hipStream_t)stream;
        StreamOrder stream_order(ctx, s);
        const size_t wb = 4 * (size_t)nlimbs;
        Staged sa_, sb_, sc_;
        lbx_status st = stage_in(ctx, "stage_a", a, wb, true, &sa_, s);
        if (st == LBX_OK) st = stage_in(ctx, "stage_b", b, wb, true, &sb_, s);
        if (st == LBX_OK) st = stage_in(ctx, "stage_c", c, wb, !(c->shift == 0 && sc >= c->storage_size), &sc_, s);
        const bool host_io = sa_.owned || sb_.owned || sc_.owned;
        if (st == LBX_OK)
            st = mp_product(ctx, P, nlimbs, devview(a, sa_.dev), devview(b, sb_.dev), devview(c, sc_.dev), m, k, n,
                            method, s, nullptr, 0, sc);
        if (st == LBX_OK && sc_.owned) {
            st = device_to_host(ctx, c->data, sc_.dev, storage_words(c) * wb, s);
        }
        if (host_io) (void)hipStreamSynchronize(s);
        release(sa_);
        release(sb_);
        release(sc_);
        if (st == LBX_OK) c->size = sc;
        return st;
    });
}

extern "C" lbx_status lbx_polymat_mul_zz(lbx_ctx *ctx, lbx_polmat *c, int c_limbs, const lbx_polmat *a,
                                         const lbx_polmat *b, int ab_limbs, size_t max_rowdeg, int method,
                                         void *stream)
{
    return guarded([&]() -> lbx_status {
        if (!ctx || !a || !b || !c) return LBX_ERR_INVALID_ARG;
        if (ab_limbs < 1 || ab_limbs > kZzMaxIn || c_limbs < 1 || c_limbs > kZzMaxOut) return LBX_ERR_UNSUPPORTED;
        if (method < 0 || method > 2) return LBX_ERR_INVALID_ARG;
        LBX_TRY(check_view(a));
        LBX_TRY(check_view(b));
        LBX_TRY(check_view(c));
        if (a->cols != b->rows || c->rows != a->rows || c->cols != b->cols) return LBX_ERR_SIZE_MISMATCH;
        if (!a->size || !b->size) return LBX_ERR_INVALID_ARG;
        const size_t m = a->rows, k = a->cols, n = b->cols;
        const size_t sc = max_rowdeg ? max_rowdeg + 1 : a->size + b->size - 1;
        if (c->size < sc) return LBX_ERR_SIZE_MISMATCH;
        size_t pts = 1;
        while (pts < sc) pts <<= 1;
        if (a->size > pts || b->size > pts) return LBX_ERR_SIZE_MISMATCH;
        if (k > 0xffffffffu || a->size > 0xffffffffu || sc > 0xffffffffu) return LBX_ERR_UNSUPPORTED;

        std::lock_guard<std::mutex> lock(ctx->mu);
        DeviceGuard guard(ctx->device);
        hipStream_t s = (hipStream_t)stream;
        StreamOrder stream_order(ctx, s);
        const size_t wi = 4 * (size_t)ab_limbs, wo = 4 * (size_t)c_limbs;
        Staged sa_, sb_, sc_;
        lbx_status st = stage_in(ctx, "stage_a", a, wi, true, &sa_, s);
        if (st == LBX_OK) st = stage_in(ctx, "stage_b", b, wi, true, &sb_, s);
        if (st == LBX_OK) st = stage_in(ctx, "stage_c", c, wo, !(c->shift == 0 && sc >= c->storage_size), &sc_, s);
        const bool host_io = sa_.owned || sb_.owned || sc_.owned;
        if (st == LBX_OK)
            st = zz_product(ctx, ab_limbs, c_limbs, devview(a, sa_.dev), devview(b, sb_.dev), devview(c, sc_.dev), m, k,
                            n, sc, method, s);
        if (st == LBX_OK && sc_.owned) {
            st = device_to_host(ctx, c->data, sc_.dev, storage_words(c) * wo, s);
        }
        if (host_io) (void)hipStreamSynchronize(s);
        release(sa_);
        release(sb_);
        release(sc_);
        if (st == LBX_OK) c->size = sc;
        return st;
    });
}
