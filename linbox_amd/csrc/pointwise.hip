// Pointwise stage of the FFT product: at every evaluation point t,
// C_t = A_t . B_t (m x k . k x n) mod p, then the 1/2^L scaling of
// mul_fft (matpoly-mult-fft-wordsize-fast.inl:160-164,183-189) folded in.
//
// The reference runs one fflas fgemm per point.  Here all points are one
// launch, in one of two forms:
//
//  * plain: vector ALUs, one point per lane, a T x T register tile of 64-bit
//    accumulators per lane.  The reduction is delayed to the end of the k loop:
//    products of centred words (below 2^60) are folded every six or more steps,
//    and the sum is reduced once with two Shoup products.  Operands are read
//    straight from the polfirst NTT output: consecutive lanes read consecutive
//    points, so every load is coalesced.
//
//  * INT8 MFMA: every residue is centred (|c| < p/2 < 2^30) and split into
//    four balanced signed 8-bit digits, c = sum_s d_s 2^(8s).  Then
//    C = sum_{s,t} 2^(8(s+t)) (A_s . B_t), and the 16 digit products are
//    accumulated on v_mfma_i32_16x16x64_i8 directly into the seven
//    anti-diagonals D_d = sum_{s+t=d} A_s.B_t (int32, exact: |D_d| <= 4 k 2^14,
//    k is processed in chunks of 4096 so |D_d| < 2^28).  The epilogue forms
//    sum_d D_d (2^(8d) / 2^L mod p) in int64 (|.| < 2^62) and reduces it.
//    The digit split happens once per element in launch_to_limbs, which also
//    transposes the NTT output into per-point blocks laid out for direct
//    16-byte operand loads.
#include "lbx_internal.h"
#include "pw_math.h"

namespace lbx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

// DEEP > 0 issues the loads of that many inner steps together (small tiles with
// few waves per CU wait for every load otherwise).
template <int TI, int TJ, int DEEP = 0>
__device__ __forceinline__ void pw_plain_body(const uint32_t *__restrict__ A, const uint32_t *__restrict__ B,
                                              uint32_t *__restrict__ C, int m, int k, int n, size_t npts,
                                              uint32_t p, const PlainConst &pc, size_t t, int i0, int j0)
{
    // acc += a*b is one v_mad_u64_u32; every pc.fold products the bits above
    // 2^62 are folded back (plain_fold), which keeps acc below 2^64
    uint64_t acc[TI][TJ];
#pragma unroll
    for (int ii = 0; ii < TI; ++ii)
#pragma unroll
        for (int jj = 0; jj < TJ; ++jj) acc[ii][jj] = 0;
    for (int q0 = 0; q0 < k; q0 += (int)pc.fold) {
        const int q1 = min(k, q0 + (int)pc.fold);
        const auto step = [&](int q) {
            uint32_t a[TI], b[TJ];
#pragma unroll
            for (int ii = 0; ii < TI; ++ii)
                a[ii] = (i0 + ii < m) ? A[((size_t)(i0 + ii) * k + q) * npts + t] : 0u;
#pragma unroll
            for (int jj = 0; jj < TJ; ++jj)
                b[jj] = (j0 + jj < n) ? B[((size_t)q * n + j0 + jj) * npts + t] : 0u;
#pragma unroll
            for (int ii = 0; ii < TI; ++ii)
#pragma unroll
                for (int jj = 0; jj < TJ; ++jj) acc[ii][jj] += (uint64_t)a[ii] * b[jj];
        };
        if constexpr (DEEP > 0) {
#pragma unroll DEEP
            for (int q = q0; q < q1; ++q) step(q);
        } else {
            for (int q = q0; q < q1; ++q) step(q);
        }
#pragma unroll
        for (int ii = 0; ii < TI; ++ii)
#pragma unroll
            for (int jj = 0; jj < TJ; ++jj)
                acc[ii][jj] = plain_fold(acc[ii][jj], pc);
    }
#pragma unroll
    for (int ii = 0; ii < TI; ++ii)
#pragma unroll
        for (int jj = 0; jj < TJ; ++jj) {
            if (i0 + ii >= m || j0 + jj >= n) continue;
            C[((size_t)(i0 + ii) * n + j0 + jj) * npts + t] = plain_finish(acc[ii][jj], p, pc);
        }
}

// Primes of one launch, in the kernel arguments.
template <class Const>
struct PlainPrimes {
    uint32_t p[kMultiPrimes];
    Const pc[kMultiPrimes];
};

// One output tile at one point per lane; item = tile * npts + t, so a wave's
// lanes take consecutive points and transforms shorter than a wave share it: the
// form of products by constants and of transforms of fewer than 64 points.
template <int T>
__global__ void __launch_bounds__(256) pw_plain_kernel(const uint32_t *__restrict__ A, const uint32_t *__restrict__ B,
                                                       uint32_t *__restrict__ C, int m, int k, int n, size_t npts,
                                                       unsigned log_npts, size_t items,
                                                       PlainPrimes<PlainConst> primes)
{
    const size_t item = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (item >= items) return;
    const unsigned i = blockIdx.y;  // prime
    const int tiles_j = (n + T - 1) / T;
    const size_t t = item & (npts - 1);
    const int tile = (int)(item >> log_npts);
    pw_plain_body<T, T, T == 2 ? 8 : 2>(A + (size_t)i * m * k * npts, B + (size_t)i * k * n * npts, C + (size_t)i * m * n * npts, m, k,
                        n, npts, primes.p[i], primes.pc[i], t, (tile / tiles_j) * T, (tile % tiles_j) * T);
}

// One T x T output tile at 64 points by one wave, on centred int32 words: per
// inner step a lane loads its point's T words of A and of B (256 contiguous
// bytes per wave and word) and adds T^2 products (v_mad_i64_i32), folding every
// pc.every-th step.
//
// Bound by the loads' latency unless enough of them are in flight: a wave of
// 8x8 tiles has 2 waves a SIMD beside it at most.  The words of the next D
// steps are therefore loaded ahead into registers, and the addresses cost no
// vector instruction or register: tile and inner index are uniform across the
// wave, so every load takes a scalar base and the lane's one 32-bit offset.  Rows
// past the edge read the last row again (their products are not stored), and
// steps past the end the last step.  Measured against unsigned words folded
// every two or three steps near 2^31 and no loads ahead: 14 primes of 32^3 at
// 2^11 points 180 -> 120 us, 5 of 24^3 at 2^11 38 -> 24 us; with the loads ahead it
// is bound by its vector instructions, 64 multiply-adds a step of some 84.
template <int T, int D>
__device__ __forceinline__ void pw_accumulate(const uint32_t *__restrict__ A, const uint32_t *__restrict__ B, int m,
                                              int k, int k0, int k1, int n, size_t npts, const PlainSConst &pc,
                                              uint32_t t, int i0, int j0, int64_t (&acc)[T][T])
{
    // uniform row and column bases of the next step to load
    const char *pa[T], *pb[T];
#pragma unroll
    for (int ii = 0; ii < T; ++ii) pa[ii] = (const char *)(A + ((size_t)min(i0 + ii, m - 1) * k + k0) * npts);
#pragma unroll
    for (int jj = 0; jj < T; ++jj) pb[jj] = (const char *)(B + ((size_t)k0 * n + min(j0 + jj, n - 1)) * npts);
    const uint32_t off = t * 4;
    const size_t step_a = npts * 4, step_b = (size_t)n * npts * 4;
    int32_t a[D][T], b[D][T];
    int q_load = k0;
    const auto load = [&](int d) {
#pragma unroll
        for (int ii = 0; ii < T; ++ii) a[d][ii] = *(const int32_t *)(pa[ii] + off);
#pragma unroll
        for (int jj = 0; jj < T; ++jj) b[d][jj] = *(const int32_t *)(pb[jj] + off);
        ++q_load;
        const size_t sa = q_load < k1 ? step_a : 0, sb = q_load < k1 ? step_b : 0;
#pragma unroll
        for (int ii = 0; ii < T; ++ii) pa[ii] += sa;
#pragma unroll
        for (int jj = 0; jj < T; ++jj) pb[jj] += sb;
    };
#pragma unroll
    for (int ii = 0; ii < T; ++ii)
#pragma unroll
        for (int jj = 0; jj < T; ++jj) acc[ii][jj] = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) load(d);
    int since = 0;  // products since the last fold
    for (int q0 = k0; q0 < k1; q0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            if (q0 + d < k1) {
#pragma unroll
                for (int ii = 0; ii < T; ++ii)
#pragma unroll
                    for (int jj = 0; jj < T; ++jj) acc[ii][jj] += (int64_t)a[d][ii] * b[d][jj];
                if (++since == (int)pc.every) {
                    since = 0;
#pragma unroll
                    for (int ii = 0; ii < T; ++ii)
#pragma unroll
                        for (int jj = 0; jj < T; ++jj) acc[ii][jj] = plain_s_fold(acc[ii][jj], pc);
                }
                load(d);
            }
        }
    }
}

template <int T, int D>
__device__ __forceinline__ void pw_tile(const uint32_t *__restrict__ A, const uint32_t *__restrict__ B,
                                        uint32_t *__restrict__ C, int m, int k, int n, size_t npts, uint32_t p,
                                        const PlainSConst &pc, uint32_t t, int i0, int j0)
{
    int64_t acc[T][T];
    pw_accumulate<T, D>(A, B, m, k, 0, k, n, npts, pc, t, i0, j0, acc);
#pragma unroll
    for (int ii = 0; ii < T; ++ii)
#pragma unroll
        for (int jj = 0; jj < T; ++jj) {
            if (i0 + ii >= m || j0 + jj >= n) continue;
            C[((size_t)(i0 + ii) * n + j0 + jj) * npts + t] = plain_s_finish(acc[ii][jj], p, pc);
        }
}

// Steps loaded ahead: some 32 words a lane whatever the tile.
template <int T>
constexpr int tile_ahead() { return T == 8 ? 2 : (T == 4 ? 3 : 6); }
// Waves per SIMD: the 128 accumulator registers and 32 ahead of an 8x8 tile leave three.
template <int T>
constexpr int tile_waves() { return T == 8 ? 3 : (T == 4 ? 5 : 8); }

// blockIdx.y is the prime.  The waves of a group take a wm x wn patch of tiles
// at the same 64 points, so its A rows and B columns come from L1 after their
// first use; groups on one XCD (blockIdx.x mod 8) share the points, so the
// operands of 64 points are read into one L2 only.
template <int T>
__global__ void __launch_bounds__(256, tile_waves<T>()) pw_tiled_kernel(const uint32_t *__restrict__ A, const uint32_t *__restrict__ B,
                                                       uint32_t *__restrict__ C, int m, int k, int n, size_t npts,
                                                       int wn, int tiles_m, int tiles_n, unsigned patches,
                                                       unsigned patches_n, PlainPrimes<PlainSConst> primes)
{
    const unsigned i = blockIdx.y, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned wm = (blockDim.x >> 6) / wn, runs = (unsigned)(npts >> 6), nb = runs < 8 ? runs : 8;
    const unsigned low = blockIdx.x % nb, g = blockIdx.x / nb, patch = g % patches, run = g / patches * nb + low;
    const int ti = (int)(patch / patches_n * wm + wave / wn), tj = (int)(patch % patches_n * wn + wave % wn);
    if (ti >= tiles_m || tj >= tiles_n) return;
    pw_tile<T, tile_ahead<T>()>(A + (size_t)i * m * k * npts, B + (size_t)i * k * n * npts,
                                C + (size_t)i * m * n * npts, m, k, n, npts, primes.p[i], primes.pc[i],
                                run * 64 + (threadIdx.x & 63), ti * T, tj * T);
}

// The same tile with its inner dimension split over the kSplitK waves of a
// group, for products too small to fill the chip with tiles: each wave sums its
// part of the steps (a chain kSplitK times as short), the folded sums (below 2^60 +
// 2^34 each, so four fit) meet in LDS and every wave finishes T^2 / kSplitK of the
// outputs.
constexpr int kSplitK = 4;
template <int T>
__global__ void __launch_bounds__(64 * kSplitK) pw_splitk_kernel(const uint32_t *__restrict__ A,
                                                                 const uint32_t *__restrict__ B,
                                                                 uint32_t *__restrict__ C, int m, int k, int n,
                                                                 size_t npts, int tiles_n, unsigned tiles,
                                                                 PlainPrimes<PlainSConst> primes)
{
    __shared__ int64_t part[kSplitK][T * T][64];
    const unsigned i = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const unsigned runs = (unsigned)(npts >> 6), nb = runs < 8 ? runs : 8;
    const unsigned low = blockIdx.x % nb, g = blockIdx.x / nb, tile = g % tiles, run = g / tiles * nb + low;
    const int i0 = (int)(tile / tiles_n) * T, j0 = (int)(tile % tiles_n) * T;
    const int per = (k + kSplitK - 1) / kSplitK, k0 = min(wave * per, k), k1 = min(k0 + per, k);
    const uint32_t t = run * 64 + lane;
    const PlainSConst &pc = primes.pc[i];
    int64_t acc[T][T];
    // a wave without steps loads the last one (in bounds) and sums nothing
    pw_accumulate<T, tile_ahead<T>()>(A + (size_t)i * m * k * npts, B + (size_t)i * k * n * npts, m, k,
                                      k0 < k1 ? k0 : k - 1, k0 < k1 ? k1 : k - 1, n, npts, pc, t, i0, j0, acc);
#pragma unroll
    for (int ii = 0; ii < T; ++ii)
#pragma unroll
        for (int jj = 0; jj < T; ++jj) part[wave][ii * T + jj][lane] = plain_s_fold(acc[ii][jj], pc);
    __syncthreads();
    uint32_t *Ci = C + (size_t)i * m * n * npts;
#pragma unroll
    for (int u = 0; u < T * T / kSplitK; ++u) {
        const int e = wave * (T * T / kSplitK) + u, ii = e / T, jj = e % T;
        int64_t sum = 0;
#pragma unroll
        for (int w = 0; w < kSplitK; ++w) sum += part[w][e][lane];
        if (i0 + ii < m && j0 + jj < n)
            Ci[((size_t)(i0 + ii) * n + j0 + jj) * npts + t] = plain_s_finish(sum, primes.p[i], pc);
    }
}

// Persistent work-queue form over the items of a batch: each workgroup takes 64
// points of four neighbouring output tiles of one job at a time, a tile a wave,
// whose A rows (mostly shared) and B columns then come from L1 after their first
// use, or 256 points of one tile.  With 256 points of one tile per group throughout
// the batch of 1024 products spent 3.44 ms here, 2.59 ms now; four tiles a group
// throughout leaves waves idle on jobs of fewer (154 products of up to 16 rows 274 ->
// 306 us).
__global__ void __launch_bounds__(256, tile_waves<8>()) batch_pointwise_kernel(const BatchJob *__restrict__ jobs,
                                                                               const PwItem *__restrict__ items,
                                                                               uint32_t nitems, uint32_t *counter)
{
    __shared__ uint32_t item_sh;
    for (;;) {
        if (threadIdx.x == 0) item_sh = atomicAdd(counter, 1u);
        __syncthreads();
        const uint32_t it = __builtin_amdgcn_readfirstlane(item_sh);  // uniform: scalar loads of the item
        __syncthreads();
        if (it >= nitems) return;
        const PwItem w = items[it];
        const BatchJob &J = jobs[w.job];
        const size_t npts = (size_t)1 << J.L;
        const uint32_t t = w.pt0 + (w.one_tile ? threadIdx.x : threadIdx.x & 63);
        const int tile = (int)w.tile0 + (w.one_tile ? 0 : (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)),
                  side = 2 << J.tile;
        const int tiles_n = ((int)J.n + side - 1) / side, i0 = tile / tiles_n * side, j0 = tile % tiles_n * side;
        const uint32_t *A = global_ptr(J.ahat), *B = global_ptr(J.bhat);
        uint32_t *Cp = global_ptr(J.chat);
        if (t < npts && i0 < (int)J.m) {
            if (J.tile == 0)
                pw_tile<2, tile_ahead<2>()>(A, B, Cp, J.m, J.k, J.n, npts, J.p, J.pc, t, i0, j0);
            else if (J.tile == 1)
                pw_tile<4, tile_ahead<4>()>(A, B, Cp, J.m, J.k, J.n, npts, J.p, J.pc, t, i0, j0);
            else
                pw_tile<8, tile_ahead<8>()>(A, B, Cp, J.m, J.k, J.n, npts, J.p, J.pc, t, i0, j0);
        }
    }
}

__global__ void zero_counters_kernel(uint32_t *c, int n)
{
    if ((int)threadIdx.x < n) c[threadIdx.x] = 0;
}

// ---- limb blocks -------------------------------------------------------
// Per point, an operand with `rows` rows and inner dimension kdim is stored as
// [rpad][kpad/64][4 planes][64 bytes]: the 64 inner-dimension digits of plane s
// of one row for one 64-wide k step are contiguous, so a lane's MFMA operand
// (16 consecutive digits) is one 16-byte load.
__host__ __device__ inline size_t rpad_of(size_t rows) { return (rows + 31) & ~(size_t)31; }
__host__ __device__ inline size_t kpad_of(size_t kdim) { return (kdim + 63) & ~(size_t)63; }
__device__ __forceinline__ size_t limb_block_bytes_dev(size_t rows, size_t kdim) { return rpad_of(rows) * kpad_of(kdim) * 4; }

// One 64-point x 64-entry tile: points t0.., inner chunk c, row r of the
// padded range; reads 64 consecutive points of 64 entries (coalesced) and
// writes, for each point, that row's 256-byte run of the limb block.
__device__ __forceinline__ void limbs_tile(const uint32_t *__restrict__ X, uint8_t *__restrict__ Y, int rows,
                                           int kdim, int row_major, size_t npts, uint32_t p, size_t block_bytes,
                                           int kchunks, size_t t0, int c, int r, int tid, uint32_t (&tile)[64][65])
{
    const int q0 = c * 64;
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
        const int ql = it * 4 + tid / 64, tl = tid % 64;
        const int q = q0 + ql;
        const size_t t = t0 + tl;
        uint32_t v = 0;
        if (r < rows && q < kdim && t < npts) {
            const size_t e = row_major ? (size_t)r * kdim + q : (size_t)q * rows + r;
            v = to_limbs(X[e * npts + t], p);
        }
        tile[ql][tl] = v;
    }
    __syncthreads();
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
        const int tl = it * 4 + tid / 64, w = tid % 64;
        const size_t t = t0 + tl;
        if (t >= npts) continue;
        const int s = w >> 4, qb = (w & 15) * 4;
        const uint32_t sh = 8 * s;
        const uint32_t word = ((tile[qb][tl] >> sh) & 0xffu) | (((tile[qb + 1][tl] >> sh) & 0xffu) << 8) |
                              (((tile[qb + 2][tl] >> sh) & 0xffu) << 16) | (((tile[qb + 3][tl] >> sh) & 0xffu) << 24);
        uint8_t *dst = Y + t * block_bytes + ((size_t)r * kchunks + c) * 256 + s * 64 + (w & 15) * 4;
        *reinterpret_cast<uint32_t *>(dst) = word;
    }
}

__global__ void __launch_bounds__(256) to_limbs_kernel(const uint32_t *__restrict__ X, uint8_t *__restrict__ Y,
                                                       int rows, int kdim, int row_major, size_t npts, uint32_t p,
                                                       size_t block_bytes, int kchunks)
{
    __shared__ uint32_t tile[64][65];
    limbs_tile(X, Y, rows, kdim, row_major, npts, p, block_bytes, kchunks, (size_t)blockIdx.x * 64, blockIdx.y,
               blockIdx.z, threadIdx.x, tile);
}

__device__ __forceinline__ uint32_t mfma_combine(const v4i (&acc)[7], int r, uint32_t p, const MfmaConst &mc)
{
    int32_t D[7];
#pragma unroll
    for (int d = 0; d < 7; ++d) D[d] = acc[d][r];
    return combine_diagonals(D, p, mc);
}

constexpr int kMaxKbPerChunk = 64;  // 64 steps of 64 = 4096 inner products per exact int32 chunk

// One wave: the 32x32 output tile (i0, j0) of one point from its limb
// blocks A and B (read from HBM/L2), as 2x2 16x16 MFMA tiles for each of the
// 16 digit pairs, k in exact int32 chunks of 4096.
__device__ __forceinline__ void mfma_tile_global(const uint8_t *__restrict__ A, const uint8_t *__restrict__ B,
                                                 uint32_t *__restrict__ Ct, int m, int n, int kchunks, int i0,
                                                 int j0, uint32_t p, const MfmaConst &mc, int l16, int lg)
{
    const size_t row_bytes = (size_t)kchunks * 256;
    {
        uint32_t res[2][2][4];
#pragma unroll
        for (int ai = 0; ai < 2; ++ai)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                for (int r = 0; r < 4; ++r) res[ai][bj][r] = 0;
        for (int kc0 = 0; kc0 < kchunks; kc0 += kMaxKbPerChunk) {
            const int kc1 = min(kchunks, kc0 + kMaxKbPerChunk);
            v4i acc[2][2][7];
#pragma unroll
            for (int ai = 0; ai < 2; ++ai)
#pragma unroll
                for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                    for (int d = 0; d < 7; ++d) acc[ai][bj][d] = v4i{0, 0, 0, 0};
            for (int kb = kc0; kb < kc1; ++kb) {
                v4i a[2][4], b[2][4];
#pragma unroll
                for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        a[sub][s] = *reinterpret_cast<const v4i *>(A + (size_t)(i0 + sub * 16 + l16) * row_bytes +
                                                                   (size_t)kb * 256 + s * 64 + lg * 16);
                        b[sub][s] = *reinterpret_cast<const v4i *>(B + (size_t)(j0 + sub * 16 + l16) * row_bytes +
                                                                   (size_t)kb * 256 + s * 64 + lg * 16);
                    }
#pragma unroll
                for (int ai = 0; ai < 2; ++ai)
#pragma unroll
                    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                        for (int s = 0; s < 4; ++s)
#pragma unroll
                            for (int u = 0; u < 4; ++u)
                                acc[ai][bj][s + u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                    a[ai][s], b[bj][u], acc[ai][bj][s + u], 0, 0, 0);
            }
#pragma unroll
            for (int ai = 0; ai < 2; ++ai)
#pragma unroll
                for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        res[ai][bj][r] = add_mod(res[ai][bj][r], mfma_combine(acc[ai][bj], r, p, mc), p);
        }
#pragma unroll
        for (int ai = 0; ai < 2; ++ai)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = i0 + ai * 16 + lg * 4 + r, j = j0 + bj * 16 + l16;
                    if (i < m && j < n) Ct[(size_t)i * n + j] = res[ai][bj][r];
                }
    }
}

// One workgroup per point; each wave computes 32x32 output tiles.
__global__ void __launch_bounds__(256) pw_mfma_kernel(const uint8_t *__restrict__ Al, const uint8_t *__restrict__ Bl,
                                                      uint32_t *__restrict__ Cmat, int m, int n, int kchunks,
                                                      int mpad, int npad, size_t a_bytes, size_t b_bytes, uint32_t p,
                                                      MfmaConst mc)
{
    const size_t t = blockIdx.x;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tiles_n = npad / 32, ntiles = (mpad / 32) * tiles_n;
    for (int tile = wave; tile < ntiles; tile += 4)
        mfma_tile_global(Al + t * a_bytes, Bl + t * b_bytes, Cmat + t * (size_t)m * n, m, n, kchunks,
                         (tile / tiles_n) * 32, (tile % tiles_n) * 32, p, mc, lane & 15, lane >> 4);
}

// LDS-staged form, used for the other shapes whose A limb block fits in 64 KiB
// (m*k <= 16384 after padding): persistent workgroups, two per CU, each takes a point, copies
// its A block to LDS once, then streams B through LDS 32 columns at a time; every
// wave computes the 32x32 tiles of one row band.  16-byte chunks are stored
// XOR-swizzled within each row (chunk c of row r at c ^ (r & 15)) so the 16 rows
// a ds_read_b128 touches fall in distinct banks.
constexpr int kLdsAMax = 65536;

__device__ __forceinline__ void mfma_tile_lds(const uint4 *__restrict__ lA, const uint4 *__restrict__ lB, int cpr,
                                              int kchunks, int arow0, int l16, int lg, v4i (&acc)[2][2][7])
{
#pragma unroll
    for (int ai = 0; ai < 2; ++ai)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
            for (int d = 0; d < 7; ++d) acc[ai][bj][d] = v4i{0, 0, 0, 0};
    for (int kb = 0; kb < kchunks; ++kb) {
        v4i a[2][4], b[2][4];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int c = (kb * 16 + s * 4 + lg) ^ l16;
                const uint4 va = lA[(arow0 + sub * 16 + l16) * cpr + c];
                const uint4 vb = lB[(sub * 16 + l16) * cpr + c];
                a[sub][s] = v4i{(int)va.x, (int)va.y, (int)va.z, (int)va.w};
                b[sub][s] = v4i{(int)vb.x, (int)vb.y, (int)vb.z, (int)vb.w};
            }
#pragma unroll
        for (int ai = 0; ai < 2; ++ai)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        acc[ai][bj][s + u] =
                            __builtin_amdgcn_mfma_i32_16x16x64_i8(a[ai][s], b[bj][u], acc[ai][bj][s + u], 0, 0, 0);
    }
}

typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void global_cvoid;

// Global -> LDS copy of `chunks` 16-byte chunks (a multiple of 64) with the
// row swizzle, using global_load_lds_dwordx4: each wave instruction fills 64
// consecutive LDS chunks (1 KiB at M0 + 16*lane) with no register staging, so
// every load of the copy is in flight at once.  Lane i of a wave's j-th
// instruction fills LDS chunk P = 64*(4j + wave) + i, i.e. row r = P / cpr,
// swizzled column P % cpr, which holds global chunk r*cpr + ((P % cpr) ^ (r & 15)).
// NW waves share the copy (P = 64*(NW*j + wave) + i).
template <int NW = 4>
__device__ __forceinline__ void copy_lds(const uint4 *__restrict__ g, uint4 *l, int chunks, int cpr, int wave,
                                         int lane)
{
    for (int base = 64 * wave; base < chunks; base += 64 * NW) {
        const int P = base + lane;
        const int r = P / cpr, c = P - r * cpr;
        __builtin_amdgcn_global_load_lds((global_cvoid *)(g + r * cpr + (c ^ (r & 15))), (lds_void *)(l + base), 16,
                                         0, 0);
    }
}

__global__ void __launch_bounds__(256, 2) pw_mfma_lds_kernel(const uint8_t *__restrict__ Al,
                                                             const uint8_t *__restrict__ Bl, uint32_t *__restrict__ Cmat,
                                                             int m, int n, int kchunks, int mpad, int npad,
                                                             size_t npts, uint32_t p, MfmaConst mc)
{
    extern __shared__ uint4 smem4[];
    const int cpr = kchunks * 16;  // 16-byte chunks per row
    uint4 *lA = smem4;
    uint4 *lB = smem4 + (size_t)mpad * cpr;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, lg = lane >> 4;
    const int a_chunks = mpad * cpr, b_chunks = 32 * cpr;
    const int nrt = mpad / 32, ncb = npad / 32;
    for (size_t t = blockIdx.x; t < npts; t += gridDim.x) {
        const uint4 *gA = reinterpret_cast<const uint4 *>(Al) + t * (size_t)a_chunks;
        const uint4 *gB = reinterpret_cast<const uint4 *>(Bl) + t * (size_t)npad * cpr;
        __syncthreads();  // the previous point is done with lA and lB
        copy_lds(gA, lA, a_chunks, cpr, wave, lane);
        uint32_t *Ct = Cmat + t * (size_t)m * n;
        for (int cb = 0; cb < ncb; ++cb) {
            if (cb) __syncthreads();
            const uint4 *gBb = gB + (size_t)cb * b_chunks;
            copy_lds(gBb, lB, b_chunks, cpr, wave, lane);
            __builtin_amdgcn_s_waitcnt(0);  // this thread's LDS-direct loads have landed
            __syncthreads();
            for (int rt = wave; rt < nrt; rt += 4) {
                v4i acc[2][2][7];
                mfma_tile_lds(lA, lB, cpr, kchunks, rt * 32, l16, lg, acc);
#pragma unroll
                for (int ai = 0; ai < 2; ++ai)
#pragma unroll
                    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int i = rt * 32 + ai * 16 + lg * 4 + r, j = cb * 32 + bj * 16 + l16;
                            if (i < m && j < n) Ct[(size_t)i * n + j] = mfma_combine(acc[ai][bj], r, p, mc);
                        }
            }
        }
    }
}

// A in registers, B in LDS: for mpad in {32, 64, 96, 128}, k <= 128 and a B block
// of at most 64 KiB.  Each wave multiplies one 32-row band of A, which it
// loads straight into registers (64 VGPRs at k = 128); only B, which every
// wave needs, goes through LDS, whole, with one LDS-direct copy.  A point
// therefore costs one wait and one barrier, with A and B (128 KiB for 128x128 operands) in
// flight together; two groups per CU overlap one's loads with the other's
// multiplies.  With nrt = mpad/32 < 4 bands, wave w takes band w % nrt and
// every (4/nrt)-th column block from w / nrt.
// Three bands (mpad = 96) take groups of three waves, one band each: 96x48x80 at
// 2^12 points 88 us, against 107 us in the LDS form above.
template <int KC, int NW>
__global__ void __launch_bounds__(64 * NW, 2) pw_mfma_rega_kernel(const uint8_t *__restrict__ Al,
                                                              const uint8_t *__restrict__ Bl,
                                                              uint32_t *__restrict__ Cmat, int m, int n, int mpad,
                                                              int npad, size_t npts, uint32_t p, MfmaConst mc)
{
    extern __shared__ uint4 smem4[];
    constexpr int cpr = KC * 16;  // 16-byte chunks per row
    uint4 *lB = smem4;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, lg = lane >> 4;
    const int a_chunks = mpad * cpr, b_chunks = npad * cpr;
    const int nrt = mpad / 32, ncb = npad / 32;
    const int band = wave % nrt, cb0 = wave / nrt, cbs = NW / nrt;
    for (size_t t = blockIdx.x; t < npts; t += gridDim.x) {
        const uint4 *gA = reinterpret_cast<const uint4 *>(Al) + t * (size_t)a_chunks;
        const uint4 *gB = reinterpret_cast<const uint4 *>(Bl) + t * (size_t)b_chunks;
        __syncthreads();  // the previous point is done with lB
        copy_lds<NW>(gB, lB, b_chunks, cpr, wave, lane);
        v4i a[2][KC][4];
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
            for (int kb = 0; kb < KC; ++kb)
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const uint4 v = gA[(band * 32 + sub * 16 + l16) * cpr + kb * 16 + s * 4 + lg];
                    a[sub][kb][s] = v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
                }
        __builtin_amdgcn_s_waitcnt(0);  // A in registers, this thread's B chunks in LDS
        __syncthreads();
        uint32_t *Ct = Cmat + t * (size_t)m * n;
        for (int cb = cb0; cb < ncb; cb += cbs) {
            v4i acc[2][2][7];
#pragma unroll
            for (int ai = 0; ai < 2; ++ai)
#pragma unroll
                for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                    for (int d = 0; d < 7; ++d) acc[ai][bj][d] = v4i{0, 0, 0, 0};
#pragma unroll
            for (int kb = 0; kb < KC; ++kb) {
                v4i b[2][4];
#pragma unroll
                for (int sub = 0; sub < 2; ++sub)
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const int c = (kb * 16 + s * 4 + lg) ^ l16;
                        const uint4 vb = lB[(cb * 32 + sub * 16 + l16) * cpr + c];
                        b[sub][s] = v4i{(int)vb.x, (int)vb.y, (int)vb.z, (int)vb.w};
                    }
#pragma unroll
                for (int ai = 0; ai < 2; ++ai)
#pragma unroll
                    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                        for (int s = 0; s < 4; ++s)
#pragma unroll
                            for (int u = 0; u < 4; ++u)
                                acc[ai][bj][s + u] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[ai][kb][s], b[bj][u],
                                                                                          acc[ai][bj][s + u], 0, 0, 0);
            }
#pragma unroll
            for (int ai = 0; ai < 2; ++ai)
#pragma unroll
                for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int i = band * 32 + ai * 16 + lg * 4 + r, j = cb * 32 + bj * 16 + l16;
                        if (i < m && j < n) Ct[(size_t)i * n + j] = mfma_combine(acc[ai][bj], r, p, mc);
                    }
        }
    }
}

// Entries e0.. x points t0.. of a point-major [t][e] array into polfirst [e][t].
__device__ __forceinline__ void point_to_entry_tile(const uint32_t *__restrict__ X, uint32_t *__restrict__ Y,
                                                    size_t entries, size_t npts, size_t e0, size_t t0, int tid,
                                                    uint32_t (&tile)[64][65])
{
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
        const int tl = it * 4 + tid / 64, el = tid % 64;
        const size_t t = t0 + tl, e = e0 + el;
        tile[tl][el] = (t < npts && e < entries) ? X[t * entries + e] : 0u;
    }
    __syncthreads();
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
        const int el = it * 4 + tid / 64, tl = tid % 64;
        const size_t t = t0 + tl, e = e0 + el;
        if (t < npts && e < entries) Y[e * npts + t] = tile[tl][el];
    }
}

__global__ void __launch_bounds__(256) point_to_entry_kernel(const uint32_t *__restrict__ X, uint32_t *__restrict__ Y,
                                                             size_t entries, size_t npts)
{
    __shared__ uint32_t tile[64][65];
    point_to_entry_tile(X, Y, entries, npts, (size_t)blockIdx.y * 64, (size_t)blockIdx.x * 64, threadIdx.x, tile);
}

// ---- INT8 stage of a batch: persistent work-queue kernels -------------------
// Each 256-thread group takes an item index from the counter, makes it
// wave-uniform (scalar loads of the job descriptor) and processes it.
__device__ __forceinline__ uint32_t next_item(uint32_t *counter, uint32_t &slot)
{
    if (threadIdx.x == 0) slot = atomicAdd(counter, 1u);
    __syncthreads();
    const uint32_t it = __builtin_amdgcn_readfirstlane(slot);
    __syncthreads();  // everyone has the index (and is done with the previous item's LDS)
    return it;
}

__global__ void __launch_bounds__(256) batch_limbs_kernel(const BatchJob *__restrict__ jobs,
                                                          const LimbItem *__restrict__ items, uint32_t nitems,
                                                          uint32_t *counter)
{
    __shared__ uint32_t tile[64][65];
    __shared__ uint32_t slot;
    for (;;) {
        const uint32_t it = next_item(counter, slot);
        if (it >= nitems) return;
        const LimbItem w = items[it];
        const BatchJob &J = jobs[w.job];
        const bool isa = w.op == 0;
        const int rows = isa ? J.m : J.n, kdim = J.k;
        const int kchunks = (kdim + 63) / 64;
        const size_t block_bytes = limb_block_bytes_dev(rows, kdim);
        limbs_tile(global_ptr(isa ? J.ahat : J.bhat), global_ptr(isa ? J.alimb : J.blimb), rows, kdim, isa ? 1 : 0,
                   (size_t)1 << J.L, J.p,
                   block_bytes, kchunks, w.t0, (int)(w.rc % kchunks), (int)(w.rc / kchunks), threadIdx.x, tile);
    }
}

__global__ void __launch_bounds__(256) batch_mfma_kernel(const BatchJob *__restrict__ jobs,
                                                         const MfmaItem *__restrict__ items, uint32_t nitems,
                                                         uint32_t *counter)
{
    __shared__ uint32_t slot;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (;;) {
        const uint32_t it = next_item(counter, slot);
        if (it >= nitems) return;
        const MfmaItem w = items[it];
        const BatchJob &J = jobs[w.job];
        const int mpad = (J.m + 31) & ~31, npad = (J.n + 31) & ~31, kchunks = (J.k + 63) / 64;
        const int tiles_n = npad / 32, tiles = (mpad / 32) * tiles_n;
        const size_t a_bytes = limb_block_bytes_dev(J.m, J.k), b_bytes = limb_block_bytes_dev(J.n, J.k);
        const uint8_t *al = global_ptr(J.alimb), *bl = global_ptr(J.blimb);
        uint32_t *cm = global_ptr(J.cmat);
        for (uint32_t u = wave; u < w.count * (uint32_t)tiles; u += 4) {
            const size_t t = w.t0 + u / tiles;
            const int tile = (int)(u % tiles);
            mfma_tile_global(al + t * a_bytes, bl + t * b_bytes, cm + t * (size_t)J.m * J.n, J.m, J.n,
                             kchunks, (tile / tiles_n) * 32, (tile % tiles_n) * 32, J.p, J.mc, lane & 15, lane >> 4);
        }
    }
}

__global__ void __launch_bounds__(256) batch_point_to_entry_kernel(const BatchJob *__restrict__ jobs,
                                                                   const TrItem *__restrict__ items, uint32_t nitems,
                                                                   uint32_t *counter)
{
    __shared__ uint32_t tile[64][65];
    __shared__ uint32_t slot;
    for (;;) {
        const uint32_t it = next_item(counter, slot);
        if (it >= nitems) return;
        const TrItem w = items[it];
        const BatchJob &J = jobs[w.job];
        point_to_entry_tile(global_ptr(J.cmat), global_ptr(J.chat), (size_t)J.m * J.n, (size_t)1 << J.L, w.e0, w.t0,
                            threadIdx.x, tile);
    }
}

}  // namespace


hipError_t launch_batch_pointwise(const BatchJob *jobs, const PwItem *items, uint32_t nitems, uint32_t *counter,
                                  unsigned grid, hipStream_t s)
{
    hipLaunchKernelGGL(batch_pointwise_kernel, dim3(grid), dim3(256), 0, s, jobs, items, nitems, counter);
    return hipGetLastError();
}

hipError_t launch_batch_limbs(const BatchJob *jobs, const LimbItem *items, uint32_t nitems, uint32_t *counter,
                              unsigned grid, hipStream_t s)
{
    hipLaunchKernelGGL(batch_limbs_kernel, dim3(grid), dim3(256), 0, s, jobs, items, nitems, counter);
    return hipGetLastError();
}

hipError_t launch_batch_mfma(const BatchJob *jobs, const MfmaItem *items, uint32_t nitems, uint32_t *counter,
                             unsigned grid, hipStream_t s)
{
    hipLaunchKernelGGL(batch_mfma_kernel, dim3(grid), dim3(256), 0, s, jobs, items, nitems, counter);
    return hipGetLastError();
}

hipError_t launch_batch_point_to_entry(const BatchJob *jobs, const TrItem *items, uint32_t nitems,
                                       uint32_t *counter, unsigned grid, hipStream_t s)
{
    hipLaunchKernelGGL(batch_point_to_entry_kernel, dim3(grid), dim3(256), 0, s, jobs, items, nitems, counter);
    return hipGetLastError();
}

hipError_t launch_zero_counters(uint32_t *counters, int n, hipStream_t s)
{
    hipLaunchKernelGGL(zero_counters_kernel, dim3(1), dim3(64), 0, s, counters, n);
    return hipGetLastError();
}

template <class Const, class F>
static PlainPrimes<Const> plain_primes(unsigned r, const uint32_t *p, const uint32_t *scale, F make)
{
    PlainPrimes<Const> primes{};
    for (unsigned i = 0; i < r; ++i) {
        primes.p[i] = p[i];
        primes.pc[i] = make(p[i], scale[i]);
    }
    return primes;
}

hipError_t launch_pointwise_plain(const uint32_t *A, const uint32_t *B, uint32_t *C, size_t m, size_t k, size_t n,
                                  size_t npts, unsigned r, const uint32_t *p, const uint32_t *scale, hipStream_t s)
{
    if (r == 0 || r > (unsigned)kMultiPrimes || (npts & (npts - 1))) return hipErrorInvalidValue;
    const auto items = [&](size_t T) { return ((m + T - 1) / T) * ((n + T - 1) / T) * npts; };
    // 2x2 tiles where 4x4 ones would leave CUs with fewer than eight waves
    const bool wide = items(4) * r >= 512 * (size_t)device_cus();
    const size_t blocks = (items(wide ? 4 : 2) + 255) / 256;
    if (items(2) / npts > 0x7fffffff || blocks > 0x7fffffff) return hipErrorInvalidValue;
    const unsigned lg = (unsigned)__builtin_ctzll(npts);
    const PlainPrimes<PlainConst> primes = plain_primes<PlainConst>(r, p, scale, plain_const);
    if (wide)
        hipLaunchKernelGGL(pw_plain_kernel<4>, dim3((unsigned)blocks, r), dim3(256), 0, s, A, B, C, (int)m, (int)k,
                           (int)n, npts, lg, items(4), primes);
    else
        hipLaunchKernelGGL(pw_plain_kernel<2>, dim3((unsigned)blocks, r), dim3(256), 0, s, A, B, C, (int)m, (int)k,
                           (int)n, npts, lg, items(2), primes);
    return hipGetLastError();
}

// Whole waves of points, and the lane's byte offset in 32 bits.
bool pointwise_tiled(size_t npts) { return npts >= 64 && npts <= ((size_t)1 << 29); }

template <int T>
static hipError_t splitk_launch(const uint32_t *A, const uint32_t *B, uint32_t *C, size_t m, size_t k, size_t n,
                                size_t npts, unsigned r, const uint32_t *p, const uint32_t *scale, hipStream_t s)
{
    const size_t tn = (n + T - 1) / T, tiles = (m + T - 1) / T * tn, blocks = tiles * (npts / 64);
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(pw_splitk_kernel<T>, dim3((unsigned)blocks, r), dim3(64 * kSplitK), 0, s, A, B, C, (int)m,
                       (int)k, (int)n, npts, (int)tn, (unsigned)tiles,
                       plain_primes<PlainSConst>(r, p, scale, plain_s_const));
    return hipGetLastError();
}

template <int T>
static hipError_t tiled_launch(const uint32_t *A, const uint32_t *B, uint32_t *C, size_t m, size_t k, size_t n,
                               size_t npts, unsigned r, const uint32_t *p, const uint32_t *scale, hipStream_t s)
{
    const size_t tm = (m + T - 1) / T, tn = (n + T - 1) / T;
    // groups of one wave where there are few, to spread them over the CUs
    const bool few = tm * tn * (npts / 64) * r < 8 * (size_t)device_cus();
    const size_t waves = few ? 1 : 4, wn = few ? 1 : (tm == 1 ? 4 : (tn == 1 ? 1 : 2)), wm = waves / wn;
    const size_t pn = (tn + wn - 1) / wn, patches = (tm + wm - 1) / wm * pn, blocks = patches * (npts / 64);
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(pw_tiled_kernel<T>, dim3((unsigned)blocks, r), dim3((unsigned)(64 * waves)), 0, s, A, B, C,
                       (int)m, (int)k, (int)n, npts, (int)wn, (int)tm, (int)tn, (unsigned)patches, (unsigned)pn,
                       plain_primes<PlainSConst>(r, p, scale, plain_s_const));
    return hipGetLastError();
}

hipError_t launch_pointwise_tiled(const uint32_t *A, const uint32_t *B, uint32_t *C, size_t m, size_t k, size_t n,
                                  size_t npts, unsigned r, const uint32_t *p, const uint32_t *scale, hipStream_t s)
{
    if (r == 0 || r > (unsigned)kMultiPrimes || (npts & (npts - 1)) || !pointwise_tiled(npts))
        return hipErrorInvalidValue;
    // the widest tile that still gives every CU eight waves: a wide tile re-reads
    // less, a narrow one fills the chip.  Whole products, us, with the 8x8 / 4x4 /
    // 2x2 tile: 24^3 at 2^12 points 53 / 51 / 54; 64^2x32 at 2^11 95 / 81 / 98, at 2^12
    // 147 / 150 / 186; 64^3 at 2^10 80 / 68 / 86, at 2^12 230 / 240 / 322.  No wider
    // than the narrow side needs, whose missing rows would be computed twice: 35x7x4
    // at 2^15 with the 8x8 tile 106, with the 4x4 one 98.
    const size_t full = 8 * (size_t)device_cus();
    const auto waves = [&](size_t T) { return ((m + T - 1) / T) * ((n + T - 1) / T) * (npts / 64) * r; };
    const size_t side = m < n ? m : n;
    if (waves(8) >= full && side > 4) return tiled_launch<8>(A, B, C, m, k, n, npts, r, p, scale, s);
    if (waves(4) >= full && side > 2) return tiled_launch<4>(A, B, C, m, k, n, npts, r, p, scale, s);
    if (waves(2) >= full && side <= 2) return tiled_launch<2>(A, B, C, m, k, n, npts, r, p, scale, s);
    // too few tiles: from eight steps on the inner dimension is split, 4x4 tiles
    // while that gives half the waves, 2x2 below.  Whole products, us, 2x2 unsplit /
    // split rule: 64^3 at 2^6 points 25 / 22, at 2^8 38 / 33; 64^2x32 at 2^9 40 / 34;
    // 16^3 at 2^9 21 / 20; 9x100x9 at 2^8 29 / 21; 3x300x5 at 2^10 60 / 32; 4x8x4 20 / 19.
    if (k >= 8) {
        if (2 * kSplitK * waves(4) >= full) return splitk_launch<4>(A, B, C, m, k, n, npts, r, p, scale, s);
        return splitk_launch<2>(A, B, C, m, k, n, npts, r, p, scale, s);
    }
    return tiled_launch<2>(A, B, C, m, k, n, npts, r, p, scale, s);
}

size_t limb_block_bytes(size_t rows, size_t kdim) { return rpad_of(rows) * kpad_of(kdim) * 4; }

hipError_t launch_to_limbs(const uint32_t *X, uint8_t *Y, size_t rows, size_t kdim, bool row_major, size_t npts,
                           uint32_t p, hipStream_t s)
{
    const size_t rpad = rpad_of(rows), kchunks = kpad_of(kdim) / 64;
    if (rpad > 65535 || kchunks > 65535) return hipErrorInvalidValue;
    dim3 grid((unsigned)((npts + 63) / 64), (unsigned)kchunks, (unsigned)rpad);
    hipLaunchKernelGGL(to_limbs_kernel, grid, dim3(256), 0, s, X, Y, (int)rows, (int)kdim, row_major ? 1 : 0, npts, p,
                       limb_block_bytes(rows, kdim), (int)kchunks);
    return hipGetLastError();
}

hipError_t launch_pointwise_mfma(const uint8_t *Al, const uint8_t *Bl, uint32_t *Cmat, size_t m, size_t k, size_t n,
                                 size_t npts, uint32_t p, uint32_t scale, hipStream_t s)
{
    const MfmaConst mc = mfma_const(p, scale);
    const size_t mpad = rpad_of(m), npad = rpad_of(n), kchunks = kpad_of(k) / 64;
    if (npts > 0x7fffffff) return hipErrorInvalidValue;
    const size_t a_bytes = limb_block_bytes(m, k);
    const int cus = device_cus();
    if (mpad <= 128 && kchunks <= 2 && npad * kchunks * 256 <= 65536) {
        const size_t lds = npad * kchunks * 256;
        const size_t grid = npts < (size_t)cus * 2 ? npts : (size_t)cus * 2;
        const int nw = mpad == 96 ? 3 : 4;
        auto k = nw == 3 ? (kchunks == 1 ? pw_mfma_rega_kernel<1, 3> : pw_mfma_rega_kernel<2, 3>)
                         : (kchunks == 1 ? pw_mfma_rega_kernel<1, 4> : pw_mfma_rega_kernel<2, 4>);
        hipError_t e = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(64 * nw), lds, s, Al, Bl, Cmat, (int)m, (int)n, (int)mpad,
                           (int)npad, npts, p, mc);
        return hipGetLastError();
    }
    if (a_bytes <= (size_t)kLdsAMax) {
        const size_t lds = a_bytes + (size_t)32 * kchunks * 256;
        hipError_t e = hipFuncSetAttribute((const void *)pw_mfma_lds_kernel,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
        const size_t grid = npts < (size_t)cus * 2 ? npts : (size_t)cus * 2;
        hipLaunchKernelGGL(pw_mfma_lds_kernel, dim3((unsigned)grid), dim3(256), lds, s, Al, Bl, Cmat, (int)m, (int)n,
                           (int)kchunks, (int)mpad, (int)npad, npts, p, mc);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(pw_mfma_kernel, dim3((unsigned)npts), dim3(256), 0, s, Al, Bl, Cmat, (int)m, (int)n,
                       (int)kchunks, (int)mpad, (int)npad, limb_block_bytes(m, k), limb_block_bytes(n, k), p, mc);
    return hipGetLastError();
}

hipError_t launch_point_to_entry(const uint32_t *X, uint32_t *Y, size_t entries, size_t npts, hipStream_t s)
{
    if (!entries || !npts) return hipSuccess;
    if ((npts + 63) / 64 > 0x7fffffff || (entries + 63) / 64 > 65535) return hipErrorInvalidValue;
    dim3 grid((unsigned)((npts + 63) / 64), (unsigned)((entries + 63) / 64));
    hipLaunchKernelGGL(point_to_entry_kernel, grid, dim3(256), 0, s, X, Y, entries, npts);
    return hipGetLastError();
}

}  // namespace lbx
