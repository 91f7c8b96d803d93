// Plain products by several primes at once: the transforms of every prime of a
// multi-prime product, or both operands of a single one, in one launch each
// way, with the pointwise stage of pointwise.hip between.
//
// Products of small and ordinary matrices modulo several primes are bound by
// launches, not by bandwidth: a prime's own product takes four kernels of some
// 5 to 10 us each with fewer groups than the chip holds (24^3 at 2^11 points:
// 576 groups of 128 threads per operand).  Here blockIdx.y is the prime and
// blockIdx.x runs over the entry groups of a, then of b.  Measured (us, a
// prime and an operand at a time / here): 16^3 at 2^9 points modulo a prime
// without roots of unity 103 / 28; 24^3 integers at 2^11, five primes, 572 / 370;
// 10x20x30 at 2^12, one prime, 58 / 45; 16^3 at 2^9, one prime, 35 / 21.
#include "ntt_device.h"

namespace lbx {
namespace {
using namespace ntt;

// Kernel arguments of the forward transforms (a's groups first).
struct FwdArgs {
    DevView a, b;
    size_t astride, bstride, rev_a, rev_b;
    uint32_t *ahat, *bhat;
    size_t ea, eb, ga;
    bool centre;  // outputs centred to int32
    uint32_t p[kMultiPrimes];
    const uint2 *twa[kMultiPrimes], *twb[kMultiPrimes];
};
struct InvArgs {
    const uint32_t *chat;
    DevView c;
    size_t cstride, count;
    size_t entries;
    uint32_t p[kMultiPrimes];
    const uint2 *twc[kMultiPrimes];
};

// One whole forward transform per TP threads.  Input coefficient t is
// coefficient t of the view, or rev-1-t of it when rev != 0 (the view has at
// most rev coefficients then), zero where that is outside the view; out may be the
// view's own storage.  One body
// serves every layout (a stride) and both zero paddings (only the first stage
// differs, behind a uniform branch): with a body for each the kernel is several
// times as long, and a launch of few groups waits for its instructions (800
// entries at 2^12 points: 21.0 us against 19.2 here; 57344 at 2^11: 164 against 149).
template <int L>
__device__ __forceinline__ void forward_entry(const DevView &in, size_t rev, size_t e, bool active, bool halfzero,
                                              const uint2 *__restrict__ tw, uint32_t p, uint32_t h,
                                              uint32_t *out, int tp, uint32_t *lds)
{
    using C = Cfg<L>;
    constexpr int RP0 = C::RLOG;
    // input coefficients [lo, hi) are inside the view
    const int lo = (int)(rev ? rev - in.size : 0), hi = (int)min(rev ? rev : in.size, (size_t)C::N);
    const size_t first = in.shift + (rev ? rev - 1 : 0);
    size_t stride = 1, base = (active ? e : 0) * in.stor;
    if (in.layout == 1) {
        stride = in.rows * in.cols;
        base = active ? e : 0;
    } else if (in.layout == 2) {
        const size_t row = (active ? e : 0) / in.cols;
        stride = in.cols;
        base = row * in.cols * in.stor + ((active ? e : 0) - row * in.cols);
    }
    const uint32_t *src = in.base + base + first * stride;
    const ptrdiff_t step = rev ? -(ptrdiff_t)stride : (ptrdiff_t)stride;
    uint32_t x[C::R];
#pragma unroll
    for (int u = 0; u < (C::R >> RP0); ++u)
#pragma unroll
        for (int q = 0; q < (1 << RP0); ++q) {
            const int t = elem<L, L - RP0, RP0>(tp, u, q);
            x[u * (1 << RP0) + q] = active && t >= lo && t < hi ? src[t * step] : 0u;
        }
    if (halfzero)
        dif_pass<L, 0, RP0, true, 0, 1>(x, tp, tw, p);
    else
        dif_pass<L, 0, RP0, false, 0, 1>(x, tp, tw, p);
    dif_pass<L, 0, RP0, false, 1, RP0>(x, tp, tw, p);
    if constexpr (RP0 < L) {
        constexpr int NRP = (L - RP0) < C::RLOG ? (L - RP0) : C::RLOG;
        scatter<L, L - RP0, RP0>(x, lds, tp);
        __syncthreads();
        gather<L, L - RP0 - NRP, NRP>(x, lds, tp);
        dif_passes<L, RP0, L, false>(x, lds, tp, tw, p);
    }
    if (active) dif_store<L, true>(x, tp, out + e * C::N, p, h);
}

template <int L>
__global__ void __launch_bounds__(Cfg<L>::BLOCK) multi_dif_kernel(FwdArgs A)
{
    using C = Cfg<L>;
    extern __shared__ uint32_t lds_all[];
    const unsigned i = blockIdx.y;
    const bool isa = blockIdx.x < A.ga;
    const size_t entries = isa ? A.ea : A.eb, rev = isa ? A.rev_a : A.rev_b;
    DevView in = isa ? A.a : A.b;
    in.base += (size_t)i * (isa ? A.astride : A.bstride);
    uint32_t *out = (isa ? A.ahat : A.bhat) + (size_t)i * entries * C::N;
    const uint2 *tw = isa ? A.twa[i] : A.twb[i];
    const int pib = threadIdx.x / C::TP, tp = threadIdx.x % C::TP;
    const size_t e = (size_t)(isa ? blockIdx.x : blockIdx.x - A.ga) * C::G + pib;
    uint32_t *lds = lds_all + pib * C::STRIDE;
    const uint32_t h = A.centre ? A.p[i] >> 1 : ~0u;
    forward_entry<L>(in, rev, e, e < entries, (rev ? rev : in.size) * 2 <= (size_t)C::N, global_ptr(tw), A.p[i], h, out,
                     tp, lds);
}

template <int L>
__global__ void __launch_bounds__(Cfg<L>::BLOCK) multi_dit_kernel(InvArgs A)
{
    extern __shared__ uint32_t lds_all[];
    const unsigned i = blockIdx.y;
    DevView out = A.c;
    out.base += (size_t)i * A.cstride;
    dit_body<L, 0, false>(A.chat + (size_t)i * A.entries * Cfg<L>::N, A.entries, global_ptr(A.twc[i]), A.p[i], out, 0,
                          A.count, 1u, 0u, (size_t)blockIdx.x * Cfg<L>::G, threadIdx.x, lds_all);
}

template <class K, class Args>
hipError_t launch_lds(K kernel, size_t grid, unsigned r, int block, size_t lds, const Args &args, hipStream_t s)
{
    if (grid > 0x7fffffff) return hipErrorInvalidValue;
    if (lds > 65536) {
        const hipError_t e =
            hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid, r), dim3(block), lds, s, args);
    return hipGetLastError();
}

template <int L>
hipError_t forward_launch(FwdArgs &A, unsigned r, hipStream_t s)
{
    using C = Cfg<L>;
    A.ga = (A.ea + C::G - 1) / C::G;
    const size_t grid = A.ga + (A.eb + C::G - 1) / C::G;
    return launch_lds(multi_dif_kernel<L>, grid, r, C::BLOCK, C::LDS_BYTES, A, s);
}

template <int L>
hipError_t inverse_launch(const InvArgs &A, unsigned r, hipStream_t s)
{
    using C = Cfg<L>;
    return launch_lds(multi_dit_kernel<L>, (A.entries + C::G - 1) / C::G, r, C::BLOCK, C::LDS_BYTES, A, s);
}

bool in_range(const MultiProduct &mp)
{
    return mp.r >= 1 && mp.r <= (unsigned)kMultiPrimes && mp.L >= 1 && mp.L <= (unsigned)kMaxLdsLog;
}

}  // namespace

#define LBX_CASES(X) \
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15)

hipError_t launch_multi_forward(const MultiProduct &mp, hipStream_t s)
{
    if (!in_range(mp) || (mp.rev_a && mp.a.size > mp.rev_a) || (mp.rev_b && mp.b.size > mp.rev_b))
        return hipErrorInvalidValue;
    FwdArgs A;
    A.a = mp.a;
    A.b = mp.b;
    A.astride = mp.astride;
    A.bstride = mp.bstride;
    A.rev_a = mp.rev_a;
    A.rev_b = mp.rev_b;
    A.ahat = mp.ahat;
    A.bhat = mp.bhat;
    A.ea = mp.m * mp.k;
    A.eb = mp.k * mp.n;
    A.centre = pointwise_tiled((size_t)1 << mp.L);
    for (int i = 0; i < kMultiPrimes; ++i) {
        const bool on = i < (int)mp.r;
        A.p[i] = on ? mp.p[i] : 0;
        A.twa[i] = on ? mp.twa[i] : nullptr;
        A.twb[i] = on ? mp.twb[i] : nullptr;
    }
    switch (mp.L) {
#define LBX_CASE(l) \
    case l: return forward_launch<l>(A, mp.r, s);
        LBX_CASES(LBX_CASE)
#undef LBX_CASE
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_multi_pointwise(const MultiProduct &mp, hipStream_t s)
{
    if (!in_range(mp)) return hipErrorInvalidValue;
    const size_t npts = (size_t)1 << mp.L;
    if (pointwise_tiled(npts))
        return launch_pointwise_tiled(mp.ahat, mp.bhat, mp.chat, mp.m, mp.k, mp.n, npts, mp.r, mp.p, mp.scale, s);
    return launch_pointwise_plain(mp.ahat, mp.bhat, mp.chat, mp.m, mp.k, mp.n, npts, mp.r, mp.p, mp.scale, s);
}

hipError_t launch_multi_inverse(const MultiProduct &mp, hipStream_t s)
{
    if (!in_range(mp)) return hipErrorInvalidValue;
    InvArgs A;
    A.chat = mp.chat;
    A.c = mp.c;
    A.cstride = mp.cstride;
    A.count = mp.count;
    A.entries = mp.m * mp.n;
    for (int i = 0; i < kMultiPrimes; ++i) {
        const bool on = i < (int)mp.r;
        A.p[i] = on ? mp.p[i] : 0;
        A.twc[i] = on ? mp.twc[i] : nullptr;
    }
    switch (mp.L) {
#define LBX_CASE(l) \
    case l: return inverse_launch<l>(A, mp.r, s);
        LBX_CASES(LBX_CASE)
#undef LBX_CASE
    default: return hipErrorInvalidValue;
    }
}

}  // namespace lbx
