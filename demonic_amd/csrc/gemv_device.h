// gemv_device.h -- device helpers that the kernel files share: buffer loads, the
// zero rule's chains, and the pieces of the MFMA layouts (the three-term split
// of x, inf/NaN screening, tiny activation rows, LDS swizzle, chunk order).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

namespace dmc {
namespace {

// 128-bit weight loads through a buffer resource, marked nontemporal: weights
// are streamed once per launch, so they should not displace x or y in the
// caches.  (Measured on MI355X: ~8% more bandwidth than plain global loads.)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t weight_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}

constexpr int kLoadNT = 2;  // cache-policy bits of a buffer load: nt

__device__ __forceinline__ u32x4 load_w16(__amdgpu_buffer_rsrc_t r, uint32_t byte_off) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, kLoadNT);
}

// The same with a wave-uniform part of the offset in the instruction's scalar
// offset.  Measured on gfx950: the range check covers the sum of both offsets
// (per dword), like a single offset.  Keeping a loop's row offset scalar and
// the lane's offset loop-invariant leaves no per-load vector address
// arithmetic, whose temporaries the register allocator otherwise places in
// registers just freed by a load -- and the compiler then waits for that
// load's whole batch before the next one may issue.
__device__ __forceinline__ u32x4 load_w16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t uniform_off) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, uniform_off, kLoadNT);
}

__device__ __forceinline__ float widen_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float widen_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// ---- zero outputs of the FMA kernels ------------------------------------------
//
// The FMA kernels split k, so an output is a sum of partial chains.  When that
// sum comes out exactly 0 it can differ from the reference chain (fmaf over
// ascending k from +0, jit.rs:29655-29670): a run of underflowing products of
// both signs leaves the chain at the zero of the last one's sign, where a sum
// of reordered partials is -0 only if every partial is; and reordered partials
// can cancel exactly where the chain keeps a subnormal residue.  Neither can
// happen when every product is an exact zero (some factor +-0): the chain then
// never leaves +0, and neither does the split sum (lanes with elements start
// at +0, idle ones add -0).  So a zero output is settled by the reference's
// rule: +0 when no product has two nonzero factors -- an all-zero activation
// row, an all-zero weight row, or factors that never meet -- and otherwise
// the chain itself (underflow or exact cancellation, which takes crafted
// data).  The common path costs one compare and one ballot per output.

// The reference chain for one output: K products x[k] * w[k * wstep], any
// alignment (2- and 4-byte loads; the rare path only).
__device__ float chain_strided(const uint16_t *__restrict__ w, int64_t wstep, const float *__restrict__ x, int K) {
    float acc = 0.0f;
    int k = 0;
    for (; k + 4 <= K; k += 4) {
        const uint16_t *p = w + (int64_t)k * wstep;
        const uint32_t b0 = p[0], b1 = p[wstep], b2 = p[2 * wstep], b3 = p[3 * wstep];
        const float x0 = x[k], x1 = x[k + 1], x2 = x[k + 2], x3 = x[k + 3];
        acc = fmaf(x0, __uint_as_float(b0 << 16), acc);
        acc = fmaf(x1, __uint_as_float(b1 << 16), acc);
        acc = fmaf(x2, __uint_as_float(b2 << 16), acc);
        acc = fmaf(x3, __uint_as_float(b3 << 16), acc);
    }
    for (; k < K; ++k) acc = fmaf(x[k], __uint_as_float((uint32_t)w[(int64_t)k * wstep] << 16), acc);
    return acc;
}

template <class T>
__device__ __forceinline__ const T *readlane_ptr(const T *p, int j) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, j);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), j);
    return reinterpret_cast<const T *>(((uint64_t)hi << 32) | lo);
}

// Wave-uniform: does some k have x[k] and (w == nullptr, or w[k * wstep])
// nonzero?  Contiguous rows (wstep <= 1, K <= 2^28): 16-byte buffer loads at
// the rows' own 4- and 2-byte alignments (exact on gfx950), 8 elements per
// lane per load, 4096 per round -- one round for K <= 4096.  The weight range
// ends exactly after element K-1: a load's dword that runs past it comes back
// as zeros (element K-1 itself when it shares such a dword), so element K-1
// is also read alone, 2 bytes, and nothing past the row is ever read.
// Strided columns: one element per lane per load, 64 * 32 per round.  All
// loads of a round are in flight together; the scan stops at the first round
// that finds a product.
__device__ bool wave_any_product(const float *x, const uint16_t *w, int64_t wstep, int K) {
    const int lane = threadIdx.x & 63;
    if (K <= 0) return false;
    if (wstep <= 1 && K <= (1 << 28)) {
        constexpr int U = 8;
        const uintptr_t wb = reinterpret_cast<uintptr_t>(w);
        const __amdgpu_buffer_rsrc_t xr = weight_rsrc(x, (uint32_t)K * 4u);
        const uintptr_t w0 = wb & ~(uintptr_t)3;
        const uint32_t wd = (uint32_t)(wb - w0);  // 0 or 2
        const __amdgpu_buffer_rsrc_t wr =
            weight_rsrc(reinterpret_cast<const void *>(w ? w0 : reinterpret_cast<uintptr_t>(x)),
                        w ? wd + 2u * (uint32_t)K : 0u);
        const uint32_t wl = w ? (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(wr, wd + 2u * (K - 1), 0, 0) : 1u;
        const uint32_t xl = __float_as_uint(x[K - 1]) & 0x7fffffffu;
        bool first = true;
        for (int k0 = 0; k0 < K; k0 += 512 * U) {
            u32x4 xa[U], xc[U], wv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t e = (uint32_t)(k0 + (u * 64 + lane) * 8);
                xa[u] = __builtin_amdgcn_raw_buffer_load_b128(xr, e * 4u, 0, 0);
                xc[u] = __builtin_amdgcn_raw_buffer_load_b128(xr, e * 4u + 16u, 0, 0);
                wv[u] = w ? __builtin_amdgcn_raw_buffer_load_b128(wr, wd + e * 2u, 0, 0) : u32x4{~0u, ~0u, ~0u, ~0u};
            }
            uint32_t hit = first && (wl & 0x7fffu) != 0 && xl != 0 ? 1u : 0u;
            first = false;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int e = k0 + (u * 64 + lane) * 8;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const uint32_t xv = (i < 4 ? xa[u][i] : xc[u][i - 4]) & 0x7fffffffu;
                    const uint32_t wv16 = (wv[u][i >> 1] >> (16 * (i & 1))) & 0x7fffu;
                    hit |= (e + i < K && xv != 0 && wv16 != 0) ? 1u : 0u;
                }
            }
            if (__builtin_amdgcn_ballot_w64(hit != 0) != 0) return true;
        }
        return false;
    }
    constexpr int U = 32;
    for (int k0 = 0; k0 < K; k0 += 64 * U) {
        uint32_t xb[U], wb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(k0 + u * 64 + lane, K - 1);
            xb[u] = __float_as_uint(x[k]) & 0x7fffffffu;
            wb[u] = w ? (uint32_t)w[(int64_t)k * wstep] & 0x7fffu : 1u;
        }
        uint32_t hit = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) hit |= (k0 + u * 64 + lane < K && xb[u] != 0 && wb[u] != 0) ? 1u : 0u;
        if (__builtin_amdgcn_ballot_w64(hit != 0) != 0) return true;
    }
    return false;
}

// The zero rule for the general row-dot kernel's outputs this wave holds, one
// per lane: `zero` marks a lane whose output s is exactly 0 and is stored; x is
// its activation row, w its first weight, wstep the elements between
// consecutive k.  All 64 lanes call it (wave-uniform control flow): rows are
// scanned by the whole wave, one output at a time, and the chains (if any) run
// one per lane.
__device__ float settle_zero(float s, bool zero, const float *x, const uint16_t *w, int64_t wstep, int K) {
    uint64_t pend = __builtin_amdgcn_ballot_w64(zero);
    if (pend == 0) return s;
    const int lane = threadIdx.x & 63;
    // activation rows that hold only +-0, each distinct row scanned once (a
    // lone zero output skips this: its product scan covers its row)
    bool xnz = true;
    if (pend & (pend - 1)) while (pend) {
        const int j = __builtin_ctzll(pend);
        const float *xj = readlane_ptr(x, j);
        const bool nz = wave_any_product(xj, nullptr, 0, K);
        const bool same = zero && x == xj;
        if (same) xnz = nz;
        pend &= ~__builtin_amdgcn_ballot_w64(same);
    }
    // outputs whose products all have a zero factor
    bool chain = false;
    for (uint64_t todo = __builtin_amdgcn_ballot_w64(zero && xnz); todo; todo &= todo - 1) {
        const int j = __builtin_ctzll(todo);
        const bool hit = wave_any_product(readlane_ptr(x, j), readlane_ptr(w, j), wstep, K);
        if (lane == j) chain = hit;
    }
    if (zero) s = chain ? chain_strided(w, wstep, x, K) : 0.0f;
    return s;
}

// ---- zero outputs of the MFMA kernels ------------------------------------------
//
// The scans and chains are functions of their own, called from rolled loops:
// expanded at the kernels' unrolled outputs, this rare path set their registers
// (gemm_sum_slices_kernel: 149 VGPRs, 3 waves per SIMD, and 199 SGPRs spilled,
// against 63, 8 waves and none).

// Least and greatest magnitude of a row: lo - 1 (zeros wrap to the top), hi.
struct Range {
    uint32_t lo1 = ~0u, hi = 0;
    __device__ __forceinline__ void put(uint32_t v) {
        lo1 = min(lo1, v - 1u);
        hi = max(hi, v);
    }
    __device__ __forceinline__ void over_wave() {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            lo1 = min(lo1, (uint32_t)__shfl_xor((int)lo1, o));
            hi = max(hi, (uint32_t)__shfl_xor((int)hi, o));
        }
    }
};

// The wave's ranges of an activation row and of a weight row or column, K <=
// 2^24, 16-byte loads at the rows' own alignments (exact on gfx950; a dword past
// the row's end comes back as zeros, which do not count, and the last weight,
// which may share one, is read alone).
__device__ __noinline__ Range wave_range(const float *x, int K) {
    Range r;
    const __amdgpu_buffer_rsrc_t xr = weight_rsrc(x, (uint32_t)K * 4u);
#pragma nounroll
    for (int k0 = 0; k0 < K; k0 += 1024) {
        u32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            v[u] = __builtin_amdgcn_raw_buffer_load_b128(xr, (uint32_t)(k0 + (u * 64 + (threadIdx.x & 63)) * 4) * 4u, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) r.put(v[u][i] & 0x7fffffffu);
    }
    r.over_wave();
    return r;
}

__device__ __noinline__ Range wave_range(const uint16_t *w, int64_t wstep, int K) {
    const int lane = threadIdx.x & 63;
    Range r;
    r.put((uint32_t)w[(int64_t)(K - 1) * wstep] & 0x7fffu);
    if (wstep <= 1) {
        const uintptr_t wb = reinterpret_cast<uintptr_t>(w);
        const uint32_t wd = (uint32_t)(wb & 3);
        const __amdgpu_buffer_rsrc_t wr = weight_rsrc(reinterpret_cast<const void *>(wb - wd), wd + 2u * (uint32_t)K);
#pragma nounroll
        for (int k0 = 0; k0 < K; k0 += 2048) {
            u32x4 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                v[u] = __builtin_amdgcn_raw_buffer_load_b128(wr, wd + (uint32_t)(k0 + (u * 64 + lane) * 8) * 2u, 0, 0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    r.put(v[u][i] & 0x7fffu);
                    r.put(v[u][i] >> 16 & 0x7fffu);
                }
        }
    } else {
#pragma nounroll
        for (int k0 = 0; k0 < K; k0 += 64 * 8) {
            uint32_t v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = w[(int64_t)min(k0 + u * 64 + lane, K - 1) * wstep];
#pragma unroll
            for (int u = 0; u < 8; ++u) r.put(v[u] & 0x7fffu);
        }
    }
    r.over_wave();
    return r;
}

// For an output whose split sum is exactly zero, from the ranges of its two
// rows: is it settled that +0 stands for the reference chain?  A product x * w
// is a multiple of 2^(ex + ew - 284) (biased exponents; 23 and 7 fraction bits).
// Where that is at least 2^-149 for the least nonzero |x| and |w|, every sum of
// the chain is a multiple of the least subnormal, none underflows, and a chain
// that ends at zero ends at +0 (an exact cancellation, or it never left +0).
// And where K products of the greatest |x| and |w| cannot reach inf, nor can
// the chain on its way (|x| < 2^(ex - 126), |w| < 2^(ew - 126), and its
// roundings grow a sum less than 4-fold up to K = 2^24).  So +0 is the answer
// where the reference is zero, and where its roundings leave a residue, +0 is
// as close to the exact sum as any other order's.
__device__ __forceinline__ bool zero_is_plus(const Range &x, const Range &w, int K) {
    const uint32_t ex = (x.lo1 + 1) >> 23, ew = (w.lo1 + 1) >> 7;
    const uint32_t lg = 32 - __builtin_clz((uint32_t)K);  // K < 2^lg
    return x.hi == 0 || w.hi == 0 ||
           (ex >= 1 && ew >= 1 && ex + ew >= 135 && (x.hi >> 23) + (w.hi >> 7) + lg <= 377);
}

// The reference chain of one output by a whole wave (w, x, K wave-uniform;
// packed weights, K <= 2^24): the lanes load 512 elements at a time, 8 each, the
// next 512 while these are summed, and the accumulator goes from lane to lane, 8
// dependent fmas and one readlane per lane.  A lane on its own waits for memory
// every 8 elements: the chain of one output of K = 14336 took 560 us that way,
// against 31 us here.  Elements past K multiply +0 by -0: adding -0 keeps the
// accumulator.
__device__ __noinline__ float wave_chain(const uint16_t *w, const float *x, int K) {
    const int lane = threadIdx.x & 63;
    const uintptr_t wb = reinterpret_cast<uintptr_t>(w);
    const uint32_t wd = (uint32_t)(wb & 3);  // 0 or 2
    const __amdgpu_buffer_rsrc_t xr = weight_rsrc(x, (uint32_t)K * 4u);
    const __amdgpu_buffer_rsrc_t wr = weight_rsrc(reinterpret_cast<const void *>(wb - wd), wd + 2u * (uint32_t)K);
    const uint32_t wlast = w[K - 1];  // its dword may straddle the range's end
    u32x4 x0, x1, wv, nx0, nx1, nwv;
    auto load = [&](int k0) __attribute__((always_inline)) {
        const uint32_t e0 = (uint32_t)(k0 + lane * 8);
        nx0 = __builtin_amdgcn_raw_buffer_load_b128(xr, e0 * 4u, 0, 0);
        nx1 = __builtin_amdgcn_raw_buffer_load_b128(xr, e0 * 4u + 16u, 0, 0);
        nwv = __builtin_amdgcn_raw_buffer_load_b128(wr, wd + e0 * 2u, 0, 0);
    };
    float acc = 0.0f;
    load(0);
#pragma nounroll
    for (int k0 = 0; k0 < K; k0 += 512) {
        x0 = nx0, x1 = nx1, wv = nwv;
        load(k0 + 512);
        const int left = K - k0 - lane * 8;  // elements of this lane's 8 (x past K is 0)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint32_t lo = 2 * v >= left ? 0x8000u : 2 * v + 1 == left ? wlast : wv[v] & 0xffffu;
            const uint32_t hi = 2 * v + 1 >= left ? 0x8000u : 2 * v + 2 == left ? wlast : wv[v] >> 16;
            wv[v] = lo | hi << 16;
        }
        const int n = min(64, (K - k0 + 7) / 8);
#pragma nounroll
        for (int l = 0; l < n; ++l) {
            float t = acc;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                t = fmaf(__uint_as_float(e < 4 ? x0[e] : x1[e - 4]), e & 1 ? widen_hi(wv[e >> 1]) : widen_lo(wv[e >> 1]),
                         t);
            acc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), l));
        }
    }
    return acc;
}

// One per lane.
__device__ __noinline__ float lane_chain(const uint16_t *w, int64_t wstep, const float *x, int K) {
    return chain_strided(w, wstep, x, K);
}

// The chains of the lanes that ask (s for the others): one after another by the
// whole wave where they are few and the weights packed, else one per lane.
__device__ __forceinline__ float few_or_lane_chains(bool ask, float s, const uint16_t *w, const float *x, int K,
                                                    int64_t wstep = 1) {
    uint64_t todo = __builtin_amdgcn_ballot_w64(ask);
    if (wstep > 1 || K > 1 << 24 || __builtin_popcountll(todo) > 6) {
        if (ask) s = lane_chain(w, wstep, x, K);
        return s;
    }
    for (; todo; todo &= todo - 1) {
        const int j = __builtin_ctzll(todo);
        const float c = wave_chain(readlane_ptr(w, j), readlane_ptr(x, j), K);
        if ((int)(threadIdx.x & 63) == j) s = c;
    }
    return s;
}

// The reference's values for outputs whose sums are exactly zero: a lane's are
// y[e] where bit e of `zeros` is set (e < 4), of its activation row x and the
// weights w + e * wpitch, wstep elements between consecutive k.  All 64 lanes
// call this.  The ranges of each distinct activation and weight row are taken
// once by the whole wave and settle almost every zero (zero_is_plus); the chains
// of the others follow.
__device__ __forceinline__ void settle_zeros(float *y, uint32_t zeros, const float *x, const uint16_t *w, int64_t wpitch,
                                          int64_t wstep, int K) {
    const bool ranges = K <= 1 << 24;
    Range rx;
    if (ranges)
        for (uint64_t todo = __builtin_amdgcn_ballot_w64(zeros != 0); todo;) {
            const float *const xj = readlane_ptr(x, __builtin_ctzll(todo));
            const Range r = wave_range(xj, K);
            if (x == xj) rx = r;
            todo &= ~__builtin_amdgcn_ballot_w64(x == xj);
        }
#pragma nounroll
    for (int e = 0; e < 4; ++e, w += wpitch) {
        const bool zero = (zeros >> e & 1) != 0;
        bool plus = ranges && rx.hi == 0;  // an activation row of +-0
        if (ranges)
            for (uint64_t todo = __builtin_amdgcn_ballot_w64(zero && !plus); todo;) {
                const uint16_t *const wj = readlane_ptr(w, __builtin_ctzll(todo));
                const Range r = wave_range(wj, wstep, K);
                if (w == wj) plus |= zero_is_plus(rx, r, K);
                todo &= ~__builtin_amdgcn_ballot_w64(w == wj);
            }
        const float v = few_or_lane_chains(zero && !plus, 0.0f, w, x, K, wstep);
        if (zero) y[e] = v;
    }
}

// ---- RD skinny M on MFMA: W [N,K] x X [M,K], K % 64 == 0 ---------------------------
//
// From M = 2 the FMA path loses to the matrix cores (M fmas per weight element,
// MT activation rows of registers; on the LM-head shape M = 2 takes 174-183 us
// there against 161-166 here, M = 3 212-240 against 166-173), so the
// products go to v_mfma_f32_16x16x32_bf16: A = a 16-row weight tile, B = x^T
// for 16 activation rows.  x is f32, so it enters as three bf16 terms,
// x == hi + mid + lo, each taken by truncation: every residual is exact in
// f32 and keeps at most 8 significant bits, so the split is exact for
// |x| >= 2^-110 (below that the error is < 2^-133 absolute).  Measured on
// gfx950 this MFMA multiplies exactly, sums a block's 32 products and the
// accumulator with one rounding, keeps bf16/f32 subnormals, and follows IEEE
// for inf and NaN -- so each output is the exact dot product up to 3
// roundings per 32 k, more accurate than the reference's sequential fma chain.
//
// Special values keep the reference's classes (fmaf(x, w, acc) semantics):
//   x = +-inf or NaN: hi carries it (a NaN is kept quiet), mid = lo = 0;
//   x != 0 tiny: hi is never 0, so inf * x stays inf;
//   w = +-inf or NaN: multiplies hi only -- the mid and lo MFMAs see 0 there,
//     because inf * (mid == 0) would be NaN where the reference has inf.
//
// Zeros: the MFMA rounds a nonzero sum smaller than half the least f32
// subnormal to +0 whatever its sign, where the reference's fmaf gives the
// signed zero (every product underflowing negative ends at -0).  So an output
// that comes out exactly zero is settled at the end: +0 where the activation or
// the weight row holds only +-0 or (the gemm layout and the slice sum,
// settle_zeros) the two rows' magnitudes leave the chain no room to underflow or
// overflow, otherwise the chain itself, fmaf over ascending k from +0.

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma_bf16(const u32x4 &a, const u32x4 &b, const f32x4 &c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
}

// Bits 0xffff in each 16-bit half of d whose bf16 exponent is all ones.
__device__ __forceinline__ uint32_t inf_nan_mask(uint32_t d) {
    const uint32_t t = ((d & 0x7f807f80u) + 0x00800080u) & 0x80008000u;
    return (t >> 15) * 0xffffu;
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// Running per-half maximum of bf16 magnitudes: a half holding an inf or NaN
// reaches 0x7f80.  Two instructions per dword (and, packed max); the exact
// per-element mask is computed only when a wave's screen fires.
__device__ __forceinline__ uint32_t max_mag(uint32_t acc, uint32_t d) {
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, acc),
                                                                  __builtin_bit_cast(u16x2, d & 0x7fff7fffu)));
}

__device__ __forceinline__ bool wave_has_inf_nan(uint32_t mx) {
    const bool mine = (mx & 0xffffu) >= 0x7f80u || (mx >> 16) >= 0x7f80u;
    return __builtin_amdgcn_ballot_w64(mine) != 0;
}

// The three bf16 terms of one f32.
__device__ __forceinline__ void split3(float v, uint32_t &h, uint32_t &m, uint32_t &l) {
    // Selects, not branches: every lane of the rows16 layout splits 16 values per line.
    const uint32_t u = __float_as_uint(v);
    const bool fin = (u & 0x7f800000u) != 0x7f800000u;
    const uint32_t t = u >> 16;
    const uint32_t nan_q = !fin && (u & 0x007fffffu) ? 0x0040u : 0u;                 // NaN: stay NaN after truncation
    const uint32_t keep = fin && (t & 0x7fffu) == 0 && (u & 0x7fffffffu) != 0 ? 1u : 0u;  // |x| < 2^-133: hi nonzero
    h = t | nan_q | keep;
    const float r1 = fin ? v - __uint_as_float(h << 16) : 0.0f;
    m = __float_as_uint(r1) >> 16;
    const float r2 = r1 - __uint_as_float(m << 16);
    l = __float_as_uint(r2) >> 16;
}

// Four values at once, two per dword of each plane.  Where all four are
// finite with |x| = 0 or |x| >= 2^-133 (bf16's least subnormal), split3's
// rule is truncation alone (no NaN quieting, no kept tiny bit, no inf
// residual), taken here without its selects: 4 operations a value and the
// packing instead of about 15.  The test is two reductions over the
// magnitudes (|x| - 1 wraps 0 to the top); a lane that fails it (an inf, a
// NaN or a tiny value among its four) takes split3.
__device__ __forceinline__ void split4(const float *v, uint32_t *hi, uint32_t *mid, uint32_t *lo) {
    uint32_t amax = 0, amin1 = 0xffffffffu;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t a = __float_as_uint(v[e]) & 0x7fffffffu;
        amax = max(amax, a);
        amin1 = min(amin1, a - 1u);
    }
    if (amax < 0x7f800000u && amin1 >= 0x0000ffffu) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t u0 = __float_as_uint(v[2 * q]), u1 = __float_as_uint(v[2 * q + 1]);
            const float r10 = v[2 * q] - __uint_as_float(u0 & 0xffff0000u);
            const float r11 = v[2 * q + 1] - __uint_as_float(u1 & 0xffff0000u);
            const uint32_t b10 = __float_as_uint(r10), b11 = __float_as_uint(r11);
            const uint32_t b20 = __float_as_uint(r10 - __uint_as_float(b10 & 0xffff0000u));
            const uint32_t b21 = __float_as_uint(r11 - __uint_as_float(b11 & 0xffff0000u));
            hi[q] = (u0 >> 16) | (u1 & 0xffff0000u);
            mid[q] = (b10 >> 16) | (b11 & 0xffff0000u);
            lo[q] = (b20 >> 16) | (b21 & 0xffff0000u);
        }
        return;
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        uint32_t h0, m0, l0, h1, m1, l1;
        split3(v[2 * q], h0, m0, l0);
        split3(v[2 * q + 1], h1, m1, l1);
        hi[q] = h0 | (h1 << 16);
        mid[q] = m0 | (m1 << 16);
        lo[q] = l0 | (l1 << 16);
    }
}

// Eight values: two halves of four.
__device__ __forceinline__ void split8(const float *v, u32x4 &hi, u32x4 &mid, u32x4 &lo) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t hq[2], mq[2], lq[2];
        split4(v + 4 * h, hq, mq, lq);
        hi[2 * h] = hq[0], hi[2 * h + 1] = hq[1];
        mid[2 * h] = mq[0], mid[2 * h + 1] = mq[1];
        lo[2 * h] = lq[0], lo[2 * h + 1] = lq[1];
    }
}

// The reference chain for one output: fmaf over ascending k from +0 (K a
// multiple of 8, rows 16-byte aligned).
__device__ float reference_chain(const uint16_t *__restrict__ w, const float *__restrict__ x, int K) {
    float acc = 0.0f;
    for (int k = 0; k < K; k += 8) {
        const u32x4 wv = *reinterpret_cast<const u32x4 *>(w + k);
        const float4 xa = *reinterpret_cast<const float4 *>(x + k);
        const float4 xb = *reinterpret_cast<const float4 *>(x + k + 4);
        const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const uint32_t bits = e & 1 ? wv[e >> 1] & 0xffff0000u : wv[e >> 1] << 16;
            acc = fmaf(xv[e], __uint_as_float(bits), acc);
        }
    }
    return acc;
}

// Tiny activation rows.  split3 is exact for |x| >= 2^-110: below that the
// third term falls under bf16's least subnormal (2^-133) and x loses its low
// bits.  That matters only when a whole activation row is that small -- then
// every product loses up to 2^-133 / |x| of itself (a row of |x| ~ 1e-37
// would be off by ~2^-10) -- while in a row with larger entries the lost
// bits are below 2^-33 of the largest one.  So each MFMA kernel keeps, per
// lane, the largest bf16 magnitude of the hi terms it split (hi keeps the
// order of |x| against 2^-100, and is nonzero for every nonzero x), takes
// the maximum per activation row over its workgroup's k range, and gives a
// row whose maximum is nonzero but below 2^-100 (bf16 0x0d80) the reference
// chain over that k range instead of its MFMA sums: bit for bit the
// reference's value when k is not split, else the slice's part of it.  Rare
// path: no real activation row is this small.
constexpr uint32_t kTinyHiBits = 0x0d80u;

__device__ __forceinline__ uint32_t hi_max(uint32_t mx) { return max(mx & 0xffffu, mx >> 16); }
__device__ __forceinline__ bool tiny_row(uint32_t mx) { return mx != 0 && mx < kTinyHiBits; }

// Wave-uniform: does the row hold an element other than +-0?  (bytes: 16 * n16)
__device__ bool wave_row_nonzero(const void *row, int n16, uint32_t mask) {
    const u32x4 *p = reinterpret_cast<const u32x4 *>(row);
    uint32_t acc = 0;
    for (int c = threadIdx.x & 63; c < n16; c += 64) {
        const u32x4 v = p[c];
        acc |= (v[0] | v[1] | v[2] | v[3]) & mask;
    }
    return __builtin_amdgcn_ballot_w64(acc != 0) != 0;
}

// One wave's outputs after the zero rule above.  Lane l holds s[t][r] for
// weight row base[t] + 4(l/16) + r of W and activation row m of X; `live`
// marks the ones it stores.  All 64 lanes call this; the rows are walked
// wave-uniformly.  Rare path: entered only when some output is exactly zero.
// The rows16 and wide layouts' rule: +0 where the activation row or the weight row
// holds only +-0, else the chain, always.  Their outputs are a few per wave and
// the scans stay in the kernel (out of it, as in settle_zeros, [102144,1024] at
// 3 activation rows took 38.0 us for 36.3).
template <int T>
__device__ void settle_tile_zeros(f32x4 (&s)[T], const bool (&live)[T][4], const int (&base)[T], const uint16_t *W,
                             const float *X, int K, int m) {
    const int g = (threadIdx.x & 63) >> 4;
    bool zero[T][4];
    bool any = false;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            zero[t][r] = live[t][r] && s[t][r] == 0.0f;
            any |= zero[t][r];
        }
    if (__builtin_amdgcn_ballot_w64(any) == 0) return;
    // Is this lane's activation row nonzero?  Lanes j = 0..15 hold every row
    // the wave has.
    bool xnz = false;
    for (int j = 0; j < 16; ++j) {
        const int mj = __builtin_amdgcn_readlane(m, j);
        if (__builtin_amdgcn_ballot_w64(any && m == mj) != 0) {
            const bool nz = wave_row_nonzero(X + (int64_t)mj * K, K / 4, 0x7fffffffu);
            if (m == mj) xnz = nz;
        }
    }
    // Zero outputs become +0, or the chain's value where both rows are nonzero.
    bool chain[T][4];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            chain[t][r] = false;
            if (zero[t][r]) s[t][r] = 0.0f;
            for (int gq = 0; gq < 4; ++gq) {
                const bool ask = zero[t][r] && xnz && g == gq;
                if (__builtin_amdgcn_ballot_w64(ask) == 0) continue;
                const int row = base[t] + 4 * gq + r;
                const bool nz = wave_row_nonzero(W + (int64_t)row * K, K / 8, 0x7fff7fffu);
                if (ask) chain[t][r] = nz;
            }
        }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            s[t][r] = few_or_lane_chains(chain[t][r], s[t][r], W + (int64_t)(base[t] + 4 * g + r) * K,
                                         X + (int64_t)m * K, K);
}

// Weight and x tiles in LDS hold rows of 128 bytes, 8 pieces of 16, back to
// back, with piece p of row r stored at position p ^ ((r / 2) mod 8).  A
// tile is written 8 rows x 128 bytes per instruction (each pair of rows then
// covers the 64 banks once) and read 16 rows x one piece (the rows' pieces
// land on 16 different groups of 4 banks).  The earlier 144-byte pitch kept
// the reads apart but let each pair of rows written together meet on 4 banks
// (11-24% of the MFMA kernels' LDS cycles lost to conflicts).
__device__ __forceinline__ int swz(int r, int p) { return r * 128 + ((p ^ ((r >> 1) & 7)) << 4); }

// Chunk order of the MFMA layouts.  A workgroup streams its weight rows
// one 128-byte column of lines (64 k) at a time; with every workgroup at
// the same k the whole device reads addresses that differ only above the
// row pitch, which for power-of-two rows (K = 4096: 8 KiB) meets a few HBM
// channels at a time.  Workgroup b therefore starts at chunk 5b mod n and
// wraps: on C4's W [128256, 4096] the read pattern alone streams in 150 us
// rotated against 178 in step (a plain read of the same bytes: 145).  The
// MFMA sums are taken in that order; the zero rule and the tiny-row chains
// recompute in k order, so only rounding inside the bound changes.
__device__ __forceinline__ int chunk_rotation(uint32_t b, int n) {
    return n > 0 ? (int)((b * 5u) % (uint32_t)n) : 0;
}
__device__ __forceinline__ int rotate_chunk(int c, int s0, int n) { return c + s0 >= n ? c + s0 - n : c + s0; }

// ---- host helpers of the launch planners -----------------------------------------

bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

int env_int(const char *name, int dflt) {
    const char *v = getenv(name);
    return (v && *v) ? atoi(v) : dflt;
}

}  // namespace
}  // namespace dmc
