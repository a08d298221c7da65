// gemm_kernels.hip -- the MFMA "gemm" layout: bf16 weights against several to
// thousands of f32 activation rows (prefill and large decode batches).
#include "gemv_device.h"
#include "gemv_launch.h"

#include <algorithm>
#include <type_traits>

namespace dmc {
namespace {

// A workgroup of NWV waves owns 32 * NWV weight rows against MT activation
// rows, so W streams from HBM once per MT rows (the 16-row layouts stream it
// once per 16).  k advances in chunks of 64: each weight row's chunk is one
// 128-byte line.  x enters as three bf16 terms (split3), either split by the
// workgroup on the way into LDS (FUSE) or once per call by
// split_x_planes_kernel into planes XS [3][M][K].
//
// What bounds it: from MT = 64 the matrix cores (3 MFMAs per product), whose
// clock falls under load (operands that are not zero run this MFMA at 1.94
// PFLOP/s out of registers, 2.4 with zeros), below that HBM.  Every wave
// taking its LDS reads, its MFMAs, its stores and a barrier in turn left the
// matrix cores ~30% busy, since the eight waves do each phase together.  So
// the operands of the next step are read from LDS while this step's MFMAs
// run, across the barrier too:
//   - a chunk is NS steps of (k-block of 32, 16 activation rows): RN MFMA
//     tiles x 3 terms, 12 to 24 MFMAs, against 3 to 7 operand reads for the
//     step after it in a second register set;
//   - one barrier per chunk, ahead of its last step: the chunk after next's
//     loads were stored to the other LDS buffer the step before, and the last
//     step's operands are already in registers, so its MFMAs cover the
//     barrier and the next chunk's first reads;
//   - the WN x WM grid of waves gives each a near-square tile (64 rows x MT/2),
//     7 to 10 operand reads per 24 MFMAs; W is shared through LDS like x;
//   - loads are unconditional and the chunk loop has no exit in its body, so
//     the compiler counts them instead of draining them (a `break` between
//     two chunks cost 5-10%).
// Measured, before (operand reads, MFMAs, stores and a barrier in turn; 64
// rows at most) / now, us, same box: C2 up m = 512 235 / 164, C2 down m = 2048
// 911 / 602 (1.2 PFLOP/s of MFMA; a large bf16 matrix product through the
// vendor library reaches 1.25 on this card), up m = 64 47.2 / 38.3.
//
// Where W lies (SRC): packed rows [N,K], K a multiple of 64, 16-byte aligned
// (kSrcPacked); rows [N,K] of any length and alignment (kSrcRows); columns, W [K,N]
// (kSrcCols).  Only the way of a chunk into the weight tile differs:
//   - kSrcRows reads the same 16-byte pieces at the rows' own 2-byte alignment
//     (exact on gfx950, checked per dword), and clears what lies past K in the
//     last chunk, in W (the next row's start, which may be an inf) and in x;
//   - kSrcCols reads 8 k rows of 512 bytes per wave, 4 columns per lane, and turns
//     each lane's 8 x 4 block with 16 byte permutes into 4 pieces of 8 k.
// A dword that runs past the matrix reads as zeros, and with K (kSrcCols: N) odd
// the matrix's last element shares one: it is read alone and put in.
//
// The kSrcRows and kSrcCols forms replace FMA kernels whose sums are spread over many
// lanes, 3 to 7 times closer to the exact value than one MFMA chain over all of
// k (each MFMA rounds the running sum; measured, K = 4096: 1.1e-7 against
// 7e-7).  They keep that: every k-block of 32 is summed from zero (lo, mid, hi:
// one rounding at full size), the blocks are added up in f32, and those sums
// once more every `fold` chunks, these and the k slices with the rounding
// errors of their sums kept.  And they keep x's 24 bits where three bf16 terms
// do not, |x| < 2^-110: a tile that holds such elements is streamed once more for
// what the terms left (kRest).
//
// When the tiles would leave the device short of workgroups, k is split over
// `slices` workgroups of kc chunks each, whose partial sums go to
// P[slice][m][n] for gemm_sum_slices_kernel.  Special values, tiny activation
// rows and the zero rule are as in the other MFMA layouts; with slices the
// zero rule runs after the sum.
typedef f32x4 f32x4_u __attribute__((aligned(4)));  // y's rows may start at any float
constexpr uint32_t kDeadLane = 0x80000000u;   // lane offset past every buffer: zeros, no traffic
enum Src { kSrcPacked, kSrcRows, kSrcCols };
constexpr uint32_t kDeadChunk = 0x7fff0000u;  // scalar offset of a chunk past the last (no 32-bit wrap with kDeadLane)

// The three bf16 terms of eight values by truncation alone: split3's terms for
// every finite |x| >= 2^-133 and 0.  Of a smaller x nothing is left, which
// matters where the row is not large either (tiny rows, settled after the
// stream) and where its larger elements meet weights of 0 or the small ones
// large weights: `cut` collects, in its low half, whether any element had more
// than the terms hold (kRest below).  An inf leaves a NaN in mid: settled after
// the stream too.
__device__ __forceinline__ void split8_finite(const float (&v)[8], u32x4 (&t)[3], uint32_t &cut) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t u0 = __float_as_uint(v[2 * q]), u1 = __float_as_uint(v[2 * q + 1]);
        const float r10 = v[2 * q] - __uint_as_float(u0 & 0xffff0000u);
        const float r11 = v[2 * q + 1] - __uint_as_float(u1 & 0xffff0000u);
        const uint32_t b10 = __float_as_uint(r10), b11 = __float_as_uint(r11);
        const uint32_t b20 = __float_as_uint(r10 - __uint_as_float(b10 & 0xffff0000u));
        const uint32_t b21 = __float_as_uint(r11 - __uint_as_float(b11 & 0xffff0000u));
        t[0][q] = (u0 >> 16) | (u1 & 0xffff0000u);
        t[1][q] = (b10 >> 16) | (b11 & 0xffff0000u);
        t[2][q] = (b20 >> 16) | (b21 & 0xffff0000u);
        cut |= b20 | b21;
    }
}

// What three terms leave of eight values, times 2^64: nothing of |x| >= 2^-110,
// else a multiple of 2^-85 under 2^-69, 16 bits, which two terms hold exactly.
__device__ __forceinline__ void split8_rest(const float (&v)[8], u32x4 (&t)[3]) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t h[2], m[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            float r = v[2 * q + e];
            const bool fin = (__float_as_uint(r) & 0x7f800000u) != 0x7f800000u;
#pragma unroll
            for (int i = 0; i < 3; ++i) r -= __uint_as_float(__float_as_uint(r) & 0xffff0000u);
            r = fin ? r * 0x1p64f : 0.0f;
            h[e] = __float_as_uint(r) & 0xffff0000u;
            m[e] = __float_as_uint(r - __uint_as_float(h[e]));
        }
        t[0][q] = (h[0] >> 16) | h[1];
        t[1][q] = (m[0] >> 16) | (m[1] & 0xffff0000u);
    }
}

// The weight tile's swizzle for columns: a lane's pieces go to rows 4 apart
// there (swz spreads rows 1 apart), so row bit 4 takes part too.
__device__ __forceinline__ int swz_cols(int r, int p) {
    return r * 128 + ((p ^ (((r >> 1) ^ (r >> 4 & 1)) & 7)) << 4);
}

// s += p, and what the rounding of that sum lost.
__device__ __forceinline__ float add_exact(float &s, float p) {
    const float t = s + p, b = t - s;
    const float e = (s - (t - b)) + (p - b);
    s = t;
    return e;
}
// (Sums that are not finite have no meaningful loss, and without one a sum keeps its bits, a -0 too.)
__device__ __forceinline__ float add_lost(float s, float e) {
    return fabsf(s) < __builtin_inff() && fabsf(e) > 0.0f ? s + e : s;
}

// Passes over the tile: the products (three terms), what the terms leave of x
// (two, times 2^64), and the hi term alone (the classes of what is not finite).
constexpr int kAll = 3, kRest = 2, kHi = 1;

template <int NWV, int MT, int SRC, bool FUSE>
__global__ void __launch_bounds__(64 * NWV) __attribute__((amdgpu_waves_per_eu(MT == 16 && SRC == kSrcPacked ? 4 : 2)))
gemv_mfma_gemm_kernel(const uint16_t *__restrict__ W, const float *__restrict__ X, const uint16_t *__restrict__ XS,
                      float *__restrict__ Y, float *__restrict__ P, int N, int K, int M, int kc, int gx, int gy,
                      int xcd, int64_t w_batch, int64_t x_batch) {
    static_assert(NWV == 4 || NWV == 8, "32 weight rows per wave");
    static_assert(SRC == kSrcPacked || (NWV == 8 && FUSE), "the general forms split x themselves, on 8 waves");
    static_assert(SRC == kSrcPacked || MT <= 64, "register budget");
    constexpr bool kTwoLevel = SRC != kSrcPacked;
    static_assert(MT == 16 || MT == 32 || MT == 64 || MT == 128, "activation rows per workgroup");
    constexpr int kRows = 32 * NWV;
    constexpr int XT = MT / 16;                    // 16-row activation tiles
    constexpr int WM = MT >= 64 ? 2 : (MT == 32 && NWV == 8) ? 2 : 1, WN = NWV / WM;
    constexpr int RN = kRows / 16 / WN, RM = XT / WM;  // MFMA tiles per wave
    constexpr int NS = 2 * RM;                     // steps per chunk
    constexpr int XI = (2 * XT + NWV - 1) / NWV;   // x staging items (16 rows x 32 k) per wave
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i16 = lane & 15;
    const int g = lane >> 4;
    const int wn = wave % WN, wm = wave / WN;
    // The tile from the linear workgroup id (a 1-D grid of gx * gy * slices).
    // With `xcd` set, workgroup L, which runs on XCD L % 8 (the dispatcher
    // deals workgroups to the 8 XCDs in turn), takes the L / 8-th tile of
    // that XCD's contiguous share, activation tiles fastest, so the
    // workgroups an XCD runs together share weight blocks through its L2;
    // otherwise tiles go in launch order, consecutive weight blocks to
    // different XCDs.
    uint32_t lin = blockIdx.x;
    if (xcd) {
        const uint32_t x = lin & 7u, q = gridDim.x >> 3, r = gridDim.x & 7u;
        lin = x * q + min(x, r) + (lin >> 3);
    }
    const int by = (int)(lin % (uint32_t)gy);
    const int bx = (int)(lin / (uint32_t)gy % (uint32_t)gx);
    const int bz = (int)(lin / (uint32_t)gy / (uint32_t)gx);
    const int row0 = bx * kRows;
    const int nrows = min(kRows, N - row0);
    const int m0 = by * MT;
    const int c0 = bz * kc;  // this slice's chunks: [c0, c0 + nch)
    const int nck = SRC == kSrcPacked ? K / 64 : (K + 63) / 64;  // chunks of k in all
    const int nch = max(0, min(nck, c0 + kc) - c0);
    if (SRC == kSrcCols) {  // batch slice blockIdx.y (P: [z][slice][m][n])
        W += blockIdx.y * w_batch;
        X += blockIdx.y * x_batch;
        Y += (int64_t)blockIdx.y * M * N;
        if (P) P += (int64_t)blockIdx.y * (gridDim.x / (uint32_t)(gx * gy)) * M * N;
    }
    const int64_t wstep = SRC == kSrcCols ? N : 1;                      // elements between a weight row's k
    const uint16_t *const wrow0 = SRC == kSrcCols ? W + row0 : W + (int64_t)row0 * K;
    const int64_t wpitch = SRC == kSrcCols ? 1 : K;                     // ... and between weight rows
    auto tile_at = [](int r, int p) { return SRC == kSrcCols ? swz_cols(r, p) : swz(r, p); };

    __shared__ __attribute__((aligned(16))) uint8_t wt[2][kRows * 128];  // swizzled 128-byte rows (swz)
    __shared__ u32x4 xp[2][XT][2][3][64];                                // operand order: conflict-free

    // kSrcRows: up to 16 bytes of the row after the block, so that only the matrix's own end cuts a dword.
    const __amdgpu_buffer_rsrc_t rs =
        SRC == kSrcCols   ? weight_rsrc(W, (uint32_t)((int64_t)K * N * 2))
        : SRC == kSrcRows ? weight_rsrc(wrow0, (uint32_t)min((int64_t)nrows * K * 2 + 16, (int64_t)(N - row0) * K * 2))
                       : weight_rsrc(wrow0, (uint32_t)((int64_t)nrows * K * 2));
    const uint32_t plane_bytes = (uint32_t)M * (uint32_t)K * 2u;
    const __amdgpu_buffer_rsrc_t xrs = FUSE ? weight_rsrc(X, 2u * plane_bytes) : weight_rsrc(XS, 3u * plane_bytes);
    // W staging: item j of a wave is rows 32 * wave + 8j + lane/8, 16 bytes per lane: whole lines
    // (kSrcCols: k rows 8 * wave + 2j and + 1, columns 4 * lane of each).
    const int slr = wave * 32 + (lane >> 3);
    uint32_t woff[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        woff[j] = SRC == kSrcCols ? (uint32_t)(row0 + 4 * lane) * 2u
                               : (uint32_t)min(slr + 8 * j, nrows - 1) * (uint32_t)K * 2u + (lane & 7) * 16;
    const uint32_t wlast = SRC == kSrcPacked ? 0 : W[(int64_t)N * K - 1];  // the matrix's last element
    // x staging: item it = (tile it/2, k-block it%2), 8 elements of row i16 per lane.
    uint32_t xoff[XI];
#pragma unroll
    for (int j = 0; j < XI; ++j) {
        const int it = wave * XI + j;
        const int xm = m0 + (it >> 1) * 16 + i16;
        const uint32_t e = (uint32_t)xm * (uint32_t)K + (it & 1) * 32 + g * 8;
        xoff[j] = it < 2 * XT && xm < M ? e * (FUSE ? 4u : 2u) : kDeadLane;
    }
    struct Regs {
        u32x4 w[4];
        u32x4 x[XI][FUSE ? 2 : 3];  // f32 halves, or the three planes
    };
    const int s0 = chunk_rotation(bx, nch);
    auto load = [&](int c, Regs &r) __attribute__((always_inline)) {
        const bool live = c < nch;
        const uint32_t cb = (uint32_t)(c0 + rotate_chunk(c, s0, nch)) * 128u;
        const uint32_t wb = live ? cb : kDeadChunk;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (SRC == kSrcCols) {
                const uint32_t k = (uint32_t)(c0 + rotate_chunk(c, s0, nch)) * 64u + wave * 8 + 2 * j;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const auto v = __builtin_amdgcn_raw_buffer_load_b64(
                        rs, woff[j], live ? (k + h) * (uint32_t)N * 2u : kDeadChunk, kLoadNT);
                    r.w[j][2 * h] = v[0];
                    r.w[j][2 * h + 1] = v[1];
                }
            } else {
                // (kSrcRows: not nontemporal, since a row's chunk spans two lines, each half another chunk's.)
                r.w[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, woff[j], wb, SRC == kSrcRows ? 0 : kLoadNT);
            }
        }
#pragma unroll
        for (int j = 0; j < XI; ++j) {
#pragma unroll
            for (int q = 0; q < (FUSE ? 2 : 3); ++q)
                r.x[j][q] = FUSE ? __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[j] + 16u * q,
                                                                         live ? 2u * cb : kDeadChunk, 0)
                                 : __builtin_amdgcn_raw_buffer_load_b128(xrs, xoff[j],
                                                                         live ? q * plane_bytes + cb : kDeadChunk, 0);
        }
    };
    uint32_t xmx[XI];  // the largest |x| staged (f32 bits; the hi term's with planes), per lane
#pragma unroll
    for (int j = 0; j < XI; ++j) xmx[j] = 0;
    uint32_t cut = 0;
    // Chunk c's staged registers into LDS buffer `buf`.
    auto store = [&](Regs &r, int c, int buf, auto TERMS) __attribute__((always_inline)) {
        constexpr int terms = decltype(TERMS)::value;
        if constexpr (SRC != kSrcPacked) {
            const int at = c < nch ? c0 + rotate_chunk(c, s0, nch) : -1;
            if (at == nck - 1) {  // the last chunk of k: wave-uniform, one in nck
                int kt = K - 64 * at;  // its elements
                asm volatile("" : "+s"(kt));  // keep the masks below out of the loop's registers
                if constexpr (SRC == kSrcRows) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int left = kt - (lane & 7) * 8;  // of this piece
                        const bool end = (K & 1) && row0 + slr + 8 * j == N - 1 && left >= 1 && left <= 8;
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            if (end && (left - 1) >> 1 == v) r.w[j][v] = wlast;
                            r.w[j][v] &= (2 * v < left ? 0xffffu : 0u) | (2 * v + 1 < left ? 0xffff0000u : 0u);
                        }
                    }
                } else if (N & 1) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                            if (wave * 8 + 2 * j + (v >> 1) == kt - 1 && row0 + 4 * lane + 2 * (v & 1) == N - 1)
                                r.w[j][v] = wlast;
                }
#pragma unroll
                for (int j = 0; j < XI; ++j) {
                    const int left = kt - ((wave * XI + j) & 1) * 32 - g * 8;
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (e >= left) r.x[j][e >> 2][e & 3] = 0;
                }
            }
        }
        if constexpr (SRC == kSrcCols) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {  // column 4 * lane + e: this wave's 8 k, two per dword
                u32x4 piece;
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    piece[v] = __builtin_amdgcn_perm(r.w[v][2 + (e >> 1)], r.w[v][e >> 1],
                                                     e & 1 ? 0x07060302u : 0x05040100u);
                *reinterpret_cast<u32x4 *>(wt[buf] + tile_at(4 * lane + e, wave)) = piece;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4 *>(wt[buf] + tile_at(slr + 8 * j, lane & 7)) = r.w[j];
        }
#pragma unroll
        for (int j = 0; j < XI; ++j) {
            const int it = wave * XI + j;
            if (it >= 2 * XT) break;  // wave-uniform
            u32x4 t[3];
            if constexpr (FUSE) {
                float v[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[e] = __uint_as_float(r.x[j][0][e]);
                    v[4 + e] = __uint_as_float(r.x[j][1][e]);
                }
                if constexpr (terms == kHi) {
                    split8(v, t[0], t[1], t[2]);
                } else if constexpr (terms == kRest) {
                    split8_rest(v, t);
                } else {
                    split8_finite(v, t, cut);
#pragma unroll
                    for (int e = 0; e < 8; ++e) xmx[j] = max(xmx[j], __float_as_uint(v[e]) & 0x7fffffffu);
                }
            } else {
#pragma unroll
                for (int q = 0; q < 3; ++q) t[q] = r.x[j][q];
                if constexpr (terms == kAll) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) xmx[j] = max_mag(xmx[j], t[0][e]);
                }
            }
#pragma unroll
            for (int q = 0; q < terms; ++q) xp[buf][it >> 1][it & 1][q][lane] = t[q];
        }
    };

    f32x4 acc[RM][RN];
    // kTwoLevel: the sums of all (with their rounding errors) and of the
    // current `fold` chunks.
    float total[kTwoLevel ? RM : 1][RN][4], lost[kTwoLevel ? RM : 1][RN][4], part[kTwoLevel ? RM : 1][RN][4];
    const int fold = kTwoLevel ? max(1, (int)(0.5f * sqrtf(2.0f * nch) + 0.5f)) : 0;
    u32x4 a[2][RN], xo[2][3];  // operands: weights per k-block, x per step
    auto read_a = [&](int buf, int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < RN; ++j)
            a[kb][j] = *reinterpret_cast<const u32x4 *>(wt[buf] + tile_at((wn * RN + j) * 16 + i16, kb * 4 + g));
    };
    auto read_x = [&](int buf, int kb, int mf, int set) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 3; ++q) xo[set][q] = xp[buf][wm * RM + mf][kb][q][lane];
    };
    // LDS only: the global loads in flight stay in flight.
    auto lds_barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    // Chunk c is in LDS buffer BUF and its first step's operands in registers;
    // chunk c + 1 is in `r`, loaded a chunk ago.
    Regs r;
    auto chunk = [&](int c, auto BUF, auto TERMS, auto AT) __attribute__((always_inline)) {
        constexpr int buf = decltype(BUF)::value;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int kb = s / RM, mf = s % RM;
            if (s + 1 < NS) {
                if ((s + 1) % RM == 0) read_a(buf, (s + 1) / RM);
                read_x(buf, (s + 1) / RM, (s + 1) % RM, (s + 1) & 1);
            }
            if (s == decltype(AT)::value) {
                store(r, c + 1, buf ^ 1, TERMS);
                load(c + 2, r);
            }
            if (s == NS - 1) {
                lds_barrier();
                read_a(buf ^ 1, 0);
                read_x(buf ^ 1, 0, 0, 0);
            }
            constexpr int terms = decltype(TERMS)::value;
            if constexpr (kTwoLevel) {
                f32x4 blk[RN];
#pragma unroll
                for (int j = 0; j < RN; ++j) blk[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int q = terms - 1; q >= 0; --q)
#pragma unroll
                    for (int j = 0; j < RN; ++j) blk[j] = mfma_bf16(a[kb][j], xo[s & 1][q], blk[j]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < RN; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        part[mf][j][v] += blk[j][v];
                        asm volatile("" : "+v"(part[mf][j][v]));  // here, not after the chunk (registers)
                    }
            } else {
#pragma unroll
                for (int q = 0; q < terms; ++q)
#pragma unroll
                    for (int j = 0; j < RN; ++j) acc[mf][j] = mfma_bf16(a[kb][j], xo[s & 1][q], acc[mf][j]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto fold_parts = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    lost[i][j][v] += add_exact(total[i][j][v], part[i][j][v]);
                    part[i][j][v] = 0.0f;
                }
    };
    auto stream = [&](auto TERMS, auto AT) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j) {
                if constexpr (kTwoLevel) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) total[i][j][v] = lost[i][j][v] = part[i][j][v] = 0.0f;
                } else {
                    acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                }
            }
        load(0, r);
        store(r, 0, 0, TERMS);
        load(1, r);
        lds_barrier();
        read_a(0, 0);
        read_x(0, 0, 0, 0);
        int c = 0;
        int until = fold;
        for (; c + 1 < nch; c += 2) {
            chunk(c, std::integral_constant<int, 0>{}, TERMS, AT);
            chunk(c + 1, std::integral_constant<int, 1>{}, TERMS, AT);
            if constexpr (kTwoLevel) {
                if (c + 2 >= until) {
                    fold_parts();
                    until = c + 2 + fold;
                }
            }
        }
        if (c < nch) chunk(c, std::integral_constant<int, 0>{}, TERMS, AT);
        if constexpr (kTwoLevel) {
            fold_parts();
#pragma unroll
            for (int i = 0; i < RM; ++i)
#pragma unroll
                for (int j = 0; j < RN; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[i][j][v] = add_lost(total[i][j][v], lost[i][j][v]);
        }
    };
    // The pass over what the terms left of x, rare: one LDS buffer and one set of
    // operands (registers), the next chunk's loads under this one's MFMAs.
    auto stream_rest = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) total[i][j][v] = lost[i][j][v] = part[i][j][v] = 0.0f;
        load(0, r);
        int until = fold;
#pragma nounroll
        for (int c = 0; c < nch; ++c) {
            lds_barrier();  // every wave is done with the buffer
            store(r, c, 0, std::integral_constant<int, kRest>{});
            load(c + 1, r);
            lds_barrier();
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                read_a(0, kb);
#pragma unroll
                for (int mf = 0; mf < RM; ++mf) {
                    read_x(0, kb, mf, 0);
                    f32x4 blk[RN];
#pragma unroll
                    for (int j = 0; j < RN; ++j) {
                        blk[j] = mfma_bf16(a[kb][j], xo[0][1], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
                        blk[j] = mfma_bf16(a[kb][j], xo[0][0], blk[j]);
                    }
#pragma unroll
                    for (int j = 0; j < RN; ++j)
#pragma unroll
                        for (int v = 0; v < 4; ++v) part[mf][j][v] += blk[j][v];
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if (c + 1 >= until) {
                fold_parts();
                until = c + 1 + fold;
            }
        }
        fold_parts();
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
            for (int j = 0; j < RN; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[i][j][v] = add_lost(total[i][j][v], lost[i][j][v]);
    };
    // Waves w and w + 4 share a SIMD: they stage (split or transpose, store) in
    // different steps, so that one's vector work runs under the other's MFMAs.
    // Same box, in the same step / staggered, us: C2 up m = 512 168 / 164, down
    // m = 2048 604 / 581, columns up m = 64 47.5 / 44.0; packed 64-row tiles
    // lose 2% where a slice has few chunks (C2 up m = 64 40.2 / 40.7).
    constexpr bool kStagger = MT == 128 || (SRC == kSrcCols && MT == 64);
    if (!kStagger || wave >= 4) stream(std::integral_constant<int, kAll>{}, std::integral_constant<int, NS - 2>{});
    else stream(std::integral_constant<int, kAll>{}, std::integral_constant<int, 0>{});

    float *const out = (P ? P + (int64_t)bz * M * N : Y) + row0;
    // The activation rows' largest magnitudes (this slice's k), in LDS bytes
    // that the stream is done with, and whether the terms left some of x.
    uint32_t *const xmax_s = reinterpret_cast<uint32_t *>(&xp[0][0][0][0][0]);
    uint32_t *const any_s = xmax_s + MT;
    auto row_maxima = [&]() __attribute__((always_inline)) {
        __syncthreads();
        for (int i = tid; i <= MT; i += 64 * NWV) xmax_s[i] = 0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < XI; ++j) {
            const int it = wave * XI + j;
            if (it < 2 * XT) atomicMax(&xmax_s[(it >> 1) * 16 + i16], FUSE ? xmx[j] : hi_max(xmx[j]) << 16);
        }
        if (kTwoLevel && (cut & 0xffffu) != 0) *any_s = 1;
        __syncthreads();
    };
    row_maxima();
    if constexpr (kTwoLevel) {
        // Rare: the tile is streamed once more for what the terms left of x, so
        // that these forms keep the 24 bits that the f32 FMA kernels keep.  With
        // and without such elements (the FMA kernels the same), us: columns
        // [4096,14336] m = 5 / 17 / 64 50 / 66 / 100 against 27.7 / 34.2 / 45.0
        // (61 / 172 / 3680), [11008,4097] m = 3 / 33 42 / 75 against 21.3 / 35.5
        // (48 / 494).
        if (*any_s != 0) {
            auto each = [&](auto body) __attribute__((always_inline)) {
#pragma unroll
                for (int f = 0; f < RM * RN * 4; ++f) {
                    const int mf = f / (RN * 4), j = f / 4 % RN, n = (wn * RN + j) * 16 + g * 4 + f % 4;
                    const int ml = (wm * RM + mf) * 16 + i16;
                    if (m0 + ml < M && n < nrows)
                        acc[mf][j][f % 4] = body(out[(int64_t)(m0 + ml) * N + n], acc[mf][j][f % 4]);
                }
            };
            each([](float &o, float v) { return o = v; });
            __syncthreads();
            stream_rest();
            each([](float &o, float v) {
                return fabsf(v) < __builtin_inff() && v != 0.0f ? o + v * 0x1p-64f : o;
            });
            cut = 0;
            row_maxima();
        }
    }
    // Outputs: lane l holds weight rows 4(l/16) + v of a tile, activation row
    // l%16.  They are stored as they are; the rare ones that the sums do not
    // settle (a tiny row, an exact zero, a value that is not finite) are redone.
    bool rare = false, big = false;  // big: some output is not finite
#pragma unroll
    for (int mf = 0; mf < RM; ++mf) {
        const int ml = (wm * RM + mf) * 16 + i16;
        if (m0 + ml >= M) continue;
        rare |= xmax_s[ml] != 0 && xmax_s[ml] < kTinyHiBits << 16;
        float *const o = out + (int64_t)(m0 + ml) * N;
#pragma unroll
        for (int j = 0; j < RN; ++j) {
            const int n = (wn * RN + j) * 16 + g * 4;
            if ((N & 3) == 0) {
                if (n < nrows) *reinterpret_cast<f32x4_u *>(o + n) = acc[mf][j];
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (n + v < nrows) o[n + v] = acc[mf][j][v];
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                rare |= n + v < nrows && acc[mf][j][v] == 0.0f;
                big |= n + v < nrows && !(fabsf(acc[mf][j][v]) < __builtin_inff());
            }
        }
    }
    // The lane's outputs of `mask` (bit f, in the order above), some lane's at a
    // time: body(is it this lane's, activation row of the tile, address, w, x).
    auto each_output = [&](uint64_t mask, auto body) __attribute__((always_inline)) {
        if (__builtin_amdgcn_ballot_w64(mask != 0) == 0) return;
#pragma nounroll
        for (int f = 0; f < RM * RN * 4; ++f) {
            const bool mine = (mask >> f & 1) != 0;
            if (__builtin_amdgcn_ballot_w64(mine) == 0) continue;
            const int mf = f / (RN * 4), n = (wn * RN + f / 4 % RN) * 16 + g * 4 + f % 4;
            const int ml = (wm * RM + mf) * 16 + i16;
            body(mine, ml, out + (int64_t)(m0 + ml) * N + n, wrow0 + min(n, nrows - 1) * wpitch,
                 X + (int64_t)min(m0 + ml, M - 1) * K);
        }
    };
    // An exact zero that stands for the reference's +0: a k slice marks it -0,
    // which its sums never are, so that the sum over the slices is -0 exactly
    // where every slice says so.
    const float plus = P ? -0.0f : 0.0f;
    uint64_t zeros = 0;  // ... and those that are not settled yet
    if (__builtin_amdgcn_ballot_w64(rare) != 0) {
        uint64_t tiny = 0, none = 0;  // outputs of tiny activation rows; zeros of rows of +-0
#pragma unroll
        for (int f = 0; f < RM * RN * 4; ++f) {
            const int mf = f / (RN * 4), n = (wn * RN + f / 4 % RN) * 16 + g * 4 + f % 4;
            const int ml = (wm * RM + mf) * 16 + i16;
            const uint32_t xm = xmax_s[ml];
            const uint64_t bit = m0 + ml < M && n < nrows ? 1ull << f : 0;
            const bool zero = acc[mf][f / 4 % RN][f % 4] == 0.0f;
            if (xm == 0) none |= zero ? bit : 0;
            else if (xm < kTinyHiBits << 16) tiny |= bit;
            else zeros |= zero ? bit : 0;
        }
        each_output(none, [&](bool mine, int, float *o, const uint16_t *, const float *) {
            if (mine) *o = plus;
        });
        each_output(tiny, [&](bool mine, int, float *o, const uint16_t *wr, const float *xr) {
            if (mine)  // this slice's chain (+0.0f: no -0 that would be taken for the mark)
                *o = (SRC == kSrcPacked ? reference_chain(wr + 64 * c0, xr + 64 * c0, 64 * nch)
                                        : chain_strided(wr + 64 * c0 * wstep, wstep, xr + 64 * c0,
                                                        min(64 * nch, K - 64 * c0))) + (P ? 0.0f : -0.0f);
        });
    }
    uint32_t *const zeros_s = any_s + 1;
    if (tid == 0) *any_s = *zeros_s = 0;
    __syncthreads();
    if (big) *any_s = 1;
    if (zeros) atomicAdd(zeros_s, (uint32_t)__builtin_popcountll(zeros));
    __syncthreads();
    const bool again = *any_s != 0;
    const int open = (int)*zeros_s;
    __syncthreads();
    if (!again && open == 0) return;
    if (open != 0) {
        // Exact zeros, of weight rows or columns that hold only +-0 (padding,
        // pruning) or of products that cancel.  One pass over the tile takes the
        // range of its weights and of each activation row, which settles them
        // all (zero_is_plus), but for a tile whose weights or x reach down to
        // underflow or up to inf.  What is left, and a few zeros alone against
        // many chunks (a range of two rows takes 4 us, a chunk here about 0.5),
        // is settled one by one, by the sum over the slices if k is split.
        // Scanning rows and columns for each zero took longer than the product,
        // most so for columns, 2N bytes between elements; with 256 zero columns,
        // so / here (without them), us: columns [4096,14336] m = 5 / 64 1166 /
        // 1252 against 46 / 72 (27.7 / 45).
        const bool ranges = open * 8 > nch && K <= 1 << 24;
        Range w;
        uint32_t *const xlo_s = zeros_s + 1, *const w_s = xlo_s + MT;
        if (ranges) {
            constexpr int kSets = MT == 16 ? 2 : 4;
            for (int i = tid; i < MT; i += 64 * NWV) xlo_s[i] = ~0u;
            if (tid == 0) w_s[0] = ~0u, w_s[1] = 0;
            __syncthreads();
            uint32_t xlo[XI];
#pragma unroll
            for (int j = 0; j < XI; ++j) xlo[j] = ~0u;
            if (SRC != kSrcPacked) w.put(wlast & 0x7fffu);  // (cut by the matrix's end)
#pragma nounroll
            for (int c = 0; c < nch; c += kSets) {
                Regs q[kSets];
#pragma unroll
                for (int u = 0; u < kSets; ++u) load(c + u, q[u]);
#pragma unroll
                for (int u = 0; u < kSets; ++u) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            w.put(q[u].w[j][v] & 0x7fffu);
                            w.put(q[u].w[j][v] >> 16 & 0x7fffu);
                        }
#pragma unroll
                    for (int j = 0; j < XI; ++j)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const u32x4 *const x = q[u].x[j];
                            if constexpr (FUSE) {
                                xlo[j] = min(xlo[j], min((x[0][v] & 0x7fffffffu) - 1u, (x[1][v] & 0x7fffffffu) - 1u));
                            } else {  // the hi term has x's exponent
                                xlo[j] = min(xlo[j], min((x[0][v] << 16 & 0x7fffffffu) - 1u, (x[0][v] & 0x7fff0000u) - 1u));
                            }
                        }
                }
            }
            w.over_wave();
            if (lane == 0) {
                atomicMin(&w_s[0], w.lo1);
                atomicMax(&w_s[1], w.hi);
            }
#pragma unroll
            for (int j = 0; j < XI; ++j) {
                const int it = wave * XI + j;
                if (it < 2 * XT) atomicMin(&xlo_s[(it >> 1) * 16 + i16], xlo[j]);
            }
            __syncthreads();
            w.lo1 = w_s[0];
            w.hi = w_s[1];
        }
        if (ranges || !P)
            each_output(zeros, [&](bool mine, int ml, float *o, const uint16_t *wr, const float *xr) {
                Range x;
                x.lo1 = ranges ? xlo_s[ml] : 0u;
                x.hi = xmax_s[ml];
                const bool settled = ranges && zero_is_plus(x, w, K);
                if (mine && settled) *o = plus;
                const bool ask = !P && mine && !settled;
                if (__builtin_amdgcn_ballot_w64(ask) != 0) settle_zeros(o, ask ? 1u : 0u, xr, wr, 0, wstep, K);
            });
        __syncthreads();
    }
    if (!again) return;
    // Outputs that are not finite: a weight or an activation is inf or NaN
    // (then every output of its row is inf or NaN in the reference), or a sum
    // overflowed.  Their class may be wrong: mid and lo are 0 against an inf
    // weight (NaN where the reference has inf), and the split of an inf leaves
    // a NaN.  The hi term alone by split3's rule, nonzero for every nonzero x
    // and carrying its inf or NaN, has the reference's classes, so the tile is
    // streamed again with it and those outputs take its result where that is
    // not finite either.  (Screening W in the loop and clearing such weights
    // for mid and lo cost 12-18% of it, for weights that hold none.)
    stream(std::integral_constant<int, kHi>{}, std::integral_constant<int, NS - 2>{});
#pragma unroll
    for (int mf = 0; mf < RM; ++mf) {
        const int ml = (wm * RM + mf) * 16 + i16;
        if (m0 + ml >= M) continue;
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int n = (wn * RN + j) * 16 + g * 4 + v;
                float *const o = out + (int64_t)(m0 + ml) * N + n;
                if (n < nrows && !(fabsf(*o) < __builtin_inff()) && !(fabsf(acc[mf][j][v]) < __builtin_inff()))
                    *o = acc[mf][j][v];
            }
    }
}

// x [M,K] f32 -> its three bf16 terms as planes XS[q][M][K] (split3 of each
// element).  count = M*K, a multiple of 8; 16-byte aligned.  Grid-stride.
__global__ void __launch_bounds__(256)
split_x_planes_kernel(const float *__restrict__ X, uint16_t *__restrict__ XS, int64_t count) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count / 8; i += (int64_t)gridDim.x * 256) {
        const float4 a = reinterpret_cast<const float4 *>(X)[2 * i];
        const float4 b = reinterpret_cast<const float4 *>(X)[2 * i + 1];
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        u32x4 hi, md, lo;
        split8(v, hi, md, lo);
        reinterpret_cast<u32x4 *>(XS)[i] = hi;
        reinterpret_cast<u32x4 *>(XS + count)[i] = md;
        reinterpret_cast<u32x4 *>(XS + 2 * count)[i] = lo;
    }
}

// y[m][n] = P[0][m][n] + P[1][m][n] + ... in slice order.  A partial of -0 says
// that its slice's products sum to a zero that stands for the reference's +0: a
// sum of -0 is +0; any other zero sum is settled (settle_zeros).  Q outputs per
// thread (4 where N is a multiple of 4, so that they share an activation row):
// 16-byte loads, up to 8 slices' in flight: 74 registers, 6 waves per SIMD (at the
// 8 waves that the compiler prefers it holds fewer loads: 18 slices of columns
// [9872,1792] at 57 rows 7.8 us against 4.5).
// PACKED: W as in kSrcPacked, else rows (wstep 1) or columns (wstep N, batch slice
// blockIdx.y) of any size.
template <int Q, bool PACKED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6, 6)))
gemm_sum_slices_kernel(const float *__restrict__ P, int slices, float *__restrict__ Y, const uint16_t *__restrict__ W,
                       const float *__restrict__ X, int M, int N, int K, int64_t wstep, int64_t w_batch,
                       int64_t x_batch) {
    typedef float vec __attribute__((ext_vector_type(Q), aligned(4)));
    const int64_t count = (int64_t)M * N;
    if (!PACKED) {
        P += (int64_t)blockIdx.y * slices * count;
        Y += (int64_t)blockIdx.y * count;
        W += blockIdx.y * w_batch;
        X += blockIdx.y * x_batch;
    }
    const int64_t first = Q * ((int64_t)blockIdx.x * 256 + threadIdx.x), step = Q * (int64_t)gridDim.x * 256;
    bool zero = false;
    for (int64_t i = first; i < count; i += step) {
        vec s = *reinterpret_cast<const vec *>(P + i);
        float lost[Q] = {};  // !PACKED: what the sum's roundings lost
#pragma unroll 8
        for (int j = 1; j < slices; ++j) {
            const vec p = *reinterpret_cast<const vec *>(P + j * count + i);
            if (PACKED) {
                s += p;
            } else {
#pragma unroll
                for (int e = 0; e < Q; ++e) {
                    float t = s[e];
                    lost[e] += add_exact(t, p[e]);
                    s[e] = t;
                }
            }
        }
        if (!PACKED) {
#pragma unroll
            for (int e = 0; e < Q; ++e) s[e] = add_lost(s[e], lost[e]);
        }
#pragma unroll
        for (int e = 0; e < Q; ++e) {
            // -0: every slice marked its zero as settled; +0: open, marked -0 in Y meanwhile.
            const bool open = s[e] == 0.0f && !__builtin_signbit(s[e]);
            zero |= open;
            s[e] = s[e] == 0.0f ? (open ? -0.0f : 0.0f) : s[e];
        }
        *reinterpret_cast<vec *>(Y + i) = s;
    }
    // Rare: the wave settles its lanes' zeros together, over the outputs again.
    if (__builtin_amdgcn_ballot_w64(zero) == 0) return;
#pragma nounroll
    for (int64_t i = first; __builtin_amdgcn_ballot_w64(i < count) != 0; i += step) {
        const int64_t at = i < count ? i : 0;
        const vec s = *reinterpret_cast<const vec *>(Y + at);
        uint32_t zeros = 0;
#pragma unroll
        for (int e = 0; e < Q; ++e) zeros |= (i < count && s[e] == 0.0f && __builtin_signbit(s[e]) ? 1u : 0u) << e;
        const int64_t m = at / N, n = at - m * N;
        if (__builtin_amdgcn_ballot_w64(zeros != 0) != 0)
            settle_zeros(Y + at, zeros, X + m * K, W + n * (wstep == 1 ? K : 1), wstep == 1 ? K : 1, wstep, K);
    }
}

unsigned grid_for(int64_t blocks) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>(blocks, 4096)); }

}  // namespace

hipError_t launch_sum_slices(const float *part, int slices, const RdProblem &p, hipStream_t s) {
    const bool packed = p.k % 64 == 0 && aligned(p.w, 16) && aligned(p.x, 16);
#define DMC_SUM(Q, PK)                                                                                         \
    hipLaunchKernelGGL((gemm_sum_slices_kernel<Q, PK>), dim3(grid_for((p.m * p.n / Q + 255) / 256)), dim3(256), 0, s, \
                       part, slices, p.y, p.w, p.x, (int)p.m, (int)p.n, (int)p.k, (int64_t)1, (int64_t)0, (int64_t)0)
    if (p.n % 4 == 0 && packed) DMC_SUM(4, true);
    else if (p.n % 4 == 0) DMC_SUM(4, false);
    else if (packed) DMC_SUM(1, true);
    else DMC_SUM(1, false);
#undef DMC_SUM
    return hipGetLastError();
}

hipError_t launch_gemm(const RdProblem &p, const RdPlan &pl, void *workspace, hipStream_t s) {
    // The workspace holds x's planes (unless the kernel splits x itself) and
    // the slice partials (when k is split): a fused single-slice plan needs
    // none and may be given none.
    const bool needs_ws = !pl.xfuse || pl.kslices > 1;
    const int mt = pl.mt * pl.mtiles;
    const bool packed = pl.vec == 8 && p.k % 64 == 0;
    if ((needs_ws && !workspace) || pl.kslices < 1 || pl.kslices > 65535 ||
        (int64_t)pl.kslices * pl.kchunks < (p.k + 63) / 64 || pl.rpw != 32 * pl.waves || pl.grid_x * pl.rpw < p.n ||
        p.ldw != p.k || p.ldx != p.k || p.ldy != p.n || p.k < 1 || (int64_t)pl.rpw * p.k * 2 + 16 > INT32_MAX ||
        (packed ? !aligned(p.w, 16) || !aligned(p.x, 16)
                : !pl.xfuse || pl.waves != 8 || p.m * p.k * 4 > INT32_MAX || !aligned(p.w, 2) || !aligned(p.x, 4)))
        return hipErrorInvalidValue;
    uint16_t *xs = pl.xfuse ? nullptr : static_cast<uint16_t *>(workspace);
    const size_t planes = pl.xfuse ? 0 : ((size_t)3 * p.m * p.k * 2 + 255) / 256 * 256;
    float *part = pl.kslices > 1 ? reinterpret_cast<float *>(static_cast<char *>(workspace) + planes) : nullptr;
    const int64_t count = p.m * p.k;
    if (!pl.xfuse)
        hipLaunchKernelGGL(split_x_planes_kernel, dim3(grid_for((count / 8 + 255) / 256)), dim3(256), 0, s, p.x, xs,
                           count);
    const int64_t gy = (p.m + mt - 1) / mt;
    const int64_t wgs = pl.grid_x * gy * (int64_t)pl.kslices;
    if (wgs > INT32_MAX) return hipErrorInvalidValue;
    // The XCD-grouped tile order where activation tiles share weight
    // blocks (DMC_HIP_GEMM_XCD: 0 never, 2 always).
    const int xenv = env_int("DMC_HIP_GEMM_XCD", 1);
    const int xcd = xenv == 2 || (xenv == 1 && gy > 1) ? 1 : 0;
#define DMC_GEMM(NW, MT, SRC, F)                                                                              \
    if (pl.waves == NW && mt == MT && packed == (SRC == kSrcPacked) && pl.xfuse == F)                            \
        hipLaunchKernelGGL((gemv_mfma_gemm_kernel<NW, MT, SRC, F>), dim3((unsigned)wgs), dim3(64 * NW), 0, s, p.w, \
                           p.x, xs, p.y, part, (int)p.n, (int)p.k, (int)p.m, pl.kchunks, (int)pl.grid_x, (int)gy, \
                           xcd, (int64_t)0, (int64_t)0);                                                      \
    else
    DMC_GEMM(8, 16, kSrcPacked, true) DMC_GEMM(8, 16, kSrcPacked, false) DMC_GEMM(8, 32, kSrcPacked, true)
    DMC_GEMM(8, 32, kSrcPacked, false) DMC_GEMM(8, 64, kSrcPacked, true) DMC_GEMM(8, 64, kSrcPacked, false)
    DMC_GEMM(8, 128, kSrcPacked, true) DMC_GEMM(8, 128, kSrcPacked, false) DMC_GEMM(4, 32, kSrcPacked, true)
    DMC_GEMM(4, 32, kSrcPacked, false) DMC_GEMM(4, 64, kSrcPacked, true) DMC_GEMM(4, 64, kSrcPacked, false)
    DMC_GEMM(8, 16, kSrcRows, true) DMC_GEMM(8, 32, kSrcRows, true) DMC_GEMM(8, 64, kSrcRows, true)
    return hipErrorInvalidValue;
#undef DMC_GEMM
    if (pl.kslices > 1) return launch_sum_slices(part, pl.kslices, p, s);
    return hipGetLastError();
}

hipError_t launch_gemm_cs(const CsProblem &p, const CsPlan &pl, void *workspace, hipStream_t s) {
    const int64_t nchunks = (p.k + 63) / 64;
    const int64_t kc = pl.kslice / 64;
    if (p.k < 1 || pl.cb != 256 || pl.waves != 8 || pl.kslice % 64 != 0 || kc < 1 || pl.slices < 1 ||
        pl.slices * kc < nchunks || (pl.slices > 1 && !workspace) || pl.grid_x * 256 < p.n || p.batch > 65535 ||
        (p.k + 64) * p.n * 2 > INT32_MAX || p.m * p.k * 4 > INT32_MAX || !aligned(p.w, 2) || !aligned(p.x, 4))
        return hipErrorInvalidValue;
    float *const part = pl.slices > 1 ? static_cast<float *>(workspace) : nullptr;
    const int64_t gy = (p.m + pl.mt - 1) / pl.mt;
    const int64_t wgs = pl.grid_x * gy * pl.slices;
    if (wgs > INT32_MAX) return hipErrorInvalidValue;
    const dim3 grid((unsigned)wgs, (unsigned)p.batch);
#define DMC_GEMM_CS(MT)                                                                                        \
    hipLaunchKernelGGL((gemv_mfma_gemm_kernel<8, MT, kSrcCols, true>), grid, dim3(512), 0, s, p.w, p.x,            \
                       (const uint16_t *)nullptr, p.y, part, (int)p.n, (int)p.k, (int)p.m, (int)kc, (int)pl.grid_x, \
                       (int)gy, gy > 1 ? 1 : 0, p.rs, p.ls)
    if (pl.mt == 16) DMC_GEMM_CS(16);
    else if (pl.mt == 32) DMC_GEMM_CS(32);
    else if (pl.mt == 64) DMC_GEMM_CS(64);
    else return hipErrorInvalidValue;
#undef DMC_GEMM_CS
    if (pl.slices <= 1) return hipGetLastError();
#define DMC_SUM_CS(Q)                                                                                          \
    hipLaunchKernelGGL((gemm_sum_slices_kernel<Q, false>), dim3(grid_for((p.m * p.n / Q + 255) / 256), (unsigned)p.batch), \
                       dim3(256), 0, s, part, (int)pl.slices, p.y, p.w, p.x, (int)p.m, (int)p.n, (int)p.k, p.n, p.rs, p.ls)
    if (p.n % 4 == 0) DMC_SUM_CS(4);
    else DMC_SUM_CS(1);
#undef DMC_SUM_CS
    return hipGetLastError();
}

}  // namespace dmc
