// gfx950 kernels of the exact negacyclic multiplier c = a*b mod (X^N+1, q).
//
// Pipeline (per product; every stage is integer-only):
//   0. pack_operands        limbs -> 64-byte-aligned K tiles of signed bytes
//   1. conversion_gemm      limb bytes x signed byte weights on INT8 MFMA
//                           (v_mfma_i32_16x16x64_i8), REDC -> residues mod p_k
//                           [reference: tensor_product<true>, solve.cu:143-250]
//   (0-2 in one kernel, convert: q of up to 256 limbs; 2 only for few rows)
//   2. ntt_columns_forward  merged-twist negacyclic NTT stages whose butterfly
//                           distance spans whole rows  [high_stages, solve.cu:280-382]
//   3. ntt_rows_product     remaining forward stages, base-case product mod
//                           (X^n1 - zeta), inverse stages, all inside one row
//                           [middle_stages*, solve.cu:385-570]
//   4. ntt_columns_inverse  inverse row-spanning stages -> v_k = x P_k^-1 mod p_k
//                           [high_stages<true>, solve.cu:317-382]
//   5. crt_gemm             residue bytes x signed digits of M_k and of
//                           floor((2^64-1)/p_k) on INT8 MFMA -> word sums of
//                           T = sum v_k M_k and of the quotient sum E
//                           [tensor_product<false>, solve.cu:143-250; CFS:1872-1881]
//   6. reconstruct          K = round(E/2^64), T += K*((-P) mod q), carries,
//                           Barrett reduction by an arbitrary q
//                           [reconstruct_direct, solve.cu:667-716, generalized]
//   (5 and 6, and 4 for few rows, in one kernel, crt_reconstruct: q of up to 60
//   limbs)
//
// Signed INT8 MFMA: data bytes u in [0,255] enter as u-128 (XOR 0x80); the
// weights are signed base-256 digits; the constant 128*sum(weights) is folded
// into per-prime offsets (conversion) and a fixed big-integer correction (CRT).
//
// Planes have a row stride of n_pad = N rounded up to 256, and word sums n_pad
// rows, so every GEMM tile load is in bounds and 16-byte aligned.
#include "kernels.hpp"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <type_traits>

namespace pm {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t u32_alias __attribute__((may_alias));

// GEMM block tile: 256 weight rows x 128 WN coefficients x 64 bytes of K, 4 x WN
// waves, each owning a 64x128 slab = 4x8 MFMA 16x16 tiles (128 int32
// accumulators per lane; two waves per SIMD).  WN is 2, or 1 where whole tiles
// would leave CUs without a block (gemm_halves).
constexpr uint32_t kTileBytes = kTile * kTK;  // one operand K step, 16 KB
constexpr uint32_t kLoads = 2;                // 16-byte loads of B per thread and K step
constexpr uint32_t kWaveM = 4, kWaveN = 8;    // 16x16 tiles per wave
constexpr uint32_t kWaveRows = kWaveM * 16, kWaveCols = kWaveN * 16;
constexpr uint32_t kGroupN = 4;               // raster group width (tiles)

constexpr uint32_t kRowWidth = 2048;          // C of every transform of more than one row

void check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

__device__ __forceinline__ uint32_t add_mod(uint32_t a, uint32_t b, uint32_t p) {
    const uint32_t t = a + b;
    return min(t, t - p);
}

__device__ __forceinline__ uint32_t sub_mod(uint32_t a, uint32_t b, uint32_t p) {
    const uint32_t t = a - b;
    return min(t, t + p);
}

// Shoup: wq = floor(w*2^32/p); for any a < 2^32, a*w - hi(a*wq)*p lies in [0, 2p).
// Both low products are taken as v_mad_u64_u32 in 64 bits, the second with the
// first as its addend, which saves the subtraction (on gfx950 all of these issue
// at the same rate, one per 4 cycles and SIMD); only the low word counts.
__device__ __forceinline__ uint32_t mul_shoup_lazy(uint32_t a, uint32_t w, uint32_t wq, uint32_t p) {
    uint64_t r = uint64_t(__umulhi(a, wq)) * (0u - p) + uint64_t(a) * w;
    asm("" : "+v"(r));  // keeps the 64-bit form, which the compiler would narrow to three instructions
    return uint32_t(r);
}

__device__ __forceinline__ uint32_t mul_shoup(uint32_t a, uint32_t w, uint32_t wq, uint32_t p) {
    const uint32_t r = mul_shoup_lazy(a, w, wq, p);
    return min(r, r - p);  // r - p wraps above r exactly when r < p
}

// Subtractive Montgomery REDC of t < p*2^32: (t - m p)/2^32, m = t p^-1 mod 2^32.
__device__ __forceinline__ uint32_t redc(uint64_t t, uint32_t p, uint32_t pinv) {
    uint32_t m = uint32_t(t) * pinv;
    uint32_t mh = __umulhi(m, p);
    uint32_t r = uint32_t(t >> 32) - mh;  // in (-p, p) mod 2^32: r + p is the smaller exactly when r < 0
    return min(r, r + p);
}

// REDC for t < 2p*2^32 (four products of residues: 4p^2 < 2p*2^32 as 2p < 2^32):
// one more conditional subtraction than redc.
__device__ __forceinline__ uint32_t redc_wide(uint64_t t, uint32_t p, uint32_t pinv) {
    const uint32_t mh = __umulhi(uint32_t(t) * pinv, p);
    uint32_t hi = uint32_t(t >> 32);
    hi = min(hi, hi - p);  // t - p*2^32, in redc's range, when that is not negative
    const uint32_t r = hi - mh;
    return min(r, r + p);
}

// Cooley-Tukey: (a, b) -> (a + wb, a - wb).  a < p; b may be any 32-bit value
// congruent to its residue.  With kReduce the outputs are below p; without,
// below 2p, which is all the next level asks of the values it multiplies (b),
// and half of every level's outputs are that: 8 instead of 11 instructions.
// (Primes just below 2^31 leave no room for Harvey's form, lazy in all of them.)
template <bool kReduce>
__device__ __forceinline__ void ct_butterfly(uint32_t& a, uint32_t& b, uint2 w, uint32_t p) {
    const uint32_t v = mul_shoup(b, w.x, w.y, p);
    if constexpr (kReduce) {
        b = sub_mod(a, v, p);
        a = add_mod(a, v, p);
    } else {
        b = a - v + p;
        a = a + v;
    }
}

// Gentleman-Sande: (a, b) -> (a + b, w (a - b)), all below p; the difference
// goes into the product as it is, below 2p.
__device__ __forceinline__ void gs_butterfly(uint32_t& a, uint32_t& b, uint2 w, uint32_t p) {
    const uint32_t u = a, v = b;
    a = add_mod(u, v, p);
    b = mul_shoup(u - v + p, w.x, w.y, p);
}

__device__ __forceinline__ uint32_t mont(uint32_t a, uint32_t b, uint32_t p, uint32_t pinv) {
    return redc(uint64_t(a) * b, p, pinv);
}

// 1, 256, 65536 and 2^24 in scalar registers the compiler cannot see through.
// With literal scales each int64 term becomes a sign extension and a 64-bit
// shift and add (about four instructions); with a register scale it is one
// v_mad_i64_i32 (32x32 signed product plus 64-bit addend).
struct DigitScales {
    int32_t s0, s8, s16, s24;
};

__device__ __forceinline__ DigitScales digit_scales() {
    DigitScales s;
    asm volatile("s_mov_b32 %0, 1" : "=s"(s.s0));
    asm volatile("s_mov_b32 %0, 0x100" : "=s"(s.s8));
    asm volatile("s_mov_b32 %0, 0x10000" : "=s"(s.s16));
    asm volatile("s_mov_b32 %0, 0x1000000" : "=s"(s.s24));
    return s;
}

// base + sum_d 256^d v[d], exact in int64.
__device__ __forceinline__ int64_t combine4(const v4i& v, const DigitScales& s, int64_t base = 0) {
    int64_t t = int64_t(v[0]) * int64_t(s.s0) + base;
    t += int64_t(v[1]) * int64_t(s.s8);
    t += int64_t(v[2]) * int64_t(s.s16);
    t += int64_t(v[3]) * int64_t(s.s24);
    return t;
}

// LDS operand tile: 256 rows of 64 bytes; the four 16-byte chunks of a row are
// XOR-swizzled by row/2.  A 128-bit LDS read serves 8 lanes (128 bytes) per
// pass; a fragment read gives those 8 lanes rows r..r+7 of one chunk, and with
// the swizzle their 16-byte slots (row*4 + chunk') mod 8 are all distinct.  The
// direct-to-LDS loads fill the slots linearly (64 consecutive slots per wave).
__device__ __forceinline__ uint32_t swz(uint32_t row, uint32_t chunk) {
    return row * kTK + (((chunk ^ (row >> 1)) & 3u) << 4);
}

// Block -> (m tile, n tile), over n groups of kGroupN tiles, each walked row by
// row.  Workgroups are dispatched to the 8 XCDs round robin, 32 at a time to
// each: those 32 get a run of the walk (8 rows x 4 tiles), so they share A and
// B tiles in their XCD's L2, and the 8 XCDs' runs follow one another, so that
// all 256 blocks at work share their few B panels, and the A panels from one n
// group to the next, in the cache behind the L2s instead of fetching them from
// HBM once per XCD.  (Each XCD walking an eighth of the grid of its own:
// conversion GEMM 10.27 ms against 9.93, CRT GEMM 5.16 against 5.03 at N =
// 65536 with 1747 limbs; the GEMMs run at the clock the card's power allows,
// and the traffic takes a part of it.)
__device__ __forceinline__ void tile_coords(uint32_t bid, uint32_t num_m, uint32_t num_n, uint32_t& tm,
                                            uint32_t& tn) {
    const uint32_t total = num_m * num_n, full = total & ~255u, x = bid % 8;
    uint32_t logical = bid;  // the last few stay where they are
    if (bid < full) {
        logical = (bid & ~255u) + x * 32 + (bid & 255u) / 8;
    } else {  // less than a round: eighths of it
        const uint32_t per = (total - full) / 8, i = bid - full;
        if (i < per * 8) logical = full + x * per + i / 8;
    }
    const uint32_t in_group = kGroupN * num_m;
    const uint32_t group = logical / in_group, first_n = group * kGroupN;
    const uint32_t width = num_n - first_n < kGroupN ? num_n - first_n : kGroupN;
    const uint32_t local = logical % in_group;
    tn = first_n + local % width;
    tm = local / width;
}

// The K loop, for a block tile of 256 weight rows (A, the pre-tiled weight
// panel [k steps][256][64]) x 256 coefficients (B, the pre-tiled data panel of
// the same layout), 64 bytes of K per step, four stages in flight:
//  * A is not staged: each wave loads its own MFMA fragments straight from
//    global memory.  Fragment mi of step ks for lane l is the 16 bytes of row
//    wm*64 + mi*16 + (l&15), chunk l>>4 -- 1 KB contiguous per fragment, one
//    coalesced load.  (Waves wn = 0 and 1 load the same fragments; the second
//    load mostly hits the CU's L1.)
//  * B goes global -> LDS with direct-to-LDS loads (global_load_lds_dwordx4):
//    lane l of a load fills LDS slot base + l, so each lane fetches the global
//    16-byte chunk that the XOR-swizzled tile layout (swz) puts in that slot.
//    No register staging and no ds_write instructions.
//  * Loads run three steps ahead: four LDS stages (64 KB) and four register
//    sets of A fragments rotate.  Step k waits until its own loads have landed
//    (the 12 loads of steps k+1, k+2 may stay in flight: 4 A + 2 B per lane and
//    step) and until this wave's LDS reads are done, then one barrier; after
//    it, no wave still reads stage (k-1)%4, which step k+3's loads refill.
// The barrier is a plain s_barrier with a compiler memory clobber, not
// __syncthreads(): the latter's release fence would wait for every
// outstanding direct-to-LDS load (vmcnt 0) and undo the prefetch.
// Measured on the conversion and CRT shapes of N=65536, L=1747 against the
// two-stage loop that staged both operands through registers and ds_write:
// 2-3 % faster on the conversion GEMM, 5-10 % on the CRT GEMM.
struct GemmStages {
    int8_t* s[4];
};

template <uint32_t WN>
__device__ __forceinline__ void gemm_mainloop(const int8_t* __restrict__ a_panel, const int8_t* __restrict__ b_panel,
                                              uint32_t ksteps, const GemmStages& st, v4i (&acc)[kWaveM][kWaveN]) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t wm = wave / WN, wn = wave % WN;
    const v4i* ap = reinterpret_cast<const v4i*>(a_panel + (wm * kWaveRows + (lane & 15)) * kTK + (lane >> 4) * 16);
    // B: slot s = tid + 256 WN j of a stage holds row s>>2, swizzled chunk s&3,
    // i.e. the row's chunk (s&3) ^ ((row>>1)&3) in the global tile.
    uint32_t boff[kLoads];
#pragma unroll
    for (uint32_t j = 0; j < kLoads; ++j) {
        const uint32_t slot = tid + 256 * WN * j, row = slot >> 2, chunk = (slot & 3) ^ ((row >> 1) & 3);
        boff[j] = row * kTK + chunk * 16;
    }
    auto clamp = [&](uint32_t k) { return k < ksteps ? k : ksteps - 1; };  // past the end: repeat the last step
    auto load_b = [&](uint32_t ks, int8_t* stage) {
        const int8_t* src = b_panel + size_t(ks) * kTileBytes;
#pragma unroll
        for (uint32_t j = 0; j < kLoads; ++j)
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const void*>(src + boff[j]),
                                             (__attribute__((address_space(3))) void*)(stage + (wave * 64 + 256 * WN * j) * 16),
                                             16, 0, 0);
    };
    auto load_a = [&](uint32_t ks, v4i (&fa)[kWaveM]) {
#pragma unroll
        for (uint32_t mi = 0; mi < kWaveM; ++mi) fa[mi] = ap[size_t(ks) * (kTileBytes / 16) + mi * 64];
    };
    v4i f0[kWaveM], f1[kWaveM], f2[kWaveM], f3[kWaveM], fb[kWaveN];
    auto step = [&](uint32_t k, const int8_t* stage, const v4i (&fa)[kWaveM], int8_t* next_stage,
                    v4i (&next_fa)[kWaveM]) {
        // vmcnt <= 12 (gfx9 encoding: low bits 3:0, high bits 15:14), lgkmcnt 0, expcnt untouched
        constexpr int kWait = (12 & 15) | ((12 >> 4) << 14) | (0x7 << 4);
        __builtin_amdgcn_s_waitcnt(kWait);
        asm volatile("s_barrier" ::: "memory");
        load_b(clamp(k + 3), next_stage);
        load_a(clamp(k + 3), next_fa);
#pragma unroll
        for (uint32_t ni = 0; ni < kWaveN; ++ni)
            fb[ni] = *reinterpret_cast<const v4i*>(stage + swz(wn * kWaveCols + ni * 16 + (lane & 15), lane >> 4));
#pragma unroll
        for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
            for (uint32_t ni = 0; ni < kWaveN; ++ni)
                acc[mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[mi], fb[ni], acc[mi][ni], 0, 0, 0);
    };
    load_b(0, st.s[0]);
    load_a(0, f0);
    load_b(clamp(1), st.s[1]);
    load_a(clamp(1), f1);
    load_b(clamp(2), st.s[2]);
    load_a(clamp(2), f2);
    uint32_t k0 = 0;
    for (; k0 + 4 <= ksteps; k0 += 4) {
        step(k0, st.s[0], f0, st.s[3], f3);
        step(k0 + 1, st.s[1], f1, st.s[0], f0);
        step(k0 + 2, st.s[2], f2, st.s[1], f1);
        step(k0 + 3, st.s[3], f3, st.s[2], f2);
    }
    if (k0 < ksteps) step(k0, st.s[0], f0, st.s[3], f3);
    if (k0 + 1 < ksteps) step(k0 + 1, st.s[1], f1, st.s[0], f0);
    if (k0 + 2 < ksteps) step(k0 + 2, st.s[2], f2, st.s[1], f1);
    // No direct-to-LDS load may outlive the block's LDS (the loads past the
    // last step refill stages nobody reads).
    __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8));  // vmcnt 0
}

// The four LDS stages of gemm_mainloop (8 KB times WN), as separate arrays of the kernel
// (so the compiler can tell a stage being filled from the one being read).
#define PM_GEMM_STAGES(name)                                                                               \
    __shared__ __attribute__((aligned(16))) int8_t name##0[kTileBytes / 2 * WN], name##1[kTileBytes / 2 * WN], \
        name##2[kTileBytes / 2 * WN], name##3[kTileBytes / 2 * WN];                                            \
    const GemmStages name{{name##0, name##1, name##2, name##3}}

// ---------------------------------------------------------------------------
// 0. operand packing: [N][L] u32 -> [2][n_pad/256][conv_k/64][256][64] bytes,
//    each byte XOR 0x80 (u -> u-128 as int8); padding words (beyond L, or rows
//    beyond N) hold the value 0.  16 lanes per coefficient row: lane l moves
//    words l, l+16, ... of the row (a block holds consecutive rows, so only
//    128-byte lines at block edges are shared).
// ---------------------------------------------------------------------------
// Rows of one wave: four rows of 16 lanes each, so that a store instruction
// writes four consecutive coefficients' 64-byte K-step chunks, 256 contiguous
// bytes of the packed tile (with one row per wave, it wrote four chunks 16 KB
// apart: 0.391 against 0.370 ms at N = 65536 with 1747 limbs).
constexpr uint32_t kPackRows = 4, kPackSpan = 64 / kPackRows;  // lanes per row

// Packs the tiles of `ts` of operands op0 .. op0+nops-1.  The k-th tile's rows
// are read from rows k*256 .. k*256+255 of a (or b): the caller passes the
// operands' rows in the set's order (all of [N][L] for the set of every tile).
__device__ __forceinline__ void pack_body(const uint32_t* __restrict__ a, const uint32_t* __restrict__ b,
                                          uint32_t* __restrict__ packed, uint32_t n, uint32_t limbs,
                                          uint32_t ksteps, uint32_t ntiles, TileSet ts, uint32_t op0,
                                          uint32_t nops, uint32_t bx) {
    constexpr uint32_t span = kPackSpan;
    const uint32_t lane = (threadIdx.x & 63) % span;
    const uint32_t per_op = ts.count * kTile;
    // row over all operands of the launch
    const uint32_t gr = (bx * 4 + (threadIdx.x >> 6)) * kPackRows + (threadIdx.x & 63) / span;
    if (gr >= nops * per_op) return;
    const uint32_t op = op0 + gr / per_op, rr = gr % per_op;
    const uint32_t tn = tile_at(ts, rr / kTile), row = rr % kTile, coef = tn * kTile + row;
    const bool live = coef < n;
    // Rows past n read (and discard) the set's first row, so every load is
    // unconditional: kPackLoads loads per lane are in flight before their
    // stores, instead of one load, a wait and a store at a time.
    const uint32_t* src = (op ? b : a) + size_t(live ? rr : 0) * limbs;
    uint32_t* dst = packed + (size_t(op) * ntiles + tn) * ksteps * (kTileBytes / 4) + row * (kTK / 4);
    const uint32_t words = ksteps * (kTK / 4);
    constexpr uint32_t kPackLoads = 8;
    for (uint32_t w0 = lane; w0 < words; w0 += span * kPackLoads) {
        uint32_t v[kPackLoads];
#pragma unroll
        for (uint32_t u = 0; u < kPackLoads; ++u) {
            const uint32_t w = w0 + span * u;
            v[u] = src[w < limbs ? w : limbs - 1];  // clamped into the row; padding words are zeroed below
        }
#pragma unroll
        for (uint32_t u = 0; u < kPackLoads; ++u) {
            const uint32_t w = w0 + span * u;
            if (w < words)
                dst[size_t(w / (kTK / 4)) * (kTileBytes / 4) + w % (kTK / 4)] =
                    ((live && w < limbs) ? v[u] : 0u) ^ 0x80808080u;
        }
    }
}

__global__ __launch_bounds__(256) void pack_operands(const uint32_t* __restrict__ a,
                                                     const uint32_t* __restrict__ b,
                                                     uint32_t* __restrict__ packed, uint32_t n, uint32_t limbs,
                                                     uint32_t ksteps, uint32_t ntiles, TileSet ts, uint32_t op0,
                                                     uint32_t nops) {
    pack_body(a, b, packed, n, limbs, ksteps, ntiles, ts, op0, nops, blockIdx.x);
}

// ---------------------------------------------------------------------------
// 1. conversion GEMM: G[4k+d][i] = sum_j digit_d(lambda*256^j mod p_k) * (byte_j(x_i)-128)
//    then x_i*lambda mod p_k = REDC(sum_d 256^d G[4k+d][i] + off_k).
// ---------------------------------------------------------------------------
template <uint32_t WN>
__device__ __forceinline__ void conversion_body(const int8_t* __restrict__ wtiles, const int8_t* __restrict__ packed,
                                                const PrimeConst* __restrict__ consts, uint32_t* __restrict__ planes,
                                                uint32_t n, uint32_t n_pad, uint32_t r, uint32_t r_pad,
                                                uint32_t conv_rows, uint32_t ksteps, TileSet ts, uint32_t op0,
                                                uint32_t nops, uint32_t bid) {
    PM_GEMM_STAGES(stages);
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t wm = wave / WN, wn = wave % WN;
    const uint32_t ntiles = n_pad / kTile, num_m = conv_rows / kTile;
    uint32_t tm, tn;
    constexpr uint32_t kParts = 2 / WN;
    tile_coords(bid, num_m, nops * ts.count * kParts, tm, tn);  // the set's coefficient tiles of nops operands
    const uint32_t part = tn % kParts;                          // of the 256-coefficient tile
    tn /= kParts;
    const uint32_t op = op0 + tn / ts.count, tcol = tile_at(ts, tn % ts.count);
    const int8_t* a_panel = wtiles + (size_t(op) * num_m + tm) * ksteps * kTileBytes;
    const int8_t* b_panel = packed + (size_t(op) * ntiles + tcol) * ksteps * kTileBytes + part * (kTileBytes / 2);

    v4i acc[kWaveM][kWaveN];
#pragma unroll
    for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
        for (uint32_t ni = 0; ni < kWaveN; ++ni) acc[mi][ni] = v4i{0, 0, 0, 0};
    gemm_mainloop<WN>(a_panel, b_panel, ksteps, stages, acc);

    // Lane holds rows 4*(lane/16)+j (j = digit) of each 16-row tile: one prime.
    // The digit sum is sum_j c_j*(byte_j - 128) with |c_j| <= p/2 over 4L bytes,
    // so |sum| <= 256*L*p; adding p*2^31 (0 mod p) to off_k makes t non-negative
    // and below p*2^32, the range of the unsigned REDC, while 256*L + 1 <= 2^31.
    // Plans allow at most 16383 primes of < 32 bits covering (q-1)^2, so
    // q < 2^262144 and L <= 8192: 256*L <= 2^21.
    const DigitScales ds = digit_scales();
    const uint32_t m0 = tm * kTile + wm * kWaveRows, c0 = tcol * kTile + (part + wn) * kWaveCols;
#pragma unroll
    for (uint32_t mi = 0; mi < kWaveM; ++mi) {
        const uint32_t kp = (m0 + mi * 16) / 4 + (lane >> 4);
        if (kp >= r) continue;
        const PrimeConst pc = consts[kp];
        const int64_t off = int64_t(op ? pc.off_b : pc.off_a) + (int64_t(pc.p) << 31);
        uint32_t* out = planes + (size_t(op) * r_pad + kp) * n_pad;
#pragma unroll
        for (uint32_t ni = 0; ni < kWaveN; ++ni) {
            const uint32_t coef = c0 + ni * 16 + (lane & 15);
            if (coef < n) out[coef] = redc(uint64_t(combine4(acc[mi][ni], ds, off)), pc.p, pc.pinv);
        }
    }
}

template <uint32_t WN>
__global__ __launch_bounds__(256 * WN, 2) void conversion_gemm(const int8_t* __restrict__ wtiles,
                                                       const int8_t* __restrict__ packed,
                                                       const PrimeConst* __restrict__ consts,
                                                       uint32_t* __restrict__ planes, uint32_t n, uint32_t n_pad,
                                                       uint32_t r, uint32_t r_pad, uint32_t conv_rows,
                                                       uint32_t ksteps, TileSet ts, uint32_t op0, uint32_t nops) {
    conversion_body<WN>(wtiles, packed, consts, planes, n, n_pad, r, r_pad, conv_rows, ksteps, ts, op0, nops, blockIdx.x);
}

// ---------------------------------------------------------------------------
// 1'. packing and conversion in one kernel, for q of up to kShortLimbs limbs:
// the coefficients' limbs go straight from [N][L] into MFMA operand registers,
// and the packed copy is never written.
//
//  * A wave owns 16 NT coefficients of one operand and holds all their bytes (at
//    most KS K steps) in registers: lane l of a fragment loads the 16 bytes of
//    coefficient l & 15, chunk l >> 4, which are only 4-byte aligned.  Bytes
//    past a coefficient's limbs are 0 there; their weights are 0 too.
//  * The block's four waves then walk the primes together, 64 weight rows (16
//    primes) at a time.  The weights come in by direct-to-LDS loads, as many
//    64-row chunks at once as kConvertStage holds, in the swizzled layout of
//    gemm_mainloop; each chunk is multiplied, reduced and stored with no wait
//    in between.
//  * gridDim.y splits the primes over blocks when there are few coefficients.
//  * ROWS > 1: a lane's fragments are the rows of whole columns, and it does the
//    forward column stages before it stores (convert_plan).
// What bounds it at N = 65536 with 55 limbs (30.7 us, packing and GEMM before:
// 14.7 + 36.5): the 29 MB of limbs read and 60 MB of residues written, about
// 18 us at a large copy's rate, with the MFMAs (7 us) and the reductions (5 us)
// beside them.  At N = 131072 with 4 limbs 11.1 against 18.4 + 21.2 us, at
// N = 128 with 128 limbs 4.8 against 2.9 + 12.0, at N = 8192 with 226 41.8
// against 7.9 + 37.5, at N = 65536 with 226 339 against 47 + 319.  Beyond 256
// limbs a wave's registers hold too few coefficients to feed the MFMAs from
// LDS.  (Operand bytes in LDS and weights straight from L2, one barrier per
// block: 37 us at N = 65536; the weight fragments then come from L2 once per
// wave.)
// ---------------------------------------------------------------------------
constexpr uint32_t kConvertStage = 48 << 10;  // LDS bytes of weights: three blocks per CU

struct ConvertArgs {
    uint32_t n, n_pad, limbs, r, r_pad, conv_rows, ksteps, n2;
    TileSet ts;  // tile k's rows are rows k*256 .. of a and b (pack_body)
    uint32_t op0;
};

constexpr uint32_t convert_stage_chunks(uint32_t ksteps) {
    const uint32_t chunk = ksteps * kWaveRows * kTK;
    return chunk < kConvertStage ? kConvertStage / chunk : 1;
}

// 16-prime chunks of one of `split` blocks that share the primes.
__host__ __device__ constexpr uint32_t convert_share(uint32_t r, uint32_t split) {
    return ((r + 15) / 16 + split - 1) / split;
}

// The staged weights, then the constants and (columns > 1) twiddles of a share's primes.
constexpr size_t convert_lds_bytes(uint32_t ksteps, uint32_t r, uint32_t split, uint32_t columns) {
    return size_t(convert_stage_chunks(ksteps)) * ksteps * kWaveRows * kTK +
           size_t(convert_share(r, split)) * 16 * (sizeof(PrimeConst) + (columns > 1 ? columns * sizeof(uint2) : 0));
}

// Blocks (bx, by) of (., ny).
template <int KS, int NT, int ROWS>
__device__ __forceinline__ void convert_body(const uint32_t* __restrict__ a, const uint32_t* __restrict__ b,
                                             const int8_t* __restrict__ wtiles,
                                             const PrimeConst* __restrict__ consts,
                                             const uint2* __restrict__ twf, uint32_t* __restrict__ planes,
                                             const ConvertArgs& args, uint32_t bx, uint32_t by, uint32_t ny,
                                             int8_t* lds) {
    typedef uint32_t v4u_word __attribute__((ext_vector_type(4), aligned(4)));  // 4-byte aligned
    constexpr uint32_t T = 64 * NT, kChunkStep = kWaveRows * kTK;                 // 4 KB: 64 rows of one K step
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t L = args.limbs, ksteps = args.ksteps;
    const uint32_t per_op = args.ts.count * kTile / T;
    // The block's coefficients: T consecutive ones of the set, fragment ni of a
    // wave 16 of them; or (ROWS > 1) T / ROWS columns of the transform's
    // [ROWS][2048] matrix, fragment ni row ni % ROWS of 16 columns, so that a lane
    // holds whole columns.
    const uint32_t op = args.op0 + bx / per_op, k0 = bx % per_op * (T / ROWS);
    const uint32_t i0 = ROWS > 1 ? k0 : tile_at(args.ts, k0 / kTile) * kTile + k0 % kTile;
    const uint32_t rows = ROWS > 1 ? T : i0 < args.n ? (args.n - i0 < T ? args.n - i0 : T) : 0;
    auto place = [](uint32_t ni) { return ni / ROWS * 16 + (ROWS > 1 ? ni % ROWS * kRowWidth : 0); };
    const uint32_t chunks = (args.r + 15) / 16, share = convert_share(args.r, ny);
    const uint32_t c0 = by * share, c1 = c0 + share < chunks ? c0 + share : chunks;
    if (!rows || c0 >= c1) return;  // whole block
    const uint32_t cl = wave * (16 * NT / ROWS) + (lane & 15);  // the lane's first coefficient of the block's

    v4i fb[KS][NT];
    {
        const uint32_t* src = (op ? b : a) + size_t(k0) * L;
        const uint32_t w0 = (lane >> 4) * 4;
#pragma unroll
        for (uint32_t ks = 0; ks < KS; ++ks)
#pragma unroll
            for (uint32_t ni = 0; ni < NT; ++ni) {
                const uint32_t row = ROWS > 1 || cl + ni * 16 < rows ? cl + place(ni) : rows - 1, w = ks * 16 + w0;
                const uint32_t* p = src + size_t(row) * L + w;
                v4u x = {0, 0, 0, 0};
                if (w + 4 <= L) {
                    x = *reinterpret_cast<const v4u_word*>(p);
                } else {
                    if (w < L) x[0] = p[0];
                    if (w + 1 < L) x[1] = p[1];
                    if (w + 2 < L) x[2] = p[2];
                }
                fb[ks][ni] = __builtin_bit_cast(v4i, x ^ 0x80808080u);
            }
    }
    const uint32_t stage = convert_stage_chunks(ksteps), num_m = args.conv_rows / kTile;
    PrimeConst* pcs = reinterpret_cast<PrimeConst*>(lds + stage * ksteps * kChunkStep);
    for (uint32_t k = c0 * 16 + tid; k < args.r && k < c1 * 16; k += 256) pcs[k - c0 * 16] = consts[k];
    // the column stages' twiddles, ROWS per prime (entry 0 unused)
    uint2* tws = reinterpret_cast<uint2*>(pcs + share * 16);
    if constexpr (ROWS > 1)
        for (uint32_t k = c0 * 16 * ROWS + tid; k < args.r * ROWS && k < c1 * 16 * ROWS; k += 256)
            tws[k - c0 * 16 * ROWS] = twf[size_t(k / ROWS) * args.n2 + k % ROWS];
    // thread tid fills slot tid of a chunk's K step: row tid>>2, chunk swizzled as in swz
    const uint32_t srow = tid >> 2, sbyte = srow * kTK + ((tid & 3) ^ ((srow >> 1) & 3)) * 16;
    const DigitScales ds = digit_scales();
    for (uint32_t s0 = c0; s0 < c1; s0 += stage) {
        const uint32_t s1 = s0 + stage < c1 ? s0 + stage : c1;
        if (s0 != c0) __syncthreads();  // every wave is done with the previous stage
        for (uint32_t c = s0; c < s1; ++c) {
            const int8_t* src = wtiles + (size_t(op) * num_m + c / 4) * ksteps * kTileBytes + (c % 4) * kChunkStep + sbyte;
            for (uint32_t ks = 0; ks < ksteps; ++ks)
                __builtin_amdgcn_global_load_lds(
                    reinterpret_cast<const void*>(src + size_t(ks) * kTileBytes),
                    (__attribute__((address_space(3))) void*)(lds + ((c - s0) * ksteps + ks) * kChunkStep + wave * 1024),
                    16, 0, 0);
        }
        __syncthreads();
        for (uint32_t c = s0; c < s1; ++c) {
            const int8_t* wl = lds + (c - s0) * ksteps * kChunkStep + swz(lane & 15, lane >> 4);
            v4i acc[kWaveM][NT];
#pragma unroll
            for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
                for (uint32_t ni = 0; ni < NT; ++ni) acc[mi][ni] = v4i{0, 0, 0, 0};
#pragma unroll
            for (uint32_t ks = 0; ks < KS; ++ks)
                if (KS <= 2 || ks < ksteps) {
                    v4i fa[kWaveM];
#pragma unroll
                    for (uint32_t mi = 0; mi < kWaveM; ++mi)
                        fa[mi] = *reinterpret_cast<const v4i*>(wl + ks * kChunkStep + mi * 16 * kTK);
#pragma unroll
                    for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
                        for (uint32_t ni = 0; ni < NT; ++ni)
                            acc[mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[mi], fb[ks][ni], acc[mi][ni], 0, 0, 0);
                }
            // the epilogue of conversion_body
#pragma unroll
            for (uint32_t mi = 0; mi < kWaveM; ++mi) {
                const uint32_t kp = c * 16 + mi * 4 + (lane >> 4);
                if (kp >= args.r) continue;
                const PrimeConst pc = pcs[kp - c0 * 16];
                const int64_t off = int64_t(op ? pc.off_b : pc.off_a) + (int64_t(pc.p) << 31);
                uint32_t* out = planes + (size_t(op) * args.r_pad + kp) * args.n_pad + i0 + cl;
                uint32_t x[NT];
#pragma unroll
                for (uint32_t ni = 0; ni < NT; ++ni) x[ni] = redc(uint64_t(combine4(acc[mi][ni], ds, off)), pc.p, pc.pinv);
                if constexpr (ROWS > 1) {  // the forward column stages (forward_reg_body)
                    const uint2* tw = tws + (kp - c0 * 16) * ROWS;
#pragma unroll
                    for (int m = 1, half = ROWS / 2; m < ROWS; m *= 2, half /= 2)
#pragma unroll
                        for (int g = 0; g < m; ++g) {
                            const uint2 t = tw[m + g];
#pragma unroll
                            for (int cg = 0; cg < NT / ROWS; ++cg)
#pragma unroll
                                for (int jr = 0; jr < half; ++jr) {
                                    uint32_t &lo = x[cg * ROWS + 2 * half * g + jr],
                                             &hi = x[cg * ROWS + 2 * half * g + jr + half];
                                    if (half == 1 || !(jr & (half / 2))) ct_butterfly<true>(lo, hi, t, pc.p);
                                    else ct_butterfly<false>(lo, hi, t, pc.p);
                                }
                        }
                }
#pragma unroll
                for (uint32_t ni = 0; ni < NT; ++ni)
                    if (ROWS > 1 || cl + ni * 16 < rows) out[place(ni)] = x[ni];
            }
        }
    }
}

template <int KS, int NT, int ROWS>
__global__ __launch_bounds__(256, KS * NT > 16 || NT == 8 ? 2 : 3) void convert(const uint32_t* __restrict__ a, const uint32_t* __restrict__ b,
                                                  const int8_t* __restrict__ wtiles,
                                                  const PrimeConst* __restrict__ consts,
                                                  const uint2* __restrict__ twf, uint32_t* __restrict__ planes,
                                                  ConvertArgs args) {
    extern __shared__ __attribute__((aligned(16))) int8_t dyn_lds[];
    convert_body<KS, NT, ROWS>(a, b, wtiles, consts, twf, planes, args, blockIdx.x, blockIdx.y, gridDim.y, dyn_lds);
}

// ---------------------------------------------------------------------------
// 5. CRT GEMM: G[c][i] = sum_{k,d} w[c][4k+d] * (byte_d(v_{k,i}) - 128),
//    D_j(i) = sum_t 256^t G[4j+t][i]   (int64, exact)
//    stored coefficient-major words[i][j] (row stride ws): a wave's 4 x 16
//    words of 16 coefficients are 128-byte runs per coefficient, written one
//    after another.
// ---------------------------------------------------------------------------
template <uint32_t WN>
__device__ __forceinline__ void crt_body(const int8_t* __restrict__ wtiles, const int8_t* __restrict__ rtiles,
                                         int64_t* __restrict__ words, uint32_t n, uint32_t crt_rows,
                                         uint32_t kstride, uint32_t ksteps, uint32_t crt_words, uint32_t ws,
                                         TileSet ts, uint32_t bid) {
    PM_GEMM_STAGES(stages);
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t wm = wave / WN, wn = wave % WN;
    const uint32_t num_m = crt_rows / kTile;
    uint32_t tm, tn;
    constexpr uint32_t kParts = 2 / WN;
    tile_coords(bid, num_m, ts.count * kParts, tm, tn);  // the set's coefficient tiles
    const uint32_t part = tn % kParts;                   // of the 256-coefficient tile
    tn = tile_at(ts, tn / kParts);
    const int8_t* a_panel = wtiles + size_t(tm) * kstride * kTileBytes;
    const int8_t* b_panel = rtiles + size_t(tn) * kstride * kTileBytes + part * (kTileBytes / 2);

    v4i acc[kWaveM][kWaveN];
#pragma unroll
    for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
        for (uint32_t ni = 0; ni < kWaveN; ++ni) acc[mi][ni] = v4i{0, 0, 0, 0};
    gemm_mainloop<WN>(a_panel, b_panel, ksteps, stages, acc);

    const DigitScales ds = digit_scales();
    const uint32_t m0 = tm * kTile + wm * kWaveRows, c0 = tn * kTile + (part + wn) * kWaveCols;
#pragma unroll
    for (uint32_t ni = 0; ni < kWaveN; ++ni) {
        const uint32_t coef = c0 + ni * 16 + (lane & 15);
        int64_t* out = words + size_t(coef) * ws;
#pragma unroll
        for (uint32_t mi = 0; mi < kWaveM; ++mi) {
            const uint32_t word = (m0 + mi * 16) / 4 + (lane >> 4);
            if (word < crt_words && coef < n) out[word] = combine4(acc[mi][ni], ds);
        }
    }
}

template <uint32_t WN>
__global__ __launch_bounds__(256 * WN, 2) void crt_gemm(const int8_t* __restrict__ wtiles,
                                                const int8_t* __restrict__ rtiles,
                                                int64_t* __restrict__ words, uint32_t n, uint32_t crt_rows,
                                                uint32_t kstride, uint32_t ksteps,
                                                uint32_t crt_words, uint32_t ws, TileSet ts) {
    crt_body<WN>(wtiles, rtiles, words, n, crt_rows, kstride, ksteps, crt_words, ws, ts, blockIdx.x);
}

// ---------------------------------------------------------------------------
// 5'. CRT GEMM for few coefficients: blocks of 64 weight rows (16 word sums) x
// 64 coefficients, whose four waves each take every fourth K step, so that even
// one tile's K loop is spread over a CU.  Both operands are read as MFMA
// fragments straight from their tiles, two steps ahead, with no barrier until
// the waves' sums meet in LDS; each wave then finishes a quarter of them.
// Consecutive tiles of one XCD share their coefficients.  crt_gemm's three
// blocks took 18.7 us at N = 128 with 128 limbs, this 6.4.  (Three waves per
// SIMD leave it 5 registers short: 24 bytes of scratch a lane.)
// ---------------------------------------------------------------------------
__device__ __forceinline__ void crt_small_body(const int8_t* __restrict__ wtiles, const int8_t* __restrict__ rtiles,
                                               int64_t* __restrict__ words, uint32_t n, uint32_t kstride,
                                               uint32_t ksteps, uint32_t crt_words, uint32_t ws, const TileSet& ts,
                                               uint32_t bid) {
    constexpr uint32_t NT = 4, T = 16 * NT;
    __shared__ v4i part[4][3][NT][64];  // [wave that finishes][wave that summed][fragment][lane]
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t num_m = (crt_words + 15) / 16, total = num_m * ts.count * (kTile / T), per = total / 8;
    const uint32_t logical = bid < per * 8 ? (bid % 8) * per + bid / 8 : bid;
    const uint32_t m = logical % num_m, k0 = logical / num_m * T;
    const uint32_t tile = tile_at(ts, k0 / kTile), i0 = tile * kTile + k0 % kTile;
    if (i0 >= n) return;  // whole block
    const uint32_t frag = (lane & 15) * kTK + (lane >> 4) * 16;
    const v4i* ap = reinterpret_cast<const v4i*>(wtiles + size_t(m / 4) * kstride * kTileBytes + m % 4 * (kWaveRows * kTK) + frag);
    const v4i* bp = reinterpret_cast<const v4i*>(rtiles + size_t(tile) * kstride * kTileBytes + k0 % kTile * kTK + frag);
    v4i acc[kWaveM][NT], fa[2][kWaveM], fb[2][NT];
#pragma unroll
    for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
        for (uint32_t ni = 0; ni < NT; ++ni) acc[mi][ni] = v4i{0, 0, 0, 0};
    auto load = [&](uint32_t ks, v4i (&a)[kWaveM], v4i (&b)[NT]) {
#pragma unroll
        for (uint32_t mi = 0; mi < kWaveM; ++mi) a[mi] = ap[size_t(ks) * (kTileBytes / 16) + mi * 64];
#pragma unroll
        for (uint32_t ni = 0; ni < NT; ++ni) b[ni] = bp[size_t(ks) * (kTileBytes / 16) + ni * 64];
    };
    auto step = [&](const v4i (&a)[kWaveM], const v4i (&b)[NT]) {
#pragma unroll
        for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
            for (uint32_t ni = 0; ni < NT; ++ni)
                acc[mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[mi], b[ni], acc[mi][ni], 0, 0, 0);
    };
    uint32_t ks = wave;
    if (ks < ksteps) load(ks, fa[0], fb[0]);
    if (ks + 4 < ksteps) load(ks + 4, fa[1], fb[1]);
    for (; ks + 12 < ksteps; ks += 8) {
        step(fa[0], fb[0]);
        load(ks + 8, fa[0], fb[0]);
        step(fa[1], fb[1]);
        load(ks + 12, fa[1], fb[1]);
    }
    if (ks < ksteps) step(fa[0], fb[0]);
    if (ks + 8 < ksteps) load(ks + 8, fa[0], fb[0]);
    if (ks + 4 < ksteps) step(fa[1], fb[1]);
    if (ks + 8 < ksteps) step(fa[0], fb[0]);
    // wave w finishes row fragment mi = w
#pragma unroll
    for (uint32_t mi = 0; mi < kWaveM; ++mi)
        if (mi != wave)
#pragma unroll
            for (uint32_t ni = 0; ni < NT; ++ni) part[mi][wave > mi ? wave - 1 : wave][ni][lane] = acc[mi][ni];
    __syncthreads();
    const DigitScales ds = digit_scales();
    const uint32_t word = m * 16 + wave * 4 + (lane >> 4);
#pragma unroll
    for (uint32_t ni = 0; ni < NT; ++ni) {
        v4i sum = wave == 0 ? acc[0][ni] : wave == 1 ? acc[1][ni] : wave == 2 ? acc[2][ni] : acc[3][ni];
#pragma unroll
        for (uint32_t w = 0; w < 3; ++w) sum += part[wave][w][ni][lane];
        const uint32_t coef = i0 + ni * 16 + (lane & 15);
        if (word < crt_words && coef < n) words[size_t(coef) * ws + word] = combine4(sum, ds);
    }
}

__global__ __launch_bounds__(256, 3) void crt_small(const int8_t* __restrict__ wtiles,
                                                    const int8_t* __restrict__ rtiles, int64_t* __restrict__ words,
                                                    uint32_t n, uint32_t kstride, uint32_t ksteps,
                                                    uint32_t crt_words, uint32_t ws, TileSet ts) {
    crt_small_body(wtiles, rtiles, words, n, kstride, ksteps, crt_words, ws, ts, blockIdx.x);
}

// ---------------------------------------------------------------------------
// 2-4. NTT.  Flat index i = row*C + col.  Forward: Cooley-Tukey with the
// negacyclic twist merged into psi^bitrev twiddles, m = 1, 2, .., n2/2 groups
// at flat distance N/(2m) down to n1.  Inverse: Gentleman-Sande, mirror order.
// Plane rows have stride ps (= n_pad).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void ntt_columns_forward(uint32_t* __restrict__ planes,
                                                           const PrimeConst* __restrict__ consts,
                                                           const uint2* __restrict__ tw, uint32_t ps,
                                                           uint32_t n2, uint32_t C, uint32_t rows,
                                                           uint32_t cw, uint32_t r, uint32_t op0) {
    extern __shared__ uint32_t tile[];  // [rows][cw]
    const uint32_t col0 = blockIdx.x * cw, k = blockIdx.y, op = op0 + blockIdx.z;
    const uint32_t p = consts[k].p;
    uint32_t* data = planes + (size_t(op) * r + k) * ps;
    const uint2* w = tw + size_t(k) * n2;
    const uint32_t total = rows * cw;
    for (uint32_t t = threadIdx.x; t < total; t += blockDim.x)
        tile[t] = data[size_t(t / cw) * C + col0 + t % cw];
    __syncthreads();
    for (uint32_t m = 1, half = rows / 2; m < rows; m *= 2, half /= 2) {
        for (uint32_t t = threadIdx.x; t < total / 2; t += blockDim.x) {
            uint32_t pr = t / cw, c = t % cw;
            uint32_t g = pr / half, jr = pr % half, row = 2 * half * g + jr;
            uint2 tw_g = w[m + g];
            uint32_t u = tile[row * cw + c];
            uint32_t v = mul_shoup(tile[(row + half) * cw + c], tw_g.x, tw_g.y, p);
            tile[row * cw + c] = add_mod(u, v, p);
            tile[(row + half) * cw + c] = sub_mod(u, v, p);
        }
        __syncthreads();
    }
    for (uint32_t t = threadIdx.x; t < total; t += blockDim.x)
        data[size_t(t / cw) * C + col0 + t % cw] = tile[t];
}

// Row stages for any row width C <= 2048 and block size n1, through LDS;
// lds32 holds 2*C words.
__device__ __forceinline__ void rows_product_body(uint32_t* __restrict__ planes, const uint32_t* __restrict__ bplanes,
                                                  const PrimeConst* __restrict__ consts,
                                                  const uint2* __restrict__ twf, const uint2* __restrict__ twi,
                                                  uint32_t ps, uint32_t n1, uint32_t n2, uint32_t C, uint32_t rows,
                                                  uint32_t* lds32, uint32_t row, uint32_t k) {
    uint32_t* A = lds32;  // A[C], B[C]
    uint32_t* B = lds32 + C;
    const uint32_t p = consts[k].p, pinv = consts[k].pinv;
    uint32_t* pa = planes + size_t(k) * ps + size_t(row) * C;
    const uint32_t* pb = bplanes + size_t(k) * ps + size_t(row) * C;
    const uint2* wf = twf + size_t(k) * n2;
    const uint2* wi = twi + size_t(k) * n2;
    for (uint32_t t = threadIdx.x; t < C; t += blockDim.x) {
        A[t] = pa[t];
        B[t] = pb[t];
    }
    __syncthreads();
    // forward stages with flat distance < C
    for (uint32_t m = rows, t = C / 2; m < n2; m *= 2, t /= 2) {
        for (uint32_t idx = threadIdx.x; idx < C / 2; idx += blockDim.x) {
            uint32_t gl = idx / t, jr = idx % t, j = 2 * t * gl + jr;
            uint2 w = wf[m + row * (C / (2 * t)) + gl];
            uint32_t u = A[j], v = mul_shoup(A[j + t], w.x, w.y, p);
            A[j] = add_mod(u, v, p);
            A[j + t] = sub_mod(u, v, p);
            u = B[j];
            v = mul_shoup(B[j + t], w.x, w.y, p);
            B[j] = add_mod(u, v, p);
            B[j + t] = sub_mod(u, v, p);
        }
        __syncthreads();
    }
    // base case: block gb holds A, B mod (X^n1 - zeta_gb), zeta_gb = psi^(2 bitrev(gb) + 1)
    uint32_t res[8];
    {
        uint32_t cnt = 0;
        for (uint32_t idx = threadIdx.x; idx < C; idx += blockDim.x, ++cnt) {
            const uint32_t s = idx % n1, blk = idx / n1, gb = row * (C / n1) + blk;
            const uint32_t* ab = A + blk * n1;
            const uint32_t* bb = B + blk * n1;
            uint32_t lo = 0, hi = 0;
            for (uint32_t t = 0; t <= s; ++t) lo = add_mod(lo, mont(ab[t], bb[s - t], p, pinv), p);
            for (uint32_t t = s + 1; t < n1; ++t) hi = add_mod(hi, mont(ab[t], bb[s + n1 - t], p, pinv), p);
            uint32_t value = lo;
            if (n1 > 1) {
                if (n2 == 1) {
                    value = sub_mod(lo, hi, p);  // zeta = -1
                } else {
                    uint2 w = wf[n2 / 2 + gb / 2];  // zeta_{2g} = w, zeta_{2g+1} = -w
                    uint32_t z = mul_shoup(hi, w.x, w.y, p);
                    value = (gb & 1) ? sub_mod(lo, z, p) : add_mod(lo, z, p);
                }
            }
            res[cnt] = value;
        }
    }
    __syncthreads();
    {
        uint32_t cnt = 0;
        for (uint32_t idx = threadIdx.x; idx < C; idx += blockDim.x, ++cnt) A[idx] = res[cnt];
    }
    __syncthreads();
    // inverse stages with flat distance < C
    for (uint32_t m = n2 / 2, t = n1; m >= rows && m > 0; m /= 2, t *= 2) {
        for (uint32_t idx = threadIdx.x; idx < C / 2; idx += blockDim.x) {
            uint32_t gl = idx / t, jr = idx % t, j = 2 * t * gl + jr;
            uint2 w = wi[m + row * (C / (2 * t)) + gl];
            uint32_t u = A[j], v = A[j + t];
            A[j] = add_mod(u, v, p);
            A[j + t] = mul_shoup(sub_mod(u, v, p), w.x, w.y, p);
        }
        __syncthreads();
    }
    for (uint32_t t = threadIdx.x; t < C; t += blockDim.x) pa[t] = A[t];
}

__global__ __launch_bounds__(256) void ntt_rows_product(uint32_t* __restrict__ planes,
                                                        const uint32_t* __restrict__ bplanes,
                                                        const PrimeConst* __restrict__ consts,
                                                        const uint2* __restrict__ twf,
                                                        const uint2* __restrict__ twi, uint32_t ps,
                                                        uint32_t n1, uint32_t n2, uint32_t C,
                                                        uint32_t rows) {
    extern __shared__ uint32_t lds32[];
    rows_product_body(planes, bplanes, consts, twf, twi, ps, n1, n2, C, rows, lds32, blockIdx.x, blockIdx.y);
}

__global__ __launch_bounds__(256) void ntt_columns_inverse(uint32_t* __restrict__ plane,
                                                           const PrimeConst* __restrict__ consts,
                                                           const uint2* __restrict__ tw, uint32_t ps,
                                                           uint32_t n2, uint32_t C, uint32_t rows,
                                                           uint32_t cw) {
    extern __shared__ uint32_t tile[];  // [rows][cw]
    const uint32_t col0 = blockIdx.x * cw, k = blockIdx.y;
    const uint32_t p = consts[k].p;
    uint32_t* data = plane + size_t(k) * ps;
    const uint2* w = tw + size_t(k) * n2;
    const uint32_t total = rows * cw;
    for (uint32_t t = threadIdx.x; t < total; t += blockDim.x)
        tile[t] = data[size_t(t / cw) * C + col0 + t % cw];
    __syncthreads();
    for (uint32_t m = rows / 2, half = 1; m >= 1; m /= 2, half *= 2) {
        for (uint32_t t = threadIdx.x; t < total / 2; t += blockDim.x) {
            uint32_t pr = t / cw, c = t % cw;
            uint32_t g = pr / half, jr = pr % half, row = 2 * half * g + jr;
            uint2 tw_g = w[m + g];
            uint32_t u = tile[row * cw + c], v = tile[(row + half) * cw + c];
            tile[row * cw + c] = add_mod(u, v, p);
            tile[(row + half) * cw + c] = mul_shoup(sub_mod(u, v, p), tw_g.x, tw_g.y, p);
        }
        __syncthreads();
    }
    for (uint32_t t = threadIdx.x; t < total; t += blockDim.x)
        data[size_t(t / cw) * C + col0 + t % cw] = tile[t];
}

// ---------------------------------------------------------------------------
// Register-resident NTT kernels for the usual shapes (rows <= 64, C = 2048).
// ---------------------------------------------------------------------------
// Forward row-spanning stages: one thread per (operand, prime, column) holding
// the column's ROWS values; the stage twiddles are uniform over the block.
// Columns col0 + [0, 256 * gridDim.x).
template <int ROWS>
__device__ __forceinline__ void forward_reg_body(uint32_t* __restrict__ planes, const PrimeConst* __restrict__ consts,
                                                 const uint2* __restrict__ tw, uint32_t ps, uint32_t n2, uint32_t C,
                                                 uint32_t r, uint32_t op0, uint32_t col0, uint32_t bx, uint32_t by,
                                                 uint32_t bz) {
    const uint32_t col = col0 + bx * 256 + threadIdx.x, k = by, op = op0 + bz;
    const uint32_t p = consts[k].p;
    uint32_t* data = planes + (size_t(op) * r + k) * ps + col;
    const uint2* w = tw + size_t(k) * n2;
    uint32_t x[ROWS];
#pragma unroll
    for (int j = 0; j < ROWS; ++j) x[j] = data[size_t(j) * C];
#pragma unroll
    for (int m = 1, half = ROWS / 2; m < ROWS; m *= 2, half /= 2)
#pragma unroll
        for (int g = 0; g < m; ++g) {
            const uint2 t = w[m + g];
#pragma unroll
            for (int jr = 0; jr < half; ++jr) {
                // the next level multiplies the rows with its distance's bit set
                uint32_t &lo = x[2 * half * g + jr], &hi = x[2 * half * g + jr + half];
                if (half == 1 || !(jr & (half / 2))) ct_butterfly<true>(lo, hi, t, p);
                else ct_butterfly<false>(lo, hi, t, p);
            }
        }
#pragma unroll
    for (int j = 0; j < ROWS; ++j) data[size_t(j) * C] = x[j];
}

template <int ROWS>
__global__ __launch_bounds__(256) void ntt_columns_forward_reg(uint32_t* __restrict__ planes,
                                                               const PrimeConst* __restrict__ consts,
                                                               const uint2* __restrict__ tw, uint32_t ps,
                                                               uint32_t n2, uint32_t C, uint32_t r, uint32_t op0,
                                                               uint32_t col0) {
    forward_reg_body<ROWS>(planes, consts, tw, ps, n2, C, r, op0, col0, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Inverse row-spanning stages for 16 primes x 16 columns per block, then the
// residues v_{k,i} are written, XOR 0x80808080, into the CRT GEMM's operand
// tiles [n_pad/256][r_pad/16][256 coefficients][16 primes x 4 bytes] through
// an LDS transpose, so each coefficient's 64-byte K chunk is one store.
// ROWS = 1 is a pure transpose (no stages).  Column groups g0 + [0, gridDim.x)
// of 16 columns each.
template <int ROWS>
__device__ __forceinline__ void inverse_tiles_body(const uint32_t* __restrict__ plane,
                                                   const PrimeConst* __restrict__ consts,
                                                   const uint2* __restrict__ tw, uint32_t ps, uint32_t n, uint32_t n2,
                                                   uint32_t C, uint32_t r, uint32_t ksteps, int8_t* __restrict__ tiles,
                                                   uint32_t g0, uint32_t bx, uint32_t by, uint32_t nx) {
    // lds[j][column][slot]: the four 16-byte groups of a column's 16 primes are
    // XOR-swizzled by column/2, so the transpose reads each 16-byte store as one
    // aligned 128-bit LDS read (8 lanes of a read pass: two columns, distinct
    // banks) and the 4-byte writes of a wave's 32-lane halves are at most 2-way
    // conflicted (4-way unswizzled).
    __shared__ __attribute__((aligned(16))) uint32_t lds[ROWS][16][16];
    auto slot = [](uint32_t c, uint32_t kk) { return ((((kk >> 2) ^ (c >> 1)) & 3u) << 2) | (kk & 3u); };
    const uint32_t kk = threadIdx.x >> 4, cc = threadIdx.x & 15;
    // A block reads 64 bytes of each row: half a 128-byte line, whose other half
    // is the next column group's.  Workgroups go to the 8 XCDs round robin by
    // linear id, so column groups 2m and 2m+1 are given to blocks 8 ids apart
    // (the same XCD when the grid's x extent is a multiple of 16): the second
    // read of each line hits that XCD's L2 instead of memory.
    const uint32_t cx = (nx & 15u) == 0 ? (bx & ~15u) | ((bx & 7u) << 1) | ((bx >> 3) & 1u) : bx;
    const uint32_t c0 = (g0 + cx) * 16, kg = by, k = kg * 16 + kk;
    uint32_t x[ROWS];
    if (k < r) {
        const uint32_t p = consts[k].p;
        const uint32_t* data = plane + size_t(k) * ps + c0 + cc;
        const uint2* w = tw + size_t(k) * n2;
#pragma unroll
        for (int j = 0; j < ROWS; ++j) x[j] = data[size_t(j) * C];
#pragma unroll
        for (int m = ROWS / 2, half = 1; m >= 1; m /= 2, half *= 2)
#pragma unroll
            for (int g = 0; g < m; ++g) {
                const uint2 t = w[m + g];
#pragma unroll
                for (int jr = 0; jr < half; ++jr) gs_butterfly(x[2 * half * g + jr], x[2 * half * g + jr + half], t, p);
            }
    } else {
#pragma unroll
        for (int j = 0; j < ROWS; ++j) x[j] = 0;
    }
#pragma unroll
    for (int j = 0; j < ROWS; ++j) lds[j][cc][slot(cc, kk)] = x[j] ^ 0x80808080u;
    __syncthreads();
    for (uint32_t idx = threadIdx.x; idx < uint32_t(ROWS) * 64; idx += 256) {
        const uint32_t q = idx & 3, c2 = (idx >> 2) & 15, j = idx >> 6;
        const uint32_t i = j * C + c0 + c2;
        if (i < n) {
            const v4u v = *reinterpret_cast<const v4u*>(&lds[j][c2][slot(c2, 4 * q)]);
            *reinterpret_cast<v4u*>(tiles + ((size_t(i >> 8) * ksteps + kg) * 256 + (i & 255)) * 64 + q * 16) = v;
        }
    }
}

template <int ROWS>
__global__ __launch_bounds__(256) void ntt_columns_inverse_tiles(const uint32_t* __restrict__ plane,
                                                                 const PrimeConst* __restrict__ consts,
                                                                 const uint2* __restrict__ tw, uint32_t ps,
                                                                 uint32_t n, uint32_t n2, uint32_t C, uint32_t r,
                                                                 uint32_t ksteps, int8_t* __restrict__ tiles,
                                                                 uint32_t g0) {
    inverse_tiles_body<ROWS>(plane, consts, tw, ps, n, n2, C, r, ksteps, tiles, g0, blockIdx.x, blockIdx.y, gridDim.x);
}

// Row stages held in registers: 256 threads x 8 values per operand, i.e. 2048
// values jj of one row of one prime (C = 2048), or, for N = C < 2048, the whole
// transforms of 2048 / C consecutive primes side by side (prime jj / C).  The
// butterfly levels are done three at a time, with an LDS exchange between
// groups:
//   layout A: jj = t + 256e      distances 1024, 512, 256
//   layout B: jj = 256(t/32) + (t%32) + 32e   distances 128, 64, 32
//   layout C: jj = 32(t/4) + (t%4) + 4e       distances 16, 8, 4
//   layout D: jj = 8t + e        distances 2, 1, and the base case (n1 <= 8)
// Forward runs the distances C/2 .. n1, the base case multiplies each n1-block
// mod (X^n1 - zeta), and the inverse climbs back from n1 to C/2.  (C <= 256
// starts and ends in layout B.)
//
// Bound by VALU issue where there are many blocks (N = 65536 with 1747 limbs:
// 1.12 ms, 95 % of the issue rate; 1.34 ms with every butterfly fully reduced),
// by latency where there are few, so each group's twiddles are fetched a group
// ahead (N = 65536 with 55 limbs 48 -> 45.5 us, N = 16384 with 28 limbs 12.8 ->
// 11.2 us).  Below C = 2048 it takes the place of the LDS kernel's one level per
// barrier: N = 1024 with 8 limbs 16.8 -> 6.3 us, a batch's N = 1024 products
// 40 -> 14 us.
// Reading the inverse twiddles out of the forward table (mirrored, half the
// twiddle bytes) and half the barriers both measured the same.
constexpr uint32_t kRowC = 2048;

__device__ __forceinline__ uint32_t layout_index(int layout, uint32_t t, int e) {
    switch (layout) {
        case 0: return t + 256u * e;
        case 1: return 256u * (t >> 5) + (t & 31u) + 32u * e;
        case 2: return 32u * (t >> 2) + (t & 3u) + 4u * e;
        default: return 8u * t + e;
    }
}

// The prime (of the block's) that value e belongs to, written so that the
// compiler sees where it is the same for a block, a wave or a thread.
template <int LOGC>
__device__ __forceinline__ uint32_t layout_prime(int layout, uint32_t t, int e) {
    if constexpr (LOGC == 11) return 0;
    if (layout == 0 && LOGC >= 8) return uint32_t(e) >> (LOGC - 8);
    if (layout == 1 && LOGC < 8) return ((t >> 5) << (8 - LOGC)) + (uint32_t(e) >> (LOGC - 5));
    const uint32_t k = t >> (LOGC - 3);
    return LOGC >= 9 ? uint32_t(__builtin_amdgcn_readfirstlane(int(k))) : k;
}

// The twiddles of one group of levels: level b (distance d = stride << b) has
// 4 >> b of them per thread, at tw[(4 >> b) - 1 ..].  In layout A they are the
// same for the whole block, in the others consecutive entries per thread.
struct RowTables {
    const uint2* tw;      // [r][n2]
    const PrimeConst* consts;
    uint32_t n2, k0, r;
    uint32_t base;        // (rows + row) * C: level d starts at base / 2d
    // primes past the last one are computed on its tables (and not stored)
    template <int LOGC>
    __device__ __forceinline__ uint32_t prime(uint32_t k) const {
        return LOGC == 11 || k0 + k < r ? k0 + k : r - 1;
    }
};

template <int LOGC>
__device__ __forceinline__ bool row_level(uint32_t d, uint32_t n1) {
    return d >= n1 && 2 * d <= (1u << LOGC);
}

template <int LOGC>
__device__ __forceinline__ void row_twiddles(uint2 (&tw)[7], const RowTables& tb, int layout, int levels, uint32_t t,
                                             uint32_t stride, uint32_t n1) {
#pragma unroll
    for (int b = 0; b < levels; ++b) {
        const uint32_t d = stride << b;
        if (!row_level<LOGC>(d, n1)) continue;
        const uint32_t shift = 31 - __clz(2 * d);
        const uint32_t first = layout == 0 ? 0 : (layout == 1 ? t >> 5 : layout == 2 ? t >> 2 : t) << (2 - b);
#pragma unroll
        for (uint32_t s = 0; s < (4u >> b); ++s) {
            const uint32_t k = layout_prime<LOGC>(layout, t, int(s << (b + 1)));
            const uint32_t g = LOGC == 11 ? first + s : (first + s) & ((1u << (LOGC - shift)) - 1);
            tw[(4u >> b) - 1 + s] = (tb.tw + size_t(tb.prime<LOGC>(k)) * tb.n2)[(tb.base >> shift) + g];
        }
    }
}

// Forward levels of one group.  `lazy_in`: the values are below 2p (left so by
// the group before); the ones the first level does not multiply are reduced
// first.  The last level of a group leaves its outputs below 2p, unless it is
// the transform's last (distance n1): then they are below p, or stay below 2p
// with `lazy_out`.
template <int LOGC>
__device__ __forceinline__ void row_forward_group(uint32_t (&x)[8], const uint2 (&tw)[7], const uint32_t (&p)[8],
                                                  int levels, uint32_t stride, uint32_t n1, bool lazy_in,
                                                  bool lazy_out) {
    if (lazy_in && row_level<LOGC>(stride << (levels - 1), n1)) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (!(e & (1 << (levels - 1)))) x[e] = min(x[e], x[e] - p[e]);
    }
#pragma unroll
    for (int b = levels - 1; b >= 0; --b) {
        const uint32_t d = stride << b;
        if (!row_level<LOGC>(d, n1)) continue;
        const bool last = d == n1;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e & (1 << b)) continue;
            const uint2 w = tw[(4 >> b) - 1 + (e >> (b + 1))];
            const bool reduce = last ? !lazy_out : b > 0 && !(e & (1 << (b - 1)));
            if (reduce) ct_butterfly<true>(x[e], x[e + (1 << b)], w, p[e]);
            else ct_butterfly<false>(x[e], x[e + (1 << b)], w, p[e]);
        }
    }
}

template <int LOGC>
__device__ __forceinline__ void row_inverse_group(uint32_t (&x)[8], const uint2 (&tw)[7], const uint32_t (&p)[8],
                                                  int levels, uint32_t stride, uint32_t n1) {
#pragma unroll
    for (int b = 0; b < levels; ++b) {
        if (!row_level<LOGC>(stride << b, n1)) continue;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (e & (1 << b)) continue;
            gs_butterfly(x[e], x[e + (1 << b)], tw[(4 >> b) - 1 + (e >> (b + 1))], p[e]);
        }
    }
}

// LDS slot of jj in the exchange buffer: jj + jj/8, one pad word after every 8.
// Unpadded, layouts C and D put 8 lanes of a wave on one bank (8-way conflicts);
// padded, no layout exceeds 2-way.  Each form is written out as a per-thread base
// plus a constant per element, so the padding costs no address arithmetic
// (a swizzle computed per element measured slower than the conflicts).
constexpr uint32_t kRowPadded = kRowC + kRowC / 8;

__device__ __forceinline__ uint32_t padded_index(int layout, uint32_t t, int e) {
    switch (layout) {
        case 0: return t + (t >> 3) + 288u * e;
        case 1: return 288u * (t >> 5) + (t & 31u) + ((t & 31u) >> 3) + 36u * e;
        case 2: return 36u * (t >> 2) + (t & 3u) + 4u * e + (e >> 1);
        default: return 9u * t + e;
    }
}

__device__ __forceinline__ void row_exchange(uint32_t* buf, uint32_t (&x)[8], int from, int to, uint32_t t) {
#pragma unroll
    for (int e = 0; e < 8; ++e) buf[padded_index(from, t, e)] = x[e];
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = buf[padded_index(to, t, e)];
    __syncthreads();
}

template <int LOGC, uint32_t N1>
__device__ __forceinline__ void rows_reg_body(uint32_t* __restrict__ planes, const uint32_t* __restrict__ bplanes,
                                              const PrimeConst* __restrict__ consts, const uint2* __restrict__ twf,
                                              const uint2* __restrict__ twi, uint32_t ps, uint32_t n2, uint32_t rows,
                                              uint32_t r, uint32_t row, uint32_t k0) {
    constexpr uint32_t n1 = N1, C = 1u << LOGC;
    constexpr int kFirst = LOGC >= 9 ? 0 : 1;  // layout of the loads and stores
    __shared__ uint32_t buf[2][kRowPadded];
    const uint32_t t = threadIdx.x;
    const RowTables fwd{twf, consts, n2, k0, r, (rows + row) * C}, inv{twi, consts, n2, k0, r, (rows + row) * C};
    uint2 wa[7], wb[7];
    uint32_t xa[8], xb[8];
    // the primes' values in each layout (D has C's)
    uint32_t pa[8], pb[8], pc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        if constexpr (kFirst == 0) pa[e] = consts[fwd.prime<LOGC>(layout_prime<LOGC>(0, t, e))].p;
        pb[e] = consts[fwd.prime<LOGC>(layout_prime<LOGC>(1, t, e))].p;
        pc[e] = consts[fwd.prime<LOGC>(layout_prime<LOGC>(2, t, e))].p;
    }
    auto place = [&](int e) {  // where value e lies in the planes, in the first layout
        const size_t k = fwd.prime<LOGC>(layout_prime<LOGC>(kFirst, t, e));
        return LOGC == 11 ? layout_index(kFirst, t, e) : k * ps + (layout_index(kFirst, t, e) & (C - 1));
    };
    if constexpr (LOGC == 11) {
        planes += size_t(k0) * ps + size_t(row) * C;
        bplanes += size_t(k0) * ps + size_t(row) * C;
    }
    if constexpr (kFirst == 0) row_twiddles<LOGC>(wa, fwd, 0, 3, t, 256, n1);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        xa[e] = planes[place(e)];
        xb[e] = bplanes[place(e)];
    }
    row_twiddles<LOGC>(wb, fwd, 1, 3, t, 32, n1);
    if constexpr (kFirst == 0) {
        row_forward_group<LOGC>(xa, wa, pa, 3, 256, n1, false, false);
        row_forward_group<LOGC>(xb, wa, pa, 3, 256, n1, false, false);
        row_exchange(buf[0], xa, 0, 1, t);
        row_exchange(buf[1], xb, 0, 1, t);
    }
    row_twiddles<LOGC>(wa, fwd, 2, 3, t, 4, n1);
    row_forward_group<LOGC>(xa, wb, pb, 3, 32, n1, kFirst == 0, false);
    row_forward_group<LOGC>(xb, wb, pb, 3, 32, n1, kFirst == 0, false);
    row_exchange(buf[0], xa, 1, 2, t);
    row_exchange(buf[1], xb, 1, 2, t);
    row_twiddles<LOGC>(wb, fwd, 3, 2, t, 1, n1);
    row_forward_group<LOGC>(xa, wa, pc, 3, 4, n1, true, false);
    row_forward_group<LOGC>(xb, wa, pc, 3, 4, n1, true, false);
    row_exchange(buf[0], xa, 2, 3, t);
    row_exchange(buf[1], xb, 2, 3, t);
    const uint32_t kd = fwd.prime<LOGC>(layout_prime<LOGC>(3, t, 0)), p = pc[0], pinv = consts[kd].pinv;
    const uint2* wf = twf + size_t(kd) * n2;
    row_twiddles<LOGC>(wa, inv, 3, 2, t, 1, n1);
    row_forward_group<LOGC>(xa, wb, pc, 2, 1, n1, true, N1 == 1);
    row_forward_group<LOGC>(xb, wb, pc, 2, 1, n1, true, false);

    // base case: thread t holds jj = 8t .. 8t+7, i.e. 8/n1 whole blocks.  Block g
    // is reduced mod (X^n1 - zeta_g): c_s = sum_{u<=s} a_u b_{s-u} + sum_{u>s}
    // a_u (zeta_g b_{s+n1-u}).  The wrapped factors zeta_g*b_v are formed once per
    // block (Shoup), so each output is one sum of n1 products and one REDC: four
    // products of residues stay below 4p^2 < 2p*2^32, and from there on p*2^32
    // is taken off (a minimum on the high word) before every second product.
    // With n1 = 1 the a values come unreduced: 2p*p < p*2^32.
    uint32_t xc[8];
    constexpr int n1i = int(N1);
#pragma unroll
    for (int blk0 = 0; blk0 < 8; blk0 += n1i) {
        uint32_t bw[n1i];  // bw[v] = zeta_g * b_v for v >= 1
        bw[0] = 0;
        if constexpr (n1i > 1) {
            const uint32_t gb = (row * C + ((8 * t + blk0) & (C - 1))) / n1;  // global block index
            uint2 w{0, 0};
            if (n2 != 1) w = wf[n2 / 2 + gb / 2];  // zeta_{2g} = w, zeta_{2g+1} = -w
#pragma unroll
            for (int v = 1; v < n1i; ++v) {
                const uint32_t b = xb[blk0 + v];
                uint32_t z;
                if (n2 == 1) {
                    z = b ? p - b : 0;  // zeta = -1
                } else {
                    z = mul_shoup(b, w.x, w.y, p);
                    if (gb & 1) z = z ? p - z : 0;
                }
                bw[v] = z;
            }
        }
#pragma unroll
        for (int s1 = 0; s1 < n1i; ++s1) {
            uint64_t acc = 0;
#pragma unroll
            for (int u = 0; u < n1i; ++u) {
                const uint32_t f = u <= s1 ? xb[blk0 + s1 - u] : bw[s1 + n1i - u];
                // at most two products on top of p*2^32, or four alone: below 2p*2^32
                if (u >= 4 && u % 2 == 0) {
                    const uint32_t hi = uint32_t(acc >> 32);
                    acc = (uint64_t(min(hi, hi - p)) << 32) | uint32_t(acc);
                }
                acc += uint64_t(xa[blk0 + u]) * f;
            }
            const uint32_t value = n1i == 1 ? redc(acc, p, pinv) : redc_wide(acc, p, pinv);
            xc[blk0 + s1] = value;
        }
    }

    row_twiddles<LOGC>(wb, inv, 2, 3, t, 4, n1);
    row_inverse_group<LOGC>(xc, wa, pc, 2, 1, n1);
    row_exchange(buf[0], xc, 3, 2, t);
    row_twiddles<LOGC>(wa, inv, 1, 3, t, 32, n1);
    row_inverse_group<LOGC>(xc, wb, pc, 3, 4, n1);
    row_exchange(buf[0], xc, 2, 1, t);
    if constexpr (kFirst == 0) row_twiddles<LOGC>(wb, inv, 0, 3, t, 256, n1);
    row_inverse_group<LOGC>(xc, wa, pb, 3, 32, n1);
    if constexpr (kFirst == 0) {
        row_exchange(buf[0], xc, 1, 0, t);
        row_inverse_group<LOGC>(xc, wb, pa, 3, 256, n1);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (LOGC == 11 || k0 + layout_prime<LOGC>(kFirst, t, e) < r) planes[place(e)] = xc[e];
}

// Blocks (row, k0): one prime per block with C = 2048, else 2048 / C from k0 on.
template <int LOGC, uint32_t N1>
__global__ __launch_bounds__(256, LOGC < 8 ? 4 : 8) void ntt_rows_reg(uint32_t* __restrict__ planes,
                                                       const uint32_t* __restrict__ bplanes,
                                                       const PrimeConst* __restrict__ consts,
                                                       const uint2* __restrict__ twf, const uint2* __restrict__ twi,
                                                       uint32_t ps, uint32_t n2, uint32_t rows, uint32_t r) {
    rows_reg_body<LOGC, N1>(planes, bplanes, consts, twf, twi, ps, n2, rows, r, blockIdx.x,
                            blockIdx.y * (kRowC >> LOGC));
}

// ---------------------------------------------------------------------------
// 6'. reconstruction, one wave per coefficient (q wider than 252 limbs, and some
// widths with few coefficients, reconstruct_variant): the coefficient's CRT word sums are coefficient-major (words[i][0 .. L+3]) and
// each lane takes one of 64 consecutive words per round, so every round is one
// 512-byte load and one 256-byte store, and N waves (not N lanes) keep the
// memory system busy.
//
//   K  = floor((E + 2^63) / 2^64), E = sum_j 2^32j D_{L+1+j} + corr_e
//   x_j = D_j + corr_t_j + K*negp_j - (Qe*q)_j            (|x_j| < 2^56)
//   R  = sum_j x_j 2^32j = T - Qe*q
// Qe is the Barrett quotient of T estimated from the four words of x from
// m = floor(s/32) - 1 up (all words from 0 when s < 64): the words below m
// shift that estimate by under 2^25 * 2^32m, i.e. under 2^-7 at the 2^s
// scale, so Ts is off by at most one and Qe lies in [Q-2, Q+1].  One pass
// normalizes x into 32-bit words (carry out of each round passed to the next)
// and compares R with q on the way; in the rare case R < 0 or R >= q, Qe is
// moved by one and the pass repeats, rewriting c.
// ---------------------------------------------------------------------------
struct WaveReconstructArgs {
    uint32_t n, ws, limbs, t_words;
    TileSet ts;  // output row k*256 + u is coefficient tile_at(ts, k)*256 + u
    uint32_t top_m, top_e, k_shift;
    uint64_t mu;
};

__device__ __forceinline__ int32_t from_lane_below(int32_t v, uint32_t lane) {
    const int32_t u = __shfl_up(v, 1, 64);
    return lane ? u : 0;
}

__device__ __forceinline__ int64_t read_lane64(int64_t v, int l) {
    const uint32_t lo = __builtin_amdgcn_readlane(int(uint32_t(v)), l);
    const uint32_t hi = __builtin_amdgcn_readlane(int(uint32_t(uint64_t(v) >> 32)), l);
    return int64_t((uint64_t(hi) << 32) | lo);
}

// Normalizes one round of 64 signed words x (lane j: |x_j| < 2^57) plus the
// wave-uniform carry into word 0 into 32-bit words; returns lane j's word and
// leaves in `carry` the carry into the next round's word 0.
__device__ __forceinline__ uint32_t normalize_round(int64_t x, int64_t& carry, uint32_t lane) {
    if (lane == 0) x += carry;
    const int32_t hi = int32_t(x >> 32);                              // |hi| < 2^25
    const int64_t v = int64_t(uint32_t(x)) + from_lane_below(hi, lane);  // (-2^25, 2^32 + 2^25)
    const int32_t cj = int32_t(v >> 32);                              // -1, 0 or 1
    const int64_t u = int64_t(uint32_t(v)) + from_lane_below(cj, lane);  // [-1, 2^32]
    const int32_t hi63 = __builtin_amdgcn_readlane(hi, 63), c63 = __builtin_amdgcn_readlane(cj, 63);
    uint32_t w = uint32_t(u);
    int64_t ripple = 0;
    if (__ballot(u < 0 || u > int64_t(0xFFFFFFFFu))) {
        // a word of -1 or 2^32 (rare): ripple its carry up the round
        int64_t r = 0;
        for (int l = 0; l < 64; ++l) {
            const int64_t t = read_lane64(u, l) + r;
            if (lane == uint32_t(l)) w = uint32_t(t);
            r = t >> 32;
        }
        ripple = r;
    }
    carry = int64_t(hi63) + c63 + ripple;
    return w;
}

__device__ __forceinline__ void reconstruct_waves_body(const int64_t* __restrict__ words, uint32_t* __restrict__ c,
                                                       const uint32_t* __restrict__ q,
                                                       const uint32_t* __restrict__ neg_p,
                                                       const uint32_t* __restrict__ corr_t,
                                                       const uint32_t* __restrict__ corr_e,
                                                       WaveReconstructArgs args, uint32_t bx) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t k = bx * 4 + (threadIdx.x >> 6);  // output row
    if (k >= args.ts.count * 256) return;  // whole waves
    const uint32_t i = tile_at(args.ts, k / 256) * 256 + k % 256;
    if (i >= args.n) return;
    const uint32_t L = args.limbs, tw = args.t_words;
    const int64_t* d = words + size_t(i) * args.ws;
    uint32_t* out = c + size_t(k) * L;

    // K = floor((E + 2^63) / 2^64)
    uint32_t ew[4];
    {
        int64_t carry = 0;
        for (uint32_t j = 0; j < 4; ++j) {
            const int64_t x = (j < 3 ? d[L + 1 + j] : 0) + int64_t(corr_e[j]) + carry;
            ew[j] = uint32_t(uint64_t(x));
            carry = x >> 32;
        }
    }
    const int64_t kq = int64_t(uint64_t(ew[2]) + (uint64_t(ew[3]) << 32) + ((uint64_t(ew[1]) + 0x80000000ull) >> 32));

    // Barrett estimate from the top four words: S = sum_t x_{m+t} 2^32t mod 2^128
    // equals (T - [words below m]) / 2^32m exactly (|S| < 2^126).
    uint64_t qe;
    {
        unsigned __int128 sum = 0;
        for (uint32_t t = 0; t < 4; ++t) {
            const uint32_t j = args.top_m + t;
            if (j >= tw) break;
            const int64_t x = (j <= L ? d[j] : 0) + int64_t(corr_t[j]) + (j < L ? kq * int64_t(neg_p[j]) : 0);
            sum += (unsigned __int128)(__int128)x << (32 * t);
        }
        __int128 ts = __int128(sum) >> args.top_e;
        if (ts < 0) ts = 0;
        qe = uint64_t(((unsigned __int128)uint64_t(ts) * args.mu) >> args.k_shift);
    }

    // A round's inputs (lane j of words j0 .. j0+63): D_j + corr_t_j + K*negp_j and
    // the three words of q that word j of Qe*q needs.  Every load is
    // unconditional, its index clamped into its table and the value selected
    // afterwards, so a round carries no divergent branches, and the loads of a
    // round are issued two rounds before it is normalized.  K < 2^32 (it is
    // below the number of primes), so K*negp_j is one 32 x 32-bit product.
    struct Round {  // the raw loads; masked and combined only when the round is used
        int64_t d;
        uint32_t ct, np, qj, qm1, qm2;
    };
    const uint32_t k32 = uint32_t(kq);
    auto fetch = [&](uint32_t j0) {
        const uint32_t j = j0 + lane;
        const uint32_t jq = j < L ? j : L - 1, jq1 = j - 1 < L ? j - 1 : 0, jq2 = j - 2 < L ? j - 2 : 0;
        return Round{d[j <= L ? j : L], corr_t[j < tw ? j : tw - 1], neg_p[jq], q[jq], q[jq1], q[jq2]};
    };
    for (int pass = 0; pass < 6; ++pass) {
        const uint64_t q0 = uint32_t(qe), q1 = uint32_t(qe >> 32);
        int64_t carry = 0;
        int cmp = 0;  // sign of R - q over the words so far (decided by the highest differing word)
        auto round = [&](const Round& in, uint32_t j0) {
            const uint32_t j = j0 + lane;
            const uint32_t qj = j < L ? in.qj : 0;
            const uint32_t qm1 = j >= 1 && j - 1 < L ? in.qm1 : 0;
            const uint32_t qm2 = j >= 2 && j - 2 < L ? in.qm2 : 0;
            // word j of Qe*q: lo(q0 q_j) + hi(q0 q_{j-1}) + lo(q1 q_{j-1}) + hi(q1 q_{j-2})
            const uint64_t pa = q0 * qj, pb = q0 * qm1, pc = q1 * qm1, pd = q1 * qm2;
            const int64_t sub = int64_t(uint32_t(pa)) + int64_t(pb >> 32) + int64_t(uint32_t(pc)) + int64_t(pd >> 32);
            const int64_t kr = j < L ? int64_t(uint64_t(k32) * in.np) : 0;
            const int64_t x = j < tw ? (j <= L ? in.d : 0) + int64_t(in.ct) + kr - sub : 0;
            const uint32_t w = normalize_round(x, carry, lane);
            if (j < L) out[j] = w;
            const uint64_t differ = __ballot(w != qj);
            if (differ) {
                const int top = 63 - __clzll(differ);
                cmp = uint32_t(__builtin_amdgcn_readlane(int(w), top)) > uint32_t(__builtin_amdgcn_readlane(int(qj), top))
                          ? 1
                          : -1;
            }
        };
        // Three register sets in rotation (no copies between them, which would
        // wait for the loads): each set is refilled right after its round.
        Round r0 = fetch(0), r1 = fetch(64), r2;
        for (uint32_t j0 = 0; j0 < tw; j0 += 192) {
            r2 = fetch(j0 + 128);
            round(r0, j0);
            if (j0 + 64 >= tw) break;
            r0 = fetch(j0 + 192);
            round(r1, j0 + 64);
            if (j0 + 128 >= tw) break;
            r1 = fetch(j0 + 256);
            round(r2, j0 + 128);
        }
        if (carry < 0) {
            --qe;  // R < 0
        } else if (carry > 0 || cmp >= 0) {
            ++qe;  // R >= q
        } else {
            break;
        }
    }
}

__global__ __launch_bounds__(256) void reconstruct_waves(const int64_t* __restrict__ words, uint32_t* __restrict__ c,
                                                         const uint32_t* __restrict__ q,
                                                         const uint32_t* __restrict__ neg_p,
                                                         const uint32_t* __restrict__ corr_t,
                                                         const uint32_t* __restrict__ corr_e,
                                                         WaveReconstructArgs args) {
    reconstruct_waves_body(words, c, q, neg_p, corr_t, corr_e, args, blockIdx.x);
}

// ---------------------------------------------------------------------------
// Reconstruction of one coefficient by G lanes, four consecutive words each (the
// formulas are those of reconstruct_waves): shared by the fused kernel and the
// one for wider q.
// ---------------------------------------------------------------------------

// What one lane needs to form K and the Barrett estimate Qe of a coefficient:
// the same constants for every lane.
struct QuotientWords {
    uint32_t ce[4], top_c[4], top_n[4];
    __device__ __forceinline__ void load(const uint32_t* __restrict__ neg_p, const uint32_t* __restrict__ corr_t,
                                         const uint32_t* __restrict__ corr_e, uint32_t L, uint32_t tw,
                                         uint32_t top_m) {
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
            const uint32_t j = top_m + t;
            const uint32_t cv = corr_t[j < tw ? j : tw - 1], nv = neg_p[j < L ? j : L - 1];
            top_c[t] = j < tw ? cv : 0;
            top_n[t] = j < L ? nv : 0;
            ce[t] = corr_e[t];
        }
    }
    // d: the coefficient's word sums.  Leaves K in k32.
    __device__ __forceinline__ uint64_t quotient(const int64_t* d, uint32_t L, uint32_t top_m, uint32_t top_e,
                                                 uint32_t k_shift, uint64_t mu, uint32_t& k32) const {
        int64_t e[3], dt[4];
#pragma unroll
        for (uint32_t j = 0; j < 3; ++j) e[j] = d[L + 1 + j];
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
            const uint32_t j = top_m + t;
            dt[t] = d[j <= L ? j : L];
            if (j > L) dt[t] = 0;
        }
        // K = floor((E + 2^63) / 2^64)
        uint32_t ew[4];
        int64_t carry = 0;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const int64_t x = (j < 3 ? e[j] : 0) + int64_t(ce[j]) + carry;
            ew[j] = uint32_t(uint64_t(x));
            carry = x >> 32;
        }
        const uint32_t k = uint32_t(ew[2] + ((uint64_t(ew[1]) + 0x80000000ull) >> 32));
        k32 = k;
        // the four words at top_m (words past the last are zero)
        unsigned __int128 sum = 0;
#pragma unroll
        for (uint32_t t = 0; t < 4; ++t) {
            const int64_t x = dt[t] + int64_t(top_c[t]) + int64_t(uint64_t(k) * top_n[t]);
            sum += (unsigned __int128)(__int128)x << (32 * t);
        }
        __int128 ts = __int128(sum) >> top_e;
        if (ts < 0) ts = 0;
        return uint64_t(((unsigned __int128)uint64_t(ts) * mu) >> k_shift);
    }
};

// Lane g of a group of G: its four words of the constants, and the group's part
// of a reconstruction.  Whole waves call reconstruct together.
template <int G>
struct LaneWords {
    uint32_t g, end;  // end: the lane of word L + 1, the last one that holds anything
    uint32_t ct[4], np[4], qv[6];  // qv[u + 2] = q[4g + u], two words below included
    __device__ __forceinline__ void load(const uint32_t* __restrict__ q, const uint32_t* __restrict__ neg_p,
                                         const uint32_t* __restrict__ corr_t, uint32_t L, uint32_t tw, uint32_t lane) {
        g = lane;
        end = (L + 1) / 4;
        // (every load unconditional, its index clamped, the value selected after)
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t j = 4 * g + u;
            const uint32_t cv = corr_t[j < tw ? j : tw - 1], nv = neg_p[j < L ? j : L - 1];
            ct[u] = j < tw ? cv : 0;
            np[u] = j < L ? nv : 0;
        }
#pragma unroll
        for (uint32_t u = 0; u < 6; ++u) {
            const uint32_t j = 4 * g + u - 2;  // wraps above L below word 0
            const uint32_t v = q[j < L ? j : L - 1];
            qv[u] = j < L ? v : 0;
        }
    }
    // Adds cin to the lane's words; returns the carry out.
    static __device__ __forceinline__ int32_t add_carry(uint32_t (&w)[4], int32_t cin) {
        int64_t t = cin;
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            t += int64_t(w[u]);
            w[u] = uint32_t(uint64_t(t));
            t >>= 32;
        }
        return int32_t(t);
    }
    // Passes each lane's carry to the next lane of its group until none is left;
    // lane `end`'s carries add up in `top` (0 on the other lanes).  The lanes above
    // it hold nothing and stay out: a coefficient's top words are often -1 until
    // the carry from below arrives, and that borrow and its undoing would walk
    // through every empty lane (128 limbs, 31 empty lanes of 64, N = 4096: 18.0
    // us with the carries added up by the last lane, 5.8 so).
    __device__ __forceinline__ void settle(uint32_t (&w)[4], int32_t carry, int32_t& top) const {
        for (;;) {
            if (g == end) top += carry;
            int32_t cin;
            if constexpr (G <= 16) cin = __builtin_amdgcn_update_dpp(0, carry, 0x111, 0xF, 0xF, true);  // row_shr:1
            else cin = __shfl_up(carry, 1, 64);
            if (g == 0 || g > end) cin = 0;
            if (!__ballot(cin != 0)) break;
            carry = add_carry(w, cin);
        }
    }
    // The lane's word sums out of the coefficient's, d (those past word L hold E
    // or nothing of the row's, and are 0 here).
    __device__ __forceinline__ void sums(const int64_t* d, uint32_t L, int64_t (&x)[4]) const {
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t j = 4 * g + u;
            const int64_t v = d[j <= L ? j : L];
            x[u] = j <= L ? v : 0;
        }
    }
    // The lane's words of (T - Qe*q) mod q, from its word sums; `valid` false:
    // they are garbage, and so are the words.
    __device__ __forceinline__ void reconstruct(const int64_t (&d)[4], uint64_t qe, uint32_t k32, bool valid,
                                                uint32_t (&w)[4]) const {
        const uint32_t lane = threadIdx.x & 63, shift = lane & ~uint32_t(G - 1), last = shift + end;
        constexpr uint64_t mask = G == 64 ? ~uint64_t(0) : (uint64_t(1) << (G & 63)) - 1;
        // R = T - Qe*q: this lane's four words and the carry out of them
        const uint64_t q0 = uint32_t(qe), q1 = uint32_t(qe >> 32);
        int32_t top = 0;
        {
            uint64_t pa = q0 * qv[1], pc = q1 * qv[1], pc2 = q1 * qv[0];
            int64_t carry = 0;
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const uint64_t a = q0 * qv[u + 2];
                const int64_t sub = int64_t(uint32_t(a)) + int64_t(pa >> 32) + int64_t(uint32_t(pc)) + int64_t(pc2 >> 32);
                carry += d[u] + int64_t(ct[u]) + int64_t(uint64_t(k32) * np[u]) - sub;
                w[u] = uint32_t(uint64_t(carry));
                carry >>= 32;
                pa = a, pc2 = pc, pc = q1 * qv[u + 2];
            }
            settle(w, int32_t(carry), top);
        }
        for (int pass = 0; pass < 6; ++pass) {
            bool gt = false, lt = false;
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {  // the highest differing word decides
                if (w[u] != qv[u + 2]) gt = w[u] > qv[u + 2], lt = !gt;
            }
            const uint64_t gm = (__ballot(gt) >> shift) & mask, lm = (__ballot(lt) >> shift) & mask;
            const bool neg = (__ballot(top < 0) >> last) & 1, pos = (__ballot(top > 0) >> last) & 1;
            const int32_t adj = !valid ? 0 : neg ? 1 : (pos || gm >= lm) ? -1 : 0;
            if (!__ballot(adj != 0)) break;
            int64_t carry = 0;
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                carry += int64_t(w[u]) + (adj > 0 ? int64_t(qv[u + 2]) : adj < 0 ? -int64_t(qv[u + 2]) : 0);
                w[u] = uint32_t(uint64_t(carry));
                carry >>= 32;
            }
            settle(w, int32_t(carry), top);
        }
    }
};

// ---------------------------------------------------------------------------
// 6''. reconstruction for q of 61 to 252 limbs, from the CRT GEMM's sums in
// memory: G = 32 or 64 lanes per coefficient (up to 128 or 256 words), blocks of
// NP passes of 256 / G coefficients, whose sums are all loaded ahead; K and Qe
// by one lane per coefficient as in the fused kernel.
// reconstruct_waves spends a whole wave on every 64 words and forms K and Qe in
// all 64 lanes: N = 8192 with 226 limbs 18.1 us, here 8.4; a
// batch of 64 small products 70 us, here 23.
// ---------------------------------------------------------------------------

template <int G, int NP>
__device__ __forceinline__ void reconstruct_wide_body(const int64_t* __restrict__ words, uint32_t* __restrict__ c,
                                                      const uint32_t* __restrict__ q,
                                                      const uint32_t* __restrict__ neg_p,
                                                      const uint32_t* __restrict__ corr_t,
                                                      const uint32_t* __restrict__ corr_e,
                                                      const WaveReconstructArgs& args, uint32_t bx) {
    typedef uint32_t v4u_word __attribute__((ext_vector_type(4), aligned(4)));  // 4-byte aligned
    constexpr uint32_t T = 256 / G * NP;
    __shared__ uint64_t quotient[T];
    __shared__ uint32_t multiple[T];
    const uint32_t tid = threadIdx.x, g = tid % G, L = args.limbs;
    const uint32_t k0 = bx * T, i0 = tile_at(args.ts, k0 / kTile) * kTile + k0 % kTile;
    if (i0 >= args.n) return;  // whole block
    const int64_t* rows = words + size_t(i0) * args.ws;
    LaneWords<G> lw;
    int64_t d[NP][4];
    lw.load(q, neg_p, corr_t, L, args.t_words, g);
#pragma unroll
    for (uint32_t ps = 0; ps < NP; ++ps) lw.sums(rows + size_t(tid / G + ps * (256 / G)) * args.ws, L, d[ps]);
    if (tid < T) {
        QuotientWords qw;
        qw.load(neg_p, corr_t, corr_e, L, args.t_words, args.top_m);
        quotient[tid] = qw.quotient(rows + size_t(tid) * args.ws, L, args.top_m, args.top_e, args.k_shift, args.mu,
                                    multiple[tid]);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t ps = 0; ps < NP; ++ps) {
        const uint32_t cl = tid / G + ps * (256 / G);
        uint32_t w[4];
        const bool valid = i0 + cl < args.n;
        lw.reconstruct(d[ps], quotient[cl], multiple[cl], valid, w);
        uint32_t* out = c + size_t(k0 + cl) * L + 4 * g;
        if (!valid) continue;
        if (4 * g + 4 <= L) {
            *reinterpret_cast<v4u_word*>(out) = v4u{w[0], w[1], w[2], w[3]};
        } else {
#pragma unroll
            for (uint32_t u = 0; u < 3; ++u)
                if (4 * g + u < L) out[u] = w[u];
        }
    }
}

template <int G, int NP>
__global__ __launch_bounds__(256) void reconstruct_wide(const int64_t* __restrict__ words, uint32_t* __restrict__ c,
                                                        const uint32_t* __restrict__ q,
                                                        const uint32_t* __restrict__ neg_p,
                                                        const uint32_t* __restrict__ corr_t,
                                                        const uint32_t* __restrict__ corr_e,
                                                        WaveReconstructArgs args) {
    reconstruct_wide_body<G, NP>(words, c, q, neg_p, corr_t, corr_e, args, blockIdx.x);
}

// ---------------------------------------------------------------------------
// 5+6. CRT GEMM and reconstruction in one kernel, for q of up to 60 limbs (at
// most 64 word sums): a block of NW waves owns 16 NW coefficients and all
// their word sums, so the sums never leave the CU.
//
//  * GEMM: every wave holds 64 weight rows (16 word sums) x 16 WM coefficients;
//    WM waves cover the word sums (16 WM >= crt_words), the others split the
//    coefficients.  The block's residue bytes (all K steps) come in by
//    direct-to-LDS loads behind one barrier; the weights are read as MFMA
//    fragments straight from global memory, two K steps ahead.  Only the K
//    steps that hold primes run (the padded ones have zero weights).
//    With up to 8 transform rows (ROWS > 0) there is no operand tile: the row
//    stage's planes are read, the inverse column stages done in registers, one
//    thread per (prime, column), and the residues written to LDS in its place
//    (N = 16384 with 28 limbs: 9.2 us, where the inverse column kernel took 5.3
//    and this one 6.6; a launch less).  Wider columns would need more
//    coefficients per block than its accumulators hold.
//  * The int64 word sums go to LDS, coefficient-major, over the operand bytes.
//  * One lane per coefficient forms K and the Barrett estimate Qe, by the
//    formulas of reconstruct_waves.
//  * Then G = 4 WM lanes per coefficient, four consecutive words each: a lane
//    carries through its own words and hands its carry to the next lane (a row
//    shift within 16 lanes); a second hand-over happens only when four words in
//    a row ripple.  A Qe that was off (by two at most) is mended by adding or
//    subtracting q in place.
//  * c is staged in LDS and stored as one contiguous run of words, each once,
//    so c may be pinned host memory.
// What bounds it at N = 65536 with 55 limbs (23.4 us, of which 17-19 us inside
// a block): the weight fragments' way from L2 (7 us: 67 MB, every block reads
// all of them) and the carry chains (4 us).  It replaces a CRT GEMM that wrote
// 8 (L+4) bytes per coefficient and a kernel that walked them with one lane per
// coefficient: 15.7 + 27.9 us there, 6.7 + 7.1 against 4.2 us at N = 1024 with
// 8 limbs, 13.8 + 8.0 against 10.0 us at N = 131072 with 4.
// ---------------------------------------------------------------------------
struct CrtFusedArgs {
    uint32_t n, limbs, t_words;
    uint32_t ksteps, kstride;  // K steps that hold primes; K steps of a residue tile
    uint32_t r, ps, n2;        // primes; plane row stride, twiddles per prime (residues read from the planes)
    TileSet ts;                // output row k*256 + u is coefficient tile_at(ts, k)*256 + u
    uint32_t top_m, top_e, k_shift;
    uint64_t mu;
};

constexpr uint32_t fused_row_words(uint32_t wm) { return 16 * wm + 2; }  // int64 per coefficient, 16-byte rows

constexpr size_t fused_lds_bytes(uint32_t wm, uint32_t nw, uint32_t ksteps) {
    const size_t operands = size_t(ksteps) * 16 * nw * kTK, sums = size_t(16) * nw * fused_row_words(wm) * 8;
    return operands > sums ? operands : sums;
}

template <int WM, int NW, int ROWS>
__device__ __forceinline__ void crt_reconstruct_body(const int8_t* __restrict__ wtiles,
                                                     const int8_t* __restrict__ rtiles,
                                                     const uint32_t* __restrict__ planes,
                                                     const PrimeConst* __restrict__ consts,
                                                     const uint2* __restrict__ twi, uint32_t* __restrict__ c,
                                                     const uint32_t* __restrict__ q,
                                                     const uint32_t* __restrict__ neg_p,
                                                     const uint32_t* __restrict__ corr_t,
                                                     const uint32_t* __restrict__ corr_e, const CrtFusedArgs& args,
                                                     uint32_t bx, int8_t* lds) {
    constexpr uint32_t NT = WM, G = 4 * WM, S = fused_row_words(WM), T = 16 * NW, NTH = 64 * NW;
    __shared__ uint64_t quotient[T];
    __shared__ uint32_t multiple[T];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t wm = wave % WM, wn = wave / WM;
    const uint32_t L = args.limbs, tw = args.t_words, ksteps = args.ksteps;
    // The block's coefficients: 16 NW consecutive ones of the set, or (ROWS > 1)
    // CW columns of the transform's [ROWS][2048] matrix, row after row.  Columns
    // are 64 or 128 bytes wide: two blocks 8 ids apart, on one XCD, share the
    // 128-byte lines (as in inverse_tiles_body).
    constexpr uint32_t CW = ROWS > 1 ? T / ROWS : T;
    const uint32_t cx = (bx & ~15u) | ((bx & 7u) << 1) | ((bx >> 3) & 1u);
    const uint32_t k0 = ROWS > 1 ? cx * CW : bx * T;
    const uint32_t tile = tile_at(args.ts, k0 / kTile), i0 = ROWS > 1 ? k0 : tile * kTile + k0 % kTile;

    // operand bytes, a row's chunk (16 bytes: four primes) swizzled as in swz
    if constexpr (ROWS > 1) {
        // inverse column stages: thread -> (prime, column), as inverse_tiles_body
        for (uint32_t w = tid; w < ksteps * 16 * CW; w += NTH) {
            const uint32_t k = w / CW, col = w % CW, kk = k < args.r ? k : args.r - 1;
            const uint32_t p = consts[kk].p;
            const uint32_t* src = planes + size_t(kk) * args.ps + k0 + col;
            const uint2* tw = twi + size_t(kk) * args.n2;
            uint32_t x[ROWS];
#pragma unroll
            for (int j = 0; j < ROWS; ++j) x[j] = src[j * kRowWidth];
#pragma unroll
            for (int m = ROWS / 2, half = 1; m >= 1; m /= 2, half *= 2)
#pragma unroll
                for (int g = 0; g < m; ++g) {
                    const uint2 t = tw[m + g];
#pragma unroll
                    for (int jr = 0; jr < half; ++jr)
                        gs_butterfly(x[2 * half * g + jr], x[2 * half * g + jr + half], t, p);
                }
#pragma unroll
            for (int j = 0; j < ROWS; ++j)
                *reinterpret_cast<u32_alias*>(lds + k / 16 * (T * kTK) + swz(j * CW + col, k % 16 / 4) + k % 4 * 4) =
                    x[j] ^ 0x80808080u;
        }
    } else if constexpr (ROWS == 1) {  // thread -> coefficient tid % T, primes 4 (tid / T) .. + 3 of each K step
        const uint32_t cf = tid % T, chunk = tid / T;
        const uint32_t* src = planes + i0 + cf;
        for (uint32_t ks = 0; ks < ksteps; ++ks) {
            v4u x;
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {  // primes past the last have zero weights: read the last one's again
                const uint32_t k = ks * 16 + chunk * 4 + u;
                x[u] = src[size_t(k < args.r ? k : args.r - 1) * args.ps];
            }
            *reinterpret_cast<v4u*>(lds + ks * (T * kTK) + swz(cf, chunk)) = x ^ 0x80808080u;
        }
    } else {  // slot tid of a K step holds row tid>>2
        const uint32_t row = tid >> 2, chunk = (tid & 3) ^ ((row >> 1) & 3);
        const int8_t* src = rtiles + size_t(tile) * args.kstride * kTileBytes + (k0 % kTile + row) * kTK + chunk * 16;
        for (uint32_t ks = 0; ks < ksteps; ++ks)
            __builtin_amdgcn_global_load_lds(reinterpret_cast<const void*>(src + size_t(ks) * kTileBytes),
                                             (__attribute__((address_space(3))) void*)(lds + ks * (T * kTK) + wave * 1024),
                                             16, 0, 0);
    }
    const v4i* ap = reinterpret_cast<const v4i*>(wtiles + (wm * kWaveRows + (lane & 15)) * kTK + (lane >> 4) * 16);
    v4i acc[kWaveM][NT], f0[kWaveM], f1[kWaveM], f2[kWaveM];
    auto load_a = [&](uint32_t ks, v4i (&f)[kWaveM]) {
#pragma unroll
        for (uint32_t mi = 0; mi < kWaveM; ++mi) f[mi] = ap[size_t(ks) * (kTileBytes / 16) + mi * 64];
    };
    load_a(0, f0);
    load_a(ksteps > 1 ? 1 : 0, f1);
#pragma unroll
    for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
        for (uint32_t ni = 0; ni < NT; ++ni) acc[mi][ni] = v4i{0, 0, 0, 0};
    __syncthreads();
    auto step = [&](uint32_t ks, const v4i (&fa)[kWaveM], v4i (&refill)[kWaveM]) {
        load_a(ks + 2 < ksteps ? ks + 2 : ksteps - 1, refill);  // past the end: the last step again
        v4i fb[NT];
#pragma unroll
        for (uint32_t ni = 0; ni < NT; ++ni)
            fb[ni] = *reinterpret_cast<const v4i*>(lds + ks * (T * kTK) +
                                                   swz((wn * NT + ni) * 16 + (lane & 15), lane >> 4));
#pragma unroll
        for (uint32_t mi = 0; mi < kWaveM; ++mi)
#pragma unroll
            for (uint32_t ni = 0; ni < NT; ++ni)
                acc[mi][ni] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[mi], fb[ni], acc[mi][ni], 0, 0, 0);
    };
    uint32_t ks = 0;  // three fragment sets in rotation
    for (; ks + 3 <= ksteps; ks += 3) {
        step(ks, f0, f2);
        step(ks + 1, f1, f0);
        step(ks + 2, f2, f1);
    }
    if (ks < ksteps) step(ks, f0, f2);
    if (ks + 1 < ksteps) step(ks + 1, f1, f0);
    const uint32_t g = tid % G;
    LaneWords<G> lw;
    lw.load(q, neg_p, corr_t, L, tw, g);
    QuotientWords qw;
    qw.load(neg_p, corr_t, corr_e, L, tw, args.top_m);
    __syncthreads();  // every wave has read the operand bytes; the sums go over them
    int64_t* sums = reinterpret_cast<int64_t*>(lds);
    const DigitScales ds = digit_scales();
#pragma unroll
    for (uint32_t ni = 0; ni < NT; ++ni)
#pragma unroll
        for (uint32_t mi = 0; mi < kWaveM; ++mi)
            sums[((wn * NT + ni) * 16 + (lane & 15)) * S + wm * 16 + mi * 4 + (lane >> 4)] = combine4(acc[mi][ni], ds);
    __syncthreads();

    // K and the Barrett quotient Qe: one lane per coefficient, for all of them
    if (tid < T) quotient[tid] = qw.quotient(sums + tid * S, L, args.top_m, args.top_e, args.k_shift, args.mu, multiple[tid]);
    __syncthreads();
#pragma unroll 1
    for (uint32_t cl = tid / G; cl < T; cl += 64 * NW / G) {  // whole waves: T G is a multiple of the threads
        uint32_t w[4];
        int64_t d[4];
        lw.sums(sums + cl * S, L, d);
        lw.reconstruct(d, quotient[cl], multiple[cl], ROWS > 1 || i0 + cl < args.n, w);
        // c over the coefficient's own sums (its lanes have read them all)
        u32_alias* cw = reinterpret_cast<u32_alias*>(lds + size_t(cl) * S * 8);
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            if (4 * g + u < L) cw[4 * g + u] = w[u];
    }
    __syncthreads();
    const uint32_t rows = ROWS > 1 ? T : i0 < args.n ? (args.n - i0 < T ? args.n - i0 : T) : 0;
    uint32_t* out = c + size_t(k0) * L;
    const u32_alias* staged = reinterpret_cast<const u32_alias*>(lds);
    const uint32_t dq = NTH / L, dr = NTH % L;  // (row, column) of word k, stepped by NTH words
    uint32_t row = tid / L, col = tid % L;
    for (uint32_t k = tid; k < rows * L; k += NTH) {
        // rows of one matrix row are consecutive coefficients
        const size_t at = ROWS > 1 ? size_t(row / CW * (kRowWidth - CW)) * L + k : k;
        out[at] = staged[row * (2 * S) + col];
        row += dq;
        col += dr;
        if (col >= L) {
            col -= L;
            ++row;
        }
    }
}

template <int WM, int NW, int ROWS>
__global__ __launch_bounds__(64 * NW, 4) void crt_reconstruct(const int8_t* __restrict__ wtiles,
                                                       const int8_t* __restrict__ rtiles,
                                                       const uint32_t* __restrict__ planes,
                                                       const PrimeConst* __restrict__ consts,
                                                       const uint2* __restrict__ twi, uint32_t* __restrict__ c,
                                                       const uint32_t* __restrict__ q,
                                                       const uint32_t* __restrict__ neg_p,
                                                       const uint32_t* __restrict__ corr_t,
                                                       const uint32_t* __restrict__ corr_e, CrtFusedArgs args) {
    extern __shared__ __attribute__((aligned(16))) int8_t dyn_lds[];
    crt_reconstruct_body<WM, NW, ROWS>(wtiles, rtiles, planes, consts, twi, c, q, neg_p, corr_t, corr_e, args, blockIdx.x, dyn_lds);
}

// ---------------------------------------------------------------------------
// 6''. Grouped launches: one stage of many products in one launch.  Entry j of
// a launch owns blocks [start[j], start[j+1]) and runs them as the blocks of
// product item[j]'s own launch of that stage (kernels.hpp, GroupItem).
// ---------------------------------------------------------------------------
// GroupItem as the kernels read it.  A pointer read from memory could point
// anywhere, which costs flat loads and stores (they wait for LDS and memory
// together); these point to global memory, and their types say so.
#ifdef __HIP_DEVICE_COMPILE__
#define PM_GLOBAL __attribute__((address_space(1)))
#else
#define PM_GLOBAL
#endif
struct GroupView {
    uint32_t n, n_pad, limbs, r, r_pad, conv_rows, conv_k, crt_rows, crt_k, crt_words, ws, t_words;
    uint32_t n1, n2, rows, row_width, k_shift, top_m, top_e;
    uint32_t conv_ks, conv_nt, conv_split, conv_columns;  // short conversion (launch_convert)
    uint64_t mu;
    const PM_GLOBAL PrimeConst* consts;
    const PM_GLOBAL int8_t* wconv;
    const PM_GLOBAL uint2* tw_fwd;
    const PM_GLOBAL uint2* tw_inv;
    const PM_GLOBAL int8_t* wcrt;
    const PM_GLOBAL uint32_t* q;
    const PM_GLOBAL uint32_t* neg_p;
    const PM_GLOBAL uint32_t* corr_t;
    const PM_GLOBAL uint32_t* corr_e;
    const PM_GLOBAL uint32_t* a;
    const PM_GLOBAL uint32_t* b;
    PM_GLOBAL uint32_t* c;
    PM_GLOBAL int8_t* packed;
    PM_GLOBAL uint32_t* planes;
    PM_GLOBAL int8_t* rtiles;
    PM_GLOBAL int64_t* words;
};
static_assert(sizeof(GroupView) == sizeof(GroupItem), "GroupView has GroupItem's layout");

template <class T>
__device__ __forceinline__ T* in_global(PM_GLOBAL T* p) {
    return (T*)p;
}

struct GroupLaunch {
    const GroupView* items;
    const uint32_t* start;  // count + 1 block offsets
    const uint32_t* item;   // the product of each entry
    uint32_t count;
};

// The product owning this block (a binary search over the offsets, the same
// for every thread of the block) and the block's index in that product's grid.
__device__ __forceinline__ const GroupView& group_entry(const GroupLaunch& g, uint32_t& local) {
    const uint32_t b = blockIdx.x;
    uint32_t lo = 0, hi = g.count;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (g.start[mid] <= b)
            lo = mid;
        else
            hi = mid;
    }
    local = b - g.start[lo];
    return g.items[g.item[lo]];
}

__device__ __forceinline__ TileSet every_tile(const GroupView& it) { return tile_range(0, it.n_pad / kTile); }

__global__ __launch_bounds__(256) void pack_group(GroupLaunch g) {
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    pack_body(in_global(it.a), in_global(it.b), reinterpret_cast<uint32_t*>(in_global(it.packed)), it.n, it.limbs, it.conv_k / kTK, it.n_pad / kTile,
              every_tile(it), 0, 2, local);
}

__global__ __launch_bounds__(512) void conversion_group(GroupLaunch g) {
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    conversion_body<2>(in_global(it.wconv), in_global(it.packed), in_global(it.consts), in_global(it.planes), it.n, it.n_pad, it.r, it.r_pad, it.conv_rows,
                    it.conv_k / kTK, every_tile(it), 0, 2, local);
}

// The grouped kernels of a stage hold several of its variants, chosen per
// product, so that products of every size share one launch and its tail (the
// batch of 64 small products: six launches of the CRT stage took 81 us, one
// takes 43).

// grid per product: (2 n_pad / 64 NT, prime splits)
__global__ __launch_bounds__(256, 3) void convert_group(GroupLaunch g) {
    extern __shared__ __attribute__((aligned(16))) int8_t dyn_lds[];
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    const uint32_t nx = 2 * it.n_pad / (64 * it.conv_nt);
    const ConvertArgs args{it.n, it.n_pad, it.limbs, it.r, it.r_pad, it.conv_rows, it.conv_k / kTK, it.n2,
                           every_tile(it), 0};
    auto run = [&](auto ks, auto nt, auto rows) {
        convert_body<ks(), nt(), rows()>(in_global(it.a), in_global(it.b), in_global(it.wconv), in_global(it.consts),
                                         in_global(it.tw_fwd), in_global(it.planes), args, local % nx, local / nx,
                                         it.conv_split, dyn_lds);
    };
    using std::integral_constant;
    auto columns = [&](auto ks, auto nt) {
        if (it.conv_columns == 1) run(ks, nt, integral_constant<int, 1>());
        else if (it.conv_columns == 2) run(ks, nt, integral_constant<int, 2>());
        else if constexpr (nt() == 4) run(ks, nt, integral_constant<int, 4>());
    };
    switch (it.conv_ks) {  // convert_plan's wide waves
        case 1: columns(integral_constant<int, 1>(), integral_constant<int, 4>()); break;
        case 2: columns(integral_constant<int, 2>(), integral_constant<int, 4>()); break;
        case 4: columns(integral_constant<int, 4>(), integral_constant<int, 4>()); break;
        default: columns(integral_constant<int, 8>(), integral_constant<int, 2>()); break;
    }
}

// grid per product: (row_width / 256, r, 2).  ROWS = 8 holds 2, 4 and 8 rows.
template <int ROWS>
__global__ __launch_bounds__(256) void forward_reg_group(GroupLaunch g) {
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    const uint32_t nx = it.row_width / 256, bx = local % nx, rest = local / nx;
    auto run = [&](auto rows) {
        forward_reg_body<rows()>(in_global(it.planes), in_global(it.consts), in_global(it.tw_fwd), it.n_pad, it.n2,
                                 it.row_width, it.r_pad, 0, 0, bx, rest % it.r, rest / it.r);
    };
    if (ROWS > 8) run(std::integral_constant<int, ROWS>());
    else if (it.rows == 2) run(std::integral_constant<int, 2>());
    else if (it.rows == 4) run(std::integral_constant<int, 4>());
    else run(std::integral_constant<int, 8>());
}

// grid per product: (rows, r / primes per block)
template <int LOGC, uint32_t N1>
__global__ __launch_bounds__(256, LOGC < 8 ? 4 : 8) void rows_reg_group(GroupLaunch g) {
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    rows_reg_body<LOGC, N1>(in_global(it.planes), in_global(it.planes) + size_t(it.r_pad) * it.n_pad,
                            in_global(it.consts), in_global(it.tw_fwd), in_global(it.tw_inv), it.n_pad, it.n2, it.rows,
                            it.r, local % it.rows, local / it.rows * (kRowC >> LOGC));
}

__global__ __launch_bounds__(256) void rows_product_group(GroupLaunch g) {
    extern __shared__ uint32_t lds32[];
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    rows_product_body(in_global(it.planes), in_global(it.planes) + size_t(it.r_pad) * it.n_pad, in_global(it.consts), in_global(it.tw_fwd), in_global(it.tw_inv), it.n_pad,
                      it.n1, it.n2, it.row_width, it.rows, lds32, local % it.rows, local / it.rows);
}

// grid per product: (row_width / 16, r_pad / 16)
// ROWS = 8 holds 1, 2, 4 and 8 rows.
template <int ROWS>
__global__ __launch_bounds__(256) void inverse_tiles_group(GroupLaunch g) {
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    const uint32_t nx = it.row_width / 16;
    auto run = [&](auto rows) {
        inverse_tiles_body<rows()>(in_global(it.planes), in_global(it.consts), in_global(it.tw_inv), it.n_pad, it.n,
                                   it.n2, it.row_width, it.r, it.r_pad / 16, in_global(it.rtiles), 0, local % nx,
                                   local / nx, nx);
    };
    if (ROWS > 8) run(std::integral_constant<int, ROWS>());
    else if (it.rows == 1) run(std::integral_constant<int, 1>());
    else if (it.rows == 2) run(std::integral_constant<int, 2>());
    else if (it.rows == 4) run(std::integral_constant<int, 4>());
    else run(std::integral_constant<int, 8>());
}

__global__ __launch_bounds__(512) void crt_group(GroupLaunch g) {
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    crt_body<2>(in_global(it.wcrt), in_global(it.rtiles), in_global(it.words), it.n, it.crt_rows,
                it.crt_k / kTK, (it.r + 15) / 16, it.crt_words, it.ws, every_tile(it), local);
}

// The variants' quotient arrays add up to 9 KB of LDS here (768 bytes in a kernel
// of one variant), so that a CU holds three blocks of the widest, not four, and
// the registers are 12 short (20 bytes of scratch a lane).
__global__ __launch_bounds__(256, 4) void crt_reconstruct_group(GroupLaunch g) {
    extern __shared__ __attribute__((aligned(16))) int8_t dyn_lds[];
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    const CrtFusedArgs args{it.n, it.limbs, it.t_words, (it.r + 15) / 16, it.r_pad / 16, it.r, it.n_pad,
                            it.n2, every_tile(it), it.top_m, it.top_e, it.k_shift, it.mu};
    auto run = [&](auto wm, auto rows) {
        crt_reconstruct_body<wm(), 4, rows()>(in_global(it.wcrt), in_global(it.rtiles), in_global(it.planes),
                                              in_global(it.consts), in_global(it.tw_inv), in_global(it.c), in_global(it.q), in_global(it.neg_p),
                                                     in_global(it.corr_t), in_global(it.corr_e), args, local, dyn_lds);
    };
    auto residues = [&](auto wm) {
        switch (it.rows) {  // residues_from_planes, up to 4 rows
            case 1: run(wm, std::integral_constant<int, 1>()); break;
            case 2: run(wm, std::integral_constant<int, 2>()); break;
            case 4: run(wm, std::integral_constant<int, 4>()); break;
            default: run(wm, std::integral_constant<int, 0>()); break;
        }
    };
    switch (fused_waves(it.crt_words)) {
        case 1: residues(std::integral_constant<int, 1>()); break;
        case 2: residues(std::integral_constant<int, 2>()); break;
        default: residues(std::integral_constant<int, 4>()); break;
    }
}

__global__ __launch_bounds__(256) void reconstruct_wide_group(GroupLaunch g) {
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    const WaveReconstructArgs args{it.n, it.ws, it.limbs, it.t_words, every_tile(it),
                                   it.top_m, it.top_e, it.k_shift, it.mu};
    auto run = [&](auto lanes, auto passes) {
        reconstruct_wide_body<lanes(), passes()>(in_global(it.words), in_global(it.c), in_global(it.q),
                                                 in_global(it.neg_p), in_global(it.corr_t), in_global(it.corr_e), args,
                                                 local);
    };
    if (it.crt_words <= 128) run(std::integral_constant<int, 32>(), std::integral_constant<int, 2>());
    else run(std::integral_constant<int, 64>(), std::integral_constant<int, 4>());
}

__global__ __launch_bounds__(256) void reconstruct_waves_group(GroupLaunch g) {
    uint32_t local;
    const GroupView& it = group_entry(g, local);
    const WaveReconstructArgs args{it.n, it.ws, it.limbs, it.t_words, every_tile(it),
                                   it.top_m, it.top_e, it.k_shift, it.mu};
    reconstruct_waves_body(in_global(it.words), in_global(it.c), in_global(it.q), in_global(it.neg_p), in_global(it.corr_t), in_global(it.corr_e), args, local);
}

__global__ void fill_zero(uint32_t* __restrict__ c, size_t words) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < words) c[i] = 0;
}

// ---------------------------------------------------------------------------
// 7. plan-time tables (host equivalents in plan.cpp, build_plan).
// ---------------------------------------------------------------------------
// x*y mod p for x, y < p < 2^31 with rcp = floor((2^64-1)/p): for t = xy < 2^62
// the estimate hi64(t*rcp) lies in (t/p - 2, t/p], so two corrections finish.
__device__ __forceinline__ uint32_t mulmod_rcp(uint32_t x, uint32_t y, uint32_t p, uint64_t rcp) {
    const uint64_t t = uint64_t(x) * y;
    uint64_t r = t - __umul64hi(t, rcp) * p;
    if (r >= p) r -= p;
    if (r >= p) r -= p;
    return uint32_t(r);
}

__device__ __forceinline__ uint32_t powmod_rcp(uint32_t b, uint32_t e, uint32_t p, uint64_t rcp) {
    uint32_t r = 1;
    for (; e; e >>= 1) {
        if (e & 1) r = mulmod_rcp(r, b, p, rcp);
        b = mulmod_rcp(b, b, p, rcp);
    }
    return r;
}

// Shoup quotient floor(w * 2^32 / p) for w < p, by the same estimate.
__device__ __forceinline__ uint32_t shoup_rcp(uint32_t w, uint32_t p, uint64_t rcp) {
    const uint64_t t = uint64_t(w) << 32;
    uint64_t q = __umul64hi(t, rcp), r = t - q * p;
    if (r >= p) { r -= p; ++q; }
    if (r >= p) ++q;
    return uint32_t(q);
}

// beta_k = n2^-1 * 2^32 * P_k^-1 mod p_k, with P_k mod p_k = prod_{j != k} p_j
// formed by one block per prime (strided products, then a tree).
__global__ __launch_bounds__(256) void table_beta(const PrimeConst* __restrict__ consts,
                                                  const uint64_t* __restrict__ rcp, uint32_t* __restrict__ beta,
                                                  uint32_t r, uint32_t n2) {
    __shared__ uint32_t part[256];
    const uint32_t k = blockIdx.x, t = threadIdx.x;
    const uint32_t p = consts[k].p;
    const uint64_t rc = rcp[k];
    uint32_t prod = 1;
    for (uint32_t j = t; j < r; j += 256)
        if (j != k) prod = mulmod_rcp(prod, consts[j].p % p, p, rc);
    part[t] = prod;
    __syncthreads();
    for (uint32_t w = 128; w; w >>= 1) {
        if (t < w) part[t] = mulmod_rcp(part[t], part[t + w], p, rc);
        __syncthreads();
    }
    if (t == 0) {
        const uint32_t radix = uint32_t((uint64_t(1) << 32) % p);
        const uint32_t n2_inv = powmod_rcp(n2 % p, p - 2, p, rc);
        const uint32_t pk_inv = powmod_rcp(part[0], p - 2, p, rc);
        beta[k] = mulmod_rcp(mulmod_rcp(n2_inv, radix, p, rc), pk_inv, p, rc);
    }
}

// tw[k][j] = (psi^e, Shoup quotient) with e = bitrev(j) over log2(n2) bits; the
// inverse table uses psi^-1.  grid (column blocks, r).
__global__ __launch_bounds__(256) void table_twiddles(const PrimeConst* __restrict__ consts,
                                                      const uint64_t* __restrict__ rcp,
                                                      const uint32_t* __restrict__ psi, uint32_t* __restrict__ fwd,
                                                      uint32_t* __restrict__ inv, uint32_t n2, uint32_t log_n2) {
    __shared__ uint32_t pf[32], pi[32];  // psi^(2^i), psi^-(2^i)
    const uint32_t k = blockIdx.y;
    const uint32_t p = consts[k].p;
    const uint64_t rc = rcp[k];
    if (threadIdx.x == 0) {
        uint32_t a = psi[2 * k], b = psi[2 * k + 1];
        for (uint32_t i = 0; i < log_n2; ++i) {
            pf[i] = a;
            pi[i] = b;
            a = mulmod_rcp(a, a, p, rc);
            b = mulmod_rcp(b, b, p, rc);
        }
    }
    __syncthreads();
    for (uint32_t j = blockIdx.x * 256 + threadIdx.x; j < n2; j += gridDim.x * 256) {
        const uint32_t e = log_n2 ? __brev(j) >> (32 - log_n2) : 0;
        uint32_t w = 1, wi = 1;
        for (uint32_t i = 0; i < log_n2; ++i)
            if ((e >> i) & 1) {
                w = mulmod_rcp(w, pf[i], p, rc);
                wi = mulmod_rcp(wi, pi[i], p, rc);
            }
        const size_t at = (size_t(k) * n2 + j) * 2;
        *reinterpret_cast<uint2*>(fwd + at) = make_uint2(w, shoup_rcp(w, p, rc));
        *reinterpret_cast<uint2*>(inv + at) = make_uint2(wi, shoup_rcp(wi, p, rc));
    }
}

// Conversion weights of operand op for prime k: columns j < 4L hold
// lambda * 256^j mod p (lambda = 2^32 for a, 2^32 * beta_k for b), centered and
// split into four signed digits (rows 4k+d); columns j >= 4L are zero.  The
// block also forms off = 128 * sum_j centered_j mod p.  Each thread writes four
// consecutive columns of a row as one word into the tiled matrix (pre-zeroed).
// grid (r, 2).
__global__ __launch_bounds__(256) void table_conversion(PrimeConst* __restrict__ consts,
                                                        const uint64_t* __restrict__ rcp,
                                                        const uint32_t* __restrict__ beta,
                                                        int8_t* __restrict__ wtiles, uint32_t conv_rows,
                                                        uint32_t conv_k, uint32_t limbs) {
    __shared__ int64_t part[256];
    const uint32_t k = blockIdx.x, op = blockIdx.y, t = threadIdx.x;
    const uint32_t p = consts[k].p;
    const uint64_t rc = rcp[k];
    const uint32_t radix = uint32_t((uint64_t(1) << 32) % p);
    const uint32_t lambda = op ? mulmod_rcp(radix, beta[k], p, rc) : radix;
    const uint32_t ksteps = conv_k / kTK, num_m = conv_rows / kTile, kbytes = 4 * limbs;
    const uint32_t step = powmod_rcp(256, 4 * 256, p, rc);  // 256^(columns per block pass)
    uint32_t cur = mulmod_rcp(lambda, powmod_rcp(256, 4 * t, p, rc), p, rc);
    int64_t sum = 0;
    for (uint32_t j0 = 4 * t; j0 < conv_k; j0 += 4 * 256) {
        uint32_t word[4] = {0, 0, 0, 0};
        uint32_t w = cur;
        for (uint32_t i = 0; i < 4; ++i) {
            if (j0 + i < kbytes) {
                int64_t x = w > p / 2 ? int64_t(w) - p : int64_t(w);
                sum += x;
                for (uint32_t d = 0; d < 4; ++d) {
                    const int64_t e = ((x + 128) & 255) - 128;
                    word[d] |= uint32_t(uint8_t(int8_t(e))) << (8 * i);
                    x = (x - e) >> 8;
                }
            }
            w = mulmod_rcp(w, 256, p, rc);
        }
        for (uint32_t d = 0; d < 4; ++d) {
            if (!word[d]) continue;
            const uint32_t row = 4 * k + d;
            const size_t at = ((size_t(op * num_m + row / kTile) * ksteps + j0 / kTK) * kTile + row % kTile) * kTK +
                              j0 % kTK;
            *reinterpret_cast<uint32_t*>(wtiles + at) = word[d];
        }
        cur = mulmod_rcp(cur, step, p, rc);
    }
    part[t] = sum;
    __syncthreads();
    for (uint32_t w = 128; w; w >>= 1) {
        if (t < w) part[t] += part[t + w];
        __syncthreads();
    }
    if (t == 0) {
        int64_t off = (128 * part[0]) % int64_t(p);
        if (off < 0) off += p;
        if (op) consts[k].off_b = uint32_t(off);
        else consts[k].off_a = uint32_t(off);
    }
}

// CRT weights of prime k (one thread each): column 4k+d of row c holds signed
// digit c-d of M_k (rows 0 .. 4L+3) and, from row 4(L+1) on, signed digit
// c-4(L+1)-d of rcp_k.  Row c's four columns are one word whose byte d is digit
// c-d: a sliding window over the digit stream.  Matrix pre-zeroed.
__global__ __launch_bounds__(64) void table_crt(const uint32_t* __restrict__ m_mod_q,
                                                const uint64_t* __restrict__ rcp, int8_t* __restrict__ wtiles,
                                                uint32_t r, uint32_t limbs, uint32_t crt_k) {
    const uint32_t k = blockIdx.x * 64 + threadIdx.x;
    if (k >= r) return;
    const uint32_t ksteps = crt_k / kTK, col = 4 * k;
    auto put = [&](uint32_t row, uint32_t word) {
        if (!word) return;
        const size_t at = ((size_t(row / kTile) * ksteps + col / kTK) * kTile + row % kTile) * kTK + col % kTK;
        *reinterpret_cast<uint32_t*>(wtiles + at) = word;
    };
    const uint32_t* m = m_mod_q + size_t(k) * limbs;
    const uint32_t md = 4 * limbs + 1;
    uint32_t window = 0;
    int carry = 0;
    for (uint32_t c = 0; c < md + 3; ++c) {
        int digit = 0;
        if (c < md) {
            const int x = (c / 4 < limbs ? int((m[c / 4] >> (8 * (c % 4))) & 255u) : 0) + carry;
            carry = x >= 128;
            digit = carry ? x - 256 : x;
        }
        window = (window << 8) | uint8_t(int8_t(digit));
        put(c, window);
    }
    const uint64_t rv = rcp[k];
    const uint32_t base = 4 * (limbs + 1);
    window = 0;
    carry = 0;
    for (uint32_t c = 0; c < 6 + 3; ++c) {
        int digit = 0;
        if (c < 6) {
            const int x = int((rv >> (8 * c)) & 255u) + carry;
            carry = x >= 128;
            digit = carry ? x - 256 : x;
        }
        window = (window << 8) | uint8_t(int8_t(digit));
        put(base + c, window);
    }
}

uint32_t column_width(const Shape& s) {
    uint32_t cw = 8192 / s.rows;
    if (cw > s.row_width) cw = s.row_width;
    if (cw < 1) cw = 1;
    return cw;
}

// Every tile of `ts` must be one of the plan's: a set past them would have the
// kernels read and write past the working buffers.
void check_tiles(const Shape& s, const TileSet& ts, const char* what) {
    const uint64_t ntiles = s.n_pad / kTile;
    const bool ok = ts.count != 0 && ts.w != 0 && ts.count % ts.w == 0 &&
                    uint64_t(ts.t0) + uint64_t(ts.count / ts.w - 1) * ts.stride + (ts.w - 1) < ntiles;
    if (!ok) throw std::invalid_argument(std::string(what) + ": coefficient tiles outside the plan's");
}

// Strips [strip_begin, strip_end) of 256 columns; (0, ~0u) is every column.
bool whole_columns(const Shape& s, uint32_t strip_begin, uint32_t strip_end, const char* what) {
    if (strip_begin == 0 && strip_end == ~0u) return true;
    if (s.row_width % 256 != 0 || s.rows < 2 || s.rows > 64 || strip_begin >= strip_end ||
        strip_end > s.row_width / 256)
        throw std::invalid_argument(std::string(what) + ": column strips outside the transform's columns");
    return false;
}

}  // namespace

size_t packed_operand_bytes(const Shape& s) { return size_t(2) * s.n_pad * s.conv_k; }

void launch_pack(const Shape& s, const uint32_t* a, const uint32_t* b, int8_t* packed, const TileSet& ts,
                 uint32_t op0, uint32_t nops, hipStream_t stream) {
    check_tiles(s, ts, "pack_operands");
    const uint32_t ksteps = s.conv_k / kTK, ntiles = s.n_pad / kTile;
    const size_t rows = size_t(nops) * ts.count * kTile;  // 4 waves per block
    const uint32_t per_block = 4 * kPackRows;
    dim3 grid(uint32_t((rows + per_block - 1) / per_block));
    hipLaunchKernelGGL(pack_operands, grid, dim3(256), 0, stream, a, b, reinterpret_cast<uint32_t*>(packed), s.n,
                       s.limbs, ksteps, ntiles, ts, op0, nops);
    check_launch("pack_operands");
}

void launch_conversion(const Shape& s, const DeviceTables& t, const int8_t* packed, uint32_t* planes,
                       const TileSet& ts, uint32_t op0, uint32_t nops, hipStream_t stream) {
    check_tiles(s, ts, "conversion_gemm");
    const uint32_t blocks = (s.conv_rows / kTile) * nops * ts.count;
    if (gemm_halves(blocks))
        hipLaunchKernelGGL(conversion_gemm<1>, dim3(2 * blocks), dim3(256), 0, stream, t.wconv, packed, t.consts,
                           planes, s.n, s.n_pad, s.r, s.r_pad, s.conv_rows, s.conv_k / kTK, ts, op0, nops);
    else
        hipLaunchKernelGGL(conversion_gemm<2>, dim3(blocks), dim3(512), 0, stream, t.wconv, packed, t.consts, planes,
                           s.n, s.n_pad, s.r, s.r_pad, s.conv_rows, s.conv_k / kTK, ts, op0, nops);
    check_launch("conversion_gemm");
}

void launch_convert(const Shape& s, const DeviceTables& t, const uint32_t* a, const uint32_t* b, uint32_t* planes,
                    const TileSet& ts, uint32_t op0, uint32_t nops, bool columns, hipStream_t stream) {
    check_tiles(s, ts, "convert");
    if (!conversion_short(s)) throw std::logic_error("convert: operands wider than a wave holds");
    if (columns && !conversion_columns(s, ts)) throw std::logic_error("convert: column stages not held by a lane");
    const uint32_t ksteps = s.conv_k / kTK;
    const ConvertArgs args{s.n, s.n_pad, s.limbs, s.r, s.r_pad, s.conv_rows, ksteps, s.n2, ts, op0};
    const ConvertPlan cp = convert_plan(s, nops * ts.count, kConvertBlocks, columns);
    const dim3 grid(nops * ts.count * 4 / cp.nt, cp.split);
    if (!convert_compiled(cp)) throw std::logic_error("convert: no kernel of the variant the shape takes");
#define PM_CONVERT(K, N, R)                                                                              \
    if (cp.ks == K && cp.nt == N && cp.rows == R)                                                        \
        hipLaunchKernelGGL((convert<K, N, R>), grid, dim3(256), convert_lds_bytes(ksteps, s.r, cp.split, R), \
                           stream, a, b, t.wconv, t.consts, t.tw_fwd, planes, args);
    PM_CONVERT_VARIANTS(PM_CONVERT)
#undef PM_CONVERT
    check_launch("convert");
}

void launch_ntt_forward_columns(const Shape& s, const DeviceTables& t, uint32_t* planes, uint32_t op0,
                                uint32_t nops, hipStream_t stream, uint32_t strip_begin, uint32_t strip_end) {
    const bool whole = whole_columns(s, strip_begin, strip_end, "ntt_columns_forward");
    if (s.rows < 2) return;
    const uint32_t ps = s.n_pad, r = s.r_pad, C = s.row_width;
    if (C % 256 == 0 && s.rows <= 64) {
        if (!columns_compiled(s.rows)) throw std::logic_error("ntt_columns_forward: no kernel of this row count");
        const uint32_t s0 = whole ? 0 : strip_begin, s1 = whole ? C / 256 : strip_end;
        dim3 grid(s1 - s0, s.r, nops);
        switch (s.rows) {
#define PM_FWD(R)                                                                                                \
    case R:                                                                                                      \
        hipLaunchKernelGGL(ntt_columns_forward_reg<R>, grid, dim3(256), 0, stream, planes, t.consts, t.tw_fwd, ps, \
                           s.n2, C, r, op0, s0 * 256);                                                           \
        break;
            PM_FWD(2) PM_FWD(4) PM_FWD(8) PM_FWD(16) PM_FWD(32) PM_FWD(64)
#undef PM_FWD
        }
    } else {
        const uint32_t cw = column_width(s);
        dim3 grid(C / cw, s.r, nops);
        hipLaunchKernelGGL(ntt_columns_forward, grid, dim3(256), size_t(s.rows) * cw * 4, stream, planes, t.consts,
                           t.tw_fwd, ps, s.n2, C, s.rows, cw, r, op0);
    }
    check_launch("ntt_columns_forward");
}

void launch_ntt_rows_product(const Shape& s, const DeviceTables& t, uint32_t* planes, const uint32_t* bplanes,
                             hipStream_t stream) {
    const uint32_t ps = s.n_pad, logc = row_variant(s.row_width, s.n1);
    if (logc) {
        const uint32_t per = kRowC >> logc;  // primes per block
        const dim3 grid(s.rows, (s.r + per - 1) / per);
        if (!rows_compiled(logc, s.n1)) throw std::logic_error("ntt_rows_product: no kernel of the variant the shape takes");
#define PM_ROWS(LC, B)                                                                                      \
    if (logc == LC && s.n1 == B)                                                                            \
        hipLaunchKernelGGL((ntt_rows_reg<LC, B>), grid, dim3(256), 0, stream, planes, bplanes, t.consts,     \
                           t.tw_fwd, t.tw_inv, ps, s.n2, s.rows, s.r);
        PM_ROWS_VARIANTS(PM_ROWS)
#undef PM_ROWS
    } else {
        const dim3 grid(s.rows, s.r);
        hipLaunchKernelGGL(ntt_rows_product, grid, dim3(256), size_t(2) * s.row_width * 4, stream, planes, bplanes,
                           t.consts, t.tw_fwd, t.tw_inv, ps, s.n1, s.n2, s.row_width, s.rows);
    }
    check_launch("ntt_rows_product");
}

void launch_ntt_inverse_columns(const Shape& s, const DeviceTables& t, uint32_t* planes, int8_t* rtiles,
                                hipStream_t stream, uint32_t strip_begin, uint32_t strip_end) {
    const bool whole = whole_columns(s, strip_begin, strip_end, "ntt_columns_inverse");
    const uint32_t ps = s.n_pad, ksteps = s.r_pad / 16;
    if (s.row_width % 16 == 0 && s.rows <= 64) {
        if (!columns_compiled(s.rows)) throw std::logic_error("ntt_columns_inverse: no kernel of this row count");
        const uint32_t g0 = whole ? 0 : strip_begin * 16, g1 = whole ? s.row_width / 16 : strip_end * 16;
        dim3 grid(g1 - g0, s.r_pad / 16);
        switch (s.rows) {
#define PM_INV(R)                                                                                              \
    case R:                                                                                                    \
        hipLaunchKernelGGL(ntt_columns_inverse_tiles<R>, grid, dim3(256), 0, stream, planes, t.consts, t.tw_inv, \
                           ps, s.n, s.n2, s.row_width, s.r, ksteps, rtiles, g0);                               \
        break;
            PM_INV(1) PM_INV(2) PM_INV(4) PM_INV(8) PM_INV(16) PM_INV(32) PM_INV(64)
#undef PM_INV
        }
    } else {
        // large or narrow shapes: LDS column stages, then a pure transpose into the tiles
        if (s.rows >= 2) {
            const uint32_t cw = column_width(s);
            dim3 grid(s.row_width / cw, s.r);
            hipLaunchKernelGGL(ntt_columns_inverse, grid, dim3(256), size_t(s.rows) * cw * 4, stream, planes,
                               t.consts, t.tw_inv, ps, s.n2, s.row_width, s.rows, cw);
            check_launch("ntt_columns_inverse");
        }
        dim3 grid((s.n + 15) / 16, s.r_pad / 16);
        hipLaunchKernelGGL(ntt_columns_inverse_tiles<1>, grid, dim3(256), 0, stream, planes, t.consts, t.tw_inv, ps,
                           s.n, s.n2, s.n, s.r, ksteps, rtiles, 0u);
    }
    check_launch("ntt_columns_inverse_tiles");
}

void launch_crt(const Shape& s, const DeviceTables& t, const int8_t* rtiles, int64_t* words, const TileSet& ts,
                hipStream_t stream) {
    check_tiles(s, ts, "crt_gemm");
    if (crt_few_blocks(s.crt_rows, ts.count)) {
        const dim3 grid((s.crt_words + 15) / 16 * ts.count * 4);
        hipLaunchKernelGGL(crt_small, grid, dim3(256), 0, stream, t.wcrt, rtiles, words, s.n, s.crt_k / kTK,
                           (s.r + 15) / 16, s.crt_words, word_stride(s), ts);
        check_launch("crt_small");
        return;
    }
    const uint32_t blocks = (s.crt_rows / kTile) * ts.count;
    if (gemm_halves(blocks))
        hipLaunchKernelGGL(crt_gemm<1>, dim3(2 * blocks), dim3(256), 0, stream, t.wcrt, rtiles, words, s.n,
                           s.crt_rows, s.crt_k / kTK, (s.r + 15) / 16, s.crt_words, word_stride(s), ts);
    else
        hipLaunchKernelGGL(crt_gemm<2>, dim3(blocks), dim3(512), 0, stream, t.wcrt, rtiles, words, s.n,
                           s.crt_rows, s.crt_k / kTK, (s.r + 15) / 16, s.crt_words, word_stride(s), ts);
    check_launch("crt_gemm");
}

namespace {

// Barrett window: the four words of x from m up (m = floor(s/32) - 1, or 0 below s = 64)
uint32_t barrett_top(const Shape& s) { return s.s_shift >= 64 ? s.s_shift / 32 - 1 : 0; }

}  // namespace

void launch_crt_reconstruct(const Shape& s, const DeviceTables& t, const int8_t* rtiles, const uint32_t* planes,
                            uint32_t* c, const TileSet& ts, hipStream_t stream) {
    check_tiles(s, ts, "crt_reconstruct");
    if (!reconstruct_fused(s)) throw std::logic_error("crt_reconstruct: more word sums than a block holds");
    const uint32_t top_m = barrett_top(s), ksteps = (s.r + 15) / 16, wm = fused_waves(s.crt_words);
    const CrtFusedArgs args{s.n, s.limbs, s.t_words, ksteps, s.r_pad / 16, s.r, s.n_pad, s.n2, ts, top_m, s.s_shift - 32 * top_m,
                            s.k_shift, s.mu};
#define PM_FUSED(W, NW, P)                                                                                       \
    hipLaunchKernelGGL((crt_reconstruct<W, NW, P>), dim3(ts.count * (kTile / (16 * NW))), dim3(64 * NW),             \
                       fused_lds_bytes(W, NW, ksteps), stream, t.wcrt, rtiles, planes, t.consts, t.tw_inv, c, t.q, t.neg_p, t.corr_t,         \
                       t.corr_e, args)
    // Blocks of eight waves read the weights half as often per coefficient (at
    // N = 65536 with 55 limbs 23.4 us against 29.2 us with four waves); below
    // 65536 coefficients there are too few of them, and smaller blocks start sooner.
    const bool wide = ts.count >= 256;
#define PM_FUSED_WM(NW, R)                    \
    do {                                      \
        if (wm == 1) PM_FUSED(1, NW, R);      \
        else if (wm == 2) PM_FUSED(2, NW, R); \
        else PM_FUSED(4, NW, R);              \
    } while (0)
    if (!residues_from_planes(s, ts)) {
        if (wide) PM_FUSED_WM(8, 0);
        else PM_FUSED_WM(4, 0);
    } else if (s.rows == 1) {
        PM_FUSED_WM(4, 1);
    } else if (s.rows == 2) {
        PM_FUSED_WM(4, 2);
    } else if (s.rows == 4) {
        PM_FUSED_WM(4, 4);
    } else {
        PM_FUSED_WM(8, 8);
    }
#undef PM_FUSED_WM
#undef PM_FUSED
    check_launch("crt_reconstruct");
}

void launch_reconstruct(const Shape& s, const DeviceTables& t, const int64_t* words, uint32_t* c, const TileSet& ts,
                        hipStream_t stream) {
    check_tiles(s, ts, "reconstruct");
    const uint32_t top_m = barrett_top(s);
    WaveReconstructArgs args{s.n, word_stride(s), s.limbs, s.t_words, ts,
                             top_m, s.s_shift - 32 * top_m, s.k_shift, s.mu};
#define PM_WIDE(G, NP)                                                                                              \
    hipLaunchKernelGGL((reconstruct_wide<G, NP>), dim3(ts.count * (kTile / (256 / G * NP))), dim3(256), 0, stream,   \
                       words, c, t.q, t.neg_p, t.corr_t, t.corr_e, args)
    switch (reconstruct_variant(s, ts.count)) {
        case Reconstruction::kLanes32: PM_WIDE(32, 2); break;
        case Reconstruction::kLanes64: PM_WIDE(64, 4); break;
        case Reconstruction::kWave:
            hipLaunchKernelGGL(reconstruct_waves, dim3(ts.count * 64), dim3(256), 0, stream, words, c, t.q, t.neg_p,
                               t.corr_t, t.corr_e, args);
            break;
    }
#undef PM_WIDE
    check_launch("reconstruct");
}

GroupItem group_item(const Shape& s, const DeviceTables& t, const DeviceWork& w, const uint32_t* a,
                     const uint32_t* b, uint32_t* c) {
    GroupItem it{};
    it.n = s.n, it.n_pad = s.n_pad, it.limbs = s.limbs, it.r = s.r, it.r_pad = s.r_pad;
    it.conv_rows = s.conv_rows, it.conv_k = s.conv_k, it.crt_rows = s.crt_rows, it.crt_k = s.crt_k;
    it.crt_words = s.crt_words, it.ws = word_stride(s), it.t_words = s.t_words;
    it.n1 = s.n1, it.n2 = s.n2, it.rows = s.rows, it.row_width = s.row_width;
    it.k_shift = s.k_shift;
    const ConvertPlan cp = convert_plan(s, 2 * s.n_pad / kTile, kConvertGroupBlocks, true);
    it.conv_ks = cp.ks, it.conv_nt = cp.nt;  // conv_split: launch_group
    it.conv_columns = s.limbs <= kGroupShortLimbs ? cp.rows : 1;
    it.top_m = barrett_top(s);
    it.top_e = s.s_shift - 32 * it.top_m;
    it.mu = s.mu;
    it.consts = t.consts, it.wconv = t.wconv, it.tw_fwd = t.tw_fwd, it.tw_inv = t.tw_inv, it.wcrt = t.wcrt;
    it.q = t.q, it.neg_p = t.neg_p, it.corr_t = t.corr_t, it.corr_e = t.corr_e;
    it.a = a, it.b = b, it.c = c;
    it.packed = w.packed, it.planes = w.planes, it.rtiles = w.rtiles, it.words = w.words;
    return it;
}

bool groupable(const Shape& s) {
    if (s.trivial) return false;
    if (s.rows >= 2 && (s.row_width % 256 != 0 || s.rows > 64)) return false;  // forward columns through LDS
    if (s.row_width % 16 != 0 || s.rows > 64) return false;                      // inverse columns through LDS
    return true;
}

namespace {

// Launches of one batch: conversion from the limbs, pack, conversion GEMM,
// forward columns (four row-count classes), rows (one per row width and block
// size n1, and the LDS kernel), inverse columns (four classes), CRT GEMM with
// reconstruction, CRT GEMM, reconstruction (two kernels).
constexpr size_t kGroupLaunches = 1 + 2 + 4 + 21 + 4 + 1 + 1 + 2;

enum GroupKind { kConvert, kPack, kConversion, kForward, kRowsReg, kRowsProduct, kInverse, kCrtRec, kCrt, kRecWide, kRecWave };

size_t group_item_bytes(size_t count) { return (count * sizeof(GroupItem) + 255) / 256 * 256; }
size_t group_table_words(size_t count) { return kGroupLaunches * (2 * count + 1); }

}  // namespace

size_t group_bytes(size_t count) { return group_item_bytes(count) + group_table_words(count) * sizeof(uint32_t); }

void launch_group(std::vector<GroupItem> items, void* dev_buffer, hipStream_t stream) {
    const uint32_t count = uint32_t(items.size());
    if (!count) return;
    uint64_t conv_blocks = 0;
    for (const GroupItem& it : items)
        if (it.limbs <= kGroupShortLimbs) conv_blocks += convert_group_blocks(it.n, it.conv_nt);
    for (GroupItem& it : items)
        if (it.limbs <= kGroupShortLimbs)
            it.conv_split = convert_group_split((it.r + 15) / 16, convert_group_blocks(it.n, it.conv_nt), conv_blocks);
    // A product none of whose variants the grouped kernels hold must not be skipped.
    for (const GroupItem& it : items) {
        const uint32_t logc = row_variant(it.row_width, it.n1);
        const ConvertPlan cp{it.conv_ks, it.conv_nt, it.conv_columns, it.conv_split};
        if (!columns_compiled(it.rows) || (logc && !rows_compiled(logc, it.n1)) ||
            (it.limbs <= kGroupShortLimbs && !convert_group_compiled(cp)))
            throw std::logic_error("launch_group: no kernel of the variant a product takes");
    }
    const size_t item_bytes = group_item_bytes(count);
    const GroupView* dev_items = static_cast<const GroupView*>(dev_buffer);  // GroupItems, uploaded below
    uint32_t* dev_tables = reinterpret_cast<uint32_t*>(static_cast<char*>(dev_buffer) + item_bytes);
    struct Launch {
        GroupKind kind;
        uint32_t variant;
        uint32_t offset, entries;
        uint64_t blocks;
        size_t lds;
    };
    std::vector<uint32_t> tables(group_table_words(count));
    std::vector<Launch> launches;
    size_t used = 0;
    // One launch over the items for which blocks(it) > 0.
    auto add = [&](GroupKind kind, uint32_t variant, auto blocks) {
        std::vector<uint32_t> sel;
        for (uint32_t i = 0; i < count; ++i)
            if (blocks(items[i]) > 0) sel.push_back(i);
        if (sel.empty()) return;
        // the longest blocks (most primes) start first, the short ones fill the tail
        std::stable_sort(sel.begin(), sel.end(), [&](uint32_t x, uint32_t y) { return items[x].r > items[y].r; });
        if (launches.size() == kGroupLaunches) throw std::logic_error("launch_group: more launches than planned");
        uint32_t* start = tables.data() + used;
        uint32_t* item = start + sel.size() + 1;
        uint64_t total = 0;
        size_t lds = 0;
        for (size_t j = 0; j < sel.size(); ++j) {
            start[j] = uint32_t(total);
            item[j] = sel[j];
            total += blocks(items[sel[j]]);
            const GroupItem& it = items[sel[j]];
            lds = std::max<size_t>(lds, kind == kCrtRec    ? fused_lds_bytes(fused_waves(it.crt_words), 4, (it.r + 15) / 16)
                                        : kind == kConvert ? convert_lds_bytes(it.conv_k / kTK, it.r, it.conv_split, it.conv_columns)
                                                           : size_t(2) * it.row_width * 4);
        }
        if (total >= (uint64_t(1) << 31)) throw std::invalid_argument("launch_group: batch too large for one grid");
        start[sel.size()] = uint32_t(total);
        launches.push_back(Launch{kind, variant, uint32_t(used), uint32_t(sel.size()), total, lds});
        used += 2 * sel.size() + 1;
    };
    auto ntiles = [](const GroupItem& it) { return uint64_t(it.n_pad / kTile); };
    add(kConvert, 0, [&](const GroupItem& it) {
        return it.limbs <= kGroupShortLimbs ? uint64_t(it.conv_split) * (8 / it.conv_nt) * ntiles(it) : 0;
    });
    add(kPack, 0, [&](const GroupItem& it) {  // as launch_pack: 2 * ntiles * 256 rows
        return it.limbs <= kGroupShortLimbs ? 0 : 128 * ntiles(it) / kPackRows;
    });
    add(kConversion, 0, [&](const GroupItem& it) {
        return it.limbs <= kGroupShortLimbs ? 0 : uint64_t(it.conv_rows / kTile) * 2 * ntiles(it);
    });
    auto row_kernel = [](const GroupItem& it) { return it.rows < 8 ? 8 : it.rows; };
    for (uint32_t R = 8; R <= 64; R *= 2)
        add(kForward, R, [&](const GroupItem& it) {
            return it.rows > 1 && it.conv_columns == 1 && row_kernel(it) == R ? uint64_t(it.row_width / 256) * it.r * 2 : 0;
        });
#define PM_GROWS(LC, B)                                                                                        \
    add(kRowsReg, LC * 16 + B, [&](const GroupItem& it) {                                                      \
        return row_variant(it.row_width, it.n1) == LC && it.n1 == B                                            \
                   ? uint64_t(it.rows) * ((it.r + (kRowC >> LC) - 1) / (kRowC >> LC))                          \
                   : 0;                                                                                        \
    });
    PM_ROWS_VARIANTS(PM_GROWS)
#undef PM_GROWS
    add(kRowsProduct, 0, [&](const GroupItem& it) {
        return row_variant(it.row_width, it.n1) ? 0 : uint64_t(it.rows) * it.r;
    });
    for (uint32_t R = 8; R <= 64; R *= 2)
        add(kInverse, R, [&](const GroupItem& it) {
            const bool skip = it.rows <= 4 && it.crt_words <= kFusedWords;  // crt_reconstruct_group does it
            return row_kernel(it) == R && !skip ? uint64_t(it.row_width / 16) * (it.r_pad / 16) : 0;
        });
    add(kCrtRec, 0, [&](const GroupItem& it) { return it.crt_words <= kFusedWords ? 4 * ntiles(it) : 0; });
    add(kCrt, 0, [&](const GroupItem& it) {  // whole tiles: the batch's products fill the GPU together
        return it.crt_words <= kFusedWords ? 0 : uint64_t(it.crt_rows / kTile) * ntiles(it);
    });
    add(kRecWide, 0, [&](const GroupItem& it) {
        return it.crt_words > kFusedWords && it.crt_words <= kWideWords ? 16 * ntiles(it) : 0;
    });
    add(kRecWave, 0, [&](const GroupItem& it) { return it.crt_words > kWideWords ? 64 * ntiles(it) : 0; });
    // the items and the work lists, one copy
    std::vector<char> upload(item_bytes + used * sizeof(uint32_t));
    std::memcpy(upload.data(), items.data(), count * sizeof(GroupItem));
    std::memcpy(upload.data() + item_bytes, tables.data(), used * sizeof(uint32_t));
    const hipError_t copied = hipMemcpy(dev_buffer, upload.data(), upload.size(), hipMemcpyHostToDevice);
    if (copied != hipSuccess) throw std::runtime_error(std::string("launch_group upload: ") + hipGetErrorString(copied));
    for (const Launch& L : launches) {
        const GroupLaunch g{dev_items, dev_tables + L.offset, dev_tables + L.offset + L.entries + 1, L.entries};
        const dim3 grid(uint32_t(L.blocks));
        switch (L.kind) {
            case kConvert:
                hipLaunchKernelGGL(convert_group, grid, dim3(256), L.lds, stream, g);
                break;
            case kPack:
                hipLaunchKernelGGL(pack_group, grid, dim3(256), 0, stream, g);
                break;
            case kConversion:
                hipLaunchKernelGGL(conversion_group, grid, dim3(512), 0, stream, g);
                break;
            case kForward:
                switch (L.variant) {
#define PM_GFWD(R)                                                                      \
    case R:                                                                             \
        hipLaunchKernelGGL(forward_reg_group<R>, grid, dim3(256), 0, stream, g);         \
        break;
                    PM_GFWD(8) PM_GFWD(16) PM_GFWD(32) PM_GFWD(64)
#undef PM_GFWD
                }
                break;
            case kRowsReg:
#define PM_GROWS(LC, B)                                                                       \
    if (L.variant == LC * 16 + B)                                                             \
        hipLaunchKernelGGL((rows_reg_group<LC, B>), grid, dim3(256), 0, stream, g);
                PM_ROWS_VARIANTS(PM_GROWS)
#undef PM_GROWS
                break;
            case kRowsProduct:
                hipLaunchKernelGGL(rows_product_group, grid, dim3(256), L.lds, stream, g);
                break;
            case kInverse:
                switch (L.variant) {
#define PM_GINV(R)                                                                      \
    case R:                                                                             \
        hipLaunchKernelGGL(inverse_tiles_group<R>, grid, dim3(256), 0, stream, g);       \
        break;
                    PM_GINV(8) PM_GINV(16) PM_GINV(32) PM_GINV(64)
#undef PM_GINV
                }
                break;
            case kCrtRec:
                hipLaunchKernelGGL(crt_reconstruct_group, grid, dim3(256), L.lds, stream, g);
                break;
            case kCrt:
                hipLaunchKernelGGL(crt_group, grid, dim3(512), 0, stream, g);
                break;
            case kRecWide:
                hipLaunchKernelGGL(reconstruct_wide_group, grid, dim3(256), 0, stream, g);
                break;
            case kRecWave:
                hipLaunchKernelGGL(reconstruct_waves_group, grid, dim3(256), 0, stream, g);
                break;
        }
        check_launch("grouped stage");
    }
}

void launch_zero(uint32_t* c, size_t words, hipStream_t stream) {
    if (!words) return;
    dim3 grid(uint32_t((words + 255) / 256));
    hipLaunchKernelGGL(fill_zero, grid, dim3(256), 0, stream, c, words);
    check_launch("fill_zero");
}

void launch_build_tables(const Shape& s, const TableBuild& t, hipStream_t stream) {
    const uint32_t r = s.r;
    launch_zero(reinterpret_cast<uint32_t*>(t.wconv), size_t(2) * s.conv_rows * s.conv_k / 4, stream);
    launch_zero(reinterpret_cast<uint32_t*>(t.wcrt), size_t(s.crt_rows) * s.crt_k / 4, stream);
    hipLaunchKernelGGL(table_beta, dim3(r), dim3(256), 0, stream, t.consts, t.rcp, t.beta, r, s.n2);
    check_launch("table_beta");
    const uint32_t cols = (s.n2 + 255) / 256;
    hipLaunchKernelGGL(table_twiddles, dim3(cols < 64 ? cols : 64, r), dim3(256), 0, stream, t.consts, t.rcp, t.psi,
                       t.tw_fwd, t.tw_inv, s.n2, s.log_n2);
    check_launch("table_twiddles");
    hipLaunchKernelGGL(table_conversion, dim3(r, 2), dim3(256), 0, stream, t.consts, t.rcp, t.beta, t.wconv,
                       s.conv_rows, s.conv_k, s.limbs);
    check_launch("table_conversion");
    hipLaunchKernelGGL(table_crt, dim3((r + 63) / 64), dim3(64), 0, stream, t.m_mod_q, t.rcp, t.wcrt, r, s.limbs,
                       s.crt_k);
    check_launch("table_crt");
}

// ---------------------------------------------------------------------------
// Static workspace of the allocation-free device entry point
// (pm_multiply_device_scratch).  The array is part of this code object: each
// GPU that loads the library holds its own copy, at its own address, until
// the process ends.  In host code `scratch` names only a host-side stand-in,
// so its device address is looked up once per device (init_scratch, called
// when the library makes a plan on that device) and only that address is
// handed to kernels.
// ---------------------------------------------------------------------------
namespace {
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kScratchDevices] = {};
hipError_t g_scratch_error[kScratchDevices] = {};
}  // namespace

void init_scratch() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kScratchDevices) {
        (void)hipGetLastError();
        return;  // pm_multiply_device_scratch reports the device as unsupported
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev]) return;
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
        (void)hipGetLastError();  // keep the failure out of later launch checks
        g_scratch_error[dev] = e != hipSuccess ? e : hipErrorInvalidSymbol;
        return;
    }
    g_scratch_ptr[dev] = ptr;
}

void* scratch_address(int device, std::string* why) {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (device < 0 || device >= kScratchDevices) {
        if (why) *why = "device " + std::to_string(device) + " is beyond the devices the static scratch supports";
        return nullptr;
    }
    if (!g_scratch_ptr[device] && why)
        *why = g_scratch_error[device] != hipSuccess
                   ? std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(g_scratch_error[device])
                   : "the static scratch was not set up on device " + std::to_string(device);
    return g_scratch_ptr[device];
}

size_t work_bytes(const Shape& s) { return carve_work(s, nullptr, nullptr); }

size_t carve_work(const Shape& s, uint8_t* base, DeviceWork* w) {
    const size_t packed = packed_operand_bytes(s);
    const size_t half = size_t(s.r_pad) * s.n_pad;
    const size_t planes = 2 * half * sizeof(uint32_t);
    const size_t words = word_sum_elements(s) * sizeof(int64_t);
    auto round = [](size_t b) { return (b + 255) / 256 * 256; };
    if (base && w) {
        w->packed = reinterpret_cast<int8_t*>(base);
        w->planes = reinterpret_cast<uint32_t*>(base + round(packed));
        w->rtiles = reinterpret_cast<int8_t*>(w->planes + half);
        w->words = reinterpret_cast<int64_t*>(base + round(packed) + round(planes));
    }
    return round(packed) + round(planes) + round(words);
}

}  // namespace pm
