// Multi-token decode on the matrix cores: the expert GEMMs of naiwa_moe_decode
// calls of several rows, exact in the weights.
//
// A block of 4 waves takes one slot segment (the sorted pairs of one slot) and a
// strip of weight rows (64 gate and the same 64 up rows, or 64 or 128 down rows);
// chunks of up to MR of the segment's tokens are the A operand of
// v_mfma_f32_16x16x32_f16.  Lane l = 16 g + m holds A[m][8 g + 0..7] (token m),
// B[8 g + 0..7][m] (weight row m of the wave's 16) and D[4 g + i][m].
//
// What bounds it: the weights are read once per chunk of tokens and nothing else
// is large, so HBM.  A lane that loads its own rows' pieces into registers
// touches 16 rows with each 16-byte load, and the cache's line lookups then cap
// the stream (4.36 TB/s for a load-only kernel on a 528 MB gate/up bank of K
// 4096, against 6.1 for a linear read).  Here each wave copies its rows' bytes
// to LDS by DMA with consecutive lanes on consecutive pieces of a row (5.5 TB/s
// for the copies alone) and the lanes unpack from LDS.  Measured, router included,
// against register loads with weights rounded to bf16 (time; bytes of weights / time):
// 8 rows of 128 experts top-8 at H 2048, I 768, Q4_K 71.2 -> 58.4-59.8 us (2.4 TB/s; the
// GEMMs are 40 us of it at 3.3), 96 rows 1,303 (the vector path then) -> 115 us (3.0 TB/s);
// 8 experts top-2 at H 4096, I 14336 16 rows 217 -> 189 us (4.2), 64 rows 258 -> 241 us
// (3.3).  The distance to a 64-bit reference fell from 3.4e-3 (1.7e-3 on the vector path)
// to 2.1e-4.
//
// Exact operands.  A quantised weight is an integer times a scale, so the B
// operand is that integer in f16 and the scales are applied in f32 afterwards:
//   Q4_K: sc * q (6-bit scale times nibble, at most 945) is exact in f16; one
//         packed fma makes two of them.  Over a 256-value block D = sum (sc q) x
//         and M = sum m6_j X_j (X_j the activation sums of the 8 sub-blocks, as
//         two f16 terms each, on one 16x16x16 MFMA): y += d D - dmin M;
//   Q8_0: q (signed byte) is exact in f16; per 32-value block y += d sum q x.
// Activations are f16 times a power of two per row chosen from the row's largest
// magnitude (2^9 <= max < 2^10), so any finite f32 row fits: a bf16 value within
// 2^-23 of the row's largest is kept exactly and smaller ones to 2^-34 of it.
//   x: one scale per token (prep kernel);
//   h: one scale per (pair, 64 features), the block's own strip, stored beside it;
//      the down kernel brings a row's strips to one scale as it reads the A operand.
// An infinity among them cancels to NaN; where h overflowed, the combine forms the sums of
// products instead (an infinite x gives NaN: some gate is -inf, and its activation NaN).
//
// Rounded operands (BF).  The layers of a chain route on activations that the layers before
// them rounded, so any change of rounding flips an expert near the cut of a top-k somewhere
// and with it all that follows: whole steps (the layered stack, the partial cache) of at most 512
// pairs a layer keep x, h and the dequantised weights in bf16 and the order of the sums that
// the first matrix-core decode had, and with them its results bit for bit.  (Larger layers ran
// on the vector path, with f32 weights, and take the exact operands now.)
//
// K order: group G = 4 s + g of 8 values is lane group g's A operand at step s.
//   Q4_K (256 values): lane group g takes 64-value chunk g; step s = 2 p + t its
//        quant bytes 8 p + 0..7, low nibbles for t = 0 and high ones for t = 1:
//        values 64 g + 32 t + 8 p + (0 2 1 3 4 6 5 7);
//   Q8_0 (128 values), exact: step s is block s, so that D has one scale: values
//        32 s + 8 g + 0..7, the natural order;
//   Q8_0, rounded: lane group g takes block g, values 32 g + 8 s + 0..7 at step s: the order
//        is part of the bits of the sums.
#include "decode_mfma.h"
#include "common.h"
#include "segments.h"
#include "unpack_bf16.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace {

typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256; // 4 waves of 16 weight rows (per matrix)
constexpr int kF = 64;        // weight rows per block and matrix
constexpr int kChunk = 64;    // features of h that share one scale: a gate/up block's strip

struct Bank {
    const uint8_t* base;
    int64_t stride;
    int64_t row_bytes;
};

template <int DT> struct KB;
template <> struct KB<NAIWA_Q4_K> {
    static constexpr int kVals = 256, kSteps = 8, kGroups = 32, kBytes = NAIWA_Q4_K_BYTES;
};
template <> struct KB<NAIWA_Q8_0> {
    static constexpr int kVals = 128, kSteps = 4, kGroups = 16, kBytes = 4 * NAIWA_Q8_0_BYTES;
};

// The group that holds run r (values 8 r .. 8 r + 7) of a K-block.
template <int DT, bool BF>
__device__ __forceinline__ int group_of_run(int r) {
    if (DT == NAIWA_Q4_K) {
        const int g = r >> 3, t = (r >> 2) & 1, p = r & 3;
        return 4 * (2 * p + t) + g;
    }
    return BF ? 4 * (r & 3) + (r >> 2) : r;
}

// The power of two that brings magnitude mx to [2^9, 2^10), as its exponent (at most
// 126, so that an all-zero or tiny row's scale and its inverse stay normal numbers).
__device__ __forceinline__ int scale_exp(float mx) { return min(126, 136 - (int)((__float_as_uint(mx) >> 23) & 255u)); }
__device__ __forceinline__ float pow2f(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// A run of 8 f32 values (natural order), scaled and rounded to f16 in the K order of DT;
// sum: the sum of the rounded values.
template <int DT>
__device__ __forceinline__ half8v pack_run(const float (&f)[8], float scale, float& sum) {
    half8v o;
    sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const _Float16 v = (_Float16)(f[DT == NAIWA_Q4_K ? q4_elem(i) : i] * scale);
        o[i] = v;
        sum += (float)v;
    }
    return o;
}

// The same in bf16, unscaled.
template <int DT>
__device__ __forceinline__ half8v pack_run_bf16(const float (&f)[8]) {
    float o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = f[DT == NAIWA_Q4_K ? q4_elem(i) : i];
    return __builtin_bit_cast(half8v, to_bf16x8(o));
}

// Slot of sub-block sum j (0..7) of a K-block: f16 halves hi [0..7] and lo [8..15].
__device__ __forceinline__ void put_sum(_Float16* s16, int j, float sum) {
    const _Float16 hi = (_Float16)sum;
    s16[j] = hi;
    s16[8 + j] = (_Float16)(sum - (float)hi);
}

// ---------------------------------------------------------------------------
// segments + activations, one launch
// ---------------------------------------------------------------------------
// Block 0 sorts the pairs into segments (tok: the token of each sorted position); block 1 + t lays out token t's row of x:
// f16 groups xa [rows][H], sub-block sums xs [rows][H / 256][16] (Q4_K) and the
// row's inverse scale xr [rows].  The two parts share nothing, and a launch of its
// own costs each about 4.5 us of a 60 us call.
template <int DT, bool BF>
__global__ void __launch_bounds__(kThreads)
seg_prep_kernel(const uint32_t* slot_ids, const float* w, int n, int width, int nslots, uint32_t* tok, uint32_t* inv,
                int* seg_count, uint32_t* seg_key, uint32_t* seg_begin, int* bad, const void* x, int x_bf16, int H,
                _Float16* xa, _Float16* xs, float* xr) {
    __shared__ NaiwaSegSmem sm;
    const int tid = threadIdx.x;
    if (blockIdx.x == 0) {
        naiwa_segment(sm, slot_ids, w, n, nslots, tok, nullptr, seg_count, seg_key, seg_begin, bad, inv, width);
        return;
    }
    const int t = blockIdx.x - 1, runs = H / 8;
    auto run_of = [&](int run, float (&f)[8]) {
        if (x_bf16) {
            const u32x4 v = *reinterpret_cast<const u32x4*>((const uint16_t*)x + (size_t)t * H + 8 * run);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f[2 * j] = __uint_as_float(v[j] << 16);
                f[2 * j + 1] = __uint_as_float(v[j] & 0xffff0000u);
            }
        } else {
            const floatx4* src = reinterpret_cast<const floatx4*>((const float*)x + (size_t)t * H + 8 * run);
            const floatx4 a = src[0], b = src[1];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f[j] = a[j];
                f[4 + j] = b[j];
            }
        }
    };
    constexpr int R = KB<DT>::kVals / 8;
    if constexpr (BF) {
        for (int run = tid; run < runs; run += kThreads) {
            float f[8];
            run_of(run, f);
            *reinterpret_cast<half8v*>(xa + (size_t)t * H + run / R * KB<DT>::kVals + 8 * group_of_run<DT, BF>(run % R)) =
                pack_run_bf16<DT>(f);
        }
        return;
    }
    float mx = 0.0f;
    for (int run = tid; run < runs; run += kThreads) {
        float f[8];
        run_of(run, f);
#pragma unroll
        for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(f[j]));
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) mx = fmaxf(mx, __shfl_xor(mx, m, 64));
    float* red = reinterpret_cast<float*>(sm.part);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const int e = scale_exp(mx);
    const float sc = pow2f(e);
    if (tid == 0) xr[t] = pow2f(-e);
    // whole rounds of the block, so that the lanes of a sub-block's 4 runs shuffle together
    for (int r0 = 0; r0 < runs; r0 += kThreads) {
        const int run = r0 + tid;
        const bool in = run < runs;
        float f[8] = {}, sum;
        if (in) run_of(run, f);
        const half8v o = pack_run<DT>(f, sc, sum);
        const int kb = run / R, r = run % R;
        if (in) *reinterpret_cast<half8v*>(xa + (size_t)t * H + kb * KB<DT>::kVals + 8 * group_of_run<DT, BF>(r)) = o;
        if (DT == NAIWA_Q4_K) {
            sum += __shfl_xor(sum, 1, 64);
            sum += __shfl_xor(sum, 2, 64);
            if (in && (r & 3) == 0) put_sum(xs + ((size_t)t * (H / 256) + kb) * 16, r >> 2, sum);
        }
    }
}

// ---------------------------------------------------------------------------
// LDS DMA
// ---------------------------------------------------------------------------
// lane i of the wave copies 16 (or 4) bytes from base + off to lds + 16 i (4 i).  Issued
// as inline assembly so that the compiler does not make every later LDS read wait for
// every copy in flight; each read of copied data follows an explicit vmcnt wait of the
// issuing wave and, where another wave reads it, a barrier.  M0 is reserved and written
// only here.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) const void*)p);
}
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const void* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
// until at most N of the wave's copies (and loads), the last ones, are in flight
template <int N>
__device__ __forceinline__ void wait_copies() { asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory"); }
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// A tile of MR token rows of one K-block.  One DMA instruction brings kRpd whole rows
// (the lanes cover them piece by piece); row m's piece c holds group c ^ (m % kRpd) and
// each instruction's rows start 16 kRpd bytes further on, so the 16 rows' pieces of one
// group fall on distinct banks while a step's read keeps a fixed offset from the lane's
// own base: (m / kRpd) kStride + (m % kRpd) 16 kGroups + 16 (g ^ m % kRpd) + 64 s.
template <int DT, int MR, bool BF> struct ATile {
    static constexpr int G = KB<DT>::kGroups, kRpd = 64 / G, kDma = MR / kRpd, kStride = 1024 + 16 * kRpd;
    static constexpr bool kSums = DT == NAIWA_Q4_K && !BF;
    __align__(16) uint8_t v[kDma * kStride];
    __align__(16) _Float16 sums[kSums ? MR * 16 : 8]; // [row][hi 0..7 | lo 0..7]
};

// Raw weight bytes of one K-block: a wave's 16 rows of NP matrices.
template <int DT, int NP> struct WTile {
    static constexpr int kMat = 16 * KB<DT>::kBytes;
    static constexpr bool k16 = DT == NAIWA_Q4_K; // 16-byte pieces; Q8_0 rows are 8-byte aligned: dwords
    static constexpr int kPieces = kMat / (k16 ? 16 : 4);
    static constexpr int kDma = (kPieces + 63) / 64;
    __align__(16) uint8_t v[NP * kMat];
};

// The lane's unpacking of its weight row's K-block, from LDS into B operands and scales.
__device__ __forceinline__ half2v h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ half2v splat(_Float16 v) { return half2v{v, v}; }

// Two bytes of w (at bits 0 and 16 after masking) as f16 integers.
__device__ __forceinline__ half2v bytes_f16(uint32_t w, uint32_t sel) {
    return h2(__builtin_amdgcn_perm(0x64646464u, w, sel)) - splat((_Float16)1024.0f);
}

// One lane's raw weight words of a K-block (NP rows), out of LDS: the stage is free for the
// next copies as soon as every lane holds its own.
template <int DT, int NP, bool BF> struct WRegs;
template <int NP, bool BF> struct WRegs<NAIWA_Q4_K, NP, BF> {
    u32x4 hd[NP], q0[NP], q1[NP]; // header; quant bytes 0-15 and 16-31 of 64-value chunk g
    __device__ __forceinline__ void load(const WTile<NAIWA_Q4_K, NP>& wt, int g, int m) {
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const uint8_t* row = wt.v + q * WTile<NAIWA_Q4_K, NP>::kMat + m * NAIWA_Q4_K_BYTES;
            hd[q] = *reinterpret_cast<const u32x4*>(row);
            q0[q] = *reinterpret_cast<const u32x4*>(row + 16 + 32 * g);
            q1[q] = *reinterpret_cast<const u32x4*>(row + 32 + 32 * g);
        }
    }
};
template <int NP> struct WRegs<NAIWA_Q8_0, NP, false> {
    // block s: d at byte 34 s, this lane's 8 codes from 34 s + 2 + 8 g; even blocks start on
    // a word (codes in 3 words from 34 s + 8 g), odd ones 2 bytes into one (codes in 2 words)
    uint32_t ev[NP][2][3], od[NP][2][2], dw[NP][4];
    __device__ __forceinline__ void load(const WTile<NAIWA_Q8_0, NP>& wt, int g, int m) {
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const uint8_t* blk = wt.v + q * WTile<NAIWA_Q8_0, NP>::kMat + m * KB<NAIWA_Q8_0>::kBytes + 2 * j * NAIWA_Q8_0_BYTES;
                const uint32_t* p = reinterpret_cast<const uint32_t*>(blk + 8 * g);
#pragma unroll
                for (int i = 0; i < 3; ++i) ev[q][j][i] = p[i];
#pragma unroll
                for (int i = 0; i < 2; ++i) od[q][j][i] = p[9 + i];
                dw[q][2 * j] = *reinterpret_cast<const uint32_t*>(blk);
                dw[q][2 * j + 1] = *reinterpret_cast<const uint32_t*>(blk + 32);
            }
    }
    __device__ __forceinline__ float d(int q, int s) const {
        return naiwa_f16_to_f32((s & 1) ? dw[q][s] >> 16 : dw[q][s] & 0xffffu);
    }
    __device__ __forceinline__ uint32_t code(int q, int s, int i) const {
        return (s & 1) ? od[q][s >> 1][i] : __builtin_amdgcn_alignbyte(ev[q][s >> 1][i + 1], ev[q][s >> 1][i], 2);
    }
};

template <int NP> struct WRegs<NAIWA_Q8_0, NP, true> {
    // block g, at byte 34 g: its d, and its codes from the word that holds the first (even g:
    // from that word's third byte on, so 9 words; odd g: 8 whole words, the eighth again)
    uint32_t w[NP][9], sh;
    uint16_t dh[NP];
    __device__ __forceinline__ void load(const WTile<NAIWA_Q8_0, NP>& wt, int g, int m) {
        sh = 2u - 2u * (uint32_t)(g & 1);
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const uint8_t* blk = wt.v + q * WTile<NAIWA_Q8_0, NP>::kMat + m * KB<NAIWA_Q8_0>::kBytes + g * NAIWA_Q8_0_BYTES;
            const uint32_t* p = reinterpret_cast<const uint32_t*>(blk + 2 * (g & 1));
            dh[q] = *reinterpret_cast<const uint16_t*>(blk);
#pragma unroll
            for (int i = 0; i < 8; ++i) w[q][i] = p[i];
            w[q][8] = p[8 - (g & 1)];
        }
    }
    __device__ __forceinline__ float d(int q, int) const { return naiwa_f16_to_f32(dh[q]); }
    __device__ __forceinline__ uint32_t code(int q, int s, int i) const {
        return __builtin_amdgcn_alignbyte(w[q][2 * s + i + 1], w[q][2 * s + i], sh);
    }
};

// One K-block of a wave: acc[q][mt] += rows q of the weights times the A tile's subtiles.
// fac (h only): the row's per-chunk f16 factors from this K-block's chunk on.
// BF: activations and dequantised weights rounded to bf16, accumulated over the K-blocks.
template <int DT, int NP, int MT, int MR, bool HF, bool BF>
__device__ __forceinline__ void kblock(const WRegs<DT, NP, BF>& wr, const ATile<DT, MR, BF>& at, const uint16_t* fac,
                                       int fst, int g, int m, const NibMask& nm, floatx4 (&acc)[NP][MT]) {
    using A = ATile<DT, MR, BF>;
    auto arow = [&](int mt) { return MR < 16 ? (m & (MR - 1)) : 16 * mt + m; };
    const uint8_t* abase[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int r = arow(mt), c = r % A::kRpd;
        abase[mt] = at.v + (r / A::kRpd) * A::kStride + c * (16 * A::G) + 16 * (g ^ c);
    }
    auto ld_a = [&](int mt, int s) {
        return __builtin_bit_cast(half8v, *reinterpret_cast<const u32x4*>(abase[mt] + 64 * s));
    };
    if constexpr (BF) {
        float sc[NP][2], mn[NP][2];
        if constexpr (DT == NAIWA_Q4_K)
#pragma unroll
            for (int q = 0; q < NP; ++q)
#pragma unroll
                for (int t = 0; t < 2; ++t) q4k_scale_min(wr.hd[q], 2 * g + t, sc[q][t], mn[q][t]);
#pragma unroll
        for (int s = 0; s < KB<DT>::kSteps; ++s) {
            bf16x8 a8[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) a8[mt] = __builtin_bit_cast(bf16x8, ld_a(mt, s));
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                bf16x8 b8;
                if constexpr (DT == NAIWA_Q4_K) {
                    const int p = s >> 1, t = s & 1;
                    const u32x4& qv = p < 2 ? wr.q0[q] : wr.q1[q];
                    b8 = q4k_unpack((p & 1) ? qv.z : qv.x, (p & 1) ? qv.w : qv.y, t, nm, sc[q][t], mn[q][t]);
                } else {
                    b8 = q8_unpack(wr.code(q, s, 0), wr.code(q, s, 1), wr.d(q, s));
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[q][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a8[mt], b8, acc[q][mt], 0, 0, 0);
            }
        }
    } else if constexpr (DT == NAIWA_Q4_K) {
        half2v sc[NP];
        half4v m6[NP];
        float d[NP], dmin[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const u32x4 hd = wr.hd[q];
            d[q] = naiwa_f16_to_f32(hd.x & 0xffffu);
            dmin[q] = naiwa_f16_to_f32(hd.x >> 16);
            // scales of sub-blocks 2 g and 2 g + 1; mins of sub-blocks 4 (g % 2) .. + 3
            const uint32_t slo = hd.y & 0x3f3f3f3fu, shi = (hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u);
            const uint32_t mlo = hd.z & 0x3f3f3f3fu, mhi = ((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u);
            const uint32_t sw = (g & 2) ? shi : slo, mw = (g & 1) ? mhi : mlo;
            sc[q] = bytes_f16(sw, (g & 1) ? 0x04030402u : 0x04010400u);
            const half2v a = bytes_f16(mw, 0x04010400u), b = bytes_f16(mw, 0x04030402u);
            m6[q] = half4v{a[0], a[1], b[0], b[1]};
        }
        half4v xs[MT];
        half2v fg[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            xs[mt] = __builtin_bit_cast(half4v, *reinterpret_cast<const u32x2*>(at.sums + arow(mt) * 16 + 4 * g));
            if constexpr (HF) {
                const uint16_t* f = fac + arow(mt) * fst;
                fg[mt] = splat(__builtin_bit_cast(_Float16, f[g]));
                const half2v fj = *reinterpret_cast<const half2v*>(f + 2 * (g & 1));
                xs[mt] *= half4v{fj[0], fj[0], fj[1], fj[1]};
            }
        }
        floatx4 D[NP][MT], M[NP][MT];
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                D[q][mt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                M[q][mt] = __builtin_amdgcn_mfma_f32_16x16x16f16(xs[mt], m6[q], D[q][mt], 0, 0, 0);
            }
#pragma unroll
        for (int s = 0; s < KB<DT>::kSteps; ++s) {
            const int p = s >> 1, t = s & 1;
            half8v a8[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                a8[mt] = ld_a(mt, s);
                if constexpr (HF) {
                    const half2v f = fg[mt];
                    a8[mt] *= half8v{f[0], f[1], f[0], f[1], f[0], f[1], f[0], f[1]};
                }
            }
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const u32x4& qv = p < 2 ? wr.q0[q] : wr.q1[q];
                const uint32_t w[2] = {(p & 1) ? qv.z : qv.x, (p & 1) ? qv.w : qv.y};
                // (magic + nibble) * sc - magic * sc = sc * nibble, exact in one f16 fma
                const uint32_t mk = nm.m[t], magic = t ? 0x54005400u : 0x64006400u;
                const half2v s2 = splat(sc[q][t]), o2 = s2 * splat((_Float16)(t ? -64.0f : -1024.0f));
                u32x4 b;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t v = (((i & 1) ? w[i >> 1] >> 8 : w[i >> 1]) & mk) | magic;
                    b[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(h2(v), s2, o2));
                }
                const half8v b8 = __builtin_bit_cast(half8v, b);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    D[q][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a8[mt], b8, D[q][mt], 0, 0, 0);
            }
        }
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc[q][mt][i] = __builtin_fmaf(d[q], D[q][mt][i], __builtin_fmaf(-dmin[q], M[q][mt][i], acc[q][mt][i]));
    } else {
        half2v fc[MT];
        if constexpr (HF) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) fc[mt] = *reinterpret_cast<const half2v*>(fac + arow(mt) * fst);
        }
#pragma unroll
        for (int s = 0; s < KB<DT>::kSteps; ++s) {
            half8v a8[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                a8[mt] = ld_a(mt, s);
                if constexpr (HF) {
                    const _Float16 f = fc[mt][s >> 1];
                    a8[mt] *= half8v{f, f, f, f, f, f, f, f};
                }
            }
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const float d = wr.d(q, s);
                uint32_t c0 = wr.code(q, s, 0), c1 = wr.code(q, s, 1);
                // byte ^ 0x80 = q + 128, as f16 1024 + 128 + q; minus 1152: q, exact
                c0 ^= 0x80808080u;
                c1 ^= 0x80808080u;
                u32x4 b;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t v = __builtin_amdgcn_perm(0x64646464u, i < 2 ? c0 : c1, (i & 1) ? 0x04030402u : 0x04010400u);
                    b[i] = __builtin_bit_cast(uint32_t, h2(v) - splat((_Float16)1152.0f));
                }
                const half8v b8 = __builtin_bit_cast(half8v, b);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const floatx4 D =
                        __builtin_amdgcn_mfma_f32_16x16x32_f16(a8[mt], b8, floatx4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[q][mt][i] = __builtin_fmaf(d, D[i], acc[q][mt][i]);
                }
            }
        }
    }
}

// LDS of one block: the weight stages of each wave and two A tiles.  More weight stages cost
// blocks: with 2 of Q4_K the 8- and 96-row calls at H 2048, I 768 took 63 and 131 us against
// 61 and 120, and 16 and 64 rows at H 4096, I 14336 the same 188 and 227.
//
// ST weight stages of each wave.
template <int DT, int NP, int MR, bool BF, int ST> struct Smem {
    WTile<DT, NP> w[ST][kThreads / 64];
    ATile<DT, MR, BF> a[2];
};

// A value every lane of the wave reads, through the scalar cache (its own counter, so it
// does not wait for copies in flight).
__device__ __forceinline__ uint32_t scalar_ld(const uint32_t* p) {
    return *(const __attribute__((address_space(4))) uint32_t*)(uintptr_t)p;
}

// The K loop of one chunk of MR tokens over NP matrices' 16 rows per wave.  start() sends
// out the first copies (weights first: they need nothing but the segment), run() goes
// through the K-blocks with one barrier each: the wave's copies for it have landed (its own
// vmcnt), the barrier makes every wave's part of the A tile visible and frees the other A
// buffer, the next A copies go out, the lanes take their weight words, the copies of the
// K-block ST further on go out into the freed stage, and the K-block is computed.
template <int DT, int NP, int MT, int MR, bool BF, int ST> struct KLoop {
    using A = ATile<DT, MR, BF>;
    using W = WTile<DT, NP>;
    static constexpr int PB = W::k16 ? 16 : 4, kPer = KB<DT>::kBytes / PB; // pieces per row
    static constexpr int kAd = (A::kDma + 3) / 4; // A copies of a wave: instructions wave, wave + 4, ...
    Smem<DT, NP, MR, BF, ST>& sm;
    const uint8_t *abase, *sums;
    const uint8_t* wrow[NP];
    int kb0, nkb, lane, wave;
    uint32_t woff[W::kDma], aoff[kAd], soff[kAd];

    __device__ __forceinline__ void issue_w(int kb, int stage) {
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            const uint8_t* wb = wrow[q] + (size_t)kb * KB<DT>::kBytes;
#pragma unroll
            for (int i = 0; i < W::kDma; ++i)
                if (64 * (i + 1) <= W::kPieces || lane < W::kPieces - 64 * i) {
                    const uint32_t l = lds_addr(sm.w[stage][wave].v + q * W::kMat + 64 * PB * i);
                    if (W::k16)
                        dma16(wb, woff[i], l);
                    else
                        dma4(wb, woff[i], l);
                }
        }
    }
    __device__ __forceinline__ void issue_a(int kb, int buf) {
        const uint8_t* ab = abase + (size_t)kb * (KB<DT>::kVals * 2);
#pragma unroll
        for (int i = 0; i < kAd; ++i) {
            const int d = wave + 4 * i;
            if (d >= A::kDma) break;
            dma16(ab, aoff[i], lds_addr(sm.a[buf].v + d * A::kStride));
            if (A::kSums && lane < 2 * A::kRpd)
                dma16(sums + (size_t)kb * 32, soff[i], lds_addr(sm.a[buf].sums + d * A::kRpd * 16));
        }
    }
    // row(i): the A row of tile row i (uniform); A rows of arow bytes, their sums of srow
    template <class F>
    __device__ __forceinline__ void start(int64_t row_bytes, uint32_t arow, uint32_t srow, const F& row) {
#pragma unroll
        for (int i = 0; i < W::kDma; ++i) {
            const int p = min(lane + 64 * i, W::kPieces - 1);
            woff[i] = (uint32_t)((p / kPer) * row_bytes) + (uint32_t)(p % kPer) * PB;
        }
        issue_w(kb0, 0);
#pragma unroll
        for (int i = 0; i < kAd; ++i) {
            const int d = min(wave + 4 * i, A::kDma - 1);
            uint32_t ra = row(d * A::kRpd), rs = ra;
#pragma unroll
            for (int k = 1; k < A::kRpd; ++k) {
                const uint32_t r = row(d * A::kRpd + k);
                ra = lane / A::G == k ? r : ra;
                rs = (lane >> 1) == k ? r : rs;
            }
            aoff[i] = ra * arow + 16u * (uint32_t)((lane % A::G) ^ (lane / A::G));
            soff[i] = rs * srow + 16u * (uint32_t)(lane & 1);
        }
        issue_a(kb0, 0);
        if (ST == 2) issue_w(kb0 + min(1, nkb - 1), 1);
    }
    template <bool HF, int NFAC>
    __device__ __forceinline__ void run(const uint16_t (*fac)[NFAC], floatx4 (&acc)[NP][MT]) {
        const int g = lane >> 4, m = lane & 15;
        const NibMask nm = nib_mask();
        for (int j = 0; j < nkb; ++j) {
            const int jn = min(j + 1, nkb - 1), stage = ST == 2 ? j & 1 : 0;
            // all but the next stage's weights, the last copies issued (every wave issues all kDma
            // of each matrix)
            wait_copies<ST == 2 ? NP * W::kDma : 0>();
            lds_barrier();
            issue_a(kb0 + jn, (j + 1) & 1);
            WRegs<DT, NP, BF> wr;
            wr.load(sm.w[stage][wave], g, m);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // held in registers: the stage is free
            issue_w(kb0 + min(j + ST, nkb - 1), stage);
            kblock<DT, NP, MT, MR, HF, BF>(wr, sm.a[j & 1], HF ? &fac[0][j * (KB<DT>::kVals / kChunk)] : nullptr, NFAC, g, m,
                                       nm, acc);
        }
        // the last K-block's copies went out once more: they land before the LDS is used for
        // anything else
        wait_copies<0>();
        lds_barrier();
    }
};

// gate/up: block (64 features, slot segment, chunks z, z + gridDim.z, ...); h = act(gate) * up
// of the pair at its sorted position, f16 in the K order of DD with a scale per (pair, 64 features).
template <int DG, int DD, int MT, int MR, bool BF, int ST>
__global__ void __launch_bounds__(kThreads, 2)
gateup_mfma_kernel(Bank gate, Bank up, const _Float16* xa, const _Float16* xs, const float* xr, int H, int I,
                   const int* seg_count, const uint32_t* seg_key, const uint32_t* seg_begin, const uint32_t* tok,
                   int act, _Float16* ha, _Float16* hs, int8_t* he) {
    constexpr int kHt = kF + 4; // floats per row of the h exchange
    __shared__ Smem<DG, 2, MR, BF, ST> sm;
    static_assert(sizeof(float) * MR * kHt <= sizeof(sm), "the h exchange reuses the tiles");
    const int sg = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tid = threadIdx.x, g = lane >> 4, m = lane & 15;
    // the arrays have an entry for every possible segment
    const uint32_t slot = scalar_ld(seg_key + sg);
    const int b = (int)scalar_ld(seg_begin + sg), e = (int)scalar_ld(seg_begin + sg + 1);
    const int segs = (int)scalar_ld((const uint32_t*)seg_count);
    asm volatile("" ::"s"(slot), "s"(b), "s"(e), "s"(segs)); // one round trip
    if (sg >= segs) return;
    const int n0 = blockIdx.x * kF;
    const int64_t r0 = n0 + 16 * wave;
    KLoop<DG, 2, MT, MR, BF, ST> kl{sm, (const uint8_t*)xa, (const uint8_t*)xs,
                                 {gate.base + (int64_t)slot * gate.stride + r0 * gate.row_bytes,
                                  up.base + (int64_t)slot * up.stride + r0 * up.row_bytes},
                                 0, H / KB<DG>::kVals, lane, wave};
    for (int c0 = b + (int)blockIdx.z * MR; c0 < e; c0 += (int)gridDim.z * MR) {
        const int cnt = min(MR, e - c0);
        // rows past the segment repeat its last token; their results are dropped
        kl.start(gate.row_bytes, (uint32_t)H * 2, (uint32_t)(H / 256) * 32,
                 [&](int r) { return scalar_ld(tok + c0 + min(r, cnt - 1)); });
        float rs[MT][4];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) rs[mt][i] = BF ? 1.0f : xr[tok[c0 + min(16 * mt + 4 * g + i, cnt - 1)]];
        floatx4 acc[2][MT] = {};
        kl.template run<false, 2>(nullptr, acc);
        float* ht = reinterpret_cast<float*>(&sm);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int mm = 16 * mt + 4 * g + i;
                if (mm < MR)
                    ht[mm * kHt + 16 * wave + m] =
                        naiwa_act(act, acc[0][mt][i] * rs[mt][i]) * (acc[1][mt][i] * rs[mt][i]);
            }
        __syncthreads();
        // thread: one run of 8 features of one token; 8 consecutive lanes hold the strip
#pragma unroll
        for (int u0 = 0; u0 < MR * 8; u0 += kThreads) {
            const int u = u0 + tid, mm = u >> 3, run = u & 7;
            if (MR * 8 < kThreads && u >= MR * 8) break;
            constexpr int KV = KB<DD>::kVals;
            const int kb = n0 / KV, r = (n0 % KV) / 8 + run;
            const size_t pos = c0 + mm;
            float f[8], mx = 0.0f, sum;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                f[j] = ht[mm * kHt + 8 * run + j];
                mx = fmaxf(mx, fabsf(f[j]));
            }
            if constexpr (BF) {
                if (mm < cnt)
                    *reinterpret_cast<half8v*>(ha + pos * I + kb * KV + 8 * group_of_run<DD, BF>(r)) = pack_run_bf16<DD>(f);
                continue;
            }
#pragma unroll
            for (int k = 1; k < 8; k <<= 1) mx = fmaxf(mx, __shfl_xor(mx, k, 64));
            const int ex = scale_exp(mx);
            const half8v o = pack_run<DD>(f, pow2f(ex), sum);
            if (DD == NAIWA_Q4_K) {
                sum += __shfl_xor(sum, 1, 64);
                sum += __shfl_xor(sum, 2, 64);
            }
            if (mm < cnt) {
                *reinterpret_cast<half8v*>(ha + pos * I + kb * KV + 8 * group_of_run<DD, BF>(r)) = o;
                if (DD == NAIWA_Q4_K && (run & 3) == 0) put_sum(hs + (pos * (I / 256) + kb) * 16, r >> 2, sum);
                if (run == 0) he[pos * (I / kChunk) + n0 / kChunk] = (int8_t)ex;
            }
        }
        __syncthreads(); // the exchange is free for the next chunk
    }
}

// down: block (NP strips of 64 rows, K part and with SPLIT chunks as gate/up's, slot segment);
// the unweighted partial dot of (K part, sorted position, row) into dpart.  Without SPLIT a block
// takes all chunks of its segment: the split's scalars, spilled around the K loop, cost 8 experts
// of H 4096, I 14336, Q4_K, at 64 rows 84.0 us against 82.1 where there is nothing to split.
template <int DD, int NP, int MT, int MR, bool BF, bool SPLIT>
__global__ void __launch_bounds__(kThreads, 2)
down_mfma_kernel(Bank down, const _Float16* ha, const _Float16* hs, const int8_t* he, int H, int I, int ks, int kparts,
                 int npairs, const int* seg_count, const uint32_t* seg_key, const uint32_t* seg_begin, float* dpart) {
    constexpr int ST = BF && DD == NAIWA_Q8_0 ? 2 : 1; // weight stages (see Smem)
    constexpr int kFac = 34; // K parts of at most 2048: 32 chunks, rows an odd number of words apart
    __shared__ Smem<DD, NP, MR, BF, ST> sm;
    __shared__ __align__(4) uint16_t fac[BF ? 1 : MR][kFac]; // read two at a time
    __shared__ float rs[BF ? 1 : MR];
    const int sg = blockIdx.z;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, m = lane & 15;
    const uint32_t slot = scalar_ld(seg_key + sg);
    const int b = (int)scalar_ld(seg_begin + sg), e = (int)scalar_ld(seg_begin + sg + 1);
    const int segs = (int)scalar_ld((const uint32_t*)seg_count);
    asm volatile("" ::"s"(slot), "s"(b), "s"(e), "s"(segs)); // one round trip
    if (sg >= segs) return;
    const int kp = SPLIT ? blockIdx.y % kparts : blockIdx.y, k0 = kp * ks, kn = min(ks, I - k0);
    const int64_t r0 = (int64_t)blockIdx.x * (NP * kF) + 16 * wave; // matrix q: rows r0 + 64 q
    KLoop<DD, NP, MT, MR, BF, ST> kl{sm, (const uint8_t*)ha, (const uint8_t*)hs, {}, k0 / KB<DD>::kVals,
                                  kn / KB<DD>::kVals, lane, wave};
#pragma unroll
    for (int q = 0; q < NP; ++q)
        kl.wrow[q] = down.base + (int64_t)slot * down.stride + (r0 + kF * q) * down.row_bytes;
    for (int c0 = b + (SPLIT ? blockIdx.y / kparts * MR : 0); c0 < e; c0 += SPLIT ? gridDim.y / kparts * MR : MR) {
        const int cnt = min(MR, e - c0);
        kl.start(down.row_bytes, (uint32_t)I * 2, (uint32_t)(I / 256) * 32,
                 [&](int r) { return (uint32_t)(c0 + min(r, cnt - 1)); });
        // each row's scales over the K part to the smallest one of them: 32 lanes a row
        if constexpr (!BF)
#pragma unroll
        for (int i = 0; i < MR; i += kThreads / 32) {
            const int r = i + (tid >> 5), c = tid & 31;
            int ex = 127;
            if (c < kn / kChunk) ex = he[(size_t)(c0 + min(r, cnt - 1)) * (I / kChunk) + k0 / kChunk + c];
            int lo = ex;
#pragma unroll
            for (int k = 1; k < 32; k <<= 1) lo = min(lo, __shfl_xor(lo, k, 64));
            fac[r][c] = __builtin_bit_cast(uint16_t, (_Float16)pow2f(max(lo - ex, -40)));
            if (c == 0) rs[r] = pow2f(-lo);
        }
        floatx4 acc[NP][MT] = {};
        kl.template run<!BF, kFac>(fac, acc);
#pragma unroll
        for (int q = 0; q < NP; ++q)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int mm = 16 * mt + 4 * g + i;
                    if (mm < cnt) dpart[((size_t)kp * npairs + c0 + mm) * H + r0 + kF * q + m] =
                            BF ? acc[q][mt][i] : acc[q][mt][i] * rs[mm];
                }
        __syncthreads(); // the scales are free for the next chunk
    }
}

// Where h overflowed: the exponent that scale_exp gives a strip with an infinity, and no other.
constexpr int8_t kInfExp = 136 - 255;
struct HArg {
    Bank down;
    const _Float16* ha;
    const int8_t* he; // null: h in bf16, whose sums of products keep infinities
    int I, ks, q4;
    const uint32_t* slot_ids;
};

// The dot of down row r of a slot with K part kp of an h that holds infinities, as sums of
// products give it: the exact operands' split sums lose it (inf - inf in d D - dmin M and in a
// sum's low half).  Next to infinities and NaNs the finite values do not count.
__device__ float infinite_dot(const HArg& a, uint32_t slot, uint32_t pos, int kp, int r) {
    const int k0 = kp * a.ks, kn = min(a.ks, a.I - k0);
    const uint16_t* h = reinterpret_cast<const uint16_t*>(a.ha) + (size_t)pos * a.I + k0;
    const uint8_t* row = a.down.base + (int64_t)slot * a.down.stride + (int64_t)r * a.down.row_bytes;
    float sum = 0.0f;
#pragma unroll 1
    for (int k = 0; k < kn; ++k) {
        const uint32_t bits = h[k]; // position k of the K order
        if ((bits & 0x7c00u) != 0x7c00u) continue;
        float w;
        if (a.q4) {
            const uint8_t* blk = row + (k0 + k) / 256 * NAIWA_Q4_K_BYTES;
            const int G = k % 256 / 8, t = (G / 4) & 1, g = G & 3;
            const uint32_t byte = blk[16 + 32 * g + 8 * (G / 8) + q4_elem(k % 8)];
            float sc, mn;
            q4k_scale_min(*reinterpret_cast<const u32x4*>(blk), 2 * g + t, sc, mn);
            w = __builtin_fmaf((float)(t ? byte >> 4 : byte & 15u), sc, mn);
        } else {
            const uint8_t* blk = row + (k0 + k) / 32 * NAIWA_Q8_0_BYTES;
            w = naiwa_f16_to_f32(*reinterpret_cast<const uint16_t*>(blk)) * (float)(int8_t)blk[2 + k % 32];
        }
        sum += w * naiwa_f16_to_f32(bits);
    }
    return sum;
}

// out (token, row) from the K parts' unweighted dots: the token's pairs in ascending sorted
// position (= ascending slot), each w * (its parts in part order), from 0 or from out.  inv
// gives a pair's position (all ones: dropped), so a token's list takes one round of loads.
// With res (bf16 [rows, H]): x = bf16(x + y) in place.  4 rows a lane.
__global__ void __launch_bounds__(64)
combine_mfma_kernel(const float* dpart, int kparts, int npairs, int H, int width, const uint32_t* inv, const float* w,
                    int accumulate, float* out, uint16_t* res, HArg h) {
    const int lane = threadIdx.x, t = blockIdx.y, r = blockIdx.x * 256 + 4 * lane;
    const bool in = r < H;
    const uint32_t pos = lane < width ? inv[(size_t)t * width + lane] : 0xffffffffu;
    const float wv = lane < width ? w[(size_t)t * width + lane] : 0.0f;
    const size_t o = (size_t)t * H + r;
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    uint16_t x0[4] = {0, 0, 0, 0};
    if (in && accumulate)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = out[o + i]; // out is only 4-byte aligned
    if (in && res)
#pragma unroll
        for (int i = 0; i < 4; ++i) x0[i] = res[o + i];
    int rank = 0;
    for (int j = 0; j < width; ++j) rank += (uint32_t)__builtin_amdgcn_readlane((int)pos, j) < pos ? 1 : 0;
    const bool valid = pos != 0xffffffffu;
    const int cnt = __popcll(__ballot(valid));
    // pair k of the list: its position and weight, in every lane
    auto pair = [&](int k, uint32_t& pk, float& wk) {
        const int src = __ffsll((long long)__ballot(valid && rank == k)) - 1;
        pk = (uint32_t)__builtin_amdgcn_readlane((int)pos, src);
        wk = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wv), src));
    };
    auto dot = [&](int p, uint32_t pk) {
        return *reinterpret_cast<const floatx4*>(dpart + ((size_t)p * npairs + pk) * H + (in ? r : 0));
    };
    auto add = [&](float wk, const floatx4& v) {
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = __builtin_fmaf(wk, v[i], acc[i]);
    };
    constexpr int kB = 8; // loads in flight
    if (kparts == 1) {
        for (int k0 = 0; k0 < cnt; k0 += kB) {
            floatx4 v[kB];
            float wk[kB];
#pragma unroll
            for (int q = 0; q < kB; ++q)
                if (k0 + q < cnt) {
                    uint32_t pk;
                    pair(k0 + q, pk, wk[q]);
                    v[q] = dot(0, pk);
                }
#pragma unroll
            for (int q = 0; q < kB; ++q)
                if (k0 + q < cnt) add(wk[q], v[q]);
        }
    } else {
        for (int k = 0; k < cnt; ++k) {
            uint32_t pk;
            float wk;
            pair(k, pk, wk);
            floatx4 sum;
            for (int p0 = 0; p0 < kparts; p0 += kB) {
                floatx4 v[kB];
#pragma unroll
                for (int i = 0; i < kB; ++i)
                    if (p0 + i < kparts) v[i] = dot(p0 + i, pk);
#pragma unroll
                for (int i = 0; i < kB; ++i)
                    if (p0 + i < kparts) sum = p0 + i == 0 ? v[i] : sum + v[i];
            }
            add(wk, sum);
        }
    }
    // a NaN may be an infinity that the dots lost: the row's pairs again, those of infinite h by
    // infinite_dot
    const bool nan = in && h.he && (acc[0] != acc[0] || acc[1] != acc[1] || acc[2] != acc[2] || acc[3] != acc[3]);
    if (__builtin_expect(__ballot(nan) != 0, 0)) {
        float sum[4];
#pragma unroll 1
        for (int i = 0; i < 4; ++i) {
            sum[i] = in && accumulate ? out[o + i] : 0.0f;
#pragma unroll 1
            for (int k = 0; k < cnt; ++k) {
                uint32_t pk;
                float wk, v = 0.0f;
                pair(k, pk, wk);
                const int src = __ffsll((long long)__ballot(valid && rank == k)) - 1;
                const uint32_t slot = h.slot_ids[(size_t)t * width + src];
#pragma unroll 1
                for (int p = 0; p < kparts; ++p) {
                    bool inf = false;
                    for (int c = p * h.ks / kChunk; c < min((p + 1) * h.ks, h.I) / kChunk; ++c)
                        inf |= h.he[(size_t)pk * (h.I / kChunk) + c] == kInfExp;
                    v += !in ? 0.0f : inf ? infinite_dot(h, slot, pk, p, r + i)
                                          : dpart[((size_t)p * npairs + pk) * H + r + i];
                }
                sum[i] = __builtin_fmaf(wk, v, sum[i]);
            }
        }
        if (nan)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = sum[i];
    }
    if (!in) return;
    if (res)
#pragma unroll
        for (int i = 0; i < 4; ++i) res[o + i] = (uint16_t)naiwa_f32_to_bf16(naiwa_bf16_to_f32(x0[i]) + acc[i]);
    if (out)
#pragma unroll
        for (int i = 0; i < 4; ++i) out[o + i] = acc[i];
}

struct Call {
    Bank g, u, d;
    int H, I, rows, n, slots, segs, ks, kparts, act;
    int* seg_count;
    uint32_t *seg_key, *seg_begin, *tok;
    _Float16 *xa, *xs, *ha, *hs;
    float *xr, *dpart;
    int8_t* he;
    hipStream_t st;
};

template <int DG, int DD, int MT, int MR, bool BF>
void experts(const Call& c) {
    // Blocks along a segment: a block takes every nz-th chunk of its tokens.  One, except where
    // the segments average so many tokens that most have several chunks and no CU has a second
    // gate/up block to turn to; then as many as chunks (of 32 tokens in about an average and a
    // deviation), up to 8 blocks a CU.  One and nz, whole calls: 4 experts, H 512, I 1024, 64 / 200
    // rows (32 / 100 tokens a segment) Q8_0 38.7 / 69.7 and 26.1 / 27.4 us, Q4_K 32.6 / 57.8 and
    // 23.0 / 25.2; 8 experts, H 4096, I 2048, 128 rows Q8_0 118 and 86.  Below: 24 tokens 66.9 and
    // 74.0 there (one chunk each).  More blocks: 8 experts, H 4096, I 8192, Q4_K, 45 tokens 246 and 258.
    const int gub = c.I / kF * c.segs;
    int nz = 1;
    if (MR == 32 && gub <= 256 && c.n >= 25 * c.segs)
        nz = (int)std::min<int64_t>(((int64_t)c.n + 42 * c.segs - 1) / (32 * c.segs), 2048 / gub);
    auto gateup = [&](auto* kernel) {
        kernel<<<dim3(c.I / kF, c.segs, nz), kThreads, 0, c.st>>>(
            c.g, c.u, c.xa, c.xs, c.xr, c.H, c.I, c.seg_count, c.seg_key, c.seg_begin, c.tok, c.act, c.ha, c.hs, c.he);
    };
    // A Q8_0 K-block is half as long as a Q4_K one, so its copies' latency shows twice as often:
    // two weight stages where the LDS for them costs no block a CU: rounded operands, and gate/up
    // of the smaller tiles while a CU has one block at most.  One and two stages, Q8_0: a layered
    // layer of 17 / 64 rows at H 2048, I 768, 128 experts 68.0 / 117.9 and 63.6 / 110.1 us; exact,
    // 4 rows, 60 experts, H 3072, I 1024 43.9 and 41.9; 16 rows, 256 experts, H 1024, I 512 (1,024
    // gate/up blocks) 53.9 and 57.1, and down at 64 rows, 128 experts, H 2048, I 768 111 and 114.
    constexpr bool q8 = DG == NAIWA_Q8_0;
    if constexpr (q8 && !BF && MR < 32) {
        if (gub <= 256)
            gateup(gateup_mfma_kernel<DG, DD, MT, MR, BF, 2>);
        else
            gateup(gateup_mfma_kernel<DG, DD, MT, MR, BF, 1>);
    } else {
        gateup(gateup_mfma_kernel<DG, DD, MT, MR, BF, q8 && BF ? 2 : 1>);
    }
    auto down = [&](auto* kernel, int np) {
        kernel<<<dim3(c.H / (np * kF), c.kparts * nz, c.segs), kThreads, 0, c.st>>>(
            c.d, c.ha, c.hs, c.he, c.H, c.I, c.ks, c.kparts, c.n, c.seg_count, c.seg_key, c.seg_begin, c.dpart);
    };
    const bool one = naiwa_decode_mfma_down_strips(c.rows, c.n / c.rows, c.slots, c.H, c.kparts,
                                                   DD == NAIWA_Q4_K && !BF) == 1;
    auto strips = [&](auto split) {
        if (one)
            down(down_mfma_kernel<DD, 1, MT, MR, BF, split>, 1);
        else
            down(down_mfma_kernel<DD, 2, MT, MR, BF, split>, 2);
    };
    if constexpr (MR == 32)
        if (nz > 1) return strips(std::true_type{});
    strips(std::false_type{});
}

// Token rows of the A tile.  8: a segment of a call of at most 8 rows holds no more (unless
// a token repeats a slot), and the smaller tile lets a fifth block fit on a CU.  32 when
// segments average more than 8 tokens: a weight is then unpacked once per 32 tokens.
template <int DG, int DD, bool BF>
void experts_rows(const Call& c) {
    if (c.rows <= 8)
        experts<DG, DD, 1, 8, BF>(c);
    else if (c.n > 8 * c.segs)
        experts<DG, DD, 2, 32, BF>(c);
    else
        experts<DG, DD, 1, 16, BF>(c);
}

template <int DG, int DD>
void experts_rounding(const Call& c, bool bf) {
    if (bf)
        experts_rows<DG, DD, true>(c);
    else
        experts_rows<DG, DD, false>(c);
}

bool fmt_ok(int dt, int k) {
    return (dt == NAIWA_Q4_K && k % KB<NAIWA_Q4_K>::kVals == 0) || (dt == NAIWA_Q8_0 && k % KB<NAIWA_Q8_0>::kVals == 0);
}

size_t a256(size_t b) { return (b + 255) & ~size_t(255); }

} // namespace

bool naiwa_decode_mfma_ok(const naiwa_bank* gate, const naiwa_bank* up, const naiwa_bank* down, const void* x) {
    const int H = gate->k, I = gate->n;
    if (gate->dtype != up->dtype || !fmt_ok(gate->dtype, H) || !fmt_ok(down->dtype, I)) return false;
    if (H % kF || I % kF) return false;
    if ((uint64_t)naiwa_row_bytes(gate->dtype, H) * 16 > UINT32_MAX || (uint64_t)naiwa_row_bytes(down->dtype, I) * 16 > UINT32_MAX)
        return false; // 32-bit offsets within a wave's rows
    return ((uintptr_t)x & 15) == 0; // 16-byte loads of x
}

NaiwaMfmaLayout::NaiwaMfmaLayout(int rows, int width, int H, int I, int kparts, int down_dtype) {
    const size_t n = (size_t)rows * width;
    off_key = 256;
    off_begin = off_key + a256(n * 4);
    off_perm = off_begin + a256((n + 1) * 4);
    off_inv = off_perm + a256(n * 4);
    off_ha = off_inv + a256(n * 4);
    off_hs = off_ha + a256(n * I * 2);
    off_he = off_hs + (down_dtype == NAIWA_Q4_K ? a256(n * (I / 256) * 32) : 0);
    // the laid-out x, which gate/up reads, and over it the dots that down writes after it
    off_xa = off_dpart = off_he + a256(n * (I / kChunk));
    off_xs = off_xa + a256((size_t)rows * H * 2);
    off_xr = off_xs + a256((size_t)rows * (H / 256) * 32);
    total = std::max(off_xr + a256((size_t)rows * 4), off_dpart + (size_t)kparts * n * H * 4);
}

// Strips of 64 down rows a block: one where two leave few blocks a CU.  A block walks its K part
// one K-block's latency after the other, and a second strip makes each of them longer (with
// exact Q4_K operands least, which unpack the least and share each A operand between strips);
// past 1.4 blocks a CU one strip pays where the halves spread evener, so that the fullest CU has
// fewer strips, up to 4 blocks a CU.  The blocks counted are those that have a segment when the rows' slots
// are drawn evenly.  Two and one strips (blocks of two, as counted), weights cold: Q8_0, 8 experts, H
// 4096, I 2048, 4 rows (175) 65.6 and 60.2 us; 60 experts, H 3072, I 1024, 4 rows (347) 51.1 and
// 48.8; H 2048, I 1408, 8 / 32 rows (407 / 854) 72.3 and 72.7 / 131.1 and 125.7; 16 experts, H 4096, I 1024, 64 rows
// (512) 63.3 and 64.5; 32 experts, H 2560, I 1536, 64 rows (640) 107.5 and 103.8; 8 experts, H
// 6144, I 4096, 16 rows (760) 136.9 and 139.6; H 4096, I 14336, 64 rows (1,792) 347 and 354.  Exact
// Q4_K, 8 experts, H 4096, I 2048, 16 rows (253) 47.3 and 45.3; 60 experts, H 3072, I 1024, 4 / 16
// rows (347 / 963) 37.8 and 36.3 / 65.9 and 68.2; 8 experts, H 4096, I 14336, 64 rows 230 and 243.
extern "C" int naiwa_decode_mfma_down_strips(int rows, int width, int slots, int H, int kparts, int exact_q4) {
    const double miss = 1.0 - std::min(1.0, (double)width / slots); // a slot's chance to be in no pair of a row
    const double fill = (double)(H / (2 * kF)) * kparts * slots * (1.0 - std::pow(miss, rows)) / 256; // blocks a CU
    if (fill <= 1.4) return 1;
    if (exact_q4 || fill >= 4.0) return 2;
    return std::ceil(2.0 * fill) < 2.0 * std::ceil(fill - 0.04) ? 1 : 2;
}

int naiwa_decode_mfma_rows_per_pass(int rows, int width, int H, int I, int kparts, int down_dtype, size_t bytes) {
    auto fits = [&](int q) {
        return NaiwaMfmaLayout(q, width, H, I, kparts, down_dtype).total <= bytes &&
               (uint64_t)q * H * 2 <= UINT32_MAX && (uint64_t)q * width * I * 2 <= UINT32_MAX; // 32-bit offsets
    };
    int passes = 1, r = rows;
    while (r > 1 && !fits(r)) r = (rows + passes) / (passes + 1), ++passes; // rows in passes + 1 passes, rounded up
    return r;
}

int naiwa_decode_mfma(const naiwa_bank* gate, const naiwa_bank* up, const naiwa_bank* down, const void* x, int x_dtype,
                      const uint32_t* slot_ids, const float* w, int rows, int width, int act, float* out,
                      int accumulate, uint16_t* res, int ks, int kparts, bool bf16, uint8_t* ws, hipStream_t st) {
    const int H = gate->k, I = gate->n, n = rows * width;
    const NaiwaMfmaLayout L(rows, width, H, I, kparts, down->dtype);
    Call c;
    c.g = Bank{(const uint8_t*)gate->base, gate->slot_stride, naiwa_row_bytes(gate->dtype, H)};
    c.u = Bank{(const uint8_t*)up->base, up->slot_stride, naiwa_row_bytes(up->dtype, H)};
    c.d = Bank{(const uint8_t*)down->base, down->slot_stride, naiwa_row_bytes(down->dtype, I)};
    c.H = H, c.I = I, c.rows = rows, c.n = n;
    c.slots = gate->slots, c.segs = std::max(1, std::min(n, gate->slots));
    c.ks = ks, c.kparts = kparts, c.act = act, c.st = st;
    c.seg_count = (int*)ws;
    c.seg_key = (uint32_t*)(ws + L.off_key);
    c.seg_begin = (uint32_t*)(ws + L.off_begin);
    c.tok = (uint32_t*)(ws + L.off_perm);
    uint32_t* inv = (uint32_t*)(ws + L.off_inv);
    c.xa = (_Float16*)(ws + L.off_xa), c.xs = (_Float16*)(ws + L.off_xs), c.xr = (float*)(ws + L.off_xr);
    c.ha = (_Float16*)(ws + L.off_ha), c.hs = (_Float16*)(ws + L.off_hs), c.he = (int8_t*)(ws + L.off_he);
    c.dpart = (float*)(ws + L.off_dpart);
    const int xb = x_dtype == NAIWA_BF16;
    const bool g4 = gate->dtype == NAIWA_Q4_K, d4 = down->dtype == NAIWA_Q4_K;
    auto* prep = g4 ? (bf16 ? seg_prep_kernel<NAIWA_Q4_K, true> : seg_prep_kernel<NAIWA_Q4_K, false>)
                    : (bf16 ? seg_prep_kernel<NAIWA_Q8_0, true> : seg_prep_kernel<NAIWA_Q8_0, false>);
    prep<<<rows + 1, kThreads, 0, st>>>(slot_ids, w, n, width, gate->slots, c.tok, inv, c.seg_count, c.seg_key,
                                        c.seg_begin, (int*)(ws + 4), x, xb, H, c.xa, c.xs, c.xr);
    if (g4 && d4)
        experts_rounding<NAIWA_Q4_K, NAIWA_Q4_K>(c, bf16);
    else if (g4)
        experts_rounding<NAIWA_Q4_K, NAIWA_Q8_0>(c, bf16);
    else if (d4)
        experts_rounding<NAIWA_Q8_0, NAIWA_Q4_K>(c, bf16);
    else
        experts_rounding<NAIWA_Q8_0, NAIWA_Q8_0>(c, bf16);
    const HArg h{c.d, c.ha, bf16 ? nullptr : c.he, I, ks, d4, slot_ids};
    combine_mfma_kernel<<<dim3((H + 255) / 256, rows), 64, 0, st>>>(c.dpart, kparts, n, H, width, inv, w, accumulate, out,
                                                                    res, h);
    return naiwa_hip_rc(hipGetLastError());
}
