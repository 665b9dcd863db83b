// Prefill's GEMMs over many rows an expert: tiles of up to 128 pairs, two weight strips a
// wave.
//
// The 64-row kernels are bound twice over at once there: a wave's 32-row strip is unpacked
// for 2 MFMAs a step (22 VALU operations x 4 cycles against 64 cycles of MFMA) and each
// of them reads its A operand from LDS (128 B/cycle a CU, 100 % of its rate).  With 4
// waves of two strips and up to four 32-row subtiles, a step unpacks two weight operands
// and reads four A operands for 8 MFMAs (256 cycles): VALU about 70 % and LDS 50 % of the
// MFMA time.  Two blocks of 4 waves share a CU (at most 256 VGPRs, 66 KB of LDS each).
//
// Measured, whole calls with the router: 4,096 tokens of 8 experts top-2, H 4096, I 14336,
// Q4_K 3,924 -> 3,061 us (0.74 -> 0.94 PFLOP/s; a library bf16 product of 8192^3 reaches
// 1.24 on this card); 1,999 tokens of 128 experts top-8, H 2048, I 768 516 -> 438 us.  In
// the first, MFMA is busy 57 % and VALU 55 % of gate/up's cycles, 50 % and 44 % of down's.
// With A loaded behind the weights it took 3,184 us; that build without the unpacking 2,558,
// without the staging of A 2,449.
// An interleaving of VALU and MFMA forced by sched_group_barrier was 2 % slower.
#pragma once

#include <type_traits>

// Whether a call of n pairs over `slots` experts takes the 128-pair tiles (prefill.hip).
extern "C" int naiwa_prefill_wide_tiles(int64_t n, int slots, int I);

namespace {

constexpr int kWide = 256;   // 4 waves, two 32-feature weight strips each
constexpr int kWideM = 128;  // pairs per tile: up to four 32-row MFMA subtiles

// One lane's share of a weight row for one K-block: raw words, unpacked step by step into
// the MFMA B operand (8 bf16).  load_part(p) fetches the words of part p (kPartSteps steps);
// a part is replaced by the next K-block's as soon as its last step is unpacked, so a lane
// holds one K-block of its rows and a whole K-block of MFMA work hides each load.
template <int DT> struct WideBRow;

template <> struct WideBRow<NAIWA_Q4_K> {
    static constexpr int kParts = 4, kPartSteps = 4;
    u32x4 hd;   // d, dmin, 12 scale bytes
    u32x4 q[4]; // per 64-value chunk: bytes 16h .. 16h + 15 of its 32 quant bytes
    float sc[2], mn[2]; // of the part being unpacked

    __device__ __forceinline__ void load_head(const uint8_t* base, uint32_t off) {
        hd = *reinterpret_cast<const u32x4*>(base + off);
    }
    __device__ __forceinline__ void load_part(const uint8_t* base, uint32_t off, int h, int p) {
        q[p] = *reinterpret_cast<const u32x4*>(base + (16 + 32 * p) + (off + 16u * h));
    }
    __device__ __forceinline__ void scales(int p) {
        q4k_scale_min(hd, 2 * p, sc[0], mn[0]);
        q4k_scale_min(hd, 2 * p + 1, sc[1], mn[1]);
    }
    __device__ __forceinline__ bf16x8 step(int s, int, const NibMask& nm) const {
        const int c = s / 4, t = s % 4;
        const uint32_t da = (t % 2) ? q[c].z : q[c].x, db = (t % 2) ? q[c].w : q[c].y;
        return q4k_unpack(da, db, t / 2, nm, sc[t / 2], mn[t / 2]);
    }
};

template <> struct WideBRow<NAIWA_Q8_0> {
    static constexpr int kParts = 2, kPartSteps = 4;
    typedef u32x4 u32x4a __attribute__((aligned(4)));
    // Block 2j + h of the K-block, at byte 2h of a word (68-byte pairs of blocks, rows of
    // whole words): its scale, and the 32 values' bytes from the word that holds the first
    // (h = 0: from its third byte on, so 9 words; h = 1: 8 whole words).
    u32x4 w[2][2];
    uint32_t last[2];
    uint16_t d[2];
    float sc;

    __device__ __forceinline__ void load_head(const uint8_t*, uint32_t) {}
    __device__ __forceinline__ void load_part(const uint8_t* base, uint32_t off, int h, int p) {
        const uint8_t* blk = base + 2 * p * NAIWA_Q8_0_BYTES;
        d[p] = *reinterpret_cast<const uint16_t*>(blk + (off + (uint32_t)NAIWA_Q8_0_BYTES * h));
        w[p][0] = *reinterpret_cast<const u32x4a*>(blk + (off + (NAIWA_Q8_0_BYTES + 2u) * h));
        w[p][1] = *reinterpret_cast<const u32x4a*>(blk + 16 + (off + (NAIWA_Q8_0_BYTES + 2u) * h));
        // h = 1 has no ninth word (it would lie past the row): its eighth again, unused
        last[p] = *reinterpret_cast<const uint32_t*>(blk + 32 + (off + (NAIWA_Q8_0_BYTES - 2u) * h));
    }
    __device__ __forceinline__ void scales(int p) { sc = naiwa_f16_to_f32(d[p]); }
    __device__ __forceinline__ bf16x8 step(int s, int h, const NibMask&) const {
        const int j = s / 4, u = s % 4;
        auto word = [&](int i) -> uint32_t { return i == 8 ? last[j] : w[j][i / 4][i % 4]; };
        const uint32_t sh = 2u - 2u * (uint32_t)h;
        const uint32_t d0 = __builtin_amdgcn_alignbyte(word(2 * u + 1), word(2 * u), sh);
        const uint32_t d1 = __builtin_amdgcn_alignbyte(word(2 * u + 2), word(2 * u + 1), sh);
        return q8_unpack(d0, d1, sc);
    }
};

// LDS A tile of one chunk of kChunk values: group g of tile row m at [g][m] (16 bytes
// each), rows of groups padded to kWideM + 1 slots.  A step's read of 32 rows of one group
// covers 32 consecutive slots at an offset fixed at compile time from the lane's own base;
// a staging store of consecutive groups of one row steps 16 (kWideM + 1) bytes (16 mod 256)
// from lane to lane, so it spreads over the banks.
constexpr int kChunk = 128, kChunkSteps = 8, kGroups = 2 * kChunkSteps;
struct WideATile {
    u32x4 v[kGroups][kWideM + 1];
};

// Each thread's share of staging one half of a chunk of the A tile's first 32 MS rows:
// global -> registers (issued early) -> LDS (half a chunk's steps later).
template <int MS> struct WideAStage {
    u32x4 r[MS]; // 16-byte pieces per thread and half: 32 MS rows x 16 groups / 256 threads / 2
    // base: the activation matrix (a kernel argument, so the loads are global ones);
    // rows[m]: byte offset of tile row m.  Piece p: row p / 16, group p % 16.
    __device__ __forceinline__ void load(const uint16_t* base, const uint32_t* rows, int chunk, int half, int tid) {
#pragma unroll
        for (int i = 0; i < MS; ++i) {
            const int p = tid + kWide * (MS * half + i), m = p / kGroups, g = p % kGroups;
            r[i] = *reinterpret_cast<const u32x4*>((const uint8_t*)(base + chunk * kChunk) + (rows[m] + 16u * g));
        }
    }
    __device__ __forceinline__ void store(WideATile& a, int half, int tid) const {
#pragma unroll
        for (int i = 0; i < MS; ++i) {
            const int p = tid + kWide * (MS * half + i);
            a.v[p % kGroups][p / kGroups] = r[i];
        }
    }
};

// The K loop of one tile: acc[n][ms] += A (32 MS rows staged through the LDS double buffer
// `as`) x B (this lane's share of the weight rows at w[n] + off; w[n] is uniform over the
// wave, so a load's address is a scalar base and one 32-bit register).  Loads run one chunk
// (A) or one K-block (B) ahead; the last ones reload themselves, so that the loads are
// unconditional and the compiler waits only for the registers each step uses.
template <int DT, int MS>
__device__ __forceinline__ void wide_k_loop(const uint16_t* abase, const uint32_t* rows, const uint8_t* const (&w)[2],
                                            uint32_t off, int nkb, WideATile* as, int tid, int lane, int h,
                                            floatx16 (&acc)[2][MS]) {
    constexpr int kPerBlock = KBlock<DT>::kVals / kChunk; // chunks of a K-block
    typedef WideBRow<DT> Row;
    const NibMask nm = nib_mask();
    WideAStage<MS> st;
    Row b[2];
    const int nchunks = nkb * kPerBlock;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        b[n].load_head(w[n], off);
#pragma unroll
        for (int p = 0; p < Row::kParts; ++p) b[n].load_part(w[n], off, h, p);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        st.load(abase, rows, 0, half, tid);
        st.store(as[0], half, tid);
    }
    st.load(abase, rows, min(1, nchunks - 1), 0, tid);
    __syncthreads();
    // this lane's A operand slot in buffer 0: step s, subtile ms reads
    // alane[buffer + 2 s (kWideM + 1) + 32 ms]
    const u32x4* alane = &as[0].v[h][lane & 31];
    constexpr int kBuf = sizeof(WideATile) / sizeof(u32x4);
    for (int kb = 0; kb < nkb; ++kb) {
        const size_t kn = (size_t)min(kb + 1, nkb - 1) * KBlock<DT>::kBytes;
#pragma unroll
        for (int c = 0; c < kPerBlock; ++c) {
            const int chunk = kb * kPerBlock + c;
            const int buf = kPerBlock == 2 ? c : (kb & 1);
            const u32x4* ab = alane + buf * kBuf;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                constexpr int kHalf = kChunkSteps / 2;
                const int part = (c * kChunkSteps + half * kHalf) / Row::kPartSteps;
#pragma unroll
                for (int n = 0; n < 2; ++n) b[n].scales(part);
                // the last part's scales are taken: the next header can replace this one
                if (part == Row::kParts - 1) {
#pragma unroll
                    for (int n = 0; n < 2; ++n) b[n].load_head(w[n] + kn, off);
                }
                __builtin_amdgcn_sched_barrier(0); // keep the prefetches where they are issued
#pragma unroll
                for (int t = 0; t < kHalf; ++t) {
                    const int cs = half * kHalf + t; // step of the chunk
                    bf16x8 x8[MS];
#pragma unroll
                    for (int ms = 0; ms < MS; ++ms)
                        x8[ms] = __builtin_bit_cast(bf16x8, ab[2 * cs * (kWideM + 1) + 32 * ms]);
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        const bf16x8 wv = b[n].step(c * kChunkSteps + cs, h, nm);
#pragma unroll
                        for (int ms = 0; ms < MS; ++ms)
                            acc[n][ms] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x8[ms], wv, acc[n][ms], 0, 0, 0);
                    }
                }
                // The next half chunk of A before the weights: the loads are waited for in
                // their order, and the store of this half a chunk on must not wait for the
                // weights issued here (their latency is HBM's).
                __builtin_amdgcn_sched_barrier(0);
                st.store(as[buf ^ 1], half, tid);
                st.load(abase, rows, min(chunk + 1 + half, nchunks - 1), half ^ 1, tid);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int n = 0; n < 2; ++n) b[n].load_part(w[n] + kn, off, h, part);
                __builtin_amdgcn_sched_barrier(0);
            }
            lds_barrier();
        }
    }
}

// fn(std::integral_constant<int, MS>) for the 32-row subtiles that cnt <= 128 rows need.
template <class F>
__device__ __forceinline__ void by_subtiles(int cnt, F&& fn) {
    const int subs = (cnt + 31) / 32;
    if (subs == 4) return fn(std::integral_constant<int, 4>{});
    if (subs == 3) return fn(std::integral_constant<int, 3>{});
    if (subs == 2) return fn(std::integral_constant<int, 2>{});
    fn(std::integral_constant<int, 1>{});
}

// gate/up: one tile of <= 128 pairs x 128 intermediate features; each wave takes the gate
// and the up rows of 32 features, so act(gate) * up needs no exchange.  xp: x in the K
// order of DG; hp (out): h in the K order of DD, bf16 [pairs, I].
template <int DG, int DD>
__global__ void __launch_bounds__(kWide, 2)
wide_gateup_kernel(Bank gate, Bank up, const uint16_t* xp, int H, int I, int k, const uint32_t* perm, Tiles tl,
              int act, uint16_t* hp, int xcd) {
    __shared__ WideATile as[2];
    __shared__ uint32_t rows[kWideM];
    int tile = 0, colb = 0;
    if (!tile_col(blockIdx.x, *tl.n, I / kTNG, xcd, &tile, &colb)) return;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int start = tl.start[tile], cnt = tl.count[tile], slot = tl.slot[tile];
    if (tid < kWideM) rows[tid] = perm[start + min(tid, cnt - 1)] / k * (uint32_t)H * 2u;
    const int n0 = colb * kTNG + 32 * wave, n = n0 + (lane & 31); // the wave's first weight row, the lane's
    const uint8_t* const w[2] = {gate.base + (int64_t)slot * gate.stride + (int64_t)n0 * gate.row_bytes,
                                 up.base + (int64_t)slot * up.stride + (int64_t)n0 * up.row_bytes};
    const uint32_t off = (uint32_t)(lane & 31) * (uint32_t)gate.row_bytes; // up has gate's format
    const int nkb = H / KBlock<DG>::kVals;
    __syncthreads();

    const int col = laid_pos<DD>(n);
    by_subtiles(cnt, [&](auto sub) {
        constexpr int MS = decltype(sub)::value;
        floatx16 acc[2][MS] = {};
        wide_k_loop<DG, MS>(xp, rows, w, off, nkb, as, tid, lane, h, acc);
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = 32 * ms + 8 * (v / 4) + 4 * h + v % 4;
                if (m < cnt)
                    hp[(size_t)(start + m) * I + col] =
                        (uint16_t)bf16x2_bits(naiwa_act(act, acc[0][ms][v]) * acc[1][ms][v], 0.0f);
            }
    });
}

// down: one tile of <= 128 pairs x 256 output features (64 per wave); pair rows scaled by
// their weight.
template <int DD>
__global__ void __launch_bounds__(kWide, 2)
wide_down_kernel(Bank down, const uint16_t* hp, int H, int I, const uint32_t* perm, const float* w, Tiles tl,
            float* ypair, int xcd) {
    __shared__ WideATile as[2];
    __shared__ uint32_t rows[kWideM], pair[kWideM]; // activation row, pair index, routing weight
    __shared__ float pw[kWideM];
    int tile = 0, col = 0;
    if (!tile_col(blockIdx.x, *tl.n, H / kTND, xcd, &tile, &col)) return;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int start = tl.start[tile], cnt = tl.count[tile], slot = tl.slot[tile];
    if (tid < kWideM) {
        const int at = start + min(tid, cnt - 1);
        rows[tid] = (uint32_t)at * (uint32_t)I * 2u;
        pair[tid] = perm[at];
        pw[tid] = w[pair[tid]];
    }
    const int n0 = col * kTND + 64 * wave, n = n0 + (lane & 31);
    const uint8_t* r0 = down.base + (int64_t)slot * down.stride + (int64_t)n0 * down.row_bytes;
    const uint8_t* const wr[2] = {r0, r0 + 32 * down.row_bytes};
    const uint32_t off = (uint32_t)(lane & 31) * (uint32_t)down.row_bytes;
    const int nkb = I / KBlock<DD>::kVals;
    __syncthreads();

    by_subtiles(cnt, [&](auto sub) {
        constexpr int MS = decltype(sub)::value;
        floatx16 acc[2][MS] = {};
        wide_k_loop<DD, MS>(hp, rows, wr, off, nkb, as, tid, lane, h, acc);
#pragma unroll
        for (int ms = 0; ms < MS; ++ms)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = 32 * ms + 8 * (v / 4) + 4 * h + v % 4;
                if (m < cnt) {
                    float* y = ypair + (size_t)pair[m] * H + n;
                    const float wp = pw[m];
#pragma unroll
                    for (int s = 0; s < 2; ++s) y[32 * s] = acc[s][ms][v] * wp;
                }
            }
    });
}

} // namespace
