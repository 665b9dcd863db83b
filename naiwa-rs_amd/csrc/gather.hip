// naiwa_moe_gather: the token->expert gather as a stable counting sort by
// expert id.  The reference groups hits per bank in row-major order
// (src/moe/stages/gpu.rs:100-133); here every (token, k) pair of a step is
// grouped by expert id, ties kept in flat index order, so the permutation and
// the per-expert offsets are bit-exact against the CPU counting sort.
#include "segments.h"

namespace {

__global__ void __launch_bounds__(NAIWA_SEG_THREADS)
gather_kernel(const uint32_t* ids, int n, int E, uint32_t* perm, uint32_t* offsets, int* bad) {
    __shared__ NaiwaSegSmem sm;
    naiwa_segment(sm, ids, nullptr, n, E, perm, offsets, nullptr, nullptr, nullptr, bad);
}

// The same stable counting sort with one block per expert id e: its segment starts at
// the number of valid ids below e, and its entries keep their flat order.  All ids in
// parallel: for many entries and few ids (a prefill chunk's routing) it replaces the
// one-block sort's serial chunks.  Every block reads all n ids, once: each of its W waves
// keeps the contiguous entries 64 R w .. 64 R (w + 1) - 1 in registers, R a lane, counts its
// own, and after one exchange of the waves' counts places them without another barrier.
// (With chunks of 256 entries and two barriers each, 16K pairs of 128 experts took 37 us.)
template <int R, int W>
__global__ void __launch_bounds__(64 * W)
gather_by_id_kernel(const uint32_t* ids, int n, int E, uint32_t* perm, uint32_t* offsets, int* bad) {
    __shared__ uint32_t sums[3][W]; // of each wave: ids below e, outside [0, E), equal to e
    const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i0 = 64 * R * wave + lane;
    uint32_t id[R];
#pragma unroll
    for (int r = 0; r < R; ++r) id[r] = i0 + 64 * r < n ? ids[i0 + 64 * r] : 0u;
    uint32_t below = 0, outside = 0, mine = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool in = i0 + 64 * r < n;
        below += (uint32_t)__popcll(__ballot(in && id[r] < (uint32_t)e));
        outside += (uint32_t)__popcll(__ballot(in && id[r] >= (uint32_t)E));
        mine += (uint32_t)__popcll(__ballot(in && id[r] == (uint32_t)e));
    }
    if (lane == 0) {
        sums[0][wave] = below;
        sums[1][wave] = outside;
        sums[2][wave] = mine;
    }
    __syncthreads();
    uint32_t start = 0, nbad = 0, before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        start += sums[0][w];
        nbad += sums[1][w];
        total += sums[2][w];
        if (w < wave) before += sums[2][w];
    }
    const uint64_t lower = (1ull << lane) - 1ull;
    uint32_t at = start + before;
    if (mine) { // the wave's count: uniform
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool me = i0 + 64 * r < n && id[r] == (uint32_t)e;
            const uint64_t m = __ballot(me);
            if (me) perm[at + (uint32_t)__popcll(m & lower)] = (uint32_t)(i0 + 64 * r);
            at += (uint32_t)__popcll(m);
        }
    }
    if (tid == 0) {
        offsets[e] = start;
        if (e == E - 1) offsets[E] = start + total;
        if (e == 0 && bad) *bad = (int)nbad;
    }
}

} // namespace

extern "C" int naiwa_moe_gather(const uint32_t* ids, int n, int E, uint32_t* perm_out,
                                uint32_t* offsets_out, int* bad_out, int64_t stream) {
    if (n < 0 || n > 65536 || E <= 0 || E > NAIWA_SEG_MAX_KEYS) return NAIWA_E_INVALID;
    if (!offsets_out || (n > 0 && (!ids || !perm_out))) return NAIWA_E_INVALID;
    // one block per id while that stays cheap (every block reads all n ids), else one block
    if (n > NAIWA_SEG_THREADS && (int64_t)n * E <= (int64_t)1 << 24) {
        // The fewest waves whose entries a lane holds in 16 registers: with more ids than CUs
        // the blocks' waves fill the chip several times over.  4, 8 and 16 waves: 257 ids of
        // 4,096 3.9 / 5.8 / 11.8 us, 2,048 of 2,048 4.1 / 4.4 / 7.6, 8,192 of 1,024 8.4 / 7.0 /
        // 9.7, 8,192 of 128 6.7 / 4.1 / 4.1, 16,384 of 128 11.9 / 7.2 / 5.4 (of 1,024 21.9 /
        // 15.0 / 16.1).
        auto launch = [&](auto* kernel, int waves) {
            kernel<<<E, 64 * waves, 0, (hipStream_t)stream>>>(ids, n, E, perm_out, offsets_out, bad_out);
        };
        if (n <= 1024)
            launch(gather_by_id_kernel<4, 4>, 4);
        else if (n <= 2048)
            launch(gather_by_id_kernel<8, 4>, 4);
        else if (n <= 4096)
            launch(gather_by_id_kernel<8, 8>, 8);
        else if (n <= 8192)
            launch(gather_by_id_kernel<16, 8>, 8);
        else if (n <= 16384)
            launch(gather_by_id_kernel<16, 16>, 16);
        else if (n <= 32768)
            launch(gather_by_id_kernel<32, 16>, 16);
        else
            launch(gather_by_id_kernel<64, 16>, 16);
    } else
        gather_kernel<<<1, NAIWA_SEG_THREADS, 0, (hipStream_t)stream>>>(ids, n, E, perm_out, offsets_out,
                                                                         bad_out);
    return naiwa_hip_rc(hipGetLastError());
}
