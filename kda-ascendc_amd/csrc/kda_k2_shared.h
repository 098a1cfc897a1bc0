// Stage-2 helpers shared by the stage-2 kernels (kda_k2.hip: one value
// tile per work-group; kda_k2w.hip: several): the record ring's direct
// buffer->LDS loads and waits, the chunk barrier, the decay broadcast and the
// fp32 state slices of a value tile.
#pragma once

#include "kda_common.h"

namespace kda {
namespace {

typedef __attribute__((address_space(3))) uint8_t lds_u8;

// The sequence of rank s when the N packed sequences are ordered longest
// first (up to 64 sequences; beyond that, or past the last, s itself).
__device__ __forceinline__ int longest_first(const Params& p, int s) {
    if (p.N > 64) return s;
    const int lane = threadIdx.x & 63;
    const int len = lane < p.N ? cu_at(p, lane + 1) - cu_at(p, lane) : -1;
    // rank of this lane's sequence: the sequences longer, or as long with a
    // lower index
    int rank = 0;
    for (int m = 0; m < p.N; ++m) {
        const int lm = __builtin_amdgcn_readlane(len, m);
        rank += (lm > len || (lm == len && m < lane)) ? 1 : 0;
    }
    const uint64_t hit = __ballot(lane < p.N && rank == s);
    if (hit == 0) return s;  // (the ranks are a permutation: past the last only)
    return __builtin_amdgcn_readfirstlane((int)__builtin_ctzll(hit));
}

// Stage 2's work-group -> (sequence or batch row, value head) bh and slice of
// the head's value tiles, NSL slices a head, XCD aware: work-group ids go to
// the XCDs round-robin, so the slices of a head, on ids of one residue class
// mod 8, share that XCD's L2 for the records.  Batch rows: XCD x takes the
// x-th eighth of the work-groups.  Packed sequences, whose chains differ in
// length: the heads are dealt to the XCDs in turn and, where the work-groups
// outnumber the CUs, longest sequences first, so that each XCD has its share
// of every sequence and starts its longest chains at once.  (An eighth of the
// heads each put whole sequences on one XCD: 6 sequences of 33 to 1311 tokens,
// HV = 16, the training forward's stage 2 109 us against 68, the reverse chain
// 129 against 90.  Where all work-groups start at once their order does not
// matter, and finding it costs a load and ~1 us.)  False past the last head
// (grid: k2_grid).
constexpr int CU_COUNT = 256;  // of a whole card; on fewer the order only differs for the sizes in between
template <int NSL>
__device__ __forceinline__ bool k2_pair(const Params& p, int wg, int& bh, int& slice) {
    const int nbh = (p.cu_seqlens ? p.N : p.B) * p.HV;
    const int xcd = wg & 7, j = wg >> 3;
    if (p.cu_seqlens) {
        slice = j % NSL;
        const int idx = (j / NSL) * 8 + xcd;
        if (idx >= nbh) return false;
        bh = idx;
        if (nbh * NSL > CU_COUNT) {
            const int s = idx / p.HV;
            bh = longest_first(p, s) * p.HV + (idx - s * p.HV);
        }
        return true;
    }
    const int total = nbh * NSL;
    const int lin = xcd * (NSL == 8 ? nbh : (total + 8 * NSL - 1) / (8 * NSL) * NSL) + j;
    bh = lin / NSL;
    slice = lin - bh * NSL;
    return lin < total;
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N));
}

// Buffer descriptor word 3 for raw byte-addressed buffers on gfx9-family
// parts (gfx950 included).
constexpr int BUF_DWORD3 = 0x00020000;

// Lane (x, q4) reads 2^G_last at [kt = x/2][q4][i = 2*(x%2) .. +1].
__device__ __forceinline__ uint32_t decay_offset(int lane) {
    const int x = lane & 15, q4 = lane >> 4;
    return REC_DECAY + (x >> 1) * 64 + q4 * 16 + (x & 1) * 8;
}

// Scales the state tile kt by its decay: element i of lane (x, q4) takes
// 2^G_last[16*kt + 4*q4 + i] from lane 2*kt + i/2 of its row (DPP
// row_newbcast, row_bcast in kda_common.h), component i % 2.
template <int KT>
__device__ __forceinline__ f32x4 decay_tile(f32x4 st, f32x2 dc) {
    return f32x4{st[0] * row_bcast<2 * KT>(dc.x), st[1] * row_bcast<2 * KT>(dc.y),
                 st[2] * row_bcast<2 * KT + 1>(dc.x), st[3] * row_bcast<2 * KT + 1>(dc.y)};
}

// s_waitcnt immediates on gfx9-family parts: vmcnt field (bits 3:0 and
// 15:14) and expcnt (bits 6:4) at their maxima, lgkmcnt (bits 11:8) 0 or 15.
constexpr int WAITCNT_LGKM0 = 0xC07F;
constexpr int WAITCNT_LGKM15 = 0xCF7F;

// Chunk barrier: the wave's LDS accesses are complete, then all waves of
// the work-group meet.  The wait and barrier are one inline asm block whose memory clobber
// keeps every LDS access on its side; as asm, the barrier carries no
// implied wait on the output wave's stores.  The builtin wait after it
// costs nothing (the count is already zero) but tells the compiler so,
// which keeps it from adding conservative waits for LDS reads issued
// before the barrier.
__device__ __forceinline__ void chunk_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_s_waitcnt(WAITCNT_LGKM0);
}

// The copy wave's side of the barrier: no clobber, so the compiler adds no
// wait for its loads in flight.
__device__ __forceinline__ void copy_barrier() { asm volatile("s_barrier"); }

// Fp32 state slice of this lane from `src` ([V, K] if v_first, else
// [K, V]; null: zeros): St[kt][i] = S[v][16*kt + 4*q4 + i].
__device__ __forceinline__ void load_state_from(const float* src, bool v_first, int v, int q4,
                                                f32x4 (&St)[8]) {
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
        St[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (src) {
            const int k0 = 16 * kt + 4 * q4;
            if (v_first) {
                St[kt] = *reinterpret_cast<const f32x4*>(src + (int64_t)v * DK + k0);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) St[kt][i] = src[(int64_t)(k0 + i) * DK + v];
            }
        }
    }
}

__device__ __forceinline__ void store_state_to(float* dst, bool v_first, int v, int q4,
                                               const f32x4 (&St)[8]) {
    if (!dst) return;
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
        const int k0 = 16 * kt + 4 * q4;
        if (v_first) {
            *reinterpret_cast<f32x4*>(dst + (int64_t)v * DK + k0) = St[kt];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[(int64_t)(k0 + i) * DK + v] = St[kt][i];
        }
    }
}

// S^T tiles of this lane: St[kt][i] = S[v][16*kt + 4*q4 + i], v = 16*vt + lane%16.
// (The layout and presence tests are outside the loads, so that all of them
// are in flight before the first wait.)
__device__ __forceinline__ void load_state(const Params& p, int64_t sbase, int v, int q4,
                                           f32x4 (&St)[8]) {
    if (!p.h0) {
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) St[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
    } else if (p.h0_v_first) {
#pragma unroll
        for (int kt = 0; kt < 8; ++kt)
            St[kt] = *reinterpret_cast<const f32x4*>(p.h0 + sbase + (int64_t)v * DK + 16 * kt + 4 * q4);
    } else {
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                St[kt][i] = p.h0[sbase + (int64_t)(16 * kt + 4 * q4 + i) * DK + v];
        }
    }
}

__device__ __forceinline__ void store_state(const Params& p, int64_t sbase, int v, int q4,
                                            const f32x4 (&St)[8]) {
    if (!p.ht) return;
    if (p.ht_v_first) {
#pragma unroll
        for (int kt = 0; kt < 8; ++kt)
            *reinterpret_cast<f32x4*>(p.ht + sbase + (int64_t)v * DK + 16 * kt + 4 * q4) = St[kt];
    } else {
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                p.ht[sbase + (int64_t)(16 * kt + 4 * q4 + i) * DK + v] = St[kt][i];
        }
    }
}

}  // namespace
}  // namespace kda
