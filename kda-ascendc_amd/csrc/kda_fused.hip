// The KDA BT=16 forward in one kernel, for shapes with more (sequence, head)
// pairs than half the CUs (batched and varlen prefill).
//
// The two-stage forward (kda_k1.hip, then kda_k2.hip / kda_k2w.hip) passes
// each chunk's 17 KiB record through HBM: written by stage 1, read back by
// stage 2.  Once the (sequence, head) pairs fill the CUs that round trip is
// most of the forward's traffic (B=16 T=2048 H=32: 3.7 GB moved per forward
// for 1.4 GB of inputs and outputs).  Here one work-group per (sequence,
// value head) keeps the records in LDS:
//   * NP producer waves each form every NP-th chunk's record with stage 1's
//     per-chunk code (k1_compute, kda_k1_chunk.h) straight into their slot of
//     a ring of RING record slots in LDS; each loads its next chunk's q, k
//     and g rows into registers once this chunk's gates are done with, and v
//     straight into the slot;
//   * four compute waves each run the recurrence for two of the head's
//     eight 16-column value tiles (wide_step, kda_k2w_step.h), reading the
//     operands every tile shares from the slot.
// Bound: the issue time of its vector and matrix instructions (an fp32 matrix
// op holds the SIMD's vector unit for all of its 32 cycles, so the grams
// alone are a sixth of it).  Twelve waves, three to a SIMD, so that two
// others issue while one waits: with four producers at two waves per SIMD
// the same work took as long as the waits it could not cover (B=16 T=2048
// H=32: 490 us, and 460 us as it is now; 16 packed sequences in 8192 tokens,
// 173 and 151 us).  The 168 registers of three waves per SIMD are the tight
// side: a few spilled registers in the compute waves' loop cost 30 %.
// The arithmetic is stage 1's and the wide stage 2's, so o and ht are bit
// for bit those of the two-stage forward.
//
// The waves meet through LDS words, never at a barrier after the start
// (a barrier would hold the compute waves' steps to the producers' chunks):
//   full[s]  = c + 1 once chunk c's record is complete in slot s = c % RING
//              (the producer's LDS writes have completed before it stores it);
//   done[s]  counts the compute waves' reads of slot s, NCW per chunk: the
//              producer of chunk c waits for NCW * (c / RING) before writing
//              slot s, that is until chunk c - RING has been read by all.
// Chunk c's producer only waits for reads of chunk c - RING, which needs
// only chunks below c, all produced by then (each producer takes its chunks
// in order), so the waits always end.  Each wait is also bounded (SPIN_LIMIT
// polls) so that a stalled work-group cannot hang the GPU: a bound that runs
// out marks the work-group aborted, after which no wave waits again; the
// work-group drains, its compute waves that had not finished write NaN over
// their o columns and final-state rows, and it adds 1 to a device-wide
// count that the host reads (fused_abort_count).
#include "kda_common.h"
#include "kda_k1_chunk.h"
#include "kda_k2_shared.h"
#include "kda_k2w_step.h"

namespace kda {

namespace {

constexpr int F_NCW = 4;  // compute waves, two value tiles each
constexpr int F_NP = 8;   // producer waves
constexpr int F_RING = 8; // record slots
constexpr int F_THREADS = 64 * (F_NCW + F_NP);
constexpr int SPIN_LIMIT = 1 << 22;
static_assert(F_RING >= F_NP, "every producer can hold a slot");

// The work-group's LDS.
__shared__ __attribute__((aligned(1024))) uint8_t f_ring[F_RING][FREC_BYTES];
__shared__ __attribute__((aligned(16))) float f_L[F_RING][BT * BT];  // the solve's L
__shared__ __attribute__((aligned(16))) float f_bias[DK];  // the head's dt_bias (zeros without it)
__shared__ int f_full[F_RING];
__shared__ int f_done[F_RING];
__shared__ int f_aborted;
__shared__ int f_counted;  // the work-group's give-up has been counted

// Work-groups that gave up a wait on this device since the library was
// loaded or the count was reset (fused_abort_count).
__device__ uint32_t g_aborts;

__device__ __forceinline__ int lds_load(const int* a) {
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
}

// Polls the LDS word `a` until it reaches `target` (bounded; see above).
__device__ __forceinline__ void wait_ge(const int* a, int target) {
    for (int i = 0; i < SPIN_LIMIT; ++i) {
        if (lds_load(a) >= target || lds_load(&f_aborted)) {
            asm volatile("" ::: "memory");
            return;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    __hip_atomic_store(&f_aborted, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    asm volatile("" ::: "memory");
}

// A work-group that gave up a wait has read slots whose chunks it cannot
// vouch for: this compute wave's o columns (its two value tiles) over the
// whole sequence and its final-state rows become NaN.
__device__ __forceinline__ void mark_lost(const Params& p, const SeqSpan& sp, int hv, int ut, int lane,
                                       f32x4 (&SA)[8], f32x4 (&SB)[8]) {
    const float nan = __builtin_nanf("");
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
        SA[kt] = f32x4{nan, nan, nan, nan};
        SB[kt] = SA[kt];
    }
    // the wave's o stores of the chunks have completed before these replace them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const u32x4 nan8 = {0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u, 0x7fc07fc0u};
    uint16_t* base = p.o + (sp.tok0 * p.HV + hv) * DK + 16 * ut + 8 * (lane & 3);
    for (int r = lane >> 2; r < sp.len; r += 16)
        *reinterpret_cast<u32x4*>(base + (int64_t)r * p.HV * DK) = nan8;
}

// The compute waves' side of the LDS flags (wide_step's hooks), and their
// share of stage 1: u of their two tiles, formed from the raw v tiles,
// bf16(A_inv) and beta the producers leave in u's place (FREC_*), with the
// matrix op stage 1 uses (form_u).
struct FlagHooks {
    int s;          // the chunk's slot
    i16x4 v[2], a;  // raw v of the two tiles in T order, bf16(A_inv) as the A operand
    f32x4 beta;     // beta of rows 4*q4 .. +3
    __device__ __forceinline__ void ready(int c) { wait_ge(&f_full[s], c + 1); }
    __device__ __forceinline__ void read_kg(const uint8_t* slot, int lane, u32x4 (&kg)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const u32x2 k0 = __builtin_bit_cast(u32x2, get_T(slot + REC_KG, 2 * j, lane));
            const u32x2 k1 = __builtin_bit_cast(u32x2, get_T(slot + REC_KG, 2 * j + 1, lane));
            kg[j] = u32x4{k0.x, k0.y, k1.x, k1.y};
        }
    }
    __device__ __forceinline__ void read_u(const uint8_t* slot, int lane, int ut) {
        // rows of 32 columns a load; the transposing read (get_T) of tile t's
        // four-column pieces (pair_col)
        typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
        const uint8_t* vs = slot + REC_U + (ut >> 1) * 1024 + (lane >> 2) * 64 + (lane & 3) * 16;
        v[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)vs);
        v[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vs + 8));
        a = *reinterpret_cast<const i16x4*>(slot + FREC_A + lane * 8);
        beta = *reinterpret_cast<const f32x4*>(slot + FREC_BETA + 16 * (lane >> 4));
    }
    __device__ __forceinline__ f32x4 u_start(int t) const {
        const u32x2 w = __builtin_bit_cast(u32x2, v[t]);
        const u32x2 vb = pack4(lo_f(w.x) * beta[0], hi_f(w.x) * beta[1], lo_f(w.y) * beta[2], hi_f(w.y) * beta[3]);
        return unpack_u(form_u(as_i16x4(vb), a));
    }
    __device__ __forceinline__ void consumed() {
        // the slot reads have completed before they are counted
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if ((threadIdx.x & 63) == 0)
            __hip_atomic_fetch_add(&f_done[s], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __device__ __forceinline__ void end() {}
};

// The LDS address of an LDS pointer (wave-uniform).
__device__ __forceinline__ uint32_t lds_addr(const uint8_t* p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_u8*)p);
}

// A raw buffer descriptor over `bytes` bytes from `base`, in SGPRs.
typedef int i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ i32x4 buffer_words(const void* base, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uintptr_t>(base);
    return i32x4{__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                 __builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)),
                 __builtin_amdgcn_readfirstlane((int)bytes), BUF_DWORD3};
}

// One direct buffer->LDS load of 16 bytes a lane (lane l's to LDS address
// lds + 16 l).  Written as inline asm so that the compiler, which cannot
// tell which LDS bytes such a load writes, does not wait for it before every
// later LDS access of the wave; the producer waits for it itself (vmcnt, in
// tail()) before it marks the slot full.  The load takes its LDS address from
// M0, which the block saves and restores (the compiler may hold a value
// there); a wait state separates each M0 write from the next use, as the
// compiler's own direct loads have.
__device__ __forceinline__ void dma16(i32x4 rs, uint32_t lds, uint32_t voff) {
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %2, %3, 0 offen lds\n\t"
        "s_mov_b32 m0, %0\n\t"
        "s_nop 0"
        : "=&s"(saved) : "s"(lds), "v"(voff), "s"(rs) : "memory");
}

// The q, k and g rows and beta of chunk c, in k1_load's layout.  Rows past
// the sequence's end read its last row (in bounds; produce clears them).
template <bool GB16>
__device__ __forceinline__ void load_chunk(const Params& p, int h, int hv, int c, const SeqSpan& sp, int lane,
                                           K1In<GB16, false>& in) {
    // a uniform base and a 32-bit offset per lane, so that the loads hold no
    // 64-bit addresses in vector registers
    const uint32_t r = min(lane & 15, sp.len - 1 - c * BT), q4 = lane >> 4;
    const int64_t tok = sp.tok0 + c * BT;
    const uint32_t qoff = r * (uint32_t)(p.H * DK * 2) + q4 * 8;
    const uint32_t hvoff = r * (uint32_t)p.HV;
    const uint8_t* qb = reinterpret_cast<const uint8_t*>(p.q + (tok * p.H + h) * DK);
    const uint8_t* kb = reinterpret_cast<const uint8_t*>(p.k + (tok * p.H + h) * DK);
    const uint8_t* gb = static_cast<const uint8_t*>(p.g) + (tok * p.HV + hv) * (DK * (GB16 ? 2 : 4));
    const uint8_t* bb = static_cast<const uint8_t*>(p.beta) + (tok * p.HV + hv) * (p.beta_bf16 ? 2 : 4);
    const uint32_t goff = hvoff * (DK * (GB16 ? 2 : 4)) + q4 * (GB16 ? 8 : 16);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) in.q.v[kt] = *reinterpret_cast<const u32x2*>(qb + 32 * kt + qoff);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) in.k.v[kt] = *reinterpret_cast<const u32x2*>(kb + 32 * kt + qoff);
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) {
        if constexpr (GB16) in.g16.v[kt] = *reinterpret_cast<const u32x2*>(gb + 32 * kt + goff);
        else in.g32[kt] = *reinterpret_cast<const f32x4*>(gb + 64 * kt + goff);
    }
    if (p.beta_bf16) in.beta_bits = *reinterpret_cast<const uint16_t*>(bb + hvoff * 2);
    else in.beta_bits = *reinterpret_cast<const uint32_t*>(bb + hvoff * 4);
}

// A producer's side of its ring slot (k1_compute's hooks).
template <bool FULL, bool GB16>
struct ProducerHooks {
    const Params& p;
    const SeqSpan& sp;
    K1In<GB16, false>& in;
    int h, hv, c, lane;
    // Before the slot is written: its previous chunk has been read by every
    // compute wave.  Then the chunk's v rows load straight into it.
    __device__ __forceinline__ void slot() {
        const int s = c % F_RING;
        wait_ge(&f_done[s], F_NCW * (c / F_RING));
        const int64_t row = ((sp.tok0 + c * BT) * p.HV + hv) * DK;
        const uint32_t stride = (uint32_t)p.HV * DK * 2;
        const i32x4 rs = buffer_words(p.v + row, min(BT, sp.len - c * BT) * stride);
        // lane l of load j moves 16 bytes of row l / 4, columns 32*j + 8*(l % 4) .. +7
        const uint32_t dst = lds_addr(f_ring[s] + REC_U);
        const uint32_t off = (lane >> 2) * stride + (lane & 3) * 16;
#pragma unroll
        for (int j = 0; j < 4; ++j) dma16(rs, dst + j * 1024, off + j * 64);
    }
    // q^, k^ and the gates are done with: the next chunk's rows load while
    // the rest of this one is formed.  v has had the gram's time to land.
    __device__ __forceinline__ void tail() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if constexpr (!FULL) {
            // v's rows past the sequence's end, which no load wrote
            if ((lane >> 2) >= sp.len - c * BT) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    *reinterpret_cast<u32x4*>(f_ring[c % F_RING] + REC_U + j * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
            }
        }
        // (past the end: the last chunk again, so that the rows of this one
        // are not held for it)
        load_chunk<GB16>(p, h, hv, min(c + F_NP, sp.nt - 1), sp, lane, in);
    }
};

// One chunk of a producer: stage 1's work on the rows in `in` into the ring
// slot; on return `in` holds the next chunk's rows.
template <bool FULL, bool GB16>
__device__ __forceinline__ void produce(const Params& p, int h, int hv, int c, const SeqSpan& sp, float ea, int lane,
                                        K1In<GB16, false>& in) {
    const int s = c % F_RING;
    if (!FULL && (lane & 15) >= sp.len - c * BT) {
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) in.q.v[kt] = in.k.v[kt] = u32x2{0u, 0u};
        in.beta_bits = 0u;
    }
    uint8_t* rec = f_ring[s];
    // kb's tiles lie in w's bytes, kg's in kg's; the solve's columns where
    // A_inv and beta go after it
    const K1Scratch scr{f_L[s], reinterpret_cast<float*>(rec + FREC_A), rec + REC_W, rec + REC_KG};
    const ProducerHooks<FULL, GB16> hk{p, sp, in, h, hv, c, lane};
    k1_compute<K1_FWD, FULL, GB16, true, true>(p, hv, c, sp, in, f_bias, ea, scr, rec, hk);
    // the record's LDS writes have completed before the slot is marked full
    // (v's rows had landed before tail() went on)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (lane == 0) __hip_atomic_store(&f_full[s], c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Producer wave pw: chunks pw, pw + NP, ... of the sequence, each into its
// slot once the slot's previous chunk has been read by every compute wave.
template <bool GB16>
__device__ __forceinline__ void producer_wave(const Params& p, int pw, int hv, const SeqSpan& sp) {
    const int lane = threadIdx.x & 63;
    const float ea = k1_ea(p, hv);
    if (pw >= sp.nt) return;
    const int h = __builtin_amdgcn_readfirstlane(hv / (p.HV / p.H));  // the q/k head of this value head
    K1In<GB16, false> in;
    load_chunk<GB16>(p, h, hv, pw, sp, lane, in);
    // the full chunks, then the sequence's partial last one
    const int nfull = sp.len / BT;
    int c = pw;
    for (; c < nfull; c += F_NP) produce<true, GB16>(p, h, hv, c, sp, ea, lane, in);
    if (c < sp.nt) produce<false, GB16>(p, h, hv, c, sp, ea, lane, in);
}

// The (sequence or batch row, value head) of work-group wg.  A work-group
// runs as long as its sequence, and work-groups start in id order as CUs
// free up: with cu_seqlens the ids go to the sequences longest first, each
// sequence's heads together, so that the longest chains start at once and the
// short ones fill in around them.  Otherwise the natural order.
__device__ __forceinline__ int fused_pair(const Params& p, int wg) {
    if (!p.cu_seqlens) return wg;
    const int s = wg / p.HV;
    return longest_first(p, s) * p.HV + (wg - s * p.HV);
}

// One work-group per (sequence or batch row, value head).
template <bool GB16>
__global__ __launch_bounds__(F_THREADS) void fused_kernel(Params p) {
    const int lane = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int bh = fused_pair(p, blockIdx.x);
    const int hv = bh - (bh / p.HV) * p.HV;
    const SeqSpan sp = seq_span(p, bh);
    const int64_t sbase = (int64_t)bh * DK * DK;
    const int q4 = lane >> 4;

    if (sp.nt == 0) {
        // an empty sequence: its final state is its initial state (no wave
        // reaches the barrier below)
        if (wave < F_NCW) {
            f32x4 St[8];
            for (int t = 0; t < 2; ++t) {
                const int v = 16 * (2 * wave + t) + (lane & 15);
                load_state(p, sbase, v, q4, St);
                store_state(p, sbase, v, q4, St);
            }
        }
        __builtin_amdgcn_endpgm();
    }
    const int tid = 64 * wave + lane;
    if (tid < F_RING) {
        f_full[tid] = 0;
        f_done[tid] = 0;
    }
    if (tid == 0) {
        f_aborted = 0;
        f_counted = 0;
    }
    if (tid < DK) f_bias[tid] = p.use_gate && p.dt_bias ? p.dt_bias[hv * DK + tid] : 0.f;
    __syncthreads();

    if (wave >= F_NCW) {
        // On the SIMD a producer shares with a compute wave it issues first:
        // one long batch runs the same either way (B=16 T=2048 H=32), 16 packed
        // sequences in 8192 tokens in 150 us against 158 with the compute waves
        // first or neither.
        __builtin_amdgcn_s_setprio(1);
        producer_wave<GB16>(p, wave - F_NCW, hv, sp);
        __builtin_amdgcn_endpgm();
    }
    const int ut = 2 * wave;                // this wave's first value tile
    // this lane's state rows of its two tiles
    const int va = 16 * ut + pair_col(0, lane & 15), vb = 16 * ut + pair_col(1, lane & 15);
    f32x4 SA[8], SB[8];
    load_state(p, sbase, va, q4, SA);
    load_state(p, sbase, vb, q4, SB);
    WideCtx cx;
    cx.scale = p.scale;
    cx.NT = sp.nt;
    cx.T = sp.len;
    cx.lane = lane;
    cx.q4 = q4;
    cx.obase = p.o + (sp.tok0 * p.HV + hv) * DK + 16 * ut + 8 * q4;
    cx.orow_stride = (int64_t)p.HV * DK;
    for (int c = 0; c < cx.NT; ++c) {
        FlagHooks hk;
        hk.s = c % F_RING;
        wide_step(cx, c, SA, SB, f_ring[hk.s], ut, hk);
    }
    // Every give-up is seen here by at least one compute wave: a producer
    // marks the work-group before it publishes the chunk it gave up on, and
    // this wave consumed every chunk; a compute wave sees its own.  The first
    // compute wave to see it counts the work-group, outside every wait loop.
    if (lds_load(&f_aborted)) {
        if (lane == 0 &&
            __hip_atomic_exchange(&f_counted, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0)
            __hip_atomic_fetch_add(&g_aborts, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        mark_lost(p, sp, hv, ut, lane, SA, SB);
    }
    store_state(p, sbase, va, q4, SA);
    store_state(p, sbase, vb, q4, SB);
    __builtin_amdgcn_endpgm();
}

}  // namespace

// Estimated times (us) of a varlen forward on `ncu` CUs, from per-chunk
// costs measured on MI355X (K = V = 128, every in-kernel flag):
//   fused: each work-group takes ~1.85 us per chunk of its sequence, in
//     parallel with the others, so the longest sequence sets the time, or
//     the chunks per CU once the work-groups run in rounds.  (Measured with
//     four producers; with eight 1.55 to 1.8, so near the line the two
//     stages are taken up to 15 % longer than the fused kernel would run.)
//   two stages: stage 1 ~7.5 ns per record slot and value head, stage 2
//     ~0.65 us per step of its longest chain (or of the chunks per CU).
// Measured at 256 (sequence, head) pairs (HV = 32): lengths 16384 + 7 x
// 1024, fused 1580 us and two stages 1019 (estimates 1894 and 1021); 8 x
// 2944, 329 against 544 (340 and 475).
double fused_estimate_us(const Params& p, int ncu) {
    const double chunks = (double)((std::min(p.max_seqlen, p.T) + BT - 1) / BT);
    const double per_cu = (double)p.HV * p.NS / ncu;
    return 1.85 * std::max(chunks, per_cu);
}

double two_stage_estimate_us(const Params& p, int ncu) {
    const double chunks = (double)((std::min(p.max_seqlen, p.T) + BT - 1) / BT);
    const double slots = (double)p.HV * p.NS;
    return 0.0075 * slots + 0.65 * std::max(chunks, slots / ncu);
}

// Whether the forward runs as one fused kernel: never when the
// reference-layout intermediates are asked for (those come from stage 1);
// as the caller asks (force_fused, the reference's use_fused_kernel, or
// two_stage); else, with fixed length, when the (sequence, head) pairs are
// more than half the CUs; with cu_seqlens and the caller's max_seqlen, when
// the fused estimate is at most the two stages'; with cu_seqlens alone,
// when the pairs fill the CUs.
//
// Below the CU count the fused kernel runs every pair in one round of
// work-groups, about 1.6 us per chunk whatever their number, while the two
// stages grow with the pairs (T=4096 forwards, two stages against fused: 80
// pairs 270 against 407 us, 128 pairs 371 against 406, 160 pairs 504 against
// 409, 224 pairs 663 against 420).  With cu_seqlens the fused kernel's time
// follows the longest sequence and stage 1's the total: a single long
// sequence among short ones makes the fused kernel up to about twice slower
// (the figures above).  Without the length of the longest sequence, the pairs
// must fill the CUs.
bool fused_forward(const Params& p, int ncu) {
    if (p.dbg_w || p.dbg_u || p.dbg_Aqk || p.dbg_A_inv || p.dbg_g) return false;
    if (p.force_fused) return true;
    if (p.two_stage) return false;
    const int64_t nbh = (int64_t)(p.cu_seqlens ? p.N : p.B) * p.HV;
    if (!p.cu_seqlens) return 2 * nbh > ncu;
    if (p.max_seqlen > 0) return fused_estimate_us(p, ncu) <= two_stage_estimate_us(p, ncu);
    return nbh >= ncu;
}

hipError_t launch_fused(const Params& p, hipStream_t stream) {
    const int64_t nbh = (int64_t)(p.cu_seqlens ? p.N : p.B) * p.HV;
    auto kern = p.g_bf16 ? fused_kernel<true> : fused_kernel<false>;
    // (a wave a row of the block: a dimension holds at most 2^32 - 1 threads, 5.6
    // M work-groups of 768 in one, which short or empty sequences reach)
    hipLaunchKernelGGL(kern, dim3((unsigned)nbh), dim3(64, F_NCW + F_NP), 0, stream, p);
    return hipGetLastError();
}

hipError_t fused_abort_count(uint32_t* count, bool reset) {
    hipError_t e = hipDeviceSynchronize();
    if (e != hipSuccess) return e;
    e = hipMemcpyFromSymbol(count, HIP_SYMBOL(g_aborts), sizeof(uint32_t), 0, hipMemcpyDeviceToHost);
    if (e != hipSuccess || !reset) return e;
    const uint32_t zero = 0;
    return hipMemcpyToSymbol(HIP_SYMBOL(g_aborts), &zero, sizeof(uint32_t), 0, hipMemcpyHostToDevice);
}

}  // namespace kda
