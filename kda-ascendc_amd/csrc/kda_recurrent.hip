// Token-by-token KDA recurrence in fp32: the decode step (T = 1) and the
// fused-recurrent form of the forward for any T.
//
// Per value head and token t, with S the [V, K] fp32 state:
//   S     = S * alpha_t[None, :]
//   v_new = beta_t * (v_t - S k^_t)
//   S     = S + v_new k^_t^T
//   o_t   = scale * S q^_t
// alpha_t = exp(lb * sigmoid(exp(A_log) * (g_t + dt_bias))) with the in-kernel
// gate; else exp(g_t) when g is the per-token log decay (g_log), else
// 2^(G_t - G_{t-1}) with G the chunk-local log2 cumsum the chunked path takes
// (G_{-1} = 0 at every 16-token chunk start of a sequence).  This is the recurrence the
// chunked path is the WY form of (kernels.py:53-302 computes it chunk-wise);
// the reference's tests use FLA's fused_recurrent_kda for it
// (/root/reference/tests/test_kda_bt16.py:26-38), and its roadmap lists the
// decode step (README.md:503-505).  No rounding happens between tokens, so
// with o in fp32 the kernel is also an on-GPU gold for the chunked path.
//
// Two kernels, which give the same bits.  recurrent_kernel: the decode step, and
// calls of few tokens over many states, where the states' bytes bound the call;
// recurrent_rows_kernel, below: everything else, bound by the latency of the
// tokens (whole_states has the line between them).
//
// recurrent_kernel: one work-group of 256 threads per (batch row or sequence, value head).
// Thread t = 32 * hw + j holds the 64 state elements at memory offsets
// 1024 * i + 4 * t + c (i = 0..15, c = 0..3) of the head's 128 x 128 state,
// so every state load and store is a 16-byte access and each wave
// instruction covers 1 KiB of consecutive memory, in either layout.  What
// those elements are depends on the layout:
//   V-first ([V, K], row v contiguous): S[v = 8i + hw][k = 4j + c].  The
//     products S k^ and S q^ reduce over k across the 32 lanes of a
//     half-wave (hw), which all hold one set of rows.
//   K-first ([K, V]): S[v = 4j + c][k = 8i + hw].  The products reduce
//     over i in registers, then over the eight half-waves: lane pairs of a
//     wave by a shuffle, the four waves through LDS.
// The state lives in registers for the whole sequence (64 floats per
// thread; 106 to 164 VGPRs in all), so three or four work-groups share a CU and the
// decode step streams the states at close to the memory system's rate.
// Grouped value heads (GVA): value head hv reads q/k head hv / (HV / H)
// (kernels.py:88).  Varlen: the work-groups of a (sequence, value head) go over
// the sequence's tokens, with states [N, HV, ...].
#include "kda_common.h"

namespace kda {

namespace {

constexpr int RT = 256;  // threads per work-group

__device__ __forceinline__ float load_scalar(const void* base, int is_bf16, int64_t i) {
    return is_bf16 ? bf2f(static_cast<const uint16_t*>(base)[i])
                   : static_cast<const float*>(base)[i];
}

// Sum over the 32 lanes of a half-wave; every lane receives it: each 16-lane
// row by DPP, then the two rows by one swizzle.  Every lane adds the same
// operands in the same order, so all receive the same bits.
__device__ __forceinline__ float half_sum(float x) {
    x = row_sum16(x);
    return x + xor16(x);
}

__device__ __forceinline__ float sigmoid_precise(float x) { return 1.0f / (1.0f + expf(-x)); }

// The decay alpha of one element of a token, in the three gate modes; gp is
// the element's G_{t-1} of the cumsum form (reset every 16 tokens).
__device__ __forceinline__ float decay_of(const Params& p, float g, float ea, float dtb, float& gp,
                                          bool chunk_start) {
    if (p.use_gate) return expf(p.lower_bound * sigmoid_precise(ea * (g + dtb)));
    if (p.g_log) return expf(g);
    if (chunk_start) gp = 0.0f;
    const float a = exp2f(g - gp);
    gp = g;
    return a;
}

// One token's raw inputs for this thread.  V-first: q, k and g at the
// thread's columns 4j .. 4j+3 and, for threads 0..31, v[4t .. 4t+3] (staged
// for the work-group).  K-first: q, k and g at columns 2l, 2l+1 for the
// lanes l of wave 0 (which form the token's vectors), and v[4j .. 4j+3]
// for every thread.  beta for all.
struct TokRaw {
    u32x2 q, k;
    float g[4];
    float beta;
    u32x2 v;
};

template <bool VFIRST>
__device__ __forceinline__ void load_tok(const Params& p, const SeqSpan& sp, int tt, int h, int hv,
                                         int t, TokRaw& r) {
    const int64_t rq = (sp.tok0 + tt) * p.H + h;
    const int64_t rv = (sp.tok0 + tt) * p.HV + hv;
    const int j = t & 31;
    r.q = r.k = r.v = u32x2{0u, 0u};
#pragma unroll
    for (int c = 0; c < 4; ++c) r.g[c] = 0.f;
    if (VFIRST) {
        const int col = 4 * j;
        r.q = *reinterpret_cast<const u32x2*>(p.q + rq * DK + col);
        r.k = *reinterpret_cast<const u32x2*>(p.k + rq * DK + col);
        if (p.g_bf16) {
            const u32x2 gw =
                *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(p.g) + rv * DK + col);
            r.g[0] = __builtin_bit_cast(float, gw.x << 16);
            r.g[1] = __builtin_bit_cast(float, gw.x & 0xffff0000u);
            r.g[2] = __builtin_bit_cast(float, gw.y << 16);
            r.g[3] = __builtin_bit_cast(float, gw.y & 0xffff0000u);
        } else {
            const f32x4 gv =
                *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.g) + rv * DK + col);
#pragma unroll
            for (int c = 0; c < 4; ++c) r.g[c] = gv[c];
        }
        if (t < 32) r.v = *reinterpret_cast<const u32x2*>(p.v + rv * DK + 4 * t);
    } else {
        if (t < 64) {
            const int col = 2 * t;
            r.q.x = *reinterpret_cast<const uint32_t*>(p.q + rq * DK + col);
            r.k.x = *reinterpret_cast<const uint32_t*>(p.k + rq * DK + col);
            if (p.g_bf16) {
                const uint32_t gw =
                    *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(p.g) + rv * DK + col);
                r.g[0] = __builtin_bit_cast(float, gw << 16);
                r.g[1] = __builtin_bit_cast(float, gw & 0xffff0000u);
            } else {
                const f32x2 gv =
                    *reinterpret_cast<const f32x2*>(static_cast<const float*>(p.g) + rv * DK + col);
                r.g[0] = gv.x;
                r.g[1] = gv.y;
            }
        }
        r.v = *reinterpret_cast<const u32x2*>(p.v + rv * DK + 4 * j);
    }
    r.beta = load_scalar(p.beta, p.beta_bf16, rv);
}

__device__ __forceinline__ void store_o(const Params& p, int64_t idx, float x) {
    if (p.o_fp32) {
        reinterpret_cast<float*>(p.o)[idx] = x;
    } else {
        p.o[idx] = f2bf(x);
    }
}

// ONE: a fixed-length batch of single tokens (the decode step): no token
// loop and no next-token prefetch, which leaves room for four waves per
// SIMD, so the 4 x 256 work-groups a CU holds stream the states in whole
// rounds.
template <bool VFIRST, bool ONE>
__global__ __launch_bounds__(RT) __attribute__((amdgpu_waves_per_eu(ONE ? 4 : 1))) void recurrent_kernel(Params p) {
    const int HV = p.HV, H = p.H;
    const int bhv = blockIdx.x;  // (batch row or sequence) * HV + hv
    const int hv = bhv - (bhv / HV) * HV;
    const int h = hv / (HV / H);
    const SeqSpan sp = seq_span(p, bhv);
    const int t = threadIdx.x;
    const int w = t >> 6, hw = t >> 5, j = t & 31;
    const int64_t sbase = (int64_t)bhv * DK * DK;

    // V-first: the token's v, double-buffered by token parity.
    __shared__ __attribute__((aligned(16))) float s_v[2][DK];
    // K-first: the token's decay, k^ and q^ (formed by wave 0), and the
    // per-wave partial sums of S k^ and S q^.
    __shared__ __attribute__((aligned(16))) float s_vec[3][DK];
    __shared__ __attribute__((aligned(16))) float s_red[2][4][DK];

    f32x4 S[16];
    const float* h0 = p.h0 ? p.h0 + sbase : nullptr;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (h0) S[i] = *reinterpret_cast<const f32x4*>(h0 + 1024 * i + 4 * t);
    }

    const float ea = p.use_gate ? expf(p.A_log[hv]) : 0.0f;
    // V-first: every thread forms its columns 4j .. 4j+3; K-first: wave 0
    // forms columns 2*lane, 2*lane+1 for the work-group.
    const int col = VFIRST ? 4 * j : 2 * (t & 63);
    const bool former = VFIRST || w == 0;
    float dtb[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.use_gate && p.dt_bias && former) {
#pragma unroll
        for (int c = 0; c < (VFIRST ? 4 : 2); ++c) dtb[c] = p.dt_bias[hv * DK + col + c];
    }
    float gp[4] = {0.f, 0.f, 0.f, 0.f};  // G_{t-1} of the cumsum form
    const bool vlane = VFIRST ? t < 32 : true;  // V-first: threads that stage v

    TokRaw cur, nxt;
    const int len = ONE ? 1 : sp.len;
    if (len > 0) load_tok<VFIRST>(p, sp, 0, h, hv, t, cur);
    for (int tt = 0; tt < len; ++tt) {
        if (!ONE && tt + 1 < len) load_tok<VFIRST>(p, sp, tt + 1, h, hv, t, nxt);
        const int64_t rv = (sp.tok0 + tt) * HV + hv;
        const bool chunk_start = (tt % BT) == 0;
        float beta = cur.beta;
        if (p.use_beta_sigmoid) beta = sigmoid_precise(beta);

        if constexpr (VFIRST) {
            // this thread's columns of q^, k^ and the decay
            float qv[4] = {lo_f(cur.q.x), hi_f(cur.q.x), lo_f(cur.q.y), hi_f(cur.q.y)};
            float kv[4] = {lo_f(cur.k.x), hi_f(cur.k.x), lo_f(cur.k.y), hi_f(cur.k.y)};
            if (p.use_l2norm) {
                float sq = 0.f, sk = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    sq = fmaf(qv[c], qv[c], sq);
                    sk = fmaf(kv[c], kv[c], sk);
                }
                const float nq = sqrtf(half_sum(sq) + L2_EPS);
                const float nk = sqrtf(half_sum(sk) + L2_EPS);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    qv[c] /= nq;
                    kv[c] /= nk;
                }
            }
            float a[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) a[c] = decay_of(p, cur.g[c], ea, dtb[c], gp[c], chunk_start);
            float* sv = s_v[tt & 1];
            if (vlane)
                *reinterpret_cast<f32x4*>(sv + 4 * t) =
                    f32x4{lo_f(cur.v.x), hi_f(cur.v.x), lo_f(cur.v.y), hi_f(cur.v.y)};
            __syncthreads();
            float ov = 0.f;  // o of row 8 * j + hw, kept by lane j < 16
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float part = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    S[i][c] *= a[c];
                    part = fmaf(S[i][c], kv[c], part);
                }
                const float pred = half_sum(part);
                const float vnew = beta * (sv[8 * i + hw] - pred);
                float po = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    S[i][c] = fmaf(vnew, kv[c], S[i][c]);
                    po = fmaf(S[i][c], qv[c], po);
                }
                const float o = half_sum(po);
                if (j == i) ov = o;
            }
            if (j < 16) store_o(p, rv * DK + 8 * j + hw, p.scale * ov);
        } else {
            // wave 0 forms the token's decay, k^ and q^ for the work-group
            if (w == 0) {
                float q0 = lo_f(cur.q.x), q1 = hi_f(cur.q.x);
                float k0 = lo_f(cur.k.x), k1 = hi_f(cur.k.x);
                if (p.use_l2norm) {
                    float sq = fmaf(q0, q0, q1 * q1), sk = fmaf(k0, k0, k1 * k1);
                    sq = half_sum(sq);
                    sk = half_sum(sk);
                    sq += __shfl_xor(sq, 32, 64);
                    sk += __shfl_xor(sk, 32, 64);
                    const float nq = sqrtf(sq + L2_EPS), nk = sqrtf(sk + L2_EPS);
                    q0 /= nq; q1 /= nq;
                    k0 /= nk; k1 /= nk;
                }
                const int e = 2 * t;
                s_vec[0][e] = decay_of(p, cur.g[0], ea, dtb[0], gp[0], chunk_start);
                s_vec[0][e + 1] = decay_of(p, cur.g[1], ea, dtb[1], gp[1], chunk_start);
                s_vec[1][e] = k0;
                s_vec[1][e + 1] = k1;
                s_vec[2][e] = q0;
                s_vec[2][e + 1] = q1;
            }
            __syncthreads();
            float kv[16], qv[16];
            float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int k = 8 * i + hw;
                const float a = s_vec[0][k];
                kv[i] = s_vec[1][k];
                qv[i] = s_vec[2][k];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    S[i][c] *= a;
                    part[c] = fmaf(S[i][c], kv[i], part[c]);
                }
            }
            // S k^ over this thread's 16 k, then the two half-waves of the
            // wave, then the four waves
#pragma unroll
            for (int c = 0; c < 4; ++c) part[c] += __shfl_xor(part[c], 32, 64);
            if ((t & 32) == 0)
                *reinterpret_cast<f32x4*>(&s_red[0][w][4 * j]) = f32x4{part[0], part[1], part[2], part[3]};
            __syncthreads();
            const float vv[4] = {lo_f(cur.v.x), hi_f(cur.v.x), lo_f(cur.v.y), hi_f(cur.v.y)};
            float vnew[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int v = 4 * j + c;
                const float pred = s_red[0][0][v] + s_red[0][1][v] + s_red[0][2][v] + s_red[0][3][v];
                vnew[c] = beta * (vv[c] - pred);
            }
            float po[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 16; ++i) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    S[i][c] = fmaf(vnew[c], kv[i], S[i][c]);
                    po[c] = fmaf(S[i][c], qv[i], po[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) po[c] += __shfl_xor(po[c], 32, 64);
            if ((t & 32) == 0)
                *reinterpret_cast<f32x4*>(&s_red[1][w][4 * j]) = f32x4{po[0], po[1], po[2], po[3]};
            __syncthreads();
            if (t < 32) {
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int v = 4 * j + c;
                    const float o = s_red[1][0][v] + s_red[1][1][v] + s_red[1][2][v] + s_red[1][3][v];
                    store_o(p, rv * DK + v, p.scale * o);
                }
            }
        }
        if (!ONE && tt + 1 < len) cur = nxt;
    }

    if (p.ht) {
        float* ht = p.ht + sbase;
#pragma unroll
        for (int i = 0; i < 16; ++i) *reinterpret_cast<f32x4*>(ht + 1024 * i + 4 * t) = S[i];
    }
}

// Several tokens.  The rows of S are independent of each other, so SPLIT
// work-groups share a (sequence, value head) and each of a work-group's SW state
// waves takes 16 rows v: lane (x, g), x = lane % 16, g = lane / 16, holds row
// v = x's 32 elements of column group g, both products of a token are 32 FMAs in
// registers and a sum over the four groups, and no state wave waits for another.
// SF further waves, the formers, take the expf, the divisions and the loads: they
// form the decays, k^, q^, beta and v of the next SF tokens, a token each, in the
// other one of two LDS buffers; one barrier every SF tokens.
//
// Bound by the latency of a token's chain (LDS reads, 32 products, the exchange,
// the update, 32 products), 0.75 us a token where recurrent_kernel's reductions
// across lanes (V-first) or waves (K-first) take 2.1 (K-first) to 3.1 (V-first).
// Four sequences of 24 tokens at 16 heads: 55 -> 21 us K-first, 77 -> 19 V-first;
// with the chip full, 2048 (sequence, head) pairs of 24 tokens: 221 -> 191 and
// 308 -> 179.  Two waves a side instead of four: V-first 244 (the formers are
// late); one former per work-group: 31 and 38 at the small size.
// 104 VGPRs and 48 KB of LDS V-first, 88 and 16 KB K-first: two work-groups a CU.
//
// The column groups and the order of the sums are recurrent_kernel's, so that
// the two, and T decode steps and one call of T tokens, give the same bits:
//   V-first: group g holds k = 32*g .. +31, as eight partial sums of four, added
//     as half_sum adds lanes 8*g .. 8*g + 7, then the groups as it adds the rest;
//   K-first: group g holds k = 8*i + 2*g + {0, 1}, one chain over i each, their
//     sum, then ((g0 + g1) + g2) + g3.
constexpr int SW = 4, SF = 4;
static_assert(16 * SW == 64, "a former's lanes load the work-group's v");
constexpr int SPLIT = DK / (16 * SW);
constexpr int VEC_GROUP = 36;  // floats between column groups in LDS (no bank conflicts)

// The sum over the four column groups, in every lane.
template <bool VFIRST>
__device__ __forceinline__ float group_sum(float r) {
    const auto swap16 = [](float x) {
        const uint32_t b = __builtin_bit_cast(uint32_t, x);
        return __builtin_amdgcn_permlane16_swap(b, b, false, false);
    };
    const auto swap32 = [](uint32_t b) { return __builtin_amdgcn_permlane32_swap(b, b, false, false); };
    const auto f = [](uint32_t b) { return __builtin_bit_cast(float, b); };
    const auto p = swap16(r);  // the groups 0, 0, 2, 2 and 1, 1, 3, 3 of the lane's row
    if constexpr (VFIRST) {
        const auto h = swap32(__builtin_bit_cast(uint32_t, f(p[0]) + f(p[1])));
        return f(h[0]) + f(h[1]);
    } else {
        const auto e = swap32(p[0]), o = swap32(p[1]);
        return f(e[0]) + f(o[0]) + f(e[1]) + f(o[1]);
    }
}

// This lane's part of the product of its 32 elements with a vector.
template <bool VFIRST>
__device__ __forceinline__ float group_part(const f32x4 (&S)[8], const f32x4 (&y)[8]) {
    if constexpr (VFIRST) {
        float q[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            q[m] = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c) q[m] = fmaf(S[m][c], y[m][c], q[m]);
        }
        return ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
    } else {
        float e = 0.f, o = 0.f;  // k even and odd
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            e = fmaf(S[m][0], y[m][0], e);
            o = fmaf(S[m][1], y[m][1], o);
            e = fmaf(S[m][2], y[m][2], e);
            o = fmaf(S[m][3], y[m][3], o);
        }
        return e + o;
    }
}

// A token's raw inputs for a lane of a former.  V-first: q and k at columns
// 4j .. 4j+3, j = lane % 32 (the norms are summed in this order), the rest for
// columns 4j + 2*(lane / 32) + {0, 1}; K-first: columns 2*lane + {0, 1}.  gp: the
// previous token's g, of the cumsum form.
struct FormRaw {
    u32x2 q, k;
    f32x2 g, gp;
    float beta;
    uint16_t v;  // row v0 + lane
};

__device__ __forceinline__ f32x2 load_g2(const Params& p, int64_t at) {
    if (p.g_bf16) {
        const uint32_t w = *reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(p.g) + at);
        return f32x2{lo_f(w), hi_f(w)};
    }
    return *reinterpret_cast<const f32x2*>(static_cast<const float*>(p.g) + at);
}

template <bool VFIRST>
__device__ __forceinline__ void load_form(const Params& p, const SeqSpan& sp, int tt, int h, int hv, int lane,
                                          int col, int v0, FormRaw& r) {
    const int64_t rq = (sp.tok0 + tt) * p.H + h;
    const int64_t rv = (sp.tok0 + tt) * p.HV + hv;
    if constexpr (VFIRST) {
        r.q = *reinterpret_cast<const u32x2*>(p.q + rq * DK + 4 * (lane & 31));
        r.k = *reinterpret_cast<const u32x2*>(p.k + rq * DK + 4 * (lane & 31));
    } else {
        r.q.x = *reinterpret_cast<const uint32_t*>(p.q + rq * DK + col);
        r.k.x = *reinterpret_cast<const uint32_t*>(p.k + rq * DK + col);
    }
    r.g = load_g2(p, rv * DK + col);
    r.gp = f32x2{0.f, 0.f};
    if (!p.use_gate && !p.g_log && tt % BT != 0) r.gp = load_g2(p, (rv - p.HV) * DK + col);
    r.beta = load_scalar(p.beta, p.beta_bf16, rv);
    r.v = p.v[rv * DK + v0 + lane];
}

// A vector's two columns of the lane, divided by its norm.
template <bool VFIRST>
__device__ __forceinline__ f32x2 unit2(const Params& p, u32x2 w, int lane) {
    f32x2 y;
    if constexpr (VFIRST) {
        const uint32_t mine = lane < 32 ? w.x : w.y;
        y = f32x2{lo_f(mine), hi_f(mine)};
    } else {
        y = f32x2{lo_f(w.x), hi_f(w.x)};
    }
    if (!p.use_l2norm) return y;
    float ss;
    if constexpr (VFIRST) {
        const float c[4] = {lo_f(w.x), hi_f(w.x), lo_f(w.y), hi_f(w.y)};
        ss = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) ss = fmaf(c[i], c[i], ss);
        ss = half_sum(ss);
    } else {
        ss = half_sum(fmaf(y.x, y.x, y.y * y.y));
        ss += __shfl_xor(ss, 32, 64);
    }
    const float n = sqrtf(ss + L2_EPS);
    return f32x2{y.x / n, y.y / n};
}

template <bool VFIRST>
__global__ __launch_bounds__(64 * (SW + SF)) void recurrent_rows_kernel(Params p) {
    const int HV = p.HV;
    const int bhv = blockIdx.x / SPLIT;  // (batch row or sequence) * HV + hv
    const int hv = bhv - (bhv / HV) * HV;
    const SeqSpan sp = seq_span(p, bhv);
    const int lane = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
    const int len = sp.len;

    // The vectors of two times SF tokens: decay, k^, q^, each as four groups of
    // 32, and beta.
    __shared__ __attribute__((aligned(16))) float s_vec[2][SF][3][4 * VEC_GROUP];
    __shared__ float s_beta[2][SF], s_v[2][SF][16 * SW];
    // V-first: a wave's 16 rows on their way between memory, which is read and
    // written in whole KiB, and the lanes; unit u (16 bytes) of row r at u ^ r.
    __shared__ __attribute__((aligned(16))) float s_rows[VFIRST ? SW : 1][VFIRST ? 16 * DK : 4];

    const int v0 = (blockIdx.x % SPLIT) * 16 * SW;  // the work-group's rows
    if (wave >= SW) {
        const int f = wave - SW;
        const int h = hv / (HV / p.H);
        const float ea = p.use_gate ? expf(p.A_log[hv]) : 0.0f;
        const int j = lane & 31;
        const int col = VFIRST ? 4 * j + 2 * (lane >> 5) : 2 * lane;
        const int at = VFIRST ? (j >> 3) * VEC_GROUP + (col & 31) : (lane & 3) * VEC_GROUP + 2 * (lane >> 2);
        f32x2 dtb = {0.f, 0.f};
        if (p.use_gate && p.dt_bias) dtb = f32x2{p.dt_bias[hv * DK + col], p.dt_bias[hv * DK + col + 1]};
        FormRaw cur, nxt;
        if (len > 0) load_form<VFIRST>(p, sp, min(f, len - 1), h, hv, lane, col, v0, cur);
        for (int t0 = 0; t0 < len; t0 += SF) {
            // (past the end the last token again: it is formed and not read)
            load_form<VFIRST>(p, sp, min(t0 + SF + f, len - 1), h, hv, lane, col, v0, nxt);
            const int buf = (t0 / SF) & 1;
            float (*vec)[4 * VEC_GROUP] = s_vec[buf][f];
            f32x2 a;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                float gp = cur.gp[c];
                a[c] = decay_of(p, cur.g[c], ea, dtb[c], gp, false);
            }
            *reinterpret_cast<f32x2*>(&vec[0][at]) = a;
            *reinterpret_cast<f32x2*>(&vec[1][at]) = unit2<VFIRST>(p, cur.k, lane);
            *reinterpret_cast<f32x2*>(&vec[2][at]) = unit2<VFIRST>(p, cur.q, lane);
            if (lane == 0) s_beta[buf][f] = p.use_beta_sigmoid ? sigmoid_precise(cur.beta) : cur.beta;
            s_v[buf][f][lane] = bf2f(cur.v);
            // tokens t0 .. t0 + SF - 1 are formed, and those before them, whose
            // buffer the next ones take, have been read
            __syncthreads();
            cur = nxt;
        }
        return;
    }

    const int x = lane & 15, g = lane >> 4;
    const int v = v0 + 16 * wave + x;
    const int64_t sbase = (int64_t)bhv * DK * DK;
    // V-first: the wave's rows, lane by lane in order of memory, and the lane's
    // element 4*m, k = 32*g + 4*m; K-first element 2*i + e: k = 8*i + 2*g + e
    float* rows = s_rows[VFIRST ? wave : 0];
    const int half = lane >> 5;
    int unit = lane & 31, xs = x;
    auto linear = [&](int m) { return rows + (2 * m + half) * DK + 4 * (unit ^ (2 * m + half)); };
    auto mine = [&](int m) { return rows + xs * DK + 4 * ((8 * g + m) ^ xs); };
    const int64_t slab = sbase + (int64_t)(v - x) * DK + 4 * lane;
    auto element = [&](int n) { return sbase + (8 * (n >> 1) + 2 * g + (n & 1)) * DK + v; };
    f32x4 S[8] = {};
    if (p.h0) {
        if constexpr (VFIRST) {
#pragma unroll
            for (int m = 0; m < 8; ++m) S[m] = *reinterpret_cast<const f32x4*>(p.h0 + slab + 256 * m);
#pragma unroll
            for (int m = 0; m < 8; ++m) *reinterpret_cast<f32x4*>(linear(m)) = S[m];
            wave_lds_fence();
#pragma unroll
            for (int m = 0; m < 8; ++m) S[m] = *reinterpret_cast<const f32x4*>(mine(m));
        } else {
#pragma unroll
            for (int n = 0; n < 32; ++n) S[n >> 2][n & 3] = p.h0[element(n)];
        }
    }
    const int64_t row0 = sp.tok0 * HV + hv;
    for (int t0 = 0; t0 < len; t0 += SF) {
        __syncthreads();  // tokens t0 .. t0 + SF - 1 are formed
        const int buf = (t0 / SF) & 1, n = min(SF, len - t0);
#pragma unroll 1
        for (int f = 0; f < n; ++f) {
            const float (*vec)[4 * VEC_GROUP] = s_vec[buf][f];
            f32x4 kv[8], qv[8];
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const f32x4 a = *reinterpret_cast<const f32x4*>(&vec[0][g * VEC_GROUP + 4 * m]);
                kv[m] = *reinterpret_cast<const f32x4*>(&vec[1][g * VEC_GROUP + 4 * m]);
                S[m] = S[m] * a;
            }
            const float pred = group_sum<VFIRST>(group_part<VFIRST>(S, kv));
#pragma unroll
            for (int m = 0; m < 8; ++m) qv[m] = *reinterpret_cast<const f32x4*>(&vec[2][g * VEC_GROUP + 4 * m]);
            const float vnew = s_beta[buf][f] * (s_v[buf][f][16 * wave + x] - pred);
#pragma unroll
            for (int m = 0; m < 8; ++m) {
#pragma unroll
                for (int c = 0; c < 4; ++c) S[m][c] = fmaf(vnew, kv[m][c], S[m][c]);
            }
            const float o = group_sum<VFIRST>(group_part<VFIRST>(S, qv));
            if (g == 0) store_o(p, (row0 + (int64_t)(t0 + f) * HV) * DK + v, p.scale * o);
        }
    }
    if (p.ht) {
        asm("" : "+v"(unit), "+v"(xs));  // (their addresses are formed again, not kept through the loop)
        if constexpr (VFIRST) {
#pragma unroll
            for (int m = 0; m < 8; ++m) *reinterpret_cast<f32x4*>(mine(m)) = S[m];
            wave_lds_fence();
#pragma unroll
            for (int m = 0; m < 8; ++m)
                *reinterpret_cast<f32x4*>(p.ht + slab + 256 * m) = *reinterpret_cast<const f32x4*>(linear(m));
        } else {
#pragma unroll
            for (int n = 0; n < 32; ++n) p.ht[element(n)] = S[n >> 2][n & 3];
        }
    }
}

}  // namespace

// Whether recurrent_kernel takes a call of `tokens` tokens a pair, one token of
// batch rows apart (that is always its).  Its three work-groups a CU hold 768
// pairs at a time, with all of their states' bytes in flight; the two of
// recurrent_rows_kernel hold 256, for a quarter to a third of the time a token.
// So few tokens and full rounds are the former's.  Us, recurrent_kernel against
// recurrent_rows_kernel (packed sequences; batch rows are within 3 % of them):
//   V-first: 1 token, 256 pairs 10.4 / 8.6, 288 10.7 / 11.7, 768 18.4 / 24.7,
//     4096 108 / 127; 2 tokens, 288 14.3 / 13.1, 384 15.2 / 15.9, 768 22.4 /
//     26.9, 4096 120 / 139; 3 tokens, 640 25.4 / 25.6, 768 26.9 / 28.6, 960
//     36.0 / 34.8, 2048 64.2 / 66.4, 4096 130 / 146; 4 tokens, 2560 98.3 /
//     97.2, 3072 114 / 119; 5 tokens, 6144 241 / 241;
//   K-first: 1 token, 256 9.5 / 8.5, 288 9.7 / 11.5, 4096 105 / 122; 2 tokens,
//     768 20.4 / 24.0, 1792 46.8 / 44.2, 2048 51.7 / 54.8, 4096 120 / 122; 3
//     tokens, 768 22.9 / 25.8, 1024 33.9 / 30.9; 5 tokens (the rows' second
//     batch), 640 25.8 / 30.1, 1024 43.1 / 41.4, 2048 73.1 / 80.7, 8192 274 /
//     320; 6 tokens, 640 29.3 / 30.4, 1024 47.6 / 42.2, 6144 228 / 238; 8
//     tokens, 640 34.8 / 31.3, 768 35.8 / 36.8.
static bool whole_states(bool v_first, int64_t pairs, int64_t tokens) {
    constexpr int64_t ROUND = 768;
    if (pairs <= 256 || tokens > 8) return false;
    if (tokens <= 2) return tokens == 1 || pairs > 320;
    const bool thin = pairs > ROUND && pairs <= 1024;  // a second round with little in it
    if (v_first) return tokens == 3 ? pairs > 640 && !thin : tokens == 4 && pairs > 2816;
    if (pairs <= ROUND) return pairs > (tokens == 5 ? 512 : tokens <= 6 ? 576 : 672);
    return tokens == 5 ? !thin : tokens == 6 && pairs > 4096;
}

hipError_t launch_recurrent(const Params& p, hipStream_t stream) {
    const int64_t nseq = p.cu_seqlens ? p.N : p.B;
    const int64_t pairs = nseq * p.HV;
    // Packed sequences' lengths are on the device.  Where the tokens are a
    // multiple of the sequences they are taken as equal, as a decode step's or
    // a draft's are; else there may be a long one among them, for which
    // recurrent_kernel takes up to four times as long a token.
    const bool equal = !p.cu_seqlens || p.T % p.N == 0;
    const int64_t tokens = p.cu_seqlens ? p.T / p.N : p.T;
    const bool one = !p.cu_seqlens && p.T == 1;
    if (!one && !(equal && whole_states(p.h0_v_first, pairs, tokens))) {
        auto rows = p.h0_v_first ? recurrent_rows_kernel<true> : recurrent_rows_kernel<false>;
        // (a wave a row of the block: a dimension holds at most 2^32 - 1 threads,
        // 8.4 M work-groups of 512 in one, which empty sequences reach)
        hipLaunchKernelGGL(rows, dim3((unsigned)(pairs * SPLIT)), dim3(64, SW + SF), 0, stream, p);
        return hipGetLastError();
    }
    auto kern = p.h0_v_first ? (one ? recurrent_kernel<true, true> : recurrent_kernel<true, false>)
                             : (one ? recurrent_kernel<false, true> : recurrent_kernel<false, false>);
    hipLaunchKernelGGL(kern, dim3((unsigned)pairs), dim3(RT), 0, stream, p);
    return hipGetLastError();
}

}  // namespace kda
