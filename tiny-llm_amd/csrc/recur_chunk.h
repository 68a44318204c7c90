// Linear recurrences over prompts in chunks of 64 tokens, on the float32 matrix pipe (v_mfma_f32_16x16x4_f32: full float32 products and sums).
//
//   KIND 0, gated delta rule:   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q      (q, k unit vectors, q also * dim^-1/2)
//   KIND 1, decay per head:     S <- a S + b k v^T;               o = S^T q
//   KIND 2, decay per channel:  S <- diag(a) S + k v^T;           o = S^T q
//
// Token by token (delta_kernel / linrec_kernel of hybrid_kernels.h) a prompt is one dependent chain of 0.2-0.27 us per token, whatever its width: 555 us
// for 2,048 tokens of the delta rule with 16 heads of 128 x 128, 392-407 us (1,900 tokens) for the other two.  In chunks: 36 + 103 us, and 24 + 59 / 54 + 60 us.
// What bounds the scan then is a chunk's chain (two products, an exchange through LDS, 1.6 us of matrix instructions of 3.2 us a chunk), half the CUs busy.  Within a chunk with decays g, R(t, i) = g_{i+1} ... g_t and
// G_t = g_0 ... g_t the recurrence is
//   U  = T (beta v) - T (beta G k) S0,   T = (I + A)^-1,  A(t, i) = beta_t R(t, i) k_t.k_i for i < t     (KIND 0;  U = v, S0 not needed, for the others)
//   O  = (G q) S0 + P U,                 P(t, i) = R(t, i) q_t.k_i (* b_i) for i <= t
//   S' = G_63 S0 + sum_i R(63, i) (b_i) k_i u_i^T
// so all that waits for the previous chunk are the three products with S0 (with U behind the first).  Two kernels:
//   chunk_prep_kernel  (head, sequence, chunk): everything that does not need S0, all chunks at once; leaves its operands in the workspace
//   chunk_scan_kernel  (head, sequence, 16 state columns): walks the chunks with its columns of the state in registers
// The products of decays are formed by multiplying, as the token loop does (no logarithms, no quotients: a decay may be 0).  Every operand of the scan lies
// in the workspace in the order in which the matrix instruction's lanes want it: a 16 x 16 block is 64 lanes x 4 floats, 1 KB, one 16-byte load a lane.
//   "A order" of a block M[rows][cols]: lane l, element e = M[l % 16][4 (l / 16) + e];  "D order": lane l, element e = M[4 (l / 16) + e][l % 16].
//   A product's result comes in D order, and D order is what the instruction wants of a second operand whose inner index runs over the rows: results chain.
#pragma once

#include "common.h"

namespace tl {
namespace hy {

__device__ __forceinline__ f32x4 mfma_f32_block(const f32x4 &a, const f32x4 &b, f32x4 c) {  // c += A (A order, 16 x 16) . B (D order, 16 x 16)
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
    return c;
}

constexpr int CHUNK = 64;

struct ChunkArgs {
    const float *src;                   // q | k | v rows of ld floats: q at q0 + (h / group) dim, k at k0 + (h / group) dim, v at v0 + h vdim
    int ld, q0, k0, v0, group;
    const int32_t *seq_row0, *seq_slot;
    float *ws, *state, *obuf;           // obuf [rows, H, vdim + ones]
    int H, vdim, ones;                  // ones: a column of the value 1 behind the values
    // KIND 0
    const float *gate_src;              // columns a0 + h (decay input) and b0 + h (beta input) of rows of ldg floats
    int ldg, a0, b0;
    const float *a_log, *dt_bias;
    float unit_eps;
    // KIND 1: gates [rows, H, 3] = (a, b, ..), or with fixed a constant decay per head and b = 1;  silu: bit 0 q and k, bit 1 v;  k_mul: factor on k
    const float *gates, *fixed;
    int silu;
    float k_mul;
    // KIND 2: decay [rows, H, dim]
    const float *decay;
};

// Floats of one (head, chunk) in the workspace: W, Q, K' (64 x dim each), P (64 x 64), U (64 x 16 VT), the chunk's whole decay (dim)
struct ChunkLayout {
    int w, q, k, p, u, g, total;
    __host__ __device__ ChunkLayout(int dim, int vt) {
        w = 0, q = w + CHUNK * dim, k = q + CHUNK * dim, p = k + CHUNK * dim, u = p + CHUNK * CHUNK, g = u + vt * 16 * CHUNK, total = g + dim;
    }
};
// the slot of a sequence's chunk: sequences start at ascending rows, so floor(row0 / 64) + sequence + chunk is taken once
__device__ __forceinline__ float *chunk_slot(const ChunkArgs &a, const ChunkLayout &lay, int h, int s, int r0, int c) {
    return a.ws + ((size_t)(r0 / CHUNK + s + c) * a.H + h) * lay.total;
}

template <int KIND, int DT>
__global__ __launch_bounds__(256) void chunk_prep_kernel(ChunkArgs a) {
    constexpr int D = 16 * DT, RS = CHUNK + 4;  // (rows of the decay products are 16-byte aligned and four banks apart)
    __shared__ f32x4 kf[4 * DT * 64];                                   // the chunk's keys, [row block][16 columns] in A order
    __shared__ __attribute__((aligned(16))) float ratio[KIND == 2 ? 4 : CHUNK * RS];                 // R(t, i), 0 for i > t
    __shared__ f32x4 af[KIND == 0 ? 16 * 64 : 1], tf[KIND == 0 ? 4 * 64 : 1], tr[KIND == 0 ? 4 * 64 : 1];  // -A [t block][i block], the inverses of its diagonal blocks, a transposition's scratch
    __shared__ __attribute__((aligned(16))) float gs[CHUNK], bs[CHUNK];
    // KIND 2: decays, and their products inside a 16-token block: up to and with t, behind t; the blocks' whole products
    __shared__ __attribute__((aligned(16))) float al[KIND == 2 ? CHUNK * (D + 4) : 1], blk[KIND == 2 ? 4 * D : 1];
    __shared__ f32x4 qf[KIND == 2 ? 4 * DT * 64 : 1];
    const int h = blockIdx.x, s = blockIdx.y, c = blockIdx.z;
    const int r0 = a.seq_row0[s], n = a.seq_row0[s + 1] - r0;
    if (c * CHUNK >= n) return;
    const int nt = min(CHUNK, n - c * CHUNK), tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64, g = lane / 16, lr = lane % 16;
    const int VE = a.vdim + a.ones, VT = (VE + 15) / 16, kh = h / a.group;
    const ChunkLayout lay(D, VT);
    float *ws = chunk_slot(a, lay, h, s, r0, c);
    const float *row0 = a.src + (size_t)(r0 + c * CHUNK) * a.ld;
    const int t = 16 * w + lr;  // the token whose q and k this lane holds a part of
    const bool live = t < nt;

    f32x4 q[DT], k[DT];
    {
        const float *qp = row0 + (size_t)(live ? t : 0) * a.ld + a.q0 + (size_t)kh * D + 4 * g, *kp = qp - a.q0 + a.k0;
#pragma unroll
        for (int j = 0; j < DT; ++j) {
            q[j] = *reinterpret_cast<const f32x4 *>(qp + 16 * j), k[j] = *reinterpret_cast<const f32x4 *>(kp + 16 * j);
            if (!live) q[j] = k[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (tid < CHUNK) {  // padding behind the prompt's end: decay 1, no input
        const bool in = tid < nt;
        const size_t row = (size_t)(r0 + c * CHUNK + (in ? tid : 0));
        float gv = 1.f, bv = 0.f;
        if constexpr (KIND == 0) {
            const float *p = a.gate_src + row * a.ldg;
            gv = expf(-expf(a.a_log[h]) * softplus_f(p[a.a0 + h] + a.dt_bias[h]));
            bv = sigmoid_f(p[a.b0 + h]);
        } else if constexpr (KIND == 1) {
            const float *p = a.gates + (row * a.H + h) * 3;
            gv = a.fixed ? a.fixed[h] : p[0];
            bv = a.fixed ? 1.f : p[1];
        }
        gs[tid] = in ? gv : 1.f;
        bs[tid] = in ? bv : 0.f;
    }
    if constexpr (KIND == 2) {
        for (int i = tid; i < CHUNK * D; i += 256) {
            const int tt = i / D, d = i % D;
            al[tt * (D + 4) + d] = tt < nt ? a.decay[((size_t)(r0 + c * CHUNK + tt) * a.H + h) * D + d] : 1.f;
        }
    }
    if constexpr (KIND == 0) {  // unit vectors
        float sq = 0.f, sk = 0.f;
#pragma unroll
        for (int j = 0; j < DT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) sq += q[j][e] * q[j][e], sk += k[j][e] * k[j][e];
        sq += lane_xor16(sq, lane), sk += lane_xor16(sk, lane);
        sq += lane_xor32(sq, lane), sk += lane_xor32(sk, lane);
        const float iq = 1.f / sqrtf((float)D) / sqrtf(sq + a.unit_eps), ik = 1.f / sqrtf(sk + a.unit_eps);
#pragma unroll
        for (int j = 0; j < DT; ++j) q[j] *= iq, k[j] *= ik;
    } else if constexpr (KIND == 1) {
#pragma unroll
        for (int j = 0; j < DT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (a.silu & 1) q[j][e] = silu_hw(q[j][e]), k[j][e] = silu_hw(k[j][e]);
                k[j][e] *= a.k_mul;
            }
    }
#pragma unroll
    for (int j = 0; j < DT; ++j) {
        kf[(w * DT + j) * 64 + lane] = k[j];
        if constexpr (KIND == 2) qf[(w * DT + j) * 64 + lane] = q[j];
    }
    __syncthreads();

    f32x4 *wq = reinterpret_cast<f32x4 *>(ws + lay.q), *wp = reinterpret_cast<f32x4 *>(ws + lay.p), *wk = reinterpret_cast<f32x4 *>(ws + lay.k);
    f32x4 *ww = reinterpret_cast<f32x4 *>(ws + lay.w), *wu = reinterpret_cast<f32x4 *>(ws + lay.u);
    if constexpr (KIND != 2) {
        if (w == 0) {  // a lane per column i: R(t, i) down the tokens
            float r = 0.f;
#pragma unroll 8
            for (int tt = 0; tt < CHUNK; ++tt) {
                r = tt < lane ? 0.f : (tt == lane ? 1.f : r * gs[tt]);
                ratio[tt * RS + lane] = r;
            }
        }
        __syncthreads();
        const float gam = ratio[t * RS] * gs[0];  // G_t
#pragma unroll
        for (int j = 0; j < DT; ++j) wq[(w * DT + j) * 64 + lane] = q[j] * gam;
        if (tid < D) ws[lay.g + tid] = ratio[(CHUNK - 1) * RS] * gs[0];
        // rows t of the wave's block against the keys of blocks 0 .. w: (k_i . q_t) comes with i = 4 g + e and t = l % 16, which is A order of [t][i]
        for (int b = 0; b <= w; ++b) {
            f32x4 pq{0.f, 0.f, 0.f, 0.f}, pk{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                const f32x4 kb = kf[(b * DT + j) * 64 + lane];
                pq = mfma_f32_block(kb, q[j], pq);
                if constexpr (KIND == 0) pk = mfma_f32_block(kb, k[j], pk);
            }
            const f32x4 r = *reinterpret_cast<const f32x4 *>(&ratio[t * RS + 16 * b + 4 * g]);
            pq *= r;
            if constexpr (KIND == 1) pq *= *reinterpret_cast<const f32x4 *>(&bs[16 * b + 4 * g]);
            wp[(w * 4 + b) * 64 + lane] = pq;
            if constexpr (KIND == 0) {
                pk *= r * -bs[t];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (16 * b + 4 * g + e >= t) pk[e] = 0.f;
                af[(w * 4 + b) * 64 + lane] = pk;
            }
        }
        if constexpr (KIND == 0) {  // (I + A)^-1 of the wave's diagonal block: a lane per column, forward substitution
            f32x4 *own = &af[(w * 4 + w) * 64];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            float x[16];
#pragma unroll
            for (int tt = 0; tt < 16; ++tt) {
                float v = tt == lr ? 1.f : 0.f;
#pragma unroll
                for (int i4 = 0; 4 * i4 < tt; ++i4) {
                    const f32x4 m = own[tt + 16 * i4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * i4 + e < tt) v += m[e] * x[4 * i4 + e];
                }
                x[tt] = v;
            }
            if (g == 0) {
#pragma unroll
                for (int tt = 0; tt < 16; ++tt) reinterpret_cast<float *>(&tf[w * 64 + tt + 16 * (lr / 4)])[lr % 4] = x[tt];
            }
            __syncthreads();
        }
    } else {
        // products of decays inside the 16-token blocks, a thread per channel and two blocks; blk = a block's whole product
        for (int i = tid; i < 4 * D; i += 256) {
            const int b = i / D, d = i % D;
            float r = 1.f;
#pragma unroll
            for (int tt = 0; tt < 16; ++tt) r *= al[(16 * b + tt) * (D + 4) + d];
            blk[b * D + d] = r;
        }
        __syncthreads();
        if (tid < D) ws[lay.g + tid] = blk[tid] * blk[D + tid] * blk[2 * D + tid] * blk[3 * D + tid];
        // the products up to (and with) the lane's token, and behind it
        f32x4 up[DT], behind[DT];
        bool wide = true;
#pragma unroll
        for (int j = 0; j < DT; ++j) {
            up[j] = behind[j] = f32x4{1.f, 1.f, 1.f, 1.f};
#pragma unroll
            for (int tt = 0; tt < 16; ++tt) {
                const f32x4 m = *reinterpret_cast<const f32x4 *>(&al[(16 * w + tt) * (D + 4) + 16 * j + 4 * g]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    up[j][e] *= tt <= lr ? m[e] : 1.f;
                    behind[j][e] *= tt > lr ? m[e] : 1.f;
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) wide = wide && up[j][e] * behind[j][e] > 1e-30f;
        }
        // Inside the wave's block: R(t, i) is the quotient of two of these products where the block's whole product is far above the smallest float (every
        // term keeps its relative precision: one product); otherwise one by one.
        if (__all(wide)) {
            f32x4 p{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < DT; ++j) p = mfma_f32_block(k[j] / up[j], q[j] * up[j], p);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * g + e > lr) p[e] = 0.f;
            wp[(w * 4 + w) * 64 + lane] = p;
        } else {  // lane (i = l % 16, a quarter of the channels g): P(t, i) = sum_d q_t k_i a_{i+1} ... a_t
            float acc[16];
#pragma unroll
            for (int tt = 0; tt < 16; ++tt) acc[tt] = 0.f;
            for (int dd = 0; dd < D / 16; ++dd) {
                const int d = (D / 4) * g + 4 * dd, at = (w * DT + d / 16) * 64 + 16 * ((d % 16) / 4);
                const f32x4 ki = kf[at + lr];
                f32x4 r{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int tt = 0; tt < 16; ++tt) {
                    const f32x4 m = *reinterpret_cast<const f32x4 *>(&al[(16 * w + tt) * (D + 4) + d]), qv = qf[at + tt];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        r[e] = tt < lr ? 0.f : (tt == lr ? ki[e] : r[e] * m[e]);
                        acc[tt] += r[e] * qv[e];
                    }
                }
            }
            float *pt = reinterpret_cast<float *>(wp + (w * 4 + w) * 64);
#pragma unroll
            for (int tt = 0; tt < 16; ++tt) {
                float v = acc[tt];
                v += lane_xor16(v, lane);
                v += lane_xor32(v, lane);
                if (g == 0) pt[(tt + 16 * (lr / 4)) * 4 + lr % 4] = v;  // A order of [t][i]
            }
        }
#pragma unroll
        for (int j = 0; j < DT; ++j) q[j] *= up[j], k[j] *= behind[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < DT; ++j) kf[(w * DT + j) * 64 + lane] = k[j];  // from here on: keys carried to their block's end
        __syncthreads();
        for (int b = w - 1; b >= 0; --b) {  // q moves back a block at a time: from its block's start to the end of block b
            f32x4 p{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < DT; ++j) {
                p = mfma_f32_block(kf[(b * DT + j) * 64 + lane], q[j], p);
                q[j] *= *reinterpret_cast<const f32x4 *>(&blk[b * D + 16 * j + 4 * g]);
            }
            wp[(w * 4 + b) * 64 + lane] = p;
        }
#pragma unroll
        for (int j = 0; j < DT; ++j) wq[(w * DT + j) * 64 + lane] = q[j];
    }

    // Columns: the keys (K' for the state's update, and T (beta G k)), then the values.  The blocks of a column chain through the inverse block by block.
    auto solve = [&](f32x4 (&x)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            f32x4 acc = x[b];
#pragma unroll
            for (int i = 0; i < b; ++i) acc = mfma_f32_block(af[(b * 4 + i) * 64 + lane], x[i], acc);
            x[b] = mfma_f32_block(tf[b * 64 + lane], acc, f32x4{0.f, 0.f, 0.f, 0.f});
        }
    };
    for (int j = w; j < DT; j += 4) {
        f32x4 x[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            f32x4 kt;
#pragma unroll
            for (int e = 0; e < 4; ++e) kt[e] = reinterpret_cast<const float *>(&kf[(b * DT + j) * 64 + 4 * g + e + 16 * (lr / 4)])[lr % 4];
            if constexpr (KIND == 2) {
                f32x4 m = kt;
                for (int i = b + 1; i < 4; ++i) m *= blk[i * D + 16 * j + lr];
                wk[(j * 4 + b) * 64 + lane] = m;
            } else {
                const f32x4 last = *reinterpret_cast<const f32x4 *>(&ratio[(CHUNK - 1) * RS + 16 * b + 4 * g]), be = *reinterpret_cast<const f32x4 *>(&bs[16 * b + 4 * g]);
                wk[(j * 4 + b) * 64 + lane] = KIND == 1 ? kt * last * be : kt * last;
                if constexpr (KIND == 0) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[b][e] = kt[e] * (be[e] * (ratio[(16 * b + 4 * g + e) * RS] * gs[0]));
                }
            }
        }
        if constexpr (KIND == 0) {
            solve(x);
#pragma unroll
            for (int b = 0; b < 4; ++b) {  // to A order, through the wave's own kilobyte
                f32x4 *scr = &tr[w * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e) reinterpret_cast<float *>(&scr[4 * g + e + 16 * (lr / 4)])[lr % 4] = -x[b][e];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                ww[(b * DT + j) * 64 + lane] = scr[lane];
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
        }
    }
    for (int ct = w; ct < VT; ct += 4) {
        const int col = 16 * ct + lr;
        f32x4 x[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int tt = 16 * b + 4 * g + e;
                float v = 0.f;
                if (tt < nt && col < VE) v = col < a.vdim ? row0[(size_t)tt * a.ld + a.v0 + (size_t)h * a.vdim + col] : 1.f;
                if (KIND == 1 && (a.silu & 2) && col < a.vdim) v = silu_hw(v);
                x[b][e] = KIND == 0 ? v * bs[tt] : v;
            }
        }
        if constexpr (KIND == 0) solve(x);
#pragma unroll
        for (int b = 0; b < 4; ++b) wu[(ct * 4 + b) * 64 + lane] = x[b];
    }
}

// grid (heads, sequences, column blocks of 16), 256 threads: wave w holds the state's key rows of blocks w, w + 4, .. for the 16 columns, in registers in D
// order.  Per chunk it forms its share of W S and Q S for all 64 tokens; the shares meet in LDS (two buffers: one barrier a chunk); then every wave has U,
// updates its own rows of the state and reads out its own 16 tokens.  A chunk's operands are on their way while the previous one is worked on.
template <int KIND, int DT>
__global__ __launch_bounds__(256, 1) void chunk_scan_kernel(ChunkArgs a) {
    constexpr int D = 16 * DT, TPW = DT / 4;
    __shared__ f32x4 part[2][4][KIND == 0 ? 8 : 4][64];
    const int h = blockIdx.x, s = blockIdx.y, ct = blockIdx.z;
    const int r0 = a.seq_row0[s], n = a.seq_row0[s + 1] - r0, slot = a.seq_slot[s];
    if (n <= 0) return;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64, g = lane / 16, lr = lane % 16;
    const int VE = a.vdim + a.ones, VT = (VE + 15) / 16, col = 16 * ct + lr;
    const ChunkLayout lay(D, VT);
    const bool active = col < VE;
    f32x4 S[TPW];
    float *sp = a.state + (((size_t)slot * a.H + h) * VE + (active ? col : 0)) * D + 4 * g;
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
        S[j] = *reinterpret_cast<const f32x4 *>(sp + 16 * (w + 4 * j));
        if (!active) S[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    struct Operands {
        f32x4 w[KIND == 0 ? 4 : 1][TPW], q[4][TPW], k[TPW][4], p[4], u[4], g[KIND == 2 ? TPW : 1];
    };
    auto fetch = [&](Operands &o, int c) __attribute__((always_inline)) {
        const float *ws = chunk_slot(a, lay, h, s, r0, c);
        const f32x4 *wq = reinterpret_cast<const f32x4 *>(ws + lay.q) + lane, *ww = reinterpret_cast<const f32x4 *>(ws + lay.w) + lane;
        const f32x4 *wk = reinterpret_cast<const f32x4 *>(ws + lay.k) + lane, *wp = reinterpret_cast<const f32x4 *>(ws + lay.p) + lane;
        const f32x4 *wu = reinterpret_cast<const f32x4 *>(ws + lay.u) + lane;
        if constexpr (KIND == 0) {
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int j = 0; j < TPW; ++j) o.w[b][j] = ww[(b * DT + w + 4 * j) * 64];
            o.u[0] = wu[(ct * 4 + w) * 64];
        } else {
#pragma unroll
            for (int b = 0; b < 4; ++b) o.u[b] = wu[(ct * 4 + b) * 64];
        }
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int j = 0; j < TPW; ++j) o.q[b][j] = wq[(b * DT + w + 4 * j) * 64];
#pragma unroll
        for (int j = 0; j < TPW; ++j)
#pragma unroll
            for (int b = 0; b < 4; ++b) o.k[j][b] = wk[((w + 4 * j) * 4 + b) * 64];
#pragma unroll
        for (int b = 0; b < 4; ++b) o.p[b] = wp[(w * 4 + min(b, w)) * 64];
        if constexpr (KIND == 2) {
#pragma unroll
            for (int j = 0; j < TPW; ++j) o.g[j] = *reinterpret_cast<const f32x4 *>(ws + lay.g + 16 * (w + 4 * j) + 4 * g);
        } else {
            o.g[0][0] = ws[lay.g];
        }
    };
    const int chunks = (n + CHUNK - 1) / CHUNK;
    auto step = [&](const Operands &cur, int c) __attribute__((always_inline)) {
        f32x4(*mine)[64] = part[c & 1][w];
        // (the token blocks' sums are independent chains: element by element across them)
        f32x4 po[4], pu[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            po[b] = pu[b] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (KIND == 0 && b == w) pu[b] = cur.u[0];
        }
#pragma unroll
        for (int j = 0; j < TPW; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if constexpr (KIND == 0) pu[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.w[b][j][e], S[j][e], pu[b], 0, 0, 0);
                    po[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.q[b][j][e], S[j][e], po[b], 0, 0, 0);
                }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            mine[b][lane] = po[b];
            if constexpr (KIND == 0) mine[4 + b][lane] = pu[b];
        }
        __syncthreads();
        f32x4 U[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if constexpr (KIND == 0) U[b] = (part[c & 1][0][4 + b][lane] + part[c & 1][1][4 + b][lane]) + (part[c & 1][2][4 + b][lane] + part[c & 1][3][4 + b][lane]);
            else U[b] = cur.u[b];
        }
#pragma unroll
        for (int j = 0; j < TPW; ++j) {
            if constexpr (KIND == 2) S[j] *= cur.g[j];
            else S[j] *= cur.g[0][0];
        }
        f32x4 o = (part[c & 1][0][w][lane] + part[c & 1][1][w][lane]) + (part[c & 1][2][w][lane] + part[c & 1][3][w][lane]);
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
#pragma unroll
                for (int j = 0; j < TPW; ++j) S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.k[j][b][e], U[b][e], S[j], 0, 0, 0);
            }
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (b <= w) o = mfma_f32_block(cur.p[b], U[b], o);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int tt = c * CHUNK + 16 * w + 4 * g + e;
            if (active && tt < n) a.obuf[((size_t)(r0 + tt) * a.H + h) * VE + col] = o[e];
        }
    };
    // (every fetch is issued, the last chunk's again at the end: with a branch around it the compiler waits for all outstanding loads instead of the current chunk's)
    Operands even, odd;
    fetch(even, 0);
    for (int c = 0; c < chunks; c += 2) {
        fetch(odd, min(c + 1, chunks - 1));
        step(even, c);
        if (c + 1 >= chunks) break;
        fetch(even, min(c + 2, chunks - 1));
        step(odd, c + 1);
    }
    if (active) {
#pragma unroll
        for (int j = 0; j < TPW; ++j) *reinterpret_cast<f32x4 *>(sp + 16 * (w + 4 * j)) = S[j];
    }
}

}  // namespace hy
}  // namespace tl
