// Decode step of dense fp32 models with up to 32 rows: five launches per layer.  Included by tship_gpt.hip only.
//   gemm_qkv   : norm of x on the way into LDS, split-K partials
//   attn_decode: sums the partials, RoPE, cache append, attention
//   gemm_wo    : split K; the last block of a column tile adds the partials, b0 and x, stores x and the tile's statistics
//   gemm_ffn13 : norm of x, activation (and gate) in the epilogue
//   gemm_ffn2  : as gemm_wo
// No launch exists only to normalise, to activate or to add partial sums.  Measured, us per layer (kernel trace of graph
// replays; eight launches with norm and activation kernels of their own -> these): one row of the 512-wide gated model
// (context 64-96) QKV 5.2, attention 5.5, output 5.0 + norm 3.9, up 6.6 + activation 3.1, down 6.3 + norm 3.9 -> 3.9, 5.4, 4.8,
// 4.1, 6.4; eight rows of the 768-wide one (context 300) 7.0, 9.4, 5.2 + 6.1, 7.8 + 3.3, 10.6 + 6.1 -> 4.6, 8.7, 5.8, 6.5, 8.6.
// Whole steps of six layers at 8 / 16 / 17 / 32 rows (from 17 on in two groups of 16, which read the weights twice): 512 wide
// 312 / 399 / 547 / 602 -> 195 / 232 / 240 / 247; 768 wide 347 / 452 / 712 / 820 -> 221 / 270 / 309 / 350; 2048 wide (ffn 5632) 689 / 941 / 1923 / 2192 -> 498 / 604 / 765 / 792 us.
// An empty launch is 1.7 us.  Rows summed and normalised from the partial sums by every consumer, without the exchange in the
// tails, were measured at one row: 1.5 us more in each consumer for 1.9 less in each producer, and 2.9 at two rows; not kept.
#pragma once

#include "tship_gpt_kernels.h"

namespace tship {

// v + the lanes N places away inside each row of 16 lanes (both partners add the same two numbers)
template <int N>
__device__ __forceinline__ float sum_ror(float v) {
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + N, 0xf, 0xf, true));
}
__device__ __forceinline__ float sum_lanes16(float v) { return sum_ror<1>(sum_ror<2>(sum_ror<4>(sum_ror<8>(v)))); }

// What a row's norm needs, per tile of 32 columns: the sum, and the sum of squared distances from the tile's own mean.  Both
// norms are put together from these without cancellation, whatever the row's mean is.
// (32 consecutive lanes hold the tile; every lane gets the result)
__device__ __forceinline__ floatx2 tile_stats(float v) {
    const float s = sum_xor16(sum_lanes16(v));
    const float d = v - s * (1.0f / 32.0f);
    return floatx2{s, sum_xor16(sum_lanes16(d * d))};
}
constexpr int F32_STEP_ROWS = 32, F32_STEP_TILES = 64;      // rows of a step; 32-column tiles of a row whose statistics a block combines

struct F32StepArgs {
    const float* X; const float* W; long ldx, ldb;
    int K, N, NT, rows, KS, kper;       // NT: column tiles; block (tile, split) multiplies k = split * kper ... of the tile
    // F32_NORM: X holds the residual stream, st [tile][32 rows] the statistics of its h / 32 tiles; g, b: the norm's gamma and
    // beta (null: none); ln: LayerNorm.  F32_ACT: the input is act(p + g[k]) with p = X, or X + X2 (a second partial sum);
    // F32_GATE: times (p of column K + k, + b[k])
    const floatx2* st; const float* X2; const float* g; const float* b; int st_nt; float inv_h; float eps; int ln; int act;
    float* xn_out; long ld_xn;          // optional: the first tile's block also stores the normalised rows
    float* out; long ld_out; long split_stride; const float* bias;
    float* x; long ld_x; floatx2* st_out; float* xchg; int* count;      // residual tail, see EPI_SPLIT_TAIL of the fp16 kernel
    int* advance_pos;
};

enum { F32_PLAIN = 0, F32_NORM = 1, F32_ACT = 2, F32_GATE = 3 };      // where the input rows come from
enum { F32_PARTIAL = 0, F32_BIAS = 1, F32_TAIL = 2 };                 // what becomes of the sums

// Y[rows][N] = f(X) W.  Block: 32 columns (8 lanes of four) x one range of k; the other lanes take groups of four k, so a
// thread reads four weight rows (16 bytes each) and, per row of X, one 16-byte broadcast from LDS.
// What bounds it: a launch of 1-10 MB of weights is a chain of round trips (input rows, weights, and for the tail the
// exchange), so all of a thread's first requests, weights included, are out before the first wait, and the weights arrive
// while the rows are normalised.  The sums over the k-lanes: halves and rows of 16 lanes with lane swaps that halve the
// values per lane, then the wavefronts through LDS, always in the same order.  The leading arguments are preloaded (st_: the
// statistics, or the second partial sum of an activation's input).
// MR: rows of a block, held in registers (a power of two up to 16; blockIdx.z: groups of MR rows; 32 rows at once take 256
// registers and one wavefront per SIMD: 13.0 against 9.2 us at 768 x 3072, the vocabulary projection 73 against 50).  U: groups of four k a thread has in
// flight.  KC: k per pass through LDS.  VEC: N and ldb are multiples of four.
template <int MR, int U, int SRC, int EPI, bool VEC = true>
__global__ __launch_bounds__(256) void step_gemm_f32_kernel(const float* __restrict__ W_, const float* __restrict__ X_, const floatx2* __restrict__ st_, int ldb_, int ldx_,
                                                            const float* __restrict__ g_, const float* __restrict__ b_, int K_, int kper_, int NT_, int rows_, F32StepArgs a) {
    constexpr int TN = 32, CL = TN / 4, KL = 256 / CL;
    constexpr int RPW = MR >= 4 ? MR / 4 : 1, WPR = MR >= 4 ? 1 : 4 / MR, QS = 64 * WPR;      // staging: rows per wavefront, wavefronts per row
    constexpr int KC = 4 * KL * U, XI = (KC / 4 + QS - 1) / QS;      // k per pass through LDS: one batch of weights
    __shared__ float sX[MR * KC];
    __shared__ float red[4][MR * TN];
    __shared__ float s_mean[MR], s_rs[MR];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    // tiles next to each other sit on one XCD
    const int tile = (blockIdx.x & 7) * ((NT_ + 7) >> 3) + (blockIdx.x >> 3), ks = blockIdx.y;
    if (tile >= NT_) return;
    const int row0 = blockIdx.z * MR, rows = min(rows_ - row0, MR);
    const int cl = t & (CL - 1), kl = t / CL;
    const int kb = ks * kper_, ke = min(K_, kb + kper_);

    floatx2 sv[SRC == F32_NORM ? F32_STEP_TILES / 16 : 1];      // 16 lanes to a row
    if constexpr (SRC == F32_NORM) {
#pragma unroll
        for (int i = 0; i < F32_STEP_TILES / 16; ++i) sv[i] = st_[(long)min((t & 15) + 16 * i, a.st_nt - 1) * F32_STEP_ROWS + row0 + min(t >> 4, MR - 1)];
    }
    float acc[MR][4];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[m][c] = 0.0f;
    const long wcol = VEC ? min((long)tile * TN + 4 * cl, (long)a.N - 4) : (long)tile * TN + 4 * cl;      // the thread's first weight column
    floatx4 wv[U][4];
    auto load_w = [&](int k0, int kn) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = k0 + min(4 * (kl + u * KL), kn - 4) + j;      // (past the range: its last rows again, and zeros below)
                if constexpr (VEC) wv[u][j] = load_once((const floatx4*)(W_ + (long)k * ldb_ + wcol));
                else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) wv[u][j][c] = W_[(long)k * ldb_ + min(wcol + c, (long)a.N - 1)];
                }
            }
    };
    const int m0 = MR >= 4 ? w * RPW : w / WPR, ql = lane + 64 * (MR >= 4 ? 0 : w % WPR);
    constexpr bool ACT = SRC == F32_ACT || SRC == F32_GATE, GATE = SRC == F32_GATE;
    floatx4 xv[XI][RPW], gv[XI], bv[XI];
    floatx4 x2[ACT ? XI : 1][RPW], xg[GATE ? XI : 1][RPW], g2[GATE ? XI : 1][RPW];      // a second partial sum, and the gate's two
    auto request = [&](int k0) {      // a pass's operands
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int k = min(k0 + 4 * (ql + i * QS), K_ - 4);
#pragma unroll
            for (int r = 0; r < RPW; ++r) {
                const long at = (long)(row0 + min(m0 + r, rows - 1)) * ldx_ + k;
                xv[i][r] = *(const floatx4*)(X_ + at);
                if constexpr (ACT) x2[i][r] = *(const floatx4*)((const float*)st_ + at);
                if constexpr (GATE) { xg[i][r] = *(const floatx4*)(X_ + at + K_); g2[i][r] = *(const floatx4*)((const float*)st_ + at + K_); }
            }
            if constexpr (SRC != F32_PLAIN) gv[i] = *(const floatx4*)(g_ + k);
            bv[i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (SRC == F32_NORM) { if (b_) bv[i] = *(const floatx4*)(b_ + k); }
            if constexpr (GATE) bv[i] = *(const floatx4*)(b_ + k);
        }
        load_w(k0, min(KC, ke - k0));
    };
    request(kb);
    // residual tail: what the last block of the tile will need
    constexpr int TI = (MR * TN + 255) / 256;
    float tail_x[TI], tail_b[TI];
    if constexpr (EPI == F32_TAIL) {
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            const int idx = min(t + 256 * i, MR * TN - 1), m = min(idx / TN, rows - 1), col = tile * TN + idx % TN;
            tail_x[i] = a.x[(long)(row0 + m) * a.ld_x + col]; tail_b[i] = a.bias[col];
        }
    }
    for (int k0 = kb; k0 < ke; k0 += KC) {
        const int kn = min(KC, ke - k0);
        if (k0 > kb) __syncthreads();                              // the pass before is consumed
        if constexpr (SRC == F32_NORM) {
            if (k0 == kb) {
                float s = 0.0f, q = 0.0f;
#pragma unroll
                for (int i = 0; i < F32_STEP_TILES / 16; ++i) if ((t & 15) + 16 * i < a.st_nt) s += sv[i][0];
                const float mean = a.ln ? sum_lanes16(s) * a.inv_h : 0.0f;
#pragma unroll
                for (int i = 0; i < F32_STEP_TILES / 16; ++i)
                    if ((t & 15) + 16 * i < a.st_nt) { const float d = sv[i][0] * (1.0f / 32.0f) - mean; q += sv[i][1] + 32.0f * d * d; }
                q = sum_lanes16(q);
                const int m = t >> 4;
                if ((t & 15) == 0 && m < MR) { s_mean[m] = mean; s_rs[m] = 1.0f / sqrtf(q * a.inv_h + a.eps); }
                __syncthreads();
            }
        }
        if constexpr (ACT) {
            const bool two = (const float*)st_ != X_;
            with_act(a.act, [&](auto A) {      // (the switch outside of the values' loops: 9.4 against 8.1 us at 8 x 3072 x 768)
#pragma unroll
                for (int i = 0; i < XI; ++i)
#pragma unroll
                    for (int r = 0; r < RPW; ++r)
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            float v = act_apply_c<decltype(A)::value>((two ? xv[i][r][c] + x2[i][r][c] : xv[i][r][c]) + gv[i][c]);
                            if constexpr (GATE) v *= (two ? xg[i][r][c] + g2[i][r][c] : xg[i][r][c]) + bv[i][c];
                            xv[i][r][c] = v;
                        }
            });
        }
#pragma unroll
        for (int i = 0; i < XI; ++i) {
            const int q = ql + i * QS;
#pragma unroll
            for (int r = 0; r < RPW; ++r) {
                const int m = m0 + r;
                floatx4 v = xv[i][r];
                if constexpr (SRC == F32_NORM) {
                    const float mean = s_mean[m], rs = s_rs[m];
#pragma unroll
                    for (int c = 0; c < 4; ++c) v[c] = gv[i][c] * ((v[c] - mean) * rs) + bv[i][c];
                }
#pragma unroll
                for (int c = 0; c < 4; ++c) v[c] = 4 * q < kn && m < rows ? v[c] : 0.0f;
                if (KC / 4 % QS == 0 || 4 * q < KC) *(floatx4*)&sX[m * KC + 4 * q] = v;
                if constexpr (SRC == F32_NORM) {
                    if (a.xn_out && tile == 0 && ks == 0 && 4 * q < kn && m < rows) *(floatx4*)(a.xn_out + (long)(row0 + m) * a.ld_xn + k0 + 4 * q) = v;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (4 * u * KL >= kn) break;                           // (the same for the whole block)
            const int g = kl + u * KL;
            const bool ok = 4 * g < kn;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) wv[u][j][c] = ok ? wv[u][j][c] : 0.0f;
#pragma unroll
            for (int m = 0; m < MR; ++m) {
                const floatx4 xm = *(const floatx4*)&sX[m * KC + 4 * g];
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[m][c] = fmaf(xm[j], wv[u][j][c], acc[m][c]);
            }
        }
        if (k0 + KC < ke) request(k0 + KC);
    }
    if (a.advance_pos && blockIdx.x == 0 && ks == 0 && blockIdx.z == 0 && t == 0) { a.advance_pos[0] += 1; a.advance_pos[1] += 1; }

    // sum over the k-lanes: after the two swaps a lane holds MR of its 4 MR values, those of index j + MR (row of 16 lanes)
    float v1[MR * 2], v2[MR];
#pragma unroll
    for (int i = 0; i < 2 * MR; ++i) {
        const int i2 = i + 2 * MR;
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i >> 2][i & 3]), __float_as_uint(acc[i2 >> 2][i2 & 3]), false, false);
        v1[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
#pragma unroll
    for (int i = 0; i < MR; ++i) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v1[i]), __float_as_uint(v1[i + MR]), false, false);
        v2[i] = sum_ror<8>(__uint_as_float(r[0]) + __uint_as_float(r[1]));
    }
    if ((lane & 15) < CL) {
        const int g = lane >> 4;
#pragma unroll
        for (int j = 0; j < MR; ++j) {
            const int idx = j + (g & 1) * MR + (g >> 1) * 2 * MR;
            red[w][(idx >> 2) * TN + cl * 4 + (idx & 3)] = v2[j];
        }
    }
    __syncthreads();
    float val[TI];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const int idx = min(t + 256 * i, MR * TN - 1);
        val[i] = ((red[0][idx] + red[1][idx]) + red[2][idx]) + red[3][idx];
    }
    if constexpr (EPI == F32_TAIL) {
        if (a.KS > 1) {
            // (the exchange of the fp16 kernel's split tail: the ordering it rests on is written there)
            __shared__ int s_last;
            const int cell = blockIdx.z * NT_ + tile;
            const long sstride = (long)gridDim.z * NT_ * (MR * TN);
            float* o = a.xchg + ks * sstride + (long)cell * (MR * TN) + t;
#pragma unroll
            for (int i = 0; i < TI; ++i) if (t + 256 * i < MR * TN) __hip_atomic_store(o + 256 * i, val[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (t == 0) s_last = __hip_atomic_fetch_add(a.count + cell, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.KS - 1;
            __syncthreads();
            if (!s_last) return;
            const float* p = a.xchg + (long)cell * (MR * TN);
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                const int idx = min(t + 256 * i, MR * TN - 1);
                float pk[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) pk[k] = k < a.KS ? __hip_atomic_load(p + k * sstride + idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0f;
                val[i] = pk[0];
#pragma unroll
                for (int k = 1; k < 16; ++k) if (k < a.KS) val[i] += pk[k];
            }
            if (t == 0) __hip_atomic_store(a.count + cell, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            const int idx = t + 256 * i, m = idx / TN, col = idx % TN;
            const float v = (val[i] + tail_b[i]) + tail_x[i];
            const floatx2 s = tile_stats(v);
            if (idx < MR * TN && m < rows) {
                a.x[(long)(row0 + m) * a.ld_x + tile * TN + col] = v;
                if (col == 0) a.st_out[(long)tile * F32_STEP_ROWS + row0 + m] = s;
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            const int idx = t + 256 * i, m = idx / TN, col = tile * TN + idx % TN;
            if (idx >= MR * TN || m >= rows || col >= a.N) continue;
            if constexpr (EPI == F32_BIAS) a.out[(long)(row0 + m) * a.ld_out + col] = val[i] + a.bias[col];
            else a.out[ks * a.split_stride + (long)(row0 + m) * a.ld_out + col] = val[i];
        }
    }
}

// Entry of the step: x = E[id] * sqrt(h) (+ segment row 0) and its tiles' statistics.  Row r of the launch, NT threads.
struct F32EmbedArgs {
    float* x; long ldx; int h; const int* ids; const float* emb; float emb_scale; const float* seg; floatx2* st;
};
template <int NT>
__device__ __forceinline__ void f32_embed_row(const F32EmbedArgs& a, int r, long erow, int t) {
    for (int c0 = t; c0 < (int)round_up(a.h, NT); c0 += NT) {
        const int c = min(c0, a.h - 1);
        float v = a.emb[erow * a.h + c] * a.emb_scale;
        if (a.seg) v += a.seg[c];
        const floatx2 s = tile_stats(v);
        if (c0 < a.h) {
            a.x[(long)r * a.ldx + c] = v;
            if ((c & 31) == 0) a.st[(long)(c >> 5) * F32_STEP_ROWS + r] = s;
        }
    }
}
__global__ __launch_bounds__(256) void f32_embed_kernel(F32EmbedArgs a) { f32_embed_row<256>(a, blockIdx.x, a.ids[blockIdx.x], threadIdx.x); }
__global__ __launch_bounds__(1024) void greedy_embed_f32_kernel(const float* __restrict__ logits, long ld, int V, int* __restrict__ next_ids,
                                                                int* __restrict__ gen_out, const int* __restrict__ d_step,
                                                                int* __restrict__ last_pos, long last_ld, const int* __restrict__ d_len,
                                                                const unsigned char* __restrict__ blocked, F32EmbedArgs ea) {
    const int tok = greedy_row(logits, ld, V, next_ids, gen_out, d_step, last_pos, last_ld, d_len, blocked);
    f32_embed_row<1024>(ea, blockIdx.x, tok, threadIdx.x);
}

}  // namespace tship
