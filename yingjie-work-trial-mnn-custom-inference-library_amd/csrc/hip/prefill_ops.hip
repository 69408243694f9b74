// prefill_ops.hip - linear attention of a prompt chunk on gfx950.
//
// The reference prefills token by token (CustomModel::prefill,
// customlib/runtime/custom_model.cpp:610-640); the arithmetic per token is the
// same as decode.  The chunk's projections are in prefill_gemm.hip, its
// attention in prefill_attn.hip; here the recurrence of the linear-attention
// layers runs as batched kernels:
//   linear_conv_prefill_tg_kernel + scan_chunk_prep_kernel + scan_chunk_state_kernel   conv1d + norms +
//                        gates for all tokens, then the gated-delta recurrence
//                        with the state in registers (one-pass kernels
//                        linear_scan_wave_kernel / linear_scan_kernel otherwise)
#include <algorithm>

#include "xqhip_common.hpp"
#include "xqhip_kernels.hpp"

namespace xqhip {

typedef float floatx4 __attribute__((ext_vector_type(4)));
// register arrays of native vectors (arrays of HIP's uint4 / uint2 structs are kept in scratch)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Linear attention over a prompt chunk: block (vh, 16-column slice) runs the
// decode step of linear_step_kernel for tokens 0..tokens-1 in order, with its
// recurrent-state columns and the conv history of the channels it computes
// held in registers for the whole chunk.  The history is read from hist_in
// and the final one written to hist_out (distinct buffers: the caller picks
// the parity copies); the q/k history is written by one block per key head,
// the value history by the block that owns the channel.
// ---------------------------------------------------------------------------
constexpr int kScanCols = 16;
constexpr int kScanIGroups = 16;
constexpr int kScanMaxK = 16;     // key dim <= 256
constexpr int kScanMaxHist = 7;   // conv kernel <= 8
constexpr int kScanMaxQkPerThread = 2;
constexpr int kScanAhead = 4;       // tokens per load group

__global__ void __launch_bounds__(256) linear_scan_kernel(LinearScanLaunch p) {
    __shared__ float qk[2 * 256];
    __shared__ float vsh[kScanCols];
    __shared__ float colsum[4][kScanCols];
    __shared__ float red[2][4];
    const int vh = blockIdx.x;
    const int j0 = blockIdx.y * kScanCols;
    const int factor = max(1, p.lv_n / max(1, p.lk_n));
    const int kh = min(p.lk_n - 1, vh / factor);
    const int dk = p.lk_hd, dv = p.lv_hd;
    const int hist = max(0, p.ksize - 1);
    const bool qk_writer = (vh % factor == 0) && blockIdx.y == 0;
    const int jl = threadIdx.x % kScanCols;
    const int ig = threadIdx.x / kScanCols;
    const int j = j0 + jl;
    const bool active = j < dv;
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    float* S = p.state + static_cast<size_t>(vh) * dk * dv;
    float sreg[kScanMaxK];
#pragma unroll
    for (int r = 0; r < kScanMaxK; ++r) {
        const int i = ig + r * kScanIGroups;
        sreg[r] = (active && i < dk) ? S[static_cast<size_t>(i) * dv + j] : 0.0f;
    }
    // channels this thread convolves: q/k channels tid and tid + 256 (< 2 dk),
    // and (threads < 16) the value channel of column j0 + tid
    int ch[kScanMaxQkPerThread + 1];
    float hreg[kScanMaxQkPerThread + 1][kScanMaxHist];
    float wreg[kScanMaxQkPerThread + 1][kScanMaxHist];
    float wx[kScanMaxQkPerThread + 1];
#pragma unroll
    for (int u = 0; u <= kScanMaxQkPerThread; ++u) {
        int c = -1;
        if (u < kScanMaxQkPerThread) {
            const int tq = threadIdx.x + u * 256;
            if (tq < 2 * dk) c = (tq >= dk ? p.lk_n * dk : 0) + kh * dk + (tq >= dk ? tq - dk : tq);
        } else if (threadIdx.x < kScanCols && j0 + static_cast<int>(threadIdx.x) < dv) {
            c = 2 * p.lk_n * dk + vh * dv + j0 + threadIdx.x;
        }
        ch[u] = c;
#pragma unroll
        for (int i = 0; i < kScanMaxHist; ++i) {
            hreg[u][i] = (c >= 0 && i < hist) ? p.hist_in[static_cast<size_t>(c) * hist + i] : 0.0f;
            wreg[u][i] = (c >= 0 && i < hist) ? p.conv_w[static_cast<size_t>(c) * p.ksize + i] : 0.0f;
        }
        wx[u] = c >= 0 ? p.conv_w[static_cast<size_t>(c) * p.ksize + hist] : 0.0f;
    }
    const float rdk = 1.0f / sqrtf(static_cast<float>(dk));
    const float neg_exp_alog = -expf(p.a_log[vh]);
    const float dtb = p.dt_bias[vh];
    // Token inputs are loaded kScanAhead tokens at a time, one group ahead of
    // the group being computed (a token's compute is shorter than a load's
    // latency), with range-checked buffer loads: rows past the last token
    // read as 0 without a memory access, so every load is unconditional.
    const uint32_t stride4 = static_cast<uint32_t>(p.mixed_stride) * 4u;
    const __amdgpu_buffer_rsrc_t r_mixed = buf_rsrc(p.mixed, static_cast<uint32_t>(p.tokens) * stride4);
    const uint32_t ab_bytes = static_cast<uint32_t>(p.tokens - 1) * stride4 + static_cast<uint32_t>(p.lv_n) * 4u;
    const __amdgpu_buffer_rsrc_t r_a = buf_rsrc(p.a, ab_bytes), r_b = buf_rsrc(p.b, ab_bytes);
    float xg[2][kScanAhead][kScanMaxQkPerThread + 1], ag[2][kScanAhead], bg[2][kScanAhead];
    auto load_group = [&](int t0, int buf) {
#pragma unroll
        for (int k = 0; k < kScanAhead; ++k) {
            const uint32_t row = static_cast<uint32_t>(t0 + k) * stride4;
#pragma unroll
            for (int u = 0; u <= kScanMaxQkPerThread; ++u)
                xg[buf][k][u] = buf_load_f32(r_mixed, ch[u] >= 0 ? row + static_cast<uint32_t>(ch[u]) * 4u : kBufOOB);
            ag[buf][k] = buf_load_f32(r_a, row + static_cast<uint32_t>(vh) * 4u);
            bg[buf][k] = buf_load_f32(r_b, row + static_cast<uint32_t>(vh) * 4u);
        }
    };
    load_group(0, 0);
    for (int t0 = 0; t0 < p.tokens; t0 += kScanAhead) {
        load_group(t0 + kScanAhead, 1);
#pragma unroll
        for (int k = 0; k < kScanAhead; ++k) {
        const int t = t0 + k;
        if (t >= p.tokens) break;  // block-uniform
        float xcur[kScanMaxQkPerThread + 1];
#pragma unroll
        for (int u = 0; u <= kScanMaxQkPerThread; ++u) xcur[u] = xg[0][k][u];
        const float a_cur = ag[0][k], b_cur = bg[0][k];
        float ssq = 0.0f, ssk = 0.0f;
#pragma unroll
        for (int u = 0; u <= kScanMaxQkPerThread; ++u) {
            const int c = ch[u];
            if (c < 0) continue;
            const float xv = xcur[u];
            float acc = 0.0f;
#pragma unroll
            for (int i = 0; i < kScanMaxHist; ++i)
                if (i < hist) acc += hreg[u][i] * wreg[u][i];
            acc += xv * wx[u];
#pragma unroll
            for (int i = 0; i < kScanMaxHist; ++i) {
                if (i + 1 < hist) hreg[u][i] = hreg[u][i + 1];
                else if (i + 1 == hist) hreg[u][i] = xv;
            }
            const float yv = silu_dev(acc);
            if (u < kScanMaxQkPerThread) {
                const int tq = threadIdx.x + u * 256;
                const bool is_k = tq >= dk;
                qk[(is_k ? 256 : 0) + (is_k ? tq - dk : tq)] = yv;
                if (is_k)
                    ssk += yv * yv;
                else
                    ssq += yv * yv;
            } else {
                vsh[threadIdx.x] = yv;
            }
        }
        ssq = wave_sum(ssq);
        ssk = wave_sum(ssk);
        if (lane == 0) {
            red[0][wid] = ssq;
            red[1][wid] = ssk;
        }
        const float beta = sigmoid_dev(b_cur);
        const float gate = neg_exp_alog * softplus_dev(a_cur + dtb);
        const float decay = expf(gate);
        __syncthreads();
        const float invq = 1.0f / sqrtf(red[0][0] + red[0][1] + red[0][2] + red[0][3] + 1.0e-6f);
        const float invk = 1.0f / sqrtf(red[1][0] + red[1][1] + red[1][2] + red[1][3] + 1.0e-6f);
        const float vj = active ? vsh[jl] : 0.0f;
        float pred = 0.0f;
#pragma unroll
        for (int r = 0; r < kScanMaxK; ++r) {
            const int i = ig + r * kScanIGroups;
            if (active && i < dk) {
                sreg[r] *= decay;
                pred += sreg[r] * (qk[256 + i] * invk);
            }
        }
        pred = xor_pair_sum<32>(xor_pair_sum<16>(pred));
        if (lane < kScanCols) colsum[wid][lane] = pred;
        __syncthreads();
        pred = colsum[0][jl] + colsum[1][jl] + colsum[2][jl] + colsum[3][jl];
        __syncthreads();
        const float delta = active ? beta * (vj - pred) : 0.0f;
        float o = 0.0f;
#pragma unroll
        for (int r = 0; r < kScanMaxK; ++r) {
            const int i = ig + r * kScanIGroups;
            if (active && i < dk) {
                sreg[r] += (qk[256 + i] * invk) * delta;
                o += sreg[r] * (qk[i] * invq);
            }
        }
        o = xor_pair_sum<32>(xor_pair_sum<16>(o));
        if (lane < kScanCols) colsum[wid][lane] = o;
        __syncthreads();
        if (threadIdx.x < kScanCols && active) {
            const float tot = colsum[0][jl] + colsum[1][jl] + colsum[2][jl] + colsum[3][jl];
            p.out[static_cast<size_t>(t) * p.out_stride + static_cast<size_t>(vh) * dv + j] = tot * rdk;
        }
        __syncthreads();  // qk, vsh, red and colsum are rewritten by the next token
        }
#pragma unroll
        for (int k = 0; k < kScanAhead; ++k) {
#pragma unroll
            for (int u = 0; u <= kScanMaxQkPerThread; ++u) xg[0][k][u] = xg[1][k][u];
            ag[0][k] = ag[1][k];
            bg[0][k] = bg[1][k];
        }
    }
#pragma unroll
    for (int r = 0; r < kScanMaxK; ++r) {
        const int i = ig + r * kScanIGroups;
        if (active && i < dk) S[static_cast<size_t>(i) * dv + j] = sreg[r];
    }
#pragma unroll
    for (int u = 0; u <= kScanMaxQkPerThread; ++u) {
        const int c = ch[u];
        if (c < 0 || (u < kScanMaxQkPerThread && !qk_writer)) continue;
#pragma unroll
        for (int i = 0; i < kScanMaxHist; ++i)
            if (i < hist) p.hist_out[static_cast<size_t>(c) * hist + i] = hreg[u][i];
    }
}

// Wave-independent form for key dim DK and conv size KS (the 9B shape: 128, 4).
// Wave w of block (vh, y) owns CPW value columns of head vh; lane l owns
// column l / (64/CPW) and key rows i = l % (64/CPW) + (64/CPW) r, so both sums
// over the key dimension (the prediction and the output) are reductions over
// the 16 lanes of a DPP row (CPW = 4) or two rows (CPW = 2, one permlane swap).  Every wave convolves the whole q/k head itself (cheap) and
// exchanges the convolved channels through its own LDS slice, so a token
// needs no block barrier at all.
template <int DK, int KS, int CPW>
__global__ void __launch_bounds__(256) linear_scan_wave_kernel(LinearScanLaunch p) {
    constexpr int CH = 2 * DK / kWave;  // q/k channels per lane
    constexpr int LPC = kWave / CPW;    // lanes per value column
    constexpr int RS = DK / LPC;        // state rows per lane
    constexpr int BC = 4 * CPW;         // value columns per block
    constexpr int H = KS - 1;
    static_assert(CH >= 1 && CH % 2 == 0 && RS >= 1, "key dim");
    __shared__ float qk_lds[4][2 * DK];
    const int vh = blockIdx.x;
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    const int factor = max(1, p.lv_n / max(1, p.lk_n));
    const int kh = min(p.lk_n - 1, vh / factor);
    const int dv = p.lv_hd;
    const int ig = lane % LPC;
    const int j = blockIdx.y * BC + wid * CPW + lane / LPC;
    const bool active = j < dv;
    float* qk_w = qk_lds[wid];
    auto qk_channel = [&](int t) { return (t >= DK ? p.lk_n * DK : 0) + kh * DK + (t % DK); };
    const int vch = 2 * p.lk_n * DK + vh * dv + j;
    // filter taps and history (history in registers across the tokens)
    float hq[CH][H > 0 ? H : 1], wq[CH][KS], hv[H > 0 ? H : 1], wvv[KS];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
        const int c = qk_channel(lane + u * kWave);
#pragma unroll
        for (int t = 0; t < H; ++t) hq[u][t] = p.hist_in[static_cast<size_t>(c) * H + t];
#pragma unroll
        for (int t = 0; t < KS; ++t) wq[u][t] = p.conv_w[static_cast<size_t>(c) * KS + t];
    }
#pragma unroll
    for (int t = 0; t < H; ++t) hv[t] = active ? p.hist_in[static_cast<size_t>(vch) * H + t] : 0.0f;
#pragma unroll
    for (int t = 0; t < KS; ++t) wvv[t] = active ? p.conv_w[static_cast<size_t>(vch) * KS + t] : 0.0f;
    float* S = p.state + static_cast<size_t>(vh) * DK * dv;
    float sreg[RS];
#pragma unroll
    for (int r = 0; r < RS; ++r) sreg[r] = active ? S[static_cast<size_t>(ig + LPC * r) * dv + j] : 0.0f;
    const float rdk = 1.0f / sqrtf(static_cast<float>(DK));
    const float neg_exp_alog = -expf(p.a_log[vh]);
    const float dtb = p.dt_bias[vh];
    // token inputs, a group of kScanAhead tokens ahead (range-checked: rows past
    // the last token read 0 without a memory access)
    const uint32_t stride4 = static_cast<uint32_t>(p.mixed_stride) * 4u;
    const __amdgpu_buffer_rsrc_t r_mixed = buf_rsrc(p.mixed, static_cast<uint32_t>(p.tokens) * stride4);
    const uint32_t ab_bytes = static_cast<uint32_t>(p.tokens - 1) * stride4 + static_cast<uint32_t>(p.lv_n) * 4u;
    const __amdgpu_buffer_rsrc_t r_a = buf_rsrc(p.a, ab_bytes), r_b = buf_rsrc(p.b, ab_bytes);
    float xg[2][kScanAhead][CH + 1], ag[2][kScanAhead], bg[2][kScanAhead];
    auto load_group = [&](int t0, int buf) {
#pragma unroll
        for (int k = 0; k < kScanAhead; ++k) {
            const uint32_t row = static_cast<uint32_t>(t0 + k) * stride4;
#pragma unroll
            for (int u = 0; u < CH; ++u)
                xg[buf][k][u] = buf_load_f32(r_mixed, row + static_cast<uint32_t>(qk_channel(lane + u * kWave)) * 4u);
            xg[buf][k][CH] = buf_load_f32(r_mixed, active ? row + static_cast<uint32_t>(vch) * 4u : kBufOOB);
            ag[buf][k] = buf_load_f32(r_a, row + static_cast<uint32_t>(vh) * 4u);
            bg[buf][k] = buf_load_f32(r_b, row + static_cast<uint32_t>(vh) * 4u);
        }
    };
    auto conv_step = [&](float (&h)[H > 0 ? H : 1], const float (&w)[KS], float x) {
        float acc = 0.0f;
#pragma unroll
        for (int t = 0; t < H; ++t) acc += h[t] * w[t];
        acc += x * w[H];
#pragma unroll
        for (int t = 0; t + 1 < H; ++t) h[t] = h[t + 1];
        if constexpr (H > 0) h[H - 1] = x;
        return silu_dev(acc);
    };
    load_group(0, 0);
    for (int t0 = 0; t0 < p.tokens; t0 += kScanAhead) {
        load_group(t0 + kScanAhead, 1);
#pragma unroll
        for (int k = 0; k < kScanAhead; ++k) {
            const int t = t0 + k;
            if (t >= p.tokens) break;  // grid-uniform
            float ssq = 0.0f, ssk = 0.0f;
#pragma unroll
            for (int u = 0; u < CH; ++u) {
                const float y = conv_step(hq[u], wq[u], xg[0][k][u]);
                qk_w[lane + u * kWave] = y;
                if (u < CH / 2) ssq += y * y; else ssk += y * y;
            }
            const float vj = conv_step(hv, wvv, xg[0][k][CH]);
            ssq = wave_sum(ssq);
            ssk = wave_sum(ssk);
            const float invq = 1.0f / sqrtf(ssq + 1.0e-6f);
            const float invk = 1.0f / sqrtf(ssk + 1.0e-6f);
            const float beta = sigmoid_dev(bg[0][k]);
            const float decay = expf(neg_exp_alog * softplus_dev(ag[0][k] + dtb));
            // the wave's own LDS writes above complete before these reads (LDS
            // operations of a wave are performed in order): no barrier
            float kr[RS], qr[RS];
#pragma unroll
            for (int r = 0; r < RS; ++r) {
                kr[r] = qk_w[DK + ig + LPC * r] * invk;
                qr[r] = qk_w[ig + LPC * r] * invq;
            }
            float pred = 0.0f;
#pragma unroll
            for (int r = 0; r < RS; ++r) {
                sreg[r] *= decay;
                pred += sreg[r] * kr[r];
            }
            pred = lanes_sum<16>(pred);
            if constexpr (LPC == 32) pred = xor_pair_sum<16>(pred);
            const float delta = beta * (vj - pred);
            float o = 0.0f;
#pragma unroll
            for (int r = 0; r < RS; ++r) {
                sreg[r] += kr[r] * delta;
                o += sreg[r] * qr[r];
            }
            o = lanes_sum<16>(o);
            if constexpr (LPC == 32) o = xor_pair_sum<16>(o);
            if (ig == 0 && active) p.out[static_cast<size_t>(t) * p.out_stride + static_cast<size_t>(vh) * dv + j] = o * rdk;
        }
#pragma unroll
        for (int k = 0; k < kScanAhead; ++k) {
#pragma unroll
            for (int u = 0; u <= CH; ++u) xg[0][k][u] = xg[1][k][u];
            ag[0][k] = ag[1][k];
            bg[0][k] = bg[1][k];
        }
    }
#pragma unroll
    for (int r = 0; r < RS; ++r)
        if (active) S[static_cast<size_t>(ig + LPC * r) * dv + j] = sreg[r];
    const bool qk_writer = (vh % factor == 0) && blockIdx.y == 0 && wid == 0;
    if (qk_writer) {
#pragma unroll
        for (int u = 0; u < CH; ++u) {
            const int c = qk_channel(lane + u * kWave);
#pragma unroll
            for (int t = 0; t < H; ++t) p.hist_out[static_cast<size_t>(c) * H + t] = hq[u][t];
        }
    }
    if (ig == 0 && active) {
#pragma unroll
        for (int t = 0; t < H; ++t) p.hist_out[static_cast<size_t>(vch) * H + t] = hv[t];
    }
}

// ---------------------------------------------------------------------------
// Two-pass form of the prefill linear-attention scan (with a workspace, key
// heads of 128 dims):
// 1. linear_conv_prefill_tg_kernel / linear_conv_prefill_kernel, parallel over
//    tokens and heads: the causal conv1d + SiLU of every channel for every
//    token of the chunk (inputs of earlier tokens from the chunk, before the
//    chunk from hist_in), the L2 norm of the q and k heads, the per-(token,
//    value head) beta = sigmoid(b) and log decay g = -exp(A_log) softplus(a +
//    dt_bias), and the final history.
// 2. the chunked recurrence (scan_chunk_prep_kernel, scan_chunk_state_kernel,
//    below): parallel over 64-token chunks except for one pass over the chunks
//    per (value head, 16 columns).
// Workspace: conv output by head, [2 lk_n][tokens][lk_hd] and [lv_n][tokens][lv_hd]
// (a block of the chunk kernels reads one head: with rows of all heads its reads
// lie a row apart and meet in few memory channels), (beta, g) [lv_n][tokens][2], then
// per (chunk, value head) the record T [64][64], Wq [64][64], gamma [64],
// gamma_last / gamma [64].
// ---------------------------------------------------------------------------
constexpr int kChunkTokens = 64;
constexpr int kChunkRecord = 2 * kChunkTokens * kChunkTokens + 2 * kChunkTokens;

size_t linear_scan_workspace_bytes(int tokens, int lk_n, int lk_hd, int lv_n, int lv_hd) {
    const size_t conv_dim = 2 * static_cast<size_t>(lk_n) * lk_hd + static_cast<size_t>(lv_n) * lv_hd;
    const size_t chunks = (static_cast<size_t>(tokens) + kChunkTokens - 1) / kChunkTokens;
    return sizeof(float) * (static_cast<size_t>(tokens) * (conv_dim + 2 * static_cast<size_t>(lv_n)) +
                            chunks * lv_n * kChunkRecord);
}

__global__ void __launch_bounds__(256) linear_conv_prefill_kernel(LinearScanLaunch p) {
    __shared__ float red[4];
    const int t = blockIdx.x, hb = blockIdx.y;
    const int dk = p.lk_hd, dv = p.lv_hd, H = p.ksize - 1;
    const int conv_dim = 2 * p.lk_n * dk + p.lv_n * dv;
    const bool is_qk = hb < 2 * p.lk_n;
    const int width = is_qk ? dk : dv;
    const int c = (is_qk ? hb * dk : 2 * p.lk_n * dk + (hb - 2 * p.lk_n) * dv) + static_cast<int>(threadIdx.x);
    const bool ok = static_cast<int>(threadIdx.x) < width;
    // input of token tau of the chunk (tau < 0: the history before it)
    auto xin = [&](int tau) {
        return tau >= 0 ? p.mixed[static_cast<size_t>(tau) * p.mixed_stride + c]
                        : p.hist_in[static_cast<size_t>(c) * H + (H + tau)];
    };
    float y = 0.0f;
    if (ok) {
        const float* w = p.conv_w + static_cast<size_t>(c) * p.ksize;
        float acc = 0.0f;
        for (int i = 0; i < H; ++i) acc += xin(t - H + i) * w[i];
        acc += xin(t) * w[H];
        y = silu_dev(acc);
        if (t == p.tokens - 1)
            for (int i = 0; i < H; ++i) p.hist_out[static_cast<size_t>(c) * H + i] = xin(p.tokens - H + i);
    }
    if (is_qk) {  // l2NormalizeHeads: x / sqrt(sum x^2 + 1e-6)
        float ss = wave_sum(y * y);
        const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
        if (lane == 0) red[wid] = ss;
        __syncthreads();
        ss = 0.0f;
        for (int i = 0; i < (width + kWave - 1) / kWave; ++i) ss += red[i];
        y *= 1.0f / sqrtf(ss + 1.0e-6f);
    } else if (threadIdx.x == 0) {
        const int vh = hb - 2 * p.lk_n;
        const size_t row = static_cast<size_t>(t) * p.mixed_stride + vh;
        float* aux = p.ws + static_cast<size_t>(p.tokens) * conv_dim + (static_cast<size_t>(vh) * p.tokens + t) * 2;
        aux[0] = sigmoid_dev(p.b[row]);
        aux[1] = -expf(p.a_log[vh]) * softplus_dev(p.a[row] + p.dt_bias[vh]);  // log of the decay
    }
    const size_t head = static_cast<size_t>(c - static_cast<int>(threadIdx.x)) * p.tokens;  // its first value
    if (ok) p.ws[head + static_cast<size_t>(t) * width + threadIdx.x] = y;
}

// The same pass for 128-channel heads and a conv kernel of KS taps, one block
// per (head, kConvTokens tokens): each thread keeps its channel's inputs for
// the tokens and the KS - 1 before them in registers (every input read once,
// range-checked buffer loads with no branch around them), and the q / k norms
// of the block's tokens share one barrier.  Same arithmetic and order as
// linear_conv_prefill_kernel.
constexpr int kConvTokens = 16;

template <int KS>
__global__ void __launch_bounds__(128) linear_conv_prefill_tg_kernel(LinearScanLaunch p) {
    constexpr int H = KS - 1, TG = kConvTokens, W = TG + H;
    __shared__ float red[2][TG];
    const int hb = blockIdx.x, g0 = blockIdx.y * TG;
    const int conv_dim = 2 * p.lk_n * 128 + p.lv_n * 128;
    const bool is_qk = hb < 2 * p.lk_n;
    const int c = (is_qk ? hb * 128 : 2 * p.lk_n * 128 + (hb - 2 * p.lk_n) * 128) + static_cast<int>(threadIdx.x);
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    // window slot i holds the input of token g0 - H + i: rows [r0, r1) of the
    // chunk, the history before token 0 (only the first group reaches it)
    const int r0 = max(0, g0 - H), r1 = min(p.tokens, g0 + TG);
    const uint32_t stride4 = static_cast<uint32_t>(p.mixed_stride) * 4u;
    const __amdgpu_buffer_rsrc_t r_x =
        buf_rsrc(p.mixed + static_cast<size_t>(r0) * p.mixed_stride, static_cast<uint32_t>(r1 - r0) * stride4);
    const __amdgpu_buffer_rsrc_t r_h = buf_rsrc(p.hist_in, static_cast<uint32_t>(conv_dim * H) * 4u);
    float xw[W], w[KS];
#pragma unroll
    for (int i = 0; i < W; ++i) {
        const int tau = g0 - H + i;
        float v = buf_load_f32(r_x, tau >= r0 ? static_cast<uint32_t>(tau - r0) * stride4 + c * 4u : kBufOOB);
        if (i < H) v += buf_load_f32(r_h, tau < 0 ? static_cast<uint32_t>(c * H + H + tau) * 4u : kBufOOB);
        xw[i] = v;
    }
#pragma unroll
    for (int i = 0; i < KS; ++i) w[i] = p.conv_w[static_cast<size_t>(c) * KS + i];
    float y[TG];
#pragma unroll
    for (int k = 0; k < TG; ++k) {
        float acc = 0.0f;
#pragma unroll
        for (int i = 0; i < H; ++i) acc += xw[k + i] * w[i];
        acc += xw[k + H] * w[H];
        y[k] = silu_dev(acc);
    }
    if (is_qk) {  // block-uniform; l2NormalizeHeads: x / sqrt(sum x^2 + 1e-6)
#pragma unroll
        for (int k = 0; k < TG; ++k) {
            const float ss = wave_sum(y[k] * y[k]);
            if (lane == 0) red[wid][k] = ss;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < TG; ++k) {
            float ss = 0.0f;
            ss += red[0][k];
            ss += red[1][k];
            y[k] *= 1.0f / sqrtf(ss + 1.0e-6f);
        }
    } else if (threadIdx.x < TG && g0 + static_cast<int>(threadIdx.x) < p.tokens) {
        const int t = g0 + threadIdx.x, vh = hb - 2 * p.lk_n;
        const size_t row = static_cast<size_t>(t) * p.mixed_stride + vh;
        float* aux = p.ws + static_cast<size_t>(p.tokens) * conv_dim + (static_cast<size_t>(vh) * p.tokens + t) * 2;
        aux[0] = sigmoid_dev(p.b[row]);
        aux[1] = -expf(p.a_log[vh]) * softplus_dev(p.a[row] + p.dt_bias[vh]);  // log of the decay
    }
#pragma unroll
    for (int k = 0; k < TG; ++k)
        if (g0 + k < p.tokens) p.ws[(static_cast<size_t>(hb) * p.tokens + g0 + k) * 128 + threadIdx.x] = y[k];
    // the history after the chunk: inputs of tokens tokens - H .. tokens - 1, slots
    // tokens - g0 + i of the group that holds the last token
    if (g0 <= p.tokens - 1 && p.tokens - 1 < g0 + TG) {
        const int base = p.tokens - g0;
#pragma unroll
        for (int i = 0; i < H; ++i) {
            float v = 0.0f;
#pragma unroll
            for (int j = 0; j < W; ++j)
                if (j == base + i) v = xw[j];
            p.hist_out[static_cast<size_t>(c) * H + i] = v;
        }
    }
}

// Chunked (parallel-in-time) form of the gated-delta recurrence over a prompt
// chunk, for key heads of 128 dims.  Within a chunk of C = 64 tokens
// (local i, decay a_i = exp(g_i), cumulative log decay G_i = g_0 + .. + g_i,
// gamma_i = exp(G_i)), the per-token update
//     S_i = a_i (I - b_i k_i k_i^T) S_{i-1} + b_i k_i v_i^T,   o_i = S_i^T q_i
// unrolls (by induction on i) to S_i = gamma_i S_0 + sum_{j<=i} exp(G_i - G_j) k_j u_j^T
// with the rows u_j^T of U solving the unit lower-triangular system
//     (I + A) U = R,   A_ij = b_i exp(G_i - G_j) (k_i . k_j) (j < i),
//     R_i = b_i (v_i - gamma_i S_0^T k_i),
// so that
//     o_i = gamma_i S_0^T q_i + sum_{j<=i} exp(G_i - G_j) (q_i . k_j) u_j,
//     S_C = gamma_{C-1} S_0 + sum_j exp(G_{C-1} - G_j) k_j u_j^T.
// scan_chunk_prep_kernel, parallel over (value head, chunk): the Gram products
// K K^T and Q K^T, T = (I + A)^{-1} (forward substitution, row by row) and
// Wq_ij = exp(G_i - G_j) (q_i . k_j) (j <= i); scan_chunk_state_kernel, one block
// per (value head, 16 value columns), walks the chunks in order with the state
// slice in LDS and the products on v_mfma_f32_16x16x4_f32 (fp32 operands, fp32
// accumulation).  The prep kernel is one block per CU as well (32 heads, 500
// tokens: 256), a chain of short phases bound by LDS latency: 16.2 us, 20.2 with
// the sums of the log decays and the block products read from LDS word by word.  Same mathematics as the per-token recurrence
// (custom_model.cpp:1074-1096), a different fp32 summation order.
constexpr int kChunk = kChunkTokens;  // tokens per chunk
constexpr int kChLd = 132;   // floats per 128-dim row in LDS (16-byte aligned rows)
constexpr int kChLdT = 68;   // floats per 64-wide row in LDS
constexpr int kChLdM = 20;   // floats per row of a 16 x 16 block in LDS
constexpr int kChRec = kChunkRecord;  // floats per (value head, chunk) record

static size_t scan_chunk_prep_lds() {
    return sizeof(float) * (2 * static_cast<size_t>(kChunk) * kChLd + 2 * kChunk * kChLdT + 4 * 16 * kChLdM + 3 * kChunk);
}
static size_t scan_chunk_state_lds() {
    return sizeof(float) * (128 * kChLdT + 2 * 16 * kChLdT + 16 * kChLd);
}

// q and k rows of key head kh for the chunk's tokens [t0, t0 + n) -> LDS rows of
// kChLd floats (rows past n are 0)
__device__ __forceinline__ void stage_qk_rows(const LinearScanLaunch& p, int kh, int t0, int n, float* Ks, float* Qs) {
    const uint32_t bytes = static_cast<uint32_t>(max(0, n)) * 512u;
    const __amdgpu_buffer_rsrc_t rq = buf_rsrc(p.ws + (static_cast<size_t>(kh) * p.tokens + t0) * 128, bytes);
    const __amdgpu_buffer_rsrc_t rk = buf_rsrc(p.ws + (static_cast<size_t>(p.lk_n + kh) * p.tokens + t0) * 128, bytes);
    u32x4 kv[8], qv[8];  // all loads in flight before the first store
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const uint32_t at = (threadIdx.x + 256u * u) * 16u;
        kv[u] = __builtin_amdgcn_raw_buffer_load_b128(rk, at, 0, 0);
        qv[u] = __builtin_amdgcn_raw_buffer_load_b128(rq, at, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int e = static_cast<int>(threadIdx.x) + 256 * u, row = e >> 5, d4 = e & 31;
        *reinterpret_cast<u32x4*>(Ks + row * kChLd + 4 * d4) = kv[u];
        *reinterpret_cast<u32x4*>(Qs + row * kChLd + 4 * d4) = qv[u];
    }
}

__global__ void __launch_bounds__(256) scan_chunk_prep_kernel(LinearScanLaunch p) {
    extern __shared__ float4 scan_lds[];
    float* Ks = reinterpret_cast<float*>(scan_lds);  // [64][kChLd]
    float* Qs = Ks + kChunk * kChLd;                 // [64][kChLd]
    float* Am = Qs + kChunk * kChLd;                 // [64][kChLdT] A (strictly lower)
    float* Tm = Am + kChunk * kChLdT;                // [64][kChLdT] T = (I + A)^{-1}, by 16 x 16 blocks
    float* Mw = Tm + kChunk * kChLdT;                // [4 waves][16][kChLdM] block products
    float* Gc = Mw + 4 * 16 * kChLdM;                   // [64] cumulative log decay
    float* Bt = Gc + kChunk;                         // [64] beta
    float* gl = Bt + kChunk;                         // [64] log decay
    const int vh = blockIdx.x, ch = blockIdx.y, t0 = ch * kChunk;
    const int n = __builtin_amdgcn_readfirstlane(min(kChunk, p.tokens - t0));  // scalar: buffer descriptors use it
    const int factor = max(1, p.lv_n / max(1, p.lk_n));
    const int kh = __builtin_amdgcn_readfirstlane(min(p.lk_n - 1, vh / factor));
    const int conv_dim = 2 * p.lk_n * 128 + p.lv_n * p.lv_hd;
    const int tid = threadIdx.x;
    stage_qk_rows(p, kh, t0, n, Ks, Qs);
    if (tid < kChunk) {  // tokens past n: beta 0, log decay 0 (the state passes unchanged)
        const float* aux = p.ws + static_cast<size_t>(p.tokens) * conv_dim;
        const size_t ai = (static_cast<size_t>(vh) * p.tokens + t0 + tid) * 2;
        Bt[tid] = tid < n ? aux[ai] : 0.0f;
        gl[tid] = tid < n ? aux[ai + 1] : 0.0f;
    }
    __syncthreads();
    if (tid < kChunk) {
        float4 g[kChunk / 4];  // every load before the chain of additions
#pragma unroll
        for (int l = 0; l < kChunk / 4; ++l) g[l] = *reinterpret_cast<const float4*>(gl + 4 * l);
        float acc = 0.0f;
#pragma unroll
        for (int l = 0; l < kChunk; ++l) {
            const float4 v = g[l >> 2];
            acc += l <= tid ? ((l & 3) == 0 ? v.x : (l & 3) == 1 ? v.y : (l & 3) == 2 ? v.z : v.w) : 0.0f;
        }
        Gc[tid] = acc;
    }
    // K K^T and Q K^T on v_mfma_f32_16x16x4_f32: wave w takes rows 16 w .. 16 w + 15
    // against the four 16-key column tiles; lane (li, lq) feeds dims 32 lq + s at
    // step s (the same permutation of the contraction for both operands)
    const int lane = tid & (kWave - 1), w = tid / kWave, li = lane & 15, lq = lane >> 4;
    float ka[32], qa[32];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const float4 kv = *reinterpret_cast<const float4*>(Ks + (16 * w + li) * kChLd + 32 * lq + 4 * u);
        const float4 qv = *reinterpret_cast<const float4*>(Qs + (16 * w + li) * kChLd + 32 * lq + 4 * u);
        ka[4 * u] = kv.x; ka[4 * u + 1] = kv.y; ka[4 * u + 2] = kv.z; ka[4 * u + 3] = kv.w;
        qa[4 * u] = qv.x; qa[4 * u + 1] = qv.y; qa[4 * u + 2] = qv.z; qa[4 * u + 3] = qv.w;
    }
    floatx4 kk[4], qk[4];
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) kk[ct] = qk[ct] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // eight independent accumulation chains, four dims of every column tile per round
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        float kb[4][4];
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) {
            const float4 v = *reinterpret_cast<const float4*>(Ks + (16 * ct + li) * kChLd + 32 * lq + 4 * u);
            kb[ct][0] = v.x; kb[ct][1] = v.y; kb[ct][2] = v.z; kb[ct][3] = v.w;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int ct = 0; ct < 4; ++ct) {
                kk[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(ka[4 * u + e], kb[ct][e], kk[ct], 0, 0, 0);
                qk[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(qa[4 * u + e], kb[ct][e], qk[ct], 0, 0, 0);
            }
    }
    __syncthreads();  // Gc is complete
    float* rec = p.ws + static_cast<size_t>(p.tokens) * (conv_dim + 2 * p.lv_n) +
                 (static_cast<size_t>(ch) * p.lv_n + vh) * kChRec;
    float* Wq = rec + kChunk * kChunk;
    // lane holds rows 16 w + 4 lq + v, column 16 ct + li of each product
#pragma unroll
    for (int ct = 0; ct < 4; ++ct)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * w + 4 * lq + v, j = 16 * ct + li;
            const float dec = j <= i ? expf(Gc[i] - Gc[j]) : 0.0f;
            Am[i * kChLdT + j] = j < i ? Bt[i] * dec * kk[ct][v] : 0.0f;
            Wq[i * kChunk + j] = dec * qk[ct][v];
        }
    __syncthreads();
    // T = (I + A)^{-1} by 16 x 16 blocks (A is strictly lower, so T is unit lower
    // triangular).  Diagonal blocks D_k = (I + A_kk)^{-1}, wave k: lane column c
    // keeps column c of D_k in registers, row r = e_r - sum_{j<r} A_rj D_j.
    const int c16 = lane & 15;
    {
        float dc[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float acc = 0.0f;
#pragma unroll
            for (int j = 0; j < r; ++j) acc += Am[(16 * w + r) * kChLdT + 16 * w + j] * dc[j];
            dc[r] = (c16 == r ? 1.0f : 0.0f) - acc;
        }
        if (lane < 16)
#pragma unroll
            for (int r = 0; r < 16; ++r) Tm[(16 * w + r) * kChLdT + 16 * w + c16] = dc[r];
    }
    __syncthreads();
    // off-diagonal blocks by distance: T_ij = -D_i sum_{k=j}^{i-1} A_ik T_kj (wave j
    // takes block (j + dist, j)); lane: row lane / 4, columns 4 (lane % 4) .. + 3
    const int br = lane >> 2, bc = 4 * (lane & 3);
    for (int dist = 1; dist < 4; ++dist) {  // block-uniform
        const int bi = w + dist, bj = w;
        const bool task = bi < 4;
        float m4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        // d += row (16 values) times the 4 columns at col (rows ld apart); every LDS read before the products
        auto madd = [](const float* row, const float* col, int ld, float (&d)[4]) {
            float4 a[4], t[16];
#pragma unroll
            for (int mm = 0; mm < 4; ++mm) a[mm] = *reinterpret_cast<const float4*>(row + 4 * mm);
#pragma unroll
            for (int mm = 0; mm < 16; ++mm) t[mm] = *reinterpret_cast<const float4*>(col + mm * ld);
#pragma unroll
            for (int mm = 0; mm < 16; ++mm) {
                const float4 q = a[mm >> 2];
                const float f = (mm & 3) == 0 ? q.x : (mm & 3) == 1 ? q.y : (mm & 3) == 2 ? q.z : q.w;
                d[0] += f * t[mm].x;
                d[1] += f * t[mm].y;
                d[2] += f * t[mm].z;
                d[3] += f * t[mm].w;
            }
        };
        if (task)
            for (int k = bj; k < bi; ++k)
                madd(Am + (16 * bi + br) * kChLdT + 16 * k, Tm + 16 * k * kChLdT + 16 * bj + bc, kChLdT, m4);
        float* mw = Mw + w * 16 * kChLdM;
        if (task) *reinterpret_cast<float4*>(mw + br * kChLdM + bc) = make_float4(m4[0], m4[1], m4[2], m4[3]);
        __syncthreads();
        if (task) {
            float t4[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            madd(Tm + (16 * bi + br) * kChLdT + 16 * bi, mw + bc, kChLdM, t4);
            *reinterpret_cast<float4*>(Tm + (16 * bi + br) * kChLdT + 16 * bj + bc) =
                make_float4(-t4[0], -t4[1], -t4[2], -t4[3]);
        }
        __syncthreads();
    }
    // buffer stores: a record need only be aligned to 4 bytes
    const __amdgpu_buffer_rsrc_t rec_r = buf_rsrc(rec, kChRec * 4u);
    for (int e = tid; e < kChunk * kChunk / 4; e += 256) {
        const int i = e >> 4, j = 4 * (e & 15);
        u32x4 v = *reinterpret_cast<const u32x4*>(Tm + i * kChLdT + j);
        if ((j >> 4) > (i >> 4)) v = u32x4{0u, 0u, 0u, 0u};  // blocks above the diagonal are 0
        __builtin_amdgcn_raw_buffer_store_b128(v, rec_r, e * 16u, 0, 0);
    }
    if (tid < kChunk) {
        rec[2 * kChunk * kChunk + tid] = expf(Gc[tid]);                          // gamma_i
        rec[2 * kChunk * kChunk + kChunk + tid] = expf(Gc[kChunk - 1] - Gc[tid]);  // gamma_last / gamma_j
    }
}

// Eight waves.  Wave w < 4 computes X = K S_0, R and U for tokens 16 w .. 16 w + 15, wave w + 4 computes
// Y = Q S_0 and the output for the same tokens, and wave w updates state rows 16 w .. 16 w + 15; the output of a chunk
// is computed under the next chunk's X, Y under U, so that each SIMD has two waves with products to issue.  What
// only a wave's own products read (its rows of K and T or Q and Wq, its values and gates) goes from memory straight
// into the lanes that feed the MFMAs, requested for the next chunk as soon as this chunk has used it.  LDS carries
// what crosses waves: K^T (for the state update), R and U (transposed: a lane's operand is a contiguous run) and
// the state slice.
// What bounds it: one block per CU (32 heads of 128 columns: 256 blocks), so a chunk is 128 fp32 MFMAs per SIMD (32
// clocks each, 1.7 us) and three barriers between dependent products.  32 heads, 500 tokens: 34.7 us (30 without the loads); four
// waves with every operand staged through LDS (five barriers, 290 KB of LDS traffic a chunk) 41.8, four waves with
// the operands straight into registers 39.4.
constexpr int kStateThreads = 512;
__global__ void __launch_bounds__(kStateThreads) scan_chunk_state_kernel(LinearScanLaunch p) {
    extern __shared__ float4 scan_lds[];
    float* Kt = reinterpret_cast<float*>(scan_lds);  // [128][kChLdT] K^T
    float* Rt = Kt + 128 * kChLdT;                   // [16][kChLdT] R^T
    float* Ut = Rt + 16 * kChLdT;                    // [16][kChLdT] U^T
    float* St = Ut + 16 * kChLdT;                    // [16][kChLd] the state slice, transposed
    const int vh = blockIdx.x, j0 = blockIdx.y * 16;
    const int factor = max(1, p.lv_n / max(1, p.lk_n));
    const int kh = __builtin_amdgcn_readfirstlane(min(p.lk_n - 1, vh / factor));
    const int dv = p.lv_hd;
    const int conv_dim = 2 * p.lk_n * 128 + p.lv_n * dv;
    const int chunks = __builtin_amdgcn_readfirstlane((p.tokens + kChunk - 1) / kChunk);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const bool outputs = w >= 4;
    const int wt = w & 3;
    const int li = lane & 15, lq = lane >> 4;  // MFMA operand row / column li, k slot lq
    const bool cact = j0 + li < dv;
    const float rdk = 1.0f / sqrtf(128.0f);
    float* S = p.state + static_cast<size_t>(vh) * 128 * dv;
    const float* aux = p.ws + static_cast<size_t>(p.tokens) * conv_dim;
    const float* recs = aux + static_cast<size_t>(p.tokens) * p.lv_n * 2;
    // byte offsets of the lane's operands: every load is a range-checked buffer load, tokens past the prompt and
    // chunks past the last read 0 (sizes and bases through readfirstlane: scalar buffer descriptors).  The
    // contraction index of every product is a permutation shared by both operands: at step 4 u + e, k slot lq takes
    // dim or token 16 u + 4 lq + e, so an operand is 16 contiguous bytes per u and four lanes read 64.
    const uint32_t xoff = static_cast<uint32_t>(16 * wt + li) * 512u + 16u * lq;  // q or k row
    const uint32_t moff = static_cast<uint32_t>(16 * wt + li) * (kChunk * 4u) + 16u * lq +
                          (outputs ? kChunk * kChunk * 4u : 0u);  // Wq or T row
    const uint32_t voff = cact ? static_cast<uint32_t>((16 * wt + 4 * lq) * dv + j0 + li) * 4u : kBufOOB;
    const uint32_t boff = static_cast<uint32_t>(16 * wt + 4 * lq) * 8u;
    const uint32_t goff = 2u * kChunk * kChunk * 4u;  // gamma, then gamma_last / gamma
    const float* xhead = p.ws + static_cast<size_t>(outputs ? kh : p.lk_n + kh) * p.tokens * 128;
    const float* vhead = p.ws + (static_cast<size_t>(2 * p.lk_n) * 128 + static_cast<size_t>(vh) * dv) * p.tokens;
    struct Rows { __amdgpu_buffer_rsrc_t x, v, rec, aux; };
    auto rows = [&](int ch) {
        const int t0 = __builtin_amdgcn_readfirstlane(min(ch * kChunk, p.tokens));
        const int n = __builtin_amdgcn_readfirstlane(max(0, min(kChunk, p.tokens - t0)));
        const int cr = __builtin_amdgcn_readfirstlane(min(ch, chunks - 1));
        return Rows{buf_rsrc(xhead + static_cast<size_t>(t0) * 128, static_cast<uint32_t>(n) * 512u),
                    buf_rsrc(vhead + static_cast<size_t>(t0) * dv, static_cast<uint32_t>(n) * dv * 4u),
                    buf_rsrc(recs + static_cast<size_t>(cr * p.lv_n + vh) * kChRec,
                             static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(ch < chunks ? kChRec * 4 : 0))),
                    buf_rsrc(aux + (static_cast<size_t>(vh) * p.tokens + t0) * 2, static_cast<uint32_t>(n) * 8u)};
    };
    auto load4 = [](__amdgpu_buffer_rsrc_t r, uint32_t off, float* d) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = __uint_as_float(v[e]);
    };
    float x[32], mt[16], v4[4], bet[4], gam[4], dl[16], glast;  // x: K or Q rows, mt: T or Wq rows
    auto load_x = [&](const Rows& r) {
#pragma unroll
        for (int u = 0; u < 8; ++u) load4(r.x, xoff + 64u * u, x + 4 * u);
    };
    auto load_m = [&](const Rows& r) {
#pragma unroll
        for (int u = 0; u < 4; ++u) load4(r.rec, moff + 64u * u, mt + 4 * u);
    };
    auto load_values = [&](const Rows& r) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            v4[v] = buf_load_f32(r.v, voff + static_cast<uint32_t>(v) * dv * 4u);
            bet[v] = buf_load_f32(r.aux, boff + 8u * v);
        }
    };
    auto load_gamma = [&](const Rows& r) { load4(r.rec, goff + (16 * wt + 4 * lq) * 4u, gam); };
    auto load_decay = [&](const Rows& r) {
        glast = buf_load_f32(r.rec, goff + (kChunk - 1) * 4u);
#pragma unroll
        for (int u = 0; u < 4; ++u) load4(r.rec, goff + (kChunk + 16 * u + 4 * lq) * 4u, dl + 4 * u);
    };
    // a float4 of LDS into four registers
    auto ld4 = [](const float* a, float* d) {
        const float4 v = *reinterpret_cast<const float4*>(a);
        d[0] = v.x; d[1] = v.y; d[2] = v.z; d[3] = v.w;
    };
    const floatx4 zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
    auto times_state = [&] {  // x S_0, two chains (even and odd steps)
        float sp[32];
#pragma unroll
        for (int u = 0; u < 8; ++u) ld4(St + li * kChLd + 16 * u + 4 * lq, sp + 4 * u);
        floatx4 r0 = zero4, r1 = zero4;
#pragma unroll
        for (int st = 0; st < 32; st += 2) {
            r0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[st], sp[st], r0, 0, 0, 0);
            r1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[st + 1], sp[st + 1], r1, 0, 0, 0);
        }
        return r0 + r1;
    };
    auto times_rows = [&](const float (&b)[16]) {  // mt b
        floatx4 r0 = zero4, r1 = zero4;
#pragma unroll
        for (int st = 0; st < 16; st += 2) {
            r0 = __builtin_amdgcn_mfma_f32_16x16x4f32(mt[st], b[st], r0, 0, 0, 0);
            r1 = __builtin_amdgcn_mfma_f32_16x16x4f32(mt[st + 1], b[st + 1], r1, 0, 0, 0);
        }
        return r0 + r1;
    };
    floatx4 Y = zero4;
    float ub[16];
    auto output = [&](int ch) {  // O = diag(gamma) Y + Wq U of chunk ch
        const floatx4 O = times_rows(ub);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int t = ch * kChunk + 16 * wt + 4 * lq + v;
            if (t < p.tokens && cact)
                p.out[static_cast<size_t>(t) * p.out_stride + static_cast<size_t>(vh) * dv + j0 + li] =
                    (gam[v] * Y[v] + O[v]) * rdk;
        }
    };
    {
        const Rows r = rows(0);
        load_x(r);
        if (!outputs) {
            load_values(r);
            load_gamma(r);
            load_m(r);
        }
        load_decay(r);
    }
    for (int e = tid; e < 128 * 16; e += kStateThreads) {
        const int d = e >> 4, cc = e & 15;
        St[cc * kChLd + d] = j0 + cc < dv ? S[static_cast<size_t>(d) * dv + j0 + cc] : 0.0f;
    }
    __syncthreads();
    // S_C = gamma_last S_0 + K^T diag(del) U: the wave's state rows.  The second and third barrier of a chunk.
    auto update_state = [&](const Rows& nx) {
        float kt[16], s4[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) ld4(Kt + (16 * w + li) * kChLdT + 16 * u + 4 * lq, kt + 4 * u);
        ld4(St + li * kChLd + 16 * w + 4 * lq, s4);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) ld4(Ut + li * kChLdT + 16 * u + 4 * lq, ub + 4 * u);
        __builtin_amdgcn_sched_barrier(0);
        floatx4 Sn, S1 = zero4;
#pragma unroll
        for (int v = 0; v < 4; ++v) Sn[v] = glast * s4[v];
#pragma unroll
        for (int st = 0; st < 16; st += 2) {
            Sn = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[st], ub[st] * dl[st], Sn, 0, 0, 0);
            S1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[st + 1], ub[st + 1] * dl[st + 1], S1, 0, 0, 0);
        }
        Sn += S1;
        *reinterpret_cast<float4*>(St + li * kChLd + 16 * w + 4 * lq) = make_float4(Sn[0], Sn[1], Sn[2], Sn[3]);
        __builtin_amdgcn_sched_barrier(0);
        load_decay(nx);
        __syncthreads();  // the new state is whole; K^T, R and U have been read
    };
    // The two kinds of wave run loops of their own with the same three barriers per chunk (a loop with branches kept
    // the loads of both alive in copies, and waited for them there).  Loads for the next chunk overwrite registers
    // behind their last use: the scheduling barriers keep them from being moved above it, which would need copies too.
    if (outputs) {  // wave-uniform
        for (int ch = 0; ch < chunks; ++ch) {
            if (ch > 0) output(ch - 1);
            __builtin_amdgcn_sched_barrier(0);
            const Rows cur = rows(ch), nx = rows(ch + 1);
            load_m(cur);
            load_gamma(cur);
            __syncthreads();
            Y = times_state();
            __builtin_amdgcn_sched_barrier(0);
            load_x(nx);
            update_state(nx);
        }
        output(chunks - 1);
    } else {
        for (int ch = 0; ch < chunks; ++ch) {
            const Rows nx = rows(ch + 1);
            __builtin_amdgcn_s_setprio(1);  // the chain that everything waits for
            // R_i = b_i (v_i - gamma_i X_i) (rows 16 wt + 4 lq + v, column li), stored transposed; K^T
            const floatx4 X = times_state();
#pragma unroll
            for (int st = 0; st < 32; ++st) Kt[(16 * (st >> 2) + 4 * lq + (st & 3)) * kChLdT + 16 * wt + li] = x[st];
            float r4[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) r4[v] = bet[v] * (v4[v] - gam[v] * X[v]);
            *reinterpret_cast<float4*>(Rt + li * kChLdT + 16 * wt + 4 * lq) = make_float4(r4[0], r4[1], r4[2], r4[3]);
            __builtin_amdgcn_sched_barrier(0);
            load_x(nx);
            load_values(nx);
            load_gamma(nx);
            __syncthreads();
            float rb[16];  // U = T R
#pragma unroll
            for (int u = 0; u < 4; ++u) ld4(Rt + li * kChLdT + 16 * u + 4 * lq, rb + 4 * u);
            __builtin_amdgcn_sched_barrier(0);
            const floatx4 U = times_rows(rb);
            *reinterpret_cast<float4*>(Ut + li * kChLdT + 16 * wt + 4 * lq) = make_float4(U[0], U[1], U[2], U[3]);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            load_m(nx);
            update_state(nx);
        }
    }
    for (int e = tid; e < 128 * 16; e += kStateThreads) {
        const int d = e >> 4, cc = e & 15;
        if (j0 + cc < dv) S[static_cast<size_t>(d) * dv + j0 + cc] = St[cc * kChLd + d];
    }
}

bool linear_scan_supported(int lk_n, int lk_hd, int lv_n, int lv_hd, int ksize) {
    return lk_n > 0 && lv_n > 0 && lv_n % lk_n == 0 && lk_hd > 0 && lk_hd <= 256 && lv_hd > 0 && ksize >= 1 &&
           ksize - 1 <= kScanMaxHist && lk_hd <= kScanIGroups * kScanMaxK;
}

hipError_t launch_linear_scan(const LinearScanLaunch& p, hipStream_t s) {
    if (p.ws && p.lk_hd == 128 && p.lv_hd <= 256) {
        if (p.lv_hd == 128 && p.ksize == 4) {
            hipLaunchKernelGGL(linear_conv_prefill_tg_kernel<4>,
                               dim3(2 * p.lk_n + p.lv_n, (p.tokens + kConvTokens - 1) / kConvTokens), dim3(128), 0, s, p);
        } else {
            const int width = max(p.lk_hd, p.lv_hd);
            hipLaunchKernelGGL(linear_conv_prefill_kernel, dim3(p.tokens, 2 * p.lk_n + p.lv_n),
                               dim3((width + kWave - 1) / kWave * kWave), 0, s, p);
        }
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        static bool attr_set = false;
        if (!attr_set) {
            if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_chunk_prep_kernel),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   static_cast<int>(scan_chunk_prep_lds()));
                e != hipSuccess)
                return e;
            if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&scan_chunk_state_kernel),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   static_cast<int>(scan_chunk_state_lds()));
                e != hipSuccess)
                return e;
            attr_set = true;
        }
        const int chunks = (p.tokens + kChunk - 1) / kChunk;
        hipLaunchKernelGGL(scan_chunk_prep_kernel, dim3(p.lv_n, chunks), dim3(256), scan_chunk_prep_lds(), s, p);
        if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
        hipLaunchKernelGGL(scan_chunk_state_kernel, dim3(p.lv_n, (p.lv_hd + 15) / 16), dim3(kStateThreads),
                           scan_chunk_state_lds(),
                           s, p);
        return hipGetLastError();
    }
    const dim3 grid(p.lv_n, (p.lv_hd + kScanCols - 1) / kScanCols);
    if (p.lk_hd == 128 && p.ksize == 4) {
        // four value columns per wave (two per wave, i.e. twice the blocks, measured
        // slower: every wave convolves the whole q/k head)
        const dim3 grid4(p.lv_n, (p.lv_hd + 15) / 16);
        hipLaunchKernelGGL((linear_scan_wave_kernel<128, 4, 4>), grid4, dim3(256), 0, s, p);
    }
    else
        hipLaunchKernelGGL(linear_scan_kernel, grid, dim3(256), 0, s, p);
    return hipGetLastError();
}

}  // namespace xqhip
