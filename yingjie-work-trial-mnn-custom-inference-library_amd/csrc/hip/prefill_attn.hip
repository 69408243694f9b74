// prefill_attn.hip - causal GQA of a prompt chunk on gfx950
// (custom_model.cpp:840-951 per token): prefill_attn_mfma_kernel on the matrix
// cores for heads of 128 and 256 dims, prefill_attn_kernel for every other
// shape or alignment.
#include <algorithm>

#include "xqhip_common.hpp"
#include "xqhip_kernels.hpp"

namespace xqhip {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef short short4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Causal GQA for a prompt chunk: a block takes query token t (position
// pos0 + t) and the `group` query heads of kv head kh over keys 0..pos0+t in
// 64-token chunks with a running max / sum (rescaled by exp(m_old - m_new)),
// then normalises by multiplying with 1/l and applies the sigmoid gate
// (custom_model.cpp:840-951 per token).
// ---------------------------------------------------------------------------
constexpr int kPAttnChunk = 64;
constexpr int kPAttnMaxGroup = 8;

// floats of LDS of attend_token
constexpr size_t attend_token_lds(int group, int hd) {
    return 2 * static_cast<size_t>(group) * hd + static_cast<size_t>(group) * (kPAttnChunk + 3);
}

// THREADS: of the block (a constant: blockDim would add the implicit arguments to every launch's)
template <int THREADS>
__device__ __forceinline__ void attend_token(const PrefillAttnLaunch& p, int t, int kh, float* smem) {
    static_assert(THREADS >= 4 * kPAttnChunk, "four threads per key");
    const int hd = p.head_dim, group = p.nq / p.nkv;
    const int ctx = *p.pos0 + t + 1;
    float* qs = smem;                        // [group][hd]
    float* sc = qs + group * hd;             // [group][64]
    float* osum = sc + group * kPAttnChunk;  // [group][hd] running output
    float* ml = osum + group * hd;           // [group][2] running max, sum
    float* fac = ml + 2 * group;             // [group] rescale of this chunk
    const float* qrow = p.q + static_cast<size_t>(t) * p.q_stride + static_cast<size_t>(kh) * group * hd;
    for (int i = threadIdx.x; i < group * hd; i += THREADS) {
        qs[i] = qrow[i];
        osum[i] = 0.0f;
    }
    if (threadIdx.x < group) {
        ml[2 * threadIdx.x] = -INFINITY;
        ml[2 * threadIdx.x + 1] = 0.0f;
    }
    __syncthreads();
    const float rscale = 1.0f / sqrtf(static_cast<float>(hd));
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    for (int c0 = 0; c0 < ctx; c0 += kPAttnChunk) {
        const int n = min(kPAttnChunk, ctx - c0);
        // scores: 4 threads per key, each a quarter of the dims
        {
            const int sub = threadIdx.x & 3, tt = threadIdx.x >> 2;
            const int dq = (hd + 3) / 4, d0 = sub * dq, d1 = min(hd, d0 + dq);
            const bool valid = tt < n;
            const _Float16* krow = p.k_cache + (static_cast<size_t>(c0 + (valid ? tt : 0)) * p.nkv + kh) * hd;
            for (int g = 0; g < group; ++g) {
                float dot = 0.0f;
                for (int d = d0; d < d1; ++d) dot += qs[g * hd + d] * static_cast<float>(krow[d]);
                dot = lanes_sum<4>(dot);
                if (valid && sub == 0) sc[g * kPAttnChunk + tt] = dot * rscale;
            }
        }
        __syncthreads();
        // online softmax update per head (one wave per head)
        for (int g = wid; g < group; g += THREADS / kWave) {
            const float sv = lane < n ? sc[g * kPAttnChunk + lane] : -INFINITY;
            const float mc = wave_max(sv);
            const float m_old = ml[2 * g];
            const float m_new = fmaxf(m_old, mc);
            const float e = lane < n ? expf(sv - m_new) : 0.0f;
            const float lsum = wave_sum(e);
            sc[g * kPAttnChunk + lane] = e;
            if (lane == 0) {
                const float f = expf(m_old - m_new);  // 0 for the first chunk
                fac[g] = f;
                ml[2 * g] = m_new;
                ml[2 * g + 1] = ml[2 * g + 1] * f + lsum;
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < group * hd; i += THREADS) {
            const int g = i / hd, d = i % hd;
            float o = osum[i] * fac[g];
            for (int j = 0; j < n; ++j)
                o += sc[g * kPAttnChunk + j] *
                     static_cast<float>(p.v_cache[(static_cast<size_t>(c0 + j) * p.nkv + kh) * hd + d]);
            osum[i] = o;
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < group * hd; i += THREADS) {
        const int g = i / hd;
        const float l = ml[2 * g + 1];
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
        const size_t oi = static_cast<size_t>(t) * p.out_stride + static_cast<size_t>(kh) * group * hd + i;
        const size_t gi = static_cast<size_t>(t) * p.q_stride + static_cast<size_t>(kh) * group * hd + i;
        p.out[oi] = (osum[i] * inv) * sigmoid_dev(p.gate[gi]);
    }
}

__global__ void __launch_bounds__(256) prefill_attn_kernel(PrefillAttnLaunch p) {
    extern __shared__ float smem[];
    attend_token<256>(p, blockIdx.x, blockIdx.y, smem);
}

// Matrix-core form.  A block takes 32 CT columns of one kv head, a column
// being one (token, query head) pair: column c is head c / T of the kv head's
// `group` and token t0 + c % T, T = 32 CT / group tokens.  CT x KS waves: wave
// (ct, ks) owns the 32 columns of tile ct and every KS-th 32-key tile, with
// its own running max / sum and output, merged through LDS at the end.  K and
// V are staged chunk by chunk (32 KS keys, shared by all column tiles), V
// loaded into registers while the scores are formed and K of the next chunk
// while the values are summed.
//
// Scores are formed transposed, S^T = K Q^T (keys are the MFMA rows): lane l
// holds column l & 31 and the keys 8 (v / 4) + 4 (l >> 5) + v % 4 of its tile,
// so a column's max is over the lane's own 16 values and lane l ^ 32, and its
// probabilities are already the B operand of O^T = V^T P^T (the MFMA's k index
// is a permutation of the keys shared by both operands).  V stays [key][dim]
// in LDS; ds_read_tr16_b64 hands each lane four keys of its dim.
//
// Precision: q (scaled per column by a power of two to [2^12, 2^13), exact)
// and p (relative to a reference within 2^6 of the column's running max, times
// 2^6) are split into fp16 hi + lo, about 22 bits together; k and v are fp16
// in the cache; fp32 accumulation.  (prefill_attn_kernel holds q and p in fp32; both are within 2^-22 of their
// value here, and the output, against 64 bits over normal data, is nearer: 2.8e-7 of its norm against 5.1e-7 at 333
// tokens after 512, 16 / 4 heads of 256.)
//
// A masked key has weight 0, but 0 times an infinity is not 0, and neither hi + lo nor the finite start of the running
// max can carry infinities or scores below -1e30.  Where that happens the output is not finite or its weights sum to
// 0: a block that finds such an output (one flag, read once at its end) computes its tokens again by attend_token.
//
// What bounds it: MFMA work is 8 pairs x hd x 2 passes of flops (q hi / lo, p hi
// / lo), 65 GFLOP at 512 tokens over 4096 keys and 32 heads; the 32-column
// tiles read each K / V fragment from LDS once per 512 MFMA cycles of a wave
// (half the LDS bandwidth), and the online softmax's VALU work is about as long
// as the MFMA work, so two waves per SIMD overlap the two.
//
// A short context's time is the chain around the keys.  q is read from memory once per block, in whole rows, and
// handed out through LDS: read by every wave in operand order (32 columns x 64 bytes an instruction) it took 3 us.
// Waves without a key neither write outputs nor are merged.
//
// Measured: 512 tokens after 3584, 32 / 8 heads of 128: 76 us (the kernel
// before, one wave per query head of 16 tokens with no key split, 181 us);
// 16 tokens after 0: 7.4 us (9.2; 10.7 with q in operand order and all eight
// waves merged); 333 tokens after 512, 16 / 4 heads of 256: 36.6 us
// (prefill_attn_kernel 3595 us).
constexpr int kFTile = 32;  // keys and columns of an MFMA tile

template <int HD, int CT, int KS>
struct FlashTile {
    static constexpr int kWaves = CT * KS, kThreads = kWave * kWaves;
    static constexpr int kCols = kFTile * CT, kKeys = kFTile * KS;
    static constexpr int kLdk = HD + 8;   // halves per K row: 16-byte rows shifted by 4 banks
    static constexpr int kLdv = HD + 16;  // halves per V row: the 4 rows of a transposed read in distinct banks
    static constexpr int kLdo = HD + 4;   // floats per column of a wave's output
    static constexpr int kRowPieces = HD / 8;
    static constexpr int kPieces = kKeys * kRowPieces / kThreads;  // 16-byte pieces of K (or V) per thread and chunk
    static constexpr int kTilePieces = kPieces / KS;               // ... and 32-key tile
    static constexpr int kQuads = HD / 4;                          // float4 of an output row
    static constexpr int kMergeCols = kThreads / kQuads;           // columns per pass of the merge
    static constexpr int kPasses = kCols / kMergeCols;
    static constexpr size_t kKvBytes = static_cast<size_t>(kKeys) * (kLdk + kLdv) * 2;
    static constexpr size_t kOutBytes = static_cast<size_t>(kWaves) * kFTile * (kLdo + 2) * 4;
    static constexpr size_t kLds = kKvBytes > kOutBytes ? kKvBytes : kOutBytes;
    static_assert(kTilePieces * KS * kThreads == kKeys * kRowPieces, "K / V staging");
    static_assert(kPasses * kThreads == kCols * kQuads, "merge");
    static_assert(kLds + 64 <= 160 * 1024, "LDS");
    static_assert(static_cast<size_t>(kKeys) * kLdk * 2 + static_cast<size_t>(kCols) * kLdo * 4 <= kLds, "q fits behind K");
    static_assert(kLds >= attend_token_lds(kPAttnMaxGroup, HD) * 4, "the general form runs in it");
};

// v[l ^ 32] paired with v[l]: the larger
__device__ __forceinline__ float half_wave_max(float v) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__builtin_bit_cast(float, static_cast<uint32_t>(r[0])),
                 __builtin_bit_cast(float, static_cast<uint32_t>(r[1])));
}

// fp32 -> fp16 hi + fp16 lo (x - hi) of 8 values
__device__ __forceinline__ void split_h8(const float (&x)[8], half8& hi, half8& lo) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const _Float16 h = static_cast<_Float16>(x[e]);
        hi[e] = h;
        lo[e] = static_cast<_Float16>(x[e] - static_cast<float>(h));
    }
}

template <int HD, int CT, int KS>
__global__ void __launch_bounds__(kWave * CT * KS, (CT * KS + 3) / 4) prefill_attn_mfma_kernel(PrefillAttnLaunch p, int tiles) {
    using F = FlashTile<HD, CT, KS>;
    constexpr int kSteps = HD / 16, kDimTiles = HD / 32;
    constexpr float kLog2e = 1.44269504088896340736f;
    constexpr float kRaise = 6.0f;  // p is held times 2^kRaise
    constexpr float kSlack = 6.0f;  // the max may outgrow the reference by 2^kSlack before it is moved
    extern __shared__ uint4 flash_lds[];
    __shared__ int redo;  // some output of the block is not finite
    _Float16* Kl = reinterpret_cast<_Float16*>(flash_lds);  // [kKeys][kLdk]
    _Float16* Vl = Kl + F::kKeys * F::kLdk;                 // [kKeys][kLdv]
    // the kv heads of a token tile are neighbours in launch order, so a head's blocks share an XCD's L2 (8
    // heads) and read its K / V from there; the tiles with the longest prefixes start first
    const int kh = blockIdx.x % p.nkv, tile = tiles - 1 - static_cast<int>(blockIdx.x) / p.nkv;
    const int group = p.nq / p.nkv, T = F::kCols / group;
    const int lane = threadIdx.x & (kWave - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int ct = wid % CT, ks = wid / CT;
    const int cl = lane & 31, g = lane >> 5;
    const int pos0 = __builtin_amdgcn_readfirstlane(*p.pos0);
    const uint32_t inv_t = (65535u + T) / T;  // c / T = c inv_t >> 16 for c < 64, T <= 64
    const int t0 = tile * T, ntok = min(T, p.tokens - t0);
    const int col = ct * kFTile + cl, ch = static_cast<int>(col * inv_t >> 16), ctok = col - ch * T;
    const bool live = ch < group && ctok < ntok;
    const int qpos = live ? pos0 + t0 + ctok : -1;           // this column's last key
    const int first = pos0 + t0, last = pos0 + t0 + ntok - 1;  // keys every / any column of the block sees

    // chunk pieces: i = threadIdx + kThreads u is key i / kRowPieces, dims 8 (i % kRowPieces) .. + 7
    const uint32_t krow = static_cast<uint32_t>(p.nkv) * HD * 2u;  // bytes per cache position
    const int pk = threadIdx.x / F::kRowPieces, pd = threadIdx.x % F::kRowPieces;
    constexpr int kKeyStep = F::kThreads / F::kRowPieces;
    u32x4 kr[F::kPieces], vr[F::kPieces];
    auto load = [&](const _Float16* cache, int c0, u32x4 (&r)[F::kPieces]) {  // keys past `last` read 0
        const int n = __builtin_amdgcn_readfirstlane(max(0, min(F::kKeys, last - c0 + 1)));
        const size_t base = static_cast<size_t>(__builtin_amdgcn_readfirstlane(max(0, min(c0, last)))) * p.nkv * HD +
                            static_cast<size_t>(kh) * HD;
        const __amdgpu_buffer_rsrc_t rs = buf_rsrc(cache + base, static_cast<uint32_t>(n) * krow);
#pragma unroll
        for (int u = 0; u < F::kPieces; ++u)
            r[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, static_cast<uint32_t>(pk + u * kKeyStep) * krow + pd * 16u,
                                                         0, 0);
    };
    auto store = [&](_Float16* d, int ld, const u32x4 (&r)[F::kPieces]) {
#pragma unroll
        for (int u = 0; u < F::kPieces; ++u)
            *reinterpret_cast<u32x4*>(d + (pk + u * kKeyStep) * ld + 8 * pd) = r[u];
    };
    // rows of q, the gate and the output: thread i takes float4 i % kQuads of columns i / kQuads, + kMergeCols, ...
    auto place = [&](int tid, int u, int stride) {  // float offset of the pass's column from token t0, or -1
        const int c = tid / F::kQuads + u * F::kMergeCols;
        const int hc = static_cast<int>(c * inv_t >> 16), tc = c - hc * T;
        return hc < group && tc < ntok ? tc * stride + (kh * group + hc) * HD + 4 * (tid % F::kQuads) : -1;
    };
    // q to LDS (V's, before it)
    u32x4 qr[F::kPasses];
    {
        const __amdgpu_buffer_rsrc_t rq =
            buf_rsrc(p.q + static_cast<size_t>(t0) * p.q_stride, static_cast<uint32_t>(ntok) * p.q_stride * 4u);
#pragma unroll
        for (int u = 0; u < F::kPasses; ++u) {  // columns without a token read 0
            const int at = place(threadIdx.x, u, p.q_stride);
            qr[u] = __builtin_amdgcn_raw_buffer_load_b128(rq, at >= 0 ? static_cast<uint32_t>(at) * 4u : kBufOOB, 0, 0);
        }
    }
    load(p.k_cache, 0, kr);
    // 256 dims: the first values with the first keys, one round trip less for a short context (16 / 4 heads, 2 tokens
    // after 0: 11.2 us, 12.5 without).  128 dims gain nothing there (7.5, 7.3 without) and lose 10 % on long contexts.
    if constexpr (HD > 128) load(p.v_cache, 0, vr);
    float* Ql = reinterpret_cast<float*>(Vl);  // [kCols][kLdo]
#pragma unroll
    for (int u = 0; u < F::kPasses; ++u)
        *reinterpret_cast<u32x4*>(Ql + (threadIdx.x / F::kQuads + u * F::kMergeCols) * F::kLdo +
                                  4 * (threadIdx.x % F::kQuads)) = qr[u];
    store(Kl, F::kLdk, kr);
    if (threadIdx.x == 0) redo = 0;
    __syncthreads();
    half8 qhi[kSteps], qlo[kSteps];  // lane supplies dims 16 s + 8 g .. + 7 of its column
    float sscale;                    // score scale in the exponent of 2
    {
        float x[kSteps][8], mx = 0.0f;
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                const float4 v = *reinterpret_cast<const float4*>(Ql + col * F::kLdo + 16 * s + 8 * g + e);
                x[s][e] = v.x;
                x[s][e + 1] = v.y;
                x[s][e + 2] = v.z;
                x[s][e + 3] = v.w;
            }
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[s][e]));
        mx = half_wave_max(mx);
        // a power of two brings the column's largest magnitude into [2^12, 2^13); an infinity or 0 stays
        int ex = 13;
        if (mx > 0.0f && mx < INFINITY) frexpf(mx, &ex);
        ex = max(ex, -100);  // 2^(13 - ex) stays finite
        const float down = ldexpf(1.0f, 13 - ex);
        sscale = ldexpf(kLog2e / sqrtf(static_cast<float>(HD)), ex - 13);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[s][e] *= down;
            split_h8(x[s], qhi[s], qlo[s]);
        }
    }
    __syncthreads();  // every wave has its q: V may take its place
    float m = -1.0e30f, l = 0.0f;  // reference of the exponents, this lane's part of the sum
    floatx16 o[kDimTiles];
#pragma unroll
    for (int j = 0; j < kDimTiles; ++j) o[j] = floatx16{};
    for (int c0 = 0; c0 <= last; c0 += F::kKeys) {  // block-uniform
        if (HD <= 128 || c0 > 0) load(p.v_cache, c0, vr);
        const int key0 = c0 + ks * kFTile;
        const bool any = key0 <= last;  // wave-uniform: this wave's tile holds a key
        half8 phi[2], plo[2];
        if (any) {
            floatx16 sh = floatx16{}, sl = floatx16{};
            const _Float16* krow_l = Kl + (ks * kFTile + cl) * F::kLdk + 8 * g;
#pragma unroll
            for (int s = 0; s < kSteps; ++s) {
                const half8 a = *reinterpret_cast<const half8*>(krow_l + 16 * s);
                sh = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qhi[s], sh, 0, 0, 0);
                sl = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qlo[s], sl, 0, 0, 0);
            }
            float sc[16], mc = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; ++v) sc[v] = sh[v] + sl[v];
            if (key0 + kFTile - 1 > first) {  // wave-uniform: the tile reaches past some column's last key
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (key0 + 8 * (v >> 2) + 4 * g + (v & 3) > qpos) sc[v] = -INFINITY;
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) mc = fmaxf(mc, sc[v]);
            mc = half_wave_max(mc) * sscale;
            // the reference moves only when a column's max has outgrown it (rarely after the first tiles)
            const bool up = mc > m + kSlack;
            if (__builtin_amdgcn_ballot_w64(up)) {
                const float to = up ? mc : m, f = exp2f(m - to);
                m = to;
                l *= f;
#pragma unroll
                for (int j = 0; j < kDimTiles; ++j) o[j] *= f;
            }
            const float off = kRaise - m;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    x[e] = __builtin_amdgcn_exp2f(fmaf(sc[8 * h + e], sscale, off));
                    l += x[e];
                }
                split_h8(x, phi[h], plo[h]);
            }
        }
        store(Vl, F::kLdv, vr);
        // block-uniform; 256 dims load on (past `last`: nothing is read): a branch around the loads costs them spilled
        // registers, one around the stores below none
        const bool more = c0 + F::kKeys <= last;
        if (HD > 128 || more) load(p.k_cache, c0 + F::kKeys, kr);
        __syncthreads();  // V is staged; every wave has read K
        if (any) {
            // transposed reads: 16 lanes cover four keys x 16 dims, lane i gets dim i of the four
            const _Float16* vb = Vl + (ks * kFTile + 4 * g + ((lane & 15) >> 2)) * F::kLdv + (lane & 16) + 4 * (lane & 3);
#pragma unroll
            for (int j = 0; j < kDimTiles; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    typedef __attribute__((address_space(3))) short4_t lds_s4;
                    const _Float16* q0 = vb + 16 * h * F::kLdv + 32 * j;
                    const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(q0));
                    const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(q0 + 8 * F::kLdv));
                    const half8 a = __builtin_bit_cast(half8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                    o[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, phi[h], o[j], 0, 0, 0);
                    o[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, plo[h], o[j], 0, 0, 0);
                }
        }
        if (more) store(Kl, F::kLdk, kr);
        __syncthreads();  // the next K is staged; every wave has read V
    }
    // merge the key splits of each column tile that have a key: outputs, then (reference, sum) of every wave's
    // columns.  The gates are requested before the outputs go to LDS, so that no load waits behind a store.
    const int splits = min(KS, last / kFTile + 1);
    const __amdgpu_buffer_rsrc_t rg =
        buf_rsrc(p.gate + static_cast<size_t>(t0) * p.q_stride, static_cast<uint32_t>(ntok) * p.q_stride * 4u);
    int mt = threadIdx.x;
    asm("" : "+v"(mt));  // (else the passes' places are kept from q's on, in registers that the loop needs)
    u32x4 gate[F::kPasses];
#pragma unroll
    for (int u = 0; u < F::kPasses; ++u) {
        const int at = place(mt, u, p.q_stride);
        gate[u] = __builtin_amdgcn_raw_buffer_load_b128(rg, at >= 0 ? static_cast<uint32_t>(at) * 4u : kBufOOB, 0, 0);
    }
    float* Ol = reinterpret_cast<float*>(flash_lds);  // [kWaves][32][kLdo]
    float* Ml = Ol + F::kWaves * kFTile * F::kLdo;    // [kWaves][32][2]
    l = xor_pair_sum<32>(l);
    if (ks < splits) {
        float* oc = Ol + (wid * kFTile + cl) * F::kLdo + 4 * g;
#pragma unroll
        for (int j = 0; j < kDimTiles; ++j)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                *reinterpret_cast<float4*>(oc + 32 * j + 8 * a) =
                    make_float4(o[j][4 * a], o[j][4 * a + 1], o[j][4 * a + 2], o[j][4 * a + 3]);
        if (g == 0) *reinterpret_cast<float2*>(Ml + (wid * kFTile + cl) * 2) = make_float2(m, l);
    }
    __syncthreads();
    bool bad = false;
#pragma unroll
    for (int u = 0; u < F::kPasses; ++u) {
        const int at = place(mt, u, p.out_stride);
        if (at < 0) continue;
        const int c = mt / F::kQuads + u * F::kMergeCols;
        const int w0 = (c / kFTile) * kFTile + (c % kFTile);  // column c of wave (ct, ks): w0 + ks CT 32
        float ml[KS], ll[KS], M = -INFINITY;
#pragma unroll
        for (int s = 0; s < KS; ++s)
            if (s < splits) {
                const float2 v = *reinterpret_cast<const float2*>(Ml + (w0 + s * F::kCols) * 2);
                ml[s] = v.x;
                ll[s] = v.y;
                M = fmaxf(M, v.x);
            }
        float L = 0.0f;
        float4 r = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int s = 0; s < KS; ++s)
            if (s < splits) {
                const float f = exp2f(ml[s] - M);
                const float4 v = *reinterpret_cast<const float4*>(Ol + (w0 + s * F::kCols) * F::kLdo + 4 * (mt % F::kQuads));
                L += f * ll[s];
                r.x += f * v.x;
                r.y += f * v.y;
                r.z += f * v.z;
                r.w += f * v.w;
            }
        const float inv = L > 0.0f ? 1.0f / L : 0.0f;  // custom_model.cpp:901-904
        bad |= !(L > 0.0f && fabsf(r.x) + fabsf(r.y) + fabsf(r.z) + fabsf(r.w) < INFINITY);
        *reinterpret_cast<float4*>(p.out + static_cast<size_t>(t0) * p.out_stride + at) =
            make_float4((r.x * inv) * sigmoid_dev(__uint_as_float(gate[u][0])),
                        (r.y * inv) * sigmoid_dev(__uint_as_float(gate[u][1])),
                        (r.z * inv) * sigmoid_dev(__uint_as_float(gate[u][2])),
                        (r.w * inv) * sigmoid_dev(__uint_as_float(gate[u][3])));
    }
    if (bad) redo = 1;
    // a barrier for the flag alone: __syncthreads() would wait for the output stores too (1 us)
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
    if (__builtin_expect(!redo, 1)) return;  // block-uniform
    __syncthreads();  // those stores, and every wave's reads of the LDS used again
    for (int t = t0; t < t0 + ntok; ++t) {
        attend_token<F::kThreads>(p, t, kh, reinterpret_cast<float*>(flash_lds));
        __syncthreads();
    }
}

bool prefill_attn_supported(int nq, int nkv, int head_dim) {
    return nkv > 0 && nq % nkv == 0 && nq / nkv <= kPAttnMaxGroup && head_dim > 0 &&
           sizeof(float) * attend_token_lds(nq / nkv, head_dim) <= 64 * 1024;
}

template <int HD, int CT, int KS>
static hipError_t launch_flash(const PrefillAttnLaunch& p, hipStream_t s) {
    using F = FlashTile<HD, CT, KS>;
    const auto fn = reinterpret_cast<const void*>(&prefill_attn_mfma_kernel<HD, CT, KS>);
    if (hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(F::kLds));
        e != hipSuccess)
        return e;
    const int T = F::kCols / (p.nq / p.nkv), tiles = (p.tokens + T - 1) / T;
    hipLaunchKernelGGL((prefill_attn_mfma_kernel<HD, CT, KS>), dim3(static_cast<unsigned>(tiles) * p.nkv),
                       dim3(F::kThreads), F::kLds, s, p, tiles);
    return hipGetLastError();
}

hipError_t launch_prefill_attn(const PrefillAttnLaunch& p, hipStream_t s) {
    const int group = p.nq / p.nkv;
    // the matrix-core kernel takes q, the gate and the output in 16-byte pieces, the caches in whole words
    const bool al16 = ((reinterpret_cast<uintptr_t>(p.q) | reinterpret_cast<uintptr_t>(p.gate) |
                        reinterpret_cast<uintptr_t>(p.out)) & 15u) == 0 && p.q_stride % 4 == 0 && p.out_stride % 4 == 0 &&
                      ((reinterpret_cast<uintptr_t>(p.k_cache) | reinterpret_cast<uintptr_t>(p.v_cache)) & 3u) == 0;
    const bool in32 = p.q_stride < 1 << 24 && p.out_stride < 1 << 24;  // offsets within a block's (at most 64) rows
    if (al16 && in32 && (p.head_dim == 128 || p.head_dim == 256)) {
        // two column tiles per block halve the K / V traffic per column; one tile with twice the key splits
        // where two would leave some of the 256 CUs without a block
        const bool wide = static_cast<long>((p.tokens + 64 / group - 1) / (64 / group)) * p.nkv >= 256;
        if (p.head_dim == 128) return wide ? launch_flash<128, 2, 4>(p, s) : launch_flash<128, 1, 8>(p, s);
        return wide ? launch_flash<256, 2, 2>(p, s) : launch_flash<256, 1, 4>(p, s);
    }
    const size_t lds = sizeof(float) * attend_token_lds(group, p.head_dim);
    hipLaunchKernelGGL(prefill_attn_kernel, dim3(p.tokens, p.nkv), dim3(256), lds, s, p);
    return hipGetLastError();
}

}  // namespace xqhip
