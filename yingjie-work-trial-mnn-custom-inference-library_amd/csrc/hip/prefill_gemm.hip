// prefill_gemm.hip - the W4A16 GEMM of a prompt chunk on gfx950: y[t] (op)= W
// prologue(x[t]) for up to a few hundred tokens at once, every token as
// gemvW4A16Neon does it (xq_gemv_w4a16_neon.cpp:259-291).
//   prep_x_kernel / prep_x_vec_kernel   per-token RMSNorm / gated head norm,
//                        x -> fp16 hi + lo in MFMA operand order, group sums
//   gemm_w4_mfma_kernel  the products on the matrix cores
//   gemm_splitk_reduce_kernel           adds the K splits of a split launch
#include <algorithm>
#include <type_traits>

#include "xqhip_common.hpp"
#include "xqhip_kernels.hpp"

namespace xqhip {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ uint32_t pack_h2(_Float16 lo, _Float16 hi) {
    return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, lo)) |
           (static_cast<uint32_t>(__builtin_bit_cast(uint16_t, hi)) << 16);
}

// ---------------------------------------------------------------------------
// Operand preparation: one block per token of x (row stride ldx) with the
// prologue applied (RMS over the row, or per-head gated norm with the gate row
// at t * ldz) -> v, stored as x_hi = fp16(v) and x_lo = fp16(v - x_hi) (about
// 22 significant bits together) in the order in which the GEMM's waves read
// them: per group of 64 columns and tile of 32 tokens 8 KiB, [hi | lo][step s
// 0..3][lane 0..63] 16-byte pieces, lane l holding token l & 31 and the columns
// 32 (l >> 5) + 8 s .. + 7 of the group in the order [0 4 1 5 2 6 3 7] (the
// order in which a word of 8 codes is unpacked).  xs[t][g] = fp32 sum of v over
// the group.  Each row is first scaled by a power of two, ts[t] = 2^k, that
// brings its largest magnitude into [2^12, 2^13): fp16 then holds any fp32
// activation (silu(gate) * up of a large residual stream can exceed 65504)
// without overflow or subnormal loss, and the GEMM multiplies its results by
// ts[t] (exact).  Rows m .. m_pad - 1 are zero-filled (ts 1).
// ---------------------------------------------------------------------------
constexpr int kPrepMaxHeads = 256;
// A row below 2^-114 is raised by 2^127, the largest power fp32 has: half the last fp16 bit is then 2^-152, less than
// fp32's own smallest value.
constexpr int kPrepMinExp = -114;
constexpr int kXTile = 512;  // 16-byte pieces of one group of a 32-token tile
constexpr int kXLo = 256;    // the x_lo pieces follow the x_hi ones

// Piece of (token t, group g) at word 0, in 16-byte units; tiles: 32-token tiles
__device__ __forceinline__ size_t x_piece(int t, int g, int tiles) {
    return (static_cast<size_t>(g) * tiles + (t >> 5)) * kXTile + (t & 31);
}
// offset of word w (columns 8 w .. 8 w + 7 of the group) from word 0
__device__ __forceinline__ int x_word(int w) { return (w & 3) * 64 + (w >> 2) * 32; }

// Token of this block.  Blocks are dealt to the 8 XCDs round robin; eight
// consecutive tokens, whose pieces share 128-byte lines, go to one XCD.
__device__ __forceinline__ int prep_token(int tokens) {
    const int b = blockIdx.x;
    return b < (tokens & ~63) ? (b & ~63) + 8 * (b & 7) + ((b >> 3) & 7) : b;
}

__global__ void __launch_bounds__(256) prep_x_kernel(const float* __restrict__ x, int ldx, int m, int cols,
                                                     Prologue pro, int ldz, uint4* __restrict__ xt,
                                                     float* __restrict__ xs, float* __restrict__ ts) {
    __shared__ float red[32];
    __shared__ float head_inv[kPrepMaxHeads];
    const int t = prep_token(gridDim.x);
    const int G = cols >> 6, nch = cols >> 3;
    uint4* xo = xt + x_piece(t, 0, gridDim.x / 32);
    const size_t gstride = static_cast<size_t>(gridDim.x / 32) * kXTile;
    float* os = xs + static_cast<size_t>(t) * G;
    if (t >= m) {
        for (int c = threadIdx.x; c < nch; c += blockDim.x) {
            uint4* d = xo + (c >> 3) * gstride + x_word(c & 7);
            d[0] = d[kXLo] = make_uint4(0u, 0u, 0u, 0u);
        }
        for (int g = threadIdx.x; g < G; g += blockDim.x) os[g] = 0.0f;
        if (threadIdx.x == 0) ts[t] = 1.0f;
        return;
    }
    const float* xr = x + static_cast<size_t>(t) * ldx;
    const float* zr = pro.mode == PRO_GATED ? pro.z + static_cast<size_t>(t) * ldz : nullptr;
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave, nw = blockDim.x / kWave;
    float inv = 1.0f;
    if (pro.mode == PRO_RMS) {
        float ss = 0.0f;
        for (int c = threadIdx.x; c < cols; c += blockDim.x) ss += xr[c] * xr[c];
        ss = block_sum(ss, red);
        inv = 1.0f / sqrtf(ss / static_cast<float>(cols) + pro.eps);
    } else if (pro.mode == PRO_GATED) {
        const int heads = cols / pro.head_dim;
        for (int h = wid; h < heads; h += nw) {  // one wave per head
            const float* xv = xr + h * pro.head_dim;
            float ss = 0.0f;
            for (int d = lane; d < pro.head_dim; d += kWave) ss += xv[d] * xv[d];
            ss = wave_sum(ss);
            if (lane == 0) head_inv[h] = 1.0f / sqrtf(ss / static_cast<float>(pro.head_dim) + pro.eps);
        }
        __syncthreads();
    }
    // one thread per 8 columns; the 8 threads of a group are consecutive lanes (nch % 8 == 0)
    auto load8 = [&](int c, float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = xr[c + e];
        if (pro.mode == PRO_RMS) {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = v[e] * inv * pro.w[c + e];
        } else if (pro.mode == PRO_GATED) {
            const int h = c / pro.head_dim, d = c - h * pro.head_dim;  // head_dim % 8 == 0
            const float ih = head_inv[h];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = v[e] * ih * pro.w[d + e] * silu_dev(zr[c + e]);
        }
    };
    // the row's power-of-two scale from its largest magnitude
    float mx = 0.0f;
    for (int c8 = threadIdx.x; c8 < nch; c8 += blockDim.x) {
        float v[8];
        load8(c8 * 8, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[e]));
    }
    mx = wave_max(mx);
    __syncthreads();  // red may still be read by the norm's block_sum
    if (lane == 0) red[wid] = mx;
    __syncthreads();
    for (int i = 0; i < nw; ++i) mx = fmaxf(mx, red[i]);
    int ex = 0;
    frexpf(mx, &ex);                                       // mx = f 2^ex, f in [0.5, 1)
    ex = max(ex, kPrepMinExp);
    const float down = mx > 0.0f ? ldexpf(1.0f, 13 - ex) : 1.0f;  // mx * down in [2^12, 2^13)
    if (threadIdx.x == 0) ts[t] = mx > 0.0f ? ldexpf(1.0f, ex - 13) : 1.0f;
    for (int c8 = threadIdx.x; c8 < nch; c8 += blockDim.x) {
        const int c = c8 * 8;
        float v[8];
        load8(c, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= down;
        uint32_t ph[4], pl[4];
        float sum = 0.0f;
#pragma unroll
        for (int p = 0; p < 4; ++p) {  // positions 2p, 2p + 1 <- columns p, p + 4
            const _Float16 ha = static_cast<_Float16>(v[p]), hb = static_cast<_Float16>(v[p + 4]);
            ph[p] = pack_h2(ha, hb);
            pl[p] = pack_h2(static_cast<_Float16>(v[p] - static_cast<float>(ha)),
                            static_cast<_Float16>(v[p + 4] - static_cast<float>(hb)));
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += v[e];
        uint4* d = xo + (c8 >> 3) * gstride + x_word(c8 & 7);
        d[0] = make_uint4(ph[0], ph[1], ph[2], ph[3]);
        d[kXLo] = make_uint4(pl[0], pl[1], pl[2], pl[3]);
        sum = lanes_sum<8>(sum);
        if ((c8 & 7) == 0) os[c8 >> 3] = sum;
    }
}

// The same for rows of NK * 2048 columns with 16-byte aligned rows, weights and
// gates, the prologue mode a template argument: thread i owns the 8-column
// pieces i, i + 256, ... of its token's row and loads each once, as 16-byte
// loads with no branch around them (the generic kernel reads the row three
// times, one float per load); the gated norm's per-head sums stay inside the
// 16 lanes that own a 128-column head.
template <int NK, int MODE>
__global__ void __launch_bounds__(256) prep_x_vec_kernel(const float* __restrict__ x, int ldx, int m, Prologue pro,
                                                         int ldz, uint4* __restrict__ xt, float* __restrict__ xs,
                                                         float* __restrict__ ts) {
    constexpr int kCols = NK * 2048, kG = kCols / 64;
    __shared__ float red_s[4], red_m[4];
    const int t = prep_token(gridDim.x);
    const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
    uint4* xo = xt + x_piece(t, 0, gridDim.x / 32);
    const size_t gstride = static_cast<size_t>(gridDim.x / 32) * kXTile;
    float* os = xs + static_cast<size_t>(t) * kG;
    if (t >= m) {  // block-uniform
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            const int c = threadIdx.x + 256 * k;
            uint4* d = xo + (c >> 3) * gstride + x_word(c & 7);
            d[0] = d[kXLo] = make_uint4(0u, 0u, 0u, 0u);
        }
        for (int g = threadIdx.x; g < kG; g += 256) os[g] = 0.0f;
        if (threadIdx.x == 0) ts[t] = 1.0f;
        return;
    }
    const float4* xr = reinterpret_cast<const float4*>(x + static_cast<size_t>(t) * ldx);
    float4 xv[NK][2], wv[NK][2], zv[NK][2];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        const int c4 = 2 * (threadIdx.x + 256 * k);  // float4 index of the piece
        xv[k][0] = xr[c4];
        xv[k][1] = xr[c4 + 1];
        if constexpr (MODE == PRO_RMS) {
            wv[k][0] = reinterpret_cast<const float4*>(pro.w)[c4];
            wv[k][1] = reinterpret_cast<const float4*>(pro.w)[c4 + 1];
        } else if constexpr (MODE == PRO_GATED) {
            // head_dim 128: the piece's offset in its head is 8 (i mod 16)
            const int d4 = 2 * (threadIdx.x & 15);
            wv[k][0] = reinterpret_cast<const float4*>(pro.w)[d4];
            wv[k][1] = reinterpret_cast<const float4*>(pro.w)[d4 + 1];
            const float4* zr = reinterpret_cast<const float4*>(pro.z + static_cast<size_t>(t) * ldz);
            zv[k][0] = zr[c4];
            zv[k][1] = zr[c4 + 1];
        }
    }
    float v[NK][8];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        const float4 a = xv[k][0], b = xv[k][1];
        v[k][0] = a.x; v[k][1] = a.y; v[k][2] = a.z; v[k][3] = a.w;
        v[k][4] = b.x; v[k][5] = b.y; v[k][6] = b.z; v[k][7] = b.w;
    }
    if constexpr (MODE == PRO_RMS) {
        float ss = 0.0f;
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += v[k][e] * v[k][e];
        ss = wave_sum(ss);
        if (lane == 0) red_s[wid] = ss;
        __syncthreads();
        ss = (red_s[0] + red_s[1]) + (red_s[2] + red_s[3]);
        const float inv = 1.0f / sqrtf(ss / static_cast<float>(kCols) + pro.eps);
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            const float w8[8] = {wv[k][0].x, wv[k][0].y, wv[k][0].z, wv[k][0].w,
                                 wv[k][1].x, wv[k][1].y, wv[k][1].z, wv[k][1].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) v[k][e] = v[k][e] * inv * w8[e];
        }
    } else if constexpr (MODE == PRO_GATED) {
#pragma unroll
        for (int k = 0; k < NK; ++k) {
            float ss = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += v[k][e] * v[k][e];
            ss = lanes_sum<16>(ss);  // the head's 16 pieces
            const float ih = 1.0f / sqrtf(ss / 128.0f + pro.eps);
            const float w8[8] = {wv[k][0].x, wv[k][0].y, wv[k][0].z, wv[k][0].w,
                                 wv[k][1].x, wv[k][1].y, wv[k][1].z, wv[k][1].w};
            const float z8[8] = {zv[k][0].x, zv[k][0].y, zv[k][0].z, zv[k][0].w,
                                 zv[k][1].x, zv[k][1].y, zv[k][1].z, zv[k][1].w};
#pragma unroll
            for (int e = 0; e < 8; ++e) v[k][e] = v[k][e] * ih * w8[e] * silu_dev(z8[e]);
        }
    }
    // the row's power-of-two scale from its largest magnitude
    float mx = 0.0f;
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(v[k][e]));
    mx = wave_max(mx);
    if (lane == 0) red_m[wid] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red_m[0], red_m[1]), fmaxf(red_m[2], red_m[3]));
    int ex = 0;
    frexpf(mx, &ex);
    ex = max(ex, kPrepMinExp);
    const float down = mx > 0.0f ? ldexpf(1.0f, 13 - ex) : 1.0f;
    if (threadIdx.x == 0) ts[t] = mx > 0.0f ? ldexpf(1.0f, ex - 13) : 1.0f;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        const int c8 = threadIdx.x + 256 * k;
        uint32_t ph[4], pl[4];
        float sum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[k][e] *= down;
#pragma unroll
        for (int q = 0; q < 4; ++q) {  // positions 2q, 2q + 1 <- columns q, q + 4
            const _Float16 ha = static_cast<_Float16>(v[k][q]), hb = static_cast<_Float16>(v[k][q + 4]);
            ph[q] = pack_h2(ha, hb);
            pl[q] = pack_h2(static_cast<_Float16>(v[k][q] - static_cast<float>(ha)),
                            static_cast<_Float16>(v[k][q + 4] - static_cast<float>(hb)));
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += v[k][e];
        uint4* d = xo + (c8 >> 3) * gstride + x_word(c8 & 7);
        d[0] = make_uint4(ph[0], ph[1], ph[2], ph[3]);
        d[kXLo] = make_uint4(pl[0], pl[1], pl[2], pl[3]);
        sum = lanes_sum<8>(sum);
        if ((c8 & 7) == 0) os[c8 >> 3] = sum;
    }
}

template <int NK>
static void launch_prep_vec(const GemmLaunch& p, int m_pad, uint4* xt, float* xs, float* ts, hipStream_t s) {
    if (p.pro.mode == PRO_RMS)
        hipLaunchKernelGGL((prep_x_vec_kernel<NK, PRO_RMS>), dim3(m_pad), dim3(256), 0, s, p.x, p.ldx, p.m, p.pro,
                           p.ldz, xt, xs, ts);
    else if (p.pro.mode == PRO_GATED)
        hipLaunchKernelGGL((prep_x_vec_kernel<NK, PRO_GATED>), dim3(m_pad), dim3(256), 0, s, p.x, p.ldx, p.m, p.pro,
                           p.ldz, xt, xs, ts);
    else
        hipLaunchKernelGGL((prep_x_vec_kernel<NK, PRO_NONE>), dim3(m_pad), dim3(256), 0, s, p.x, p.ldx, p.m, p.pro,
                           p.ldz, xt, xs, ts);
}

static bool prep_vec_ok(const GemmLaunch& p) {
    auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; };
    if (p.cols % 2048 != 0 || !al16(p.x) || p.ldx % 4 != 0) return false;
    if (p.pro.mode == PRO_RMS) return al16(p.pro.w);
    if (p.pro.mode == PRO_GATED) return p.pro.head_dim == 128 && al16(p.pro.w) && al16(p.pro.z) && p.ldz % 4 == 0;
    return p.pro.mode == PRO_NONE;
}

// ---------------------------------------------------------------------------
// y[t][r] (op)= sum_k w[r][k] x[t][k].
//
// In column group g (64 columns) a row's weights are w = sn s + c0 with
// sn = q - 8 the signed code, s the group scale and c0 = (8 - z) s for
// w = (q - z) s, or 8 s + z for w = q s + z.  Hence
//     y[t][r] = sum_g s[r][g] A[r][t][g] + sum_g c0[r][g] xs[t][g],
//     A[r][t][g] = sum_{k in g} sn[r][k] x[t][k],  xs[t][g] = sum_{k in g} x[t][k].
// 16 sn is exact in fp16, so 16 A takes two v_mfma_f32_32x32x16_f16 passes (x_hi and
// x_lo) into a per-group accumulator, which is scaled by s into the fp32
// result.  The c0 term is a K = G contraction done after the group loop in
// three fp16 hi/lo passes (c0 scaled by 64 and xs by 1/64, both exact, to stay
// in fp16 range), skipped where every zero is 8.
//
// Block: WGR x WGT waves, each owning TI x TJ tiles of 32 rows x 32 tokens.
// The tokens are the MFMA's rows and the weight rows its columns, so a lane
// holds one weight row: its scale is one register.  Everything the block reads
// goes straight from memory into LDS, XS - 1 groups ahead for x (an LDS image in
// operand order, read back one conflict-free KiB per fragment), two for the codes
// (two groups of a row at a time) and a quad of groups for the scales; one
// barrier per group, before the group's last step: the next group's first reads
// and the transfers that reuse its LDS run under that step's MFMAs, one transfer
// between two of them (with the barrier after the step and a group's transfers
// requested together: 12352x4096, 512 tokens 103 us, now 99; 10240 rows 95, now
// 90; 24576 rows 128 tokens 66, now 62.5).  A lane reads 16 bytes of codes per tile and group and
// unpacks a word of 8 with one shift, four three-input bit ops and four packed
// fp16 subtractions.  The LDS reads, the unpacking and the scaling of a finished
// group's sums are placed between the MFMAs.
//
// What bounds it: the MFMAs, at the clock that their power leaves.  gate/up (24576x4096, 512 tokens) issues 206 GFLOP in
// 188 us = 1.1 PFLOP/s, the matrix cores busy for 58 % of the cycles at 1.8 GHz (the card's clock is 2.4); a loop of
// nothing but these MFMAs on random operands runs at 1.35 PFLOP/s (2.2 on zeros).  Leaving out the unpacking, the
// scaling, the barriers or the LDS reads (timing only) changes it by at most 5 %.  The kernel before (weights as
// the row operand, 32-row waves that each read every token's fragments, x staged through registers) took 255 us.
// ---------------------------------------------------------------------------
constexpr int kGemmPad = 128;  // tokens are padded to at most a multiple of this
constexpr int kGemmMaxSplits = 8;
constexpr size_t kGemmPartMax = size_t{8} << 20;  // floats of partial products of one call

struct GemmArgs {
    const uint8_t* nib;
    const uint32_t* meta;
    int rows, cols, affine;
    int zero_is_8;    // c0 = (8 - z) s is 0 for every group: the c0 pass is skipped
    const uint4* xt;  // prepared x, [G][tiles][512] pieces
    const float* xs;  // [32 tiles][G]
    const float* ts;  // [32 tiles] per-token power-of-two scale of xt and xs
    int tiles;        // 32-token tiles (padded)
    int gps;          // column groups per K split, a multiple of 4
    float* part;      // split K: [splits][m][rows] partial products (the reduce applies the epilogue)
    int m;
    float* y;
    int ldy, epi;
};

template <int WGR, int WGT, int TI, int TJ, int XS>
struct GemmTile {
    static constexpr int kWaves = WGR * WGT, kThreads = kWave * kWaves;
    static constexpr int kBR = 32 * TI * WGR, kBT = 32 * TJ * WGT;
    static constexpr int kXU = kBT * 16 / kThreads;  // 16-byte pieces of x per thread and group
    static constexpr int kAU = kBR * 4 / kThreads;   // 16-byte pieces of codes per thread and half-quad
    static constexpr int kSU = kBR * 4 / kThreads;  // scales per thread and quad
    static constexpr int kXStage = kBT * 16;         // pieces per x stage
    static constexpr size_t kLds = 16 * (XS * static_cast<size_t>(kXStage) + 9 * static_cast<size_t>(kBR));
    static_assert(kXU * kThreads == kBT * 16 && kAU * kThreads == kBR * 4 && kSU * kThreads == kBR * 4, "staging");
};

// 8 stored codes (q ^ 8; column n of the word in bits 4n..4n+3) -> fp16 16 (q - 8),
// in the column order [0 4 1 5 2 6 3 7].  (w & 0x000F000F) ^ 0x74087408 is fp16
// 16384 + 16 q for codes 0 and 4 (one step of fp16 there is 16), (w & 0x00F000F0) ^
// 0x64806480 is 1024 + 16 q for codes 1 and 5, and w >> 8 gives the other four; both
// differences are exact.  The 16 leaves the sums once, at the end: x is the same
// fp16 pair in every column (held divided by 16 in the odd ones, for codes of q - 8
// and 16 (q - 8), its lo half met fp16's subnormals 16 times earlier beside an outlier).
template <int P>  // codes 2 P, 2 P + 1 of that order
__device__ __forceinline__ uint32_t unpack_pair(uint32_t w) {
    const uint32_t v = P & 2 ? w >> 8 : w;
    const _Float16 bias = static_cast<_Float16>(P & 1 ? 1152.0f : 16512.0f);
    const uint32_t m = P & 1 ? (v & 0x00F000F0u) ^ 0x64806480u : (v & 0x000F000Fu) ^ 0x74087408u;
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, m) - half2_t{bias, bias});
}

// 16 bytes per lane from a buffer straight into LDS, lane l to byte lds + 16 l (lds wave-uniform).  Written as asm
// because the compiler makes every LDS read after the builtin wait for all outstanding loads; it has no register
// output, and the kernel waits for its own transfers (wait_transfers) before the barrier that publishes them.
// The s_nop is the wait state a transfer needs behind a scalar write of m0 (the compiler adds it for the builtin, not
// inside an asm block).  Naming the reserved m0 as clobbered is sound here because nothing else in the kernel uses it:
// no builtin transfer, no indexed register move, no LDS access that is bounded by it.
__device__ __forceinline__ void buffer_to_lds16(u32x4 rsrc, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory", "m0");
}
// the same for 2 (zero-extended) or 4 bytes per lane, lane l to byte lds + 4 l
template <int BYTES>
__device__ __forceinline__ void buffer_to_lds(u32x4 rsrc, uint32_t voff, uint32_t soff, uint32_t lds) {
    if constexpr (BYTES == 2)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_ushort %1, %2, %3 offen lds"
                     :
                     : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                     : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                     :
                     : "s"(lds), "v"(voff), "s"(rsrc), "s"(soff)
                     : "memory", "m0");
}
// at most N of the wave's loads (transfers and register loads, in issue order) still outstanding
template <int N>
__device__ __forceinline__ void wait_transfers() {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ __forceinline__ u32x4 buf_words(const void* p, uint32_t bytes) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    return u32x4{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a))),
                 static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32))) & 0xffffu,
                 static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(bytes)), kBufWord3};
}

template <typename V>
__device__ __forceinline__ V lds_at(uint32_t byte) {
    return *reinterpret_cast<const __attribute__((address_space(3))) V*>(byte);
}

template <int WGR, int WGT, int TI, int TJ, int XS, int META>
__global__ void __launch_bounds__(kWave * WGR * WGT) __attribute__((amdgpu_waves_per_eu(TI * TJ <= 2 ? 4 : 2)))
gemm_w4_mfma_kernel(GemmArgs a) {
    constexpr uint32_t kMetaBytes = kMetaGroupBytes<META>;
    constexpr bool kSplits = WGR * WGT == 4;  // the 8-wave tile is never split over K (gemm_plan)
    using T = GemmTile<WGR, WGT, TI, TJ, XS>;
    constexpr int BR = T::kBR, BT = T::kBT, XU = T::kXU, AU = T::kAU, SU = T::kSU, NT = T::kThreads;
    extern __shared__ u32x4 gemm_lds[];
    // LDS: x [XS stages][kXStage], codes [BR][8], metadata words of the quad's groups [BR]
    // Tile of this block.  Blocks are dealt to the 8 XCDs round robin in
    // launch order; a weight slab (BR rows of one K split, a "unit") is read
    // by every token tile, so the token tiles of a unit are given launch
    // indices b = 8 k + (unit mod 8) and share one XCD's L2: the weights come
    // from memory once instead of once per XCD.  Units past the last multiple
    // of 8 keep the plain order.
    int tt, unit;
    {
        const int nt = gridDim.x;
        const int b = blockIdx.x + nt * (blockIdx.y + gridDim.y * blockIdx.z);
        const int units8 = (gridDim.y * gridDim.z) & ~7;
        if (b < units8 * nt) {
            const int k = b >> 3;
            unit = (k / nt) * 8 + (b & 7);
            tt = k % nt;
        } else {
            const int b2 = b - units8 * nt;
            unit = units8 + b2 / nt;
            tt = b2 % nt;
        }
    }
    const int split = unit / static_cast<int>(gridDim.y);
    const int t0 = tt * BT, r0 = (unit - split * static_cast<int>(gridDim.y)) * BR;
    const int G = a.cols >> 6;
    // this block's column groups: [g0, g1) of K split `split`, g0 a multiple of 4
    const int g0 = split * a.gps, g1 = min(G, g0 + a.gps), glast = g1 - 1;
    const uint32_t row_bytes = static_cast<uint32_t>(a.cols) >> 1;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int lr = lane & 31, lh = lane >> 5;
    const int wr = (wid / WGT) * 32 * TI, wj = (wid % WGT) * TJ;  // the wave's first row and token tile in the block

    // x of a group: piece tid + NT j of the block's image, one transfer per wave and j
    const u32x4 x_r = buf_words(a.xt, static_cast<uint32_t>(a.tiles) * 32u * a.cols * 4u);
    const uint32_t x_group = static_cast<uint32_t>(a.tiles) * kXTile * 16u;  // bytes per group
    const uint32_t x_tile = static_cast<uint32_t>(t0 >> 5) * kXTile * 16u;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        reinterpret_cast<__attribute__((address_space(3))) uint8_t*>(reinterpret_cast<uintptr_t>(gemm_lds)))) ;
    auto load_x = [&](int g, int st, int j) {
        buffer_to_lds16(x_r, static_cast<uint32_t>(tid) * 16u, static_cast<uint32_t>(g) * x_group + x_tile + NT * 16u * j,
                        lds0 + (st * T::kXStage + wid * kWave + NT * j) * 16u);
    };

    // codes, two groups (half a quad) at a time: LDS row r (64 bytes) of half-quad p holds in slot n the piece
    // n ^ ((r >> 2) & 3), piece = 2 half + group (the swizzle keeps the pieces eight neighbouring rows read in
    // distinct banks).  Pieces past a row's last group are whatever follows it, rows past the end 0: neither is used.
    const u32x4 nib_r = buf_words(a.nib, static_cast<uint32_t>(a.rows) * row_bytes);
    const int lastc = (G - 1) >> 6, gc_last = G - (lastc << 6);
    const int apiece = (tid ^ (tid >> 4)) & 3;
    const uint32_t aoff = static_cast<uint32_t>(r0 + (tid >> 2)) * row_bytes + (apiece & 1) * 16u;
    // (the whole offset in the vector operand: the range check must see all of it)
    auto load_a = [&](int g, int hq, int j) {  // half-quad hq of the quad at g
        const int c = g >> 6;
        const uint32_t half = static_cast<uint32_t>(c == lastc ? gc_last : 64) * 16u;
        const uint32_t off = aoff + (apiece & 2 ? half : 0u) + static_cast<uint32_t>(c) * 2048u + ((g & 63) + 2 * hq) * 16u;
        buffer_to_lds16(nib_r, off + (NT / 4) * j * row_bytes, 0,
                        lds0 + (XS * T::kXStage + hq * BR * 4 + wid * kWave + NT * j) * 16u);
    };
    // scales: word i = tid + NT j is group i & 3 of the quad, row i >> 2
    const u32x4 meta_w = buf_words(a.meta, meta_total_bytes<META>(static_cast<uint32_t>(a.rows), static_cast<uint32_t>(G)));
    const uint32_t soff = (static_cast<uint32_t>(r0 + (tid >> 2)) * G + (tid & 3)) * kMetaBytes;
    auto load_s = [&](int g, int j) {
        buffer_to_lds<META == 2 ? 2 : 4>(meta_w, soff + static_cast<uint32_t>(g + (NT / 4) * j * G) * kMetaBytes, 0,
                                         lds0 + (XS * T::kXStage + 8 * BR) * 16u + (wid * kWave + NT * j) * 4u);
    };
    // One MFMA step (16 of the group's 64 columns) multiplies every tile pair by x_hi and x_lo, in a fixed
    // order with the next step's LDS reads and unpacking between the MFMAs; a group's sums are scaled into the
    // result from its last step to the next group's first, tile by tile before the tile's sums start again from 0.
    u32x4 cw[2][TI];    // codes of the group and of the next
    u32x4 sq[TI];       // metadata words of the quad
    float sv[2][TI];    // scales of the group and of the one before
    half8 xf[2][TJ][2]; // x_hi, x_lo fragments of this step and the next
    u32x4 cf[2][TI];    // unpacked codes of this step and the next
    floatx16 acc[TI][TJ], t[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = t[i][j] = floatx16{};
    // LDS addresses of the lane, one register each (opaque: the compiler otherwise keeps one per read, hoisted out
    // of the loop); everything else is a constant offset
    uint32_t x16 = lds0 + (wj * kXTile + lane) * 16u;
    const uint32_t arow = lds0 + XS * T::kXStage * 16u + (wr + lr) * 64u;
    uint32_t a_even = arow + ((2 * lh) ^ ((lr >> 2) & 3)) * 16u, a_odd = arow + ((2 * lh + 1) ^ ((lr >> 2) & 3)) * 16u;
    uint32_t s16 = lds0 + (XS * T::kXStage + 8 * BR + wr + lr) * 16u;
    asm("" : "+v"(x16), "+v"(a_even), "+v"(a_odd), "+v"(s16));
    auto read_x = [&](int st, int s, int b) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const uint32_t at = x16 + (st * T::kXStage + s * 64 + j * kXTile) * 16u;
            xf[b][j][0] = lds_at<half8>(at);
            xf[b][j][1] = lds_at<half8>(at + kXLo * 16u);
        }
    };
    auto read_codes = [&](int u) {
#pragma unroll
        for (int i = 0; i < TI; ++i) cw[u & 1][i] = lds_at<u32x4>((u & 1 ? a_odd : a_even) + ((u >> 1) * BR + 32 * i) * 64u);
    };
    auto read_scales = [&] {
#pragma unroll
        for (int i = 0; i < TI; ++i) sq[i] = lds_at<u32x4>(s16 + 512u * i);
    };
    auto set_scale = [&](int u, bool in) {  // groups past g1 get scale 0
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            const float v = META == 1 || META == 3 ? __uint_as_float(sq[i][u]) : half_lo(sq[i][u]);
            sv[u & 1][i] = in ? v : 0.0f;
        }
    };
    auto scale_in = [&](int n, int part, int b) {  // a quarter of tile pair n
        const int i = n / TJ, j = n % TJ;
#pragma unroll
        for (int v = 4 * part; v < 4 * part + 4; ++v) acc[i][j][v] = fmaf(sv[b][i], t[i][j][v], acc[i][j][v]);
    };
    auto unpack = [&](int b, int p, int s, int n) {  // piece n of step s's unpacking: word n / 4
        const int i = n >> 2;
        const uint32_t w = cw[p][i][s];
        switch (n & 3) {
            case 0: cf[b][i][0] = unpack_pair<0>(w); break;
            case 1: cf[b][i][1] = unpack_pair<1>(w); break;
            case 2: cf[b][i][2] = unpack_pair<2>(w); break;
            default: cf[b][i][3] = unpack_pair<3>(w); break;
        }
    };
    const floatx16 zero = floatx16{};

    constexpr int NP = TI * TJ, NM = 2 * NP;  // tile pairs, MFMAs per step (each pair's hi and lo)
    // Quarter part of a pair's sums goes into the result before this MFMA, counted from the group's last step
    // on: from two MFMAs after the pair's last one up to its first one of the next group, spread evenly.
    auto scale_slot = [](int pair, int part) {
        const int s0 = 2 * pair + 3 + part * (NM - 2) / 4, s1 = NM + 2 * pair;
        return s0 < s1 ? s0 : s1;
    };
    static_assert(XS == 2 || XS == 4, "the stage of a group is a constant of its place in the quad");
#pragma unroll
    for (int j = 0; j < SU; ++j) load_s(g0, j);
#pragma unroll
    for (int j = 0; j < 2 * AU; ++j) load_a(g0, j / AU, j % AU);
#pragma unroll
    for (int e = 0; e < (XS - 1) * XU; ++e) load_x(min(g0 + e / XU, glast), e / XU, e % XU);
#pragma unroll
    for (int i = 0; i < TI; ++i) sv[1][i] = 0.0f;
    wait_transfers<0>();
    __syncthreads();
    // A group's phase runs from the barrier before its first reads to the next.  It requests the x that is XS - 1
    // groups ahead (the stage was last read before the barrier), then the next quad's scales (u = 0) or half of its
    // codes (u odd), whose LDS was last read before it too, at most one transfer before each MFMA.
    auto request = [&](int g, int u, int slot) {  // slot: MFMAs of the phase before
        const int gq = min((g & ~3) + 4, glast & ~3);
#pragma unroll
        for (int j = 0; j < XU; ++j)
            if (slot == j) load_x(min(g + XS - 1, glast), (u + XS - 1) % XS, j);
#pragma unroll
        for (int j = 0; j < SU; ++j)
            if (u == 0 && slot == XU + j) load_s(gq, j);
#pragma unroll
        for (int j = 0; j < AU; ++j)
            if ((u & 1) && slot == XU + j) load_a(gq, u >> 1, j);
    };
    static_assert(XU + AU <= 4 * NM && XU + SU <= 4 * NM, "every request within the phase");
    read_x(0, 0, 0);
    read_scales();
    read_codes(0);
    __syncthreads();  // the first scales are read before the next are requested
#pragma unroll
    for (int n = 0; n < NM; ++n) request(g0, 0, n);
#pragma unroll
    for (int n = 0; n < 4 * TI; ++n) unpack(0, 0, 0, n);
    for (int g = g0; g < g1; g += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {  // group g + u (past g1: scales 0), x stage u % XS
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int b = k & 1;
                if (k == 1) read_codes((u + 1) & 3);
                if (k == 2) set_scale(u, g + u < g1);
                if (k == 2 && u == 3) read_scales();
                if (k < 3) {
                    read_x(u % XS, k + 1, b ^ 1);
                } else {
                    // All of the group's x is in registers: the barrier, and the next group's first reads under this
                    // step's MFMAs.  Landed before it: the next group's x, the codes requested in the phase before
                    // (each has had XS - 1 or two phases' time), the scales (three phases').
                    if constexpr (XS == 2) {
                        if (u == 0) wait_transfers<SU>();
                        else if (u == 2) wait_transfers<0>();
                        else wait_transfers<AU>();
                    } else {
                        if (u == 0) wait_transfers<XU + SU>();
                        else if (u == 1) wait_transfers<2 * XU + SU + AU>();
                        else if (u == 2) wait_transfers<XU>();
                        else wait_transfers<2 * XU + AU>();
                    }
                    __syncthreads();
                    read_x((u + 1) % XS, 0, b ^ 1);
                }
#pragma unroll
                for (int n = 0; n < NM; ++n) {
                    const int pair = n >> 1, i = pair / TJ, j = pair % TJ;
                    if (k == 3) request(g + u + 1, (u + 1) & 3, n);
                    else request(g + u, u, NM * (k + 1) + n);
                    if (k == 3 || k == 0) {
#pragma unroll
                        for (int q = 0; q < 4 * NP; ++q)
                            if (scale_slot(q >> 2, q & 3) == (k == 0 ? NM : 0) + n) scale_in(q >> 2, q & 3, (k == 0 ? u + 1 : u) & 1);
                    }
                    if (k == 0 && (n & 1) == 0) t[i][j] = zero;
                    t[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(xf[b][j][n & 1], __builtin_bit_cast(half8, cf[b][i]),
                                                                     t[i][j], 0, 0, 0);
                    // the next step's codes, spread over this step's MFMAs
#pragma unroll
                    for (int q = 0; q < 4 * TI; ++q)
                        if (q * NM / (4 * TI) == n) unpack(b ^ 1, k == 3 ? (u + 1) & 1 : u & 1, (k + 1) & 3, q);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4 * NP; ++q)
        if (scale_slot(q >> 2, q & 3) >= NM) scale_in(q >> 2, q & 3, 1);
    wait_transfers<0>();  // the last phase's requests, which nothing reads
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] *= 0.0625f;  // the codes' 16

    // c0 term: K = G, lane half h takes groups gb + 8 h + 0..7 of its token / row.  All loads of a step are
    // issued before any use; groups past g1 read out of range (zero), so c0 and xs are 0.
    const __amdgpu_buffer_rsrc_t meta_r =
        buf_rsrc(a.meta, meta_total_bytes<META>(static_cast<uint32_t>(a.rows), static_cast<uint32_t>(G)));
    const __amdgpu_buffer_rsrc_t xs_r = buf_rsrc(a.xs, static_cast<uint32_t>(a.tiles) * 32u * G * 4u);
    for (int gb = g0; gb < (a.zero_is_8 ? g0 : g1); gb += 16) {
        const int g8 = gb + 8 * lh;
        MetaWord<META> mw[TI][8];
        uint32_t xw[TJ][8];
#pragma unroll
        for (int i = 0; i < TI; ++i) {
            const uint32_t row = static_cast<uint32_t>(min(r0 + wr + 32 * i + lr, a.rows - 1));
            const uint32_t off = (row * G + static_cast<uint32_t>(g8)) * kMetaBytes;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool in = g8 + e < g1;
                const uint32_t o = in ? off + kMetaBytes * e : kBufOOB;
                const uint32_t zo =
                    META == 3 && in ? z4_offset(static_cast<uint32_t>(a.rows), static_cast<uint32_t>(G), row,
                                                static_cast<uint32_t>(g8 + e))
                                    : kBufOOB;
                mw[i][e] = load_meta<META, 0>(meta_r, o, zo);
            }
        }
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const uint32_t off = (static_cast<uint32_t>(t0 + 32 * (wj + j) + lr) * G + static_cast<uint32_t>(g8)) * 4u;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                xw[j][e] = __builtin_amdgcn_raw_buffer_load_b32(xs_r, g8 + e < g1 ? off + 4u * e : kBufOOB, 0, 0);
        }
        half8 ch[TI], cl[TI], sh[TJ], so[TJ];
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float sc = meta_scale(mw[i][e]);
                const float z = meta_zero_at(mw[i][e], static_cast<uint32_t>((g8 + e) & 7) * 4u);
                const float c0 = 64.0f * (a.affine ? fmaf(8.0f, sc, z) : (8.0f - z) * sc);
                ch[i][e] = static_cast<_Float16>(c0);
                cl[i][e] = static_cast<_Float16>(c0 - static_cast<float>(ch[i][e]));
            }
#pragma unroll
        for (int j = 0; j < TJ; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = __builtin_bit_cast(float, xw[j][e]) * 0.015625f;
                sh[j][e] = static_cast<_Float16>(v);
                so[j][e] = static_cast<_Float16>(v - static_cast<float>(sh[j][e]));
            }
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sh[j], cl[i], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(so[j], ch[i], acc[i][j], 0, 0, 0);
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(sh[j], ch[i], acc[i][j], 0, 0, 0);
            }
    }

    // epilogue: lane holds row lr of tile i and the tokens 8 (v >> 2) + 4 lh + (v & 3) of tile j
    auto finish = [&](auto whole) {  // whole: every row and token of the block exists
        constexpr bool kWhole = decltype(whole)::value;
        const bool part = kSplits && a.part, pair = a.epi == 2 && !part, add = a.epi == 1 && !part;
        const size_t ld = part ? static_cast<size_t>(a.rows) : static_cast<size_t>(a.ldy);
        float* out = part ? a.part + static_cast<size_t>(split) * a.m * a.rows : a.y;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int tb = t0 + 32 * (wj + j) + 4 * lh;
            float4 ts4[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) ts4[q] = *reinterpret_cast<const float4*>(a.ts + tb + 8 * q);
#pragma unroll
            for (int i = 0; i < TI; ++i) {
                const int r = r0 + wr + 32 * i + lr;
                const bool rin = kWhole || r < a.rows;
                float* yr = out + static_cast<size_t>(tb) * ld + (pair ? r >> 1 : r);
                float val[16], old[16];
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const float4 f = ts4[v >> 2];
                    val[v] = acc[i][j][v] * ((v & 3) == 0 ? f.x : (v & 3) == 1 ? f.y : (v & 3) == 2 ? f.z : f.w);
                }
                if (pair) {  // interleaved (gate, up) rows -> silu(gate) * up
#pragma unroll
                    for (int v = 0; v < 16; ++v) val[v] = silu_dev(val[v]) * dpp_f32<kDppXor1>(val[v]);
                } else if (add) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int dt = 8 * (v >> 2) + (v & 3);
                        old[v] = kWhole || (rin && tb + dt < a.m) ? yr[dt * ld] : 0.0f;
                    }
#pragma unroll
                    for (int v = 0; v < 16; ++v) val[v] = old[v] + val[v];
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int dt = 8 * (v >> 2) + (v & 3);
                    if ((kWhole || (rin && tb + dt < a.m)) && (!pair || (lr & 1) == 0)) yr[dt * ld] = val[v];
                }
            }
        }
    };
    if (t0 + BT <= a.m && r0 + BR <= a.rows) finish(std::true_type{});  // block-uniform
    else finish(std::false_type{});
}

// y[t][r] (op)= sum over splits z (in order) of part[z][t][r]; op: store, add, or 2:
// the interleaved (gate, up) rows' silu(gate) * up.
// A thread takes V consecutive rows of a token (V the largest of 4, 2, 1 that divides
// rows: every load is then aligned to its size), all splits' loads in flight.
template <int V>
__global__ void __launch_bounds__(256) gemm_splitk_reduce_kernel(const float* __restrict__ part, int splits, int m,
                                                                 int rows, float* __restrict__ y, int ldy, int op) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const int r = (blockIdx.x * 256 + threadIdx.x) * V, t = blockIdx.y;
    if (r >= rows) return;
    const size_t n = static_cast<size_t>(m) * rows, at = static_cast<size_t>(t) * rows + r;
    float* yp = y + static_cast<size_t>(t) * ldy + (op == 2 ? r >> 1 : r);
    vec p[kGemmMaxSplits];
    float old[V];
#pragma unroll
    for (int z = 0; z < kGemmMaxSplits; ++z)
        if (z < splits) p[z] = *reinterpret_cast<const vec*>(part + z * n + at);
#pragma unroll
    for (int e = 0; e < V; ++e) old[e] = op == 1 ? yp[e] : 0.0f;
    vec s = p[0];
#pragma unroll
    for (int z = 1; z < kGemmMaxSplits; ++z)
        if (z < splits) s += p[z];
    if (op == 2) {
#pragma unroll
        for (int e = 0; e < V; e += 2) yp[e >> 1] = silu_dev(s[e]) * s[e + 1];
        return;
    }
#pragma unroll
    for (int e = 0; e < V; ++e) yp[e] = op == 1 ? old[e] + s[e] : s[e];
}

bool gemm_supported(int rows, int cols, int group, int layout, const Prologue& pro) {
    if ((layout != 0 && layout != 2 && layout != 3 && layout != 4) || group != 64 || cols % 64 != 0 || cols / 64 > 256 ||
        rows <= 0)
        return false;
    if (pro.mode == PRO_GATED)
        return pro.head_dim > 0 && pro.head_dim % 8 == 0 && cols % pro.head_dim == 0 &&
               cols / pro.head_dim <= kPrepMaxHeads;
    return true;
}


static size_t gemm_prep_bytes(int m, int cols) {
    const size_t m_pad = static_cast<size_t>((m + kGemmPad - 1) / kGemmPad) * kGemmPad;
    return m_pad * static_cast<size_t>(cols) * (2 * sizeof(_Float16)) +
           m_pad * static_cast<size_t>(cols / 64) * sizeof(float) + m_pad * sizeof(float);
}

// Grows with m and with rows, so that a workspace sized for a chunk's most
// tokens and widest matrix serves every smaller call (gemm_plan keeps the
// partial products of a split launch, which fewer tokens or rows can split
// into more, within both bounds).
size_t gemm_workspace_bytes(int m, int cols, int rows) {
    const size_t all = static_cast<size_t>(kGemmMaxSplits) * m * std::max(0, rows);
    return gemm_prep_bytes(m, cols) + (std::min(all, kGemmPartMax) * sizeof(float) + 255) / 256 * 256;
}

template <int WGR, int WGT, int TI, int TJ, int XS, int META>
static hipError_t launch_gemm_cfg(const GemmArgs& a, int splits, hipStream_t s) {
    using T = GemmTile<WGR, WGT, TI, TJ, XS>;
    const auto fn = reinterpret_cast<const void*>(&gemm_w4_mfma_kernel<WGR, WGT, TI, TJ, XS, META>);
    if constexpr (T::kLds > 64 * 1024) {  // beyond the default dynamic-LDS limit (gfx950 has 160 KiB per CU)
        if (hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(T::kLds));
            e != hipSuccess)
            return e;
    }
    const dim3 grid((a.m + T::kBT - 1) / T::kBT, (a.rows + T::kBR - 1) / T::kBR, splits);
    hipLaunchKernelGGL((gemm_w4_mfma_kernel<WGR, WGT, TI, TJ, XS, META>), grid, dim3(T::kThreads), T::kLds, s, a);
    return hipGetLastError();
}

template <int WGR, int WGT, int TI, int TJ, int XS>
static hipError_t launch_gemm_tile(const GemmArgs& a, int meta, int splits, hipStream_t s) {
    switch (meta) {
        case 0: return launch_gemm_cfg<WGR, WGT, TI, TJ, XS, 0>(a, splits, s);
        case 1: return launch_gemm_cfg<WGR, WGT, TI, TJ, XS, 1>(a, splits, s);
        case 2: return launch_gemm_cfg<WGR, WGT, TI, TJ, XS, 2>(a, splits, s);
        default: return launch_gemm_cfg<WGR, WGT, TI, TJ, XS, 3>(a, splits, s);
    }
}

enum GemmTileKind { kTileSmall, kTileMid, kTileLarge };
struct GemmPlan {
    GemmTileKind tile;
    int bt, splits, gps;  // tokens per block, K splits, column groups per split (a multiple of 4)
};

// us that a block spends on a group of 64 columns where `blocks` share the CUs: a part for each block of the fullest
// CU and a part for the load of the whole chip (memory, power).  Fitted to 2000 launches: 512 to 24600 rows, 1024 to
// 12288 columns, 2 to 512 tokens, every tile and split.  3 small or 2 middle blocks are resident on a CU at once.
static double group_us(GemmTileKind tile, long blocks) {
    const double per_cu = blocks / 256.0, n = static_cast<double>((blocks + 255) / 256);
    if (tile == kTileMid) return 0.22 + 0.48 * n + 0.35 * per_cu;
    if (tile == kTileLarge) return 0.05 + 1.02 * n + 0.43 * per_cu;
    return n == 1 ? 0.30 + 0.11 * per_cu : n == 2 ? 0.37 + 0.16 * per_cu : n == 3 ? 0.43 + 0.23 * per_cu : 0.16 * n + 0.18 * per_cu;
}

// Tile and K splits of a launch: the least time by group_us, a split launch with its second kernel and the partial
// products' traffic added.  That kernel adds the splits in a fixed order: deterministic.
//   128 rows x 32 tokens (4 waves): the most blocks, no padding of short prompts.
//   256 x 64 (4 waves): half the LDS reads per product.
//   256 x 128 (8 waves, one block per CU): half the x again, where one round of blocks covers the launch.  Never
//     split: with fewer blocks than CUs to split for, the middle tile has twice as many.
// Measured, us with prep and reduce (small, middle, large tile; splits in brackets), the choice first:
//   4096x4096, 8 tokens: small 15.4 (8), 24.5 (1).            24576x4096, 64: small 41.5 (1), 46.1 (2), middle 44.0 (2)
//   24576x4096, 300: middle 118.6, small 160, large 182.       12352x4096, 512: large 99.5, middle 109, small 142
//   24576x4096, 512: middle 181, large 195, small 246.         4096x12288, 512: middle 114 (2), 152 (1), small 136
//   10240x10240, 128: middle 68 (3), 122 (1), small 88.
// Over 240 sizes the choice is 1 % behind the fastest tile and split on average, 8 % at most.
static GemmPlan gemm_plan(int rows, int m, int cols) {
    const int G = cols / 64;
    auto blocks = [&](int br, int bt) { return static_cast<long>((m + bt - 1) / bt) * ((rows + br - 1) / br); };
    struct Option { GemmTileKind tile; int br, bt, splits; };
    GemmPlan best{};
    double least = 1.0e30;
    for (const Option& o : {Option{kTileSmall, 128, 32, kGemmMaxSplits}, Option{kTileMid, 256, 64, 4}, Option{kTileLarge, 256, 128, 1}})
        for (int s = 1; s <= std::min(o.splits, std::max(1, G / 8)); ++s) {  // at least two quads of groups per split
            if (s > 1 && static_cast<size_t>(s) * m * rows > kGemmPartMax) break;  // the workspace's bound
            const int gps = ((G + s - 1) / s + 3) / 4 * 4, splits = (G + gps - 1) / gps;
            const double t = (gps + 5) * group_us(o.tile, blocks(o.br, o.bt) * splits) +  // 5: a block's start and end
                             (splits > 1 ? 2.5 + 2.5e-6 * splits * m * rows : 0.0);
            if (t < least) {
                least = t;
                best = GemmPlan{o.tile, o.bt, splits, gps};
            }
        }
    return best;
}

hipError_t launch_gemm(const GemmLaunch& p, hipStream_t s) {
    const GemmPlan plan = gemm_plan(p.rows, p.m, p.cols);
    const int m_pad = (p.m + plan.bt - 1) / plan.bt * plan.bt;
    uint4* xt = static_cast<uint4*>(p.workspace);
    float* xs = reinterpret_cast<float*>(xt + static_cast<size_t>(m_pad) * (p.cols / 4));
    float* ts = xs + static_cast<size_t>(m_pad) * (p.cols / 64);
    // one instance per width up to 12288, the widest in use; 10240 columns, 2 tokens, RMS: the launches take 19.3 us,
    // 25.0 with the general kernel
    switch (prep_vec_ok(p) ? p.cols / 2048 : 0) {
        case 1: launch_prep_vec<1>(p, m_pad, xt, xs, ts, s); break;
        case 2: launch_prep_vec<2>(p, m_pad, xt, xs, ts, s); break;
        case 3: launch_prep_vec<3>(p, m_pad, xt, xs, ts, s); break;
        case 4: launch_prep_vec<4>(p, m_pad, xt, xs, ts, s); break;
        case 5: launch_prep_vec<5>(p, m_pad, xt, xs, ts, s); break;
        case 6: launch_prep_vec<6>(p, m_pad, xt, xs, ts, s); break;
        default:
            hipLaunchKernelGGL(prep_x_kernel, dim3(m_pad), dim3(256), 0, s, p.x, p.ldx, p.m, p.cols, p.pro, p.ldz, xt, xs, ts);
    }
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    float* part = plan.splits > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(p.workspace) +
                                                             gemm_prep_bytes(p.m, p.cols)) : nullptr;
    GemmArgs a{p.nib, static_cast<const uint32_t*>(p.meta), p.rows, p.cols, p.affine, p.zero_is_8, xt, xs, ts,
               m_pad / 32, plan.gps, part, p.m, p.y, p.ldy, p.epi};
    // metadata form: 0 fp16 (scale, zero), 1 fp32 pair (layout 2), 2 fp16 scale, zero 8 (layout 3),
    // 3 fp32 scale and 4-bit zero (layout 4)
    const int meta = p.layout == 2 ? 1 : (p.layout == 3 ? 2 : (p.layout == 4 ? 3 : 0));
    hipError_t e = hipErrorInvalidValue;
    switch (plan.tile) {
        case kTileSmall: e = launch_gemm_tile<4, 1, 1, 1, 4>(a, meta, plan.splits, s); break;
        case kTileMid: e = launch_gemm_tile<4, 1, 2, 2, 2>(a, meta, plan.splits, s); break;
        case kTileLarge: e = launch_gemm_tile<4, 2, 2, 2, 2>(a, meta, plan.splits, s); break;
    }
    if (e != hipSuccess || plan.splits == 1) return e;
    const int v = p.rows % 4 == 0 ? 4 : 2 - p.rows % 2;
    const dim3 grid((p.rows + 256 * v - 1) / (256 * v), p.m);
    if (v == 4)
        hipLaunchKernelGGL(gemm_splitk_reduce_kernel<4>, grid, dim3(256), 0, s, part, plan.splits, p.m, p.rows, p.y, p.ldy, p.epi);
    else if (v == 2)
        hipLaunchKernelGGL(gemm_splitk_reduce_kernel<2>, grid, dim3(256), 0, s, part, plan.splits, p.m, p.rows, p.y, p.ldy, p.epi);
    else
        hipLaunchKernelGGL(gemm_splitk_reduce_kernel<1>, grid, dim3(256), 0, s, part, plan.splits, p.m, p.rows, p.y, p.ldy, p.epi);
    return hipGetLastError();
}

}  // namespace xqhip
