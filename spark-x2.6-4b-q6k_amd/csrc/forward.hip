/* forward.hip — one decode token through the whole model on gfx950: the
 * embedding row, every layer's norm / attention / MLP around the library's
 * matvecs, the final norm and the tied-head logits.
 *
 * Semantics are the reference's CPU forward (tools/vq-runtime/src/
 * model.rs:441-591), which its GPU runtime mirrors launch by launch
 * (tools/vq/gpu/vq-model-gpu.cu:776-835):
 *
 *   h = embed[token]
 *   per layer:  xn = rms_norm(h, in_norm)                  (f64 sum of squares)
 *               [q k v] = qkv xn ; g = attn_gate xn
 *               rope over the first head_dim * partial elements of each q, k head
 *               K[pos], V[pos] = k, v
 *               per head: softmax over the layer's window of q.K/sqrt(hd), times V,
 *                         times sigmoid(g[head])
 *               h += out attn
 *               xn = rms_norm(h, post_norm)
 *               h += down (gelu(gate xn) * (up xn))        (exact erf gelu)
 *   logits = embed rms_norm(h, norm)                        (tied head)
 *
 * The matvecs are the library's own (VQ trunk, VQ or Q8_0 head). The
 * elementwise kernels here are small and latency-bound: one token is a few
 * thousand values. What matters for them is a short chain, so rope and the
 * KV store are one launch, and the norms and activations write the
 * matvecs' input in the form they read (f32, or bf16 when the model runs its
 * matvecs on bf16 activations). Activations stay f32 between kernels.
 *
 * The token and position live in device memory (two ints the chain's first
 * launch sets), and every kernel that depends on them reads them there: the
 * embedding row, rope and the KV row, the attention window. The chain's
 * launches are then the same for every token, so it is recorded once as a
 * HIP graph and replayed per token (sparkmv_model_capture / _replay); each
 * attention launch is shaped for its longest window.
 */
#include "act.h"
#include "kq.h"
#include "model.h"
#include "prefill.h"
#include "vq.h"

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <vector>

#include "../../include/sparkmv.h"

namespace sparkmv {

/* f32 -> bf16, round to nearest even (NaN stays NaN) */
__device__ __forceinline__ uint16_t fw_bf16(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t) ((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t) (u >> 16);
}

__global__ void fw_fill_kernel(float * p, int n, float v) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += blockDim.x * gridDim.x) p[i] = v;
}

/* st[0] = token, st[1] = position, and the position's rope tables for the
 * full and the sliding layers (model.rs:416-428, f32): tab[r][0][i] = cos,
 * tab[r][1][i] = sin of pos * theta_r^(-2i / pdim_r), i < pdim_r / 2 <= 128. */
__global__ void fw_set_state_kernel(int * st, int token, int pos, float theta0, int pdim0, float theta1, int pdim1,
                                    float * tab) {
    const int i = threadIdx.x;
    if (i == 0) {
        st[0] = token;
        st[1] = pos;
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const float theta = r ? theta1 : theta0;
        const int pdim = r ? pdim1 : pdim0;
        if (i < pdim / 2) {
            const float freq = 1.0f / powf(theta, (float) (2 * i) / (float) pdim);
            const float a = (float) pos * freq;
            tab[r * 256 + i] = cosf(a);
            tab[r * 256 + 128 + i] = sinf(a);
        }
    }
}

/* The embedding row of a Q8_0 tied head: row st[0], d * q exactly. */
__global__ void fw_q8_0_row_kernel(const uint8_t * blocks, int cols, const int * st, float * out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= cols) return;
    const uint8_t * b = blocks + ((size_t) st[0] * (cols >> 5) + (i >> 5)) * 34;
    _Float16 d;
    __builtin_memcpy(&d, b, 2);
    out[i] = (float) d * (float) (int8_t) b[2 + (i & 31)];
}

/* out = x * inv * w with inv = 1 / sqrt(mean(x^2) + eps), the sum of squares in
 * f64 and inv rounded once to f32 (model.rs:236-245). One workgroup. */
template <int PER>
__global__ __launch_bounds__(256) void fw_rmsnorm_kernel(const float * x, const float * w, float * out,
                                                         uint16_t * out16, int n, float eps) {
    __shared__ double part[4];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    /* workgroup b normalizes column b (a verify block's tokens) */
    x += (size_t) blockIdx.x * n;
    if (out) out += (size_t) blockIdx.x * n;
    if (out16) out16 += (size_t) blockIdx.x * n;
    /* x and w of this thread's elements requested together: one memory
     * round trip before the reduction */
    float xv[PER], wv[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int i = t + 256 * k;
        xv[k] = i < n ? x[i] : 0.0f;
        wv[k] = i < n ? w[i] : 0.0f;
    }
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < PER; k++) s += (double) xv[k] * (double) xv[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) part[wave] = s;
    __syncthreads();
    const double tot = (part[0] + part[1]) + (part[2] + part[3]);
    const float inv = (float) (1.0 / sqrt(tot / (double) n + (double) eps));
#pragma unroll
    for (int k = 0; k < PER; k++) {
        const int i = t + 256 * k;
        if (i < n) {
            const float v = xv[k] * inv * wv[k];
            if (out) out[i] = v;
            if (out16) out16[i] = fw_bf16(v);
        }
    }
}

/* ---- attention of one token, or of a verify block of up to 8 ----
 * Softmax attention over the layer's window of the cache (model.rs:505-557;
 * window 0: every position), split by positions over workgroups whose
 * partial results a second launch combines:
 *
 *   fw_attn_split_kernel: workgroup (split, kv head, 16 columns). The window's
 *     positions are cut into tiles of 16 and split s takes `per` consecutive
 *     tiles, per = ceil(tiles / nsplit): one tile each up to 16 * nsplit
 *     positions, so a short window still spreads over the chip, and a long one
 *     costs nsplit partials per head whatever its length. Columns that read a
 *     kv head's rows run together on the f32 matrix cores: column t * G + g is
 *     token t (of N) and query head g of the group's G, at most 32. More than
 *     16 take a second workgroup, which finds K and V in a cache: both blocks
 *     in one workgroup was slower in short windows (a block of 8 at position
 *     20: 8.6 us, 6.4 now; the four-layer call 336 -> 329, 330 with a
 *     workgroup per 16 positions and token) and in long ones (6001: 22.3 us
 *     and 19.8).
 *   fw_attn_combine_kernel: per (head, token), rescales the partials to their
 *     overall reference M, divides by L = sum_s l_s e^(m_s - M) and applies the
 *     head's sigmoid gate.
 *
 * The split kernel's four waves share each tile by head elements: wave w
 * contracts elements DW w .. DW w + DW - 1 (DW = HD / 4) of K against Q
 * (S^T = K Q^T, positions x columns), the four partial scores meet in LDS
 * (one barrier per tile, two buffers), every wave forms the same weights and
 * adds its own elements of O^T += V^T P^T. So one tile takes a quarter of a
 * wave's matrix time, which a short window needs, and a wave holds only
 * DW / 2 registers per tile of K and V, which lets the next tile be in flight
 * under this one, which a long window needs (two tiles ahead: 45.3 -> 47.0 us
 * at 30000 positions).
 *
 * Operand layout (lane 16 g + c), as in the prompt kernel below: a lane
 * reads its K row c as runs of 4 elements (k-step ks contracts element
 * 16 (ks / 4) + 4 g + ks % 4 of the wave's range), holds the scores of
 * positions 4 g + i for column c, and reads elements VW c .. + VW - 1
 * (VW = DW / 16) of the V rows 4 g + ks: O^T block r holds element
 * VW (4 g + i) + r of column c.
 *
 * The weights are exp(score - m) for a reference m per column that moves only
 * when a score passes it by more than kPaLag (the prompt kernel's rule): the
 * quotient does not depend on m, and most tiles skip the rescale.
 *
 * DEC (one decode token): position and rope tables come from device memory
 * (the state kernel's), the kernel rotates its query heads itself, and the
 * split whose tile ends at pos rotates the new key, uses it and the new value
 * from LDS, and stores both in the cache (model.rs:498-503); no other split
 * reads row pos, which before the store may hold anything. The launch shape
 * is fixed by the longest window, so a captured graph serves every position:
 * splits past the current window do nothing.
 *
 * Otherwise (a block): queries and keys are rotated and every key and value
 * is in the cache. A tile that some column sees only in part (causal end or
 * window start) must not weight a hidden V row by zero when it holds an
 * infinity or NaN; such a tile adds its rows one by one instead.
 *
 * What bounds it: HBM at long context (8 KB per position, read once, 5.2
 * TB/s); latency at short. Measured with four kv heads of 256 elements
 * (before: a workgroup per 16 positions, a wave per query head and token, all
 * partials combined by four waves per head): one token at position 30007 70 +
 * 56 -> 47 + 4.7 us (partials + combine), at 1003 9.4 + 4.7 -> 7.4 + 4.6, a
 * 512-position window 7.5 + 4.7 -> 6.1 + 4.6; a block of 8 at 6001 79 + 13 ->
 * 20 + 4.8, its 512-position windows 10.2 + 4.8 -> 7.9 + 4.1.
 * kAttnSplits: 64 against 128 costs the split kernel 1.7 us at 30007 and saves
 * every combine 0.6; 256 splits 54 + 6.3 at 30007. */
constexpr int kAttnChunk = 16;     /* positions per tile */
constexpr int kAttnSplits = 64;    /* partials per head and token, at most */
constexpr float kPaLag = 8.0f;     /* how far a score may pass the reference maximum */

struct AttnArgs {
    const float * qkv;   /* [N][ldq]: q, k, v of each token */
    float * kc, * vc;    /* the layer's cache rows [max_ctx][kvd] */
    const int * st;      /* DEC: token, position */
    const float * rtab;  /* DEC: the position's rope table [cos, sin][128] */
    float * po, * pml;   /* partials: [N * heads][nsplit][HD], [N * heads][nsplit][m, l] */
    int ldq, qd, kvd, pos0, N, window, heads, kv_heads, pdim, nsplit;
    float scale;
};

/* the splits of a window of n positions: tiles per split */
__host__ __device__ __forceinline__ int attn_per(int n, int nsplit) {
    const int tiles = (n + kAttnChunk - 1) / kAttnChunk;
    return (tiles + nsplit - 1) / nsplit;
}

template <int HD, int DEC>
__global__ __launch_bounds__(256, 2) void fw_attn_split_kernel(const AttnArgs A) {
    constexpr int DW = HD / 4, KQ = DW / 16, VW = DW / 16, QS = HD + 4;
    typedef float f4v __attribute__((ext_vector_type(4)));
    typedef float vv __attribute__((ext_vector_type(VW)));
    __shared__ __attribute__((aligned(16))) float lq[16 * QS];
    __shared__ f4v ls[2][4][64];
    __shared__ __attribute__((aligned(16))) float lkv[DEC ? 2 * HD : 4];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int pos = DEC ? A.st[1] : A.pos0, N = DEC ? 1 : A.N, kvh = blockIdx.y;
    const int G = A.heads / A.kv_heads, kvd = A.kvd;
    const int pfirst = A.window > 0 && pos + 1 > A.window ? pos + 1 - A.window : 0;
    const int plast = pos + N - 1, n = plast - pfirst + 1;
    const int per = attn_per(n, A.nsplit), ntile = (n + kAttnChunk - 1) / kAttnChunk;
    const int tb = blockIdx.x * per, te = min(tb + per, ntile);
    if (tb >= ntile) return;   /* uniform: the combine reads splits < ceil(ntile / per) */
    const bool newest = DEC && te == ntile;
    /* rows past the last stored one repeat it */
    const int rlast = DEC ? max(pos - 1, 0) : plast;
    const int d0 = DW * wave;
    const float * kb = A.kc + (size_t) kvh * HD + d0 + 4 * g;
    const float * vb = A.vc + (size_t) kvh * HD + d0 + VW * c;
    f4v kf[2][KQ];
    vv vf[2][4];
    auto fetch = [&](int tile, int s) {
        const int p = pfirst + kAttnChunk * min(tile, te - 1);
        const float * kp = kb + (size_t) min(p + c, rlast) * kvd;
#pragma unroll
        for (int j = 0; j < KQ; j++) kf[s][j] = *(const f4v *) (kp + 16 * j);
#pragma unroll
        for (int ks = 0; ks < 4; ks++) vf[s][ks] = *(const vv *) (vb + (size_t) min(p + 4 * g + ks, rlast) * kvd);
    };
    fetch(tb, 0);
    __builtin_amdgcn_sched_barrier(0);
    /* the queries (rows past the last column repeat it), from column col0 on */
    const int ncol = N * G, col0 = DEC ? 0 : 16 * (int) blockIdx.z;
    if constexpr (DEC) {
        /* rotated here (model.rs:416-438): element e < half pairs with
         * e + half, e in [half, 2 half) with e - half */
        const int half = A.pdim / 2, rows = newest ? G + 2 : G;
        constexpr int PER = (6 * HD + 255) / 256;   /* G <= 4 query rows, the new key and value */
        float x[PER], y[PER], cs[PER], sn[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = tid + 256 * k, r = min(i / HD, rows - 1), e = i & (HD - 1);
            const float * src = A.qkv + (r < G ? (size_t) (kvh * G + r) * HD : (size_t) A.qd + (size_t) (r - G) * kvd + (size_t) kvh * HD);
            const int q = e < half ? e : (e < 2 * half ? e - half : 0);
            x[k] = src[e];
            y[k] = src[e < half ? e + half : (e < 2 * half ? e - half : e)];
            cs[k] = A.rtab[q];
            sn[k] = A.rtab[128 + q];
        }
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int i = tid + 256 * k, r = i / HD, e = i & (HD - 1);
            if (r >= rows) continue;
            float v = x[k];
            if (r <= G && e < 2 * half) v = e < half ? x[k] * cs[k] - y[k] * sn[k] : x[k] * cs[k] + y[k] * sn[k];
            if (r < G) {
                lq[r * QS + e] = v;
            } else {
                lkv[(r - G) * HD + e] = v;
                float * dst = r == G ? A.kc : A.vc;
                dst[(size_t) pos * kvd + (size_t) kvh * HD + e] = v;
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < 16 * HD / 4 / 256; k++) {
            const int i = tid + 256 * k, col = min(col0 + i / (HD / 4), ncol - 1), e = 4 * (i & (HD / 4 - 1));
            const int t = col / G, h = kvh * G + col - t * G;
            *(f4v *) (lq + (i / (HD / 4)) * QS + e) = *(const f4v *) (A.qkv + (size_t) t * A.ldq + (size_t) h * HD + e);
        }
    }
    __syncthreads();
    const int col = min(col0 + c, ncol - 1);
    float qv[4 * KQ];
#pragma unroll
    for (int j = 0; j < KQ; j++) {
        const f4v q4 = *(const f4v *) (lq + (DEC ? col : c) * QS + d0 + 16 * j + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) qv[4 * j + i] = q4[i];
    }
    const int pos_t = pos + col / G, start_t = A.window > 0 && pos_t + 1 > A.window ? pos_t + 1 - A.window : 0;
    /* positions every column sees: the tiles inside need no mask */
    const int allfirst = A.window > 0 && plast + 1 > A.window ? plast + 1 - A.window : 0;
    f4v o[VW];
    float m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int r = 0; r < VW; r++) o[r] = f4v{0.f, 0.f, 0.f, 0.f};
    auto step = [&](int tile, int s) {
        const int p = pfirst + kAttnChunk * tile;
        const bool edge = p + kAttnChunk > pos + (DEC ? 0 : 1) || p < allfirst;   /* uniform */
        if (DEC && edge) {
            /* the last tile: row pos is the new key and value. Rows past it
             * weigh zero, as their scores are masked, and their values are
             * zero too: the new value again would add 0 times its infinities */
            if (p + c >= pos) {
#pragma unroll
                for (int j = 0; j < KQ; j++) kf[s][j] = *(const f4v *) (lkv + d0 + 16 * j + 4 * g);
            }
#pragma unroll
            for (int ks = 0; ks < 4; ks++) {
                const int pp = p + 4 * g + ks;
                if (pp >= pos) vf[s][ks] = pp == pos ? *(const vv *) (lkv + HD + d0 + VW * c) : (vv) 0.0f;
            }
        }
        /* this wave's elements of S^T in four chains: two round often enough
         * at the size of the score to show in sharp weights (deviation 12 at
         * position 20000: a token's row 1.08e-6 from 64 bits, 6.8e-7 with four
         * and 8.6e-7 with a lane-local dot and butterfly per score) */
        f4v sa[4];
#pragma unroll
        for (int i = 0; i < 4; i++) sa[i] = f4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KQ; j++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                sa[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s][j][i], qv[4 * j + i], sa[i], 0, 0, 0);
        ls[s][wave][lane] = (sa[0] + sa[1]) + (sa[2] + sa[3]);
        __syncthreads();
        const f4v sc = (ls[s][0][lane] + ls[s][1][lane]) + (ls[s][2][lane] + ls[s][3][lane]);
        float e[4];
        float mc = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int pp = p + 4 * g + i;
            e[i] = !edge || (pp >= start_t && pp <= pos_t) ? sc[i] * A.scale : -INFINITY;
            mc = fmaxf(mc, e[i]);
        }
        if (__any(mc > m + kPaLag)) {   /* uniform, and the same in every wave */
            mc = fmaxf(mc, __shfl_xor(mc, 16, 64));
            mc = fmaxf(mc, __shfl_xor(mc, 32, 64));
            const float mn = fmaxf(m, mc);
            const float a = mn == -INFINITY ? 1.0f : expf(m - mn);   /* nothing seen yet: no rescale */
            l *= a;
#pragma unroll
            for (int r = 0; r < VW; r++) o[r] *= a;
            m = mn;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            e[i] = e[i] == -INFINITY ? 0.0f : expf(e[i] - m);
            l += e[i];
        }
        if constexpr (!DEC) {
            bool bad = false;
            if (edge) {
#pragma unroll
                for (int ks = 0; ks < 4; ks++)
#pragma unroll
                    for (int r = 0; r < VW; r++) bad = bad || !__builtin_isfinite(vf[s][ks][r]);
            }
            if (edge && __any(bad)) {
                /* a hidden row may hold an infinity or NaN: row by row, hidden rows left out */
#pragma unroll 1
                for (int q = 0; q < 4; q++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const int pp = p + 4 * q + k;
                        const float * vr = A.vc + (size_t) min(pp, rlast) * kvd + (size_t) kvh * HD + d0 + 4 * VW * g;
                        const float w = __shfl(e[k], 16 * q + c, 64);
                        if (pp >= start_t && pp <= pos_t)
#pragma unroll
                            for (int i = 0; i < 4; i++)
#pragma unroll
                                for (int r = 0; r < VW; r++) o[r][i] += w * vr[VW * i + r];
                    }
                return;
            }
        }
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
#pragma unroll
            for (int r = 0; r < VW; r++)
                o[r] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[s][ks][r], e[ks], o[r], 0, 0, 0);
    };
    /* tile t in slot and score buffer (t - tb) & 1, the next one requested
     * before it is worked (past the end the last one again: a branch between
     * the loads would make the waits for this tile cover them too) */
    for (int t = tb; t < te;) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (t < te) {
                __builtin_amdgcn_sched_barrier(0);
                fetch(t + 1, u ^ 1);
                __builtin_amdgcn_sched_barrier(0);
                step(t, u);
            }
            t++;
        }
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (col0 + c >= ncol) return;
    const int t = col / G, h = kvh * G + col - t * G;
    const size_t at = ((size_t) t * A.heads + h) * A.nsplit + blockIdx.x;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        vv v;
#pragma unroll
        for (int r = 0; r < VW; r++) v[r] = o[r][i];
        *(vv *) (A.po + at * HD + d0 + VW * (4 * g + i)) = v;
    }
    if (wave == 0 && g == 0) {
        A.pml[2 * at] = m;
        A.pml[2 * at + 1] = l;
    }
}

/* The combine of (head blockIdx.x, token blockIdx.y): M = max m_s, L = sum_s
 * l_s e^(m_s - M), wave w summing e^(m_s - M) o_s over splits
 * w, w + 8, ... in increasing order, then the waves' sums in wave order, over
 * L, times the head's sigmoid gate. All of the partials' vectors that a wave
 * needs are requested at once (kPre each, kAttnSplits in all), behind the m
 * and l loads whose reductions they overlap: one memory round trip. */
template <int VPL>
__global__ __launch_bounds__(512) void fw_attn_combine_kernel(const AttnArgs A, int dec, const float * gate, int ldg,
                                                              float * out, uint16_t * out16) {
    constexpr int HD = 64 * VPL, W = 8, kPre = kAttnSplits / W;
    typedef float fv __attribute__((ext_vector_type(VPL)));
    __shared__ float wts[kAttnSplits];
    __shared__ fv acc[W][64];
    __shared__ float red;
    const int h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float gl = gate[(size_t) t * ldg + h];
    const int pos = dec ? A.st[1] : A.pos0, N = dec ? 1 : A.N;
    const int pfirst = A.window > 0 && pos + 1 > A.window ? pos + 1 - A.window : 0;
    const int n = pos + N - pfirst, per = attn_per(n, A.nsplit);
    const int ns = ((n + kAttnChunk - 1) / kAttnChunk + per - 1) / per;
    const size_t row = (size_t) t * A.heads + h, at = row * A.nsplit;
    static_assert(kAttnSplits == 64, "wave 0 holds one split per lane");
    float mc = -INFINITY, lc = 0.0f;
    if (tid < ns) {
        mc = A.pml[2 * (at + tid)];
        lc = A.pml[2 * (at + tid) + 1];
    }
    fv pre[kPre];
    const float * P = A.po + at * HD + lane * VPL;
#pragma unroll
    for (int k = 0; k < kPre; k++) pre[k] = *(const fv *) (P + (size_t) min(wave + W * k, ns - 1) * HD);
    if (wave == 0) {
        float M = mc;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
        const float w = tid < ns ? expf(mc - M) : 0.0f;
        wts[tid] = w;
        float L = w * lc;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) L += __shfl_xor(L, o, 64);
        if (lane == 0) red = L;
    }
    __syncthreads();
    fv o = (fv) 0.0f;
#pragma unroll
    for (int k = 0; k < kPre; k++)
        if (wave + W * k < ns) o += wts[wave + W * k] * pre[k];
    acc[wave][lane] = o;
    __syncthreads();
    if (wave == 0) {
        const float inv = 1.0f / red;
        const float g = 1.0f / (1.0f + expf(-gl));
        fv r = acc[0][lane];
#pragma unroll
        for (int w = 1; w < W; w++) r += acc[w][lane];
        r *= inv * g;
#pragma unroll
        for (int v = 0; v < VPL; v++) {
            out[row * HD + lane * VPL + v] = r[v];
            if (out16) out16[row * HD + lane * VPL + v] = fw_bf16(r[v]);
        }
    }
}

/* ---- a verify block: ntok <= 8 consecutive tokens at positions pos0 .. ----
 * (vq-model-gpu.cu:858-969 forward_batch + verify_logits). Each step of the
 * forward runs once for the whole block; token t attends causally to the
 * positions up to pos0 + t. Positions and tokens are kernel arguments: the
 * block path runs eagerly. */
struct FwTok8 {
    int t[8];
};

/* Embedding rows of a Q8_0 head for the block's tokens: column t = row tok[t]. */
__global__ void fw_q8_0_rows_kernel(const uint8_t * blocks, int cols, FwTok8 tok, float * out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
    if (i >= cols) return;
    const uint8_t * b = blocks + ((size_t) tok.t[t] * (cols >> 5) + (i >> 5)) * 34;
    _Float16 d;
    __builtin_memcpy(&d, b, 2);
    out[(size_t) t * cols + i] = (float) d * (float) (int8_t) b[2 + (i & 31)];
}

/* Rope and the KV store for token t = blockIdx.x at position pos0 + t: pair
 * i's cos and sin computed once per token with the expressions of the decode
 * tables (model.rs:416-438, f32), then pair i of every q and k head rotated
 * in place, a rotated k pair stored to the cache too; v and the k elements
 * past pdim stored to the cache. pdim <= 256. */
__global__ __launch_bounds__(256) void fw_rope_kv_n_kernel(float * qkv, int ldq, int qd, int kvd, int heads,
                                                            int kv_heads, int hd, int pdim, float theta, int pos0,
                                                            float * kc, float * vc) {
    __shared__ float cs[2][128];
    const int half = pdim / 2, t = blockIdx.x, pos = pos0 + t, tid = threadIdx.x;
    float * row = qkv + (size_t) t * ldq;
    if (tid < half) {
        const float freq = 1.0f / powf(theta, (float) (2 * tid) / (float) pdim);
        const float a = (float) pos * freq;
        cs[0][tid] = cosf(a);
        cs[1][tid] = sinf(a);
    }
    __syncthreads();
    /* four items per thread at a time, every load issued before the stores
     * (which write the rows read) */
    constexpr int B = 4;
    const int nrot = (heads + kv_heads) * half;
    for (int j0 = tid; j0 < nrot; j0 += B * blockDim.x) {
        float x0[B], x1[B];
#pragma unroll
        for (int b = 0; b < B; b++) {
            const int j = j0 + b * blockDim.x;
            if (j < nrot) {
                const int h = j / half, i = j - h * half;
                const float * base = h < heads ? row + (size_t) h * hd : row + qd + (size_t) (h - heads) * hd;
                x0[b] = base[i];
                x1[b] = base[i + half];
            }
        }
#pragma unroll
        for (int b = 0; b < B; b++) {
            const int j = j0 + b * blockDim.x;
            if (j < nrot) {
                const int h = j / half, i = j - h * half;
                const float c = cs[0][i], sn = cs[1][i];
                float * base = h < heads ? row + (size_t) h * hd : row + qd + (size_t) (h - heads) * hd;
                const float r0 = x0[b] * c - x1[b] * sn, r1 = x1[b] * c + x0[b] * sn;
                base[i] = r0;
                base[i + half] = r1;
                if (h >= heads) {
                    float * k = kc + (size_t) pos * kvd + (size_t) (h - heads) * hd;
                    k[i] = r0;
                    k[i + half] = r1;
                }
            }
        }
    }
    for (int j0 = tid; j0 < kvd; j0 += B * blockDim.x) {
        float v[B], k[B];
#pragma unroll
        for (int b = 0; b < B; b++) {
            const int j = j0 + b * blockDim.x;
            if (j < kvd) {
                v[b] = row[qd + kvd + j];
                k[b] = row[qd + j];
            }
        }
#pragma unroll
        for (int b = 0; b < B; b++) {
            const int j = j0 + b * blockDim.x;
            if (j < kvd) {
                vc[(size_t) pos * kvd + j] = v[b];
                if (j % hd >= 2 * half) kc[(size_t) pos * kvd + j] = k[b];
            }
        }
    }
}

/* fw_rope_kv_n_kernel's work for up to kMaxCols tokens, spread over
 * N x (heads + kv_heads) workgroups: token t = blockIdx.x, head h =
 * blockIdx.y (query heads, then kv heads), thread i < pdim / 2 computing
 * pair i's cos and sin with the same expressions and rotating the head's
 * pair in place; a kv head's rotated pair, its elements past pdim and its v
 * go to the cache too. One load, rotation and store per thread: an 8-token
 * verify block 3141-3145 -> 3061 us against fw_rope_kv_n_kernel's eight
 * workgroups looping over the heads (5.8 us per launch). Long chunks keep
 * fw_rope_kv_n_kernel: this shape (or head groups looped per workgroup)
 * made a 512-token chunk 100-260 us slower. blockDim.x = 128 >= pdim / 2. */
__global__ __launch_bounds__(128) void fw_rope_kv_heads_kernel(float * qkv, int ldq, int qd, int kvd, int heads,
                                                                int hd, int pdim, float theta, int pos0, float * kc,
                                                                float * vc) {
    const int half = pdim / 2, t = blockIdx.x, h = blockIdx.y, i = threadIdx.x, pos = pos0 + t;
    float * row = qkv + (size_t) t * ldq;
    const bool kv = h >= heads;
    const int kh = h - heads;
    float * base = kv ? row + qd + (size_t) kh * hd : row + (size_t) h * hd;
    float * kr = kv ? kc + (size_t) pos * kvd + (size_t) kh * hd : nullptr;
    if (kv) {
        /* elements past pdim and v (neither is written by the rotation) */
        const float * vr = row + qd + kvd + (size_t) kh * hd;
        float * vo = vc + (size_t) pos * kvd + (size_t) kh * hd;
        for (int e = i; e < hd; e += blockDim.x) {
            vo[e] = vr[e];
            if (e >= 2 * half) kr[e] = base[e];
        }
    }
    if (i < half) {
        const float freq = 1.0f / powf(theta, (float) (2 * i) / (float) pdim);
        const float a = (float) pos * freq;
        const float c = cosf(a), sn = sinf(a);
        const float x0 = base[i], x1 = base[i + half];
        const float r0 = x0 * c - x1 * sn, r1 = x1 * c + x0 * sn;
        base[i] = r0;
        base[i + half] = r1;
        if (kv) {
            kr[i] = r0;
            kr[i + half] = r1;
        }
    }
}

/* act = gelu(g) * u with torch's exact gelu, erf in f64 as model.rs:253-258
 * calls it. */
__global__ void fw_gelu_mul_kernel(const float * g, const float * u, float * act, uint16_t * act16, int n) {
    /* four elements per thread through 16-byte loads (g, u and act 16-byte
     * aligned, act16 8-byte aligned: the callers' buffers), the tail apart;
     * act null: only act16 is written (the bf16 model reads nothing else) */
    typedef float f4v __attribute__((ext_vector_type(4)));
    typedef uint16_t u4v __attribute__((ext_vector_type(4)));
    const int n4 = n / 4;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += blockDim.x * gridDim.x) {
        const f4v a = ((const f4v *) g)[i], b = ((const f4v *) u)[i];
        f4v r;
        u4v r16;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            r[k] = gelu_mul(a[k], b[k]);
            r16[k] = fw_bf16(r[k]);
        }
        if (act) ((f4v *) act)[i] = r;
        if (act16) ((u4v *) act16)[i] = r16;
    }
    const int i = 4 * n4 + blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const float r = gelu_mul(g[i], u[i]);
        if (act) act[i] = r;
        if (act16) act16[i] = fw_bf16(r);
    }
}

/* Layer-input capture: rows h[0 .. n) into slot rows pos .. pos + n - 1,
 * the position read from st[1] when st is given (a replayed graph) */
__global__ void fw_capture_kernel(const float * h, float * slot, const int * st, int pos, int n, int hidden) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
    if (i >= hidden || t >= n) return;
    const int p = (st ? st[1] : pos) + t;
    slot[(size_t) p * hidden + i] = h[(size_t) t * hidden + i];
}

/* The index of the largest value (Model::argmax, model.rs:594-605): the
 * first of equal maxima, NaN never chosen, 0 when nothing beats -inf. One
 * workgroup of 1024 threads: each scans a stride, then a tree keeps the
 * larger value or, on a tie, the lower index. */
__global__ __launch_bounds__(1024) void fw_argmax_kernel(const float * v, int n, int * out) {
    __shared__ float bv[1024];
    __shared__ int bi[1024];
    const int t = threadIdx.x;
    float best = -INFINITY;
    int b = -1;
    for (int i = t; i < n; i += 1024) {
        const float x = v[i];
        if (x > best) { best = x; b = i; }
    }
    bv[t] = best;
    bi[t] = b;
    __syncthreads();
    for (int off = 512; off > 0; off >>= 1) {
        if (t < off) {
            const float o = bv[t + off];
            const int oi = bi[t + off];
            if (oi >= 0 && (bi[t] < 0 || o > bv[t] || (o == bv[t] && oi < bi[t]))) { bv[t] = o; bi[t] = oi; }
        }
        __syncthreads();
    }
    if (t == 0) out[0] = bi[0] < 0 ? 0 : bi[0];
}

/* ---- a prompt chunk: up to kPromptMax consecutive tokens at pos0 .. ----
 * (vq-model-gpu.cu:858-943 forward_batch). The steps are the verify
 * block's; the tokens come from device memory, and attention runs without
 * per-chunk partials (whose buffer grows with tokens x context). */
constexpr int kPromptMax = 512;

/* Embedding rows of a Q8_0 head: column t = row tok[t] (device). */
__global__ void fw_q8_0_rows_dev_kernel(const uint8_t * blocks, int cols, const int * tok, float * out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, t = blockIdx.y;
    if (i >= cols) return;
    const uint8_t * b = blocks + ((size_t) tok[t] * (cols >> 5) + (i >> 5)) * 34;
    _Float16 d;
    __builtin_memcpy(&d, b, 2);
    out[(size_t) t * cols + i] = (float) d * (float) (int8_t) b[2 + (i & 31)];
}

/* Attention of token t = blockIdx.y (query rotated in qkv, every key of its
 * window in the cache) for the query heads of kv head blockIdx.x, one wave
 * per query head: the window in chunks of kAttnChunk positions with a
 * running maximum m, sum l and output o (each chunk's terms scaled to the
 * new maximum, the old ones by e^(m_old - m_new)), then o / l times the
 * head's sigmoid gate. The same softmax as the CPU's (model.rs:520-557),
 * summed chunk by chunk in position order. */
template <int VPL>
__global__ __launch_bounds__(256) void fw_attn_prompt_kernel(const float * qkv, int ldq, int kvd, const float * kc,
                                                              const float * vc, const float * gate, int ldg, int pos0,
                                                              int window, int heads, int kv_heads, float scale,
                                                              float * out, uint16_t * out16) {
    constexpr int hd = 64 * VPL, C = kAttnChunk;
    typedef float fv __attribute__((ext_vector_type(VPL)));
    const int t = blockIdx.y, pos = pos0 + t;
    const int start = window > 0 && pos + 1 > window ? pos + 1 - window : 0;
    const int n = pos + 1 - start;
    const int kvh = blockIdx.x, G = heads / kv_heads;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int h = kvh * G + wave;
    const fv q = *(const fv *) (qkv + (size_t) t * ldq + (size_t) h * hd + lane * VPL);
    const float * kb = kc + (size_t) start * kvd + (size_t) kvh * hd + lane * VPL;
    const float * vb = vc + (size_t) start * kvd + (size_t) kvh * hd + lane * VPL;
    float m = -INFINITY, l = 0.0f;
    fv o = (fv) 0.0f;
    for (int j0 = 0; j0 < n; j0 += C) {
        const int jn = min(C, n - j0);
        fv kr[C], vr[C];
#pragma unroll
        for (int j = 0; j < C; j++) kr[j] = *(const fv *) (kb + (size_t) (j0 + min(j, jn - 1)) * kvd);
#pragma unroll
        for (int j = 0; j < C; j++) vr[j] = *(const fv *) (vb + (size_t) (j0 + min(j, jn - 1)) * kvd);
        float sc[C];
        float mc = -INFINITY;
#pragma unroll
        for (int j = 0; j < C; j++) {
            float sv = 0.0f;
#pragma unroll
            for (int v = 0; v < VPL; v++) sv += q[v] * kr[j][v];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) sv += __shfl_xor(sv, off, 64);
            sc[j] = sv * scale;
            if (j < jn) mc = fmaxf(mc, sc[j]);
        }
        const float mn = fmaxf(m, mc);
        const float a = expf(m - mn);          /* 0 on the first chunk (m = -inf) */
        l *= a;
        o *= a;
#pragma unroll
        for (int j = 0; j < C; j++) {
            /* rows past jn are padding that may hold anything (the row at pos
             * before its store): skipped, not weighted by zero */
            if (j < jn) {
                const float e = expf(sc[j] - mn);
                l += e;
                o += e * vr[j];
            }
        }
        m = mn;
    }
    const float g = 1.0f / (1.0f + expf(-gate[(size_t) t * ldg + h]));
    const fv r = o * (1.0f / l) * g;
    const size_t ob = (size_t) t * heads * hd + (size_t) h * hd + lane * VPL;
#pragma unroll
    for (int v = 0; v < VPL; v++) {
        out[ob + v] = r[v];
        if (out16) out16[ob + v] = fw_bf16(r[v]);
    }
}

/* The same prompt attention on the f32 matrix cores, for 256-element heads
 * (the reference model's): one workgroup per (query head, 16 query tokens),
 * the grid ordered so that the blocks with the longest causal range start
 * first. The block's positions are cut into tiles of 16; wave w of the 4
 * takes tiles w, w + 4, w + 8, ..., with its own running maximum, sum and
 * output, merged at the end. No wave reads another's K or V rows, so a wave
 * loads them from global memory straight into the MFMA operand layout, with
 * no LDS staging and no barrier in the loop: V of a tile is requested before
 * the tile's scores are formed and K of the next tile right after, so both
 * arrive while MFMAs run. Per tile a wave forms the 16 x 16 scores
 * S^T = K Q^T (positions x tokens) with 64 v_mfma_f32_16x16x4f32 (four
 * accumulators, so consecutive MFMAs do not wait for each other), masks
 * positions outside each token's window (causal, and the sliding window),
 * weights them by exp(score - m) for a per-token reference m, and adds
 * O^T += V^T P^T with 64 more. Unlike the kernel above, m is not the running
 * maximum itself: it moves (the sums and outputs rescaled) only when a score
 * passes it by more than kPaLag, which keeps every weight below e^8 and
 * spares most tiles the exchange between lanes and the rescale. The quotient
 * of outputs and sums does not depend on m; products and sums stay in f32,
 * and only the rounding and the order of the additions differ from the
 * kernel above.
 *
 * Operand layouts (lane l = 16 g + c): an A operand is A[l % 16][l / 16]
 * (16 x 4), a B operand B[l / 16][l % 16] (4 x 16), and the 16 x 16 result
 * sits as D[4 (l / 16) + i][l % 16], i < 4. Which head element a (k-step,
 * lane group) pair contracts over is free as long as both operands agree:
 * lane (g, c) feeds K[c][pa_k(ks, g)] and Q[c][pa_k(ks, g)] at k-step ks:
 * it reads its K row as 16 runs of 4 floats, the 4 lane groups of a row
 * together 64 contiguous bytes (a load instruction touches 16 cache lines,
 * not 64), and holds the scores of token c at positions 4 g + i. For O^T, k-step ks takes positions 4 g + ks: the B
 * value is the lane's own probability i = ks, and the A value is
 * V[4 g + ks][d], with the rows of O^T permuted (pa_d) so that d too runs in
 * groups of 4: the 16 lanes of a group read 256 contiguous bytes of a row. */
constexpr int kPaTok = 16;     /* query tokens per workgroup */

/* head element contracted at k-step ks by lane group g in S^T = K Q^T */
static __device__ __forceinline__ int pa_k(int ks, int g) { return 16 * (ks >> 2) + 4 * g + (ks & 3); }
/* head element of row R of O^T block b */
static __device__ __forceinline__ int pa_d(int b, int R) { return 64 * (b >> 2) + 4 * R + (b & 3); }

__global__ __launch_bounds__(256) void fw_attn_prompt_mfma_kernel(const float * qkv, int ldq, int kvd,
                                                                   const float * kc, const float * vc,
                                                                   const float * gate, int ldg, int pos0, int N,
                                                                   int window, int heads, int kv_heads, float scale,
                                                                   float * out, uint16_t * out16,
                                                                   const uint32_t * redo, int nredo) {
    typedef float f4v __attribute__((ext_vector_type(4)));
    /* the merge after the loop: outputs handed between waves, 3 x 4 blocks
     * of 64 x 4 floats per wave, and the maximum and sum per token of each;
     * before the loop the block's Q rows pass through the first part */
    __shared__ f4v lds_o[48 * 64];
    __shared__ float lds_s[4 * 32];
    const int h = blockIdx.x, t0 = ((int) gridDim.y - 1 - (int) blockIdx.y) * kPaTok;
    const int kvh = h / (heads / kv_heads);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, c = lane & 15;
    if (redo) {
        /* after the split kernel below: only the blocks that it could not do */
        const int nb = ((int) gridDim.y + 1) / 2;   /* its blocks are two of these */
        uint32_t any = 0;
        for (int z = 0; z < nredo; z++) any |= redo[((size_t) z * nb + t0 / (2 * kPaTok)) * kv_heads + kvh];
        if (!any) return;   /* uniform */
    }
    /* this lane's token (column c); tokens past N compute a copy of the last
     * one and store nothing */
    const int tv = min(t0 + c, N - 1), pos_t = pos0 + tv;
    const int start_t = window > 0 && pos_t + 1 > window ? pos_t + 1 - window : 0;
    /* the block's positions: from the first token's window start to the last token */
    const int tl = min(t0 + kPaTok - 1, N - 1);
    const int pfirst = window > 0 && pos0 + t0 + 1 > window ? pos0 + t0 + 1 - window : 0;
    const int plast = pos0 + tl;
    /* the gate, requested first: it is needed at the end */
    const float gate_t = gate[(size_t) tv * ldg + h];
    /* Q^T as the B operand: Q[c][pa_k(ks, g)], ks < 64. The block's 16 Q rows
     * are read once per workgroup into LDS (rows of 65 x 4 floats, so the 16
     * rows of a lane group fall on distinct banks), in the space the merge
     * uses after the loop */
    float qv[64];
    {
        f4v * lds_q = lds_o;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int i = tid + 256 * k, tk = i >> 6, c4 = i & 63;
            lds_q[tk * 65 + c4] = *(const f4v *) (qkv + (size_t) min(t0 + tk, N - 1) * ldq + (size_t) h * 256 + 4 * c4);
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 64; ks += 4) {
            const f4v q4 = lds_q[c * 65 + pa_k(ks, g) / 4];
            qv[ks] = q4[0];
            qv[ks + 1] = q4[1];
            qv[ks + 2] = q4[2];
            qv[ks + 3] = q4[3];
        }
        __syncthreads();   /* every wave holds its Q before any writes the merge */
    }
    f4v o[16];
#pragma unroll
    for (int db = 0; db < 16; db++) o[db] = f4v{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.0f;
    const float * kbase = kc + (size_t) kvh * 256;
    const float * vbase = vc + (size_t) kvh * 256;
    /* K rows pw + c and V rows pw + 4 g + ks of the tile at pw; rows past
     * plast repeat it and are masked. Each is requested for the next tile as
     * soon as this tile's MFMAs have read it, so it has most of a tile's time
     * to arrive. The requests are unconditional (past the last tile they all
     * read row plast again): behind a branch, the waits for this tile's V
     * would also cover the next tile's K */
    f4v kf[16], vf[16];
    auto fetch_k = [&](int pw) {
        const float * kp = kbase + (size_t) min(pw + c, plast) * kvd;
#pragma unroll
        for (int j = 0; j < 16; j++) kf[j] = *(const f4v *) (kp + pa_k(4 * j, g));
    };
    auto fetch_v = [&](int pw) {
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            const float * vp = vbase + (size_t) min(pw + 4 * g + ks, plast) * kvd + 4 * c;
#pragma unroll
            for (int q = 0; q < 4; q++) vf[4 * ks + q] = *(const f4v *) (vp + 64 * q);
        }
    };
    const int pbeg = (pfirst & ~15) + 16 * wave;
    /* Q, then K, then V, in the order the loop waits for them */
    __builtin_amdgcn_sched_barrier(0);
    fetch_k(pbeg);
    __builtin_amdgcn_sched_barrier(0);
    fetch_v(pbeg);
    __builtin_amdgcn_sched_barrier(0);
    for (int pw = pbeg; pw <= plast; pw += 64) {
        /* S^T = K Q^T */
        f4v s0 = f4v{0.f, 0.f, 0.f, 0.f}, s1 = s0, s2 = s0, s3 = s0;
#pragma unroll
        for (int j = 0; j < 16; j++) {
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][0], qv[4 * j], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][1], qv[4 * j + 1], s1, 0, 0, 0);
            s2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][2], qv[4 * j + 2], s2, 0, 0, 0);
            s3 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][3], qv[4 * j + 3], s3, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch_k(pw + 64);
        __builtin_amdgcn_sched_barrier(0);
        const f4v s = (s0 + s1) + (s2 + s3);
        /* scale and mask: position pw + 4 g + i for token c */
        float e[4];
        float mc = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int pp = pw + 4 * g + i;
            const bool ok = pp >= start_t && pp <= pos_t;
            e[i] = ok ? s[i] * scale : -INFINITY;
            mc = fmaxf(mc, e[i]);
        }
        /* the weights are exp(score - m) for a reference m per token that
         * moves only when a score passes it by more than kPaLag (then to the
         * token's maximum so far, the sum and outputs rescaled): the weights
         * stay below e^kPaLag, and most tiles need neither an exchange
         * between lanes nor a rescale */
        if (__any(mc > m + kPaLag)) {   /* uniform */
            mc = fmaxf(mc, __shfl_xor(mc, 16, 64));
            mc = fmaxf(mc, __shfl_xor(mc, 32, 64));
            const float mn = fmaxf(m, mc);
            /* nothing seen yet for this token: no rescale */
            const float a = mn == -INFINITY ? 1.0f : expf(m - mn);
            l *= a;
#pragma unroll
            for (int db = 0; db < 16; db++) o[db] *= a;
            m = mn;
        }
        /* l holds this lane's share of the sum (its 4 positions), reduced
         * over the lane groups after the loop */
#pragma unroll
        for (int i = 0; i < 4; i++) {
            e[i] = e[i] == -INFINITY ? 0.0f : expf(e[i] - m);
            l += e[i];
        }
        /* O^T += V^T P^T; row c of block db is element pa_d(db, c) */
#pragma unroll
        for (int ks = 0; ks < 4; ks++)
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    o[4 * q + r] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[4 * ks + q][r], e[ks], o[4 * q + r], 0, 0,
                                                                        0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_v(pw + 64);
        __builtin_amdgcn_sched_barrier(0);
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    /* merge: wave w finishes head elements 64 w .. 64 w + 63 (blocks
     * 4 w .. 4 w + 3 of O^T) of the 16 tokens. The other waves hand it their
     * outputs for those blocks through LDS in their register layout, a slot
     * of 64 x 4 floats per (source wave, owner, block), owners' own blocks
     * not stored; every wave hands over its maximum and sum per token */
#pragma unroll
    for (int w = 0; w < 4; w++) {
        if (w == wave) continue;   /* uniform */
        const int k = (w - wave + 3) & 3;   /* 0 .. 2: the owner's index among the others */
#pragma unroll
        for (int b = 0; b < 4; b++) lds_o[((wave * 3 + k) * 4 + b) * 64 + lane] = o[4 * w + b];
    }
    if (g == 0) {
        lds_s[wave * 32 + c] = m;
        lds_s[wave * 32 + 16 + c] = l;
    }
    __syncthreads();
    float mw[4], aw[4];
#pragma unroll
    for (int w = 0; w < 4; w++) mw[w] = lds_s[w * 32 + c];
    const float mt = fmaxf(fmaxf(mw[0], mw[1]), fmaxf(mw[2], mw[3]));
    float lt = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        aw[w] = mw[w] == -INFINITY ? 0.0f : expf(mw[w] - mt);
        lt += lds_s[w * 32 + 16 + c] * aw[w];
    }
    /* sum over the source waves in wave order, this wave's own blocks from
     * its registers */
    f4v v[4];
#pragma unroll
    for (int w = 0; w < 4; w++) {
#pragma unroll
        for (int b = 0; b < 4; b++) {
            f4v x;
            if (w == wave) {   /* uniform */
                x = o[4 * w + b];
            } else {
                const int k = (wave - w + 3) & 3;
                x = lds_o[((w * 3 + k) * 4 + b) * 64 + lane];
            }
            v[b] = w == 0 ? x * aw[0] : v[b] + x * aw[w];
        }
    }
    if (t0 + c >= N) return;
    const float gs = 1.0f / (1.0f + expf(-gate_t));
    const float inv = 1.0f / lt;
    /* element pa_d(4 wave + b, 4 g + i) = 64 wave + 16 g + 4 i + b: four
     * consecutive elements per i */
    const size_t ob = (size_t) tv * heads * 256 + (size_t) h * 256 + 64 * wave + 16 * g;
    /* the bf16 copy when one is asked for (the next matvec reads only it),
     * else the f32 output */
    f4v r[4];
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = f4v{v[0][i], v[1][i], v[2][i], v[3][i]} * inv * gs;
    if (out16) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint2 p;
            p.x = (uint32_t) fw_bf16(r[i][0]) | ((uint32_t) fw_bf16(r[i][1]) << 16);
            p.y = (uint32_t) fw_bf16(r[i][2]) | ((uint32_t) fw_bf16(r[i][3]) << 16);
            *(uint2 *) (out16 + ob + 4 * i) = p;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) *(f4v *) (out + ob + 4 * i) = r[i];
    }
}

/* Prompt attention over long spans, for 256-element heads in groups of four
 * query heads per kv head: the products on the f16 matrix cores, f32 in
 * value. Every f32 operand is brought to the top of f16's range by a power of
 * two (exact) and split into two f16 halves; hi hi, hi lo and lo hi are taken
 * (lo lo is below 2^-24). q has a scale per token, k and v one per position,
 * and the weights, times their rows' v scales, one per token and tile, which
 * the token's output column carries back. No scale is shared between
 * positions, so what a token does not see (or weighs little) takes no bits
 * from what it sees. hi + lo is x to 2^-23 of x, or to 2^-39 of the largest
 * operand under the same scale where x is below 2^-16 of it: of the largest
 * element of the same row, or, for a weight, of the token's largest in the
 * tile. (The out matvec that reads the result splits all of a token's heads
 * under one scale in the same way.) Three f16 products run in 3/16 of the f32
 * products' matrix-core time. Sums stay f32: the scores' hi hi products have
 * two accumulators, their small products one (one and one rounded often enough
 * at the size of the score to show in sharp weights), and the outputs of 32
 * positions are summed apart, small products first, then added to the running
 * output: it rounds once per 32 positions (the f32 kernel above, every 4).
 * Distance of a token's row from 64 bits, mean of 160, f32 kernel and here (one
 * hi hi accumulator): scores of deviation 3 at position 2070 8.5e-7 and 6.3e-7
 * (8.0e-7), of 12 there 1.10e-6 and 1.02e-6 (1.26e-6), at 3000 1.12e-6 and
 * 9.3e-7 (1.20e-6).
 *
 * One workgroup per (kv head, 32 tokens, span split): of its eight waves,
 * wave w is query head w % 4 of the group and tokens 16 (w / 4) .. against all
 * of the workgroup's K and V, so a position's rows are read, split and put
 * into LDS once for 128 columns (the f32 kernel reads them per head and 16
 * tokens). Positions go 32 at a time. The query halves and the outputs (64
 * registers each) stay in registers; K is converted while the outputs' MFMAs
 * run, V while the scores' do, each requested a phase earlier.
 *
 * 512 tokens at 16384, 16 heads: 610 us, 1378 in the f32 kernel (101 TFLOP/s
 * of f32 products; 229 here). What bounds it is the conversions' and
 * softmax's VALU work and the two barriers per tile (MFMAs are busy a quarter
 * of the time). Nothing may spill here: a wave's loads return in order, so a
 * reload in the loop waits for the K and V requests before it (59 spilled
 * registers: 1400 us). Three bf16 planes and six products need no scales but
 * spilled, at 1390 us. Scales per v row and per token, exponents for keys and
 * queries and the second accumulator cost 18 us of 592 against one v scale per
 * tile, which lost the weights of rows beside a much larger or an all-zero one.
 * Taking lo lo too costs 28 us more and gains 2 % of the distance.
 *
 * Layouts (16x16x32: lane l = 16 g + c holds A[c][8 g + j], B[8 g + j][c],
 * D[4 g + i][c]): scores are positions x tokens, so a lane's 8 weights are of
 * its own token, and the output product takes weight j as it lies: position
 * 16 (j / 4) + 4 g + j % 4, with V stored to match. Output block b, row r is
 * head element 16 r + b.
 *
 * A workgroup that meets an infinity or NaN says so in redo [split][token
 * block][kv head], and the f32 kernel above then does those blocks again. */
constexpr int kPsTok = 32;                          /* tokens per workgroup, positions per tile */
constexpr int kPsPlane = 16384;                     /* LDS bytes of one half of a tile */
constexpr int kPsLds = 4 * kPsPlane + 320;          /* K and V halves, scales, the waves' flags */
constexpr int kPsMaxSplit = 8;

typedef uint32_t ps_u4 __attribute__((ext_vector_type(4)));
typedef _Float16 ps_h8 __attribute__((ext_vector_type(8)));

/* f[0 .. 7] * sc as two halves of eight f16 */
static __device__ __forceinline__ void ps_split(const float * f, float sc, ps_h8 * pl) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const float x = f[j] * sc;
        pl[0][j] = (_Float16) x;
        pl[1][j] = (_Float16) (x - (float) pl[0][j]);
    }
}

/* The largest of m over the 16 lanes of a row, in every lane */
static __device__ __forceinline__ uint32_t ps_max16(uint32_t m) {
    m = max(m, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) m, 0xB1, 0xf, 0xf, false));    /* lane ^ 1 */
    m = max(m, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) m, 0x4E, 0xf, 0xf, false));    /* lane ^ 2 */
    m = max(m, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) m, 0x141, 0xf, 0xf, false));   /* mirrored in 8 */
    return max(m, (uint32_t) __builtin_amdgcn_update_dpp(0, (int) m, 0x140, 0xf, 0xf, false)); /* in 16 */
}

/* The largest of m over the lanes l, l ^ 16, l ^ 32 and l ^ 48, in each of
 * them: register swaps (odd rows of 16 lanes with even ones, then halves of
 * the wave), no LDS round trip ahead of the output products */
static __device__ __forceinline__ uint32_t ps_max_rows(uint32_t m) {
    const auto a = __builtin_amdgcn_permlane16_swap(m, m, false, false);
    m = max(a[0], a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(m, m, false, false);
    return max(b[0], b[1]);
}

/* The power of two that brings the largest magnitude (f32 bits) to [2^14,
 * 2^15) (as far as 2^126 takes it), and its inverse's exponent, -126 .. 113;
 * zero gives the smallest, so that nothing is scaled down for it */
static __device__ __forceinline__ float ps_scale(uint32_t mag, int & ex) {
    const uint32_t f = min(268u - min(mag >> 23, 254u), 253u);
    ex = 127 - (int) f;
    return __uint_as_float(f << 23);
}

/* 2^ex, ex in -126 .. 127 */
static __device__ __forceinline__ float ps_pow2(int ex) { return __uint_as_float((uint32_t) (ex + 127) << 23); }

typedef float ps_f4 __attribute__((ext_vector_type(4)));

static __device__ __forceinline__ ps_f4 ps_mfma(ps_h8 a, ps_h8 b, ps_f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

__global__ __launch_bounds__(512) void fw_attn_prompt_split_kernel(const float * qkv, int ldq, int kvd,
                                                                    const float * kc, const float * vc, int pos0, int N,
                                                                    int heads, float scale, float * po, float * pml,
                                                                    uint32_t * redo) {
    typedef ps_f4 f4v;
    typedef int i4v __attribute__((ext_vector_type(4)));
    typedef _Float16 h4v __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) uint8_t ps_lds[];
    int * kexp = (int *) (ps_lds + 4 * kPsPlane);              /* exponent of K's inverse scale per position */
    float * vinv = (float *) (kexp + 32);                      /* V's inverse scale */
    uint32_t * flags = (uint32_t *) (vinv + 32);               /* per wave, at the end */
    /* the wave as a scalar: what depends on it alone takes no vector register */
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, g = lane >> 4, c = lane & 15;
    /* the blocks with the longest causal range first */
    const int kvh = blockIdx.z, t0 = ((int) gridDim.y - 1 - (int) blockIdx.y) * kPsTok, h = 4 * kvh + (wave & 3);
    const int tk = t0 + 16 * (wave >> 2) + c;
    const int tv = min(tk, N - 1), pos_t = pos0 + tv;
    const int plast = pos0 + min(t0 + kPsTok - 1, N - 1);
    const int nt = plast / 32 + 1, nz = gridDim.x, z = blockIdx.x;
    const int ta = (int) ((long) nt * z / nz), tb = (int) ((long) nt * (z + 1) / nz);
    const float * kb = kc + (size_t) kvh * 256, * vb = vc + (size_t) kvh * 256;
    const float * qrow = qkv + (size_t) tv * ldq + (size_t) h * 256;

    /* K: piece i is position 16 i + tid / 32, elements 8 kg .. + 7; positions
     * past plast repeat it and are masked */
    const int kg = tid & 31, kp = tid >> 5;
    f4v kr[4], vr[4];
    auto load_k = [&](int p0) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const f4v * r = (const f4v *) (kb + (size_t) min(p0 + 16 * i + kp, plast) * kvd + 8 * kg);
            kr[2 * i] = r[0];
            kr[2 * i + 1] = r[1];
        }
    };
    float ksc[2];
    bool bad = false;   /* an infinity or NaN */
    /* the pieces' scales, from their positions' largest magnitudes (32 lanes) */
    auto scale_k = [&]() {
        uint32_t all = 0;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            uint32_t m = 0;
#pragma unroll
            for (int j = 0; j < 8; j++) m = max(m, __float_as_uint(kr[2 * i + (j >> 2)][j & 3]) & 0x7fffffffu);
            m = ps_max16(m);
            m = max(m, (uint32_t) __shfl_xor((int) m, 16, 64));
            all = max(all, m);
            int ex;
            ksc[i] = ps_scale(m, ex);
            if (kg == 0) kexp[16 * i + kp] = ex;
        }
        bad |= all >= 0x7f800000u;
    };
    /* a half's 16-byte pieces by (element group, position), the positions of
     * a group permuted so that neither side meets bank conflicts */
    auto store_k = [&](int i) {
        float f[8];
#pragma unroll
        for (int j = 0; j < 8; j++) f[j] = kr[2 * i + (j >> 2)][j & 3];
        ps_h8 pl[2];
        ps_split(f, ksc[i], pl);
#pragma unroll
        for (int p = 0; p < 2; p++)
            *(ps_h8 *) (ps_lds + p * kPsPlane + kg * 512 + 16 * ((16 * i + kp) ^ (kg & 15))) = pl[p];
    };
    /* V: wave 2 vg + pb takes positions 16 pb + 4 vg .. + 3, elements 4 lane .. + 3 */
    const int vg = wave >> 1, vp = wave & 1;
    auto load_v = [&](int p0) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            vr[j] = *(const f4v *) (vb + (size_t) min(p0 + 16 * vp + 4 * vg + j, plast) * kvd + 4 * lane);
    };
    float vsc[4];
    auto scale_v = [&]() {
        uint32_t all = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t m = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) m = max(m, __float_as_uint(vr[j][e]) & 0x7fffffffu);
            m = ps_max16(m);
            /* the row's largest in a scalar register, its scale with it */
            uint32_t w = 0;
#pragma unroll
            for (int r = 0; r < 4; r++) w = max(w, (uint32_t) __builtin_amdgcn_readlane((int) m, 16 * r));
            all = max(all, w);
            int ex;
            vsc[j] = ps_scale(w, ex);
            if (lane == 0) vinv[16 * vp + 4 * vg + j] = ps_pow2(ex);
        }
        bad |= all >= 0x7f800000u;
    };
    /* element 4 lane + e is row lane / 4 of block 4 (lane % 4) + e */
    auto store_v = [&](int e) {
        h4v hi, lo;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float x = vr[j][e] * vsc[j];
            hi[j] = (_Float16) x;
            lo[j] = (_Float16) (x - (float) hi[j]);
        }
        uint8_t * d = ps_lds + 2 * kPsPlane + (4 * (lane & 3) + e) * 1024 + vg * 256 + (lane >> 2) * 16 + vp * 8;
        *(h4v *) d = hi;
        *(h4v *) (d + kPsPlane) = lo;
    };

    if (ta < tb) {
        load_k(32 * ta);
        load_v(32 * ta);
    }
    /* the token's query: halves of the row's 8 steps, the row's scale over the
     * four lanes that hold it */
    ps_h8 q[8][2];
    int qexp;
    {
        f4v qf[16];
        uint32_t mx = 0;
#pragma unroll
        for (int ks = 0; ks < 16; ks++) {
            qf[ks] = *(const f4v *) (qrow + 32 * (ks >> 1) + 8 * g + 4 * (ks & 1));
#pragma unroll
            for (int j = 0; j < 4; j++) mx = max(mx, __float_as_uint(qf[ks][j]) & 0x7fffffffu);
        }
        mx = max(mx, (uint32_t) __shfl_xor((int) mx, 16, 64));
        mx = max(mx, (uint32_t) __shfl_xor((int) mx, 32, 64));
        const float qs = ps_scale(mx, qexp);
        bad |= mx >= 0x7f800000u;
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            float f[8];
#pragma unroll
            for (int j = 0; j < 8; j++) f[j] = qf[2 * ks + (j >> 2)][j & 3];
            ps_split(f, qs, q[ks]);
        }
    }
    f4v o[16];
#pragma unroll
    for (int b = 0; b < 16; b++) o[b] = f4v{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.0f;
    if (ta < tb) {
        scale_k();
#pragma unroll
        for (int i = 0; i < 2; i++) store_k(i);
        __syncthreads();
    }
    for (int ti = ta; ti < tb; ti++) {
        const int p0 = 32 * ti;
        load_k(p0 + 32);
        f4v s0[2][2], s1[2];
#pragma unroll
        for (int pb = 0; pb < 2; pb++) s0[pb][0] = s0[pb][1] = s1[pb] = f4v{0.f, 0.f, 0.f, 0.f};
        ps_h8 kf[2][2][2];
        auto read_k = [&](int ks) {
#pragma unroll
            for (int pb = 0; pb < 2; pb++)
#pragma unroll
                for (int p = 0; p < 2; p++)
                    kf[ks & 1][pb][p] = *(const ps_h8 *) (ps_lds + p * kPsPlane + (4 * ks + g) * 512 +
                                                          16 * ((16 * pb + c) ^ ((4 * ks + g) & 15)));
        };
        read_k(0);
#pragma unroll
        for (int ks = 0; ks < 8; ks++) {
            __builtin_amdgcn_sched_barrier(0);   /* no reads further ahead: no registers */
            if (ks < 7) read_k(ks + 1);
#pragma unroll
            for (int pb = 0; pb < 2; pb++) s1[pb] = ps_mfma(kf[ks & 1][pb][1], q[ks][0], s1[pb]);
#pragma unroll
            for (int pb = 0; pb < 2; pb++) s0[pb][ks & 1] = ps_mfma(kf[ks & 1][pb][0], q[ks][0], s0[pb][ks & 1]);
#pragma unroll
            for (int pb = 0; pb < 2; pb++) s1[pb] = ps_mfma(kf[ks & 1][pb][0], q[ks][1], s1[pb]);
            if (ks == 0) scale_v();
            if (ks >= 3 && ks < 7) store_v(ks - 3);
        }
        __builtin_amdgcn_sched_barrier(0);
        const i4v ki[2] = {*(const i4v *) (kexp + 4 * g), *(const i4v *) (kexp + 16 + 4 * g)};
        float e[8];
        float mc = -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; i++)
            /* both scales in one step: a large key's alone may pass f32's range */
            e[i] = __builtin_ldexpf((s0[i >> 2][0][i & 3] + s0[i >> 2][1][i & 3]) + s1[i >> 2][i & 3], ki[i >> 2][i & 3] + qexp);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int pp = p0 + 16 * (i >> 2) + 4 * g + (i & 3);
            e[i] = pp <= pos_t ? e[i] * scale : -INFINITY;
            mc = fmaxf(mc, e[i]);
        }
        /* the lagging reference maximum of the kernel above */
        if (__any(mc > m + kPaLag)) {   /* uniform */
            mc = fmaxf(mc, __shfl_xor(mc, 16, 64));
            mc = fmaxf(mc, __shfl_xor(mc, 32, 64));
            const float mn = fmaxf(m, mc);
            const float a = mn == -INFINITY ? 1.0f : expf(m - mn);
            l *= a;
#pragma unroll
            for (int b = 0; b < 16; b++) o[b] *= a;
            m = mn;
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            e[i] = e[i] == -INFINITY ? 0.0f : expf(e[i] - m);
            l += e[i];
        }
        __syncthreads();   /* V is whole, K read by all */
        {
            /* the token's weights in units of its V rows' scales, brought to the
             * top of f16's range by a power of two of the token's own: only
             * what it sees has a weight. e^kPaLag < 2^12 and inverse scales of
             * at most 2^113 stay finite */
            const f4v va[2] = {*(const f4v *) (vinv + 4 * g), *(const f4v *) (vinv + 16 + 4 * g)};
            uint32_t wm = 0;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                e[i] *= va[i >> 2][i & 3];
                wm = max(wm, __float_as_uint(e[i]));
            }
            wm = ps_max_rows(wm);
            int wexp;
            const float ws = ps_scale(wm, wexp), vo = ps_pow2(wexp);
            ps_h8 pw[2];
            ps_split(e, ws, pw);
            load_v(p0 + 32);
            ps_h8 v[2][2][2];
            auto read_v = [&](int st) {
#pragma unroll
                for (int k = 0; k < 2; k++)
#pragma unroll
                    for (int p = 0; p < 2; p++)
                        v[st & 1][k][p] = *(const ps_h8 *) (ps_lds + (2 + p) * kPsPlane + (2 * st + k) * 1024 + 16 * lane);
            };
            read_v(0);
#pragma unroll
            for (int st = 0; st < 8; st++) {   /* two output blocks a step */
                __builtin_amdgcn_sched_barrier(0);
                if (st < 7) read_v(st + 1);
                f4v r[2];
#pragma unroll
                for (int k = 0; k < 2; k++) r[k] = ps_mfma(v[st & 1][k][1], pw[0], f4v{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                for (int k = 0; k < 2; k++) r[k] = ps_mfma(v[st & 1][k][0], pw[1], r[k]);
#pragma unroll
                for (int k = 0; k < 2; k++) r[k] = ps_mfma(v[st & 1][k][0], pw[0], r[k]);
                if (st == 0) scale_k();
                if (st == 3 || st == 5) store_k((st - 3) / 2);
#pragma unroll
                for (int k = 0; k < 2; k++)
#pragma unroll
                    for (int i = 0; i < 4; i++) o[2 * st + k][i] = __builtin_fmaf(r[k][i], vo, o[2 * st + k][i]);
            }
        }
        __syncthreads();   /* K is whole, V read by all */
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const bool wbad = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (lane == 0) flags[wave] = wbad ? 1u : 0u;
    __syncthreads();
    if (tid == 0) {
        uint32_t any = 0;
        for (int w = 0; w < 8; w++) any |= flags[w];
        redo[((size_t) z * gridDim.y + t0 / kPsTok) * gridDim.z + kvh] = any;
    }
    if (tk >= N) return;
    const size_t at = ((size_t) z * N + tv) * heads + h;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        f4v * d = (f4v *) (po + at * 256 + 16 * (4 * g + i));
#pragma unroll
        for (int k = 0; k < 4; k++) d[k] = f4v{o[4 * k][i], o[4 * k + 1][i], o[4 * k + 2][i], o[4 * k + 3][i]};
    }
    if (g == 0) {
        pml[2 * at] = m;
        pml[2 * at + 1] = l;
    }
}

/* The splits of a token and head in order: outputs and sums brought to the
 * largest reference, then o / l times the head's sigmoid gate. One wave per
 * (token, head), four elements per lane. */
__global__ __launch_bounds__(256) void fw_attn_prompt_merge_kernel(const float * po, const float * pml, int nz, int N,
                                                                    int heads, const float * gate, int ldg, float * out,
                                                                    uint16_t * out16) {
    typedef float f4v __attribute__((ext_vector_type(4)));
    const int t = blockIdx.x, h = 4 * blockIdx.y + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (h >= heads) return;
    f4v p[kPsMaxSplit];
    float ms[kPsMaxSplit], ls[kPsMaxSplit];
    float mt = -INFINITY;
#pragma unroll
    for (int z = 0; z < kPsMaxSplit; z++) {
        if (z >= nz) continue;   /* uniform */
        const size_t at = ((size_t) z * N + t) * heads + h;
        p[z] = *(const f4v *) (po + at * 256 + 4 * lane);
        ms[z] = pml[2 * at];
        ls[z] = pml[2 * at + 1];
        mt = fmaxf(mt, ms[z]);
    }
    f4v o = f4v{0.f, 0.f, 0.f, 0.f};
    float l = 0.0f;
#pragma unroll
    for (int z = 0; z < kPsMaxSplit; z++) {
        if (z >= nz || ms[z] == -INFINITY) continue;
        const float a = expf(ms[z] - mt);
        o += p[z] * a;
        l += ls[z] * a;
    }
    const f4v r = o * (1.0f / l) * (1.0f / (1.0f + expf(-gate[(size_t) t * ldg + h])));
    const size_t ob = ((size_t) t * heads + h) * 256 + 4 * lane;
    if (out16) {
        uint2 w;
        w.x = (uint32_t) fw_bf16(r[0]) | ((uint32_t) fw_bf16(r[1]) << 16);
        w.y = (uint32_t) fw_bf16(r[2]) | ((uint32_t) fw_bf16(r[3]) << 16);
        *(uint2 *) (out16 + ob) = w;
    } else {
        *(f4v *) (out + ob) = r;
    }
}

/* ------------------------------------------------------------------ host -- */

namespace {

struct Model {
    sparkmv_model_cfg c;
    std::vector<sparkmv_model_layer> layers;
    std::vector<int> layer_set;
    int head_kind = -1;                  /* 0 VQ container, 8 Q8_0 blocks */
    const void * head_stages[4] = {nullptr, nullptr, nullptr, nullptr};
    const void * head_blocks = nullptr;
    const float * final_norm = nullptr;
    /* device memory, one allocation */
    void * mem = nullptr;
    float * h, * xn, * qkv, * g, * attn, * mg, * mu, * act, * kv;
    uint16_t * xn16, * attn16, * act16;
    uint64_t * pslot;                    /* the gate/up launches' exchange, intermediate * kMaxCols words, kept zero */
    /* exchange words of the several-column launches over hidden rows (the
     * chunk-split tiles' tree), kept zero; the launches share them, one at
     * a time on the model's stream */
    uint64_t * kslot;
    long kslot_cap;
    /* gelu * up written by the gate/up launch (1), or by the activation
     * kernel (0: SPARKMV_SEPARATE_ACT=1 at creation; the same bits, slower) */
    int fuse_act = 1;
    int * st;                            /* token, position */
    float * part, * pml;                 /* attention partials [heads][nsplit][head_dim], [heads][nsplit][2] */
    float * rtab;                        /* rope tables [full, sliding][cos, sin][128] */
    int nsplit;                          /* kAttnSplits, or the tiles of a shorter cache */
    /* the recorded chain */
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    /* cached positions (model.rs:453, :361-381) */
    int len = 0;
    /* tuned kernels per (rows, cols) of a VQ matvec: variant, threads */
    std::map<std::pair<int, int>, std::pair<int, int>> picks;
    /* device memory the model frees at destroy: weights a loader uploaded */
    std::vector<void *> owned;
    /* block buffers (verify blocks and prompt chunks), one allocation at
     * sparkmv_model_reserve or the first block: vcap columns of each
     * activation, gate rows at the qkv stride, the tokens, and attention
     * partials for verify blocks of up to 8 tokens */
    void * vmem = nullptr;
    int vcap = 0;
    /* the prompt matrices' K-split slices, for chunks of up to vcap tokens: a
     * pool allocation and release per matrix left 20-40 us gaps on the GPU */
    void * vsplit = nullptr;
    size_t vsplit_bytes = 0;
    float * vh, * vxn, * vqkv, * vg, * vattn, * vmg, * vmu, * vact, * vpart, * vpml;
    uint16_t * vxn16, * vattn16, * vact16;
    int * vtok;
    /* layer-input capture (model.rs:322-348, vq-model-gpu.cu:632-639):
     * cap_slot[li] is layer li's slot or -1; cap is [cap_n][max_ctx][hidden] */
    std::vector<int> cap_slot;
    int cap_n = 0;
    float * cap = nullptr;
};

size_t align256(size_t b) { return (b + 255) & ~(size_t) 255; }

/* the rotated prefix of a head: (head_dim * partial) as usize, at most head_dim (model.rs:419) */
int rope_dim(int hd, double partial) {
    const int d = (int) ((float) hd * (float) partial);
    return d > hd ? hd : d;
}

int check_launch(const char * what) {
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail_hip(what, e);
}

int gemv(const Model & m, const void * const * st, int rows, int cols, const void * x, float * y, int acc,
         hipStream_t s, int ncol = 1, int ldy = 0) {
    VqMatDesc d;
    memset(&d, 0, sizeof d);
    for (int i = 0; i < m.c.nstages; i++) d.stages[i] = st[i];
    d.y = y;
    d.rows = rows;
    VqCall c;
    memset(&c, 0, sizeof c);
    c.dim = m.c.dim; c.nc = m.c.nc; c.cols = cols; c.v3 = m.c.v3; c.nst = m.c.nstages;
    c.mats = &d; c.nmat = 1;
    c.x = x; c.ldx = cols; c.xf32 = m.c.x_dtype == SPARKMV_X_F32; c.ncol = ncol; c.ldy = ldy ? ldy : rows;
    c.accumulate = acc; c.stream = s;
    if (ncol > 1) {
        c.kslot = m.kslot;
        c.kslot_cap = m.kslot_cap;
    }
    const auto it = m.picks.find({rows, cols});
    if (it != m.picks.end()) { c.variant = it->second.first; c.threads = it->second.second; }
    return vq_launch(c);
}

int gemv2(const Model & m, const void * const * st0, int rows0, float * y0, const void * const * st1, int rows1,
          float * y1, int cols, const void * x, hipStream_t s, int ncol = 1, int ldy = 0) {
    VqMatDesc d[2];
    memset(d, 0, sizeof d);
    for (int i = 0; i < m.c.nstages; i++) { d[0].stages[i] = st0[i]; d[1].stages[i] = st1[i]; }
    d[0].y = y0; d[0].rows = rows0;
    d[1].y = y1; d[1].rows = rows1;
    VqCall c;
    memset(&c, 0, sizeof c);
    c.dim = m.c.dim; c.nc = m.c.nc; c.cols = cols; c.v3 = m.c.v3; c.nst = m.c.nstages;
    c.mats = d; c.nmat = 2;
    c.x = x; c.ldx = cols; c.xf32 = m.c.x_dtype == SPARKMV_X_F32; c.ncol = ncol; c.ldy = ldy ? ldy : rows0;
    c.accumulate = 0; c.stream = s;
    /* two matrices in one launch take a tuned kernel when both are tuned alike */
    const auto a = m.picks.find({rows0, cols}), b = m.picks.find({rows1, cols});
    if (a != m.picks.end() && b != m.picks.end() && a->second == b->second) {
        c.variant = a->second.first;
        c.threads = a->second.second;
    }
    return vq_launch(c);
}

/* rms_norm(h) * w into the bf16 activations, then the two matrices over
 * them: with bf16 activations and untuned kernels, ONE launch whose
 * workgroups stage the norm of h themselves (vq_norm_launch); otherwise the
 * norm launch and gemv2. */
int rmsnorm(const Model & m, const float * x, const float * w, hipStream_t s, int ncol = 1, float * out = nullptr,
            uint16_t * out16 = nullptr);

/* gate and up over the N columns of x (bf16 or f32 [N][cols]) into mg / mu
 * [N][rows], then act / act16 = gelu(gate) * up: written by the gate/up
 * launch itself where the several-column kernel takes the shape (bf16
 * activations, no tuning profile, the activation not switched apart), else
 * by the activation kernel. */
int gate_up_act_n(const Model & m, const void * const * gate, const void * const * up, int rows, int cols,
                  const void * x, float * mg, float * mu, float * act, uint16_t * act16, hipStream_t s, int N) {
    const bool b16 = m.c.x_dtype == SPARKMV_X_BF16;
    if (b16 && m.fuse_act && m.picks.empty()) {
        VqMatDesc d[2];
        memset(d, 0, sizeof d);
        for (int i = 0; i < m.c.nstages; i++) { d[0].stages[i] = gate[i]; d[1].stages[i] = up[i]; }
        d[0].y = mg; d[0].rows = rows;
        d[1].y = mu; d[1].rows = rows;
        VqCall c;
        memset(&c, 0, sizeof c);
        c.dim = m.c.dim; c.nc = m.c.nc; c.cols = cols; c.v3 = m.c.v3; c.nst = m.c.nstages;
        c.mats = d; c.nmat = 2;
        c.x = x; c.ldx = cols; c.xf32 = 0; c.ncol = N; c.ldy = rows;
        c.accumulate = 0; c.stream = s;
        const VqPair pair{m.pslot, rows * kMaxCols, act, act16};
        const int rc = vq_pair_launch(c, pair);
        if (rc <= 0) return rc;
    }
    if (gemv2(m, gate, rows, mg, up, rows, mu, cols, x, s, N, rows)) return -1;
    hipLaunchKernelGGL(fw_gelu_mul_kernel, dim3((N * rows / 4 + 255) / 256 + 1), dim3(256), 0, s, mg, mu, act, act16,
                       N * rows);
    return check_launch("gelu launch");
}

int norm_gemv2(const Model & m, const float * h, const float * w, const void * const * st0, int rows0, float * y0,
               const void * const * st1, int rows1, float * y1, int cols, hipStream_t s, const VqPair * pair = nullptr,
               bool * act_done = nullptr) {
    const bool b16 = m.c.x_dtype == SPARKMV_X_BF16;
    if (act_done) *act_done = false;
    VqMatDesc d[2];
    memset(d, 0, sizeof d);
    for (int i = 0; i < m.c.nstages; i++) { d[0].stages[i] = st0[i]; d[1].stages[i] = st1[i]; }
    d[0].y = y0; d[0].rows = rows0;
    d[1].y = y1; d[1].rows = rows1;
    VqCall c;
    memset(&c, 0, sizeof c);
    c.dim = m.c.dim; c.nc = m.c.nc; c.cols = cols; c.v3 = m.c.v3; c.nst = m.c.nstages;
    c.mats = d; c.nmat = 2;
    c.ncol = 1; c.ldy = rows0;
    c.accumulate = 0; c.stream = s;
    if (b16 && m.picks.empty()) {
        c.x = h; c.ldx = cols; c.xf32 = 1;
        if (pair) {
            /* one launch for the norm, both matrices and the activation */
            const int rc = vq_norm_launch(c, w, m.c.eps, nullptr, pair);
            if (rc <= 0) {
                if (rc == 0 && act_done) *act_done = true;
                return rc;
            }
        }
        const int rc = vq_norm_launch(c, w, m.c.eps, nullptr);
        if (rc <= 0) return rc;
    }
    if (rmsnorm(m, h, w, s, 1, nullptr, nullptr)) return -1;
    if (pair && b16 && m.picks.empty()) {
        c.x = m.xn16; c.ldx = cols; c.xf32 = 0;
        const int rc = vq_pair_launch(c, *pair);
        if (rc <= 0) {
            if (rc == 0 && act_done) *act_done = true;
            return rc;
        }
    }
    return gemv2(m, st0, rows0, y0, st1, rows1, y1, cols, b16 ? (const void *) m.xn16 : (const void *) m.xn, s);
}

int rmsnorm(const Model & m, const float * x, const float * w, hipStream_t s, int ncol, float * out,
            uint16_t * out16) {
    const bool b16 = m.c.x_dtype == SPARKMV_X_BF16;
    const int per = (m.c.hidden + 255) / 256;
    float * o = out ? out : m.xn;
    uint16_t * o16 = b16 ? (out16 ? out16 : m.xn16) : nullptr;
    const dim3 g((unsigned) ncol);
    if (per <= 4) hipLaunchKernelGGL(fw_rmsnorm_kernel<4>, g, dim3(256), 0, s, x, w, o, o16, m.c.hidden, m.c.eps);
    else if (per <= 12) hipLaunchKernelGGL(fw_rmsnorm_kernel<12>, g, dim3(256), 0, s, x, w, o, o16, m.c.hidden, m.c.eps);
    else if (per <= 32) hipLaunchKernelGGL(fw_rmsnorm_kernel<32>, g, dim3(256), 0, s, x, w, o, o16, m.c.hidden, m.c.eps);
    else { set_error("hidden %d is above 8192", m.c.hidden); return -1; }
    return check_launch("rms norm launch");
}

}  // namespace

}  // namespace sparkmv

using namespace sparkmv;

extern "C" {

void * sparkmv_model_create(const sparkmv_model_cfg * cfg) {
    if (!cfg) { set_error("model config is null"); return nullptr; }
    const sparkmv_model_cfg & c = *cfg;
    if (c.hidden <= 0 || c.layers <= 0 || c.heads <= 0 || c.kv_heads <= 0 || c.head_dim <= 0 || c.intermediate <= 0 ||
        c.vocab <= 0 || c.max_ctx <= 0 || c.sliding_window <= 0) {
        set_error("model config has a non-positive size");
        return nullptr;
    }
    if (c.heads % c.kv_heads) { set_error("heads %d is not a multiple of kv_heads %d", c.heads, c.kv_heads); return nullptr; }
    if (c.head_dim % 2) { set_error("head_dim %d is odd", c.head_dim); return nullptr; }
    if (c.x_dtype != SPARKMV_X_F32 && c.x_dtype != SPARKMV_X_BF16) { set_error("unknown x dtype %d", c.x_dtype); return nullptr; }
    if (c.nstages < 1 || c.nstages > 4) { set_error("stage count %d is outside 1..4", c.nstages); return nullptr; }
    if (!(c.eps > 0.0f)) { set_error("eps must be positive"); return nullptr; }
    if (c.head_dim != 64 && c.head_dim != 128 && c.head_dim != 256) {
        set_error("head_dim %d is not 64, 128 or 256", c.head_dim);
        return nullptr;
    }
    if (c.heads / c.kv_heads > 4) { set_error("more than 4 query heads per kv head"); return nullptr; }
    for (double partial : {c.rope_full_partial, c.rope_slide_partial}) {
        const int half = rope_dim(c.head_dim, partial) / 2;
        if (half % (c.head_dim / 64)) {
            set_error("rope half-width %d is not a multiple of head_dim / 64", half);
            return nullptr;
        }
    }
    /* the interface's limit (sparkmv.h); the kernels here hold kAttnSplits
     * partials per head whatever the length */
    constexpr int kMaxCtx = 131072;
    if (c.max_ctx > kMaxCtx) { set_error("max_ctx %d is above %d", c.max_ctx, kMaxCtx); return nullptr; }
    const long nch_max = ((long) c.max_ctx + kAttnChunk - 1) / kAttnChunk;
    if (c.hidden > 8192) { set_error("hidden %d is above 8192", c.hidden); return nullptr; }
    Model * m = new Model;
    m->c = c;
    m->layers.resize(c.layers);
    m->layer_set.assign(c.layers, 0);
    m->cap_slot.assign(c.layers, -1);
    const size_t qd = (size_t) c.heads * c.head_dim, kvd = (size_t) c.kv_heads * c.head_dim;
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += align256(bytes); return o; };
    const size_t o_h = take(c.hidden * 4), o_xn = take(c.hidden * 4), o_qkv = take((qd + 2 * kvd) * 4);
    const size_t o_g = take(c.heads * 4), o_attn = take(qd * 4), o_mg = take(c.intermediate * 4);
    const size_t o_mu = take(c.intermediate * 4), o_act = take(c.intermediate * 4);
    const size_t o_xn16 = take(c.hidden * 2), o_attn16 = take(qd * 2), o_act16 = take(c.intermediate * 2);
    const size_t o_kv = take((size_t) c.layers * c.max_ctx * kvd * 4 * 2);
    const size_t o_st = take(2 * sizeof(int));
    const size_t nsplit = nch_max < kAttnSplits ? (size_t) nch_max : kAttnSplits;
    const size_t o_part = take((size_t) c.heads * nsplit * c.head_dim * 4), o_pml = take((size_t) c.heads * nsplit * 8);
    const size_t o_rtab = take(512 * 4);
    const size_t n_pslot = (size_t) c.intermediate * kMaxCols;
    const size_t o_pslot = take(n_pslot * 8);
    const size_t n_kslot = (size_t) c.hidden * kMaxCols * vq_ck_words(kVqCkMaxGroups);
    const size_t o_kslot = take(n_kslot * 8);
    hipError_t e = hipMalloc(&m->mem, off);
    if (e != hipSuccess) {
        fail_hip("model buffers", e);
        delete m;
        return nullptr;
    }
    uint8_t * b = (uint8_t *) m->mem;
    e = hipMemset(b + o_pslot, 0, n_pslot * 8);
    if (e == hipSuccess) e = hipMemset(b + o_kslot, 0, n_kslot * 8);
    if (e != hipSuccess) {
        fail_hip("model exchange words", e);
        (void) hipFree(m->mem);
        delete m;
        return nullptr;
    }
    m->pslot = (uint64_t *) (b + o_pslot);
    m->kslot = (uint64_t *) (b + o_kslot);
    m->kslot_cap = (long) n_kslot;
    const char * sep = getenv("SPARKMV_SEPARATE_ACT");
    m->fuse_act = !(sep && sep[0] == '1');
    m->h = (float *) (b + o_h); m->xn = (float *) (b + o_xn); m->qkv = (float *) (b + o_qkv);
    m->g = (float *) (b + o_g); m->attn = (float *) (b + o_attn); m->mg = (float *) (b + o_mg);
    m->mu = (float *) (b + o_mu); m->act = (float *) (b + o_act);
    m->xn16 = (uint16_t *) (b + o_xn16); m->attn16 = (uint16_t *) (b + o_attn16); m->act16 = (uint16_t *) (b + o_act16);
    m->kv = (float *) (b + o_kv);
    m->st = (int *) (b + o_st);
    m->part = (float *) (b + o_part);
    m->pml = (float *) (b + o_pml);
    m->rtab = (float *) (b + o_rtab);
    m->nsplit = (int) nsplit;
    return m;
}

void sparkmv_model_destroy(void * model) {
    Model * m = (Model *) model;
    if (!m) return;
    if (m->exec) (void) hipGraphExecDestroy(m->exec);
    if (m->graph) (void) hipGraphDestroy(m->graph);
    if (m->mem) (void) hipFree(m->mem);
    if (m->vmem) (void) hipFree(m->vmem);
    if (m->cap) (void) hipFree(m->cap);
    for (void * p : m->owned) (void) hipFree(p);
    delete m;
}

int sparkmv_model_set_layer(void * model, int li, const sparkmv_model_layer * L) {
    Model * m = (Model *) model;
    if (!m || !L) { set_error("model or layer is null"); return -1; }
    if (li < 0 || li >= m->c.layers) { set_error("layer %d is outside 0..%d", li, m->c.layers - 1); return -1; }
    if (!L->in_norm || !L->post_norm) { set_error("layer %d has a null norm", li); return -1; }
    const void * const * mats[6] = {L->qkv, L->attn_gate, L->out, L->gate, L->up, L->down};
    for (int k = 0; k < 6; k++)
        for (int s = 0; s < m->c.nstages; s++)
            if (!mats[k][s]) { set_error("layer %d matrix %d stage %d is null", li, k, s); return -1; }
    m->layers[li] = *L;
    m->layer_set[li] = 1;
    return 0;
}

int sparkmv_model_set_head(void * model, int kind, const void * const * stages, const void * blocks,
                           const float * final_norm) {
    Model * m = (Model *) model;
    if (!m || !final_norm) { set_error("model or final norm is null"); return -1; }
    if (kind == 0) {
        if (!stages) { set_error("VQ head without stages"); return -1; }
        for (int s = 0; s < m->c.nstages; s++) {
            if (!stages[s]) { set_error("VQ head stage %d is null", s); return -1; }
            m->head_stages[s] = stages[s];
        }
    } else if (kind == 8) {
        if (!blocks) { set_error("Q8_0 head without blocks"); return -1; }
        if (m->c.hidden % 32) { set_error("a Q8_0 head needs hidden %% 32 == 0"); return -1; }
        m->head_blocks = blocks;
    } else {
        set_error("head kind %d is neither 0 (VQ) nor 8 (Q8_0)", kind);
        return -1;
    }
    m->head_kind = kind;
    m->final_norm = final_norm;
    return 0;
}

}  // extern "C"

int sparkmv::model_adopt(void * model, void * dev_ptr) {
    Model * m = (Model *) model;
    if (!m || !dev_ptr) { set_error("model or pointer is null"); return -1; }
    m->owned.push_back(dev_ptr);
    return 0;
}

namespace {

/* Layer li's input rows into its capture slot (model.rs:466-471, before the
 * layer runs; vq-model-gpu.cu:888-895): n rows of h at pos (from st[1] when
 * st is given). */
int capture_rows(const Model & m, int li, const float * h, const int * st, int pos, int n, hipStream_t s) {
    if (!m.cap_n || m.cap_slot[(size_t) li] < 0) return 0;
    float * slot = m.cap + (size_t) m.cap_slot[(size_t) li] * m.c.max_ctx * m.c.hidden;
    hipLaunchKernelGGL(fw_capture_kernel, dim3((m.c.hidden + 255) / 256, n), dim3(256), 0, s, h, slot, st, pos, n,
                       m.c.hidden);
    return check_launch("capture launch");
}

int ready(const Model * m) {
    if (m->head_kind < 0) { set_error("the model has no head"); return -1; }
    for (int li = 0; li < m->c.layers; li++)
        if (!m->layer_set[li]) { set_error("layer %d has no weights", li); return -1; }
    return 0;
}

int check_step(const Model * m, uint32_t token, int pos) {
    if ((long) token >= m->c.vocab) { set_error("token %u is outside the vocabulary", token); return -1; }
    if (pos < 0 || pos >= m->c.max_ctx) { set_error("position %d exceeds the %d-token cache", pos, m->c.max_ctx); return -1; }
    return 0;
}

int set_state(Model * m, uint32_t token, int pos, hipStream_t s) {
    const sparkmv_model_cfg & c = m->c;
    hipLaunchKernelGGL(fw_set_state_kernel, dim3(1), dim3(128), 0, s, m->st, (int) token, pos,
                       (float) c.rope_full_theta, rope_dim(c.head_dim, c.rope_full_partial), (float) c.rope_slide_theta,
                       rope_dim(c.head_dim, c.rope_slide_partial), m->rtab);
    return check_launch("state launch");
}

/* The split attention and its combine for one decode token (dec) or the
 * block's A.N tokens, whose windows span at most `span` positions. */
int attn_launch(const AttnArgs & A, int hd, int span, const float * gate, int ldg, float * out, uint16_t * out16,
                bool dec, hipStream_t s) {
    const int tiles = (span + kAttnChunk - 1) / kAttnChunk;
    const dim3 grid((unsigned) (tiles < A.nsplit ? tiles : A.nsplit), (unsigned) A.kv_heads,
                    (unsigned) ((A.N * (A.heads / A.kv_heads) + 15) / 16)), b(256);
#define FW_ATTN(H)                                                                                                   \
    do {                                                                                                             \
        if (dec) hipLaunchKernelGGL((fw_attn_split_kernel<H, 1>), grid, b, 0, s, A);                                 \
        else hipLaunchKernelGGL((fw_attn_split_kernel<H, 0>), grid, b, 0, s, A);                                     \
        hipLaunchKernelGGL(fw_attn_combine_kernel<H / 64>, dim3(A.heads, A.N), dim3(512), 0, s, A, dec ? 1 : 0, gate, \
                           ldg, out, out16);                                                                         \
    } while (0)
    if (hd == 64) FW_ATTN(64);
    else if (hd == 128) FW_ATTN(128);
    else FW_ATTN(256);
#undef FW_ATTN
    return check_launch("attention launch");
}

/* Every launch of one token, reading token and position from m->st. */
int chain(Model * m, float * logits, hipStream_t s) {
    const sparkmv_model_cfg & c = m->c;
    const bool b16 = c.x_dtype == SPARKMV_X_BF16;
    const int qd = c.heads * c.head_dim, kvd = c.kv_heads * c.head_dim, hd = c.head_dim;

    /* the embedding row (model.rs:462-464): the tied head's row `token` */
    if (m->head_kind == 0) {
        hipLaunchKernelGGL(fw_fill_kernel, dim3((c.hidden + 255) / 256), dim3(256), 0, s, m->h, c.hidden, 0.0f);
        if (check_launch("fill launch")) return -1;
        const Layout L = make_layout(c.dim, c.nc, c.vocab, c.hidden, c.v3);
        for (int st = 0; st < c.nstages; st++)
            if (vq_row_dequant_dev_launch(m->head_stages[st], L, m->st, m->h, s)) return -1;
    } else {
        hipLaunchKernelGGL(fw_q8_0_row_kernel, dim3((c.hidden + 255) / 256), dim3(256), 0, s,
                           (const uint8_t *) m->head_blocks, c.hidden, (const int *) m->st, m->h);
        if (check_launch("embedding launch")) return -1;
    }

    const float scale = 1.0f / sqrtf((float) hd);
    for (int li = 0; li < c.layers; li++) {
        const sparkmv_model_layer & L = m->layers[li];
        const bool full = L.full != 0;
        float * kc = m->kv + (size_t) li * 2 * c.max_ctx * kvd;
        float * vc = kc + (size_t) c.max_ctx * kvd;

        if (capture_rows(*m, li, m->h, m->st, 0, 1, s)) return -1;
        if (norm_gemv2(*m, m->h, L.in_norm, L.qkv, qd + 2 * kvd, m->qkv, L.attn_gate, c.heads, m->g, c.hidden, s))
            return -1;

        /* rope, the KV store and attention (model.rs:484-557), launched for
         * the longest window this layer can see */
        const int pdim = rope_dim(hd, full ? c.rope_full_partial : c.rope_slide_partial);
        const float * rtab = m->rtab + (full ? 0 : 256);
        const int span = full || c.sliding_window > c.max_ctx ? c.max_ctx : c.sliding_window;
        AttnArgs at;
        at.qkv = m->qkv; at.kc = kc; at.vc = vc; at.st = m->st; at.rtab = rtab; at.po = m->part; at.pml = m->pml;
        at.ldq = qd + 2 * kvd; at.qd = qd; at.kvd = kvd; at.pos0 = 0; at.N = 1; at.window = full ? 0 : c.sliding_window;
        at.heads = c.heads; at.kv_heads = c.kv_heads; at.pdim = pdim; at.nsplit = m->nsplit; at.scale = scale;
        if (attn_launch(at, hd, span, m->g, 1, m->attn, b16 ? m->attn16 : nullptr, true, s)) return -1;
        if (gemv(*m, L.out, c.hidden, qd, b16 ? (const void *) m->attn16 : (const void *) m->attn, m->h, 1, s))
            return -1;

        /* MLP (model.rs:566-581): the gate/up launch writes the activation
         * itself when its shape allows, else the activation kernel does */
        const VqPair pair{m->pslot, c.intermediate, m->act, b16 ? m->act16 : nullptr};
        bool act_done = false;
        if (norm_gemv2(*m, m->h, L.post_norm, L.gate, c.intermediate, m->mg, L.up, c.intermediate, m->mu, c.hidden, s,
                       m->fuse_act ? &pair : nullptr, &act_done))
            return -1;
        if (!act_done) {
            hipLaunchKernelGGL(fw_gelu_mul_kernel, dim3((c.intermediate / 4 + 255) / 256 + 1), dim3(256), 0, s, m->mg,
                               m->mu, m->act, b16 ? m->act16 : nullptr, c.intermediate);
            if (check_launch("gelu launch")) return -1;
        }
        if (gemv(*m, L.down, c.hidden, c.intermediate, b16 ? (const void *) m->act16 : (const void *) m->act, m->h,
                 1, s))
            return -1;
    }

    /* final norm and the tied head (model.rs:583-590) */
    if (rmsnorm(*m, m->h, m->final_norm, s)) return -1;
    const void * xin = b16 ? (const void *) m->xn16 : (const void *) m->xn;
    if (m->head_kind == 0) return gemv(*m, m->head_stages, c.vocab, c.hidden, xin, logits, 0, s);
    return kq_gemv_launch(8, m->head_blocks, c.vocab, c.hidden, xin, b16 ? 0 : 1, c.hidden, 1, logits, c.vocab, 0, s);
}

/* The block buffers for up to cap tokens (at least 8). A smaller or equal
 * reservation keeps what is there; a larger one replaces it (the caller
 * synchronizes first: work in flight may still use the old buffers). */
int alloc_block(Model * m, int cap) {
    cap = cap < 8 ? 8 : cap;
    if (m->vmem && cap <= m->vcap) return 0;
    const sparkmv_model_cfg & c = m->c;
    const size_t qd = (size_t) c.heads * c.head_dim, kvd = (size_t) c.kv_heads * c.head_dim, N = (size_t) cap;
    size_t off = 0;
    auto take = [&](size_t bytes) { const size_t o = off; off += align256(bytes); return o; };
    const size_t o_h = take(N * c.hidden * 4), o_xn = take(N * c.hidden * 4), o_qkv = take(N * (qd + 2 * kvd) * 4);
    const size_t o_g = take(N * (qd + 2 * kvd) * 4), o_attn = take(N * qd * 4), o_mg = take(N * c.intermediate * 4);
    const size_t o_mu = take(N * c.intermediate * 4), o_act = take(N * c.intermediate * 4);
    const size_t o_xn16 = take(N * c.hidden * 2), o_attn16 = take(N * qd * 2), o_act16 = take(N * c.intermediate * 2);
    const size_t o_part = take((size_t) 8 * c.heads * m->nsplit * c.head_dim * 4);
    const size_t o_pml = take((size_t) 8 * c.heads * m->nsplit * 8);
    const size_t o_tok = take(N * sizeof(int));
    size_t split = 0;
    if (cap > kMaxCols) {
        const int n = cap < kPromptMax ? cap : kPromptMax, ldq = (int) (qd + 2 * kvd);
        const int shapes[][2] = {{ldq, c.hidden}, {c.heads, c.hidden}, {c.hidden, (int) qd}, {c.intermediate, c.hidden},
                                 {c.hidden, c.intermediate}};
        for (const auto & rc : shapes) {
            const size_t b = prefill_split_bytes(rc[0], rc[1], n);
            split = b > split ? b : split;
        }
    }
    const size_t o_split = take(split);
    void * mem = nullptr;
    hipError_t e = hipMalloc(&mem, off);
    if (e != hipSuccess) return fail_hip("block buffers", e);
    if (m->vmem) (void) hipFree(m->vmem);
    m->vmem = mem;
    m->vcap = cap;
    uint8_t * b = (uint8_t *) m->vmem;
    m->vsplit = split ? b + o_split : nullptr;
    m->vsplit_bytes = split;
    m->vh = (float *) (b + o_h); m->vxn = (float *) (b + o_xn); m->vqkv = (float *) (b + o_qkv);
    m->vg = (float *) (b + o_g); m->vattn = (float *) (b + o_attn); m->vmg = (float *) (b + o_mg);
    m->vmu = (float *) (b + o_mu); m->vact = (float *) (b + o_act); m->vpart = (float *) (b + o_part);
    m->vpml = (float *) (b + o_pml);
    m->vxn16 = (uint16_t *) (b + o_xn16); m->vattn16 = (uint16_t *) (b + o_attn16);
    m->vact16 = (uint16_t *) (b + o_act16);
    m->vtok = (int *) (b + o_tok);
    return 0;
}

/* y[t * ldy + r] (+)= W x_t for N tokens of x ([N][cols], the model's x
 * dtype): up to kMaxCols tokens through the batched GEMV (each column the
 * decode arithmetic), more through the prefill GEMM (the reference's prompt
 * path, vq-model-gpu.cu:838-851: x enters the matrix cores as f16). */
int mat_n(const Model & m, const void * const * st, int rows, int cols, const void * x, float * y, int acc,
          hipStream_t s, int N, int ldy) {
    if (N <= kMaxCols) return gemv(m, st, rows, cols, x, y, acc, s, N, ldy);
    const Layout L = make_layout(m.c.dim, m.c.nc, rows, cols, m.c.v3);
    const int xf32 = m.c.x_dtype == SPARKMV_X_F32;
    if (m.c.nstages <= 2 && prefill_mfma_ready(L, m.c.nstages, x, xf32, cols, 0, N))
        return prefill_mfma_launch(st, m.c.nstages, L, x, xf32, cols, 0, N, y, ldy, acc, s, m.vsplit, m.vsplit_bytes);
    return prefill_simple_launch(st, m.c.nstages, L, x, xf32, (size_t) cols, 1, N, y, ldy, acc, s);
}

/* Rope and the KV store of N tokens at pos0 .. pos0 + N - 1 (rows of qkv at
 * stride ldq), the shape chosen by N. */
int rope_kv_launch(float * qkv, int N, int ldq, int qd, int kvd, int heads, int kv_heads, int hd, int pdim,
                          float theta, int pos0, float * kc, float * vc, hipStream_t s) {
    if (N <= kMaxCols)
        hipLaunchKernelGGL(fw_rope_kv_heads_kernel, dim3(N, heads + kv_heads), dim3(128), 0, s, qkv, ldq, qd, kvd,
                           heads, hd, pdim, theta, pos0, kc, vc);
    else
        hipLaunchKernelGGL(fw_rope_kv_n_kernel, dim3(N), dim3(256), 0, s, qkv, ldq, qd, kvd, heads, kv_heads, hd,
                           pdim, theta, pos0, kc, vc);
    return check_launch("rope launch");
}

/* A verify block: the forward of ntok consecutive tokens at pos .. pos + ntok - 1
 * with every matvec over ntok columns (weights decoded once for the block),
 * then the head over the same columns; logits are [ntok][vocab]. */
int block(Model * m, const uint32_t * tokens, int N, int pos, float * logits, hipStream_t s) {
    const sparkmv_model_cfg & c = m->c;
    const bool b16 = c.x_dtype == SPARKMV_X_BF16;
    const int qd = c.heads * c.head_dim, kvd = c.kv_heads * c.head_dim, hd = c.head_dim, ldq = qd + 2 * kvd;
    FwTok8 tk;
    for (int t = 0; t < 8; t++) tk.t[t] = t < N ? (int) tokens[t] : 0;
    if (m->head_kind == 0) {
        hipLaunchKernelGGL(fw_fill_kernel, dim3((N * c.hidden + 255) / 256), dim3(256), 0, s, m->vh, N * c.hidden, 0.0f);
        if (check_launch("fill launch")) return -1;
        const Layout L = make_layout(c.dim, c.nc, c.vocab, c.hidden, c.v3);
        for (int t = 0; t < N; t++)
            for (int st = 0; st < c.nstages; st++)
                if (vq_row_dequant_launch(m->head_stages[st], L, (int) tokens[t], m->vh + (size_t) t * c.hidden, s))
                    return -1;
    } else {
        hipLaunchKernelGGL(fw_q8_0_rows_kernel, dim3((c.hidden + 255) / 256, N), dim3(256), 0, s,
                           (const uint8_t *) m->head_blocks, c.hidden, tk, m->vh);
        if (check_launch("embedding launch")) return -1;
    }
    const float scale = 1.0f / sqrtf((float) hd);
    const void * xin = b16 ? (const void *) m->vxn16 : (const void *) m->vxn;
    for (int li = 0; li < c.layers; li++) {
        const sparkmv_model_layer & L = m->layers[li];
        const bool full = L.full != 0;
        float * kc = m->kv + (size_t) li * 2 * c.max_ctx * kvd;
        float * vc = kc + (size_t) c.max_ctx * kvd;
        if (capture_rows(*m, li, m->vh, nullptr, pos, N, s)) return -1;
        if (rmsnorm(*m, m->vh, L.in_norm, s, N, m->vxn, m->vxn16)) return -1;
        if (gemv2(*m, L.qkv, ldq, m->vqkv, L.attn_gate, c.heads, m->vg, c.hidden, xin, s, N, ldq)) return -1;
        const double theta = full ? c.rope_full_theta : c.rope_slide_theta;
        const int pdim = rope_dim(hd, full ? c.rope_full_partial : c.rope_slide_partial);
        if (rope_kv_launch(m->vqkv, N, ldq, qd, kvd, c.heads, c.kv_heads, hd, pdim, (float) theta, pos, kc, vc, s))
            return -1;
        AttnArgs at;
        at.qkv = m->vqkv; at.kc = kc; at.vc = vc; at.st = nullptr; at.rtab = nullptr; at.po = m->vpart; at.pml = m->vpml;
        at.ldq = ldq; at.qd = qd; at.kvd = kvd; at.pos0 = pos; at.N = N; at.window = full ? 0 : c.sliding_window;
        at.heads = c.heads; at.kv_heads = c.kv_heads; at.pdim = pdim; at.nsplit = m->nsplit; at.scale = scale;
        /* the block's positions: from the first token's window start to the last token */
        const int span = full || pos + 1 < c.sliding_window ? pos + N : c.sliding_window + N - 1;
        if (attn_launch(at, hd, span, m->vg, ldq, m->vattn, b16 ? m->vattn16 : nullptr, false, s)) return -1;
        if (gemv(*m, L.out, c.hidden, qd, b16 ? (const void *) m->vattn16 : (const void *) m->vattn, m->vh, 1, s, N,
                 c.hidden))
            return -1;
        if (rmsnorm(*m, m->vh, L.post_norm, s, N, m->vxn, m->vxn16)) return -1;
        if (gate_up_act_n(*m, L.gate, L.up, c.intermediate, c.hidden, xin, m->vmg, m->vmu, m->vact,
                          b16 ? m->vact16 : nullptr, s, N))
            return -1;
        if (gemv(*m, L.down, c.hidden, c.intermediate, b16 ? (const void *) m->vact16 : (const void *) m->vact, m->vh,
                 1, s, N, c.hidden))
            return -1;
    }
    if (rmsnorm(*m, m->vh, m->final_norm, s, N, m->vxn, m->vxn16)) return -1;
    /* the head over the block's columns; the Q8_0 kernel gives each column
     * exactly its one-column result (the verify-head requirement,
     * Spark-X2.6-4B-Base-handoff.md:299-302) */
    if (m->head_kind == 0) return gemv(*m, m->head_stages, c.vocab, c.hidden, xin, logits, 0, s, N, c.vocab);
    return kq_gemv_launch(8, m->head_blocks, c.vocab, c.hidden, xin, b16 ? 0 : 1, c.hidden, N, logits, c.vocab, 0, s);
}

/* Span splits of the split-product prompt attention for a chunk, or 0 where
 * it does not run: full layers, four query heads per kv head, and a span of
 * 2048 positions, whatever the chunk. Below, the partials and two more
 * launches take what the products save (whole prompt call of the four-layer
 * model, 33 tokens at 1500: 1155-1184 us without, 1158-1224 with it). From
 * there on no chunk is slower: 3, 9, 16 and 64 tokens at 2048 523, 690, 824
 * and 821 us without, 487, 682, 817 and 818 with it; 3, 9, 16 and 33 at 4096
 * 586, 604, 678 and 862, and 496, 573, 648 and 843; 9 at 16000 1093 and 936;
 * 512 at 16384 2901 and 2050. As many splits as fill the CUs,
 * leave a split 256 positions and fit the FFN's buffers. */
int prompt_splits(const Model & m, int N, int pos, int window) {
    const sparkmv_model_cfg & c = m.c;
    const int span = pos + N;
    if (window > 0 || c.heads != 4 * c.kv_heads || span < 2048) return 0;
    const int wgs = c.kv_heads * ((N + kPsTok - 1) / kPsTok);
    const size_t one = (size_t) N * (c.heads * 256 + 2 * c.heads) + (size_t) wgs, room = (size_t) (m.vact - m.vmg);
    int n = (cu_count() + wgs - 1) / wgs;
    if (n > span / 256) n = span / 256;
    if (n > kPsMaxSplit) n = kPsMaxSplit;
    if ((size_t) n * one > room) n = (int) (room / one);
    return n;
}

int prompt_split_launch(const float * qkv, int ldq, int kvd, const float * kc, const float * vc, int pos, int N,
                        int heads, int kv_heads, float scale, int nz, float * po, float * pml, uint32_t * redo,
                        hipStream_t s) {
    static LdsAllowed allowed;
    if (lds_allow(allowed, (const void *) fw_attn_prompt_split_kernel, kPsLds,
                  "LDS opt-in for the split prompt attention"))
        return -1;
    hipLaunchKernelGGL(fw_attn_prompt_split_kernel,
                       dim3((unsigned) nz, (unsigned) ((N + kPsTok - 1) / kPsTok), (unsigned) kv_heads), dim3(512),
                       kPsLds, s, qkv, ldq, kvd, kc, vc, pos, N, heads, scale, po, pml, redo);
    return check_launch("split prompt attention launch");
}

/* A prompt chunk (vq-model-gpu.cu:858-943 forward_batch): N tokens at
 * pos .. pos + N - 1 through every layer, the tokens already in m->vtok.
 * With logits, the final norm and the head of the last token
 * (vq-model-gpu.cu:946-953 tail_logits). */
int prompt(Model * m, int N, int pos, float * logits, hipStream_t s) {
    const sparkmv_model_cfg & c = m->c;
    const bool b16 = c.x_dtype == SPARKMV_X_BF16;
    const int qd = c.heads * c.head_dim, kvd = c.kv_heads * c.head_dim, hd = c.head_dim, ldq = qd + 2 * kvd;
    if (m->head_kind == 0) {
        hipLaunchKernelGGL(fw_fill_kernel, dim3((N * c.hidden + 255) / 256), dim3(256), 0, s, m->vh, N * c.hidden, 0.0f);
        if (check_launch("fill launch")) return -1;
        const Layout L = make_layout(c.dim, c.nc, c.vocab, c.hidden, c.v3);
        for (int st = 0; st < c.nstages; st++)
            if (vq_row_dequant_dev_launch(m->head_stages[st], L, m->vtok, m->vh, s, N, (size_t) c.hidden)) return -1;
    } else {
        hipLaunchKernelGGL(fw_q8_0_rows_dev_kernel, dim3((c.hidden + 255) / 256, N), dim3(256), 0, s,
                           (const uint8_t *) m->head_blocks, c.hidden, (const int *) m->vtok, m->vh);
        if (check_launch("embedding launch")) return -1;
    }
    const float scale = 1.0f / sqrtf((float) hd);
    const void * xin = b16 ? (const void *) m->vxn16 : (const void *) m->vxn;
    for (int li = 0; li < c.layers; li++) {
        const sparkmv_model_layer & L = m->layers[li];
        const bool full = L.full != 0;
        float * kc = m->kv + (size_t) li * 2 * c.max_ctx * kvd;
        float * vc = kc + (size_t) c.max_ctx * kvd;
        if (capture_rows(*m, li, m->vh, nullptr, pos, N, s)) return -1;
        if (rmsnorm(*m, m->vh, L.in_norm, s, N, m->vxn, m->vxn16)) return -1;
        if (N <= kMaxCols) {
            if (gemv2(*m, L.qkv, ldq, m->vqkv, L.attn_gate, c.heads, m->vg, c.hidden, xin, s, N, ldq)) return -1;
        } else {
            if (mat_n(*m, L.qkv, ldq, c.hidden, xin, m->vqkv, 0, s, N, ldq)) return -1;
            if (mat_n(*m, L.attn_gate, c.heads, c.hidden, xin, m->vg, 0, s, N, ldq)) return -1;
        }
        const double theta = full ? c.rope_full_theta : c.rope_slide_theta;
        const int pdim = rope_dim(hd, full ? c.rope_full_partial : c.rope_slide_partial);
        if (rope_kv_launch(m->vqkv, N, ldq, qd, kvd, c.heads, c.kv_heads, hd, pdim, (float) theta, pos, kc, vc, s))
            return -1;
        const int window = full ? 0 : c.sliding_window;
        const dim3 ag((unsigned) c.kv_heads, (unsigned) N), ab((unsigned) (64 * (c.heads / c.kv_heads)));
        uint16_t * a16 = b16 ? m->vattn16 : nullptr;
        const int psplit = hd == 256 ? prompt_splits(*m, N, pos, window) : 0;
        uint32_t * redo = nullptr;
        if (psplit > 0) {
            /* partials in the FFN's buffers, idle here */
            float * po = m->vmg, * pml = po + (size_t) psplit * N * qd;
            redo = (uint32_t *) (pml + (size_t) psplit * N * c.heads * 2);
            if (prompt_split_launch(m->vqkv, ldq, kvd, kc, vc, pos, N, c.heads, c.kv_heads, scale, psplit, po, pml,
                                    redo, s))
                return -1;
            hipLaunchKernelGGL(fw_attn_prompt_merge_kernel, dim3((unsigned) N, (unsigned) ((c.heads + 3) / 4)), dim3(256),
                               0, s, po, pml, psplit, N, c.heads, m->vg, ldq, m->vattn, a16);
            if (check_launch("prompt attention merge launch")) return -1;
        }
        if (hd == 256) {
            hipLaunchKernelGGL(fw_attn_prompt_mfma_kernel, dim3((unsigned) c.heads, (unsigned) ((N + kPaTok - 1) / kPaTok)),
                               dim3(256), 0, s, m->vqkv, ldq, kvd, kc, vc, m->vg, ldq, pos, N, window,
                               c.heads, c.kv_heads, scale, m->vattn, a16, (const uint32_t *) redo, psplit);
        }
        else if (hd == 64)
            hipLaunchKernelGGL(fw_attn_prompt_kernel<1>, ag, ab, 0, s, m->vqkv, ldq, kvd, kc, vc, m->vg, ldq, pos,
                               window, c.heads, c.kv_heads, scale, m->vattn, a16);
        else if (hd == 128)
            hipLaunchKernelGGL(fw_attn_prompt_kernel<2>, ag, ab, 0, s, m->vqkv, ldq, kvd, kc, vc, m->vg, ldq, pos,
                               window, c.heads, c.kv_heads, scale, m->vattn, a16);
        else
            hipLaunchKernelGGL(fw_attn_prompt_kernel<4>, ag, ab, 0, s, m->vqkv, ldq, kvd, kc, vc, m->vg, ldq, pos,
                               window, c.heads, c.kv_heads, scale, m->vattn, a16);
        if (check_launch("attention launch")) return -1;
        if (mat_n(*m, L.out, c.hidden, qd, b16 ? (const void *) m->vattn16 : (const void *) m->vattn, m->vh, 1, s, N,
                  c.hidden))
            return -1;
        if (rmsnorm(*m, m->vh, L.post_norm, s, N, m->vxn, m->vxn16)) return -1;
        if (N <= kMaxCols) {
            if (gate_up_act_n(*m, L.gate, L.up, c.intermediate, c.hidden, xin, m->vmg, m->vmu, m->vact,
                              b16 ? m->vact16 : nullptr, s, N))
                return -1;
        } else {
            if (mat_n(*m, L.gate, c.intermediate, c.hidden, xin, m->vmg, 0, s, N, c.intermediate)) return -1;
            if (mat_n(*m, L.up, c.intermediate, c.hidden, xin, m->vmu, 0, s, N, c.intermediate)) return -1;
            /* bf16: down reads act16 only, so the f32 copy is not written */
            hipLaunchKernelGGL(fw_gelu_mul_kernel, dim3((N * c.intermediate / 4 + 255) / 256 + 1), dim3(256), 0, s,
                               m->vmg, m->vmu, b16 ? nullptr : m->vact, b16 ? m->vact16 : nullptr,
                               N * c.intermediate);
            if (check_launch("gelu launch")) return -1;
        }
        if (mat_n(*m, L.down, c.hidden, c.intermediate, b16 ? (const void *) m->vact16 : (const void *) m->vact, m->vh,
                  1, s, N, c.hidden))
            return -1;
    }
    if (!logits) return 0;
    /* the last token's row: final norm and the head, as one decode step's */
    if (rmsnorm(*m, m->vh + (size_t) (N - 1) * c.hidden, m->final_norm, s, 1, m->vxn, m->vxn16)) return -1;
    if (m->head_kind == 0) return gemv(*m, m->head_stages, c.vocab, c.hidden, xin, logits, 0, s);
    return kq_gemv_launch(8, m->head_blocks, c.vocab, c.hidden, xin, b16 ? 0 : 1, c.hidden, 1, logits, c.vocab, 0, s);
}

}  // namespace

extern "C" {

int sparkmv_model_forward(void * model, uint32_t token, int pos, float * logits, void * stream) {
    Model * m = (Model *) model;
    if (!m || !logits) { set_error("model or logits is null"); return -1; }
    if (check_step(m, token, pos) || ready(m)) return -1;
    hipStream_t s = (hipStream_t) stream;
    if (set_state(m, token, pos, s)) return -1;
    if (chain(m, logits, s)) return -1;
    m->len = pos + 1;
    return 0;
}

int sparkmv_model_capture(void * model, float * logits, void * stream) {
    Model * m = (Model *) model;
    if (!m || !logits) { set_error("model or logits is null"); return -1; }
    if (!stream) { set_error("capture needs a created stream, not the null stream"); return -1; }
    if (ready(m)) return -1;
    hipStream_t s = (hipStream_t) stream;
    hipError_t e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return fail_hip("begin capture", e);
    const int rc = chain(m, logits, s);
    hipGraph_t g = nullptr;
    e = hipStreamEndCapture(s, &g);
    if (rc) { if (g) (void) hipGraphDestroy(g); return -1; }
    if (e != hipSuccess) return fail_hip("end capture", e);
    hipGraphExec_t x = nullptr;
    e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    if (e != hipSuccess) { (void) hipGraphDestroy(g); return fail_hip("graph instantiate", e); }
    if (m->exec) (void) hipGraphExecDestroy(m->exec);
    if (m->graph) (void) hipGraphDestroy(m->graph);
    m->graph = g;
    m->exec = x;
    return 0;
}

int sparkmv_model_replay(void * model, uint32_t token, int pos, void * stream) {
    Model * m = (Model *) model;
    if (!m) { set_error("model is null"); return -1; }
    if (!m->exec) { set_error("the model has no recorded forward: call sparkmv_model_capture first"); return -1; }
    if (check_step(m, token, pos)) return -1;
    hipStream_t s = (hipStream_t) stream;
    if (set_state(m, token, pos, s)) return -1;
    hipError_t e = hipGraphLaunch(m->exec, s);
    if (e != hipSuccess) return fail_hip("graph launch", e);
    m->len = pos + 1;
    return 0;
}

int sparkmv_model_verify(void * model, const uint32_t * tokens, int ntok, int pos, float * logits, void * stream) {
    Model * m = (Model *) model;
    if (!m || !tokens || !logits) { set_error("model, tokens or logits is null"); return -1; }
    if (ntok < 1 || ntok > 8) { set_error("a verify block holds 1..8 tokens, not %d", ntok); return -1; }
    if (pos < 0 || pos + ntok > m->c.max_ctx) {
        set_error("positions %d..%d exceed the %d-token cache", pos, pos + ntok - 1, m->c.max_ctx);
        return -1;
    }
    for (int t = 0; t < ntok; t++)
        if ((long) tokens[t] >= m->c.vocab) { set_error("token %u is outside the vocabulary", tokens[t]); return -1; }
    if (ready(m)) return -1;
    if (!m->vmem && alloc_block(m, 8)) return -1;
    if (block(m, tokens, ntok, pos, logits, (hipStream_t) stream)) return -1;
    m->len = pos + ntok;
    return 0;
}

int sparkmv_model_reserve(void * model, int ntok) {
    Model * m = (Model *) model;
    if (!m) { set_error("model is null"); return -1; }
    if (ntok < 1 || ntok > kPromptMax) { set_error("a reservation covers 1..%d tokens, not %d", kPromptMax, ntok); return -1; }
    if (m->vmem && ntok > m->vcap) {
        /* the old buffers may still be in use by queued work */
        hipError_t e = hipDeviceSynchronize();
        if (e != hipSuccess) return fail_hip("synchronize before a larger reservation", e);
    }
    return alloc_block(m, ntok);
}

int sparkmv_model_forward_batch(void * model, const uint32_t * tokens, int ntok, int pos, float * logits,
                                void * stream) {
    Model * m = (Model *) model;
    if (!m || !tokens) { set_error("model or tokens is null"); return -1; }
    if (ntok < 1 || ntok > kPromptMax) { set_error("a prompt chunk holds 1..%d tokens, not %d", kPromptMax, ntok); return -1; }
    if (pos < 0 || pos + ntok > m->c.max_ctx) {
        set_error("positions %d..%d exceed the %d-token cache", pos, pos + ntok - 1, m->c.max_ctx);
        return -1;
    }
    for (int t = 0; t < ntok; t++)
        if ((long) tokens[t] >= m->c.vocab) { set_error("token %u is outside the vocabulary", tokens[t]); return -1; }
    if (ready(m)) return -1;
    if (!m->vmem || ntok > m->vcap) {
        if (m->vmem) {
            hipError_t e = hipDeviceSynchronize();
            if (e != hipSuccess) return fail_hip("synchronize before larger block buffers", e);
        }
        if (alloc_block(m, ntok)) return -1;
    }
    hipStream_t s = (hipStream_t) stream;
    /* the tokens go to device memory on the stream; the host array is read
     * before the call returns */
    static_assert(sizeof(uint32_t) == sizeof(int), "token width");
    hipError_t e = hipMemcpyAsync(m->vtok, tokens, (size_t) ntok * sizeof(int), hipMemcpyHostToDevice, s);
    if (e != hipSuccess) return fail_hip("token upload", e);
    e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail_hip("token upload", e);
    if (prompt(m, ntok, pos, logits, s)) return -1;
    m->len = pos + ntok;
    return 0;
}

int sparkmv_model_rollback(void * model, int pos) {
    Model * m = (Model *) model;
    if (!m) { set_error("model is null"); return -1; }
    if (pos < 0 || pos > m->len) { set_error("rollback to %d exceeds the %d cached positions", pos, m->len); return -1; }
    m->len = pos;
    return 0;
}

int sparkmv_model_len(void * model) {
    Model * m = (Model *) model;
    return m ? m->len : -1;
}

/* Apply a trusted tuning profile to the model's VQ matvecs, per geometry,
 * as the reference's loader does (tools/vq/gpu/vq-model-gpu.cu:300-324): a
 * geometry with a runnable gemv entry takes its kernel and width; an entry
 * that is not runnable here leaves the heuristic; an untrusted profile
 * changes nothing. Returns the number of geometries tuned, or -1. Drops a
 * captured graph (capture again to replay the tuned kernels). */
int sparkmv_model_apply_profile(void * model, const void * profile, uint64_t artifact, const char * gpu) {
    Model * m = (Model *) model;
    if (!m || !profile || !gpu) { set_error("model, profile or gpu name is null"); return -1; }
    const int t = sparkmv_profile_trusted(profile, artifact, gpu);
    if (t < 0) return -1;
    if (t == 0) {
        set_error("profile: measured for another artifact or device; the heuristic stays");
        return 0;
    }
    const auto & c = m->c;
    const int qd = c.heads * c.head_dim, kvd = c.kv_heads * c.head_dim;
    const int geoms[][2] = {{qd + 2 * kvd, c.hidden}, {c.heads, c.hidden}, {c.hidden, qd},
                            {c.intermediate, c.hidden}, {c.hidden, c.intermediate}, {c.vocab, c.hidden}};
    int applied = 0, refused = 0;
    m->picks.clear();
    for (const auto & g : geoms) {
        if (m->picks.count({g[0], g[1]})) continue;
        int v = 0, th = 0;
        const int r = profile_gemv_pick(profile, c.dim, c.nc, g[0], g[1], c.v3, &v, &th);
        if (r < 0) refused++;
        if (r == 1) {
            m->picks[{g[0], g[1]}] = {v, th};
            applied++;
        }
    }
    if (m->exec) { (void) hipGraphExecDestroy(m->exec); m->exec = nullptr; }
    if (m->graph) { (void) hipGraphDestroy(m->graph); m->graph = nullptr; }
    set_error("profile: %d geometries take their tuned kernel, %d entries are not runnable here (heuristic kept)",
              applied, refused);
    return applied;
}

/* The kernel the model runs for a (rows, cols) VQ matvec: variant and width
 * as sparkmv_plan_op_kernel reports them (0, 0 = the heuristic). */
int sparkmv_model_matvec_kernel(void * model, int rows, int cols, int * variant, int * threads) {
    Model * m = (Model *) model;
    if (!m) { set_error("model is null"); return -1; }
    const auto it = m->picks.find({rows, cols});
    if (variant) *variant = it == m->picks.end() ? 0 : it->second.first;
    if (threads) *threads = it == m->picks.end() ? 0 : it->second.second;
    return 0;
}

/* The layer's KV cache rows (device pointers), for tests and inspection. */
int sparkmv_model_kv(void * model, int li, float ** k, float ** v) {
    Model * m = (Model *) model;
    if (!m || li < 0 || li >= m->c.layers || !k || !v) { set_error("bad model, layer or output"); return -1; }
    const size_t kvd = (size_t) m->c.kv_heads * m->c.head_dim;
    *k = m->kv + (size_t) li * 2 * m->c.max_ctx * kvd;
    *v = *k + (size_t) m->c.max_ctx * kvd;
    return 0;
}

int sparkmv_model_enable_capture(void * model, const int * layers, int n) {
    Model * m = (Model *) model;
    if (!m || (n > 0 && !layers)) { set_error("model or layer list is null"); return -1; }
    /* the runtime's limits and messages (vq-model-gpu.cu:707-736) */
    if (n <= 0 || n > 8) { set_error("capture: %d layers requested, the limit is 8", n); return -1; }
    if (m->cap) { set_error("capture: already enabled"); return -1; }
    std::vector<int> slot((size_t) m->c.layers, -1);
    for (int k = 0; k < n; k++) {
        const int li = layers[k];
        if (li < 0 || li >= m->c.layers) { set_error("capture: layer %d is outside 0..%d", li, m->c.layers); return -1; }
        if (slot[(size_t) li] >= 0) { set_error("capture: layer %d is listed twice", li); return -1; }
        slot[(size_t) li] = k;
    }
    void * mem = nullptr;
    hipError_t e = hipMalloc(&mem, (size_t) n * m->c.max_ctx * m->c.hidden * sizeof(float));
    if (e != hipSuccess) {
        set_error("capture: cannot allocate %d x %d x %d floats", n, m->c.max_ctx, m->c.hidden);
        return -1;
    }
    m->cap = (float *) mem;
    m->cap_n = n;
    m->cap_slot = slot;
    /* a recorded graph lacks the copies: record it again */
    if (m->exec) { (void) hipGraphExecDestroy(m->exec); m->exec = nullptr; }
    if (m->graph) { (void) hipGraphDestroy(m->graph); m->graph = nullptr; }
    return 0;
}

int sparkmv_model_captured(void * model, int k, float ** rows) {
    Model * m = (Model *) model;
    if (!m || !rows) { set_error("model or output is null"); return -1; }
    if (k < 0 || k >= m->cap_n) { set_error("capture slot %d is outside 0..%d", k, m->cap_n - 1); return -1; }
    *rows = m->cap + (size_t) k * m->c.max_ctx * m->c.hidden;
    return m->len;
}

int sparkmv_model_embed_row(void * model, uint32_t id, float * out, void * stream) {
    Model * m = (Model *) model;
    if (!m || !out) { set_error("model or output is null"); return -1; }
    if (m->head_kind < 0) { set_error("the model has no head"); return -1; }
    if ((long) id >= m->c.vocab) { set_error("token %u is outside the vocabulary", id); return -1; }
    const hipStream_t s = (hipStream_t) stream;
    const sparkmv_model_cfg & c = m->c;
    if (m->head_kind == 0) {
        hipLaunchKernelGGL(fw_fill_kernel, dim3((c.hidden + 255) / 256), dim3(256), 0, s, out, c.hidden, 0.0f);
        if (check_launch("fill launch")) return -1;
        const Layout L = make_layout(c.dim, c.nc, c.vocab, c.hidden, c.v3);
        for (int st = 0; st < c.nstages; st++)
            if (vq_row_dequant_launch(m->head_stages[st], L, (int) id, out, s)) return -1;
        return 0;
    }
    FwTok8 tk;
    for (int t = 0; t < 8; t++) tk.t[t] = (int) id;
    hipLaunchKernelGGL(fw_q8_0_rows_kernel, dim3((c.hidden + 255) / 256, 1), dim3(256), 0, s,
                       (const uint8_t *) m->head_blocks, c.hidden, tk, out);
    return check_launch("embedding launch");
}

int sparkmv_argmax(const float * logits, int n, int * out, void * stream) {
    if (!logits || !out) { set_error("logits or output is null"); return -1; }
    if (n < 1) { set_error("argmax needs at least one value, not %d", n); return -1; }
    hipLaunchKernelGGL(fw_argmax_kernel, dim3(1), dim3(1024), 0, (hipStream_t) stream, logits, n, out);
    return check_launch("argmax launch");
}

}  // extern "C"
