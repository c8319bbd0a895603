// gfx950 batched prefill: P prompt tokens through the model at once, bitwise equal to P
// sequential forwards (the reference's prompt loop, src/main.c:127-130, calling
// qm_model_forward, src/model.c:158-191).
//
// Exactness, layer by layer:
//   * activations are quantized per token row exactly as qm_quantize_row_q8 does (src/quant.c);
//   * a matmul row (r, token p) is the reference's serial chain s = +0; s = s + (float)acc_b *
//     (dw_b * dx_b) over blocks b in order (src/kernels_scalar.c:12-34). acc_b, the exact int32
//     dot of one 32-element block, comes from one i8 MFMA with a zero accumulator (32 rows x 32
//     tokens x one block per v_mfma_i32_32x32x32_i8, or 16 x 16 per v_mfma_i32_16x16x32_i8); the
//     float chains are extended in block order;
//   * attention scores, softmax and the weighted V sum keep the decode kernels' per-element
//     orders (serial over head_dim, the reference softmax, serial over positions).
//
// MFMA operand layouts (checked on the device): v_mfma_i32_16x16x32_i8 has A[i][k] in lane
// i + 16*(k/8), byte k%8; B[k][j] in lane j + 16*(k/8), byte k%8; D[i][j] in lane j + 16*(i/4),
// element i%4. v_mfma_i32_32x32x32_i8 has A[i][k] in lane i + 32*(k/16), byte k%16, B alike, and
// D[i][j] in lane j + 32*((i/4)%2), element 4*(i/8) + i%4. Any permutation of k applied to both operands leaves the dot unchanged; for
// Q4_0 weights each 8-element group is taken as [e0 e2 e4 e6 e1 e3 e5 e7] (the low nibbles of
// 4 bytes, then the high nibbles), and activations are stored in the same order.
#include "qmh_device.h"
#include "qmh_launch.h"

#define QMH_Q8 2
#define QMH_Q4 3

typedef int pf_v4i __attribute__((ext_vector_type(4)));
typedef float pf_v4f __attribute__((ext_vector_type(4)));
typedef _Float16 pf_v4h __attribute__((ext_vector_type(4)));
typedef int pf_v16i __attribute__((ext_vector_type(16)));
typedef float pf_v16f __attribute__((ext_vector_type(16)));

// ============================================================================ embedding

__global__ void k_pf_embed(const uint8_t *__restrict__ E, int dtype, int dim, int vocab, const int32_t *tokens,
                           float *X) {
    const int p = blockIdx.x;
    int tok = tokens[p];
    tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);  // the host validated the ids
    const size_t nbr = (size_t)(dim + 31) / 32;
    float *xr = X + (size_t)p * dim;
    if (dtype == QMH_Q8 || dtype == QMH_Q4) {
        // a quarter block (8 values) per thread: the scale, then the codes as 16-bit loads (a block's
        // codes start 2 bytes in, so they are only 2-byte aligned)
        const int bs = dtype == QMH_Q8 ? 34 : 18;
        for (int g = threadIdx.x; g < (int)nbr * 4; g += blockDim.x) {
            const int b = g >> 2, k0 = (g & 3) * 8;
            if (b * 32 + k0 >= dim) continue;
            const uint8_t *blk = E + ((size_t)tok * nbr + b) * bs;
            const float d = qmh_h2f(*(const uint16_t *)blk);
            float v[8];
            if (dtype == QMH_Q8) {
                const uint16_t *c = (const uint16_t *)(blk + 2 + k0);
#pragma unroll
                for (int h = 0; h < 4; h++) {
                    const uint16_t w = c[h];
                    v[2 * h] = d * (float)(int8_t)(w & 0xff);
                    v[2 * h + 1] = d * (float)(int8_t)(w >> 8);
                }
            } else {
                const uint16_t *c = (const uint16_t *)(blk + 2 + k0 / 2);  // element k: byte k/2, low nibble first
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const uint16_t w = c[h];
#pragma unroll
                    for (int q = 0; q < 4; q++) v[4 * h + q] = d * (float)((int)((w >> (4 * q)) & 15) - 8);
                }
            }
#pragma unroll
            for (int k = 0; k < 8; k++)
                if (b * 32 + k0 + k < dim) xr[b * 32 + k0 + k] = v[k];
        }
    } else {
        for (int i = threadIdx.x; i < dim; i += blockDim.x) xr[i] = ((const float *)E)[(size_t)tok * dim + i];
    }
}

extern "C" int qmh_launch_pf_embed(const uint8_t *tok_embd, int dtype, int dim, int vocab, const int32_t *tokens,
                                   int P, float *X, void *stream) {
    hipLaunchKernelGGL(k_pf_embed, dim3(P), dim3(256), 0, (hipStream_t)stream, tok_embd, dtype, dim, vocab, tokens, X);
    return (int)hipGetLastError();
}

// ============================================================================ activation quantization
//
// Row p of x (n values, optionally RMSNorm'd with gain w: src/ops.c:93-98) -> Q8_0 blocks of the
// token-major-within-block image: codes xc[(b*PP + p)*32 + k], scales xd[b*PP + p] (fp32 of the
// fp16 d). perm8: codes of each 8-group in the order e0 e2 e4 e6 e1 e3 e5 e7 (Q4_0 consumers).
// One workgroup per token; 8 lanes per block, 4 values each, as the decode prologue.
// One thread's share of a block quantization: block b = 32*r + tid/8 (round r), values 4*(tid%8)
// .. +3 of it, as the decode prologue (amax over 8 lanes by DPP), then the codes and the scale.
__device__ __forceinline__ void pf_quant_block(const float (&v)[4], int b, int nb, int p, int sub, int8_t *xc,
                                               float *xd, int PP, int perm8) {
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float av = fabsf(v[j]);
        m = av > m ? av : m;
    }
    m = qmh_amax8(m);
    const float dd = qmh_h2f(qmh_f2h(qmh_div127(m)));
    int q[4];
    qmh_q8_codes4(v, dd, qmh_rcp(dd), q);
    const uint32_t b0 = (uint32_t)q[0] & 0xffu, b1 = (uint32_t)q[1] & 0xffu, b2 = (uint32_t)q[2] & 0xffu,
                   b3 = (uint32_t)q[3] & 0xffu;
    // one dword per lane: bytes 4*sub .. +3 of the block. perm8 (elements 8g+e, e = 0..7, at
    // 8g + {0,4,1,5,2,6,3,7}[e]): the lane pair of a group (elements 0-3, 4-7) swaps half-words,
    // {e0 e2 | e1 e3} against {e4 e6 | e5 e7}, and writes {e0 e2 e4 e6} (even lane) or {e1 e3 e5 e7}.
    const uint32_t pk = b0 | (b2 << 8) | (b1 << 16) | (b3 << 24);
    const uint32_t pp = (uint32_t)qmh_dpp<QMH_DPP_QXOR1>((int)pk);  // every lane of the block is active here
    const uint32_t w = !perm8 ? (b0 | (b1 << 8) | (b2 << 16) | (b3 << 24))
                       : (sub & 1) == 0 ? ((pk & 0xffffu) | (pp << 16)) : ((pp >> 16) | (pk & 0xffff0000u));
    if (b < nb) {
        *(uint32_t *)(xc + ((size_t)b * PP + p) * 32 + 4 * sub) = w;
        if (sub == 0) xd[(size_t)b * PP + p] = dd;
    }
}

// One workgroup per token; 8 lanes per block, 4 values each. Rows of up to PQ_R*1024 values are
// loaded once into registers (one round of loads), larger ones round by round.
#define PQ_R 16
template <int NT>
__global__ __launch_bounds__(NT) void k_pf_quant(const float *__restrict__ x, int ldx, const float *w, float eps,
                                                     int n, int8_t *xc, float *xd, int PP, int perm8) {
    __shared__ double red[NT / 64 + 1];  // the waves' partial sums, then the serial sum
    const int p = blockIdx.x, tid = threadIdx.x, nb = (n + 31) / 32, sub = tid & 7;
    const int R = (nb + NT / 8 - 1) / (NT / 8);  // rounds of 32 blocks
    const float *row = x + (size_t)p * ldx;
    const bool held = R <= PQ_R;
    float xv[PQ_R][4];
    double ss = 0.0;
    if (held) {
#pragma unroll
        for (int r = 0; r < PQ_R; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = (r * (NT / 8) + (tid >> 3)) * 32 + sub * 4 + j;
                xv[r][j] = (r < R && i < n) ? row[i] : 0.0f;
            }
        if (w)
#pragma unroll
            for (int r = 0; r < PQ_R; r++)
#pragma unroll
                for (int j = 0; j < 4; j++) ss += (double)xv[r][j] * (double)xv[r][j];
    } else if (w) {
        for (int i = tid; i < n; i += NT) ss += (double)row[i] * (double)row[i];
    }
    float inv = 1.0f;
    if (w) {
        ss = qmh_block_sum_d(ss, red);
        const double d = qmh_sum_slack(ss, n);
        inv = qmh_rms_inv(ss - d, n, eps);
        if (inv != qmh_rms_inv(ss + d, n, eps)) {  // uniform; serial sum as the reference
            if (tid == 0) {
                double s2 = 0.0;
                for (int i = 0; i < n; i++) s2 += (double)row[i] * (double)row[i];
                red[NT / 64] = s2;
            }
            __syncthreads();
            inv = qmh_rms_inv(red[NT / 64], n, eps);
        }
    }
    // (x*inv)*w as the reference; rounds are uniform (DPP needs all 8 lanes of a block)
    if (held) {
#pragma unroll
        for (int r = 0; r < PQ_R; r++)
            if (r < R) {
                const int b = r * (NT / 8) + (tid >> 3), i4 = b * 32 + sub * 4;
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    v[j] = w ? ((b < nb && i4 + j < n) ? xv[r][j] * inv * w[i4 + j] : 0.0f) : xv[r][j];
                pf_quant_block(v, b, nb, p, sub, xc, xd, PP, perm8);
            }
    } else {
        for (int r = 0; r < R; r++) {
            const int b = r * (NT / 8) + (tid >> 3), i4 = b * 32 + sub * 4;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const bool in = b < nb && i4 + j < n;
                v[j] = in ? (w ? row[i4 + j] * inv * w[i4 + j] : row[i4 + j]) : 0.0f;
            }
            pf_quant_block(v, b, nb, p, sub, xc, xd, PP, perm8);
        }
    }
}

// k_pf_quant for rows of n % 4 == 0 values (16-byte aligned rows and gain) in RR rounds: each
// thread's 4 values of a round are one 16-byte buffer load whose range check (n*4 bytes) zeroes
// what lies past the row, so all of a thread's loads (row and gain) issue at once, before the
// sum. The scale 1/sqrt(ss/n + eps) takes the margin test first, as the decode prologue.
typedef uint32_t pf_v4u __attribute__((ext_vector_type(4)));
template <int NT, int RR, bool NORM>
__global__ __launch_bounds__(NT) void k_pf_quant4(const float *__restrict__ x, int ldx, const float *w, float eps,
                                                      int n, int8_t *xc, float *xd, int PP, int perm8) {
    __shared__ double red[NT / 64 + 1];
    const int p = blockIdx.x, tid = threadIdx.x, nb = (n + 31) / 32, sub = tid & 7;
    const float *row = x + (size_t)p * ldx;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)row, (short)0, n * 4, 0x00020000);
    pf_v4u xv[RR], wv[RR];
#pragma unroll
    for (int r = 0; r < RR; r++) xv[r] = __builtin_amdgcn_raw_buffer_load_b128(rx, (r * NT + tid) * 16, 0, 0);
    float inv = 1.0f;
    if (NORM) {
        const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)w, (short)0, n * 4, 0x00020000);
#pragma unroll
        for (int r = 0; r < RR; r++) wv[r] = __builtin_amdgcn_raw_buffer_load_b128(rw, (r * NT + tid) * 16, 0, 0);
        double ss = 0.0;  // values past the row load as +0
#pragma unroll
        for (int r = 0; r < RR; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double v = (double)__uint_as_float(xv[r][j]);
                ss += v * v;
            }
        // wave butterflies, then the waves in order; red is not reused, so one barrier publishes
        ss = qmh_wave_sum_d(ss);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
        __syncthreads();
        ss = 0.0;
#pragma unroll
        for (int k = 0; k < NT / 64; k++) ss += red[k];
        // the same ss in every thread: uniform branches
        if (!qmh_rms_inv_margin(ss, n, nb * 32, eps, &inv)) {
            const double d = qmh_sum_slack(ss, nb * 32);
            inv = qmh_rms_inv(ss - d, n, eps);
            if (inv != qmh_rms_inv(ss + d, n, eps)) {  // the reference's serial sum
                if (tid == 0) {
                    double s2 = 0.0;
                    for (int i = 0; i < n; i++) s2 += (double)row[i] * (double)row[i];
                    red[NT / 64] = s2;
                }
                __syncthreads();
                inv = qmh_rms_inv(red[NT / 64], n, eps);
            }
        }
    }
    // (x*inv)*w as the reference; rounds are uniform (DPP needs all 8 lanes of a block)
#pragma unroll
    for (int r = 0; r < RR; r++)
        if (r * (NT / 8) < nb) {
            const int b = r * (NT / 8) + (tid >> 3), i4 = b * 32 + sub * 4;
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float xe = __uint_as_float(xv[r][j]);
                v[j] = NORM ? ((b < nb && i4 + j < n) ? xe * inv * __uint_as_float(wv[r][j]) : 0.0f) : xe;
            }
            pf_quant_block(v, b, nb, p, sub, xc, xd, PP, perm8);
        }
}

template <int NT, bool NORM>
static void pf_quant4_launch(int RR, int P, hipStream_t s, const float *x, int ldx, const float *w, float eps, int n,
                             int8_t *xc, float *xd, int PP, int perm8) {
#define PQ4(R_) hipLaunchKernelGGL((k_pf_quant4<NT, R_, NORM>), dim3(P), dim3(NT), 0, s, x, ldx, w, eps, n, xc, xd, PP, perm8)
    switch (RR) {
    case 1: PQ4(1); break;
    case 2: PQ4(2); break;
    case 4: PQ4(4); break;
    case 8: PQ4(8); break;
    default: PQ4(16); break;
    }
#undef PQ4
}

extern "C" int qmh_launch_pf_quant(const float *x, int ldx, const float *w, float eps, int n, int P, int8_t *xc,
                                   float *xd, int PP, int perm8, void *stream) {
    // a few rows (batched decode): 1024 threads per row, one round of loads for a 4096-value row
    // and 16 waves to wait on them; many rows (prefill): 512 threads (256 and 1024 were 0.3-0.5%
    // slower at 512 rows)
    const int NT = P <= 16 ? 1024 : 512, nb = (n + 31) / 32, R = (nb + NT / 8 - 1) / (NT / 8);
    const bool vec = n % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0;
    hipStream_t s = (hipStream_t)stream;
    if (vec && R <= PQ_R) {
        const int RR = R <= 1 ? 1 : R <= 2 ? 2 : R <= 4 ? 4 : R <= 8 ? 8 : 16;
        if (NT == 1024) {
            if (w) pf_quant4_launch<1024, true>(RR, P, s, x, ldx, w, eps, n, xc, xd, PP, perm8);
            else pf_quant4_launch<1024, false>(RR, P, s, x, ldx, w, eps, n, xc, xd, PP, perm8);
        } else {
            if (w) pf_quant4_launch<512, true>(RR, P, s, x, ldx, w, eps, n, xc, xd, PP, perm8);
            else pf_quant4_launch<512, false>(RR, P, s, x, ldx, w, eps, n, xc, xd, PP, perm8);
        }
    } else if (NT == 1024) {
        hipLaunchKernelGGL(k_pf_quant<1024>, dim3(P), dim3(1024), 0, s, x, ldx, w, eps, n, xc, xd, PP, perm8);
    } else {
        hipLaunchKernelGGL(k_pf_quant<QMH_WG>, dim3(P), dim3(QMH_WG), 0, s, x, ldx, w, eps, n, xc, xd, PP, perm8);
    }
    return (int)hipGetLastError();
}

// ============================================================================ matmul
//
__device__ __forceinline__ long pf_q4_operand(uint32_t w) {
    // 8 nibbles -> 8 signed int8 (q - 8): low nibbles (e0 e2 e4 e6), then high (e1 e3 e5 e7).
    // Per byte, q + 0x78 stays below 0x100 (no carry into the next byte), and flipping its top
    // bit gives q - 8 in two's complement: 0 -> 0xf8, 8 -> 0x00, 15 -> 0x07.
    const uint32_t lo = ((w & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
    const uint32_t hi = (((w >> 4) & 0x0f0f0f0fu) + 0x78787878u) ^ 0x80808080u;
    return (long)(((uint64_t)hi << 32) | lo);
}

// slot of block 0 of a weight row: plain tiles, or interleaved (W1 | W3) tiles with tile_r/2
// rows of each matrix (half 0: W1, 1: W3); block b adds b*tile_r
__device__ __forceinline__ uint32_t pf_slot0(const qmh_pf_args &a, int row, int half) {
    if (a.il) {
        const int h = a.tile_r / 2;
        return (uint32_t)(row / h) * a.nb * a.tile_r + row % h + half * h;
    }
    return (uint32_t)(row / a.tile_r) * a.nb * a.tile_r + row % a.tile_r;
}

// The skinny matmul's operands of one block: NM matrices (2 for the W1 | W3 SwiGLU pair), one 16-row
// tile, TW 16-token tiles
template <int NM, int TW>
struct PfBlock {
    long A[NM];       // raw weight codes: 8 int8 (Q8_0) or 4 nibble bytes (Q4_0, low word)
    uint32_t wh[NM];  // the fp16 scale of the lane's A row
    long B[TW];
    float dx[TW];
};

// Per-lane byte/element offsets of the operands, fixed over the blocks: the loop adds only the
// block's uniform base, so the loads take a scalar base and these offsets. Rows past the
// allocated slots read row 0 instead: each D row depends only on its own A row, and those rows
// are never stored.
template <int NM>
struct PfLane {
    uint32_t a[NM], w[NM];  // weight codes (bytes) and the scale (element) of the lane's A row at block 0
    uint32_t x, d;          // activation codes (bytes), scales (elements) of token tile 0
};

// Loads only: no value is used here, so the wait for these loads falls where the block is multiplied.
template <int WT, int NM, int TW>
__device__ __forceinline__ void pf_load(const qmh_pf_args &a, int b, const PfLane<NM> &ln, PfBlock<NM, TW> &o) {
    constexpr int CB = WT == QMH_Q8 ? 32 : 16;
    const uint8_t *cb = a.codes + (size_t)b * a.tile_r * CB;
    const uint16_t *sb = a.scales + (size_t)b * a.tile_r;
#pragma unroll
    for (int m = 0; m < NM; m++) {
        if (WT == QMH_Q8) o.A[m] = *(const long *)(cb + ln.a[m]);
        else o.A[m] = (long)*(const uint32_t *)(cb + ln.a[m]);
        o.wh[m] = sb[ln.w[m]];
    }
    const int8_t *xb = a.xc + (size_t)b * a.PP * 32;
    const float *db = a.xd + (size_t)b * a.PP;
#pragma unroll
    for (int tt = 0; tt < TW; tt++) {
        o.B[tt] = *(const long *)(xb + ln.x + tt * 512);
        o.dx[tt] = db[ln.d + tt * 16];
    }
}

// one output of the matmul: y = row's value for token p (up: the W3 value of the SwiGLU pair;
// partner: the value of row ^ 1, RoPE's pair), stored as the epilogue asks
__device__ __forceinline__ void pf_store(const qmh_pf_args &a, int row, int p, float y, float up, float partner) {
    if (a.epi == QMH_PF_STORE) {
        a.out0[(size_t)p * a.ld0 + row] = y;
    } else if (a.epi == QMH_PF_ADD) {  // x += W x' (src/model.c:179,186)
        a.out0[(size_t)p * a.ld0 + row] = a.out0[(size_t)p * a.ld0 + row] + y;
    } else if (a.epi == QMH_PF_SWIGLU) {  // silu(g)*u (src/ops.c:128-133)
        a.out0[(size_t)p * a.ld0 + row] = y / (1.0f + qmh_expf(-y)) * up;
    } else {  // QKV: rope on q and k (src/ops.c:114-126), k/v into the caches
        const int pos = a.pos_arr ? a.pos_arr[p] : a.pos0 + p;
        float *kc = a.out1 + (size_t)p * a.kv_stride, *vc = a.out2 + (size_t)p * a.kv_stride;
        if (row < a.seg2) {
            const int local = row < a.seg1 ? row : row - a.seg1;
            const float *cs = a.rope + ((size_t)pos * (a.head_dim >> 1) + ((local % a.head_dim) >> 1)) * 2;
            const float c = cs[0], sn = cs[1];
            const float v = (local & 1) == 0 ? (y * c - partner * sn) : (partner * sn + y * c);
            if (row < a.seg1) a.out0[(size_t)p * a.ld0 + local] = v;
            else kc[(size_t)local * a.max_seq + pos] = v;
        } else {
            vc[(size_t)pos * a.kvd + (row - a.seg2)] = y;
        }
    }
}

// ---- tiled matmul (qmh_pf_tiled says when)
//
// A workgroup owns RT 32-row tiles x TT 32-token tiles, one (row tile, token tile) pair per wave, and
// takes all blocks in order. IL (W1 | W3): the first RT/2 row tiles are W1 rows, the others the same
// rows of W3, whose values pass to the W1 waves through LDS at the end.
//
// What bounds it. Per 1024 outputs (32 x 32) and block a wave issues 48 VALU instructions (convert,
// multiply, add: the reference's three roundings) and two MFMAs of 32 cycles. On this device a SIMD takes
// a VALU instruction every 2 cycles from two or more waves (every 4 from one), and an MFMA's cycles
// largely add to the VALU's: about 163 cycles per pair of tile and block, and the clock falls to
// ~1.9 GHz under it. So the shape that needs the fewest cycles wins, not the one with the most work per
// load: v_mfma_i32_32x32x32_i8 gives 1024 dots in 32 cycles where 16x16x32 takes 64, and likewise the
// f16 32x32x8 for the scale products. Timed at 512 tokens (us, 16x16 tiles in registers -> this, launches in a
// graph over 8 copies of the weights): 12288x4096 125 -> 81, 4096x4096 53 -> 34, W1|W3 2x11008x4096 195 -> 155,
// 4096x11008 128 -> 81. Counters at W1|W3: 264 cycles per pair of tile and block, 64 of MFMA and 117 of VALU issue;
// the rest is waves waiting and the last round of workgroups (LDS conflicts 2%).
// Tried and slower: the int8 accumulator started at the bits of 1.5*2^23 with a second scale product
// -1.5*2^23*dw*dx, for two VALU instructions per term (an f32 MFMA runs on the VALU's own units, and
// the third MFMA costs what the conversion saved); 32x32 tiles with operands straight from
// memory (6 to 10% slower: the loads bound it); two token tiles per wave (one wave per SIMD). Four waves per
// SIMD are asked of every instance: the 2 x 1 ones hold three (the compiler warns), but asked for three they were 1-2%
// slower; the Q8_0 2 x 2 ones spill 3-4 registers for the fourth.
//
// Operands pass through LDS in stages of PG_KB blocks, two buffers: a thread's pieces of stage i + 2
// (+ DEEP) are loaded to registers during stage i and written when stage i has been read. The loads'
// offsets are fixed per thread (buffer loads, the block in the scalar offset, which a buffer's range check
// need not cover). The stages run past the last block, in a last stage that is not whole and in those
// loaded ahead: these load the last block again, so that every address lies in the matrix, and what they
// hold is never multiplied. The barrier waits for LDS only, so loads stay in flight across it. Q4_0 codes
// are written as 16*(q - 8) (two operations per four codes; a chain of 16 x the terms is 16 x the
// reference's chain exactly, so one multiply by 1/16 ends it: no term is below 2^-48 or above 2^52). In LDS
// each half block of every row (or token) is contiguous over the rows, with 1-2% of the cycles lost to bank
// conflicts; the four fp16 scales of a row sit side by side, and the scale product of
// block j takes all four as k = 0..3 of A against B with only entry j (others 0).
//
// Inside a block: convert and multiply by the scale products, issue the next block's integer MFMA
// (its accumulators are free), add to the chains, issue the next block's scale MFMA.
//
// Infinite or NaN scales: 0 * inf in the scale MFMA makes a NaN where the reference might not, and
// leaves a NaN in every chain it touches, so rows that end as NaN are computed again from memory
// (pg_row). Finite scales never give a NaN or an infinity.
#define PG_KB 4
#define PG_FENCE() __builtin_amdgcn_sched_barrier(0)  // keeps the order above

// every LDS access done, then the barrier: the vector memory loads in flight are not waited for
__device__ __forceinline__ void pg_lds_barrier() { __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int RT, int TT>
struct PgLds {
    static constexpr int A = PG_KB * RT * 1024, B = PG_KB * TT * 1024, W = RT * 32 * 8, D = TT * 32 * 8;
    static constexpr int STG = A + B + W + D;
};

// one row's chain from memory, block by block as the reference (a row or token with an infinite or NaN
// scale, see k_pf_gemm)
template <int WT>
__device__ float pg_row(const qmh_pf_args &a, uint32_t slot, int p) {
    constexpr int CB = WT == QMH_Q8 ? 32 : 16;
    float s = 0.0f;
#pragma unroll 1
    for (int b = 0; b < a.nb; b++) {
        const uint8_t *c = a.codes + ((size_t)slot + (size_t)b * a.tile_r) * CB;
        const int8_t *x = a.xc + ((size_t)b * a.PP + p) * 32;
        int acc = 0;
#pragma unroll 1
        for (int g = 0; g < 8; g++) {  // 4 image bytes; Q4_0: group 8 * (g / 2), low nibbles then high
            const uint32_t xw = *(const uint32_t *)(x + 4 * g);
            uint32_t w;
            if (WT == QMH_Q8) w = *(const uint32_t *)(c + 4 * g);
            else w = (uint32_t)(pf_q4_operand(*(const uint32_t *)(c + 4 * (g >> 1))) >> (32 * (g & 1)));
            acc = __builtin_amdgcn_sdot4((int)w, (int)xw, acc, false);
        }
        const float dw = qmh_h2f(a.scales[(size_t)slot + (size_t)b * a.tile_r]);
        s = s + (float)acc * (dw * a.xd[(size_t)b * a.PP + p]);
    }
    return s;
}

template <int WT, bool IL, int RT, int TT, int DEEP>
__global__ __launch_bounds__(64 * RT * TT, 4) void k_pf_gemm(qmh_pf_args a) {
    constexpr int KB = PG_KB, CB = WT == QMH_Q8 ? 32 : 16, AH = CB / 16, WG = 64 * RT * TT;
    constexpr int NR = RT * 32, NTK = TT * 32, RS = WG / NR, TS = WG / NTK;
    constexpr int NA = KB / RS, NB = 2 * KB / TS, ND = (KB + TS - 1) / TS;
    using L = PgLds<RT, TT>;
    __shared__ __align__(16) uint8_t lds[2 * L::STG];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, hi = l >> 5, lr = l & 31;
    // workgroups go round robin over the 8 XCDs: the token groups of a row group share one XCD's L2
    // (W1 | W3 at 512 tokens 217 -> 208 us)
    const int gx = gridDim.x, gy = gridDim.y, lin = blockIdx.y * gx + blockIdx.x;
    int bx = blockIdx.x, by = blockIdx.y;
    if (lin < gy / 8 * 8 * gx) {
        by = (lin >> 3) / gx * 8 + (lin & 7);
        bx = (lin >> 3) % gx;
    }
    const int rg0 = by * (IL ? NR / 2 : NR), t0 = bx * NTK, nb = a.nb;
    // A: row of the tile, blocks j0 + k*RS (a wave's lanes share j0)
    static_assert(NR % 64 == 0, "whole waves per block of A");
    const int row = tid % NR, j0 = wave * 64 / NR;
    // B: token, (half, block) q0 + k*TS: a wave's lanes share the block, q0 / 2 + k*TS/2
    const int tok = tid % NTK, q0 = tid / NTK, qb = wave * 64 / NTK / 2;
    // offsets from the workgroup's first slot; rows past the allocated ones read its first row
    const uint32_t slot_w = pf_slot0(a, rg0, 0);
    auto slot_of = [&](int r) {
        const int rr = rg0 + (IL ? r % (NR / 2) : r);
        return pf_slot0(a, rr < a.rows_alloc ? rr : rg0, IL ? r / (NR / 2) : 0);
    };
    const uint32_t slot_r = slot_of(row) - slot_w;
    const size_t nslots = (size_t)(IL ? a.rows_alloc / (a.tile_r / 2) * a.tile_r : a.rows_alloc) * nb - slot_w;
    auto rsrc = [](const void *q, size_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)q, (short)0, (int)(bytes < 0xffffffffu ? bytes : 0xffffffffu), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rca = rsrc(a.codes + (size_t)slot_w * CB, nslots * CB), rcw = rsrc(a.scales + slot_w, nslots * 2);
    const __amdgpu_buffer_rsrc_t rcb = rsrc(a.xc + (size_t)t0 * 32, ((size_t)nb * a.PP - t0) * 32);
    const __amdgpu_buffer_rsrc_t rcd = rsrc(a.xd + t0, ((size_t)nb * a.PP - t0) * 4);
    const uint32_t ast = (uint32_t)a.tile_r * CB, bst = (uint32_t)a.PP * 32;
    const uint32_t va = slot_r * CB, vw = slot_r * 2, vb = tok * 32 + (q0 & 1) * 16, vd = tok * 4;
    auto blk = [&](int b) { return (uint32_t)(b < nb ? b : nb - 1); };
    pf_v4u ra_[1 + DEEP][NA][AH], rb_[1 + DEEP][NB];
    uint32_t rw_[1 + DEEP][NA], rd_[1 + DEEP][ND];
    // stage of blocks b0.. into register set q, and from there to the LDS buffer at base
    auto gload = [&](int b0, int q) {
#pragma unroll
        for (int k = 0; k < NA; k++) {
#pragma unroll
            for (int h = 0; h < AH; h++)
                ra_[q][k][h] = __builtin_amdgcn_raw_buffer_load_b128(rca, va + 16 * h, blk(b0 + j0 + k * RS) * ast, 0);
            rw_[q][k] = __builtin_amdgcn_raw_buffer_load_b16(rcw, vw, blk(b0 + j0 + k * RS) * (uint32_t)a.tile_r * 2, 0);
        }
#pragma unroll
        for (int k = 0; k < NB; k++)
            rb_[q][k] = __builtin_amdgcn_raw_buffer_load_b128(rcb, vb, blk(b0 + qb + k * (TS / 2)) * bst, 0);
#pragma unroll
        for (int k = 0; k < ND; k++) {  // block q0 + k*TS: shared by a wave's lanes from 64 tokens on
            const uint32_t o = blk(b0 + (NTK < 64 ? q0 : wave * 64 / NTK) + k * TS) * (uint32_t)a.PP * 4;
            if (TS <= KB || wave * 64 / NTK < KB)
                rd_[q][k] = __builtin_amdgcn_raw_buffer_load_b32(rcd, NTK < 64 ? vd + o : vd, NTK < 64 ? 0 : o, 0);
        }
    };
    auto swrite = [&](uint32_t base, int q) {
#pragma unroll
        for (int k = 0; k < NA; k++) {
            pf_v4u lo = ra_[q][k][0], hh = ra_[q][k][AH - 1];
            if (WT == QMH_Q4) {
                const pf_v4u v = lo;
                lo[0] = ((v[0] << 4) & 0xf0f0f0f0u) ^ 0x80808080u, lo[1] = (v[0] & 0xf0f0f0f0u) ^ 0x80808080u;
                lo[2] = ((v[1] << 4) & 0xf0f0f0f0u) ^ 0x80808080u, lo[3] = (v[1] & 0xf0f0f0f0u) ^ 0x80808080u;
                hh[0] = ((v[2] << 4) & 0xf0f0f0f0u) ^ 0x80808080u, hh[1] = (v[2] & 0xf0f0f0f0u) ^ 0x80808080u;
                hh[2] = ((v[3] << 4) & 0xf0f0f0f0u) ^ 0x80808080u, hh[3] = (v[3] & 0xf0f0f0f0u) ^ 0x80808080u;
            }
            uint8_t *o = lds + base + (j0 + k * RS) * (NR * 32) + row * 16;
            *(pf_v4u *)o = lo;
            *(pf_v4u *)(o + NR * 16) = hh;
            *(uint16_t *)(lds + base + L::A + L::B + row * 8 + 2 * (j0 + k * RS)) = (uint16_t)rw_[q][k];
        }
#pragma unroll
        for (int k = 0; k < NB; k++)
            *(pf_v4u *)(lds + base + L::A + (q0 + k * TS) * (NTK * 16) + tok * 16) = rb_[q][k];
#pragma unroll
        for (int k = 0; k < ND; k++)
            if (TS <= KB || wave * 64 / NTK < KB)
                *(_Float16 *)(lds + base + L::A + L::B + L::W + tok * 8 + 2 * (q0 + k * TS)) = (_Float16)__uint_as_float(rd_[q][k]);
    };
    // the wave's operands: codes by block parity, scales by stage parity
    const int wr = wave / TT, wt = wave % TT;
    const uint32_t oa = hi * (NR * 16) + (uint32_t)(wr * 32 + lr) * 16, ob = L::A + hi * (NTK * 16) + (uint32_t)(wt * 32 + lr) * 16;
    const uint32_t ow = L::A + L::B + (uint32_t)(wr * 32 + lr) * 8, od = L::A + L::B + L::W + (uint32_t)(wt * 32 + lr) * 8;
    const uint32_t mlo = hi ? 0 : 0xffffu, mhi = hi ? 0 : 0xffff0000u;
    pf_v4i A[2], B[2];
    uint2 w[2], d[2];
    auto rd = [&](uint32_t base, int j, int k) {
        A[k] = *(const pf_v4i *)(lds + base + oa + j * (NR * 32));
        B[k] = *(const pf_v4i *)(lds + base + ob + j * (NTK * 32));
    };
    auto rs = [&](uint32_t base, int k) {
        w[k] = *(const uint2 *)(lds + base + ow);
        d[k] = *(const uint2 *)(lds + base + od);
    };
    float s[16];
    pf_v16i acc, zi;
    pf_v16f pw, zf;
#pragma unroll
    for (int e = 0; e < 16; e++) s[e] = 0.0f, zi[e] = 0, zf[e] = 0.0f;
    auto isp = [&](int k, int j) {
        const uint2 m = j == 0 ? make_uint2(d[k].x & mlo, 0u) : j == 1 ? make_uint2(d[k].x & mhi, 0u)
                        : j == 2 ? make_uint2(0u, d[k].y & mlo) : make_uint2(0u, d[k].y & mhi);
        pw = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(pf_v4h, w[k]), __builtin_bit_cast(pf_v4h, m), zf, 0, 0, 0);
    };
    auto isi = [&](int k) { acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[k], B[k], zi, 0, 0, 0); };
    // the block whose MFMAs are in flight into the chains; the next block's MFMAs from operand set k,
    // entry j of scale set sk
    auto mul = [&](int k, int sk, int j) {
        PG_FENCE();
        float f[16];
#pragma unroll
        for (int e = 0; e < 16; e++) f[e] = (float)acc[e];
        PG_FENCE();
#pragma unroll
        for (int e = 0; e < 16; e++) f[e] = f[e] * pw[e];
        PG_FENCE();
        isi(k);
        PG_FENCE();
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] = s[e] + f[e];
        PG_FENCE();
        isp(sk, j);
        PG_FENCE();
    };
    const int nst = (nb + KB - 1) / KB;
    gload(0, 0);
    if (DEEP) gload(KB, DEEP);
    swrite(0, 0);
    if (!DEEP) gload(KB, 0);
    else gload(2 * KB, 0);
    pg_lds_barrier();
    swrite(L::STG, DEEP);
    gload((2 + DEEP) * KB, DEEP);
    rd(0, 0, 0);
    rd(0, 1, 1);
    rs(0, 0);
    isi(0), isp(0, 0);
    for (int i0 = 0; i0 < nst; i0 += 2) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int b0 = (i0 + h) * KB;
            const uint32_t base = h * L::STG, oth = L::STG - base;
#pragma unroll
            for (int j = 0; j < KB; j++) {
                if (j == KB - 2) {
                    pg_lds_barrier();  // this stage's operands are read, the next stage is written
                    rd(oth, 0, j & 1);
                    rs(oth, h ^ 1);
                    swrite(base, DEEP ? h : 0);
                    gload(b0 + (3 + DEEP) * KB, DEEP ? h : 0);
                } else {
                    rd(j < KB - 2 ? base : oth, (j + 2) % KB, j & 1);
                }
                if (b0 + j < nb) mul((j & 1) ^ 1, j == KB - 1 ? h ^ 1 : h, (j + 1) % KB);
            }
        }
    }
    if (WT == QMH_Q4)
#pragma unroll
        for (int e = 0; e < 16; e++) s[e] = s[e] * 0.0625f;
    const int p = t0 + 32 * wt + lr, wrow = rg0 + 32 * (IL ? wr % (RT / 2) : wr);
    // a NaN here means an infinite or NaN scale: that row's chain again, from memory
    uint32_t nan = 0;
#pragma unroll
    for (int e = 0; e < 16; e++)
        nan |= (s[e] != s[e] && p < a.P && wrow + 8 * (e >> 2) + 4 * hi + (e & 3) < a.rows) ? 1u << e : 0u;
    if (__any(nan != 0)) {
#pragma unroll 1
        for (int e = 0; e < 16; e++) {
            if (!((nan >> e) & 1)) continue;
            const float v = pg_row<WT>(a, pf_slot0(a, wrow + 8 * (e >> 2) + 4 * hi + (e & 3), IL ? wr / (RT / 2) : 0), p);
#pragma unroll
            for (int k = 0; k < 16; k++) s[k] = k == e ? v : s[k];
        }
    }
    if (!IL) {
        if (p >= a.P) return;
        // 4 consecutive rows per lane: 16-byte accesses where they are whole and aligned
        if ((a.epi == QMH_PF_STORE || a.epi == QMH_PF_ADD) && a.ld0 % 4 == 0 && ((uintptr_t)a.out0 & 15) == 0 &&
            rg0 + NR <= a.rows) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                pf_v4f *o = (pf_v4f *)(a.out0 + (size_t)p * a.ld0 + wrow + 8 * g + 4 * hi);
                pf_v4f y = {s[4 * g], s[4 * g + 1], s[4 * g + 2], s[4 * g + 3]};
                if (a.epi == QMH_PF_ADD) {  // x += W x' (src/model.c:179,186)
                    const pf_v4f x = *o;
#pragma unroll
                    for (int e = 0; e < 4; e++) y[e] = x[e] + y[e];
                }
                *o = y;
            }
            return;
        }
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int r = wrow + 8 * (e >> 2) + 4 * hi + (e & 3);
            if (r < a.rows) pf_store(a, r, p, s[e], 0.0f, s[e ^ 1]);
        }
        return;
    }
    // W3's values to the waves of W1
    __syncthreads();
    constexpr int HW = RT / 2 * TT;  // waves of W1
    float *x = (float *)lds + (wave % HW) * 1024 + l;
    static_assert(2 * L::STG >= HW * 4096, "the exchange fits the stages");
    if (wave >= HW)
#pragma unroll
        for (int e = 0; e < 16; e++) x[e * 64] = s[e];
    __syncthreads();
    if (wave >= HW) return;
    float up[16];
#pragma unroll
    for (int e = 0; e < 16; e++) up[e] = x[e * 64];
    if (!a.qxc) {
        if (p >= a.P) return;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int r = wrow + 8 * (e >> 2) + 4 * hi + (e & 3);
            if (r < a.rows) pf_store(a, r, p, s[e], up[e], 0.0f);
        }
        return;
    }
    // W2's input as its Q8_0 image: the wave's 32 rows are one block of each of its tokens, 16 values in
    // lane l and 16 in l ^ 32. The same steps as k_pf_quant's block (src/quant.c:27-52): amax, the fp16
    // scale, the codes (Q4_0 order: 8g + e at 8g + {0,4,1,5,2,6,3,7}[e], by a half-word swap with
    // lane l ^ 32); rows past `rows` are 0 there and here.
    float v[16], m = 0.0f;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const float y = s[e];
        v[e] = wrow + 8 * (e >> 2) + 4 * hi + (e & 3) < a.rows ? y / (1.0f + qmh_expf(-y)) * up[e] : 0.0f;  // src/ops.c:128-133
        const float av = fabsf(v[e]);
        m = av > m ? av : m;
    }
    const float o = __shfl_xor(m, 32);
    m = o > m ? o : m;
    const float dd = qmh_h2f(qmh_f2h(qmh_div127(m))), rinv = qmh_rcp(dd);
    const int b = wrow >> 5;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        int q[4];
        qmh_q8_codes4(v + 4 * g, dd, rinv, q);
        const uint32_t c0 = (uint32_t)q[0] & 0xffu, c1 = (uint32_t)q[1] & 0xffu, c2 = (uint32_t)q[2] & 0xffu, c3 = (uint32_t)q[3] & 0xffu;
        const uint32_t pk = c0 | (c2 << 8) | (c1 << 16) | (c3 << 24);
        const uint32_t pp = (uint32_t)__shfl_xor((int)pk, 32);
        const uint32_t wv = !a.qperm8 ? (c0 | (c1 << 8) | (c2 << 16) | (c3 << 24))
                            : hi == 0 ? ((pk & 0xffffu) | (pp << 16)) : ((pp >> 16) | (pk & 0xffff0000u));
        if (p < a.P) *(uint32_t *)(a.qxc + ((size_t)b * a.PP + p) * 32 + 8 * g + 4 * hi) = wv;
    }
    if (p < a.P && hi == 0) a.qxd[(size_t)b * a.PP + p] = dd;
}

// Skinny matmul for decode-sized batches (P <= 16*TT tokens, TT <= 4; qmh_pf_tiled says when): one workgroup per 16-row group
// streams every block of its rows once for all tokens. The blocks pass in rounds of as many as
// fit the LDS budget at this P: wave w takes blocks base + 8j + w in batches of PD (each batch's
// loads all in flight, no barrier inside a round), takes each block's exact int32 dot for TT
// token tiles from MFMAs with a zero accumulator, and stores the term (float)acc*(dw*dx) in LDS
// at [matrix][block in round][token][row]; after the round one thread per (row, token) pair
// extends that pair's serial chain over the round's blocks in order (the reference's order).
// After the last round each pair runs the epilogue. Dynamic LDS: one round's terms, at most SK_LDS.
#define SK_WG 512
#define SK_LDS (128 * 1024)
// blocks per round: a multiple of 8 that fits the LDS budget at P tokens (the launch gives the
// kernel exactly NM*16*P*4 bytes per block of a round)
__host__ __device__ inline int sk_round(int nb, int nm, int P) {
    const int fit = (SK_LDS / (nm * 16 * P * 4)) & ~7, all = (nb + 7) & ~7;
    return fit < all ? fit : all;
}
template <int WT, int NM, int TT, int PD>
__global__ __launch_bounds__(SK_WG) void k_sk_gemm(qmh_pf_args a) {
    constexpr int PT = 16 * TT;
    constexpr int NPAIR = 16 * PT / SK_WG > 0 ? 16 * PT / SK_WG : 1;  // (row, token) pairs per thread
    extern __shared__ float T[];
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, kq = l >> 4, tok = l & 15;
    const int r0 = blockIdx.x * 16, P = a.P, nb = a.nb;
    const int rblk = sk_round(nb, NM, P);
    constexpr int CB = WT == QMH_Q8 ? 32 : 16;
    PfLane<NM> ln;
    {
        const int row = r0 + tok;  // the lane's A row
#pragma unroll
        for (int m = 0; m < NM; m++) {
            ln.a[m] = pf_slot0(a, row < a.rows_alloc ? row : 0, m) * CB + (WT == QMH_Q8 ? 8 : 4) * kq;
            ln.w[m] = pf_slot0(a, row < a.rows_alloc ? row : 0, m);
        }
    }
    const uint32_t kmask = kq == 0 ? 0xffffu : 0u;  // lanes of k = 0..3
    ln.x = (uint32_t)tok * 32 + 8 * kq;
    ln.d = (uint32_t)tok;
    float s[NPAIR][NM];
#pragma unroll
    for (int k = 0; k < NPAIR; k++)
#pragma unroll
        for (int m = 0; m < NM; m++) s[k][m] = 0.0f;
    for (int base = 0; base < nb; base += rblk) {
        const int nr = min(rblk, nb - base);
        for (int k0 = 0; 8 * k0 + wave < nr; k0 += PD) {  // uniform per wave
            PfBlock<NM, TT> blk[PD];
#pragma unroll
            for (int j = 0; j < PD; j++) {
                const int jb = 8 * (k0 + j) + wave;
                pf_load<WT, NM, TT>(a, base + (jb < nr ? jb : nr - 1), ln, blk[j]);
            }
#pragma unroll
            for (int j = 0; j < PD; j++) {
                const int jb = 8 * (k0 + j) + wave;
                if (jb < nr) {  // uniform per wave
                    // every MFMA of the block first, each into its own registers, then the terms:
                    // the multiplies overlap instead of each waiting for the previous results. The
                    // scale products dw * dx come from an f16 MFMA with the scales at k = 0 (exact: a
                    // product of two fp16 values), as in k_pf_gemm
                    pf_v4i acc[NM][TT];
                    pf_v4f pw[NM][TT];
                    pf_v4h Bs[TT];
#pragma unroll
                    for (int tt = 0; tt < TT; tt++) {
                        const uint32_t h = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)blk[j].dx[tt]) & kmask;
                        Bs[tt] = __builtin_bit_cast(pf_v4h, make_uint2(h, 0u));
                    }
#pragma unroll
                    for (int m = 0; m < NM; m++) {
                        const long Am = WT == QMH_Q8 ? blk[j].A[m] : pf_q4_operand((uint32_t)blk[j].A[m]);
                        const pf_v4h As = __builtin_bit_cast(pf_v4h, make_uint2(blk[j].wh[m] & kmask, 0u));
#pragma unroll
                        for (int tt = 0; tt < TT; tt++) {
                            const pf_v4i z = {0, 0, 0, 0};
                            const pf_v4f zf = {0.0f, 0.0f, 0.0f, 0.0f};
                            acc[m][tt] = __builtin_amdgcn_mfma_i32_16x16x32_i8(Am, blk[j].B[tt], z, 0, 0, 0);
                            pw[m][tt] = __builtin_amdgcn_mfma_f32_16x16x16f16(As, Bs[tt], zf, 0, 0, 0);
                        }
                    }
#pragma unroll
                    for (int m = 0; m < NM; m++)
#pragma unroll
                        for (int tt = 0; tt < TT; tt++) {
                            const int p = 16 * tt + tok;
                            if (p < P) {  // rows 4*kq .. +3 of token p: one 16-byte store
                                pf_v4f t;
#pragma unroll
                                for (int e = 0; e < 4; e++) t[e] = (float)acc[m][tt][e] * pw[m][tt][e];
                                *(pf_v4f *)(T + ((m * rblk + jb) * P + p) * 16 + 4 * kq) = t;
                            }
                        }
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NPAIR; k++) {
            const int c = threadIdx.x + k * SK_WG, row = c & 15, p = c >> 4;
            if (p < P)
                for (int jb = 0; jb < nr; jb++)  // the matrices' chains side by side, each in block order
#pragma unroll
                    for (int m = 0; m < NM; m++) s[k][m] = s[k][m] + T[((m * rblk + jb) * P + p) * 16 + row];
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < NPAIR; k++) {
        const int c = threadIdx.x + k * SK_WG, row = c & 15, p = c >> 4;
        const float partner = __shfl_xor(s[k][0], 1);  // row ^ 1 of the same token: RoPE's pair
        if (p < P && r0 + row < a.rows) pf_store(a, r0 + row, p, s[k][0], s[k][NM - 1], partner);
    }
}

// ============================================================================ multi-token matvec
//
// Up to BMV_P tokens (batched decode, short prompts): the decode matvec's organisation with one
// record and one term per token. A workgroup owns a contiguous range of whole tiles (contiguous
// slots: tile-major, then block, then row in tile). Its threads stream every slot once (8 Q4_0 or 4
// Q8_0 slots per thread per register set, two sets), and for each token form the block's exact int32
// dot with sdot4 against that token's activation record in LDS, then the term (float)acc * (dw * dx)
// into LDS at [token][slot]. After the stream one lane per (row, token) walks its terms in block order
// from +0 (the reference's chain) and runs the prefill epilogue (pf_store).
//
// Records: 48 bytes per (block, token), codes in the order the weights pair with (Q8_0: element
// order; Q4_0: even elements, then odd), then d (fp32), then the code sum (Q4_0: sum (q - 8) x =
// sum q x - 8 sum x, exact). They are built either from the Q8_0 image of k_pf_quant (its perm8
// groups [e0 e2 e4 e6 e1 e3 e5 e7] give their first 4 bytes to the even half and the last 4 to the
// odd half) or, for a plain input, straight from the f32 rows (bmv_records_f32).
#define BMV_P 3
#define BMV_NT 512
#define BMV_REC 48
#define BMV_CH 4  // (row, token) pairs per thread: rows of a workgroup x tokens <= 4*BMV_NT
#define BMV_LDS (160 * 1024)
__host__ __device__ inline int bmv_ntiles(const qmh_pf_args &a) {
    return a.il ? a.rows_alloc / (a.tile_r / 2) : a.rows_alloc / a.tile_r;
}
__host__ __device__ inline int bmv_tile0(int w, int ntiles, int G) { return (int)((long long)w * ntiles / G); }

// Records straight from the f32 rows of a plain (not RMSNorm'd) input, as k_pf_quant computes them:
// item k = p*nb + b is block b of token p, 8 lanes per item with 4 values each, four rounds of
// items at a time. Q4_0 consumers get the split code order.
template <int WT>
__device__ __forceinline__ void bmv_quant_item(const qmh_pf_args &a, uint8_t *rec, int k, int nk, const float (&v)[4]) {
    const int sub = threadIdx.x & 7, P = a.P, nb = a.nb, p = k / nb, b = k - p * nb;
    float m = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float av = fabsf(v[j]);
        m = av > m ? av : m;
    }
    m = qmh_amax8(m);
    const float dd = qmh_h2f(qmh_f2h(qmh_div127(m)));
    int q[4];
    qmh_q8_codes4(v, dd, qmh_rcp(dd), q);
    const int qs = qmh_sum8(q[0] + q[1] + q[2] + q[3]);
    if (k < nk) {
        uint8_t *rp = rec + (size_t)(b * P + p) * BMV_REC;
        if (WT == QMH_Q4) {  // elements 4s, 4s+2 at 2s, 2s+1; 4s+1, 4s+3 at 16+2s, 16+2s+1
            *(uint16_t *)(rp + 2 * sub) = (uint16_t)((q[0] & 0xff) | (q[2] & 0xff) << 8);
            *(uint16_t *)(rp + 16 + 2 * sub) = (uint16_t)((q[1] & 0xff) | (q[3] & 0xff) << 8);
        } else {
            *(uint32_t *)(rp + 4 * sub) =
                (uint32_t)((q[0] & 0xff) | (q[1] & 0xff) << 8 | (q[2] & 0xff) << 16 | (q[3] & 0xff) << 24);
        }
        if (sub == 0) {
            *(float *)(rp + 32) = dd;
            *(int *)(rp + 36) = qs;
        }
    }
}

template <int WT>
__device__ __forceinline__ void bmv_records_f32(const qmh_pf_args &a, uint8_t *rec) {
    const int tid = threadIdx.x, sub = tid & 7, P = a.P, nb = a.nb, n = a.nxf;
    const int nk = P * nb, NR = (nk + BMV_NT / 8 - 1) / (BMV_NT / 8);
    for (int r0 = 0; r0 < NR; r0 += 4) {  // uniform: DPP needs all 8 lanes of an item
        float xv[4][4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int k = (r0 + u) * (BMV_NT / 8) + (tid >> 3), p = k / nb, i0 = (k - p * nb) * 32 + 4 * sub;
#pragma unroll
            for (int j = 0; j < 4; j++)
                xv[u][j] = (r0 + u < NR && k < nk && i0 + j < n) ? a.xf[(size_t)p * a.ldxf + i0 + j] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (r0 + u < NR) bmv_quant_item<WT>(a, rec, (r0 + u) * (BMV_NT / 8) + (tid >> 3), nk, xv[u]);
    }
}

// MP: the largest token count P the instance serves (its per-token loop is unrolled MP times)
template <int WT, int MP>
__global__ __launch_bounds__(BMV_NT, 4) void k_bmv(qmh_pf_args a) {  // 4 waves per SIMD: two per CU
    constexpr int CB = WT == QMH_Q8 ? 32 : 16;  // code bytes per slot
    constexpr int NV = CB / 16;
    constexpr int U = WT == QMH_Q8 ? 4 : 8;      // slots per thread per register set
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, P = a.P, nb = a.nb, R = a.tile_r, lgR = __builtin_ctz((unsigned)R);
    const int ntiles = bmv_ntiles(a);
    const int t0 = bmv_tile0(blockIdx.x, ntiles, gridDim.x), t1 = bmv_tile0(blockIdx.x + 1, ntiles, gridDim.x);
    const int ntw = t1 - t0;
    if (ntw <= 0) return;  // the host launches at most ntiles workgroups
    // blocks per LDS round: all of them, or (one tile per workgroup) as many as let two workgroups
    // share a CU; each round's terms extend the chains before the next round overwrites them
    const int bq = a.bmv_bq > 0 && a.bmv_bq < nb && ntw == 1 ? a.bmv_bq : nb;
    float *T = (float *)(smem + (size_t)nb * P * BMV_REC);
    const uint8_t *cbase = a.codes + (size_t)t0 * nb * R * CB;
    const uint16_t *sbase = a.scales + (size_t)t0 * nb * R;
    uint4 cA[U][NV], cB[U][NV];
    uint32_t sA[U], sB[U];
    int q0 = 0, nbq = bq, TS = ntw * bq * R;  // the round's first block, blocks, slots
    // slot l = j*BMV_NT + tid of the round: block column (l >> lgR) = (tid >> lgR) + j*(BMV_NT >> lgR);
    // its block index in the round is that mod nbq, kept incrementally (step < nbq). With several
    // tiles there is one round (q0 = 0); with rounds there is one tile, so slot q0*R + l of the range
    auto load = [&](uint4 (&c)[U][NV], uint32_t (&sc)[U], int j0) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int l0 = (j0 + u) * BMV_NT + tid, l = (l0 < TS ? l0 : TS - 1) + q0 * R;
#pragma unroll
            for (int v = 0; v < NV; v++) c[u][v] = *(const uint4 *)(cbase + (size_t)l * CB + 16 * v);
            sc[u] = sbase[l];
        }
    };
    load(cA, sA, 0);

    if (a.xf) {
        bmv_records_f32<WT>(a, smem);
    } else {
    // records from the quantized image
    const int nitems = nb * P * 4;  // (block, token, 8-byte group); groups of one record in adjacent lanes
    for (int i0 = 0; i0 < nitems; i0 += BMV_NT) {
        const int it = i0 + tid, g = it & 3, bp = it >> 2, b = bp / P, p = bp - b * P;
        const bool ok = it < nitems;
        int2 v = make_int2(0, 0);
        if (ok) v = *(const int2 *)(a.xc + ((size_t)b * a.PP + p) * 32 + 8 * g);
        int sum = __builtin_amdgcn_sdot4(v.x, 0x01010101, 0, false);
        sum = __builtin_amdgcn_sdot4(v.y, 0x01010101, sum, false);
        sum += __shfl_xor(sum, 1);
        sum += __shfl_xor(sum, 2);
        if (ok) {
            uint8_t *rec = smem + (size_t)bp * BMV_REC;
            if (WT == QMH_Q4) {
                *(int *)(rec + 4 * g) = v.x;
                *(int *)(rec + 16 + 4 * g) = v.y;
            } else {
                *(int2 *)(rec + 8 * g) = v;
            }
            if (g == 0) {
                *(float *)(rec + 32) = a.xd[(size_t)b * a.PP + p];
                *(int *)(rec + 36) = sum;
            }
        }
    }
    }
    __syncthreads();

    // the rounds: stream (terms to LDS), then every chain extended over the round's blocks in order
    const int rows_w = ntw * R, npair = rows_w * P;  // pair c = p*rows_w + i: row i of the range, token p
    float yk[BMV_CH];
#pragma unroll
    for (int kc = 0; kc < BMV_CH; kc++) yk[kc] = 0.0f;
    for (q0 = 0; q0 < nb; q0 += bq) {
        nbq = nb - q0 < bq ? nb - q0 : bq;
        TS = ntw * nbq * R;
        const int nper = (TS + BMV_NT - 1) / BMV_NT, bstep = (BMV_NT >> lgR) % nbq;
        int bcur = (tid >> lgR) % nbq;
        auto compute = [&](const uint4 (&c)[U][NV], const uint32_t (&sc)[U], int j0) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int l = (j0 + u) * BMV_NT + tid;
                if (j0 + u < nper) {  // uniform
                    const float dw = qmh_h2f((uint16_t)sc[u]);
#pragma unroll
                    for (int p = 0; p < MP; p++)
                        if (p < P) {
                            const uint8_t *rp = smem + (size_t)((q0 + bcur) * P + p) * BMV_REC;
                            const int4 x0 = *(const int4 *)rp, x1 = *(const int4 *)(rp + 16);
                            const float2 ds = *(const float2 *)(rp + 32);
                            int acc;
                            if (WT == QMH_Q4) {
                                const uint4 w = c[u][0];
                                acc = -8 * __float_as_int(ds.y);
                                acc = __builtin_amdgcn_sdot4((int)(w.x & 0x0f0f0f0fu), x0.x, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)((w.x >> 4) & 0x0f0f0f0fu), x1.x, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)(w.y & 0x0f0f0f0fu), x0.y, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)((w.y >> 4) & 0x0f0f0f0fu), x1.y, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)(w.z & 0x0f0f0f0fu), x0.z, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)((w.z >> 4) & 0x0f0f0f0fu), x1.z, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)(w.w & 0x0f0f0f0fu), x0.w, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)((w.w >> 4) & 0x0f0f0f0fu), x1.w, acc, false);
                            } else {
                                const uint4 w0 = c[u][0], w1 = c[u][NV - 1];
                                acc = __builtin_amdgcn_sdot4((int)w0.x, x0.x, 0, false);
                                acc = __builtin_amdgcn_sdot4((int)w0.y, x0.y, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)w0.z, x0.z, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)w0.w, x0.w, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)w1.x, x1.x, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)w1.y, x1.y, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)w1.z, x1.z, acc, false);
                                acc = __builtin_amdgcn_sdot4((int)w1.w, x1.w, acc, false);
                            }
                            if (l < TS) T[(size_t)p * TS + l] = (float)acc * (dw * ds.x);
                        }
                }
                bcur += bstep;
                bcur -= bcur >= nbq ? nbq : 0;
            }
        };
        if (q0 > 0) load(cA, sA, 0);  // the first round's set was issued before the records
        for (int j0 = 0; j0 < nper; j0 += 2 * U) {
            if (j0 + U < nper) load(cB, sB, j0 + U);
            compute(cA, sA, j0);
            if (j0 + 2 * U < nper) load(cA, sA, j0 + 2 * U);
            if (j0 + U < nper) compute(cB, sB, j0 + U);
        }
        __syncthreads();
#pragma unroll
        for (int kc = 0; kc < BMV_CH; kc++) {
            const int c = kc * BMV_NT + tid, p = c / rows_w, i = c - p * rows_w, tl = i >> lgR, r = i & (R - 1);
            if (c < npair) {
                const float *tp = T + (size_t)p * TS + (size_t)tl * nbq * R + r;
                float y = yk[kc];
                int b = 0;
                for (; b + 16 <= nbq; b += 16) {
                    float v[16];
#pragma unroll
                    for (int k = 0; k < 16; k++) v[k] = tp[(b + k) * R];
#pragma unroll
                    for (int k = 0; k < 16; k++) y = y + v[k];
                }
                for (; b < nbq; b++) y = y + tp[b * R];
                yk[kc] = y;
            }
        }
        __syncthreads();  // the next round's terms overwrite these
    }

    // epilogues: a tile's rows are consecutive lanes of one wave (R divides 64, rows_w is a multiple of R)
#pragma unroll
    for (int kc = 0; kc < BMV_CH; kc++)
        if (kc * BMV_NT < npair) {  // uniform
            const int c = kc * BMV_NT + tid, p = c / rows_w, i = c - p * rows_w, tl = i >> lgR, r = i & (R - 1);
            const float y = yk[kc];
            const int tile = t0 + tl;
            if (a.il) {  // rows r < R/2 of a tile are W1 rows, r + R/2 their W3 rows
                const float up = __shfl_down(y, R >> 1);
                const int row = tile * (R >> 1) + r;
                if (c < npair && r < (R >> 1) && row < a.rows) pf_store(a, row, p, y, up, 0.0f);
            } else {
                const float partner = __shfl_xor(y, 1);  // row ^ 1: RoPE's pair
                const int row = tile * R + r;
                if (c < npair && row < a.rows) pf_store(a, row, p, y, y, partner);
            }
        }
}

extern "C" int qmh_launch_pf_gemm(const qmh_pf_args *a, void *stream) {
    if (a->PP % 128 || a->P > a->PP || a->P < 1 || a->nb < 1) return (int)hipErrorInvalidValue;
    if ((a->epi == QMH_PF_SWIGLU) != (a->il != 0)) return (int)hipErrorInvalidValue;
    if (a->dtype != QMH_Q4 && a->dtype != QMH_Q8) return (int)hipErrorInvalidValue;
    // the image output exists only in the tiled matmul's SwiGLU epilogue
    if (a->qxc && (a->epi != QMH_PF_SWIGLU || !a->qxd || !qmh_pf_tiled(a->P, a->rows, a->nb, a->il))) return (int)hipErrorInvalidValue;
    hipStream_t s = (hipStream_t)stream;
    if (a->xf && (a->nxf < 1 || a->nxf > 32 * a->nb || a->ldxf < a->nxf)) return (int)hipErrorInvalidValue;
    // the multi-token matvec when one tile's terms fit its LDS with the records. It quantizes a plain
    // input (Wo's, W2's) itself: timed on MI355X at 1-4 tokens, that saves 5-9 us per matmul over
    // k_pf_quant's launch, while an RMSNorm'd input quantized in every workgroup was 6 us slower.
    const int ntiles = bmv_ntiles(*a);
    const size_t rec = (size_t)a->nb * a->P * BMV_REC, per_tile = (size_t)a->P * a->tile_r * a->nb * sizeof(float);
    const bool bmv = a->P <= BMV_P && rec + per_tile <= BMV_LDS &&
                     (size_t)a->tile_r * a->P * ((ntiles + 255) / 256) <= (size_t)BMV_CH * BMV_NT;
    const bool fuse = bmv && a->xf && !a->norm_w;
    if (a->xf && !fuse) {  // the quantized image first
        const int rc = qmh_launch_pf_quant(a->xf, a->ldxf, a->norm_w, a->eps, a->nxf, a->P, (int8_t *)a->xc,
                                           (float *)a->xd, a->PP, a->dtype == QMH_Q4, stream);
        if (rc) return rc;
    }
    if (bmv) {
        qmh_pf_args b = *a;
        if (!fuse) b.xf = nullptr;
        // whole tiles per workgroup: about one workgroup per CU (256), fewer tiles if LDS asks
        const int fit = (int)((BMV_LDS - rec) / per_tile), want = ntiles / 256 > 1 ? ntiles / 256 : 1;
        const int k = want < fit ? want : fit, G = (ntiles + k - 1) / k;
        size_t lds = rec + (size_t)((ntiles + G - 1) / G) * per_tile;
        // one tile per workgroup, more workgroups than CUs and room for one per CU: LDS rounds of bq
        // blocks so that two share a CU
        b.bmv_bq = 0;
        const size_t per_block = (size_t)a->P * a->tile_r * sizeof(float);
        if (k == 1 && ntiles > 256 && 2 * lds > BMV_LDS && 2 * rec < BMV_LDS) {
            const int bq = (int)((BMV_LDS / 2 - rec) / per_block);
            if (bq >= 16 && bq < a->nb) {
                b.bmv_bq = bq;
                lds = rec + (size_t)bq * per_block;
            }
        }
#define BMV_GO(MP_)                                                                                    \
    do {                                                                                                 \
        if (a->dtype == QMH_Q4) hipLaunchKernelGGL((k_bmv<QMH_Q4, MP_>), dim3(G), dim3(BMV_NT), lds, s, b); \
        else hipLaunchKernelGGL((k_bmv<QMH_Q8, MP_>), dim3(G), dim3(BMV_NT), lds, s, b);                  \
    } while (0)
        // one instance for 1-2 tokens, one for 3 (the single-token instance was 2% slower at one
        // sequence than the 2-token one)
        static_assert(BMV_P == 3, "k_bmv instances for up to 3 tokens");
        if (a->P <= 2) BMV_GO(2);
        else BMV_GO(3);
#undef BMV_GO
        return (int)hipGetLastError();
    }
    if (!qmh_pf_tiled(a->P, a->rows, a->nb, a->il)) {  // decode-sized batches: the skinny matmul streams every weight once
        const dim3 g((a->rows + 15) / 16);
        const int nm = a->il ? 2 : 1;
        const size_t lds = (size_t)sk_round(a->nb, nm, a->P) * nm * 16 * a->P * sizeof(float);
#define SK_LAUNCH(NMV, TTV, PDV)                                                                              \
    do {                                                                                                      \
        if (a->dtype == QMH_Q4)                                                                               \
            hipLaunchKernelGGL((k_sk_gemm<QMH_Q4, NMV, TTV, PDV>), g, dim3(SK_WG), lds, s, *a);               \
        else                                                                                                  \
            hipLaunchKernelGGL((k_sk_gemm<QMH_Q8, NMV, TTV, PDV>), g, dim3(SK_WG), lds, s, *a);               \
    } while (0)
        // load depths timed on MI355X over the 7B shapes: for W1 | W3 up to 4 tokens, 3 blocks
        // ahead (113 VGPRs: two workgroups per CU) beat 8 by 5%; from 5 tokens 8 is ahead
        if (a->P <= 4 && a->il) {
            SK_LAUNCH(2, 1, 3);
        } else if (a->P <= 16) {
            if (a->il) SK_LAUNCH(2, 1, 8);
            else SK_LAUNCH(1, 1, 6);
        } else if (a->P <= 32) {
            if (a->il) SK_LAUNCH(2, 2, 4);
            else SK_LAUNCH(1, 2, 8);
        } else {  // 33..64 tokens: a round holds 16 (W1 | W3) or 32 blocks, 2 or 4 per wave; 2 ahead
            if (a->il) SK_LAUNCH(2, 4, 2);
            else SK_LAUNCH(1, 4, 2);
        }
#undef SK_LAUNCH
        return (int)hipGetLastError();
    }
    // the tiled matmul. Token groups past P are not launched, and 64 divides PP, so every read of the
    // activations stays in the PP-token image. 4 x 2 tiles per workgroup, two waves per SIMD of a CU;
    // 2 x 2 where 4 x 2 would leave half of the CUs idle or more (timed, us, 4 x 2 -> 2 x 2: 4096x11008 at
    // 96 tokens, 64 workgroups, 82 -> 66; 2048x5632 at 512, 128, 47 -> 39; 4096x4096 at 300, 160,
    // 36.7 -> 37.8) and for W1 | W3, whose 64-slot tiles it reads whole (4096 columns: 197 -> 186; 2048:
    // 59 -> 60), both with the loads two stages ahead. Up to 32 tokens 2 x 1, which has no second token
    // tile to compute for nothing (2 x 2 -> 2 x 1: 32000x4096 36 -> 33, W1 | W3 40 -> 36, 12288x4096
    // 34 -> 32).
    const int tg = (a->P + 63) / 64, g4 = tg * ((a->rows + 127) / 128);
#define PG_LAUNCH(IL_, RT_, TT_, DEEP_, ROWS_)                                                                \
    do {                                                                                                      \
        const dim3 g((a->P + 32 * (TT_)-1) / (32 * (TT_)), (a->rows + (ROWS_)-1) / (ROWS_));                  \
        if (a->dtype == QMH_Q4)                                                                               \
            hipLaunchKernelGGL((k_pf_gemm<QMH_Q4, IL_, RT_, TT_, DEEP_>), g, dim3(64 * RT_ * TT_), 0, s, *a); \
        else                                                                                                  \
            hipLaunchKernelGGL((k_pf_gemm<QMH_Q8, IL_, RT_, TT_, DEEP_>), g, dim3(64 * RT_ * TT_), 0, s, *a); \
    } while (0)
    if (a->il && a->P <= 32) PG_LAUNCH(true, 2, 1, 1, 32);
    else if (a->il) PG_LAUNCH(true, 2, 2, 1, 32);
    else if (a->P <= 32) PG_LAUNCH(false, 2, 1, 1, 64);
    else if (g4 <= 128) PG_LAUNCH(false, 2, 2, 1, 64);
    else PG_LAUNCH(false, 4, 2, 0, 128);
#undef PG_LAUNCH
    return (int)hipGetLastError();
}

// ============================================================================ attention
//
// Scores of 16 tokens against 256 positions per workgroup (lane = position; 16 serial dot
// chains over head_dim per lane, K^T read once for the 16 tokens), each times the scale as
// src/model.c:146. Rows of att: (head, token) with max_seq entries; entries past the token's
// position are not written.
#define QMH_PF_TOK 16
__global__ __launch_bounds__(QMH_WG) void k_pf_scores(const float *__restrict__ Q, const float *__restrict__ Kt,
                                                      float *att, int P, int pos0, int n_heads, int n_kv, int hd,
                                                      int max_seq, float scale) {
    const int h = blockIdx.x, g = blockIdx.y, t = blockIdx.z * QMH_WG + threadIdx.x;
    const int p0 = g * QMH_PF_TOK, np = min(QMH_PF_TOK, P - p0);
    // a wave whose 64 positions are all past the group's last token has nothing to store (the
    // kernel has no barrier, so waves leave independently)
    if ((int)(blockIdx.z * QMH_WG + (threadIdx.x & ~63u)) > pos0 + p0 + np - 1) return;
    const int kvh = h / (n_heads / n_kv), D = n_heads * hd;
    // the group's queries, read with uniform (scalar) loads: every lane needs the same values.
    // Tokens past P read the last token's row (their scores are never stored).
    const float *qg = Q + (size_t)h * hd;
    const int tc = t < max_seq ? t : max_seq - 1;
    const float *kc = Kt + (size_t)kvh * hd * max_seq + tc;
    float s[QMH_PF_TOK];
#pragma unroll
    for (int k = 0; k < QMH_PF_TOK; k++) s[k] = 0.0f;
    // 64 K values of the lane's position in flight, then four dimensions per step (hd is a
    // multiple of 4)
    for (int d0 = 0; d0 < hd; d0 += 64) {
        float kv[64];
#pragma unroll
        for (int j = 0; j < 64; j++) kv[j] = kc[(size_t)(d0 + j < hd ? d0 + j : hd - 1) * max_seq];
#pragma unroll
        for (int j = 0; j < 64; j += 4)
            if (d0 + j < hd) {
#pragma unroll
                for (int k = 0; k < QMH_PF_TOK; k++) {
                    const float *qk = qg + (size_t)(p0 + k < P ? p0 + k : P - 1) * D + d0 + j;
                    const float4 q4 = make_float4(qk[0], qk[1], qk[2], qk[3]);
                    s[k] = s[k] + q4.x * kv[j];
                    s[k] = s[k] + q4.y * kv[j + 1];
                    s[k] = s[k] + q4.z * kv[j + 2];
                    s[k] = s[k] + q4.w * kv[j + 3];
                }
            }
    }
#pragma unroll
    for (int k = 0; k < QMH_PF_TOK; k++)
        if (k < np && t <= pos0 + p0 + k) att[((size_t)h * P + p0 + k) * max_seq + t] = s[k] * scale;
}

// The same scores with the products from MFMAs, for head_dim 128, 64 and 48: v_mfma_f32_16x16x1_4b_f32
// with a zero accumulator is 1024 correctly rounded products q[d] * k[d] (16 tokens x 4 x 16 positions;
// checked on the device over every exponent, subnormals and special values included), and the VALU
// adds them to the chains: s = +0, s = s + q[d] * k[d] over d in order, then s * scale. (A product of
// -0 may come out as +0: a chain is never -0, so the sum is the same.) The f32 MFMA runs on the VALU's
// units at the rate of its multiplies, but it takes one register each of query and key per 1024 products,
// where register blocking on the VALU (4 x 4 per thread) read 32 bytes of LDS per 16 products and filled the
// LDS return path. Keys come straight from memory; below 128 dimensions a wave's queries go through LDS of its
// own, loaded as whole rows (read from memory by token, each lane of a load is another cache line: 46 us
// where this takes 42); at 128 the longer start and 34 KB of LDS per workgroup cost what that saves (29 -> 31). One wave per tile of 16 tokens x 64 positions; a workgroup's
// 4 waves take 4 consecutive token tiles of the same positions, whose keys they share in L1. Timed, us,
// register blocking -> this: 512 tokens, 32 heads x 128 dimensions 33 -> 29; a 1901-token prompt of 32
// heads x 64, per 512-token pass, 49 -> 42 (two VALU operations per pair and dimension at two waves per
// SIMD would be 14 and 24; the score writes are 12 of the 42). 32 x 64 tiles, and queries in scalar
// registers (8 tokens x 128 positions per wave), took 36-39 at the first shape.
template <int HD>
__global__ __launch_bounds__(QMH_WG, 4) void k_pf_scores_m(const float *__restrict__ Q, const float *__restrict__ Kt,
                                                           float *att, int P, int pos0, int n_heads, int n_kv,
                                                           int max_seq, float scale) {
    constexpr int DG = 8;  // dimensions per register set; the next set loads while one is used
    static_assert(HD % (2 * DG) == 0, "whole pairs of sets");
    constexpr bool QL = HD < 128;  // queries through LDS
    const int h = blockIdx.x, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), l = threadIdx.x & 63;
    const int p0 = blockIdx.y * 64 + 16 * wave, c0 = blockIdx.z * 64;
    if (p0 >= P || c0 > pos0 + min(p0 + 15, P - 1)) return;  // past the prompt, or past every token (whole wave)
    const int kvh = h / (n_heads / n_kv);
    const int tc = min(c0 + l, max_seq - 1);
    const float *q = Q + ((size_t)min(p0 + (l & 15), P - 1) * n_heads + h) * HD;
    if (QL) {  // the wave's queries, whole rows at a time
        __shared__ __align__(16) float qs[QL ? 4 : 1][16][HD + 4];
#pragma unroll
        for (int i = 0; i < HD / 16; i++) {
            const int r = (64 * i + l) / (HD / 4), d = 4 * ((64 * i + l) % (HD / 4));
            *(pf_v4f *)&qs[wave][r][d] = *(const pf_v4f *)(Q + ((size_t)min(p0 + r, P - 1) * n_heads + h) * HD + d);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // within the wave: LDS operations stay in order
        __builtin_amdgcn_wave_barrier();
        q = qs[wave][l & 15];
    }
    // every offset below lies in the kv head's keys: positions clamped to max_seq - 1, dimensions below HD
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void *)(Kt + (size_t)kvh * HD * max_seq), (short)0, (int)((uint32_t)HD * (uint32_t)max_seq * 4u), 0x00020000);
    pf_v4f qv[2][DG / 4];
    float kv[2][DG];
    auto load = [&](int d0, int w) {
#pragma unroll
        for (int d = 0; d < DG / 4; d++) qv[w][d] = *(const pf_v4f *)(q + d0 + 4 * d);
#pragma unroll
        for (int d = 0; d < DG; d++) kv[w][d] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rk, tc * 4, (uint32_t)(d0 + d) * (uint32_t)max_seq * 4u, 0));
    };
    float s[16];
    pf_v16f z;
#pragma unroll
    for (int e = 0; e < 16; e++) s[e] = z[e] = 0.0f;
    load(0, 0);
#pragma unroll 1
    for (int d0 = 0; d0 < HD; d0 += 2 * DG) {
#pragma unroll
        for (int w = 0; w < 2; w++) {
            const int dn = d0 + (w + 1) * DG;
            load(dn < HD ? dn : 0, w ^ 1);
            // the next dimension's products go out before this one's are added
            pf_v16f f[2];
            auto mul = [&](int d) { f[d & 1] = __builtin_amdgcn_mfma_f32_16x16x1f32(qv[w][d / 4][d % 4], kv[w][d], z, 0, 0, 0); };
            mul(0);
#pragma unroll
            for (int d = 0; d < DG; d++) {
                if (d + 1 < DG) mul(d + 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int e = 0; e < 16; e++) s[e] = s[e] + f[d & 1][e];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // element 4*b + e: token 4*(l/16) + e, position 16*b + l%16
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int pt = p0 + 4 * (l >> 4) + e;
        float *row = att + ((size_t)h * P + pt) * max_seq + c0 + (l & 15);
#pragma unroll
        for (int b = 0; b < 4; b++)
            if (pt < P && c0 + 16 * b + (l & 15) <= pos0 + pt) row[16 * b] = s[4 * b + e] * scale;
    }
}

// softmax of one (head, token) row in place (src/ops.c:100-112), one wave per row (4 rows per
// workgroup): the max and the double sum of the exponentials by shuffles, no barrier. The final
// pass recomputes each exponential instead of storing and re-reading it (the same bits), so the
// serial fallback of the sum works from the untouched scores.
__global__ __launch_bounds__(QMH_WG) void k_pf_softmax(float *att, int P, int pos0, int max_seq) {
    const int h = blockIdx.x, p = blockIdx.y * (QMH_WG / 64) + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (p >= P) return;  // the whole wave
    const int n = pos0 + p + 1;
    float *x = att + ((size_t)h * P + p) * max_seq;
    const float x0 = x[0];
    float m = -__builtin_inff();
    for (int t = lane; t < n; t += 64) m = x[t] > m ? x[t] : m;
    m = qmh_wave_max(m);
    if (x0 != x0) m = x0;  // the reference's scan starts from x[0]: a NaN there stays
    double sum = 0.0;
    for (int t = lane; t < n; t += 64) sum += (double)qmh_expf(x[t] - m);
    sum = qmh_wave_sum_d(sum);
    const double d = qmh_sum_slack(sum, n);
    float inv = qmh_recip_of_sum(sum - d);
    if (inv != qmh_recip_of_sum(sum + d)) {  // uniform; serial sum as the reference
        double ser = 0.0;
        if (lane == 0)
            for (int t = 0; t < n; t++) ser += (double)qmh_expf(x[t] - m);
        inv = qmh_recip_of_sum(__shfl(ser, 0));
    }
    for (int t = lane; t < n; t += 64) x[t] = qmh_expf(x[t] - m) * inv;
}

// k_pf_softmax with the row in registers (rows of up to 64*W*R positions, W waves per row): one
// range-checked load per value, all issued at once; each exponential is computed once and kept for both
// the sum and the probability (the same values k_pf_softmax computes twice). The exponentials take no
// branch (qmh_expf_nonpos) and their table from LDS, so a lane's R of them overlap; with the branches of
// qmh_expf each waited for the one before. Timed, us per 512-token pass of 32 heads, before ->
// after: rows up to 512 31 -> 14, up to 1901 140 -> 41 (one wave per row recomputing each exponential); the
// serial sum, below, was most of it.
template <int R, int W>
__global__ __launch_bounds__(QMH_WG) void k_pf_softmax_r(float *att, int P, int pos0, int max_seq) {
    __shared__ uint64_t tab[32];
    __shared__ float redf[4];
    __shared__ double redd[4];
    constexpr int RW = 4 / W, LN = 64 * W;  // rows per workgroup, lanes per row
    __shared__ float ex[W > 1 ? LN * R : 1];  // the exponentials, for the serial sum
    const int tid = threadIdx.x;
    const int rw = __builtin_amdgcn_readfirstlane(tid / LN);  // uniform per wave: a scalar resource
    const int h = blockIdx.x, p = blockIdx.y * RW + rw, lane = tid % LN;
    if (tid < 32) tab[tid] = qmh_exp2_tab[tid];
    const int pc = p < P ? p : P - 1;
    const int n = pos0 + pc + 1;
    float *x = att + ((size_t)h * P + pc) * max_seq;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)x, (short)0, n * 4, 0x00020000);
    float xv[R];
#pragma unroll
    for (int r = 0; r < R; r++) xv[r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, (r * LN + lane) * 4, 0, 0));
    const float x0 = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rx, 0, 0, 0));
    __syncthreads();
    if (p >= P) return;  // W == 1: whole waves, and no barrier follows
    float m = -__builtin_inff();
#pragma unroll
    for (int r = 0; r < R; r++)
        if (r * LN + lane < n) m = xv[r] > m ? xv[r] : m;
    m = qmh_wave_max(m);
    if (W > 1) {
        if ((tid & 63) == 0) redf[tid >> 6] = m;
        __syncthreads();
        m = redf[0];
#pragma unroll
        for (int w = 1; w < W; w++) m = fmaxf(m, redf[w]);
    }
    if (x0 != x0) m = x0;  // the reference's scan starts from x[0]: a NaN there stays
    float e[R];
    double sum = 0.0;
#pragma unroll
    for (int r = 0; r < R; r++) {
        e[r] = 0.0f;
        if (r * LN < n) {  // uniform: rounds past the row cost nothing
            e[r] = qmh_expf_nonpos(xv[r] - m, tab);
            e[r] = r * LN + lane < n ? e[r] : 0.0f;  // + 0 leaves the sum as it is
            sum += (double)e[r];
        }
    }
    sum = qmh_wave_sum_d(sum);
    if (W > 1) {
        if ((tid & 63) == 0) redd[tid >> 6] = sum;
        __syncthreads();
        sum = redd[0];
#pragma unroll
        for (int w = 1; w < W; w++) sum += redd[w];
    }
    const double d = qmh_sum_slack(sum, n);
    float inv = qmh_recip_of_sum(sum - d);
    if (inv != qmh_recip_of_sum(sum + d)) {  // uniform over the row; serial sum as the reference
        // every lane of a wave adds the row's exponentials in order, broadcast from the lanes that hold
        // them (about 20 cycles each; one lane recomputing them took 140 ns each, 83 us for a row that
        // most calls of 512 rows x 32 heads have one of in thirty)
        double ser = 0.0;
        if (W > 1) {
#pragma unroll
            for (int r = 0; r < R; r++) ex[r * LN + lane] = e[r];
            __syncthreads();
        }
#pragma unroll 1
        for (int c = 0; c < n; c += 64) {
            float v;
            if (W > 1) {
                v = ex[c + (tid & 63)];
            } else {
                v = e[0];
#pragma unroll
                for (int r = 1; r < R; r++) v = c == 64 * r ? e[r] : v;
            }
            const int nc = n - c < 64 ? n - c : 64;
#pragma unroll 1
            for (int i = 0; i < nc; i++)
                ser += (double)__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), i));
        }
        inv = qmh_recip_of_sum(ser);
    }
#pragma unroll
    for (int r = 0; r < R; r++)
        if (r * LN + lane < n) x[r * LN + lane] = e[r] * inv;
}

// out[token][h*hd + i] = +0 + p_0 v_0[i] + p_1 v_1[i] + ... in position order (src/model.c:147-154);
// one workgroup per (head, 16 tokens), head_dim <= 128. V and the probabilities pass through LDS
// in chunks of 64 positions (cooperative float4 loads, the next chunk's held in registers while
// the current one is used); thread (i, half) runs column i's chains of tokens 8*half .. +7.
// The probabilities sit in LDS as [position][token], so a thread's 8 per position are two
// 16-byte reads. Positions up to pos0 + p0 are seen by every token of the group and run four at a
// time with no mask; the last 15 positions of the group (its causal diagonal) extend only the
// chains of the tokens that see them (a select, never an added zero: that would turn -0 into +0
// and propagate a NaN from V).
#define QMH_PF_VC 64
__global__ __launch_bounds__(QMH_WG) void k_pf_pv(const float *__restrict__ att, const float *__restrict__ V,
                                                  float *out, int P, int pos0, int n_heads, int n_kv, int hd,
                                                  int max_seq) {
    __shared__ __align__(16) float ps[QMH_PF_VC * QMH_PF_TOK];  // [t][token]
    __shared__ __align__(16) float vs[QMH_PF_VC * 128];         // [t][column]
    const int h = blockIdx.x, p0 = blockIdx.y * QMH_PF_TOK, np = min(QMH_PF_TOK, P - p0);
    const int kvh = h / (n_heads / n_kv), kvd = hd * n_kv, tid = threadIdx.x;
    const int tmax = pos0 + p0 + np;  // positions 0 .. tmax-1 are used by some token
    const int tall = pos0 + p0 + 1;   // positions 0 .. tall-1 are used by every token of the group
    const float *vbase = V + (size_t)kvh * hd;
    const int hd4 = hd >> 2;
    constexpr int VR = QMH_PF_VC * 128 / 4 / QMH_WG;     // float4 of V per thread per chunk
    constexpr int PR = QMH_PF_TOK * QMH_PF_VC / QMH_WG;  // probabilities per thread per chunk
    float4 vr[VR];
    float pr[PR];
    auto load = [&](int c0) {
#pragma unroll
        for (int k = 0; k < VR; k++) {
            const int e = k * QMH_WG + tid, t = e >> 5, c4 = e & 31;  // 32 float4 slots per row
            const int tc = c0 + t < tmax ? c0 + t : tmax - 1;
            vr[k] = c4 < hd4 ? *(const float4 *)(vbase + (size_t)tc * kvd + 4 * c4) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int k = 0; k < PR; k++) {
            const int e = k * QMH_WG + tid, kk = e / QMH_PF_VC, t = c0 + e % QMH_PF_VC;
            pr[k] = (kk < np && t <= pos0 + p0 + kk) ? att[((size_t)h * P + p0 + kk) * max_seq + t] : 0.0f;
        }
    };
    const int i = tid & 127, half = tid >> 7;
    float acc[8];
#pragma unroll
    for (int k = 0; k < 8; k++) acc[k] = 0.0f;
    load(0);
    for (int c0 = 0; c0 < tmax; c0 += QMH_PF_VC) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < VR; k++) {
            const int e = k * QMH_WG + tid;
            *(float4 *)(vs + (e >> 5) * 128 + 4 * (e & 31)) = vr[k];
        }
#pragma unroll
        for (int k = 0; k < PR; k++) {
            const int e = k * QMH_WG + tid;
            ps[(e % QMH_PF_VC) * QMH_PF_TOK + e / QMH_PF_VC] = pr[k];
        }
        if (c0 + QMH_PF_VC < tmax) load(c0 + QMH_PF_VC);
        __syncthreads();
        if (i < hd) {
            const int nt = min(QMH_PF_VC, tmax - c0);
            const int nall = min(nt, max(tall - c0, 0));  // positions of this chunk every token sees
            const float *pp = ps + 8 * half;
            int t = 0;
            for (; t + 4 <= nall; t += 4) {
                float v[4];
                float4 pa[4], pb[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    v[u] = vs[(t + u) * 128 + i];
                    pa[u] = *(const float4 *)(pp + (t + u) * QMH_PF_TOK);
                    pb[u] = *(const float4 *)(pp + (t + u) * QMH_PF_TOK + 4);
                }
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    acc[0] = acc[0] + pa[u].x * v[u];
                    acc[1] = acc[1] + pa[u].y * v[u];
                    acc[2] = acc[2] + pa[u].z * v[u];
                    acc[3] = acc[3] + pa[u].w * v[u];
                    acc[4] = acc[4] + pb[u].x * v[u];
                    acc[5] = acc[5] + pb[u].y * v[u];
                    acc[6] = acc[6] + pb[u].z * v[u];
                    acc[7] = acc[7] + pb[u].w * v[u];
                }
            }
            for (; t < nt; t++) {
                const float v = vs[t * 128 + i];
                const float4 pa = *(const float4 *)(pp + t * QMH_PF_TOK), pb = *(const float4 *)(pp + t * QMH_PF_TOK + 4);
                const float pk[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
                const int kmin = c0 + t - (pos0 + p0);  // tokens kk >= kmin see position c0 + t
#pragma unroll
                for (int k = 0; k < 8; k++) {
                    const float nx = acc[k] + pk[k] * v;
                    acc[k] = 8 * half + k >= kmin ? nx : acc[k];
                }
            }
        }
    }
    if (i < hd)
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int kk = 8 * half + k;
            if (kk < np) out[(size_t)(p0 + kk) * n_heads * hd + h * hd + i] = acc[k];
        }
}

// The same P.V with the products from MFMAs, for head_dim 128, 64 and 48: v_mfma_f32_16x16x1_4b_f32 with a
// zero accumulator gives the products p_t * v_t[i] (rounded as the reference rounds them, see
// k_pf_scores_m) of 16 tokens x 32 columns at two positions, t + j in its first two 16x16 blocks and
// t + 4 + j in the others; four of them (j = 0..3) hold 8 positions, and 64 VALU adds then extend the 8
// chains of each lane position by position. Per 8 positions a wave loads one 16-byte piece of probabilities
// and four V values per lane, with no LDS and no barrier. The number of chains bounds the parallelism: with
// 32 columns per wave, 512 tokens x 32 heads x 64 columns are two waves per SIMD (64 columns per wave and
// one position per MFMA left one, which issues VALU work at half the rate: 81 us where this takes 50).
// Register blocking on the VALU (4 tokens x 2 columns per thread) read 24 bytes of LDS per 8 products;
// probabilities in scalar registers waited for the scalar cache. Positions up to the first token's are
// seen by every token; the last 15 extend only the chains of the tokens that see them (a select, never an
// added zero: a NaN from V must not pass). Wo's input image (xc): the tile through LDS, then the
// quantizer's steps. Timed, us, register blocking -> this: 512 tokens, 32 heads x 128 columns 44 -> 26; a
// 1901-token prompt of 32 heads x 64, per 512-token pass, 98 -> 50.
template <int HD>
__global__ __launch_bounds__(QMH_WG, 4) void k_pf_pv_m(const float *__restrict__ att, const float *__restrict__ V,
                                                       float *out, int P, int pos0, int n_heads, int n_kv, int max_seq,
                                                       int8_t *xc, float *xd, int PP, int perm8) {
    constexpr int CG = (HD + 31) / 32;             // 32-column groups of a head
    constexpr int CW = CG % 4 == 0 ? 4 : CG % 2 == 0 ? 2 : 1, TW = 4 / CW;  // waves: CW column groups x TW token groups
    __shared__ __align__(16) float tile[4][16][36];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), l = threadIdx.x & 63, hi = l >> 5;
    // token groups, the long ones first and the second half reversed, so that the workgroups a CU gets
    // carry equal work in sum
    const int G = gridDim.y, half = (G + 1) / 2, y = blockIdx.y;
    const int grp = y < half ? G - 1 - y : y - half;
    const int h = blockIdx.x / (CG / CW), c0 = ((blockIdx.x % (CG / CW)) * CW + wave % CW) * 32;
    const int p0 = (grp * TW + wave / CW) * 16;
    if (p0 >= P) return;  // the whole wave; no barrier follows
    const int np = min(16, P - p0), kvh = h / (n_heads / n_kv), kvd = HD * n_kv;
    const int tall = pos0 + p0 + 1, tmax = pos0 + p0 + np;  // positions seen by every token, by some token
    const int pl = p0 + (l & 15), cl = c0 + (l & 31);
    // Resources: the token group's probabilities, and per j the kv head's V from row j. The sets loaded ahead
    // run past the last position, and a 4-position load past the last row's end: the range check reads those
    // as 0, and they are not used. It need cover the lane's offset only, so the position is in there and nothing
    // in the scalar offset.
    const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc((void *)(att + ((size_t)h * P + p0) * max_seq), (short)0, (int)((uint32_t)np * (uint32_t)max_seq * 4u), 0x00020000);
    __amdgpu_buffer_rsrc_t rv[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const uint32_t n = j < max_seq ? ((uint32_t)(max_seq - j) * (uint32_t)kvd - (uint32_t)(kvh * HD)) * 4u : 0u;
        rv[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(V + (size_t)kvh * HD + (size_t)j * kvd), (short)0, (int)n, 0x00020000);
    }
    uint32_t po = ((uint32_t)(pl < P ? l & 15 : np - 1) * (uint32_t)max_seq + 4u * hi) * 4u;
    uint32_t vo = ((uint32_t)(cl < HD ? cl : 0) + 4u * hi * (uint32_t)kvd) * 4u;
    const uint32_t vst = 32u * (uint32_t)kvd;
    constexpr int NB = 3;  // sets of 8 positions: one used, two in flight
    pf_v4u pr[NB];
    float vr[NB][4];
    auto load = [&](int w) {  // the next set
        pr[w] = __builtin_amdgcn_raw_buffer_load_b128(rp, po, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; j++) vr[w][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv[j], vo, 0, 0));
        po += 32u, vo += vst;
    };
    float s[8];  // element 4*b + e: token row0 + e, column 16*b + l%16
    pf_v16f z;
#pragma unroll
    for (int e = 0; e < 16; e++) z[e] = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) s[e] = 0.0f;
    const int row0 = 4 * (l >> 4);
    auto group = [&](int w, int t0, bool diag) {
        pf_v16f f[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            f[j] = __builtin_amdgcn_mfma_f32_16x16x1f32(__uint_as_float(pr[w][j]), vr[w][j], z, 0, 0, 0);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int kmin = t0 + k - (pos0 + p0);  // tokens >= kmin see the position
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float nx = s[e] + f[k % 4][8 * (k / 4) + e];
                s[e] = !diag || row0 + (e & 3) >= kmin ? nx : s[e];
            }
        }
    };
#pragma unroll
    for (int w = 0; w < NB - 1; w++) load(w);
#pragma unroll 1
    for (int t = 0; t < tmax; t += 8 * NB) {
#pragma unroll
        for (int w = 0; w < NB; w++) {
            const int tw = t + 8 * w;
            if (tw < tmax) {  // uniform
                load((w + NB - 1) % NB);
                if (tw + 8 <= tall) group(w, tw, false);
                else group(w, tw, true);
            }
        }
    }
    if (!xc) {
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (row0 + e < np && c0 + 16 * b + (l & 15) < HD)
                    out[((size_t)(p0 + row0 + e) * n_heads + h) * HD + c0 + 16 * b + (l & 15)] = s[4 * b + e];
        return;
    }
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int e = 0; e < 4; e++) tile[wave][row0 + e][16 * b + (l & 15)] = s[4 * b + e];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // within the wave: LDS operations stay in order
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < 2; r++) {  // 8 lanes per token, 4 values each: one block of 32
        const int kk = 8 * r + (l >> 3);
        const pf_v4f x = *(const pf_v4f *)&tile[wave][kk][4 * (l & 7)];
        const float v4[4] = {x[0], x[1], x[2], x[3]};
        pf_quant_block(v4, h * (HD / 32) + c0 / 32, kk < np ? 0x7fffffff : 0, p0 + kk, l & 7, xc, xd, PP, perm8);
    }
}

extern "C" int qmh_launch_pf_attention(const float *Q, const float *Kt, const float *V, float *att, float *out, int P,
                                       int pos0, int n_heads, int n_kv, int hd, int max_seq, float scale, int8_t *xc,
                                       float *xd, int PP, int perm8, void *stream) {
    if (hd > 128 || hd % 4 || pos0 + P > max_seq || P < 1) return (int)hipErrorInvalidValue;
    // the output's quantized image: from k_pf_pv_m (head_dim 128 or 64: whole blocks), or from out after k_pf_pv
    if (xc && (!xd || (hd != 128 && hd != 64) || P > PP)) return (int)hipErrorInvalidValue;
    hipStream_t s = (hipStream_t)stream;
    const int ng = (P + QMH_PF_TOK - 1) / QMH_PF_TOK, nz = (pos0 + P + QMH_WG - 1) / QMH_WG;
    const int rlen = pos0 + P;  // the longest row
    const dim3 wg(QMH_WG);
    // head_dim 48, 64, 128: products from MFMAs (a layer's V, with the sets loaded past it, within 32-bit
    // offsets; queries read as float4s)
    const bool mf = (hd == 128 || hd == 64 || hd == 48) && (uint64_t)(max_seq + 64ull) * hd * n_kv * 4 < 1ull << 32 &&
                    ((uintptr_t)Q & 15) == 0;
#define PF_HD(K_, G_, ...)                                                         \
    do {                                                                           \
        if (hd == 128) hipLaunchKernelGGL(K_<128>, G_, wg, 0, s, __VA_ARGS__);     \
        else if (hd == 64) hipLaunchKernelGGL(K_<64>, G_, wg, 0, s, __VA_ARGS__);  \
        else hipLaunchKernelGGL(K_<48>, G_, wg, 0, s, __VA_ARGS__);                \
    } while (0)
    if (mf)
        PF_HD(k_pf_scores_m, dim3(n_heads, (P + 63) / 64, (rlen + 63) / 64), Q, Kt, att, P, pos0, n_heads, n_kv,
              max_seq, scale);
    else
        hipLaunchKernelGGL(k_pf_scores, dim3(n_heads, ng, nz), wg, 0, s, Q, Kt, att, P, pos0, n_heads, n_kv, hd,
                           max_seq, scale);
    // one wave per row up to 512 positions, four beyond, the fewest rounds that hold the longest row
    const dim3 g1(n_heads, (P + 3) / 4), g4(n_heads, P);
#define PF_SM(R_, W_, G_) hipLaunchKernelGGL((k_pf_softmax_r<R_, W_>), G_, wg, 0, s, att, P, pos0, max_seq)
    if (rlen <= 64 * 2) PF_SM(2, 1, g1);
    else if (rlen <= 64 * 4) PF_SM(4, 1, g1);
    else if (rlen <= 64 * 8) PF_SM(8, 1, g1);
    else if (rlen <= 256 * 4) PF_SM(4, 4, g4);
    else if (rlen <= 256 * 8) PF_SM(8, 4, g4);
    else if (rlen <= 256 * 16) PF_SM(16, 4, g4);
    else hipLaunchKernelGGL(k_pf_softmax, g1, wg, 0, s, att, P, pos0, max_seq);
#undef PF_SM
    if (mf)
        PF_HD(k_pf_pv_m, dim3(n_heads, hd == 128 ? (P + 15) / 16 : (P + 31) / 32), att, V, out, P, pos0, n_heads, n_kv, max_seq,
              xc, xd, PP, perm8);
    else
        hipLaunchKernelGGL(k_pf_pv, dim3(n_heads, ng), wg, 0, s, att, V, out, P, pos0, n_heads, n_kv, hd, max_seq);
#undef PF_HD
    const int rc = (int)hipGetLastError();
    if (rc || !xc || mf) return rc;
    return qmh_launch_pf_quant(out, n_heads * hd, nullptr, 0.0f, n_heads * hd, P, xc, xd, PP, perm8, stream);
}
