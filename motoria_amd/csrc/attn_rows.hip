// The Q/K/V and O rows of a prompt batch on the matrix cores
// (src/tensor/matmul.c:19-28 of the reference for n tokens):
// v_mfma_f32_16x16x32_f16 over one 32-code block multiplies Q8 codes held as
// fp16 integers and gives the exact int32 block dot (32 products below 2^14
// each, every partial sum an integer below 2^24), so the block term
// ((float)dot * d_w) * d_x and the sum in block order are the reference's.
//
// Both operands lie in memory as the fragments the instruction takes: for 16
// rows (tokens) and one block, 64 lanes x 8 codes, lane l holding codes
// 8 (l / 16) .. + 7 of row l % 16: 1 KB that a wavefront copies into LDS with
// one instruction and reads back conflict-free without a swizzle. The weights
// are repacked so once (mhip_attention_pack), the tokens' codes by the kernel
// that makes them; the scales of both are block-major.
//
// A workgroup takes 64 weight rows x 32 NJ tokens, a wavefront half of each
// (2 x NJ tiles of 16 x 16), one block per step of an RS-stage LDS ring
// filled RS - 1 steps ahead. What bounds it is the vector ALUs: twelve
// operations per matrix instruction, beside which the matrix cores run for
// about 40 % of their time; the small tiles buy four wavefronts per SIMD, and
// one wavefront alone issues a vector operation at half the rate of several.
// Measured at 777 tokens (QKV 5120 x 2048, O 2048 x 4096): 51 us a launch,
// against 145-160 us for operands in registers one block ahead (about 17 us is
// what the products and their terms take).
#include "attn_common.h"
#include "mhip_internal.h"

namespace {

using mhip_attn::dma16;
using mhip_attn::dma4;
using mhip_attn::wait_vm;

constexpr int QK = mhip::QK;
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // of a caller's x

constexpr int RM_R = 64;  // weight rows of a workgroup
constexpr int FRAG = 16 * QK;  // codes of a fragment
constexpr int RS = 4;          // ring stages (3, 5, 6 and 8 measured 1-3% slower)

// Row r of a .mia Q8_0 matrix (36-byte blocks) into fragments [R / 16][nb]
// and block-major scales [nb][R], one thread per block.
__global__ __launch_bounds__(256) void k_pack_rows(const uint8_t *__restrict__ w, int R, int nb,
                                                   _Float16 *__restrict__ qh,
                                                   float *__restrict__ sc) {
    const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= (size_t)R * nb) return;
    const int r = (int)(q / nb), b = (int)(q % nb);
    const uint8_t *blk = w + q * 36;
    sc[(size_t)b * R + r] = *(const float *)blk;
    const int8_t *c = (const int8_t *)(blk + 4);
    _Float16 *o = qh + ((size_t)(r / 16) * nb + b) * FRAG + (r % 16) * 8;
#pragma unroll
    for (int i = 0; i < QK; i++) o[(i / 8) * 128 + i % 8] = (_Float16)c[i];
}

// The tokens' Q8 codes [n][nb * 32] and scales [n][nb] as fragments
// [n / 16][nb] and block-major scales [nb][ld], a thread per 8 codes: the 16
// tokens of a tile on 16 consecutive lanes, so a wavefront writes a whole
// fragment at a time.
__global__ __launch_bounds__(256) void k_token_frags(const int8_t *__restrict__ q,
                                                     const float *__restrict__ s, int n, int nb,
                                                     int ld, _Float16 *__restrict__ o,
                                                     float *__restrict__ os) {
    const int lane = threadIdx.x & 63, b = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int t = blockIdx.x * 16 + (lane & 15), c = lane >> 4;
    if (b >= nb || t >= n) return;
    const int2 v = *(const int2 *)(q + ((size_t)t * nb + b) * QK + 8 * c);
    h8 h;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        h[i] = (_Float16)(int8_t)(v.x >> (8 * i));
        h[4 + i] = (_Float16)(int8_t)(v.y >> (8 * i));
    }
    *(h8 *)(o + ((size_t)blockIdx.x * nb + b) * FRAG + 8 * lane) = h;
    if (c == 0) os[(size_t)b * ld + t] = s[(size_t)t * nb + b];
}

struct RowPack {
    const _Float16 *q[3];  // fragments of segment k
    const float *s[3];     // its block-major scales
    float *out[3];
    int r0[4];             // rows of segment k: [r0[k], r0[k+1]), multiples of RM_R
};

template <int NJ> struct alignas(16) Step {
    _Float16 w[RM_R / 16][FRAG];  // 4 KB
    _Float16 x[2 * NJ][FRAG];     // 2 NJ KB
    float sw[RM_R];
    float sx[64];  // (NJ = 1: the 32 scales twice)
};

// out[k][t * ld_k + r] = (resid ? resid[t * ld_r + r] : 0) + the Q8 dot of row
// r of segment k with token t. xs: block-major, ld floats a block.
template <int NJ>
__global__ __launch_bounds__(256, 4) void k_rows_mfma(RowPack sg, int nb, int n,
                                                      const _Float16 *__restrict__ xh,
                                                      const float *__restrict__ xs, int ld,
                                                      const float *resid, int ld_r) {
    __shared__ Step<NJ> ring[RS];
    const int lane = threadIdx.x & 63, l16 = lane & 15, c = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = blockIdx.x * RM_R;
    const int k = row0 >= sg.r0[1] ? (row0 >= sg.r0[2] ? 2 : 1) : 0;
    const int rl0 = row0 - sg.r0[k], R = sg.r0[k + 1] - sg.r0[k];
    const int t0 = blockIdx.y * 32 * NJ;
    // this wavefront's share of a step: weight fragment `wave`, a token
    // fragment and 64 scales (wavefront 0 the weights', the others the tokens')
    constexpr int NLOAD = 3;
    const _Float16 *wsrc = sg.q[k] + (size_t)(rl0 / 16 + wave) * nb * FRAG + 8 * lane;
    const int xf = wave % (2 * NJ);
    const _Float16 *xsrc = xh + (size_t)(t0 / 16 + xf) * nb * FRAG + 8 * lane;
    const float *ssrc = wave == 0 ? sg.s[k] + rl0 + lane : xs + t0 + lane % (32 * NJ);
    const int sstep = wave == 0 ? R : ld;
    const unsigned ring0 = (unsigned)(uintptr_t)&ring[0];
    const unsigned so = wave == 0 ? (unsigned)offsetof(Step<NJ>, sw)
                                  : (unsigned)offsetof(Step<NJ>, sx);
    auto issue = [&](int b) {
        const int bb = min(b, nb - 1);  // past the end: the last block again
        const unsigned st = ring0 + (unsigned)((b % RS) * sizeof(Step<NJ>));
        dma16(st + wave * 1024, wsrc + (size_t)bb * FRAG);
        dma16(st + (unsigned)offsetof(Step<NJ>, x) + xf * 1024, xsrc + (size_t)bb * FRAG);
        dma4(st + so, ssrc + (size_t)bb * sstep);
    };
    const int wr = 2 * (wave >> 1), wt = NJ * (wave & 1);  // first fragments of the wavefront
    f4v acc[2][NJ];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) acc[i][j] = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < RS - 1; s++) issue(s);
    for (int b = 0; b < nb; b++) {
        wait_vm<(RS - 2) * NLOAD>();  // this wavefront's part of step b is in LDS ...
        __syncthreads();              // ... and every other's; step b - 1 is read
        issue(b + RS - 1);
        const Step<NJ> &S = ring[b % RS];
        h8 a[2], x[NJ];
        f4v dw[2];
        float dx[NJ];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            a[i] = *(const h8 *)&S.w[wr + i][8 * lane];
            dw[i] = *(const f4v *)&S.sw[16 * (wr + i) + 4 * c];
        }
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            x[j] = *(const h8 *)&S.x[wt + j][8 * lane];
            dx[j] = S.sx[16 * (wt + j) + l16];
        }
        const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const f4v blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], x[j], z, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float t = blk[r] * dw[i][r];
                    acc[i][j][r] = acc[i][j][r] + t * dx[j];  // (no contraction)
                }
            }
    }
    wait_vm<0>();  // the copies past the end
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int t = t0 + 16 * (wt + j) + l16;
        if (t < n) {
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int row = rl0 + 16 * (wr + i) + 4 * c;
                f4v v = acc[i][j];
                if (resid) v = *(const f4u *)(resid + (size_t)t * ld_r + row) + v;
                *(f4u *)(sg.out[k] + (size_t)t * R + row) = v;
            }
        }
    }
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// The packed weights of one layer (mhip_attention_pack): the fragments of Q,
// K, V and O, then their block-major scales, each 256-byte aligned.
struct AttnPack {
    _Float16 *q[4];
    float *s[4];
};
AttnPack pack_carve(const mhip_attn_dims *s, const void *base) {
    const size_t d = s->dim, qd = (size_t)s->n_heads * s->head_dim,
                 kvd = (size_t)s->n_kv_heads * s->head_dim;
    const size_t rows[4] = {qd, kvd, kvd, d}, cols[4] = {d, d, d, qd};
    AttnPack a;
    uint8_t *p = (uint8_t *)base;
    for (int m = 0; m < 4; m++) {
        a.q[m] = (_Float16 *)p;
        p += align256(rows[m] * cols[m] * 2);
    }
    for (int m = 0; m < 4; m++) {
        a.s[m] = (float *)p;
        p += align256(rows[m] * (cols[m] / QK) * 4);
    }
    return a;
}

// Tokens per workgroup: 32 while that leaves workgroups for the chip's CUs,
// 64 from RN2 tokens on, where each token fragment then feeds twice the
// products. A layer's call at 32/4 heads and position 0, us, 32 / 64: 16
// tokens 81/90, 200 119/126, 400 171/175, 550 222/219, 1024 402/384 (128
// tokens a workgroup: 117 at 16, 201 at 400, 406 at 1024).
constexpr int RN2 = 512;

template <int NJ>
void launch(hipStream_t st, const RowPack &g, int nb, int n, const _Float16 *xh, const float *xs,
            int ld, const float *resid, int ld_r) {
    k_rows_mfma<NJ><<<dim3((unsigned)(g.r0[3] / RM_R), (unsigned)((n + 32 * NJ - 1) / (32 * NJ))),
                      256, 0, st>>>(g, nb, n, xh, xs, ld, resid, ld_r);
}

void rows(hipStream_t st, const RowPack &g, int nb, int n, const _Float16 *xh, const float *xs,
          int ld, const float *resid, int ld_r) {
    if (n >= RN2) launch<2>(st, g, nb, n, xh, xs, ld, resid, ld_r);
    else launch<1>(st, g, nb, n, xh, xs, ld, resid, ld_r);
}

}  // namespace

namespace mhip {

bool rows_pack_fits(const mhip_attn_dims *s) {
    const int qd = s->n_heads * s->head_dim, kvd = s->n_kv_heads * s->head_dim;
    return qd % RM_R == 0 && kvd % RM_R == 0 && s->dim % RM_R == 0;
}

void rows_pack(hipStream_t st, const mhip_attn_dims *s, const void *const *w, void *pack) {
    const int d = s->dim, qd = s->n_heads * s->head_dim, kvd = s->n_kv_heads * s->head_dim;
    const AttnPack a = pack_carve(s, pack);
    const int rows[4] = {qd, kvd, kvd, d}, nbs[4] = {d / QK, d / QK, d / QK, qd / QK};
    for (int m = 0; m < 4; m++)
        k_pack_rows<<<blocks_for((size_t)rows[m] * nbs[m], 256), 256, 0, st>>>(
            (const uint8_t *)w[m], rows[m], nbs[m], a.q[m], a.s[m]);
}

void rows_token_frags(hipStream_t st, const int8_t *q, const float *s, int n, int nb, int ld,
                      _Float16 *o, float *os) {
    k_token_frags<<<dim3(blocks_for(n, 16), blocks_for(nb, 4)), 256, 0, st>>>(q, s, n, nb, ld, o, os);
}

void rows_qkv(hipStream_t st, const mhip_attn_dims *s, const void *pack, int n, const _Float16 *xh,
              const float *xs, int ld, float *q, float *k, float *v) {
    const AttnPack a = pack_carve(s, pack);
    const int qd = s->n_heads * s->head_dim, kvd = s->n_kv_heads * s->head_dim;
    rows(st, {{a.q[0], a.q[1], a.q[2]}, {a.s[0], a.s[1], a.s[2]}, {q, k, v}, {0, qd, qd + kvd, qd + 2 * kvd}},
         s->dim / QK, n, xh, xs, ld, nullptr, 0);
}

void rows_o(hipStream_t st, const mhip_attn_dims *s, const void *pack, int n, const _Float16 *xh,
            const float *xs, int ld, float *x) {
    const AttnPack a = pack_carve(s, pack);
    const int d = s->dim;
    rows(st, {{a.q[3], nullptr, nullptr}, {a.s[3], nullptr, nullptr}, {x, nullptr, nullptr}, {0, d, d, d}},
         s->n_heads * s->head_dim / QK, n, xh, xs, ld, x, d);
}

}  // namespace mhip
