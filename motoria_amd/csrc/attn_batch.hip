// The scores, softmax and mix of a prompt batch (head_dim 128): src/model/
// forward.c:141-163 of the reference for n tokens at positions pos .. pos +
// n - 1, every value in the reference's order (each score one sequential
// fp32 dot, the softmax's sum and the mix sequential over positions, every
// product rounded before its addition).
//
// The work is two triangular products, S = Q K^T and O = P V, over the rows
// (token, head of the key/value group): a group's heads share each key and
// value row, so a tile of rows is group x tokens. A row's sum runs over its
// 128 elements (positions) in order, and the rounded product and the rounded
// addition of a term are two operations of the vector ALUs' rate either way,
// so what there is to gain is everything else: each operand read must feed
// many terms, and every SIMD must hold several wavefronts (a wavefront alone
// issues a vector operation every ~4.3 cycles, several together one every
// ~2.1; measured). The products come from the matrix cores, as outer
// products with K = 1 and C = 0 (v_mfma_f32_16x16x1_4b_f32: 1024 products,
// each rounded once, subnormals kept; checked against the vector product
// over all exponents), the additions from the vector ALUs: 36 T terms/s, the
// rate of multiply + add on the vector ALUs (the two kinds of instruction do
// not overlap on a SIMD), for two operand registers per 1024 terms instead of
// a register per 8 terms, which leaves room for 4-6 wavefronts per SIMD.
// (A product -0 is added to a sum that started at +0 and so is never -0.)
// Measured, 777 tokens at position 1200, 32/4 heads of 128 (10.1 G terms,
// 280 us at that rate): scores 238, max and sum 49, mix 315 us, against 1260
// for a workgroup per (key/value head, token); fewer workgroups per CU are
// slower (mix 309 us with four, 331 with three, 357 with two).
#include "mhip_internal.h"

namespace {

constexpr int HD = 128;
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // of a caller's cache rows
typedef float f16v __attribute__((ext_vector_type(16)));

// acc += p; gives `next` back for a product that then does not start before
// it (left free, the compiler starts every product of a loop's body at once,
// 16 registers each).
__device__ __forceinline__ float add(f16v &acc, const f16v &p, float next) {
    acc = acc + p;
    asm volatile("" : "+v"(acc), "+v"(next));
    return next;
}

__device__ __forceinline__ f16v outer(float a, float b) {
    const f16v z = {0.0f};
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, z, 0, 0, 0);
}

// A tile's place: the blocks of an XCD (blockIdx.x % 8) work on one key/value
// group where the groups divide the XCDs (or the XCDs the groups), so that
// XCD's L2 holds that group's cache rows only.
constexpr int NXCD = 8;
struct Tiles {
    int nkv, nrt;  // groups, row tiles per group
    __host__ __device__ int blocks() const {
        if (NXCD % nkv == 0) {
            const int sub = NXCD / nkv;
            return NXCD * ((nrt + sub - 1) / sub);
        }
        return nkv * nrt;
    }
    __device__ bool place(int b, int *g, int *rt) const {
        if (NXCD % nkv == 0) {
            const int sub = NXCD / nkv, x = b % NXCD;
            *g = x / sub;
            *rt = (b / NXCD) * sub + x % sub;
            return *rt < nrt;
        }
        *g = b % nkv;
        *rt = b / nkv;
        return true;
    }
};

// The maximum over each 16 lanes, in every one of them (row rotations).
template <int CTRL>
__device__ __forceinline__ float ror_max(float v) {
    const int b = __float_as_int(v);
    return fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, false)));
}
__device__ __forceinline__ float max16(float v) {
    return ror_max<0x121>(ror_max<0x122>(ror_max<0x124>(ror_max<0x128>(v))));
}

// Scores of SR rows x SU positions per workgroup, a 32 x 32 tile per
// wavefront (blocks of 16 rows x 16 positions); the operands in LDS SI
// elements at a time (row stride SI + 4 floats: the 16 rows a block reads 16
// bytes of lie on distinct banks). S[(t * nh + h) * sld + u], and the
// largest score of each 32 positions of a row in pmax (stride pld).
constexpr int SR = 64, SU = 64, SI = 64, SLD = SI + 4;

__global__ __launch_bounds__(256, 4) void k_ab_scores(const float *__restrict__ q,
                                                      const float *__restrict__ kc, Tiles tl,
                                                      int pos, int n, int nh, int group, int kvd,
                                                      float scale, float *__restrict__ S, int sld,
                                                      float *__restrict__ pmax, int pld) {
    __shared__ __align__(16) float qs[SR * SLD], ks[SU * SLD];
    __shared__ int rid[SR], rlim[SR];  // of the tile's rows: S row from the tile's token on, last position
    int g, rt;
    if (!tl.place(blockIdx.x, &g, &rt)) return;
    const int rows = n * group, r0 = rt * SR, u0 = blockIdx.y * SU;
    const int rlast = min(r0 + SR, rows) - 1;
    if (u0 > pos + rlast / group) return;  // no row of the tile reads these positions
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c16 = lane & 15, blk = lane >> 4;
    const int wr = 32 * (wave >> 1), wc = 32 * (wave & 1);
    // staging: thread -> (row tid / 16 + 16 k, 16 bytes tid % 16)
    const int s4 = tid & 15, t0 = r0 / group, un = pos + n - 1 - u0;
    const float *qb = q + ((size_t)t0 * nh + (size_t)g * group) * HD;
    const float *kb = kc + (size_t)u0 * kvd + (size_t)g * HD;
    unsigned qp[4], kp[4];  // in floats, from the tile's first row
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int r = min(r0 + (tid >> 4) + 16 * k, rlast);
        const int t = r / group, hh = r - t * group;
        qp[k] = (unsigned)(((t - t0) * nh + hh) * HD + 4 * s4);
        kp[k] = (unsigned)(min((tid >> 4) + 16 * k, un) * kvd + 4 * s4);
    }
    if (tid < SR) {
        const int t = (r0 + tid) / group, hh = r0 + tid - t * group;
        rid[tid] = (t - t0) * nh + hh;
        rlim[tid] = r0 + tid < rows ? pos + t - u0 : -1;
    }
    f4v qv[4], kv[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        qv[k] = *(const f4v *)(qb + qp[k]);
        kv[k] = *(const f4u *)(kb + kp[k]);
    }
    f16v acc = {0.0f};
    const f4v *A = (const f4v *)&qs[(wr + 16 * (blk >> 1) + c16) * SLD];
    const f4v *B = (const f4v *)&ks[(wc + 16 * (blk & 1) + c16) * SLD];
#pragma unroll 1
    for (int i0 = 0; i0 < HD; i0 += SI) {
        if (i0) __syncthreads();
#pragma unroll
        for (int k = 0; k < 4; k++) {
            *(f4v *)&qs[((tid >> 4) + 16 * k) * SLD + 4 * s4] = qv[k];
            *(f4v *)&ks[((tid >> 4) + 16 * k) * SLD + 4 * s4] = kv[k];
        }
        __syncthreads();
        if (i0 + SI < HD) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                qv[k] = *(const f4v *)(qb + i0 + SI + qp[k]);
                kv[k] = *(const f4u *)(kb + i0 + SI + kp[k]);
            }
        }
        // the products of a term are formed while the previous term's are added
        f4v a = A[0], b = B[0];
        f16v p = outer(a.x, b.x);
#pragma unroll 1
        for (int i = 1; i <= SI / 4; i++) {
            const int j = i < SI / 4 ? i : 0;  // (the last round's operands are not used)
            const f4v an = A[j], bn = B[j];
            f16v p1 = outer(a.y, b.y);
            a.z = add(acc, p, a.z);
            p = outer(a.z, b.z);
            a.w = add(acc, p1, a.w);
            p1 = outer(a.w, b.w);
            a = an;
            b = bn;
            a.x = add(acc, p, a.x);
            if (i < SI / 4) p = outer(a.x, b.x);
            a.y = add(acc, p1, a.y);
        }
    }
    // lane: positions wc + 16 (q & 1) + c16, rows wr + 16 (q >> 1) + 4 blk + r
    const size_t Rt = (size_t)t0 * nh + (size_t)g * group;
    float *St = S + Rt * sld + u0;
    float *pm = pmax + Rt * pld + (u0 + wc) / 32;
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = wr + 16 * rb + 4 * blk + r, last = rlim[row];
            float *Sr = St + (size_t)rid[row] * sld;
            float mx = -__builtin_inff();
#pragma unroll
            for (int cb = 0; cb < 2; cb++) {
                const int u = wc + 16 * cb + c16;
                const float s = acc[4 * (2 * rb + cb) + r] * scale;
                if (u <= last) {
                    Sr[u] = s;
                    mx = fmaxf(mx, s);  // (keeps the larger of a number and a NaN)
                }
            }
            mx = max16(mx);
            if (c16 == 0 && wc <= last) pm[(size_t)rid[row] * pld] = mx;
        }
}

// The softmax's maximum and sequential sum of MR rows per workgroup: the
// maximum from k_ab_scores' parts, the exponentials formed MU positions at a
// time by wavefronts 0-3 into one of two LDS buffers while lanes 0 .. MR - 1
// of wavefront 4 add the other one's in position order (positions past the
// row's end as +0, which leaves the sum as it is). stat[R] = (max, sum).
constexpr int MR = 16, MU = 128, MLD = MU + 4;

__global__ __launch_bounds__(320) void k_ab_stat(const float *__restrict__ S, int sld,
                                                 const float *__restrict__ pmax, int pld, int pos,
                                                 int nrows, int nh, float2 *__restrict__ stat) {
    __shared__ __align__(16) float eb[2][MR * MLD];
    __shared__ float mxs[MR];
    __shared__ uint64_t etab[32];
    const int tid = threadIdx.x, R0 = blockIdx.x * MR;
    if (tid < 32) etab[tid] = mia_expf_tab[tid];
    const bool prod = tid < 256;
    const int row = prod ? tid >> 4 : tid & 15, c = tid & 15;
    const int R = min(R0 + row, nrows - 1), np = pos + R / nh + 1;
    const int npw = pos + (min(R0 + MR, nrows) - 1) / nh + 1;  // the longest row
    if (prod) {
        float mx = -__builtin_inff();
        for (int k = c; 32 * k < np; k += 16) mx = fmaxf(mx, pmax[(size_t)R * pld + k]);
        mx = max16(mx);
        if (c == 0) mxs[row] = mx;
    }
    __syncthreads();
    const float mx = mxs[row];
    const float *s = S + (size_t)R * sld;
    float sum = 0.0f;
    f4v nx[2];
    auto fetch = [&](int u0) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int u = u0 + 64 * k + 4 * c;
            nx[k] = u < np ? *(const f4v *)(s + u) : (f4v){0, 0, 0, 0};
        }
    };
    if (prod) fetch(0);
    int b = 0;
    for (int u0 = 0; u0 < npw + MU; u0 += MU, b ^= 1) {
        if (prod) {
            if (u0 < npw) {
                f4v v[2] = {nx[0], nx[1]};
                if (u0 + MU < npw) fetch(u0 + MU);
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const int u = u0 + 64 * k + 4 * c;
                    f4v e;
                    e.x = u < np ? mia_expf_glibc_tab(v[k].x - mx, etab) : 0.0f;
                    e.y = u + 1 < np ? mia_expf_glibc_tab(v[k].y - mx, etab) : 0.0f;
                    e.z = u + 2 < np ? mia_expf_glibc_tab(v[k].z - mx, etab) : 0.0f;
                    e.w = u + 3 < np ? mia_expf_glibc_tab(v[k].w - mx, etab) : 0.0f;
                    *(f4v *)&eb[b][row * MLD + 64 * k + 4 * c] = e;
                }
            }
        } else if (u0 && tid < 256 + MR) {
            const f4v *e4 = (const f4v *)&eb[b ^ 1][row * MLD];
#pragma unroll 2
            for (int k = 0; k < MU / 4; k += 4) {
                f4v e[4];
#pragma unroll
                for (int j = 0; j < 4; j++) e[j] = e4[k + j];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    sum = sum + e[j].x;
                    sum = sum + e[j].y;
                    sum = sum + e[j].z;
                    sum = sum + e[j].w;
                }
            }
        }
        __syncthreads();
    }
    if (!prod && tid < 256 + MR && R0 + row < nrows) stat[R0 + row] = make_float2(mx, sum);
}

// The mix of XR rows per workgroup, 32 rows x 32 elements per wavefront
// (blocks of 16 x 16): the rows' probabilities (the exponential again, over
// the sum) and the value rows staged in LDS XU positions at a time, the next
// ones requested ahead; then Q8 of each row's 32 values (a wavefront's 32
// elements are one block, quant.c:11-27): codes as int8 (attq) and scales
// [t][nh * 4], or (atth) as the row kernels read them: fp16 integers in
// fragments of 16 tokens from token tb on, scales [nh * 4][ld]. A position that only some rows of
// the tile read (the batch's own tokens) is added to those alone.
constexpr int XR = 32, XU = 32, XLD = XU + 4;

__global__ __launch_bounds__(256, 4) void k_ab_mix(const float *__restrict__ S, int sld,
                                                   const float2 *__restrict__ stat,
                                                   const float *__restrict__ vc, Tiles tl, int pos,
                                                   int n, int nh, int group, int kvd,
                                                   int8_t *__restrict__ attq,
                                                   _Float16 *__restrict__ atth,
                                                   float *__restrict__ atts, int tb, int ld) {
    __shared__ __align__(16) float ps[XR * XLD], vs[XU * HD];
    __shared__ uint64_t etab[32];
    int g, rt;
    // (the tiles of the last tokens, the longest, first)
    if (!tl.place(tl.blocks() - 1 - (int)blockIdx.x, &g, &rt)) return;
    const int rows = n * group, r0 = rt * XR, rlast = min(r0 + XR, rows) - 1;
    const int nfull = pos + r0 / group + 1, np = pos + rlast / group + 1;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c16 = lane & 15, blk = lane >> 4;
    if (tid < 32) etab[tid] = mia_expf_tab[tid];
    // staging: probabilities of row tid / 8, four positions; four 16-byte
    // pieces of the value rows
    const int prow = min(r0 + (tid >> 3), rlast), pt = prow / group;
    const size_t PR = (size_t)pt * nh + (size_t)g * group + (prow - pt * group);
    const float2 st = stat[PR];
    const float *sp = S + PR * sld + 4 * (tid & 7);
    const float *vp = vc + (size_t)g * HD + 4 * (tid & 31);
    f4v sv, vv[4];
    auto fetch = [&](int u0) {
        const int u = u0 + 4 * (tid & 7);
        sv = u < np ? *(const f4v *)(sp + u0) : (f4v){0, 0, 0, 0};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int w = min(u0 + (tid >> 5) + 8 * k, np - 1);  // (past the end: not used)
            vv[k] = *(const f4u *)(vp + (size_t)w * kvd);
        }
    };
    fetch(0);
    f16v acc = {0.0f};
    const float *A = &ps[(16 * (blk >> 1) + c16) * XLD];
    const float *B = &vs[32 * wave + 16 * (blk & 1) + c16];
#pragma unroll 1
    for (int u0 = 0; u0 < np; u0 += XU) {
        __syncthreads();
        {
            f4v p;
            p.x = mia_expf_glibc_tab(sv.x - st.x, etab) / st.y;
            p.y = mia_expf_glibc_tab(sv.y - st.x, etab) / st.y;
            p.z = mia_expf_glibc_tab(sv.z - st.x, etab) / st.y;
            p.w = mia_expf_glibc_tab(sv.w - st.x, etab) / st.y;
            *(f4v *)&ps[(tid >> 3) * XLD + 4 * (tid & 7)] = p;
#pragma unroll
            for (int k = 0; k < 4; k++)
                *(f4v *)&vs[((tid >> 5) + 8 * k) * HD + 4 * (tid & 31)] = vv[k];
        }
        __syncthreads();
        if (u0 + XU < np) fetch(u0 + XU);
        if (u0 + XU <= nfull) {
            f4v a = *(const f4v *)A;
            f16v p = outer(a.x, B[0]);
#pragma unroll 1
            for (int u = 0; u < XU; u += 4) {
                const f4v an = *(const f4v *)(A + ((u + 4) & (XU - 1)));
                f16v p1 = outer(a.y, B[(u + 1) * HD]);
                a.z = add(acc, p, a.z);
                p = outer(a.z, B[(u + 2) * HD]);
                a.w = add(acc, p1, a.w);
                p1 = outer(a.w, B[(u + 3) * HD]);
                a = an;
                a.x = add(acc, p, a.x);
                if (u + 4 < XU) p = outer(a.x, B[(u + 4) * HD]);
                a.y = add(acc, p1, a.y);
            }
        } else {
            const int ue = min(XU, np - u0);
            for (int u = 0; u < ue; u++) {
                const f16v p = outer(A[u], B[u * HD]);
#pragma unroll
                for (int k = 0; k < 16; k++) {
                    const int row = r0 + 16 * (k >> 3) + 4 * blk + (k & 3);
                    if (u0 + u <= pos + row / group) acc[k] = acc[k] + p[k];
                }
            }
        }
    }
    // element 32 wave + 16 (q & 1) + c16 of rows 16 (q >> 1) + 4 blk + r
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = r0 + 16 * rb + 4 * blk + r;
            const float o0 = acc[8 * rb + r], o1 = acc[8 * rb + 4 + r];
            const float am = max16(fmaxf(fmaxf(0.0f, fabsf(o0)), fabsf(o1)));  // a NaN counts as 0
            const float d = am / 127.0f;
            const float qi = d != 0.0f ? 1.0f / d : 0.0f;
            if (row >= rows) continue;
            const int t = row / group, h = g * group + (row - t * group);
            const int8_t q0 = (int8_t)roundf(o0 * qi), q1 = (int8_t)roundf(o1 * qi);
            const int ob = h * (HD / 32) + wave;  // the block of the output row
            if (atth) {
                // codes 8 c .. + 7 of token t at lane 16 c + t % 16
                _Float16 *f = atth + ((size_t)((tb + t) / 16) * (nh * (HD / 32)) + ob) * 512 +
                              (c16 / 8) * 128 + ((tb + t) % 16) * 8 + c16 % 8;
                f[0] = (_Float16)q0;
                f[256] = (_Float16)q1;
                if (c16 == 0) atts[(size_t)ob * ld + tb + t] = d;
            } else {
                const size_t o = ((size_t)(tb + t) * nh + h) * HD + 32 * wave + c16;
                attq[o] = q0;
                attq[o + 16] = q1;
                if (c16 == 0) atts[(size_t)(tb + t) * nh * (HD / 32) + ob] = d;
            }
        }
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }
int part_ld(int sld) { return (sld + 31) / 32; }
size_t token_bytes(int nh, int sld) {  // scores, maxima and (max, sum) of a token's rows
    return (size_t)nh * (sld + part_ld(sld) + 2) * 4;
}
// The score matrix of a pass is kept under this size (and held whole by the
// memory-side cache when it is much smaller); 64 tokens' at least.
constexpr size_t PASS_BYTES = 512u << 20;
constexpr int PASS_MIN = 64;

}  // namespace

namespace mhip {

size_t attn_batch_scratch(int nh, int n, int max_seq) {
    const size_t tb = token_bytes(nh, (max_seq + 3) & ~3), want = tb * (size_t)n;
    const size_t floor = tb * (size_t)(n < PASS_MIN ? n : PASS_MIN);
    return align256(want < PASS_BYTES ? want : floor > PASS_BYTES ? floor : PASS_BYTES) + 3 * 256;
}

void launch_attn_batch(hipStream_t st, const float *q, const float *kc, const float *vc, int pos,
                       int n, int nh, int nkv, float scale, void *scratch, size_t bytes,
                       int8_t *attq, _Float16 *atth, float *atts, int ld) {
    const int group = nh / nkv, kvd = nkv * HD, qd = nh * HD;
    const int sld = (pos + n + 3) & ~3, pld = part_ld(sld);
    const size_t fit = (bytes - 3 * 256) / token_bytes(nh, sld);
    // passes of equal size
    const int np = fit < (size_t)n ? (int)((n + fit - 1) / fit) : 1, pass = (n + np - 1) / np;
    float *S = (float *)scratch;
    float *pmax = (float *)((uint8_t *)S + align256((size_t)pass * nh * sld * 4));
    float2 *stat = (float2 *)((uint8_t *)pmax + align256((size_t)pass * nh * pld * 4));
    for (int t0 = 0; t0 < n; t0 += pass) {
        const int ns = n - t0 < pass ? n - t0 : pass, p0 = pos + t0;
        const Tiles ts = {nkv, (ns * group + SR - 1) / SR}, tx = {nkv, (ns * group + XR - 1) / XR};
        k_ab_scores<<<dim3((unsigned)ts.blocks(), (unsigned)((p0 + ns + SU - 1) / SU)), 256, 0, st>>>(
            q + (size_t)t0 * qd, kc, ts, p0, ns, nh, group, kvd, scale, S, sld, pmax, pld);
        k_ab_stat<<<blocks_for((size_t)ns * nh, MR), 320, 0, st>>>(S, sld, pmax, pld, p0, ns * nh,
                                                                   nh, stat);
        k_ab_mix<<<(unsigned)tx.blocks(), 256, 0, st>>>(
            S, sld, stat, vc, tx, p0, ns, nh, group, kvd, attq, atth, atts, t0, ld);
    }
}

}  // namespace mhip
