// The token sampler on device logits: mia_sample of the reference
// (src/tokenizer/sampler.c:33-66) with the same picks.
//
//   greedy:  the first maximum (k_argmax_part / k_argmax_final; NaN never
//            wins except at index 0, as the reference's strict comparison)
//   else:    e_i = expf((l_i - l_best) / T)            (k_sample_exp)
//            sum = e_0 + e_1 + ... in index order       (k_sum_runs, k_sum_walk;
//                                                        k_chain_sum)
//            candidates p_i = e_i / sum >= cutoff as keys (descending
//            p) and indices, sorted stably              (k_sample_keys, rocPRIM)
//            the running sum of the sorted p up to top_p, r = u * cum, the
//            first candidate whose running sum exceeds r (k_sample_pick)
//
// The running sums are fp32 chains in a fixed order, as the reference adds
// them. They are computed exactly but not one addition at a time: while a
// running sum stays inside one binade every addition adds a whole number of
// that binade's ulps, so a workgroup turns 8192 additions at a time into an
// integer prefix sum and walks only the few additions that leave the binade
// (seq_scan). Everything else is parallel.
#include <rocprim/device/device_radix_sort.hpp>

#include "mhip_internal.h"

namespace {

constexpr int NT = 256;          // threads of every sampler kernel
constexpr int PARTS = 256;       // workgroups of the argmax's first pass
constexpr uint32_t NONE = ~0u;    // key of a dropped token

struct SampleState {
    int best;
    float sum;
    int walked;  // how the sum was taken: pieces that k_sum_walk noted, -1 by seq_scan alone
    int last;
    float cum;
};

struct Best {
    float v;
    int i;  // -1: no non-NaN value seen
};

// The better of two candidates from disjoint index ranges: the larger value,
// the lower index among equal values (+0 and -0 are equal).
__device__ __forceinline__ Best better(Best a, Best b) {
    if (b.i < 0) return a;
    if (a.i < 0) return b;
    if (b.v > a.v) return b;
    if (a.v > b.v) return a;
    return b.i < a.i ? b : a;
}

__device__ Best block_best(Best m, Best *sh) {
    const int tid = threadIdx.x;
    sh[tid] = m;
    __syncthreads();
    for (int o = NT / 2; o > 0; o >>= 1) {
        if (tid < o) sh[tid] = better(sh[tid], sh[tid + o]);
        __syncthreads();
    }
    return sh[0];
}

__global__ __launch_bounds__(NT) void k_argmax_part(const float *__restrict__ l, int n,
                                                    Best *__restrict__ part) {
    __shared__ Best sh[NT];
    Best m = {0.0f, -1};
    for (int i = blockIdx.x * NT + threadIdx.x; i < n; i += gridDim.x * NT) {
        const float v = l[i];
        if (v == v && (m.i < 0 || v > m.v)) m = {v, i};  // indices rise: ties keep the first
    }
    m = block_best(m, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// sampler.c:34-37: best = 0, replaced by every later index whose value is
// strictly larger. With l[0] NaN nothing is larger; otherwise that is the
// first maximum of the non-NaN values.
__global__ __launch_bounds__(NT) void k_argmax_final(const float *__restrict__ l,
                                                     const Best *__restrict__ part, int nparts,
                                                     SampleState *st, int *token) {
    __shared__ Best sh[NT];
    Best m = {0.0f, -1};
    for (int p = threadIdx.x; p < nparts; p += NT) m = better(m, part[p]);
    m = block_best(m, sh);
    if (threadIdx.x == 0) {
        const float l0 = l[0];
        const int best = (l0 != l0 || m.i < 0) ? 0 : m.i;
        st->best = best;
        if (token) *token = best;
    }
}

// The sum's pieces (k_sum_runs): a thread takes PIECE consecutive values, 64
// pieces make a group (a wavefront), RUN_T / 64 groups a workgroup.
constexpr int RUN_T = 256, PIECE = 8, RUN_W = RUN_T * PIECE;
// Sizes whose sum is taken so: from where it is faster (a whole draw, us, on
// one workgroup / so: 4096 95/65, 32768 152/83, 151936 236/131 with spread
// logits) up to where their groups fit the walk's workgroup, and the
// workgroups' sums the argmax's partial results.
constexpr int RUN_MIN_N = 2048, RUN_MAX_N = PARTS * RUN_W;

// sampler.c:41-44, the exponentials (the sum is k_sum_runs' and k_sum_walk's),
// and (bsum not null) each workgroup's sum of its RUN_W values in double.
__global__ __launch_bounds__(RUN_T) void k_sample_exp(const float *__restrict__ l, int n,
                                                      float temperature,
                                                      const SampleState *__restrict__ st,
                                                      float *__restrict__ e,
                                                      double *__restrict__ bsum) {
    __shared__ uint64_t etab[32];
    __shared__ double part[RUN_T / 64];
    const int tid = threadIdx.x;
    if (tid < 32) etab[tid] = mia_expf_tab[tid];
    __syncthreads();
    const float mx = l[st->best];
    const int i0 = blockIdx.x * RUN_W, i1 = min(n, i0 + RUN_W);
    double s = 0.0;
    for (int i = i0 + tid; i < i1; i += RUN_T) {
        const float v = mia_expf_glibc_tab((l[i] - mx) / temperature, etab);
        e[i] = v;
        s = s + (double)v;
    }
    if (!bsum) return;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s = s + __shfl_xor(s, o);
    if ((tid & 63) == 0) part[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
        double t = 0.0;
        for (int k = 0; k < RUN_T / 64; k++) t = t + part[k];
        bsum[blockIdx.x] = t;
    }
}

// ---- exact running sums, 8192 additions at a time -------------------------------
//
// The chains s_0 = 0, s_{k+1} = fl(s_k + v_k) over v_k >= 0 (sampler.c:43,
// 55, 64). Let s lie on the grid of spacing u = 2^(P-23) below 2^(P+1):
// the binade [2^P, 2^(P+1)) for P >= -126, together with the subnormals for
// P = -126 (spacing 2^-149 below 2^-125). Then s = M u with an integer
// M < 2^24, and while s + v stays below 2^(P+1) - u/2 the rounded sum is
// u (M + n) with n the integer nearest to v / u: every value of the grid
// below 2^(P+1) is representable, and only an exact half (a tie, broken
// towards an even M + n) makes the result depend on M. So as long as
// M + n_0 + ... + n_j <= 2^24 - 1 (and no v_j / u is a tie), the chain's
// values are u times an integer prefix sum. The workgroup holds a window
// of SQ_W values (SQ_V consecutive per thread), forms every n_j and their
// prefix sums, and finds the first element at which the chain leaves the
// binade, meets a tie or a value that is not a finite v >= 0, or makes
// the caller's predicate true; that one addition is done in fp32 by its
// thread, the grid is taken from the new s, and the window goes on after
// it, first over its next SQ_SHORT values only (exits come in bursts while
// the sum is small; a short pass costs the waves that hold those values),
// then over the rest. Ties, exits from a binade (at most one per binade the
// sum passes through) and the stop are the only additions done one at a
// time. The prefix sums are fp32 sums of whole numbers: exact below 2^24,
// and at least 2^24 when the exact sum is, which is all the test needs (an
// n too large for the binade is entered as 2^25). A chain that becomes
// infinite, NaN or negative finishes one addition at a time on one lane.
constexpr int SQ_T = 1024, SQ_V = 8, SQ_W = SQ_T * SQ_V, SQ_SHORT = 1024;
constexpr float SQ_TOP = 16777216.0f;  // 2^24: a mantissa at or above it left the binade
constexpr int SQ_PF = 2;               // windows loaded ahead
constexpr size_t SQ_LDS = (size_t)(SQ_PF + 1) * SQ_W * sizeof(float);  // the window ring

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
// 16 bytes from global memory straight into LDS at lds + 16 * lane.
__device__ __forceinline__ void sq_dma16(unsigned lds, const void *g) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(g)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
enum { SQ_SUM = 0, SQ_GE = 1, SQ_GT = 2 };

template <int MODE>
__device__ __forceinline__ bool sq_pred(float s, float thr) {
    return MODE == SQ_GE ? s >= thr : MODE == SQ_GT ? thr < s : false;
}

// The grid of s >= 0 finite: P with s = M 2^(P-23), M an integer < 2^24.
__device__ __forceinline__ int sq_grid(float s) {
    return s >= 0x1p-126f ? ilogbf(s) : -126;
}

// Runs the chain over v[0 .. n) (16-byte aligned) on a workgroup of SQ_T
// threads, every thread calling. Returns the index of the first element
// after whose addition MODE's predicate holds (n if none) and leaves in *s
// the chain's value after that addition (after all n if none).
template <int MODE>
__device__ int seq_scan(const float *__restrict__ v, int n, float thr, float *s_out) {
    __shared__ float wtot[2][SQ_T / 64];
    __shared__ int wstop[2][SQ_T / 64];
    __shared__ float s1_sh[2];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int P = -126;
    float M = 0.0f;       // s = M 2^(P-23) = 0
    int lo = 0;           // the chain has added v[0 .. lo)
    int it = 0;           // parity of the LDS buffers
    float s = 0.0f;
    int stop = n;
    bool seq = false;     // the chain left the finite non-negative values
    const int nw = (n + SQ_W - 1) / SQ_W;
    // Windows stream into an LDS ring of SQ_PF + 1 windows, SQ_PF ahead,
    // straight from global memory (thread t's values land where it reads
    // them: load q of a wavefront puts lane l's 16 bytes at 16 l); every
    // load is a whole 16-byte vector at an in-range index (the last one
    // reaches up to 3 values past n: callers pad to a multiple of 4), and
    // values past n are zeroed when a window is taken.
    extern __shared__ __align__(16) float sq_ring[];
    const unsigned ring = (unsigned)(uintptr_t)sq_ring;
    const int nl = n > 4 ? (n - 1) & ~3 : 0;
    auto issue = [&](int w) {
        const int i0 = w * SQ_W + SQ_V * tid;
        const unsigned st = ring + (unsigned)(((w % (SQ_PF + 1)) * SQ_W + SQ_V * 64 * wave) * 4);
#pragma unroll
        for (int q = 0; q < SQ_V / 4; q++)
            sq_dma16(st + (unsigned)(q * 64 * 16), v + min(i0 + 4 * q, nl));
    };
    if (n > 0) {
#pragma unroll
        for (int q = 0; q < SQ_PF; q++) issue(q);
    }
    bool short_pass = false;
    for (int w = 0; w < nw && stop == n && !seq; w++) {
        // this wavefront's loads of window w are in (later ones may not be)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SQ_PF - 1) * (SQ_V / 4)) : "memory");
        const int base = w * SQ_W + SQ_V * tid;
        float x[SQ_V];
        {
            const float4 *src = (const float4 *)(sq_ring + (w % (SQ_PF + 1)) * SQ_W + SQ_V * 64 * wave) + lane;
#pragma unroll
            for (int q = 0; q < SQ_V / 4; q++) {
                const float4 r = src[64 * q];
                x[4 * q] = base + 4 * q < n ? r.x : 0.0f;
                x[4 * q + 1] = base + 4 * q + 1 < n ? r.y : 0.0f;
                x[4 * q + 2] = base + 4 * q + 2 < n ? r.z : 0.0f;
                x[4 * q + 3] = base + 4 * q + 3 < n ? r.w : 0.0f;
            }
        }
        // window w + SQ_PF goes into the stage of window w - 1 (read before)
        issue(w + SQ_PF);
        const int wend = min(w * SQ_W + SQ_W, n);
        const int wbase = w * SQ_W + SQ_V * 64 * wave;  // this wavefront's values
        for (;;) {
            const int hi = short_pass ? min(lo + SQ_SHORT, wend) : wend;
            // a wavefront with none of [lo, hi) skips the element work
            const bool busy = wbase + SQ_V * 64 > lo && wbase < hi;
            const float lim = ldexpf(1.0f, P + 1);
            float L[SQ_V];
            bool sp[SQ_V];
            float run = 0.0f;
            if (busy) {
#pragma unroll
                for (int e = 0; e < SQ_V; e++) {
                    const int i = base + e;
                    const float xv = x[e];
                    float k = 0.0f;
                    bool special = false;
                    if (i >= lo && i < hi) {
                        if (!(xv >= 0.0f) || xv == __builtin_inff()) {
                            special = true;  // NaN, infinite or negative
                        } else if (xv >= lim) {
                            k = 2.0f * SQ_TOP;  // leaves the binade
                        } else {
                            const float t = ldexpf(xv, 23 - P);  // < 2^24, exact
                            k = rintf(t);
                            special = t - truncf(t) == 0.5f;  // a tie
                        }
                    }
                    sp[e] = special;
                    run = run + k;
                    L[e] = run;
                }
            }
            // exclusive prefix of the thread totals over the workgroup
            float incl = run;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const float y = __shfl_up(incl, o);
                if (lane >= o) incl = incl + y;
            }
            const float up = __shfl_up(incl, 1);
            const float exw = lane > 0 ? up : 0.0f;
            if (lane == 63) wtot[it][wave] = incl;
            __syncthreads();
            float before = 0.0f, total = 0.0f;
#pragma unroll
            for (int k = 0; k < SQ_T / 64; k++) {
                const float t = wtot[it][k];
                if (k < wave) before = before + t;
                total = total + t;
            }
            const float ex = M + (before + exw);
            // the first element that leaves the binade, is special or stops
            int first = SQ_V;
            if (busy) {
#pragma unroll
                for (int e = SQ_V - 1; e >= 0; e--) {
                    const float Me = ex + L[e];
                    bool st = sp[e] || Me >= SQ_TOP;
                    if (MODE != SQ_SUM && !st && base + e >= lo && base + e < hi)
                        st = sq_pred<MODE>(ldexpf(Me, P - 23), thr);
                    if (st) first = e;
                }
            }
            const unsigned long long b = __ballot(first < SQ_V);
            if (lane == (b ? __ffsll((long long)b) - 1 : 0))
                wstop[it][wave] = b ? SQ_V * tid + first : SQ_W;
            __syncthreads();
            int f = SQ_W;
#pragma unroll
            for (int k = 0; k < SQ_T / 64; k++) f = min(f, wstop[it][k]);
            it ^= 1;
            if (f == SQ_W) {  // [lo, hi) stays in the binade
                M = M + total;
                s = ldexpf(M, P - 23);
                lo = hi;
                short_pass = false;
                if (hi == wend) break;
                continue;
            }
            // element f: its thread adds it in fp32
            if (tid == f / SQ_V) {
                const int e = f % SQ_V;
                float Lp = 0.0f;
#pragma unroll
                for (int q = 0; q < SQ_V; q++)
                    if (q < e) Lp = L[q];
                float xe = x[0];
#pragma unroll
                for (int q = 1; q < SQ_V; q++)
                    if (q == e) xe = x[q];
                s1_sh[it ^ 1] = ldexpf(ex + Lp, P - 23) + xe;
            }
            __syncthreads();
            s = s1_sh[it ^ 1];
            const int fi = w * SQ_W + f;
            lo = fi + 1;
            short_pass = true;
            if (MODE != SQ_SUM && sq_pred<MODE>(s, thr)) {
                stop = fi;
                break;
            }
            if (!(s >= 0.0f) || s == __builtin_inff()) {
                seq = true;
                break;
            }
            P = sq_grid(s);
            M = ldexpf(s, 23 - P);
            if (lo == wend) break;
        }
    }
    if (seq) {  // the rest one addition at a time (NaN, infinite or negative sums)
        if (tid == 0) {
            int i = lo;
            for (; i < n; i++) {
                s = s + v[i];
                if (MODE != SQ_SUM && sq_pred<MODE>(s, thr)) break;
            }
            s1_sh[0] = s;
            wstop[0][0] = i;
        }
        __syncthreads();
        s = s1_sh[0];
        stop = MODE == SQ_SUM ? n : wstop[0][0];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the end
    *s_out = s;
    return stop;
}

// sampler.c:43: sum = e_0 + e_1 + ... + e_{n-1} (fp32, index order).
__global__ __launch_bounds__(SQ_T) void k_chain_sum(const float *__restrict__ e, int n,
                                                    SampleState *st) {
    float s;
    seq_scan<SQ_SUM>(e, n, 0.0f, &s);
    if (threadIdx.x == 0) {
        st->sum = s;
        st->walked = -1;
    }
}

// ---- the same over the whole chip ---------------------------------------------------
//
// A run of additions s <- fl(s + v), v >= 0, that stays inside one binade of
// s is a map of s's bits that depends on their lowest one alone (s = M u;
// fl(s + v) = (M + k) u, k the integer nearest v / u, a tie to the even M +
// k), and such maps compose. A double scan of the workgroups' sums tells in
// which binade nearly every piece will lie. k_sum_runs (all CUs) makes each
// such piece a map and composes the maps of every 64 pieces between the
// others, whose places it notes (the first, and those within 2^-14 of a power
// of two). k_sum_walk, one workgroup, composes what is left over the groups
// and then goes from one noted piece to the next: a map, the piece's own
// additions. The scan only predicts (the fp32 sum drifts from the exact one
// by its roundings); the walk checks each map before it counts: s lies in the
// binade the map was made for, and still does after it, so, the additions
// being of values >= 0, it did all along. Where that fails, or with more
// than WALK_MAX noted pieces (NaN or infinite values, sums among the
// subnormals), seq_scan runs over all values instead. 151936 values: 108 us
// for seq_scan on one workgroup, 4 + 8 us for the two; 3-8 % of draws over
// model-like logits at T = 0.6-1 still need seq_scan (many values too small
// to be added move a power of two past its noted pieces) and take what every
// draw took on one workgroup.
struct Run {
    int a0, a1;  // added to even (odd) bits
    int P;       // the exponent field of the binade; 0: nothing is added
};
__device__ __forceinline__ Run then(Run a, Run b) {
    return {a.a0 + ((a.a0 & 1) ? b.a1 : b.a0), a.a1 + ((a.a1 & 1) ? b.a0 : b.a1), b.P ? b.P : a.P};
}
__device__ __forceinline__ Run run_up(Run r, int o) {
    return {__shfl_up(r.a0, o), __shfl_up(r.a1, o), __shfl_up(r.P, o)};
}
// The runs of the lanes before and this one's, from the last lane with `head`
// set on (its own included); head: whether there was one.
__device__ __forceinline__ void wave_runs(Run &r, int &head, int lane) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const Run p = run_up(r, o);
        const int ph = __shfl_up(head, o);
        if (lane >= o && !head) {
            r = then(p, r);
            head = ph;
        }
    }
}

// run[k]: the maps of piece k and those before it in its group, from the last
// noted piece on (which has none of its own); noted[group]: a bit per piece.
__global__ __launch_bounds__(RUN_T) void k_sum_runs(const float *__restrict__ e, int n,
                                                    const double *__restrict__ bsum,
                                                    Run *__restrict__ run,
                                                    unsigned long long *__restrict__ noted) {
    __shared__ double part[RUN_T / 64], before[RUN_T / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double b = 0.0;
    for (int k = tid; k < (int)blockIdx.x; k += RUN_T) b = b + bsum[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) b = b + __shfl_xor(b, o);
    if (lane == 0) before[wave] = b;
    const int p = blockIdx.x * RUN_T + tid, i0 = p * PIECE;
    float v[PIECE];
#pragma unroll
    for (int j = 0; j < PIECE; j += 4) {
        const float4 q = i0 + j < n ? *(const float4 *)(e + i0 + j) : make_float4(0, 0, 0, 0);
        v[j] = q.x;
        v[j + 1] = i0 + j + 1 < n ? q.y : 0.0f;
        v[j + 2] = i0 + j + 2 < n ? q.z : 0.0f;
        v[j + 3] = i0 + j + 3 < n ? q.w : 0.0f;
    }
    double own = 0.0;
#pragma unroll
    for (int j = 0; j < PIECE; j++) own = own + (double)v[j];
    double incl = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const double y = __shfl_up(incl, o);
        if (lane >= o) incl = incl + y;
    }
    if (lane == 63) part[wave] = incl;
    __syncthreads();
    double base = 0.0;
    for (int k = 0; k < RUN_T / 64; k++) base = base + before[k];
    for (int k = 0; k < wave; k++) base = base + part[k];
    const double S1 = base + incl, S0 = S1 - own, dl = 0x1p-14;
    const unsigned b0 = (unsigned)((uint64_t)__double_as_longlong(S0 * (1.0 - dl)) >> 52);
    const unsigned b1 = (unsigned)((uint64_t)__double_as_longlong(S1 * (1.0 + dl)) >> 52);
    const bool zero = own == 0.0;  // (every value is +0, or past the end)
    const bool in = zero || (b0 == b1 && b0 >= 1023 - 100 && b0 < 1023 + 100);
    Run r = {0, 0, 0};
    if (in && !zero) {
        // v / u, u = 2^(P - 23), P = b0 - 1023: exact, or too small to count
        const float scale = __int_as_float((int)(127 + 23 + 1023 - b0) << 23);
        r.P = (int)b0 - 1023 + 127;
#pragma unroll
        for (int j = 0; j < PIECE; j++) {
            const float q = v[j] * scale, f = floorf(q), fr = q - f;
            const int k = (int)f, up = fr > 0.5f ? 1 : 0;
            const bool tie = fr == 0.5f;
            r.a0 = r.a0 + k + (tie ? (r.a0 + k) & 1 : up);
            r.a1 = r.a1 + k + (tie ? (r.a1 + k + 1) & 1 : up);
        }
    }
    const unsigned long long mask = __ballot(!in);
    int head = in ? 0 : 1;
    wave_runs(r, head, lane);
    run[p] = r;
    if (lane == 0) noted[p >> 6] = mask;
}

constexpr int WALK_MAX = 128;  // noted pieces of the walk, at most
static_assert(RUN_MAX_N / (64 * PIECE) <= SQ_T, "a thread per group");
__global__ __launch_bounds__(SQ_T) void k_sum_walk(const float *__restrict__ e, int n, int groups,
                                                   const Run *__restrict__ run,
                                                   const unsigned long long *__restrict__ noted,
                                                   SampleState *st) {
    __shared__ Run pre[WALK_MAX + 1], wlast[SQ_T / 64];
    __shared__ int piece[WALK_MAX], whead[SQ_T / 64], wcnt[SQ_T / 64], bad;
    __shared__ float vals[WALK_MAX][PIECE];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned long long mask = tid < groups ? noted[tid] : 0;
    Run r = {0, 0, 0};
    if (tid < groups) r = run[64 * tid + 63];
    // runs over the groups, from the last noted piece on, and the count of
    // noted pieces before each group
    int head = mask ? 1 : 0, cnt = __popcll(mask);
    wave_runs(r, head, lane);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(cnt, o);
        if (lane >= o) cnt = cnt + y;
    }
    if (lane == 63) {
        wlast[wave] = r;
        whead[wave] = head;
        wcnt[wave] = cnt;
    }
    if (tid == 0) bad = 0;
    __syncthreads();
    Run wb = {0, 0, 0};  // the wavefronts before this one
    int c0 = 0, total = 0;
    for (int k = 0; k < SQ_T / 64; k++) {
        if (k < wave) {
            wb = whead[k] ? wlast[k] : then(wb, wlast[k]);
            c0 = c0 + wcnt[k];
        }
        total = total + wcnt[k];
    }
    if (total <= WALK_MAX) {  // (uniform)
        const Run incl = head ? r : then(wb, r), up = run_up(incl, 1);
        const Run before = lane > 0 ? up : wb;  // from the last noted piece up to this group
        if (tid == SQ_T - 1) pre[total] = incl;
        int k = c0 + cnt - __popcll(mask), prev = -1;
        for (unsigned long long left = mask; left; left &= left - 1, k++) {
            const int i = __ffsll((long long)left) - 1;
            // the pieces between the noted one before (or the group's start)
            // and this one: piece i - 1's run starts there
            Run g = {0, 0, 0};
            if (i - 1 > prev) g = run[64 * tid + i - 1];
            pre[k] = prev < 0 ? then(before, g) : g;
            piece[k] = 64 * tid + i;
            prev = i;
        }
        __syncthreads();
        for (int q = tid; q < total * PIECE; q += SQ_T) {
            const int i = piece[q / PIECE] * PIECE + q % PIECE;
            vals[q / PIECE][q % PIECE] = i < n ? e[i] : 0.0f;
        }
        __syncthreads();
        if (wave == 0) {
            float s = 0.0f;
            bool ok = true;
            for (int q = 0; q <= total; q++) {
                const Run g = pre[q];
                const int b = __float_as_int(s), a = (b & 1) ? g.a1 : g.a0;
                ok = ok && (g.P == 0 || (b >> 23 == g.P && (b + a) >> 23 == g.P));
                s = __int_as_float(b + a);
                if (q < total) {
#pragma unroll
                    for (int j = 0; j < PIECE; j++) s = s + vals[q][j];
                }
            }
            if (tid == 0) {
                st->sum = s;
                st->walked = total;
                bad = !ok;
            }
        }
        __syncthreads();
        if (!bad) return;
    }
    float s;
    seq_scan<SQ_SUM>(e, n, 0.0f, &s);
    if (tid == 0) {
        st->sum = s;
        st->walked = -1;
    }
}

// sampler.c:46-51: p_i = e_i / sum; a candidate when p_i >= cutoff, as the
// key 0x7fffffff - bits(p) with i beside it: ascending keys are descending p
// (bits of p >= 0 order as p does), and the sort keeps equal ones in index
// order. (Against 64-bit keys of probability and index: 60 -> 54 us at 151936
// values.)
__global__ __launch_bounds__(NT) void k_sample_keys(const float *__restrict__ e, int n,
                                                    float cutoff,
                                                    const SampleState *__restrict__ st,
                                                    uint32_t *__restrict__ keys,
                                                    int *__restrict__ ids) {
    const int i = blockIdx.x * NT + threadIdx.x;
    if (i >= n) return;
    const float p = e[i] / st->sum;
    keys[i] = p >= cutoff ? 0x7fffffffu - __float_as_uint(p) : NONE;
    ids[i] = i;
}

// The sorted keys as probabilities pf[]; the candidates are the keys before
// the first NONE: their count goes to st->last (as m - 1, the default last
// candidate).
__global__ __launch_bounds__(NT) void k_keys_split(const uint32_t *__restrict__ keys, int n,
                                                   float *__restrict__ pf, SampleState *st) {
    const int i = blockIdx.x * NT + threadIdx.x;
    if (i >= n) return;
    const uint32_t k = keys[i];
    if (k == NONE) {
        if (i == 0) st->last = -1;
        return;
    }
    pf[i] = __uint_as_float(0x7fffffffu - k);
    if (i + 1 == n || keys[i + 1] == NONE) st->last = i;
}

// sampler.c:53-66 on the m candidates (pf, pi; m - 1 in st->last): cum =
// p_0 + p_1 + ... until cum >= top_p (last = that candidate) or the
// candidates end; r = u * cum; the pick is the first candidate up to last
// whose running sum (the same additions from 0) exceeds r, else last.
__global__ __launch_bounds__(SQ_T) void k_sample_pick(const float *__restrict__ pf,
                                                      const int *__restrict__ pi, float top_p,
                                                      float u, SampleState *st, int *token) {
    const int m = st->last + 1;
    if (m == 0) {  // no candidate
        if (threadIdx.x == 0) *token = st->best;
        return;
    }
    float cum;
    const int j = seq_scan<SQ_GE>(pf, m, top_p, &cum);
    const int last = j < m ? j : m - 1;
    const float r = u * cum;
    float acc;
    const int k = seq_scan<SQ_GT>(pf, last + 1, r, &acc);
    if (threadIdx.x == 0) {
        st->cum = cum;
        st->last = last;
        *token = pi[k <= last ? k : last];
    }
}

template <int MODE>
__global__ __launch_bounds__(SQ_T) void k_chain(const float *__restrict__ v, int n, float thr,
                                                int *__restrict__ out) {
    float s;
    const int k = seq_scan<MODE>(v, n, thr, &s);
    if (threadIdx.x == 0) {
        out[0] = __float_as_int(s);
        out[1] = k;
    }
}

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// The LDS ring of the running-sum kernels is above the default limit.
int sq_lds_attr(mhip_ctx *c) {
    const void *fns[] = {(const void *)k_chain_sum, (const void *)k_sum_walk, (const void *)k_sample_pick,
                         (const void *)k_chain<SQ_SUM>, (const void *)k_chain<SQ_GE>,
                         (const void *)k_chain<SQ_GT>};
    for (const void *f : fns)
        if (mhip::check(c, hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                               (int)SQ_LDS),
                        "sampler LDS attribute"))
            return -1;
    return 0;
}

struct SampleScratch {
    SampleState *st;
    Best *part;
    float *e;
    uint64_t *kin, *kout;
    // of the sum, in the places of what is dead or not yet there
    double *bsum;               // [workgroups of k_sum_runs]: the argmax's partial results
    Run *run;                   // [pieces]: the first keys
    unsigned long long *noted;  // [groups]: the sorted keys
    void *tmp;
    size_t tmp_bytes;
};

size_t sort_bytes(int n) {
    size_t b = 0;
    if (rocprim::radix_sort_pairs(nullptr, b, (const uint32_t *)nullptr, (uint32_t *)nullptr,
                                  (const int *)nullptr, (int *)nullptr, (unsigned)n, 0, 32) != hipSuccess)
        return 0;
    return b;
}

SampleScratch carve(int n, void *base) {
    uint8_t *p = (uint8_t *)base;
    SampleScratch s;
    s.st = (SampleState *)p;
    p += align256(sizeof(SampleState));
    s.part = (Best *)p;
    p += align256(sizeof(Best) * PARTS);
    s.e = (float *)p;
    p += align256((size_t)n * 4);
    s.kin = (uint64_t *)p;
    p += align256((size_t)n * 8);
    s.kout = (uint64_t *)p;
    p += align256((size_t)n * 8);
    s.bsum = (double *)s.part;
    s.run = (Run *)s.kin;
    s.noted = (unsigned long long *)s.kout;
    static_assert(sizeof(Best) >= sizeof(double), "a sum per partial result");
    static_assert((RUN_MIN_N + RUN_W) / PIECE * sizeof(Run) <= RUN_MIN_N * sizeof(uint64_t),
                  "whole workgroups of runs fit the keys");
    s.tmp = p;
    s.tmp_bytes = sort_bytes(n);
    return s;
}

// sampler.c:20-25: xorshift64* (shifts 12, 25, 27; multiplier
// 2685821657736338717), its top 24 bits over 2^24.
float rand01(mhip_sampler *s) {
    uint64_t x = s->rng;
    x ^= x >> 12;
    x ^= x << 25;
    x ^= x >> 27;
    s->rng = x;
    return (float)((x * 0x2545F4914F6CDD1DULL) >> 40) / 16777216.0f;
}

}  // namespace

extern "C" {

void mhip_sampler_init(mhip_sampler *s, float temperature, float top_p, int n, uint64_t seed) {
    s->temperature = temperature;
    s->top_p = (top_p > 0.0f && top_p <= 1.0f) ? top_p : 1.0f;
    s->n = n;
    s->rng = seed ? seed : 0x2545F4914F6CDD1DULL;
}

size_t mhip_sample_scratch_bytes(int n) {
    if (n < 1 || n > MHIP_SAMPLE_MAX_N) return 0;
    const size_t sb = sort_bytes(n);
    if (!sb) return 0;
    return align256(sizeof(SampleState)) + align256(sizeof(Best) * PARTS) +
           align256((size_t)n * 4) + 2 * align256((size_t)n * 8) + align256(sb);
}

int mhip_sample(mhip_ctx *c, mhip_sampler *s, const float *d_logits, void *d_scratch,
                int *d_token) {
    const int n = s ? s->n : 0;
    if (!s || n < 1 || n > MHIP_SAMPLE_MAX_N)
        return mhip::fail(c, "sampler: n=%d outside [1, %d]", n, MHIP_SAMPLE_MAX_N);
    if (!d_logits || !d_scratch || !d_token) return mhip::fail(c, "sampler: null pointer");
    if (mhip::use_device(c)) return -1;
    SampleScratch sc = carve(n, d_scratch);
    if (!sc.tmp_bytes) return mhip::fail(c, "sampler: sort workspace query failed");
    hipStream_t st = c->stream;
    const int greedy = s->temperature <= 0.0f;
    const unsigned parts = std::min<unsigned>(PARTS, mhip::blocks_for(n, NT));
    k_argmax_part<<<parts, NT, 0, st>>>(d_logits, n, sc.part);
    k_argmax_final<<<1, NT, 0, st>>>(d_logits, sc.part, parts, sc.st, greedy ? d_token : nullptr);
    if (greedy) return mhip::check_launch(c, "sampler (greedy)");
    // the host-side draw and cutoff, in the reference's order (sampler.c:47,63)
    const float u = rand01(s);
    const float cutoff = (1.0f - s->top_p) / (float)(n > 1 ? n - 1 : 1);
    const unsigned nb = mhip::blocks_for(n, NT);
    const unsigned rb = mhip::blocks_for(n, RUN_W);
    const bool runs = n >= RUN_MIN_N && n <= RUN_MAX_N;
    k_sample_exp<<<rb, RUN_T, 0, st>>>(d_logits, n, s->temperature, sc.st, sc.e,
                                       runs ? sc.bsum : nullptr);
    if (sq_lds_attr(c)) return -1;
    if (runs) {
        k_sum_runs<<<rb, RUN_T, 0, st>>>(sc.e, n, sc.bsum, sc.run, sc.noted);
        k_sum_walk<<<1, SQ_T, SQ_LDS, st>>>(sc.e, n, (int)rb * (RUN_T / 64), sc.run, sc.noted, sc.st);
    } else {
        k_chain_sum<<<1, SQ_T, SQ_LDS, st>>>(sc.e, n, sc.st);
    }
    uint32_t *key = (uint32_t *)sc.kin, *sorted = (uint32_t *)sc.kout;
    int *id = (int *)sc.kin + n, *pi = (int *)sc.kout + n;
    k_sample_keys<<<nb, NT, 0, st>>>(sc.e, n, cutoff, sc.st, key, id);
    if (mhip::check_launch(c, "sampler")) return -1;
    size_t tb = sc.tmp_bytes;
    if (mhip::check(c, rocprim::radix_sort_pairs(sc.tmp, tb, key, sorted, id, pi, (unsigned)n, 0, 32, st),
                    "sampler sort"))
        return -1;
    float *pf = (float *)sc.kin;  // the unsorted keys are dead after the sort
    k_keys_split<<<nb, NT, 0, st>>>(sorted, n, pf, sc.st);
    k_sample_pick<<<1, SQ_T, SQ_LDS, st>>>(pf, pi, s->top_p, u, sc.st, d_token);
    return mhip::check_launch(c, "sampler pick");
}

int mhip_chain_f32(mhip_ctx *c, const float *d_v, int n, int mode, float thr, int *d_out) {
    if (n < 0 || !d_out || (n > 0 && !d_v)) return mhip::fail(c, "chain: bad arguments (n=%d)", n);
    if ((uintptr_t)d_v % 16) return mhip::fail(c, "chain: d_v is not 16-byte aligned");
    if (mode != MHIP_CHAIN_SUM && mode != MHIP_CHAIN_GE && mode != MHIP_CHAIN_GT)
        return mhip::fail(c, "chain: mode %d", mode);
    if (mhip::use_device(c)) return -1;
    if (sq_lds_attr(c)) return -1;
    hipStream_t st = c->stream;
    if (mode == MHIP_CHAIN_SUM)
        k_chain<SQ_SUM><<<1, SQ_T, SQ_LDS, st>>>(d_v, n, thr, d_out);
    else if (mode == MHIP_CHAIN_GE)
        k_chain<SQ_GE><<<1, SQ_T, SQ_LDS, st>>>(d_v, n, thr, d_out);
    else
        k_chain<SQ_GT><<<1, SQ_T, SQ_LDS, st>>>(d_v, n, thr, d_out);
    return mhip::check_launch(c, "chain");
}

}  // extern "C"
