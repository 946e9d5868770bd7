// Expert products of the batched / prefill MoE layer on the matrix cores.
//
// For T tokens the T*K assignments are bucketed by expert (k_disp_*); each
// expert's bucket is a dense contraction with that expert's weights:
//
//   k_gateup_mfma  h = SwiGLU(Wg x, Wu x), then Q8_0(h)   forward.c:186-192
//   k_down_mfma    tmp = Wd Q8(h)                           forward.c:192-193
//
// Both products run on the Q8_0 codes themselves, as fp16 integers:
// v_mfma_f32_16x16x32_f16 over one 32-value block gives the exact int32
// block dot (every partial sum is an integer below 2^24). The reference's
// block term ((float)acc * d_w) * d_x is added to the row sum in block order
// by the vector ALUs (matmul.c:19-28) with the reference's three roundings, so
// h, Q8(h) after it and the expert outputs are bit-equal to the reference's.
// In gate/up that is needed: h is requantized, and a code that flips on a
// last-ulp difference moves a token's layer output by up to ~1.5e-3 relative
// (measured over 48 layers of 4096 tokens with one fused multiply-add there).
// down, whose output is not requantized, has the fused form as an option
// (MHIP_FAST_DOWN: the second product's rounding and the addition's become
// one, within a few fp32 ulps). gate/up writes Q8(h) as fp16 codes plus
// block-major scales, which down reads the same way as gate/up reads Q8(xn);
// no operand is ever rounded to fp16.
//
// Tiles: 256 weight rows x 128 assignments (rows of one expert's bucket),
// one 32-value Q8_0 block of k per step, eight wavefronts and two workgroups
// per CU. The weights are the A operand, so each lane's four results share
// one assignment (one x scale) and four consecutive weight rows (one float4
// of weight scales). A tile of more than 64 rows gives a wavefront 64 weight
// rows against one half of the assignments (4 x 4 tiles of 16 x 16), a tile
// of fewer 32 weight rows against all of them (2 x up to 4), so that both
// keep every wavefront busy on at most 64 accumulator registers: four
// wavefronts per SIMD, of which a vector operation of one runs beside another
// wavefront's (one alone issues one every ~4.3 cycles, several together one
// every ~2.1). Against four wavefronts of 64 weight rows x 128 assignments
// (two per SIMD), same-box: gate/up + down 151 + 80 -> 133 + 75 us at T =
// 512; the layer 598 -> 576 at T = 2048 skewed; T = 4096 the same (895, 898).
//
// Operands move from global memory straight into an NS-stage LDS ring with
// global_load_lds (no registers on the way), NS-1 steps ahead of the
// products. Each wavefront issues a fixed number of such loads per step, so
// a wait for the oldest step is one immediate vmcnt count. The loads are
// issued from inline assembly (which sets M0, the LDS base they use) so the
// compiler does not wait for all of them before every LDS read; the waits
// are explicit. Rows past a bucket's end load a valid row; their results are
// never stored.
#include "mhip_internal.h"

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int GT = 512;           // threads per workgroup (8 wavefronts)
constexpr int TM = MHIP_GEMM_TM;  // assignment rows per tile
constexpr int TN = 256;           // weight rows per tile
constexpr int KB = 32;            // k per step: one Q8_0 block
constexpr int WN = TN / 4;        // weight rows of a heavy tile's wavefront (64)
constexpr int MI = WN / 16;       // its 16-row weight tiles (4)
constexpr int NJ = TM / 32;       // its 16-row assignment tiles (4)
constexpr int NS = 4;             // ring stages (two workgroups per CU)
constexpr int OLD = TM + 4;       // gate/up epilogue tile row stride (floats): 128 columns + pad
constexpr int DLD = TN / 2 + 4;   // down epilogue tile row stride: 128 columns + pad

static_assert(TM == 128 && TN == 256 && GT == 512, "tiling");

// One step of the ring.
//   x:  assignment rows, 32 fp16 codes = 4 chunks of 16 bytes; chunk c
//       of row m sits at slot c ^ ((m >> 1) & 3), so the eight rows that
//       eight consecutive lanes read at one chunk fall on distinct banks;
//   w:  weight rows, 32 int8 codes = 2 halves of 16 bytes; half h of row n
//       sits at slot h ^ ((n >> 3) & 1), so the sixteen rows that sixteen
//       consecutive lanes read (8 bytes each) fall on distinct banks;
//   sw: block scales of the weight rows, sx: of the assignment rows.
struct alignas(16) Step {
    _Float16 x[TM][KB];  // 8 KB
    int8_t w[TN][KB];    // 8 KB
    float sw[TN];        // 1 KB
    float sx[TM];        // 512 B: the scale of row 16 j + l at 8 l + j
};
static_assert(sizeof(Step) == 17920, "step layout");

__device__ __forceinline__ int xslot(int m, int chunk) { return chunk ^ ((m >> 1) & 3); }
__device__ __forceinline__ int wslot(int n, int half) { return half ^ ((n >> 3) & 1); }

// The group g < G with f(g) <= p < f(g + 1), for a non-decreasing f over
// 0..G with f(0) <= p < f(G).
template <typename F>
__device__ __forceinline__ int find_group(F f, int G, int p) {
    int lo = 0, hi = G;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (f(mid) <= p)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// Tile coordinates shared by both kernels.
//
// A bucket's row tiles are TM rows each but its last, which holds the rest;
// that one is light when it has at most TM / 2 rows (its products run on at
// most four 16-row assignment tiles), heavy otherwise. The 1-D grid is
// ordered for balance and for the XCDs' L2 caches: workgroup b runs on XCD
// b % 8, and XCD k takes a contiguous eighth of the heavy row tiles (in
// bucket order, so consecutive tiles of one expert share its weights), then
// a contiguous eighth of the light ones, each row tile's ny weight-row tiles
// back to back (they share its A rows). Every XCD thus starts the same number
// of heavy tiles (within one) before any light tile, and the light tiles fill
// the last round. Workgroups beyond an XCD's shares exit.
struct TileRef {
    int e, base, nrows, y;
};
constexpr int NXCD = 8;
__device__ __forceinline__ bool tile_of(const int *groups, const int *gtile, const int *glight,
                                        int ny, TileRef &t) {
    const int G = groups[0];
    if (G == 0) return false;
    const int nl = glight[G], nh = gtile[G] - nl;
    const int hs = (nh + NXCD - 1) / NXCD, ls = (nl + NXCD - 1) / NXCD;
    const int b = blockIdx.x, xcd = b % NXCD, r = b / NXCD;
    const int q = r / ny;
    const int hk = max(0, min(hs, nh - xcd * hs)), lk = max(0, min(ls, nl - xcd * ls));
    int g, mt;
    if (q < hk) {
        // heavy tile p: group g's heavy tiles are its first
        // (gtile - glight)(g + 1) - (gtile - glight)(g)
        const int p = xcd * hs + q;
        auto heavy_before = [&](int k) { return gtile[k] - glight[k]; };
        g = find_group(heavy_before, G, p);
        mt = gtile[g] + (p - heavy_before(g));
    } else if (q < hk + lk) {
        // light tile p: the last tile of the group with glight(g) == p
        const int p = xcd * ls + (q - hk);
        g = find_group([&](int k) { return glight[k]; }, G, p);
        mt = gtile[g + 1] - 1;
    } else {
        return false;
    }
    t.y = r % ny;
    t.e = groups[1 + 3 * g];
    t.base = groups[2 + 3 * g] + (mt - gtile[g]) * TM;
    t.nrows = min(TM, groups[3 + 3 * g] - t.base);
    return true;
}

// global -> LDS, 16 (resp. 4) bytes per lane; lane i writes LDS at
// lds + 16 i (resp. 4 i). lds must be wavefront-uniform.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(unsigned lds, const void *g) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(g)
                 : "memory", "m0");
}
__device__ __forceinline__ void dma4(unsigned lds, const void *g) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(g)
                 : "memory", "m0");
}
#pragma clang diagnostic pop
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ unsigned lds_addr(const void *p) {
    return (unsigned)(uintptr_t)p;
}

// 8 Q8_0 codes (two little-endian words) as fp16 integers, in byte order:
// flipping the sign bit gives the code + 128 as a byte u, the fp16 with bits
// 0x64 u is 1024 + u, and subtracting 1152 is exact.
__device__ __forceinline__ h8 codes8(unsigned w0, unsigned w1) {
    const unsigned u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u;
    const unsigned d[4] = {__builtin_amdgcn_perm(0x64646464u, u0, 0x04010400u),
                           __builtin_amdgcn_perm(0x64646464u, u0, 0x04030402u),
                           __builtin_amdgcn_perm(0x64646464u, u1, 0x04010400u),
                           __builtin_amdgcn_perm(0x64646464u, u1, 0x04030402u)};
    const h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    h8 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const h2 v = __builtin_bit_cast(h2, d[i]) - off;
        r[2 * i] = v[0];
        r[2 * i + 1] = v[1];
    }
    return r;
}

// Per-thread global sources of one tile, advanced by one block per step:
// every wavefront copies 16 assignment rows, 32 weight rows and 64 scales
// (wavefronts 0-3 the weight rows', 4 and 5 the assignment rows', 6 and 7
// those again).
struct Src {
    const _Float16 *x;  // assignment-row chunk (KB halves per step)
    const int8_t *w;    // weight-row half (KB bytes per step)
    const float *s;     // scale, block-major ...
    int sstep;          // ... blocks sstep floats apart
};

// This thread's 16-byte pieces of a step: x row 16 w + lane / 4 (the chunk
// that lands in slot lane % 4), weight row 32 w + lane / 2 (the half that
// lands in slot lane % 2); the place of its scale among sx.
struct Pieces {
    int xr, xc, wr, wh, sx;
};
__device__ __forceinline__ Pieces pieces() {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    Pieces p;
    p.xr = 16 * wave + (lane >> 2);
    p.xc = xslot(p.xr, lane & 3);  // slot ^ swizzle = the chunk stored there
    p.wr = 32 * wave + (lane >> 1);
    p.wh = wslot(p.wr, lane & 1);
    p.sx = 64 * (wave & 1) + lane;
    return p;
}

// This lane's places in a step, in bytes from its start, at the wavefront's
// first tiles: tiles are whole 16-row groups, and a row's slots depend on the
// low bits of its index alone, so the other tiles lie at fixed distances.
struct Lanes {
    unsigned x, w, sw, sx;
};

// One step's products and terms of a wavefront: MIA 16-row weight tiles,
// nstep rows apart, against NJA assignment tiles.
template <bool EXACT, int MIA, int NJA>
__device__ __forceinline__ void step(const char *S, const Lanes &la, int nstep,
                                     f4v (&acc)[MI * NJ]) {
    const f4v z = {0.0f, 0.0f, 0.0f, 0.0f};
    h8 x[NJA];
#pragma unroll
    for (int j = 0; j < NJA; j++) x[j] = *(const h8 *)(S + la.x + j * 16 * KB * 2);
    const f4v sx = *(const f4v *)(S + la.sx);
    uint2 q = *(const uint2 *)(S + la.w);
    f4v sw = *(const f4v *)(S + la.sw);
#pragma unroll
    for (int i = 0; i < MIA; i++) {
        const h8 a = codes8(q.x, q.y);
        f4v blk[NJA];
#pragma unroll
        for (int j = 0; j < NJA; j++)
            blk[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, x[j], z, 0, 0, 0);
        const f4v s4 = sw;
        if (i + 1 < MIA) {
            q = *(const uint2 *)(S + la.w + (i + 1) * nstep * KB);
            sw = *(const f4v *)(S + la.sw + (i + 1) * nstep * 4);
        }
#pragma unroll
        for (int j = 0; j < NJA; j++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float t = blk[j][r] * s4[r];
                if (EXACT)
                    acc[i * NJ + j][r] = acc[i * NJ + j][r] + t * sx[j];  // no contraction (-ffp-contract=off)
                else
                    acc[i * NJ + j][r] = __builtin_fmaf(t, sx[j], acc[i * NJ + j][r]);
            }
            // the next tile's products start after this one's terms: started
            // all at once they would hold 64 registers
            asm volatile("" : "+v"(acc[i * NJ + j]), "+v"(q.x), "+v"(q.y));
        }
    }
}

// A wavefront's place in a tile. A heavy tile (over TM / 2 rows): weight rows
// 64 (w % 4) .. + 63, half w / 4 of the assignment tiles (of an odd count the
// second half's last one is empty, so that every wavefront of the workgroup
// runs the same code and meets the same barriers). A light one: 32 weight rows
// against all its rows.
struct Place {
    bool heavy;
    int n0, j0;      // LDS weight row, LDS assignment tile of its first tiles
    int r0, nj;      // its assignment tiles r0 .. + nj of the bucket's
};
// The assignment tiles of the halves of a heavy tile, and the bucket row at
// row m of the ring: the second half starts at ring tile NJ.
__device__ __forceinline__ int half_tiles(int nrows) { return (nrows + 31) / 32; }
__device__ __forceinline__ int ring_row(int m, int nrows) {
    const int r = nrows > TM / 2 && m >= TM / 2 ? m - TM / 2 + 16 * half_tiles(nrows) : m;
    return min(r, nrows - 1);  // (past the end: a valid row, its results unused)
}
__device__ __forceinline__ Place place_of(int nrows, int wave, bool paired) {
    Place p;
    p.heavy = nrows > TM / 2;
    if (p.heavy) {
        p.n0 = WN * (wave & 3);
        p.nj = half_tiles(nrows);
        p.j0 = NJ * (wave >> 2);
        p.r0 = p.nj * (wave >> 2);
    } else {
        // gate/up pairs a gate tile with the up tile 32 rows on
        p.n0 = paired ? WN * (wave >> 1) + 16 * (wave & 1) : 32 * wave;
        p.j0 = p.r0 = 0;
        p.nj = (nrows + 15) / 16;
    }
    return p;
}

// The k loop over nk steps (nk >= NS - 1). On return acc[NJ i + j][r] holds
//   C[n0 + 16 i + 4 (lane / 16) + r][16 (r0 + j) + lane % 16]
// (weight row, assignment row; a light tile's second weight tile lies NSTEP
// rows on) for j < nj: the exact block dots, each block
// term added with its two scales in block order.
// EXACT: the reference's three roundings, s = s + ((float)acc * d_w) * d_x
// (bit-equal row sums); otherwise the second product and the addition are
// one fused multiply-add (within a few ulps).
template <bool EXACT, int MIA, int NJA, int NSTEP>
__device__ __forceinline__ void gemm_tile(Step *ring, const Src &src, int nk, const Place &pl,
                                          f4v (&acc)[MI * NJ]) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int NLOAD = 3;  // global_load_lds per wavefront per step
    const unsigned ring0 = lds_addr(ring);
    const unsigned ox = (unsigned)offsetof(Step, x) + wave * 1024;
    const unsigned ow = (unsigned)offsetof(Step, w) + wave * 1024;
    const unsigned os = wave < 4 ? (unsigned)offsetof(Step, sw) + wave * 256
                                 : (unsigned)offsetof(Step, sx) + (wave & 1) * 256;
    auto issue = [&](int kb) {
        const int k = min(kb, nk - 1);  // past the end: reload the last step
        const unsigned st = ring0 + (unsigned)((kb % NS) * sizeof(Step));
        dma16(st + ox, src.x + (size_t)k * KB);
        dma16(st + ow, src.w + (size_t)k * KB);
        dma4(st + os, src.s + (size_t)k * src.sstep);
    };
#pragma unroll
    for (int s = 0; s < NS - 1; s++) issue(s);
    const int c = lane >> 4, l16 = lane & 15;
    Lanes la;
    la.x = (unsigned)offsetof(Step, x) + (16 * pl.j0 + l16) * KB * 2 + 16 * xslot(l16, c);
    la.w = (unsigned)offsetof(Step, w) + (pl.n0 + l16) * KB + 16 * wslot(l16, c >> 1) + 8 * (c & 1);
    la.sw = (unsigned)offsetof(Step, sw) + (pl.n0 + 4 * c) * 4;
    la.sx = (unsigned)offsetof(Step, sx) + (8 * l16 + pl.j0) * 4;
    for (int kb = 0; kb < nk; kb++) {
        // this wavefront's loads of step kb are done (NS - 2 later steps may
        // still be in flight); then every wavefront's are
        wait_vm<(NS - 2) * NLOAD>();
        __syncthreads();
        // step kb + NS - 1 reuses the slot read in step kb - 1, which every
        // wavefront has finished with (the LDS reads completed before the
        // barrier)
        issue(kb + NS - 1);
        step<EXACT, MIA, NJA>((const char *)&ring[kb % NS], la, NSTEP, acc);
    }
    wait_vm<0>();  // the reloads past the end
    __syncthreads();
}

// The k loop in the form of the tile (every wavefront of the workgroup the
// same): one per count of 16-row assignment tiles of a wavefront, so a
// bucket's last tile runs at most one empty tile.
template <bool EXACT, int NSTEP>
__device__ __forceinline__ void gemm_tile_rows(Step *ring, const Src &src, int nk, const Place &pl,
                                               f4v (&acc)[MI * NJ]) {
    if (pl.heavy) {
        switch (pl.nj) {
        case 4: gemm_tile<EXACT, MI, 4, 16>(ring, src, nk, pl, acc); break;
        default: gemm_tile<EXACT, MI, 3, 16>(ring, src, nk, pl, acc); break;
        }
    } else {
        switch (pl.nj) {
        case 4: gemm_tile<EXACT, MI / 2, 4, NSTEP>(ring, src, nk, pl, acc); break;
        case 3: gemm_tile<EXACT, MI / 2, 3, NSTEP>(ring, src, nk, pl, acc); break;
        case 2: gemm_tile<EXACT, MI / 2, 2, NSTEP>(ring, src, nk, pl, acc); break;
        default: gemm_tile<EXACT, MI / 2, 1, NSTEP>(ring, src, nk, pl, acc); break;
        }
    }
}

// ---- x block scales in bucketed, block-major order --------------------------------
//
// xsb[k][p] = xs[t][k] for the assignment p = (t, j) in bucketed order, so a
// tile's 128 rows read their scales of block k as one contiguous run.
// Thread p copies blocks XB y .. XB y + XB - 1 of its token's row: four
// 16-byte reads of one row (rather than a 4-byte gather per block), then
// stores that are contiguous across the wavefront for each block.
constexpr int XB = 16;
__global__ __launch_bounds__(256) void k_xs_bucket(const float *__restrict__ xs,
                                                   const int *__restrict__ perm,
                                                   float *__restrict__ xsb, int A, int nb, int K) {
    const int p = blockIdx.x * 256 + threadIdx.x, k0 = blockIdx.y * XB;
    if (p >= A) return;
    const float *row = xs + (size_t)(perm[p] / K) * nb + k0;
    float *dst = xsb + (size_t)k0 * A + p;
    if (nb % 4 == 0 && k0 + XB <= nb) {
        float v[XB];
#pragma unroll
        for (int q = 0; q < XB / 4; q++) {
            const float4 f = *(const float4 *)(row + 4 * q);
            v[4 * q] = f.x;
            v[4 * q + 1] = f.y;
            v[4 * q + 2] = f.z;
            v[4 * q + 3] = f.w;
        }
#pragma unroll
        for (int k = 0; k < XB; k++) dst[(size_t)k * A] = v[k];
    } else {
        for (int k = 0; k < XB && k0 + k < nb; k++) dst[(size_t)k * A] = row[k];
    }
}

union alignas(16) GateUpLds {
    Step ring[NS];
    float o[TM][OLD];  // epilogue: 128 assignment rows x 128 h columns
};
union alignas(16) DownLds {
    Step ring[NS];
    float o[TM][DLD];  // epilogue: 128 assignment rows x 128 down rows
};
static_assert(sizeof(GateUpLds) == NS * sizeof(Step) && sizeof(DownLds) == NS * sizeof(Step),
              "epilogue tiles fit the rings");
static_assert(2 * sizeof(DownLds) <= 160 * 1024, "two workgroups per CU");

// ---- gate/up + SwiGLU + Q8(h) ----------------------------------------------------
//
// blockIdx.x = tile of assignment rows (gtile numbering) x 6 column tiles of
// 128 consecutive h columns h0..h0+127. Wavefront w's 64 weight rows are the
// gate rows then the up rows of h columns h0+32w..h0+32w+31, so SwiGLU pairs
// its accumulator tiles i and i + 2 lane by lane.
__global__ __launch_bounds__(GT, 4) void k_gateup_mfma(
    const uint8_t *__restrict__ table, mhip_layout lay, const _Float16 *__restrict__ xq16,
    const float *__restrict__ xsb, const int *__restrict__ groups, const int *__restrict__ gtile,
    const int *__restrict__ glight, const int *__restrict__ perm, _Float16 *__restrict__ hq16,
    float *__restrict__ hsb, int d, int eh, int K, int A) {
    __shared__ GateUpLds L;
    __shared__ uint64_t etab[32];  // the expf table, for the SwiGLU lookups
    TileRef tr;
    if (!tile_of(groups, gtile, glight, eh / (TN / 2), tr)) return;
    if (threadIdx.x < 32) etab[threadIdx.x] = mia_expf_tab[threadIdx.x];  // read after the k loop's barriers
    const int base = tr.base, nrows = tr.nrows;
    const int h0 = tr.y * (TN / 2);
    const uint8_t *ex = table + (size_t)tr.e * lay.expert_bytes;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    Src src;
    {
        const Pieces p = pieces();
        src.x = xq16 + (size_t)(perm[base + ring_row(p.xr, nrows)] / K) * d + p.xc * 8;
        // tile row n: wavefront n / 64; within it gate rows then up rows
        auto wrow = [&](int n, int half) {
            const int r = n % WN;
            const int hc = h0 + (n / WN) * (WN / 2) + r % (WN / 2);
            return (const int8_t *)(ex + (r < WN / 2 ? lay.gate_q : lay.up_q)) + (size_t)hc * d +
                   16 * half;
        };
        src.w = wrow(p.wr, p.wh);
        if (wave < 4) {
            // scale of tile row 64 wave + lane
            const int hc = h0 + wave * (WN / 2) + lane % (WN / 2);
            src.s = (const float *)(ex + (lane < WN / 2 ? lay.gate_st : lay.up_st)) + hc;
            src.sstep = eh;
        } else {
            // sx slot p holds ring row 16 (p % 8) + p / 8
            src.s = xsb + base + ring_row(16 * (p.sx & 7) + (p.sx >> 3), nrows);
            src.sstep = A;
        }
    }

    f4v acc[MI * NJ];
#pragma unroll
    for (int i = 0; i < MI * NJ; i++) acc[i] = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
    const Place pl = place_of(nrows, __builtin_amdgcn_readfirstlane(wave), true);
    gemm_tile_rows<true, 32>(L.ring, src, d / KB, pl, acc);

    // SwiGLU into the h tile (LDS, reused): row = assignment, column = h - h0
    const int c = lane >> 4, l16 = lane & 15;
    auto swiglu = [&](const f4v &g, const f4v &u, int row, int col) {
        f4v hv;
#pragma unroll
        for (int r = 0; r < 4; r++)
            hv[r] = (g[r] / (1.0f + mia_expf_glibc_tab(-g[r], etab))) * u[r];
        *(f4v *)&L.o[row][col] = hv;
    };
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        if (j < pl.nj) {
            const int row = 16 * (pl.r0 + j) + l16;
            if (pl.heavy) {
#pragma unroll
                for (int i = 0; i < MI / 2; i++)
                    swiglu(acc[i * NJ + j], acc[(i + 2) * NJ + j], row,
                           (WN / 2) * (wave & 3) + 16 * i + 4 * c);
            } else {
                swiglu(acc[j], acc[NJ + j], row, 16 * wave + 4 * c);
            }
        }
    }
    __syncthreads();
    {
        // Q8_0 of 32-blocks of h (quant.c:11-27): the codes as fp16 integers
        // (bucketed rows) and the scales block-major (hsb[block][row], the
        // down kernel's x scales); a thread per (row, block)
        const int m = tid >> 2, blk = tid & 3;
        if (m < nrows) {
            const f4v *hs = (const f4v *)&L.o[m][32 * blk];
            float v[32];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const f4v q = hs[k];
                v[4 * k] = q[0];
                v[4 * k + 1] = q[1];
                v[4 * k + 2] = q[2];
                v[4 * k + 3] = q[3];
            }
            float amax = 0.0f;
#pragma unroll
            for (int k = 0; k < 32; k++) amax = fmaxf(amax, fabsf(v[k]));
            const float dsc = amax / 127.0f;
            const float qi = dsc != 0.0f ? 1.0f / dsc : 0.0f;
            h8 o[4];
#pragma unroll
            for (int k = 0; k < 32; k++) o[k >> 3][k & 7] = (_Float16)roundf(v[k] * qi);
            h8 *dst = (h8 *)(hq16 + (size_t)(base + m) * eh + h0 + 32 * blk);
#pragma unroll
            for (int k = 0; k < 4; k++) dst[k] = o[k];
            hsb[(size_t)(h0 / KB + blk) * A + base + m] = dsc;
        }
    }
}

// ---- down -----------------------------------------------------------------------------
//
// blockIdx.x = tile of assignment rows x 8 column tiles of 256 consecutive
// down rows n0..n0+255. The x operand is the tile's Q8(h) (fp16 codes,
// bucketed order, contiguous) with its block-major scales. Results go out
// through LDS 128 columns at a time, so every assignment row is written as
// 512 contiguous bytes.
// EXACT: the reference's roundings of each block term (the expert outputs
// bit-equal); otherwise one fused multiply-add per term (a few ulps).
template <bool EXACT>
__global__ __launch_bounds__(GT, 4) void k_down_mfma(const uint8_t *__restrict__ table,
                                                     mhip_layout lay,
                                                     const _Float16 *__restrict__ hq16,
                                                     const float *__restrict__ hsb,
                                                     const int *__restrict__ groups,
                                                     const int *__restrict__ gtile,
                                                     const int *__restrict__ glight,
                                                     float *__restrict__ tmp, int d, int eh,
                                                     int A) {
    __shared__ DownLds L;
    TileRef tr;
    if (!tile_of(groups, gtile, glight, d / TN, tr)) return;
    const int base = tr.base, nrows = tr.nrows;
    const int n0 = tr.y * TN;
    const uint8_t *ex = table + (size_t)tr.e * lay.expert_bytes;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    Src src;
    {
        const Pieces p = pieces();
        src.x = hq16 + (size_t)(base + ring_row(p.xr, nrows)) * eh + p.xc * 8;
        src.w = (const int8_t *)(ex + lay.down_q) + (size_t)(n0 + p.wr) * eh + 16 * p.wh;
        if (wave < 4) {
            src.s = (const float *)(ex + lay.down_st) + n0 + WN * wave + lane;
            src.sstep = d;
        } else {
            // sx slot p holds ring row 16 (p % 8) + p / 8
            src.s = hsb + base + ring_row(16 * (p.sx & 7) + (p.sx >> 3), nrows);
            src.sstep = A;
        }
    }

    f4v acc[MI * NJ];
#pragma unroll
    for (int i = 0; i < MI * NJ; i++) acc[i] = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
    const Place pl = place_of(nrows, __builtin_amdgcn_readfirstlane(wave), false);
    gemm_tile_rows<EXACT, 16>(L.ring, src, eh / KB, pl, acc);

    const int c = lane >> 4, l16 = lane & 15;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        // the tile's columns 128 half .. + 127, then every thread writes them out
        if (pl.n0 / (TN / 2) == half) {
#pragma unroll
            for (int j = 0; j < NJ; j++)
                if (j < pl.nj) {
#pragma unroll
                    for (int i = 0; i < MI; i++)
                        if (pl.heavy || i < MI / 2)
                            *(f4v *)&L.o[16 * (pl.r0 + j) + l16][pl.n0 % (TN / 2) + 16 * i + 4 * c] =
                                acc[i * NJ + j];
                }
        }
        __syncthreads();
        // 128 rows x 32 float4: thread tid writes float4 tid % 32 of rows tid / 32 + 16 k
#pragma unroll
        for (int k = 0; k < TM / 16; k++) {
            const int m = tid / 32 + 16 * k, f = tid % 32;
            if (m < nrows)
                *(f4v *)(tmp + (size_t)(base + m) * d + n0 + (TN / 2) * half + 4 * f) =
                    *(const f4v *)&L.o[m][4 * f];
        }
        __syncthreads();
    }
}

}  // namespace

namespace mhip {

bool gemm_path_fits(const mhip_dims *s) {
    // whole tiles of weight rows, and enough k steps to fill the rings
    return s->dim % TN == 0 && s->expert_hidden % (TN / 2) == 0 && s->dim / KB >= NS - 1 &&
           s->expert_hidden / KB >= NS - 1;
}

int gemm_max_tiles(int A, int E) { return (A + TM - 1) / TM + (A < E ? A : E); }

// Workgroups for ny weight-row tiles: every XCD's heavy and light shares
// (ceil(H / 8) + ceil(L / 8) <= ceil((H + L) / 8) + 1 row tiles) fit.
static unsigned gemm_grid(int A, int E, int ny) {
    const int share = (gemm_max_tiles(A, E) + NXCD - 1) / NXCD + 1;
    return (unsigned)(NXCD * share * ny);
}

int launch_gateup_mfma(hipStream_t st, const mhip_dims *s, const mhip_layout *lay,
                       const void *d_table_layer, const mhip_scratch *sc, int A) {
    const int d = s->dim, eh = s->expert_hidden;
    k_xs_bucket<<<dim3((A + 255) / 256, (d / KB + XB - 1) / XB), 256, 0, st>>>(
        sc->xs, sc->perm, sc->xsb, A, d / KB, s->n_active);
    const unsigned grid = gemm_grid(A, s->n_experts, eh / (TN / 2));
    k_gateup_mfma<<<grid, GT, 0, st>>>((const uint8_t *)d_table_layer, *lay,
                                       (const _Float16 *)sc->xdq, sc->xsb, sc->groups,
                                       sc->gtile, sc->glight, sc->perm, (_Float16 *)sc->hdq,
                                       sc->hs, d, eh, s->n_active, A);
    return (int)hipGetLastError();
}

int launch_down_mfma(hipStream_t st, const mhip_dims *s, const mhip_layout *lay,
                     const void *d_table_layer, const mhip_scratch *sc, int A, bool exact) {
    const int d = s->dim, eh = s->expert_hidden;
    const unsigned grid = gemm_grid(A, s->n_experts, d / TN);
    if (exact)
        k_down_mfma<true><<<grid, GT, 0, st>>>((const uint8_t *)d_table_layer, *lay,
                                               (const _Float16 *)sc->hdq, sc->hs, sc->groups,
                                               sc->gtile, sc->glight, sc->tmp, d, eh, A);
    else
        k_down_mfma<false><<<grid, GT, 0, st>>>((const uint8_t *)d_table_layer, *lay,
                                                (const _Float16 *)sc->hdq, sc->hs, sc->groups,
                                                sc->gtile, sc->glight, sc->tmp, d, eh, A);
    return (int)hipGetLastError();
}

}  // namespace mhip
