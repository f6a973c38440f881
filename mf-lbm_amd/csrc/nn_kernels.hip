// Kernels of the learned warm start: a 3-D convolutional encoder-decoder trained on steady velocity fields
// that the single-phase solver produces (no reference counterpart; the reference starts every run at rest).
//
// Tensors are channels-last, x[n][z][y][x][c] in BF16; channel counts are multiples of 8 so a lane loads 8
// consecutive channels (16 bytes) at once.  A 3x3x3 convolution (stride 1, zero padding 1) is an implicit GEMM
// out[p][co] = sum_k A[p][k] B[k][co] with k = off * cin + ci (off = 9 (dz+1) + 3 (dy+1) + (dx+1)), run on the
// gfx950 matrix cores (v_mfma_f32_16x16x32_bf16, FP32 accumulation).  Weights are stored per output channel as
// rows of kpad = roundup(27 cin, 32) BF16 values (zero beyond 27 cin); the FP32 master copy (rows of 27 cin)
// lives with the optimiser.  The input gradient of a convolution is the same kernel run on the output gradient with the
// kernel flipped and its channel roles swapped (mflbm_nn_weights_to_bf16 writes both forms).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>

#include "mflbm.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int NT = 256;
constexpr unsigned NOWHERE = 1u << 31;   // a byte offset beyond every buffer resource: such a load reads zero
constexpr int NXCD = 8;   // gfx950: 8 dies, work-groups dispatched to them in turn

__device__ __forceinline__ float bf2f(__bf16 v) { return (float)v; }
__device__ __forceinline__ __bf16 f2bf(float v) { return (__bf16)v; }

struct Shape {
    int n, d, h, w;
    __host__ __device__ __forceinline__ long count() const { return (long)n * d * h * w; }
};

// Matrix-core fragment layout of v_mfma_f32_16x16x32_bf16 for lane l (64 lanes): A row l % 16 with k
// 8 (l / 16) .. +7; B column l % 16 with the same k; D holds rows 4 (l / 16) + t, t = 0..3, of column l % 16.
__device__ __forceinline__ f32x4 mfma(const bf16x8& a, const bf16x8& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// 16 x 16 x 32 product of row-major A (16 x 32) and column-major B (columns of 32): the layout check.
__global__ void k_mfma_probe(const __bf16* __restrict__ a, const __bf16* __restrict__ b, float* __restrict__ d) {
    const int l = threadIdx.x;
    const int r = l & 15, q = l >> 4;
    bf16x8 fa, fb;
    for (int j = 0; j < 8; ++j) {
        fa[j] = a[r * 32 + q * 8 + j];
        fb[j] = b[r * 32 + q * 8 + j];
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    acc = mfma(fa, fb, acc);
    for (int t = 0; t < 4; ++t) d[(q * 4 + t) * 16 + r] = acc[t];
}

// One wave computes 32 positions x 32 output channels; 4 waves per block along positions.
template <int RELU>
__global__ void __launch_bounds__(NT) k_conv_fwd(const __bf16* __restrict__ x, const __bf16* __restrict__ wt,
                                                 const float* __restrict__ bias, __bf16* __restrict__ y, Shape S,
                                                 int cin, int cout, int kpad) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const long M = S.count();
    const long p0 = ((long)blockIdx.x * 4 + wv) * 32;
    const int co0 = blockIdx.y * 32;
    if (p0 >= M) return;
    const int r = lane & 15, q = lane >> 4;
    int pz[2], py[2], px[2], pn[2];
    bool pv[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        long p = p0 + h * 16 + r;
        pv[h] = p < M;
        if (!pv[h]) p = 0;
        px[h] = (int)(p % S.w);
        p /= S.w;
        py[h] = (int)(p % S.h);
        p /= S.h;
        pz[h] = (int)(p % S.d);
        pn[h] = (int)(p / S.d);
    }
    const int K = 27 * cin;
    f32x4 acc[2][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < 2; ++g) acc[h][g] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x8 zero = {};
    for (int k0 = 0; k0 < kpad; k0 += 32) {
        const int k = k0 + q * 8;
        bf16x8 a[2] = {zero, zero}, b[2] = {zero, zero};
        if (k < K) {
            const int off = k / cin, ci = k - off * cin;
            const int dz = off / 9 - 1, dy = (off / 3) % 3 - 1, dx = off % 3 - 1;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int zz = pz[h] + dz, yy = py[h] + dy, xx = px[h] + dx;
                if (pv[h] && zz >= 0 && zz < S.d && yy >= 0 && yy < S.h && xx >= 0 && xx < S.w)
                    a[h] = *(const bf16x8*)(x + ((((long)pn[h] * S.d + zz) * S.h + yy) * S.w + xx) * cin + ci);
            }
        }
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int co = co0 + g * 16 + r;
            if (co < cout) b[g] = *(const bf16x8*)(wt + (long)co * kpad + k);   // zero padded beyond K
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int g = 0; g < 2; ++g) acc[h][g] = mfma(a[h], b[g], acc[h][g]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const int co = co0 + g * 16 + r;
            if (co >= cout) continue;
            const float bb = bias ? bias[co] : 0.f;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const long p = p0 + h * 16 + q * 4 + t;
                if (p >= M) continue;
                float v = acc[h][g][t] + bb;
                if (RELU && v < 0.f) v = 0.f;
                y[p * cout + co] = f2bf(v);
            }
        }
}

// The same convolution from a spatial tile in LDS: a work-group owns TZ x TY x TX positions and 16 NCO WC output
// channels, stages the tile's input with its one-node halo once (all cin channels; zero outside the domain) and takes all
// 27 offsets from there, so each input value is read from memory about 2.3 times instead of 27.  Wave (wp, wc) computes
// 16 MT positions x 16 NCO channels; the weights of KG steps of 32 k come through LDS in fragment order (16 bytes per
// lane, linear), two buffers in turn, the next stage's loads in flight.  Rows of the input tile are an odd number of
// 16-byte chunks apart, so the 16 positions of a fragment fall on different banks.  The k order, and so every sum, is
// that of k_conv_fwd; weights are the A operand, so a lane ends with four consecutive channels of one position.
// Bound by LDS: 32 -> 32 channels at 4 x 64^3, 105 us (552 TFLOP/s), the LDS is active 67 % of the cycles and the matrix
// cores 21 %; a wave of 2 x 2 fragments reads four of them from LDS for four products.
template <int MT, int NCO, int WP, int WC, int TZ, int TY, int TX, int KG>
struct ConvTile {
    static constexpr int THREADS = 64 * WP * WC, POS = TZ * TY * TX, CO = 16 * NCO * WC;
    static constexpr int HX = TX + 2, HY = TY + 2, HZ = TZ + 2, ROWS = HX * HY * HZ;
    static constexpr int WITEMS = KG * CO * 4;   // 16-byte chunks of a weight stage
    static_assert(POS == 16 * MT * WP && WITEMS % THREADS == 0, "tile split");
    static int lds_bytes(int cin) { return ((ROWS * ((cin / 8) | 1) + 1) + 2 * WITEMS) * 16; }
};
template <int RELU, bool UNI, int MT, int NCO, int WP, int WC, int TZ, int TY, int TX, int KG>
__global__ void __launch_bounds__(64 * WP * WC) k_conv_tile(const __bf16* __restrict__ x, const __bf16* __restrict__ wt,
                                                            const float* __restrict__ bias, __bf16* __restrict__ y, Shape S,
                                                            int cin, int cout, int kpad, int nxt, int nyt, int nzt, int ncg,
                                                            int total) {
    using T = ConvTile<MT, NCO, WP, WC, TZ, TY, TX, KG>;
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    const int g0 = (int)(blockIdx.x % NXCD) * (int)(gridDim.x / NXCD) + (int)(blockIdx.x / NXCD);   // a die: consecutive tiles
    if (g0 >= total) return;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wp = wv % WP, wc = wv / WP;
    const int r = lane & 15, q = lane >> 4;
    int t = g0;
    const int co0 = (t % ncg) * T::CO;
    t /= ncg;
    const int x0 = (t % nxt) * TX;
    t /= nxt;
    const int y0 = (t % nyt) * TY;
    t /= nyt;
    const int z0 = (t % nzt) * TZ;
    const int nn = t / nzt;
    const int nch = cin / 8, sc = nch | 1;
    u32x4* const xs = lds;                              // ROWS rows of sc chunks, then a zero chunk
    u32x4* const ws = lds + T::ROWS * sc + 1;           // two stages of weight fragments
    const u32x4 none = {};
    // input tile through a buffer resource over its planes (the launcher keeps the window below 2 GiB); an item outside
    // the domain takes an offset beyond it and reads zero
    const long plane = (long)S.h * S.w;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(x + ((long)nn * S.d + z0 - 1) * plane * cin), 0, (int)(T::HZ * plane * cin * 2), 0x00027000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)wt, 0, cout * kpad * 2, 0x00027000);
    const int nk = kpad / 32, ns = (nk + KG - 1) / KG;
    // weight items: chunk q of step kk of channel c: 64 KG contiguous bytes of a channel's row per 4 KG threads
    constexpr int NW = T::WITEMS / T::THREADS;
    unsigned wo[NW];
    int wl[NW];
#pragma unroll
    for (int v = 0; v < NW; ++v) {
        const int u = tid + T::THREADS * v, uq = u & 3, kk = (u >> 2) % KG, c = (u >> 2) / KG;
        wo[v] = co0 + c < cout ? 2u * (unsigned)((co0 + c) * kpad + kk * 32 + uq * 8) : NOWHERE;
        wl[v] = ((kk * (T::CO / 16) + (c >> 4)) * 4 + uq) * 16 + (c & 15);
    }
    u32x4 rw[NW];
    auto wload = [&](int s) {
#pragma unroll
        for (int v = 0; v < NW; ++v) {
            const int kk = ((tid + T::THREADS * v) >> 2) % KG;   // (a step past the row's end is not read)
            rw[v] = __builtin_amdgcn_raw_buffer_load_b128(wr, (int)(s * KG + kk < nk ? wo[v] : NOWHERE), s * KG * 64, 0);
        }
    };
    auto wstore = [&](int buf) {
#pragma unroll
        for (int v = 0; v < NW; ++v) ws[buf * T::WITEMS + wl[v]] = rw[v];
    };
    wload(0);
    {
        const int items = T::ROWS * nch;
        constexpr int UN = 8;   // loads in flight per thread
        for (int u0 = tid; u0 < items; u0 += UN * T::THREADS) {
            u32x4 v[UN];
            int at[UN];
#pragma unroll
            for (int k = 0; k < UN; ++k) {
                const int u = u0 + k * T::THREADS;
                const int row = u / nch, c = u - row * nch;
                const int hx = row % T::HX, hy = (row / T::HX) % T::HY, hz = row / (T::HX * T::HY);
                const int zz = z0 - 1 + hz, yy = y0 - 1 + hy, xx = x0 - 1 + hx;
                const bool in = (u < items) & ((unsigned)zz < (unsigned)S.d) & ((unsigned)yy < (unsigned)S.h) & ((unsigned)xx < (unsigned)S.w);
                at[k] = row * sc + c;
                v[k] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(in ? (((unsigned)hz * S.h + yy) * S.w + xx) * (unsigned)cin * 2u + 16u * c : NOWHERE), 0, 0);
            }
#pragma unroll
            for (int k = 0; k < UN; ++k)
                if (u0 + k * T::THREADS < items) xs[at[k]] = v[k];
        }
        if (tid == 0) xs[T::ROWS * sc] = none;
    }
    wstore(0);
    // first chunk of the row of this lane's position in each fragment
    int rb[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int p = (wp * MT + m) * 16 + r;
        rb[m] = ((p / (TX * TY) * T::HY + p / TX % TY) * T::HX + p % TX) * sc;
    }
    f32x4 acc[MT][NCO];
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int c = 0; c < NCO; ++c) acc[m][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    // One step of 32 k: this lane's eight k are one channel chunk of one offset; with cin a multiple of 32 (UNI) the
    // offset is the whole wave's, else the division goes by a multiplication (k8 / nch = k8 * inv >> 16 for k8 < 65536 /
    // nch) and the last step may reach beyond the 27 offsets (zero chunk).
    const unsigned inv = (65536u + nch - 1) / nch;
    auto products = [&](const u32x4* w, int ks) {
        const unsigned k8 = UNI ? (unsigned)ks * 4u : (unsigned)(ks * 4 + q);
        const unsigned off = k8 * inv >> 16, c8 = k8 - off * nch + (UNI ? q : 0);
        const unsigned dz = off * 57u >> 9, e = off - 9u * dz, dyy = e * 11u >> 5;
        const int ko = (int)(((dz * T::HY + dyy) * T::HX + (e - 3u * dyy)) * (unsigned)sc + c8);
        bf16x8 fw[NCO], fx[MT];
#pragma unroll
        for (int c = 0; c < NCO; ++c) fw[c] = __builtin_bit_cast(bf16x8, w[c * 64]);
#pragma unroll
        for (int m = 0; m < MT; ++m) fx[m] = __builtin_bit_cast(bf16x8, xs[UNI || off < 27u ? rb[m] + ko : T::ROWS * sc]);
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < NCO; ++c) acc[m][c] = mfma(fw[c], fx[m], acc[m][c]);
    };
    __syncthreads();
    for (int s = 0; s < ns; ++s) {
        if (s + 1 < ns) wload(s + 1);
        const u32x4* const w = ws + (s & 1) * T::WITEMS + wc * NCO * 64 + lane;
        if ((s + 1) * KG <= nk) {   // (whole stages without a branch between their products)
#pragma unroll
            for (int kk = 0; kk < KG; ++kk) products(w + kk * T::CO * 4, s * KG + kk);
        } else {
            for (int kk = 0; s * KG + kk < nk; ++kk) products(w + kk * T::CO * 4, s * KG + kk);
        }
        if (s + 1 < ns) wstore((s + 1) & 1);
        __syncthreads();
    }
    const bool quad = cout % 4 == 0 && ((uintptr_t)y & 7) == 0;
#pragma unroll
    for (int c = 0; c < NCO; ++c) {
        const int co = co0 + (wc * NCO + c) * 16 + 4 * q;
        float bb[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) bb[k] = bias && co + k < cout ? bias[co + k] : 0.f;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int p = (wp * MT + m) * 16 + r;
            const int zz = z0 + p / (TX * TY), yy = y0 + p / TX % TY, xx = x0 + p % TX;
            if (zz >= S.d || yy >= S.h || xx >= S.w) continue;
            __bf16* const out = y + (((long)nn * S.d + zz) * plane + (long)yy * S.w + xx) * cout + co;
            bf16x4 o;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                float v = acc[m][c][k] + bb[k];
                if (RELU && v < 0.f) v = 0.f;
                o[k] = f2bf(v);
            }
            if (quad) {
                if (co < cout) *(bf16x4*)out = o;
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (co + k < cout) out[k] = o[k];
            }
        }
    }
}
template <int MT, int NCO, int WP, int WC, int TZ, int TY, int TX, int KG>
int launch_conv_tile(const void* x, const void* wf, const float* bias, void* y, const Shape& S, int cin, int cout, int kpad,
                     int relu, hipStream_t st) {
    using T = ConvTile<MT, NCO, WP, WC, TZ, TY, TX, KG>;
    const int nxt = (S.w + TX - 1) / TX, nyt = (S.h + TY - 1) / TY, nzt = (S.d + TZ - 1) / TZ, ncg = (cout + T::CO - 1) / T::CO;
    const long total = (long)nxt * nyt * nzt * S.n * ncg;
    const int bytes = T::lds_bytes(cin);
    const bool uni = cin % 32 == 0;
    const auto kern = relu ? (uni ? k_conv_tile<1, true, MT, NCO, WP, WC, TZ, TY, TX, KG> : k_conv_tile<1, false, MT, NCO, WP, WC, TZ, TY, TX, KG>)
                           : (uni ? k_conv_tile<0, true, MT, NCO, WP, WC, TZ, TY, TX, KG> : k_conv_tile<0, false, MT, NCO, WP, WC, TZ, TY, TX, KG>);
    if (bytes > 65536 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
        return MFLBM_ERR_HIP;
    hipLaunchKernelGGL(kern, dim3((unsigned)((total + NXCD - 1) / NXCD * NXCD)), dim3(T::THREADS), bytes, st, (const __bf16*)x,
                       (const __bf16*)wf, bias, (__bf16*)y, S, cin, cout, kpad, nxt, nyt, nzt, ncg, (int)total);
    return hipGetLastError() == hipSuccess ? MFLBM_OK : MFLBM_ERR_HIP;
}

// Weight gradient: dw[co][k] += sum_p dy[p][co] * x[p + off(k)][ci(k)] (rows of 27 cin, the layout of the FP32
// master weights), the positions split into chunks of `chunk` (a multiple of 32) over grid z.  A work-group computes
// 16 NC output channels x 16 input channels x all 27 offsets and walks its chunk 32 positions at a time; wave v takes
// the offsets 7 v .. 7 v + 6, so one dy fragment serves seven products.  w is a multiple of 8, so eight positions from
// a multiple of 8 on lie in one x row: per such octet and per (dz, dy) the rows x - 1 .. x + 8 are staged (zero outside
// the domain), and an offset's operand is those rows from dx on.  Both tiles are staged as they lie in memory,
// [position][channel], 16 bytes at a time, two buffers in turn, and the transposing LDS read of gfx950 hands each lane
// the positions of its channel (of 16 lanes, lane 4 j + c / 4 addresses row j, channels 4 (c / 4) .., and lane c receives
// rows 0 .. 3 of channel c).  The fragments, and so the sums, are those of a lane-by-lane gather: lane l takes the
// 8 consecutive positions from 8 (l / 16) on of one output channel (A) or one input channel (B).
// Bound by the latency of a tile (load, barrier, LDS reads, 7 NC products) with few waves on each compute unit: the
// chunk fixes the order of the sums, so a work-group walks all 128 tiles.  4 x 32^3, 64 -> 64, with the chunk sums: 567
// us with scalar transposing stores, 88 us so; 4 x 64^3, 32 -> 32: 1010 and 154 us (377 TFLOP/s).
// The chunk sums go to dw with FP32 atomics, or (ORDERED) are stored to the chunk's own slice dw + z * cout * K,
// every element written by exactly one lane, for a fixed-order sum after.
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bf16x8 read_transposed(const __bf16* lo, const __bf16* hi) {
    union {
        s16x4 h[2];
        bf16x8 v;
    } u;
    u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)lo);
    u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)hi);
    return u.v;
}
// Global reads go through a buffer resource over the chunk and its neighbours: an item outside the domain or the layer
// takes an offset beyond it and reads zero, so no load sits under a branch (it would have to arrive before the branch
// is left) and nothing is cleared on the way to LDS.  Wave v stages octet v of the tile, whose coordinates are scalar;
// each item needs some of seven conditions on them (a lane constant).  FAR: the window is 2 GiB or more (planes of
// hundreds of millions of values); the same loads by 64-bit addresses.
constexpr int DW_OFF = 7;    // offsets per wave
constexpr int DW_ROWS = 9 * 4 * 10;   // staged x rows of a tile: (dz, dy) x octet x (x - 1 .. x + 8)
__host__ __device__ inline long dw_window(const Shape& S, int cin, long chunk) {   // bytes of x a chunk may touch
    return (chunk + 8 + 2 * ((long)S.h * S.w + S.w + 1)) * cin * 2;
}
template <bool ORDERED, int NC, bool FAR>
__global__ void __launch_bounds__(NT, 2) k_conv_dw(const __bf16* __restrict__ x, const __bf16* __restrict__ dy,
                                                   float* __restrict__ dw, Shape S, int cin, int cout, long chunk,
                                                   int nco, int nci, int total, int zfirst) {
    __shared__ __attribute__((aligned(16))) __bf16 xs[2][DW_ROWS][16];
    __shared__ __attribute__((aligned(16))) __bf16 ys[2][NC][32][16];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, q = lane >> 4;
    // each die takes a run of consecutive chunks, all channel groups of one next to each other: they share its L2
    const int g = (int)(blockIdx.x % NXCD) * (int)(gridDim.x / NXCD) + (int)(blockIdx.x / NXCD);
    if (g >= total) return;
    const int zc = zfirst + g / (nco * nci);
    const int co0 = (g % nco) * (16 * NC);
    const int ci0 = (g / nco % nci) * 16;
    const int K = 27 * cin;
    const long M = S.count();
    const long pbeg = (long)zc * chunk;
    const int npos = (int)((pbeg + chunk < M ? pbeg + chunk : M) - pbeg);
    const int ntile = (npos + 31) / 32;
    // the x window: position pbeg - lead is its start (before x's own start only where no item is valid)
    const long lead = (long)S.h * S.w + S.w + 1;
    const __bf16* const xwin = x + (pbeg - lead) * cin;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)xwin, 0, FAR ? 0 : (int)dw_window(S, cin, chunk), 0x00027000);
    const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc((void*)(dy + pbeg * cout), 0, FAR ? 0 : npos * cout * 2, 0x00027000);
    // this lane's x items of octet wv: item u = lane + 64 v: channels 8 (u % 2) .. of row u / 2 = (dz, dy) x (x - 1 .. x + 8)
    constexpr int NX = 3;
    unsigned req[NX], xo[NX];
    long xl[NX];
    int xrow[NX];
#pragma unroll
    for (int v = 0; v < NX; ++v) {
        const int u = lane + 64 * v, row = u >> 1, e = row / 10, c = row % 10;
        const int dz = e / 3 - 1, dyy = e % 3 - 1, ci = ci0 + 8 * (u & 1);
        // conditions on the octet: 0 y > 0, 1 y < h - 1, 2 z > 0, 3 z < d - 1, 4 x > 0, 5 x + 8 < w, 6 in the chunk, 7 never
        req[v] = (dyy < 0 ? 1u : dyy > 0 ? 2u : 0u) | (dz < 0 ? 4u : dz > 0 ? 8u : 0u) | (c == 0 ? 16u : c == 9 ? 32u : 0u) |
                 64u | (u < 180 && ci < cin ? 0u : 128u);
        xl[v] = (lead + 8 * wv + ((long)dz * S.h + dyy) * S.w + c - 1) * cin + ci;   // elements from the window's start
        xo[v] = (unsigned)(2 * xl[v]);
        xrow[v] = min(e, 8) * 40 + wv * 10 + c;
    }
    int ox, oy, oz;   // the octet's coordinates
    {
        int t = (int)(pbeg + 8 * wv);   // (positions are below 2^31: 32-bit decode)
        ox = t % S.w;
        t /= S.w;
        oy = t % S.h;
        t /= S.h;
        oz = t % S.d;
    }
    const int ax = 32 % S.w, ay = (32 / S.w) % S.h, az = (32 / S.w) / S.h % S.d;   // 32 positions on: one carry an axis
    const int yc = tid % (2 * NC), yp = tid / (2 * NC);   // dy item: channels 8 yc .. of position yp
    const bool yact = tid < 64 * NC;
    const unsigned yo = yact && co0 + 8 * yc < cout ? 2u * (unsigned)(yp * cout + co0 + 8 * yc) : NOWHERE;
    auto load = [&](int it, u32x4& ra, u32x4 (&rb)[NX]) {
        const unsigned have = (oy > 0 ? 1u : 0u) | (oy < S.h - 1 ? 2u : 0u) | (oz > 0 ? 4u : 0u) | (oz < S.d - 1 ? 8u : 0u) |
                              (ox > 0 ? 16u : 0u) | (ox + 8 < S.w ? 32u : 0u) | (32 * it + 8 * wv < npos ? 64u : 0u);
        if constexpr (FAR) {
            const u32x4 none = {};
            ra = yo != NOWHERE && 32 * it + yp < npos
                     ? *(const u32x4*)(dy + (pbeg + 32L * it + yp) * cout + co0 + 8 * yc) : none;
#pragma unroll
            for (int v = 0; v < NX; ++v) rb[v] = (req[v] & ~have) == 0 ? *(const u32x4*)(xwin + xl[v] + 32L * it * cin) : none;
        } else {
            ra = __builtin_amdgcn_raw_buffer_load_b128(yr, (int)(32 * it + yp < npos ? yo : NOWHERE), 64 * it * cout, 0);
#pragma unroll
            for (int v = 0; v < NX; ++v)
                rb[v] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)((req[v] & ~have) == 0 ? xo[v] : NOWHERE), 64 * it * cin, 0);
        }
        ox += ax;
        const int cx = ox >= S.w;
        ox -= cx ? S.w : 0;
        oy += ay + cx;
        const int cy = oy >= S.h;
        oy -= cy ? S.h : 0;
        oz += az + cy;
        oz -= oz >= S.d ? S.d : 0;
    };
    auto store = [&](int buf, const u32x4& ra, const u32x4 (&rb)[NX]) {
        if (yact) *(u32x4*)&ys[buf][yc >> 1][yp][8 * (yc & 1)] = ra;
#pragma unroll
        for (int v = 0; v < NX; ++v)
            if (lane + 64 * v < 180) *(u32x4*)&xs[buf][xrow[v]][8 * (lane & 1)] = rb[v];
    };
    f32x4 acc[NC][DW_OFF];
#pragma unroll
    for (int h = 0; h < NC; ++h)
#pragma unroll
        for (int o = 0; o < DW_OFF; ++o) acc[h][o] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int tr = r >> 2, tc = 4 * (r & 3);   // row and first channel this lane addresses in a transposing read
    int row[DW_OFF];
#pragma unroll
    for (int o = 0; o < DW_OFF; ++o) {
        const int off = min(wv * DW_OFF + o, 26);   // (the last wave's seventh is computed twice and not stored)
        row[o] = (off / 3) * 40 + off % 3 + 10 * q + tr;
    }
    // tile `it` is in buffer it % 2; its successor is already in one set of registers, and the loads of the one after
    // that go to the other set, so a load has two tiles of products to arrive
    u32x4 ra[2], rb[2][NX];
    auto step = [&](int it, int cur) {
        if (it + 2 < ntile) load(it + 2, ra[cur], rb[cur]);
        bf16x8 fa[NC], fb[DW_OFF];
#pragma unroll
        for (int h = 0; h < NC; ++h) fa[h] = read_transposed(&ys[cur][h][8 * q + tr][tc], &ys[cur][h][8 * q + 4 + tr][tc]);
#pragma unroll
        for (int o = 0; o < DW_OFF; ++o) fb[o] = read_transposed(&xs[cur][row[o]][tc], &xs[cur][row[o] + 4][tc]);
#pragma unroll
        for (int o = 0; o < DW_OFF; ++o)
#pragma unroll
            for (int h = 0; h < NC; ++h) acc[h][o] = mfma(fa[h], fb[o], acc[h][o]);
        if (it + 1 < ntile) store(cur ^ 1, ra[cur ^ 1], rb[cur ^ 1]);
        __syncthreads();
    };
    if (ntile > 0) load(0, ra[0], rb[0]);
    if (ntile > 1) load(1, ra[1], rb[1]);
    if (ntile > 0) store(0, ra[0], rb[0]);
    __syncthreads();
    int it = 0;
    for (; it + 1 < ntile; it += 2) {
        step(it, 0);
        step(it + 1, 1);
    }
    if (it < ntile) step(it, 0);
    const int ci = ci0 + r;
    if (ci >= cin) return;
#pragma unroll
    for (int o = 0; o < DW_OFF; ++o) {
        const int off = wv * DW_OFF + o;
        if (off >= 27) continue;
        const int kcol = off * cin + ci;
#pragma unroll
        for (int h = 0; h < NC; ++h)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int co = co0 + h * 16 + q * 4 + t;
                if (co >= cout) continue;
                if (ORDERED)
                    dw[((long)zc * cout + co) * K + kcol] = acc[h][o][t];
                else
                    atomicAdd(&dw[(long)co * K + kcol], acc[h][o][t]);
            }
    }
}
// Output channels per work-group: 32 (fewer fragment reads per product) where that leaves a work-group for each of the
// 256 compute units, else 16.  Measured, 32 against 16: 4 x 32^3 64 -> 64 (256 work-groups of 32) 88 / 101 us, 4 x 16^3
// 256 -> 128 (256) 83 / 86, 4 x 64^3 32 -> 32 (512) 154 / 188; 4 x 32^3 32 -> 64 (128) 76 / 70, 4 x 16^3 128 -> 128
// (128) 70 / 64, 4 x 8^3 256 -> 256 (128) 44 / 41.  (64 channels: within 2 % at best, 190 at 4 x 64^3 32 -> 32.)
template <bool ORDERED>
void launch_conv_dw(const void* x, const void* dy, float* dw, const Shape& S, int cin, int cout, long chunk, hipStream_t st) {
    const long nz = (S.count() + chunk - 1) / chunk, ny = (cin + 15) / 16;
    const int nc = cout > 16 && (cout + 31) / 32 * ny * nz >= 256 ? 2 : 1;
    const bool far = dw_window(S, cin, chunk) >= (1L << 31) || chunk * cout * 2 >= (1L << 31);
    const auto kern = far ? k_conv_dw<ORDERED, 1, true> : nc == 2 ? k_conv_dw<ORDERED, 2, false> : k_conv_dw<ORDERED, 1, false>;
    const long nco = (cout + 16 * (far ? 1 : nc) - 1) / (16 * (far ? 1 : nc));
    // a launch has less than 2^32 threads: beyond 2^24 work-groups the chunks take several (any weight matrix that fits the
    // memory has fewer than 2^24 channel groups)
    const long zper = std::max(1L, ((1L << 24) - NXCD) / (nco * ny));
    for (long z0 = 0; z0 < nz; z0 += zper) {
        const long total = nco * ny * std::min(zper, nz - z0);
        hipLaunchKernelGGL(kern, dim3((unsigned)((total + NXCD - 1) / NXCD * NXCD)), dim3(NT), 0, st, (const __bf16*)x,
                           (const __bf16*)dy, dw, S, cin, cout, chunk, (int)nco, (int)ny, (int)total, (int)z0);
    }
}

// positions per chunk of the weight- and bias-gradient sums
constexpr long DW_CHUNK = 4096, DB_CHUNK = 8192;

// bias gradient: db[co] += sum over positions of dy[p][co].  A work-group sums a chunk of 32 channels as eight partial
// sums over every eighth position, added in order; ORDERED: the chunk's sum is stored to db[chunk * cout + co], else
// every partial sum is added to db[co].  The positions come 256 at a time through LDS, 16 bytes a load and the next
// tile's loads in flight, and each thread adds its 32 from there: one 2-byte load per addition had the additions wait
// for memory one after the other (4 x 32^3, 64 channels: 250 us, 26 us so).
constexpr int DB_TILE = 256, DB_LD = 40;   // positions a tile; LDS row (32 channels + 8)
template <bool ORDERED>
__global__ void __launch_bounds__(NT) k_bias_grad(const __bf16* __restrict__ dy, float* __restrict__ db, long M, int cout,
                                                  long chunk) {
    __shared__ __attribute__((aligned(16))) __bf16 tile[2][DB_TILE][DB_LD];
    __shared__ float part[NT];
    const int tid = threadIdx.x, cl = tid % 32, lane_p = tid / 32;
    const int c0 = blockIdx.y * 32, co = cl + c0;
    const long pbeg = (long)blockIdx.x * chunk;
    const int npos = (int)((pbeg + chunk < M ? pbeg + chunk : M) - pbeg);
    const int ntile = (npos + DB_TILE - 1) / DB_TILE;
    const bf16x8 zero = {};
    // load v of this thread: channels 8 (tid % 4) .. of position tid / 4 + 64 v (cout is a multiple of 8)
    const int lc = 8 * (tid % 4), lp = tid / 4;
    const bool chan = c0 + lc < cout;
    const __bf16* const src = dy + (pbeg + lp) * cout + c0 + lc;
    auto load = [&](int t, bf16x8 (&r)[4]) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int p = t * DB_TILE + lp + 64 * v;
            r[v] = zero;
            if (chan && p < npos) r[v] = *(const bf16x8*)(src + ((long)t * DB_TILE + 64 * v) * cout);
        }
    };
    auto store = [&](int buf, const bf16x8 (&r)[4]) {
#pragma unroll
        for (int v = 0; v < 4; ++v) *(bf16x8*)&tile[buf][lp + 64 * v][lc] = r[v];
    };
    float s = 0.f;
    bf16x8 reg[4];
    load(0, reg);
    store(0, reg);
    __syncthreads();
    for (int t = 0; t < ntile; ++t) {
        const bool more = t + 1 < ntile;
        if (more) load(t + 1, reg);
        const int n = min(DB_TILE, npos - t * DB_TILE);
        if (n == DB_TILE) {
#pragma unroll
            for (int k = 0; k < DB_TILE / 8; ++k) s += bf2f(tile[t & 1][lane_p + 8 * k][cl]);
        } else {
            for (int p = lane_p; p < n; p += 8) s += bf2f(tile[t & 1][p][cl]);
        }
        if (more) store((t + 1) & 1, reg);
        __syncthreads();
    }
    if (!ORDERED) {
        if (co < cout) atomicAdd(&db[co], s);
        return;
    }
    part[tid] = s;
    __syncthreads();
    if (lane_p == 0 && co < cout) {
        float t = part[tid];
        for (int k = 1; k < NT / 32; ++k) t += part[tid + 32 * k];
        db[(long)blockIdx.x * cout + co] = t;
    }
}
// out[e] += sum over z = 0 .. nz-1 of part[z * ne + e], in that order.  The loads of 16 slices are issued together
// (one after the other the sum waited for each: 19 us on average over a training step's layers, 6 us so).
__global__ void __launch_bounds__(NT) k_sum_slices(const float* __restrict__ part, float* __restrict__ out, long ne, int nz) {
    const long e = (long)blockIdx.x * NT + threadIdx.x;
    if (e >= ne) return;
    float s = 0.f;
    int z = 0;
    for (; z + 16 <= nz; z += 16) {
        float v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = part[(long)(z + k) * ne + e];
#pragma unroll
        for (int k = 0; k < 16; ++k) s += v[k];
    }
    for (; z < nz; ++z) s += part[(long)z * ne + e];
    out[e] += s;
}

// Elementwise kernels: V = 8 consecutive values per thread (16-byte accesses; the launchers take it where the channel
// count or length is a multiple of 8 and every tensor starts on 16 bytes), else V = 1.  Bound by HBM; one 2-byte value per
// thread was bound by the number of accesses instead (ReLU gradient, mean over the layers of a training step: 23 us, 13 us so; addition 29 and 15).
template <int V>
struct alignas(2 * V) Pack {
    __bf16 v[V];
};
template <int V>
__global__ void k_relu_bwd(__bf16* __restrict__ g, const __bf16* __restrict__ y, long n) {
    const long i = (long)blockIdx.x * NT + threadIdx.x;
    if (i * V >= n) return;
    Pack<V> a = ((const Pack<V>*)g)[i];
    const Pack<V> b = ((const Pack<V>*)y)[i];
#pragma unroll
    for (int k = 0; k < V; ++k)
        if (!(bf2f(b.v[k]) > 0.f)) a.v[k] = f2bf(0.f);
    ((Pack<V>*)g)[i] = a;
}

// 2x average pooling (fine shape S, coarse S/2) and its adjoint; nearest 2x upsampling and its adjoint.  One thread per
// V channels of a coarse position, c counted in units of V.
template <int V>
__device__ __forceinline__ bool coarse_at(const Shape& S, int c, long& i, long (&fine)[8]) {
    i = (long)blockIdx.x * NT + threadIdx.x;
    const int D = S.d / 2, H = S.h / 2, W = S.w / 2;
    if (i >= (long)S.n * D * H * W * c) return false;
    const int ch = (int)(i % c);
    long t = i / c;
    const int xx = (int)(t % W);
    t /= W;
    const int yy = (int)(t % H);
    t /= H;
    const int zz = (int)(t % D);
    const int nn = (int)(t / D);
#pragma unroll
    for (int o = 0; o < 8; ++o)
        fine[o] = ((((long)nn * S.d + 2 * zz + (o >> 2)) * S.h + 2 * yy + ((o >> 1) & 1)) * S.w + 2 * xx + (o & 1)) * c + ch;
    return true;
}
// SUM: the sum of the fine values (scaled by 1/8 as pooling, unscaled as the upsampling's adjoint); else each fine value
// takes the coarse one (scaled by 1/8 as the pooling's adjoint)
template <int V, bool SUM, bool EIGHTH>
__global__ void k_coarse(const __bf16* __restrict__ x, __bf16* __restrict__ y, Shape S, int c) {
    long i, f[8];
    if (!coarse_at<V>(S, c, i, f)) return;
    const Pack<V>* const X = (const Pack<V>*)x;
    Pack<V>* const Y = (Pack<V>*)y;
    if (SUM) {
        Pack<V> a[8], r;
#pragma unroll
        for (int o = 0; o < 8; ++o) a[o] = X[f[o]];
#pragma unroll
        for (int k = 0; k < V; ++k) {
            float s = 0.f;
#pragma unroll
            for (int o = 0; o < 8; ++o) s += bf2f(a[o].v[k]);
            r.v[k] = f2bf(EIGHTH ? 0.125f * s : s);
        }
        Y[i] = r;
    } else {
        Pack<V> a = X[i];
        if (EIGHTH) {
#pragma unroll
            for (int k = 0; k < V; ++k) a.v[k] = f2bf(0.125f * bf2f(a.v[k]));
        }
#pragma unroll
        for (int o = 0; o < 8; ++o) Y[f[o]] = a;
    }
}
template <int V>
__global__ void k_add(const __bf16* __restrict__ a, const __bf16* __restrict__ b, __bf16* __restrict__ y, long n) {
    const long i = (long)blockIdx.x * NT + threadIdx.x;
    if (i * V >= n) return;
    const Pack<V> u = ((const Pack<V>*)a)[i], w = ((const Pack<V>*)b)[i];
    Pack<V> r;
#pragma unroll
    for (int k = 0; k < V; ++k) r.v[k] = f2bf(bf2f(u.v[k]) + bf2f(w.v[k]));
    ((Pack<V>*)y)[i] = r;
}
// mean squared error over the first `used` of `c` channels; writes the gradient (BF16) and adds the sum of
// squares to *loss (FP32).  At most MSE_BLOCKS work-groups walk the tensor: one atomic addition to the one address per
// 256 values took 420 us of a training step (4 x 64^3 x 8), 23 us so.
constexpr int MSE_BLOCKS = 1024;
template <int V>
__global__ void __launch_bounds__(NT) k_mse(const __bf16* __restrict__ y, const __bf16* __restrict__ t,
                                            __bf16* __restrict__ g, float* __restrict__ loss, long n, int c, int used,
                                            float scale) {
    __shared__ float red[NT];
    float s = 0.f;
    for (long i = (long)blockIdx.x * NT + threadIdx.x; i * V < n; i += (long)gridDim.x * NT) {
        const Pack<V> a = ((const Pack<V>*)y)[i], b = ((const Pack<V>*)t)[i];
        Pack<V> r;
        const int ch = (int)(i * V % c);
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const float d = ch + k < used ? bf2f(a.v[k]) - bf2f(b.v[k]) : 0.f;
            r.v[k] = f2bf(2.f * scale * d);
            s += d * d;
        }
        ((Pack<V>*)g)[i] = r;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = NT / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(loss, red[0]);
}
// Adam on FP32 master weights (bias-corrected, Kingma & Ba 2015)
__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       long n, float lr, float b1, float b2, float eps, float c1, float c2) {
    const long i = (long)blockIdx.x * NT + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}
// FP32 master weights w[co][27 cin] -> BF16 forward rows wf[co][kpad] and the flipped, transposed rows of the
// input-gradient convolution wb[ci][kpadb] (wb[ci][off' cout + co] = w[co][(26 - off') cin + ci])
__global__ void k_weights(const float* __restrict__ w, __bf16* __restrict__ wf, __bf16* __restrict__ wb, int cin,
                          int cout, int kpad, int kpadb) {
    const long i = (long)blockIdx.x * NT + threadIdx.x;
    const long nf = (long)cout * kpad, nb = (long)cin * kpadb;
    if (i < nf) {
        const int co = (int)(i / kpad), k = (int)(i % kpad);
        wf[i] = f2bf(k < 27 * cin ? w[(long)co * 27 * cin + k] : 0.f);
    }
    if (wb && i < nb) {
        const int ci = (int)(i / kpadb), k = (int)(i % kpadb);
        float v = 0.f;
        if (k < 27 * cout) {
            const int off = k / cout, co = k % cout;
            v = w[(long)co * 27 * cin + (26 - off) * cin + ci];
        }
        wb[i] = f2bf(v);
    }
}

inline unsigned blocks(long n) { return (unsigned)((n + NT - 1) / NT); }
inline int launched(hipStream_t) {
    return hipGetLastError() == hipSuccess ? MFLBM_OK : MFLBM_ERR_HIP;
}
inline int kpad_of(int cin) { return (27 * cin + 31) / 32 * 32; }

}  // namespace

extern "C" int mflbm_nn_mfma_probe(const void* a, const void* b, float* d, void* stream) {
    hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, (hipStream_t)stream, (const __bf16*)a, (const __bf16*)b, d);
    return launched((hipStream_t)stream);
}

namespace {
// Estimated us of the two forward kernels: the latency of a work-group, which grows with the input channels, or, with more
// work-groups than the device holds, so many times it; in whole rounds where a compute unit holds one work-group.
// Fitted to both kernels' times over 240 shapes (sides 1 to 256, 1 to 512 images, 8 to 264 channels in, 8 to 256 out): the
// kernel that the estimates prefer is within 2 % of the faster one on each, and on 117 random shapes beside them within 3 %
// but for three of 10 to 17 us (at most 1.4 us).
// k_conv_fwd: 128 positions x 32 channels a work-group; along an axis one node long a third of the offsets is inside,
// and a wave skips the loads of the others.
double untiled_us(const Shape& S, int cin, int cout) {
    const double thin = (S.d == 1 ? 1.0 / 3 : 1.0) * (S.h == 1 ? 1.0 / 3 : 1.0) * (S.w == 1 ? 1.0 / 3 : 1.0);
    const double rounds = (double)((S.count() + 127) / 128) * ((cout + 31) / 32) / 256;
    const double latency = 0.45 * cin * (cin >= 64 ? 1 + cin / 1024.0 * std::min(1.0, rounds) : 1.0);
    const double round = cin >= 64 ? 0.37 * cin * std::ceil(rounds) : (cin >= 32 ? 0.23 : 0.4) * cin * rounds;
    return std::max(4.5 + latency * (0.7 + 0.3 * thin), round * (0.5 + 0.5 * thin));
}
// k_conv_tile: whole tiles, however much of them lies in the domain; base and per: us of a work-group and per input channel
template <int MT, int NCO, int WP, int WC, int TZ, int TY, int TX, int KG>
double tile_us(const Shape& S, int cin, int cout, double base, double per, double in_flight) {
    using T = ConvTile<MT, NCO, WP, WC, TZ, TY, TX, KG>;
    const double groups = (double)S.n * ((S.d + TZ - 1) / TZ) * ((S.h + TY - 1) / TY) * ((S.w + TX - 1) / TX) * ((cout + T::CO - 1) / T::CO);
    if ((groups + NXCD) * T::THREADS >= 4294967296.0) return HUGE_VAL;   // a launch has less than 2^32 threads
    const double rounds = std::max(1.0, groups / in_flight);
    return (base + per * cin) * (in_flight == 256 ? std::ceil(rounds) : rounds);
}
}  // namespace

extern "C" int mflbm_nn_conv3d_fwd(const void* x, const void* wf, const float* bias, void* y, int32_t n, int32_t d,
                                   int32_t h, int32_t w, int32_t cin, int32_t cout, int32_t relu, void* stream) {
    if (!x || !wf || !y || n < 1 || d < 1 || h < 1 || w < 1 || cin < 8 || cin % 8 || cout < 1) return MFLBM_ERR_ARG;
    const Shape S{n, d, h, w};
    const long M = S.count();
    hipStream_t st = (hipStream_t)stream;
    const int kp = kpad_of(cin);
    // Tile by channels (the tile of all cin channels, up to 256 of them, in the 160 KB of LDS) and by the number of
    // work-groups: the large tiles read less halo and fewer fragments per product, but need 256 work-groups to use every
    // compute unit.  Without the tile: more than 256 input channels, planes beyond a 2 GiB window, and domains that fill so
    // little of their tiles that the whole tiles would take longer than k_conv_fwd, which pays for no position outside the
    // domain.  us tiled / untiled: 1 x 1 x 256 x 256 32 -> 32 29 / 18, 256 -> 256 3491 / 1017, 4 x 1 x 64 x 64 64 -> 64
    // 39 / 27, 512 x 1 x 1 x 1 64 -> 64 71 / 25, 8 x 9^3 256 -> 256 219 / 182; but 16 x 1 x 1 x 64 64 -> 64 20 / 25, 4 x 4^3
    // 256 -> 256 56 / 118, 4 x 64 x 3 x 16 128 -> 128 34 / 89.
    if (cin <= 256 && 10L * h * w * cin * 2 < (1L << 31) && (long)cout * kp * 2 < (1L << 31)) {
        const double tu = untiled_us(S, cin, cout);
        const long tiles8 = (long)n * ((d + 7) / 8) * ((h + 7) / 8) * ((w + 7) / 8);   // 8 x 8 x 8 tiles
        // BASE, PER, FLIGHT: tile_us; then fragments of positions and of channels, waves along positions and channels, tile,
        // steps per weight stage
#define TILE_US(BASE, PER, FLIGHT, ...) tile_us<__VA_ARGS__>(S, cin, cout, BASE, PER, FLIGHT)
#define TILE(BASE, PER, FLIGHT, ...) \
    if (TILE_US(BASE, PER, FLIGHT, __VA_ARGS__) <= tu) return launch_conv_tile<__VA_ARGS__>(x, wf, bias, y, S, (int)cin, (int)cout, kp, (int)relu, st)
#define TILES(BIG, SMALL) \
    if (tiles8 * ((cout + 63) / 64) >= 256 && TILE_US BIG <= TILE_US SMALL) { TILE BIG; } else { TILE SMALL; }
        if (cin <= 32) {   // 4 x 64^3, us before / after: 8 -> 32 75 / 44, 32 -> 8 196 / 85, 32 -> 32 254 / 116, 32 -> 64 483 / 175
            if (cout <= 16) { TILE(4, 0.15, 300, 2, 1, 8, 1, 4, 8, 8, 8); }
            else if (cout > 32) { TILE(7, 0.29, 400, 4, 4, 4, 1, 4, 8, 8, 1); }
            else if (cin <= 16) { TILE(4, 0.19, 400, 4, 2, 4, 1, 4, 8, 8, 4); }
            else { TILE(4, 0.22, 370, 2, 2, 8, 1, 4, 8, 8, 4); }
        } else if (cin <= 64) {   // 4 x 64^3 64 -> 32 782 / 204; 4 x 32^3 64 -> 64 206 / 46 (61 in the small tile); 4 x 16^3 64 -> 128 52 / 23 (40 in the large)
            if (cout <= 32) { TILES((4, 0.33, 256, 4, 2, 8, 1, 8, 8, 8, 4), (4, 0.24, 256, 2, 2, 8, 1, 4, 8, 8, 4)) }
            else { TILES((4, 0.55, 256, 4, 4, 8, 1, 8, 8, 8, 2), (4, 0.25, 256, 2, 2, 4, 2, 4, 4, 8, 4)) }
        } else if (cin <= 128) {   // 4 x 16^3 128 -> 128 100 / 36, 4 x 32^3 128 -> 64 400 / 139
            TILE(4, 0.22, 256, 2, 2, 4, 2, 4, 4, 8, 8);
        } else {   // 4 x 8^3 256 -> 256 125 / 57, 4 x 16^3 256 -> 128 195 / 118
            TILE(4, 0.2, 256, 1, 2, 4, 2, 4, 4, 4, 4);
        }
#undef TILES
#undef TILE
#undef TILE_US
    }
    const dim3 grid((unsigned)((M + 127) / 128), (unsigned)((cout + 31) / 32));
    if (relu)
        hipLaunchKernelGGL(k_conv_fwd<1>, grid, dim3(NT), 0, (hipStream_t)stream, (const __bf16*)x, (const __bf16*)wf,
                           bias, (__bf16*)y, S, (int)cin, (int)cout, kpad_of(cin));
    else
        hipLaunchKernelGGL(k_conv_fwd<0>, grid, dim3(NT), 0, (hipStream_t)stream, (const __bf16*)x, (const __bf16*)wf,
                           bias, (__bf16*)y, S, (int)cin, (int)cout, kpad_of(cin));
    return launched((hipStream_t)stream);
}

extern "C" int mflbm_nn_conv3d_dw(const void* x, const void* dy, float* dw, float* dbias, int32_t n, int32_t d, int32_t h,
                                  int32_t w, int32_t cin, int32_t cout, void* stream) {
    if (!x || !dy || !dw || n < 1 || d < 1 || h < 1 || w < 8 || w % 8 || cin < 8 || cin % 8 || cout < 8 || cout % 8 ||
        (long)n * d * h * w >= (1L << 31))
        return MFLBM_ERR_ARG;
    const Shape S{n, d, h, w};
    const long M = S.count();
    launch_conv_dw<false>(x, dy, dw, S, cin, cout, DW_CHUNK, (hipStream_t)stream);
    if (dbias)
        hipLaunchKernelGGL(k_bias_grad<false>, dim3((unsigned)((M + DB_CHUNK - 1) / DB_CHUNK), (unsigned)((cout + 31) / 32)),
                           dim3(NT), 0, (hipStream_t)stream, (const __bf16*)dy, dbias, M, (int)cout, DB_CHUNK);
    return launched((hipStream_t)stream);
}

extern "C" int64_t mflbm_nn_conv3d_dw_work(int32_t n, int32_t d, int32_t h, int32_t w, int32_t cin, int32_t cout) {
    if (n < 1 || d < 1 || h < 1 || w < 1 || cin < 1 || cout < 1) return -1;
    const long M = (long)n * d * h * w;
    return ((M + DW_CHUNK - 1) / DW_CHUNK) * cout * 27L * cin + ((M + DB_CHUNK - 1) / DB_CHUNK) * cout;
}

namespace {

// The launches of the fixed-order weight and bias gradients on a workspace of at least
// mflbm_nn_conv3d_dw_work(...) floats.  Every workspace element the sums read is written first by the same
// call (each chunk slice of the weight and bias partials is stored whole), so the workspace needs no clearing.
int dw_ordered_launch(const void* x, const void* dy, float* dw, float* dbias, float* work, const Shape& S, int cin,
                      int cout, hipStream_t st) {
    const long M = S.count();
    const long K = 27L * cin, nzw = (M + DW_CHUNK - 1) / DW_CHUNK, nzb = (M + DB_CHUNK - 1) / DB_CHUNK;
    float* bpart = work + nzw * cout * K;
    launch_conv_dw<true>(x, dy, work, S, cin, cout, DW_CHUNK, st);
    hipLaunchKernelGGL(k_sum_slices, dim3((unsigned)((cout * K + NT - 1) / NT)), dim3(NT), 0, st, (const float*)work, dw,
                       cout * K, (int)nzw);
    if (dbias) {
        hipLaunchKernelGGL(k_bias_grad<true>, dim3((unsigned)nzb, (unsigned)((cout + 31) / 32)), dim3(NT), 0, st,
                           (const __bf16*)dy, bpart, M, (int)cout, DB_CHUNK);
        hipLaunchKernelGGL(k_sum_slices, dim3((unsigned)((cout + NT - 1) / NT)), dim3(NT), 0, st, (const float*)bpart, dbias,
                           (long)cout, (int)nzb);
    }
    return launched(st);
}

// Workspace of the allocation-free weight gradient: one array per GPU in the library's code object, held until
// the process ends.  Host code never passes its name to a kernel (on the host it is a stand-in, not a device
// address): the device address of each GPU's copy comes from hipGetSymbolAddress once per device, with that
// device current, and only that address is used.
constexpr long DW_SCRATCH_FLOATS = 4L << 20;   // 16 MiB
static __device__ __align__(256) float scratch[DW_SCRATCH_FLOATS];

constexpr int MAX_DEVICES = 64;
std::mutex scratch_mutex;
float* scratch_ptr[MAX_DEVICES] = {};

// the current device's scratch address, resolved on the first call on that device
int scratch_of_current_device(float** out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) return MFLBM_ERR_NODEV;
    if (dev < 0 || dev >= MAX_DEVICES) return MFLBM_ERR_ARG;
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return MFLBM_ERR_HIP;
        scratch_ptr[dev] = (float*)p;
    }
    *out = scratch_ptr[dev];
    return MFLBM_OK;
}

bool dw_args_ok(const void* x, const void* dy, const float* dw, int32_t n, int32_t d, int32_t h, int32_t w, int32_t cin,
                int32_t cout) {
    return x && dy && dw && n >= 1 && d >= 1 && h >= 1 && w >= 8 && w % 8 == 0 && cin >= 8 && cin % 8 == 0 && cout >= 8 &&
           cout % 8 == 0 && (long)n * d * h * w < (1L << 31);
}

}  // namespace

extern "C" int mflbm_nn_conv3d_dw_ordered(const void* x, const void* dy, float* dw, float* dbias, float* work,
                                          int64_t work_floats, int32_t n, int32_t d, int32_t h, int32_t w, int32_t cin,
                                          int32_t cout, void* stream) {
    if (!work || !dw_args_ok(x, dy, dw, n, d, h, w, cin, cout)) return MFLBM_ERR_ARG;
    if (work_floats < mflbm_nn_conv3d_dw_work(n, d, h, w, cin, cout)) return MFLBM_ERR_ARG;
    return dw_ordered_launch(x, dy, dw, dbias, work, Shape{n, d, h, w}, cin, cout, (hipStream_t)stream);
}

extern "C" int64_t mflbm_nn_conv3d_dw_scratch_floats(void) { return DW_SCRATCH_FLOATS; }

extern "C" int mflbm_nn_conv3d_dw_ordered_noalloc(const void* x, const void* dy, float* dw, float* dbias, int32_t n,
                                                  int32_t d, int32_t h, int32_t w, int32_t cin, int32_t cout,
                                                  void* stream) {
    if (!dw_args_ok(x, dy, dw, n, d, h, w, cin, cout)) return MFLBM_ERR_ARG;
    if (mflbm_nn_conv3d_dw_work(n, d, h, w, cin, cout) > DW_SCRATCH_FLOATS) return MFLBM_ERR_ARG;
    float* work = nullptr;
    const int rc = scratch_of_current_device(&work);
    if (rc) return rc;
    return dw_ordered_launch(x, dy, dw, dbias, work, Shape{n, d, h, w}, cin, cout, (hipStream_t)stream);
}

extern "C" int mflbm_nn_weights_to_bf16(const float* w, void* wf, void* wb, int32_t cin, int32_t cout, void* stream) {
    if (!w || !wf || cin < 1 || cout < 1) return MFLBM_ERR_ARG;
    const int kp = kpad_of(cin), kpb = kpad_of(cout);
    const long n = (long)cout * kp > (long)cin * kpb ? (long)cout * kp : (long)cin * kpb;
    hipLaunchKernelGGL(k_weights, dim3(blocks(n)), dim3(NT), 0, (hipStream_t)stream, w, (__bf16*)wf, (__bf16*)wb, (int)cin,
                       (int)cout, kp, kpb);
    return launched((hipStream_t)stream);
}

namespace {
// every tensor on a 16-byte boundary and the length (or channel count) whole packs of 8
template <class... P>
bool packs(long n, const P*... p) {
    return n % 8 == 0 && (... && (((uintptr_t)p & 15) == 0));
}
}  // namespace

extern "C" int mflbm_nn_relu_bwd(void* g, const void* y, int64_t n, void* stream) {
    if (!g || !y || n < 0) return MFLBM_ERR_ARG;
    const bool v = packs(n, (const char*)g, (const char*)y);
    if (n) hipLaunchKernelGGL(v ? k_relu_bwd<8> : k_relu_bwd<1>, dim3(blocks(v ? n / 8 : n)), dim3(NT), 0, (hipStream_t)stream,
                              (__bf16*)g, (const __bf16*)y, (long)n);
    return launched((hipStream_t)stream);
}

// Input features of the warm-start network: the fluid indicator, d / 8 and (d / 8)^2 with d the Euclidean
// distance from a node to the nearest solid node capped at 16, in channels 0..2 of a channels-last BF16 tensor.
// The squared distance is a separable minimum over offsets of at most 16 per axis (exact below the cap: the
// nearest solid within 16 lies inside that cube), wrapped along periodic axes and cut at the others.
constexpr int DCAP = 16;
constexpr int DBIG = 1 << 20;
__device__ __forceinline__ int wrap_or_cut(int a, int n, int per) { return per ? ((a % n) + n) % n : (a >= 0 && a < n ? a : -1); }
__global__ void k_dist_x(const int8_t* __restrict__ fluid, int* __restrict__ g, int d, int h, int w, int per) {
    const long t = (long)blockIdx.x * NT + threadIdx.x;
    if (t >= (long)d * h * w) return;
    const int x = (int)(t % w);
    const long row = t - x;
    int best = DBIG;
    for (int a = -DCAP; a <= DCAP; ++a) {
        const int xx = wrap_or_cut(x + a, w, per);
        if (xx >= 0 && fluid[row + xx] == 0) best = min(best, a * a);
    }
    g[t] = best;
}
__global__ void k_dist_y(const int* __restrict__ gin, int* __restrict__ gout, int d, int h, int w, int per) {
    const long t = (long)blockIdx.x * NT + threadIdx.x;
    if (t >= (long)d * h * w) return;
    const int x = (int)(t % w), y = (int)((t / w) % h);
    const long base = t - (long)y * w;
    int best = DBIG;
    for (int a = -DCAP; a <= DCAP; ++a) {
        const int yy = wrap_or_cut(y + a, h, per);
        if (yy >= 0) best = min(best, gin[base + (long)yy * w] + a * a);
    }
    gout[t] = best;
    (void)x;
}
__global__ void k_dist_z_features(const int8_t* __restrict__ fluid, const int* __restrict__ gin, __bf16* __restrict__ out,
                                  int d, int h, int w, int cin, int per) {
    const long t = (long)blockIdx.x * NT + threadIdx.x;
    const long plane = (long)h * w;
    if (t >= (long)d * plane) return;
    const int z = (int)(t / plane);
    const long base = t - (long)z * plane;
    int best = DBIG;
    for (int a = -DCAP; a <= DCAP; ++a) {
        const int zz = wrap_or_cut(z + a, d, per);
        if (zz >= 0) best = min(best, gin[base + (long)zz * plane] + a * a);
    }
    const double dist = fmin(sqrt((double)best), (double)DCAP) / 8.0;
    __bf16* o = out + t * cin;
    o[0] = f2bf((float)fluid[t]);
    o[1] = f2bf((float)dist);
    o[2] = f2bf((float)(dist * dist));
}
extern "C" int mflbm_nn_distance_features(const int8_t* fluid, int32_t* work, void* x, int32_t d, int32_t h, int32_t w,
                                          int32_t cin, int32_t zper, int32_t yper, int32_t xper, void* stream) {
    if (!fluid || !work || !x || d < 1 || h < 1 || w < 1 || cin < 3) return MFLBM_ERR_ARG;
    const long cnt = (long)d * h * w;
    hipStream_t st = (hipStream_t)stream;
    hipLaunchKernelGGL(k_dist_x, dim3(blocks(cnt)), dim3(NT), 0, st, fluid, (int*)work, (int)d, (int)h, (int)w, (int)xper);
    hipLaunchKernelGGL(k_dist_y, dim3(blocks(cnt)), dim3(NT), 0, st, (const int*)work, (int*)work + cnt, (int)d, (int)h,
                       (int)w, (int)yper);
    hipLaunchKernelGGL(k_dist_z_features, dim3(blocks(cnt)), dim3(NT), 0, st, fluid, (const int*)work + cnt, (__bf16*)x,
                       (int)d, (int)h, (int)w, (int)cin, (int)zper);
    return launched(st);
}

namespace {
template <bool SUM, bool EIGHTH>
int launch_coarse(const void* x, void* y, const Shape& S, int c, hipStream_t st) {
    const bool v = packs(c, (const char*)x, (const char*)y);
    const int cv = v ? c / 8 : c;
    const long cnt = (long)S.n * (S.d / 2) * (S.h / 2) * (S.w / 2) * cv;
    hipLaunchKernelGGL((v ? k_coarse<8, SUM, EIGHTH> : k_coarse<1, SUM, EIGHTH>), dim3(blocks(cnt)), dim3(NT), 0, st,
                       (const __bf16*)x, (__bf16*)y, S, cv);
    return launched(st);
}
}  // namespace

extern "C" int mflbm_nn_pool2(const void* x, void* y, int32_t n, int32_t d, int32_t h, int32_t w, int32_t c, int32_t bwd,
                              void* stream) {
    if (!x || !y || d % 2 || h % 2 || w % 2 || c < 1) return MFLBM_ERR_ARG;
    const Shape S{n, d, h, w};
    return bwd ? launch_coarse<false, true>(x, y, S, c, (hipStream_t)stream) : launch_coarse<true, true>(x, y, S, c, (hipStream_t)stream);
}

extern "C" int mflbm_nn_up2(const void* x, void* y, int32_t n, int32_t d, int32_t h, int32_t w, int32_t c, int32_t bwd,
                            void* stream) {
    if (!x || !y || d % 2 || h % 2 || w % 2 || c < 1) return MFLBM_ERR_ARG;
    const Shape S{n, d, h, w};
    return bwd ? launch_coarse<true, false>(x, y, S, c, (hipStream_t)stream) : launch_coarse<false, false>(x, y, S, c, (hipStream_t)stream);
}

extern "C" int mflbm_nn_add(const void* a, const void* b, void* y, int64_t n, void* stream) {
    if (!a || !b || !y || n < 0) return MFLBM_ERR_ARG;
    const bool v = packs(n, (const char*)a, (const char*)b, (const char*)y);
    if (n) hipLaunchKernelGGL(v ? k_add<8> : k_add<1>, dim3(blocks(v ? n / 8 : n)), dim3(NT), 0, (hipStream_t)stream,
                              (const __bf16*)a, (const __bf16*)b, (__bf16*)y, (long)n);
    return launched((hipStream_t)stream);
}

extern "C" int mflbm_nn_mse(const void* y, const void* t, void* g, float* loss, int64_t npos, int32_t c, int32_t used,
                            float scale, void* stream) {
    if (!y || !t || !g || !loss || npos < 0 || c < 1 || used < 0 || used > c) return MFLBM_ERR_ARG;
    const long n = (long)npos * c;
    const bool v = packs(c, (const char*)y, (const char*)t, (const char*)g);
    const unsigned nb = blocks(v ? n / 8 : n);
    if (n) hipLaunchKernelGGL(v ? k_mse<8> : k_mse<1>, dim3(nb < MSE_BLOCKS ? nb : MSE_BLOCKS), dim3(NT), 0, (hipStream_t)stream,
                              (const __bf16*)y, (const __bf16*)t, (__bf16*)g, loss, n, (int)c, (int)used, scale);
    return launched((hipStream_t)stream);
}

extern "C" int mflbm_nn_adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2,
                             float eps, int32_t step, void* stream) {
    if (!w || !g || !m || !v || n < 0 || step < 1) return MFLBM_ERR_ARG;
    float c1 = 1.f, c2 = 1.f;
    for (int s = 0; s < step; ++s) {
        c1 *= b1;
        c2 *= b2;
    }
    if (n) hipLaunchKernelGGL(k_adam, dim3(blocks(n)), dim3(NT), 0, (hipStream_t)stream, w, g, m, v, (long)n, lr, b1, b2,
                              eps, 1.f - c1, 1.f - c2);
    return launched((hipStream_t)stream);
}
