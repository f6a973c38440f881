// Pieces shared by the two-phase and the single-phase gfx950 paths: the padded dense layout, the compact
// node set the populations are stored on, the XCD-aware block order, host-side halo packing and the error
// plumbing of the C ABI.
//
// Dense layout (every dense field: phase field, normals, walls, macroscopic fields):
//
//   offset(i, j, k) = (i + XO) + (j + YO) * px + (k + ZO) * px * py      (1-based interior indices)
//
// with XO = 15 so that i = 1 sits on a 128-byte boundary, px = round_up(nx + 20, 16), py = ny + 8,
// pz = nz + 8 (at least the 4-layer halo of the phase field in every direction).
//
// Compact population storage: one slot per interior fluid node (compact indices [0, nf), x-fastest order)
// followed by the "support" nodes: every non-fluid node a fluid node reaches in one lattice link (solid
// neighbours, whose slots carry the wall reflection of the AA update, and halo nodes) and every node of the
// planes the boundary conditions and the periodic exchange address.  A dense int32 map gives the compact
// index of a padded offset (-1 where nothing is stored).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdlib>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "lattice.h"
#include "layout.h"
#include "mflbm.h"

namespace mflbm_dev {

constexpr int BLOCK = 256;
constexpr int NXCD = 8;   // gfx950: 8 accelerator complex dies, work-groups dispatched round-robin

// Logical block index with each XCD taking one contiguous range of blocks: node lists are in x-fastest
// order, so a die then works on a z-slab and stencil neighbours stay in its own L2.  The grid is launched
// as NXCD * per blocks.  (The lattice updates take update_block.)
__device__ __forceinline__ int xcd_block(int per) { return (int)(blockIdx.x % NXCD) * per + (int)(blockIdx.x / NXCD); }

// Logical block index of the lattice updates: the dies take runs of UPDATE_RUN consecutive blocks in turn.  In the odd
// step a slot line is shared by the rows its run boundaries fall on (neighbouring blocks) and read by the planes above
// and below (some 8 blocks on), so a run keeps most sharers on one die's L2, while all dies still stream one region.
// Odd step, us, runs of 1 / 8 / 16 / 32 / 128 blocks: two-phase 256^3 FP64 667 / 651 / 652 / 652 / 685, 160^3 FP32 89 / 85 /
// 86 / 83 / 88, single-phase 160^3 FP64 88 / 81 / 82 / 82 / 84 (whole eighths: 88), 125x131x119 FP32 21.7 / 19.8 / 19.4 /
// 19.6 / 20.1: 8 to 32 alike.  The even step shares nothing but finds in its die what the odd step left there (runs of 1 / 16):
// 538 / 525 us at 256^3, 61 / 60 and 12.5 / 11.8 us in the single-phase cases, 55 / 50 us for ten REVs.  The grid is update_grid(blocks).
constexpr int UPDATE_RUN = 16;
__device__ __forceinline__ int update_block() {
    const int x = (int)blockIdx.x % NXCD, i = (int)blockIdx.x / NXCD;
    return (i / UPDATE_RUN * NXCD + x) * UPDATE_RUN + i % UPDATE_RUN;
}
inline unsigned update_grid(long blocks) {
    return (unsigned)((blocks + NXCD * UPDATE_RUN - 1) / (NXCD * UPDATE_RUN) * (NXCD * UPDATE_RUN));
}
inline unsigned nblocks(long n) { return (unsigned)((n + BLOCK - 1) / BLOCK); }
// grid of a list kernel that uses xcd_block(): per = blocks per die
inline int xcd_per(long n) { return (int)((nblocks(n) + NXCD - 1) / NXCD); }

// link slot of fluid node x (compact index) in direction r, or -1 when x + e_r is a fluid node
__device__ __forceinline__ int link_slot(int nc, const int* wbase, const unsigned long long* wmask, int x, int r) {
    const int e = 18 * (x >> 6) + r - 1;
    const unsigned long long wm = wmask[e];
    const unsigned l = (unsigned)x & 63u;
    if (!((wm >> l) & 1ull)) return -1;
    return nc + wbase[e] + __popcll(wm & ((1ull << l) - 1ull));
}

// A pointer that a kernel read from memory is generic to the compiler: accesses through it are flat instructions with a
// 64-bit vector address each.  Named as global it takes the scalar-base form that a kernel argument gets by itself.
#define MFLBM_GLOBAL __attribute__((address_space(1)))

// The odd step's neighbour slots of fluid node m (compact index; m & 63 its lane, every lane of the wave in one link
// mask word) at dense offset n: per direction r, the index of the slot (x + e_r, opp(r)) in slice opp(r), which is
// the link slot of (m, r) where the wave's link mask has m's bit, else the compact index of the fluid node x + e_r.
// The wave-uniform masks and bases are scalar loads issued together; the eight row records around the node's own row
// (layout.h) are loaded unconditionally, all in flight at once (a conditional load per direction compiles to a branch
// that waits for every earlier load), and every fluid neighbour's index is its row's rank or one next to it.
__device__ __forceinline__ void odd_neighbour_slots(const RowRec* rows_, const Layout& L, int nc, const int* wbase_,
                                                    const unsigned long long* wmask_, int m, int n, unsigned nb[19]) {
    const MFLBM_GLOBAL long* const rows = (const MFLBM_GLOBAL long*)rows_;
    const MFLBM_GLOBAL int* const wbase = (const MFLBM_GLOBAL int*)wbase_;
    const MFLBM_GLOBAL unsigned long long* const wmask = (const MFLBM_GLOBAL unsigned long long*)wmask_;
    const int e0 = 18 * __builtin_amdgcn_readfirstlane(m >> 6) - 1;
    const unsigned lane = (unsigned)m & 63u;
    const unsigned long long below = (1ull << lane) - 1ull;
    const int g = n >> 4, sx = L.px >> 4, sxy = L.pxy >> 4;
    RowRec row[9];   // entry 3 (ez + 1) + ey + 1
#pragma unroll
    for (int k = 0; k < 9; ++k)
        if (k != 4) row[k] = __builtin_bit_cast(RowRec, rows[g + (k % 3 - 1) * sx + (k / 3 - 1) * sxy]);
#pragma unroll
    for (int r = 1; r < 19; ++r) {
        const int ex = lat::EX[r], k = 3 * (lat::EZ[r] + 1) + lat::EY[r] + 1;
        unsigned mv;
        if (k == 4) mv = (unsigned)(m + ex);
        else mv = row_rank(row[k], n) + (ex < 0 ? ~0u : ex > 0 ? row_fluid(row[k], n, 0) : 0u);
        const unsigned long long wm = wmask[e0 + r];
        const unsigned li = (unsigned)(nc + wbase[e0 + r]) + (unsigned)__popcll(wm & below);
        nb[r] = ((wm >> lane) & 1ull) ? li : mv;
    }
}

// Whether the even step of a state of these bytes (fluid nodes only; of a batch, those of the samples still running)
// reads and writes its slots non-temporally.  The
// even step touches every slot line once, whole: beyond what the 256 MB last-level cache keeps from step to step its
// lines only push out those that are read again (the odd step's shared lines, normals, phi, row records).  us per step
// (even and odd mean), cached / streamed: two-phase FP64 90 MB 71 / 77, 196 MB 137 / 130, 362 MB 247 / 211, 1349 MB
// 791 / 723; FP32 181 MB 185 / 172; single-phase FP64 98 MB 37 / 39, 181 MB 77 / 69, 674 MB 307 / 273; FP32 150 MB
// 54 / 61, 231 MB 110 / 95, 337 MB 159 / 140.  (The odd step's lines are shared by neighbouring rows: streamed loads
// took its 256^3 update from 689 to 923 us, streamed stores to 698.)
inline bool stream_even(long pop_bytes) { return pop_bytes > (160L << 20); }

// Slot access with a scalar slice base and a 32-bit per-lane byte offset (one global load/store with an SGPR
// base instead of a 64-bit vector address per slot); slices are kept below 2^32 bytes.
// STREAM: a non-temporal access, for the even step of a state that no cache holds (stream_even).
template <bool STREAM = false, class T>
__device__ __forceinline__ T slot_ld(const T* slice, unsigned i) {
    const MFLBM_GLOBAL T* const p = (const MFLBM_GLOBAL T*)((const MFLBM_GLOBAL char*)slice + i * (unsigned)sizeof(T));
    return STREAM ? __builtin_nontemporal_load(p) : *p;
}
template <bool STREAM = false, class T>
__device__ __forceinline__ void slot_st(T* slice, unsigned i, T v) {
    MFLBM_GLOBAL T* const p = (MFLBM_GLOBAL T*)((MFLBM_GLOBAL char*)slice + i * (unsigned)sizeof(T));
    if (STREAM) __builtin_nontemporal_store(v, p);
    else *p = v;
}
// Exchanged halo slots of a folded domain (layout.h, Fold): the halo slot (q, h) of a direction q that points
// into the domain along h's halo axes, and the slot (q, y) of h's image.  The reference's self-exchange leaves them
// equal after every step.
//   fold_exchanged: calls f(h, y, q) for each such pair of the one-layer halo node (i, j, k) (x interior).
//   k_fold_dense (downloads): the compact storage kept the value at y, except where y is not fluid and the
//     interior node x = h + e_q is: then it is x's link slot of direction opp(q), which the link download wrote
//     at h, and y takes it from there; and where y holds no slot at all (no step touches the pair, and the first
//     push exchange left (q, y) equal to the (q, h) the staging still holds).  One thread per node of the
//     one-layer halo box; `ncol` population sets of 19 arrays each in the dense staging.
template <class Fn>
__device__ __forceinline__ void fold_exchanged(const Layout& L, const Fold& F, long t, Fn&& f) {
    const long ny2 = L.ny + 2, nz2 = L.nz + 2;
    if (t >= (long)L.nx * ny2 * nz2) return;
    const int i = (int)(t % L.nx) + 1;
    const int j = (int)((t / L.nx) % ny2);
    const int k = (int)(t / ((long)L.nx * ny2));
    int y;
    if (!fold_image(L, F, i, j, k, y)) return;
    const int h = L.at(i, j, k);
    const bool gy = j == 0 || j == L.ny + 1, gz = k == 0 || k == L.nz + 1;
    const int ey = j == 0 ? 1 : -1, ez = k == 0 ? 1 : -1;
#pragma unroll
    for (int q = 1; q < 19; ++q) {
        if ((gy && lat::EY[q] != ey) || (gz && lat::EZ[q] != ez)) continue;
        f(h, y, q);
    }
}
inline unsigned fold_blocks(const Layout& L) { return nblocks((long)L.nx * (L.ny + 2) * (L.nz + 2)); }
static __global__ void k_fold_dense(Layout L, Fold F, const int* __restrict__ map, int nf, double* __restrict__ dense,
                                    long ps, int ncol) {
    fold_exchanged(L, F, (long)blockIdx.x * BLOCK + threadIdx.x, [&](int h, int y, int q) {
        const bool y_fluid = (unsigned)map[y] < (unsigned)nf;
        const int x = h + L.off(q);
        int xi, xj, xk;
        decode(L, x, xi, xj, xk);
        const bool x_inside = xi >= 1 && xi <= L.nx && xj >= 1 && xj <= L.ny && xk >= 1 && xk <= L.nz;
        const bool from_h = map[y] < 0 || (!y_fluid && x_inside && (unsigned)map[x] < (unsigned)nf);
        for (int c = 0; c < ncol; ++c) {
            double* a = dense + (long)(19 * c + q) * ps;
            if (from_h) a[y] = a[h];
            else a[h] = a[y];
        }
    });
}

// message of the last failed create call (contexts keep their own)
inline thread_local std::string g_create_error;

// record an error on a context (or, for a NULL context, as the create error) and return its code
inline int vfail(std::string* dst, int code, const char* fmt, va_list ap) {
    char buf[512];
    vsnprintf(buf, sizeof buf, fmt, ap);
    *(dst ? dst : &g_create_error) = buf;
    return code;
}
template <class Ctx>
int fail(Ctx* c, int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    const int r = vfail(c ? &c->err : nullptr, code, fmt, ap);
    va_end(ap);
    return r;
}
inline int fail(std::nullptr_t, int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    const int r = vfail(nullptr, code, fmt, ap);
    va_end(ap);
    return r;
}

}  // namespace mflbm_dev

#define HIPCHK(c, call)                                                                                      \
    do {                                                                                                     \
        hipError_t e_ = (call);                                                                              \
        if (e_ != hipSuccess) return fail((c), MFLBM_ERR_HIP, "%s failed: %s", #call, hipGetErrorString(e_)); \
    } while (0)

#define LAUNCH(c, kern, grid, ...)                                                                           \
    do {                                                                                                     \
        if ((grid) > 0) {                                                                                    \
            hipLaunchKernelGGL(kern, dim3(grid), dim3(BLOCK), 0, (c)->stream, __VA_ARGS__);                  \
            hipError_t e_ = hipGetLastError();                                                               \
            if (e_ != hipSuccess) return fail((c), MFLBM_ERR_HIP, "launch %s: %s", #kern, hipGetErrorString(e_)); \
        }                                                                                                    \
    } while (0)
