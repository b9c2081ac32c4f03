// Goldstein branch-cut unwrapping for gfx950, bit-exact with the host specification
// (reference cudaGoldsteinUnwrap2D, Goldstein.cu:5-50; residues :52-103, cuts :105-248, flood fill
// :263-641). Integer work throughout: residues int8, cuts uint8, 2*pi counts int32.
//
//   1. k_gs_residues  one thread per pixel: the reference's wrapped differences with its float /
//                     double promotions, summed in float, thresholded at +-6.
//   2. branch cuts, deterministic raster order (the reference runs its search for all residues
//      concurrently, which is racy; the raster order makes it reproducible): k_gs_pair (one workgroup per
//      map) pairs the residues, with rows side by side where no decision can reach another's (maps of few
//      columns: k_gs_walk, one residue after the other), and k_gs_draw draws the chosen cuts in parallel.
//   3. fill           a pixel's 2 pi count is the sum of the steps along the path by which a level-synchronous
//                     breadth-first search over non-cut pixels reaches it from a fixed start, each new pixel
//                     from its first neighbour of the previous level in the order right, left, below,
//                     above. Maps whose cut bits fit in LDS (up to 1.3 M pixels): a spanning forest gives the
//                     counts without a search (k_gs_tile, k_gs_merge, k_gs_anchor; whole device), and every
//                     step is checked against them; a map whose counts would depend on the path takes the search:
//                     k_gs_bfs_lev (one workgroup per map, one barrier per level) stores each pixel's
//                     level, k_gs_ptr_init takes the parents from the levels and k_gs_ptr_jump
//                     (whole device) sums the steps along the parent chains by pointer
//                     jumping. Larger maps: k_gs_bfs, with k along the levels.
//   4. k_gs_finish    one thread per pixel: interior cut pixels next to a reached pixel take k from
//                     it (same order); unwrapped = phi + 2 pi k, or 0 where unreached.
// Float operations that decide integers are written as single rounded operations and this file is
// built with -ffp-contract=off (the _rn intrinsics are plain operations that the compiler would
// otherwise fuse into FMAs), matching the host specification compiled without contraction.
#include <climits>
#include <type_traits>

#include "internal.hpp"

namespace ctdm {

static constexpr float kTWO_PI_F = 6.28318530717958647692f;
static constexpr float kINV_2PI_F = 0.15915494309189533577f;

// fmodf(a, b) for b > 0, then shifted into [0, b). For |a| < 2b, fmodf is a itself or a - sign(a) b,
// and |a| - b is exact there (b <= |a| <= 2b); other a (wrapped phases far outside [-pi, pi]) take fmodf.
__device__ __forceinline__ float gs_mod(float a, float b)
{
    const float aa = fabsf(a);
    float r = aa < b ? a : (aa < __fmul_rn(2.f, b) ? copysignf(__fsub_rn(aa, b), a) : fmodf(a, b));
    if (r < 0.f) r = __fadd_rn(r, b);
    return r;
}

__device__ __forceinline__ float gs_wrap_step(float a, float b)
{
    const float d = __fsub_rn(a, b);
    const float x = (float)__dadd_rn((double)d, M_PI);
    const float m = gs_mod(x, (float)(M_PI * 2.0));
    return (float)__dsub_rn((double)m, M_PI);
}

__device__ __forceinline__ int gs_step2pi(float d) { return (int)rintf(__fmul_rn(d, kINV_2PI_F)); }

// Per-pixel kernels run on a grid of (column tiles, rows, maps): column, row and map come from the
// grid, with no division.
__device__ __forceinline__ void pixel_of_grid(int W, int& x, int& y, long long& map)
{
    x = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    y = (int)blockIdx.y;
    map = blockIdx.z;
}

// ---------------------------------------------------------------- 1. residues
// Also starts the cut mask: a residue on the border is its own cut, every other pixel is clear.
__global__ void k_gs_residues(const float* __restrict__ phi, int batch, int H, int W, int8_t* __restrict__ res,
                              uint8_t* __restrict__ cuts)
{
    const long long n = (long long)H * W;
    int i, j;
    long long b;
    pixel_of_grid(W, i, j, b);
    if (i >= W) return;
    const int p = i + W * j;
    const long long g = b * n + p;
    const float* m = phi + b * n;
    int8_t q = 0;
    if (i < W - 1 && j < H - 1) {
        const float a = m[p], bb = m[p + 1], c = m[p + 1 + W], d = m[p + W];
        const float s = __fadd_rn(__fadd_rn(__fadd_rn(gs_wrap_step(a, bb), gs_wrap_step(bb, c)), gs_wrap_step(c, d)),
                                  gs_wrap_step(d, a));
        q = s >= 6.0f ? 1 : (s <= -6.0f ? -1 : 0);
    }
    res[g] = q;
    cuts[g] = q != 0 && (i == 0 || j == 0);
}

// ---------------------------------------------------------------- 2. branch cuts
// Word w of the bit array of a byte map's nonzero entries (bit b: byte 32 w + b; bytes past n read as 0).
// Two 16-byte loads where the word's bytes sit on a 16-byte boundary, else byte loads at clamped
// addresses, all issued before use.
__device__ __forceinline__ unsigned nonzero_bits(const uint8_t* __restrict__ m, long long n, int w)
{
    const long long p0 = (long long)w * 32;
    unsigned v = 0;
    if (p0 + 32 <= n && ((reinterpret_cast<uintptr_t>(m + p0) & 15) == 0)) {
        const uint4 a = *reinterpret_cast<const uint4*>(m + p0);
        const uint4 b = *reinterpret_cast<const uint4*>(m + p0 + 16);
        const unsigned q[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) v |= (unsigned)(((q[k] >> (8 * e)) & 0xffu) != 0) << (4 * k + e);
    } else {
        uint8_t q[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) q[k] = m[min(p0 + k, n - 1)];
#pragma unroll
        for (int k = 0; k < 32; ++k) v |= (unsigned)(p0 + k < n && q[k] != 0) << k;
    }
    return v;
}

// Words w of the bit arrays of a residue map's charges, x: positive, y: negative (bit b: pixel 32 w + b;
// pixels past n: 0). Bytes are 0, 1 or -1: bit 0 tells a charge, bit 7 its sign, and a multiplication moves
// the four flags of a 32-bit load (bits 0, 8, 16, 24) to bits 28-31 without carries.
__device__ __forceinline__ uint2 charge_bits(const int8_t* __restrict__ m, long long n, int w)
{
    const long long p0 = (long long)w * 32;
    unsigned any = 0, neg = 0;
    if (p0 + 32 <= n && ((reinterpret_cast<uintptr_t>(m + p0) & 15) == 0)) {
        const uint4 a = *reinterpret_cast<const uint4*>(m + p0);
        const uint4 b = *reinterpret_cast<const uint4*>(m + p0 + 16);
        const unsigned q[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            any |= (((q[k] & 0x01010101u) * 0x10204080u) >> 28) << (4 * k);
            neg |= ((((q[k] >> 7) & 0x01010101u) * 0x10204080u) >> 28) << (4 * k);
        }
    } else {
        int8_t q[32];
#pragma unroll
        for (int k = 0; k < 32; ++k) q[k] = m[min(p0 + k, n - 1)];
#pragma unroll
        for (int k = 0; k < 32; ++k) {
            any |= (unsigned)(p0 + k < n && q[k] != 0) << k;
            neg |= (unsigned)(p0 + k < n && q[k] < 0) << k;
        }
    }
    return make_uint2(any & ~neg, neg);
}

// ---------------------------------------------------------------- 2b. branch cuts: rows in a pipeline
// The search visits the residues in raster order: a residue that is still present takes the first point of
// its box scan (rings of radius 1, 2, ..., below R) that is a border point or a present charge of the opposite
// sign, and both charges are removed. A residue on the border takes itself; no other residue removes it (the
// border is met first), so those are left out here and marked as cuts beside the residues (k_gs_residues).
//
// A decision only reads and changes pixels within its reach (the ring of its hit), so rows can run side by
// side when each stays behind the one above. One workgroup per map, one group of GS_LANES lanes per row in
// flight. Each group publishes the pixel up to which its row is decided (raster index; a wave's LDS
// operations execute in order, so removals precede the index that covers them). With c the first column the
// row above has not published and rho a bound on every reach, a residue at column x takes a hit on ring r
// once x + r + rho < c, and a row publishes at most c. If every reach is at most rho, its scan then
// sees
//   - every earlier residue's removals: undecided ones lie at columns >= c in the row above and no further left
//     in the rows before, so they change columns >= c - rho only;
//   - no later residue's: one decided in a row below, at x' on ring r', had x' + r' + rho < c' with c' at most what this row
//     had published, which is at most x, so it changed columns < x - rho.
// so all decisions are those of the raster order. A hit beyond rho ends the attempt, and the map starts again
// with 4 rho, then with R, which no reach exceeds. A small rho keeps the rows close together and more of them
// in flight; it follows the residue density, as the nearest opposite charges are close where residues are
// many. Reaches over maps of 8 Gaussians plus uniform noise of +-a pi: at most 7 at densities 0.28 (a = 0.8;
// one in 150 000 is 6) and 0.20 (0.7), 10 at 0.10 (0.6, 256^2), 12 at 0.09, 16 at 0.04 (0.55), each ring
// further 3 to 15 times rarer, so a second attempt stays below one map in a hundred.
//
// Bound: the chain of dependent decisions along the front (about 1 900 steps for 512 rows of density 0.28,
// 19 decisions side by side). In a step a group reads the row above's index, its row's next 31 pixels and the
// opposite charges on rings 1-3 of the pixel it stands on (one LDS round trip), looks the first hit up (another)
// and removes the pair; the work of a step is done on vectors of rows, one instruction for the eight rows of a
// wave, since a wavefront alone on its SIMD takes about five cycles per instruction whatever its lanes do.
// Measured: 64 maps of 512^2 at density 0.28 in 0.97 ms, one 256^2 map at 0.09 in 0.40 ms, against 7.1 and
// 0.60 ms one residue after the other (2c). (With a row publishing c - rho - 1 at most: 1.03 and 0.46 ms.)
constexpr int GS_LANES = 8;                       // lanes per row: rows -3 .. 3 around it (the last lane idle)
constexpr int GS_WAVES = 4;                       // wavefronts per map
constexpr int GS_ROWS = GS_WAVES * 64 / GS_LANES; // rows in flight
constexpr int GS_LEFT = INT_MIN;                  // published by a group that leaves its rows undecided

// The charges still present as two bit arrays, positive and negative, with the border's bits set in both; nw
// words each, one spare word before them and two after. In LDS when they fit (maps up to 0.63 M pixels), else in global memory, read and
// cleared by atomics at device scope, which bypass the vector L1.
template <bool LDSW>
struct Charges {
    unsigned* w;   // positive charges, then negative ones from word nw + 3
    int nw;
    __device__ __forceinline__ unsigned ld(int i) const
    {
        if constexpr (LDSW)
            return __hip_atomic_load(w + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        else
            return __hip_atomic_load(w + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // first word of the charges of one sign
    __device__ __forceinline__ int plane(bool negative) const { return negative ? nw + 3 : 0; }
    __device__ __forceinline__ void clear(int p, bool negative) const
    {
        unsigned* a = w + plane(negative) + (p >> 5);
        const unsigned m = ~(1u << (p & 31));
        if constexpr (LDSW)
            atomicAnd(a, m);
        else
            __hip_atomic_fetch_and(a, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void set_border(int p) const
    {
        for (int s = 0; s < 2; ++s) {
            if constexpr (LDSW)
                atomicOr(w + plane(s) + (p >> 5), 1u << (p & 31));
            else
                __hip_atomic_fetch_or(w + plane(s) + (p >> 5), 1u << (p & 31), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        }
    }
};

// Position q of ring r's scan order, unclipped: left column top to bottom, then the columns between on the
// top and bottom rows in turn, then the right column top to bottom.
__device__ __forceinline__ void ring_position(int r, int q, int& dx, int& dy)
{
    const int side = 2 * r + 1, q2 = q - side, nmid = 2 * (side - 2);
    dx = q < side ? -r : (q2 < nmid ? 1 - r + (q2 >> 1) : r);
    dy = q < side ? q - r : (q2 < nmid ? ((q2 & 1) ? r : -r) : q2 - nmid - r);
}

// The scan of one residue beyond ring 3 by a whole wavefront, 64 positions of the scan order per round (the
// first hit is the lowest lane with one). Returns the hit's pixel, -1 for no hit; sets `far` for a hit beyond ring
// rho, or none up to it. No ring is clipped before the one that touches the border, which holds a hit, so the
// first round (ring 4 and 32 positions of ring 5, fixed offsets) needs no look at the borders. at(q): whether pixel q, at most five
// rows outside the map, is a hit.
template <class At>
__device__ int gs_scan(const At& at, int H, int W, int R, int p, int i, int j, int lane, int rho, bool& far)
{
    if (R <= 4) return -1;
    int rc = 4, o0 = 0;  // next position: ring rc, index o0
    if (R > 5 && rho >= 5) {
        int dx, dy;
        ring_position(lane < 32 ? 4 : 5, lane & 31, dx, dy);
        const int q = p + dx + W * dy;
        const unsigned long long hit = __ballot(at(q));
        if (hit) {
            const int l = __builtin_ctzll(hit);
            return __builtin_amdgcn_readlane(q, l);
        }
        rc = 5;
        o0 = 32;
    }
    while (rc < R) {
        if (rc > rho) {
            far = true;
            return -1;
        }
        int lr = R, lq = 0;  // lanes past the last ring scan nothing
        int start = 0, rr = rc, off = o0;
        while (start < 64 && rr < R) {
            const int P = 2 * (min(j + rr, H - 1) - max(j - rr, 0) + 1) +
                          2 * (min(i + rr, W - 1) - max(i - rr, 0) - 1);
            const int take = min(P - off, 64 - start);
            if (lane >= start && lane < start + take) {
                lr = rr;
                lq = off + lane - start;
            }
            start += take;
            off += take;
            if (off == P) {
                ++rr;
                off = 0;
            }
        }
        int c = 0;
        bool here = false;
        if (lr < R) {
            const int m1 = max(i - lr, 0), m2 = min(i + lr, W - 1);
            const int n1 = max(j - lr, 0), n2 = min(j + lr, H - 1);
            const int nrow = n2 - n1 + 1, nmid = 2 * (m2 - m1 - 1);
            const int q2 = lq - nrow;
            const bool left = lq < nrow, mid = !left && q2 < nmid;
            const int mm = left ? m1 : (mid ? m1 + 1 + (q2 >> 1) : m2);
            const int nn = left ? n1 + lq : (mid ? ((q2 & 1) ? n2 : n1) : n1 + (q2 - nmid));
            const int q = mm + W * nn;
            c = q;
            here = at(q);
        }
        const unsigned long long hit = __ballot(here);
        if (hit) {
            const int l = __builtin_ctzll(hit);
            far = __builtin_amdgcn_readlane(lr, l) > rho;
            return __builtin_amdgcn_readlane(c, l);
        }
        rc = rr;
        o0 = off;
    }
    return -1;
}

// Minimum over the eight lanes of a row's group.
__device__ __forceinline__ unsigned group_min(unsigned v)
{
    static_assert(GS_LANES == 8, "group reduction");
    auto step = [&](auto ctrl) {
        const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(-1, (int)v, decltype(ctrl)::value, 0xf, 0xf, false);
        v = o < v ? o : v;
    };
    step(std::integral_constant<int, 0xb1>{});   // quad_perm 1 0 3 2
    step(std::integral_constant<int, 0x4e>{});   // quad_perm 2 3 0 1
    step(std::integral_constant<int, 0x141>{});  // mirrored within 8 lanes
    return v;
}

// Scan key of the point (dx, dy) on rings 1-3, ordered as the scan: order << 10 | ring << 8 | dx + 8 << 4 | dy + 8.
constexpr unsigned GS_NONE = 0xffffu;
__device__ __forceinline__ unsigned ring_key(int dx, int dy)
{
    const int r = max(abs(dx), abs(dy)), side = 2 * r + 1;
    const int q = dx == -r ? dy + r : (dx == r ? side + 2 * (side - 2) + dy + r : side + 2 * (dx + r - 1) + (dy > 0));
    return (unsigned)((q + (r == 1 ? 0 : (r == 2 ? 8 : 24))) << 10 | r << 8 | (dx + 8) << 4 | (dy + 8));
}

template <bool LDSW>
__global__ __launch_bounds__(64 * GS_WAVES) void k_gs_pair(const int8_t* __restrict__ res, int H, int W,
                                                           unsigned* __restrict__ gwords, int2* __restrict__ pairs,
                                                           int* __restrict__ rowpairs, int* __restrict__ flags)
{
    extern __shared__ unsigned lwords[];
    // prog[first lane of a group]: its published index (the other lanes write the words beside it, which
    // costs less than masking them)
    __shared__ int prog[64 * GS_WAVES], failed, nres;
    __shared__ unsigned short first_key[8 * 128];  // [row dy + 3][charges at dx = -3 .. 3]: key of the first hit
    constexpr int NT = 64 * GS_WAVES;
    const int tid = threadIdx.x, lane = tid & 63, l = lane % GS_LANES, slot = tid / GS_LANES;
    const long long n = (long long)H * W;
    const int nw = (int)((n + 31) / 32);
    const int8_t* r = res + blockIdx.x * n;
    if (tid == 0) {  // the fill's flag of this map, and behind the last one the longest chain
        flags[blockIdx.x] = 0;
        if (blockIdx.x == 0) flags[gridDim.x] = 0;
    }
    int2* out = pairs + blockIdx.x * n;  // row y's choices start at out[y W], nrow[y] of them
    int* nrow = rowpairs + (long long)blockIdx.x * H;
    const Charges<LDSW> ch{(LDSW ? lwords : gwords + (long long)blockIdx.x * 2 * (nw + 3)) + 1, nw};
    const int R = min(901, W / 2);
    for (int e = tid; e < 8 * 128; e += NT) {
        unsigned best = GS_NONE;
        const int dy = (e >> 7) - 3;
        for (int k = 0; k < 7; ++k) {
            const int dx = k - 3, rg = max(abs(dx), abs(dy));
            if (dy <= 3 && rg > 0 && rg < R && ((e >> k) & 1)) best = min(best, ring_key(dx, dy));
        }
        first_key[e] = (unsigned short)best;
    }
    const int off = W * (l - 3) - 3;  // this lane's row around a pixel, from dx = -3
    const unsigned short* const keys = first_key + (l << 7);
    // group g starts on row 1 + g (those past the map publish the same, as the first row reads the last group)
    const int start = (int)min((1ll + slot) * W, (long long)INT_MAX);
    int* const my_prog = &prog[tid];
    const int* const above = &prog[(slot + GS_ROWS - 1) % GS_ROWS * GS_LANES];
    if (tid == 0) nres = 0;
    __syncthreads();
    int rho = 0;  // set from the density on the first attempt
    for (int attempt = 0;; ++attempt) {
        int mine = 0;
        for (int w = tid - 1; w < nw + 2; w += NT) {
            const uint2 b = w >= 0 && w < nw ? charge_bits(r, n, w) : make_uint2(0, 0);
            ch.w[w] = b.x;
            ch.w[nw + 3 + w] = b.y;
            mine += __popc(b.x | b.y);
        }
        if (attempt == 0 && mine) atomicAdd(&nres, mine);
        prog[tid] = start;
        if (tid == 0) failed = 0;
        if constexpr (!LDSW) __threadfence();
        __syncthreads();
        for (int y = tid; y < H; y += NT) {
            ch.set_border(y * W);
            ch.set_border(y * W + W - 1);
        }
        for (int x = tid; x < W; x += NT) {
            ch.set_border(x);
            ch.set_border((H - 1) * W + x);
        }
        if constexpr (!LDSW) __threadfence();
        __syncthreads();
        rho = attempt == 0 ? (nres >= 0.25f * n ? 8 : (nres >= 0.1f * n ? 12 : (nres >= 0.05f * n ? 20 : 40)))
                           : (attempt == 1 ? 4 * rho : R);  // no scan reaches R
        // Per row in flight (equal in all lanes of its group): the row, its first pixel and the end of its
        // interior, the pixel it stands on (the first undecided one), whether a charge is expected there and its
        // sign, the published index and the choices so far. Groups without a row stand still on a valid pixel.
        int y = 1 + slot;
        bool active = y <= H - 2 && nres > 0, known = false, qn = false;
        int row0 = active ? y * W : 0, hi = row0 + W - 1, pos = row0 + 1, pub = start, np = 0;
        // Every step moves the topmost undecided row on (it waits for nothing), and a group that leaves its
        // rows publishes GS_LEFT, which the group after it passes on: the loop ends.
        while (__ballot(active)) {
            const int v = __hip_atomic_load(above, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if constexpr (!LDSW) __builtin_amdgcn_s_waitcnt(0);  // the index before the charges it covers
            asm volatile("" ::: "memory");
            const int wi = pos >> 5;
            const unsigned a0 = ch.ld(wi), a1 = ch.ld(wi + 1), b0 = ch.ld(nw + 3 + wi), b1 = ch.ld(nw + 4 + wi);
            // the seven pixels of this lane's row (outside the map: any words, those rings come after a border hit)
            const int opp = ch.plane(!qn), ring = pos + off;
            const int wr = opp + max(min(ring >> 5, nw), -1);
            const unsigned r0 = ch.ld(wr), r1 = ch.ld(wr + 1);
            asm volatile("" ::: "memory");
            const unsigned best = group_min(keys[__builtin_amdgcn_alignbit(r1, r0, ring) & 127u]);
            // the row's charges from pos on (bit b: pixel pos + b)
            const int nb = min(31, hi - pos);
            const unsigned neg = __builtin_amdgcn_alignbit(b1, b0, pos);
            unsigned any = __builtin_amdgcn_ubfe(__builtin_amdgcn_alignbit(a1, a0, pos) | neg, 0, nb);
            const bool all = v >= row0;                           // the row above is decided
            const int lim = all ? INT_MAX - 2 * rho : v + W;      // else: below the pixel under its published index
            const bool here = active && known && (any & 1u);
            const int dx = (int)((best >> 4) & 15u) - 8, dy = (int)(best & 15u) - 8;
            bool decided = here && best != GS_NONE && pos + (int)((best >> 8) & 3u) + rho < lim;
            int t = pos + dx + (LDSW ? __mul24(W, dy) : W * dy);
            bool pair = (unsigned)(pos - row0 + dx - 1) < (unsigned)(W - 2) && (unsigned)(y + dy - 1) < (unsigned)(H - 2);
            // no hit on rings 1-3: the rest of the scan, once every ring up to rho is settled
            bool far = false;
            for (unsigned long long slow = __ballot(here && best == GS_NONE && pos + 2 * rho < lim); slow;) {
                const int f = __builtin_ctzll(slow);
                slow &= ~(((1ull << GS_LANES) - 1) << (f & ~(GS_LANES - 1)));
                bool beyond = false;
                const int sp = __builtin_amdgcn_readlane(pos, f);
                const int so = __builtin_amdgcn_readlane(opp, f);
                auto at = [&](int q) -> bool {
                    return (ch.ld(so + (int)min((unsigned)(q >> 5), (unsigned)nw)) >> (q & 31)) & 1u;
                };
                const int c = gs_scan(at, H, W, R, sp, sp - __builtin_amdgcn_readlane(row0, f),
                                      __builtin_amdgcn_readlane(y, f), lane, rho, beyond);
                if ((lane ^ f) < GS_LANES) {
                    t = c;
                    const int tx = c % W, ty = c / W;
                    pair = tx > 0 && tx < W - 1 && ty > 0 && ty < H - 1;
                    decided = !beyond;
                    far = beyond;
                }
            }
            if (decided) {
                any &= ~1u;
                if (t >= 0) {  // else nothing within reach: the residue stays unbalanced
                    // the residue goes, and the charge it takes; a border point stays
                    const unsigned dt = (unsigned)(t - pos);
                    if (pair && dt < 31u) any &= ~(1u << dt);
                    if (l == 0 || (l == 1 && pair)) {
                        ch.clear(l ? t : pos, l ? !qn : qn);
                        out[row0 + np] = make_int2(pos, t);
                    }
                    ++np;
                }
            }
            // the next charge, and how far the row is decided
            known = any != 0;
            const int nx = known ? __builtin_ctz(any) : nb;
            qn = (neg >> nx) & 1u;
            pos += nx;
            pub = pub == GS_LEFT ? GS_LEFT : max(pub, min(pos, lim));
            if (active && all && pos >= hi) {
                pub = row0 + W;
                if (l == 0) nrow[y] = np;
                active = y + GS_ROWS <= H - 2;
                if (active) {
                    y += GS_ROWS;
                    row0 = y * W;
                    hi = row0 + W - 1;
                    pos = row0 + 1;
                    known = false;
                    np = 0;
                }
            }
            if (active && (far || v == GS_LEFT)) {
                if (far) failed = 1;
                active = false;
                pub = GS_LEFT;
            }
            if constexpr (!LDSW) __builtin_amdgcn_s_waitcnt(0);  // removals before the index that covers them
            asm volatile("" ::: "memory");
            __hip_atomic_store(my_prog, pub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        __syncthreads();
        if (!failed) break;
        __syncthreads();  // every wave has read the flag before the next attempt clears it
    }
    for (int y = tid; y < H; y += NT)
        if (nres == 0 || y == 0 || y == H - 1) nrow[y] = 0;
}

// ---------------------------------------------------------------- 2c. branch cuts: one residue after the other
// Maps of few columns leave the pipeline no room, since each row stays more than rho columns behind the one above: the
// search as it is stated, by one wavefront, with a residue's first 64 positions (rings 1-3 and 16 of ring 4) side by side and
// the rest by gs_scan. The pixels' states stand in LDS in two bits each (1, 2: a present charge of either sign, 3: border),
// with zeros for five rows before and after, so that one read tells a position's state and no position needs a look at the
// map's edges (no ring is clipped before the one that touches the border, which holds a hit).
// Bound by the instructions from one residue to the next, about 90 ns a residue, hence the common case as a loop of its
// own. Against the pipeline, at noise of 0.6 and 0.8 pi (density 0.09 and 0.28), in us: one map of 4000 x 16 560 and 1619 (2445,
// 4265), 2000 x 40 734 and 2061 (1924, 2764), 520 x 48 239 and 637 (557, 737), 1000 x 60 561 and 1549 (1145, 1465), 520 x 64
// 330 and 869 (515, 780). The line lies where the densest maps begin to lose more than the others gain.
constexpr int GS_WALK = 60;
constexpr __host__ __device__ int gs_ahead(int W) { return 5 * (W + 1) / 16 + 2; }
__device__ __forceinline__ unsigned spread_bits(unsigned v)  // bit b of the low half to bit 2 b
{
    v = (v | (v << 8)) & 0x00ff00ffu;
    v = (v | (v << 4)) & 0x0f0f0f0fu;
    v = (v | (v << 2)) & 0x33333333u;
    return (v | (v << 1)) & 0x55555555u;
}

__global__ __launch_bounds__(256) void k_gs_walk(const int8_t* __restrict__ res, int H, int W, int2* __restrict__ pairs,
                                                 int* __restrict__ rowpairs, int* __restrict__ flags)
{
    extern __shared__ unsigned lwords[];
    __shared__ int total;
    const int tid = threadIdx.x, lane = tid & 63, R = min(901, W / 2), ahead = gs_ahead(W);
    const long long n = (long long)H * W;
    const int nw = (int)((n + 15) / 16);
    unsigned* const state = lwords + ahead;
    const int8_t* r = res + blockIdx.x * n;
    if (tid == 0) {  // the fill's flag of this map, and behind the last one the longest chain
        flags[blockIdx.x] = 0;
        if (blockIdx.x == 0) flags[gridDim.x] = 0;
    }
    int2* out = pairs + blockIdx.x * n;
    for (int w = tid; w < ahead; w += 256) lwords[w] = state[nw + w] = 0;
    for (int w = tid; w < (nw + 1) / 2; w += 256) {
        const uint2 b = charge_bits(r, n, w);
        state[2 * w] = spread_bits(b.x & 0xffffu) | spread_bits(b.y & 0xffffu) << 1;
        if (2 * w + 1 < nw) state[2 * w + 1] = spread_bits(b.x >> 16) | spread_bits(b.y >> 16) << 1;
    }
    __syncthreads();
    auto border = [&](int p) { atomicOr(state + (p >> 4), 3u << (2 * (p & 15))); };
    for (int y = tid; y < H; y += 256) {
        border(y * W);
        border(y * W + W - 1);
    }
    for (int x = tid; x < W; x += 256) {
        border(x);
        border((H - 1) * W + x);
    }
    __syncthreads();
    if (tid < 64) {
        auto ld = [&](int w) { return __hip_atomic_load(state + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
        const int ring = lane < 8 ? 1 : (lane < 24 ? 2 : (lane < 48 ? 3 : 4));
        int dx, dy;
        ring_position(ring, lane - (lane < 8 ? 0 : (lane < 24 ? 8 : (lane < 48 ? 24 : 48))), dx, dy);
        const int off = 2 * (dx + W * dy);  // positions as bit numbers, two a pixel
        const unsigned in = ring < R ? 3u : 0u;
        int2* o = out;
        for (int c = 0; c < nw; c += 64) {
            const unsigned w = c + lane < nw ? ld(c + lane) : 0u;
            unsigned m = (w ^ (w >> 1)) & 0x55555555u;  // charges left to visit (at their lower bits)
            const int base = 32 * (c + lane);
            int p = 0;  // the residue visited
            unsigned opp = 0, self = 0;
            auto settle = [&](int t, bool pair) {  // lane 0 removes the residue, lane 1 the charge that it takes
                const int gone = pair ? t : p;
                if (lane < 2) {
                    const int x = lane ? gone : p;
                    atomicAnd(state + (x >> 5), ~(3u << (x & 31)));
                    reinterpret_cast<int*>(o)[lane] = (lane ? t : p) >> 1;
                }
                ++o;
                const unsigned x = gone - base, taken = x < 32u ? 1u << x : 0u;
                m = m & ~self & ~taken;
                asm volatile("" ::: "memory");  // the removals before later reads (in order in the LDS)
            };
            for (;;) {
                unsigned long long hit = ~0ull;
                for (unsigned long long live; (live = __ballot(m != 0)) != 0;) {
                    const int f = __builtin_ctzll(live), bit = __builtin_ctz(__builtin_amdgcn_readlane(m, f));
                    p = 32 * (c + f) + bit;
                    const int q = p + off;
                    opp = ((unsigned)__builtin_amdgcn_readlane(w, f) >> (bit | 1)) & 1u ? 1u : 2u;
                    const unsigned v = (ld(q >> 5) >> (q & 31)) & in;
                    hit = __ballot((v & opp) != 0);
                    const unsigned long long edge = __ballot(v == 3u);
                    self = lane == f ? 1u << bit : 0u;
                    if (__builtin_expect(hit == 0, 0)) break;
                    const int k = __builtin_ctzll(hit);
                    settle(__builtin_amdgcn_readlane(q, k), !((edge >> k) & 1u));
                }
                if (hit) break;
                bool far = false;
                auto at = [&](int x) { return ((ld(x >> 4) >> (2 * (x & 15))) & opp) != 0; };
                const int pp = p >> 1, t = gs_scan(at, H, W, R, pp, pp % W, pp / W, lane, R, far);
                if (t >= 0)
                    settle(2 * t, t % W > 0 && t % W < W - 1 && t / W > 0 && t / W < H - 1);
                else
                    m &= ~self;  // nothing within reach: the residue stays unbalanced
            }
        }
        const int np = (int)(o - out);
        if (lane == 0) total = np;
    }
    __syncthreads();
    // the choices are one list: rows of W of them
    for (int y = tid; y < H; y += 256) rowpairs[(long long)blockIdx.x * H + y] = max(min(total - y * W, W), 0);
}

// The chosen cuts: one thread per choice, one grid row per row of the map (cut pixels are only set, so the
// order does not matter).
__global__ void k_gs_draw(const int2* __restrict__ pairs, const int* __restrict__ rowpairs, int H, int W,
                          uint8_t* __restrict__ cuts)
{
    const long long n = (long long)H * W;
    const long long map = blockIdx.z;
    const int k = (int)(blockIdx.x * blockDim.x + threadIdx.x), y = blockIdx.y;
    if (k >= rowpairs[map * H + y]) return;
    const int2 pr = pairs[map * n + (long long)y * W + k];
    uint8_t* cut = cuts + map * n;
    const int p = pr.x, r1 = p % W, c1 = p / W;
    // to an opposite charge straight; to a column border along the row, else to a row border along the column
    int r2 = pr.y % W, c2 = pr.y / W;
    if (r2 == 0 || r2 == W - 1) c2 = c1;
    else if (c2 == 0 || c2 == H - 1) r2 = r1;
    const long long t = r2 + (long long)W * c2;
    cut[p] = 1;
    cut[t] = 1;
    const float dR = (float)(r2 - r1), dC = (float)(c2 - c1);
    const float rad = __fsqrt_rn(__fadd_rn(__fmul_rn(dR, dR), __fmul_rn(dC, dC)));
    const float ct = __fdiv_rn(dR, rad), st = __fdiv_rn(dC, rad);
    const int nseg = (int)rintf(rad);
    const int rlo = min(r1, r2), rhi = max(r1, r2), clo = min(c1, c2), chi = max(c1, c2);
    for (int ii = 1; ii <= nseg; ++ii) {
        const int rf = r1 + (int)rintf(__fmul_rn((float)ii, ct));
        const int cf = c1 + (int)rintf(__fmul_rn((float)ii, st));
        if (rf >= rlo && rf <= rhi && cf >= clo && cf <= chi) cut[rf + (long long)W * cf] = 1;
    }
}

// ---------------------------------------------------------------- 3. flood fill (BFS levels)
__device__ __forceinline__ int ld_rel(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// The same at workgroup scope, for data one workgroup owns until its kernel ends (its waves share a
// CU, so the loads may be served by that CU's cache).
__device__ __forceinline__ int ld_wg(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
__device__ __forceinline__ void st_wg(int* p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }

// Queue slot for each calling lane: one atomic per wavefront for the lanes that call it together
// (this module is built without the compiler's atomic optimizer, so the aggregation is explicit).
__device__ __forceinline__ int reserve_slot(int* counter)
{
    const unsigned long long m = __ballot(1);
    const int rank = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    int base = 0;
    if (rank == 0) base = atomicAdd(counter, __popcll(m));  // the first active lane
    return __builtin_amdgcn_readfirstlane(base) + rank;
}
__device__ __forceinline__ void st_rel(int* p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

__global__ __launch_bounds__(1024) void k_gs_bfs(const float* __restrict__ phi, const uint8_t* __restrict__ cuts,
                                                 int H, int W, int* __restrict__ level, int* __restrict__ kk,
                                                 int* __restrict__ qa, int* __restrict__ qb)
{
    __shared__ int ncur, nnext;
    const long long n = (long long)H * W;
    const float* ph = phi + blockIdx.x * n;
    const uint8_t* cut = cuts + blockIdx.x * n;
    int* lev = level + blockIdx.x * n;
    int* k = kk + blockIdx.x * n;
    int* cur = qa + blockIdx.x * n;
    int* nxt = qb + blockIdx.x * n;
    for (long long p = threadIdx.x; p < n; p += blockDim.x) {
        st_wg(lev + p, -1);
        st_wg(k + p, INT_MIN);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int sx = W / 2, sy = min(20, H - 1);
        while (sx >= 0 && sy < H && cut[sx + (long long)W * sy]) {
            --sx;
            ++sy;
        }
        ncur = 0;
        if (sx >= 0 && sy < H) {
            const int s = sx + W * sy;
            st_wg(lev + s, 0);
            st_wg(k + s, 0);
            st_wg(cur, s);
            ncur = 1;
        }
        nnext = 0;
    }
    __syncthreads();
    const int dx4[4] = {1, -1, 0, 0}, dy4[4] = {0, 0, 1, -1};
    for (int d = 0;; ++d) {
        const int nc = ncur;
        if (nc == 0) break;
        for (int e = threadIdx.x; e < nc; e += blockDim.x) {
            const int p = ld_wg(cur + e);
            const int x = p % W, y = p / W;
            for (int t = 0; t < 4; ++t) {
                const int nx = x + dx4[t], ny = y + dy4[t];
                if (nx < 0 || nx >= W || ny < 0 || ny >= H) continue;
                const int q = nx + W * ny;
                if (cut[q]) continue;
                int expected = -1;
                if (__hip_atomic_compare_exchange_strong(lev + q, &expected, d + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_WORKGROUP)) {
                    const int pos = reserve_slot(&nnext);
                    st_wg(nxt + pos, q);
                }
            }
        }
        __syncthreads();
        const int nn = nnext;
        for (int e = threadIdx.x; e < nn; e += blockDim.x) {
            const int q = ld_wg(nxt + e);
            const int x = q % W, y = q / W;
            for (int t = 0; t < 4; ++t) {
                const int nx = x + dx4[t], ny = y + dy4[t];
                if (nx < 0 || nx >= W || ny < 0 || ny >= H) continue;
                const int pp = nx + W * ny;
                if (ld_wg(lev + pp) == d) {
                    st_wg(k + q, ld_wg(k + pp) - gs_step2pi(__fsub_rn(ph[q], ph[pp])));
                    break;
                }
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            ncur = nn;
            nnext = 0;
        }
        int* t = cur;
        cur = nxt;
        nxt = t;
        __syncthreads();
    }
}

// Bit p of a bit mask.
__device__ __forceinline__ bool tbit(const unsigned* b, long long p) { return (b[p >> 5] >> (p & 31)) & 1u; }

// ---------------------------------------------------------------- 3b. fill without a search
// The 2 pi count of a reached pixel is the sum of the steps along the search's path to it. Where every loop of free
// (not cut) pixels has steps that sum to zero, which is what the cuts are for, any path gives the same count, and the
// paths need no levels: a spanning forest of the free pixels does. k_gs_tile joins the pixels of a tile in LDS,
// k_gs_merge the tiles' trees over the tile borders, k_gs_anchor lets each tile's roots point to the map's root and
// finds the start pixel's; k_gs_finish then adds two offsets per pixel. Each pixel's pair (ptr, sum), k(p) =
// sum + k(ptr), is read and written as one 64-bit word; a root points to itself. Roots are hooked to roots of smaller
// index by compare-and-swap, so pointers only fall, every walk ends, and a failed swap means that another one joined that root.
// Every edge between free pixels is then checked (k_gs_tile within tiles, k_gs_anchor across their borders). A map with
// an edge that disagrees, or with a step outside 32 bits, is flagged and takes the search of 3c, whose kernels return at
// once for the others: whatever the input, the counts are the search's own. 64 maps of 512^2 (noise +-0.8 pi; about one
// map in 1000 is flagged): fill and outputs 0.41 ms in place of 1.92 (k_gs_tile 0.10, merge 0.04, anchor 0.03, the idle search
// 0.03, finish 0.21), 1.2 to 1.5 with a flagged map among them; one map of 256^2 60 us in place of 320. Tiles of 16 rows:
// 0.42, of 64 (1024 threads) 0.41.
constexpr int GS_TX = 64, GS_TY = 32;  // a tile: a wave's width, four rows for each of eight waves
__device__ __forceinline__ unsigned long long gs_pack(int ptr, unsigned sum)
{
    return (unsigned long long)(unsigned)ptr | ((unsigned long long)sum << 32);
}
template <int SCOPE>
__device__ __forceinline__ unsigned long long gs_pair_load(const unsigned long long* p)
{
    if constexpr (SCOPE == 0)
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int SCOPE>
__device__ __forceinline__ void gs_pair_store(unsigned long long* p, unsigned long long v)
{
    if constexpr (SCOPE == 0)
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Root of node a; off gains the sums on the way. Pointers fall strictly, so the walk ends.
template <int SCOPE>
__device__ __forceinline__ int gs_root(const unsigned long long* node, int a, unsigned& off)
{
    for (;;) {
        const unsigned long long v = gs_pair_load<SCOPE>(node + a);
        const int up = (int)(unsigned)v;
        if (up == a) return a;
        off += (unsigned)(v >> 32);
        a = up;
    }
}
// Joins the trees of p and q, given k(p) = k(a) + oa, k(q) = k(b) + ob and k(q) = k(p) - s.
template <int SCOPE>
__device__ __forceinline__ void gs_unite(unsigned long long* node, int a, unsigned oa, int b, unsigned ob, unsigned s)
{
    for (;;) {
        a = gs_root<SCOPE>(node, a, oa);
        b = gs_root<SCOPE>(node, b, ob);
        if (a == b) return;
        const unsigned d = oa - s - ob;  // k(b) - k(a)
        const int hi = a < b ? b : a;
        unsigned long long self = gs_pack(hi, 0);
        const unsigned long long link = a < b ? gs_pack(a, d) : gs_pack(b, 0u - d);
        bool done;
        if constexpr (SCOPE == 0)
            done = __hip_atomic_compare_exchange_strong(node + hi, &self, link, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP);
        else
            done = __hip_atomic_compare_exchange_strong(node + hi, &self, link, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
        if (done) return;
    }
}
// A step outside 32 bits (the conversion saturates): its two directions are not each other's negative.
__device__ __forceinline__ bool gs_step_bad(int s) { return s == INT_MIN || s == INT_MAX; }

// One tile per workgroup, a row at a time per wave: the offsets within a run of free pixels are a prefix sum of the
// row's steps, so the nodes are the runs (at their first pixels) and the edges to join the first of each overlap of a
// run with one of the row above.
__global__ __launch_bounds__(512) void k_gs_tile(const float* __restrict__ phi, const uint8_t* __restrict__ cuts, int H,
                                                 int W, unsigned long long* __restrict__ pr, int* __restrict__ flag)
{
    constexpr int RW = GS_TY / 8;  // rows per wave
    __shared__ unsigned long long node[GS_TX * GS_TY];
    const long long n = (long long)H * W, b = blockIdx.z;
    const float* ph = phi + b * n;
    const uint8_t* cut = cuts + b * n;
    const int lane = threadIdx.x & 63, r0 = (threadIdx.x >> 6) * RW;
    const int x = blockIdx.x * GS_TX + lane, y0 = blockIdx.y * GS_TY;
    float f[RW + 1];
    unsigned long long m[RW + 1];  // free pixels of rows r0 - 1 .. r0 + RW - 1 (none above the tile's first row)
    unsigned off[RW + 1];          // k(p) - k(first pixel of p's run)
    int st[RW + 1];                // node of p's run
    bool bad = false;
#pragma unroll
    for (int i = 0; i <= RW; ++i) {
        const int row = r0 + i - 1, y = y0 + row;
        const bool in = row >= 0 && y < H && x < W;
        const long long g = in ? (long long)y * W + x : 0;
        f[i] = ph[g];
        const bool fr = in && cut[g] == 0;
        m[i] = __ballot(fr);
    }
#pragma unroll
    for (int i = 0; i <= RW; ++i) {
        const float left = __shfl_up(f[i], 1);
        const unsigned long long joined = m[i] & (m[i] << 1);  // free with a free left neighbour
        const int s = (joined >> lane) & 1 ? gs_step2pi(__fsub_rn(f[i], left)) : 0;
        bad |= gs_step_bad(s);
        unsigned v = 0u - (unsigned)s;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned u = __shfl_up(v, o);
            if (lane >= o) v += u;
        }
        const unsigned long long first = m[i] & ~joined & (~0ull >> (63 - lane));  // run starts up to this lane
        const int sl = first ? 63 - __clzll(first) : lane;
        off[i] = v - __shfl(v, sl);
        st[i] = max(r0 + i - 1, 0) * GS_TX + sl;
        if (i > 0 && sl == lane && ((m[i] >> lane) & 1)) node[st[i]] = gs_pack(st[i], 0);
    }
    __syncthreads();
#pragma unroll
    for (int i = 1; i <= RW; ++i) {
        const unsigned long long e = m[i] & m[i - 1];
        if (((e & ~(e << 1)) >> lane) & 1)
            gs_unite<0>(node, st[i - 1], off[i - 1], st[i], off[i], (unsigned)gs_step2pi(__fsub_rn(f[i], f[i - 1])));
    }
    __syncthreads();
#pragma unroll
    for (int i = 1; i <= RW; ++i) {
        if (((m[i] >> lane) & 1) && (st[i] & 63) == lane) {
            unsigned o = 0;
            const int r = gs_root<0>(node, st[i], o);
            gs_pair_store<0>(node + st[i], gs_pack(r, o));
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 1; i <= RW; ++i) {
        const int y = y0 + r0 + i - 1;
        if (x >= W || y >= H) continue;
        unsigned long long out = gs_pack(-1, 0);
        if ((m[i] >> lane) & 1) {
            const unsigned long long v = node[st[i]];
            const int r = (int)(unsigned)v;
            const unsigned k = off[i] + (unsigned)(v >> 32);
            if ((m[i - 1] >> lane) & 1) {
                const int s = gs_step2pi(__fsub_rn(f[i], f[i - 1]));
                bad |= gs_step_bad(s) || k != off[i - 1] + (unsigned)(node[st[i - 1]] >> 32) - (unsigned)s;
            }
            out = gs_pack((y0 + r / GS_TX) * W + (int)blockIdx.x * GS_TX + r % GS_TX, k);
        }
        pr[b * n + (long long)y * W + x] = out;
    }
    if (__any(bad) && lane == 0) atomicOr(flag + b, 1);
}

// Edge e of a map's tile borders: pixels p and q = right of or below p, of two tiles. `before`: how far back the pair before it
// along the border lies when it joins the same two tiles (else 0): where that pair is free too the edge joins nothing new.
__device__ __forceinline__ bool gs_border_edge(long long e, int H, int W, int& p, int& q, int& before)
{
    const long long nv = (long long)((W - 1) / GS_TX) * H, nh = (long long)((H - 1) / GS_TY) * W;
    if (e >= nv + nh) return false;
    if (e < nv) {
        const int y = (int)(e % H), x = ((int)(e / H) + 1) * GS_TX;
        q = y * W + x;
        p = q - 1;
        before = y % GS_TY ? W : 0;
    } else {
        const int x = (int)((e - nv) % W), y = ((int)((e - nv) / W) + 1) * GS_TY;
        q = y * W + x;
        p = q - W;
        before = x % GS_TX ? 1 : 0;
    }
    return true;
}

__global__ __launch_bounds__(256) void k_gs_merge(const float* __restrict__ phi, const uint8_t* __restrict__ cuts, int H,
                                                  int W, unsigned long long* __restrict__ pr)
{
    const long long n = (long long)H * W, base = blockIdx.y * n;
    int p, q, before;
    if (!gs_border_edge((long long)blockIdx.x * 256 + threadIdx.x, H, W, p, q, before)) return;
    const uint8_t* cut = cuts + base;
    if (cut[p] || cut[q] || (before && !cut[p - before] && !cut[q - before])) return;
    const unsigned s = (unsigned)gs_step2pi(__fsub_rn(phi[base + q], phi[base + p]));
    gs_unite<1>(pr + base, p, 0, q, 0, s);
}

// After the merge: every border edge is checked and its pixels, with the tile roots that they point to, are pointed to
// the map's root; the last workgroup of a map writes the root of its start pixel with the start's offset (-1: none).
__global__ __launch_bounds__(256) void k_gs_anchor(const float* __restrict__ phi, const uint8_t* __restrict__ cuts, int H,
                                                   int W, unsigned long long* __restrict__ pr,
                                                   unsigned long long* __restrict__ start, int* __restrict__ flag)
{
    const long long n = (long long)H * W, base = blockIdx.y * n;
    const uint8_t* cut = cuts + base;
    unsigned long long* node = pr + base;
    if (blockIdx.x == gridDim.x - 1) {
        if (threadIdx.x != 0) return;
        int sx = W / 2, sy = min(20, H - 1);
        while (sx >= 0 && sy < H && cut[sx + (long long)W * sy]) {
            --sx;
            ++sy;
        }
        unsigned long long v = gs_pack(-1, 0);
        if (sx >= 0 && sy < H) {
            unsigned o = 0;
            const int r = gs_root<1>(node, sx + W * sy, o);
            v = gs_pack(r, o);
        }
        start[blockIdx.y] = v;
        return;
    }
    int p, q, before;
    if (!gs_border_edge((long long)blockIdx.x * 256 + threadIdx.x, H, W, p, q, before) || cut[p] || cut[q]) return;
    const int s = gs_step2pi(__fsub_rn(phi[base + q], phi[base + p]));
    // the pixel's own pair, then the node it points to: both get the root
    auto settle = [&](int a, unsigned& k) {
        const unsigned long long v = gs_pair_load<1>(node + a);
        const int t = (int)(unsigned)v;
        unsigned o = 0;
        const int r = gs_root<1>(node, t, o);
        k = (unsigned)(v >> 32) + o;
        if (t != r) {
            gs_pair_store<1>(node + t, gs_pack(r, o));
            gs_pair_store<1>(node + a, gs_pack(r, k));
        }
        return r;
    };
    unsigned kp, kq;
    const int rp = settle(p, kp), rq = settle(q, kq);
    if (gs_step_bad(s) || rp != rq || kq != kp - (unsigned)s) atomicOr(flag + blockIdx.y, 1);
}

// ---------------------------------------------------------------- 3c. flood fill in two stages
// For flagged maps (see 3b) whose cut bits fit in LDS (up to 1.3 M pixels in 160 KiB). Stage 1 (k_gs_bfs_lev, one
// workgroup per map) finds the levels of the search of k_gs_bfs. Stage 2 (the whole device): k_gs_ptr_init gives every
// reached pixel the pair (parent, -step2pi(phi - phi_parent)), the parent being the first neighbour of the previous
// level in the order right, left, below, above, and k_gs_ptr_jump contracts the parent chains by pointer jumping,
// (ptr, sum) <- (ptr[ptr], sum + sum[ptr]), until each pointer is the start pixel, whose pair is (itself, 0). Then sum
// is the pixel's 2 pi count: the same integers k_gs_bfs adds level by level, in another order (integer
// sums do not depend on it). Unreached pixels keep ptr = -1.
//
// The search keeps one bit per pixel in LDS, set for cut pixels and for visited ones, so that an atomic
// OR claims a pixel (the returned word tells whether it was still free; a level is one pass and one
// barrier); each claimed pixel's level goes to global memory (stored, never read during the search). The
// parents are taken afterwards from the final levels: levels are the shortest path lengths from the start
// pixel, the same whatever order the search claims pixels in.
__global__ __launch_bounds__(1024) void k_gs_bfs_lev(const uint8_t* __restrict__ cuts, int H, int W, int Q,
                                                     int* __restrict__ level, int* __restrict__ qa,
                                                     int* __restrict__ qb, int* __restrict__ maxdepth,
                                                     const int* __restrict__ flag)
{
    if (!flag[blockIdx.x]) return;
    extern __shared__ unsigned sm[];
    __shared__ int cnt[3];  // entries of levels d, d + 1, d + 2 (mod 3)
    const long long n = (long long)H * W;
    const int nb = (int)((n + 31) / 32);
    unsigned* blk = sm;  // cut or visited
    int* lq[2] = {reinterpret_cast<int*>(sm + nb), reinterpret_cast<int*>(sm + nb) + Q};
    const uint8_t* cut = cuts + blockIdx.x * n;
    int* lev = level + blockIdx.x * n;
    for (long long p = threadIdx.x; p < n; p += blockDim.x) lev[p] = -1;  // unreached
    int* gq[2] = {qa + blockIdx.x * n, qb + blockIdx.x * n};
    auto qget = [&](int which, int i) -> int { return i < Q ? lq[which][i] : ld_wg(gq[which] + i); };
    auto qput = [&](int which, int i, int v) {
        if (i < Q)
            lq[which][i] = v;
        else
            st_wg(gq[which] + i, v);
    };
    for (int w = threadIdx.x; w < nb; w += blockDim.x) blk[w] = nonzero_bits(cut, n, w);
    __syncthreads();
    if (threadIdx.x == 0) {
        int sx = W / 2, sy = min(20, H - 1);
        while (sx >= 0 && sy < H && tbit(blk, sx + (long long)W * sy)) {
            --sx;
            ++sy;
        }
        cnt[0] = 0;
        if (sx >= 0 && sy < H) {
            const int s0 = sx + W * sy;
            blk[s0 >> 5] |= 1u << (s0 & 31);
            lev[s0] = 0;
            qput(0, 0, (int)((unsigned)sx | ((unsigned)sy << 16)));
            cnt[0] = 1;
        }
        cnt[1] = 0;
        cnt[2] = 0;
    }
    __syncthreads();
    const int dx4[4] = {1, -1, 0, 0}, dy4[4] = {0, 0, 1, -1};
    int d = 0;
    for (;; ++d) {  // one barrier per level
        const int cur = d & 1, nxt = cur ^ 1;                           // queues
        const int c0 = d % 3, c1 = (d + 1) % 3, c2 = (d + 2) % 3;       // counters
        const int nc = cnt[c0];
        if (nc == 0) break;
        if (threadIdx.x == 0) cnt[c2] = 0;  // level d + 2 appends there only after this pass's barrier
        for (int e = threadIdx.x; e < 4 * nc; e += blockDim.x) {  // one (pixel, direction) per thread
            const unsigned v = (unsigned)qget(cur, e >> 2);  // x | y << 16
            const int t = e & 3;
            const int nx = (int)(v & 0xffffu) + dx4[t], ny = (int)(v >> 16) + dy4[t];
            if (nx < 0 || nx >= W || ny < 0 || ny >= H) continue;
            const int q = nx + W * ny;
            const unsigned bit = 1u << (q & 31);
            if (blk[q >> 5] & bit) continue;
            if (atomicOr(blk + (q >> 5), bit) & bit) continue;  // cut, or claimed by another thread
            lev[q] = d + 1;
            qput(nxt, reserve_slot(&cnt[c1]), (int)((unsigned)nx | ((unsigned)ny << 16)));
        }
        __syncthreads();
    }
    if (threadIdx.x == 0 && d > 1) atomicMax(maxdepth, d - 1);  // longest parent chain of the map
}

// Pair (ptr, sum) per pixel of a flagged map from its levels, map-local ptr: a reached pixel of level d + 1 points to
// its first neighbour of level d in the order right, left, below, above (cut and unreached pixels have level -1), the
// start pixel (level 0) to itself.
__global__ __launch_bounds__(256) void k_gs_ptr_init(const float* __restrict__ phi, const int* __restrict__ level, int H,
                                                     int W, unsigned long long* __restrict__ pr,
                                                     const int* __restrict__ flag)
{
    const int b = blockIdx.y;
    if (!flag[b]) return;
    const long long n = (long long)H * W;
    const int* lev = level + b * n;
    const float* ph = phi + b * n;
    for (long long p = (long long)blockIdx.x * 256 + threadIdx.x; p < n; p += (long long)gridDim.x * 256) {
        const int x = (int)(p % W), y = (int)(p / W), d = lev[p];
        unsigned long long v = gs_pack(-1, 0);
        if (d == 0) {
            v = gs_pack((int)p, 0);
        } else if (d > 0) {
            long long pp = -1;
            if (x + 1 < W && lev[p + 1] == d - 1)
                pp = p + 1;
            else if (x > 0 && lev[p - 1] == d - 1)
                pp = p - 1;
            else if (y + 1 < H && lev[p + W] == d - 1)
                pp = p + W;
            else if (y > 0 && lev[p - W] == d - 1)
                pp = p - W;
            v = gs_pack((int)pp, 0u - (unsigned)gs_step2pi(__fsub_rn(ph[p], ph[pp])));
        }
        pr[b * n + p] = v;
    }
}

// Pointer jumping, in place: each pixel follows its pointer GS_HOPS times, reading the pairs as they are,
// and keeps the last pointer with the summed steps. Pairs are read and written as single 64-bit accesses,
// so every read sees a consistent pair: an update keeps k(p) = sum(p) + k(ptr(p)) whichever version of a
// pair it reads, and a newer version only shortens the chain. A launch multiplies every pointer's reach by
// at least GS_HOPS + 1 (the pairs read within it may be older than the launch's own updates), so launch
// `step` is needed only while (GS_HOPS + 1)^step is below the longest chain (maxdepth, from the search);
// later launches return at once.
constexpr int GS_HOPS = 15;
__global__ __launch_bounds__(256) void k_gs_ptr_jump(unsigned long long* __restrict__ a, long long n, int step,
                                                     const int* __restrict__ maxdepth, const int* __restrict__ flag)
{
    if (!flag[blockIdx.y]) return;
    long long reach = 1;
    for (int i = 0; i < step; ++i) reach *= GS_HOPS + 1;
    if (reach >= (long long)*maxdepth) return;
    const long long base = (long long)blockIdx.y * n;  // the grid's y is the map
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const long long g = base + i;
        const unsigned long long mine = __hip_atomic_load(a + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int P = (int)(unsigned)mine;
        if (P < 0) continue;
        int sum = (int)(mine >> 32);
#pragma unroll
        for (int h = 0; h < GS_HOPS; ++h) {  // a reached pixel's pointer is a reached pixel (never negative)
            const unsigned long long up = __hip_atomic_load(a + base + P, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sum += (int)(up >> 32);
            P = (int)(unsigned)up;
        }
        const unsigned long long nv = (unsigned long long)(unsigned)P | ((unsigned long long)(unsigned)sum << 32);
        if (nv != mine) __hip_atomic_store(a + g, nv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------- 4. cut fill + outputs
// k of a pixel: from the fill's int32 counts, or (PTR) from the pairs. A flagged map's are contracted (ptr < 0:
// unreached), the others' lead to the map's root in two steps at most.
template <bool PTR>
__global__ void k_gs_finish(const float* __restrict__ phi, const uint8_t* __restrict__ cuts, const int* __restrict__ kk,
                            const int2* __restrict__ pr, const int2* __restrict__ start, const int* __restrict__ flag,
                            int H, int W, int* __restrict__ kout, float* __restrict__ unwrapped)
{
    const long long n = (long long)H * W;
    int x, y;
    long long b;
    pixel_of_grid(W, x, y, b);
    if (x >= W) return;
    const int p = x + W * y;
    const long long g = b * n + p;
    const uint8_t* cut = cuts + b * n;
    const float* ph = phi + b * n;
    const int2 anchor = PTR ? start[b] : make_int2(0, 0);
    const bool searched = PTR ? flag[b] != 0 : false;
    // k of four pixels, or fewer (q < 0: none, INT_MIN): every load of a level is under way before the next level's
    auto kat = [&](const int (&q)[4], int (&kv)[4]) {
        if constexpr (PTR) {
            int2 v[4], u[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) v[t] = q[t] >= 0 ? pr[b * n + q[t]] : make_int2(-1, 0);
#pragma unroll
            for (int t = 0; t < 4; ++t) u[t] = v[t].x >= 0 && !searched ? pr[b * n + v[t].x] : make_int2(anchor.x, anchor.y);
#pragma unroll
            for (int t = 0; t < 4; ++t)
                kv[t] = v[t].x >= 0 && u[t].x == anchor.x ? (int)((unsigned)v[t].y + (unsigned)u[t].y - (unsigned)anchor.y) : INT_MIN;
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t) kv[t] = q[t] >= 0 ? kk[b * n + q[t]] : INT_MIN;
        }
    };
    const bool is_cut = cut[p];
    int own[4] = {p, -1, -1, -1}, kp[4];
    kat(own, kp);
    int kv = kp[0];
    if (is_cut && x > 0 && x < W - 1 && y > 0 && y < H - 1) {
        const int nb[4] = {p + 1, p - 1, p + W, p - W};
        int q[4], kq[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) q[t] = cut[nb[t]] ? -1 : nb[t];
        kat(q, kq);
#pragma unroll
        for (int t = 3; t >= 0; --t)  // the first one that the fill reached
            if (kq[t] != INT_MIN) kv = kq[t] - gs_step2pi(__fsub_rn(ph[p], ph[nb[t]]));
    }
    if (kout) kout[g] = kv;
    unwrapped[g] = kv == INT_MIN ? 0.f : __fadd_rn(ph[p], __fmul_rn((float)kv, kTWO_PI_F));
}

void goldstein(Ctx& c, const float* wrapped, int batch, int H, int W, int8_t* res, uint8_t* cuts, int32_t* k2pi,
               float* unwrapped)
{
    CTDM_REQUIRE(wrapped && unwrapped, "goldstein: null pointer");
    CTDM_REQUIRE(batch >= 0 && H >= 3 && W >= 3, "goldstein: maps must be at least 3 x 3");
    CTDM_REQUIRE((long long)H * W < (1LL << 30), "goldstein: map too large");
    CTDM_REQUIRE(H <= 65535 && batch <= 65535, "goldstein: at most 65535 rows and 65535 maps per call");
    if (batch == 0) return;
    const long long n = (long long)H * W, tot = n * batch;
    int8_t* r = res ? res : (int8_t*)c.buf("gs.res", tot);
    uint8_t* ct = cuts ? cuts : (uint8_t*)c.buf("gs.cut", tot);
    int* qa = (int*)c.buf("gs.qa", sizeof(int) * tot);
    int* qb = (int*)c.buf("gs.qb", sizeof(int) * tot);
    const dim3 pgrid((unsigned)((W + 255) / 256), (unsigned)H, (unsigned)batch);  // per-pixel kernels
    hipLaunchKernelGGL(k_gs_residues, pgrid, dim3(256), 0, c.stream, wrapped, batch, H, W, r, ct);
    const long long nw = (n + 31) / 32, nb = (n + 31) / 32;
    const size_t lds_max = (size_t)(c.max_lds > 0 ? c.max_lds : 64 * 1024);
    // branch cuts: the pairs of the raster-order search, then their cuts
    const size_t words = 2 * ((size_t)nw + 3) * sizeof(unsigned);  // the charges' two bit arrays
    int* npairs = (int*)c.buf("gs.npairs", sizeof(int) * (size_t)batch * H);
    int2* pairs = (int2*)c.buf("gs.pairs", sizeof(int2) * (size_t)tot);
    int* flag = (int*)c.buf("gs.flag", sizeof(int) * ((size_t)batch + 1));
    int* maxd = flag + batch;
    // up to GS_WALK columns one residue after the other (where a map's states fit in LDS beside the kernel's own word)
    const size_t states = sizeof(unsigned) * ((size_t)(n + 15) / 16 + 2 * (size_t)gs_ahead(W));
    if (W <= GS_WALK && states + 64 <= lds_max) {
        hipLaunchKernelGGL(k_gs_walk, dim3(batch), dim3(256), states, c.stream, r, H, W, pairs, npairs, flag);
    } else if (words + 4096 <= lds_max) {  // beside the kernel's own 3 KiB
        hipLaunchKernelGGL(k_gs_pair<true>, dim3(batch), dim3(64 * GS_WAVES), words, c.stream, r, H, W, nullptr,
                           pairs, npairs, flag);
    } else {
        unsigned* gw = (unsigned*)c.buf("gs.words", words * batch);
        hipLaunchKernelGGL(k_gs_pair<false>, dim3(batch), dim3(64 * GS_WAVES), 0, c.stream, r, H, W, gw, pairs,
                           npairs, flag);
    }
    CTDM_CHECK_LAUNCH("k_gs_pair");
    hipLaunchKernelGGL(k_gs_draw, pgrid, dim3(256), 0, c.stream, pairs, npairs, H, W, ct);
    CTDM_CHECK_LAUNCH("k_gs_draw");
    const size_t bits = sizeof(unsigned) * (size_t)nb;  // cut-or-visited bits
    const bool searchable = bits + 64 + 2 * sizeof(int) * 256 <= lds_max && W < 65536 && H < 65536;
    // the queues get what LDS has left (>= 256 each); their entries pack x and y in 16 bits each
    if (searchable) {
        unsigned long long* pr = (unsigned long long*)c.buf("gs.pr", sizeof(unsigned long long) * (size_t)tot);
        unsigned long long* start = (unsigned long long*)c.buf("gs.start", sizeof(unsigned long long) * (size_t)batch);
        int* lev = (int*)c.buf("gs.level", sizeof(int) * tot);
        hipLaunchKernelGGL(k_gs_tile, dim3((unsigned)((W + GS_TX - 1) / GS_TX), (unsigned)((H + GS_TY - 1) / GS_TY), (unsigned)batch),
                           dim3(512), 0, c.stream, wrapped, ct, H, W, pr, flag);
        CTDM_CHECK_LAUNCH("k_gs_tile");
        const long long edges = (long long)((W - 1) / GS_TX) * H + (long long)((H - 1) / GS_TY) * W;
        if (edges) {
            hipLaunchKernelGGL(k_gs_merge, dim3((unsigned)grid1d(edges, 256), (unsigned)batch), dim3(256), 0, c.stream,
                               wrapped, ct, H, W, pr);
            CTDM_CHECK_LAUNCH("k_gs_merge");
        }
        hipLaunchKernelGGL(k_gs_anchor, dim3((unsigned)(edges ? grid1d(edges, 256) : 0) + 1, (unsigned)batch), dim3(256), 0,
                           c.stream, wrapped, ct, H, W, pr, start, flag);
        CTDM_CHECK_LAUNCH("k_gs_anchor");
        // the search, for flagged maps: levels, parents from them, 2 pi counts by pointer jumping
        const int Q = (int)std::min<long long>(n, (long long)((lds_max - 64 - bits) / (2 * sizeof(int))));
        hipLaunchKernelGGL(k_gs_bfs_lev, dim3(batch), dim3(1024), bits + 2 * sizeof(int) * (size_t)Q, c.stream, ct,
                           H, W, Q, lev, qa, qb, maxd, (const int*)flag);
        CTDM_CHECK_LAUNCH("k_gs_bfs_lev");
        // about 8 workgroups per CU in all, split over the maps (the grid's y), but 128 for the one map of many that
        // may be flagged
        const long long per_map = std::max<long long>(128, (long long)std::max(c.cus, 1) * 8 / batch);
        const dim3 jg((unsigned)std::min<long long>(grid1d(n, 256), per_map), (unsigned)batch);
        hipLaunchKernelGGL(k_gs_ptr_init, jg, dim3(256), 0, c.stream, wrapped, lev, H, W, pr, (const int*)flag);
        // enough launches for any chain in a map ((GS_HOPS + 1)^launches >= n); launches past the longest
        // chain return at once
        int launches = 0;
        for (long long reach = 1; reach < n; reach *= GS_HOPS + 1) ++launches;
        for (int r = 0; r < launches; ++r)
            hipLaunchKernelGGL(k_gs_ptr_jump, jg, dim3(256), 0, c.stream, pr, n, r, (const int*)maxd, (const int*)flag);
        CTDM_CHECK_LAUNCH("k_gs_ptr_jump");
        hipLaunchKernelGGL(k_gs_finish<true>, pgrid, dim3(256), 0, c.stream, wrapped, ct, nullptr, (const int2*)pr,
                           (const int2*)start, (const int*)flag, H, W, k2pi, unwrapped);
    } else {
        int* kk = (int*)c.buf("gs.k", sizeof(int) * tot);
        int* lev = (int*)c.buf("gs.level", sizeof(int) * tot);
        hipLaunchKernelGGL(k_gs_bfs, dim3(batch), dim3(1024), 0, c.stream, wrapped, ct, H, W, lev, kk, qa, qb);
        CTDM_CHECK_LAUNCH("k_gs_bfs");
        hipLaunchKernelGGL(k_gs_finish<false>, pgrid, dim3(256), 0, c.stream, wrapped, ct, kk, nullptr, nullptr,
                           nullptr, H, W, k2pi, unwrapped);
    }
    CTDM_CHECK_LAUNCH("k_gs_finish");
}

}  // namespace ctdm
