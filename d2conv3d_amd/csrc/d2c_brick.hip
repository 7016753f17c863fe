// Offset / mask gradient and grad_input of a three-dimensional problem as dense matrix products over bricks of the
// input volume (dconv3d_gpu.cu:562-643, :708-864 in another formulation).
//
// A sampling point reaches the 2 x 2 x 2 voxels above its base voxel floor(z, y, x).  All points whose base voxel
// lies in a block of 1 x 3 x 3 voxels reach the same brick of 2 x 4 x 4 = 32 voxels.  With the points sorted by block
//
//   T[v, s]   = x[v, :] . gcol[s, :]           32 voxels x 32 points x channels: one matrix product; a point's eight
//                                              corner dots are among its 32, and grad_offset / grad_mask follow
//   gx[v, :] += W[v, s] * gcol[s, :]           W = the points' corner weights times modulation, zero off the corners
//
// Three quarters of the products are with zeros, on matrix cores that have them to spare; in exchange nothing is
// gathered: a grad-column row is read once, for both results, and a brick's input rows stay in LDS.  (The kernels
// that gather -- eight corner rows per point through the L1, grad-column rows 3.4 times -- took 1.73 + 1.47 ms for
// 256 channels on 32x60x108, bound by the L1 path, the vector ALU and row latency; this one takes 0.82, at 2.6 TB/s to and
// from device memory, and 0.22 for 512 channels in 8 groups on 2x8x30x54, where they took 0.50 + 0.35.)

#include <algorithm>
#include <cmath>
#include "d2c_mma.hpp"
#include "d2c_tiled.hpp"
#include "d2c_brick.hpp"

namespace {

typedef short v4s __attribute__((ext_vector_type(4)));

// One sampling point as the sort sees it.
struct BrickPoint {
    bool in;              // a corner is inside the volume
    int zi, yq, xq;       // its block
    unsigned cell;        // its base voxel in the block: y | x << 2
    float hz, hy, hx;     // fractions, as make_tap3 gives them
};
D2C_DEV int brick_seg(const BrickDims &d, int bg, int zi, int by, int bx) { return ((bg * d.nz + zi) * d.nby + by) * d.nbx + bx; }
// ---- the sort: count the points of every block, give every block a range, file -------------------------------------
// A workgroup works on 256 positions and up to 28 taps, 4 threads to a position, and requests what it reads of all of
// them first.  Points of neighbouring positions fall into few blocks: they are counted in LDS, in a window of the blocks
// around the workgroup's positions (all blocks of the sample and group where those fit), and a block's number goes to the
// global count in one addition.  The filing pass counts in LDS again: a point's place among the workgroup's points of
// its block is what the addition returned, and the workgroup takes its range of a block's entries in one addition.
// So neither pass writes or reads anything per point that is not wanted in the end.  Points outside the window take
// the global additions one by one; those outside the volume are counted per workgroup too (additions to one address
// follow each other at about 10 ns: with one for every wavefront the list of them took half of the filing pass).
// Bound: scattered stores of 20 bytes to a point, and the instructions of a point's place.  5.6 M points in 8
// offset groups on 2x8x30x54, us for counting + ranges + filing: 134 + 8 + 146 with a hash table per workgroup, places
// of the counting pass kept in memory and an addition per wavefront for the points outside; 46 + 5 + 89 this way.
// 32x60x108 in one group 95 + 7 + 136 and 48 + 5 + 100; 2x8x30x54 in one group 24 + 4 + 35 and 12 + 5 + 21.
// Workgroups: an XCD takes a contiguous part of the positions, the tap groups of a block of 256 one after the other, so
// that the lines which several workgroups write or read in parts meet in one L2.
constexpr int kTaps = 7, kTapGroups = 4, kSortThreads = 256 * kTapGroups;
constexpr int kSortTaps = kTaps * kTapGroups;
struct SortWindow {
    int wz, wy, wx;       // blocks of the window along each axis
    int ngrp, taps;       // groups of taps, taps to a group (up to kSortTaps)
    int ly, lx;           // a workgroup's positions: 2^(8 - ly - lx) planes of 2^ly x 2^lx
    int ny, nx, ntile;    // such tiles along y and x, and of a sample
    FastDiv dkw, dkh;     // divisions by the filter's extents
};
struct SortUnit {
    int b, g, bg, k0, k1; // taps k0, k0 + kTapGroups, ... below k1
    int oz, oy, ox, p;    // the thread's position
    int bz, by, bx;       // ... in the input, without a tap
    bool ok;              // ... is one
    int z0, y0, x0;       // first block of the window
};
D2C_DEV SortUnit sort_unit(const TiledShape &s, const BrickDims &d, const SortWindow &w)
{
    const int nt = (int)gridDim.x, q = nt >> 3, r = nt & 7, xcd = blockIdx.x & 7;
    const int u = xcd * q + (xcd < r ? xcd : r) + (int)(blockIdx.x >> 3);
    const int blk = u / w.ngrp;
    SortUnit t;
    t.bg = blk / w.ntile; t.b = t.bg / s.G; t.g = t.bg - t.b * s.G;
    const int tile = blk - t.bg * w.ntile, tzy = tile / w.nx, tx = tile - tzy * w.nx, tz = tzy / w.ny, ty = tzy - tz * w.ny;
    const int lz = 8 - w.ly - w.lx, i = threadIdx.x & 255;
    t.oz = (tz << lz) + (i >> (w.ly + w.lx)); t.oy = (ty << w.ly) + ((i >> w.lx) & ((1 << w.ly) - 1)); t.ox = (tx << w.lx) + (i & ((1 << w.lx) - 1));
    t.ok = t.oz < s.Do && t.oy < s.Ho && t.ox < s.Wo;
    t.p = t.ok ? (t.oz * s.Ho + t.oy) * s.Wo + t.ox : 0;
    t.bz = t.oz * s.geo.sd - s.geo.pd; t.by = t.oy * s.geo.sh - s.geo.ph; t.bx = t.ox * s.geo.sw - s.geo.pw;
    t.k0 = (u - blk * w.ngrp) * w.taps;
    t.k1 = min(t.k0 + w.taps, s.K);
    t.k0 += __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    // the window lies around the middle of the workgroup's positions and taps
    const int cz = ((tz << lz) + (1 << lz) / 2) * s.geo.sd - s.geo.pd + (s.geo.kd - 1) * s.geo.dd / 2 + 1;
    const int cy = (((ty << w.ly) + (1 << w.ly) / 2) * s.geo.sh - s.geo.ph + (s.geo.kh - 1) * s.geo.dh / 2 + 1) / 3;
    const int cx = (((tx << w.lx) + (1 << w.lx) / 2) * s.geo.sw - s.geo.pw + (s.geo.kw - 1) * s.geo.dw / 2 + 1) / 3;
    t.z0 = max(0, min(cz - w.wz / 2, d.nz - w.wz));
    t.y0 = max(0, min(cy - w.wy / 2, d.nby - w.wy));
    t.x0 = max(0, min(cx - w.wx / 2, d.nbx - w.wx));
    return t;
}
// Tap k of the thread's position from its offsets (sort_offsets): make_tap3 with what the sort needs of it.  A
// position is clamped to where no corner is inside, which is also what the median makes of one that is no number; along an axis that
// is fixed the far plane has no corners.  All of a point's instructions count here: the passes are bound by them.
template <bool AUX16, bool SIZED>
D2C_DEV BrickPoint brick_point(const TiledShape &s, const SortWindow &w, const SortUnit &t, const float *craw, int k)
{
    const int kr = fdiv(k, w.dkw), kx = k - kr * s.geo.kw, kz = fdiv(kr, w.dkh), ky = kr - kz * s.geo.kh;
    float c[3] = {craw[0], craw[1], craw[2]};
    if constexpr (SIZED) size_tap_offsets<AUX16>(s, kz, ky, kx, c, c);
    else tap_offsets_finish<AUX16, false>(s, k, c);
    const float z = (float)(t.bz + kz * s.geo.dd) + c[0], y = (float)(t.by + ky * s.geo.dh) + c[1], x = (float)(t.bx + kx * s.geo.dw) + c[2];
    const float fz = floorf(__builtin_amdgcn_fmed3f(z, -4.f, (float)(s.D + 4))), fy = floorf(__builtin_amdgcn_fmed3f(y, -4.f, (float)(s.H + 4))),
                fx = floorf(__builtin_amdgcn_fmed3f(x, -4.f, (float)(s.W + 4)));
    const int z0 = (int)fz, y0 = (int)fy, x0 = (int)fx;
    const int ez = (s.keep & 0xF0u) != 0, ey = (s.keep & 0xCCu) != 0, ex = (s.keep & 0xAAu) != 0;
    BrickPoint r;
    r.in = (unsigned)(z0 + ez) < (unsigned)(s.D + ez) && (unsigned)(y0 + ey) < (unsigned)(s.H + ey) && (unsigned)(x0 + ex) < (unsigned)(s.W + ex);
    // (base voxels start at -1)
    r.zi = z0 + 1;
    r.yq = brick_block(y0); r.xq = brick_block(x0);
    r.cell = ((unsigned)(y0 + 1) - (unsigned)r.yq * 3u) | ((unsigned)(x0 + 1) - (unsigned)r.xq * 3u) << 2;
    r.hz = z - fz; r.hy = y - fy; r.hx = x - fx;
    return r;
}
// slot of a point's block in the window, -1: outside
D2C_DEV int sort_slot(const SortWindow &w, const SortUnit &t, const BrickPoint &q)
{
    const int z = q.zi - t.z0, y = q.yq - t.y0, x = q.xq - t.x0;
    return (unsigned)z < (unsigned)w.wz && (unsigned)y < (unsigned)w.wy && (unsigned)x < (unsigned)w.wx ? (z * w.wy + y) * w.wx + x : -1;
}
D2C_DEV int sort_slot_seg(const BrickDims &d, const SortWindow &w, const SortUnit &t, int i)
{
    const int r = i / w.wx, x = i - r * w.wx, z = r / w.wy, y = r - z * w.wy;
    return brick_seg(d, t.bg, t.z0 + z, t.y0 + y, t.x0 + x);
}
// the offsets of the thread's taps k0, k0 + kTapGroups, ...; of a size map: size - 1 of the position, in the first place
template <bool AUX16, bool SIZED>
D2C_DEV void sort_offsets(const TiledShape &s, const void *off, const SortUnit &t, float (&c)[kTaps][3])
{
    if constexpr (SIZED) {
        tap_offsets_issue<AUX16, true>(s, off, t.b, t.g, 0, t.p, c[0]);
        if (s.ss.on == 1) size_minus_one<AUX16>(s, c[0]);
    } else {
#pragma unroll
        for (int i = 0; i < kTaps; i++)
            if (t.k0 + i * kTapGroups < t.k1) tap_offsets_issue<AUX16, false>(s, off, t.b, t.g, t.k0 + i * kTapGroups, t.p, c[i]);
    }
}
template <bool AUX16, bool SIZED>
__global__ void __launch_bounds__(kSortThreads, 8)     // (two workgroups to a compute unit)
brick_count_kernel(TiledShape s, BrickDims d, BrickLists L, const void *off, SortWindow w)
{
    extern __shared__ __align__(16) unsigned char smem[];
    int *const s_cnt = reinterpret_cast<int *>(smem);
    const int nslot = w.wz * w.wy * w.wx;
    const SortUnit t = sort_unit(s, d, w);
    float c[kTaps][3];
    sort_offsets<AUX16, SIZED>(s, off, t, c);
    for (int i = threadIdx.x; i < nslot; i += kSortThreads) s_cnt[i] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kTaps; i++) {
        const int k = t.k0 + i * kTapGroups;
        if (!t.ok || k >= t.k1) continue;
        const BrickPoint q = brick_point<AUX16, SIZED>(s, w, t, c[SIZED ? 0 : i], k);
        if (!q.in) continue;
        const int sl = sort_slot(w, t, q);
        if (sl >= 0) atomicAdd(&s_cnt[sl], 1);
        else atomicAdd(&L.count[brick_seg(d, t.bg, q.zi, q.yq, q.xq)], 1);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nslot; i += kSortThreads) {
        const int n = s_cnt[i];
        if (n) atomicAdd(&L.count[sort_slot_seg(d, w, t, i)], n);
    }
}
// (the order of the ranges does not matter: a workgroup adds up its 1024 counts and takes one range for all; additions to
// one address follow each other at about 10 ns)
__global__ void __launch_bounds__(1024) brick_range_kernel(BrickLists L, int nseg)
{
    __shared__ int s_sum[16];
    const int i = blockIdx.x * 1024 + threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = i < nseg ? L.count[i] : 0;
    int sum = n;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(sum, d, 64);
        if (lane >= d) sum += v;
    }
    if (lane == 63) s_sum[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int all = 0;
        for (int w = 0; w < 16; w++) { const int v = s_sum[w]; s_sum[w] = all; all += v; }
        const int base = atomicAdd(L.cursor, all);
        for (int w = 0; w < 16; w++) s_sum[w] += base;
    }
    __syncthreads();
    if (i < nseg) L.end[i] = s_sum[wave] + sum - n;       // (the filing pass takes entries from here on and leaves the end)
}
template <bool AUX16, bool SIZED>
__global__ void __launch_bounds__(kSortThreads, 8)     // (two workgroups to a compute unit, for 16 - 20 bytes of spills a lane)
brick_file_kernel(TiledShape s, BrickDims d, BrickLists L, const void *off, const void *mask, SortWindow w, long n)
{
    typedef typename std::conditional<AUX16, bf16_t, float>::type AT;
    extern __shared__ __align__(16) unsigned char smem[];
    int *const s_cnt = reinterpret_cast<int *>(smem);
    const int nslot = w.wz * w.wy * w.wx;
    const SortUnit t = sort_unit(s, d, w);
    float c[kTaps][3], al[kTaps];
    sort_offsets<AUX16, SIZED>(s, off, t, c);
#pragma unroll
    for (int i = 0; i < kTaps; i++) {
        const int k = t.k0 + i * kTapGroups;
        al[i] = mask && k < t.k1 ? ld_auxT<AUX16>(mask, mask_index(s, t.b, t.g, k, t.p)) : 1.f;
    }
    for (int i = threadIdx.x; i <= nslot; i += kSortThreads) s_cnt[i] = 0;
    __syncthreads();
    const float size[3] = {c[0][0], c[0][1], c[0][2]};
    // slot << 4 | base voxel (slot -1: outside the window, `rank` is the entry; all ones: no point)
    int slot[kTaps], rank[kTaps];
#pragma unroll
    for (int i = 0; i < kTaps; i++) {
        const int k = t.k0 + i * kTapGroups;
        slot[i] = -1; rank[i] = 0;
        if (!t.ok || k >= t.k1) continue;
        const BrickPoint q = brick_point<AUX16, SIZED>(s, w, t, SIZED ? size : c[i], k);
        c[i][0] = q.hz; c[i][1] = q.hy; c[i][2] = q.hx;
        if (!q.in) continue;
        const int sl = sort_slot(w, t, q);
        slot[i] = (int)((unsigned)sl << 4 | q.cell);
        rank[i] = sl >= 0 ? atomicAdd(&s_cnt[sl], 1) : atomicAdd(&L.end[brick_seg(d, t.bg, q.zi, q.yq, q.xq)], 1);
    }
    // points outside the volume: behind the window's counts, a wavefront's together
    unsigned long long m[kTaps];
    int total = 0, out = 0;
#pragma unroll
    for (int i = 0; i < kTaps; i++) {
        m[i] = __ballot(t.ok && t.k0 + i * kTapGroups < t.k1 && slot[i] == -1);
        total += __popcll(m[i]);
    }
    const int lane = threadIdx.x & 63;
    if (total && lane == 0) out = atomicAdd(&s_cnt[nslot], total);
    __syncthreads();
    if (threadIdx.x == 0 && s_cnt[nslot]) s_cnt[nslot] = atomicAdd(L.cursor + 1, s_cnt[nslot]);
    for (int i = threadIdx.x; i < nslot; i += kSortThreads) {
        const int m = s_cnt[i];
        if (m) s_cnt[i] = atomicAdd(&L.end[sort_slot_seg(d, w, t, i)], m);
    }
    __syncthreads();
    // (everything that has been asked for is here: the stores below wait for nothing, least of all for one another)
    __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
    for (int i = 0; i < kTaps; i++) {
        const int k = t.k0 + i * kTapGroups;
        if (!t.ok || k >= t.k1) continue;
        const int at = slot[i] >= 0 ? s_cnt[slot[i] >> 4] + rank[i] : (slot[i] == -1 ? -1 : rank[i]);
        L.place[((long)t.bg * s.K + k) * s.P + t.p] = at;
        if (at < 0) continue;
        L.pt[at] = make_uint4((unsigned)(k * s.M + t.b * s.P + t.p) * 128u | (unsigned)(slot[i] & 15), __float_as_uint(c[i][1]),
                              __float_as_uint(c[i][2]), __float_as_uint(c[i][0]));
        L.alpha[at] = (mask && s.mact) ? mask_act<AT>(s.mact, al[i]) : al[i];
    }
    // points outside the volume: their rows among all groups' rows, listed downwards from the end of the entries (which the
    // points inside leave free)
    if (total == 0) return;
    int at = __builtin_amdgcn_readfirstlane(out) + s_cnt[nslot];
    unsigned *const end = reinterpret_cast<unsigned *>(L.pt + n) - 1;
#pragma unroll
    for (int i = 0; i < kTaps; i++) {
        if ((m[i] >> lane) & 1)
            end[-(long)(at + __popcll(m[i] & ((1ull << lane) - 1)))] =
                (unsigned)((t.g * s.K + t.k0 + i * kTapGroups) * s.M + t.b * s.P + t.p);
        at += __popcll(m[i]);
    }
}
// Workgroups of a pass over all points that needs no window: 256 positions, kPassTaps taps.  (A wavefront waits for the places,
// then for the sums they name: few taps in each of many.  Results of 27 and 7 taps, C3 and 2048 channels on 8x30x54, us: 9 taps
// 61, 36; 3 52, 16; 2 54, 12; 1 56, 10.)
constexpr int kPassTaps = 2;
struct PointUnit {
    int b, g, bg, k0, p;
};
D2C_DEV PointUnit point_unit(const TiledShape &s, int ngrp)
{
    const int nt = (int)gridDim.x, q = nt >> 3, r = nt & 7, xcd = blockIdx.x & 7;
    const int u = xcd * q + (xcd < r ? xcd : r) + (int)(blockIdx.x >> 3);
    const int npb = (s.P + 255) / 256, blk = u / ngrp;
    PointUnit t;
    t.bg = blk / npb; t.b = t.bg / s.G; t.g = t.bg - t.b * s.G;
    t.k0 = (u - blk * ngrp) * kPassTaps; t.p = (blk - t.bg * npb) * 256 + threadIdx.x;
    return t;
}

// ---- the weights as matrix operands -----------------------------------------------------------------------------------
// A corner weight is a float and stays one: it travels as three bfloat16 terms that add up to it exactly (its top 8
// significant bits, the next 8, the last 8), each multiplied with the bfloat16 rows and summed in float32 -- what fmaf
// of the float weight gives.  (Truncated, not rounded: no term is larger than the weight.)
// The pair of a row of two corners along x, in the row of four voxels of a brick: 16-bit elements x .. x + 1 of 8 bytes
// (`xs`: 16 x), zeros beside them.  The zeros are not products: a weight that is no number stays at its corners.
struct WeightRow {
    unsigned long long t[3];
};
D2C_DEV WeightRow weight_row(float w0, float w1, unsigned xs)
{
    WeightRow r;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const unsigned b0 = __float_as_uint(w0), b1 = __float_as_uint(w1);
        r.t[i] = (unsigned long long)__builtin_amdgcn_perm(b1, b0, 0x07060302u) << xs;
        w0 -= __uint_as_float(b0 & 0xffff0000u); w1 -= __uint_as_float(b1 & 0xffff0000u);
    }
    return r;
}

// ---- infinities and NaN ---------------------------------------------------------------------------------------------
// A product with a weight of zero is no product where the other factor is no number: 0 * inf would carry one bad voxel, or one
// bad grad_out position, into everything that shares a brick with it.  Weights that are no number stay at their corners
// (weight_row); bad rows are noticed -- the sampling kernel looks at every plane it takes, the gradient kernel at the sums
// of every plane it hands over, which such a row turns into no numbers -- and the points concerned are then worked out
// one by one, corner by corner, as the gathering kernels do: corners inside the volume whose distance along each axis is
// less than one voxel.  (Looking costs 0 - 0.3 % of a step: 2x256x8x30x54 700 -> 702 us, long clip 4704 and 4704.)
D2C_DEV bool any_lane(bool v) { return __builtin_amdgcn_ballot_w64(v) != 0; }
D2C_DEV bool no_number(float v) { return !(fabsf(v) < __builtin_inff()); }
// (of the pairs of bfloat16 of `n` words)
D2C_DEV bool no_number_bf16(const unsigned *w, int n)
{
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 m = {0, 0};
#pragma unroll
    for (int i = 0; i < n; i++) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu));
    return m.x >= 0x7f80 || m.y >= 0x7f80;
}
// one point of the block at (z, y0, x0), the same for all lanes
struct PointValues {
    unsigned row;                 // byte offset of its row
    int y, x;                     // base voxel
    float hz, hy, hx, alpha;
};
D2C_DEV PointValues point_of_lane(const uint4 &e, float alpha, int l, int y0, int x0)
{
    PointValues p;
    const unsigned q = (unsigned)__builtin_amdgcn_readlane((int)e.x, l);
    p.row = q & ~127u; p.y = y0 + (int)(q & 3u); p.x = x0 + (int)((q >> 2) & 3u);
    p.hy = lane_value(__uint_as_float(e.y), l); p.hx = lane_value(__uint_as_float(e.z), l); p.hz = lane_value(__uint_as_float(e.w), l);
    p.alpha = lane_value(alpha, l);
    return p;
}

// ---- the products -------------------------------------------------------------------------------------------------
// A workgroup takes a column of bricks (one 3 x 3 block of base voxels along y and x, a range of z) and up to four chunks
// of 64 channels, a wavefront each; all walk the same points, 32 at a time.  Going up in z, the upper plane of a brick is the
// lower one of the next: a plane's input rows and its grad_input sums stay where they are (plane z in slot z & 1),
// one plane is loaded and one is added to the accumulator per step.
//
// Matrix operands (v_mfma_f32_32x32x16_bf16):
//   T:  A = x rows (lane = voxel), B = grad-column rows (lane = point), both from LDS
//   gx: A = the weights, three bfloat16 terms, B = the rows, both through LDS (lane = point there, transposing reads)
// Voxel m of the brick: plane slot m / 16, y (m / 4) % 4, x m % 4.  A lane of T holds point lane % 32 and, in
// register r, voxel 8 * (r / 4) + 4 * (lane / 32) + r % 4: x = r % 4, slot = r / 8, y = 2 * ((r / 4) % 2) + lane / 32, so
// that of a point's two corner rows along y each half of the wavefront holds one.
struct BrickArgs {
    BrickDims d;
    BrickLists L;
    const void *xcl;         // [N][vol][Cin]
    const void *gcol;        // [chunk][tap][N*P][64 bfloat16 / 32 float]
    float *gxcl;             // [N][vol][Cin] sums (cleared), or NULL
    float2 *res;             // [set][point][2]: sum over its channels of (mask, x), (z, y) per unit of modulation; or NULL
    long nres;               // points per set
    int zlen, nzr;           // base planes per workgroup, ranges of them
    int nset;                // sets of up to kMaxWaves chunks
    int G, cpc, Cin, D, H, W, vol;
    long chunk_rows;         // K * M
};

constexpr int kMaxWaves = 4;
constexpr int kWeightLds = 3 * 32 * 64;                       // weights of 32 points
constexpr int kRowLds = 32 * 128, kRowLdsF = 3 * 32 * 64;     // a wavefront's rows of 32 points; float32: as three terms
D2C_DEV void lds_only_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
D2C_DEV void wave_fence() { asm volatile("" ::: "memory"); __builtin_amdgcn_wave_barrier(); }

// The wavefronts of a workgroup need the same weights.  SHARE: they take turns in making those of the next 32 points, a step
// ahead (the barrier in front of the sums over chunks keeps them in step), in two buffers of the workgroup; the first ones of a plane are waited for.
// Else, where there is one wavefront or a plane has few points, a buffer for each, filled when it is wanted.  (us, each its own first: 256 channels on
// 32x60x108, 27 taps, 862, 830; float32 on 2x8x30x54 283, 259; 2048 channels on 8x30x54, 7 taps, two steps to a plane, 230, 236.)
template <bool SHARE>
__global__ void __launch_bounds__(64 * kMaxWaves, 3) brick_grad_kernel(BrickArgs a, const int *__restrict__ seg_end, const int *__restrict__ seg_count)
{
    const int lane = threadIdx.x & 63, h = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    // A wavefront's grad-column rows of 32 points x 64 channels, and their weights [term][point][voxel of 32].  16-byte pieces of a row are
    // permuted so that neither the row-wise accesses (16 lanes on the same piece of 16 rows) nor the transposing reads
    // (4 rows x 64 bytes) meet a bank twice.
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *const s_g = smem + wave * kRowLds, *const s_w = smem + nw * kRowLds + (SHARE ? 0 : wave * kWeightLds);
    float2 *const s_part = reinterpret_cast<float2 *>(smem + nw * kRowLds + (SHARE ? 2 : nw) * kWeightLds);       // [2][wave][lane]: sums over a chunk each
    auto g_swz = [](int row) INLINE { return (((row >> 1) & 1) << 2) | (((row >> 2) & 1) << 1) | ((row >> 3) & 1); };

    // task: set of chunks, then block column along x, y, then z range, group and sample; an XCD takes a contiguous part of them
    const int nt = (int)gridDim.x, xq = nt >> 3, xr = nt & 7, xcd = blockIdx.x & 7;
    int t = xcd * xq + (xcd < xr ? xcd : xr) + (int)(blockIdx.x >> 3);
    const int set = t % a.nset; t /= a.nset;
    const int bx = t % a.d.nbx; t /= a.d.nbx;
    const int by = t % a.d.nby; t /= a.d.nby;
    const int zr = t % a.nzr; const int bg = t / a.nzr;
    const int b = bg / a.G, g = bg - b * a.G;
    const bool here = set * nw + wave < a.cpc;                       // (the last set can be short: a wavefront that only keeps step)
    const int cc0 = g * a.cpc + (here ? set * nw + wave : 0);        // its chunk
    const bool want_gx = a.gxcl != nullptr && here;
    const int res_bytes = a.res ? 16 : 0;
    const int y0 = by * 3 - 1, x0 = bx * 3 - 1;
    const int zi_lo = zr * a.zlen, zi_hi = min(zi_lo + a.zlen, a.d.nz);
    constexpr unsigned kNone = 0xFFFFFFF0u;                          // an offset past every buffer: nothing is stored

    f32x16 gacc[2];
#pragma unroll
    for (int r = 0; r < 16; r++) gacc[0][r] = gacc[1][r] = 0.f;

    // input rows as the operand of T: lane = voxel n of the brick, its 8 channels of every k-step.  load_plane changes
    // the lanes of slot z & 1 (zeros outside the volume).
    u32x4_t xa[4];
    auto load_plane = [&](int z) INLINE {
        int fn = n;
        opaque_v(fn);
        if ((fn >> 4) != (z & 1)) return;
        const int vox_y = y0 + ((fn >> 2) & 3), vox_x = x0 + (fn & 3);
        const bool in = vox_y >= 0 && vox_y < a.H && vox_x >= 0 && vox_x < a.W && z >= 0 && z < a.D;
        const bf16_t *xp = (const bf16_t *)a.xcl + ((long)b * a.vol + ((long)(in ? z : 0) * a.H + (in ? vox_y : 0)) * a.W + (in ? vox_x : 0)) * a.Cin
                           + cc0 * 64 + h * 8;
        for_each_const([&](auto I) INLINE {
            constexpr int ks = decltype(I)::value;
            xa[ks] = u32x4_t{0u, 0u, 0u, 0u};
            if (in && here) xa[ks] = *reinterpret_cast<const u32x4_t *>(xp + ks * 16);
        }, std::make_integer_sequence<int, 4>{});
    };
    // sums of plane z (slot z & 1) -> accumulator, and cleared.  (Through a buffer descriptor of the plane: an add that
    // goes nowhere has an offset past its end, and no branch stands between the adds.)
    int bad_from = 0x7fffffff;                           // the planes from here on are left to the end
    const unsigned plane_bytes = (unsigned)a.H * (unsigned)a.W * (unsigned)a.Cin * 4u;
    auto flush_plane = [&](int z) INLINE {
        const bool odd = z & 1;
        // (looked at: the sums of both planes, the points of the other one are among this one's)
        float all[2] = {0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 16; r++) { all[0] += gacc[0][r]; all[1] += gacc[1][r]; }
        if (any_lane(no_number(all[0] + all[1]))) bad_from = min(bad_from, z);
        const bool zin = z >= 0 && z < a.D && z < bad_from;
        // (worked out anew each time: kept across the points, these offsets would take the registers of the products)
        int fn = n, fh = h;
        opaque_v(fn); opaque_v(fh);
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.gxcl + ((long)b * a.vol + (long)(zin ? z : 0) * a.H * a.W) * a.Cin, 0,
                                                          (int)plane_bytes, 0x00020000);
        for_each_const([&](auto I) INLINE {
            constexpr int r = decltype(I)::value;
            constexpr int dy = 2 * (r >> 2), dx = r & 3;
            const int y = y0 + fh + dy, x = x0 + dx;
            const bool in = zin && y >= 0 && y < a.H && x >= 0 && x < a.W;
            const unsigned o = in ? (unsigned)((y * a.W + x) * a.Cin + cc0 * 64 + fn) * 4u : kNone;
            for_each_const([&](auto Q) INLINE {
                constexpr int q = decltype(Q)::value;
                const float v = odd ? gacc[q][8 + r] : gacc[q][r];
                gacc[q][r] = odd ? gacc[q][r] : 0.f;
                gacc[q][8 + r] = odd ? 0.f : gacc[q][8 + r];
                __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(v, rs, (int)o, q * 128, 0);
            }, std::make_integer_sequence<int, 2>{});
        }, std::make_integer_sequence<int, 8>{});
    };

    // LDS places of this lane: rows as they are loaded (8 lanes to a row: lanes of one load that each take 16 bytes of
    // another row cost the L1 four times the lookups), as the operand of T, weights as they are made, and transposing
    // reads of both (within 16 lanes, lane l element j comes from lane 4j + l/4, element l%4)
    const int pv = lane >> 3, pc = lane & 7;
    const unsigned g_st = lds_address(s_g) + pv * 128 + ((pc ^ g_swz(pv)) << 4);
    const unsigned g_ld = lds_address(s_g) + n * 128 + ((h ^ g_swz(n)) << 4);
    const unsigned w_st = lds_address(s_w) + n * 64 + (((h * 2) ^ ((n >> 2) & 3)) << 4);     // (^ 8 y: the lane's row y of voxels)
    const int tr_row = h * 8 + ((lane & 15) >> 2), tr_pc = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1), tr_in = (lane & 1) * 8;
    const unsigned g_tr = lds_address(s_g) + tr_row * 128 + ((tr_pc ^ g_swz(tr_row)) << 4) + tr_in;
    unsigned w_tr = lds_address(s_w) + tr_row * 64 + ((tr_pc ^ (h * 2)) << 4) + tr_in;
    auto tr_read = [](unsigned addr) INLINE {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(size_t)addr));
    };
    auto operand = [](uint2 lo, uint2 hi) INLINE { return __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y)); };

    // Points are worked on 32 at a time; entries are requested three such steps ahead, grad-column rows two.
    uint4 e0, e1, e2, e3;
    float a0, a1, a2, a3;
    u32x4_t row_a[4], row_b[4];
    int e_lo = 0, cnt = 0;
    auto entry = [&](int i, uint4 &q, float &al) INLINE {
        const int e = max(e_lo + min(i + n, cnt - 1), 0);
        q = a.L.pt[e]; al = a.L.alpha[e];
    };
    const auto rsg = __builtin_amdgcn_make_buffer_rsrc((bf16_t *)const_cast<void *>(a.gcol) + (long)cc0 * a.chunk_rows * 64, 0, (int)(unsigned)(a.chunk_rows * 128), 0x00020000);
    auto rows = [&](const uint4 &q, u32x4_t (&row)[4]) INLINE {
        for_each_const([&](auto I) INLINE {
            constexpr int i = decltype(I)::value;
            row[i] = __builtin_amdgcn_raw_buffer_load_b128(rsg, __builtin_amdgcn_ds_bpermute((i * 8 + pv) << 2, (int)(q.x & ~127u)) + pc * 16, 0, 0);
        }, std::make_integer_sequence<int, 4>{});
    };
    // what base plane zi - 1 needs: its points (the range `range` asked for) and the plane above it
    int r_lo, r_n;
    auto range = [&](int zi) INLINE {
        const int sg = brick_seg(a.d, bg, min(zi, zi_hi - 1), by, bx);
        r_lo = seg_end[sg]; r_n = seg_count[sg];
    };
    // weights of points i .. (lane = point, the 16 voxels of slot h): rows yb, yb + 1 of four voxels, zeros in the other two
    int wofs = 0;                                    // the buffer of this step's weights
    auto weights = [&](const uint4 &e, float al, int i, int to, bool low) INLINE {
        const unsigned yb = e.x & 3u, xs = (e.x & 12u) << 2;
        const float hy = __uint_as_float(e.y), hx = __uint_as_float(e.z), hz = __uint_as_float(e.w);
        const float wz = (i + n < cnt ? al : 0.f) * ((h != 0) == low ? 1.f - hz : hz);
        const float wy0 = wz * (1.f - hy), wy1 = wz * hy, lx = 1.f - hx;
        const WeightRow r0 = weight_row(wy0 * lx, wy0 * hx, xs), r1 = weight_row(wy1 * lx, wy1 * hx, xs);
        typedef __attribute__((address_space(3))) unsigned long long *lds64;
        const unsigned sy = yb << 3, st = w_st + to;
        const unsigned at0 = st ^ sy, at1 = st ^ (sy + 8), at2 = st ^ ((sy + 16) & 24), at3 = st ^ ((sy + 24) & 24);
#pragma unroll
        for (int q = 0; q < 3; q++) {
            *(lds64)(size_t)(at0 + q * 2048) = r0.t[q];
            *(lds64)(size_t)(at1 + q * 2048) = r1.t[q];
            *(lds64)(size_t)(at2 + q * 2048) = 0;
            *(lds64)(size_t)(at3 + q * 2048) = 0;
        }
    };
    auto begin = [&](int zi) INLINE {
        cnt = __builtin_amdgcn_readfirstlane(r_n); e_lo = __builtin_amdgcn_readfirstlane(r_lo) - cnt;
        if (cnt > 0) {
            entry(0, e0, a0);
            entry(32, e1, a1);
            entry(64, e2, a2);
        }
        load_plane(zi);
        if (cnt > 0) {
            rows(e0, row_a);
            rows(e1, row_b);
        }
    };
    int par = 0, turn = 0, turn2 = nw / 2;           // whose turn it is to store sums, to make weights
    range(zi_lo);
    load_plane(zi_lo - 1);
    begin(zi_lo);
    for (int zi = zi_lo; zi < zi_hi; zi++) {
        const int z = zi - 1;
        const bool low = z & 1;                      // slot of the base plane
        range(zi + 1);
        if (SHARE && cnt > 0) {
            if (turn2 == wave) weights(e0, a0, 0, wofs, low);
            lds_only_barrier();
        }
        auto step = [&](int i0, u32x4_t (&row)[4]) INLINE {
            // the rows to LDS, others requested in their place.  (The entry first: loads complete in order, and it is
            // wanted first.  Past the last point: its row again.)
            entry(i0 + 96, e3, a3);
            __builtin_amdgcn_sched_barrier(0);
            typedef __attribute__((address_space(3))) u32x4_t *lds128;
            *(lds128)(size_t)g_st = row[0];
            *(lds128)(size_t)((g_st ^ 16) + 1024) = row[1];
            *(lds128)(size_t)(g_st + 2048) = row[2];
            *(lds128)(size_t)((g_st ^ 16) + 3072) = row[3];
            rows(e2, row);
            __builtin_amdgcn_sched_barrier(0);
            const unsigned yb = e0.x & 3u, xs = (e0.x & 12u) << 2;
            const float hy = __uint_as_float(e0.y), hx = __uint_as_float(e0.z), hz = __uint_as_float(e0.w), lz = 1.f - hz;
            if constexpr (!SHARE) weights(e0, a0, i0, 0, low);
            else if (turn2 == wave && i0 + 32 < cnt) weights(e1, a1, i0 + 32, wofs ^ kWeightLds, low);
            wave_fence();
            // ---- the two products
            f32x16 T;
#pragma unroll
            for (int r = 0; r < 16; r++) T[r] = 0.f;
            for_each_const([&](auto KG) INLINE {
                constexpr int kg = decltype(KG)::value;            // 16 points, and half of T's channels
                const bf16x8_t wh = operand(tr_read(w_tr + kg * 1024), tr_read((w_tr ^ 16) + kg * 1024 + 256));
                const bf16x8_t wm = operand(tr_read(w_tr + kg * 1024 + 2048), tr_read((w_tr ^ 16) + kg * 1024 + 2304));
                const bf16x8_t wl = operand(tr_read(w_tr + kg * 1024 + 4096), tr_read((w_tr ^ 16) + kg * 1024 + 4352));
                for_each_const([&](auto Q) INLINE {
                    constexpr int q = decltype(Q)::value, ks = kg * 2 + q;
                    const u32x4_t gq = *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t *>((size_t)(g_ld ^ (ks * 32)));
                    T = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, xa[ks]), __builtin_bit_cast(bf16x8_t, gq), T, 0, 0, 0);
                    const bf16x8_t gb = operand(tr_read((g_tr ^ (q * 64)) + kg * 2048), tr_read((g_tr ^ (q * 64) ^ 32) + kg * 2048 + 512));
                    gacc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wh, gb, gacc[q], 0, 0, 0);
                    gacc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wm, gb, gacc[q], 0, 0, 0);
                    gacc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wl, gb, gacc[q], 0, 0, 0);
                }, std::make_integer_sequence<int, 2>{});
            }, std::make_integer_sequence<int, 2>{});
            wave_fence();
            // ---- grad_offset / grad_mask from the point's corner dots
            {
                const bool y1 = yb >= 1, y2 = yb >= 2, x1 = xs >= 16, x2 = xs >= 32;
                const bool q = h ? y2 : y1;                       // the corner row along y this half holds ...
                const bool hi = (y1 != y2) != (h != 0);           // ... and whether it is the upper one
                // (single registers from here on: a choice between two elements of T is not to become a variable index)
                float tv[16];
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    tv[r] = T[r];
                    opaque_v(tv[r]);
                }
                float sx[2], ex[2];
#pragma unroll
                for (int zz = 0; zz < 2; zz++) {
                    float ty[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) ty[i] = q ? tv[zz * 8 + 4 + i] : tv[zz * 8 + i];
                    const float d0 = x2 ? ty[2] : (x1 ? ty[1] : ty[0]);
                    const float d1 = x2 ? ty[3] : (x1 ? ty[2] : ty[1]);
                    sx[zz] = fmaf(hx, d1 - d0, d0);
                    ex[zz] = d1 - d0;
                }
                const float w0 = low ? hz : lz, w1 = low ? lz : hz;
                const float sz = fmaf(w1, sx[1], w0 * sx[0]), ez = fmaf(w1, ex[1], w0 * ex[0]);
                const float dz = low ? sx[0] - sx[1] : sx[1] - sx[0];
                const float wy = hi ? hy : 1.f - hy;
                const float r_m = wy * sz, r_y = hi ? sz : -sz, r_x = wy * ez, r_z = wy * dz;
                // the two halves of a point: lanes 0 - 31 end with (mask, x), the others with (z, y)
                const auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(r_m), __float_as_uint(r_z), false, false);
                const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(r_x), __float_as_uint(r_y), false, false);
                float2 r = make_float2(__uint_as_float(u[0]) + __uint_as_float(u[1]), __uint_as_float(v[0]) + __uint_as_float(v[1]));
                if (SHARE || nw > 1) {
                    // the chunks of the other wavefronts, which take turns in adding up and storing
                    s_part[(par * nw + wave) * 64 + lane] = r;
                    lds_only_barrier();
                    if (turn == wave) {
                        r = make_float2(0.f, 0.f);
                        for (int w = 0; w < nw; w++) {
                            const float2 q2 = s_part[(par * nw + w) * 64 + lane];
                            r.x += q2.x; r.y += q2.y;
                        }
                    }
                }
                // (a store of every lane through a descriptor of the 32 results: no branch, see flush_plane)
                typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
                const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.res + (set * a.nres + e_lo + i0) * 2, 0,
                                                                  turn == wave ? min(cnt - i0, 32) * res_bytes : 0, 0x00020000);
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(r.x), __float_as_uint(r.y)}, rs, n * 16 + h * 8, 0, 0);
                par ^= 1;
                if (++turn == nw) turn = 0;
                if (++turn2 == nw) turn2 = 0;
                if (SHARE) { w_tr += wofs ? -kWeightLds : kWeightLds; wofs ^= kWeightLds; }
            }
            e0 = e1; a0 = a1;
            e1 = e2; a1 = a2;
            e2 = e3; a2 = a3;
        };
        for (int i0 = 0; i0 < cnt; i0 += 64) {
            step(i0, row_a);
            if (i0 + 32 < cnt) step(i0 + 32, row_b);
        }
        // (the loads of the next base plane first: a wait for them then is no wait for the adds)
        if (zi + 1 < zi_hi) begin(zi + 1);
        if (want_gx) flush_plane(z);
    }
    if (want_gx) flush_plane(zi_hi - 1);
    if (bad_from >= zi_hi || !want_gx) return;
    // The planes whose sums hold infinities or NaN, and those above them, point by point (see above; lane = channel).
    for (int zi = max(bad_from, zi_lo); zi < zi_hi; zi++) {
        const int sg = brick_seg(a.d, bg, zi, by, bx);
        const int np = __builtin_amdgcn_readfirstlane(seg_count[sg]), lo = __builtin_amdgcn_readfirstlane(seg_end[sg]) - np;
        for (int i = 0; i < np; i += 64) {
            const int e = lo + min(i + lane, np - 1);
            const uint4 q = a.L.pt[e];
            const float al = a.L.alpha[e];
            for (int j = 0; j < min(np - i, 64); j++) {
                const PointValues p = point_of_lane(q, al, j, y0, x0);
                const float gv = bf16_to_f32(((const bf16_t *)a.gcol)[(long)cc0 * a.chunk_rows * 64 + (p.row >> 1) + lane]);
                for (int c = 0; c < 8; c++) {
                    const int z = zi - 1 + (c >> 2), y = p.y + ((c >> 1) & 1), x = p.x + (c & 1);
                    const float wz = c & 4 ? p.hz : 1.f - p.hz, wy = c & 2 ? p.hy : 1.f - p.hy, wx = c & 1 ? p.hx : 1.f - p.hx;
                    if (wz > 0.f && wy > 0.f && wx > 0.f && z >= bad_from && z >= 0 && z < a.D && y >= 0 && y < a.H && x >= 0 && x < a.W)
                        atomicAdd(a.gxcl + ((long)b * a.vol + ((long)z * a.H + y) * a.W + x) * a.Cin + cc0 * 64 + lane, p.alpha * wz * wy * wx * gv);
                }
            }
        }
    }
}

// ---- the same for float32 -------------------------------------------------------------------------------------------
// Rows are 32 channels (128 bytes).  Weights, rows and input each travel as three bfloat16 terms that add up to the float
// (what the third leaves is below 2^-26 of it); of the nine products of two numbers the six largest are summed in float32:
// what is left out is below 2^-25 of a product, less than a rounding in float32 leaves.  A wavefront takes its
// rows apart as they come (16 floats to a lane) into three planes [point][32 channels] in LDS, laid out like the weights'.
// A number that is none, or that the first term would round to an infinity, has no such terms: where a plane of the input or
// the rows of a step hold one, the corner dots of the step are worked out point by point; the sums of grad_input as above.
// To 32 points x 32 channels 24 matrix instructions, 364 of the vector ALU and 57 of LDS: the matrix pipes are busy 29 % of
// the time, instruction issue as a whole about 60 %, and the rows alone (0.72 GB) would take 0.14 ms.  Sized operator, 256 -> 256 channels on 2x8x30x54, us:
// 279 and 70 for the sort and the results; gathering (a dot product per corner and channel, then the lists of a voxel's points) 389 + 311.
// Not it: two wavefronts per SIMD with the rows of two steps in flight, 333.
// (numbers that the first term would round to an infinity count as none)
D2C_DEV void split3(float a, float b, uint32_t (&o)[3])
{
#pragma unroll
    for (int i = 0; i < 3; i++) {
        o[i] = pack_bf16x2(a, b);
        a -= __uint_as_float(o[i] << 16); b -= __uint_as_float(o[i] & 0xffff0000u);
    }
}
template <bool SHARE>
__global__ void __launch_bounds__(64 * kMaxWaves, 3) brick_grad_f32_kernel(BrickArgs a, const int *__restrict__ seg_end, const int *__restrict__ seg_count)
{
    const int lane = threadIdx.x & 63, h = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *const s_g = smem + wave * kRowLdsF, *const s_w = smem + nw * kRowLdsF + (SHARE ? 0 : wave * kWeightLds);   // rows and weights: [term][point][32]
    float2 *const s_part = reinterpret_cast<float2 *>(smem + nw * kRowLdsF + (SHARE ? 2 : nw) * kWeightLds);     // [2][wave][lane]: sums over a chunk each

    // task: as in brick_grad_kernel
    const int nt = (int)gridDim.x, xq = nt >> 3, xr = nt & 7, xcd = blockIdx.x & 7;
    int t = xcd * xq + (xcd < xr ? xcd : xr) + (int)(blockIdx.x >> 3);
    const int set = t % a.nset; t /= a.nset;
    const int bx = t % a.d.nbx; t /= a.d.nbx;
    const int by = t % a.d.nby; t /= a.d.nby;
    const int zr = t % a.nzr; const int bg = t / a.nzr;
    const int b = bg / a.G, g = bg - b * a.G;
    const bool here = set * nw + wave < a.cpc;
    const int cc0 = g * a.cpc + (here ? set * nw + wave : 0);
    const bool want_gx = a.gxcl != nullptr && here;
    const int res_bytes = a.res ? 16 : 0;
    const int y0 = by * 3 - 1, x0 = bx * 3 - 1;
    const int zi_lo = zr * a.zlen, zi_hi = min(zi_lo + a.zlen, a.d.nz);
    constexpr unsigned kNone = 0xFFFFFFF0u;
    const float *const xin = reinterpret_cast<const float *>(a.xcl), *const rows_in = reinterpret_cast<const float *>(a.gcol);

    f32x16 gacc;
#pragma unroll
    for (int r = 0; r < 16; r++) gacc[r] = 0.f;

    // input rows as the operand of T: lane = voxel n of the brick, 8 channels of each of two k-steps, three terms.
    // load_plane changes the lanes of slot z & 1.
    u32x4_t xa[2][3];
    bool bad_x = false;                                  // this lane's row holds infinities or NaN
    auto load_plane = [&](int z) INLINE {
        int fn = n;
        opaque_v(fn);
        if ((fn >> 4) != (z & 1)) return;
        const int vox_y = y0 + ((fn >> 2) & 3), vox_x = x0 + (fn & 3);
        const bool in = vox_y >= 0 && vox_y < a.H && vox_x >= 0 && vox_x < a.W && z >= 0 && z < a.D;
        const float *xp = xin + ((long)b * a.vol + ((long)(in ? z : 0) * a.H + (in ? vox_y : 0)) * a.W + (in ? vox_x : 0)) * a.Cin + cc0 * 32 + h * 8;
        float4 v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (in && here) v[i] = *reinterpret_cast<const float4 *>(xp + (i >> 1) * 16 + (i & 1) * 4);
        }
        unsigned top[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t lo[3], hi[3];
            split3(v[i].x, v[i].y, lo);
            split3(v[i].z, v[i].w, hi);
            top[2 * i] = lo[0]; top[2 * i + 1] = hi[0];
#pragma unroll
            for (int q = 0; q < 3; q++) { xa[i >> 1][q][(i & 1) * 2] = lo[q]; xa[i >> 1][q][(i & 1) * 2 + 1] = hi[q]; }
        }
        bad_x = no_number_bf16(top, 8);
    };
    int bad_from = 0x7fffffff;
    const unsigned plane_bytes = (unsigned)a.H * (unsigned)a.W * (unsigned)a.Cin * 4u;
    auto flush_plane = [&](int z) INLINE {
        const bool odd = z & 1;
        float all = 0.f;
#pragma unroll
        for (int r = 0; r < 16; r++) all += gacc[r];
        if (any_lane(no_number(all))) bad_from = min(bad_from, z);
        const bool zin = z >= 0 && z < a.D && z < bad_from;
        int fn = n, fh = h;
        opaque_v(fn); opaque_v(fh);
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.gxcl + ((long)b * a.vol + (long)(zin ? z : 0) * a.H * a.W) * a.Cin, 0,
                                                          (int)plane_bytes, 0x00020000);
        for_each_const([&](auto I) INLINE {
            constexpr int r = decltype(I)::value;
            constexpr int dy = 2 * (r >> 2), dx = r & 3;
            const int y = y0 + fh + dy, x = x0 + dx;
            const bool in = zin && y >= 0 && y < a.H && x >= 0 && x < a.W;
            const unsigned o = in ? (unsigned)((y * a.W + x) * a.Cin + cc0 * 32 + fn) * 4u : kNone;
            const float v = odd ? gacc[8 + r] : gacc[r];
            gacc[r] = odd ? gacc[r] : 0.f;
            gacc[8 + r] = odd ? 0.f : gacc[8 + r];
            __builtin_amdgcn_raw_ptr_buffer_atomic_fadd_f32(v, rs, (int)o, 0, 0);
        }, std::make_integer_sequence<int, 8>{});
    };

    // LDS places of this lane: rows and weights in the same layout, 64 bytes to a point, its 16-byte pieces permuted
    const int pv = lane >> 3, pc = lane & 7;
    const unsigned g_ld = lds_address(s_g) + n * 64, g_sw = (unsigned)((n >> 2) & 3);
    const unsigned w_st = lds_address(s_w) + n * 64 + (((h * 2) ^ ((n >> 2) & 3)) << 4);
    const int tr_row = h * 8 + ((lane & 15) >> 2), tr_pc = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1), tr_in = (lane & 1) * 8;
    const unsigned tr = tr_row * 64 + ((tr_pc ^ (h * 2)) << 4) + tr_in;
    const unsigned g_tr = lds_address(s_g) + tr;
    unsigned w_tr = lds_address(s_w) + tr;              // (of this step's buffer)
    auto tr_read = [](unsigned addr) INLINE {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(size_t)addr));
    };
    auto operand = [&](unsigned at, int kg, int term) INLINE {
        const uint2 lo = tr_read(at + kg * 1024 + term * 2048), hi = tr_read((at ^ 16) + kg * 1024 + 256 + term * 2048);
        return __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
    };

    uint4 e0, e1, e2;
    float a0, a1, a2;
    u32x4_t row_a[4];
    int e_lo = 0, cnt = 0;
    auto entry = [&](int i, uint4 &q, float &al) INLINE {
        const int e = max(e_lo + min(i + n, cnt - 1), 0);
        q = a.L.pt[e]; al = a.L.alpha[e];
    };
    const auto rsg = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(rows_in) + (long)cc0 * a.chunk_rows * 32, 0, (int)(unsigned)(a.chunk_rows * 128), 0x00020000);
    auto rows = [&](const uint4 &q, u32x4_t (&row)[4]) INLINE {
        for_each_const([&](auto I) INLINE {
            constexpr int i = decltype(I)::value;
            row[i] = __builtin_amdgcn_raw_buffer_load_b128(rsg, __builtin_amdgcn_ds_bpermute((i * 8 + pv) << 2, (int)(q.x & ~127u)) + pc * 16, 0, 0);
        }, std::make_integer_sequence<int, 4>{});
    };
    int r_lo, r_n;
    auto range = [&](int zi) INLINE {
        const int sg = brick_seg(a.d, bg, min(zi, zi_hi - 1), by, bx);
        r_lo = seg_end[sg]; r_n = seg_count[sg];
    };
    // weights of points i .. (lane = point, the 16 voxels of slot h): rows yb, yb + 1 of four voxels, zeros in the other two
    int wofs = 0;                                    // the buffer of this step's weights
    auto weights = [&](const uint4 &e, float al, int i, int to, bool low) INLINE {
        const unsigned yb = e.x & 3u, xs = (e.x & 12u) << 2;
        const float hy = __uint_as_float(e.y), hx = __uint_as_float(e.z), hz = __uint_as_float(e.w);
        const float wz = (i + n < cnt ? al : 0.f) * ((h != 0) == low ? 1.f - hz : hz);
        const float wy0 = wz * (1.f - hy), wy1 = wz * hy, lx = 1.f - hx;
        const WeightRow r0 = weight_row(wy0 * lx, wy0 * hx, xs), r1 = weight_row(wy1 * lx, wy1 * hx, xs);
        typedef __attribute__((address_space(3))) unsigned long long *lds64;
        const unsigned sy = yb << 3, st = w_st + to;
        const unsigned at0 = st ^ sy, at1 = st ^ (sy + 8), at2 = st ^ ((sy + 16) & 24), at3 = st ^ ((sy + 24) & 24);
#pragma unroll
        for (int q = 0; q < 3; q++) {
            *(lds64)(size_t)(at0 + q * 2048) = r0.t[q];
            *(lds64)(size_t)(at1 + q * 2048) = r1.t[q];
            *(lds64)(size_t)(at2 + q * 2048) = 0;
            *(lds64)(size_t)(at3 + q * 2048) = 0;
        }
    };
    auto begin = [&](int zi) INLINE {
        cnt = __builtin_amdgcn_readfirstlane(r_n); e_lo = __builtin_amdgcn_readfirstlane(r_lo) - cnt;
        if (cnt > 0) {
            entry(0, e0, a0);
            entry(32, e1, a1);
        }
        load_plane(zi);
        if (cnt > 0) {
            rows(e0, row_a);
        }
    };
    int par = 0, turn = 0, turn2 = nw / 2;           // whose turn it is to store sums, to make weights
    range(zi_lo);
    load_plane(zi_lo - 1);
    begin(zi_lo);
    for (int zi = zi_lo; zi < zi_hi; zi++) {
        const int z = zi - 1;
        const bool low = z & 1;                      // slot of the base plane
        range(zi + 1);
        const bool bad_plane = any_lane(bad_x);
        if (SHARE && cnt > 0) {
            if (turn2 == wave) weights(e0, a0, 0, wofs, low);
            lds_only_barrier();
        }
        auto step = [&](int i0, u32x4_t (&row)[4]) INLINE {
            entry(i0 + 64, e2, a2);
            __builtin_amdgcn_sched_barrier(0);
            // the rows to LDS, term by term; others requested in their place
            unsigned top[8];
            for_each_const([&](auto I) INLINE {
                constexpr int i = decltype(I)::value;
                const float v[4] = {__uint_as_float(row[i][0]), __uint_as_float(row[i][1]), __uint_as_float(row[i][2]), __uint_as_float(row[i][3])};
                uint32_t lo[3], hi[3];
                split3(v[0], v[1], lo);
                split3(v[2], v[3], hi);
                top[2 * i] = lo[0]; top[2 * i + 1] = hi[0];
                const int pt = i * 8 + pv;
                const unsigned at = lds_address(s_g) + pt * 64 + (((pc >> 1) ^ ((pt >> 2) & 3)) << 4) + (pc & 1) * 8;
                typedef __attribute__((address_space(3))) unsigned long long *lds64;
#pragma unroll
                for (int q = 0; q < 3; q++) *(lds64)(size_t)(at + q * 2048) = (unsigned long long)hi[q] << 32 | lo[q];
            }, std::make_integer_sequence<int, 4>{});
            const bool bad = bad_plane || any_lane(no_number_bf16(top, 8));
            rows(e1, row);
            __builtin_amdgcn_sched_barrier(0);
            const unsigned yb = e0.x & 3u, xs = (e0.x & 12u) << 2;
            const float hy = __uint_as_float(e0.y), hx = __uint_as_float(e0.z), hz = __uint_as_float(e0.w), lz = 1.f - hz;
            if constexpr (!SHARE) weights(e0, a0, i0, 0, low);
            else if (turn2 == wave && i0 + 32 < cnt) weights(e1, a1, i0 + 32, wofs ^ kWeightLds, low);
            wave_fence();
            // ---- the two products, the smallest terms first
            f32x16 T;
#pragma unroll
            for (int r = 0; r < 16; r++) T[r] = 0.f;
            constexpr int order[6][2] = {{1, 1}, {0, 2}, {2, 0}, {0, 1}, {1, 0}, {0, 0}};
            for_each_const([&](auto KG) INLINE {
                constexpr int kg = decltype(KG)::value;            // 16 channels
                bf16x8_t gq[3];
#pragma unroll
                for (int q = 0; q < 3; q++)
                    gq[q] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const __attribute__((address_space(3))) u32x4_t *>(
                                                   (size_t)(g_ld + (((kg * 2 + h) ^ g_sw) << 4) + q * 2048)));
#pragma unroll
                for (int i = 0; i < 6; i++)
                    T = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, xa[kg][order[i][0]]), gq[order[i][1]], T, 0, 0, 0);
            }, std::make_integer_sequence<int, 2>{});
            __builtin_amdgcn_sched_barrier(0);
            for_each_const([&](auto KG) INLINE {
                constexpr int kg = decltype(KG)::value;            // 16 points
                bf16x8_t w[3], gb[3];
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    w[q] = operand(w_tr, kg, q);
                    gb[q] = operand(g_tr, kg, q);
                }
#pragma unroll
                for (int i = 0; i < 6; i++) gacc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[order[i][0]], gb[order[i][1]], gacc, 0, 0, 0);
            }, std::make_integer_sequence<int, 2>{});
            wave_fence();
            // ---- grad_offset / grad_mask from the point's corner dots
            {
                const bool y1 = yb >= 1, y2 = yb >= 2, x1 = xs >= 16, x2 = xs >= 32;
                const bool q = h ? y2 : y1;
                const bool hi = (y1 != y2) != (h != 0);
                float tv[16];
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    tv[r] = T[r];
                    opaque_v(tv[r]);
                }
                float d[2][2];                                    // [plane slot][corner along x] of the row along y that this half holds
#pragma unroll
                for (int zz = 0; zz < 2; zz++) {
                    float ty[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) ty[i] = q ? tv[zz * 8 + 4 + i] : tv[zz * 8 + i];
                    d[zz][0] = x2 ? ty[2] : (x1 ? ty[1] : ty[0]);
                    d[zz][1] = x2 ? ty[3] : (x1 ? ty[2] : ty[1]);
                }
                if (__builtin_expect(bad, 0)) {
                    // point by point (lane = channel of either half, which takes one plane): corner dots as plain sums
                    for (int j = 0; j < min(cnt - i0, 32); j++) {
                        const PointValues p = point_of_lane(e0, a0, j, y0, x0);
                        const float gv = rows_in[(long)cc0 * a.chunk_rows * 32 + (p.row >> 2) + n];
                        float dot[4];                             // y, x of plane z + h
#pragma unroll
                        for (int c = 0; c < 4; c++) {
                            const int zc = z + h, yc = p.y + (c >> 1), xc = p.x + (c & 1);
                            const bool in = here && zc >= 0 && zc < a.D && yc >= 0 && yc < a.H && xc >= 0 && xc < a.W;
                            float v = in ? gv * xin[((long)b * a.vol + ((long)zc * a.H + yc) * a.W + xc) * a.Cin + cc0 * 32 + n] : 0.f;
#pragma unroll
                            for (int m = 1; m < 32; m <<= 1) v += __shfl_xor(v, m, 64);
                            dot[c] = v;
                        }
                        // (plane z + h lies in slot low ^ h: what lane j of half 0, 1 wants of either half)
                        const int ry = hi ? 1 : 0;
#pragma unroll
                        for (int zz = 0; zz < 2; zz++)
#pragma unroll
                            for (int xx = 0; xx < 2; xx++) {
                                const float v0 = lane_value(dot[xx], ((zz != 0) != low) ? 32 : 0), v1 = lane_value(dot[2 + xx], ((zz != 0) != low) ? 32 : 0);
                                if (n == j) d[zz][xx] = ry ? v1 : v0;
                            }
                    }
                }
                float sx[2], ex[2];
#pragma unroll
                for (int zz = 0; zz < 2; zz++) {
                    sx[zz] = fmaf(hx, d[zz][1] - d[zz][0], d[zz][0]);
                    ex[zz] = d[zz][1] - d[zz][0];
                }
                const float w0 = low ? hz : lz, w1 = low ? lz : hz;
                const float sz = fmaf(w1, sx[1], w0 * sx[0]), ez = fmaf(w1, ex[1], w0 * ex[0]);
                const float dz = low ? sx[0] - sx[1] : sx[1] - sx[0];
                const float wy = hi ? hy : 1.f - hy;
                const float r_m = wy * sz, r_y = hi ? sz : -sz, r_x = wy * ez, r_z = wy * dz;
                const auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(r_m), __float_as_uint(r_z), false, false);
                const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(r_x), __float_as_uint(r_y), false, false);
                float2 r = make_float2(__uint_as_float(u[0]) + __uint_as_float(u[1]), __uint_as_float(v[0]) + __uint_as_float(v[1]));
                if (SHARE || nw > 1) {
                    s_part[(par * nw + wave) * 64 + lane] = r;
                    lds_only_barrier();
                    if (turn == wave) {
                        r = make_float2(0.f, 0.f);
                        for (int w = 0; w < nw; w++) {
                            const float2 q2 = s_part[(par * nw + w) * 64 + lane];
                            r.x += q2.x; r.y += q2.y;
                        }
                    }
                }
                typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
                const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.res + (set * a.nres + e_lo + i0) * 2, 0,
                                                                  turn == wave ? min(cnt - i0, 32) * res_bytes : 0, 0x00020000);
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(r.x), __float_as_uint(r.y)}, rs, n * 16 + h * 8, 0, 0);
                par ^= 1;
                if (++turn == nw) turn = 0;
                if (++turn2 == nw) turn2 = 0;
                if (SHARE) { w_tr += wofs ? -kWeightLds : kWeightLds; wofs ^= kWeightLds; }
            }
            e0 = e1; a0 = a1;
            e1 = e2; a1 = a2;
        };
        for (int i0 = 0; i0 < cnt; i0 += 32) step(i0, row_a);
        if (zi + 1 < zi_hi) begin(zi + 1);
        if (want_gx) flush_plane(z);
    }
    if (want_gx) flush_plane(zi_hi - 1);
    if (bad_from >= zi_hi || !want_gx) return;
    // (as in brick_grad_kernel; lane = channel)
    for (int zi = max(bad_from, zi_lo); zi < zi_hi; zi++) {
        const int sg = brick_seg(a.d, bg, zi, by, bx);
        const int np = __builtin_amdgcn_readfirstlane(seg_count[sg]), lo = __builtin_amdgcn_readfirstlane(seg_end[sg]) - np;
        for (int i = 0; i < np; i += 64) {
            const int e = lo + min(i + lane, np - 1);
            const uint4 q = a.L.pt[e];
            const float al = a.L.alpha[e];
            for (int j = 0; j < min(np - i, 64); j++) {
                const PointValues p = point_of_lane(q, al, j, y0, x0);
                if (h) continue;
                const float gv = rows_in[(long)cc0 * a.chunk_rows * 32 + (p.row >> 2) + n];
                for (int c = 0; c < 8; c++) {
                    const int z = zi - 1 + (c >> 2), y = p.y + ((c >> 1) & 1), x = p.x + (c & 1);
                    const float wz = c & 4 ? p.hz : 1.f - p.hz, wy = c & 2 ? p.hy : 1.f - p.hy, wx = c & 1 ? p.hx : 1.f - p.hx;
                    if (wz > 0.f && wy > 0.f && wx > 0.f && z >= bad_from && z >= 0 && z < a.D && y >= 0 && y < a.H && x >= 0 && x < a.W)
                        atomicAdd(a.gxcl + ((long)b * a.vol + ((long)z * a.H + y) * a.W + x) * a.Cin + cc0 * 32 + n, p.alpha * wz * wy * wx * gv);
                }
            }
        }
    }
}

// ---- sampled columns ------------------------------------------------------------------------------------------------
// col[chunk][tap][rows][64] = modulation * interpolated input of every point (rows: N*P and a few): x^T[64 channels, 32 voxels] * W[32 voxels, 32
// points], three bfloat16 terms of the weights.  W is made by the lanes that hold the points, in the operand's own order
// (lane = point, half h of the wavefront: the voxels of rows y = 2h, 2h + 1 of each plane); the brick's input is kept as
// the other operand, one plane changed per step in z.  Rows leave whole, through LDS.  Bound by the rows it writes:
// 5.6 M points x 256 channels (32x60x108, 27 taps), 2.9 GB: 730 us (the whole forward pass: 2.3 ms gathering, 1.7 ms sorted).
// (Workgroups as in brick_grad_kernel: a column of bricks, a wavefront per chunk.)
struct BrickSampleArgs {
    BrickDims d;
    BrickLists L;
    const bf16_t *xcl;       // [N][vol][Cin]
    bf16_t *col;
    int zlen, nzr, nset, G, cpc, Cin, D, H, W, vol;
    long chunk_rows;         // K * rows of a tap
    int K, rows, pad;        // taps; rows of a tap, those beyond N*P
    int M, nzero;            // N*P; workgroups in front that clear rows
    long npoint;
    FastDiv dM, dKM;
};
__global__ void __launch_bounds__(64 * kMaxWaves, 4) brick_sample_kernel(BrickSampleArgs a, const int *__restrict__ seg_end, const int *__restrict__ seg_count)
{
    const int lane = threadIdx.x & 63, h = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nw = blockDim.x >> 6;
    // (of as many wavefronts as there are: with four times what one needs, workgroups of one were ten to a compute unit: 512 channels in 8
    // groups on 2x8x30x54 206 us, with sixteen 194)
    extern __shared__ __align__(16) unsigned char smem[];
    unsigned char *const s_r = smem + wave * kRowLds;                // a plane's 16 input rows; 32 rows on their way out
    const int pv = lane >> 3, pc = lane & 7;
    if ((int)blockIdx.x < a.nzero) {
        // rows of the points outside the volume, and those behind the last position: zeros (8 lanes to a chunk's row)
        const int w = (int)blockIdx.x * nw + wave, nwave = a.nzero * nw, nout = a.L.cursor[1];
        const unsigned *const end = reinterpret_cast<const unsigned *>(a.L.pt + a.npoint) - 1;
        for (int o0 = w * 64; o0 < nout; o0 += nwave * 64) {
            const unsigned e = o0 + lane < nout ? end[-(long)(o0 + lane)] : 0u;
            for (int i = 0; i < 64 && o0 + i < nout; i += 8) {
                const int o = __builtin_amdgcn_ds_bpermute((i + pv) << 2, (int)e);
                if (o0 + i + pv >= nout) continue;
                const int g = fdiv(o, a.dKM), r = o - g * (a.K * a.M), row = r + fdiv(r, a.dM) * a.pad;
                for (int c = 0; c < a.cpc; c++)
                    reinterpret_cast<uint4 *>(a.col + ((long)(g * a.cpc + c) * a.chunk_rows + row) * 64)[pc] = make_uint4(0, 0, 0, 0);
            }
        }
        const int tails = a.G * a.cpc * a.K * a.pad;
        for (int i = w * 8 + pv; i < tails; i += nwave * 8) {
            const int t = i / a.pad;
            reinterpret_cast<uint4 *>(a.col + ((long)t * a.rows + a.M + (i - t * a.pad)) * 64)[pc] = make_uint4(0, 0, 0, 0);
        }
        return;
    }
    const int bid = (int)blockIdx.x - a.nzero, nt = (int)gridDim.x - a.nzero, xq = nt >> 3, xr = nt & 7, xcd = bid & 7;
    int t = xcd * xq + (xcd < xr ? xcd : xr) + (bid >> 3);
    const int set = t % a.nset; t /= a.nset;
    const int bx = t % a.d.nbx; t /= a.d.nbx;
    const int by = t % a.d.nby; t /= a.d.nby;
    const int zr = t % a.nzr; const int bg = t / a.nzr;
    const int b = bg / a.G, g = bg - b * a.G;
    if (set * nw + wave >= a.cpc) return;
    const int cc0 = g * a.cpc + set * nw + wave;
    const int y0 = by * 3 - 1, x0 = bx * 3 - 1;
    const int zi_lo = zr * a.zlen, zi_hi = min(zi_lo + a.zlen, a.d.nz);

    uint4 pl[2];
    auto load_plane = [&](int z) INLINE {
        for_each_const([&](auto I) INLINE {
            constexpr int i = decltype(I)::value;
            const int v = i * 8 + pv, y = y0 + (v >> 2), x = x0 + (v & 3);
            pl[i] = make_uint4(0, 0, 0, 0);
            if (z >= 0 && z < a.D && y >= 0 && y < a.H && x >= 0 && x < a.W)
                pl[i] = *reinterpret_cast<const uint4 *>(a.xcl + ((long)b * a.vol + ((long)z * a.H + y) * a.W + x) * a.Cin + cc0 * 64 + pc * 8);
        }, std::make_integer_sequence<int, 2>{});
    };
    // the plane as matrix operand: lane = channel, 8 voxels (half h: y = 2h, 2h + 1).  The channel of a lane is the one that
    // makes a lane of the result hold 16 consecutive channels of its point: row m of the operand = channel
    // 16 * ((m >> 2) & 1) + 4 * (m >> 3) + (m & 3).
    const int q4 = ((lane >> 4) & 1) * 4 + (lane & 3), ch = (q4 & 1) * 16 + (q4 >> 1) * 4;
    const unsigned p_tr = lds_address(s_r) + (h * 8 + ((lane & 15) >> 2)) * 128 + ch * 2;
    auto tr_read = [](unsigned addr) INLINE {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s *)(size_t)addr));
    };
    bf16x8_t xl[2], xh[2];                                           // [channels 0-31, 32-63] of the lower and the upper plane
    bool bad_l, bad_h = false;                                       // infinities or NaN in them
    auto take_plane = [&]() INLINE {
        const unsigned w[8] = {pl[0].x, pl[0].y, pl[0].z, pl[0].w, pl[1].x, pl[1].y, pl[1].z, pl[1].w};
        bad_h = any_lane(no_number_bf16(w, 8));
        for_each_const([&](auto I) INLINE {
            constexpr int i = decltype(I)::value;
            *reinterpret_cast<uint4 *>(s_r + (i * 8 + pv) * 128 + pc * 16) = pl[i];
        }, std::make_integer_sequence<int, 2>{});
        wave_fence();
        for_each_const([&](auto C) INLINE {
            constexpr int c = decltype(C)::value;
            const uint2 lo = tr_read(p_tr + c * 64), hi = tr_read(p_tr + c * 64 + 512);
            xh[c] = __builtin_bit_cast(bf16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
        }, std::make_integer_sequence<int, 2>{});
        wave_fence();
    };
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.col + (long)cc0 * a.chunk_rows * 64, 0, (int)(unsigned)(a.chunk_rows * 128), 0x00020000);
    constexpr unsigned kNone = 0xFFFFFFF0u;
    // rows on their way out: written 16 bytes a time by the lane of the point, read 8 lanes to a row; pieces permuted against
    // bank conflicts (16 lanes on one piece of 16 rows)
    const int swz = (n >> 1) & 7;

    auto range = [&](int zi, int &lo, int &cnt) INLINE {
        const int sg = brick_seg(a.d, bg, min(zi, zi_hi - 1), by, bx);
        cnt = __builtin_amdgcn_readfirstlane(seg_count[sg]); lo = __builtin_amdgcn_readfirstlane(seg_end[sg]) - cnt;
    };
    uint4 e0, e1;
    float a0, a1;
    auto entry = [&](int lo, int cnt, int i, uint4 &q, float &al) INLINE {
        const int e = max(lo + min(i + n, cnt - 1), 0);
        q = a.L.pt[e]; al = a.L.alpha[e];
    };
    int lo, cnt;
    range(zi_lo, lo, cnt);
    load_plane(zi_lo - 1);
    entry(lo, cnt, 0, e0, a0);
    take_plane();
    load_plane(zi_lo);
    for (int zi = zi_lo; zi < zi_hi; zi++) {
        xl[0] = xh[0]; xl[1] = xh[1];
        bad_l = bad_h;
        take_plane();
        int nlo, ncnt;
        range(zi + 1, nlo, ncnt);
        load_plane(zi + 1);
        for (int i0 = 0; i0 < cnt; i0 += 32) {
            // (the next entries: of this block, or the first of the next plane's)
            if (i0 + 32 < cnt) entry(lo, cnt, i0 + 32, e1, a1);
            else entry(nlo, ncnt, 0, e1, a1);
            const unsigned xs = (e0.x & 12u) << 2;
            const int dy = 2 * h - (int)(e0.x & 3u);                     // the half's first row of voxels, from the base voxel
            const float hy = __uint_as_float(e0.y), hx = __uint_as_float(e0.z), hz = __uint_as_float(e0.w), lx = 1.f - hx;
            f32x16 r0, r1;
#pragma unroll
            for (int r = 0; r < 16; r++) r0[r] = r1[r] = 0.f;
            for_each_const([&](auto S) INLINE {
                constexpr int slot = decltype(S)::value;
                const float wz = a0 * (slot ? hz : 1.f - hz), wy0 = wz * (1.f - hy), wy1 = wz * hy;
                const float u0 = dy == 0 ? wy0 : (dy == 1 ? wy1 : 0.f), u1 = dy == -1 ? wy0 : (dy == 0 ? wy1 : 0.f);
                const WeightRow w0 = weight_row(u0 * lx, u0 * hx, xs), w1 = weight_row(u1 * lx, u1 * hx, xs);
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const bf16x8_t wt = __builtin_bit_cast(bf16x8_t, make_uint4((unsigned)w0.t[i], (unsigned)(w0.t[i] >> 32),
                                                                                (unsigned)w1.t[i], (unsigned)(w1.t[i] >> 32)));
                    r0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(slot ? xh[0] : xl[0], wt, r0, 0, 0, 0);
                    r1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(slot ? xh[1] : xl[1], wt, r1, 0, 0, 0);
                }
            }, std::make_integer_sequence<int, 2>{});
            for_each_const([&](auto P) INLINE {
                constexpr int q = decltype(P)::value, c = q >> 1, r = (q & 1) * 8;      // channels 32 c + 16 h + r ..
                const f32x16 &v = c ? r1 : r0;
                *reinterpret_cast<uint4 *>(s_r + n * 128 + (((c * 4 + h * 2 + (q & 1)) ^ swz) << 4)) =
                    make_uint4(pack_bf16x2(v[r], v[r + 1]), pack_bf16x2(v[r + 2], v[r + 3]), pack_bf16x2(v[r + 4], v[r + 5]),
                               pack_bf16x2(v[r + 6], v[r + 7]));
            }, std::make_integer_sequence<int, 4>{});
            if (__builtin_expect(bad_l || bad_h, 0)) {
                // point by point (lane = channel), over what the products have left in LDS (stores of another type: kept behind those)
                wave_fence();
                for (int j = 0; j < min(cnt - i0, 32); j++) {
                    const PointValues p = point_of_lane(e0, a0, j, y0, x0);
                    float v = 0.f;
                    for (int c = 0; c < 8; c++) {
                        const int z = zi - 1 + (c >> 2), y = p.y + ((c >> 1) & 1), x = p.x + (c & 1);
                        const float wz = c & 4 ? p.hz : 1.f - p.hz, wy = c & 2 ? p.hy : 1.f - p.hy, wx = c & 1 ? p.hx : 1.f - p.hx;
                        if (wz > 0.f && wy > 0.f && wx > 0.f && p.alpha != 0.f && z >= 0 && z < a.D && y >= 0 && y < a.H && x >= 0 && x < a.W)
                            v = fmaf(wz * wy * wx * p.alpha,
                                     bf16_to_f32(a.xcl[((long)b * a.vol + ((long)z * a.H + y) * a.W + x) * a.Cin + cc0 * 64 + lane]), v);
                    }
                    *reinterpret_cast<bf16_t *>(s_r + j * 128 + (((lane >> 3) ^ ((j >> 1) & 7)) << 4) + (lane & 7) * 2) = f32_to_bf16(v);
                }
            }
            wave_fence();
            const unsigned to = (e0.x & ~127u) + (unsigned)(fdiv((int)(e0.x >> 7), a.dM) * a.pad) * 128u;      // (the entry counts N*P rows per tap)
            for_each_const([&](auto I) INLINE {
                constexpr int i = decltype(I)::value;
                const int row = i * 8 + pv;
                const u32x4_t v = *reinterpret_cast<const u32x4_t *>(s_r + row * 128 + ((pc ^ ((row >> 1) & 7)) << 4));
                const unsigned o = (unsigned)__builtin_amdgcn_ds_bpermute(row << 2, (int)to) + pc * 16;
                __builtin_amdgcn_raw_buffer_store_b128(v, rs, i0 + row < cnt ? (int)o : (int)kNone, 0, 2);
            }, std::make_integer_sequence<int, 4>{});
            wave_fence();
            e0 = e1; a0 = a1;
        }
        // (a plane without points has asked for nothing: the next one's entries)
        if (cnt == 0) entry(nlo, ncnt, 0, e0, a0);
        lo = nlo; cnt = ncnt;
    }
}

// ---- per-point sums -> gradients in their storage type and layout --------------------------------------------------
D2C_DEV void brick_point_sums(const float2 *res, long nres, int nset, int at, float2 &mx, float2 &zy)
{
    mx = zy = make_float2(0.f, 0.f);
    if (at < 0) return;
    for (int i = 0; i < nset; i++) {
        const float4 v = reinterpret_cast<const float4 *>(res)[i * nres + at];
        mx.x += v.x; mx.y += v.y; zy.x += v.z; zy.y += v.w;
    }
}
template <bool AUX16>
__global__ void __launch_bounds__(256)
brick_finish_kernel(TiledShape s, BrickLists L, const float2 *res, long nres, int nset, const void *mask, void *goff, void *gmask,
                    int ngrp)
{
    typedef typename std::conditional<AUX16, bf16_t, float>::type AT;
    const PointUnit un = point_unit(s, ngrp);
    const int k0 = un.k0, bg = un.bg, b = un.b, g = un.g, p = un.p;
    if (p >= s.P) return;
    int at[kPassTaps];
    float al[kPassTaps];
    float2 mx[kPassTaps], zy[kPassTaps];
#pragma unroll
    for (int i = 0; i < kPassTaps; i++) {
        const int k = min(k0 + i, s.K - 1);
        at[i] = L.place[((long)bg * s.K + k) * s.P + p];
        al[i] = mask ? ld_auxT<AUX16>(mask, mask_index(s, b, g, k, p)) : 1.f;
    }
#pragma unroll
    for (int i = 0; i < kPassTaps; i++) brick_point_sums(res, nres, nset, at[i], mx[i], zy[i]);
#pragma unroll
    for (int i = 0; i < kPassTaps; i++) {
        const int k = k0 + i;
        if (k >= s.K) break;
        const bool in = at[i] >= 0;
        if (mask && s.mact) { al[i] = mask_act<AT>(s.mact, al[i]); mx[i].x *= mask_act_grad(s.mact, al[i]); }
        if (gmask) reinterpret_cast<AT *>(gmask)[mask_index(s, b, g, k, p)] = f32_to_elem<AT>(in ? mx[i].x : 0.f);
        if (goff) {
            AT *o = reinterpret_cast<AT *>(goff) + offset_index(s, b, g, k, p);
            o[0] = f32_to_elem<AT>(in && (s.axes & 1) ? al[i] * zy[i].x : 0.f);
            o[s.P] = f32_to_elem<AT>(in && (s.axes & 2) ? al[i] * zy[i].y : 0.f);
            o[2 * (long)s.P] = f32_to_elem<AT>(in && (s.axes & 4) ? al[i] * mx[i].y : 0.f);
        }
    }
}
// Size-map source: d(offset_a) / d(size_a) = base_a[k_a], so the taps of a position add up; the axes that a channel of
// the raw map feeds add up, times the derivative of the size activation.  A workgroup is 64 positions x kTapShares shares of the
// taps.  (Four shares leave a third of the chip's wavefronts out: 1024 -> 256 channels on 8x30x54, 27 taps, 4, 9 and 14 shares 28, 18
// and 17 us; 256 channels on 2x8x30x54, float32, 24, 18 and 20.)
constexpr int kTapShares = 9;
template <bool AUX16>
__global__ void __launch_bounds__(64 * kTapShares)
brick_finish_size_kernel(TiledShape s, BrickLists L, const float2 *res, long nres, int nset, const void *mask, const void *raw,
                         void *graw, void *gmask)
{
    typedef typename std::conditional<AUX16, bf16_t, float>::type AT;
    __shared__ float s_sum[kTapShares][3][64];
    const int b = blockIdx.y, lane = threadIdx.x & 63, part = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    float sum[3] = {0.f, 0.f, 0.f};
    if (p < s.P)
#pragma unroll 4
        for (int k = part; k < s.K; k += kTapShares) {
            const int at = L.place[((long)b * s.K + k) * s.P + p];
            float2 mx, zy;
            brick_point_sums(res, nres, nset, at, mx, zy);
            float al = 1.f;
            if (mask) {
                const long mi = mask_index(s, b, 0, k, p);
                al = ld_auxT<AUX16>(mask, mi);
                if (s.mact) { al = mask_act<AT>(s.mact, al); mx.x *= mask_act_grad(s.mact, al); }
                if (gmask) reinterpret_cast<AT *>(gmask)[mi] = f32_to_elem<AT>(at < 0 ? 0.f : mx.x);
            }
            if (at < 0) continue;
            const int kx = k % s.geo.kw, ky = (k / s.geo.kw) % s.geo.kh, kz = k / (s.geo.kw * s.geo.kh);
            sum[0] += s.ss.base[0][kz] * (al * zy.x);
            sum[1] += s.ss.base[1][ky] * (al * zy.y);
            sum[2] += s.ss.base[2][kx] * (al * mx.y);
        }
#pragma unroll
    for (int ax = 0; ax < 3; ax++) s_sum[part][ax][lane] = sum[ax];
    __syncthreads();
    const int c = part;                               // channel of the map
    if (!graw || p >= s.P || c >= mode_channels(s.ss.mode)) return;
    float v = 0.f;
#pragma unroll
    for (int ax = 0; ax < 3; ax++)
        if (axis_channel(s.ss.mode, ax) == c)
#pragma unroll
            for (int i = 0; i < kTapShares; i++) v += s_sum[i][ax][lane];
    const long ri = (long)b * s.obs + (long)c * s.P + p;
    v *= size_act_grad(s.ss.act, ld_auxT<AUX16>(raw, ri));
    reinterpret_cast<AT *>(graw)[ri] = f32_to_elem<AT>(v);
}

BrickDims brick_dims(const TiledShape &s) { return BrickDims{s.D + 1, (s.H + 3) / 3, (s.W + 3) / 3}; }
long brick_nseg(const TiledShape &s)
{
    const BrickDims d = brick_dims(s);
    return (long)s.N * s.G * d.nz * d.nby * d.nbx;
}
long brick_points(const TiledShape &s) { return (long)s.N * s.G * s.K * s.P; }
double brick_mean(const TiledShape &s) { return 9.0 * s.K * s.P / s.vol; }      // points per block, were all inside
// Blocks that a workgroup of the sort counts in LDS: all of a sample and group, or what fits of those around its
// positions, planes first, then rows (a point displaced out of the window costs a global addition of its own).
constexpr int kSortSlots = 8192;
SortWindow sort_window(const TiledShape &s, const BrickDims &d)
{
    SortWindow w{d.nz, d.nby, d.nbx, 0, 0, 0, 0, 0, 0, 0, make_fastdiv(s.geo.kw), make_fastdiv(s.geo.kh)};
    // A tile of 4 x 8 x 8 positions reaches fewer blocks than 64 positions of a few rows (filing 32x60x108: 122 us, 136).  With
    // few tiles the taps of one are dealt to several workgroups (counting + filing 1024 -> 256 channels on 8x30x54: 20 + 32 us
    // on 56 workgroups, 10 + 15 on 224; on four times as many as compute units no faster).
    const int lz = s.Do >= 3 ? 2 : (s.Do >= 2 ? 1 : 0);
    w.lx = 3; w.ly = 5 - lz;
    w.ny = (s.Ho + (1 << w.ly) - 1) >> w.ly; w.nx = (s.Wo + (1 << w.lx) - 1) >> w.lx;
    w.ntile = ((s.Do + (1 << lz) - 1) >> lz) * w.ny * w.nx;
    w.taps = std::min(s.K, kSortTaps);
    while (w.taps > kTapGroups && (long)w.ntile * s.N * s.G * ((s.K + w.taps - 1) / w.taps) < 256) w.taps = (w.taps + 1) / 2;
    w.ngrp = (s.K + w.taps - 1) / w.taps;
    const int least[3] = {(s.geo.kd - 1) * s.geo.dd + 9, ((s.geo.kh - 1) * s.geo.dh + 2) / 3 + 7, ((s.geo.kw - 1) * s.geo.dw + 2) / 3 + 7};
    auto shrink = [](int &v, int lo, long others, int slots) {
        if ((long)v * others > slots) v = (int)std::max<long>(std::min(v, lo), slots / others);
    };
    shrink(w.wz, least[0], (long)w.wy * w.wx, kSortSlots);
    shrink(w.wy, least[1], (long)w.wz * w.wx, kSortSlots);
    shrink(w.wx, least[2], (long)w.wz * w.wy, kSortSlots);
    // (a kernel of great extent: whatever still fits)
    shrink(w.wz, 1, (long)w.wy * w.wx, kSortSlots);
    shrink(w.wy, 1, (long)w.wz * w.wx, kSortSlots);
    shrink(w.wx, 1, (long)w.wz * w.wy, kSortSlots);
    return w;
}
// Base planes per workgroup of the gradient kernel: a range costs one plane more than it has bases, to be loaded and added, and
// the last round of workgroups (twelve wavefronts to a compute unit) leaves the chip part empty; half of that is taken for lost.  us, planes
// per range: 256 channels on 2x8x30x54 1 115, 2 116, 3 104; float32 2 262, 3 232, 5 253; 1024 channels on 8x30x54 1 227, 2 240, 3 230,
// 5 234; 2048, 7 taps, 2 260, 3 227, 5 224, 9 209; 512, 8 groups, 2x8x30x54 1 229, 2 223, 3 225, 5 232; 256 on 32x60x108 3 824, 5 822, 9 890.
// Below three quarters of a round the shortest ranges even out best (steps: 256 -> 64 channels, float32, 8x20x32, 0.6 rounds of 3 planes
// 294, of 1 289; bfloat16 8x40x50 0.9 rounds of 3 planes 332, of 1 340; 8x60x107 one round of 9 931, of 1 956).
int brick_range_planes(int nz, long cols, int nw)
{
    const double slots = 12.0 / nw * std::max(d2c_num_cus(), 1);
    int best = nz;
    double least = 1e300;
    for (int z = nz;; z = (z + 1) / 2) {
        const double r = cols * ((nz + z - 1) / z) / slots, t = 0.5 * (r + 0.5 + std::ceil(r)) * (z + 1.25);
        if (z == 1 ? t < least : (r >= 0.75 && t < least)) { least = t; best = z; }
        if (z == 1) return best;
    }
}
int brick_sets(const TiledShape &s) { return (s.cpg / s.bkc + kMaxWaves - 1) / kMaxWaves; }
BrickLists brick_lists(const TiledShape &s, char *base)
{
    const BrickWs w = d2c_brick_ws(s);
    return BrickLists{(int *)(base + w.count), (int *)(base + w.count) + brick_nseg(s), (int *)(base + w.end), (int *)(base + w.place),
                      (uint4 *)(base + w.pt), (float *)(base + w.alpha)};
}

}  // namespace

// The bricks serve problems in three dimensions whose blocks hold enough points to fill most of a matrix
// product of 32: below about half a product on average (few taps, strided outputs) the gathering kernels are as good.
// (Float32: grad_input, grad_offset and grad_mask; sampled columns are bfloat16 only.)
bool d2c_brick_supported(const TiledShape &s, int dtype)
{
    if (s.nd != 3 || (dtype != D2C_BF16 && dtype != D2C_F32) || s.cpg % s.bkc) return false;
    return brick_mean(s) >= 16.0 && s.K <= 65535 && (long)s.N * s.G <= 65535 && brick_nseg(s) < (1L << 31) - 1024 &&
           brick_points(s) < (1L << 31) - 64 && (size_t)s.K * (s.M + 64) * 128 < 0xFFFFFF00u &&
           (size_t)s.H * s.W * s.Cin * 4 < 0xFFFFFFF0u;
}
BrickWs d2c_brick_ws(const TiledShape &s)
{
    const size_t n = (size_t)brick_points(s), nseg = (size_t)brick_nseg(s);
    BrickWs w;
    w.count = 0;                                                   // [nseg] counts, then the cursor and the number of points outside: one clear
    w.end = d2c_align_up((nseg + 2) * 4);
    w.place = w.end + d2c_align_up(nseg * 4);
    w.pt = w.place + d2c_align_up(n * 4);
    w.alpha = w.pt + d2c_align_up(n * 16);
    w.total = w.alpha + d2c_align_up(n * 4);
    w.res_bytes = d2c_align_up(n * 16) * brick_sets(s);
    return w;
}

// What has to be zero in front of the sort.
void *d2c_brick_zero(const TiledShape &s, void *ws, size_t *bytes)
{
    *bytes = ((size_t)brick_nseg(s) + 2) * 4;
    return (char *)ws + d2c_brick_ws(s).count;
}
// Sorts the points (`cleared`: d2c_brick_zero() has been).
int d2c_brick_sort(const TiledShape &s, const void *off, const void *mask, void *ws, hipStream_t st, bool cleared)
{
    D2cProfScope prof(D2C_PROF_PACK, st);
    const BrickDims d = brick_dims(s);
    const BrickLists L = brick_lists(s, (char *)ws);
    const int nseg = (int)brick_nseg(s);
    if (!cleared) d2c_fill_zero(L.count, ((size_t)nseg + 2) * 4, st);
    const SortWindow w = sort_window(s, d);
    const size_t lds = ((size_t)w.wz * w.wy * w.wx + 1) * 4;
    const dim3 grid((unsigned)((long)w.ntile * w.ngrp * s.N * s.G)), blk(kSortThreads);
    auto go = [&](auto A, auto Z) {
        constexpr bool A16 = decltype(A)::value, SZ = decltype(Z)::value;
        hipLaunchKernelGGL((brick_count_kernel<A16, SZ>), grid, blk, lds, st, s, d, L, off, w);
        hipLaunchKernelGGL(brick_range_kernel, dim3((nseg + 1023) / 1024), dim3(1024), 0, st, L, nseg);
        hipLaunchKernelGGL((brick_file_kernel<A16, SZ>), grid, blk, lds, st, s, d, L, off, mask, w, brick_points(s));
    };
    if (s.adt == D2C_BF16) {
        if (s.ss.on) go(std::true_type{}, std::true_type{});
        else go(std::true_type{}, std::false_type{});
    } else {
        if (s.ss.on) go(std::false_type{}, std::true_type{});
        else go(std::false_type{}, std::false_type{});
    }
    return d2c_check_launch("brick_file_kernel");
}

// `gxcl` (cleared), `goff` (size-map source: the gradient of the raw map `raw`) and `gmask` may be NULL.
int d2c_brick_grad(const TiledShape &s, const void *xcl, const void *gcol, const void *mask, const void *raw, float *gxcl,
                   void *goff, void *gmask, const void *lists, void *res, hipStream_t st)
{
    const long n = brick_points(s);
    BrickArgs a{};
    a.d = brick_dims(s); a.L = brick_lists(s, (char *)const_cast<void *>(lists));
    a.xcl = xcl; a.gcol = gcol; a.gxcl = gxcl;
    a.res = (goff || gmask) ? (float2 *)res : nullptr;
    a.nres = (long)(d2c_align_up((size_t)n * 16) / 16);
    a.G = s.G; a.cpc = s.cpg / s.bkc; a.Cin = s.Cin; a.D = s.D; a.H = s.H; a.W = s.W; a.vol = s.vol;
    a.chunk_rows = (long)s.K * s.M;
    a.nset = brick_sets(s);
    const int nw = (a.cpc + a.nset - 1) / a.nset;
    const long cols = (long)a.d.nbx * a.d.nby * s.N * s.G * a.nset;
    a.zlen = brick_range_planes(a.d.nz, cols, nw);
    a.nzr = (a.d.nz + a.zlen - 1) / a.zlen;
    const unsigned grid = (unsigned)(cols * a.nzr);
    {
        D2cProfScope prof(D2C_PROF_BWD_AUX, st, s.bkc == 64 ? "brick_grad_kernel" : "brick_grad_f32_kernel");
        const bool share = nw > 1 && brick_mean(s) >= 128.0;      // (four steps to a plane)
        const int lds = nw * (s.bkc == 64 ? kRowLds : kRowLdsF) + (share ? 2 : nw) * kWeightLds + (nw > 1 ? nw * 1024 : 0);
        auto kern = s.bkc == 64 ? (share ? &brick_grad_kernel<true> : &brick_grad_kernel<false>)
                                : (share ? &brick_grad_f32_kernel<true> : &brick_grad_f32_kernel<false>);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * nw), lds, st, a, a.L.end, a.L.count);
        if (int rc = d2c_check_launch("brick_grad_kernel")) return rc;
    }
    if (!a.res) return D2C_OK;
    D2cProfScope prof(D2C_PROF_PACK, st);
    const bool a16 = s.adt == D2C_BF16;
    if (s.ss.on) {
        auto fin = a16 ? &brick_finish_size_kernel<true> : &brick_finish_size_kernel<false>;
        hipLaunchKernelGGL(fin, dim3((s.P + 63) / 64, s.N), dim3(64 * kTapShares), 0, st, s, a.L, a.res, a.nres, a.nset, mask, raw, goff, gmask);
    } else {
        auto fin = a16 ? &brick_finish_kernel<true> : &brick_finish_kernel<false>;
        const int ngrp = (s.K + kPassTaps - 1) / kPassTaps;
        hipLaunchKernelGGL(fin, dim3((unsigned)((long)((s.P + 255) / 256) * ngrp * s.N * s.G)), dim3(256), 0, st, s, a.L, a.res, a.nres, a.nset, mask,
                           goff, gmask, ngrp);
    }
    return d2c_check_launch("brick_finish_kernel");
}

// The sampled columns [chunk][tap][rows][64] of sorted points.
int d2c_brick_columns(const TiledShape &s, const void *xcl, void *col, int rows, const void *lists, hipStream_t st)
{
    BrickSampleArgs a{};
    a.d = brick_dims(s); a.L = brick_lists(s, (char *)const_cast<void *>(lists));
    a.xcl = (const bf16_t *)xcl; a.col = (bf16_t *)col;
    a.G = s.G; a.cpc = s.cpg / 64; a.Cin = s.Cin; a.D = s.D; a.H = s.H; a.W = s.W; a.vol = s.vol;
    a.K = s.K; a.rows = rows; a.M = s.M; a.chunk_rows = (long)s.K * rows; a.pad = rows - s.M;
    a.dM = make_fastdiv(s.M); a.dKM = make_fastdiv(s.K * s.M);
    a.nset = brick_sets(s);
    const int nw = (a.cpc + a.nset - 1) / a.nset;
    const int ncu = d2c_num_cus();
    const long cols = (long)a.d.nbx * a.d.nby * s.N * s.G * a.nset;
    a.zlen = a.d.nz;
    // (enough workgroups to fill the chip several times over, fewer where a plane has few points: 2048 channels, 7 taps, 100 us, 88)
    const long want = (brick_mean(s) >= 128.0 ? 64L : 16L) * ncu;
    while (a.zlen > 1 && cols * ((a.d.nz + a.zlen - 1) / a.zlen) * nw < want) a.zlen = (a.zlen + 1) / 2;
    a.nzr = (a.d.nz + a.zlen - 1) / a.zlen;
    a.npoint = brick_points(s);
    a.nzero = (int)std::min<long>(2048, (a.npoint + 511) / 512) / nw + 1;
    D2cProfScope prof(D2C_PROF_SAMPLE, st, "brick_sample_kernel");
    hipLaunchKernelGGL(brick_sample_kernel, dim3((unsigned)(cols * a.nzr + a.nzero)), dim3(64 * nw), nw * kRowLds, st, a, a.L.end, a.L.count);
    return d2c_check_launch("brick_sample_kernel");
}
