// The ordinary convolution of a layer's deformation branch (`deform_params`, network/layers.py:66-68), bfloat16, on
// the matrix cores.  It has no sampling points: a tap of an output position is one voxel, so the three products below
// read 128-byte pieces of channels-last rows straight into LDS, one per (position, tap), where the deformable operator
// at zero offsets interpolates eight and the backward pass goes through grad-column rows, sample lists and kept columns.
//
//   forward       out[o, m]   = bias[o] + sum_{tap, c} W[o, c, tap] * x[vox(m, tap), c]      conv_rows_kernel
//   grad_input    gx[c, v]    = sum_{tap, o} W[o, c, tap] * gout[pos(v, tap), o]             ... and conv_wide_kernel
//   grad_weight   gW[o, c, tap] = sum_m gout[o, m] * x[vox(m, tap), c]                       conv_weight_kernel
//
// (m: output positions over the whole batch, v: input voxels; a row that a tap puts outside the volume is a row of
// zeros.)  Everything the kernels need in another order is made by one launch per direction (conv_prepare_kernel).
// Sums that are shared out between workgroups are written as float partial results and added up in a fixed order by
// the finishing kernels: nothing is cleared, and equal inputs give equal bits.
//
// 1024 -> 30 channels on 8x30x54 (forward): 0.51 ms at zero offsets on the gather kernel; figures of these kernels
// are at each one.
#include "d2c_mma.hpp"
#include <algorithm>

namespace {

constexpr int kThreads = 256;
constexpr int kMT = 128;              // rows (positions) per workgroup of conv_rows_kernel
constexpr int kWMT = 256;             // ... of conv_wide_kernel
constexpr int kCW = 64;               // positions per step of conv_weight_kernel

D2C_DEV int xcd_swizzle(int bid, int n)
{
    const int x = bid & 7, idx = bid >> 3;
    const int q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + idx;
}

// One spatial axis triple of a gather: rows on the grid (d, h, w) read rows on the grid (sd, sh, sw).
struct RowMap {
    int N, P;                         // samples, rows per sample (the grid's points)
    int d, h, w;                      // grid of the result rows
    int sd, sh, sw;                   // grid of the source rows
    TapGeom g;
    int back;                         // 0: source = o * stride - pad + tap * dilation; 1: the transposed map
    FastDiv dP, dHW, dW;
};
inline RowMap row_map(const d2c_conv3d_desc &q, bool back)
{
    RowMap r;
    r.N = q.N;
    r.back = back ? 1 : 0;
    r.g = make_geom(q);
    r.d = back ? q.D : q.Do; r.h = back ? q.H : q.Ho; r.w = back ? q.W : q.Wo;
    r.sd = back ? q.Do : q.D; r.sh = back ? q.Ho : q.H; r.sw = back ? q.Wo : q.W;
    r.P = r.d * r.h * r.w;
    r.dP = make_fastdiv(r.P); r.dHW = make_fastdiv(r.h * r.w); r.dW = make_fastdiv(r.w);
    return r;
}

// grid point of row m: sample and the source coordinates of tap (0, 0, 0), unclipped (transposed map: before the
// division by the stride)
struct RowPos {
    int b, z, y, x;
    bool ok;
};
D2C_DEV RowPos row_pos(const RowMap &r, int m)
{
    RowPos p;
    p.ok = m < r.N * r.P;
    const int mm = p.ok ? m : 0;
    p.b = fdiv(mm, r.dP);
    const int q = mm - p.b * r.P, z = fdiv(q, r.dHW), rem = q - z * (r.h * r.w), y = fdiv(rem, r.dW), x = rem - y * r.w;
    p.z = r.back ? z + r.g.pd : z * r.g.sd - r.g.pd;
    p.y = r.back ? y + r.g.ph : y * r.g.sh - r.g.ph;
    p.x = r.back ? x + r.g.pw : x * r.g.sw - r.g.pw;
    return p;
}
// source row of (row, tap (kz, ky, kx)), or -1
D2C_DEV int source_row(const RowMap &r, const RowPos &p, int kz, int ky, int kx)
{
    int z, y, x;
    bool ok = p.ok;
    if (r.back) {
        z = p.z - kz * r.g.dd; y = p.y - ky * r.g.dh; x = p.x - kx * r.g.dw;
        ok = ok && z >= 0 && y >= 0 && x >= 0;
        if (r.g.sd != 1 || r.g.sh != 1 || r.g.sw != 1) {
            const int qz = z / r.g.sd, qy = y / r.g.sh, qx = x / r.g.sw;
            ok = ok && qz * r.g.sd == z && qy * r.g.sh == y && qx * r.g.sw == x;
            z = qz; y = qy; x = qx;
        }
    } else {
        z = p.z + kz * r.g.dd; y = p.y + ky * r.g.dh; x = p.x + kx * r.g.dw;
        ok = ok && z >= 0 && y >= 0 && x >= 0;
    }
    ok = ok && z < r.sd && y < r.sh && x < r.sw;
    return ok ? ((p.b * r.sd + z) * r.sh + y) * r.sw + x : -1;
}

// ---- LDS reads of data that DMA transfers filled (see lds_row_read in d2c_mma.hpp), and counted waits
template <int N> D2C_DEV void wait_lds(u32x4_t &a) { asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(a) : "n"(N)); }
template <int N> D2C_DEV void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
D2C_DEV void group_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
D2C_DEV void dma16(const void *src, unsigned char *lds)
{
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                     (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
}
D2C_DEV u32x4_t lds_read16(unsigned a)
{
    u32x4_t v;
    asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(a));
    return v;
}

template <int OFF> D2C_DEV u32x4_t lds_read16_at(unsigned a)
{
    u32x4_t v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(a), "n"(OFF));
    return v;
}

// 16-byte slot of channel vector v of row r in an LDS tile of KC-channel rows: consecutive rows spread over all 16
// slots of the 64 banks, so that the reads of 16 lanes, one row each, do not meet.  The copies in device memory that
// are read as whole tiles (the weights) have it built in.
template <int KC> __host__ __device__ inline int tile_slot(int r, int v)
{
    return KC == 64 ? (v ^ ((r >> 1) & 7)) : (v ^ ((r >> 2) & 3));
}

// ============================================================ forward and grad_input
//   D[n, m] = sum_{step} B[step][n][KC] * A[source_row(m, tap of the step)][chunk of the step][KC]
// One workgroup = 128 rows m x NT columns n, four wavefronts; a step is one tap and KC channels.  Both tiles of a step
// go to LDS by DMA (1 KiB requests; a lane's 16 bytes come from the row its position and tap name), NST stages deep;
// the source rows of a tap are worked out once by the lanes of the wavefront that fetches them and handed round by
// permutes.  Steps are tap-major, so that happens once per tap.
// What bounds it: with 32 columns the row requests (64 bytes per clock and compute unit: every position's row once
// per tap), with 128 the matrix instructions and the requests alike (32 KiB and 512 matrix clocks per step).
struct ConvRowsArgs {
    RowMap map;
    const unsigned char *src;         // rows of `rowb` bytes, then a row of zeros at byte `zrow`
    const unsigned char *wt;          // [step][column tile][NT][KC] bfloat16, slots swizzled
    const bf16_t *bias;               // or NULL
    bf16_t *out;                      // [N][C][P], or NULL: partial sums
    float *part;                      // [split][C][N * P]; conv_wide_kernel: [piece][column / 4][row of the tile][4]
    unsigned rowb, zrow;
    int C;                            // columns that exist
    int nchunk, S;                    // KC-channel chunks per row, steps
    int ntile, nctile, nsplit;
    int nfull;                        // conv_wide_kernel: tiles (row tile major) whose steps are not shared out
    // COLS: `src` is [chunk][tap][row][KC], a step's rows lie one after the other
    int K, tap_rows;                  // taps, rows of a tap
    int act;                          // epilogue (d2c_epilogue)
    float act_scale;
    int wide_out;                     // rows of `out` come in fours: P a multiple of four, `out` on eight bytes
};

template <int NT, int KC, bool COLS>
__global__ void __launch_bounds__(kThreads, 2) conv_rows_kernel(ConvRowsArgs a)
{
    constexpr int WO = NT == 128 ? 2 : 1, WP = 4 / WO;     // wavefronts along columns / rows
    constexpr int OB = NT / 32 / WO, PB = kMT / 32 / WP;   // 32-blocks of a wavefront
    constexpr int ROWB = KC * 2, RPD = 1024 / ROWB, VPR = ROWB / 16;
    constexpr int ABYTES = kMT * ROWB, BBYTES = NT * ROWB, STAGE = ABYTES + BBYTES;
    constexpr int NST = STAGE > 24 * 1024 ? 2 : 3;
    constexpr int AD = ABYTES / 4096;                      // DMA requests per wavefront and step: rows,
    constexpr int BD = (BBYTES + 4095) / 4096;             // ... weights (2 KiB of them: the first two wavefronts)
    constexpr int NKG = KC / 16;
    __shared__ __align__(1024) unsigned char s_t[NST * STAGE];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int id = xcd_swizzle(blockIdx.x, gridDim.x);
    const int ct = id % a.nctile; id /= a.nctile;
    const int split = id % a.nsplit, tile = id / a.nsplit;
    const int st_lo = (int)((long)a.S * split / a.nsplit), st_hi = (int)((long)a.S * (split + 1) / a.nsplit);
    const int m0 = tile * kMT;

    // --- rows this wavefront fetches: wave * 32 + (0 .. 31), lane l works out row l & 31
    const RowPos rp = COLS ? RowPos{} : row_pos(a.map, m0 + wave * 32 + (lane & 31));
    const unsigned char *asrc = a.src;                     // (COLS: the rows of the step)
    const long tap_bytes = (long)a.tap_rows * ROWB;
    const int lrow = lane / VPR, lslot = lane % VPR;       // this lane's row within a request, its 16-byte slot
    unsigned aoff[AD], ainc[AD];
    int chunk = st_lo % a.nchunk, tap = st_lo / a.nchunk;
    auto tap_rows = [&](int k, int j) {
        if constexpr (COLS) {
            asrc = a.src + ((long)j * a.K + k) * tap_bytes;
#pragma unroll
            for (int i = 0; i < AD; i++) {
                const int rl = i * RPD + lrow;
                // (a tile's rows past the last one: the last one again, stored nowhere)
                aoff[i] = (unsigned)min(m0 + wave * 32 + rl, a.map.N * a.map.P - 1) * ROWB + (unsigned)tile_slot<KC>(rl, lslot) * 16u;
            }
            return;
        }
        const int kx = k % a.map.g.kw, ky = (k / a.map.g.kw) % a.map.g.kh, kz = k / (a.map.g.kw * a.map.g.kh);
        const int row = source_row(a.map, rp, kz, ky, kx);
#pragma unroll
        for (int i = 0; i < AD; i++) {
            const int rl = i * RPD + lrow;                  // row of this request and lane, 0 .. 31
            const int sr = __builtin_amdgcn_ds_bpermute(rl << 2, row);
            const unsigned vb = (unsigned)tile_slot<KC>(rl, lslot) * 16u;    // (wave * 32 is a multiple of the pattern)
            aoff[i] = sr >= 0 ? (unsigned)sr * a.rowb + (unsigned)j * ROWB + vb : a.zrow + vb;
            ainc[i] = sr >= 0 ? ROWB : 0u;
        }
    };
    static_assert(AD * RPD == 32, "a wavefront fetches 32 rows per step");
    const unsigned char *bsrc = a.wt + ((long)st_lo * a.nctile + ct) * BBYTES + (wave % (BBYTES >= 4096 ? 4 : BBYTES / 1024)) * 1024 + lane * 16;
    const long bstep = (long)a.nctile * BBYTES;
    auto issue = [&](int buf) {
        unsigned char *sa = s_t + buf * STAGE + wave * (32 * ROWB), *sb = s_t + buf * STAGE + ABYTES;
#pragma unroll
        for (int i = 0; i < AD; i++) {
            dma16(asrc + aoff[i], sa + i * 1024);
            if constexpr (!COLS) aoff[i] += ainc[i];
        }
        if constexpr (COLS) asrc += a.K * tap_bytes;       // (the next chunk of the tap)
#pragma unroll
        for (int i = 0; i < BD; i++) {
            // (fewer than four pieces: wavefronts fetch the same one twice, which keeps the counts equal)
            const int piece = BBYTES >= 4096 ? i * 4 + wave : wave % (BBYTES / 1024);
            dma16(bsrc + (BBYTES >= 4096 ? i * 4096 : 0), sb + piece * 1024);
        }
        bsrc += bstep;
        if (++chunk == a.nchunk) {
            chunk = 0; tap++;
            if (tap * a.nchunk < st_hi) tap_rows(tap, 0);
        }
    };

    f32x16 acc[OB][PB];
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int pb = 0; pb < PB; pb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[ob][pb][r] = 0.f;
    const int wo = wave % WO, wp = wave / WO;
    // byte offsets of this lane's operand vectors of k-group 0 .. NKG-1 within a tile (blocks of 32 rows repeat them)
    unsigned slot[NKG];
#pragma unroll
    for (int kg = 0; kg < NKG; kg++)
        slot[kg] = (unsigned)((lane & 31) * ROWB + tile_slot<KC>(lane & 31, kg * 2 + (lane >> 5)) * 16);
    const unsigned ra = lds_address(s_t) + wp * PB * 32 * ROWB, rb = lds_address(s_t) + ABYTES + wo * OB * 32 * ROWB;

    tap_rows(tap, chunk);
    issue(0);
    if (NST == 3 && st_lo + 1 < st_hi) issue(1);
    int buf = 0, nbuf = NST - 1;
    for (int st = st_lo; st < st_hi; st++) {
        if (NST == 3 && st + 1 < st_hi) wait_vm<AD + BD>(); else wait_vm<0>();
        group_barrier();
        if (st + NST - 1 < st_hi) issue(nbuf);
        const unsigned pa = ra + buf * STAGE, pb_ = rb + buf * STAGE;
        u32x4_t fa[2][PB], fb[2][OB];
        auto fetch = [&](int kg, int s) {
#pragma unroll
            for (int ob = 0; ob < OB; ob++) fb[s][ob] = lds_read16(pb_ + slot[kg] + ob * 32 * ROWB);
#pragma unroll
            for (int pb = 0; pb < PB; pb++) fa[s][pb] = lds_read16(pa + slot[kg] + pb * 32 * ROWB);
        };
        fetch(0, 0);
#pragma unroll
        for (int kg = 0; kg < NKG; kg++) {
            const int s = kg & 1;
            if (kg + 1 < NKG) fetch(kg + 1, s ^ 1);
#pragma unroll
            for (int ob = 0; ob < OB; ob++) { if (kg + 1 < NKG) wait_lds<OB + PB>(fb[s][ob]); else wait_lds<0>(fb[s][ob]); }
#pragma unroll
            for (int pb = 0; pb < PB; pb++) { if (kg + 1 < NKG) wait_lds<OB + PB>(fa[s][pb]); else wait_lds<0>(fa[s][pb]); }
#pragma unroll
            for (int ob = 0; ob < OB; ob++)
#pragma unroll
                for (int pb = 0; pb < PB; pb++)
                    mma_kgroup<bf16_t, false>(acc[ob][pb], __builtin_bit_cast(uint4, fb[s][ob]), __builtin_bit_cast(uint4, fa[s][pb]));
        }
        buf = buf + 1 == NST ? 0 : buf + 1;
        nbuf = nbuf + 1 == NST ? 0 : nbuf + 1;
    }

    const int M = a.map.N * a.map.P;
#pragma unroll
    for (int pb = 0; pb < PB; pb++) {
        const int m = m0 + (wp * PB + pb) * 32 + (lane & 31);
        if (m >= M) continue;
        const int b = fdiv(m, a.map.dP), p = m - b * a.map.P;
#pragma unroll
        for (int ob = 0; ob < OB; ob++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int n = ct * NT + (wo * OB + ob) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (n >= a.C) continue;
                if (a.out)
                    a.out[((long)b * a.C + n) * a.map.P + p] =
                        f32_to_bf16(d2c_epilogue(acc[ob][pb][r] + (a.bias ? bf16_to_f32(a.bias[n]) : 0.f), a.act, a.act_scale));
                else a.part[((long)split * a.C + n) * M + m] = acc[ob][pb][r];
            }
    }
}

typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
// Operands that take one LDS read, and those that take two (a transposing read brings half of the vector).
struct TrVec { u32x2_t lo, hi; };
template <int N> D2C_DEV void wait_lds(TrVec &a) { asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a.lo), "+v"(a.hi) : "n"(N)); }
D2C_DEV void landed(u32x4_t &a) { asm volatile("" : "+v"(a)); }
D2C_DEV void landed(TrVec &a) { asm volatile("" : "+v"(a.lo), "+v"(a.hi)); }
D2C_DEV uint4 operand_of(const u32x4_t &a) { return __builtin_bit_cast(uint4, a); }
D2C_DEV uint4 operand_of(const TrVec &a) { return make_uint4(a.lo.x, a.lo.y, a.hi.x, a.hi.y); }

// One k-group of the wide kernels below: OB x PB matrix instructions on operand set KG & 1, and between them the reads of the
// next k-group's operands into the other set and whatever `request` has for a slot.  The reads are spread over the group (the
// four wavefronts share the LDS)
// and waited for one by one, in the order in which the instructions need them: weights 0, rows 0 .. PB-1, weights 1 ...
// The last k-group of a step meets `sync` in slot kSync and reads from the next step's buffers after it.
template <int OB, int PB, int KG, class FB, class Read, class Request, class Sync>
D2C_DEV void wide_group(f32x16 (&acc)[OB][PB], u32x4_t (&fa)[2][PB], FB (&fb)[2][OB], Read read, Request request, Sync sync)
{
    constexpr int NM = OB * PB, NR = OB + PB, s = KG & 1, lo = KG == 3 ? NM * 3 / 8 : 0;
    for_each_const([&](auto I) INLINE {
        constexpr int i = decltype(I)::value, ob = i / PB, pb = i % PB;
        // (LDS reads that the first r operands take)
        constexpr auto reads = [](int r) { return r + (std::is_same<FB, TrVec>::value ? (r > 0) + (r > PB + 1 ? r - PB - 1 : 0) : 0); };
        constexpr int issued = i <= lo ? 0 : ((i - lo) * NR + NM - lo - 1) / (NM - lo);        // operands of this group before slot i
        if constexpr (KG == 3 && i == lo) sync();
        if constexpr (pb == 0 || ob == 0) {
            // the operand(s) that this instruction is the first to need
            constexpr int need = ob == 0 ? 1 + pb : PB + ob, later = reads(NR) - reads(need + 1) + reads(issued);
            static_assert(later <= 15, "the counter of LDS reads");
            if constexpr (KG == 3 && i >= lo) {
                if constexpr (pb == 0) landed(fb[s][ob]);
                if constexpr (ob == 0) landed(fa[s][pb]);
            } else {
                if constexpr (pb == 0) wait_lds<later>(fb[s][ob]);
                if constexpr (ob == 0) wait_lds<later>(fa[s][pb]);
            }
        }
        mma_kgroup<bf16_t, false>(acc[ob][pb], operand_of(fb[s][ob]), operand_of(fa[s][pb]));
        constexpr int next = i < lo ? 0 : ((i + 1 - lo) * NR + NM - lo - 1) / (NM - lo);
        for_each_const([&](auto R) INLINE {
            constexpr int r = issued + decltype(R)::value;
            if constexpr (r == 0) read(std::integral_constant<int, 0>{}, fb[s ^ 1][0]);
            else if constexpr (r <= PB) read(std::integral_constant<int, OB + r - 1>{}, fa[s ^ 1][r - 1]);
            else read(std::integral_constant<int, r - PB>{}, fb[s ^ 1][r - PB]);
        }, std::make_integer_sequence<int, next - issued>{});
        request(I);
        __builtin_amdgcn_sched_barrier(0);
    }, std::make_integer_sequence<int, NM>{});
}

// The same product for larger problems: a workgroup = 256 rows x NT columns (256 or 128), four wavefronts of 128 x NT/2,
// one workgroup per compute unit.  A step of 64 channels is 2048 matrix clocks (NT = 256) against 1024 clocks of LDS
// reads and 512 of DMA writes; the 128 x 128 tile above has 768 clocks of LDS traffic for 512 matrix clocks.  Rows are
// fetched two steps ahead (three buffers; they come from device memory), weights one (two buffers; they come from L2),
// each into the buffer that the step's barrier has just freed.
// The operand reads of a k-group and the DMA requests go between the matrix instructions of the k-group before; a step's
// only barrier stands in front of its last k-group, when every wavefront holds the last operands of the step in
// registers: from there on the buffers of the step are free and the next step's first operands are read.
// Over sampled columns, 512 -> 512 channels on 2x8x30x54: 520 us with the tile above (its partial sums included), 341 us
// (1.08 PFLOP/s); 256 -> 256 on 32x60x108: 1015 and 683 us, of which reading 2.9 GB of columns once takes 520.
template <int NT, bool COLS>
__global__ void __launch_bounds__(kThreads, 1) conv_wide_kernel(ConvRowsArgs a)
{
    constexpr int OB = NT / 64, PB = 4;                    // 32-blocks of a wavefront: columns, rows
    constexpr int ROWB = 128, ABYTES = kWMT * ROWB, BBYTES = NT * ROWB;
    constexpr int AD = 8, BD = BBYTES / 4096, NM = OB * PB;
    __shared__ __align__(1024) unsigned char s_t[3 * ABYTES + 2 * BBYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the first `nfull` tiles are whole ones, the rest is shared out to nsplit workgroups each
    const bool whole = (int)blockIdx.x < a.nfull;
    const int piece = whole ? 0 : xcd_swizzle((int)blockIdx.x - a.nfull, (int)gridDim.x - a.nfull);
    const int item = whole ? xcd_swizzle(blockIdx.x, a.nfull) : a.nfull + piece / a.nsplit;
    const int split = whole ? 0 : piece % a.nsplit, nsplit = whole ? 1 : a.nsplit;
    const int ct = item % a.nctile, tile = item / a.nctile;
    const int st_lo = (int)((long)a.S * split / nsplit), st_hi = (int)((long)a.S * (split + 1) / nsplit);
    const int m0 = tile * kWMT, M = a.map.N * a.map.P;

    // --- rows this wavefront fetches: wave * 64 + (0 .. 63), eight per request; lane l works out row l
    const RowPos rp = COLS ? RowPos{} : row_pos(a.map, m0 + wave * 64 + lane);
    const unsigned char *asrc = a.src;                     // (COLS: the rows of the step)
    const long tap_bytes = (long)a.tap_rows * ROWB;
    const int lrow = lane >> 3;                            // this lane's row within a request
    unsigned aoff[AD], ainc[AD];
    int achunk = st_lo % a.nchunk, atap = st_lo / a.nchunk, ast = st_lo;      // the step that the next rows belong to
    if (COLS) {
#pragma unroll
        for (int i = 0; i < AD; i++) {
            // (a tile's rows past the last one: the last one again, stored nowhere)
            const int rl = i * 8 + lrow;
            aoff[i] = (unsigned)min(m0 + wave * 64 + rl, M - 1) * ROWB + (unsigned)tile_slot<64>(rl, lane & 7) * 16u;
        }
    }
    auto tap_rows = [&]() {
        if constexpr (COLS) {
            asrc = a.src + ((long)achunk * a.K + atap) * tap_bytes;
        } else {
            const int kx = atap % a.map.g.kw, ky = (atap / a.map.g.kw) % a.map.g.kh, kz = atap / (a.map.g.kw * a.map.g.kh);
            const int row = source_row(a.map, rp, kz, ky, kx);
#pragma unroll
            for (int i = 0; i < AD; i++) {
                const int rl = i * 8 + lrow;
                const int sr = __builtin_amdgcn_ds_bpermute(rl << 2, row);
                const unsigned vb = (unsigned)tile_slot<64>(rl, lane & 7) * 16u;
                aoff[i] = sr >= 0 ? (unsigned)sr * a.rowb + (unsigned)achunk * ROWB + vb : a.zrow + vb;
                ainc[i] = sr >= 0 ? ROWB : 0u;
            }
        }
    };
    // to the next step's rows (after the last step: its rows again, which nothing reads)
    auto advance = [&]() {
        if (ast + 1 >= st_hi) return;
        ast++;
        if (++achunk == a.nchunk) {
            achunk = 0; atap++;
            tap_rows();
        } else if constexpr (COLS) {
            asrc += a.K * tap_bytes;
        } else {
#pragma unroll
            for (int i = 0; i < AD; i++) aoff[i] += ainc[i];
        }
    };
    const unsigned char *bsrc = a.wt + ((long)st_lo * a.nctile + ct) * BBYTES + wave * 1024 + lane * 16;
    const long bstep = (long)a.nctile * BBYTES;
    unsigned char *const sa = s_t + wave * (64 * ROWB), *const sb = s_t + 3 * ABYTES + wave * 1024;
    auto row_request = [&](int i, int buf) { dma16(asrc + aoff[i], sa + buf * ABYTES + i * 1024); };
    auto weight_request = [&](int i, int buf) { dma16(bsrc + i * 4096, sb + buf * BBYTES + i * 4096); };

    f32x16 acc[OB][PB];
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int pb = 0; pb < PB; pb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[ob][pb][r] = 0.f;
    const int wo = wave & 1, wp = wave >> 1;
    unsigned slot[4];
#pragma unroll
    for (int kg = 0; kg < 4; kg++)
        slot[kg] = (unsigned)((lane & 31) * ROWB + tile_slot<64>(lane & 31, kg * 2 + (lane >> 5)) * 16);
    const unsigned ra = lds_address(s_t) + wp * PB * 32 * ROWB, rb = lds_address(s_t) + 3 * ABYTES + wo * OB * 32 * ROWB;
    u32x4_t fa[2][PB], fb[2][OB];
    // operand vector i of a k-group: weights, then rows
    auto operand = [&](auto I, u32x4_t &v, unsigned pa, unsigned pb, unsigned sl) INLINE {
        constexpr int i = decltype(I)::value;
        v = i < OB ? lds_read16(pb + sl + i * 32 * ROWB) : lds_read16(pa + sl + (i - OB) * 32 * ROWB);
    };

    // the bias of this wavefront's columns, one to a lane.  (Read here: a load between the stores at the end would wait for
    // those in front of it.)
    float bias_l[OB / 2];
#pragma unroll
    for (int i = 0; i < OB / 2; i++) {
        const int n = ct * NT + wo * OB * 32 + i * 64 + lane;
        bias_l[i] = a.bias && n < a.C ? bf16_to_f32(a.bias[n]) : 0.f;
    }

    tap_rows();
    for (int i = 0; i < AD; i++) row_request(i, 0);
    for (int i = 0; i < BD; i++) weight_request(i, 0);
    advance();
    for (int i = 0; i < AD; i++) row_request(i, 1);
    advance();
    if (st_lo + 1 < st_hi) bsrc += bstep;
    for (int i = 0; i < BD; i++) weight_request(i, 1);
    wait_vm<AD + BD>();
    group_barrier();
    // (in the order of wide_group)
    operand(std::integral_constant<int, 0>{}, fb[0][0], ra, rb, slot[0]);
    for_each_const([&](auto I) INLINE { operand(std::integral_constant<int, OB + decltype(I)::value>{}, fa[0][decltype(I)::value], ra, rb, slot[0]); },
                   std::make_integer_sequence<int, PB>{});
    for_each_const([&](auto I) INLINE { operand(std::integral_constant<int, 1 + decltype(I)::value>{}, fb[0][1 + decltype(I)::value], ra, rb, slot[0]); },
                   std::make_integer_sequence<int, OB - 1>{});
    int abuf = 0, bbuf = 0;
    for (int st = st_lo; st < st_hi; st++) {
        if (st + 2 < st_hi) bsrc += bstep;
        const int a1 = abuf == 2 ? 0 : abuf + 1, a2 = a1 == 2 ? 0 : a1 + 1, b1 = bbuf ^ 1;
        for_each_const([&](auto KG) INLINE {
            constexpr int kg = decltype(KG)::value;
            const unsigned pa = ra + (kg == 3 ? a1 : abuf) * ABYTES, pb_ = rb + (kg == 3 ? b1 : bbuf) * BBYTES;
            wide_group<OB, PB, kg>(acc, fa, fb, [&](auto I, u32x4_t &v) INLINE { operand(I, v, pa, pb_, slot[(kg + 1) & 3]); },
                [&](auto I) INLINE {
                    constexpr int i = decltype(I)::value, n = NM / (AD / 2);
                    if constexpr ((kg == 1 || kg == 2) && i % n == 0) row_request((kg - 1) * (AD / 2) + i / n, a2);
                    if constexpr (kg == 3 && i >= NM * 3 / 8 && i - NM * 3 / 8 < BD) weight_request(i - NM * 3 / 8, bbuf);
                },
                // (the rows of the step after the next one may be under way)
                [&]() INLINE { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(AD) : "memory"); });
        }, std::make_integer_sequence<int, 4>{});
        advance();
        abuf = a1; bbuf = b1;
    }
    // (the reads and requests behind the last step)
#pragma unroll
    for (int ob = 0; ob < OB; ob++) wait_lds<0>(fb[0][ob]);
#pragma unroll
    for (int pb = 0; pb < PB; pb++) asm volatile("" : "+v"(fa[0][pb]));
    wait_vm<0>();

    // Results, by stores that drop what lies outside (offset kNone).  A lane holds four consecutive columns of its row in four
    // registers: partial sums leave as they lie (16 bytes a lane); results, where rows come in fours (wide_out), after
    // the lanes of four rows have exchanged theirs (8 bytes a lane, a column of four rows), else one by one.
    // (256 -> 256 channels on 32x60x108, the kernel: 655 us one by one with the bias read in between, where each read waits for the
    // stores in front of it; 638 with the bias read ahead; 618 this way.  Without sampling, 8x60x107: 127, 126, 120.)
    constexpr unsigned kNone = 0xFFFFFFF0u;
    const int h4 = (lane >> 5) * 4, q = lane & 3;
    const unsigned step = (unsigned)a.map.P * 2u;
    if (!whole) {
        const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.part + (long)piece * NT * kWMT, 0, NT * kWMT * 4, 0x00020000);
        for_each_const([&](auto I) INLINE {
            constexpr int ob = decltype(I)::value / 4, r4 = decltype(I)::value % 4;
            for_each_const([&](auto J) INLINE {
                constexpr int pb = decltype(J)::value;
                const f32x16 &v = acc[ob][pb];
                const u32x4_t t = {__float_as_uint(v[r4 * 4]), __float_as_uint(v[r4 * 4 + 1]), __float_as_uint(v[r4 * 4 + 2]), __float_as_uint(v[r4 * 4 + 3])};
                const int c4 = (wo * OB + ob) * 8 + r4 * 2 + (lane >> 5), mt = (wp * PB + pb) * 32 + (lane & 31);
                __builtin_amdgcn_raw_buffer_store_b128(t, rs, (c4 * kWMT + mt) * 16, 0, 0);
            }, std::make_integer_sequence<int, PB>{});
            __builtin_amdgcn_sched_barrier(0);
        }, std::make_integer_sequence<int, OB * 4>{});
        return;
    }
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.out, 0, (int)((unsigned)a.C * (unsigned)M * 2u), 0x00020000);
    auto finish = [&](auto WIDE, auto ACT) INLINE {
        constexpr bool wide = decltype(WIDE)::value, act = decltype(ACT)::value;
        unsigned at[PB];
#pragma unroll
        for (int pb = 0; pb < PB; pb++) {
            const int m = m0 + (wp * PB + pb) * 32 + (wide ? lane & 28 : lane & 31), b = fdiv(m, a.map.dP), p = m - b * a.map.P;
            at[pb] = m >= M ? kNone : ((unsigned)b * a.C * a.map.P + p) * 2u + (unsigned)(h4 + (wide ? q : 0)) * step;
        }
        const unsigned sel = q & 1 ? 0x07060302u : 0x01000504u;        // the odd rows' lanes take the upper column of a pair
        for_each_const([&](auto I) INLINE {
            constexpr int ob = decltype(I)::value / 4, r4 = decltype(I)::value % 4, bl = (ob & 1) * 32 + 8 * r4;
            const int n0 = ct * NT + (wo * OB + ob) * 32 + 8 * r4;
            float bias[4], bv = bias_l[ob >> 1];
            opaque_v(bv);
#pragma unroll
            for (int e = 0; e < 4; e++) bias[e] = h4 ? lane_value(bv, bl + 4 + e) : lane_value(bv, bl + e);
            for_each_const([&](auto J) INLINE {
                constexpr int pb = decltype(J)::value;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[e] = acc[ob][pb][r4 * 4 + e];
                    opaque_v(v[e]);                        // (from here on its own: what the four ways share is not to be made in front of them, at once)
                    v[e] += bias[e];
                    if constexpr (act) v[e] = d2c_epilogue(v[e], a.act, a.act_scale);
                }
                if constexpr (wide) {
                    // columns (0, 1), (2, 3) of a row -> column q & 1, 2 + (q & 1) of two rows -> column q of four rows
                    const unsigned u0 = pack_bf16x2(v[0], v[1]), u1 = pack_bf16x2(v[2], v[3]);
                    const unsigned w0 = __builtin_amdgcn_perm(u0, (unsigned)__builtin_amdgcn_mov_dpp((int)u0, 0xB1, 0xF, 0xF, true), sel);
                    const unsigned w1 = __builtin_amdgcn_perm(u1, (unsigned)__builtin_amdgcn_mov_dpp((int)u1, 0xB1, 0xF, 0xF, true), sel);
                    const unsigned t = (unsigned)__builtin_amdgcn_mov_dpp((int)(q & 2 ? w0 : w1), 0x4E, 0xF, 0xF, true);
                    const unsigned o = n0 + h4 + q < a.C && at[pb] != kNone ? at[pb] + (unsigned)n0 * step : kNone;
                    __builtin_amdgcn_raw_buffer_store_b64(q & 2 ? u32x2_t{t, w1} : u32x2_t{w0, t}, rs, (int)o, 0, 0);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const unsigned o = n0 + h4 + e < a.C && at[pb] != kNone ? at[pb] + (unsigned)(n0 + e) * step : kNone;
                        __builtin_amdgcn_raw_buffer_store_b16((short)f32_to_bf16(v[e]), rs, (int)o, 0, 0);
                    }
                }
            }, std::make_integer_sequence<int, PB>{});
            __builtin_amdgcn_sched_barrier(0);
        }, std::make_integer_sequence<int, OB * 4>{});
    };
    const bool act = a.act != D2C_EPILOGUE_NONE;
    if (a.wide_out) { if (act) finish(std::true_type{}, std::true_type{}); else finish(std::true_type{}, std::false_type{}); }
    else if (act) finish(std::false_type{}, std::true_type{});
    else finish(std::false_type{}, std::false_type{});
}

// out = bias + the partial sums of conv_wide_kernel's tiles from `nfull` on ([piece][column / 4][row][4]): a workgroup = four
// columns of a tile, a thread = a row; four pieces are requested at a time.  (2048 -> 256 channels, 7 taps, on 8x30x54, five pieces: 21 us
// with a column to a workgroup, 13 this way; 64 -> 108 on 4x14x25 4.8 with a column to a workgroup, 5.15 with a piece at a time, 4.1)
__global__ void __launch_bounds__(kWMT) conv_wide_finish_kernel(ConvRowsArgs a, int NT)
{
    const int nq = NT / 4, rest = blockIdx.x / nq, c4 = blockIdx.x - rest * nq, item = a.nfull + rest, ct = item % a.nctile, tile = item / a.nctile;
    const int n = ct * NT + c4 * 4, m = tile * kWMT + threadIdx.x;
    if (n >= a.C || m >= a.map.N * a.map.P) return;
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = a.bias && n + e < a.C ? bf16_to_f32(a.bias[n + e]) : 0.f;
    const float4 *q = reinterpret_cast<const float4 *>(a.part) + ((long)rest * a.nsplit * nq + c4) * kWMT + threadIdx.x;
    for (int s0 = 0; s0 < a.nsplit; s0 += 4) {
        float4 t[4];
#pragma unroll
        for (int s = 0; s < 4; s++)
            if (s0 + s < a.nsplit) t[s] = q[(long)(s0 + s) * nq * kWMT];
#pragma unroll
        for (int s = 0; s < 4; s++)
            if (s0 + s < a.nsplit) { v[0] += t[s].x; v[1] += t[s].y; v[2] += t[s].z; v[3] += t[s].w; }
    }
    const int b = fdiv(m, a.map.dP), p = m - b * a.map.P;
#pragma unroll
    for (int e = 0; e < 4; e++)
        if (n + e < a.C) a.out[((long)b * a.C + n + e) * a.map.P + p] = f32_to_bf16(d2c_epilogue(v[e], a.act, a.act_scale));
}

// out[b][n][p] = bias[n] + the partial sums of (n, b * P + p)
__global__ void __launch_bounds__(256) conv_rows_finish_kernel(const float *part, const bf16_t *bias, bf16_t *out, int nsplit,
                                                               int C, int P, FastDiv dP, int M, int act, float act_scale)
{
    const int m = blockIdx.x * 256 + threadIdx.x, n = blockIdx.y;
    if (m >= M) return;
    float v = bias ? bf16_to_f32(bias[n]) : 0.f;
    const float *q = part + (long)n * M + m;
    for (int s = 0; s < nsplit; s++) v += q[(long)s * C * M];
    const int b = fdiv(m, dP), p = m - b * P;
    out[((long)b * C + n) * P + p] = f32_to_bf16(d2c_epilogue(v, act, act_scale));
}

// ============================================================ grad-column rows of the deformable operator
//   gcol[pair][m][c] = sum_o gout[m][o] * W[o][64 j + c][tap]     (pair = chunk j of 64 input channels and tap)
// The reduction is short (S steps of 64 output channels), the results are many.  A wavefront holds its 64 rows of grad_out in
// registers, all output channels of them (S * 32 registers), and goes along the pairs; a workgroup = 4 wavefronts, 256 rows,
// one per compute unit.  Only the weights go through LDS: 64 columns x 64 output channels a step, kGradBuf steps deep.
// Each is read by four wavefronts for 64 rows each: LDS is busy half of the matrix instructions' time, and a step brings
// 8 KB for 512 matrix clocks.  Two sets of accumulators: the results of a tile leave between the matrix instructions
// of the next one.  Column n of the two blocks of 32 holds the channels 2n and 2n + 1, so that a lane has both in its own
// registers and 32 lanes write a whole row, without LDS and without an exchange between lanes.
// An XCD's workgroups share a range of pairs whose weights fit its L2 (cgroups ranges) and, where there are fewer than
// eight, a range of row tiles; runs go along the pairs of a row tile.
// Bound: the rows it writes (256 -> 256 channels on 32x60x108: 2.9 GB at 3.9 TB/s), with more output channels the matrix instructions beside them
// (512 -> 512 in 8 groups on 2x8x30x54: matrix cores busy for 61 % of the cycles, at the 1.9 GHz that the chip holds meanwhile, 2.4 TB/s).
// us, tiles of 256 x 256 with both operands and the results through LDS (above 256 output channels: tiled_bwd_col32_kernel), and this way:
// 256 -> 256 on 2x8x30x54 142, 106; on 32x60x108 965, 731; 1024 -> 256 on 8x30x54 263, 191; 512 -> 512 in 8 groups 427, 360.
struct GradColArgs {
    const unsigned char *src;         // channels-last grad_out, rows of `rowb` bytes
    const unsigned char *wt;          // [pair][step][64 columns][64] bfloat16, slots swizzled
    bf16_t *gcol;
    unsigned rowb;
    int M, npair, ntile, cgroups;
};
constexpr int kGradBuf = 8;
template <int S>
__global__ void __launch_bounds__(kThreads, 1) grad_col_kernel(GradColArgs a)
{
    constexpr int RB = 2, CB = 2, NB = kGradBuf, WB = 8192, RQ = 2, NM = RB * CB;          // RQ: requests of a wavefront and step
    constexpr int TS = S * 4 * NM, NST = RB * 16;                                          // matrix instructions and stores of a tile
    // requests and stores of a wavefront between the requests for a step and the wait for it, at least: while the pipeline
    // fills, and later
    constexpr int kYoung = RQ * (NB - 2), kOld = kYoung + NST * (NB - 2) / S - 2, kLater = kOld < kYoung ? kYoung : (kOld > 63 ? 63 : kOld);
    __shared__ __align__(1024) unsigned char s_t[NB * WB];

    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xcd = blockIdx.x & 7, j = (int)blockIdx.x >> 3, per = (int)gridDim.x >> 3, rgroups = 8 / a.cgroups;
    const int cg = xcd % a.cgroups, rg = xcd / a.cgroups;
    const int c_lo = a.npair * cg / a.cgroups, c_hi = a.npair * (cg + 1) / a.cgroups, nc = c_hi - c_lo;
    const int r_lo = a.ntile * rg / rgroups, r_hi = a.ntile * (rg + 1) / rgroups;
    const long units = (long)(r_hi - r_lo) * nc;
    const int u_lo = (int)(units * j / per), u_hi = (int)(units * (j + 1) / per);
    if (u_lo >= u_hi) return;

    // --- requests: the steps of the weights in the order in which they are wanted (after the last one: that one again, which
    // nothing reads)
    int row = r_lo + u_lo / nc, col = c_lo + u_lo % nc;
    int bj = 0, bcol = col, bleft = (u_hi - u_lo) * S - 1;
    const unsigned char *bsrc = a.wt + (long)bcol * S * WB + wave * 1024 + lane * 16;
    auto advance = [&]() {
        if (bleft == 0) return;
        bleft--;
        bsrc += WB;
        if (++bj < S) return;
        bj = 0;
        if (++bcol < c_hi) return;
        bcol = c_lo;
        bsrc -= (long)nc * S * WB;
    };
    auto request = [&](int i, int buf) { dma16(bsrc + i * 4096, s_t + buf * WB + wave * 1024 + i * 4096); };

    // --- this wavefront's rows (those past the last one: the last one, stored nowhere)
    u32x4_t x[RB][S * 4];
    auto load_rows = [&]() {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const unsigned char *p = a.src + (unsigned)min(row * kWMT + wave * 64 + rb * 32 + n, a.M - 1) * (size_t)a.rowb + h * 16;
#pragma unroll
            for (int k = 0; k < S * 4; k++) x[rb][k] = *reinterpret_cast<const u32x4_t *>(p + k * 32);
        }
        // (waited for here: a wait behind the branch would be one of every tile)
        __builtin_amdgcn_s_waitcnt(0x0F70);
    };

    f32x16 acc[2][RB][CB];
    u32x4_t fb[2][CB];
    unsigned slot[4];
#pragma unroll
    for (int kg = 0; kg < 4; kg++) slot[kg] = lds_address(s_t) + (unsigned)(n * 128 + tile_slot<64>(n, kg * 2 + h) * 16);
    // --- the tile whose results are on their way out: the first of its rows, a descriptor of it that ends with the pair's last
    unsigned long long out_p = reinterpret_cast<unsigned long long>(a.gcol);
    unsigned out_bytes = 0;
    const unsigned lane_at = (unsigned)(wave * 64 + h * 4) * 128u + n * 4u;
    auto store = [&](auto SET, auto Q, auto &rs, const unsigned (&base)[2]) INLINE {
        constexpr int set = decltype(SET)::value, rb = decltype(Q)::value / 16, r = decltype(Q)::value % 16, at = (8 * (r >> 2) + (r & 3)) * 128;
        __builtin_amdgcn_raw_buffer_store_b32(pack_bf16x2(acc[set][rb][0][r], acc[set][rb][1][r]), rs, (int)(base[rb] + at), 0, 2);
    };
    auto out_rsrc = [&]() INLINE {
        const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)out_p), hi = __builtin_amdgcn_readfirstlane((unsigned)(out_p >> 32));
        return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>((unsigned long long)hi << 32 | lo), 0,
                                                 (int)__builtin_amdgcn_readfirstlane(out_bytes), 0x00020000);
    };

    for (int b = 0; b < NB; b++) {
#pragma unroll
        for (int i = 0; i < RQ; i++) request(i, b);
        advance();
    }
    load_rows();
    group_barrier();
#pragma unroll
    for (int cb = 0; cb < CB; cb++) fb[0][cb] = lds_read16(slot[0] + cb * 4096);
    int buf = 0, done = 0;                                 // steps done, as far as it matters
    auto tile = [&](auto SET) INLINE {
        constexpr int set = decltype(SET)::value;
        const auto rs = out_rsrc();
        // (anew for every tile: what is added to these stays in the stores)
        unsigned base[2] = {lane_at, lane_at + 4096u};
        opaque_v(base[0]); opaque_v(base[1]);
        for_each_const([&](auto ST) INLINE {
            constexpr int st = decltype(ST)::value;
            const int nbuf = buf + 1 == NB ? 0 : buf + 1;
            for_each_const([&](auto KG) INLINE {
                constexpr int kg = decltype(KG)::value, s = kg & 1, lo = kg == 3 ? NM * 3 / 8 : 0;
                const unsigned p = slot[(kg + 1) & 3] + (kg == 3 ? nbuf : buf) * WB;
                for_each_const([&](auto I) INLINE {
                    constexpr int i = decltype(I)::value, cb = i / RB, rb = i % RB, e = (st * 4 + kg) * NM + i;
                    constexpr int issued = i <= lo ? 0 : ((i - lo) * CB + NM - lo - 1) / (NM - lo), next = i < lo ? 0 : ((i + 1 - lo) * CB + NM - lo - 1) / (NM - lo);
                    if constexpr (kg == 3 && i == lo) {
                        // every wavefront holds the last operands of the step, its buffer is free; the next step's are there
                        if (done >= NB) wait_vm<kLater>(); else wait_vm<kYoung>();
                        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
                    }
                    if constexpr (rb == 0) {
                        if constexpr (kg == 3 && i >= lo) landed(fb[s][cb]);
                        else wait_lds<CB - 1 - cb + issued>(fb[s][cb]);
                    }
                    const bf16x8_t xv = __builtin_bit_cast(bf16x8_t, x[rb][st * 4 + kg]), wv = __builtin_bit_cast(bf16x8_t, fb[s][cb]);
                    if constexpr (st == 0 && kg == 0) {
                        f32x16 z;
#pragma unroll
                        for (int r = 0; r < 16; r++) z[r] = 0.f;
                        acc[set][rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, wv, z, 0, 0, 0);
                    } else acc[set][rb][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, wv, acc[set][rb][cb], 0, 0, 0);
                    for_each_const([&](auto R) INLINE {
                        constexpr int r = issued + decltype(R)::value;
                        fb[s ^ 1][r] = lds_read16_at<r * 4096>(p);
                    }, std::make_integer_sequence<int, next - issued>{});
                    if constexpr (kg == 3 && i >= lo && i - lo < RQ) request(i - lo, buf);
                    constexpr int q = (e * NST + TS - 1) / TS, q1 = ((e + 1) * NST + TS - 1) / TS;
                    for_each_const([&](auto Q) INLINE { store(std::integral_constant<int, set ^ 1>{}, std::integral_constant<int, q + decltype(Q)::value>{}, rs, base); },
                                   std::make_integer_sequence<int, q1 - q>{});
                    __builtin_amdgcn_sched_barrier(0);
                }, std::make_integer_sequence<int, NM>{});
            }, std::make_integer_sequence<int, 4>{});
            advance();
            buf = nbuf;
            done = min(done + 1, NB);
        }, std::make_integer_sequence<int, S>{});
        out_p = reinterpret_cast<unsigned long long>(a.gcol) + ((unsigned long long)col * a.M + row * kWMT) * 128;
        out_bytes = (unsigned)(a.M - row * kWMT) * 128u;
    };
    auto next_tile = [&]() {
        if (++col < c_hi) return;
        col = c_lo; row++;
        load_rows();
    };
    auto drain = [&](auto SET) INLINE {
        const auto rs = out_rsrc();
        const unsigned base[2] = {lane_at, lane_at + 4096u};
        for_each_const([&](auto Q) INLINE { store(SET, Q, rs, base); __builtin_amdgcn_sched_barrier(0); }, std::make_integer_sequence<int, NST>{});
    };
    constexpr std::integral_constant<int, 0> k0{};
    constexpr std::integral_constant<int, 1> k1{};
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[1][rb][cb][r] = 0.f;
    for (int u = u_lo;;) {
        tile(k0);
        if (++u == u_hi) { drain(k0); break; }
        next_tile();
        tile(k1);
        if (++u == u_hi) { drain(k1); break; }
        next_tile();
    }
    // (the reads and requests behind the last step)
#pragma unroll
    for (int cb = 0; cb < CB; cb++) wait_lds<0>(fb[0][cb]);
    wait_vm<0>();
}
// W[o][c][tap] -> the operand order above: a thread makes vector v of eight o of (channel, tap) e
D2C_DEV void grad_col_weight(const bf16_t *w, uint4 *wt, int Cout, int Cin, int K, const FastDiv &dK, int S, int e, int v)
{
    const int CK = Cin * K;
    if (e >= CK) return;
    alignas(16) bf16_t t[8];
#pragma unroll
    for (int q = 0; q < 8; q++) t[q] = v * 8 + q < Cout ? w[(long)(v * 8 + q) * CK + e] : (bf16_t)0;
    const int c = fdiv(e, dK), k = e - c * K, pair = (c >> 6) * K + k, ch = c & 63;
    wt[(((long)pair * S + (v >> 3)) * 64 + (ch & 1) * 32 + (ch >> 1)) * 8 + tile_slot<64>(ch >> 1, v & 7)] = *reinterpret_cast<const uint4 *>(t);
}

// ============================================================ grad_weight over sampled columns
//   gW[o][(pair, c)] = sum_m gout[o][m] * col[pair][m][c]          (pair = chunk of 64 input channels and tap)
// The pipeline of conv_wide_kernel once more, the reduction over positions: a workgroup = four pairs (256 columns) x OT output
// channels over a share of the 64-position tiles, four wavefronts of 128 columns x OT / 2, one workgroup per compute unit.  A
// step's columns (three buffers, two steps ahead: they come from device memory) are read with the transposing LDS load,
// grad_out comes in fragment order (pack_gout_kernel; two buffers).  Bound as conv_wide_kernel: OT * 8 matrix clocks a step
// against 64 KB of operands.  Shares of all items run side by side on an XCD, so that grad_out is read there once.
// Every workgroup stores its sums; col_weight_finish_kernel adds them up on their way into grad_weight.  (Float atomics into one
// accumulator, all workgroups at the end of the launch, take 40 us for the 62 MB of 256 -> 256 channels, these stores 10.)
// The kernel it took the place of (tiled_bwd_weight_col_kernel: 512 output channels x 128 columns, with 256 channels half of its
// wavefronts multiply nothing; it still serves several weight groups, columns in the rows' place, slices, calls that want grad_weight alone
// over kept columns, and sums that have no room where the grad-column rows were), us, the sums brought into grad_weight included:
// 512 -> 512 in 8 groups on 2x8x30x54 413, 332; 256 -> 256 there 146, 114; on 32x60x108 869, 619 (reading 2.9 GB of columns once takes
// 520); 1024 -> 256 on 8x30x54 230, 192; 2048 -> 256 with 7 taps 130, 116.  Whole training steps of small problems gain too:
// 128 -> 64 on 420 positions 104, 101; 128 -> 128 on 1400 122, 112; 512 -> 512 267, 238; tiles that are mostly padding lose nothing (both
// products' kernels of before, and these: 256 -> 1 on 12960 308, 285; 256 -> 40 291, 290; 256 -> 130 332, 323; 512 -> 144 564, 543).
// One weight group.
struct ColWeightArgs {
    const unsigned char *gp;          // [tile of 128 positions][row block of 32][k-group of 16][lane] 16 bytes
    const unsigned char *col;         // [pair][position][64] bfloat16
    float *part;                      // [piece][item][pair of 4][16 x 4 channels][OT][4]
    long pair_bytes;
    int npair, otiles, nitem;         // pairs, tiles of OT output channels, items (tiles x sets of four pairs)
    int OBT;                          // row blocks of the fragments
    int ntile, nsplit;
};
template <int OT>
__global__ void __launch_bounds__(kThreads, 1) col_weight_kernel(ColWeightArgs a)
{
    constexpr int OB = 4, PB = OT / 64;                    // 32-blocks of a wavefront: columns, output channels
    constexpr int ABYTES = 4 * 64 * 128, BBYTES = OT * 128;
    constexpr int AD = 8, BD = BBYTES / 4096, NM = OB * PB;
    __shared__ __align__(1024) unsigned char s_t[3 * ABYTES + 2 * BBYTES];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int id = xcd_swizzle(blockIdx.x, gridDim.x), piece = id / a.nitem, item = id - piece * a.nitem;
    const int ot = item % a.otiles, ci = item / a.otiles;
    const int t_lo = (int)((long)a.ntile * piece / a.nsplit), t_hi = (int)((long)a.ntile * (piece + 1) / a.nsplit);

    // --- requests: a wavefront fetches the columns of a pair (past the last pair: that one again, stored in no gradient), eight
    // rows at a time; 16-byte pieces of a row are permuted so that the transposing reads, 64 bytes of four consecutive rows,
    // meet no bank twice
    const int pair = min(ci * 4 + wave, a.npair - 1);
    const unsigned char *asrc = a.col + pair * a.pair_bytes + (long)t_lo * 8192 + (lane >> 3) * 128 +
                                ((lane & 7) ^ ((lane >> 4) & 1) << 2) * 16;
    int at = t_lo, bt = t_lo;                              // the tiles that the next requests belong to
    // (after the last tile: that one again, which nothing reads)
    auto advance_cols = [&]() { if (at + 1 < t_hi) { at++; asrc += 8192; } };
    // ... and k-group `wave` of every row block (past the last block: that one again)
    const unsigned char *bsrc = a.gp + ((long)(t_lo >> 1) * a.OBT * 8 + (t_lo & 1) * 4 + wave) * 1024 + lane * 16;
    unsigned bo[BD];
#pragma unroll
    for (int i = 0; i < BD; i++) bo[i] = (unsigned)min(ot * (OT / 32) + i, a.OBT - 1) * 8192u;
    auto advance_gout = [&]() {
        if (bt + 1 >= t_hi) return;
        bsrc += bt & 1 ? (long)a.OBT * 8192 - 4096 : 4096;
        bt++;
    };
    unsigned char *const sa = s_t + wave * 8192, *const sb = s_t + 3 * ABYTES + wave * 1024;
    auto col_request = [&](int i, int buf) { dma16(asrc + i * 1024, sa + buf * ABYTES + i * 1024); };
    auto gout_request = [&](int i, int buf) { dma16(bsrc + bo[i], sb + buf * BBYTES + i * 4096); };

    f32x16 acc[OB][PB];
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int pb = 0; pb < PB; pb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[ob][pb][r] = 0.f;
    const int wo = wave & 1, wp = wave >> 1;               // halves of the columns, of the output channels
    // transposing reads: position (lane / 32) * 8 + (lane % 16) / 4 (and four more), channel (lane / 16 % 2) * 16 + lane % 4 * 4
    const unsigned tr = (unsigned)((lane >> 5) * 8 + ((lane & 15) >> 2)) * 128u + (unsigned)(((lane >> 4) & 1) * 32 + (lane & 3) * 8);
    const unsigned fl = (unsigned)((lane >> 3) & 1) * 64u; // (rows 2, 3 of four: the 64-byte halves changed over)
    const unsigned ra0 = lds_address(s_t) + wo * 16384 + tr + fl, ra1 = lds_address(s_t) + wo * 16384 + tr + (64u - fl);
    const unsigned rb = lds_address(s_t) + 3 * ABYTES + wp * PB * 4096 + lane * 16;
    TrVec fb[2][OB];
    u32x4_t fa[2][PB];
    // operand vector i of k-group KG: columns, then output channels
    auto cols = [](auto I, auto KG, TrVec &v, unsigned p0, unsigned p1) INLINE {
        constexpr int i = decltype(I)::value, o = (i >> 1) * 8192 + decltype(KG)::value * 2048;
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v.lo) : "v"(i & 1 ? p1 : p0), "n"(o));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v.hi) : "v"(i & 1 ? p1 : p0), "n"(o + 512));
    };
    auto gout = [](auto I, auto KG, u32x4_t &v, unsigned p) INLINE {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(p), "n"((decltype(I)::value - OB) * 4096 + decltype(KG)::value * 1024));
    };

    for (int i = 0; i < AD; i++) col_request(i, 0);
#pragma unroll
    for (int i = 0; i < BD; i++) gout_request(i, 0);
    advance_cols();
    for (int i = 0; i < AD; i++) col_request(i, 1);
    advance_cols();
    advance_gout();
#pragma unroll
    for (int i = 0; i < BD; i++) gout_request(i, 1);
    wait_vm<AD + BD>();
    group_barrier();
    // (in the order of wide_group)
    constexpr std::integral_constant<int, 0> k0{};
    cols(k0, k0, fb[0][0], ra0, ra1);
    for_each_const([&](auto I) INLINE { gout(std::integral_constant<int, OB + decltype(I)::value>{}, k0, fa[0][decltype(I)::value], rb); },
                   std::make_integer_sequence<int, PB>{});
    for_each_const([&](auto I) INLINE { cols(std::integral_constant<int, 1 + decltype(I)::value>{}, k0, fb[0][1 + decltype(I)::value], ra0, ra1); },
                   std::make_integer_sequence<int, OB - 1>{});
    int abuf = 0, bbuf = 0;
    for (int t = t_lo; t < t_hi; t++) {
        advance_gout();
        const int a1 = abuf == 2 ? 0 : abuf + 1, a2 = a1 == 2 ? 0 : a1 + 1, b1 = bbuf ^ 1;
        for_each_const([&](auto KG) INLINE {
            constexpr int kg = decltype(KG)::value;
            constexpr std::integral_constant<int, (kg + 1) & 3> nk{};
            const unsigned ab = (kg == 3 ? a1 : abuf) * ABYTES, p0 = ra0 + ab, p1 = ra1 + ab, pb_ = rb + (kg == 3 ? b1 : bbuf) * BBYTES;
            wide_group<OB, PB, kg>(acc, fa, fb,
                [&](auto I, auto &v) INLINE {
                    if constexpr (decltype(I)::value < OB) cols(I, nk, v, p0, p1);
                    else gout(I, nk, v, pb_);
                },
                [&](auto I) INLINE {
                    constexpr int i = decltype(I)::value, n = NM / (AD / 2), lo = NM * 3 / 8, g = (BD + NM - lo - 1) / (NM - lo);
                    if constexpr ((kg == 1 || kg == 2) && i % n == 0) col_request((kg - 1) * (AD / 2) + i / n, a2);
                    if constexpr (kg == 3 && i >= lo)
                        for_each_const([&](auto Q) INLINE {
                            constexpr int q = (i - lo) * g + decltype(Q)::value;
                            if constexpr (q < BD) gout_request(q, bbuf);
                        }, std::make_integer_sequence<int, g>{});
                },
                // (the columns of the step after the next one may be under way)
                [&]() INLINE { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(AD) : "memory"); });
        }, std::make_integer_sequence<int, 4>{});
        advance_cols();
        abuf = a1; bbuf = b1;
    }
    // (the reads and requests behind the last step)
#pragma unroll
    for (int ob = 0; ob < OB; ob++) wait_lds<0>(fb[0][ob]);
#pragma unroll
    for (int pb = 0; pb < PB; pb++) landed(fa[0][pb]);
    wait_vm<0>();

    // a lane holds four consecutive channels of its output channel
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.part + (long)id * (256 * OT), 0, 256 * OT * 4, 0x00020000);
    for_each_const([&](auto I) INLINE {
        constexpr int ob = decltype(I)::value / 4, r4 = decltype(I)::value % 4;
        for_each_const([&](auto J) INLINE {
            constexpr int pb = decltype(J)::value;
            const f32x16 &v = acc[ob][pb];
            const u32x4_t t = {__float_as_uint(v[r4 * 4]), __float_as_uint(v[r4 * 4 + 1]), __float_as_uint(v[r4 * 4 + 2]), __float_as_uint(v[r4 * 4 + 3])};
            const int c4 = (wo * 4 + ob) * 8 + r4 * 2 + (lane >> 5), o = (wp * PB + pb) * 32 + (lane & 31);
            __builtin_amdgcn_raw_buffer_store_b128(t, rs, (c4 * OT + o) * 16, 0, 0);
        }, std::make_integer_sequence<int, PB>{});
        __builtin_amdgcn_sched_barrier(0);
    }, std::make_integer_sequence<int, OB * 4>{});
}

// grad_weight[o][c][tap] = the sums above: a workgroup = kFinOut output channels x 16 input channels, all taps, through LDS
constexpr int kFinOut = 8;
struct ColWeightFinishArgs {
    const float *part;
    bf16_t *gw;
    int nsplit, nitem, otiles, OT, K, Cout, Cin, nob;      // nob: sets of kFinOut output channels
    int wide;                                              // `gw` on 16 bytes
};
__global__ void __launch_bounds__(256) col_weight_finish_kernel(ColWeightFinishArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int ob = blockIdx.x % a.nob, c16 = blockIdx.x / a.nob;
    const int j = c16 >> 2, run = 16 * a.K, rs = run * 2 + 16;         // chunk; elements of a row, bytes of it in LDS
    const int o0 = ob * kFinOut, ot = o0 / a.OT, nr = min(kFinOut, a.Cout - o0);
    const float4 *const part = reinterpret_cast<const float4 *>(a.part) + (o0 - ot * a.OT);
    const long piece = (long)a.nitem * 64 * a.OT;
    for (int i = threadIdx.x; i < a.K * 32; i += 256) {
        const int o = i & 7, c4 = (i >> 3) & 3, k = i >> 5, pair = j * a.K + k;
        const float4 *q = part + (((long)(pair >> 2) * a.otiles + ot) * 64 + (pair & 3) * 16 + (c16 & 3) * 4 + c4) * a.OT + o;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
        for (int s = 0; s < a.nsplit; s++) {
            const float4 t = q[s * piece];
            v.x += t.x; v.y += t.y; v.z += t.z; v.w += t.w;
        }
        bf16_t *d = reinterpret_cast<bf16_t *>(smem + o * rs) + c4 * 4 * a.K + k;
        d[0] = f32_to_bf16(v.x); d[a.K] = f32_to_bf16(v.y); d[2 * a.K] = f32_to_bf16(v.z); d[3 * a.K] = f32_to_bf16(v.w);
    }
    __syncthreads();
    bf16_t *const dst = a.gw + ((long)o0 * a.Cin + c16 * 16) * a.K;
    const long row = (long)a.Cin * a.K;
    if (a.wide) {
        const int nv = run / 8;
        for (int i = threadIdx.x; i < nr * nv; i += 256) {
            const int r = i / nv, v = i - r * nv;
            *reinterpret_cast<uint4 *>(dst + r * row + v * 8) = *reinterpret_cast<const uint4 *>(smem + r * rs + v * 16);
        }
    } else {
        for (int i = threadIdx.x; i < nr * run; i += 256) {
            const int r = i / run, v = i - r * run;
            dst[r * row + v] = *reinterpret_cast<const bf16_t *>(smem + r * rs + v * 2);
        }
    }
}

// ============================================================ grad_weight
// One workgroup = one tap, 128 input channels, 32 * OBT output channels, over its share of the 64-position tiles.  A
// step brings 64 input rows of 256 bytes and the grad_out fragments of 64 positions to LDS by DMA; the rows are read
// with the transposing LDS load (the reduction runs over positions).  Wavefronts share the step: WO along the output
// channels, 4 / WO along the input channels.  Bound by the requests (20 - 32 KiB per step and 128 - 512 matrix clocks).
struct ConvWeightArgs {
    RowMap map;                       // forward map
    const unsigned char *src;         // channels-last input, rows of `rowb` bytes, a row of zeros at `zrow`
    const uint4 *gp;                  // grad_out fragments [tile of 64][row block of 32][k-group][lane]
    float *part;                      // [split][tap][128-channel block][C][128]
    unsigned rowb, zrow;
    int C, OBP;                       // output channels; row blocks of the fragment copy
    int ncb, K, notile, nsplit, ntile;
    int half_last;                    // the last block of 128 channels has 64 only
};

template <int OBT>
__global__ void __launch_bounds__(kThreads, 2) conv_weight_kernel(ConvWeightArgs a)
{
    constexpr int WO = OBT == 4 ? 2 : 1;
    constexpr int OB = OBT / WO, CB = WO;                  // 32-blocks of a wavefront: output / input channels
    constexpr int XB = kCW * 256, GB = OBT * 4096, STAGE = XB + GB;
    constexpr int NST = STAGE > 24 * 1024 ? 2 : 3;
    constexpr int XD = 4, GD = OBT;
    __shared__ __align__(1024) unsigned char s_t[NST * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int id = xcd_swizzle(blockIdx.x, gridDim.x);
    // (neighbouring workgroups: the taps of one channel block and share of positions, whose rows overlap)
    const int ot = id % a.notile; id /= a.notile;
    const int k = id % a.K; id /= a.K;
    const int split = id % a.nsplit, cb = id / a.nsplit;
    const int t_lo = (int)((long)a.ntile * split / a.nsplit), t_hi = (int)((long)a.ntile * (split + 1) / a.nsplit);
    const int kx = k % a.map.g.kw, ky = (k / a.map.g.kw) % a.map.g.kh, kz = k / (a.map.g.kw * a.map.g.kh);

    // rows of a request: 4 x 256 bytes; wavefront w fetches rows 16 w .. 16 w + 15
    const int lrow = lane >> 4, lslot = lane & 15;
    const bool cut = a.half_last && cb == a.ncb - 1;
    auto issue = [&](int t, int buf) {
        const RowPos rp = row_pos(a.map, t * kCW + wave * 16 + (lane & 15));
        const int row = source_row(a.map, rp, kz, ky, kx);
        unsigned char *sx = s_t + buf * STAGE + wave * 4096, *sg = s_t + buf * STAGE + XB;
#pragma unroll
        for (int i = 0; i < XD; i++) {
            const int rl = i * 4 + lrow;
            const int sr = __builtin_amdgcn_ds_bpermute(rl << 2, row);
            const int v = lslot ^ ((rl & 3) << 2);         // channel vector of this slot, see the reads below
            const bool ok = sr >= 0 && !(cut && v >= 8);
            const unsigned o = ok ? (unsigned)sr * a.rowb + (unsigned)(cb * 256 + v * 16) : a.zrow + (unsigned)(v & 7) * 16u;
            dma16(a.src + o, sx + i * 1024);
        }
        const unsigned char *g = reinterpret_cast<const unsigned char *>(a.gp) +
                                 ((long)t * a.OBP + ot * OBT) * 4096 + wave * 1024 + lane * 16;
#pragma unroll
        for (int i = 0; i < GD; i++) dma16(g + i * 4096, sg + i * 4096 + wave * 1024);
    };

    f32x16 acc[OB][CB];
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int c = 0; c < CB; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[ob][c][r] = 0.f;
    const int wo = wave % WO, wc = wave / WO;
    // transposing reads: lane -> position (g16 >> 1) * 8 + (l16 >> 2), channel block + (g16 & 1) * 16 + (l16 & 3) * 4;
    // the 64-byte segments of four consecutive rows lie in different quarters of the banks
    const int l16 = lane & 15, g16 = lane >> 4;
    const int prow = (g16 >> 1) * 8 + (l16 >> 2);
    unsigned xo[CB];
#pragma unroll
    for (int c = 0; c < CB; c++)
        xo[c] = lds_address(s_t) + prow * 256 + (((wc * CB + c) ^ (prow & 3)) * 64) + (g16 & 1) * 32 + (l16 & 3) * 8;
    const unsigned go = lds_address(s_t) + XB + wo * OB * 4096 + lane * 16;
    typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));

    if (t_lo < t_hi) {
        issue(t_lo, 0);
        if (NST == 3 && t_lo + 1 < t_hi) issue(t_lo + 1, 1);
    }
    int buf = 0, nbuf = NST - 1;
    for (int t = t_lo; t < t_hi; t++) {
        if (NST == 3 && t + 1 < t_hi) wait_vm<XD + GD>(); else wait_vm<0>();
        group_barrier();
        if (t + NST - 1 < t_hi) issue(t + NST - 1, nbuf);
        const unsigned bo = buf * STAGE;
#pragma unroll
        for (int kg = 0; kg < 4; kg++) {
            u32x4_t fg[OB];
            u32x2_t lo[CB], hi[CB];
#pragma unroll
            for (int ob = 0; ob < OB; ob++) fg[ob] = lds_read16(go + bo + ob * 4096 + kg * 1024);
#pragma unroll
            for (int c = 0; c < CB; c++) {
                asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(lo[c]) : "v"(xo[c] + bo + kg * 4096));
                asm volatile("ds_read_b64_tr_b16 %0, %1 offset:1024" : "=v"(hi[c]) : "v"(xo[c] + bo + kg * 4096));
            }
#pragma unroll
            for (int ob = 0; ob < OB; ob++) wait_lds<0>(fg[ob]);
#pragma unroll
            for (int c = 0; c < CB; c++) asm volatile("" : "+v"(lo[c]), "+v"(hi[c]));
#pragma unroll
            for (int ob = 0; ob < OB; ob++)
#pragma unroll
                for (int c = 0; c < CB; c++)
                    mma_kgroup<bf16_t, false>(acc[ob][c], __builtin_bit_cast(uint4, fg[ob]),
                                              make_uint4(lo[c].x, lo[c].y, hi[c].x, hi[c].y));
        }
        buf = buf + 1 == NST ? 0 : buf + 1;
        nbuf = nbuf + 1 == NST ? 0 : nbuf + 1;
    }
    float *part = a.part + (((long)split * a.K + k) * a.ncb + cb) * a.C * 128;
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int c = 0; c < CB; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int o = (ot * OBT + wo * OB + ob) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (o < a.C) part[(long)o * 128 + (wc * CB + c) * 32 + (lane & 31)] = acc[ob][c][r];
            }
}

// partial sums -> gW[o][c][tap]: a workgroup takes one output channel and one block of 128 input channels, through LDS
// (the sums of a tap are rows of channels, grad_weight has the taps of a channel side by side)
constexpr int kFinishTaps = 64;       // taps per round
__global__ void __launch_bounds__(256) conv_weight_finish_kernel(const float *part, bf16_t *gw, int nsplit, int K, int ncb, int C,
                                                                 int Cin)
{
    __shared__ bf16_t t[128 * (kFinishTaps + 1)];
    const int cb = blockIdx.x % ncb, o = blockIdx.x / ncb;
    const int nc = min(128, Cin - cb * 128);
    const long sstr = (long)K * ncb * C * 128;
    for (int k0 = 0; k0 < K; k0 += kFinishTaps) {
        const int nk = min(kFinishTaps, K - k0);
        for (int i = threadIdx.x; i < nk * 128; i += 256) {
            const int c = i & 127, k = i >> 7;
            const float *q = part + (((long)(k0 + k) * ncb + cb) * C + o) * 128 + c;
            float v = 0.f;
            for (int s = 0; s < nsplit; s++) v += q[s * sstr];
            t[c * nk + k] = f32_to_bf16(v);
        }
        __syncthreads();
        bf16_t *d = gw + ((long)o * Cin + cb * 128) * K + k0;
        if (nk == K) {
            for (int i = threadIdx.x; i < nc * nk; i += 256) d[i] = t[i];
        } else {
            for (int i = threadIdx.x; i < nc * nk; i += 256) d[(long)(i / nk) * K + i % nk] = t[i];
        }
        __syncthreads();
    }
}

// ============================================================ operand orders, one launch per direction
struct ConvPrepArgs {
    // input -> channels-last rows, then zeros
    const bf16_t *x;
    bf16_t *xcl;
    int C, vol, N, nbx, nby, nblk_x, zrow_words;
    // weights: column tiles [step][tile][NT][KC]; back: the transposed product (columns = input channels)
    const bf16_t *w;
    uint4 *wt;
    int Cout, Cin, K, NT, KC, nchunk, nct, back, nblk_w;
    long nvec;
    // grad_out -> channels-last rows of Cp channels (+ a row of zeros) and fragments of tiles of 64 << gp_wide positions
    const bf16_t *gout;
    bf16_t *gcl;
    uint4 *gp;
    int Cp, OBP, P, M, ngt, ngc, nblk_g, gp_wide;
    FastDiv dP;
    // bias gradient
    bf16_t *gb;
    int nblk_b;
    // weights of grad_col_kernel
    uint4 *gcw;
    int gcS, ngcw, nblk_gcw;          // steps; workgroups per vector, in all
    FastDiv dK;
    // ranges of the workspace to clear
    uint32_t *zero[2];
    size_t zwords[2];
    int nblk_z;
};

__global__ void __launch_bounds__(256) conv_prepare_kernel(ConvPrepArgs a)
{
    constexpr int RS = 66;            // LDS row stride in elements
    __shared__ __align__(16) bf16_t s_t[64 * 72];
    int b = blockIdx.x;
    if (b < a.nblk_x) {
        // 64 voxels x 64 channels
        const int bx = b % a.nbx, by = (b / a.nbx) % a.nby, n = b / (a.nbx * a.nby);
        const int v0 = bx * 64, c0 = by * 64;
        const bf16_t *xb = a.x + (long)n * a.C * a.vol;
        bf16_t *ob = a.xcl + (long)n * a.C * a.vol;
        if (b == 0 && (int)threadIdx.x < a.zrow_words) reinterpret_cast<unsigned *>(a.xcl + (long)a.N * a.C * a.vol)[threadIdx.x] = 0u;
        for (int i = threadIdx.x; i < 512; i += 256) {
            const int c = c0 + i / 8, v = v0 + (i % 8) * 8;
            if (v < a.vol) {
                const uint4 q = load_run<bf16_t>(xb + (long)c * a.vol + v, a.vol - v);
                const unsigned u[4] = {q.x, q.y, q.z, q.w};
                bf16_t *t = s_t + ((i % 8) * 8) * RS + i / 8;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    t[(2 * e) * RS] = (bf16_t)(u[e] & 0xffffu);
                    t[(2 * e + 1) * RS] = (bf16_t)(u[e] >> 16);
                }
            }
        }
        __syncthreads();
        for (int i = threadIdx.x; i < 512; i += 256) {
            const int v = v0 + i / 8, c = c0 + (i % 8) * 8;
            if (v < a.vol) {
                const unsigned *t = reinterpret_cast<const unsigned *>(s_t + (i / 8) * RS + (i % 8) * 8);
                *reinterpret_cast<uint4 *>(ob + (long)v * a.C + c) = make_uint4(t[0], t[1], t[2], t[3]);
            }
        }
        return;
    }
    b -= a.nblk_x;
    if (b < a.nblk_w) {
        // one 16-byte vector of the result per thread and turn, taps fastest (the runs of W)
        const int R = a.back ? a.Cin : a.Cout;              // columns that exist
        const int Rp = a.nct * a.NT, D = a.back ? a.Cout : a.Cin, VPR = a.KC / 8, nv = a.nchunk * VPR;
        for (long i = (long)b * 256 + threadIdx.x; i < a.nvec; i += (long)a.nblk_w * 256) {
            const int k = (int)(i % a.K);
            long r = i / a.K;
            int col, v;                                      // column, channel vector along the reduction
            if (a.back) { col = (int)(r % Rp); v = (int)(r / Rp); }
            else { v = (int)(r % nv); col = (int)(r / nv); }
            alignas(16) bf16_t e[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int d = v * 8 + q;
                const bool ok = col < R && d < D;
                const long src = a.back ? ((long)d * a.Cin + col) * a.K + k : ((long)col * a.Cin + d) * a.K + k;
                e[q] = ok ? a.w[src] : (bf16_t)0;
            }
            const int ct = col / a.NT, cr = col % a.NT, j = v / VPR, vv = v % VPR;
            const int slot = a.KC == 64 ? tile_slot<64>(cr, vv) : tile_slot<32>(cr, vv);
            a.wt[((((long)k * a.nchunk + j) * a.nct + ct) * a.NT + cr) * VPR + slot] = *reinterpret_cast<const uint4 *>(e);
        }
        return;
    }
    b -= a.nblk_w;
    if (b < a.nblk_g) {
        // 64 positions x 64 channels of grad_out, into both orders
        const int gt = b % a.ngt, gc = b / a.ngt;
        constexpr int GS = 72;                               // [channel][position], 16-byte aligned rows
        for (int i = threadIdx.x; i < 512; i += 256) {
            const int c = gc * 64 + i / 8, m = gt * 64 + (i % 8) * 8;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (c < a.Cout && m < a.M) {
                const int n = fdiv(m, a.dP), p = m - n * a.P;
                const bf16_t *const src = a.gout + ((long)n * a.Cout + c) * a.P + p;
                if (p + 8 <= a.P) {
                    v = __builtin_bit_cast(uint4, load_any<bf16_t>(src));
                } else {
                    // (the rows of a channel in the next samples are Cout * P apart)
                    alignas(16) bf16_t e[8];
                    long at = 0;
                    int r = p;
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        e[q] = m + q < a.M ? src[at] : (bf16_t)0;
                        at++;
                        if (++r == a.P) { r = 0; at += (long)(a.Cout - 1) * a.P; }
                    }
                    v = *reinterpret_cast<const uint4 *>(e);
                }
            }
            *reinterpret_cast<uint4 *>(s_t + (i / 8) * GS + (i % 8) * 8) = v;
        }
        __syncthreads();
        if (a.gp) {
            for (int i = threadIdx.x; i < 512; i += 256) {
                const int ln = i & 63, kg = (i >> 6) & 3, ob = i >> 8;
                if (gc * 2 + ob < a.OBP)
                    a.gp[((((long)(gt >> a.gp_wide) * a.OBP + gc * 2 + ob) * (4 << a.gp_wide)) + (gt & ((1 << a.gp_wide) - 1)) * 4 + kg) * 64 + ln] =
                        *reinterpret_cast<const uint4 *>(s_t + (ob * 32 + (ln & 31)) * GS + kg * 16 + (ln >> 5) * 8);
            }
        }
        if (a.gcl) {
            if (b == 0 && threadIdx.x < 128) reinterpret_cast<unsigned *>(a.gcl + (long)a.M * a.Cp)[threadIdx.x] = 0u;
            for (int i = threadIdx.x; i < 512; i += 256) {
                const int m = gt * 64 + i / 8, c = (i % 8) * 8;
                if (m < a.M && gc * 64 + c < a.Cp) {
                    alignas(16) bf16_t e[8];
#pragma unroll
                    for (int q = 0; q < 8; q++) e[q] = s_t[(c + q) * GS + i / 8];
                    *reinterpret_cast<uint4 *>(a.gcl + (long)m * a.Cp + gc * 64 + c) = *reinterpret_cast<const uint4 *>(e);
                }
            }
        }
        return;
    }
    b -= a.nblk_g;
    if (b < a.nblk_b) {
        bias_grad_body<bf16_t, 256>(a.gout, a.gb, a.N, a.Cout, a.P, b);
        return;
    }
    b -= a.nblk_b;
    if (b < a.nblk_gcw) {
        grad_col_weight(a.w, a.gcw, a.Cout, a.Cin, a.K, a.dK, a.gcS, b % a.ngcw * 256 + threadIdx.x, b / a.ngcw);
        return;
    }
    b -= a.nblk_gcw;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        uint4 *z = reinterpret_cast<uint4 *>(a.zero[j]);
        const size_t n = a.zwords[j] / 4;
        for (size_t i = (size_t)b * 256 + threadIdx.x; i < n; i += (size_t)a.nblk_z * 256) z[i] = make_uint4(0, 0, 0, 0);
        if (b == 0 && threadIdx.x < a.zwords[j] % 4) a.zero[j][n * 4 + threadIdx.x] = 0u;
    }
}

// ============================================================ host side
struct RowsPlan {
    int MT, NT, KC, nchunk, nct, S, ntile, nsplit, nfull;
    size_t wt_bytes, part_bytes;
};
// columns C, reduction over `depth` channels per tap, M rows
RowsPlan rows_plan(int C, int depth, int K, int M, int ncu)
{
    RowsPlan p;
    p.KC = depth <= 32 ? 32 : 64;
    p.nchunk = (depth + p.KC - 1) / p.KC;
    p.S = K * p.nchunk;
    // Tile, and number of pieces that the steps of a tile are shared out to, by what they cost in clocks of a compute unit:
    // rounds over the workgroups that run at a time, each its steps and about four more for its start and end; partial sums
    // are written and read once more.  (clocks of a step: from the rates on large problems)
    long best = -1;
    auto take = [&](long cost, int MT, int NT, int s, long full) {
        if (best >= 0 && cost * 20 >= best * 19) return;
        best = cost;
        p.MT = MT; p.NT = NT; p.nsplit = s; p.nfull = (int)full; p.nct = (C + NT - 1) / NT; p.ntile = (M + MT - 1) / MT;
    };
    auto parts = [&](long pieces, int MT, int NT) { return (pieces * (MT / 32) * (NT / 32) + ncu - 1) / ncu * 600 + 8000; };
    {
        // two workgroups to a compute unit; all tiles are shared out alike
        const int NT = C <= 32 ? 32 : (C <= 64 ? 64 : 128);
        const long items = (long)((M + kMT - 1) / kMT) * ((C + NT - 1) / NT), slots = 2L * ncu, clocks = C <= 32 ? 1500 : (C <= 64 ? 2000 : 2700);
        for (int s = 1; s <= 16 && s <= p.S; s++)
            take((items * s + slots - 1) / slots * ((p.S + s - 1) / s + 4) * clocks + (s > 1 ? parts(items * s, kMT, NT) : 0), kMT, NT, s, 0);
    }
    // one workgroup to a compute unit; the tiles of the last, partly filled round are shared out (results are written through
    // 32-bit offsets)
    for (int NT = 128; NT <= 256 && C > NT / 2 && p.KC == 64 && (size_t)C * M * 2 < 0xFFFF0000u; NT *= 2) {
        const long items = (long)((M + kWMT - 1) / kWMT) * ((C + NT - 1) / NT), full = items / ncu * ncu, rest = items - full,
                   clocks = NT == 256 ? 3500 : 2100;
        for (int s = 1; s <= 16 && s <= p.S; s++)
            take(full / ncu * (p.S + 4) * clocks + (rest * s + ncu - 1) / ncu * ((p.S + s - 1) / s + 4) * clocks + (s > 1 ? parts(rest * s, kWMT, NT) : 0),
                 kWMT, NT, s, s == 1 ? items : full);
    }
    p.wt_bytes = d2c_align_up((size_t)p.S * p.nct * p.NT * p.KC * 2);
    p.part_bytes = p.nsplit == 1 ? 0
                 : d2c_align_up((p.MT == kWMT ? ((size_t)p.ntile * p.nct - p.nfull) * p.nsplit * kWMT * p.NT : (size_t)p.nsplit * C * M) * sizeof(float));
    return p;
}

template <int NT, int KC, bool COLS = false> int launch_rows(const ConvRowsArgs &a, hipStream_t st)
{
    D2cProfScope prof(D2C_PROF_FWD, st, "conv_rows_kernel");
    hipLaunchKernelGGL((conv_rows_kernel<NT, KC, COLS>), dim3((unsigned)(a.ntile * a.nsplit * a.nctile)), dim3(kThreads), 0, st, a);
    return d2c_check_launch("conv_rows_kernel");
}

template <int NT, bool COLS> int launch_wide(const ConvRowsArgs &a, hipStream_t st)
{
    D2cProfScope prof(D2C_PROF_FWD, st, "conv_wide_kernel");
    const int rest = a.ntile * a.nctile - a.nfull;
    hipLaunchKernelGGL((conv_wide_kernel<NT, COLS>), dim3((unsigned)(a.nfull + rest * a.nsplit)), dim3(kThreads), 0, st, a);
    if (rest > 0) hipLaunchKernelGGL(conv_wide_finish_kernel, dim3((unsigned)(rest * (NT / 4))), dim3(kWMT), 0, st, a, NT);
    return d2c_check_launch("conv_wide_kernel");
}

int run_rows(const RowsPlan &p, const RowMap &map, const void *src, unsigned rowb, unsigned zrow, const void *wt, const void *bias,
             void *out, float *part, int C, hipStream_t st, int cols_K = 0, int cols_rows = 0, int act = 0, float act_scale = 1.f)
{
    const bool wide = p.MT == kWMT, sums = p.nsplit > 1 && !wide;
    ConvRowsArgs a{map, (const unsigned char *)src, (const unsigned char *)wt, sums ? nullptr : (const bf16_t *)bias,
                   sums ? nullptr : (bf16_t *)out, part, rowb, zrow, C, p.nchunk, p.S, p.ntile, p.nct, p.nsplit, p.nfull,
                   cols_K, cols_rows, act, act_scale, map.P % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0};
    int rc;
    if (wide)
        rc = p.NT == 256 ? (cols_K > 0 ? launch_wide<256, true>(a, st) : launch_wide<256, false>(a, st))
                         : (cols_K > 0 ? launch_wide<128, true>(a, st) : launch_wide<128, false>(a, st));
    else if (cols_K > 0) rc = p.NT == 32 ? launch_rows<32, 64, true>(a, st) : (p.NT == 64 ? launch_rows<64, 64, true>(a, st) : launch_rows<128, 64, true>(a, st));
    else if (p.KC == 32) rc = p.NT == 32 ? launch_rows<32, 32>(a, st) : (p.NT == 64 ? launch_rows<64, 32>(a, st) : launch_rows<128, 32>(a, st));
    else rc = p.NT == 32 ? launch_rows<32, 64>(a, st) : (p.NT == 64 ? launch_rows<64, 64>(a, st) : launch_rows<128, 64>(a, st));
    if (rc || !sums) return rc;
    const int M = map.N * map.P;
    D2cProfScope prof(D2C_PROF_PACK, st);
    hipLaunchKernelGGL(conv_rows_finish_kernel, dim3((M + 255) / 256, C), dim3(256), 0, st, part, (const bf16_t *)bias, (bf16_t *)out,
                       p.nsplit, C, map.P, map.dP, M, act, act_scale);
    return d2c_check_launch("conv_rows_finish_kernel");
}

struct WeightPlan {
    int obt, OBP, notile, ncb, ntile, nsplit;
    size_t gp_bytes, part_bytes;
};
WeightPlan weight_plan(const d2c_conv3d_desc &q, int K, int ncu)
{
    WeightPlan p;
    const int M = q.N * q.Do * q.Ho * q.Wo;
    p.obt = q.Cout <= 32 ? 1 : (q.Cout <= 64 ? 2 : 4);
    p.notile = (q.Cout + 32 * p.obt - 1) / (32 * p.obt);
    p.OBP = p.notile * p.obt;
    p.ncb = (q.Cin + 127) / 128;
    p.ntile = (M + kCW - 1) / kCW;
    const long items = (long)K * p.ncb * p.notile, slots = 2L * ncu;
    long best = -1;
    p.nsplit = 1;
    for (int s = 1; s <= 16 && s <= p.ntile; s++) {
        const long rounds = (items * s + slots - 1) / slots;
        const long cost = rounds * ((p.ntile + s - 1) / s + 6) + (s > 1 ? (items * s * p.obt + slots - 1) / slots : 0);
        if (best < 0 || cost * 20 < best * 19) { best = cost; p.nsplit = s; }
    }
    p.gp_bytes = d2c_align_up((size_t)p.ntile * p.OBP * 4096);
    p.part_bytes = d2c_align_up((size_t)p.nsplit * K * p.ncb * q.Cout * 128 * sizeof(float));
    return p;
}

inline int padded_channels(int c) { return c <= 32 ? 32 : (c + 63) / 64 * 64; }
inline bool plain_shape_ok(const d2c_conv3d_desc &q)
{
    const size_t lim = (size_t)1 << 32, P = (size_t)q.Do * q.Ho * q.Wo;
    return q.dtype == D2C_BF16 && q.groups == 1 && q.Cin % 64 == 0 &&
           (size_t)q.N * q.Cin * q.D * q.H * q.W * 2 + 1024 < lim && (size_t)q.N * padded_channels(q.Cout) * P * 2 + 1024 < lim &&
           (size_t)q.N * P < (1u << 30) && (size_t)q.N * q.D * q.H * q.W < (1u << 30);
}
inline int weight_blocks(long nvec) { return (int)std::min<long>((nvec + 255) / 256, 4096); }
void prep_input(ConvPrepArgs &a, const d2c_conv3d_desc &q, const void *x, void *xcl, int zrow_words)
{
    const int vol = q.D * q.H * q.W;
    a.x = (const bf16_t *)x; a.xcl = (bf16_t *)xcl; a.C = q.Cin; a.vol = vol; a.N = q.N; a.zrow_words = zrow_words;
    a.nbx = (vol + 63) / 64; a.nby = q.Cin / 64; a.nblk_x = a.nbx * a.nby * q.N;
}
void prep_weights(ConvPrepArgs &a, const d2c_conv3d_desc &q, const RowsPlan &p, const void *w, void *wt, bool back)
{
    a.w = (const bf16_t *)w; a.wt = (uint4 *)wt; a.Cout = q.Cout; a.Cin = q.Cin; a.K = q.kd * q.kh * q.kw;
    a.NT = p.NT; a.KC = p.KC; a.nchunk = p.nchunk; a.nct = p.nct; a.back = back;
    a.nvec = (long)p.nct * p.NT * p.nchunk * (p.KC / 8) * a.K;
    a.nblk_w = weight_blocks(a.nvec);
}
void prep_zero(ConvPrepArgs &a, int j, void *p, size_t bytes)
{
    a.zero[j] = (uint32_t *)p; a.zwords[j] = p ? bytes / 4 : 0;
    a.nblk_z = (int)std::min<size_t>((std::max(a.zwords[0], a.zwords[1]) + 4095) / 4096, 2048);
}
int prep_launch(const ConvPrepArgs &a, hipStream_t st)
{
    const long n = (long)a.nblk_x + a.nblk_w + a.nblk_g + a.nblk_b + a.nblk_gcw + a.nblk_z;
    if (n == 0) return D2C_OK;
    D2cProfScope prof(D2C_PROF_PACK, st);
    hipLaunchKernelGGL(conv_prepare_kernel, dim3((unsigned)n), dim3(256), 0, st, a);
    return d2c_check_launch("conv_prepare_kernel");
}

}  // namespace

// ---- the same product over sampled columns [chunk][tap][rows][64] (d2c_brick.hip): the forward pass of the deformable
// operator, one weight group
size_t d2c_col_forward_ws(const d2c_conv3d_desc &q)
{
    const int ncu = d2c_num_cus();
    if (ncu <= 0) return 0;
    const RowsPlan p = rows_plan(q.Cout, q.Cin, q.kd * q.kh * q.kw, q.N * q.Do * q.Ho * q.Wo, ncu);
    return p.wt_bytes + p.part_bytes;
}
// What the sorted points, the sampling and the product need in front, as one launch: the input channels-last with a row of
// zeros of 256 bytes (x == nullptr: it is there), the weights, the counts of the sort cleared.
int d2c_col_forward_prepare(const d2c_conv3d_desc &q, const void *x, void *xcl, const void *w, void *ws, void *zero, size_t zero_bytes,
                            hipStream_t st)
{
    const int ncu = d2c_num_cus();
    if (ncu <= 0) return D2C_ERR_LAUNCH;
    ConvPrepArgs a{};
    if (x) prep_input(a, q, x, xcl, 64);
    prep_weights(a, q, rows_plan(q.Cout, q.Cin, q.kd * q.kh * q.kw, q.N * q.Do * q.Ho * q.Wo, ncu), w, ws, false);
    prep_zero(a, 0, zero, zero_bytes);
    return prep_launch(a, st);
}
int d2c_col_forward(const d2c_conv3d_desc &q, const void *col, int rows, const void *bias, void *out, void *ws, hipStream_t st)
{
    const int K = q.kd * q.kh * q.kw, ncu = d2c_num_cus();
    if (ncu <= 0) return D2C_ERR_LAUNCH;
    const RowsPlan p = rows_plan(q.Cout, q.Cin, K, q.N * q.Do * q.Ho * q.Wo, ncu);
    return run_rows(p, row_map(q, false), col, 0, 0, ws, bias, out, (float *)((char *)ws + p.wt_bytes), q.Cout, st, K, rows, q.epilogue,
                    q.epilogue_scale);
}

// ---- grad-column rows [chunk][tap][N*P][64] of the deformable operator's backward pass, one weight group
namespace {
struct GradColPlan {
    int Cp, S, ntile, npair, cgroups;
    size_t wt_bytes;
};
GradColPlan grad_col_plan(const d2c_conv3d_desc &q)
{
    GradColPlan p;
    const int M = q.N * q.Do * q.Ho * q.Wo;
    p.Cp = (q.Cout + 63) / 64 * 64;
    p.S = p.Cp / 64;
    p.ntile = (M + kWMT - 1) / kWMT;
    p.npair = q.Cin / 64 * q.kd * q.kh * q.kw;
    p.wt_bytes = d2c_align_up((size_t)p.npair * p.S * 8192);
    p.cgroups = 1;
    while (p.cgroups < 8 && p.wt_bytes / p.cgroups > (2u << 20)) p.cgroups *= 2;
    return p;
}
}  // namespace
// One weight group, as many output channels as the registers hold; grad_out and the rows of a pair within 32-bit offsets.  Of any
// size: training steps, us, with the kernel of the other shapes (tiled_bwd_col32_kernel) and with this one: 64 -> 64 on 49
// positions 84, 79; 512 -> 512 on 63 188, 142; 256 -> 256 on 420 160, 139; 1400 141, 126; 128 -> 128 on 12960 215, 204.
bool d2c_grad_col_supported(const d2c_conv3d_desc &q)
{
    const GradColPlan p = grad_col_plan(q);
    const size_t M = (size_t)q.N * q.Do * q.Ho * q.Wo;
    return q.dtype == D2C_BF16 && q.groups == 1 && q.Cin % 64 == 0 && q.Cout <= 512 && M * p.Cp * 2 + 1024 < 0xFFFF0000u &&
           (long)p.ntile * p.npair * p.S < (1L << 30) &&
           M * 128 < 0xFFFF0000u;
}
// its operand of grad_out, channels-last (the weights, in its order, take as much as those of tiled_bwd_col32_kernel or less)
size_t d2c_grad_col_gout_bytes(const d2c_conv3d_desc &q)
{
    return d2c_align_up((size_t)q.N * q.Do * q.Ho * q.Wo * grad_col_plan(q).Cp * 2 + 1024);
}
// What the backward pass over sorted points needs of grad_out and the weights, and what it adds into, as one launch (one
// weight group): the operands of d2c_grad_col (both or none), grad_out in fragment order for the grad_weight
// product (`goutp`, see pack_gout_kernel), the bias gradient, two ranges cleared; any of them NULL.  grad_out is read once
// for both orders.
int d2c_brick_bwd_prepare(const d2c_conv3d_desc &q, const void *gout, const void *w, void *col_wt, void *col_gout, void *goutp, void *gb,
                          void *zero0, size_t zero0_bytes, void *zero1, size_t zero1_bytes, hipStream_t st)
{
    const GradColPlan p = grad_col_plan(q);
    const int K = q.kd * q.kh * q.kw, P = q.Do * q.Ho * q.Wo, M = q.N * P;
    ConvPrepArgs a{};
    a.w = (const bf16_t *)w; a.Cout = q.Cout; a.Cin = q.Cin; a.K = K; a.N = q.N; a.dK = make_fastdiv(K);
    if (col_wt) {
        a.gcw = (uint4 *)col_wt; a.gcS = p.S; a.ngcw = (q.Cin * K + 255) / 256; a.nblk_gcw = a.ngcw * p.S * 8;
        a.gcl = (bf16_t *)col_gout;
    }
    a.gout = (const bf16_t *)gout; a.gp = (uint4 *)goutp; a.gp_wide = 1;
    a.Cp = p.Cp; a.OBP = p.Cp / 32; a.P = P; a.M = M; a.dP = make_fastdiv(P);
    a.ngt = (M + 127) / 128 * 2; a.ngc = p.Cp / 64; a.nblk_g = col_wt || goutp ? a.ngt * a.ngc : 0;
    a.gb = (bf16_t *)gb; a.nblk_b = gb ? q.Cout : 0;
    prep_zero(a, 0, zero0, zero0_bytes);
    prep_zero(a, 1, zero1, zero1_bytes);
    return prep_launch(a, st);
}
int d2c_grad_col(const d2c_conv3d_desc &q, void *gcol, const void *wt, const void *gcl, hipStream_t st)
{
    const GradColPlan p = grad_col_plan(q);
    const int M = q.N * q.Do * q.Ho * q.Wo, ncu = d2c_num_cus();
    if (ncu <= 0) return D2C_ERR_LAUNCH;
    GradColArgs a{(const unsigned char *)gcl, (const unsigned char *)wt, (bf16_t *)gcol, (unsigned)p.Cp * 2u, M, p.npair, p.ntile, p.cgroups};
    D2cProfScope prof(D2C_PROF_BWD_DATA, st, "grad_col_kernel");
    const dim3 grid((unsigned)std::max(8, ncu / 8 * 8));
    auto launch = [&](auto S) { hipLaunchKernelGGL((grad_col_kernel<decltype(S)::value>), grid, dim3(kThreads), 0, st, a); };
    switch (p.S) {
    case 1: launch(std::integral_constant<int, 1>{}); break;
    case 2: launch(std::integral_constant<int, 2>{}); break;
    case 3: launch(std::integral_constant<int, 3>{}); break;
    case 4: launch(std::integral_constant<int, 4>{}); break;
    case 5: launch(std::integral_constant<int, 5>{}); break;
    case 6: launch(std::integral_constant<int, 6>{}); break;
    case 7: launch(std::integral_constant<int, 7>{}); break;
    default: launch(std::integral_constant<int, 8>{}); break;
    }
    return d2c_check_launch("grad_col_kernel");
}

// ---- grad_weight over sampled columns, sums in `scratch`
namespace {
struct ColWeightPlan {
    int OT, otiles, nitem, ntile, nsplit;
    size_t bytes;                     // of the sums; 0: not on this kernel
};
ColWeightPlan col_weight_plan(const TiledShape &s, size_t scratch, int ncu)
{
    ColWeightPlan p{};
    p.OT = s.Cout > 128 ? 256 : 128;
    p.otiles = (s.Cout + p.OT - 1) / p.OT;
    p.nitem = (s.nchunk * s.K + 3) / 4 * p.otiles;
    p.ntile = (s.M + 63) / 64;
    if (kFinOut * ((size_t)s.K * 32 + 16) > 64 * 1024) return p;
    // pieces by what they cost in steps of a compute unit: rounds, each its steps and about eight more for its start and end, and
    // the sums, written and read once more
    double best = -1;
    for (int n = 1; n <= 32 && n <= p.ntile; n++) {
        const size_t bytes = (size_t)p.nitem * n * p.OT * 1024;
        if (bytes > scratch) break;
        const double cost = (double)(((long)p.nitem * n + ncu - 1) / ncu) * ((p.ntile + n - 1) / n + 8) + (double)p.nitem * n * p.OT / 2560;
        if (best < 0 || cost < best) { best = cost; p.nsplit = n; p.bytes = bytes; }
    }
    return p;
}
}  // namespace
bool d2c_col_weight_use(const TiledShape &s, size_t scratch) { return col_weight_plan(s, scratch, 1).bytes > 0; }
int d2c_col_weight(const TiledShape &s, const void *goutp, const void *col, long col_rows, void *gw, void *scratch, size_t scratch_bytes,
                   hipStream_t st)
{
    const int ncu = d2c_num_cus();
    if (ncu <= 0) return D2C_ERR_LAUNCH;
    const ColWeightPlan p = col_weight_plan(s, scratch_bytes, ncu);
    {
        ColWeightArgs a{(const unsigned char *)goutp, (const unsigned char *)col, (float *)scratch, col_rows * 128, s.nchunk * s.K, p.otiles,
                        p.nitem, (s.Cout + 63) / 64 * 2, p.ntile, p.nsplit};
        D2cProfScope prof(D2C_PROF_BWD_WEIGHT, st, "col_weight_kernel");
        const dim3 grid((unsigned)(p.nitem * p.nsplit));
        if (p.OT == 256) hipLaunchKernelGGL(col_weight_kernel<256>, grid, dim3(kThreads), 0, st, a);
        else hipLaunchKernelGGL(col_weight_kernel<128>, grid, dim3(kThreads), 0, st, a);
        if (int rc = d2c_check_launch("col_weight_kernel")) return rc;
    }
    D2cProfScope prof(D2C_PROF_PACK, st);
    ColWeightFinishArgs f{(const float *)scratch, (bf16_t *)gw, p.nsplit, p.nitem, p.otiles, p.OT, s.K, s.Cout, s.Cin,
                          (s.Cout + kFinOut - 1) / kFinOut, reinterpret_cast<uintptr_t>(gw) % 16 == 0};
    hipLaunchKernelGGL(col_weight_finish_kernel, dim3((unsigned)(s.Cin / 16 * f.nob)), dim3(256), kFinOut * ((size_t)s.K * 32 + 16), st, f);
    return d2c_check_launch("col_weight_finish_kernel");
}

bool d2c_plain_supported(const d2c_conv3d_desc &q) { return plain_shape_ok(q); }
size_t d2c_plain_input_bytes(const d2c_conv3d_desc &q) { return (size_t)q.N * q.Cin * q.D * q.H * q.W * 2 + 1024; }

size_t d2c_plain_forward_ws(const d2c_conv3d_desc &q)
{
    const int K = q.kd * q.kh * q.kw, ncu = d2c_num_cus();
    if (ncu <= 0) return 0;
    const RowsPlan p = rows_plan(q.Cout, q.Cin, K, q.N * q.Do * q.Ho * q.Wo, ncu);
    return p.wt_bytes + p.part_bytes;
}

int d2c_plain_forward(const d2c_conv3d_desc &q, const void *x, const void *w, const void *bias, void *out, void *xcl, void *ws,
                      hipStream_t st)
{
    const int K = q.kd * q.kh * q.kw, ncu = d2c_num_cus(), vol = q.D * q.H * q.W;
    if (ncu <= 0) return D2C_ERR_LAUNCH;
    const RowsPlan p = rows_plan(q.Cout, q.Cin, K, q.N * q.Do * q.Ho * q.Wo, ncu);
    char *base = (char *)ws;
    {
        ConvPrepArgs a{};
        prep_input(a, q, x, xcl, 128);
        prep_weights(a, q, p, w, base, false);
        if (int rc = prep_launch(a, st)) return rc;
    }
    return run_rows(p, row_map(q, false), xcl, (unsigned)q.Cin * 2u, (unsigned)((size_t)q.N * q.Cin * vol * 2), base, bias, out,
                    (float *)(base + p.wt_bytes), q.Cout, st);
}

namespace {
struct PlainBwdWs {
    size_t gcl, gp, wt, part, total;
};
PlainBwdWs plain_bwd_ws(const d2c_conv3d_desc &q, const RowsPlan &r, const WeightPlan &w)
{
    PlainBwdWs l;
    l.gcl = 0;
    l.gp = d2c_align_up((size_t)q.N * q.Do * q.Ho * q.Wo * padded_channels(q.Cout) * 2 + 1024);
    l.wt = l.gp + w.gp_bytes;
    l.part = l.wt + r.wt_bytes;
    // (grad_input's partial sums are done with before grad_weight's are written)
    l.total = l.part + std::max(r.part_bytes, w.part_bytes);
    return l;
}
}  // namespace

size_t d2c_plain_backward_ws(const d2c_conv3d_desc &q)
{
    const int K = q.kd * q.kh * q.kw, ncu = d2c_num_cus();
    if (ncu <= 0) return 0;
    return plain_bwd_ws(q, rows_plan(q.Cin, padded_channels(q.Cout), K, q.N * q.D * q.H * q.W, ncu), weight_plan(q, K, ncu)).total;
}

int d2c_plain_backward(const d2c_conv3d_desc &q, const void *gout, const void *xcl, const void *w, void *gx, void *gw, void *gb,
                       void *ws, hipStream_t st)
{
    const int K = q.kd * q.kh * q.kw, ncu = d2c_num_cus(), vol = q.D * q.H * q.W, P = q.Do * q.Ho * q.Wo, M = q.N * P;
    if (ncu <= 0) return D2C_ERR_LAUNCH;
    if (!gx && !gw && !gb) return D2C_OK;
    const int Cp = padded_channels(q.Cout);
    const RowsPlan r = rows_plan(q.Cin, Cp, K, q.N * vol, ncu);
    const WeightPlan p = weight_plan(q, K, ncu);
    const PlainBwdWs l = plain_bwd_ws(q, r, p);
    char *base = (char *)ws;
    {
        ConvPrepArgs a{};
        a.N = q.N; a.Cout = q.Cout;
        if (gx) prep_weights(a, q, r, w, base + l.wt, true);
        a.gout = (const bf16_t *)gout;
        a.gcl = gx ? (bf16_t *)(base + l.gcl) : nullptr;
        a.gp = gw ? (uint4 *)(base + l.gp) : nullptr;
        a.Cp = Cp; a.OBP = p.OBP; a.P = P; a.M = M; a.dP = make_fastdiv(P);
        a.ngt = (M + 63) / 64;
        a.ngc = std::max((Cp + 63) / 64, (p.OBP + 1) / 2);
        a.nblk_g = (gx || gw) ? a.ngt * a.ngc : 0;
        a.gb = (bf16_t *)gb;
        a.nblk_b = gb ? q.Cout : 0;
        if (int rc = prep_launch(a, st)) return rc;
    }
    if (gx) {
        if (int rc = run_rows(r, row_map(q, true), base + l.gcl, (unsigned)Cp * 2u, (unsigned)((size_t)M * Cp * 2), base + l.wt, nullptr,
                              gx, (float *)(base + l.part), q.Cin, st))
            return rc;
    }
    if (gw) {
        ConvWeightArgs a{row_map(q, false), (const unsigned char *)xcl, (const uint4 *)(base + l.gp), (float *)(base + l.part),
                         (unsigned)q.Cin * 2u, (unsigned)((size_t)q.N * q.Cin * vol * 2), q.Cout, p.OBP, p.ncb, K, p.notile,
                         p.nsplit, p.ntile, q.Cin % 128 != 0};
        const dim3 grid((unsigned)((long)K * p.ncb * p.notile * p.nsplit));
        {
            D2cProfScope prof(D2C_PROF_BWD_WEIGHT, st, "conv_weight_kernel");
            if (p.obt == 1) hipLaunchKernelGGL(conv_weight_kernel<1>, grid, dim3(kThreads), 0, st, a);
            else if (p.obt == 2) hipLaunchKernelGGL(conv_weight_kernel<2>, grid, dim3(kThreads), 0, st, a);
            else hipLaunchKernelGGL(conv_weight_kernel<4>, grid, dim3(kThreads), 0, st, a);
            if (int rc = d2c_check_launch("conv_weight_kernel")) return rc;
        }
        D2cProfScope prof(D2C_PROF_PACK, st);
        hipLaunchKernelGGL(conv_weight_finish_kernel, dim3((unsigned)(q.Cout * p.ncb)), dim3(256), 0, st, (const float *)a.part,
                           (bf16_t *)gw, p.nsplit, K, p.ncb, q.Cout, q.Cin);
        return d2c_check_launch("conv_weight_finish_kernel");
    }
    return D2C_OK;
}
