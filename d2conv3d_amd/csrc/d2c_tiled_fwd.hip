// Forward pass as an implicit GEMM on the matrix cores.
//
//   out[b, o, p] = bias[o] + sum_{c, k} W[o, c, k] * alpha[b,g,k,p] * trilinear(x[b, c], pos(b,g,k,p))
//
// GEMM view: rows = output channels, columns = output positions (N*P of
// them), reduction = (channel chunk, tap).  The sampled operand is produced on
// the fly: for one (chunk, tap) step every thread gathers the 8 corners of its
// position as 16-byte channel vectors from the channels-last copy of the
// input, interpolates in fp32 with the modulation folded into the corner
// weights, and drops the result into an LDS tile in MFMA operand order.  The
// im2col column buffer of the reference (dconv3d_gpu.cu:297) never exists.
//
// Here: the DMA-gather kernel, whose corner rows go to LDS without passing through registers, for weight groups wide enough or
// problems large enough to fill its output tile; and the choice between it and the kernel of the other problems
// (d2c_tiled_wave.hip).
#include "d2c_mma.hpp"
#include "d2c_tiled.hpp"

// the kernel of the small problems (d2c_tiled_wave.hip)
size_t d2c_wave_count_bytes(const TiledShape &s, int nt);
size_t d2c_wave_split_bytes(const TiledShape &s, int nt);
template <typename T>
int d2c_wave_launch(const TiledShape &s, int nt, bool skip_zero, const void *xcl, const void *off, const void *mask, const void *wp,
                    const void *bias, void *out, float *split, void *col, hipStream_t st);

namespace {

constexpr int kNV = 8;         // 16-byte vectors per sampled row (one chunk)
constexpr int kRS = kNV * 16 + 16;  // LDS row stride in bytes (padded: conflict-free 16-byte reads)
constexpr int kThreads = 512;

struct FwdArgs {
    TiledShape s;
    const void *xcl;   // [N][vol][Cin]
    const void *off, *mask;
    const void *wp;    // packed weights, see pack_weight_fwd
    const void *bias;
    void *out;
    float *outacc;     // fp32 tiles of the work items whose steps are shared out
    unsigned zrow;     // byte offset (from xcl) of a 128-byte row of zeros: what dead corners read
    // Schedule of the DMA-gather kernel, whose workgroups are persistent (one per compute unit).  A work item is
    // one (position tile, output tile, weight group) with all its steps.  Items [0, sk_full) are dealt whole,
    // round-robin.  The remaining items, fewer than one round, have their steps cut into sk_cut equal ranges;
    // the (range, item) pieces are dealt round-robin in range-major order, so that the workgroups running at
    // one time are at about the same steps and share their weight fragments in L2.  The pieces add into
    // `outacc`, here laid out [item - sk_full][output channel of the tile][position of the tile].
    int sk_items, sk_full, sk_ntile, sk_otiles, sk_cut;
    // The sampled, modulated columns kept for the backward pass (or NULL): what the matrix step multiplies with the
    // weights, [chunk][tap][col_rows][BKC] in the element type, col_rows = position tiles x 64 (zeros past the last
    // position) -- the layout tiled_bwd_weight_col_kernel reads.  Written by the DMA-gather kernel.
    void *col;
    long col_rows;
};

// Tiles that are neighbours in space go to the same XCD (workgroups are dealt
// round-robin over the 8 XCDs), so that its L2 sees a compact part of the input.
D2C_DEV int xcd_swizzle(int bid, int n)
{
    const int x = bid & 7, idx = bid >> 3;
    const int q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + idx;
}

// ---------------------------------------------------------------------------
// The same forward pass with the corner rows moved global -> LDS by DMA loads
// (global_load_lds_dwordx4: no staging registers; the rows of step s+2 are
// requested during the matrix-core phase of iteration s, a few requests
// between each pair of MFMAs, and are in flight over the interpolation of
// step s+1 and the barrier).
// One workgroup = 512 + 64 threads = 64 positions x NT output channels.  One DMA
// instruction of a wavefront fetches the 8 corner rows (8 x 128 bytes) of one
// position: lane = (corner, 16-byte vector); corners that are out of range or
// cut off by the early-out read a row of zeros instead.
//
// Workgroups are persistent: each walks a list of segments (a work item and a
// range of its steps, see FwdArgs) as ONE sequence of steps, so that the
// pipeline stays full from one segment into the next; only the matrix-core
// wavefronts notice a segment's end (they store or add their accumulators).
constexpr int kDMT = 64;                   // positions per workgroup

// Workgroup barrier that waits for this wavefront's LDS operations only: its global loads and DMA transfers
// stay in flight across it (a __syncthreads() would wait for them as well).
D2C_DEV void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

constexpr int kMaxSeg = 128;               // segments per workgroup (the launcher sizes the grid for this)

// A position in the step sequence of a workgroup.  The segments are listed in LDS once, at the start; all
// fields are uniform over the workgroup and live in scalar registers.
//
// Step order within a work item: offset group (outer), tap, chunk of that offset group (inner), so that the chunks
// that share the sampling points of a (group, tap) follow each other and the coordinate wavefront computes a table
// once for all of them.  The walker counts chunk, tap and group along (no division per step).
struct SegWalk {
    int seg;                      // index of the current segment
    int item;                     // its work item, -1 past the end of the sequence
    int st, st_hi;                // current step, end of the current segment
    int tile, otile, wg;          // the item's position tile, output tile, weight group
    int j, k, g;                  // the step's chunk within the weight group, tap, offset group
    int jj;                       // chunk within the offset group
    bool fresh;                   // first step of its (group, tap) in this segment: sampling points not seen yet
};
D2C_DEV void seg_load(SegWalk &w, const int4 *s_seg, int nseg, const TiledShape &s)
{
    if (w.seg < nseg) {
        const int4 u = s_seg[2 * w.seg], v = s_seg[2 * w.seg + 1];
        w.item = __builtin_amdgcn_readfirstlane(u.x);
        w.st = __builtin_amdgcn_readfirstlane(u.y);
        w.st_hi = __builtin_amdgcn_readfirstlane(u.z);
        w.tile = __builtin_amdgcn_readfirstlane(v.x);
        w.otile = __builtin_amdgcn_readfirstlane(v.y);
        w.wg = __builtin_amdgcn_readfirstlane(v.z);
        const int t = w.st / s.cpc, gi = t / s.K;
        w.jj = w.st - t * s.cpc;
        w.k = t - gi * s.K;
        w.j = gi * s.cpc + w.jj;
        w.g = (w.wg * s.cg + w.j * s.bkc) / s.cpg;
    } else {
        w.item = -1; w.st = 0; w.st_hi = 0x7fffffff;
        w.j = 0; w.k = 0; w.g = 0; w.jj = 0;
    }
    w.fresh = true;
}
// one step on; true when that entered a new segment
D2C_DEV bool seg_advance(SegWalk &w, const int4 *s_seg, int nseg, const TiledShape &s)
{
    if (++w.st < w.st_hi) {
        if (++w.jj < s.cpc) {
            w.j++; w.fresh = false;
        } else {
            w.jj = 0; w.fresh = true;
            if (++w.k < s.K) w.j -= s.cpc - 1;
            else { w.k = 0; w.j++; w.g++; }
        }
        return false;
    }
    w.seg++;
    seg_load(w, s_seg, nseg, s);
    return true;
}

// (The LDS regions are passed as restrict-qualified pointers: that gives their accesses alias scopes, without
// which the compiler makes every LDS store wait for all DMA transfers in flight, whatever region they fill.)
// NC: corner rows fetched and interpolated per sampling point: 8, or 4 / 2 when offsets along one / two axes are fixed
// (TiledShape::axes; the corners on the far side of a fixed axis have weight zero and no slot at all).
template <typename T, bool AUX16, int WAVES_O, int WAVES_P, bool SIZED, int NC, bool COLS>
D2C_DEV void fwd_dma_body(const FwdArgs &a, unsigned char *__restrict__ s_raw, unsigned char *__restrict__ s_tile,
                          float *__restrict__ s_w, int2 *__restrict__ s_if,
                          int *__restrict__ s_meta, int4 *__restrict__ s_seg)
{
    constexpr int MT = kDMT;
    constexpr int VEC = Elem<T>::VEC;
    constexpr int BKC = kNV * VEC;
    constexpr int WPOS = MT / WAVES_P;    // positions per MMA wave
    constexpr int PB = WPOS / 32;         // 32-position blocks per MMA wave
    constexpr int OB = 2;                 // 32-channel blocks per MMA wave
    constexpr int NT = 64 * WAVES_O;      // output channels per workgroup
    constexpr int NKG = kNV / 2;          // k-groups per step
    static_assert(MT * kNV == kThreads, "one (position, vector) item per thread");
    static_assert(WAVES_O * WAVES_P <= kThreads / 64 && PB >= 1, "MMA wave layout");
    constexpr int RAWPOS = NC * kNV * 16;   // raw bytes per position
    constexpr int PPI = 8 / NC;             // positions per DMA instruction

    const TiledShape &s = a.s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int S = s.nchunk * s.K;
    const int OBT = s.ogp / 32;
    const int dzc = s.H * s.W * s.Cin, dyc = s.W * s.Cin;

    // --- the step sequence of this workgroup: its whole items, then its pieces of the last round's items
    const int nwg = (int)gridDim.x;
    const int bid = xcd_swizzle(blockIdx.x, nwg);
    const int ntail = a.sk_items - a.sk_full, npiece = ntail * a.sk_cut;
    const int nwhole_mine = bid < a.sk_full ? (a.sk_full - bid + nwg - 1) / nwg : 0;
    const int npiece_mine = bid < npiece ? (npiece - bid + nwg - 1) / nwg : 0;
    const int nseg = nwhole_mine + npiece_mine;        // <= kMaxSeg
    if (nseg == 0) return;
    if (tid < nseg) {
        int item, lo, hi;
        if (tid < nwhole_mine) {
            item = bid + tid * nwg; lo = 0; hi = S;
        } else {
            const int piece = bid + (tid - nwhole_mine) * nwg, range = piece / ntail;
            item = a.sk_full + (piece - range * ntail);
            lo = (int)((long)S * range / a.sk_cut);
            hi = (int)((long)S * (range + 1) / a.sk_cut);
        }
        s_seg[2 * tid] = make_int4(item, lo, hi, 0);
        s_seg[2 * tid + 1] = make_int4(item % a.sk_ntile, (item / a.sk_ntile) % a.sk_otiles,
                                       item / (a.sk_ntile * a.sk_otiles), 0);
    }
    __syncthreads();
    int total = 0;
    for (int q = 0; q < nseg; q++) total += __builtin_amdgcn_readfirstlane(s_seg[2 * q].z - s_seg[2 * q].y);
    SegWalk w0;
    w0.seg = 0;
    seg_load(w0, s_seg, nseg, s);

    // --- coordinates: a ninth wavefront (one position per lane) that does nothing else, so that this
    // arithmetic runs beside the work of the other eight instead of in front of their barrier
    const bool cwave = wave == 8;        // coordinates
    const bool worker = wave < 8;
    const int ctid = tid - kThreads;
    // The lane's position within a work item.  Offsets are requested (issue) one iteration before they are
    // turned into a table row (finish).
    // (size-map source: the part of the offsets that the taps of a position share, size - 1 per axis, is formed
    // here once per work item; a step then costs three multiplications and no load)
    typedef typename std::conditional<AUX16, bf16_t, float>::type AT;
    const CoordConst cc = coord_const(s);
    const int ncomp = s.nd == 3 ? 3 : 1;                               // offset components per tap
    const long cstride = s.nd == 3 ? (long)s.P * (long)sizeof(AT) : 0;
    const long off_tap = (long)ncomp * s.P * (long)sizeof(AT);         // bytes per (sample, group, tap) of the offsets
    const long mask_tap = (long)s.P * (long)sizeof(AT);                // ... of the mask
    // Lane l of the coordinate wavefront keeps the constants of tap l (taps 64 and up are computed when met):
    // where the tap sits in the kernel, as float, and for the size-map source its kernel-grid coordinates.
    float tap_z = 0.f, tap_y = 0.f, tap_x = 0.f, tap_bz = 0.f, tap_by = 0.f, tap_bx = 0.f;
    auto tap_consts = [&](int k, float &tz, float &ty, float &tx, float &bz, float &by, float &bx) {
        const int kx = k % s.geo.kw, ky = (k / s.geo.kw) % s.geo.kh, kz = k / (s.geo.kw * s.geo.kh);
        tz = (float)(kz * s.geo.dd); ty = (float)(ky * s.geo.dh); tx = (float)(kx * s.geo.dw);
        if constexpr (SIZED) {
            bz = rnd<AT>(s.ss.base[0][kz]); by = rnd<AT>(s.ss.base[1][ky]); bx = rnd<AT>(s.ss.base[2][kx]);
        }
    };
    if (cwave && ctid < s.K) tap_consts(ctid, tap_z, tap_y, tap_x, tap_bz, tap_by, tap_bx);
    struct PosC {
        float fz, fy, fx;          // o * stride - pad per axis, as float
        int vox0;                  // voxel index of the sample's origin
        unsigned aoff, moff;       // byte offsets of (sample - first sample of the tile, position) in offsets / mask
        bool valid;
        float s0, s1, s2;
    };
    const char *off_item = nullptr, *mask_item = nullptr;      // uniform: the tile's first sample
    auto pos_of = [&](const SegWalk &w) {
        PosC c{0.f, 0.f, 0.f, 0, 0u, 0u, false, 0.f, 0.f, 0.f};
        const int m0 = w.item >= 0 ? w.tile * MT : 0;
        const int b_lo = fdiv(m0, s.dP);
        off_item = reinterpret_cast<const char *>(a.off) + (long)b_lo * s.obs * (long)sizeof(AT);
        mask_item = reinterpret_cast<const char *>(a.mask) + (long)b_lo * s.mbs * (long)sizeof(AT);
        const int m = m0 + ctid;
        c.valid = w.item >= 0 && m < s.M;
        if (c.valid) {
            const int b = fdiv(m, s.dP), p = m - b * s.P;
            const int oz = fdiv(p, s.dHW), rem = p - oz * (s.Wo * s.Ho);
            const int oy = fdiv(rem, s.dW), ox = rem - oy * s.Wo;
            c.fz = (float)(oz * s.geo.sd - s.geo.pd);
            c.fy = (float)(oy * s.geo.sh - s.geo.ph);
            c.fx = (float)(ox * s.geo.sw - s.geo.pw);
            c.vox0 = b * s.vol;
            // (a lane without a position keeps offset 0: its loads read the tile's first position)
            c.aoff = (unsigned)(b - b_lo) * ((unsigned)s.obs * (unsigned)sizeof(AT)) + (unsigned)p * (unsigned)sizeof(AT);
            c.moff = (unsigned)(b - b_lo) * ((unsigned)s.mbs * (unsigned)sizeof(AT)) + (unsigned)p * (unsigned)sizeof(AT);
            if (SIZED && cwave) {
                float t[3];
                tap_offsets_issue<AUX16, true>(s, a.off, b, 0, 0, p, t);
                size_minus_one<AUX16>(s, t);
                c.s0 = t[0]; c.s1 = t[1]; c.s2 = t[2];
            }
        }
        return c;
    };
    float craw[4] = {0.f, 0.f, 0.f, 1.f};
    auto coords_issue = [&](const SegWalk &w, const PosC &c) {
        if (cwave && w.fresh) {
            const int gk = w.g * s.K + w.k;
            if constexpr (!SIZED) coord_offsets_issue<AUX16>(off_item + gk * off_tap, cstride, c.aoff, craw);
            if (a.mask) craw[3] = ld_aux_at<AUX16>(mask_item + gk * mask_tap, c.moff);
        }
    };
    auto coords_finish = [&](const SegWalk &w, const PosC &c, int buf) {
        if (cwave && !w.fresh) {
            // same sampling points as the step before (another chunk of the offset group): its table, copied
            const int pbuf = (buf + 2) % 3;
#pragma unroll
            for (int q = 0; q < 8; q++) s_w[(buf * 8 + q) * MT + ctid] = s_w[(pbuf * 8 + q) * MT + ctid];
            s_if[buf * MT + ctid] = s_if[pbuf * MT + ctid];
        } else if (cwave) {
            float tz, ty, tx, bz = 0.f, by = 0.f, bx = 0.f;
            if (w.k < 64) {
                tz = lane_value(tap_z, w.k);
                ty = lane_value(tap_y, w.k);
                tx = lane_value(tap_x, w.k);
                if constexpr (SIZED) {
                    bz = lane_value(tap_bz, w.k);
                    by = lane_value(tap_by, w.k);
                    bx = lane_value(tap_bx, w.k);
                }
            } else {
                tap_consts(w.k, tz, ty, tx, bz, by, bx);
            }
            if constexpr (SIZED) {
                craw[0] = rnd<AT>(bz * c.s0); craw[1] = rnd<AT>(by * c.s1); craw[2] = rnd<AT>(bx * c.s2);
            }
            coord_offsets_select(cc, craw);
            if (s.mact && a.mask) craw[3] = mask_act<AT>(s.mact, craw[3]);
            const CornerRow r = corner_row(cc, (c.fz + tz) + craw[0], (c.fy + ty) + craw[1], (c.fx + tx) + craw[2],
                                           craw[3], c.vox0, c.valid);
#pragma unroll
            for (int q = 0; q < 8; q++) s_w[(buf * 8 + q) * MT + ctid] = r.w[q];
            s_if[buf * MT + ctid] = make_int2(r.idx, (int)r.live);
        }
        // what the workers need to know of the step: its first input channel and where its weight fragments start
        // (they walk no step sequence of their own)
        if (cwave && ctid == 0) {
            s_meta[buf * 4] = w.wg * s.cg + w.j * BKC;
            s_meta[buf * 4 + 1] = (w.wg * S + w.j * s.K + w.k) * OBT + w.otile * (NT / 32);
            // COLS: the row of the column buffer where this step's tile goes (the first output tile writes it)
            if constexpr (COLS)
                s_meta[buf * 4 + 2] = w.otile == 0 ? (int)((((long)(w.wg * s.nchunk + w.j)) * s.K + w.k) * a.col_rows) + w.tile * MT
                                                   : -1;
        }
    };
    // a table that fetches rows of zeros: steps past the end of a sequence shorter than the pipeline
    auto coords_none = [&](int buf) {
        if (cwave) {
#pragma unroll
            for (int q = 0; q < 8; q++) s_w[(buf * 8 + q) * MT + ctid] = 0.f;
            s_if[buf * MT + ctid] = make_int2(0, 0);
            if (ctid == 0) { s_meta[buf * 4] = 0; s_meta[buf * 4 + 1] = 0; s_meta[buf * 4 + 2] = -1; }
        }
    };

    // --- corner rows of a step -> s_raw[rbuf]: worker wavefront w requests positions 8w .. 8w+7, one
    // instruction per position, lane = (corner, 16-byte vector)
    // (with fewer than 8 corners an instruction covers 8 / NC positions: lane = (position, corner slot, vector); slot j
    // is the corner whose bits are those of j spread over the free axes)
    const int dslot = (lane >> 3) % NC, dsub = (lane >> 3) / NC, dvec = lane & 7;
    const int dcorner = NC == 8 ? dslot : corner_of_slot(dslot, s.axes);
    const int dcoff = ((dcorner >> 2) & 1) * dzc + ((dcorner >> 1) & 1) * dyc + (dcorner & 1) * s.Cin;
    // one request: the rows of position(s) wave * 8 + i * PPI (+ dsub); `vidx` / `vflag` hold the table entries of the
    // wavefront's 8 positions (lane i: position i)
    auto dma_request = [&](int i, int vidx, int vflag, int c0, int rbuf) {
        const char *base = reinterpret_cast<const char *>(a.xcl);
        const int pos0 = wave * (MT / 8) + i * PPI;
        int idx;
        unsigned live;
        if constexpr (PPI == 1) {
            idx = __builtin_amdgcn_readlane(vidx, i);
            live = (unsigned)__builtin_amdgcn_readlane(vflag, i);
        } else {
            idx = __builtin_amdgcn_ds_bpermute((i * PPI + dsub) << 2, vidx);
            live = (unsigned)__builtin_amdgcn_ds_bpermute((i * PPI + dsub) << 2, vflag);
        }
        const unsigned o = ((live >> dcorner) & 1u)
                               ? (unsigned)(idx + c0 + dcoff + dvec * VEC) * (unsigned)sizeof(T)
                               : a.zrow + (unsigned)dvec * 16u;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(base + o),
                                         (__attribute__((address_space(3))) void *)(s_raw + (rbuf * MT + pos0) * RAWPOS),
                                         16, 0, 0);
    };
    // (past the end of the sequence the tables are those of three steps before, or the ones of coords_none: the
    // same number of transfers in every iteration, which lets the compiler count the loads in flight instead of
    // waiting for all)
    auto dma_issue = [&](int rbuf, int tbuf) {
        if (!worker) return;
        const int c0 = __builtin_amdgcn_readfirstlane(s_meta[tbuf * 4]);
        // table entries of this wavefront's 8 positions: one LDS read (lane i holds position i), then
        // lane-indexed moves to scalar registers
        const int2 vif = s_if[tbuf * MT + wave * (MT / 8) + (lane & 7)];
#pragma unroll
        for (int i = 0; i < MT / 8 / PPI; i++) dma_request(i, vif.x, vif.y, c0, rbuf);
    };
    // --- interpolation: thread = (position, 16-byte vector)
    const int ipos = tid >> 3, ivec = tid & 7;
    int wslot[NC];      // row of the weight table that belongs to corner slot c
#pragma unroll
    for (int c = 0; c < NC; c++) wslot[c] = (NC == 8 ? c : corner_of_slot(c, s.axes)) * MT;
    // (the rows are read behind the compiler's back, see lds_row_read: the transfers requested during the matrix
    // step, for the step after the one interpolated here, stay in flight; `between(c)` runs after corner slot c)
    auto interp_rows = [&](int rbuf, int tbuf, auto between) {
        const unsigned rp = lds_address(s_raw + (rbuf * MT + ipos) * RAWPOS + ivec * 16);
        VecAcc<T> va;
        va.zero();
        if constexpr (NC == 2) {
            u32x4_t r0 = lds_row_read<0>(rp), r1 = lds_row_read<kNV * 16>(rp);
            const float w0 = s_w[tbuf * 8 * MT + wslot[0] + ipos], w1 = s_w[tbuf * 8 * MT + wslot[1] + ipos];
            lds_rows_wait(r0, r1);
            va.fma(w0, __builtin_bit_cast(uint4, r0));
            between(0);
            va.fma(w1, __builtin_bit_cast(uint4, r1));
            between(1);
        } else {
#pragma unroll
            for (int h = 0; h < NC / 4; h++) {
                constexpr int R = kNV * 16;
                u32x4_t r0 = h ? lds_row_read<4 * R>(rp) : lds_row_read<0>(rp);
                u32x4_t r1 = h ? lds_row_read<5 * R>(rp) : lds_row_read<R>(rp);
                u32x4_t r2 = h ? lds_row_read<6 * R>(rp) : lds_row_read<2 * R>(rp);
                u32x4_t r3 = h ? lds_row_read<7 * R>(rp) : lds_row_read<3 * R>(rp);
                float w[4];
#pragma unroll
                for (int c = 0; c < 4; c++) w[c] = s_w[tbuf * 8 * MT + wslot[h * 4 + c] + ipos];
                lds_rows_wait(r0, r1, r2, r3);
                va.fma(w[0], __builtin_bit_cast(uint4, r0));
                between(h * 4);
                va.fma(w[1], __builtin_bit_cast(uint4, r1));
                between(h * 4 + 1);
                va.fma(w[2], __builtin_bit_cast(uint4, r2));
                between(h * 4 + 2);
                va.fma(w[3], __builtin_bit_cast(uint4, r3));
                between(h * 4 + 3);
            }
        }
        return va;
    };
    // COLS: the tile of a step also goes to the column buffer, one 16-byte streaming store per thread.  It is kept
    // for one step and issued in the matrix step of the next iteration, behind that step's last row request
    // (col_flush): it then has most of a step to complete before the wait at the top of the iteration comes round
    // again (that wait counts stores as well as loads), and meets the vector-memory path when the row requests are
    // out (N=2, C=512, 8x30x54: kernel +10 % with the store right behind the wait, +6 % in front of the
    // interpolation, +4 % here; as a plain instead of a streaming store +26 %).
    typedef unsigned u32x4_c __attribute__((ext_vector_type(4)));
    u32x4_c col_v = {0u, 0u, 0u, 0u};
    int col_row = -1;                                  // (wavefront-uniform)
    // (float: the interpolated values themselves, not the two-term operand form the matrix step reads)
    auto col_keep = [&](const VecAcc<T> &va, const uint4 &v, int tbuf) {
        if constexpr (COLS) {
            if constexpr (sizeof(T) == 4)
                col_v = u32x4_c{__float_as_uint(va.a[0]), __float_as_uint(va.a[1]), __float_as_uint(va.a[2]),
                                __float_as_uint(va.a[3])};
            else col_v = u32x4_c{v.x, v.y, v.z, v.w};
            col_row = __builtin_amdgcn_readfirstlane(s_meta[tbuf * 4 + 2]);
        }
    };
    auto col_flush = [&]() {
        if constexpr (COLS) {
            // (a thread's 16 bytes of its tile: position tid / 8, vector tid % 8 of a 128-byte row)
            if (col_row >= 0)
                __builtin_nontemporal_store(col_v, reinterpret_cast<u32x4_c *>(reinterpret_cast<char *>(a.col)
                                                       + (long)col_row * (BKC * (long)sizeof(T)) + tid * 16));
        }
    };
    auto interp_store = [&](int rbuf, int tbuf, int dbuf) {
        if (!worker) return;
        VecAcc<T> va = interp_rows(rbuf, tbuf, [](int) {});
        const uint4 v = va.pack();
        *reinterpret_cast<uint4 *>(s_tile + (dbuf * MT + ipos) * kRS + ivec * 16) = v;
        col_keep(va, v, tbuf);
    };

    // --- MMA role
    const bool mma_wave = wave < WAVES_O * WAVES_P;
    const int wave_o = wave % WAVES_O, wave_p = wave / WAVES_O;
    f32x16 acc[OB][PB];
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int pb = 0; pb < PB; pb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[ob][pb][r] = 0.f;
    const uint4 *wp4 = reinterpret_cast<const uint4 *>(a.wp);
    uint4 af[NKG][OB];
    // (wstep: the table's entry for the step; past the end of the sequence a stale one, the fragments are not used)
    auto wfrag = [&](int wstep, int kg, int ob) {
        const long wbase = ((long)wstep + wave_o * OB) * NKG * 64 + lane;
        return wp4[wbase + ((long)ob * NKG + kg) * 64];
    };
    // The vector-memory path of a CU takes one request of a wavefront at a time (1 KiB = 16 clocks) and a wavefront
    // stalls at issue while the path is busy: requests issued back to back serialise with everything else the
    // wavefront does.  So they are spread over the iteration: the DMA requests of step it+2 between the MFMAs of
    // step it (in its first half, so that they have landed when the interpolation starts), the weight-fragment
    // loads of step it+1 between the corners of the interpolation.
    static_assert(WAVES_O * WAVES_P == 8 && NKG * OB == 8, "all workers are matrix wavefronts; a fragment per corner");
    auto mma_dma_step = [&](int dbuf, int rbuf, int tbuf) {
        const unsigned char *tb = s_tile + (dbuf * MT + wave_p * WPOS + (lane & 31)) * kRS + (lane >> 5) * 16;
        const int c0 = __builtin_amdgcn_readfirstlane(s_meta[tbuf * 4]);
        // table entries of this wavefront's 8 positions: one LDS read (lane i holds position i), then
        // lane-indexed moves to scalar registers
        const int2 vif = s_if[tbuf * MT + wave * (MT / 8) + (lane & 7)];
        constexpr int DPK = 4;                                // requests per k-group
#pragma unroll
        for (int kg = 0; kg < NKG; kg++) {
            uint4 bf[PB];
#pragma unroll
            for (int pb = 0; pb < PB; pb++)
                bf[pb] = *reinterpret_cast<const uint4 *>(tb + pb * 32 * kRS + kg * 32);
#pragma unroll
            for (int ob = 0; ob < OB; ob++)
#pragma unroll
                for (int pb = 0; pb < PB; pb++) mma_kgroup<T, kF32SplitFwd>(acc[ob][pb], af[kg][ob], bf[pb]);
#pragma unroll
            for (int q = 0; q < DPK; q++) {
                const int i = kg * DPK + q;
                if (i >= MT / 8 / PPI) break;
                dma_request(i, vif.x, vif.y, c0, rbuf);
            }
            // (the kept columns of this step's tile: behind the last row requests, while matrix instructions remain)
            if (kg == (MT / 8 / PPI + DPK - 1) / DPK) col_flush();
        }
    };
    // interpolation of one step; the weight fragments of that step are fetched on the way
    auto interp_wload_store = [&](int rbuf, int tbuf, int dbuf) {
        const int wstep = __builtin_amdgcn_readfirstlane(s_meta[tbuf * 4 + 1]);
        VecAcc<T> va = interp_rows(rbuf, tbuf, [&](int c) {
#pragma unroll
            for (int f = c * (8 / NC); f < (c + 1) * (8 / NC); f++) af[f / OB][f % OB] = wfrag(wstep, f / OB, f % OB);
        });
        const uint4 v = va.pack();
        *reinterpret_cast<uint4 *>(s_tile + (dbuf * MT + ipos) * kRS + ivec * 16) = v;
        col_keep(va, v, tbuf);
    };
    // end of a segment: whole items get bias, conversion and store; pieces of an item add into its fp32 tile
    auto flush_acc = [&](const SegWalk &w) {
        if (!mma_wave) return;
        // (an opaque copy of the lane number: the address arithmetic below depends on nothing else that changes
        // from step to step, and must not be computed ahead of the step loop and kept in registers)
        int elane = lane;
        asm volatile("" : "+v"(elane));
        const int ot0 = wave_o * 64 + 4 * (elane >> 5);      // first output channel of this lane within the tile
        const int nvalid = s.og - (w.otile * NT + ot0);       // channels from there on that exist
        const int o0 = w.wg * s.og + w.otile * NT + ot0;
        if (w.item >= a.sk_full) {
            float *tp = a.outacc + ((long)(w.item - a.sk_full) * NT + ot0) * MT + wave_p * WPOS + (elane & 31);
#pragma unroll
            for (int pb = 0; pb < PB; pb++)
#pragma unroll
                for (int ob = 0; ob < OB; ob++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int oo = ob * 32 + 8 * (r >> 2) + (r & 3);
                        if (oo < nvalid) atomicAdd(tp + oo * MT + pb * 32, acc[ob][pb][r]);
                        acc[ob][pb][r] = 0.f;
                    }
        } else {
            const T *bias = reinterpret_cast<const T *>(a.bias);
#pragma unroll
            for (int pb = 0; pb < PB; pb++) {
                const int m = w.tile * MT + wave_p * WPOS + pb * 32 + (elane & 31);
                const bool ok = m < s.M;
                const int b = m / s.P, p = m - b * s.P;
                T *op = reinterpret_cast<T *>(a.out) + ((long)b * s.Cout + o0) * s.P + p;
#pragma unroll
                for (int ob = 0; ob < OB; ob++)
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const int oo = ob * 32 + 8 * (r >> 2) + (r & 3);
                        if (ok && oo < nvalid) {
                            float v = acc[ob][pb][r];
                            if (bias) v += elem_to_f32<T>(bias[o0 + oo]);
                            op[(long)oo * s.P] = f32_to_elem<T>(d2c_epilogue(v, s.act, s.act_scale));
                        }
                        acc[ob][pb][r] = 0.f;
                    }
            }
        }
    };

    // --- pipeline.  Iteration `it` of the step sequence: step it on the matrix cores with the rows of step it+2
    // requested on the way, step it+1 interpolated with its weight fragments requested on the way, coordinates
    // of step it+3 computed.  Corner tables rotate over 3 buffers,
    // raw rows and tiles over 2.  A wavefront interpolates the positions whose rows it requested itself, so the
    // rows need no barrier, only that wavefront's own wait.
    SegWalk wc = w0;                  // coordinates: the step whose table is computed next (its offsets are requested
                                      // one iteration before)
    PosC pc = pos_of(wc);
    for (int q = 0; q < 3; q++) {
        if (q < total) {
            coords_issue(wc, pc);
            coords_finish(wc, pc, q);
            if (seg_advance(wc, s_seg, nseg, s)) pc = pos_of(wc);
        } else {
            coords_none(q);
        }
    }
    SegWalk wm = w0;                  // the step on the matrix cores
    __syncthreads();
    if (mma_wave) {
        const int wstep = __builtin_amdgcn_readfirstlane(s_meta[1]);
#pragma unroll
        for (int kg = 0; kg < NKG; kg++)
#pragma unroll
            for (int ob = 0; ob < OB; ob++) af[kg][ob] = wfrag(wstep, kg, ob);
    }
    dma_issue(0, 0);
    dma_issue(1, 1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    interp_store(0, 0, 0);
    if (3 < total) {
        coords_issue(wc, pc);
    }
    // One loop per role (separate register budgets), the same synchronisation point per iteration in each.
    if (worker) {
        // (one inner loop per segment, so that the code that stores the accumulators stays out of the loop
        // over steps; nothing but the accumulators knows where a segment ends)
        int it = 0;
        while (wm.item >= 0) {
            for (; wm.st < wm.st_hi; wm.st++, it++) {
                lds_barrier();
                // everything this wavefront has in flight is due: the weight fragments of this step (requested
                // during the last interpolation) and the rows of step it+1 (requested during the last matrix step)
                __builtin_amdgcn_s_waitcnt(0x0F70);     // vmcnt(0)
                mma_dma_step(it & 1, it & 1, (it + 2) % 3);
                // (past the end of the sequence the interpolation works on stale rows into the tile nobody reads)
                interp_wload_store((it + 1) & 1, (it + 1) % 3, (it + 1) & 1);
            }
            flush_acc(wm);
            wm.seg++;
            seg_load(wm, s_seg, nseg, s);
        }
    } else {
        // (at default priority: with its short instruction sequence, issuing ahead of the two workers of its SIMD
        // costs 3 % on the 512-channel tile and gains nothing on the 256-channel one)
        for (int it = 0; it < total; it++) {
            lds_barrier();
            if (it + 3 < total) {                      // offsets requested one iteration ago
                coords_finish(wc, pc, it % 3);
                if (seg_advance(wc, s_seg, nseg, s)) pc = pos_of(wc);
            }
            if (it + 4 < total) {
                coords_issue(wc, pc);
            }
        }
    }
}

template <typename T, bool AUX16, int WAVES_O, int WAVES_P, bool SIZED, int NC, bool COLS = false>
__global__ void __launch_bounds__(kThreads + 64) tiled_fwd_dma_kernel(FwdArgs a)
{
    constexpr int MT = kDMT;
    // (separate arrays, not slices of one: the compiler then knows which of them a DMA transfer fills, and
    // lets accesses to the others go ahead while transfers are in flight)
    __shared__ __align__(16) unsigned char s_raw[2 * MT * NC * kNV * 16];   // [2][MT][NC corners][128 B]
    __shared__ __align__(16) unsigned char s_tile[2 * MT * kRS];      // [2][MT][kRS]
    __shared__ float s_w[3 * 8 * MT];                                 // [3][8][MT]
    __shared__ int2 s_if[3 * MT];                                     // [3][MT] (offset of corner 000, live corners)
    __shared__ int s_meta[3 * 4];                                     // [3][first channel, weight-fragment row]
    __shared__ int4 s_seg[2 * kMaxSeg];                               // [kMaxSeg][2]
    fwd_dma_body<T, AUX16, WAVES_O, WAVES_P, SIZED, NC, COLS>(a, s_raw, s_tile, s_w, s_if, s_meta, s_seg);
}

// out = fp32 tile + bias for the items whose steps were shared out (see FwdArgs).  One block = 32 output
// channels of one such item.
template <typename T>
__global__ void __launch_bounds__(256) fwd_dma_finish_kernel(FwdArgs a, int NT)
{
    constexpr int MT = kDMT;
    const TiledShape &s = a.s;
    const int item = a.sk_full + blockIdx.x;
    const int tile = item % a.sk_ntile, otile = (item / a.sk_ntile) % a.sk_otiles, wg = item / (a.sk_ntile * a.sk_otiles);
    const float *acc = a.outacc + (long)blockIdx.x * NT * MT;
    const T *bias = reinterpret_cast<const T *>(a.bias);
    T *out = reinterpret_cast<T *>(a.out);
    for (int e = threadIdx.x; e < 32 * MT; e += 256) {
        const int ot = blockIdx.y * 32 + e / MT, pl = e % MT;
        const int ol = otile * NT + ot, m = tile * MT + pl;
        if (ol >= s.og || m >= s.M) continue;
        const int o = wg * s.og + ol, b = m / s.P, p = m - b * s.P;
        float v = acc[(long)ot * MT + pl];
        if (bias) v += elem_to_f32<T>(bias[o]);
        out[((long)b * s.Cout + o) * s.P + p] = f32_to_elem<T>(d2c_epilogue(v, s.act, s.act_scale));
    }
}

template <typename T, bool AUX16, int WO, int WP>
int launch_fwd_dma(FwdArgs a, float *outacc, hipStream_t st)
{
    const bool sized = a.s.ss.on != 0;
    constexpr int NT = 64 * WO;
    const int ncu = d2c_num_cus();
    if (ncu <= 0) return D2C_ERR_LAUNCH;
    a.sk_ntile = (a.s.M + kDMT - 1) / kDMT;
    a.sk_otiles = a.s.ogp / NT;
    a.sk_items = a.sk_ntile * a.sk_otiles * a.s.groups;
    // The last, partial round: cut its items into the number of step ranges that is estimated to finish first
    // (a piece costs its steps plus about two steps' time for adding its result; the launches that clear the sums and store them
    // take as long as four.  Without those counted, us: 64 -> 512 channels, float32, three taps, on 5184 positions 54 -> 35, on 19440 69 -> 63; 128 -> 512 71 -> 58,
    // one tap; seven taps, 64 -> 256, on 6600 46 -> 38).
    // A workgroup lists at most kMaxSeg segments: very large problems get more workgroups than compute units
    // (and no cut of their last round, which is a small part of them).
    const int S = a.s.nchunk * a.s.K;
    const int maxwhole = kMaxSeg / 2;
    const int nwg_whole = a.sk_items > (long)ncu * maxwhole ? (a.sk_items + maxwhole - 1) / maxwhole : ncu;
    const int tail = nwg_whole == ncu ? a.sk_items % ncu : 0;
    a.sk_full = a.sk_items;
    a.sk_cut = 1;
    if (tail && outacc) {
        long best = S;
        for (int k = 2; k <= kMaxSeg / 2 && k <= S; k++) {
            const long rounds = ((long)tail * k + ncu - 1) / ncu;
            const long cost = rounds * ((S + k - 1) / k + 2);
            if (cost < best) { best = cost; a.sk_cut = k; }
        }
        if (a.sk_cut > 1 && (best + 4) * 10 < (long)S * 9) a.sk_full = a.sk_items - tail; else a.sk_cut = 1;
    }
    const int nshare = a.sk_items - a.sk_full;
    a.outacc = nshare ? outacc : nullptr;
    if (nshare) {
        D2cProfScope prof(D2C_PROF_PACK, st);
        d2c_fill_zero(outacc, (size_t)nshare * NT * kDMT * sizeof(float), st);
    }
    {
        const int nwg = nshare ? ncu : (a.sk_items < nwg_whole ? a.sk_items : nwg_whole);
        D2cProfScope prof(D2C_PROF_FWD, st, "tiled_fwd_dma_kernel");
        // offsets fixed along one / two axes (the layers that deform in space or in time only): 4 / 2 corner rows
        const int nfree = a.s.nd == 3 ? __builtin_popcount(a.s.axes & 7) : 3;
        // (the variants that also write the columns: all three offset axes)
        if (a.col && nfree == 3) {
            if (sized) hipLaunchKernelGGL((tiled_fwd_dma_kernel<T, AUX16, WO, WP, true, 8, true>), dim3(nwg), dim3(kThreads + 64), 0, st, a);
            else hipLaunchKernelGGL((tiled_fwd_dma_kernel<T, AUX16, WO, WP, false, 8, true>), dim3(nwg), dim3(kThreads + 64), 0, st, a);
        } else if (sized) hipLaunchKernelGGL((tiled_fwd_dma_kernel<T, AUX16, WO, WP, true, 8>), dim3(nwg), dim3(kThreads + 64), 0, st, a);
        else if (nfree == 2) hipLaunchKernelGGL((tiled_fwd_dma_kernel<T, AUX16, WO, WP, false, 4>), dim3(nwg), dim3(kThreads + 64), 0, st, a);
        else if (nfree == 1) hipLaunchKernelGGL((tiled_fwd_dma_kernel<T, AUX16, WO, WP, false, 2>), dim3(nwg), dim3(kThreads + 64), 0, st, a);
        else hipLaunchKernelGGL((tiled_fwd_dma_kernel<T, AUX16, WO, WP, false, 8>), dim3(nwg), dim3(kThreads + 64), 0, st, a);
        if (int rc = d2c_check_launch("tiled_fwd_dma_kernel")) return rc;
    }
    if (nshare) {
        D2cProfScope prof(D2C_PROF_PACK, st);
        hipLaunchKernelGGL(fwd_dma_finish_kernel<T>, dim3(nshare, NT / 32), dim3(256), 0, st, a, NT);
        return d2c_check_launch("fwd_dma_finish_kernel");
    }
    return 0;
}

}  // namespace

// Which of the two forward kernels a shape runs on: the DMA-gather kernel (64-position tiles, 512 or 256 output channels
// per workgroup, persistent, the steps of its last round of work items shared out) or the one whose wavefronts work alone
// (32-position tiles, 128 or 64 output channels, d2c_tiled_wave.hip).  Measured on both, us per forward call, DMA first:
//   up to 128 output channels the DMA kernel's output tile stays mostly empty.  64 -> 64, float32: 16000 positions 100,
//   64; 51360 positions 281, 187.  128 -> 128: 171, 125; 509, 404.  256 -> 40: 319, 202; 1002, 705; bfloat16 128 -> 128:
//   99, 75; 277, 229; 1024 -> 128 325, 299; 1396, 1340.  But wavefronts at different steps share no fragments, and weights that the L2
//   of an XCD does not hold come from further away, as do rows of many channels.  Float32, 10496, 20000 and 51200 positions: 512 -> 128 (7 MB)
//   426, 460; 807, 751; 2080, 2059.  576 -> 128 477, 529; 916, 870; 2341, 2458.  768 -> 96 (10 MB in tiles of 128) 631, 745; 1211, 1259; 3267, 3659.
//   768 -> 64 626, 664; 1203, 1131; 3245, 3213.  1024 -> 64 800, 928; 1598, 1646; 4616, 4847.
//   In thin maps many taps lie outside, whose rows the other kernel leaves out and the DMA kernel fetches as zeros.  3x3x3, 1, 2, 3 and 4 planes:
//   768 -> 96 1112, 775; 1130, 791; 2200, 1490; 1159, 970.  1024 -> 128 1491, 1030; 1524, 1068; 3032, 2148; 1564, 1347.  2048 -> 64 2918, 1628; 3011, 1826; 1606, 1289;
//   3126, 2936.  2048 -> 128 2938, 2086; 3112, 2258; 1656, 1479; 3213, 3397.  8, 16 and 32 planes: 768 -> 96 661, 733; 649, 701; 618, 612.  1024 -> 64 855, 928; 837, 848;
//   795, 715.  2048 -> 64 1666, 2131; 1612, 1934; 1554, 1703.
//   With offsets fixed along an axis the rows that are not read count less here than there: 576 -> 128, two free 463, 394; 2060, 1421; one 366, 395;
//   1702, 1430.  1024 -> 64 777, 536; 3620, 2063; 609, 536; 2992, 1945;
//   bfloat16 with one axis free has few rows to fetch, and coordinates and weights, which the DMA kernel takes once for all output channels,
//   decide.  12960, 20736, 25600 and 51360 positions (203, 324, 400, 803 tiles): 64 -> 128 46, 47; 69, 68; 83, 88; 127, 147.  128 -> 128 70, 68; 98, 97;
//   119, 124; 194, 212.  192 -> 96 93, 89; 126, 127; 154, 166; 261, 281.  3 taps, 128 -> 128 25, 25; 43, 37; 40, 45; 66, 73.  Up to 64 output channels they decide too,
//   but a layer's call (modulation by a sigmoid in the sampler) is faster there: 64 -> 64 on 51360 positions, with its branch, 199, 190.  Two axes free: 128 -> 128
//   on 51360 248, 212;
//   A few steps leave some of the eight wavefronts of the other kernel without work.  25600, 51360 and 102720 positions: one step 64 -> 128, bfloat16, 31, 38; 51, 65;
//   76, 113; two, float32, 35, 42; 54, 66; 78, 112; 64 -> 64 34, 33; 51, 52; 73, 84.  Three, bfloat16, 64 -> 128 37, 39; 60, 66; 93, 114; 64 -> 64 87, 90 on 102720.  Four, float32,
//   128 -> 128 41, 46; 64, 71; 106, 130.  Six 45, 45; 73, 72; 112, 124.  Twelve 62, 62; 100, 103; 175, 189.  18 121, 101; 199, 174; 379, 318;
//   Offsets formed from a size map make coordinates dearer, which the chunks of a tap share.  12960, 25600 and 51360 positions, bfloat16, 64 -> 128, 9 taps 30, 36; 50, 65;
//   84, 109; 7 28, 28; 45, 48; 78, 80; 27 55, 60; 98, 111; 158, 188.  128 -> 128 9 43, 46; 75, 84; 122, 142; 27 94, 88; 157, 162; 267, 280.  192 -> 128 27 130, 117; 211, 222; 379, 384.
//   64 -> 64 9 29, 30; 48, 54; 80, 90; 27 54, 51; 96, 95; 154, 161; 7, a step to a wavefront, 27, 22; 43, 39; 74, 65.  128 -> 64 9 73, 73 on 25600; 27 152, 142.  Float32,
//   64 -> 128 9 42, 44; 74, 78; 119, 132; 27 93, 83; 156, 152; 266, 260.  128 -> 128 9 68, 60; 119, 111; 195, 187.  64 -> 64 9 41, 36; 73, 66; 117, 113;
//   above 128 the wavefronts sample once per 128 output channels.  256 -> 256, float32: 5120 positions 139, 200; 8192
//   189, 232.  With few tiles both share out steps, and the DMA kernel's pieces are too many: 512 -> 512, bfloat16, 324
//   positions 65, 53 (float32 70, 72), 1400 positions 82, 102; below about a thousand steps over all tiles (4 tiles of 48 steps,
//   conv1d) its pipeline is not filled either.  Where a tile's steps times the other kernel's samplings are many, it wins from four tiles on: 4, 6 and
//   9 tiles, float32, 2560 and more: 1024 -> 512 88, 96; 97, 106; 117, 143.  2048 -> 512 130, 178; 151, 206; 185, 270.  512 -> 1024 88, 94; 100, 113; 119, 191.
//   1536 -> 256 74, 80; 86, 87; 102, 108.  768 -> 512 79, 76; 82, 84; 99, 110; bfloat16 2048 -> 512 86, 96; 92, 106; 107, 140; fewer: 1024 -> 256 61, 57; 70, 62;
//   81, 74.  512 -> 512 68, 55; 72, 60; 82, 80.  2048 -> 512, 9 taps, 78, 71; 84, 80; 94, 102; and on three tiles 512 -> 1024 81, 79.
//   Few steps on a hundred tiles and more, that kernel samples four times and more: 64 -> 512 on 5184, 6600 and 7920 positions, float32, one tap 28, 30; 29, 38; 30, 38;
//   three 35, 32; 36, 41; 37, 42; bfloat16 31, 29; 32, 37; 32, 37, nine 40, 42; 41, 54; 41, 62.  64 -> 320 three taps 34, 24; 35, 32; 35, 33.
constexpr int kDmaTilesNarrow = 160, kDmaTilesWide = 128, kDmaTilesLeast = 10, kDmaStepsWide = 1024, kDmaTilesOneAxis = 384,
              kDmaTilesShort = 384, kDmaStepsShort = 4, kDmaTilesShortLong = 1600, kDmaStepsShortLong = 12,
              kDmaTilesFew = 4, kDmaStepsFew = 2560, kDmaTilesWidest = 100, kColsTiles = 48, kColsStepsNarrowF32 = 2048, kColsTilesWideF32 = 20;
constexpr size_t kDmaWeightBytes = 8u << 20, kDmaRowsF32 = 27 * 1024;
// Share of the (position, tap) pairs along an axis whose undisplaced sampling point lies in the volume
static double taps_inside(int n, int out, int k, int stride, int pad, int dil)
{
    long inside = 0;
    for (int t = 0; t < k; t++) {
        const int at = t * dil - pad;                     // of output position 0
        const int lo = at < 0 ? (-at + stride - 1) / stride : 0, hi = at < n ? std::min(out, (n - 1 - at) / stride + 1) : 0;
        inside += std::max(0, hi - lo);
    }
    return (double)inside / ((double)out * k);
}
static long dma_tiles(const TiledShape &s) { return (long)((s.M + kDMT - 1) / kDMT) * s.groups; }
bool d2c_fwd_use_dma(const TiledShape &s)
{
    const long tiles = dma_tiles(s);
    if (s.og <= 128) {
        size_t rows = (size_t)s.cg * s.K;
        if (tiles < kDmaTilesNarrow) return false;
        if (s.nd == 3 && (s.axes & 7) == 7) {
            const long steps = (long)s.nchunk * s.K;
            if (s.og > 64 ? (tiles >= kDmaTilesShort && steps <= kDmaStepsShort) || (tiles >= kDmaTilesShortLong && steps <= kDmaStepsShortLong)
                          : tiles >= kDmaTilesShortLong && 2 * steps <= kDmaStepsShort)
                return true;
            // (384 tiles as above)
            if (s.ss.on && (s.bkc == 32 ? s.og > 64 && steps <= 18 && tiles >= kDmaTilesShort
                                        : s.og > 64 ? s.nchunk == 1 || (s.nchunk == 2 && tiles >= kDmaTilesShort)
                                                    : s.nchunk == 1 && steps > 8 && tiles >= kDmaTilesShort))
                return true;
        }
        if (s.bkc == 32 && s.nd == 3 && (s.axes & 7) == 7) {
            const double in = taps_inside(s.D, s.Do, s.geo.kd, s.geo.sd, s.geo.pd, s.geo.dd) *
                              taps_inside(s.H, s.Ho, s.geo.kh, s.geo.sh, s.geo.ph, s.geo.dh) *
                              taps_inside(s.W, s.Wo, s.geo.kw, s.geo.sw, s.geo.pw, s.geo.dw);
            if (in < 0.8) return false;
            if (in < 0.85) rows = rows * 9 / 20;          // (four planes: above, the line lies between 1024 -> 128 and 2048 -> 128, short of 2048 -> 64)
            return rows * (s.og > 64 ? 128 : 64) * 4 >= kDmaWeightBytes || rows >= kDmaRowsF32;
        }
        if (s.bkc == 64 && s.nd == 3 && __builtin_popcount(s.axes & 7) == 1 && s.og > 64 && tiles >= kDmaTilesOneAxis) return true;
        return s.og > 64 && (size_t)s.og * rows * (128 / s.bkc) >= kDmaWeightBytes;
    }
    const long steps = (long)s.nchunk * s.K;
    return tiles >= (s.og > 384 ? kDmaTilesWidest : kDmaTilesWide) || (tiles >= kDmaTilesLeast && tiles * steps >= kDmaStepsWide) ||
           (tiles >= (long)kDmaTilesFew * s.groups && steps * ((s.og + 127) / 128) >= kDmaStepsFew);
}

// Whether an infinity in a corner of weight zero stays out of the result: in the DMA-gather kernel and over sorted points always.
// The other kernel keeps to that for problems of the size that those serve otherwise; in smaller ones such a
// corner is multiplied like any other (0 * inf is NaN), as the direct kernels do.
static bool d2c_fwd_skips_zero_weights(const TiledShape &s)
{
    const long tiles = dma_tiles(s);
    return s.og <= 128 ? tiles >= kDmaTilesNarrow : tiles >= kDmaTilesWide || tiles * s.nchunk * s.K >= kDmaStepsWide;
}

// Output channels per workgroup.  The sampled tile of the DMA-gather kernel is produced once for all of them.
int d2c_fwd_out_tile(const TiledShape &s)
{
    if (d2c_fwd_use_dma(s)) return s.og > 256 ? 512 : 256;
    return s.og > 64 ? 128 : 64;
}

// Scratch of the other kernel where it shares the steps of a tile out between workgroups: the counters, all of it
size_t d2c_fwd_split_count_bytes(const TiledShape &s) { return d2c_fwd_use_dma(s) ? 0 : d2c_wave_count_bytes(s, d2c_fwd_out_tile(s)); }
size_t d2c_fwd_split_bytes(const TiledShape &s) { return d2c_fwd_use_dma(s) ? 0 : d2c_wave_split_bytes(s, d2c_fwd_out_tile(s)); }

// Whether the forward kernel of this shape can write the sampled columns for the backward pass: on problems with
// offsets along all three axes, wide weight groups from kColsTiles position tiles on (below that the backward kernels
// that read the columns lose to the ones that sample again: 256 -> 256 channels on 4x15x27, 26 tiles: 0.25 -> 0.30 ms),
// narrow ones from kDmaTilesNarrow tiles on.  Float32, whose backward pass over sorted points samples again where no columns are
// kept, from fewer: wide groups from kColsTilesWideF32 tiles, narrow ones from kColsTiles on or by the steps of all tiles.  Training steps, us, columns kept,
// sampling again; narrow, 27 taps: 64 -> 64 24 tiles 119, 117; 32 120, 124; 48 135, 147.  128 -> 128 8 130, 127; 12 128, 133; 20 134, 151.
// 256 -> 128 4 141, 142; 8 146, 156; 12 154, 172.  512 -> 128 4 174, 191.  9 taps, 256 -> 64: 24 127, 124; 32 125, 135.  7 taps, 128 -> 128: 60 129,
// 129; 80 127, 144.  Wide: 64 -> 200 20 154, 157; 32 166, 171.  256 -> 256 12 209, 218; 20 235, 259.  512 -> 512 12 534, 542; 20 522, 632.
bool d2c_fwd_writes_columns(const TiledShape &s, int dtype)
{
    const long tiles = dma_tiles(s);
    if ((dtype != D2C_BF16 && dtype != D2C_F32) || s.nd != 3 || (s.axes & 7) != 7) return false;
    if (s.og <= 128) return dtype == D2C_F32 ? tiles >= kColsTiles || tiles * s.nchunk * s.K >= kColsStepsNarrowF32 : tiles >= kDmaTilesNarrow;
    return d2c_fwd_use_dma(s) && tiles >= (dtype == D2C_F32 ? kColsTilesWideF32 : kColsTiles);
}
long d2c_columns_rows(const TiledShape &s) { return (long)((s.M + kDMT - 1) / kDMT) * kDMT; }
// `col`: where the sampled columns go (d2c_fwd_writes_columns), or NULL.
// `outacc`: partial sums of the DMA-gather kernel's shared work items, or the d2c_fwd_split_bytes() of the other kernel
// (the counters first, cleared), NULL where that one is not to split its steps.
template <typename T>
int d2c_tiled_fwd_launch(const TiledShape &s, const void *xcl, const void *off, const void *mask, const void *wp,
                         const void *bias, void *out, float *outacc, hipStream_t st, void *col)
{
    const int nt = d2c_fwd_out_tile(s);
    if (col && !d2c_fwd_writes_columns(s, (int)Elem<T>::DT)) col = nullptr;
    if (!d2c_fwd_use_dma(s)) return d2c_wave_launch<T>(s, nt, d2c_fwd_skips_zero_weights(s), xcl, off, mask, wp, bias, out, outacc, col, st);
    // the channels-last input is followed by a row of zeros (see forward_t)
    const unsigned zrow = (unsigned)((size_t)s.N * s.vol * s.Cin * sizeof(T));
    FwdArgs a{s, xcl, off, mask, wp, bias, out, nullptr, zrow, 0, 0, 0, 0, 1, nullptr, 0};
    bool aux16 = false;
    if constexpr (sizeof(T) == 2) aux16 = s.adt == D2C_BF16;
    if (col) {
        a.col = col;
        a.col_rows = d2c_columns_rows(s);
    }
    if (nt == 512) {
        if constexpr (sizeof(T) == 2) {
            if (aux16) return launch_fwd_dma<T, true, 8, 1>(a, outacc, st);
        }
        return launch_fwd_dma<T, false, 8, 1>(a, outacc, st);
    }
    if constexpr (sizeof(T) == 2) {
        if (aux16) return launch_fwd_dma<T, true, 4, 2>(a, outacc, st);
    }
    return launch_fwd_dma<T, false, 4, 2>(a, outacc, st);
}
template int d2c_tiled_fwd_launch<bf16_t>(const TiledShape &, const void *, const void *, const void *, const void *,
                                          const void *, void *, float *, hipStream_t, void *);
template int d2c_tiled_fwd_launch<float>(const TiledShape &, const void *, const void *, const void *, const void *,
                                         const void *, void *, float *, hipStream_t, void *);
