// Forward pass of small problems as an implicit GEMM on the matrix cores (see d2c_tiled_fwd.hip for the view), one chain of
// steps per wavefront.
#include "d2c_mma.hpp"
#include "d2c_tiled.hpp"

long d2c_columns_rows(const TiledShape &s);

namespace {

constexpr int kNV = 8;              // 16-byte vectors per sampled row (one chunk)
constexpr int kRS = kNV * 16 + 16;  // LDS row stride in bytes (padded: conflict-free 16-byte reads)
constexpr int kThreads = 512;

struct WaveArgs {
    TiledShape s;
    const void *xcl;   // [N][vol][Cin]
    const void *off, *mask;
    const void *wp;    // packed weights, see pack_weight_fwd
    const void *bias;
    void *out;
    // Few tiles: the steps are dealt to `nsplit` workgroups per tile, which leave their partial sums in `part`,
    // [tile][split][channel][position], and count themselves in `arrived` (zero in front of the launch).
    float *part;
    unsigned *arrived;
    int nsplit;
    unsigned xbytes;   // size of the channels-last input
    // The sampled, modulated columns kept for the backward pass (or NULL), [chunk][tap][col_rows][BKC] in the element type,
    // zeros past the last position (col_rows is a whole number of tiles, and the grid has that many)
    void *col;
    long col_rows;
    // Corners of weight zero (a point on a voxel plane, a modulation of exactly zero): not read, so that an infinity there
    // reaches nothing, or read and multiplied like any other, which makes NaN of it (see d2c_fwd_skips_zero_weights)
    int skip_zero;
};

// Tiles that are neighbours in space go to the same XCD (workgroups are dealt
// round-robin over the 8 XCDs), so that its L2 sees a compact part of the input.
D2C_DEV int xcd_swizzle(int bid, int n)
{
    const int x = bid & 7, idx = bid >> 3;
    const int q = n >> 3, r = n & 7;
    return x * q + (x < r ? x : r) + idx;
}

// Small problems: every wavefront on its own.  A workgroup owns 32 positions x NT output channels; its eight wavefronts
// (and, where the tiles are fewer than the compute units, those of the nsplit workgroups of a tile) share out the steps
// of the reduction.  A wavefront samples the 32 positions of its step into a tile of its own in LDS and multiplies it:
// there is no barrier between the first step and the sum of the partial results, so eight chains of dependent
// latencies (offsets, corner rows, fragments) run side by side instead of one.  The corners of step i + 1 and the
// fragments of step i + 1 are in flight while step i is multiplied.  The corners of an item are requested into the
// registers of the one that has just been interpolated, and a tap's offsets before the corners of the step in front of it, as they
// are stored: a wait for them is no wait for corners.  (us per forward call, with all corners of a step requested behind the
// interpolation and the offsets behind those, and this way: 64 -> 64 on 8x32x32 37.8, 35.6; bfloat16 28.3, 26.1; sized 42.0, 36.1;
// 128 -> 64 on 8x30x54, bfloat16 71.3, 65.0; 64 -> 64 on 16x60x100 343.8, 327.)
// Partial sums of workgroups go to the workspace; the one that finishes last adds them up, in a fixed order, applies bias
// and activation and stores: no clear in front, no kernel behind.
// Bound: few steps, by latency (64 -> 64 channels on 4x14x25, float32: one or two steps to a wavefront); many, by the corner
// rows through L1 and the vector ALU's 4 clocks per instruction, about equally (8x32x32: 453 MB through L1, 12 us of 28).
// Against workgroups that take a step of 128 positions together, barrier by barrier, with atomic partial sums, a clear
// and a finishing kernel, us per forward call: 4x14x25 37.5 -> 18.1, 8x32x32 62.2 -> 34.9; 128 -> 128 on 8x32x32 310 ->
// 69; 1024 -> 128 on 4x14x25 425 -> 97; conv1d 4 x 512 -> 512 on 64 positions 31.8 -> 21.9.
constexpr int kWP = 32, kWWaves = 8;
constexpr int kWTab = kWP * 8;                          // table entries of a tap: 8 corners of every position
constexpr int kWBytes = kWP * kRS + 2 * kWTab * 8;      // LDS of a wavefront: tile, two tables (weights, row offsets)
constexpr unsigned kWOutside = 0xFFFFFF00u;             // row offset of a corner that is not read: past every buffer
// LDS of a workgroup; the partial sums take the tiles' place
constexpr int wave_lds(int nt) { return kWWaves * (kWBytes > nt * kWP * 4 ? kWBytes : nt * kWP * 4); }

// A wavefront's place in the steps of its reduction: offset group, tap, chunk of that group (uniform, scalar registers).
struct WaveWalk {
    int st, j, jj, k, kz, ky, kx, g;
};
D2C_DEV WaveWalk wave_walk(const TiledShape &s, int wg, int st)
{
    WaveWalk w;
    const int t = st / s.cpc, gi = t / s.K;
    w.st = st;
    w.jj = st - t * s.cpc;
    w.k = t - gi * s.K;
    w.j = gi * s.cpc + w.jj;
    w.g = (wg * s.cg + w.j * s.bkc) / s.cpg;
    w.kx = w.k % s.geo.kw; w.ky = (w.k / s.geo.kw) % s.geo.kh; w.kz = w.k / (s.geo.kw * s.geo.kh);
    return w;
}
// one step on; true when that is another tap
D2C_DEV bool wave_advance(WaveWalk &w, const TiledShape &s)
{
    w.st++;
    if (++w.jj < s.cpc) { w.j++; return false; }
    w.jj = 0;
    if (++w.k < s.K) {
        w.j -= s.cpc - 1;
        if (++w.kx == s.geo.kw) { w.kx = 0; if (++w.ky == s.geo.kh) { w.ky = 0; w.kz++; } }
    } else {
        w.k = w.kx = w.ky = w.kz = 0;
        w.j++; w.g++;
    }
    return true;
}

// NG: items whose corners are in flight at a time
template <typename T, bool AUX16, int OB, int NG, bool SIZED, bool COLS>
__global__ void __launch_bounds__(kThreads) tiled_fwd_wave_kernel(WaveArgs a)
{
    constexpr int NT = 32 * OB;           // output channels per workgroup
    constexpr int NKG = kNV / 2;          // k-groups per step
    constexpr int ITEMS = kWP * kNV / 64; // (position, vector) items per lane
    typedef typename std::conditional<AUX16, bf16_t, float>::type AT;

    __shared__ __align__(16) unsigned char smem[wave_lds(NT)];
    __shared__ int s_last;

    const TiledShape &s = a.s;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = xcd_swizzle(blockIdx.x, gridDim.x);
    const int otile = blockIdx.y / a.nsplit, split = blockIdx.y - otile * a.nsplit, wg = blockIdx.z;
    const int m0 = tile * kWP;
    const int S = s.nchunk * s.K;                           // steps of the whole reduction
    const int wg_lo = (int)((long)S * split / a.nsplit), wg_n = (int)((long)S * (split + 1) / a.nsplit) - wg_lo;
    const int st_lo = wg_lo + wg_n * wave / kWWaves, st_hi = wg_lo + wg_n * (wave + 1) / kWWaves;

    f32x16 acc[OB];
#pragma unroll
    for (int ob = 0; ob < OB; ob++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[ob][r] = 0.f;

    if (st_lo < st_hi) {
        unsigned char *tb = smem + wave * kWBytes;
        float *tab_w = reinterpret_cast<float *>(tb + kWP * kRS);                        // [2][position][corner]
        unsigned *tab_o = reinterpret_cast<unsigned *>(tb + kWP * kRS + 2 * kWTab * 4);  // ... byte offset of the row

        // coordinates: lane = position (both halves of the wavefront work out the same ones)
        int cb = 0, cp = 0, coz = 0, coy = 0, cox = 0;
        const bool cvalid = m0 + (lane & 31) < s.M;
        if (cvalid) {
            const int m = m0 + (lane & 31);
            cb = fdiv(m, s.dP); cp = m - cb * s.P;
            coz = fdiv(cp, s.dHW);
            const int r = cp - coz * s.Ho * s.Wo;
            coy = fdiv(r, s.dW); cox = r - coy * s.Wo;
        }
        const unsigned dx = (unsigned)s.Cin * (unsigned)sizeof(T), dy = (unsigned)s.W * dx, dz = (unsigned)s.H * dy;
        float craw[4] = {0.f, 0.f, 0.f, 1.f};
        // (as it is stored: nothing here waits for what it reads; a lane without a position reads the first one's)
        auto coords_issue = [&](const WaveWalk &w) INLINE {
            tap_offsets_issue<AUX16, SIZED>(s, a.off, cb, w.g, w.k, cp, craw);
            if (a.mask) {
                const long at = mask_index(s, cb, w.g, w.k, cp);
                craw[3] = AUX16 ? __uint_as_float((unsigned)reinterpret_cast<const bf16_t *>(a.mask)[at]) : reinterpret_cast<const float *>(a.mask)[at];
            }
        };
        auto coords_finish = [&](const WaveWalk &w, int buf) INLINE {
            float cw[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            unsigned co[8];
#pragma unroll
            for (int c = 0; c < 8; c++) co[c] = kWOutside;
            if (cvalid) {
                tap_offsets_finish<AUX16, SIZED>(s, w.k, craw);
                const Tap3<float> t = tiled_tap3(s, coz * s.geo.sd - s.geo.pd + w.kz * s.geo.dd,
                                                 coy * s.geo.sh - s.geo.ph + w.ky * s.geo.dh,
                                                 cox * s.geo.sw - s.geo.pw + w.kx * s.geo.dw, craw[0], craw[1], craw[2]);
                const float am = AUX16 && a.mask ? __uint_as_float(__float_as_uint(craw[3]) << 16) : craw[3];
                const float al = (s.mact && a.mask) ? mask_act<AT>(s.mact, am) : am;
                const unsigned o0 = (unsigned)(cb * s.vol + (t.z0 * s.H + t.y0) * s.W + t.x0) * dx;
                unsigned read = t.live;
                if (__builtin_expect(a.skip_zero, 0))
                    read &= (t.hz > 0.f ? 0xFFu : 0x0Fu) & (t.hy > 0.f ? 0xFFu : 0x33u) & (t.hx > 0.f ? 0xFFu : 0x55u) & (al != 0.f ? 0xFFu : 0u);
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    const bool live = (read >> c) & 1u;
                    cw[c] = live ? tap3_weight(t, c) * al : 0.f;
                    if (live) co[c] = o0 + (c >> 2) * dz + ((c >> 1) & 1) * dy + (c & 1) * dx;
                }
            }
            if (lane < 32) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    *reinterpret_cast<float4 *>(tab_w + buf * kWTab + lane * 8 + h * 4) =
                        make_float4(cw[4 * h], cw[4 * h + 1], cw[4 * h + 2], cw[4 * h + 3]);
                    *reinterpret_cast<uint4 *>(tab_o + buf * kWTab + lane * 8 + h * 4) =
                        make_uint4(co[4 * h], co[4 * h + 1], co[4 * h + 2], co[4 * h + 3]);
                }
            }
            __builtin_amdgcn_wave_barrier();
        };

        // gather: item i of a lane = (position i * 8 + lane / 8, 16-byte vector lane % 8): one load of the wavefront
        // takes eight whole rows.  The descriptor begins at the step's first channel; corners that are not read have
        // an offset past its end, which loads zeros without a request.
        const int gpos = lane >> 3, gvec = lane & 7;
        uint4 gv[NG][8];
        auto gather_issue = [&](const WaveWalk &w, int buf, auto I) INLINE {
            constexpr int item = decltype(I)::value, i = item % NG;
            const unsigned c0 = (unsigned)(wg * s.cg + w.j * s.bkc) * (unsigned)sizeof(T);
            const __amdgpu_buffer_rsrc_t res = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<char *>(reinterpret_cast<const char *>(a.xcl)) + c0, 0, (int)(a.xbytes - c0), 0x00020000);
            unsigned co[8];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint4 v = *reinterpret_cast<const uint4 *>(tab_o + buf * kWTab + (item * 8 + gpos) * 8 + h * 4);
                co[4 * h] = v.x; co[4 * h + 1] = v.y; co[4 * h + 2] = v.z; co[4 * h + 3] = v.w;
            }
#pragma unroll
            for (int c = 0; c < 8; c++) {
                typedef unsigned u32x4_b __attribute__((ext_vector_type(4)));
                const u32x4_b v = __builtin_amdgcn_raw_buffer_load_b128(res, (int)(co[c] + (unsigned)gvec * 16u), 0, 0);
                gv[i][c] = make_uint4(v[0], v[1], v[2], v[3]);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto interp = [&](const WaveWalk &w, int buf, auto I) INLINE {
            constexpr int item = decltype(I)::value, i = item % NG;
            {
                const int pos = item * 8 + gpos;
                const float4 w0 = *reinterpret_cast<const float4 *>(tab_w + buf * kWTab + pos * 8);
                const float4 w1 = *reinterpret_cast<const float4 *>(tab_w + buf * kWTab + pos * 8 + 4);
                const float cw[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
                VecAcc<T> va;
                va.zero();
#pragma unroll
                for (int c = 0; c < 8; c++) va.fma(cw[c], gv[i][c]);
                const uint4 q = va.pack();
                *reinterpret_cast<uint4 *>(tb + pos * kRS + gvec * 16) = q;
                if constexpr (COLS) {
                    // (float: the interpolated values themselves, not the two-term operands of pack(); streaming stores,
                    // written once and read by another call)
                    u32x4_t cv = {q.x, q.y, q.z, q.w};
                    if constexpr (sizeof(T) == 4)
                        cv = u32x4_t{__float_as_uint(va.a[0]), __float_as_uint(va.a[1]), __float_as_uint(va.a[2]), __float_as_uint(va.a[3])};
                    if (otile == 0)
                        __builtin_nontemporal_store(cv, reinterpret_cast<u32x4_t *>(reinterpret_cast<char *>(a.col)
                            + (((long)(wg * s.nchunk + w.j) * s.K + w.k) * a.col_rows + m0 + pos) * (kNV * 16) + gvec * 16));
                }
            }
        };

        // weight fragments: those of the next step are requested as soon as the matrix cores have taken the current ones
        const uint4 *wp4 = reinterpret_cast<const uint4 *>(a.wp);
        const int OBT = s.ogp / 32;
        uint4 af[NKG][OB];
        auto frag_row = [&](const WaveWalk &w) INLINE {
            return wp4 + (((long)wg * S + w.j * s.K + w.k) * OBT + otile * OB) * (NKG * 64) + lane;
        };

        // The step being multiplied, whose first corners are under way, and the next one, whose tap's coordinates are (where it
        // is another tap).  Requests are waited for in their order: the coordinates of a step go in front of the corners of the step
        // before, so that working them out leaves those in flight.
        WaveWalk wm = wave_walk(s, wg, st_lo), wn = wm;
        coords_issue(wm);
        int cur = 0;
        coords_finish(wm, 0);
        bool fresh = wave_advance(wn, s);
        if (fresh && wn.st < st_hi) coords_issue(wn);
        for_each_const([&](auto I) INLINE { gather_issue(wm, 0, I); }, std::make_integer_sequence<int, NG>{});
        {
            const uint4 *fr = frag_row(wm);
#pragma unroll
            for (int kg = 0; kg < NKG; kg++)
#pragma unroll
                for (int ob = 0; ob < OB; ob++) af[kg][ob] = fr[(ob * NKG + kg) * 64];
        }
        const unsigned char *const t0 = tb + (lane & 31) * kRS + (lane >> 5) * 16;
        while (wn.st < st_hi) {
            int nxt = cur;
            if (fresh) { nxt ^= 1; coords_finish(wn, nxt); }
            WaveWalk w2 = wn;
            fresh = wave_advance(w2, s);
            if (fresh && w2.st < st_hi) coords_issue(w2);
            // (the corners of the item NG further on, of this step or the next, into the registers that have just been read)
            for_each_const([&](auto I) INLINE {
                constexpr int item = decltype(I)::value;
                interp(wm, cur, I);
                if constexpr (item + NG < ITEMS) gather_issue(wm, cur, std::integral_constant<int, item + NG>{});
                else gather_issue(wn, nxt, std::integral_constant<int, (item + NG) % ITEMS>{});
            }, std::make_integer_sequence<int, ITEMS>{});
            __builtin_amdgcn_wave_barrier();
            const uint4 *fr = frag_row(wn);
#pragma unroll
            for (int kg = 0; kg < NKG; kg++) {
                const uint4 bf = *reinterpret_cast<const uint4 *>(t0 + kg * 32);
#pragma unroll
                for (int ob = 0; ob < OB; ob++) mma_kgroup<T, kF32SplitFwd>(acc[ob], af[kg][ob], bf);
#pragma unroll
                for (int ob = 0; ob < OB; ob++) af[kg][ob] = fr[(ob * NKG + kg) * 64];
            }
            __builtin_amdgcn_wave_barrier();
            wm = wn; wn = w2; cur = nxt;
        }
        for_each_const([&](auto I) INLINE {
            constexpr int item = decltype(I)::value;
            interp(wm, cur, I);
            if constexpr (item + NG < ITEMS) gather_issue(wm, cur, std::integral_constant<int, item + NG>{});
        }, std::make_integer_sequence<int, ITEMS>{});
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int kg = 0; kg < NKG; kg++) {
            const uint4 bf = *reinterpret_cast<const uint4 *>(t0 + kg * 32);
#pragma unroll
            for (int ob = 0; ob < OB; ob++) mma_kgroup<T, kF32SplitFwd>(acc[ob], af[kg][ob], bf);
        }
    }

    // --- sum over the wavefronts (fixed order)
    __syncthreads();
    {
        float *red = reinterpret_cast<float *>(smem) + wave * (NT * kWP);        // [output channel][position]
#pragma unroll
        for (int ob = 0; ob < OB; ob++)
#pragma unroll
            for (int r = 0; r < 16; r++)
                red[(ob * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * kWP + (lane & 31)] = acc[ob][r];
    }
    __syncthreads();
    constexpr int PER = NT * kWP / kThreads;      // results per thread: channel e / 32, position e % 32
    float v[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const float *red = reinterpret_cast<const float *>(smem) + i * kThreads + tid;
        float t = red[0];
#pragma unroll
        for (int q = 1; q < kWWaves; q++) t += red[q * (NT * kWP)];
        v[i] = t;
    }
    if (a.nsplit > 1) {
        const int item = (wg * (gridDim.y / a.nsplit) + otile) * gridDim.x + tile;
        // (stores and loads of agent scope go past the L2 of the XCD by themselves: what orders them is the wait for the
        // stores, the barrier and the counter; a release and an acquire would write back and drop whole caches)
        float *part = a.part + (long)item * a.nsplit * (NT * kWP) + tid;
#pragma unroll
        for (int i = 0; i < PER; i++)
            __hip_atomic_store(part + (long)split * (NT * kWP) + i * kThreads, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0)
            s_last = __hip_atomic_fetch_add(a.arrived + item, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)a.nsplit - 1;
        __syncthreads();
        if (!s_last) return;
#pragma unroll
        for (int i = 0; i < PER; i++) v[i] = 0.f;
#pragma unroll 4
        for (int q = 0; q < a.nsplit; q++)
#pragma unroll
            for (int i = 0; i < PER; i++)
                v[i] += __hip_atomic_load(part + (long)q * (NT * kWP) + i * kThreads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // --- bias, activation, store (a half of a wavefront holds the 32 positions of one channel)
    T *out = reinterpret_cast<T *>(a.out);
    const T *bias = reinterpret_cast<const T *>(a.bias);
    const int m = m0 + (tid & 31);
    const bool ok = m < s.M;
    const int b = ok ? fdiv(m, s.dP) : -1, p = ok ? m - b * s.P : 0;
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int ol = otile * NT + (i * kThreads + tid) / kWP;
        if (ol >= s.og) continue;                           // (uniform over the half)
        const int o = wg * s.og + ol;
        if (ok) {
            float t = v[i];
            if (bias) t += elem_to_f32<T>(bias[o]);
            out[((long)b * s.Cout + o) * s.P + p] = f32_to_elem<T>(d2c_epilogue(t, s.act, s.act_scale));
        }
    }
}

size_t wave_items(const TiledShape &s, int nt, bool cols)
{
    const size_t tiles = cols ? d2c_columns_rows(s) / kWP : (s.M + kWP - 1) / kWP;
    return tiles * (s.ogp / nt) * s.groups;
}

template <typename T, bool AUX16, int OB, int NG>
int launch_wave(const WaveArgs &a, hipStream_t st)
{
    const int NT = 32 * OB;
    const dim3 grid(a.col ? a.col_rows / kWP : (a.s.M + kWP - 1) / kWP, a.s.ogp / NT * a.nsplit, a.s.groups);
    D2cProfScope prof(D2C_PROF_FWD, st, "tiled_fwd_wave_kernel");
#define D2C_WAVE(NG_, SIZED, COLS) hipLaunchKernelGGL((tiled_fwd_wave_kernel<T, AUX16, OB, NG_, SIZED, COLS>), grid, dim3(kThreads), 0, st, a)
    if (a.s.ss.on) { if (a.col) D2C_WAVE(2, true, true); else D2C_WAVE(2, true, false); }
    else if (a.col) D2C_WAVE(2, false, true);
    else D2C_WAVE(NG, false, false);
#undef D2C_WAVE
    return d2c_check_launch("tiled_fwd_wave_kernel");
}

}  // namespace

// Workgroups per (position tile, output tile of nt channels): 1 when the tiles alone fill the chip, or as many as there are
// compute units for (us per forward call with 1, 2 and as many as this: 64 -> 64 on 4x14x25 31.5, 24.5, 19.2; on 8x15x27, 2 of
// them, 33.5, 26.2, 25.8; 1024 -> 128 on 4x9x9 340, 181, 43).
static int wave_split(const TiledShape &s, int nt)
{
    const long wgs = (long)wave_items(s, nt, false), most = s.nchunk * s.K / kWWaves;      // (every wavefront has a step)
    long n = 256 / wgs;
    if (n > most) n = most;
    if (n > 32) n = 32;                // (the last one adds that many up)
    return n > 1 ? (int)n : 1;
}
// Scratch of the split: arrival counters (cleared in front of the launch), partial sums behind them
size_t d2c_wave_count_bytes(const TiledShape &s, int nt) { return wave_split(s, nt) > 1 ? wave_items(s, nt, true) * sizeof(unsigned) : 0; }
size_t d2c_wave_split_bytes(const TiledShape &s, int nt)
{
    const size_t n = d2c_wave_count_bytes(s, nt);
    return n ? d2c_align_up(n) + d2c_align_up(wave_items(s, nt, true) * wave_split(s, nt) * nt * kWP * sizeof(float)) : 0;
}

// `split`: d2c_wave_split_bytes() of scratch, or NULL: the steps of a tile stay with one workgroup
template <typename T>
int d2c_wave_launch(const TiledShape &s, int nt, bool skip_zero, const void *xcl, const void *off, const void *mask, const void *wp,
                    const void *bias, void *out, float *split, void *col, hipStream_t st)
{
    WaveArgs a{s, xcl, off, mask, wp, bias, out, nullptr, nullptr, 1, (unsigned)((size_t)s.N * s.vol * s.Cin * sizeof(T)),
               col, d2c_columns_rows(s), skip_zero};
    if (split && d2c_wave_split_bytes(s, nt)) {
        a.nsplit = wave_split(s, nt);
        a.arrived = reinterpret_cast<unsigned *>(split);
        a.part = reinterpret_cast<float *>(reinterpret_cast<char *>(split) + d2c_align_up(d2c_wave_count_bytes(s, nt)));
    }
    if constexpr (sizeof(T) == 2) {
        if (s.adt == D2C_BF16) return nt == 128 ? launch_wave<T, true, 4, 2>(a, st) : launch_wave<T, true, 2, 4>(a, st);
    }
    return nt == 128 ? launch_wave<T, false, 4, 2>(a, st) : launch_wave<T, false, 2, 4>(a, st);
}
template int d2c_wave_launch<bf16_t>(const TiledShape &, int, bool, const void *, const void *, const void *, const void *, const void *,
                                     void *, float *, void *, hipStream_t);
template int d2c_wave_launch<float>(const TiledShape &, int, bool, const void *, const void *, const void *, const void *, const void *,
                                    void *, float *, void *, hipStream_t);
