// Backward pass of small problems of the 1-D operator: three launches (bfloat16: a fourth converts the sums), everything read in the
// layout it has.
//
//   grad-column product, its uses, columns      conv1d_data_kernel
//     gcol[c, pos] = sum_o W[o, c, k] * gout[o, pos]                               (dconv1d_gpu.cu:392-397)
//     gx[c, corner] += a_corner * alpha * gcol[c, pos]                             (atomics; :196-243)
//     goff, gmask:  sums over c of gcol[c, pos] * x[c, corner]                     (:291-364)
//     col[c, k][pos] = alpha * interpolated x, for
//   gW[o, c, k] = sum_pos gout[o, pos] * col[c, k][pos]                            conv1d_weight_kernel  (:399-455)
//
// A row of positions is contiguous in grad_out, in the input and in the columns: it is what the lanes of a wavefront lie
// along when a tile is read, and what the reduction of the second product runs along.  The matrix instruction of float
// problems is the float32 one.
//
// Bound: launches and latency (512 -> 512 channels on 4 x 64 positions, float32: 5, 27 and 11 us, where the kernels of the
// larger problems, with their layouts, clears and conversions, took 120 in 15 launches).
#include <algorithm>
#include "d2c_mma.hpp"
#include "d2c_tiled.hpp"

namespace {

constexpr int kThreads = 512, kWaves = kThreads / 64;

struct Conv1dArgs {
    TiledShape s;
    const void *gout, *x, *off, *mask, *w;
    float *gx;                // [N][Cin][L] sums (cleared), or NULL
    float *goff, *gmask;      // [N][G * K][P] sums (cleared), or NULL
    void *col;                // [Cin][K][N * Pp], zeros past the last position of a sample, or NULL
    void *gw;
    float *part;              // few tiles of grad_weight: partial sums [tile][split][64][32] of the workgroups that share one ...
    unsigned *arrived;        // ... and how many have left theirs (cleared)
    int Pp;                   // positions of a sample, rounded up to whole vectors
    int tpw;                  // taps per workgroup
    FastDiv dPp;
};

template <typename T> D2C_DEV float ld_elem(const void *p, long i) { return elem_to_f32<T>(reinterpret_cast<const T *>(p)[i]); }

// One workgroup = 32 positions (of the padded samples), 32 channels, `tpw` taps.  The eight wavefronts share out the
// reduction over the output channels (nothing is staged: a lane reads the grad_out values of its position and the
// weights of its channel) and add up through LDS; then a thread holds two channels of one position.
template <typename T, bool AUX16>
__global__ void __launch_bounds__(kThreads) conv1d_data_kernel(Conv1dArgs a)
{
    constexpr int KS = sizeof(T) == 2 ? 16 : 2;           // output channels per matrix instruction
    constexpr int UN = sizeof(T) == 2 ? 2 : 16;           // instructions whose operands are requested together
    __shared__ float s_g[kWaves][32 * 32];
    __shared__ float2 s_dot[kWaves][32];

    const TiledShape &s = a.s;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = blockIdx.y * 32, wg = c0 / s.cg, g = c0 / s.cpg;
    const int k_lo = blockIdx.z * a.tpw, k_hi = min(k_lo + a.tpw, s.K);
    const bool product = a.gx || a.goff || a.gmask;

    // lane n / thread: the position
    const int mp = blockIdx.x * 32 + n, b = fdiv(mp, a.dPp), p = mp - b * a.Pp;
    const bool there = b < s.N, ok = there && p < s.P;
    const int bb = there ? b : 0, pp = ok ? p : 0;

    const int slab = ((s.og + kWaves * KS - 1) / (kWaves * KS)) * KS;
    const int o_lo = wave * slab, o_hi = min(o_lo + slab, s.og);
    const T *const go = reinterpret_cast<const T *>(a.gout) + ((long)bb * s.Cout + wg * s.og) * s.P + pp;
    const long wrow = (long)s.cg * s.K;

    for (int k = k_lo; k < k_hi; k++) {
        // sampling point of (position, tap)
        float x1 = 0.f, al = 1.f;
        const long ai = ((long)(bb * s.G + g) * s.K + k) * s.P + pp;
        x1 = ld_auxT<AUX16>(a.off, ai);
        if (a.mask) al = ld_auxT<AUX16>(a.mask, ai);

        if (product) {
            const T *const wp = reinterpret_cast<const T *>(a.w) + (long)(wg * s.og) * wrow + (long)(c0 - wg * s.cg + n) * s.K + k;
            f32x16 acc;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] = 0.f;
            for (int o = o_lo; o < o_hi; o += UN * KS) {
                if constexpr (sizeof(T) == 4) {
                    float wv[UN], gv[UN];
#pragma unroll
                    for (int i = 0; i < UN; i++) {
                        const int oo = o + i * KS + h;
                        const bool in = oo < o_hi;
                        wv[i] = in ? wp[oo * wrow] : 0.f;
                        gv[i] = in && ok ? go[(long)oo * s.P] : 0.f;
                    }
#pragma unroll
                    for (int i = 0; i < UN; i++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[i], gv[i], acc, 0, 0, 0);
                } else {
                    alignas(16) T wv[UN][8], gv[UN][8];
#pragma unroll
                    for (int i = 0; i < UN; i++)
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            const int oo = o + i * KS + h * 8 + e;
                            const bool in = oo < o_hi;
                            wv[i][e] = in ? wp[oo * wrow] : (T)0;
                            gv[i][e] = in && ok ? go[(long)oo * s.P] : (T)0;
                        }
#pragma unroll
                    for (int i = 0; i < UN; i++)
                        mma_kgroup<T, false>(acc, operand_vec<T, false>(wv[i]), operand_vec<T, false>(gv[i]));
                }
            }
#pragma unroll
            for (int r = 0; r < 16; r++) s_g[wave][(8 * (r >> 2) + 4 * h + (r & 3)) * 32 + n] = acc[r];
        }

        // (both corners are gated by range; at integer positions the low corner of the gradients steps down by one while the
        // high one stays, and they interpolate with x - (x0 - 1): dconv1d_gpu.cu:332-339)
        const int bx = pp * s.geo.sw - s.geo.pw + k * s.geo.dw;
        const Tap3<float> t = tiled_tap3(s, 0, 0, bx, 0.f, 0.f, x1);
        const bool l0 = ok && (t.live & 1u), l1 = ok && (t.live & 2u);
        int x0q = t.x0;
        float qlo = t.lx, qhi = t.hx;
        if (s.quirks && (double)t.hx < 1e-8) {
            x0q -= 1;
            const float tq = ((float)bx + x1) - (float)x0q;
            qlo = 1.f - tq; qhi = tq;
        }
        const bool r0 = ok && x0q >= 0 && x0q < s.W, r1 = ok && t.x0 + 1 >= 0 && t.x0 + 1 < s.W;
        // the two channels of this thread: values at the corners
        const int cl = tid >> 5;
        float v0[2], v1[2], vq[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const long xi = ((long)bb * s.Cin + c0 + cl + i * 16) * s.W;
            v0[i] = l0 ? ld_elem<T>(a.x, xi + t.x0) : 0.f;
            v1[i] = l1 || r1 ? ld_elem<T>(a.x, xi + t.x0 + 1) : 0.f;
            vq[i] = x0q == t.x0 && l0 ? v0[i] : (r0 ? ld_elem<T>(a.x, xi + x0q) : 0.f);
        }
        if (a.col && there) {
            // (a corner of weight zero, of a point on a voxel or a modulation of exactly zero, is left out: an infinity there
            // reaches nothing, as in the kernels of the larger problems)
            const bool has0 = l0 && al != 0.f, has1 = l1 && t.hx > 0.f && al != 0.f;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const float v = (has0 ? t.lx * al * v0[i] : 0.f) + (has1 ? t.hx * al * v1[i] : 0.f);
                reinterpret_cast<T *>(a.col)[((long)(c0 + cl + i * 16) * s.K + k) * ((long)s.N * a.Pp) + mp] = f32_to_elem<T>(ok ? v : 0.f);
            }
        }
        if (product) {
            __syncthreads();
            float d0 = 0.f, d1 = 0.f;
#pragma unroll
            for (int i = 0; i < 2; i++) {
                float gc = 0.f;
#pragma unroll
                for (int q = 0; q < kWaves; q++) gc += s_g[q][(cl + i * 16) * 32 + n];
                if (a.gx) {
                    float *const gx = a.gx + ((long)bb * s.Cin + c0 + cl + i * 16) * s.W + t.x0;
                    if (l0) atomicAdd(gx, t.lx * al * gc);
                    if (l1) atomicAdd(gx + 1, t.hx * al * gc);
                }
                if (r0) d0 = fmaf(gc, vq[i], d0);
                if (r1) d1 = fmaf(gc, v1[i], d1);
            }
            if (a.goff || a.gmask) {
                d0 += __shfl_xor(d0, 32, 64);
                d1 += __shfl_xor(d1, 32, 64);
                if (h == 0) s_dot[wave][n] = make_float2(d0, d1);
            }
            __syncthreads();                              // (and the sums may be overwritten)
            if ((a.goff || a.gmask) && tid < 32 && ok) {
                float2 d = s_dot[0][n];
#pragma unroll
                for (int q = 1; q < kWaves; q++) { d.x += s_dot[q][n].x; d.y += s_dot[q][n].y; }
                if (a.goff) atomicAdd(a.goff + ai, al * (d.y - d.x));
                if (a.gmask) atomicAdd(a.gmask + ai, (r0 ? qlo * d.x : 0.f) + (r1 ? qhi * d.y : 0.f));
            }
        }
    }
}

// One workgroup = 64 output channels, 32 columns (channel, tap); the eight wavefronts share out the positions and add up
// through LDS.  A vector of grad_out is one load wherever its row starts (rows of an odd length went value by value: 256 -> 512 channels on 2665
// positions, backward and forward, 239 -> 196 us, bfloat16 200 -> 172; on 2656 193 either way).  Where such tiles are few, gridDim.z workgroups share one; the one that comes last adds their sums up, in a
// fixed order (as in tiled_fwd_wave_kernel).
template <typename T>
__global__ void __launch_bounds__(kThreads) conv1d_weight_kernel(Conv1dArgs a)
{
    constexpr int VEC = Elem<T>::VEC, PS = 2 * VEC;       // positions per k-group
    typedef T row_vec __attribute__((ext_vector_type(VEC), aligned(sizeof(T))));      // rows of grad_out start where they start
    __shared__ float s_g[kWaves][64 * 32];
    const TiledShape &s = a.s;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5, n = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nct = s.cg * s.K / 32, wg = blockIdx.x / nct, ct = blockIdx.x - wg * nct;
    const int o0 = blockIdx.y * 64;                       // within the weight group
    const int gp = a.Pp / PS, groups = s.N * gp;          // k-groups of a sample, of all
    const int part = blockIdx.z * kWaves + wave, parts = gridDim.z * kWaves;
    const int q_lo = (int)((long)groups * part / parts), q_hi = (int)((long)groups * (part + 1) / parts);
    const T *const cp = reinterpret_cast<const T *>(a.col) + ((long)wg * s.cg * s.K + ct * 32 + n) * ((long)s.N * a.Pp) + h * VEC;
    f32x16 acc[2];
#pragma unroll
    for (int r = 0; r < 16; r++) acc[0][r] = acc[1][r] = 0.f;
    int b = q_lo / gp, q = q_lo - b * gp;
    for (int i = q_lo; i < q_hi; i++) {
        const uint4 cv = *reinterpret_cast<const uint4 *>(cp + (long)i * PS);
        uint4 gv[2];
        const int p = q * PS + h * VEC;
#pragma unroll
        for (int ob = 0; ob < 2; ob++) {
            const int o = o0 + ob * 32 + n;
            const T *const go = reinterpret_cast<const T *>(a.gout) + ((long)b * s.Cout + wg * s.og + (o < s.og ? o : 0)) * s.P + p;
            alignas(16) T e[VEC];
            if (p + VEC <= s.P) *reinterpret_cast<uint4 *>(e) = __builtin_bit_cast(uint4, *reinterpret_cast<const row_vec *>(go));
            else
#pragma unroll
                for (int j = 0; j < VEC; j++) e[j] = p + j < s.P ? go[j] : (T)0;
            gv[ob] = *reinterpret_cast<const uint4 *>(e);
        }
#pragma unroll
        for (int ob = 0; ob < 2; ob++) mma_kgroup<T, false>(acc[ob], gv[ob], cv);
        if (++q == gp) { q = 0; b++; }
    }
#pragma unroll
    for (int ob = 0; ob < 2; ob++)
#pragma unroll
        for (int r = 0; r < 16; r++) s_g[wave][(ob * 32 + 8 * (r >> 2) + 4 * h + (r & 3)) * 32 + n] = acc[ob][r];
    __syncthreads();
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        v[i] = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; w++) v[i] += s_g[w][i * kThreads + tid];
    }
    if (gridDim.z > 1) {
        // (agent scope: past the L2 of the XCD; ordered by the wait for the stores, the barrier and the counter)
        __shared__ int s_last;
        const int item = blockIdx.x * gridDim.y + blockIdx.y;
        float *const part_p = a.part + (long)item * gridDim.z * (64 * 32) + tid;
#pragma unroll
        for (int i = 0; i < 4; i++)
            __hip_atomic_store(part_p + (long)blockIdx.z * (64 * 32) + i * kThreads, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) s_last = __hip_atomic_fetch_add(a.arrived + item, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.z - 1;
        __syncthreads();
        if (!s_last) return;
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = 0.f;
#pragma unroll 4
        for (int q = 0; q < (int)gridDim.z; q++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                v[i] += __hip_atomic_load(part_p + (long)q * (64 * 32) + i * kThreads, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int e = i * kThreads + tid, o = o0 + e / 32;
        if (o < s.og)
            reinterpret_cast<T *>(a.gw)[(long)(wg * s.og + o) * s.cg * s.K + ct * 32 + (e & 31)] = f32_to_elem<T>(v[i]);
    }
}

// What is cleared in front (up to four ranges), and the bias gradient behind it in the grid
struct Conv1dPrepArgs {
    uint32_t *zero[4];
    long words[4];
    int nblk_z;
    const void *gout;
    void *gb;
    int N, Cout, P;
};
template <typename T> __global__ void __launch_bounds__(256) conv1d_prepare_kernel(Conv1dPrepArgs a)
{
    if ((int)blockIdx.x < a.nblk_z) {
#pragma unroll
        for (int j = 0; j < 4; j++)
            for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < a.words[j]; i += (long)a.nblk_z * 256) a.zero[j][i] = 0u;
        return;
    }
    bias_grad_body<T, 256>((const T *)a.gout, (T *)a.gb, a.N, a.Cout, a.P, (int)blockIdx.x - a.nblk_z);
}

// sums -> storage type
struct Conv1dFinishArgs {
    const float *src[3];
    bf16_t *dst[3];
    long n[3];
};
__global__ void __launch_bounds__(256) conv1d_finish_kernel(Conv1dFinishArgs a)
{
#pragma unroll
    for (int j = 0; j < 3; j++)
        for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < a.n[j]; i += (long)gridDim.x * 256) a.dst[j][i] = f32_to_bf16(a.src[j][i]);
}

struct Conv1dWs {
    int Pp, nsplit;
    size_t gx, goff, gmask, col, arrived, part, total;
};
Conv1dWs conv1d_ws(const TiledShape &s, int dtype)
{
    const size_t es = dtype == D2C_BF16 ? 2 : 4, ps = 32 / es;
    Conv1dWs w;
    w.Pp = (int)((s.P + ps - 1) / ps * ps);
    const size_t na = (size_t)s.N * s.G * s.K * s.P * sizeof(float);
    w.gx = 0;
    w.goff = dtype == D2C_BF16 ? d2c_align_up((size_t)s.N * s.Cin * s.W * sizeof(float)) : 0;
    w.gmask = w.goff + (s.adt == D2C_BF16 ? d2c_align_up(na) : 0);
    w.col = w.gmask + (s.adt == D2C_BF16 ? d2c_align_up(na) : 0);
    w.arrived = w.col + d2c_align_up((size_t)s.Cin * s.K * s.N * w.Pp * es);
    const long tiles = (long)s.groups * (s.cg * s.K / 32) * ((s.og + 63) / 64), steps = (long)s.N * w.Pp / ps;
    w.nsplit = (int)std::max<long>(1, std::min<long>(std::min<long>(512 / tiles, 32), steps / (2 * kWaves)));
    w.part = w.arrived + (w.nsplit > 1 ? d2c_align_up(tiles * sizeof(unsigned)) : 0);
    w.total = w.part + (w.nsplit > 1 ? d2c_align_up((size_t)tiles * w.nsplit * 64 * 32 * sizeof(float)) : 0);
    return w;
}

}  // namespace

// Small problems: few (32 positions, 32 channels, tap) items of the first kernel, whose operands nobody shares; the others
// run on the kernels of d2c_tiled_bwd.hip.  us per forward + backward call, those first (N x Cin -> Cout, positions, taps):
//   384 items, 4 x 512 -> 512, 64, 3: float32 151, 95; bfloat16 144, 98       2016, 4 x 512 -> 512, 333, 3: 358, 220; 215, 183
//   2350, 320 -> 192, 1500, 5: 190, 169; 152, 163                             2880, 3 x 192 -> 64, 1024, 5: 151, 180; 133, 168
//   9600, 4 x 2048 -> 256, 400, 3: 614, 540; 345, 487                         18000, 4 x 1024 -> 512, 1500, 3: 1217, 1287; 397, 1327
// (Float32 problems of few input channels to an output channel are faster there from fewer items on -- 512 -> 256 on 4640 positions 291, 434 here, 512 -> 384 on 6000
// 616, 675 -- but the grad-column product there adds up in longer chains, and on two-term operands with up to 256 output channels: grad_input
// 4.4e-6 off float64 against 1.3e-7 here, 2.7e-7 against 1.5e-7 with more.)
bool d2c_conv1d_bwd_use(const TiledShape &s, int dtype)
{
    const long items = ((long)s.N * s.P + 31) / 32 * (s.Cin / 32) * s.K;
    return s.nd == 1 && s.cg % 32 == 0 && s.cpg % 32 == 0 && items <= (dtype == D2C_F32 && s.og >= 256 ? 10240 : 2048);
}
size_t d2c_conv1d_bwd_ws(const TiledShape &s, int dtype) { return conv1d_ws(s, dtype).total; }

template <typename T>
int d2c_conv1d_bwd(const TiledShape &s, const void *gout, const void *x, const void *off, const void *mask, const void *w, void *gx,
                   void *goff, void *gmask, void *gw, void *gb, void *ws, hipStream_t st)
{
    const Conv1dWs l = conv1d_ws(s, Elem<T>::DT);
    char *const base = (char *)ws;
    const bool x16 = sizeof(T) == 2, a16 = s.adt == D2C_BF16;
    const long nx = (long)s.N * s.Cin * s.W, na = (long)s.N * s.G * s.K * s.P;
    Conv1dArgs a{s, gout, x, off, mask, w, nullptr, nullptr, nullptr, gw ? base + l.col : nullptr, gw, (float *)(base + l.part),
                 (unsigned *)(base + l.arrived), l.Pp, s.K, make_fastdiv(l.Pp)};
    if (gx) a.gx = x16 ? (float *)(base + l.gx) : (float *)gx;
    if (goff) a.goff = a16 ? (float *)(base + l.goff) : (float *)goff;
    if (gmask) a.gmask = a16 ? (float *)(base + l.gmask) : (float *)gmask;
    {
        Conv1dPrepArgs z{};
        z.zero[0] = (uint32_t *)a.gx; z.words[0] = gx ? nx : 0;
        z.zero[1] = (uint32_t *)a.goff; z.words[1] = goff ? na : 0;
        z.zero[2] = (uint32_t *)a.gmask; z.words[2] = gmask ? na : 0;
        z.zero[3] = (uint32_t *)a.arrived; z.words[3] = gw ? (long)(l.part - l.arrived) / 4 : 0;
        z.nblk_z = (int)std::min<long>((std::max(std::max(z.words[0], z.words[3]), std::max(z.words[1], z.words[2])) + 1023) / 1024, 1024);
        z.gout = gout; z.gb = gb; z.N = s.N; z.Cout = s.Cout; z.P = s.P;
        const int nblk = z.nblk_z + (gb ? s.Cout : 0);
        if (nblk) {
            D2cProfScope prof(D2C_PROF_PACK, st);
            hipLaunchKernelGGL(conv1d_prepare_kernel<T>, dim3(nblk), dim3(256), 0, st, z);
            if (int rc = d2c_check_launch("conv1d_prepare_kernel")) return rc;
        }
    }
    if (gx || goff || gmask || gw) {
        const long tiles = ((long)s.N * l.Pp + 31) / 32, chunks = s.Cin / 32;
        // (all taps of a tile in one workgroup where that fills the chip: it has read their lines of the weights)
        while (a.tpw > 1 && tiles * chunks * ((s.K + a.tpw - 1) / a.tpw) < 512) a.tpw = (a.tpw + 1) / 2;
        const dim3 grid((unsigned)tiles, (unsigned)chunks, (unsigned)((s.K + a.tpw - 1) / a.tpw));
        D2cProfScope prof(D2C_PROF_BWD_DATA, st, "conv1d_data_kernel");
        if (sizeof(T) == 2 && a16) hipLaunchKernelGGL((conv1d_data_kernel<T, sizeof(T) == 2>), grid, dim3(kThreads), 0, st, a);
        else hipLaunchKernelGGL((conv1d_data_kernel<T, false>), grid, dim3(kThreads), 0, st, a);
        if (int rc = d2c_check_launch("conv1d_data_kernel")) return rc;
    }
    if (gw) {
        D2cProfScope prof(D2C_PROF_BWD_WEIGHT, st, "conv1d_weight_kernel");
        hipLaunchKernelGGL(conv1d_weight_kernel<T>, dim3((unsigned)(s.groups * (s.cg * s.K / 32)), (unsigned)((s.og + 63) / 64), (unsigned)l.nsplit),
                           dim3(kThreads), 0, st, a);
        if (int rc = d2c_check_launch("conv1d_weight_kernel")) return rc;
    }
    if ((x16 && gx) || (a16 && (goff || gmask))) {
        Conv1dFinishArgs f{{a.gx, a.goff, a.gmask}, {(bf16_t *)gx, (bf16_t *)goff, (bf16_t *)gmask},
                           {x16 && gx ? nx : 0, a16 && goff ? na : 0, a16 && gmask ? na : 0}};
        const long n = std::max(f.n[0], std::max(f.n[1], f.n[2]));
        D2cProfScope prof(D2C_PROF_PACK, st);
        hipLaunchKernelGGL(conv1d_finish_kernel, dim3((unsigned)std::min<long>((n + 255) / 256, 4096)), dim3(256), 0, st, f);
        return d2c_check_launch("conv1d_finish_kernel");
    }
    return D2C_OK;
}
template int d2c_conv1d_bwd<bf16_t>(const TiledShape &, const void *, const void *, const void *, const void *, const void *, void *, void *,
                                    void *, void *, void *, void *, hipStream_t);
template int d2c_conv1d_bwd<float>(const TiledShape &, const void *, const void *, const void *, const void *, const void *, void *, void *,
                                   void *, void *, void *, void *, hipStream_t);
