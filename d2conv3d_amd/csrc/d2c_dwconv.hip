// Plain depthwise conv3d (one filter per output channel, no sampling): the
// operator of the reference's second extension (ops/fast-depthwise-conv3d,
// csrc/grouped_conv3d.cu), whose kernels take one thread per output element
// and read every input value from memory (:25-92 forward, :97-175 grad_input,
// :178-276 grad_weight with a shared-memory reduction per output channel).
//
// The usual filter of the backbone -- 3x3x3, unit stride and dilation, padding 1, one output channel per input channel --
// runs on kernels that march along z (dwc_march_*): a thread owns kVW x kMR elements of a plane, every plane is read
// once and serves three output planes from registers; the backward kernel forms grad_input, grad_weight and grad_bias
// from the same reads.  The other shapes:
//
// Here the tensors stay NCDHW (W contiguous) and a thread owns kVW consecutive
// elements along W: for 3x3x3 filters with unit stride and dilation along W
// (the backbone's case) an input row segment of kVW + 2 values serves 3 taps of
// kVW outputs, i.e. 13.5 instead of 27 loads per output, all of them coalesced
// along W.  A workgroup works on one (sample, output channel): its 27 weights
// are wavefront-uniform.  Other filter shapes take one element per thread with
// run-time loops.  Sums are float (double for float64 tensors).
//
//   forward     : out[n,co,o]   = bias[co] + sum_k w[co,k] * x[n, co/m, o*s - p + k*d]
//   grad_input  : gx[n,ci,i]    = sum_{co in ci*m..} sum_k w[co,k] * gout[n,co,(i + p - k*d)/s]   (where divisible)
//   grad_weight : gw[co,k]      = sum_{n,o} gout[n,co,o] * x[n, co/m, o*s - p + k*d]   (registers, wavefront and
//                                  workgroup reduction, one atomic per workgroup and tap into a scratch array)
//   grad_bias   : gb[co]        = sum_{n,o} gout[n,co,o]
#include "d2c_mma.hpp"

namespace {

constexpr int kVW = 4;         // elements along W per thread (blocked kernels)
constexpr int kThreadsDw = 256;
constexpr int kTX = 16, kTY = 16;   // blocked kernels: a workgroup = kTX groups of kVW elements along W x kTY rows

struct DwcShape {
    d2c_dwconv3d_desc q;
    int mult;       // output channels per input channel
    int K;          // taps
    long P, vol;    // output positions / input voxels per (sample, channel)
};

// storage type -> type of the sums
template <typename ST> struct Acc { typedef float type; };
template <> struct Acc<double> { typedef double type; };
template <typename ST> D2C_DEV typename Acc<ST>::type ldv(const ST *p, long i) { return (typename Acc<ST>::type)p[i]; }
template <> D2C_DEV float ldv<bf16_t>(const bf16_t *p, long i) { return bf16_to_f32(p[i]); }
template <typename ST> D2C_DEV void stv(ST *p, long i, typename Acc<ST>::type v) { p[i] = (ST)v; }
template <> D2C_DEV void stv<bf16_t>(bf16_t *p, long i, float v) { p[i] = f32_to_bf16(v); }

// Tile of a workgroup of the blocked kernels over a volume of `nz` x `ny` rows of `nx4` groups of kVW elements:
// blockIdx.y = (z, tile of rows, tile of groups); the divisions are per workgroup, in scalar registers.
struct Tile2 {
    int z, y, x0;
    bool ok;
};
D2C_DEV Tile2 tile_of(int nz, int ny, int nx4)
{
    const int tx = (nx4 + kTX - 1) / kTX, ty = (ny + kTY - 1) / kTY;
    int b = blockIdx.y;
    const int bx = b % tx; b /= tx;
    const int by = b % ty;
    Tile2 t;
    t.z = b / ty;
    t.y = by * kTY + (int)(threadIdx.x / kTX);
    const int g = bx * kTX + (int)(threadIdx.x % kTX);
    t.x0 = g * kVW;
    t.ok = t.y < ny && g < nx4 && t.z < nz;
    return t;
}
inline unsigned tiles_of(int nz, int ny, int nx4) { return (unsigned)(nz * ((ny + kTY - 1) / kTY) * ((nx4 + kTX - 1) / kTX)); }

// The kVW + 2 values  src[row + first .. row + first + kVW + 1]  of a row of `width` elements, zero outside the row
// or when the row itself is outside the volume (`row_ok` false; `row` is then any row inside the volume).
// VEC: first + 1 is a multiple of kVW, the row is kVW-aligned in memory and `width` a multiple of kVW, so the middle
// kVW values are one vector load (lane-contiguous: a wavefront's request is 1 KiB of whole lines, where scalar
// loads of lanes 16 bytes apart keep the vector-memory path busy four times as long); the two outer values come
// from the neighbouring lanes of the same row (a row of the tile = 16 consecutive lanes = one DPP row), and from
// memory only at the tile's edges.  All lanes of the wavefront must take part.
template <typename ST, bool VEC>
D2C_DEV void row_segment(const ST *src, long row, int first, int width, bool row_ok, typename Acc<ST>::type *v)
{
    typedef typename Acc<ST>::type CT;
    if constexpr (VEC) {
        static_assert(sizeof(CT) == 4 && kVW == 4, "float sums, 4 elements per lane");
        const int x0 = first + 1;
        const bool in = row_ok && x0 < width;       // x0 >= 0 always; whole vector inside when its start is
        float m[4] = {0.f, 0.f, 0.f, 0.f};
        if (in) {
            if constexpr (sizeof(ST) == 4) {
                const float4 t = *reinterpret_cast<const float4 *>(src + row + x0);
                m[0] = t.x; m[1] = t.y; m[2] = t.z; m[3] = t.w;
            } else {
                const uint2 t = *reinterpret_cast<const uint2 *>(src + row + x0);
                m[0] = __uint_as_float(t.x << 16); m[1] = __uint_as_float(t.x & 0xffff0000u);
                m[2] = __uint_as_float(t.y << 16); m[3] = __uint_as_float(t.y & 0xffff0000u);
            }
        }
        // lane i-1's last value / lane i+1's first value; 0 at the ends of the 16-lane row
        float left = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m[3]), 0x111, 0xF, 0xF, true));   // row_shr 1
        float right = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m[0]), 0x101, 0xF, 0xF, true));  // row_shl 1
        const int tx = threadIdx.x % kTX;
        if (tx == 0 && in && first >= 0) left = ldv<ST>(src, row + first);
        if (tx == kTX - 1 && row_ok && first + kVW + 1 < width) right = ldv<ST>(src, row + first + kVW + 1);
        v[0] = left; v[1] = m[0]; v[2] = m[1]; v[3] = m[2]; v[4] = m[3]; v[5] = right;
    } else {
#pragma unroll
        for (int i = 0; i < kVW + 2; i++) {
            const int ix = first + i;
            const CT t = ldv<ST>(src, row + min(max(ix, 0), width - 1));
            v[i] = (row_ok && ix >= 0 && ix < width) ? t : (CT)0;
        }
    }
}

// ---------------------------------------------------------------- forward
template <typename ST, int MODE>
__global__ void __launch_bounds__(kThreadsDw) dwc_fwd_kernel(DwcShape s, const ST *x, const ST *w, const ST *bias, ST *out)
{
    typedef typename Acc<ST>::type CT;
    const d2c_dwconv3d_desc &q = s.q;
    const int nc = blockIdx.x, n = nc / q.Cout, co = nc - n * q.Cout, ci = co / s.mult;
    const long xb = ((long)n * q.C + ci) * s.vol, ob = (long)nc * s.P;
    const long wb = (long)co * s.K;
    const CT bv = bias ? ldv<ST>(bias, co) : (CT)0;
    if constexpr (MODE > 0) {
        CT wv[27];
#pragma unroll
        for (int k = 0; k < 27; k++) wv[k] = ldv<ST>(w, wb + k);
        const Tile2 t = tile_of(q.Do, q.Ho, (q.Wo + kVW - 1) / kVW);   // (lanes without an item go along: see row_segment)
        const int oz = t.z, oy = t.y, ox0 = t.x0, ix0 = ox0 - q.pw;
        CT acc[kVW];
#pragma unroll
        for (int i = 0; i < kVW; i++) acc[i] = bv;
        // Every load is made, from an address clamped into the volume, and dropped afterwards if it was outside:
        // without branches around them all 54 loads of a thread are in flight together.
#pragma unroll
        for (int kz = 0; kz < 3; kz++) {
            const int iz = oz * q.sd - q.pd + kz * q.dd;
#pragma unroll
            for (int ky = 0; ky < 3; ky++) {
                const int iy = oy * q.sh - q.ph + ky * q.dh;
                const bool row_ok = t.ok && iz >= 0 && iz < q.D && iy >= 0 && iy < q.H;
                const long rb = xb + ((long)min(max(iz, 0), q.D - 1) * q.H + min(max(iy, 0), q.H - 1)) * q.W;
                CT v[kVW + 2];
                row_segment<ST, MODE == 2>(x, rb, ix0, q.W, row_ok, v);
#pragma unroll
                for (int kx = 0; kx < 3; kx++)
#pragma unroll
                    for (int i = 0; i < kVW; i++) acc[i] = d2c_fma<CT>(wv[(kz * 3 + ky) * 3 + kx], v[i + kx], acc[i]);
            }
        }
        if (!t.ok) return;
        const long o = ob + ((long)oz * q.Ho + oy) * q.Wo + ox0;
#pragma unroll
        for (int i = 0; i < kVW; i++)
            if (ox0 + i < q.Wo) stv<ST>(out, o + i, acc[i]);
    } else {
        for (long it = (long)blockIdx.y * blockDim.x + threadIdx.x; it < s.P; it += (long)gridDim.y * blockDim.x) {
            const int ox = (int)(it % q.Wo), oy = (int)((it / q.Wo) % q.Ho), oz = (int)(it / ((long)q.Wo * q.Ho));
            CT acc = bv;
            for (int kz = 0; kz < q.kd; kz++) {
                const int iz = oz * q.sd - q.pd + kz * q.dd;
                if (iz < 0 || iz >= q.D) continue;
                for (int ky = 0; ky < q.kh; ky++) {
                    const int iy = oy * q.sh - q.ph + ky * q.dh;
                    if (iy < 0 || iy >= q.H) continue;
                    const long rb = xb + ((long)iz * q.H + iy) * q.W;
                    for (int kx = 0; kx < q.kw; kx++) {
                        const int ix = ox * q.sw - q.pw + kx * q.dw;
                        if (ix >= 0 && ix < q.W)
                            acc = d2c_fma<CT>(ldv<ST>(w, wb + (kz * q.kh + ky) * q.kw + kx), ldv<ST>(x, rb + ix), acc);
                    }
                }
            }
            stv<ST>(out, ob + it, acc);
        }
    }
}

// ------------------------------------------------------------- grad_input
// Output position along an axis that tap k of input index i belongs to, or -1.
D2C_DEV int out_index(int i, int p, int k, int d, int s, int n_out)
{
    const int t = i + p - k * d;
    if (t < 0) return -1;
    const int o = t / s;
    return (o * s == t && o < n_out) ? o : -1;
}

template <typename ST, int MODE>
__global__ void __launch_bounds__(kThreadsDw) dwc_bwd_input_kernel(DwcShape s, const ST *gout, const ST *w, ST *gx)
{
    typedef typename Acc<ST>::type CT;
    const d2c_dwconv3d_desc &q = s.q;
    const int nc = blockIdx.x, n = nc / q.C, ci = nc - n * q.C;
    const long xb = (long)nc * s.vol;
    if constexpr (MODE > 0) {
        const Tile2 t = tile_of(q.D, q.H, (q.W + kVW - 1) / kVW);     // (lanes without an item go along: see row_segment)
        const int iz = t.z, iy = t.y, ix0 = t.x0;
        CT acc[kVW];
#pragma unroll
        for (int i = 0; i < kVW; i++) acc[i] = (CT)0;
        for (int m = 0; m < s.mult; m++) {
            const int co = ci * s.mult + m;
            const long gb = ((long)n * q.Cout + co) * s.P, wb = (long)co * 27;
#pragma unroll
            for (int kz = 0; kz < 3; kz++) {
                const int oz = out_index(iz, q.pd, kz, q.dd, q.sd, q.Do);
#pragma unroll
                for (int ky = 0; ky < 3; ky++) {
                    const int oy = out_index(iy, q.ph, ky, q.dh, q.sh, q.Ho);
                    const bool row_ok = t.ok && oz >= 0 && oy >= 0;
                    const long rb = gb + ((long)max(oz, 0) * q.Ho + max(oy, 0)) * q.Wo;
                    // unit stride and dilation along W: ox = ix + pw - kx, so element i of this thread and tap kx
                    // read g[i + 2 - kx] of the segment that starts at ox = ix0 + pw - 2
                    CT g[kVW + 2];
                    row_segment<ST, MODE == 2>(gout, rb, ix0 + q.pw - 2, q.Wo, row_ok, g);
#pragma unroll
                    for (int kx = 0; kx < 3; kx++) {
                        const CT wk = ldv<ST>(w, wb + (kz * 3 + ky) * 3 + kx);
#pragma unroll
                        for (int i = 0; i < kVW; i++) acc[i] = d2c_fma<CT>(wk, g[i + 2 - kx], acc[i]);
                    }
                }
            }
        }
        if (!t.ok) return;
        const long o = xb + ((long)iz * q.H + iy) * q.W + ix0;
#pragma unroll
        for (int i = 0; i < kVW; i++)
            if (ix0 + i < q.W) stv<ST>(gx, o + i, acc[i]);
    } else {
        for (long it = (long)blockIdx.y * blockDim.x + threadIdx.x; it < s.vol; it += (long)gridDim.y * blockDim.x) {
            const int ix = (int)(it % q.W), iy = (int)((it / q.W) % q.H), iz = (int)(it / ((long)q.W * q.H));
            CT acc = (CT)0;
            for (int m = 0; m < s.mult; m++) {
                const int co = ci * s.mult + m;
                const long gb = ((long)n * q.Cout + co) * s.P, wb = (long)co * s.K;
                for (int kz = 0; kz < q.kd; kz++) {
                    const int oz = out_index(iz, q.pd, kz, q.dd, q.sd, q.Do);
                    if (oz < 0) continue;
                    for (int ky = 0; ky < q.kh; ky++) {
                        const int oy = out_index(iy, q.ph, ky, q.dh, q.sh, q.Ho);
                        if (oy < 0) continue;
                        for (int kx = 0; kx < q.kw; kx++) {
                            const int ox = out_index(ix, q.pw, kx, q.dw, q.sw, q.Wo);
                            if (ox >= 0)
                                acc = d2c_fma<CT>(ldv<ST>(w, wb + (kz * q.kh + ky) * q.kw + kx),
                                                  ldv<ST>(gout, gb + ((long)oz * q.Ho + oy) * q.Wo + ox), acc);
                        }
                    }
                }
            }
            stv<ST>(gx, xb + it, acc);
        }
    }
}

// ------------------------------------------------------------ grad_weight
template <typename CT> D2C_DEV CT wave_sum(CT v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// sum of `v` over the workgroup, added to *dst by one thread
template <typename CT> D2C_DEV void block_add(CT v, CT *dst, CT *s_red)
{
    v = wave_sum<CT>(v);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __syncthreads();
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        CT t = (CT)0;
        for (int i = 0; i < kThreadsDw / 64; i++) t += s_red[i];
        atomicAdd(dst, t);
    }
}

// grid = (output channels, shares of the (sample, position) items); gwacc[co][k] and gbacc[co] zeroed beforehand.
// The bias gradient is the sum of the grad_out values that pass through here anyway (gbacc may be NULL).
template <typename ST, int MODE>
__global__ void __launch_bounds__(kThreadsDw) dwc_bwd_weight_kernel(DwcShape s, const ST *gout, const ST *x,
                                                                    typename Acc<ST>::type *gwacc,
                                                                    typename Acc<ST>::type *gbacc)
{
    typedef typename Acc<ST>::type CT;
    __shared__ CT s_red[kThreadsDw / 64];
    const d2c_dwconv3d_desc &q = s.q;
    const int co = blockIdx.x, ci = co / s.mult;
    CT gsum = (CT)0;
    if constexpr (MODE > 0) {
        CT acc[27];
#pragma unroll
        for (int k = 0; k < 27; k++) acc[k] = (CT)0;
        const int wo4 = (q.Wo + kVW - 1) / kVW;
        // items = (sample, z, row); a thread walks the groups of a row, so that no division is in the inner loop
        const int rows = q.N * q.Do * q.Ho;     // < 2^30 (d2c_dwconv3d_check)
        const int tx = threadIdx.x % kTX, ty = threadIdx.x / kTX;
        for (int row = (int)blockIdx.y * kTY + ty; row < rows; row += (int)gridDim.y * kTY) {
            const int oy = row % q.Ho, oz = (row / q.Ho) % q.Do, n = row / (q.Ho * q.Do);
            const long xb = ((long)n * q.C + ci) * s.vol;
            const long grow = ((long)n * q.Cout + co) * s.P + ((long)oz * q.Ho + oy) * q.Wo;
            for (int g0 = 0; g0 < wo4; g0 += kTX) {       // the 16 lanes of a row stay together (see row_segment)
                const int g4 = g0 + tx;
                const int ox0 = g4 * kVW, ix0 = ox0 - q.pw;
                CT g[kVW];
                if constexpr (MODE == 2) {
                    // (Wo is a multiple of kVW here: a group is inside the row or past it as a whole)
                    float m[4] = {0.f, 0.f, 0.f, 0.f};
                    if (ox0 < q.Wo) {
                        if constexpr (sizeof(ST) == 4) {
                            const float4 t = *reinterpret_cast<const float4 *>(gout + grow + ox0);
                            m[0] = t.x; m[1] = t.y; m[2] = t.z; m[3] = t.w;
                        } else {
                            const uint2 t = *reinterpret_cast<const uint2 *>(gout + grow + ox0);
                            m[0] = __uint_as_float(t.x << 16); m[1] = __uint_as_float(t.x & 0xffff0000u);
                            m[2] = __uint_as_float(t.y << 16); m[3] = __uint_as_float(t.y & 0xffff0000u);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < kVW; i++) g[i] = (CT)m[i];
                } else {
#pragma unroll
                    for (int i = 0; i < kVW; i++) g[i] = ox0 + i < q.Wo ? ldv<ST>(gout, grow + ox0 + i) : (CT)0;
                }
#pragma unroll
                for (int i = 0; i < kVW; i++) gsum += g[i];
#pragma unroll
                for (int kz = 0; kz < 3; kz++) {
                    const int iz = oz * q.sd - q.pd + kz * q.dd;
#pragma unroll
                    for (int ky = 0; ky < 3; ky++) {
                        const int iy = oy * q.sh - q.ph + ky * q.dh;
                        const bool row_ok = iz >= 0 && iz < q.D && iy >= 0 && iy < q.H;
                        const long rb = xb + ((long)min(max(iz, 0), q.D - 1) * q.H + min(max(iy, 0), q.H - 1)) * q.W;
                        CT v[kVW + 2];
                        row_segment<ST, MODE == 2>(x, rb, ix0, q.W, row_ok, v);
#pragma unroll
                        for (int kx = 0; kx < 3; kx++)
#pragma unroll
                            for (int i = 0; i < kVW; i++)
                                acc[(kz * 3 + ky) * 3 + kx] = d2c_fma<CT>(g[i], v[i + kx], acc[(kz * 3 + ky) * 3 + kx]);
                    }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < 27; k++) block_add<CT>(acc[k], gwacc + (long)co * 27 + k, s_red);
    } else {
        const long items = s.P * q.N;
        for (int k = 0; k < s.K; k++) {
            const int kx = k % q.kw, ky = (k / q.kw) % q.kh, kz = k / (q.kw * q.kh);
            CT acc = (CT)0;
            for (long it = (long)blockIdx.y * blockDim.x + threadIdx.x; it < items; it += (long)gridDim.y * blockDim.x) {
                const int n = (int)(it / s.P);
                const long r = it - (long)n * s.P;
                const int ox = (int)(r % q.Wo), oy = (int)((r / q.Wo) % q.Ho), oz = (int)(r / ((long)q.Wo * q.Ho));
                const int iz = oz * q.sd - q.pd + kz * q.dd, iy = oy * q.sh - q.ph + ky * q.dh,
                          ix = ox * q.sw - q.pw + kx * q.dw;
                const CT gv = ldv<ST>(gout, ((long)n * q.Cout + co) * s.P + r);
                if (k == 0) gsum += gv;
                if (iz >= 0 && iz < q.D && iy >= 0 && iy < q.H && ix >= 0 && ix < q.W)
                    acc = d2c_fma<CT>(gv, ldv<ST>(x, ((long)n * q.C + ci) * s.vol + ((long)iz * q.H + iy) * q.W + ix), acc);
            }
            block_add<CT>(acc, gwacc + (long)co * s.K + k, s_red);
        }
    }
    if (gbacc) block_add<CT>(gsum, gbacc + co, s_red);
}

template <typename ST>
__global__ void __launch_bounds__(256) dwc_cvt_kernel(const typename Acc<ST>::type *src, ST *dst, long n)
{
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
        stv<ST>(dst, i, src[i]);
}

// grad_bias alone (grad_weight not wanted): shares of the positions per output channel, partial sums added to gbacc
template <typename ST>
__global__ void __launch_bounds__(kThreadsDw) dwc_bias_grad_kernel(DwcShape s, const ST *gout,
                                                                   typename Acc<ST>::type *gbacc)
{
    typedef typename Acc<ST>::type CT;
    __shared__ CT s_red[kThreadsDw / 64];
    const d2c_dwconv3d_desc &q = s.q;
    const int co = blockIdx.x;
    CT acc = (CT)0;
    const long items = s.P * q.N;
    for (long it = (long)blockIdx.y * blockDim.x + threadIdx.x; it < items; it += (long)gridDim.y * blockDim.x) {
        const long n = it / s.P, r = it - n * s.P;
        acc += ldv<ST>(gout, (n * q.Cout + co) * s.P + r);
    }
    block_add<CT>(acc, gbacc + co, s_red);
}

// ---------------------------------------------------------------- marching kernels
// A workgroup = one (sample, channel), kTY * kMR rows, kTX * kVW columns, a range of planes.  What bounds them is memory, and close behind
// it the vector ALU (27 and 54 products to an element at a quarter of the lanes per clock): 2x256x8x56x56 float moves 103 MB
// forward, 154 MB backward (20 and 30 us at the rate of a large copy) and takes 21 and 32.  With all taps of every plane it took 30
// and 59, with those of its planes 24 and 45; the rest were registers moved from plane to plane, cleared and branched around in front of every load, and
// sums of the workgroup through LDS, 350 of 878 instructions.  bfloat16 25 and 59, 21 and 30; rows that are not vectors, 1x256x7x59x107: float 28 and
// 50, 27 and 39, bfloat16 41 and 91, 25 and 38.
constexpr int kMR = 2;                          // rows per thread
constexpr int kMTaps = 28;                      // 27 taps and the bias
struct MarchTiles {
    int ty, tx, nz, zlen;                       // tiles along y and x, ranges of planes and their length
};
MarchTiles march_tiles(const d2c_dwconv3d_desc &q)
{
    MarchTiles t;
    t.ty = (q.H + kTY * kMR - 1) / (kTY * kMR); t.tx = (q.W + kTX * kVW - 1) / (kTX * kVW);
    t.zlen = q.D;
    // (a range reads two planes more than it has: shorter than 8 for the sake of 1024 workgroups only, never than 4.  Forward +
    // backward, us, float32: 2x256x8x56x56 in one range 72, in two 80; 1x64x32x112x112 in two 150, in four 141)
    while (t.zlen > 4 && (long)q.N * q.C * t.ty * t.tx * ((q.D + t.zlen - 1) / t.zlen) < (t.zlen > 8 ? 2048 : 1024)) t.zlen = (t.zlen + 1) / 2;
    t.nz = (q.D + t.zlen - 1) / t.zlen;
    return t;
}
bool march_ok(const d2c_dwconv3d_desc &q)
{
    return q.dtype != D2C_F64 && q.Cout == q.C && q.kd == 3 && q.kh == 3 && q.kw == 3 && q.sd == 1 && q.sh == 1 && q.sw == 1 &&
           q.pd == 1 && q.ph == 1 && q.pw == 1 && q.dd == 1 && q.dh == 1 && q.dw == 1;
}
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned short u16x4_any __attribute__((ext_vector_type(4), aligned(2)));
template <typename ST> D2C_DEV void march_store(ST *row, int x0, int width, const float *m)
{
    if (x0 + kVW <= width) {
        if constexpr (sizeof(ST) == 4) *reinterpret_cast<f32x4_any *>(row + x0) = f32x4_any{m[0], m[1], m[2], m[3]};
        else {
            const uint32_t a = pack_bf16x2(m[0], m[1]), b = pack_bf16x2(m[2], m[3]);
            *reinterpret_cast<u16x4_any *>(row + x0) = u16x4_any{(unsigned short)a, (unsigned short)(a >> 16), (unsigned short)b, (unsigned short)(b >> 16)};
        }
    } else {
#pragma unroll
        for (int i = 0; i < kVW - 1; i++)
            if (x0 + i < width) stv<ST>(row, x0 + i, m[i]);
    }
}
// Rows are read through a buffer descriptor of what is left of the channel from a plane on (65535 tiles of 16 x 64 elements to a channel, the
// limit of d2c_dwconv3d_check, are far below 2 GiB).  What lies outside the volume has an offset
// past the descriptor's end and is zero, without a branch and without registers cleared in front of the load; what a vector brings from
// behind its row is cleared afterwards (not VEC).  bfloat16 rows that are not vectors: the words around their elements, shifted; the descriptor begins and
// ends with a whole word then, `skip` bytes in front of the plane.
constexpr unsigned kMarchNone = 0x80000000u;
template <typename ST, bool VEC> struct MarchPlane {
    decltype(__builtin_amdgcn_make_buffer_rsrc((void *)nullptr, 0, 0, 0)) rs;
    unsigned skip;
    D2C_DEV MarchPlane(const ST *channel, int z, long HW, int D, bool ok)
    {
        const bool in = ok && z >= 0 && z < D;
        const uintptr_t at = reinterpret_cast<uintptr_t>(channel + (in ? z : 0) * HW);
        const long bytes = (D - z) * HW * (long)sizeof(ST);
        skip = sizeof(ST) == 2 && !VEC ? (unsigned)(at & 2) : 0u;
        rs = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void *>(at - skip), 0,
                                               in ? (int)(sizeof(ST) == 2 && !VEC ? (bytes + skip + 3) & ~3l : bytes) : 0, 0x00020000);
    }
};
// byte offsets in a plane of a thread's rows y0 - 1 .. y0 + kMR, and of the element beside the tile (of its first and last lane)
struct MarchOffsets {
    unsigned o[kMR + 2], e[kMR + 2];
};
template <typename ST, bool EDGE> D2C_DEV MarchOffsets march_offsets(int y0, int x0, int H, int W)
{
    const int tx = threadIdx.x % kTX;
    const int beside = tx == 0 ? x0 - 1 : (tx == kTX - 1 && x0 + kVW < W ? x0 + kVW : -1);
    MarchOffsets r;
#pragma unroll
    for (int j = 0; j < kMR + 2; j++) {
        const int y = y0 - 1 + j;
        const bool ok = y >= 0 && y < H;
        r.o[j] = ok && x0 < W ? (unsigned)((y * W + x0) * (int)sizeof(ST)) : kMarchNone;
        if constexpr (EDGE) r.e[j] = ok && beside >= 0 ? (unsigned)((y * W + beside) * (int)sizeof(ST)) : kMarchNone;
    }
    return r;
}
// kVW elements from byte `o` of a plane on, the first of them element x0 of its row
template <typename ST, bool VEC> D2C_DEV void march_load(const MarchPlane<ST, VEC> &p, unsigned o, int x0, int width, float *m)
{
    if constexpr (sizeof(ST) == 4) {
        const auto t = __builtin_amdgcn_raw_buffer_load_b128(p.rs, (int)o, 0, 0);
#pragma unroll
        for (int i = 0; i < kVW; i++) m[i] = __uint_as_float(t[i]);
    } else {
        unsigned lo, hi;
        if constexpr (VEC) {
            const auto t = __builtin_amdgcn_raw_buffer_load_b64(p.rs, (int)o, 0, 0);
            lo = t[0]; hi = t[1];
        } else {
            const unsigned at = o + p.skip;
            const auto t = __builtin_amdgcn_raw_buffer_load_b96(p.rs, (int)(at & ~3u), 0, 0);
            lo = __builtin_amdgcn_alignbit(t[1], t[0], (at & 2u) * 8u); hi = __builtin_amdgcn_alignbit(t[2], t[1], (at & 2u) * 8u);
        }
        m[0] = __uint_as_float(lo << 16); m[1] = __uint_as_float(lo & 0xffff0000u);
        m[2] = __uint_as_float(hi << 16); m[3] = __uint_as_float(hi & 0xffff0000u);
    }
    // (the first element is zero already where it lies outside, shifted or not)
    if constexpr (!VEC) {
#pragma unroll
        for (int i = 1; i < kVW; i++) m[i] = x0 + i < width ? m[i] : 0.f;
    }
}
template <typename ST, bool VEC> D2C_DEV float march_element(const MarchPlane<ST, VEC> &p, unsigned o)
{
    if constexpr (sizeof(ST) == 4) return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(p.rs, (int)o, 0, 0));
    else return __uint_as_float((unsigned)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(p.rs, (int)(o + p.skip), 0, 0) << 16);
}
// One plane's rows y0 - 1 .. y0 + kMR of a thread, as they come from memory ...
struct MarchRows {
    float m[kMR + 2][kVW];
    float e[kMR + 2];                           // the element beside the tile (its first and last lane)
};
// (EDGE: more than one tile along x)
template <typename ST, bool VEC, bool EDGE>
D2C_DEV void march_rows(const ST *channel, int z, bool plane_ok, const MarchOffsets &f, const d2c_dwconv3d_desc &q, int x0, MarchRows &o)
{
    const MarchPlane<ST, VEC> p(channel, z, (long)q.H * q.W, q.D, plane_ok);
#pragma unroll
    for (int j = 0; j < kMR + 2; j++) {
        march_load<ST, VEC>(p, f.o[j], x0, q.W, o.m[j]);
        if constexpr (EDGE) o.e[j] = march_element<ST, VEC>(p, f.e[j]);
    }
}
template <bool EDGE> D2C_DEV void march_clear(MarchRows &o)
{
#pragma unroll
    for (int j = 0; j < kMR + 2; j++) {
        o.m[j][0] = o.m[j][1] = o.m[j][2] = o.m[j][3] = 0.f;
        if constexpr (EDGE) o.e[j] = 0.f;
    }
}
// ... and row j with its neighbours along x: v[i] is element x0 - 1 + i.  (The 16 lanes of a row are one DPP row.)
template <bool EDGE> D2C_DEV void march_segment(const MarchRows &o, int j, float *v)
{
    const int tx = threadIdx.x % kTX;
    const float left = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(o.m[j][3]), 0x111, 0xF, 0xF, true));    // row_shr 1
    const float right = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(o.m[j][0]), 0x101, 0xF, 0xF, true));   // row_shl 1
    // (a lane without a neighbour in its row of 16 gets zero)
    v[0] = EDGE && tx == 0 ? o.e[j] : left;
    v[1] = o.m[j][0]; v[2] = o.m[j][1]; v[3] = o.m[j][2]; v[4] = o.m[j][3];
    v[5] = EDGE && tx == kTX - 1 ? o.e[j] : right;
}
// rows y0 .. y0 + kMR - 1 of plane z, from v
template <typename ST, bool VEC>
D2C_DEV void march_put(ST *channel, int z, const MarchOffsets &f, const d2c_dwconv3d_desc &q, int y0, int x0, const float (&v)[kMR][kVW])
{
    const long HW = (long)q.H * q.W;
    if constexpr (VEC) {
        const MarchPlane<ST, VEC> p(channel, z, HW, q.D, true);
#pragma unroll
        for (int r = 0; r < kMR; r++) {
            if constexpr (sizeof(ST) == 4)
                __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{__float_as_uint(v[r][0]), __float_as_uint(v[r][1]), __float_as_uint(v[r][2]), __float_as_uint(v[r][3])},
                                                       p.rs, (int)f.o[r + 1], 0, 0);
            else {
                typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
                __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf16x2(v[r][0], v[r][1]), pack_bf16x2(v[r][2], v[r][3])}, p.rs, (int)f.o[r + 1], 0, 0);
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < kMR; r++)
            if (y0 + r < q.H) march_store<ST>(channel + z * HW + (long)(y0 + r) * q.W, x0, q.W, v[r]);
    }
}
struct MarchPos {
    int nc, c, y0, x0, z_lo, z_hi, tile;
};
D2C_DEV MarchPos march_pos(const d2c_dwconv3d_desc &q, const MarchTiles &t)
{
    MarchPos p;
    p.nc = blockIdx.x;
    p.c = p.nc % q.C;
    int b = blockIdx.y;
    const int bx = b % t.tx; b /= t.tx;
    const int by = b % t.ty, bz = b / t.ty;
    p.y0 = (by * kTY + (int)(threadIdx.x / kTX)) * kMR;
    p.x0 = (bx * kTX + (int)(threadIdx.x % kTX)) * kVW;
    p.z_lo = bz * t.zlen; p.z_hi = min(p.z_lo + t.zlen, q.D);
    p.tile = (p.nc / q.C) * (int)gridDim.y + (int)blockIdx.y;
    return p;
}

// f(z, phase) for the planes z0 .. z1.  What belongs to planes z - 1, z, z + 1 is entry (0, 1, 2 + phase) % 3 of its array: nothing moves from
// plane to plane (the moves were a sixth of the instructions).
template <class F> D2C_DEV void march_planes(int z0, int z1, F f)
{
    for (int z = z0; z <= z1; z += 3) {
        f(z, std::integral_constant<int, 0>{});
        if (z + 1 > z1) break;
        f(z + 1, std::integral_constant<int, 1>{});
        if (z + 2 > z1) break;
        f(z + 2, std::integral_constant<int, 2>{});
    }
}
// The wavefront's sums of kMTaps values a lane: two values change places half by half, those pairs row by row of 16 lanes, and each row adds up: 70
// instructions (kMTaps sums of their own, six steps through the LDS path each: 340).  Lanes of row r end with values 7 r .. 7 r + 6.
D2C_DEV void march_sums(const float (&v)[kMTaps], float (&o)[kMTaps / 4])
{
    static_assert(kMTaps == 28, "four rows of seven");
    float h[14];
#pragma unroll
    for (int k = 0; k < 14; k++) {
        const auto u = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[k]), __float_as_uint(v[k + 14]), false, false);
        h[k] = __uint_as_float(u[0]) + __uint_as_float(u[1]);
    }
#pragma unroll
    for (int k = 0; k < 7; k++) {
        const auto u = __builtin_amdgcn_permlane16_swap(__float_as_uint(h[k]), __float_as_uint(h[k + 7]), false, false);
        float t = __uint_as_float(u[0]) + __uint_as_float(u[1]);
        auto turned = [&](auto N) INLINE {
            return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(t), 0x120 + decltype(N)::value, 0xF, 0xF, true));   // row_ror
        };
        t += turned(std::integral_constant<int, 8>{}); t += turned(std::integral_constant<int, 4>{});
        t += turned(std::integral_constant<int, 2>{}); t += turned(std::integral_constant<int, 1>{});
        o[k] = t;
    }
}

// A plane of input touches three planes of results; those of another range are not worked on (the planes in front of and
// behind a range of four, with all 27 taps, were a third of the instructions), nor are rows by wavefronts below the volume.
template <typename ST, bool VEC, bool EDGE>
__global__ void __launch_bounds__(kThreadsDw) dwc_march_fwd_kernel(d2c_dwconv3d_desc q, MarchTiles t, const ST *__restrict__ x,
                                                                   const ST *__restrict__ w, const ST *__restrict__ bias,
                                                                   ST *__restrict__ out)
{
    const MarchPos p = march_pos(q, t);
    if (__builtin_amdgcn_readfirstlane(p.y0) >= q.H) return;
    const long HW = (long)q.H * q.W;
    const ST *xc = x + (long)p.nc * q.D * HW;
    ST *oc = out + (long)p.nc * q.D * HW;
    float wv[27];
#pragma unroll
    for (int k = 0; k < 27; k++) wv[k] = ldv<ST>(w, (long)p.c * 27 + k);
    const float bv = bias ? ldv<ST>(bias, p.c) : 0.f;
    float acc[3][kMR][kVW];                     // output planes z - 1, z, z + 1 while input plane z is worked on
#pragma unroll
    for (int i = 0; i < 3 * kMR * kVW; i++) (&acc[0][0][0])[i] = bv;
    MarchRows cur, nxt;
    const MarchOffsets f = march_offsets<ST, EDGE>(p.y0, p.x0, q.H, q.W);
    march_rows<ST, VEC, EDGE>(xc, p.z_lo - 1, true, f, q, p.x0, cur);
    march_planes(p.z_lo - 1, p.z_hi, [&](int z, auto PHASE) INLINE {
        auto a = [&](int i) INLINE -> float (&)[kMR][kVW] { return acc[(i + decltype(PHASE)::value) % 3]; };
        // (a plane that is not there: a branch; requests of nothing take as long as others.  512x4x120x190, two of six planes, 124 us without the branch, 109;
        // the backward kernel is slower with it, 193 and 214 us)
        if (z + 1 < q.D && z < p.z_hi) march_rows<ST, VEC, EDGE>(xc, z + 1, true, f, q, p.x0, nxt);
        else march_clear<EDGE>(nxt);
        float v[kMR + 2][kVW + 2];
#pragma unroll
        for (int j = 0; j < kMR + 2; j++) march_segment<EDGE>(cur, j, v[j]);
#pragma unroll
        for (int kz = 0; kz < 3; kz++) {
            const int zo = z + 1 - kz;          // the plane that tap kz of this one adds to
            if (zo < p.z_lo || zo >= p.z_hi) continue;
#pragma unroll
            for (int j = 0; j < kMR + 2; j++)
#pragma unroll
                for (int r = 0; r < kMR; r++) {
                    const int ky = j - r;       // row y0 + r reads rows y0 + r - 1 + ky
                    if (ky < 0 || ky > 2) continue;
#pragma unroll
                    for (int kx = 0; kx < 3; kx++)
#pragma unroll
                        for (int i = 0; i < kVW; i++)
                            a(2 - kz)[r][i] = fmaf(wv[(kz * 3 + ky) * 3 + kx], v[j][i + kx], a(2 - kz)[r][i]);
                }
        }
        if (z - 1 >= p.z_lo) march_put<ST, VEC>(oc, z - 1, f, q, p.y0, p.x0, a(0));
#pragma unroll
        for (int r = 0; r < kMR; r++)
#pragma unroll
            for (int i = 0; i < kVW; i++) a(0)[r][i] = bv;
        cur = nxt;
    });
}

// part[tile][channel][kMTaps]: the workgroup's sums of grad_weight and grad_bias (or NULL); gx or NULL
// (float32 rows that are not vectors, several tiles along x, spill 24 bytes a lane: a training step of 512 channels on 4x120x190 takes 302 us with
// them, of 64 on 16x120x213 156; the kernel that moved its registers from plane to plane and spilt none 316, 171)
template <typename ST, bool VEC, bool EDGE>
__global__ void __launch_bounds__(kThreadsDw, 3) dwc_march_bwd_kernel(d2c_dwconv3d_desc q, MarchTiles t, const ST *__restrict__ gout,
                                                                   const ST *__restrict__ x, const ST *__restrict__ w,
                                                                   ST *__restrict__ gx, float *__restrict__ part)
{
    const MarchPos p = march_pos(q, t);
    const long HW = (long)q.H * q.W;
    const ST *gc = gout + (long)p.nc * q.D * HW, *xc = x + (long)p.nc * q.D * HW;
    float wv[27];
#pragma unroll
    for (int k = 0; k < 27; k++) wv[k] = ldv<ST>(w, (long)p.c * 27 + k);
    float acc[3][kMR][kVW], xv[3][kMR][kVW];    // grad_input and input of planes z - 1, z, z + 1 while grad_out plane z is worked on
    float gw[kMTaps];
#pragma unroll
    for (int i = 0; i < 3 * kMR * kVW; i++) (&acc[0][0][0])[i] = (&xv[0][0][0])[i] = 0.f;
#pragma unroll
    for (int k = 0; k < kMTaps; k++) gw[k] = 0.f;
    const MarchOffsets f = march_offsets<ST, EDGE>(p.y0, p.x0, q.H, q.W);
    // (input outside the range is another workgroup's)
    auto load_x = [&](int z, float (*o)[kVW]) INLINE {
        const MarchPlane<ST, VEC> xp(xc, z, HW, q.D, part && z < p.z_hi);
#pragma unroll
        for (int r = 0; r < kMR; r++) march_load<ST, VEC>(xp, f.o[r + 1], p.x0, q.W, o[r]);
    };
    MarchRows cur, nxt;
    float xn[kMR][kVW];
    // (a wavefront below the volume only takes part in the sums)
    const int z_end = __builtin_amdgcn_readfirstlane(p.y0) < q.H ? p.z_hi : p.z_lo - 2;
    if (z_end >= p.z_lo) {
        march_rows<ST, VEC, EDGE>(gc, p.z_lo - 1, true, f, q, p.x0, cur);
        load_x(p.z_lo, xv[2]);
    }
    march_planes(p.z_lo - 1, z_end, [&](int z, auto PHASE) INLINE {
        constexpr int P = decltype(PHASE)::value;
        march_rows<ST, VEC, EDGE>(gc, z + 1, z < p.z_hi, f, q, p.x0, nxt);
        load_x(z + 2, xn);
        float v[kMR + 2][kVW + 2];
#pragma unroll
        for (int j = 0; j < kMR + 2; j++) {
            march_segment<EDGE>(cur, j, v[j]);
            if (j >= 1 && j <= kMR && z >= p.z_lo && z < p.z_hi) gw[27] += (v[j][1] + v[j][2]) + (v[j][3] + v[j][4]);
        }
        // grad_input plane z' takes tap kz of grad_out plane z = z' + 1 - kz: z' = z - 1 + kz; and grad_weight the same pair
#pragma unroll
        for (int kz = 0; kz < 3; kz++) {
            const int zo = z - 1 + kz;
            if (zo < p.z_lo || zo >= p.z_hi) continue;
#pragma unroll
            for (int j = 0; j < kMR + 2; j++)
#pragma unroll
                for (int r = 0; r < kMR; r++) {
                    const int ky = r + 2 - j;   // row y0 + r takes tap ky from row y0 + r + 1 - ky
                    if (ky < 0 || ky > 2) continue;
#pragma unroll
                    for (int kx = 0; kx < 3; kx++) {
                        const int k = (kz * 3 + ky) * 3 + kx;
#pragma unroll
                        for (int i = 0; i < kVW; i++) {
                            acc[(kz + P) % 3][r][i] = fmaf(wv[k], v[j][i + 2 - kx], acc[(kz + P) % 3][r][i]);
                            gw[k] = fmaf(xv[(kz + P) % 3][r][i], v[j][i + 2 - kx], gw[k]);
                        }
                    }
                }
        }
        if (gx && z - 1 >= p.z_lo) march_put<ST, VEC>(gx + (long)p.nc * q.D * HW, z - 1, f, q, p.y0, p.x0, acc[P]);
#pragma unroll
        for (int r = 0; r < kMR; r++)
#pragma unroll
            for (int i = 0; i < kVW; i++) {
                acc[P][r][i] = 0.f;
                xv[P][r][i] = xn[r][i];
            }
        cur = nxt;
    });
    if (!part) return;
    // Pairs with a position outside the volume, or an input of another range, were zero times something, which is no number
    // where the something is infinite or none: then pair by pair.
    float all = 0.f;
#pragma unroll
    for (int k = 0; k < 27; k++) all += gw[k];
    if (__builtin_expect(!(fabsf(all) < __builtin_inff()), 0)) {
#pragma unroll
        for (int k = 0; k < 27; k++) gw[k] = 0.f;
#pragma unroll 1
        for (int e = 0; e < (p.z_hi - p.z_lo) * kMR * kVW; e++) {
            const int z = p.z_lo + e / (kMR * kVW), y = p.y0 + e / kVW % kMR, xx = p.x0 + e % kVW;
            if (y >= q.H || xx >= q.W) continue;
            const float v = ldv<ST>(xc, z * HW + (long)y * q.W + xx);
#pragma unroll
            for (int k = 0; k < 27; k++) {
                const int gz = z + 1 - k / 9, gy = y + 1 - k / 3 % 3, gxx = xx + 1 - k % 3;
                if (gz >= 0 && gz < q.D && gy >= 0 && gy < q.H && gxx >= 0 && gxx < q.W)
                    gw[k] = fmaf(v, ldv<ST>(gc, gz * HW + (long)gy * q.W + gxx), gw[k]);
            }
        }
    }
    __shared__ float s_red[kThreadsDw / 64][kMTaps];
    float sum[kMTaps / 4];
    march_sums(gw, sum);
    if ((threadIdx.x & 15) == 0) {
#pragma unroll
        for (int k = 0; k < kMTaps / 4; k++) s_red[threadIdx.x >> 6][(threadIdx.x >> 4 & 3) * (kMTaps / 4) + k] = sum[k];
    }
    __syncthreads();
    if (threadIdx.x < kMTaps) {
        float v = 0.f;
#pragma unroll
        for (int i = 0; i < kThreadsDw / 64; i++) v += s_red[i][threadIdx.x];
        part[((long)p.tile * q.C + p.c) * kMTaps + threadIdx.x] = v;
    }
}
// One workgroup per channel: the tiles' sums -> grad_weight, grad_bias (either may be NULL)
template <typename ST>
__global__ void __launch_bounds__(256) dwc_march_finish_kernel(const float *part, int C, int ntile, ST *gw, ST *gb)
{
    __shared__ float s_sum[8][32];
    const int k = threadIdx.x & 31, sl = threadIdx.x >> 5, c = blockIdx.x;
    float v = 0.f;
    if (k < kMTaps)
        for (int i = sl; i < ntile; i += 8) v += part[((long)i * C + c) * kMTaps + k];
    s_sum[sl][k] = v;
    __syncthreads();
    if (threadIdx.x >= kMTaps) return;
    v = 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) v += s_sum[i][k];
    if (k < 27) {
        if (gw) stv<ST>(gw, (long)c * 27 + k, v);
    } else if (gb) stv<ST>(gb, c, v);
}

DwcShape make_shape(const d2c_dwconv3d_desc &q)
{
    DwcShape s;
    s.q = q;
    s.mult = q.Cout / q.C;
    s.K = q.kd * q.kh * q.kw;
    s.P = (long)q.Do * q.Ho * q.Wo;
    s.vol = (long)q.D * q.H * q.W;
    return s;
}

bool host_blocked(const d2c_dwconv3d_desc &q) { return q.kd == 3 && q.kh == 3 && q.kw == 3 && q.sw == 1 && q.dw == 1; }

unsigned blocks_for(long items, long cap)
{
    long g = (items + kThreadsDw - 1) / kThreadsDw;
    return (unsigned)(g < 1 ? 1 : (g > cap ? cap : g));
}

// vector loads of kVW elements: rows that start kVW-aligned in memory, segments that start one element left of a
// multiple of kVW (padding 1 along W)
template <typename ST> bool vec_ok(const d2c_dwconv3d_desc &q, const void *a, const void *b)
{
    const uintptr_t al = kVW * sizeof(ST);
    return sizeof(ST) <= 4 && q.pw == 1 && q.W % kVW == 0 && q.Wo == q.W && reinterpret_cast<uintptr_t>(a) % al == 0 &&
           (b == nullptr || reinterpret_cast<uintptr_t>(b) % al == 0);
}

template <typename ST>
int forward_t(const d2c_dwconv3d_desc &q, const void *x, const void *w, const void *bias, void *out, hipStream_t st)
{
    if constexpr (sizeof(ST) <= 4) {
        if (march_ok(q)) {
            const MarchTiles t = march_tiles(q);
            const dim3 grid((unsigned)(q.N * q.C), (unsigned)(t.ty * t.tx * t.nz));
            auto kern = vec_ok<ST>(q, x, out) ? (t.tx > 1 ? &dwc_march_fwd_kernel<ST, true, true> : &dwc_march_fwd_kernel<ST, true, false>)
                                              : (t.tx > 1 ? &dwc_march_fwd_kernel<ST, false, true> : &dwc_march_fwd_kernel<ST, false, false>);
            hipLaunchKernelGGL(kern, grid, dim3(kThreadsDw), 0, st, q, t, (const ST *)x, (const ST *)w, (const ST *)bias, (ST *)out);
            return d2c_check_launch("dwc_march_fwd_kernel");
        }
    }
    const DwcShape s = make_shape(q);
    const unsigned nc = (unsigned)(q.N * q.Cout);
    const dim3 tiles(nc, tiles_of(q.Do, q.Ho, (q.Wo + kVW - 1) / kVW));
    bool done = false;
    if constexpr (sizeof(ST) <= 4) {
        if (host_blocked(q) && vec_ok<ST>(q, x, nullptr)) {
            hipLaunchKernelGGL((dwc_fwd_kernel<ST, 2>), tiles, dim3(kThreadsDw), 0, st, s, (const ST *)x, (const ST *)w,
                               (const ST *)bias, (ST *)out);
            done = true;
        }
    }
    if (!done) {
        if (host_blocked(q))
            hipLaunchKernelGGL((dwc_fwd_kernel<ST, 1>), tiles, dim3(kThreadsDw), 0, st, s, (const ST *)x, (const ST *)w,
                               (const ST *)bias, (ST *)out);
        else
            hipLaunchKernelGGL((dwc_fwd_kernel<ST, 0>), dim3(nc, blocks_for(s.P, 4096)), dim3(kThreadsDw), 0, st, s,
                               (const ST *)x, (const ST *)w, (const ST *)bias, (ST *)out);
    }
    return d2c_check_launch("dwc_fwd_kernel");
}

template <typename ST>
int backward_t(const d2c_dwconv3d_desc &q, const void *gout, const void *x, const void *w, void *gx, void *gw, void *gb,
               void *ws, hipStream_t st)
{
    typedef typename Acc<ST>::type CT;
    if constexpr (sizeof(ST) <= 4) {
        if (march_ok(q)) {
            if (!gx && !gw && !gb) return D2C_OK;
            const MarchTiles t = march_tiles(q);
            const dim3 grid((unsigned)(q.N * q.C), (unsigned)(t.ty * t.tx * t.nz));
            float *part = gw || gb ? (float *)ws : nullptr;
            auto kern = vec_ok<ST>(q, gout, x) && reinterpret_cast<uintptr_t>(gx) % (kVW * sizeof(ST)) == 0
                            ? (t.tx > 1 ? &dwc_march_bwd_kernel<ST, true, true> : &dwc_march_bwd_kernel<ST, true, false>)
                            : (t.tx > 1 ? &dwc_march_bwd_kernel<ST, false, true> : &dwc_march_bwd_kernel<ST, false, false>);
            hipLaunchKernelGGL(kern, grid, dim3(kThreadsDw), 0, st, q, t, (const ST *)gout, (const ST *)x, (const ST *)w, (ST *)gx, part);
            if (int rc = d2c_check_launch("dwc_march_bwd_kernel")) return rc;
            if (!part) return D2C_OK;
            hipLaunchKernelGGL(dwc_march_finish_kernel<ST>, dim3((unsigned)q.C), dim3(256), 0, st, part, q.C, q.N * (int)grid.y, (ST *)gw,
                               (ST *)gb);
            return d2c_check_launch("dwc_march_finish_kernel");
        }
    }
    const DwcShape s = make_shape(q);
    const bool blocked = host_blocked(q);
    if (gx) {
        const unsigned nc = (unsigned)(q.N * q.C);
        const dim3 tiles(nc, tiles_of(q.D, q.H, (q.W + kVW - 1) / kVW));
        bool done = false;
        if constexpr (sizeof(ST) <= 4) {
            if (blocked && vec_ok<ST>(q, gout, nullptr)) {
                hipLaunchKernelGGL((dwc_bwd_input_kernel<ST, 2>), tiles, dim3(kThreadsDw), 0, st, s, (const ST *)gout,
                                   (const ST *)w, (ST *)gx);
                done = true;
            }
        }
        if (!done) {
            if (blocked)
                hipLaunchKernelGGL((dwc_bwd_input_kernel<ST, 1>), tiles, dim3(kThreadsDw), 0, st, s, (const ST *)gout,
                                   (const ST *)w, (ST *)gx);
            else
                hipLaunchKernelGGL((dwc_bwd_input_kernel<ST, 0>), dim3(nc, blocks_for(s.vol, 4096)), dim3(kThreadsDw), 0,
                                   st, s, (const ST *)gout, (const ST *)w, (ST *)gx);
        }
        if (int rc = d2c_check_launch("dwc_bwd_input_kernel")) return rc;
    }
    if (!gw && !gb) return D2C_OK;
    // scratch: gwacc [Cout][K], then gbacc [Cout]
    const long nw = (long)q.Cout * s.K;
    CT *gwacc = reinterpret_cast<CT *>(ws), *gbacc = gwacc + nw;
    d2c_fill_zero(gwacc, (size_t)(nw + q.Cout) * sizeof(CT), st);
    // shares of the work per output channel: enough workgroups to fill the chip, each with some work
    const long work = blocked ? (long)q.N * q.Do * q.Ho / kTY : (long)q.N * s.P / (4 * kThreadsDw);
    long shares = (2048 + q.Cout - 1) / q.Cout;
    if (shares > work) shares = work;
    if (shares < 1) shares = 1;
    if (shares > 4096) shares = 4096;
    const dim3 grid((unsigned)q.Cout, (unsigned)shares);
    if (gw) {
        bool done = false;
        if constexpr (sizeof(ST) <= 4) {
            if (blocked && vec_ok<ST>(q, x, gout)) {
                hipLaunchKernelGGL((dwc_bwd_weight_kernel<ST, 2>), grid, dim3(kThreadsDw), 0, st, s, (const ST *)gout,
                                   (const ST *)x, gwacc, gb ? gbacc : nullptr);
                done = true;
            }
        }
        if (!done) {
            if (blocked)
                hipLaunchKernelGGL((dwc_bwd_weight_kernel<ST, 1>), grid, dim3(kThreadsDw), 0, st, s, (const ST *)gout,
                                   (const ST *)x, gwacc, gb ? gbacc : nullptr);
            else
                hipLaunchKernelGGL((dwc_bwd_weight_kernel<ST, 0>), grid, dim3(kThreadsDw), 0, st, s, (const ST *)gout,
                                   (const ST *)x, gwacc, gb ? gbacc : nullptr);
        }
        if (int rc = d2c_check_launch("dwc_bwd_weight_kernel")) return rc;
        hipLaunchKernelGGL(dwc_cvt_kernel<ST>, dim3(blocks_for(nw, 1024)), dim3(256), 0, st, gwacc, (ST *)gw, nw);
    } else {
        hipLaunchKernelGGL(dwc_bias_grad_kernel<ST>, grid, dim3(kThreadsDw), 0, st, s, (const ST *)gout, gbacc);
        if (int rc = d2c_check_launch("dwc_bias_grad_kernel")) return rc;
    }
    if (gb) hipLaunchKernelGGL(dwc_cvt_kernel<ST>, dim3(blocks_for(q.Cout, 1024)), dim3(256), 0, st, gbacc, (ST *)gb, (long)q.Cout);
    return d2c_check_launch("dwc_cvt_kernel");
}

template <typename F32, typename F64, typename B16> int by_dtype(int dt, F32 f32, F64 f64, B16 b16)
{
    return dt == D2C_F64 ? f64() : (dt == D2C_F32 ? f32() : b16());
}

}  // namespace

extern "C" {

int d2c_dwconv3d_check(const d2c_dwconv3d_desc *q)
{
    if (!q) { d2c_set_error("null description"); return D2C_ERR_SHAPE; }
    if (q->dtype != D2C_F32 && q->dtype != D2C_F64 && q->dtype != D2C_BF16) {
        d2c_set_error("unsupported dtype %d", q->dtype);
        return D2C_ERR_DTYPE;
    }
    if (q->N < 1 || q->C < 1 || q->Cout < 1 || q->D < 1 || q->H < 1 || q->W < 1) {
        d2c_set_error("tensor sizes must be positive");
        return D2C_ERR_SHAPE;
    }
    if (q->Cout % q->C != 0) {   // grouped_conv3d.cu:306-309
        d2c_set_error("Depthwise out channels should be a multiple of in channels, got %d and %d", q->Cout, q->C);
        return D2C_ERR_SHAPE;
    }
    const int k[3] = {q->kd, q->kh, q->kw}, s[3] = {q->sd, q->sh, q->sw}, p[3] = {q->pd, q->ph, q->pw},
              d[3] = {q->dd, q->dh, q->dw}, in[3] = {q->D, q->H, q->W}, out[3] = {q->Do, q->Ho, q->Wo};
    for (int i = 0; i < 3; i++) {
        if (k[i] < 1) { d2c_set_error("kernel size should be at least 1"); return D2C_ERR_SHAPE; }
        if (s[i] < 1) { d2c_set_error("stride should be at least 1, got %d", s[i]); return D2C_ERR_SHAPE; }          // :314
        if (p[i] < 0) { d2c_set_error("padding should be non-negative, got %d", p[i]); return D2C_ERR_SHAPE; }      // :316
        if (d[i] < 1) { d2c_set_error("dilation should be at least 1, got %d", d[i]); return D2C_ERR_SHAPE; }       // :318
        const int span = in[i] + 2 * p[i] - (d[i] * (k[i] - 1) + 1);
        const int want = span >= 0 ? span / s[i] + 1 : 0;
        if (want < 1) { d2c_set_error("Output size should be positive, got %d at dim %d", want, i + 2); return D2C_ERR_SHAPE; }   // :409
        if (out[i] != want) {
            d2c_set_error("output size %d at dim %d does not match the computed size %d", out[i], i + 2, want);
            return D2C_ERR_SHAPE;
        }
    }
    const long lim = 1L << 31;   // 32-bit indices inside a (sample, channel) volume and over the grid
    if ((long)q->D * q->H * q->W >= lim || (long)q->Do * q->Ho * q->Wo >= lim || (long)q->N * q->Cout >= lim ||
        (long)q->N * q->C >= lim || (long)q->N * q->Do * q->Ho >= lim / 2) {
        d2c_set_error("tensor too large for 32-bit indices");
        return D2C_ERR_UNSUPPORTED;
    }
    // one workgroup per 16 rows x 64 elements of a (sample, channel) volume, counted in the grid's y extent
    const long tiles_in = (long)q->D * ((q->H + 15) / 16) * ((q->W + 63) / 64);
    const long tiles_out = (long)q->Do * ((q->Ho + 15) / 16) * ((q->Wo + 63) / 64);
    if (tiles_in > 65535 || tiles_out > 65535) {
        d2c_set_error("volume too large for the launch grid (%ld tiles per channel)", tiles_in > tiles_out ? tiles_in : tiles_out);
        return D2C_ERR_UNSUPPORTED;
    }
    return D2C_OK;
}

size_t d2c_dwconv3d_backward_workspace_bytes(const d2c_dwconv3d_desc *q)
{
    if (d2c_dwconv3d_check(q) != D2C_OK) return 0;
    if (march_ok(*q)) {
        const MarchTiles t = march_tiles(*q);
        return d2c_align_up((size_t)q->N * t.ty * t.tx * t.nz * q->C * kMTaps * sizeof(float));
    }
    return d2c_align_up((size_t)q->Cout * (q->kd * q->kh * q->kw + 1) * (q->dtype == D2C_F64 ? 8 : 4));
}

int d2c_dwconv3d_forward(const d2c_dwconv3d_desc *q, const void *x, const void *weight, const void *bias, void *out,
                         void *stream)
{
    if (int rc = d2c_dwconv3d_check(q)) return rc;
    if (!x || !weight || !out) { d2c_set_error("null tensor pointer"); return D2C_ERR_SHAPE; }
    hipStream_t st = (hipStream_t)stream;
    return by_dtype(q->dtype, [&] { return forward_t<float>(*q, x, weight, bias, out, st); },
                    [&] { return forward_t<double>(*q, x, weight, bias, out, st); },
                    [&] { return forward_t<bf16_t>(*q, x, weight, bias, out, st); });
}

int d2c_dwconv3d_backward(const d2c_dwconv3d_desc *q, const void *grad_out, const void *x, const void *weight,
                          void *grad_x, void *grad_weight, void *grad_bias, void *workspace, size_t workspace_bytes,
                          void *stream)
{
    if (int rc = d2c_dwconv3d_check(q)) return rc;
    if (!grad_out || !x || !weight) { d2c_set_error("null tensor pointer"); return D2C_ERR_SHAPE; }
    if (grad_weight || grad_bias) {
        const size_t need = d2c_dwconv3d_backward_workspace_bytes(q);
        if (!workspace || workspace_bytes < need || reinterpret_cast<uintptr_t>(workspace) % 256 != 0) {
            d2c_set_error("workspace of %zu bytes (256-byte aligned) needed, got %zu", need, workspace_bytes);
            return D2C_ERR_WORKSPACE;
        }
    }
    hipStream_t st = (hipStream_t)stream;
    return by_dtype(
        q->dtype, [&] { return backward_t<float>(*q, grad_out, x, weight, grad_x, grad_weight, grad_bias, workspace, st); },
        [&] { return backward_t<double>(*q, grad_out, x, weight, grad_x, grad_weight, grad_bias, workspace, st); },
        [&] { return backward_t<bf16_t>(*q, grad_out, x, weight, grad_x, grad_weight, grad_bias, workspace, st); });
}

}  // extern "C"
