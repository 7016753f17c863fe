// Normalisation behind the convolution: the GroupNorm that follows every deformable convolution + activation of the
// reference's refinement modules (network/modules/refinement.py:38-43), from per-channel statistics of the
// convolution's output, made by a pass over it.
//
//   chan_stats[n][c] = (sum_p x[n,c,p], sum_p x[n,c,p]^2)                       fp32, per (sample, channel)
//   group g of sample n:  mean = sum / m,  var = sumsq / m - mean^2,  m = (C / groups) * P    (biased, as torch)
//   y = (x - mean) * rstd * gamma[c] + beta[c],   rstd = 1 / sqrt(var + eps)
//   backward, with xh = (x - mean) * rstd and per channel r1 = sum_p gy, r2 = sum_p gy * x:
//     grad_x = rstd * (gamma[c] * gy - A / m - xh * B / m),
//         A = sum_{c' in g} gamma[c'] * r1[c'],  B = sum_{c' in g} gamma[c'] * (r2[c'] - mean * r1[c']) * rstd
//     grad_gamma[c] = sum_n (r2 - mean * r1) * rstd,   grad_beta[c] = sum_n r1
//
// One workgroup per (sample, channel) row of P values, or per piece of one where the output depends on single values; 16-byte
// accesses, of rows of any alignment.
#include <algorithm>
#include "d2c_common.hpp"
#include "d2c_mma.hpp"

namespace {

constexpr int kGnThreads = 256;

struct GnArgs {
    d2c_group_norm_desc q;
    const void *x, *gy;          // [N][C][P]
    const float *stats;          // [N][C][2]
    const void *gamma, *beta;    // [C] or NULL (1 / 0)
    void *y;                     // forward: y; backward: grad_x
    float *part;                 // backward: [N][C][2] (r1, r2)
    void *ggamma, *gbeta;
    int pieces;                  // workgroups to a row
};

D2C_DEV float block_sum(float v, float *red)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < kGnThreads / 64; i++) t += red[i];
    return t;
}

// out[i] = f(in[0][i], ...) for a piece of a row, f = make().  Bound: memory; a thread requests up to kGnVectors vectors of each row, then works
// out f (sums over a group, double).  Few rows are several workgroups each: four to a compute unit in all, since each works out f.  (One workgroup
// to a row, a vector at a time, rows of odd lengths element by element; us, before and after, forward and gradient, bfloat16: 256 rows of 51360
// 19.6, 11.4 and 21.1, 15.0; of 51361 62, 13 and 74, 17; 1024 rows of 12960 12.3, 11.4 and 15.7, 14.9; float32 21.3, 17.3 and 25.8, 24.8; 55.8, 17.4 and
// 59.8, 24.7; 64 rows of 50 3.4, 3.9; of 1400 3.8, 3.7.)
constexpr int kGnVectors = 4;
inline int row_pieces(const d2c_group_norm_desc &q)
{
    const long rows = (long)q.N * q.C, run = (long)kGnThreads * kGnVectors * (q.dtype == D2C_BF16 ? 8 : 4), want = 4L * std::max(d2c_num_cus(), 1);
    return (int)std::max(std::min((q.P + run - 1) / run, (want + rows - 1) / rows), 1L);
}
template <typename T, int NIN, typename Make> D2C_DEV void map_piece(const T *const (&in)[NIN], T *out, int P, int piece, int pieces, Make make)
{
    constexpr int VEC = 16 / (int)sizeof(T);
    const int nv = P / VEC, len = (nv + pieces - 1) / pieces, v1 = min(nv, (piece + 1) * len);
    AnyVec<T> q[kGnVectors][NIN];
    auto request = [&](int v0) INLINE {
#pragma unroll
        for (int k = 0; k < kGnVectors; k++)
#pragma unroll
            for (int j = 0; j < NIN; j++)
                if (v0 + k * kGnThreads < v1) q[k][j] = load_any(in[j] + (long)(v0 + k * kGnThreads) * VEC);
    };
    int v0 = piece * len + (int)threadIdx.x;
    request(v0);
    const auto f = make();
    while (v0 < v1) {
#pragma unroll
        for (int k = 0; k < kGnVectors; k++) {
            if (v0 + k * kGnThreads >= v1) continue;
            alignas(16) T e[NIN][VEC], o[VEC];
#pragma unroll
            for (int j = 0; j < NIN; j++) *reinterpret_cast<AnyVec<T> *>(e[j]) = q[k][j];
#pragma unroll
            for (int i = 0; i < VEC; i++) {
                float v[NIN];
#pragma unroll
                for (int j = 0; j < NIN; j++) v[j] = elem_to_f32<T>(e[j][i]);
                o[i] = f32_to_elem<T>(f(v));
            }
            *reinterpret_cast<AnyVec<T> *>(out + (long)(v0 + k * kGnThreads) * VEC) = *reinterpret_cast<const AnyVec<T> *>(o);
        }
        v0 += kGnThreads * kGnVectors;
        request(v0);
    }
    if (piece + 1 == pieces && (int)threadIdx.x < P - nv * VEC) {
        const int i = nv * VEC + threadIdx.x;
        float v[NIN];
#pragma unroll
        for (int j = 0; j < NIN; j++) v[j] = elem_to_f32<T>(in[j][i]);
        out[i] = f32_to_elem<T>(f(v));
    }
}
// A thread's values go in sixteens, added up pairwise, then to sums in double: one chain of float additions loses up to 5e-6 of
// a sum of squares on 205440 positions (bfloat16 squares are short and round to one side), this way 6e-8.  Bound: memory, and
// latency where the rows are few.  us, chains first: 256 channels, float32, 51360 positions 18.1, 10.1; 51361 (rows of any alignment, which
// went element by element) 52.1, 10.2; bfloat16 7.2, 6.1 and 24.9, 6.5; 64 channels on 50 2.6, 2.6.
template <typename T> __global__ void __launch_bounds__(kGnThreads) channel_stats_kernel(GnArgs a)
{
    constexpr int RUN = 16, VEC = 16 / (int)sizeof(T), NV = RUN / VEC;
    __shared__ double2 red[kGnThreads / 64];
    const long rowi = blockIdx.x;
    const int P = a.q.P;
    const T *row = reinterpret_cast<const T *>(a.x) + rowi * P;
    double s = 0.0, sq = 0.0;
    auto add = [&](const float *v) {
        float t[RUN], u[RUN];
#pragma unroll
        for (int i = 0; i < RUN; i++) { t[i] = v[i]; u[i] = v[i] * v[i]; }
#pragma unroll
        for (int n = RUN / 2; n > 0; n >>= 1)
#pragma unroll
            for (int i = 0; i < n; i++) { t[i] += t[i + n]; u[i] += u[i + n]; }
        s += (double)t[0]; sq += (double)u[0];
    };
    const int nv = P / VEC;
    for (int i0 = threadIdx.x; i0 < nv; i0 += kGnThreads * NV) {
        float v[RUN];
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int i = i0 + k * kGnThreads;
            AnyVec<T> q = {0u, 0u, 0u, 0u};
            if (i < nv) q = load_any(row + (long)i * VEC);
            const uint4 w = make_uint4(q[0], q[1], q[2], q[3]);
            const T *e = reinterpret_cast<const T *>(&w);
#pragma unroll
            for (int j = 0; j < VEC; j++) v[k * VEC + j] = elem_to_f32<T>(e[j]);
        }
        add(v);
    }
    if ((int)threadIdx.x < P - nv * VEC) {
        const float v = elem_to_f32<T>(row[nv * VEC + threadIdx.x]);
        s += (double)v; sq += (double)(v * v);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) { s += __shfl_xor(s, d, 64); sq += __shfl_xor(sq, d, 64); }
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = make_double2(s, sq);
    __syncthreads();
    if (threadIdx.x == 0) {
        double2 t = red[0];
#pragma unroll
        for (int i = 1; i < kGnThreads / 64; i++) { t.x += red[i].x; t.y += red[i].y; }
        const_cast<float *>(a.stats)[rowi * 2] = (float)t.x;
        const_cast<float *>(a.stats)[rowi * 2 + 1] = (float)t.y;
    }
}

// mean and 1 / sqrt(var + eps) of a group from the sums over its (C / groups) * P values.  The per-channel fp32 sums
// are combined, and the variance sum_sq / m - mean^2 is taken, in double: with |mean| far above the standard
// deviation the two terms agree in their leading digits and a float difference would lose the variance.
D2C_DEV void moments_from_sums(double s, double sq, double m, float eps, float &mean, float &rstd)
{
    const double mu = s / m;
    const double var = fmax(sq / m - mu * mu, 0.0);
    mean = (float)mu;
    rstd = (float)(1.0 / sqrt(var + (double)eps));
}

// mean and rstd of the group that channel c of sample n belongs to
D2C_DEV void group_moments(const GnArgs &a, int n, int c, float &mean, float &rstd)
{
    const int cpg = a.q.C / a.q.groups, g = c / cpg;
    const float *st = a.stats + ((long)n * a.q.C + g * cpg) * 2;
    double s = 0.0, sq = 0.0;
    for (int i = 0; i < cpg; i++) { s += (double)st[2 * i]; sq += (double)st[2 * i + 1]; }
    moments_from_sums(s, sq, (double)cpg * (double)a.q.P, a.q.eps, mean, rstd);
}

// the same for a workgroup: its first wavefront works it out (a division and a square root in double, on every SIMD as often as it
// has wavefronts that do)
D2C_DEV void group_moments_block(const GnArgs &a, int n, int c, float &mean, float &rstd)
{
    __shared__ float2 res;
    if (threadIdx.x < 64) {
        const int cpg = a.q.C / a.q.groups, g = c / cpg;
        const float *st = a.stats + ((long)n * a.q.C + g * cpg) * 2;
        double s = 0.0, sq = 0.0;
        for (int i = threadIdx.x; i < cpg; i += 64) { s += (double)st[2 * i]; sq += (double)st[2 * i + 1]; }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) { s += __shfl_xor(s, d, 64); sq += __shfl_xor(sq, d, 64); }
        moments_from_sums(s, sq, (double)cpg * (double)a.q.P, a.q.eps, mean, rstd);
        if (threadIdx.x == 0) res = make_float2(mean, rstd);
    }
    __syncthreads();
    mean = res.x; rstd = res.y;
}

template <typename T> __global__ void __launch_bounds__(kGnThreads) gn_fwd_kernel(GnArgs a)
{
    const int row = (int)(blockIdx.x / (unsigned)a.pieces), piece = (int)blockIdx.x - row * a.pieces, n = row / a.q.C, c = row % a.q.C;
    const T *const in[1] = {reinterpret_cast<const T *>(a.x) + (long)row * a.q.P};
    map_piece<T, 1>(in, reinterpret_cast<T *>(a.y) + (long)row * a.q.P, a.q.P, piece, a.pieces, [&] {
        float mean, rstd;
        group_moments_block(a, n, c, mean, rstd);
        const float ga = a.gamma ? elem_to_f32<T>(reinterpret_cast<const T *>(a.gamma)[c]) : 1.f;
        const float be = a.beta ? elem_to_f32<T>(reinterpret_cast<const T *>(a.beta)[c]) : 0.f;
        const float sc = rstd * ga, sh = be - mean * sc;
        return [=](const float (&v)[1]) { return fmaf(v[0], sc, sh); };
    });
}

template <typename T> __global__ void __launch_bounds__(kGnThreads) gn_bwd_reduce_kernel(GnArgs a)
{
    __shared__ float red[kGnThreads / 64];
    const long rowi = blockIdx.x;
    const T *xr = reinterpret_cast<const T *>(a.x) + rowi * a.q.P;
    const T *gr = reinterpret_cast<const T *>(a.gy) + rowi * a.q.P;
    float r1 = 0.f, r2 = 0.f;
    constexpr int VEC = 16 / (int)sizeof(T);
    const int nv = a.q.P / VEC;
    // (a thread's vectors in the order of their addresses, kGnVectors of them requested at a time)
    for (int i0 = threadIdx.x; i0 < nv; i0 += kGnThreads * kGnVectors) {
        AnyVec<T> q[kGnVectors][2];
#pragma unroll
        for (int k = 0; k < kGnVectors; k++) {
            const int i = i0 + k * kGnThreads;
            q[k][0] = q[k][1] = AnyVec<T>{0u, 0u, 0u, 0u};
            if (i < nv) { q[k][0] = load_any(xr + (long)i * VEC); q[k][1] = load_any(gr + (long)i * VEC); }
        }
#pragma unroll
        for (int k = 0; k < kGnVectors; k++) {
            if (i0 + k * kGnThreads >= nv) continue;
            alignas(16) T xe[VEC], ge[VEC];
            *reinterpret_cast<AnyVec<T> *>(xe) = q[k][0]; *reinterpret_cast<AnyVec<T> *>(ge) = q[k][1];
#pragma unroll
            for (int j = 0; j < VEC; j++) {
                const float g = elem_to_f32<T>(ge[j]);
                r1 += g;
                r2 = fmaf(g, elem_to_f32<T>(xe[j]), r2);
            }
        }
    }
    if ((int)threadIdx.x < a.q.P - nv * VEC) {
        const float g = elem_to_f32<T>(gr[nv * VEC + threadIdx.x]);
        r1 += g;
        r2 = fmaf(g, elem_to_f32<T>(xr[nv * VEC + threadIdx.x]), r2);
    }
    r1 = block_sum(r1, red);
    r2 = block_sum(r2, red);
    if (threadIdx.x == 0) {
        a.part[rowi * 2] = r1;
        a.part[rowi * 2 + 1] = r2;
    }
}

template <typename T> __global__ void __launch_bounds__(kGnThreads) gn_bwd_apply_kernel(GnArgs a)
{
    __shared__ float red[kGnThreads / 64];
    const int row = (int)(blockIdx.x / (unsigned)a.pieces), piece = (int)blockIdx.x - row * a.pieces, n = row / a.q.C, c = row % a.q.C;
    const int cpg = a.q.C / a.q.groups, g = c / cpg;
    const T *const in[2] = {reinterpret_cast<const T *>(a.x) + (long)row * a.q.P, reinterpret_cast<const T *>(a.gy) + (long)row * a.q.P};
    map_piece<T, 2>(in, reinterpret_cast<T *>(a.y) + (long)row * a.q.P, a.q.P, piece, a.pieces, [&] {
        float mean, rstd;
        group_moments_block(a, n, c, mean, rstd);
        float A = 0.f, B = 0.f;
        for (int i = threadIdx.x; i < cpg; i += kGnThreads) {
            const int cc = g * cpg + i;
            const float gm = a.gamma ? elem_to_f32<T>(reinterpret_cast<const T *>(a.gamma)[cc]) : 1.f;
            const float r1 = a.part[((long)n * a.q.C + cc) * 2], r2 = a.part[((long)n * a.q.C + cc) * 2 + 1];
            A = fmaf(gm, r1, A);
            B = fmaf(gm, (r2 - mean * r1) * rstd, B);
        }
        A = block_sum(A, red);
        B = block_sum(B, red);
        const float m = (float)cpg * (float)a.q.P;
        const float ga = a.gamma ? elem_to_f32<T>(reinterpret_cast<const T *>(a.gamma)[c]) : 1.f;
        // grad_x = rstd * (ga * gy - A / m - xh * B / m) = c1 * gy + c2 * x + c3
        const float c1 = rstd * ga, c2 = -rstd * rstd * B / m, c3 = -rstd * A / m - c2 * mean;
        return [=](const float (&v)[2]) { return fmaf(c1, v[1], fmaf(c2, v[0], c3)); };
    });
}

// grad_gamma / grad_beta: one thread per channel, loop over the samples
template <typename T> __global__ void __launch_bounds__(256) gn_bwd_affine_kernel(GnArgs a)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= a.q.C) return;
    float gg = 0.f, gb = 0.f;
    for (int n = 0; n < a.q.N; n++) {
        float mean, rstd;
        group_moments(a, n, c, mean, rstd);
        const float r1 = a.part[((long)n * a.q.C + c) * 2], r2 = a.part[((long)n * a.q.C + c) * 2 + 1];
        gg += (r2 - mean * r1) * rstd;
        gb += r1;
    }
    if (a.ggamma) reinterpret_cast<T *>(a.ggamma)[c] = f32_to_elem<T>(gg);
    if (a.gbeta) reinterpret_cast<T *>(a.gbeta)[c] = f32_to_elem<T>(gb);
}

int check(const d2c_group_norm_desc *q)
{
    if (!q) { d2c_set_error("group norm: null description"); return D2C_ERR_SHAPE; }
    if (q->N <= 0 || q->C <= 0 || q->P <= 0 || q->groups <= 0 || q->C % q->groups != 0) {
        d2c_set_error("group norm: N, C, P, groups must be positive and groups must divide C");
        return D2C_ERR_SHAPE;
    }
    if ((long)q->N * q->C >= (1L << 31)) { d2c_set_error("group norm: too many rows"); return D2C_ERR_SHAPE; }
    if (q->dtype != D2C_F32 && q->dtype != D2C_BF16) { d2c_set_error("group norm: float32 or bfloat16 only"); return D2C_ERR_DTYPE; }
    if (!(q->eps >= 0.f)) { d2c_set_error("group norm: eps must be non-negative"); return D2C_ERR_SHAPE; }
    return D2C_OK;
}

#define GN_LAUNCH(kernel, grid, block)                                                              \
    do {                                                                                            \
        if (q->dtype == D2C_BF16) hipLaunchKernelGGL(kernel<bf16_t>, grid, block, 0, st, a);        \
        else hipLaunchKernelGGL(kernel<float>, grid, block, 0, st, a);                              \
    } while (0)

}  // namespace

extern "C" int d2c_channel_stats(const d2c_group_norm_desc *q, const void *x, float *chan_stats, void *stream)
{
    if (int rc = check(q)) return rc;
    if (!x || !chan_stats) { d2c_set_error("null tensor pointer"); return D2C_ERR_SHAPE; }
    hipStream_t st = (hipStream_t)stream;
    GnArgs a{*q, x, nullptr, chan_stats, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 1};
    GN_LAUNCH(channel_stats_kernel, dim3((unsigned)(q->N * q->C)), dim3(kGnThreads));
    return d2c_check_launch("channel_stats_kernel");
}

extern "C" int d2c_group_norm_forward(const d2c_group_norm_desc *q, const void *x, const float *chan_stats,
                                      const void *gamma, const void *beta, void *y, void *stream)
{
    if (int rc = check(q)) return rc;
    if (!x || !chan_stats || !y) { d2c_set_error("null tensor pointer"); return D2C_ERR_SHAPE; }
    hipStream_t st = (hipStream_t)stream;
    GnArgs a{*q, x, nullptr, chan_stats, gamma, beta, y, nullptr, nullptr, nullptr, row_pieces(*q)};
    GN_LAUNCH(gn_fwd_kernel, dim3((unsigned)(q->N * q->C) * (unsigned)a.pieces), dim3(kGnThreads));
    return d2c_check_launch("gn_fwd_kernel");
}

extern "C" size_t d2c_group_norm_backward_workspace_bytes(const d2c_group_norm_desc *q)
{
    if (check(q) != D2C_OK) return 0;
    return d2c_align_up((size_t)q->N * q->C * 2 * sizeof(float));
}

extern "C" int d2c_group_norm_backward(const d2c_group_norm_desc *q, const void *grad_y, const void *x,
                                       const float *chan_stats, const void *gamma, void *grad_x, void *grad_gamma,
                                       void *grad_beta, void *ws, size_t ws_bytes, void *stream)
{
    if (int rc = check(q)) return rc;
    if (!grad_y || !x || !chan_stats) { d2c_set_error("null tensor pointer"); return D2C_ERR_SHAPE; }
    const size_t need = d2c_group_norm_backward_workspace_bytes(q);
    if (!ws || ws_bytes < need || ((uintptr_t)ws & 255u)) {
        d2c_set_error("workspace of %zu bytes (256-byte aligned) required, got %zu at %p", need, ws_bytes, ws);
        return D2C_ERR_WORKSPACE;
    }
    hipStream_t st = (hipStream_t)stream;
    GnArgs a{*q, x, grad_y, chan_stats, gamma, nullptr, grad_x, (float *)ws, grad_gamma, grad_beta, row_pieces(*q)};
    GN_LAUNCH(gn_bwd_reduce_kernel, dim3((unsigned)(q->N * q->C)), dim3(kGnThreads));
    if (int rc = d2c_check_launch("gn_bwd_reduce_kernel")) return rc;
    if (grad_x) {
        GN_LAUNCH(gn_bwd_apply_kernel, dim3((unsigned)(q->N * q->C) * (unsigned)a.pieces), dim3(kGnThreads));
        if (int rc = d2c_check_launch("gn_bwd_apply_kernel")) return rc;
    }
    if (grad_gamma || grad_beta) {
        GN_LAUNCH(gn_bwd_affine_kernel, dim3((unsigned)((q->C + 255) / 256)), dim3(256));
        if (int rc = d2c_check_launch("gn_bwd_affine_kernel")) return rc;
    }
    return D2C_OK;
}
