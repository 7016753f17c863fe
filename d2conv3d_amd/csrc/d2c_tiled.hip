// Tiled kernel families: eligibility, workspace carving, operand packing and
// dispatch.  Forward / backward kernels live in d2c_tiled_fwd.hip and
// d2c_tiled_bwd.hip.
#include "d2c_tiled.hpp"
#include "d2c_brick.hpp"
#include "d2c_mma.hpp"

size_t d2c_col_forward_ws(const d2c_conv3d_desc &q);
int d2c_col_forward_prepare(const d2c_conv3d_desc &q, const void *x, void *xcl, const void *w, void *ws, void *zero, size_t zero_bytes,
                            hipStream_t st);
int d2c_col_forward(const d2c_conv3d_desc &q, const void *col, int rows, const void *bias, void *out, void *ws, hipStream_t st);
bool d2c_grad_col_supported(const d2c_conv3d_desc &q);
size_t d2c_grad_col_gout_bytes(const d2c_conv3d_desc &q);
int d2c_brick_bwd_prepare(const d2c_conv3d_desc &q, const void *gout, const void *w, void *col_wt, void *col_gout, void *goutp, void *gb,
                          void *zero0, size_t zero0_bytes, void *zero1, size_t zero1_bytes, hipStream_t st);
int d2c_grad_col(const d2c_conv3d_desc &q, void *gcol, const void *wt, const void *gcl, hipStream_t st);
bool d2c_col_weight_use(const TiledShape &s, size_t scratch);
int d2c_col_weight(const TiledShape &s, const void *goutp, const void *col, long col_rows, void *gw, void *scratch, size_t scratch_bytes,
                   hipStream_t st);
int d2c_fwd_out_tile(const TiledShape &s);
template <typename T>
int d2c_tiled_fwd_launch(const TiledShape &s, const void *xcl, const void *off, const void *mask, const void *wp,
                         const void *bias, void *out, float *outacc, hipStream_t st, void *col = nullptr);
bool d2c_fwd_writes_columns(const TiledShape &s, int dtype);
long d2c_columns_rows(const TiledShape &s);
bool d2c_fwd_use_dma(const TiledShape &s);
size_t d2c_fwd_split_count_bytes(const TiledShape &s);
size_t d2c_fwd_split_bytes(const TiledShape &s);

bool d2c_tiled_bwd_data_supported(const TiledShape &s, int dtype);
bool d2c_tiled_bwd_weight_supported(const TiledShape &s, int dtype);
int d2c_bwd_ogk(int og, int dtype);
int d2c_bwd_pass_channels(int dtype);
bool d2c_tiled_bwd_single_pass(const TiledShape &s, int dtype);
template <typename T>
int d2c_tiled_bwd_data_launch(const TiledShape &s, const void *gout, const void *xcl, const void *off,
                              const void *mask, const void *w, void *wt, float *gxcl, void *gcolbuf, void *goff,
                              void *gmask, float *auxacc, hipStream_t st, int phase = 3, int g_lo = 0, int g_n = 0,
                              bool weights_packed = false);
bool d2c_bwd_sliceable(const TiledShape &s, int dtype);
int d2c_backward_slices();
int d2c_bwd_data_split(const TiledShape &s, int dtype);
template <typename T>
int d2c_gx_owner_launch(const TiledShape &s, const void *gcol, const SampleLists &L, float *gxcl, hipStream_t st,
                        int c_lo = 0, int c_n = 0);
void d2c_lists_ws(const TiledShape &s, int dtype, size_t *counts, size_t *entries, size_t *ovf);
SampleLists d2c_lists_make(const TiledShape &s, int dtype, void *counts, void *entries, void *ovf);
int d2c_lists_clear(const SampleLists &L, hipStream_t st);
bool d2c_lists_supported(const TiledShape &s);
int d2c_lists_build(const TiledShape &s, const void *off, const void *mask, const SampleLists &L, hipStream_t st);
int d2c_lists_fill(const TiledShape &s, const void *off, const void *mask, const SampleLists &L, hipStream_t st);
int d2c_gx_mode();
int d2c_col_weight_mode();
template <typename T>
int d2c_aux_grad_launch(const TiledShape &s, const void *xcl, const void *off, const void *mask, const void *gcol,
                        void *goff, void *gmask, const SampleLists *lists, void *col, bool col_in_place, hipStream_t st,
                        int g_lo = 0, int g_n = 0);
template <typename T>
int d2c_tiled_bwd_weight_launch(const TiledShape &s, const void *gout, const void *xcl, const void *off,
                                const void *mask, void *goutp, float *gwacc, void *gw, const void *col, long col_rows,
                                hipStream_t st, int phase = 7, int jp_lo = 0, int jp_n = 0);
bool d2c_bwd_weight_from_col(const TiledShape &s, int dtype);
bool d2c_bwd_weight_from_kept_col(const TiledShape &s, int dtype);
size_t d2c_bwd_col_bytes(const TiledShape &s, int dtype, int nchunks = 0);
size_t d2c_bwd_goutp_bytes(const TiledShape &s, int dtype);
template <typename T> int d2c_tiled_unpack_gx(const TiledShape &s, const float *gxcl, void *gx, hipStream_t st);
template <typename T> int d2c_tiled_bias_grad(const TiledShape &s, const void *gout, void *gb, hipStream_t st);

bool d2c_conv1d_bwd_use(const TiledShape &s, int dtype);
size_t d2c_conv1d_bwd_ws(const TiledShape &s, int dtype);
template <typename T>
int d2c_conv1d_bwd(const TiledShape &s, const void *gout, const void *x, const void *off, const void *mask, const void *w, void *gx,
                   void *goff, void *gmask, void *gw, void *gb, void *ws, hipStream_t st);
bool d2c_depthwise_supported(const TiledShape &s);
template <typename T>
int d2c_depthwise_forward(const TiledShape &s, const void *xcl, const void *off, const void *mask, const void *wt,
                          const void *bias, void *out, hipStream_t st);
template <typename T>
int d2c_dw_gx_owner_launch(const TiledShape &s, const void *goutcl, const void *wt, const SampleLists &L, float *gxcl,
                           hipStream_t st);
template <typename T>
int d2c_depthwise_backward(const TiledShape &s, const void *goutcl, const void *xcl, const void *off, const void *mask,
                           const void *wt, float *gxcl, void *goff, void *gmask, float *auxacc, float *gwacc, void *gw,
                           hipStream_t st);

static bool mfma_channels_ok(const d2c_conv3d_desc &q);

namespace {

inline int vec_of(int dtype) { return dtype == D2C_BF16 ? 8 : 4; }
inline int bkc_of(int dtype) { return 8 * vec_of(dtype); }

// The 1-D operator as a 3-D problem on a 1 x 1 x L volume with a 1 x 1 x k kernel.
d2c_conv3d_desc as_3d(const d2c_conv1d_desc &q)
{
    d2c_conv3d_desc r;
    r.N = q.N; r.Cin = q.Cin; r.Cout = q.Cout; r.D = 1; r.H = 1; r.W = q.L;
    r.kd = 1; r.kh = 1; r.kw = q.k; r.sd = 1; r.sh = 1; r.sw = q.s; r.pd = 0; r.ph = 0; r.pw = q.p;
    r.dd = 1; r.dh = 1; r.dw = q.d; r.groups = q.groups; r.offset_groups = q.offset_groups;
    r.Do = 1; r.Ho = 1; r.Wo = q.Lo; r.dtype = q.dtype; r.aux_dtype = q.aux_dtype;
    r.epilogue = D2C_EPILOGUE_NONE; r.epilogue_scale = 1.f; r.offset_axes = 0; r.backward_flags = 0;
    r.deform_channels = 0; r.mask_activation = D2C_MASK_ACT_NONE;
    return r;
}

TiledShape tiled_shape(const d2c_conv3d_desc &q, int nd = 3, int quirks = 0, const d2c_size_map_desc *sz = nullptr)
{
    TiledShape s;
    s.ss.on = sz ? 1 : 0;
    s.ss.mode = sz ? sz->mode : 0;
    s.ss.act = sz ? sz->activation : 0;
    for (int i = 0; i < D2C_SIZE_MAX_K; i++) {
        s.ss.base[0][i] = sz ? sz->base_z[i] : 0.f;
        s.ss.base[1][i] = sz ? sz->base_y[i] : 0.f;
        s.ss.base[2][i] = sz ? sz->base_x[i] : 0.f;
    }
    s.nd = nd; s.quirks = quirks;
    s.N = q.N; s.Cin = q.Cin; s.Cout = q.Cout; s.D = q.D; s.H = q.H; s.W = q.W;
    s.K = q.kd * q.kh * q.kw; s.G = q.offset_groups; s.groups = q.groups;
    s.Do = q.Do; s.Ho = q.Ho; s.Wo = q.Wo;
    s.cg = q.Cin / q.groups; s.og = q.Cout / q.groups; s.cpg = q.Cin / q.offset_groups;
    s.nchunk = s.cg / bkc_of(q.dtype);
    s.bkc = bkc_of(q.dtype);
    s.cpc = (s.cg < s.cpg ? s.cg : s.cpg) / s.bkc;
    s.adt = q.aux_dtype;
    s.act = q.epilogue; s.act_scale = q.epilogue_scale;
    s.P = q.Do * q.Ho * q.Wo; s.vol = q.D * q.H * q.W; s.M = q.N * s.P;
    s.axes = (nd == 3 && (q.offset_axes & 7)) ? (q.offset_axes & 7) : 7;
    s.keep = 0xffu;
    if (!(s.axes & 1)) s.keep &= 0x0fu;     // z fixed: dz = 0 corners
    if (!(s.axes & 2)) s.keep &= 0x33u;     // y fixed: dy = 0
    if (!(s.axes & 4)) s.keep &= 0x55u;     // x fixed: dx = 0
    s.dP = make_fastdiv(s.P); s.dHW = make_fastdiv(q.Ho * q.Wo); s.dW = make_fastdiv(q.Wo);
    // samples of the offsets (or the size map) and of the mask: tensors of their own, or both inside the layer's
    // deformation tensor of `deform_channels` channels
    s.obs = q.deform_channels > 0 ? (long)q.deform_channels * s.P
                                  : (sz ? (long)mode_channels(sz->mode) * s.P : (long)s.G * s.K * (nd == 3 ? 3 : 1) * s.P);
    s.mbs = q.deform_channels > 0 ? (long)q.deform_channels * s.P : (long)s.G * s.K * s.P;
    s.mact = q.mask_activation;
    // float problems: 1 = every backward matrix kernel on two-term bfloat16 operands (asked for in the description),
    // 2 = the grad-column product alone, like the forward kernels (the default: every tolerance gate stays green)
    s.f32split = q.dtype != D2C_F32 ? 0 : ((q.backward_flags & D2C_BWD_F32_SPLIT) ? 1 : (kF32SplitFwd ? 2 : 0));
    s.geo = make_geom(q);
    const int nt = d2c_fwd_out_tile(s);                   // (of all that is filled in above)
    s.ogp = (s.og + nt - 1) / nt * nt;
    return s;
}

// The tiled kernels let dead corners read a 256-byte row of zeros that follows the channels-last input; the first
// workgroup of the pack kernel writes it (the batch size is the grid's z extent; C is a multiple of the channel
// chunk there, so the row is 128-byte aligned).
template <typename T> D2C_DEV void pack_zero_row(T *xcl, int C, int vol, int zero_row)
{
    if (zero_row && blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0 && threadIdx.x < 64)
        reinterpret_cast<unsigned *>(xcl + (long)gridDim.z * C * vol)[threadIdx.x] = 0u;
}

// x [C][vol] -> xcl [vol][C] of one batch element: a 32 x 32 element tile through LDS
template <typename T> D2C_DEV void pack_tile32(const T *xb, T *ob, int C, int vol, int v0, int c0)
{
    __shared__ T tile[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
    for (int i = 0; i < 32; i += 8) {
        const int c = c0 + ty + i, v = v0 + tx;
        if (c < C && v < vol) tile[ty + i][tx] = xb[(long)c * vol + v];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32; i += 8) {
        const int v = v0 + ty + i, c = c0 + tx;
        if (c < C && v < vol) ob[(long)v * C + c] = tile[tx][ty + i];
    }
}

// The same for bfloat16 with 16-byte accesses on both sides (2-byte accesses of 32 lanes move 64 bytes per
// request): a 64 x 64 element tile; needs C to be a multiple of 8 and a 16-byte aligned `ob`.
D2C_DEV void pack_tile64_bf16(const bf16_t *xb, bf16_t *ob, int C, int vol, int v0, int c0)
{
    constexpr int RS = 66;                             // LDS row stride in elements (33 words)
    __shared__ bf16_t tile[64 * RS];                   // [v][c]
    for (int i = threadIdx.x; i < 512; i += 256) {     // 64 channels x 8 vectors of 8 positions
        const int c = c0 + i / 8, v = v0 + (i % 8) * 8;
        if (c < C && v < vol) {
            const uint4 q = load_run<bf16_t>(xb + (long)c * vol + v, vol - v);
            const unsigned u[4] = {q.x, q.y, q.z, q.w};
            bf16_t *t = tile + ((i % 8) * 8) * RS + i / 8;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                t[(2 * e) * RS] = (bf16_t)(u[e] & 0xffffu);
                t[(2 * e + 1) * RS] = (bf16_t)(u[e] >> 16);
            }
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 512; i += 256) {     // 64 positions x 8 vectors of 8 channels
        const int v = v0 + i / 8, c = c0 + (i % 8) * 8;
        if (c < C && v < vol) {
            const unsigned *t = reinterpret_cast<const unsigned *>(tile + (i / 8) * RS + (i % 8) * 8);
            *reinterpret_cast<uint4 *>(ob + (long)v * C + c) = make_uint4(t[0], t[1], t[2], t[3]);
        }
    }
}

// x [N][C][vol] -> xcl [N][vol][C]
template <typename T>
__global__ void __launch_bounds__(256) pack_input_kernel(const T *x, T *xcl, int C, int vol, int zero_row)
{
    pack_zero_row(xcl, C, vol, zero_row);
    const long bo = (long)blockIdx.z * C * vol;
    pack_tile32<T>(x + bo, xcl + bo, C, vol, blockIdx.x * 32, blockIdx.y * 32);
}

__global__ void __launch_bounds__(256) pack_input_bf16_kernel(const bf16_t *x, bf16_t *xcl, int C, int vol, int zero_row)
{
    pack_zero_row(xcl, C, vol, zero_row);
    const long bo = (long)blockIdx.z * C * vol;
    pack_tile64_bf16(x + bo, xcl + bo, C, vol, blockIdx.x * 64, blockIdx.y * 64);
}

// Forward weight operand in MFMA fragment order:
//   wp[wg][step = chunk*K + k][o-block of 32][k-group][lane] = 16 bytes =
//   W[wg*og + ob*32 + lane%32][chunk*BKC + (2*kg + lane/32)*VEC + 0..VEC-1][k]
// (rows past og are zero), so a wavefront's fragment load is 1 KiB contiguous.
template <typename T> D2C_DEV void pack_weight_fwd(const T *w, T *wp, const TiledShape &s, int b, int nb)
{
    constexpr int VEC = Elem<T>::VEC, BKC = 8 * VEC;
    const int OBT = s.ogp / 32, S = s.nchunk * s.K;
    const long total = (long)s.groups * S * OBT * 4 * 64;
    for (long i = (long)b * 256 + threadIdx.x; i < total; i += (long)nb * 256) {
        const int lane = (int)(i & 63);
        const int kg = (int)((i >> 6) & 3);
        long r = i >> 8;
        const int obg = (int)(r % OBT); r /= OBT;
        const int st = (int)(r % S);
        const int wg = (int)(r / S);
        const int j = st / s.K, k = st - j * s.K;
        const int ol = obg * 32 + (lane & 31);
        const int ch = j * BKC + (2 * kg + (lane >> 5)) * VEC;
        alignas(16) T tmp[VEC];
#pragma unroll
        for (int e = 0; e < VEC; e++)
            tmp[e] = ol < s.og ? w[((long)(wg * s.og + ol) * s.cg + ch + e) * s.K + k] : (T)0;
        *reinterpret_cast<uint4 *>(wp + i * VEC) = operand_vec<T, kF32SplitFwd>(tmp);
    }
}

// The same re-layout through LDS: a workgroup takes kPackRows output channels of one channel chunk, whose
// weights are runs of BKC * K consecutive elements in W, reads them with 16-byte loads and writes whole
// 16-byte fragment vectors (kPackRows consecutive lanes each).  Needs a 16-byte aligned W and rows that fit LDS.
constexpr int kPackRows = 8;
template <typename T> D2C_DEV void pack_weight_fwd_lds(const T *w, T *wp, const TiledShape &s, int b, unsigned char *smem)
{
    constexpr int VEC = Elem<T>::VEC, BKC = 8 * VEC, R = kPackRows;
    const int OBT = s.ogp / 32, S = s.nchunk * s.K;
    const int part = b % (32 / R); b /= 32 / R;
    const int obg = b % OBT; b /= OBT;
    const int j = b % s.nchunk;
    const int wg = b / s.nchunk;
    const int run = BKC * s.K;                       // elements of a row
    const int rs = run * (int)sizeof(T) + 4;         // LDS row stride in bytes (an odd number of banks)
    const int ol0 = obg * 32 + part * R;
    const int vpr = run * (int)sizeof(T) / 16;       // 16-byte vectors of a row
    for (int i = threadIdx.x; i < R * vpr; i += 256) {
        const int r = i / vpr, v = i - r * vpr;
        const int ol = ol0 + r;
        uint4 val = make_uint4(0, 0, 0, 0);
        if (ol < s.og)
            val = *reinterpret_cast<const uint4 *>(
                reinterpret_cast<const char *>(w + ((long)(wg * s.og + ol) * s.cg + j * BKC) * s.K) + (size_t)v * 16);
        unsigned *d = reinterpret_cast<unsigned *>(smem + r * rs + v * 16);
        d[0] = val.x; d[1] = val.y; d[2] = val.z; d[3] = val.w;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < s.K * 8 * R; i += 256) {
        const int r = i % R, q = i / R;
        const int khi = q & 7, k = q >> 3;           // khi = 2 * k-group + lane / 32
        const T *src = reinterpret_cast<const T *>(smem + r * rs) + khi * VEC * s.K + k;
        alignas(16) T tmp[VEC];
#pragma unroll
        for (int e = 0; e < VEC; e++) tmp[e] = src[e * s.K];
        const int lane = (khi & 1) * 32 + part * R + r;
        const long vi = ((((long)wg * S + j * s.K + k) * OBT + obg) * 4 + (khi >> 1)) * 64 + lane;
        *reinterpret_cast<uint4 *>(wp + vi * VEC) = operand_vec<T, kF32SplitFwd>(tmp);
    }
}

// What a call needs before its main kernels, as one launch: up to two tensors to channels-last (the input, grad_out) with
// zeros behind the first, the weights in the order of the kernels behind, a range of the workspace cleared, the bias
// gradient.  A workgroup finds its job from its index; jobs a call does not need have no workgroups.  (Each of these as
// a kernel of its own costs 2 - 3 us of launch and drain: 64 -> 64 channels on 4x14x25, float32, 37 us in five launches.)
enum { PREP_W_DEPTHWISE, PREP_W_FWD, PREP_W_FWD_LDS };
struct PrepArgs {
    struct Pack {
        const void *src;
        void *dst;
        int C, vol, wide;     // wide: 64 x 64 tiles (see pack_tile64_bf16, transpose_tile64)
        int nbx, nby, nblk;   // tiles along vol and C; workgroups of the job (tiles x batch)
    } pack[2];
    uint32_t *zrow;            // zeros behind the channels-last input
    int zrow_words;
    const void *w;
    void *wt;
    int wkind, wC, wK, nblk_w;
    struct Zero {
        uint32_t *p;
        size_t words;
        int nblk;
    } zero[3];
    const void *gout;          // bias gradient: one workgroup per channel
    void *gb;
    int bN, bC, bP, nblk_b;
    size_t lds;
    TiledShape s;
};
// WIDE: with large float32 tiles (a kernel of its own: their code costs a small call 1 %)
template <typename T, bool WIDE> __global__ void __launch_bounds__(256) prepare_kernel(PrepArgs a)
{
    extern __shared__ __align__(16) unsigned char smem[];
    int b = blockIdx.x;
    if (b == 0 && (int)threadIdx.x < a.zrow_words)
        for (int i = threadIdx.x; i < a.zrow_words; i += 256) a.zrow[i] = 0u;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const PrepArgs::Pack &pk = a.pack[j];
        if (b < pk.nblk) {
            const int bx = b % pk.nbx, by = (b / pk.nbx) % pk.nby;
            const long bo = (long)(b / (pk.nbx * pk.nby)) * pk.C * pk.vol;
            if constexpr (sizeof(T) == 2) {
                if (pk.wide) {
                    pack_tile64_bf16((const bf16_t *)pk.src + bo, (bf16_t *)pk.dst + bo, pk.C, pk.vol, bx * 64, by * 64);
                    return;
                }
            } else if constexpr (WIDE) if (pk.wide) {
                transpose_tile64((float *)smem, (const float *)pk.src + bo, (float *)pk.dst + bo, pk.C, pk.vol, by * 64, bx * 64);
                return;
            }
            pack_tile32<T>((const T *)pk.src + bo, (T *)pk.dst + bo, pk.C, pk.vol, bx * 32, by * 32);
            return;
        }
        b -= pk.nblk;
    }
    if (b < a.nblk_w) {
        const T *w = (const T *)a.w;
        T *wt = (T *)a.wt;
        if (a.wkind == PREP_W_DEPTHWISE) {
            const int n = a.wC * a.wK;
            for (int i = b * 256 + threadIdx.x; i < n; i += a.nblk_w * 256) wt[i] = w[(i % a.wC) * a.wK + i / a.wC];
        } else if (a.wkind == PREP_W_FWD) pack_weight_fwd<T>(w, wt, a.s, b, a.nblk_w);
        else pack_weight_fwd_lds<T>(w, wt, a.s, b, smem);
        return;
    }
    b -= a.nblk_w;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const PrepArgs::Zero &z = a.zero[j];
        if (b < z.nblk) {
            for (size_t i = (size_t)b * 256 + threadIdx.x; i < z.words; i += (size_t)z.nblk * 256) z.p[i] = 0u;
            return;
        }
        b -= z.nblk;
    }
    if (b < a.nblk_b) bias_grad_body<T, 256>((const T *)a.gout, (T *)a.gb, a.bN, a.bC, a.bP, b);
}

// Size-map source, backward: fp32 sums per axis [N][3][P] -> gradient of the raw size prediction [N][channels][P]
// (the axes a channel feeds add up; times the derivative of the size activation), in the storage type of the map.
template <bool AUX16>
__global__ void __launch_bounds__(256) size_grad_finish_kernel(TiledShape s, const float *acc, const void *raw, void *graw)
{
    const int nc = mode_channels(s.ss.mode);
    const long total = (long)s.N * s.P;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const long n = i / s.P, p = i - n * s.P;
        for (int c = 0; c < nc; c++) {
            float v = 0.f;
#pragma unroll
            for (int ax = 0; ax < 3; ax++)
                if (axis_channel(s.ss.mode, ax) == c) v += acc[(n * 3 + ax) * s.P + p];
            const long ri = n * s.obs + (long)c * s.P + p;
            v *= size_act_grad(s.ss.act, ld_auxT<AUX16>(raw, ri));
            if constexpr (AUX16) reinterpret_cast<bf16_t *>(graw)[ri] = f32_to_bf16(v);
            else reinterpret_cast<float *>(graw)[ri] = v;
        }
    }
}

// Size-map source, backward: raw map -> (size - 1) per axis as float [N][3][P] (0 for an axis the mode does not
// predict), once per call: the kernels of the backward pass form a tap's offsets from it per (tile, tap).
template <bool AUX16>
__global__ void __launch_bounds__(256) size_minus_one_kernel(TiledShape s, const void *raw, float *sm1)
{
    const long total = (long)s.N * s.P;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const long n = i / s.P, p = i - n * s.P;
        float c[3];
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {
            const int ch = axis_channel(s.ss.mode, ax);
            c[ax] = ch < 0 ? 0.f : ld_auxT<AUX16>(raw, n * s.obs + (long)ch * s.P + p);
        }
        size_minus_one<AUX16>(s, c);
#pragma unroll
        for (int ax = 0; ax < 3; ax++) sm1[(n * 3 + ax) * s.P + p] = c[ax];
    }
}

struct FwdWs {
    size_t xcl, wp, outacc;
    size_t least;                   // what the gathering kernels need
    size_t gemm, lists, col, end;   // forward over sampled columns: operands of the product, sorted points, columns
    size_t keep;                    // ... in a call that holds input, points and columns in the caller's buffer: those operands, in front
    size_t total;                   // what the call is fastest with
};
bool use_brick_forward(const d2c_conv3d_desc &q, const TiledShape &s, bool kept);
// columns; and what a forward call can leave for its backward call: behind them the sorted points, then the input channels-last
size_t brick_col_bytes(const TiledShape &s) { return (size_t)(s.Cin / 64) * s.K * d2c_columns_rows(s) * 128; }
size_t brick_keep_input(const TiledShape &s) { return brick_col_bytes(s) + d2c_brick_ws(s).total; }
size_t brick_keep_bytes(const TiledShape &s) { return brick_keep_input(s) + d2c_align_up((size_t)s.N * s.vol * s.Cin * 2 + 256); }
// Caller-held prepared region (d2c_conv3d_prepared_bytes): channels-last input + zero row | forward weights in
// fragment order | backward weights transposed per step (single-pass reductions only)
struct PreparedLayout {
    size_t xcl, wp, wt, wt_bytes, total;
};
FwdWs fwd_ws(const d2c_conv3d_desc &q, const TiledShape &s)
{
    const size_t es = d2c_elem_size(q.dtype);
    FwdWs w{};
    w.xcl = 0;
    w.wp = d2c_align_up((size_t)s.N * s.vol * s.Cin * es + 256);   // input, then a 256-byte row of zeros
    w.outacc = w.wp + d2c_align_up((size_t)s.groups * s.nchunk * s.K * s.ogp * bkc_of(q.dtype) * es);
    // fp32 partial sums of the output for the work items whose steps the DMA-gather kernel shares out: whole tiles of
    // 64 positions x padded output channels
    w.least = w.outacc;
    if (d2c_fwd_use_dma(s)) w.least += d2c_align_up((size_t)((s.M + 63) / 64 * 64) * s.ogp * s.groups * sizeof(float));
    w.total = w.least + d2c_fwd_split_bytes(s);      // (the kernel of the small problems: fastest with its steps split)
    const bool plain = use_brick_forward(q, s, false), keep = use_brick_forward(q, s, true);
    if (plain || keep) {
        w.gemm = w.wp;
        w.lists = w.gemm + d2c_align_up(d2c_col_forward_ws(q));
        w.col = w.lists + d2c_brick_ws(s).total;
        w.end = w.col + brick_col_bytes(s);
        if (plain) w.total = std::max(w.total, w.end);
        // (where the gathering kernel writes no columns, every forward workspace has to do for a call that keeps them)
        w.keep = w.lists - w.gemm;
        if (keep && !d2c_fwd_writes_columns(s, q.dtype)) w.total = std::max(w.total, w.keep);
    }
    return w;
}

PreparedLayout prepared_layout(const d2c_conv3d_desc &q, const TiledShape &s)
{
    const size_t es = d2c_elem_size(q.dtype);
    PreparedLayout p;
    p.xcl = 0;
    p.wp = d2c_align_up((size_t)s.N * s.vol * s.Cin * es + 256);
    p.wt = p.wp + d2c_align_up((size_t)s.groups * s.nchunk * s.K * s.ogp * bkc_of(q.dtype) * es);
    const int omax = d2c_bwd_pass_channels(q.dtype);
    p.wt_bytes = s.og <= omax ? d2c_align_up((size_t)s.groups * s.K * s.nchunk * bkc_of(q.dtype) * d2c_bwd_ogk(s.og, q.dtype) * es) : 0;
    p.total = p.wt + p.wt_bytes;
    return p;
}

template <typename T>
int pack_input(const TiledShape &s, const void *x, void *xcl, hipStream_t st, bool zero_row = false)
{
    dim3 grid((s.vol + 31) / 32, (s.Cin + 31) / 32, s.N);
    D2cProfScope prof(D2C_PROF_PACK, st);
    if constexpr (sizeof(T) == 2) {
        if (s.Cin % 8 == 0 && reinterpret_cast<uintptr_t>(xcl) % 16 == 0) {
            hipLaunchKernelGGL(pack_input_bf16_kernel, dim3((s.vol + 63) / 64, (s.Cin + 63) / 64, s.N), dim3(256), 0, st,
                               (const bf16_t *)x, (bf16_t *)xcl, s.Cin, s.vol, (int)zero_row);
            return d2c_check_launch("pack_input_bf16_kernel");
        }
    }
    hipLaunchKernelGGL(pack_input_kernel<T>, grid, dim3(256), 0, st, (const T *)x, (T *)xcl, s.Cin, s.vol, (int)zero_row);
    return d2c_check_launch("pack_input_kernel");
}

// The jobs of prepare_kernel.
template <typename T> void prep_pack(PrepArgs::Pack &pk, const void *src, void *dst, int N, int C, int vol)
{
    pk.src = src; pk.dst = dst; pk.C = C; pk.vol = vol;
    constexpr int V = 16 / (int)sizeof(T);
    pk.wide = C % V == 0 && reinterpret_cast<uintptr_t>(dst) % 16 == 0;
    // (float32: where large tiles give every compute unit one; below, the small ones are no slower and their kernel holds less code:
    // 64 x 1400 elements 18.3 us, 18.1 of a forward call)
    if (sizeof(T) == 4 && (long)((vol + 63) / 64) * ((C + 63) / 64) * N < 256) pk.wide = 0;
    const int tl = pk.wide ? 64 : 32;
    pk.nbx = (vol + tl - 1) / tl; pk.nby = (C + tl - 1) / tl;
    pk.nblk = pk.nbx * pk.nby * N;
}
void prep_zero(PrepArgs &a, int j, void *p, size_t bytes)
{
    a.zero[j] = PrepArgs::Zero{(uint32_t *)p, bytes / 4, (int)std::min<size_t>((bytes / 4 + 1023) / 1024, 2048)};
}
template <typename T> void prep_weight_fwd(PrepArgs &a, const TiledShape &s, const void *w, void *wp)
{
    a.s = s; a.w = w; a.wt = wp;
    const size_t lds = (size_t)kPackRows * ((size_t)s.bkc * s.K * sizeof(T) + 4);
    if (lds <= 48 * 1024 && reinterpret_cast<uintptr_t>(w) % 16 == 0) {
        a.wkind = PREP_W_FWD_LDS; a.lds = lds;
        a.nblk_w = s.groups * s.nchunk * (s.ogp / 32) * (32 / kPackRows);
    } else {
        a.wkind = PREP_W_FWD;
        a.nblk_w = (int)std::min<long>(((long)s.groups * s.nchunk * s.K * (s.ogp / 32) * 4 * 64 + 255) / 256, 8192);
    }
}
template <typename T> int prep_launch(const PrepArgs &a, hipStream_t st)
{
    const long nblk = (long)a.pack[0].nblk + a.pack[1].nblk + a.nblk_w + a.zero[0].nblk + a.zero[1].nblk + a.zero[2].nblk + a.nblk_b;
    if (nblk == 0) return D2C_OK;
    D2cProfScope prof(D2C_PROF_PACK, st);
    const bool wide = sizeof(T) == 4 && (a.pack[0].wide || a.pack[1].wide);
    auto kern = wide ? &prepare_kernel<T, sizeof(T) == 4> : &prepare_kernel<T, false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(256), wide ? std::max<size_t>(a.lds, kTransposeLds) : a.lds, st, a);
    return d2c_check_launch("prepare_kernel");
}
// ... for a depthwise call (gout == nullptr: no grad_out copy; zero_bytes == 0: nothing to clear; gb == nullptr: no
// bias gradient)
template <typename T>
int dw_prepare(const TiledShape &s, const void *x, void *xcl, const void *gout, void *goutcl, const void *w, void *wt,
               void *zero, size_t zero_bytes, void *gb, hipStream_t st)
{
    PrepArgs a{};
    prep_pack<T>(a.pack[0], x, xcl, s.N, s.Cin, s.vol);
    if (gout) prep_pack<T>(a.pack[1], gout, goutcl, s.N, s.Cout, s.P);
    a.wkind = PREP_W_DEPTHWISE; a.w = w; a.wt = wt; a.wC = s.Cin; a.wK = s.K;
    a.nblk_w = std::min((s.Cin * s.K + 255) / 256, 1024);
    a.zrow = (uint32_t *)((T *)xcl + (size_t)s.N * s.vol * s.Cin); a.zrow_words = s.Cin * (int)sizeof(T) / 4;
    prep_zero(a, 0, zero, zero_bytes);
    a.gout = gout; a.gb = gb; a.bN = s.N; a.bC = s.Cout; a.bP = s.P;
    a.nblk_b = (gb && gout) ? s.Cout : 0;
    return prep_launch<T>(a, st);
}

bool is_depthwise(const d2c_conv3d_desc &q)
{
    if (q.dtype != D2C_BF16 && q.dtype != D2C_F32) return false;
    return q.groups == q.Cin && q.Cout == q.Cin && q.Cin > 1 && d2c_depthwise_supported(tiled_shape(q));
}

// depthwise workspace: channels-last input + one row of zeros | weights [K][C] | grad_input accumulator | grad_weight accumulator |
// channels-last grad_out | sample lists (bucket counts, buckets of 32-byte entries, overflow array)
struct DwWs {
    size_t xcl, wt, gxcl, gwacc, auxacc, goutcl, counts, entries, ovf, total_fwd, total_bwd;
};
DwWs dw_ws(const d2c_conv3d_desc &q, const TiledShape &s)
{
    const size_t es = d2c_elem_size(q.dtype);
    DwWs w;
    w.xcl = 0;
    w.wt = d2c_align_up(((size_t)s.N * s.vol + 1) * s.Cin * es);   // input, then a row of zeros
    w.total_fwd = w.wt + d2c_align_up((size_t)s.K * s.Cin * es);
    w.gxcl = w.total_fwd;
    w.gwacc = w.gxcl + d2c_align_up((size_t)s.N * s.vol * s.Cin * sizeof(float));
    w.auxacc = w.gwacc + d2c_align_up((size_t)s.K * s.Cin * sizeof(float));
    // (grad_weight sums, offset / mask gradient sums and bucket counts follow each other: one clear)
    size_t c, en, ov;
    d2c_lists_ws(s, D2C_F32, &c, &en, &ov);      // (32-byte entries whatever the element type)
    w.counts = w.auxacc + d2c_align_up((size_t)s.N * s.G * s.K * s.P * 4 * sizeof(float));
    w.goutcl = w.counts + c;
    w.entries = w.goutcl + d2c_align_up((size_t)s.N * s.P * s.Cout * es);
    w.ovf = w.entries + en;
    w.total_bwd = w.ovf + ov;
    return w;
}

template <typename T>
int forward_t(const d2c_conv3d_desc &q, const void *x, const void *off, const void *mask, const void *w,
              const void *bias, void *out, void *ws, hipStream_t st, int nd = 3, const d2c_size_map_desc *sz = nullptr,
              const D2cPrepared *prep = nullptr, void *columns = nullptr, size_t columns_bytes = 0,
              size_t ws_bytes = 0)
{
    const TiledShape s = tiled_shape(q, nd, 0, sz);
    char *base = (char *)ws;
    if (nd == 3 && is_depthwise(q)) {
        const DwWs d = dw_ws(q, s);
        if (int rc = dw_prepare<T>(s, x, base + d.xcl, nullptr, nullptr, w, base + d.wt, nullptr, 0, nullptr, st)) return rc;
        return d2c_depthwise_forward<T>(s, base + d.xcl, off, mask, base + d.wt, bias, out, st);
    }
    const FwdWs l = fwd_ws(q, s);
    // (a caller-held prepared region takes the place of the workspace's channels-last input and packed weights; what it
    // already holds from an earlier call is not made again)
    const PreparedLayout pl = prepared_layout(q, s);
    char *xcl_p = prep ? (char *)prep->base + pl.xcl : base + l.xcl;
    char *wp_p = prep ? (char *)prep->base + pl.wp : base + l.wp;
    const bool have_x = prep && (prep->reuse & D2C_REUSE_INPUT);
    if (nd == 3 && !prep && use_brick_forward(q, s, columns != nullptr)) {
        // sort the points, sample the columns (the caller's buffer, with the sorted points and the input behind them for its
        // backward call, or the workspace), multiply.  A smaller workspace: the gathering kernels, below.
        const bool keep = columns && columns_bytes >= brick_keep_bytes(s);
        const bool fits = ws_bytes >= (keep ? l.keep : (columns ? l.col : l.end));
        char *const gemm = base + (keep ? 0 : l.gemm);
        char *col = columns ? (char *)columns : base + l.col;
        char *lists = keep ? col + brick_col_bytes(s) : base + l.lists;
        if (keep) xcl_p = col + brick_keep_input(s);
        if (fits) {
            size_t zb;
            void *const zp = d2c_brick_zero(s, lists, &zb);
            if (int rc = d2c_col_forward_prepare(q, x, xcl_p, w, gemm, zp, zb, st)) return rc;
        }
        if (fits || keep)
            if (int rc = d2c_brick_sort(s, off, mask, lists, st, fits)) return rc;
        if (fits) {
            if (int rc = d2c_brick_columns(s, xcl_p, col, (int)d2c_columns_rows(s), lists, st)) return rc;
            return d2c_col_forward(q, col, (int)d2c_columns_rows(s), bias, out, gemm, st);
        }
    }
    // input, weights, and the counters of the steps' split (which needs its scratch: a smaller workspace goes without)
    PrepArgs pa{};
    if (!have_x) {
        prep_pack<T>(pa.pack[0], x, xcl_p, s.N, s.Cin, s.vol);
        pa.zrow = (uint32_t *)((T *)xcl_p + (size_t)s.N * s.vol * s.Cin); pa.zrow_words = 64;
    }
    if (!(prep && (prep->reuse & D2C_REUSE_FORWARD_WEIGHTS))) prep_weight_fwd<T>(pa, s, w, wp_p);
    const size_t split = d2c_fwd_split_bytes(s);
    const bool shared = d2c_fwd_use_dma(s) || (split && (nd != 3 || ws_bytes >= l.outacc + split));
    if (shared && split) prep_zero(pa, 0, base + l.outacc, d2c_fwd_split_count_bytes(s));
    if (int rc = prep_launch<T>(pa, st)) return rc;
    return d2c_tiled_fwd_launch<T>(s, xcl_p, off, mask, wp_p, bias, out, shared ? (float *)(base + l.outacc) : nullptr, st, columns);
}

// grad_input by sample lists (see d2c_invlist.hip): from whole grad-column rows, i.e. the reduction over all output
// channels of a weight group (in one pass of the product-only kernels, or in several whose rows are added up).
bool use_lists(const d2c_conv3d_desc &q, const TiledShape &s)
{
    return d2c_gx_mode() >= 1 && d2c_lists_supported(s) && d2c_tiled_bwd_data_supported(s, q.dtype) &&
           (s.nd == 3 || d2c_tiled_bwd_single_pass(s, q.dtype));
}

// grad_offset / grad_mask by the kernel of d2c_aux_grad.hip (from the grad-column rows).  (Weight groups wider than
// one pass of the grad-column product get whole rows too: the later passes over their output channels add to the
// rows, see d2c_tiled_bwd_data_launch.
// That needs the product-only kernels, i.e. grad_input from sample lists: where grad_input is scattered with
// atomics by the fused kernel, wide weight groups keep the fused kernel's passes.)
bool use_aux_kernel(const d2c_conv3d_desc &q, const TiledShape &s)
{
    if (!d2c_tiled_bwd_data_supported(s, q.dtype)) return false;
    // (1-D problems with wide weight groups keep the fused kernel: their float32 gradients are held to the literal
    // gate, which the two-term operands of the product-only kernel miss there)
    return d2c_tiled_bwd_single_pass(s, q.dtype) || (s.nd == 3 && d2c_gx_mode() >= 1 && d2c_lists_supported(s));
}

// grad_offset, grad_mask and grad_input from bricks of sorted points (d2c_brick.hip): wherever whole grad-column rows are
// at hand.  (A bucket capacity asked for by the test hook is a matter of the lists.)
bool use_brick(const d2c_conv3d_desc &q, const TiledShape &s)
{
    // (float32 weight groups that take several passes of the grad-column product: from 128 positions on.  Training steps without kept
    // columns, us, lists first: 64 -> 320 channels on 50 positions 136, 129; 144 152, 129; 504 177, 147; 256 -> 512 50 239, 201; 256 293, 242;
    // 512 -> 1024 50 579, 508; 256 729, 678; with kept columns 64 -> 320 on 12960 573, 531; 512 -> 1024 5765, 5331.  Fewer than two tiles of
    // positions stay with the lists, which cost them 5 - 20 %: test_wide_weight_groups_stay_on_the_list_based_backward holds 50 and 75 positions
    // to that way.)
    return d2c_gx_mode() == 1 && use_lists(q, s) && use_aux_kernel(q, s) && d2c_brick_supported(s, q.dtype) &&
           (q.dtype == D2C_BF16 || d2c_tiled_bwd_single_pass(s, q.dtype) || s.M >= 128);
}

// The forward pass over sampled columns: sort, sample, multiply.  `kept`: the caller keeps the columns, where the backward call can
// multiply over them, and that one takes the sorted points over.  Picoseconds per point and chunk of 64 channels, C columns: sort 60 / chunks of a
// group, sampling 33, product 0.13 C; the gathering kernel 55 + 0.15 C (192 - 512 columns).  So with the sort paid for by
// the backward pass the columns win throughout, without it from four chunks on.
// Small problems, where launches and half-filled rounds of tiles count, in us, gathering first (27 taps but for the last; the line lies
// where the columns stop losing):
//   training step:  128 -> 128: 405 positions 133, 140; 810 151, 145; 1296 176, 152; 5760 308, 190   128 -> 40: 810 132, 141; 1296 149, 138
//                   256 -> 64: 405 143, 144; 810 168, 153    256 -> 256: 5760 338, 288    1024 -> 256: 810 308, 288; 5760 772, 674
//   forward alone:  256 -> 256: 4000 75, 80; 5120 88, 85; 6912 120, 96    192 -> 192: 5120 71, 71; 6912 94, 81; 28800 247, 195
//                   512 -> 512: 1600 84, 85; 2560 106, 102; 4000 139, 129; in 2 groups 2560 105, 101; 6400 209, 180
//                   1024 -> 256: 1600 92, 106; 2560 129, 121; 4000 178, 154   128 -> 128: 28800 135, 139
//                   up to 128 output channels (the gathering kernel there is the one of the small problems): 256 -> 128: 6912 65, 83; 8880 105, 103;
//                   512 -> 64: 4000 61, 87; 5120 97, 95; 1024 -> 128: 2560 78, 102; 4000 130, 132
//                   7 taps: 256 -> 256: 5120 49, 52; 8880 64, 63    2048 -> 256: 3240 97, 101; 4000 111, 109
bool use_brick_forward(const d2c_conv3d_desc &q, const TiledShape &s, bool kept)
{
    const long chunks = s.Cin / 64, of_group = s.cpg / 64;
    const bool large = kept ? s.M >= 400 && s.M * chunks >= 2048
                            : (of_group >= 4 && s.M >= 4096 && s.M * of_group >= 32768) ||
                              (of_group >= 3 && s.K >= 27 && s.og > 128 && s.M >= 2560 && s.M * chunks >= 20480);
    return large && q.dtype == D2C_BF16 && use_brick(q, s) && s.groups == 1 && brick_col_bytes(s) < (4ull << 30) &&
           (!kept || d2c_bwd_weight_from_kept_col(s, q.dtype));
}

// grad_weight as a matrix product over sampled columns that the offset / mask gradient kernel writes on its way
// (needs that kernel to run: the caller wants grad_offset or grad_mask)
// (0 sample again, 1 columns in a buffer of their own, 2 columns over the grad-column rows: the description's
// backward_flags, or where those say nothing the process-wide test hook)
int gw_mode(const d2c_conv3d_desc &q)
{
    const int f = q.backward_flags & D2C_BWD_GW_MASK;
    return f == D2C_BWD_GW_DEFAULT ? d2c_col_weight_mode() : (f == D2C_BWD_GW_RESAMPLE ? 0 : f);
}
// Float32 problems that the bricks serve and that bring no columns have two ways: the bricks, which write none, and a second
// sampling for grad_weight; or the gathering kernels, which write columns, and the product over them.  The second sampling multiplies on
// the float32 instruction, in passes and tiles of 256 output channels, the product over whole sets of four chunks on the bfloat16 one; the
// bricks gain most where the points are few.  Training steps, bricks and second sampling / gathering and columns, us:
//   up to 128 output channels: 128 -> 64 on 2560 positions 1.05, 8192 1.23; 256 -> 128 1400 0.94, 3240 1.08, 12960 1.05; 1024 -> 128 1400 0.95, 3240 1.07
//   up to 256 (the tile is full): 256 -> 256 on 1400 254, 283; 5120 557, 571; 12960 1259, 1257; 64 -> 256 1400 153, 173; 25600 768, 798
//   more: 256 -> 512 on 504 270, 310; 1400 382, 392; 2560 516, 500; 12960 1940, 1793;  256 -> 1024 504 465, 474; 1008 576, 544; 12960 3994, 2985
//   offset groups, whose points are sorted each on its own: 512 -> 512, 8 groups, 256 369, 370; 504 427, 410; 12960 4078, 3340;
//   512 -> 128, 8 groups, 256 0.96, 784 1.11;  256 -> 128, 2 groups, 1008 0.96, 2000 1.09
//   fewer taps: 256 -> 256, 9, 5120 269, 299; 12960 504, 489;  7 5120 235, 278; 25600 766, 741
//   chunks that make no whole sets, on the float32 instruction both ways: 64 -> 64 on 5120 182, 192; 25600 602, 630;  320 -> 256 12960 0.94
bool columns_pay(const d2c_conv3d_desc &q, const TiledShape &s)
{
    const int pass = d2c_bwd_pass_channels(q.dtype);
    if (s.nchunk % 4 || (s.og > 128 && s.og <= pass)) return false;
    return (double)s.M * s.K * ((s.og + pass - 1) / pass) * (s.G / s.groups + 1) >= 150000.0;
}
bool use_col_weight(const d2c_conv3d_desc &q, const TiledShape &s)
{
    if (q.dtype != D2C_BF16 && (gw_mode(q) != 1 || ((q.backward_flags & D2C_BWD_GW_MASK) == D2C_BWD_GW_DEFAULT && use_brick(q, s) && !columns_pay(q, s))))
        return false;
    return gw_mode(q) && use_aux_kernel(q, s) && d2c_bwd_weight_from_col(s, q.dtype);
}
// ... written over the grad-column rows (mode 2): grad_input is taken from those rows first, from sample lists
// that a pass of their own files
// (bfloat16 only: float problems asked for it sample again, as they always did)
bool col_in_place(const d2c_conv3d_desc &q, const TiledShape &s)
{
    return gw_mode(q) == 2 && q.dtype == D2C_BF16 && use_col_weight(q, s);
}

// The backward pass slice by slice over the offset groups (see d2c_bwd_sliceable): `gs` groups per slice of the
// grad-column rows (0: not sliced), `cgs` groups per block of sampled columns that one launch of the grad-weight
// product takes (a multiple of gs that holds an even number of channel chunks).
struct BwdSlices {
    int gs, cgs;
};
BwdSlices bwd_slices(const d2c_conv3d_desc &q, const TiledShape &s)
{
    BwdSlices r{0, 0};
    // the description's backward_flags, or where those say nothing the process-wide test hook; by default the pass
    // is not sliced (one pass over all groups is the faster one: the grad_input kernel needs the parallelism of all
    // channel chunks at once)
    int n = (q.backward_flags >> 8) & 0xff;
    if (n == 0) n = d2c_backward_slices();
    if (n < 2 || gw_mode(q) == 2 || d2c_gx_mode() < 1 || s.ss.on || !d2c_bwd_sliceable(s, q.dtype) ||
        !d2c_tiled_bwd_data_supported(s, q.dtype) || !d2c_lists_supported(s))
        return r;
    if (n > s.G) n = s.G;
    r.gs = (s.G + n - 1) / n;
    r.cgs = ((r.gs * (s.cpg / 64)) % 2 == 0) ? r.gs : 2 * r.gs;
    return r;
}

// Whether a backward call runs on the bricks: not one slice by slice, and not one that writes its columns over the rows.
// `saved_columns`: the caller brings the sampled columns of the forward call (no column region, no slices).  `col_weight`: the call
// would multiply over columns of its own if there were any (it wants grad_weight, and grad_offset or grad_mask)
bool brick_backward(const d2c_conv3d_desc &q, const TiledShape &s, bool saved_columns, bool col_weight = true)
{
    if (!use_brick(q, s)) return false;
    if (saved_columns) return true;
    // (float32 columns come from the gathering kernel)
    return gw_mode(q) != 2 && bwd_slices(q, s).gs == 0 && !(q.dtype == D2C_F32 && col_weight && use_col_weight(q, s));
}

// grad_weight by col_weight_kernel, its sums in the place of the grad-column rows: where there are columns.  (The rows' place has room for
// at least as much as `gwacc`.)
size_t grad_rows_bytes(const d2c_conv3d_desc &q, const TiledShape &s) { return (size_t)s.Cin * s.K * s.M * d2c_elem_size(q.dtype); }
bool use_wide_weight(const d2c_conv3d_desc &q, const TiledShape &s, bool brick)
{
    return brick && q.dtype == D2C_BF16 && s.groups == 1 && d2c_col_weight_use(s, grad_rows_bytes(q, s));
}

struct BwdWs {
    size_t xcl, wt, gxcl, gwacc, goutp, auxacc, gcol, counts, entries, ovf, gsacc, sm1, brick, res, gcl, col, least, total;
};
// `sorted`: ... and the sorted points and the input behind them
BwdWs bwd_ws(const d2c_conv3d_desc &q, const TiledShape &s, bool saved_columns = false, bool sorted = false, bool col_weight = true)
{
    const bool brick = brick_backward(q, s, saved_columns, col_weight);
    const size_t es = d2c_elem_size(q.dtype);
    const bool wide = use_wide_weight(q, s, brick);
    BwdWs w;
    w.xcl = 0;
    w.wt = sorted ? 0 : d2c_align_up((size_t)s.N * s.vol * s.Cin * es + 256);   // input, then a 256-byte row of zeros
    const int omax = d2c_bwd_pass_channels(q.dtype);
    const int ogk = d2c_bwd_ogk(s.og < omax ? s.og : omax, q.dtype);
    w.gxcl = w.wt + d2c_align_up((size_t)s.groups * s.K * s.nchunk * bkc_of(q.dtype) * ogk * es);
    w.gwacc = w.gxcl + d2c_align_up((size_t)s.N * s.vol * s.Cin * sizeof(float));
    w.goutp = w.gwacc + (wide ? 0 : d2c_align_up((size_t)s.Cout * s.cg * s.K * sizeof(float)));
    w.auxacc = w.goutp + d2c_align_up(d2c_bwd_goutp_bytes(s, q.dtype));
    // fp32 scratch of the offset / mask gradient, used when the data kernel splits its steps or reduces the output
    // channels in several passes (the partial sums then add up in fp32, whatever the storage type of the result)
    w.total = w.auxacc;
    if (d2c_bwd_data_split(s, q.dtype) > 1 || !d2c_tiled_bwd_single_pass(s, q.dtype))
        w.total += d2c_align_up((size_t)s.N * s.G * s.K * s.P * (s.nd + 1) * sizeof(float));
    w.gcol = w.counts = w.entries = w.ovf = 0;
    const BwdSlices sl = saved_columns ? BwdSlices{0, 0} : bwd_slices(q, s);
    if (use_lists(q, s) || use_aux_kernel(q, s)) {
        w.gcol = w.total;
        // (+ 64 rows behind the last one: what the last tile of the grad-weight product reads when the columns took
        // the rows' place)
        const size_t chunks = sl.gs ? (size_t)sl.gs * (s.cpg / bkc_of(q.dtype)) : (size_t)(s.Cin / bkc_of(q.dtype));
        w.total = w.gcol + d2c_align_up((chunks * s.K * s.M + 64) * bkc_of(q.dtype) * es);
        // (calls that bring no columns, or want no other gradient, add grad_weight up once the rows are done with, or were not made)
        if (wide) w.gwacc = w.gcol;
    }
    if (use_lists(q, s) && !brick) {
        size_t c, en, ov;
        d2c_lists_ws(s, q.dtype, &c, &en, &ov);
        w.counts = w.total;
        w.entries = w.counts + c;
        w.ovf = w.entries + en;
        w.total = w.ovf + ov;
    }
    // size-map source: fp32 sums of the size gradient per axis
    w.gsacc = w.total;
    if (s.ss.on) w.total += d2c_align_up((size_t)s.N * 3 * s.P * sizeof(float));
    w.sm1 = w.total;       // ... and (size - 1) per axis
    if (s.ss.on) w.total += d2c_align_up((size_t)s.N * 3 * s.P * sizeof(float));
    w.brick = w.total;     // sorted points
    if (brick && !sorted) w.total += d2c_brick_ws(s).total;
    w.res = w.total;       // ... and sums per point
    if (brick) w.total += d2c_brick_ws(s).res_bytes;
    w.col = w.total;       // sampled columns for the grad-weight product
    if (!saved_columns && col_weight && use_col_weight(q, s) && !col_in_place(q, s))
        w.total += d2c_align_up(d2c_bwd_col_bytes(s, q.dtype, sl.cgs ? sl.cgs * (s.cpg / 64) : 0));
    // Operands of grad_col_kernel: the weights in the place of `wt`, grad_out in that of the sums per point and the columns, which are
    // written later.  Where it takes more than those have, a call with less workspace runs without, on tiled_bwd_col32_kernel.
    w.gcl = w.res;
    w.least = w.total;
    if (brick && d2c_grad_col_supported(q)) w.total = std::max(w.total, w.gcl + d2c_grad_col_gout_bytes(q));
    return w;
}

template <typename T>
int backward_t(const d2c_conv3d_desc &q, const void *gout, const void *x, const void *off, const void *mask,
               const void *w, void *gx, void *goff, void *gmask, void *gw, void *gb, void *ws, hipStream_t st,
               int nd = 3, int quirks = 0, const d2c_size_map_desc *sz = nullptr, const D2cPrepared *prep = nullptr,
               const void *columns = nullptr, size_t columns_bytes = 0, size_t ws_bytes = 0)
{
    TiledShape s = tiled_shape(q, nd, quirks, sz);
    char *base = (char *)ws;
    if (!mask) gmask = nullptr;
    const void *size_raw = off;   // (size-map source; `off` becomes the per-axis (size - 1) below)
    if (nd == 3 && is_depthwise(q)) {
        const DwWs d = dw_ws(q, s);
        float *gxcl = gx ? (float *)(base + d.gxcl) : nullptr;
        float *gwacc = gw ? (float *)(base + d.gwacc) : nullptr;
        const bool grads = gx || goff || gmask || gw;
        // one launch: input and grad_out channels-last ([N][P][C]), the weights [K][C], the clear of the grad_weight sums,
        // offset / mask gradient sums and bucket counts (which follow each other), the bias gradient
        if (!grads) return gb ? d2c_tiled_bias_grad<T>(s, gout, gb, st) : D2C_OK;
        if (int rc = dw_prepare<T>(s, x, base + d.xcl, gout, base + d.goutcl, w, base + d.wt,
                                   grads ? base + d.gwacc : nullptr, grads ? d.goutcl - d.gwacc : 0, gb, st))
            return rc;
        if (grads) {
            const bool lists = gx && d2c_gx_mode() >= 1 && d2c_lists_supported(s);
            SampleLists L{nullptr, nullptr, nullptr, 0, 0, 0};
            if (lists) {
                L = d2c_lists_make(s, D2C_F32, base + d.counts, base + d.entries, base + d.ovf);
                if (int rc = d2c_lists_fill(s, off, mask, L, st)) return rc;
            }
            if (goff || gmask || gw || !lists)
                if (int rc = d2c_depthwise_backward<T>(s, base + d.goutcl, base + d.xcl, off, mask, base + d.wt,
                                                      lists ? nullptr : gxcl, goff, gmask, (float *)(base + d.auxacc),
                                                      gwacc, gw, st))
                    return rc;
            if (lists)
                if (int rc = d2c_dw_gx_owner_launch<T>(s, base + d.goutcl, base + d.wt, L, gxcl, st)) return rc;
            if (gx)
                if (int rc = d2c_tiled_unpack_gx<T>(s, gxcl, gx, st)) return rc;
        }
        return D2C_OK;
    }
    // (kept columns of a forward call over sorted points: those follow the columns)
    const bool sorted = columns && use_brick_forward(q, s, true) && columns_bytes >= brick_keep_bytes(s);
    const bool col_weight = gw && (goff || gmask);
    const bool brick = nd == 3 && brick_backward(q, s, columns != nullptr, col_weight);
    const BwdWs l = bwd_ws(q, s, columns != nullptr, sorted, col_weight);
    const PreparedLayout pl = prepared_layout(q, s);
    // (a forward call over sorted points has left the input behind them)
    const bool have_x = (prep && (prep->reuse & D2C_REUSE_INPUT)) || (sorted && !prep);
    char *xcl_p = prep ? (char *)prep->base + pl.xcl : (sorted ? (char *)const_cast<void *>(columns) + brick_keep_input(s) : base + l.xcl);
    // (the transposed weights of the region serve single-pass reductions; wider weight groups re-pack per pass)
    const bool wt_prep = prep && pl.wt_bytes > 0;
    char *wt_p = wt_prep ? (char *)prep->base + pl.wt : base + l.wt;
    const bool wt_packed = wt_prep && (prep->reuse & D2C_REUSE_BACKWARD_WEIGHTS);
    bool gw_cleared = false;
    if (brick && sizeof(T) == 4) {
        // one launch: the input with the row of zeros behind it, the clear of what is added into, the bias gradient
        PrepArgs pa{};
        if (!have_x) {
            prep_pack<T>(pa.pack[0], x, xcl_p, s.N, s.Cin, s.vol);
            pa.zrow = (uint32_t *)((T *)xcl_p + (size_t)s.N * s.vol * s.Cin); pa.zrow_words = 64;
        }
        if (gx) prep_zero(pa, 0, base + l.gxcl, (size_t)s.N * s.vol * s.Cin * sizeof(float));
        if (gx || goff || gmask) {
            size_t zb;
            void *const zp = d2c_brick_zero(s, base + l.brick, &zb);
            prep_zero(pa, 1, zp, zb);
        }
        if (gw) {
            prep_zero(pa, 2, base + l.gwacc, (size_t)s.Cout * s.cg * s.K * sizeof(float));
            gw_cleared = true;
        }
        pa.gout = gout; pa.gb = gb; pa.bN = s.N; pa.bC = s.Cout; pa.bP = s.P; pa.nblk_b = gb ? s.Cout : 0;
        if (int rc = prep_launch<T>(pa, st)) return rc;
        gb = nullptr;
    } else if (!have_x)
        if (int rc = pack_input<T>(s, x, xcl_p, st, true)) return rc;   // with the row of zeros behind it
    if (s.ss.on && !(brick && sorted && (goff || gmask || gx))) {
        D2cProfScope prof(D2C_PROF_PACK, st);
        long gr = ((long)s.N * s.P + 255) / 256;
        if (gr > 8192) gr = 8192;
        float *sm1 = (float *)(base + l.sm1);
        if (s.adt == D2C_BF16)
            hipLaunchKernelGGL(size_minus_one_kernel<true>, dim3((unsigned)gr), dim3(256), 0, st, s, size_raw, sm1);
        else
            hipLaunchKernelGGL(size_minus_one_kernel<false>, dim3((unsigned)gr), dim3(256), 0, st, s, size_raw, sm1);
        if (int rc = d2c_check_launch("size_minus_one_kernel")) return rc;
        s.ss.on = 2;
        off = sm1;
    }
    bool gw_from_col = false, gw_in_place = false, gw_done = false, gw_ready = false, gw_wide = false;
    // (`columns`: the sampled columns the forward call kept -- the offset / mask gradient kernel then writes none, the
    // grad-weight product takes these, and the settings that save workspace by other means do not apply)
    const BwdSlices sl = columns ? BwdSlices{0, 0} : bwd_slices(q, s);
    if ((gx || goff || gmask) && sl.gs > 0) {
        // Slice by slice over the offset groups: the grad-column rows of a slice are made, read by the offset / mask
        // gradient kernel (which files the slice's samples and writes its sampled columns) and by the grad_input
        // kernel, and the grad-weight product takes the columns of a block of slices, before the next slice
        // overwrites the rows: the buffers hold one slice (one block), and what a kernel reads was written a moment ago.
        constexpr int BKC = 8 * Elem<T>::VEC;
        const size_t es = sizeof(T);
        float *gxcl = gx ? (float *)(base + l.gxcl) : nullptr;
        const bool lists = gx != nullptr, auxk = goff || gmask;
        gw_from_col = gw && auxk && use_col_weight(q, s);
        SampleLists L{nullptr, nullptr, nullptr, 0, 0, 0};
        if (lists) {
            L = d2c_lists_make(s, Elem<T>::DT, base + l.counts, base + l.entries, base + l.ovf);
            if (int rc = auxk ? d2c_lists_clear(L, st) : d2c_lists_build(s, off, mask, L, st)) return rc;
        }
        if (int rc = d2c_tiled_bwd_data_launch<T>(s, gout, xcl_p, off, mask, w, wt_p, nullptr, base + l.gcol,
                                                 nullptr, nullptr, (float *)(base + l.auxacc), st, 1, 0, 0, wt_packed))
            return rc;
        if (gw_from_col)
            if (int rc = d2c_tiled_bwd_weight_launch<T>(s, gout, xcl_p, off, mask, base + l.goutp,
                                                       (float *)(base + l.gwacc), gw, base + l.col, 0, st, 1))
                return rc;
        const int cpc = s.cpg / BKC;
        const long mpad = (long)((s.M + 63) / 64) * 64;
        for (int g0 = 0; g0 < s.G; g0 += sl.gs) {
            const int gn = s.G - g0 < sl.gs ? s.G - g0 : sl.gs;
            const int c_lo = g0 * cpc, blk_lo = g0 / sl.cgs * sl.cgs;
            // (the kernels address chunk c at c * K * rows * BKC elements from the pointer they get: the pointer that
            // puts the slice's first chunk at the start of the buffer)
            char *gcol_v = reinterpret_cast<char *>(reinterpret_cast<uintptr_t>(base + l.gcol)
                                                    - (uintptr_t)((size_t)c_lo * s.K * s.M * BKC * es));
            char *col_v = reinterpret_cast<char *>(reinterpret_cast<uintptr_t>(base + l.col)
                                                   - (uintptr_t)((size_t)blk_lo * cpc * s.K * mpad * BKC * es));
            if (int rc = d2c_tiled_bwd_data_launch<T>(s, gout, xcl_p, off, mask, w, wt_p, nullptr, gcol_v,
                                                     nullptr, nullptr, (float *)(base + l.auxacc), st, 2, g0, gn))
                return rc;
            if (auxk)
                if (int rc = d2c_aux_grad_launch<T>(s, xcl_p, off, mask, gcol_v, goff, gmask, lists ? &L : nullptr,
                                                    gw_from_col ? col_v : nullptr, false, st, g0, gn))
                    return rc;
            if (lists)
                if (int rc = d2c_gx_owner_launch<T>(s, gcol_v, L, gxcl, st, c_lo, gn * cpc)) return rc;
            const int g1 = g0 + gn;
            if (gw_from_col && (g1 == s.G || g1 % sl.cgs == 0))
                if (int rc = d2c_tiled_bwd_weight_launch<T>(s, gout, xcl_p, off, mask, base + l.goutp,
                                                           (float *)(base + l.gwacc), gw, col_v, mpad, st, 2,
                                                           blk_lo * cpc / 2, (g1 - blk_lo) * cpc / 2))
                    return rc;
        }
        if (gx)
            if (int rc = d2c_tiled_unpack_gx<T>(s, gxcl, gx, st)) return rc;
        if (gw_from_col) {
            if (int rc = d2c_tiled_bwd_weight_launch<T>(s, gout, xcl_p, off, mask, base + l.goutp,
                                                       (float *)(base + l.gwacc), gw, base + l.col, 0, st, 4))
                return rc;
            gw_done = true;
        }
    } else if (gx || goff || gmask) {
        if (d2c_tiled_bwd_data_supported(s, q.dtype)) {
            float *gxcl = gx ? (float *)(base + l.gxcl) : nullptr;
            const bool lists = gx && use_lists(q, s);
            const bool auxk = (goff || gmask) && use_aux_kernel(q, s);
            // grad_input from sample lists: filled by the offset / mask gradient kernel on its way when that
            // runs, by a pass of their own otherwise
            // size-map source: `goff` is the gradient of the raw size map; the offset / mask gradient kernel adds
            // into fp32 sums per axis, which a finishing kernel folds into it
            gw_from_col = gw && (columns ? d2c_bwd_weight_from_kept_col(s, q.dtype) : (auxk && use_col_weight(q, s)));
            void *goff_k = goff;
            if (s.ss.on && goff && !brick) {
                goff_k = base + l.gsacc;
                D2cProfScope prof(D2C_PROF_PACK, st);
                d2c_fill_zero(goff_k, (size_t)s.N * 3 * s.P * sizeof(float), st);
            }
            // (the sampled columns over the grad-column rows: grad_input has to be done with the rows before the
            // offset / mask gradient kernel runs, so the samples are filed by a pass of their own)
            gw_in_place = gw_from_col && !columns && col_in_place(q, s);
            SampleLists L{nullptr, nullptr, nullptr, 0, 0, 0};
            char *const lists_p = sorted ? (char *)const_cast<void *>(columns) + brick_col_bytes(s) : base + l.brick;
            if (brick) {
                if (!sorted)
                    if (int rc = d2c_brick_sort(s, off, mask, lists_p, st, sizeof(T) == 4)) return rc;
            } else if (lists) {
                L = d2c_lists_make(s, Elem<T>::DT, base + l.counts, base + l.entries, base + l.ovf);
                if (int rc = (auxk && !gw_in_place) ? d2c_lists_clear(L, st) : d2c_lists_build(s, off, mask, L, st)) return rc;
            }
            const bool grad_col = brick && !prep && ws_bytes >= l.total && d2c_grad_col_supported(q);
            if (brick && sizeof(T) == 2 && s.groups == 1) {
                // grad_out and the weights in the orders of the products, the bias gradient, what is added into cleared
                gw_ready = gw_from_col;
                gw_wide = gw_ready && use_wide_weight(q, s, brick);
                if (int rc = d2c_brick_bwd_prepare(q, gout, w, grad_col ? base + l.wt : nullptr, base + l.gcl, gw_ready ? base + l.goutp : nullptr,
                                                   gb, gxcl, gxcl ? (size_t)s.N * s.vol * s.Cin * sizeof(float) : 0,
                                                   gw_ready && !gw_wide ? base + l.gwacc : nullptr, (size_t)s.Cout * s.cg * s.K * sizeof(float), st))
                    return rc;
                gb = nullptr;
            } else if (brick && sizeof(T) == 2 && gxcl) {
                D2cProfScope prof(D2C_PROF_PACK, st);
                d2c_fill_zero(gxcl, (size_t)s.N * s.vol * s.Cin * sizeof(float), st);
            }
            if (grad_col) {
                if (int rc = d2c_grad_col(q, base + l.gcol, base + l.wt, base + l.gcl, st)) return rc;
            } else if (int rc = d2c_tiled_bwd_data_launch<T>(s, gout, xcl_p, off, mask, w, wt_p,
                                                     lists ? nullptr : gxcl, (lists || auxk) ? base + l.gcol : nullptr,
                                                     auxk ? nullptr : goff, auxk ? nullptr : gmask,
                                                     (float *)(base + l.auxacc), st, 3, 0, 0, wt_packed))
                return rc;
            if (lists && gw_in_place)
                if (int rc = d2c_gx_owner_launch<T>(s, base + l.gcol, L, gxcl, st)) return rc;
            if (gw_in_place) {
                D2cProfScope prof(D2C_PROF_PACK, st);
                d2c_fill_zero(base + l.gcol + (size_t)(s.Cin / bkc_of(q.dtype)) * s.K * s.M * bkc_of(q.dtype) * sizeof(T),
                              (size_t)64 * bkc_of(q.dtype) * sizeof(T), st);
            }
            if (brick) {
                if (gw_from_col && !columns) {
                    if (int rc = d2c_brick_columns(s, xcl_p, base + l.col, (int)d2c_columns_rows(s), lists_p, st)) return rc;
                }
                if (int rc = d2c_brick_grad(s, xcl_p, base + l.gcol, mask, size_raw, gxcl, goff, gmask, lists_p,
                                            base + l.res, st)) return rc;
            } else if (auxk)
                if (int rc = d2c_aux_grad_launch<T>(s, xcl_p, off, mask, base + l.gcol, goff_k, gmask,
                                                    (lists && !gw_in_place) ? &L : nullptr,
                                                    (gw_from_col && !columns) ? (gw_in_place ? base + l.gcol : base + l.col) : nullptr,
                                                    gw_in_place, st))
                    return rc;
            if (s.ss.on && goff && !brick) {
                D2cProfScope prof(D2C_PROF_PACK, st);
                long gr = ((long)s.N * s.P + 255) / 256;
                if (gr > 8192) gr = 8192;
                if (s.adt == D2C_BF16)
                    hipLaunchKernelGGL(size_grad_finish_kernel<true>, dim3((unsigned)gr), dim3(256), 0, st, s,
                                       (const float *)goff_k, size_raw, goff);
                else
                    hipLaunchKernelGGL(size_grad_finish_kernel<false>, dim3((unsigned)gr), dim3(256), 0, st, s,
                                       (const float *)goff_k, size_raw, goff);
                if (int rc = d2c_check_launch("size_grad_finish_kernel")) return rc;
            }
            if (lists && !gw_in_place && !brick)
                if (int rc = d2c_gx_owner_launch<T>(s, base + l.gcol, L, gxcl, st)) return rc;
            if (gx)
                if (int rc = d2c_tiled_unpack_gx<T>(s, gxcl, gx, st)) return rc;
        } else {
            // shapes the fused kernel does not hold on chip: direct kernels (f32 staging in the same region)
            if (int rc = d2c_generic_conv3d_backward(q, gout, x, off, mask, w, gx, goff, gmask, nullptr, nullptr,
                                                     base + l.gxcl, st))
                return rc;
        }
    }
    if (gw && !gw_done) {
        if (columns && d2c_bwd_weight_from_kept_col(s, q.dtype)) gw_from_col = true;   // (also when nothing else was wanted)
        if (gw_wide) {
            // (its sums take the place of the grad-column rows, which are done with)
            if (int rc = d2c_col_weight(s, base + l.goutp, columns ? columns : base + l.col, (long)((s.M + 63) / 64) * 64, gw, base + l.gcol,
                                        grad_rows_bytes(q, s), st))
                return rc;
        } else if (d2c_tiled_bwd_weight_supported(s, q.dtype)) {
            if (int rc = d2c_tiled_bwd_weight_launch<T>(s, gout, xcl_p, off, mask, base + l.goutp,
                                                       (float *)(base + l.gwacc),
                                                       gw, gw_from_col ? (columns ? (char *)columns : (gw_in_place ? base + l.gcol : base + l.col)) : nullptr,
                                                       gw_in_place ? (long)s.M : (long)((s.M + 63) / 64) * 64, st, (gw_ready ? 6 : 7) | (gw_cleared ? 8 : 0)))
                return rc;
        } else {
            if (int rc = d2c_generic_conv3d_backward(q, gout, x, off, mask, w, nullptr, nullptr, nullptr, gw, nullptr,
                                                     nullptr, st))
                return rc;
        }
    }
    if (gb) return d2c_tiled_bias_grad<T>(s, gout, gb, st);
    return D2C_OK;
}

}  // namespace

static bool mfma_channels_ok(const d2c_conv3d_desc &q)
{
    if (q.dtype != D2C_BF16 && q.dtype != D2C_F32) return false;
    // the tiled kernels address the channels-last input with 32-bit byte offsets
    if ((size_t)q.N * q.Cin * q.D * q.H * q.W * d2c_elem_size(q.dtype) + 256 >= (1ull << 32)) return false;
    // ... form voxel indices with 24-bit multiplications (corner_row), and address the offsets of the (at most two)
    // samples a position tile meets with 32-bit byte offsets from the first one
    if ((long)q.D * q.H >= (1 << 23) || q.W >= (1 << 23)) return false;
    if ((size_t)2 * q.offset_groups * q.kd * q.kh * q.kw * 3 * q.Do * q.Ho * q.Wo * 4 >= (1ull << 32)) return false;
    // ... and the grad-column rows of one (chunk, tap), 128 bytes per position, through a buffer descriptor
    if ((size_t)q.N * q.Do * q.Ho * q.Wo * 128 + 256 >= (1ull << 32)) return false;
    const int bkc = bkc_of(q.dtype);
    const int cg = q.Cin / q.groups, cpg = q.Cin / q.offset_groups;
    return cg % bkc == 0 && cpg % bkc == 0;
}

// ---- 1-D operator on the matrix-core kernels -----------------------------
// Served when the channel counts fit the chunking and both backward kernels
// can take the shape; otherwise the direct 1-D kernels run.
bool d2c_tiled1d_supported(const d2c_conv1d_desc &q1)
{
    const d2c_conv3d_desc q = as_3d(q1);
    if (!mfma_channels_ok(q)) return false;
    const TiledShape s = tiled_shape(q, 1, q1.reference_quirks);
    return d2c_tiled_bwd_data_supported(s, q.dtype) && d2c_tiled_bwd_weight_supported(s, q.dtype);
}
size_t d2c_tiled1d_forward_ws(const d2c_conv1d_desc &q1)
{
    const d2c_conv3d_desc q = as_3d(q1);
    return fwd_ws(q, tiled_shape(q, 1, 0)).total;
}
size_t d2c_tiled1d_backward_ws(const d2c_conv1d_desc &q1)
{
    const d2c_conv3d_desc q = as_3d(q1);
    const TiledShape s = tiled_shape(q, 1, 0);
    return d2c_conv1d_bwd_use(s, q.dtype) ? d2c_conv1d_bwd_ws(s, q.dtype) : bwd_ws(q, s).total;
}
int d2c_tiled1d_forward(const d2c_conv1d_desc &q1, const void *x, const void *off, const void *mask, const void *w,
                        const void *bias, void *out, void *ws, hipStream_t st)
{
    const d2c_conv3d_desc q = as_3d(q1);
    if (q.dtype == D2C_BF16) return forward_t<bf16_t>(q, x, off, mask, w, bias, out, ws, st, 1);
    return forward_t<float>(q, x, off, mask, w, bias, out, ws, st, 1);
}
int d2c_tiled1d_backward(const d2c_conv1d_desc &q1, const void *gout, const void *x, const void *off,
                         const void *mask, const void *w, void *gx, void *goff, void *gmask, void *gw, void *gb,
                         void *ws, hipStream_t st)
{
    const d2c_conv3d_desc q = as_3d(q1);
    const TiledShape s = tiled_shape(q, 1, q1.reference_quirks);
    if (!mask) gmask = nullptr;
    if (d2c_conv1d_bwd_use(s, q.dtype))
        return q.dtype == D2C_BF16 ? d2c_conv1d_bwd<bf16_t>(s, gout, x, off, mask, w, gx, goff, gmask, gw, gb, ws, st)
                                   : d2c_conv1d_bwd<float>(s, gout, x, off, mask, w, gx, goff, gmask, gw, gb, ws, st);
    if (q.dtype == D2C_BF16)
        return backward_t<bf16_t>(q, gout, x, off, mask, w, gx, goff, gmask, gw, gb, ws, st, 1, q1.reference_quirks);
    return backward_t<float>(q, gout, x, off, mask, w, gx, goff, gmask, gw, gb, ws, st, 1, q1.reference_quirks);
}

bool d2c_tiled_supported(const d2c_conv3d_desc &q)
{
    if (q.dtype != D2C_BF16 && q.dtype != D2C_F32) return false;
    if (is_depthwise(q)) return true;
    return mfma_channels_ok(q);
}

int d2c_tiled_algo(const d2c_conv3d_desc &q) { return is_depthwise(q) ? D2C_ALGO_DEPTHWISE : D2C_ALGO_MFMA; }

// Offsets and mask read inside the layer's deformation tensor, modulation activation in the sampler
// (d2c_conv3d_desc::deform_channels, mask_activation): matrix-core kernels whose backward pass runs the offset / mask
// gradient kernel.
bool d2c_tiled_packed_supported(const d2c_conv3d_desc &q)
{
    if (is_depthwise(q) || !mfma_channels_ok(q)) return false;
    const size_t P = (size_t)q.Do * q.Ho * q.Wo;
    if (q.deform_channels > 0 && (size_t)2 * q.deform_channels * P * 4 >= (1ull << 32)) return false;
    return use_aux_kernel(q, tiled_shape(q));
}

// Offsets held at zero along some axes (offset_axes) are honoured by the tiled kernels only: every part of the
// backward pass has to stay on them too, or the direct kernels that take over would sample with the unzeroed offsets.
bool d2c_tiled_axes_supported(const d2c_conv3d_desc &q)
{
    if (is_depthwise(q) || !mfma_channels_ok(q)) return false;
    const TiledShape s = tiled_shape(q);
    return d2c_tiled_bwd_data_supported(s, q.dtype) && d2c_tiled_bwd_weight_supported(s, q.dtype);
}

size_t d2c_tiled_forward_ws(const d2c_conv3d_desc &q, D2cForwardWs which)
{
    const TiledShape s = tiled_shape(q);
    if (is_depthwise(q)) return dw_ws(q, s).total_fwd;
    const FwdWs l = fwd_ws(q, s);
    switch (which) {
    case D2C_FWD_WS_GATHER: return l.least + d2c_fwd_split_bytes(s);
    case D2C_FWD_WS_LEAST: return l.least;
    case D2C_FWD_WS_KEEP: return use_brick_forward(q, s, true) ? l.keep : l.least + d2c_fwd_split_bytes(s);
    case D2C_FWD_WS_KEEP_LEAST:
        return !use_brick_forward(q, s, true) ? l.least : (d2c_fwd_writes_columns(s, q.dtype) ? std::min(l.least, l.keep) : l.keep);
    default: return l.total;
    }
}

size_t d2c_tiled_backward_ws(const d2c_conv3d_desc &q, const d2c_size_map_desc *sz, bool saved_columns, bool keep, bool least)
{
    const TiledShape s = tiled_shape(q, 3, 0, sz);
    if (is_depthwise(q)) return dw_ws(q, s).total_bwd;
    // (which gradients a call wants is not known here)
    const bool sorted = keep && use_brick_forward(q, s, true);
    const BwdWs a = bwd_ws(q, s, saved_columns, sorted, true), b = bwd_ws(q, s, saved_columns, sorted, false);
    return least ? std::max(a.least, b.least) : std::max(a.total, b.total);
}

// Bytes of the sampled columns that a forward call can keep for the backward call of the same step:
// [chunk][tap][rows][64 bfloat16 / 32 float], rows = position tiles x 64.  0 where the forward kernel does not write them or
// the backward pass cannot multiply over them.
size_t d2c_tiled_columns_bytes(const d2c_conv3d_desc &q, const d2c_size_map_desc *sz)
{
    if (is_depthwise(q) || !mfma_channels_ok(q)) return 0;
    if (sz && !d2c_tiled_sized_supported(q, true)) return 0;
    const TiledShape s = tiled_shape(q, 3, 0, sz);
    // (where only the sorted points give columns, they are kept with them)
    if (use_brick_forward(q, s, true)) return d2c_fwd_writes_columns(s, q.dtype) ? brick_col_bytes(s) : brick_keep_bytes(s);
    if (!d2c_fwd_writes_columns(s, q.dtype) || !d2c_bwd_weight_from_kept_col(s, q.dtype) || !use_aux_kernel(q, s)) return 0;
    const long rows = d2c_columns_rows(s), chunks = s.Cin / bkc_of(q.dtype);
    if (chunks * s.K * rows >= (1L << 31)) return 0;      // (the kernel counts rows in 32 bits)
    return (size_t)chunks * s.K * rows * bkc_of(q.dtype) * d2c_elem_size(q.dtype);
}

// ... and what is worth keeping beside them: the sampling points that the forward pass sorted, behind the columns
size_t d2c_tiled_keep_bytes(const d2c_conv3d_desc &q, const d2c_size_map_desc *sz)
{
    const size_t n = d2c_tiled_columns_bytes(q, sz);
    const TiledShape s = tiled_shape(q, 3, 0, sz);
    return n > 0 && use_brick_forward(q, s, true) ? brick_keep_bytes(s) : n;
}

// The matrix-core kernels can form the offsets from a size map themselves; the backward pass then needs the
// offset / mask gradient kernel (one pass over the output channels of a weight group).
bool d2c_tiled_sized_supported(const d2c_conv3d_desc &q, bool backward)
{
    if (q.offset_groups != 1 || is_depthwise(q) || !mfma_channels_ok(q)) return false;
    if (!backward) return true;
    return use_aux_kernel(q, tiled_shape(q));
}

int d2c_tiled_forward(const d2c_conv3d_desc &q, const void *x, const void *off, const void *mask, const void *w,
                      const void *bias, void *out, void *ws, size_t ws_bytes, hipStream_t st, const d2c_size_map_desc *sz,
                      const D2cPrepared *prep, void *columns, size_t columns_bytes)
{
    if (q.dtype == D2C_BF16) return forward_t<bf16_t>(q, x, off, mask, w, bias, out, ws, st, 3, sz, prep, columns, columns_bytes, ws_bytes);
    return forward_t<float>(q, x, off, mask, w, bias, out, ws, st, 3, sz, prep, columns, columns_bytes, ws_bytes);
}

// Bytes of the caller-held prepared region of a description (0: the kernel family keeps nothing worth holding)
size_t d2c_tiled_prepared_bytes(const d2c_conv3d_desc &q)
{
    if (is_depthwise(q) || !mfma_channels_ok(q)) return 0;
    return prepared_layout(q, tiled_shape(q)).total;
}

int d2c_tiled_backward(const d2c_conv3d_desc &q, const void *gout, const void *x, const void *off,
                       const void *mask, const void *w, void *gx, void *goff, void *gmask, void *gw, void *gb,
                       void *ws, size_t ws_bytes, hipStream_t st, const d2c_size_map_desc *sz, const D2cPrepared *prep,
                       const void *columns, size_t columns_bytes)
{
    if (q.dtype == D2C_BF16)
        return backward_t<bf16_t>(q, gout, x, off, mask, w, gx, goff, gmask, gw, gb, ws, st, 3, 0, sz, prep, columns, columns_bytes, ws_bytes);
    return backward_t<float>(q, gout, x, off, mask, w, gx, goff, gmask, gw, gb, ws, st, 3, 0, sz, prep, columns, columns_bytes, ws_bytes);
}
