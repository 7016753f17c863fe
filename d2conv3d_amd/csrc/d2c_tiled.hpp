// Host interface of the tiled kernel families (matrix-core implicit GEMM and
// the depthwise bandwidth kernels).
#pragma once
#include "d2c_common.hpp"

bool d2c_tiled_supported(const d2c_conv3d_desc &q);
int d2c_tiled_algo(const d2c_conv3d_desc &q);  // D2C_ALGO_MFMA or D2C_ALGO_DEPTHWISE
// whether a description that reads offsets and mask inside one deformation tensor, or applies a modulation
// activation in the sampler, is served (in both directions)
bool d2c_tiled_packed_supported(const d2c_conv3d_desc &q);
// whether a description with some offset axes fixed (offset_axes != 7) stays on the tiled kernels in both directions
bool d2c_tiled_axes_supported(const d2c_conv3d_desc &q);
// Workspace of a forward call: what it is fastest with; what the gathering kernels are fastest with (with room for the
// partial sums of a small problem); the least it runs with; what a call that keeps its columns is fastest with, given a
// buffer of d2c_tiled_keep_bytes(); the least that one runs with
enum D2cForwardWs { D2C_FWD_WS_FAST, D2C_FWD_WS_GATHER, D2C_FWD_WS_LEAST, D2C_FWD_WS_KEEP, D2C_FWD_WS_KEEP_LEAST };
size_t d2c_tiled_forward_ws(const d2c_conv3d_desc &q, D2cForwardWs which = D2C_FWD_WS_FAST);
// `sz` != nullptr: the offsets are formed from a raw size map (`off` is that map [N, channels(mode), P], `goff` the
// gradient with respect to it); only where d2c_tiled_sized_supported() says so.
// `saved_columns`: for a backward call that is handed the sampled columns of its forward call (d2c_tiled_columns_bytes);
// `keep`: in a buffer of d2c_tiled_keep_bytes(); `least`: what the call runs with
size_t d2c_tiled_backward_ws(const d2c_conv3d_desc &q, const d2c_size_map_desc *sz = nullptr, bool saved_columns = false,
                             bool keep = false, bool least = false);
size_t d2c_tiled_columns_bytes(const d2c_conv3d_desc &q, const d2c_size_map_desc *sz = nullptr);
size_t d2c_tiled_keep_bytes(const d2c_conv3d_desc &q, const d2c_size_map_desc *sz = nullptr);
bool d2c_tiled_sized_supported(const d2c_conv3d_desc &q, bool backward);
// `prep` != nullptr: a caller-held region of d2c_tiled_prepared_bytes() bytes that takes the place of the
// workspace's channels-last input and packed weights; the parts named in `reuse` (D2C_REUSE_*) are taken as they are.
struct D2cPrepared {
    void *base;
    int reuse;
};
size_t d2c_tiled_prepared_bytes(const d2c_conv3d_desc &q);
int d2c_tiled_forward(const d2c_conv3d_desc &q, const void *x, const void *off, const void *mask, const void *w,
                      const void *bias, void *out, void *ws, size_t ws_bytes, hipStream_t st, const d2c_size_map_desc *sz = nullptr,
                      const D2cPrepared *prep = nullptr, void *columns = nullptr, size_t columns_bytes = 0);
int d2c_tiled_backward(const d2c_conv3d_desc &q, const void *gout, const void *x, const void *off,
                       const void *mask, const void *w, void *gx, void *goff, void *gmask, void *gw, void *gb,
                       void *ws, size_t ws_bytes, hipStream_t st, const d2c_size_map_desc *sz = nullptr,
                       const D2cPrepared *prep = nullptr, const void *columns = nullptr, size_t columns_bytes = 0);

// 1-D operator served by the same matrix-core kernels (1 x 1 x L volume).
bool d2c_tiled1d_supported(const d2c_conv1d_desc &q);
size_t d2c_tiled1d_forward_ws(const d2c_conv1d_desc &q);
size_t d2c_tiled1d_backward_ws(const d2c_conv1d_desc &q);
int d2c_tiled1d_forward(const d2c_conv1d_desc &q, const void *x, const void *off, const void *mask, const void *w,
                        const void *bias, void *out, void *ws, hipStream_t st);
int d2c_tiled1d_backward(const d2c_conv1d_desc &q, const void *gout, const void *x, const void *off,
                         const void *mask, const void *w, void *gx, void *goff, void *gmask, void *gw, void *gb,
                         void *ws, hipStream_t st);

// The ordinary convolution of a deformation branch (d2c_conv.hip).
bool d2c_plain_supported(const d2c_conv3d_desc &q);
size_t d2c_plain_input_bytes(const d2c_conv3d_desc &q);
size_t d2c_plain_forward_ws(const d2c_conv3d_desc &q);
size_t d2c_plain_backward_ws(const d2c_conv3d_desc &q);
int d2c_plain_forward(const d2c_conv3d_desc &q, const void *x, const void *w, const void *bias, void *out, void *xcl, void *ws,
                      hipStream_t st);
int d2c_plain_backward(const d2c_conv3d_desc &q, const void *gout, const void *xcl, const void *w, void *gx, void *gw, void *gb,
                       void *ws, hipStream_t st);
