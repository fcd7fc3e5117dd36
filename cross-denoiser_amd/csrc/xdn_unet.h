// The reference's bandwidth U-Net (scripts/main.py:83-118) on gfx950: frame descriptions and
// launchers of its kernels (internal header).
//
// Network (Keras order; H0 = full resolution, H1 = H0/2, H2 = H0/4; activations bf16 NHWC):
//   0 c1_1  conv3x3 15->8  ReLU  H0      (input: the five 3-channel FP32 images)
//   1 c1_2  conv3x3  8->8  ReLU  H0
//     pool  2x2 max             H0->H1
//   2 c2_1  conv3x3  8->16 ReLU  H1
//   3 c2_2  conv3x3 16->16 ReLU  H1
//     pool  2x2 max             H1->H2
//   4 c3_1  conv3x3 16->32 ReLU  H2
//   5 c3_2  conv3x3 32->32 ReLU  H2
//   6 c3_3  convT 1x1 stride 2 32->32 (linear) H2->H1: out(2y,2x) = W^T in(y,x) + b, else b
//   7 c4_1  conv3x3 48->16 ReLU  H1      (input: concat[c3_3, c2_2])
//   8 c4_2  conv3x3 16->16 ReLU  H1
//   9 c4_3  convT 1x1 stride 2 16->16 H1->H0
//  10 c5_1  conv3x3 24->8  ReLU  H0      (input: concat[c4_3, c1_2])
//  11 head  conv1x1  8->6        H0      FP32 output (the band/alpha head follows in the filter)
// 31,414 parameters.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "xdn_common.h"
#include "xdn_cnn.h"

namespace xdn {

// UC_SRC_UPCAT: the first source is a transposed 1x1 stride-2 layer's output. Off the even positions it
// holds that layer's bias, so only the even ones are read; the rest take the pixel (0, 1).
enum { UC_SRC_BF16 = 0, UC_SRC_IMAGES = 1, UC_SRC_UPCAT = 2 };
enum { UC_EPI_RELU = 0, UC_EPI_MASK = 1, UC_EPI_PLAIN = 2 };

// The 3x3 kernels address a tile with 32-bit offsets from its first row, below kUOob. Widest frames at full
// resolution, by the bytes a pixel column takes in the 18 rows of a tile: 16 channels to c5_1 (and 32 to c4_1 at
// half the width), the 24 of c5_1's data gradient (48 of c4_1's). Checked before a call launches anything.
constexpr uint32_t kUOob = 0xFFFFFFF0u;
constexpr int UNET_MAX_W_FORWARD = (int)((kUOob - 1) / (18 * 32));   // 7,456,540
constexpr int UNET_MAX_W_BACKWARD = (int)((kUOob - 1) / (18 * 48));  // 4,971,026

// 3x3 'same' convolution over concat[a (CA ch), b (CB ch)] (or the five images), forward or data
// gradient (the data gradient is the same kernel on dY with the flipped, transposed fragments).
struct UcFrame {
    const void *a, *b;          // bf16 sources (b may be null when CB == 0)
    const float *img[5];        // FP32 3-channel images (UC_SRC_IMAGES)
    void *out;                  // bf16 [H][W][CO]
    const uint16_t *mask;       // bf16 [H][W][CO] activation whose ReLU masks the output (MASK)
    const void *wfrag;          // 16-byte B fragments [9][KC][NT][64]
    const float *bias;          // [NT * 32] (RELU)
    const float *head_w;        // UC_F_24_8_HEAD: the 1x1 head, FP32 [8][6] then [6]
    float *head_out;            // UC_F_24_8_HEAD: its output, FP32 [H][W][6]
    void *pooled;               // *_POOL: the 2x2 maximum of out, bf16 [H/2][W/2][CO] (H, W even)
    int H, W;
};
// kind = index into the instantiated (SRC, CA, CB, CO, EPI) table of k_unet.hip
hipError_t launch_uconv(int kind, int n, const UcFrame *fr, hipStream_t st);
enum {
    UC_F_0 = 0,   // images -> 8, ReLU
    UC_F_8_8_POOL,  // 8 -> 8 ReLU and its 2x2 max pool
    UC_F_8_16,    // 8 -> 16 ReLU
    UC_F_16_16,   // 16 -> 16 ReLU
    UC_F_16_16_POOL,  // the same and its 2x2 max pool
    UC_F_16_32,   // 16 -> 32 ReLU
    UC_F_32_32,   // 32 -> 32 ReLU
    UC_F_48_16,   // concat 32+16 -> 16 ReLU
    UC_F_24_8_HEAD,  // concat 16 (upsampled) + 8 -> 8 ReLU, then the 1x1 head 8 -> 6 (FP32) on the bf16 output
    UC_KINDS
};

// Weight gradient of a 3x3 layer over concat[a (CA), b (CB)] (or the images) and dY (CO ch): per
// block one compact partial [9][cs][CO] + [CO] of the input slice [32 * mtile, 32 * mtile + cs)
// (cs = min(32, channels - 32 * mtile); compact_part(9, cs, CO) floats).
struct UwFrame {
    const void *a, *b;
    const float *img[5];
    const uint16_t *dy;         // bf16 [H][W][CO]
    float *part;                // [nblk][compact_part(9, cs, CO)]
    float *part_m1;             // the same of input channels 32 and up
    int H, W, nblk;
};
hipError_t launch_uwgrad_images(int n, const UwFrame *fr, hipStream_t st);  // images (15) x dY 8

// The gradients of a 3x3 layer below the first: weights (wfr: input and dY) and data (cfr: dY into the input's
// gradient), in one launch.
hipError_t launch_ubackward(int kind, int n, const UwFrame *wfr, const UcFrame *cfr, hipStream_t st);
enum {
    UBW_8_8 = 0,  // layer 8 -> 8, data gradient masked
    UBW_8_16,     // 8 -> 16, unmasked (pool input)
    UBW_16_16,    // 16 -> 16, masked
    UBW_16_32,    // 16 -> 32, unmasked (pool input)
    UBW_32_32,    // 32 -> 32, masked
    UBW_48_16,    // concat 32 (upsampled) + 16 -> 16, unmasked
    UBW_24_8,     // concat 16 (upsampled) + 8 -> 8, unmasked
};

// Gradient into a pooled activation act [H][W][C]: the pooled gradient (bf16 [H/2][W/2][C]) goes to
// the first maximum of each 2x2 window (row-major), the skip gradient (bf16 [H][W][sstride], channels
// soff..soff+C-1) is added in FP32, and the ReLU of act masks the sum -> bf16 dY [H][W][C].
struct PoolBwFrame {
    const uint16_t *dpool;
    const uint16_t *act;
    const uint16_t *dskip;
    uint16_t *dy;
    int H, W, sstride, soff;
};
hipError_t launch_pool_bwd(int C, int n, const PoolBwFrame *fr, hipStream_t st);

// Transposed 1x1 convolution, stride 2 ('same'): out(2y,2x) = W^T in(y,x) + b, other positions b.
// W is the Keras kernel [co][ci] (shape 1x1xCOxCI). Backward: dIn(y,x) = W dOut(2y,2x) masked by
// the ReLU of in -> bf16; per block one compact partial: dW [ci][co] then db (all output positions).
struct CtFrame {
    const uint16_t *in;         // bf16 [h][w][C]
    uint16_t *out;              // bf16 [2h][2w][C] (forward)
    const uint16_t *dout;       // bf16 [2h][2w][dstride], channels 0..C-1 (backward)
    uint16_t *din;              // bf16 [h][w][C] (backward)
    const float *w, *b;         // FP32 master
    float *part;                // [nblk][C * C + C] (backward)
    int h, w_, dstride, nblk;
};
hipError_t launch_convT(int C, int n, const CtFrame *fr, hipStream_t st);
hipError_t launch_convT_bwd(int C, int n, const CtFrame *fr, hipStream_t st);

// Head (1x1 convolution 8 -> 6, FP32 output; its forward is UC_F_24_8_HEAD) backward: d(in) =
// W dparam masked by the ReLU of in (bf16), per block one compact partial [8][6] + [6].
struct HeadFrame {
    const uint16_t *in;         // bf16 [H][W][8]
    const float *dparam;        // FP32 [H][W][6]
    uint16_t *din;              // bf16 [H][W][8]
    const float *w, *b;         // FP32 master [8][6], [6]
    float *part;
    int H, W, nblk;
};
hipError_t launch_head_bwd(int n, const HeadFrame *fr, hipStream_t st);

// Weight packing of one 3x3 layer: forward fragments [9][KC][NT][64] (K = ci, N = co) and, when
// frag_dgrad is set, data-gradient fragments (K = co, N = ci, taps flipped). A job with copy_n > 0
// instead copies copy_n floats from w to frag_fwd (the FP32 1x1 layers).
struct UPackJob {
    const float *w, *b;         // FP32 master [3][3][ci][co], [co]
    void *frag_fwd, *frag_dgrad;
    float *bias32;              // [NT * 32]
    int ci, co, copy_n;
};
hipError_t launch_upack(int n, const UPackJob *jobs, hipStream_t st);

int ublocks(int H, int W);      // weight-gradient blocks per image

}  // namespace xdn
