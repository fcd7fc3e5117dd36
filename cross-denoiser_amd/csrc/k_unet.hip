// Kernels of the reference's bandwidth U-Net (scripts/main.py:83-118) on gfx950.
//
//   uconv3x3<SRC, CA, CB, CO, EPI>  3x3 'same' convolution as an implicit GEMM on
//     v_mfma_f32_32x32x16_bf16 (M = 32 output channels per channel tile, N = 32 px of a row, K = 16
//     input channels per chunk) over concat[a (CA ch), b (CB ch)] staged in LDS; 16x32-px tiles,
//     every B fragment feeds up to three output rows. Forward
//     (bias + ReLU -> bf16) and data gradient (flipped, transposed fragments; ReLU-masked, or
//     plain for concat and pooled inputs). Channel counts are the stored ones (8, 16, 24, 32, 48).
//   uwgrad_block<SRC, CA, CB, CO, MT, DEPTH>  weight gradient over 8x32-px strips, operands from pixel-major
//     LDS tiles through ds_read_b64_tr_b16, one 32-channel input slice (MT) per instantiation,
//     software-pipelined strip loop.
//   ubackward                    weight and data gradient of a layer in one launch (uwgrad_images: the
//                                first layer's weight gradient alone).
//   pool_bwd                     gradient of the 2x2 max pool (to the first maximum, plus the
//     skip-connection gradient, ReLU-masked); the pool itself is in the epilogue of the layer before it,
//     uconv3x3<..., POOL>.
//   convT1x1s2 / convT_bwd       transposed 1x1 stride-2 convolution and its gradients.
//   head_bwd                     gradients of the 1x1 8->6 output convolution (its forward runs in
//                                the epilogue of the last 3x3 layer, uconv3x3<..., HEAD>).
//   upack                        FP32 master weights -> bf16 fragments.
#include "xdn_common.h"
#include "xdn_unet.h"

namespace xdn {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s lds_v4s;

__device__ __forceinline__ uint32_t u_f2bf(float f)
{
    const uint32_t u = __float_as_uint(f);
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ uint32_t u_pack2(float a, float b) { return u_f2bf(a) | (u_f2bf(b) << 16); }
__device__ __forceinline__ float u_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float u_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ f32x16 u_mfma(u32x4 a, u32x4 b, f32x16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}
// transposing LDS read, see ld_tr of k_cnn.hip
__device__ __forceinline__ uint2 u_ld_tr(const uint16_t *p)
{
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)p));
}
// bf16 word pair: keep each half where the mask half is > 0
__device__ __forceinline__ uint32_t u_keep(uint32_t mw, uint32_t vw)
{
    const uint32_t lo = mw & 0xFFFFu, hi = mw >> 16;
    const uint32_t klo = ((lo & 0x8000u) == 0 && lo != 0) ? 0xFFFFu : 0u;
    const uint32_t khi = ((hi & 0x8000u) == 0 && hi != 0) ? 0xFFFF0000u : 0u;
    return vw & (klo | khi);
}
__device__ __forceinline__ float u_bf(const uint16_t *p, int i) { return __uint_as_float((uint32_t)p[i] << 16); }

// Sum over the 64 lanes in every lane, pairing lanes 32, 16, 8, 4, 2 and 1 apart: lane swaps and DPP row
// rotations (after each sum the values repeat with that period, so a rotation meets the same partner)
// instead of six LDS permutes, with the sums of a __shfl_xor tree bit for bit (54 sums of head_bwd, 32 of
// convT_bwd<32>: 1 us of a block each).
template <int R>
__device__ __forceinline__ float u_ror_add(float v)
{
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + R, 0xf, 0xf, true));
}
__device__ __forceinline__ float u_wave_sum(float v)
{
    const uint32_t a = __float_as_uint(v);
    const auto s32 = __builtin_amdgcn_permlane32_swap(a, a, false, false);
    v = __uint_as_float((uint32_t)s32[0]) + __uint_as_float((uint32_t)s32[1]);
    const uint32_t b = __float_as_uint(v);
    const auto s16 = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    v = __uint_as_float((uint32_t)s16[0]) + __uint_as_float((uint32_t)s16[1]);
    return u_ror_add<1>(u_ror_add<2>(u_ror_add<4>(u_ror_add<8>(v))));
}

static int udiv_up(int a, int b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------------------------------------
// 3x3 convolution (forward / data gradient)
// ---------------------------------------------------------------------------------------------
struct UcBatch {
    TileMap map;
    UcFrame f[XDN_MAX_FRAMES];
};
static_assert(sizeof(UcBatch) <= 4096, "kernel argument too large");

constexpr int UT_W = 32, UT_H = 16;

// Raw buffer accesses with 32-bit offsets from a tile's first row: a load at kUOob returns zero and a
// store there is dropped, so image borders and partial tiles need no branch and all loads of a
// staging are in flight together.
typedef __amdgpu_buffer_rsrc_t u_rsrc;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(3))) unsigned int u32x3;
__device__ __forceinline__ u_rsrc u_buf(const void *p, size_t off, size_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(static_cast<const char *>(p) + off), (short)0, (int)(uint32_t)bytes,
                                             0x00020000);
}
// Two floats -> packed bf16 {a, b}, round to nearest even (one v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t u_cvt2(float a, float b)
{
    typedef __attribute__((ext_vector_type(2))) float f32x2;
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// The kernel fragments are the MFMA A operand (M = output channels) and 32 pixels of a row the B
// operand, so a lane ends with 4 of every 8 output channels of one pixel, c = 8j + 4h + 0..3, and the
// epilogue works in registers: bias, ReLU or mask, one conversion per channel pair, a permlane32 swap
// per two groups of 8 channels and whole-pixel 16-B (or 8-B) stores. With the pixels on the A side a
// lane held one channel of 16 pixels: at 8 channels three quarters of the lanes converted padding and
// the tile went back through LDS in 2-byte writes. Only the CI real channels are staged, in pixels of
// an odd number of 16-B units (conflict-free b128 reads); the upper half of an odd last K chunk is
// masked to zero as it is read. Bound by HBM at 8 output channels (1920x1080, before -> now: 8 -> 8
// 28.3 -> 19.5 us for 66 MB, images -> 8 38.7 -> 34.0 us for 158 MB, 24 -> 8 and the head 50 -> 46 us
// with only the even pixels of the upsampled source read), by staging latency and MFMA issue elsewhere
// (48 -> 16 at half resolution 37.7 -> 20.4 us); registers for four waves per SIMD with one K
// chunk, three with two, two with three chunks or two channel tiles. 16 -> 32 spills 8 VGPRs (36 B a lane) at four
// waves and 32 -> 32 four (20 B) at three; a scheduling barrier that removes the spills changed no time.
constexpr int uconv_lds(int src, int ci, bool head)  // 16-bit elements
{
    const int q = (src == UC_SRC_IMAGES ? 16 : ci) / 8;
    return (UT_W + 2) * (UT_H + 2) * 8 * (q | 1) + (head ? 2 * 54 : 0);
}

template <int SRC, int CA, int CB, int CO, int EPI, bool HEAD, bool POOL = false>
__device__ __forceinline__ void uconv_block(const UcBatch &b, int bid, uint16_t *lds)
{
    static_assert(!HEAD || (CO == 8 && EPI == UC_EPI_RELU), "the head follows the 8-channel ReLU layer");
    static_assert(!POOL || (CO <= 16 && EPI == UC_EPI_RELU), "the pool takes nonnegative activations");
    constexpr int CI = SRC == UC_SRC_IMAGES ? 16 : CA + CB;
    constexpr int KC = (CI + 15) / 16, QL = CI / 8, PS = 8 * (QL | 1);
    constexpr int NT = (CO + 31) / 32, NG = CO / 8;
    constexpr int LW = UT_W + 2, LH = UT_H + 2, NPX = LW * LH;
    float *hws = reinterpret_cast<float *>(lds + NPX * PS);  // head weights [8][6], bias [6], read behind the MFMAs
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, px = lane & 31, h = lane >> 5;
    const TileLoc L = locate(b.map, xcd_tile(bid, b.map.total));
    const UcFrame &F = b.f[L.f];
    const int H = F.H, W = F.W;
    const int x0 = L.tx * UT_W, y0 = L.ty * UT_H;
    const int yb = max(0, y0 - 1);                                  // first staged image row
    const size_t row0 = (size_t)yb * W, npx = (size_t)(min(H, y0 + UT_H + 1) - yb) * W;
    // offset of a staged pixel from row yb (in pixels), or kUOob
    auto pixel = [&](int pix) -> uint32_t {
        const int ly = pix / LW, lx = pix - ly * LW;
        const int gy = y0 + ly - 1, gx = x0 + lx - 1;
        return pix < NPX && gy >= 0 && gy < H && gx >= 0 && gx < W ? (uint32_t)(gy - yb) * (uint32_t)W + (uint32_t)gx : kUOob;
    };
    // UPCAT: off the even image positions (odd tile-local ones: tiles start at even rows and columns) the
    // first source is its layer's bias, staged from pixel (0, 1) while the other loads are in flight
    u32x4 fill;
    if constexpr (SRC == UC_SRC_UPCAT)
        fill = *reinterpret_cast<const u32x4 *>(static_cast<const uint16_t *>(F.a) + CA + 8 * (tid % (CA / 8)));
    // kernel fragments first: their loads are in flight together with the tile's
    u32x4 wf[9][KC][NT];
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                wf[t][kc][nt] = static_cast<const u32x4 *>(F.wfrag)[((t * KC + kc) * NT + nt) * 64 + lane];
    if constexpr (HEAD)
        if (tid < 54) hws[tid] = F.head_w[tid];
    if constexpr (SRC != UC_SRC_IMAGES)
    {
        constexpr int QA = CA / 8, QB = CB / 8;
        static_assert(256 % QA == 0, "a thread stages the same chunk of every pixel");
        constexpr bool UP = SRC == UC_SRC_UPCAT;
        constexpr int NPA = UP ? (LW / 2) * (LH / 2) : NPX;  // pixels loaded of the first source
        auto apix = [](int e) { return UP ? (2 * (e / (LW / 2)) + 1) * LW + 2 * (e % (LW / 2)) + 1 : e; };
        constexpr int NA = (NPA * QA + 255) / 256, NB = QB ? (NPX * QB + 255) / 256 : 0;
        const u_rsrc ra = u_buf(F.a, row0 * (CA * 2), npx * (CA * 2));
        u32x4 va[NA];
        u32x4 vb[NB ? NB : 1];
#pragma unroll
        for (int u = 0; u < NA; ++u)
        {
            const int i = tid + 256 * u;
            const uint32_t p = i < NPA * QA ? pixel(apix(i / QA)) : kUOob;
            va[u] = __builtin_amdgcn_raw_buffer_load_b128(ra, p == kUOob ? kUOob : p * (CA * 2) + (i % QA) * 16, 0, 0);
        }
        if constexpr (QB > 0)
        {
            const u_rsrc rb = u_buf(F.b, row0 * (CB * 2), npx * (CB * 2));
#pragma unroll
            for (int u = 0; u < NB; ++u)
            {
                const int i = tid + 256 * u;
                const uint32_t p = pixel(i / QB);
                vb[u] = __builtin_amdgcn_raw_buffer_load_b128(rb, p == kUOob ? kUOob : p * (CB * 2) + (i % QB) * 16, 0, 0);
            }
        }
        if constexpr (UP)
#pragma unroll
            for (int u = 0; u < (NPX * QA + 255) / 256; ++u)
            {
                const int i = tid + 256 * u, pix = i / QA;
                if (i >= NPX * QA || (pix / LW & (pix % LW) & 1)) continue;
                *reinterpret_cast<u32x4 *>(&lds[pix * PS + (i % QA) * 8]) = pixel(pix) != kUOob ? fill : u32x4{0u, 0u, 0u, 0u};
            }
#pragma unroll
        for (int u = 0; u < NA; ++u)
        {
            const int i = tid + 256 * u;
            if (i < NPA * QA) *reinterpret_cast<u32x4 *>(&lds[apix(i / QA) * PS + (i % QA) * 8]) = va[u];
        }
        if constexpr (QB > 0)
#pragma unroll
            for (int u = 0; u < NB; ++u)
            {
                const int i = tid + 256 * u;
                if (i < NPX * QB) *reinterpret_cast<u32x4 *>(&lds[(i / QB) * PS + CA + (i % QB) * 8]) = vb[u];
            }
    }
    else
    {
        constexpr int NP = (NPX + 255) / 256;
        u32x3 v[NP][5];
#pragma unroll
        for (int im = 0; im < 5; ++im)
        {
            const u_rsrc r = u_buf(F.img[im], row0 * 12, npx * 12);
#pragma unroll
            for (int u = 0; u < NP; ++u)
            {
                const uint32_t p = pixel(tid + 256 * u);
                v[u][im] = __builtin_amdgcn_raw_buffer_load_b96(r, p == kUOob ? kUOob : p * 12, 0, 0);
            }
        }
#pragma unroll
        for (int u = 0; u < NP; ++u)
        {
            const int pix = tid + 256 * u;
            if (pix >= NPX) continue;
            float f[16];
#pragma unroll
            for (int im = 0; im < 5; ++im)
#pragma unroll
                for (int k = 0; k < 3; ++k) f[3 * im + k] = __uint_as_float(v[u][im][k]);
            f[15] = 0.f;
#pragma unroll
            for (int q = 0; q < 2; ++q)
                *reinterpret_cast<u32x4 *>(&lds[pix * PS + 8 * q]) =
                    u32x4{u_cvt2(f[8 * q], f[8 * q + 1]), u_cvt2(f[8 * q + 2], f[8 * q + 3]),
                          u_cvt2(f[8 * q + 4], f[8 * q + 5]), u_cvt2(f[8 * q + 6], f[8 * q + 7])};
        }
    }
    // the lane's output pixel of tile row 4 wv + orow, in pixels from row y0 (kUOob outside the image)
    const size_t orow0 = (size_t)y0 * W, onpx = (size_t)(min(H, y0 + UT_H) - y0) * W;
    auto opixel = [&](int orow) -> uint32_t {
        const int r = 4 * wv + orow;
        return y0 + r < H && x0 + px < W ? (uint32_t)r * (uint32_t)W + (uint32_t)(x0 + px) : kUOob;
    };
    const u_rsrc ro = u_buf(F.out, orow0 * (CO * 2), onpx * (CO * 2));
    float4 bias[EPI == UC_EPI_RELU ? NG : 1];  // channels 8j + 4h + 0..3
    if constexpr (EPI == UC_EPI_RELU)
#pragma unroll
        for (int j = 0; j < NG; ++j) bias[j] = *reinterpret_cast<const float4 *>(F.bias + 8 * j + 4 * h);
    __syncthreads();

    f32x16 acc[4][NT];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int k = 0; k < 16; ++k) acc[r][nt][k] = 0.f;
    const uint32_t hi0 = h ? 0u : 0xFFFFFFFFu;  // zeroes the upper half of an odd last K chunk
#pragma unroll
    for (int ir = 0; ir < 6; ++ir)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
#pragma unroll
            for (int kc = 0; kc < KC; ++kc)
            {
                const bool odd = (QL & 1) && kc == KC - 1;
                u32x4 a = *reinterpret_cast<const u32x4 *>(
                    &lds[((4 * wv + ir) * LW + px + dx) * PS + kc * 16 + (odd ? 0 : 8 * h)]);
                if (odd) a &= u32x4{hi0, hi0, hi0, hi0};
#pragma unroll
                for (int orow = 0; orow < 4; ++orow)
                {
                    const int dy = ir - orow;
                    if (dy < 0 || dy > 2) continue;
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) acc[orow][nt] = u_mfma(wf[dy * 3 + dx][kc][nt], a, acc[orow][nt]);
                }
            }

    uint32_t above[POOL ? 2 * NG : 1];  // POOL: the packed channels of the row above
    // head: output channels 3h .. 3h + 2 of the lane's pixel
    float hw[HEAD ? 24 : 1], hb[3] = {0.f, 0.f, 0.f};
    if constexpr (HEAD)
    {
        // the reads stay behind the MFMAs: hoisted above them they spill at three waves per SIMD (46 -> 67 us)
        asm volatile("" ::: "memory");
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int k = 0; k < 3; ++k) hw[c * 3 + k] = hws[c * 6 + 3 * h + k];
#pragma unroll
        for (int k = 0; k < 3; ++k) hb[k] = hws[48 + 3 * h + k];
    }
#pragma unroll
    for (int orow = 0; orow < 4; ++orow)
    {
        const uint32_t p = opixel(orow);
        const bool in = p != kUOob;
        uint32_t d[2 * NG];  // d[2j + e] = channels 8j + 4h + 2e, +1
#pragma unroll
        for (int j = 0; j < NG; ++j)
        {
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = acc[orow][j / 4][4 * (j & 3) + k];
            if constexpr (EPI == UC_EPI_RELU)
            {
                v[0] = fmaxf(v[0] + bias[j].x, 0.f); v[1] = fmaxf(v[1] + bias[j].y, 0.f);
                v[2] = fmaxf(v[2] + bias[j].z, 0.f); v[3] = fmaxf(v[3] + bias[j].w, 0.f);
            }
            d[2 * j] = u_cvt2(v[0], v[1]);
            d[2 * j + 1] = u_cvt2(v[2], v[3]);
        }
        if constexpr (POOL)
        {
            // 2x2 maximum of the stored activations: row pairs in a lane, column pairs in adjacent lanes.
            // Nonnegative bf16 values order as int16. A launch of its own read them all again:
            // the step of four 256x256 streams 414 -> 407 us, the network at 1920x1080 630 -> 621.
            typedef __attribute__((ext_vector_type(2))) short s16x2;
            auto max2 = [](uint32_t x, uint32_t y) {
                return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(s16x2, x), __builtin_bit_cast(s16x2, y)));
            };
            uint32_t m[2 * NG];
#pragma unroll
            for (int k = 0; k < 2 * NG; ++k)
            {
                if (!(orow & 1))
                {
                    above[k] = d[k];
                    continue;
                }
                const uint32_t v = max2(above[k], d[k]);
                m[k] = max2(v, (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xf, 0xf, true));
            }
            if (orow & 1)
            {
                const u_rsrc rp = u_buf(F.pooled, orow0 / 4 * (CO * 2), onpx / 4 * (CO * 2));
                const uint32_t p2 = (uint32_t)((4 * wv + orow) >> 1) * (uint32_t)(W / 2) + (uint32_t)((x0 + px) >> 1);
                const bool st = in && !(px & 1);
                if constexpr (NG == 1)
                    __builtin_amdgcn_raw_buffer_store_b64(u32x2{m[0], m[1]}, rp, st ? p2 * 16 + 8 * h : kUOob, 0, 0);
                else
                {
                    u32x4 v;
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                    {
                        const auto sw = __builtin_amdgcn_permlane32_swap(m[e], m[2 + e], false, false);
                        v[e] = (uint32_t)sw[0];
                        v[2 + e] = (uint32_t)sw[1];
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(v, rp, st ? p2 * 32 + 16 * h : kUOob, 0, 0);
                }
            }
        }
        // two groups of 8 channels: each half-wave gathers one whole group of its pixels
#pragma unroll
        for (int g = 0; g < NG / 2; ++g)
        {
            u32x4 v;
#pragma unroll
            for (int e = 0; e < 2; ++e)
            {
                const auto sw = __builtin_amdgcn_permlane32_swap(d[4 * g + e], d[4 * g + 2 + e], false, false);
                v[e] = (uint32_t)sw[0];
                v[2 + e] = (uint32_t)sw[1];
            }
            const uint32_t o = in ? p * (CO * 2) + 32 * g + 16 * h : kUOob;
            if constexpr (EPI == UC_EPI_MASK)
            {
                const u_rsrc rm = u_buf(F.mask, orow0 * (CO * 2), onpx * (CO * 2));
                const u32x4 m = __builtin_amdgcn_raw_buffer_load_b128(rm, o, 0, 0);
                v.x = u_keep(m.x, v.x); v.y = u_keep(m.y, v.y); v.z = u_keep(m.z, v.z); v.w = u_keep(m.w, v.w);
            }
            __builtin_amdgcn_raw_buffer_store_b128(v, ro, o, 0, 0);
        }
        if constexpr (NG & 1)
        {
            u32x2 v = {d[2 * NG - 2], d[2 * NG - 1]};
            const uint32_t o = in ? p * (CO * 2) + 16 * (NG - 1) + 8 * h : kUOob;
            if constexpr (EPI == UC_EPI_MASK)
            {
                const u_rsrc rm = u_buf(F.mask, orow0 * (CO * 2), onpx * (CO * 2));
                const u32x2 m = __builtin_amdgcn_raw_buffer_load_b64(rm, o, 0, 0);
                v.x = u_keep(m.x, v.x); v.y = u_keep(m.y, v.y);
            }
            __builtin_amdgcn_raw_buffer_store_b64(v, ro, o, 0, 0);
        }
        if constexpr (HEAD)
        {
            // the head on the stored bf16 activation: bias, then the 8 inputs in order
            const auto s0 = __builtin_amdgcn_permlane32_swap(d[0], d[0], false, false);
            const auto s1 = __builtin_amdgcn_permlane32_swap(d[1], d[1], false, false);
            const uint32_t w4[4] = {(uint32_t)s0[0], (uint32_t)s1[0], (uint32_t)s0[1], (uint32_t)s1[1]};
            float sum[3] = {hb[0], hb[1], hb[2]};
#pragma unroll
            for (int c = 0; c < 8; ++c)
            {
                const float in_c = (c & 1) ? u_hi(w4[c / 2]) : u_lo(w4[c / 2]);
#pragma unroll
                for (int k = 0; k < 3; ++k) sum[k] += in_c * hw[c * 3 + k];
            }
            const u_rsrc rh = u_buf(F.head_out, orow0 * 24, onpx * 24);
            __builtin_amdgcn_raw_buffer_store_b96(
                u32x3{__float_as_uint(sum[0]), __float_as_uint(sum[1]), __float_as_uint(sum[2])}, rh,
                in ? p * 24 + 12 * h : kUOob, 0, 0);
        }
    }
}

template <int SRC, int CA, int CB, int CO, int EPI, bool HEAD, bool POOL>
__global__ __launch_bounds__(256, CO > 32 || CA + CB > 32 ? 2 : (CA + CB > 16 ? 3 : 4)) void uconv3x3(UcBatch b)
{
    __shared__ __attribute__((aligned(16))) uint16_t lds[uconv_lds(SRC, CA + CB, HEAD)];
    uconv_block<SRC, CA, CB, CO, EPI, HEAD, POOL>(b, blockIdx.x, lds);
}

// Bytes of the widest pixel that a tile stages or stores (a source, the output or mask, the FP32 head).
constexpr int widest_pixel(int src, int ca, int cb, int co, bool head)
{
    const int in = src == UC_SRC_IMAGES ? 12 : 2 * (ca > cb ? ca : cb), out = head ? 24 : 2 * co;
    return in > out ? in : out;
}

// False: a row is too wide for this instantiation's 32-bit offsets (at its own level of the network; the entry
// points refuse such frames before they launch anything, see UNET_MAX_W_FORWARD).
template <int SRC, int CA, int CB, int CO, bool HEAD>
static bool uconv_batch(UcBatch &b, int n, const UcFrame *fr)
{
    constexpr uint64_t row = (UT_H + 2) * widest_pixel(SRC, CA, CB, CO, HEAD);
    for (int i = 0; i < n; ++i)
        if (row * (uint64_t)fr[i].W >= kUOob) return false;
    int tx[XDN_MAX_FRAMES], ty[XDN_MAX_FRAMES];
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        tx[i] = udiv_up(fr[i].W, UT_W);
        ty[i] = udiv_up(fr[i].H, UT_H);
    }
    b.map = make_tilemap(n, tx, ty);
    return true;
}

template <int SRC, int CA, int CB, int CO, int EPI, bool HEAD = false, bool POOL = false>
static hipError_t uconv_t(int n, const UcFrame *fr, hipStream_t st)
{
    UcBatch b{};
    if (!uconv_batch<SRC, CA, CB, CO, HEAD>(b, n, fr)) return hipErrorInvalidValue;
    if (b.map.total == 0) return hipSuccess;
    if (POOL)
        for (int i = 0; i < n; ++i)
            if (fr[i].H % 2 || fr[i].W % 2) return hipErrorInvalidValue;
    hipLaunchKernelGGL((uconv3x3<SRC, CA, CB, CO, EPI, HEAD, POOL>), dim3(b.map.total), dim3(256), 0, st, b);
    return hipGetLastError();
}

hipError_t launch_uconv(int kind, int n, const UcFrame *fr, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (n > XDN_MAX_FRAMES) return hipErrorInvalidValue;
    switch (kind)
    {
    case UC_F_0: return uconv_t<UC_SRC_IMAGES, 0, 0, 8, UC_EPI_RELU>(n, fr, st);
    case UC_F_8_8_POOL: return uconv_t<UC_SRC_BF16, 8, 0, 8, UC_EPI_RELU, false, true>(n, fr, st);
    case UC_F_8_16: return uconv_t<UC_SRC_BF16, 8, 0, 16, UC_EPI_RELU>(n, fr, st);
    case UC_F_16_16: return uconv_t<UC_SRC_BF16, 16, 0, 16, UC_EPI_RELU>(n, fr, st);
    case UC_F_16_16_POOL: return uconv_t<UC_SRC_BF16, 16, 0, 16, UC_EPI_RELU, false, true>(n, fr, st);
    case UC_F_16_32: return uconv_t<UC_SRC_BF16, 16, 0, 32, UC_EPI_RELU>(n, fr, st);
    case UC_F_32_32: return uconv_t<UC_SRC_BF16, 32, 0, 32, UC_EPI_RELU>(n, fr, st);
    case UC_F_48_16: return uconv_t<UC_SRC_BF16, 32, 16, 16, UC_EPI_RELU>(n, fr, st);
    case UC_F_24_8_HEAD: return uconv_t<UC_SRC_UPCAT, 16, 8, 8, UC_EPI_RELU, true>(n, fr, st);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------------------------
// Weight gradient of a 3x3 layer: input slice [32 MT, 32 MT + 32) of concat[a, b] (or the images).
// A block walks strips, at most two blocks a CU (their number fixes the partial sums), so what it spends
// is the time between strips: staging without branches, strip-invariant offsets, DEPTH strips in flight,
// only the even pixels of an upsampled source. HBM and the halo's L2 reads bound the images (1920x1080:
// 41.4 us, 158 MB), LDS reads, barriers and latency the rest (in launches of their own with two strips in
// flight, 24 channels 45 -> 33.6 us, 8 channels 26.7 -> 20.3 us, 48 in two slices 18.8 + 11.8 -> 17.5 + 11.4 us).
// ---------------------------------------------------------------------------------------------
struct UwBatch {
    int n;
    int blk_begin[XDN_MAX_FRAMES + 1];
    UwFrame f[XDN_MAX_FRAMES];
};
static_assert(sizeof(UwBatch) <= 4096, "kernel argument too large");

constexpr int US_W = 32, US_H = 8;                // strip: 8 rows x 32 px
constexpr int UX_C = US_W + 2, UX_R = US_H + 2;   // staged X: 10 rows x 34 px (1-px halo)

constexpr int uw_slice(int src, int ci, int mt) { return src == UC_SRC_IMAGES ? 15 : (ci - 32 * mt < 32 ? ci - 32 * mt : 32); }
constexpr int uwgrad_tile(int src, int ci, int co, int mt)  // 16-bit elements, at least 4 x 1024 floats
{
    const int n = UX_R * UX_C * (uw_slice(src, ci, mt) <= 16 ? 16 : 32) + US_H * US_W * (co <= 16 ? 16 : 32);
    return n > 8192 ? n : 8192;
}
constexpr int uwgrad_lds(int src, int ci, int co, int mt) { return uwgrad_tile(src, ci, co, mt) + 2 * 4 * 32; }

template <int SRC, int CA, int CB, int CO, int MT, int DEPTH>
__device__ __forceinline__ void uwgrad_block(const UwBatch &b, int bid, uint16_t *lds)
{
    // input-slice channels of this instantiation; staged channel counts (pixel strides) 16 or 32,
    // zero-padded: with 16 the lane groups 0 and 1 read the same channels, so the accumulator rows
    // (or columns) 16-31 repeat 0-15 and are not written out
    constexpr int CS = uw_slice(SRC, CA + CB, MT);
    constexpr int XS = CS <= 16 ? 16 : 32, DS = CO <= 16 ? 16 : 32;
    constexpr int X_ELEMS = UX_R * UX_C * XS;
    float(*dbs)[32] = reinterpret_cast<float(*)[32]>(lds + uwgrad_tile(SRC, CA + CB, CO, MT));
    uint16_t *xs = lds, *ds = lds + X_ELEMS;
    int f = 0;
    while (f + 1 < b.n && bid >= b.blk_begin[f + 1]) ++f;
    const UwFrame &F = b.f[f];
    const int li = bid - b.blk_begin[f], nblk = b.blk_begin[f + 1] - b.blk_begin[f];
    const int H = F.H, W = F.W;
    const int sx = (W + US_W - 1) / US_W, sy = (H + US_H - 1) / US_H;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, h = lane >> 5, ch = lane & 31;
    const int rr = 2 * wv + h;
    const int grp = (lane >> 4) & 1, s16 = lane & 15, jq = s16 >> 2, qq = s16 & 3;
    const int cbx = (XS > 16 ? 16 * grp : 0) + 4 * qq, cbd = (DS > 16 ? 16 * grp : 0) + 4 * qq;

    // Staging: 16-byte chunks of the sources' real channels (a slice lies in a, in b, or takes all of
    // both), raw buffer loads as in uconv3x3 and no branch, so a strip's loads stay in flight
    // through the two strips computed before it; the padding of the LDS pixels is cleared once.
    constexpr int CAS = SRC == UC_SRC_IMAGES ? 0 : (CA - 32 * MT > 0 ? CS < CA ? CS : CA : 0);
    constexpr int CBS = SRC == UC_SRC_IMAGES ? 0 : CS - CAS;
    constexpr int AOFF = CAS ? 32 * MT : 0, BOFF = CAS ? 0 : 32 * MT - CA;
    constexpr int QA = CAS / 8, QB = CBS / 8, QX = XS / 8, QD = DS / 8, QDR = CO / 8, NPX = UX_R * UX_C;
    constexpr bool UP = SRC == UC_SRC_UPCAT && QA > 0;
    constexpr int NPA = UP ? (UX_C / 2) * (UX_R / 2) : NPX;  // pixels loaded of a
    auto apix = [](int e) { return UP ? (2 * (e / (UX_C / 2)) + 1) * UX_C + 2 * (e % (UX_C / 2)) + 1 : e; };
    constexpr int NA = (NPA * QA + 255) / 256, NB = (NPX * QB + 255) / 256;
    constexpr int NI = SRC == UC_SRC_IMAGES ? (NPX + 255) / 256 : 0;
    static_assert(SRC == UC_SRC_IMAGES || ((QA == 0 || 256 % QA == 0) && CAS + CBS == CS), "slice of the concatenation");
    struct Strip {
        u32x4 a[NA ? NA : 1], b[NB ? NB : 1], d[QDR];
        u32x3 im[NI ? NI : 1][5];
        int ylo, yhi, xlo, xhi;  // UPCAT: staged rows and columns that lie in the image
    };
    u32x4 fill = {0u, 0u, 0u, 0u};
    bool refill = true;  // UPCAT: the bias pixels of the staged tile have to be written (see uconv3x3)
    if constexpr (UP)
        fill = *reinterpret_cast<const u32x4 *>(static_cast<const uint16_t *>(F.a) + CA + AOFF + 8 * (tid % (QA ? QA : 1)));
    // byte offsets from the strip's first staged pixel (row y0 - 1, column x0 - 1), the same for all
    // strips; a strip at the image border replaces those outside by kUOob
    auto offset = [&](int pix, int stride, int chunk) -> uint32_t {
        const int r = pix / UX_C, col = pix - r * UX_C;
        return ((uint32_t)r * (uint32_t)W + (uint32_t)col) * (uint32_t)stride + (uint32_t)chunk;
    };
    auto fetch = [&](Strip &R, int strip, bool on) {  // !on: no strip, every load out of range
        // 32 -> 32: the offsets are computed anew for every strip (an identity DPP move keeps
        // them in the loop); kept in registers they cost spills, 15.6 -> 20.4 us
        const int ti = CO > 16 && CS > 16 ? __builtin_amdgcn_mov_dpp(tid, 0xE4, 0xf, 0xf, true) : tid;
        const int s = on ? strip : 0, y0 = (s / sx) * US_H, x0 = (s % sx) * US_W;
        // staged rows [ylo, yhi) and columns [xlo, xhi) lie in the image (readfirstlane: keeps the
        // compiler from giving `on` a copy of the loads of its own, and a full wait where both meet)
        const int ylo = y0 == 0, yhi = __builtin_amdgcn_readfirstlane(on ? min(UX_R, H - y0 + 1) : 0);
        const int xlo = x0 == 0, xhi = min(UX_C, W - x0 + 1);
        const bool inner = ylo == 0 && yhi == UX_R && xlo == 0 && xhi == UX_C;
        const long base = ((long)y0 - 1) * W + x0 - 1;  // may lie before the image: only masked lanes do
        const size_t span = (size_t)UX_R * W + UX_C;
        auto outside = [&](int r, int col) { return r < ylo || r >= yhi || col < xlo || col >= xhi; };
        uint32_t oa[NA ? NA : 1], ob[NB ? NB : 1], od[QDR], oi[NI ? NI : 1];
#pragma unroll
        for (int u = 0; u < NA; ++u)
        {
            const int i = ti + 256 * u, e = i / (QA ? QA : 1);
            oa[u] = e < NPA ? offset(apix(e), CA * 2, AOFF * 2 + (i % (QA ? QA : 1)) * 16) : kUOob;
        }
#pragma unroll
        for (int u = 0; u < NB; ++u)
        {
            const int i = ti + 256 * u, pix = i / (QB ? QB : 1);
            ob[u] = pix < NPX ? offset(pix, CB * 2, BOFF * 2 + (i % (QB ? QB : 1)) * 16) : kUOob;
        }
#pragma unroll
        for (int u = 0; u < NI; ++u) oi[u] = ti + 256 * u < NPX ? offset(ti + 256 * u, 12, 0) : kUOob;
#pragma unroll
        for (int u = 0; u < QDR; ++u)
        {
            const int i = ti + 256 * u, pix = i / QDR;
            od[u] = ((uint32_t)(pix / US_W + 1) * (uint32_t)W + (uint32_t)(pix % US_W + 1)) * (CO * 2) + (i % QDR) * 16;
        }
        R.ylo = ylo; R.yhi = yhi; R.xlo = xlo; R.xhi = xhi;
        if (!inner)
        {
#pragma unroll
            for (int u = 0; u < NA; ++u)
            {
                const int pix = apix((ti + 256 * u) / (QA ? QA : 1));
                if (outside(pix / UX_C, pix % UX_C)) oa[u] = kUOob;
            }
#pragma unroll
            for (int u = 0; u < NB; ++u)
            {
                const int pix = (ti + 256 * u) / (QB ? QB : 1);
                if (outside(pix / UX_C, pix % UX_C)) ob[u] = kUOob;
            }
#pragma unroll
            for (int u = 0; u < NI; ++u)
                if (outside((ti + 256 * u) / UX_C, (ti + 256 * u) % UX_C)) oi[u] = kUOob;
#pragma unroll
            for (int u = 0; u < QDR; ++u)
            {
                const int pix = (ti + 256 * u) / QDR;
                if (outside(pix / US_W + 1, pix % US_W + 1)) od[u] = kUOob;
            }
        }
        if constexpr (QA > 0)
        {
            const u_rsrc r = u_buf(F.a, base * (CA * 2), span * (CA * 2));
#pragma unroll
            for (int u = 0; u < NA; ++u) R.a[u] = __builtin_amdgcn_raw_buffer_load_b128(r, oa[u], 0, 0);
        }
        if constexpr (QB > 0)
        {
            const u_rsrc r = u_buf(F.b, base * (CB * 2), span * (CB * 2));
#pragma unroll
            for (int u = 0; u < NB; ++u) R.b[u] = __builtin_amdgcn_raw_buffer_load_b128(r, ob[u], 0, 0);
        }
        if constexpr (SRC == UC_SRC_IMAGES)
#pragma unroll
            for (int im = 0; im < 5; ++im)
            {
                const u_rsrc r = u_buf(F.img[im], base * 12, span * 12);
#pragma unroll
                for (int u = 0; u < NI; ++u) R.im[u][im] = __builtin_amdgcn_raw_buffer_load_b96(r, oi[u], 0, 0);
            }
        const u_rsrc rd = u_buf(F.dy, base * (CO * 2), span * (CO * 2));
#pragma unroll
        for (int u = 0; u < QDR; ++u) R.d[u] = __builtin_amdgcn_raw_buffer_load_b128(rd, od[u], 0, 0);
    };
    auto commit = [&](Strip &R) {
        if constexpr (UP)
        {
            // bias pixels stay from strip to strip but where a strip meets the image border
            const bool border = R.ylo != 0 || R.yhi != UX_R || R.xlo != 0 || R.xhi != UX_C;
            if (refill || border)
                for (int i = tid; i < NPX * QA; i += 256)
                {
                    const int pix = i / QA, r = pix / UX_C, col = pix % UX_C;
                    if (r & col & 1) continue;
                    const bool in = r >= R.ylo && r < R.yhi && col >= R.xlo && col < R.xhi;
                    *reinterpret_cast<u32x4 *>(&xs[pix * XS + (i % QA) * 8]) = in ? fill : u32x4{0u, 0u, 0u, 0u};
                }
            refill = border;
        }
        if constexpr (QA > 0)
#pragma unroll
            for (int u = 0; u < NA; ++u)
            {
                const int i = tid + 256 * u;
                if (i < NPA * QA) *reinterpret_cast<u32x4 *>(&xs[apix(i / QA) * XS + (i % QA) * 8]) = R.a[u];
            }
        if constexpr (QB > 0)
#pragma unroll
            for (int u = 0; u < NB; ++u)
            {
                const int i = tid + 256 * u;
                if (i < NPX * QB) *reinterpret_cast<u32x4 *>(&xs[(i / QB) * XS + CAS + (i % QB) * 8]) = R.b[u];
            }
        if constexpr (SRC == UC_SRC_IMAGES)
#pragma unroll
            for (int u = 0; u < NI; ++u)
            {
                const int pix = tid + 256 * u;
                if (pix >= NPX) continue;
                float f[16];
#pragma unroll
                for (int im = 0; im < 5; ++im)
#pragma unroll
                    for (int k = 0; k < 3; ++k) f[3 * im + k] = __uint_as_float(R.im[u][im][k]);
                f[15] = 0.f;
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    *reinterpret_cast<u32x4 *>(&xs[pix * XS + 8 * q]) =
                        u32x4{u_cvt2(f[8 * q], f[8 * q + 1]), u_cvt2(f[8 * q + 2], f[8 * q + 3]),
                              u_cvt2(f[8 * q + 4], f[8 * q + 5]), u_cvt2(f[8 * q + 6], f[8 * q + 7])};
            }
#pragma unroll
        for (int u = 0; u < QDR; ++u)
        {
            const int i = tid + 256 * u;
            *reinterpret_cast<u32x4 *>(&ds[(i / QDR) * DS + (i % QDR) * 8]) = R.d[u];
        }
    };
    // padding chunks of the staged pixels
    if constexpr (SRC != UC_SRC_IMAGES && QA + QB < QX)
        for (int i = tid; i < NPX * (QX - QA - QB); i += 256)
            *reinterpret_cast<u32x4 *>(&xs[i / (QX - QA - QB) * XS + 8 * (QA + QB + i % (QX - QA - QB))]) = u32x4{0u, 0u, 0u, 0u};
    if constexpr (QDR < QD)
        for (int i = tid; i < US_H * US_W * (QD - QDR); i += 256)
            *reinterpret_cast<u32x4 *>(&ds[i / (QD - QDR) * DS + 8 * (QDR + i % (QD - QDR))]) = u32x4{0u, 0u, 0u, 0u};

    const StripWalk sw = xcd_strips(li, nblk, sx * sy);
    Strip R[DEPTH];
#pragma unroll
    for (int k = 0; k < DEPTH; ++k) fetch(R[k], sw.first + k * sw.step, sw.first + k * sw.step < sw.end);

    // CO > 16: 32x32x16 MFMA, M = 32 input channels, N = 32 output channels, K = 16 px (8 px of row
    // 2wv + h per lane half). CO <= 16: 16x16x32 MFMA, M = 16 input channels (MTI tiles), N = 16
    // output channels, K = 32 px = one strip row (8 px per lane group kg = lane / 16), a quarter of
    // the MFMA work and of the accumulator registers.
    constexpr bool N16 = CO <= 16;
    constexpr int MTI = XS / 16;
    typedef __attribute__((ext_vector_type(4))) float f32x4;
    f32x16 acc[N16 ? 1 : 9];
    f32x4 acc16[N16 ? 9 : 1][N16 ? MTI : 1];
    if constexpr (N16)
    {
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int m = 0; m < MTI; ++m)
#pragma unroll
                for (int k = 0; k < 4; ++k) acc16[t][m][k] = 0.f;
    }
    else
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int k = 0; k < 16; ++k) acc[t][k] = 0.f;
    float db = 0.f;
    const int kg = lane >> 4;
    auto compute = [&]() {
        if constexpr (N16)
        {
            // lane group kg takes pixels 8kg .. 8kg+7 of the row; lane L of the group reads the
            // transposed channel L (4 pixels per ds_read_b64_tr_b16)
#pragma unroll
            for (int r = 0; r < 2; ++r)
            {
                const int row = 2 * wv + r;
                const uint16_t *dp = &ds[(row * US_W + 8 * kg + jq) * DS + 4 * qq];
                const uint2 b0 = u_ld_tr(dp), b1 = u_ld_tr(dp + 4 * DS);
                const u32x4 B = {b0.x, b0.y, b1.x, b1.y};
                db += (u_lo(B.x) + u_hi(B.x)) + (u_lo(B.y) + u_hi(B.y)) + (u_lo(B.z) + u_hi(B.z)) +
                      (u_lo(B.w) + u_hi(B.w));
#pragma unroll
                for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                    for (int sh = 0; sh < 3; ++sh)
#pragma unroll
                        for (int m = 0; m < MTI; ++m)
                        {
                            const uint16_t *xp = &xs[((row + dy) * UX_C + 8 * kg + sh + jq) * XS + 16 * m + 4 * qq];
                            const uint2 a0 = u_ld_tr(xp), a1 = u_ld_tr(xp + 4 * XS);
                            acc16[dy * 3 + sh][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                __builtin_bit_cast(bf16x8, u32x4{a0.x, a0.y, a1.x, a1.y}),
                                __builtin_bit_cast(bf16x8, B), acc16[dy * 3 + sh][m], 0, 0, 0);
                        }
            }
            return;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
        {
            const uint16_t *dp = &ds[(rr * US_W + 8 * c + jq) * DS + cbd];
            const uint2 b0 = u_ld_tr(dp), b1 = u_ld_tr(dp + 4 * DS);
            const u32x4 B = {b0.x, b0.y, b1.x, b1.y};
            db += (u_lo(B.x) + u_hi(B.x)) + (u_lo(B.y) + u_hi(B.y)) + (u_lo(B.z) + u_hi(B.z)) + (u_lo(B.w) + u_hi(B.w));
#pragma unroll
            for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                for (int sh = 0; sh < 3; ++sh)
                {
                    const uint16_t *xp = &xs[((rr + dy) * UX_C + 8 * c + sh + jq) * XS + cbx];
                    const uint2 a0 = u_ld_tr(xp), a1 = u_ld_tr(xp + 4 * XS);
                    acc[dy * 3 + sh] = u_mfma(u32x4{a0.x, a0.y, a1.x, a1.y}, B, acc[dy * 3 + sh]);
                }
        }
    };
    for (int s = sw.first; s < sw.end; s += DEPTH * sw.step)
#pragma unroll
        for (int k = 0; k < DEPTH; ++k)
        {
            const int c = s + k * sw.step;
            if (c >= sw.end) break;  // uniform across the block
            __syncthreads();
            commit(R[k]);
            __syncthreads();
            // unconditional at two strips in flight: the next commit then waits for its own strip alone
            if (DEPTH > 1 || c + sw.step < sw.end) fetch(R[k], c + DEPTH * sw.step, c + DEPTH * sw.step < sw.end);
            compute();
        }
    // compact partial [9][CS][CO] + [CO] of this input slice
    float *out = (MT ? F.part_m1 : F.part) + (size_t)li * compact_part(9, CS, CO);
    float *red = reinterpret_cast<float *>(lds);  // [4 waves][1024]
#pragma unroll
    for (int t = 0; t < 9; ++t)
    {
        __syncthreads();
        if constexpr (N16)
        {
            // 16x16 accumulators: column co = lane % 16, rows ci = 16m + 4kg + i
#pragma unroll
            for (int m = 0; m < MTI; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i) red[wv * 1024 + (16 * m + 4 * kg + i) * 32 + (lane & 15)] = acc16[t][m][i];
        }
        else
#pragma unroll
            for (int k = 0; k < 16; ++k)
            {
                const int ci = 8 * (k >> 2) + 4 * h + (k & 3);
                red[wv * 1024 + ci * 32 + ch] = acc[t][k];
            }
        __syncthreads();
        for (int e = tid; e < CS * CO; e += 256)
        {
            const int ci = e / CO, co = e - ci * CO, r = ci * 32 + co;
            out[t * CS * CO + e] = (red[r] + red[1024 + r]) + (red[2048 + r] + red[3072 + r]);
        }
    }
    if constexpr (N16)
    {
        db += __shfl_xor(db, 16);
        db += __shfl_xor(db, 32);
        if (lane < 16) dbs[wv][lane] = db;
    }
    else
    {
        db += __shfl_xor(db, 32);
        if (h == 0) dbs[wv][ch] = db;
    }
    __syncthreads();
    if (tid < CO) out[9 * CS * CO + tid] = (dbs[0][tid] + dbs[1][tid]) + (dbs[2][tid] + dbs[3][tid]);
}

// up to 512 blocks per image (two per CU): the quarter- and half-resolution layers have few strips
int ublocks(int H, int W)
{
    const int strips = udiv_up(W, US_W) * udiv_up(H, US_H);
    return strips < 1 ? 1 : (strips < 512 ? strips : 512);
}

template <int DEPTH>
__global__ __launch_bounds__(256, 2) void uwgrad_images(UwBatch b)
{
    __shared__ __attribute__((aligned(16))) uint16_t lds[uwgrad_lds(UC_SRC_IMAGES, 0, 8, 0)];
    uwgrad_block<UC_SRC_IMAGES, 0, 0, 8, 0, DEPTH>(b, blockIdx.x, lds);
}

// False: a row is too wide for the 32-bit offsets.
template <int SRC, int CA, int CB, int CO>
static bool uwgrad_batch(UwBatch &b, int n, const UwFrame *fr, int &blocks)
{
    constexpr int pix = widest_pixel(SRC, CA, CB, CO, false);
    for (int i = 0; i < n; ++i)  // a strip's 32-bit offsets
        if ((uint64_t)pix * (UX_R * (uint64_t)fr[i].W + UX_C) >= kUOob) return false;
    b.n = n;
    blocks = 0;
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        b.blk_begin[i] = blocks;
        blocks += fr[i].nblk;
    }
    b.blk_begin[n] = blocks;
    return true;
}

// The first layer's weight gradient. Two strips in flight where a block walks more than two, one below
// (256x256, one strip: 10.6 us, 13.8 with two).
hipError_t launch_uwgrad_images(int n, const UwFrame *fr, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (n > XDN_MAX_FRAMES) return hipErrorInvalidValue;
    UwBatch b{};
    int blocks;
    if (!uwgrad_batch<UC_SRC_IMAGES, 0, 0, 8>(b, n, fr, blocks)) return hipErrorInvalidValue;
    if (blocks == 0) return hipSuccess;
    bool deep = false;
    for (int i = 0; i < n; ++i) deep |= udiv_up(fr[i].W, US_W) * udiv_up(fr[i].H, US_H) > 2 * fr[i].nblk;
    if (deep)
        hipLaunchKernelGGL((uwgrad_images<2>), dim3(blocks), dim3(256), 0, st, b);
    else
        hipLaunchKernelGGL((uwgrad_images<1>), dim3(blocks), dim3(256), 0, st, b);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// A layer's weight gradient and data gradient in one launch. Both wait for dY alone; as two launches they
// were two latencies in a row on small images (four 256x256 streams: 32 tiles and 64 strips at quarter
// resolution) and two nearly empty last waves on large ones. The first blocks take the weight gradient (both
// slices of the 48-channel layer), at most two a CU and the longest to run, the others the data gradient's
// tiles, which fill in behind them; each part starts at a multiple of eight blocks, so that its XCD order
// holds. The block bodies are those of separate kernels: the same bits. U-Net backward, two launches -> one:
// 256x256 153 -> 108 us, four of them 187 -> 147, 512x512 172 -> 132, 1280x720 281 -> 235, 1920x1080
// 442 -> 391, 3840x2160 1393 -> 1311. One strip in flight (two: 397 at 1920x1080); three waves per SIMD
// where two are given: 409; data gradient first: 422; both parts interleaved: 433.
// ---------------------------------------------------------------------------------------------
struct UbBatch {
    UwBatch w;
    UcBatch c;
    int w_blocks;
};
static_assert(sizeof(UbBatch) <= 4096, "kernel argument too large");

__host__ __device__ constexpr int up8(int n) { return (n + 7) & ~7; }

template <int SRC, int CA, int CB, int CO, int EPI, int WAVES>
__global__ __launch_bounds__(256, WAVES) void ubackward(UbBatch b)
{
    constexpr int CI = CA + CB;
    constexpr bool two = CI > 32;  // input slices
    constexpr int LW = uwgrad_lds(SRC, CI, CO, 0), LC = uconv_lds(UC_SRC_BF16, CO, false);
    __shared__ __attribute__((aligned(16))) uint16_t lds[LW > LC ? LW : LC];
    int bid = blockIdx.x;
    const int wb = up8(b.w_blocks);
    if (bid < wb)
    {
        if (bid < b.w_blocks) uwgrad_block<SRC, CA, CB, CO, 0, 1>(b.w, bid, lds);
        return;
    }
    bid -= wb;
    if constexpr (two)
    {
        if (bid < wb)
        {
            if (bid < b.w_blocks) uwgrad_block<UC_SRC_BF16, CA, CB, CO, 1, 1>(b.w, bid, lds);
            return;
        }
        bid -= wb;
    }
    uconv_block<UC_SRC_BF16, CO, 0, CI, EPI, false>(b.c, bid, lds);
}

template <int SRC, int CA, int CB, int CO, int EPI, int WAVES>
static hipError_t ubackward_t(int n, const UwFrame *wfr, const UcFrame *cfr, hipStream_t st)
{
    constexpr int CI = CA + CB;
    UbBatch b{};
    if (!uwgrad_batch<SRC, CA, CB, CO>(b.w, n, wfr, b.w_blocks)) return hipErrorInvalidValue;
    if (!uconv_batch<UC_SRC_BF16, CO, 0, CI, false>(b.c, n, cfr)) return hipErrorInvalidValue;
    if (b.c.map.total == 0) return hipSuccess;
    const int blocks = up8(b.w_blocks) * (CI > 32 ? 2 : 1) + b.c.map.total;
    hipLaunchKernelGGL((ubackward<SRC, CA, CB, CO, EPI, WAVES>), dim3(blocks), dim3(256), 0, st, b);
    return hipGetLastError();
}

hipError_t launch_ubackward(int kind, int n, const UwFrame *wfr, const UcFrame *cfr, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (n > XDN_MAX_FRAMES) return hipErrorInvalidValue;
    switch (kind)
    {
    case UBW_8_8: return ubackward_t<UC_SRC_BF16, 8, 0, 8, UC_EPI_MASK, 4>(n, wfr, cfr, st);
    case UBW_8_16: return ubackward_t<UC_SRC_BF16, 8, 0, 16, UC_EPI_PLAIN, 4>(n, wfr, cfr, st);
    case UBW_16_16: return ubackward_t<UC_SRC_BF16, 16, 0, 16, UC_EPI_MASK, 4>(n, wfr, cfr, st);
    case UBW_16_32: return ubackward_t<UC_SRC_BF16, 16, 0, 32, UC_EPI_PLAIN, 2>(n, wfr, cfr, st);
    case UBW_32_32: return ubackward_t<UC_SRC_BF16, 32, 0, 32, UC_EPI_MASK, 2>(n, wfr, cfr, st);
    case UBW_48_16: return ubackward_t<UC_SRC_UPCAT, 32, 16, 16, UC_EPI_PLAIN, 2>(n, wfr, cfr, st);
    case UBW_24_8: return ubackward_t<UC_SRC_UPCAT, 16, 8, 8, UC_EPI_PLAIN, 2>(n, wfr, cfr, st);
    default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------------------------
// Gradient of the max pool (its forward is in uconv3x3<..., POOL>)
// ---------------------------------------------------------------------------------------------
struct PoolBwBatch {
    int n, total;
    int begin[XDN_MAX_FRAMES + 1];
    PoolBwFrame f[XDN_MAX_FRAMES];
};

__device__ __forceinline__ int item_frame(const int *begin, int n, int i)
{
    int f = 0;
    while (f + 1 < n && i >= begin[f + 1]) ++f;
    return f;
}

// one item = one 2x2 window x one 8-channel chunk: vector loads of the window's four activations,
// skip gradients and outputs
template <int C>
__global__ __launch_bounds__(256) void pool_bwd(PoolBwBatch b)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= b.total) return;
    const int f = item_frame(b.begin, b.n, i);
    const PoolBwFrame &F = b.f[f];
    const int W = F.W, W2 = W / 2;
    const int li = i - b.begin[f], q = li % (C / 8), p2 = li / (C / 8);
    const int y2 = p2 / W2, x2 = p2 - y2 * W2;
    size_t pix[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) pix[k] = (size_t)(2 * y2 + (k >> 1)) * W + 2 * x2 + (k & 1);
    u32x4 a[4], sk[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        a[k] = *reinterpret_cast<const u32x4 *>(F.act + pix[k] * C + q * 8);
        sk[k] = *reinterpret_cast<const u32x4 *>(F.dskip + pix[k] * F.sstride + F.soff + q * 8);
    }
    const u32x4 dpw = *reinterpret_cast<const u32x4 *>(F.dpool + (size_t)p2 * C + q * 8);
    auto half = [](const u32x4 &w, int c) {
        const uint32_t x = c < 2 ? w.x : (c < 4 ? w.y : (c < 6 ? w.z : w.w));
        return (c & 1) ? u_hi(x) : u_lo(x);
    };
    float r[4][8];
#pragma unroll
    for (int c = 0; c < 8; ++c)
    {
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = half(a[k], c);
        // first maximum of the window in row-major order
        int arg = 0;
        float best = v[0];
#pragma unroll
        for (int k = 1; k < 4; ++k)
            if (v[k] > best) best = v[k], arg = k;
        const float dp = half(dpw, c);
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            const float g = (arg == k ? dp : 0.f) + half(sk[k], c);
            r[k][c] = v[k] > 0.f ? g : 0.f;
        }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
        *reinterpret_cast<u32x4 *>(F.dy + pix[k] * C + q * 8) =
            u32x4{u_pack2(r[k][0], r[k][1]), u_pack2(r[k][2], r[k][3]), u_pack2(r[k][4], r[k][5]),
                  u_pack2(r[k][6], r[k][7])};
}

template <int C>
static hipError_t pool_bwd_t(int n, const PoolBwFrame *fr, hipStream_t st)
{
    PoolBwBatch b{};
    b.n = n;
    int acc = 0;
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        b.begin[i] = acc;
        acc += (fr[i].H / 2) * (fr[i].W / 2) * (C / 8);
    }
    b.begin[n] = b.total = acc;
    if (acc == 0) return hipSuccess;
    hipLaunchKernelGGL(pool_bwd<C>, dim3(udiv_up(acc, 256)), dim3(256), 0, st, b);
    return hipGetLastError();
}

hipError_t launch_pool_bwd(int C, int n, const PoolBwFrame *fr, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (n > XDN_MAX_FRAMES) return hipErrorInvalidValue;
    if (C == 8) return pool_bwd_t<8>(n, fr, st);
    if (C == 16) return pool_bwd_t<16>(n, fr, st);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------------------------
// Transposed 1x1 stride-2 convolution
// ---------------------------------------------------------------------------------------------
struct CtBatch {
    int n, gpw;  // gpw: 32-pixel groups per wave (forward)
    int blk_begin[XDN_MAX_FRAMES + 1];
    CtFrame f[XDN_MAX_FRAMES];
};
static_assert(sizeof(CtBatch) <= 4096, "kernel argument too large");

// forward: out(2y,2x) = W in(y,x) + b, the other three outputs of the 2x2 block = b. FP32 MFMA
// (v_mfma_f32_32x32x2_f32: M = output channels, N = 32 coarse pixels, K = 2 input channels per
// step; a wave takes four such pixel groups with the weights in registers) on the FP32 master
// weights, so the products are those of FP32 arithmetic;
// a lane ends with 16 (C = 32) or 8 (C = 16) channels c(i) = 8(i/4) + 4h + i%4 of its pixel, and a
// permlane32 swap gives it 8 consecutive channels per 16-B store.
template <int C>
__global__ __launch_bounds__(256) void convT1x1s2(CtBatch b)
{
    constexpr int NI = C == 32 ? 16 : 8;  // accumulator rows holding output channels
    constexpr int NG = NI / 8;            // 16-B stores per output pixel and lane
    int f = 0;
    while (f + 1 < b.n && (int)blockIdx.x >= b.blk_begin[f + 1]) ++f;
    const CtFrame &F = b.f[f];
    const int li = blockIdx.x - b.blk_begin[f], GPW = b.gpw;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, px = lane & 31, h = lane >> 5;
    const int w = F.w_, np = F.h * w, W2 = 2 * w;
    // A operand of step s: W[co = px][ci = 2s + h]; the bias of the lane's outputs
    float wa[C / 2], bo[NI];
#pragma unroll
    for (int s2 = 0; s2 < C / 2; ++s2) wa[s2] = px < C ? F.w[px * C + 2 * s2 + h] : 0.f;
#pragma unroll
    for (int i = 0; i < NI; ++i) bo[i] = F.b[8 * (i >> 2) + 4 * h + (i & 3)];
    u32x4 vb[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g)
    {
        const int cb = 16 * g + 8 * h;
        vb[g] = u32x4{u_pack2(F.b[cb], F.b[cb + 1]), u_pack2(F.b[cb + 2], F.b[cb + 3]),
                      u_pack2(F.b[cb + 4], F.b[cb + 5]), u_pack2(F.b[cb + 6], F.b[cb + 7])};
    }
    for (int gi = 0; gi < GPW; ++gi)
    {
        const int p = ((li * 4 + wv) * GPW + gi) * 32 + px;
        if (p - px >= np) break;  // uniform across the wave
        // B operand: in[p][ci = 2s + h]
        float xb[C / 2];
#pragma unroll
        for (int s2 = 0; s2 < C / 2; ++s2) xb[s2] = 0.f;
        if (p < np)
#pragma unroll
            for (int c = 0; c < C; c += 8)
            {
                const u32x4 v = *reinterpret_cast<const u32x4 *>(F.in + (size_t)p * C + c);
                const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) xb[c / 2 + j] = h ? u_hi(wd[j]) : u_lo(wd[j]);
            }
        f32x16 acc;
#pragma unroll
        for (int k = 0; k < 16; ++k) acc[k] = 0.f;
#pragma unroll
        for (int s2 = 0; s2 < C / 2; ++s2) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[s2], xb[s2], acc, 0, 0, 0);
        uint32_t d[NI / 2];
#pragma unroll
        for (int q = 0; q < NI / 2; ++q) d[q] = u_pack2(acc[2 * q] + bo[2 * q], acc[2 * q + 1] + bo[2 * q + 1]);
        // lane h gathers channels 16g + 8h .. +7 (see conv3x3_l1 of k_cnn.hip)
        u32x4 v[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
            for (int e = 0; e < 2; ++e)
            {
                const auto sw = __builtin_amdgcn_permlane32_swap(d[4 * g + e], d[4 * g + 2 + e], false, false);
                v[g][e] = (uint32_t)sw[0];
                v[g][2 + e] = (uint32_t)sw[1];
            }
        if (p < np)
        {
            const int y = p / w, x = p - y * w;
#pragma unroll
            for (int k = 0; k < 4; ++k)
            {
                uint16_t *o = F.out + ((size_t)(2 * y + (k >> 1)) * W2 + 2 * x + (k & 1)) * C + 8 * h;
#pragma unroll
                for (int g = 0; g < NG; ++g) *reinterpret_cast<u32x4 *>(o + 16 * g) = k == 0 ? v[g] : vb[g];
            }
        }
    }
}

// backward: blocks walk coarse pixels in chunks of 256, one per thread for the loads: the chunk's
// inputs and dOut(2y,2x) go to LDS as they are (bf16, pixel-major) and each thread adds the sum of
// dOut over its 2x2 output block to its bias-gradient sums. Each wave then takes 64 pixels of the
// chunk: dIn = W^T dOut(2y,2x) on FP32 MFMA for 32 channels (FP32 VALU for 16), FP32 master
// weights, masked by the input's ReLU; dW[ci][co] = sum in (x) dOut(2y,2x) on bf16 MFMA (M = ci,
// N = co, K = pixels; operands through ds_read_b64_tr_b16). The waves' accumulators and the
// threads' bias sums are reduced through LDS in a fixed order at the end.
template <int C>
__global__ __launch_bounds__(256) void convT_bwd(CtBatch b)
{
    static_assert(C == 16 || C == 32, "channel count");
    constexpr int Q = C / 8;
    __shared__ __attribute__((aligned(16))) uint16_t tile[2][256 * C];  // inputs, dOut(2y,2x)
    __shared__ float red[4][C * C + C];
    __shared__ __attribute__((aligned(16))) float ws[C == 16 ? C * C : 4];  // [co][ci] (VALU dIn)
    int f = 0;
    while (f + 1 < b.n && (int)blockIdx.x >= b.blk_begin[f + 1]) ++f;
    const CtFrame &F = b.f[f];
    const int li = blockIdx.x - b.blk_begin[f], nblk = b.blk_begin[f + 1] - b.blk_begin[f];
    const int h = F.h, w = F.w_, np = h * w, W2 = 2 * w;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    constexpr int NI = C == 32 ? 16 : 8;  // dIn accumulator rows holding input channels
    // C = 32: A operand of the dIn product, step s: W^T[ci = lane%32][co = 2s + lane/32]
    float wt[C == 32 ? C / 2 : 1];
    if constexpr (C == 32)
#pragma unroll
        for (int s2 = 0; s2 < C / 2; ++s2) wt[s2] = F.w[(2 * s2 + (lane >> 5)) * C + (lane & 31)];
    else
        for (int e = tid; e < C * C; e += 256) ws[e] = F.w[e];
    float bacc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) bacc[c] = 0.f;
    typedef __attribute__((ext_vector_type(C == 32 ? 16 : 4))) float accv;
    accv acc;
#pragma unroll
    for (int k = 0; k < (C == 32 ? 16 : 4); ++k) acc[k] = 0.f;
    // transposing-read addressing (see ld_tr of k_cnn.hip): lane s of a 16-lane group addresses
    // pixel +s/4, channels +4(s%4)
    const int s16 = lane & 15, jq = s16 >> 2, qq = s16 & 3;
    for (int base = li * 256; base < np; base += nblk * 256)
    {
        __syncthreads();  // the previous chunk's tiles are read
        const int p = base + tid;
        u32x4 xv[Q], gv[Q];
#pragma unroll
        for (int k = 0; k < Q; ++k) xv[k] = gv[k] = u32x4{0u, 0u, 0u, 0u};
        float gs[C];
#pragma unroll
        for (int c = 0; c < C; ++c) gs[c] = 0.f;
        if (p < np)
        {
            const int y = p / w, xx = p - y * w;
#pragma unroll
            for (int k = 0; k < Q; ++k) xv[k] = *reinterpret_cast<const u32x4 *>(F.in + (size_t)p * C + 8 * k);
#pragma unroll
            for (int t = 0; t < 4; ++t)
            {
                const uint16_t *gp = F.dout + ((size_t)(2 * y + (t >> 1)) * W2 + 2 * xx + (t & 1)) * F.dstride;
#pragma unroll
                for (int k = 0; k < Q; ++k)
                {
                    const u32x4 v = *reinterpret_cast<const u32x4 *>(gp + 8 * k);
                    if (t == 0) gv[k] = v;
                    const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        gs[8 * k + 2 * j] += u_lo(wd[j]);
                        gs[8 * k + 2 * j + 1] += u_hi(wd[j]);
                    }
                }
            }
        }
#pragma unroll
        for (int k = 0; k < Q; ++k)
        {
            *reinterpret_cast<u32x4 *>(&tile[0][tid * C + 8 * k]) = xv[k];
            *reinterpret_cast<u32x4 *>(&tile[1][tid * C + 8 * k]) = gv[k];
        }
#pragma unroll
        for (int c = 0; c < C; ++c) bacc[c] += gs[c];
        __syncthreads();  // this chunk's tiles are visible
        // dIn. C = 32: FP32 MFMA (A = W^T from registers, B = dOut(2y,2x) of the wave's 32-pixel group
        // from the tile), masked by the staged input and stored through the permlane32 swap. C = 16
        // (half the MFMA rows would be padding): FP32 VALU per thread, output channels in order.
        if constexpr (C == 16)
        {
            if (p < np)
            {
                float x[C], g[C];
#pragma unroll
                for (int k = 0; k < Q; ++k)
                {
                    const uint32_t xw[4] = {xv[k].x, xv[k].y, xv[k].z, xv[k].w};
                    const uint32_t gw[4] = {gv[k].x, gv[k].y, gv[k].z, gv[k].w};
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                    {
                        x[8 * k + 2 * j] = u_lo(xw[j]); x[8 * k + 2 * j + 1] = u_hi(xw[j]);
                        g[8 * k + 2 * j] = u_lo(gw[j]); g[8 * k + 2 * j + 1] = u_hi(gw[j]);
                    }
                }
                float d[C];
#pragma unroll
                for (int c = 0; c < C; ++c) d[c] = 0.f;
#pragma unroll
                for (int co = 0; co < C; ++co)
#pragma unroll
                    for (int c = 0; c < C; c += 4)
                    {
                        const float4 wq = *reinterpret_cast<const float4 *>(&ws[co * C + c]);
                        d[c] += wq.x * g[co]; d[c + 1] += wq.y * g[co]; d[c + 2] += wq.z * g[co]; d[c + 3] += wq.w * g[co];
                    }
#pragma unroll
                for (int c = 0; c < C; c += 8)
                    *reinterpret_cast<u32x4 *>(F.din + (size_t)p * C + c) =
                        u32x4{u_pack2(x[c] > 0.f ? d[c] : 0.f, x[c + 1] > 0.f ? d[c + 1] : 0.f),
                              u_pack2(x[c + 2] > 0.f ? d[c + 2] : 0.f, x[c + 3] > 0.f ? d[c + 3] : 0.f),
                              u_pack2(x[c + 4] > 0.f ? d[c + 4] : 0.f, x[c + 5] > 0.f ? d[c + 5] : 0.f),
                              u_pack2(x[c + 6] > 0.f ? d[c + 6] : 0.f, x[c + 7] > 0.f ? d[c + 7] : 0.f)};
            }
        }
        else
#pragma unroll
        for (int gq = 0; gq < 2; ++gq)
        {
            const int pl = 64 * wv + 32 * gq + (lane & 31), hh = lane >> 5;
            float xb[C / 2];
#pragma unroll
            for (int k = 0; k < Q; ++k)
            {
                const u32x4 v = *reinterpret_cast<const u32x4 *>(&tile[1][pl * C + 8 * k]);
                const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) xb[4 * k + j] = hh ? u_hi(wd[j]) : u_lo(wd[j]);
            }
            f32x16 dacc;
#pragma unroll
            for (int k = 0; k < 16; ++k) dacc[k] = 0.f;
#pragma unroll
            for (int s2 = 0; s2 < C / 2; ++s2) dacc = __builtin_amdgcn_mfma_f32_32x32x2f32(wt[s2], xb[s2], dacc, 0, 0, 0);
            // rows c(i) = 8(i/4) + 4hh + i%4: four bf16 inputs at 8j + 4hh per j
            uint32_t d[NI / 2];
#pragma unroll
            for (int j = 0; j < NI / 4; ++j)
            {
                const uint2 xm = *reinterpret_cast<const uint2 *>(&tile[0][pl * C + 8 * j + 4 * hh]);
                const float xs[4] = {u_lo(xm.x), u_hi(xm.x), u_lo(xm.y), u_hi(xm.y)};
                d[2 * j] = u_pack2(xs[0] > 0.f ? dacc[4 * j] : 0.f, xs[1] > 0.f ? dacc[4 * j + 1] : 0.f);
                d[2 * j + 1] = u_pack2(xs[2] > 0.f ? dacc[4 * j + 2] : 0.f, xs[3] > 0.f ? dacc[4 * j + 3] : 0.f);
            }
            u32x4 v[NI / 8];
#pragma unroll
            for (int g = 0; g < NI / 8; ++g)
#pragma unroll
                for (int e = 0; e < 2; ++e)
                {
                    const auto sw = __builtin_amdgcn_permlane32_swap(d[4 * g + e], d[4 * g + 2 + e], false, false);
                    v[g][e] = (uint32_t)sw[0];
                    v[g][2 + e] = (uint32_t)sw[1];
                }
            const int pp = base + pl;
            if (pp < np)
#pragma unroll
                for (int g = 0; g < NI / 8; ++g)
                    *reinterpret_cast<u32x4 *>(F.din + (size_t)pp * C + 16 * g + 8 * hh) = v[g];
        }
        // dW: pixels past the end of the image were staged as zeros
        if constexpr (C == 32)
        {
            // 32x32x16: lane l holds row ci = l%32, k = pixels 8(l/32) + 0..7 of the K step
            const int grp = (lane >> 4) & 1, hh = lane >> 5;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
            {
                const int pb = 64 * wv + 16 * ks + 8 * hh + jq;
                const uint16_t *xp = &tile[0][pb * C + 16 * grp + 4 * qq];
                const uint16_t *gp = &tile[1][pb * C + 16 * grp + 4 * qq];
                const uint2 a0 = u_ld_tr(xp), a1 = u_ld_tr(xp + 4 * C);
                const uint2 b0 = u_ld_tr(gp), b1 = u_ld_tr(gp + 4 * C);
                acc = u_mfma(u32x4{a0.x, a0.y, a1.x, a1.y}, u32x4{b0.x, b0.y, b1.x, b1.y}, acc);
            }
        }
        else
        {
            // 16x16x32: lane l holds row ci = l%16, k = pixels 8(l/16) + 0..7 of the K step
            const int kg = lane >> 4;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
            {
                const int pb = 64 * wv + 32 * ks + 8 * kg + jq;
                const uint16_t *xp = &tile[0][pb * C + 4 * qq];
                const uint16_t *gp = &tile[1][pb * C + 4 * qq];
                const uint2 a0 = u_ld_tr(xp), a1 = u_ld_tr(xp + 4 * C);
                const uint2 b0 = u_ld_tr(gp), b1 = u_ld_tr(gp + 4 * C);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    __builtin_bit_cast(bf16x8, u32x4{a0.x, a0.y, a1.x, a1.y}),
                    __builtin_bit_cast(bf16x8, u32x4{b0.x, b0.y, b1.x, b1.y}), acc, 0, 0, 0);
            }
        }
    }
    // bias sums: wave reduction in a fixed order, then the four waves
#pragma unroll
    for (int c = 0; c < C; ++c) bacc[c] = u_wave_sum(bacc[c]);
    // accumulators: C[row = ci][col = co]
#pragma unroll
    for (int k = 0; k < (C == 32 ? 16 : 4); ++k)
    {
        const int ci = C == 32 ? 8 * (k >> 2) + 4 * (lane >> 5) + (k & 3) : 4 * (lane >> 4) + k;
        const int co = C == 32 ? (lane & 31) : (lane & 15);
        red[wv][ci * C + co] = acc[k];
    }
    if (lane == 0)
#pragma unroll
        for (int c = 0; c < C; ++c) red[wv][C * C + c] = bacc[c];
    __syncthreads();
    // compact partial: dW [ci][co], then db
    float *out = F.part + (size_t)li * compact_part(1, C, C);
    for (int e = tid; e < C * C + C; e += 256) out[e] = (red[0][e] + red[1][e]) + (red[2][e] + red[3][e]);
}

template <int C, bool BWD>
static hipError_t convT_t(int n, const CtFrame *fr, hipStream_t st)
{
    CtBatch b{};
    b.n = n;
    int acc = 0;
    if (!BWD)
    {
        // Pixel groups per wave (a wave loads the weights once): four where that leaves 192 blocks,
        // fewer below. 254 blocks at four (C = 32, 1920x1080): 14.2 us, 15.4 at two, 18.8 at one; 128
        // (C = 16, four 256x256 images): 8.2, 6.5, 6.6; 32 (C = 32): 12.0, 8.4, 6.6.
        long np = 0;
        for (int i = 0; i < n; ++i) np += (long)fr[i].h * fr[i].w_;
        for (b.gpw = 4; b.gpw > 1 && np < (long)192 * b.gpw * 4 * 32; b.gpw >>= 1) {}
    }
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        b.blk_begin[i] = acc;
        acc += BWD ? fr[i].nblk : udiv_up(fr[i].h * fr[i].w_, b.gpw * 4 * 32);
    }
    b.blk_begin[n] = acc;
    if (acc == 0) return hipSuccess;
    if (BWD)
        hipLaunchKernelGGL(convT_bwd<C>, dim3(acc), dim3(256), 0, st, b);
    else
        hipLaunchKernelGGL(convT1x1s2<C>, dim3(acc), dim3(256), 0, st, b);
    return hipGetLastError();
}

hipError_t launch_convT(int C, int n, const CtFrame *fr, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (n > XDN_MAX_FRAMES) return hipErrorInvalidValue;
    if (C == 16) return convT_t<16, false>(n, fr, st);
    if (C == 32) return convT_t<32, false>(n, fr, st);
    return hipErrorInvalidValue;
}

hipError_t launch_convT_bwd(int C, int n, const CtFrame *fr, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (n > XDN_MAX_FRAMES) return hipErrorInvalidValue;
    if (C == 16) return convT_t<16, true>(n, fr, st);
    if (C == 32) return convT_t<32, true>(n, fr, st);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------------------------
// Head backward: 1x1 convolution 8 -> 6
// ---------------------------------------------------------------------------------------------
struct HeadBatch {
    int n;
    int blk_begin[XDN_MAX_FRAMES + 1];
    HeadFrame f[XDN_MAX_FRAMES];
};
static_assert(sizeof(HeadBatch) <= 4096, "kernel argument too large");

__global__ __launch_bounds__(256) void head_bwd(HeadBatch b)
{
    __shared__ float red[4][54];
    int f = 0;
    while (f + 1 < b.n && (int)blockIdx.x >= b.blk_begin[f + 1]) ++f;
    const HeadFrame &F = b.f[f];
    const int li = blockIdx.x - b.blk_begin[f], nblk = b.blk_begin[f + 1] - b.blk_begin[f];
    const int np = F.H * F.W, tid = threadIdx.x;
    float w[48];
#pragma unroll
    for (int e = 0; e < 48; ++e) w[e] = F.w[e];
    float g[54];
#pragma unroll
    for (int e = 0; e < 54; ++e) g[e] = 0.f;
    // The loads of four pixels are in flight together; each thread sums its pixels in order. At the
    // HBM floor for 1920x1080 (116 MB, 27.7 -> 22.9 us); four 256x256 images: a chain of 16 pixels
    // a thread in 64 blocks, 15.8 -> 10.7 us.
    constexpr int U = 4;
    const int step = nblk * 256;
    for (int p0 = li * 256 + tid; p0 < np; p0 += U * step)
    {
        u32x4 v[U];
        float d[U][6];
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            const int p = p0 + u * step < np ? p0 + u * step : p0;
            v[u] = *reinterpret_cast<const u32x4 *>(F.in + (size_t)p * 8);
#pragma unroll
            for (int k = 0; k < 6; ++k) d[u][k] = F.dparam[(size_t)p * 6 + k];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            const int p = p0 + u * step;
            if (p >= np) break;
            const float in[8] = {u_lo(v[u].x), u_hi(v[u].x), u_lo(v[u].y), u_hi(v[u].y),
                                 u_lo(v[u].z), u_hi(v[u].z), u_lo(v[u].w), u_hi(v[u].w)};
            const float(&dp)[6] = d[u];
            uint32_t o[4];
#pragma unroll
            for (int c = 0; c < 8; c += 2)
            {
                float s0 = 0.f, s1 = 0.f;
#pragma unroll
                for (int k = 0; k < 6; ++k)
                {
                    s0 += w[c * 6 + k] * dp[k];
                    s1 += w[(c + 1) * 6 + k] * dp[k];
                }
                o[c / 2] = u_pack2(in[c] > 0.f ? s0 : 0.f, in[c + 1] > 0.f ? s1 : 0.f);
            }
            *reinterpret_cast<u32x4 *>(F.din + (size_t)p * 8) = u32x4{o[0], o[1], o[2], o[3]};
#pragma unroll
            for (int c = 0; c < 8; ++c)
#pragma unroll
                for (int k = 0; k < 6; ++k) g[c * 6 + k] += in[c] * dp[k];
#pragma unroll
            for (int k = 0; k < 6; ++k) g[48 + k] += dp[k];
        }
    }
#pragma unroll
    for (int e = 0; e < 54; ++e) g[e] = u_wave_sum(g[e]);
    if ((tid & 63) == 0)
#pragma unroll
        for (int e = 0; e < 54; ++e) red[tid >> 6][e] = g[e];
    __syncthreads();
    float *out = F.part + (size_t)li * compact_part(1, 8, 6);  // [8][6] then [6]
    if (tid < 54) out[tid] = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
}

hipError_t launch_head_bwd(int n, const HeadFrame *fr, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    if (n > XDN_MAX_FRAMES) return hipErrorInvalidValue;
    HeadBatch b{};
    b.n = n;
    int acc = 0;
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        b.blk_begin[i] = acc;
        acc += fr[i].nblk;
    }
    b.blk_begin[n] = acc;
    if (acc == 0) return hipSuccess;
    hipLaunchKernelGGL(head_bwd, dim3(acc), dim3(256), 0, st, b);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------
// Weight packing: fwd frag[t][kc][nt][lane] = W[t][kc*16 + 8h + j][nt*32 + lane%32],
// dgrad frag[t][kc][nt][lane] = W[8-t][nt*32 + lane%32][kc*16 + 8h + j]; zero outside ci x co
// ---------------------------------------------------------------------------------------------
constexpr int UPACK_MAX = 24;  // jobs per launch
struct UPackBatch {
    int n;
    UPackJob j[UPACK_MAX];
};
static_assert(sizeof(UPackBatch) <= 4096, "kernel argument too large");

__host__ __device__ inline int upack_items(const UPackJob &J)
{
    if (J.copy_n > 0) return (J.copy_n + 63) / 64;
    return 9 * ((J.ci + 15) / 16) * ((J.co + 31) / 32) + (J.frag_dgrad ? 9 * ((J.co + 15) / 16) * ((J.ci + 31) / 32) : 0);
}

__global__ __launch_bounds__(64) void upack(UPackBatch b)
{
    const UPackJob &J = b.j[blockIdx.y];
    const int lane = threadIdx.x, h = lane >> 5, n = lane & 31;
    const int item = blockIdx.x;
    if (J.copy_n > 0)
    {
        const int e = item * 64 + lane;
        if (e < J.copy_n) static_cast<float *>(J.frag_fwd)[e] = J.w[e];
        return;
    }
    const int kcf = (J.ci + 15) / 16, ntf = (J.co + 31) / 32;
    const int kcd = (J.co + 15) / 16, ntd = (J.ci + 31) / 32;
    const int nf = 9 * kcf * ntf, nd = J.frag_dgrad ? 9 * kcd * ntd : 0;
    if (item < nf)
    {
        const int t = item / (kcf * ntf), r = item - t * kcf * ntf, kc = r / ntf, nt = r - kc * ntf;
        const int co = nt * 32 + n;
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 8; j += 2)
        {
            const int c0 = kc * 16 + 8 * h + j, c1 = c0 + 1;
            const float a = (c0 < J.ci && co < J.co) ? J.w[(t * J.ci + c0) * J.co + co] : 0.f;
            const float bb = (c1 < J.ci && co < J.co) ? J.w[(t * J.ci + c1) * J.co + co] : 0.f;
            w[j >> 1] = u_pack2(a, bb);
        }
        static_cast<u32x4 *>(J.frag_fwd)[item * 64 + lane] = u32x4{w[0], w[1], w[2], w[3]};
        if (t == 0 && kc == 0 && h == 0) J.bias32[nt * 32 + n] = co < J.co ? J.b[co] : 0.f;
    }
    else if (item < nf + nd)
    {
        const int it = item - nf;
        const int t = it / (kcd * ntd), r = it - t * kcd * ntd, kc = r / ntd, nt = r - kc * ntd;
        const int ci = nt * 32 + n;
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 8; j += 2)
        {
            const int o0 = kc * 16 + 8 * h + j, o1 = o0 + 1;
            const float a = (o0 < J.co && ci < J.ci) ? J.w[((8 - t) * J.ci + ci) * J.co + o0] : 0.f;
            const float bb = (o1 < J.co && ci < J.ci) ? J.w[((8 - t) * J.ci + ci) * J.co + o1] : 0.f;
            w[j >> 1] = u_pack2(a, bb);
        }
        static_cast<u32x4 *>(J.frag_dgrad)[it * 64 + lane] = u32x4{w[0], w[1], w[2], w[3]};
    }
}

hipError_t launch_upack(int n, const UPackJob *jobs, hipStream_t st)
{
    for (int c0 = 0; c0 < n; c0 += UPACK_MAX)
    {
        const int m = n - c0 < UPACK_MAX ? n - c0 : UPACK_MAX;
        UPackBatch b{};
        b.n = m;
        int maxi = 0;
        for (int i = 0; i < m; ++i)
        {
            b.j[i] = jobs[c0 + i];
            const int items = upack_items(b.j[i]);
            maxi = items > maxi ? items : maxi;
        }
        if (maxi == 0) continue;
        hipLaunchKernelGGL(upack, dim3(maxi, m), dim3(64), 0, st, b);
        if (hipError_t e = hipGetLastError()) return e;
    }
    return hipSuccess;
}

}  // namespace xdn
