// Bandwidth-driven bilateral spatial filter on gfx950 (SpatialFilterKernel / SpatialFilterGradKernel,
// regression.cu.cc:33-195) and the fused per-frame training kernel.
//
// Weights w^X = exp(-b0|dX|^2 - b2|dalb|^2 - b3|dn|^2 - b4 ((dx/h)^2 + (dy/h)^2)) over an 11x11
// reflect-101 window, X in {A (band 0), B (band 1)}; the bands are pre-scaled by -log2(e) so each
// weight is one v_exp_f32. Nothing per tap is stored: every backward recomputes the weights.
//
// Kernels (16x16 output tile per 256-lane workgroup, the tile plus a 5-px halo staged in LDS as
// three float4 planes per pixel: (A.xyz, B.x), (B.yz, alb.xy), (alb.z, n.xyz)):
//   sf_tile<FWD>     unnormalized sums and weight sums                          VALU-bound
//   sf_tile<GRAD>    band gradient from upstream grads, weights recomputed     VALU-bound
//   sf_tile<TRAIN>   forward sums + the 32 band-gradient moments in registers, then the temporal
//                    accumulation, loss and the whole pointwise backward (aggregation ->
//                    weights -> band transform) in the epilogue; writes the output image and
//                    d loss / d network output                                  VALU-bound
//   sf_grad_inputs   gradient w.r.t. the four images (and the bands with BAND), gather form (no atomics): every pixel
//                    collects its own-center term and the terms of all centers whose (mirrored)
//                    window contains it, both from one pass over its window; two threads a pixel
//   sf_generic       windows past 15x15, direct loads (forward / grad)
#include "xdn_common.h"
#include "xdn_kernels.h"

namespace xdn {

enum { SF_FWD = 0, SF_GRAD = 1, SF_TRAIN = 2 };

struct SfBatch {
    TileMap map;
    SfFrame f[XDN_MAX_FRAMES];
    int half;
};
struct TrBatch {
    TileMap map;
    TrainFrame f[XDN_MAX_FRAMES];
};
static_assert(sizeof(SfBatch) <= 4096, "kernel argument too large");
static_assert(sizeof(TrBatch) <= 4096, "kernel argument too large");

constexpr int SF_T = 16;

// Per-tap state of one center pixel.
struct SfCenter {
    float3 cA, cB, ca, cn;
    float k0, k1, k2, k3, k4;  // -log2e * band, k4 already divided by half^2
};

struct SfAcc {
    float3 aA, aB;
    float sA, sB;
    float4 MA[4], MB[4];  // TRAIN: moments sum w*d_k*(c,1)
};

// One tap of the band gradient: g[k] += u * distance, with r2 the squared pixel distance. The roundings are
// spelled out so that every kernel that computes the band gradient gives the same bits.
__device__ __forceinline__ float2 sf_grad_tap(float (&g)[5], const float4 k, float k4, float DA, float DB, float Da,
                                              float Dn, float r2, float3 gA, float hA, float3 iA, float3 gB, float hB,
                                              float3 iB)
{
#pragma clang fp contract(off)
    const float sh = fmaf(k.z, Da, fmaf(k.w, Dn, k4 * r2));
    const float uA = fast_exp2(fmaf(k.x, DA, sh)) * fmaf(gA.z, iA.z, fmaf(gA.y, iA.y, fmaf(gA.x, iA.x, hA)));
    const float uB = fast_exp2(fmaf(k.y, DB, sh)) * fmaf(gB.z, iB.z, fmaf(gB.y, iB.y, fmaf(gB.x, iB.x, hB)));
    const float u = uA + uB;
    g[0] = fmaf(uA, DA, g[0]);
    g[1] = fmaf(uB, DB, g[1]);
    g[2] = fmaf(u, Da, g[2]);
    g[3] = fmaf(u, Dn, g[3]);
    g[4] = fmaf(u, r2, g[4]);
    return make_float2(uA, uB);
}

// |v|^2 in the roundings of dist2.
__device__ __forceinline__ float norm2(float3 v) { return fmaf(v.z, v.z, fmaf(v.x, v.x, v.y * v.y)); }
__device__ __forceinline__ float3 sub3(float3 a, float3 b) { return make_float3(a.x - b.x, a.y - b.y, a.z - b.z); }

// One tap of sf_tap<SF_FWD> at the squared pixel distances y2 and x2, with the roundings spelled out: an image's sums
// are the same bits in every kernel that takes its window rows in the same groups. (sf_tile leaves them to the
// compiler: the images it serves are served by no other kernel.)
__device__ __forceinline__ void sf_fwd_tap(const SfCenter &C, SfAcc &acc, float3 iA, float3 iB, float3 ia, float3 in,
                                           float y2, float x2)
{
#pragma clang fp contract(off)
    const float sh = fmaf(C.k2, norm2(sub3(C.ca, ia)), fmaf(C.k3, norm2(sub3(C.cn, in)), fmaf(C.k4, y2, C.k4 * x2)));
    const float wA = fast_exp2(fmaf(C.k0, norm2(sub3(C.cA, iA)), sh));
    const float wB = fast_exp2(fmaf(C.k1, norm2(sub3(C.cB, iB)), sh));
    acc.aA.x = fmaf(wA, iA.x, acc.aA.x); acc.aA.y = fmaf(wA, iA.y, acc.aA.y); acc.aA.z = fmaf(wA, iA.z, acc.aA.z);
    acc.aB.x = fmaf(wB, iB.x, acc.aB.x); acc.aB.y = fmaf(wB, iB.y, acc.aB.y); acc.aB.z = fmaf(wB, iB.z, acc.aB.z);
    acc.sA += wA;
    acc.sB += wB;
}

template <int MODE>
__device__ __forceinline__ void sf_tap(const SfCenter &C, SfAcc &acc, float3 iA, float3 iB, float3 ia, float3 in,
                                       float pd, float kpd)
{
    const float dA = dist2(C.cA, iA), dB = dist2(C.cB, iB), dal = dist2(C.ca, ia), dn = dist2(C.cn, in);
    const float sh = C.k2 * dal + (C.k3 * dn + kpd);
    const float wA = fast_exp2(C.k0 * dA + sh);
    const float wB = fast_exp2(C.k1 * dB + sh);
    acc.aA.x += wA * iA.x; acc.aA.y += wA * iA.y; acc.aA.z += wA * iA.z;
    acc.aB.x += wB * iB.x; acc.aB.y += wB * iB.y; acc.aB.z += wB * iB.z;
    acc.sA += wA;
    acc.sB += wB;
    if (MODE == SF_TRAIN)
    {
        const float mA[4] = {wA * dA, wA * dal, wA * dn, wA * pd};
        const float mB[4] = {wB * dB, wB * dal, wB * dn, wB * pd};
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            acc.MA[k].x += mA[k] * iA.x; acc.MA[k].y += mA[k] * iA.y; acc.MA[k].z += mA[k] * iA.z;
            acc.MA[k].w += mA[k];
            acc.MB[k].x += mB[k] * iB.x; acc.MB[k].y += mB[k] * iB.y; acc.MB[k].z += mB[k] * iB.z;
            acc.MB[k].w += mB[k];
        }
    }
}

__device__ __forceinline__ void sf_zero(SfAcc &a)
{
    a.aA = a.aB = make_float3(0.f, 0.f, 0.f);
    a.sA = a.sB = 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) a.MA[k] = a.MB[k] = make_float4(0.f, 0.f, 0.f, 0.f);
}

__device__ __forceinline__ void sf_center_bands(SfCenter &C, const float *band, size_t c, int half)
{
    const float *b = band + 5 * c;
    C.k0 = -kLog2e * b[0];
    C.k1 = -kLog2e * b[1];
    C.k2 = -kLog2e * b[2];
    C.k3 = -kLog2e * b[3];
    C.k4 = -kLog2e * b[4] / (float)(half * half);
}

// The same from the network's raw output (band transform of scripts/main.py:110-113).
__device__ __forceinline__ void sf_center_param(SfCenter &C, const float *param, uint32_t c, int half)
{
    const float *pr = param + 6 * (size_t)c;
    float bnd[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) bnd[k] = 1.f / (pr[k] * pr[k] + 1e-4f);
    C.k0 = -kLog2e * bnd[0]; C.k1 = -kLog2e * bnd[1]; C.k2 = -kLog2e * bnd[2];
    C.k3 = -kLog2e * bnd[3]; C.k4 = -kLog2e * bnd[4] / (float)(half * half);
}

// Epilogue of the fused training kernel for one pixel; returns the pixel's loss sum.
// Follows aggregation_loss (scripts/main.py:214-248), its analytic gradient, the band-gradient
// contraction (regression.cu.cc:58-80) and the band/alpha transform (main.py:111-113).
__device__ __forceinline__ float train_epilogue(const TrainFrame &F, uint32_t c, const SfAcc &acc, float inv_count,
                                                float3 lab2, float3 lab1)
{
    // the five bandwidth outputs are read again at the end, where the band transform needs them:
    // kept live from here they push the epilogue past the registers of five resident blocks
    const float *pr = F.param + 6 * (size_t)c;
    const float alpha = 1.f / (1.f + __expf(-pr[5]));
    const float d1 = acc.sA + 1e-4f, d2 = acc.sB + 1e-4f;
    const float i1 = 1.f / d1, i2 = 1.f / d2, i12 = 1.f / (acc.sA + acc.sB + 1e-4f);
    const float op = F.opacity[c] > 0.f ? 1.f : 0.f;
    const float s = F.succ_e[c] * F.succ_prev[c];
    const float a = s * alpha + (1.f - s);
    const float3 pv = ld3(F.prev_out, c);
    const float3 plab1 = ld3(F.prev_ols2, c), plab2 = ld3(F.prev_ols1, c);
    const float o1v[3] = {acc.aA.x * i1, acc.aA.y * i1, acc.aA.z * i1};
    const float o2v[3] = {acc.aB.x * i2, acc.aB.y * i2, acc.aB.z * i2};
    const float ov[3] = {(acc.aA.x + acc.aB.x) * i12, (acc.aA.y + acc.aB.y) * i12, (acc.aA.z + acc.aB.z) * i12};
    const float pvv[3] = {pv.x, pv.y, pv.z};
    const float l1v[3] = {lab1.x, lab1.y, lab1.z}, l2v[3] = {lab2.x, lab2.y, lab2.z};
    const float p1v[3] = {plab1.x, plab1.y, plab1.z}, p2v[3] = {plab2.x, plab2.y, plab2.z};
    const float cg = 0.25f * op * inv_count;
    float lsum = 0.f, ga = 0.f;
    float outl[3], outv[3], gA[3], gB[3], lossv[3];
    float hA = 0.f, hB = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k)
    {
        const float o = (a * ov[k] + (1.f - a) * pvv[k]) * op;
        outl[k] = o;
        outv[k] = fmaxf(0.f, expm1f(o));
        const float o1 = a * o1v[k] + (1.f - a) * pvv[k];
        const float o2 = a * o2v[k] + (1.f - a) * pvv[k];
        const float r1 = 1.f / (l1v[k] * l1v[k] + 1e-2f), r2 = 1.f / (l2v[k] * l2v[k] + 1e-2f);
        const float q1 = 1.f / (p1v[k] * p1v[k] + 1e-2f), q2 = 1.f / (p2v[k] * p2v[k] + 1e-2f);
        const float e1 = o1 - l1v[k], e2 = o2 - l2v[k], f1 = o1 - p1v[k], f2 = o2 - p2v[k];
        const float l = ((e1 * e1 * r1 + e2 * e2 * r2) * 0.5f + (f1 * f1 * q1 + f2 * f2 * q2) * 0.5f) * 0.5f * op;
        lossv[k] = l;
        lsum += l;
        const float g1 = cg * 2.f * (e1 * r1 + f1 * q1);
        const float g2 = cg * 2.f * (e2 * r2 + f2 * q2);
        ga += g1 * (o1v[k] - pvv[k]) + g2 * (o2v[k] - pvv[k]);
        const float go1 = a * g1, go2 = a * g2;
        gA[k] = go1 * i1;
        gB[k] = go2 * i2;
        hA -= go1 * o1v[k] * i1;  // d out1 / d sumw1 = -sum1 / d1^2 = -out1 / d1
        hB -= go2 * o2v[k] * i2;
    }
    st3(F.out_log, c, make_float3(outl[0], outl[1], outl[2]));
    st3(F.out, c, make_float3(outv[0], outv[1], outv[2]));
    if (F.loss) st3(F.loss, c, make_float3(lossv[0], lossv[1], lossv[2]));
    // band gradients: d w / d b_k = -d_k w  ->  dL/db_k = -(<g, M_k.xyz> + h M_k.w)
    float oA[4], oB[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
    {
        oA[k] = -(gA[0] * acc.MA[k].x + gA[1] * acc.MA[k].y + gA[2] * acc.MA[k].z + hA * acc.MA[k].w);
        oB[k] = -(gB[0] * acc.MB[k].x + gB[1] * acc.MB[k].y + gB[2] * acc.MB[k].z + hB * acc.MB[k].w);
    }
    const float gb[5] = {oA[0], oB[0], oA[1] + oB[1], oA[2] + oB[2], oA[3] + oB[3]};
    float x[5];  // all five loaded before the first store (the stores may alias them as far as the
#pragma unroll  // compiler knows)
    for (int k = 0; k < 5; ++k) x[k] = pr[k];
    float *dp = F.dparam + 6 * (size_t)c;
#pragma unroll
    for (int k = 0; k < 5; ++k)
    {
        const float band = 1.f / (x[k] * x[k] + 1e-4f);
        dp[k] = gb[k] * (-2.f * x[k] * band * band);
    }
    dp[5] = s * ga * alpha * (1.f - alpha);
    return lsum;
}

template <int HALF, int MODE, class Batch>
__device__ __forceinline__ void sf_tile_body(const Batch &b, float *red)
{
    constexpr int E = SF_T + 2 * HALF;
    __shared__ float4 s0[E * E], s1[E * E], s2[E * E];
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const auto &F = b.f[L.f];
    const int H = F.H, W = F.W;
    const int x0 = L.tx * SF_T, y0 = L.ty * SF_T;
    const float *IA, *IB;
    if constexpr (MODE == SF_TRAIN) { IA = F.ols1; IB = F.ols2; }
    else { IA = F.ia; IB = F.ib; }
    for (int i = threadIdx.x; i < E * E; i += 256)
    {
        const int ly = i / E, lx = i - ly * E;
        // halo rows/columns past the last live pixel + HALF are never read: clamp them so the mirror
        // stays inside the image for partial tiles
        const int gy = mirror(min(y0 + ly - HALF, H - 1 + HALF), H), gx = mirror(min(x0 + lx - HALF, W - 1 + HALF), W);
        const size_t p = (size_t)gy * W + gx;
        const float3 a = ld3(IA, p), bb = ld3(IB, p), al = ld3(F.alb, p), n = ld3(F.nrm, p);
        s0[i] = make_float4(a.x, a.y, a.z, bb.x);
        s1[i] = make_float4(bb.y, bb.z, al.x, al.y);
        s2[i] = make_float4(al.z, n.x, n.y, n.z);
    }
    __syncthreads();
    const int lx = threadIdx.x & (SF_T - 1), ly = threadIdx.x / SF_T;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cx = x0 + lx, cy = y0 + ly;
    const bool live = cx < W && cy < H;
    float lsum = 0.f;
    if (live)
    {
        const uint32_t c = (uint32_t)cy * (uint32_t)W + (uint32_t)cx;  // a frame has < 2^32 pixels
        const int q0 = (ly + HALF) * E + lx + HALF;
        SfCenter C;
        {
            const float4 P0 = s0[q0], P1 = s1[q0], P2 = s2[q0];
            C.cA = make_float3(P0.x, P0.y, P0.z);
            C.cB = make_float3(P0.w, P1.x, P1.y);
            C.ca = make_float3(P1.z, P1.w, P2.x);
            C.cn = make_float3(P2.y, P2.z, P2.w);
        }
        if constexpr (MODE == SF_TRAIN)
        {
            sf_center_param(C, F.param, c, HALF);
        }
        else
            sf_center_bands(C, F.band, c, HALF);
        SfAcc acc;
        sf_zero(acc);
        constexpr float inv_h2 = 1.f / (float)(HALF * HALF);
        for (int dy = -HALF; dy <= HALF; ++dy)
        {
            const float pdy = (float)(dy * dy) * inv_h2;
            const float kdy = C.k4 * (float)(dy * dy);
            const int base = (ly + HALF + dy) * E + lx + HALF;
#pragma unroll
            for (int dx = -HALF; dx <= HALF; ++dx)
            {
                const int q = base + dx;
                const float4 P0 = s0[q], P1 = s1[q], P2 = s2[q];
                const float pd = pdy + (float)(dx * dx) * inv_h2;
                const float kpd = kdy + C.k4 * (float)(dx * dx);
                sf_tap<MODE>(C, acc, make_float3(P0.x, P0.y, P0.z), make_float3(P0.w, P1.x, P1.y),
                             make_float3(P1.z, P1.w, P2.x), make_float3(P2.y, P2.z, P2.w), pd, kpd);
            }
        }
        if constexpr (MODE == SF_FWD)
        {
            st3(F.accA, c, acc.aA);
            st3(F.accB, c, acc.aB);
            F.wsA[c] = acc.sA;
            F.wsB[c] = acc.sB;
        }
        else
        {
            const float inv_count = 1.f / (3.f * (float)H * (float)W);
            lsum = train_epilogue(F, c, acc, inv_count, C.cA, C.cB);
        }
    }
    if constexpr (MODE == SF_TRAIN)
    {
        // deterministic per-tile loss partial: wave reduction then 4 waves through LDS (wave and lane
        // from a wave-uniform value and the lane count, so no thread index stays live across the taps)
        for (int off = 32; off > 0; off >>= 1) lsum += __shfl_down(lsum, off);
        const bool lane0 = __lane_id() == 0;
        if (lane0) red[wave] = lsum;
        __syncthreads();
        if (wave == 0 && lane0) F.loss_part[tile - b.map.begin[L.f]] = (red[0] + red[1]) + (red[2] + red[3]);
    }
}

// Five waves per SIMD, what the LDS of the 11x11 tile allows: win 7 at 1920x1080 125 -> 113 us, win 11 as before.
template <int HALF>
__global__ __launch_bounds__(256, 5) void sf_tile(SfBatch b)
{
    sf_tile_body<HALF, SF_FWD>(b, nullptr);
}

// First of the window rows of group p of P, from the middle row.
template <int HALF, int P>
__device__ __forceinline__ int sf_row0(int p)
{
    return (2 * HALF + 1) * p / P - HALF;
}

// The window rows of a pixel are summed in P groups, each from zero and the groups' sums added in order, by G
// threads (groups of 256 threads of the block, each taking P / G row groups, whose sums meet in LDS): G = 4 or 2
// for launches that leave the chip idle, where a 16x16 tile then runs 4 G waves instead of a chain of 121 taps in
// four, and GRAD at every size. P is the image's, so that its bits do not depend on what it is launched with.
template <int HALF, int MODE, int G, int P>
__global__ __launch_bounds__(256 * G, G == 1 ? 5 : 1) void sf_tile_split(SfBatch b)
{
    static_assert(MODE == SF_FWD || MODE == SF_GRAD, "the training tile is not split");
    static_assert(P % G == 0, "whole row groups a thread");
    constexpr int E = SF_T + 2 * HALF, NV = MODE == SF_FWD ? 8 : 5, Q = P / G;
    constexpr int RED = (P - Q) * NV * 256;  // floats of the reduction, which reuses the tile
    __shared__ float4 s[3][E * E > RED / 12 ? E * E : (RED + 11) / 12];
    const TileLoc L = locate(b.map, xcd_tile(blockIdx.x, b.map.total));
    const SfFrame &F = b.f[L.f];
    const int H = F.H, W = F.W;
    const int x0 = L.tx * SF_T, y0 = L.ty * SF_T;
    for (int i = threadIdx.x; i < E * E; i += 256 * G)
    {
        const int ly = i / E, lx = i - ly * E;
        const int gy = mirror(min(y0 + ly - HALF, H - 1 + HALF), H), gx = mirror(min(x0 + lx - HALF, W - 1 + HALF), W);
        const size_t p = (size_t)gy * W + gx;
        const float3 a = ld3(F.ia, p), bb = ld3(F.ib, p), al = ld3(F.alb, p), n = ld3(F.nrm, p);
        s[0][i] = make_float4(a.x, a.y, a.z, bb.x);
        s[1][i] = make_float4(bb.y, bb.z, al.x, al.y);
        s[2][i] = make_float4(al.z, n.x, n.y, n.z);
    }
    const int t = threadIdx.x & 255, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int lx = t & (SF_T - 1), ly = t / SF_T;
    const int cx = x0 + lx, cy = y0 + ly;
    const bool live = cx < W && cy < H;
    // lanes past the image run along on the last pixel (nothing of theirs is stored)
    const size_t c = (size_t)min(cy, H - 1) * W + min(cx, W - 1);
    SfCenter C;
    sf_center_bands(C, F.band, c, HALF);
    float3 gA = make_float3(0.f, 0.f, 0.f), gB = gA;
    float hA = 0.f, hB = 0.f;
    if constexpr (MODE == SF_GRAD)
    {
        gA = ld3(F.gaccA, c); gB = ld3(F.gaccB, c); hA = F.gwA[c]; hB = F.gwB[c];
    }
    __syncthreads();
    const int q0 = (ly + HALF) * E + lx + HALF;
    {
        const float4 P0 = s[0][q0], P1 = s[1][q0], P2 = s[2][q0];
        C.cA = make_float3(P0.x, P0.y, P0.z);
        C.cB = make_float3(P0.w, P1.x, P1.y);
        C.ca = make_float3(P1.z, P1.w, P2.x);
        C.cn = make_float3(P2.y, P2.z, P2.w);
    }
    constexpr float inv_h2 = 1.f / (float)(HALF * HALF);
    float sum[Q][NV];  // of the thread's row groups
#pragma unroll
    for (int q = 0; q < Q; ++q)
    {
        SfAcc acc;
        sf_zero(acc);
        float g[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        const int dy1 = sf_row0<HALF, P>(Q * grp + q + 1);
#pragma unroll 1
        for (int dy = sf_row0<HALF, P>(Q * grp + q); dy < dy1; ++dy)
        {
            const float y2 = (float)(dy * dy);
            const int base = q0 + dy * E;
#pragma unroll
            for (int dx = -HALF; dx <= HALF; ++dx)
            {
                const float4 P0 = s[0][base + dx], P1 = s[1][base + dx], P2 = s[2][base + dx];
                const float3 iA = make_float3(P0.x, P0.y, P0.z), iB = make_float3(P0.w, P1.x, P1.y);
                const float3 ia = make_float3(P1.z, P1.w, P2.x), in = make_float3(P2.y, P2.z, P2.w);
                if constexpr (MODE == SF_FWD)
                    sf_fwd_tap(C, acc, iA, iB, ia, in, y2, (float)(dx * dx));
                else
                    sf_grad_tap(g, make_float4(C.k0, C.k1, C.k2, C.k3), C.k4, norm2(sub3(C.cA, iA)),
                                norm2(sub3(C.cB, iB)), norm2(sub3(C.ca, ia)), norm2(sub3(C.cn, in)),
                                y2 + (float)(dx * dx), gA, hA, iA, gB, hB, iB);
            }
        }
        if constexpr (MODE == SF_FWD)
        {
            const float a[8] = {acc.aA.x, acc.aA.y, acc.aA.z, acc.aB.x, acc.aB.y, acc.aB.z, acc.sA, acc.sB};
#pragma unroll
            for (int k = 0; k < NV; ++k) sum[q][k] = a[k];
        }
        else
#pragma unroll
            for (int k = 0; k < NV; ++k) sum[q][k] = g[k];
        if (G == 1 && q > 0)
#pragma unroll
            for (int k = 0; k < NV; ++k) sum[0][k] += sum[q][k];
    }
    float(&v)[NV] = sum[0];
    if constexpr (G > 1)
    {
        __syncthreads();  // the tile is dead
        float *red = reinterpret_cast<float *>(&s[0][0]);  // [P - Q][NV][256]
        static_assert(sizeof(s) >= sizeof(float) * RED, "reduction space");
        if (grp)
#pragma unroll
            for (int q = 0; q < Q; ++q)
#pragma unroll
                for (int k = 0; k < NV; ++k) red[((Q * (grp - 1) + q) * NV + k) * 256 + t] = sum[q][k];
        __syncthreads();
        if (grp) return;
#pragma unroll
        for (int p = 1; p < P; ++p)
#pragma unroll
            for (int k = 0; k < NV; ++k) v[k] += p < Q ? sum[p][k] : red[((p - Q) * NV + k) * 256 + t];
    }
    if (!live) return;
    if constexpr (MODE == SF_FWD)
    {
        st3(F.accA, c, make_float3(v[0], v[1], v[2]));
        st3(F.accB, c, make_float3(v[3], v[4], v[5]));
        F.wsA[c] = v[6];
        F.wsB[c] = v[7];
    }
    else
    {
        float *o = F.gband + 5 * c;
#pragma unroll
        for (int k = 0; k < NV; ++k) o[k] = (k == 4 ? -inv_h2 : -1.f) * v[k];
    }
}

// Five resident blocks per CU (32.5 KB of LDS each): 96 VGPRs instead of 106. The epilogue is kept
// lean for it (see train_epilogue); one 8-byte value is still spilled there, none in the tap loop.
template <int HALF>
__global__ __launch_bounds__(256, 5) void sf_train_tile(TrBatch b)
{
    __shared__ float red[4];
    sf_tile_body<HALF, SF_TRAIN>(b, red);
}

// The training tile for launches that leave the chip idle: the window rows of a pixel are split over two
// threads as in sf_tile_split, their 40 sums joined in LDS twenty at a time, over the tile.
template <int HALF>
__global__ __launch_bounds__(512) void sf_train_split(TrBatch b)
{
    constexpr int G = 2, E = SF_T + 2 * HALF, NV = 40, CH = 20, R = 2 * HALF + 1;
    __shared__ float4 s[3][E * E];
    __shared__ float red[4];
    static_assert(sizeof(s) >= sizeof(float) * CH * 256, "reduction space");
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const TrainFrame &F = b.f[L.f];
    const int H = F.H, W = F.W;
    const int x0 = L.tx * SF_T, y0 = L.ty * SF_T;
    for (int i = threadIdx.x; i < E * E; i += 256 * G)
    {
        const int ly = i / E, lx = i - ly * E;
        const int gy = mirror(min(y0 + ly - HALF, H - 1 + HALF), H), gx = mirror(min(x0 + lx - HALF, W - 1 + HALF), W);
        const size_t p = (size_t)gy * W + gx;
        const float3 a = ld3(F.ols1, p), bb = ld3(F.ols2, p), al = ld3(F.alb, p), n = ld3(F.nrm, p);
        s[0][i] = make_float4(a.x, a.y, a.z, bb.x);
        s[1][i] = make_float4(bb.y, bb.z, al.x, al.y);
        s[2][i] = make_float4(al.z, n.x, n.y, n.z);
    }
    const int t = threadIdx.x & 255, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int lx = t & (SF_T - 1), ly = t / SF_T;
    const int cx = x0 + lx, cy = y0 + ly;
    const bool live = cx < W && cy < H;
    // lanes past the image run along on the last pixel (nothing of theirs is stored)
    const uint32_t c = (uint32_t)min(cy, H - 1) * (uint32_t)W + (uint32_t)min(cx, W - 1);
    SfCenter C;
    sf_center_param(C, F.param, c, HALF);
    __syncthreads();
    const int q0 = (ly + HALF) * E + lx + HALF;
    {
        const float4 P0 = s[0][q0], P1 = s[1][q0], P2 = s[2][q0];
        C.cA = make_float3(P0.x, P0.y, P0.z);
        C.cB = make_float3(P0.w, P1.x, P1.y);
        C.ca = make_float3(P1.z, P1.w, P2.x);
        C.cn = make_float3(P2.y, P2.z, P2.w);
    }
    SfAcc acc;
    sf_zero(acc);
    constexpr float inv_h2 = 1.f / (float)(HALF * HALF);
#pragma unroll 1
    for (int dy = R * grp / G - HALF; dy < R * (grp + 1) / G - HALF; ++dy)
    {
        const float y2 = (float)(dy * dy), kdy = C.k4 * y2, pdy = y2 * inv_h2;
        const int base = q0 + dy * E;
#pragma unroll
        for (int dx = -HALF; dx <= HALF; ++dx)
        {
            const float4 P0 = s[0][base + dx], P1 = s[1][base + dx], P2 = s[2][base + dx];
            sf_tap<SF_TRAIN>(C, acc, make_float3(P0.x, P0.y, P0.z), make_float3(P0.w, P1.x, P1.y),
                             make_float3(P1.z, P1.w, P2.x), make_float3(P2.y, P2.z, P2.w),
                             pdy + (float)(dx * dx) * inv_h2, kdy + C.k4 * (float)(dx * dx));
        }
    }
    float *const v[NV] = {&acc.aA.x, &acc.aA.y, &acc.aA.z, &acc.aB.x, &acc.aB.y, &acc.aB.z, &acc.sA, &acc.sB,
                          &acc.MA[0].x, &acc.MA[0].y, &acc.MA[0].z, &acc.MA[0].w, &acc.MA[1].x, &acc.MA[1].y,
                          &acc.MA[1].z, &acc.MA[1].w, &acc.MA[2].x, &acc.MA[2].y, &acc.MA[2].z, &acc.MA[2].w,
                          &acc.MA[3].x, &acc.MA[3].y, &acc.MA[3].z, &acc.MA[3].w, &acc.MB[0].x, &acc.MB[0].y,
                          &acc.MB[0].z, &acc.MB[0].w, &acc.MB[1].x, &acc.MB[1].y, &acc.MB[1].z, &acc.MB[1].w,
                          &acc.MB[2].x, &acc.MB[2].y, &acc.MB[2].z, &acc.MB[2].w, &acc.MB[3].x, &acc.MB[3].y,
                          &acc.MB[3].z, &acc.MB[3].w};
    float *part = reinterpret_cast<float *>(&s[0][0]);  // [CH][256]
#pragma unroll
    for (int k0 = 0; k0 < NV; k0 += CH)
    {
        __syncthreads();  // the tile, or the first half of the sums, is read
        if (grp)
#pragma unroll
            for (int k = 0; k < CH; ++k) part[k * 256 + t] = *v[k0 + k];
        __syncthreads();
        if (!grp)
#pragma unroll
            for (int k = 0; k < CH; ++k) *v[k0 + k] += part[k * 256 + t];
    }
    float lsum = 0.f;
    if (!grp && live) lsum = train_epilogue(F, c, acc, 1.f / (3.f * (float)H * (float)W), C.cA, C.cB);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_down(lsum, off);
    const bool lane0 = __lane_id() == 0;
    if (!grp && lane0) red[wave] = lsum;
    __syncthreads();
    if (wave == 0 && lane0) F.loss_part[tile - b.map.begin[L.f]] = (red[0] + red[1]) + (red[2] + red[3]);
}

// Any window size: direct loads with the mirror boundary.
template <int MODE>
__global__ __launch_bounds__(256) void sf_generic(SfBatch b)
{
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const SfFrame &F = b.f[L.f];
    const int H = F.H, W = F.W, HALF = b.half;
    const int cx = L.tx * SF_T + (threadIdx.x & 15), cy = L.ty * SF_T + (threadIdx.x >> 4);
    if (cx >= W || cy >= H) return;
    const size_t c = (size_t)cy * W + cx;
    SfCenter C;
    C.cA = ld3(F.ia, c); C.cB = ld3(F.ib, c); C.ca = ld3(F.alb, c); C.cn = ld3(F.nrm, c);
    sf_center_bands(C, F.band, c, HALF);
    float3 gA = make_float3(0.f, 0.f, 0.f), gB = gA;
    float hA = 0.f, hB = 0.f;
    if (MODE == SF_GRAD)
    {
        gA = ld3(F.gaccA, c); gB = ld3(F.gaccB, c); hA = F.gwA[c]; hB = F.gwB[c];
    }
    SfAcc acc;
    sf_zero(acc);
    float g[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    for (int dy = -HALF; dy <= HALF; ++dy)
        for (int dx = -HALF; dx <= HALF; ++dx)
        {
            const size_t i = (size_t)mirror(cy + dy, H) * W + mirror(cx + dx, W);
            const float r2 = (float)(dx * dx + dy * dy);
            const float3 iA = ld3(F.ia, i), iB = ld3(F.ib, i), ia = ld3(F.alb, i), in = ld3(F.nrm, i);
            if (MODE == SF_FWD)
                sf_tap<MODE>(C, acc, iA, iB, ia, in, 0.f, C.k4 * r2);
            else
                sf_grad_tap(g, make_float4(C.k0, C.k1, C.k2, C.k3), C.k4, norm2(sub3(C.cA, iA)), norm2(sub3(C.cB, iB)),
                            norm2(sub3(C.ca, ia)), norm2(sub3(C.cn, in)), r2, gA, hA, iA, gB, hB, iB);
        }
    if (MODE == SF_FWD)
    {
        st3(F.accA, c, acc.aA);
        st3(F.accB, c, acc.aB);
        F.wsA[c] = acc.sA;
        F.wsB[c] = acc.sB;
    }
    else
    {
        float *o = F.gband + 5 * c;
#pragma unroll
        for (int k = 0; k < 5; ++k) o[k] = k == 4 ? -g[k] / (float)(HALF * HALF) : -g[k];
    }
}

// ---------------------------------------------------------------------------------------------
// Gradient w.r.t. the images (the reference returns None for them, scripts/ops.py:32).
// For every pixel q:
//   own term   (q as the center): for each tap i = mirror(q+d), with u = w (<g_q, c_i> + h_q):
//              dq += -2 b_q u (c_q - c_i)  (per image and band)
//   tap terms  (q as the tap of center p, mirror(p+d) = q):
//              dq += w g_p (direct, colour images only) + 2 b_p u_pq (c_p - c_q)
// For a neighbour r of q inside the image both terms run over the same pair (q, r): r is a tap of q and
// q a tap of r at the same distances, so one pass over the window computes each pair's four distances
// once and adds both terms with one coefficient per image,
//   dq += -2 (b_q u_qr + b_r u_rq) (c_q - c_r) + w_rq g_r,
// 79 FMA-class instructions and four exponentials a pair instead of about 120 and the index work of a
// tap-by-tap enumeration. Pixels within
// HALF of an image edge are also reached through the reflection: with q' = -q or 2n - 2 - q along an
// axis, they are taps of the centers p around q' too, at the distances of (p, q) and the pixel
// distance of p - q'; those pairs are a second loop that only blocks at an edge run.
// LDS: the tile plus halo of every per-pixel quantity (25 floats), 26x26 pixels for win 11: 67.6 KB, two
// blocks per CU, so a pixel's window rows are split over two threads (rows dy < 0 and dy >= 0, joined
// through LDS) for four waves per SIMD instead of two. VALU-bound: 512x512, win 11: 247 -> 102 us
// (128 us with one thread per pixel).
// BAND: the band gradient too. Its terms are the own terms' u against the pair's distances, which are at
// hand here: five FMAs a pair instead of a second launch that recomputes distances and weights (forward and
// both gradients at 512x512 163 -> 145 us, at 1920x1080 1044 -> 770 us).
// ---------------------------------------------------------------------------------------------
struct Yes {
    static constexpr bool value = true;
};
struct No {
    static constexpr bool value = false;
};

template <int HALF, bool BAND, int P>
__global__ __launch_bounds__(512) void sf_grad_inputs_tile(SfBatch b)
{
    constexpr int E = SF_T + 2 * HALF;
    constexpr float inv_h2 = 1.f / (float)(HALF * HALF);
    // per pixel: (A.xyz, B.x) (B.yz, alb.xy) (alb.z, n.xyz) (k0..k3) (k4, gA.xyz) (hA, gB.xyz) (hB) with
    // k = -log2e * band, k4 divided by HALF^2
    __shared__ float4 s[6][E * E];
    __shared__ float shB[E * E];
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const SfFrame &F = b.f[L.f];
    const int H = F.H, W = F.W;
    const int x0 = L.tx * SF_T, y0 = L.ty * SF_T;
    for (int i = threadIdx.x; i < E * E; i += 512)
    {
        const int ly = i / E, lx = i - ly * E;
        const int gy = mirror(min(y0 + ly - HALF, H - 1 + HALF), H), gx = mirror(min(x0 + lx - HALF, W - 1 + HALF), W);
        const size_t p = (size_t)gy * W + gx;
        const float3 a = ld3(F.ia, p), bb = ld3(F.ib, p), al = ld3(F.alb, p), n = ld3(F.nrm, p);
        SfCenter C;
        sf_center_bands(C, F.band, p, HALF);
        float3 gA = ld3(F.gaccA, p), gB = ld3(F.gaccB, p);
        float hA = F.gwA[p], hB = F.gwB[p];
        // a window position outside the image is a tap (of the mirrored pixel's values) but no center: its
        // weights are exp2(-inf) = 0, also at an infinite distance (-1 inf, where 0 inf would be NaN), and its
        // upstream gradients zero
        const int ux = x0 + lx - HALF, uy = y0 + ly - HALF;
        if (ux < 0 || uy < 0 || ux >= W || uy >= H)
        {
            C.k0 = C.k1 = C.k2 = C.k3 = -1.f;
            C.k4 = -__builtin_inff();
            hA = hB = 0.f;
            gA = gB = make_float3(0.f, 0.f, 0.f);
        }
        s[0][i] = make_float4(a.x, a.y, a.z, bb.x);
        s[1][i] = make_float4(bb.y, bb.z, al.x, al.y);
        s[2][i] = make_float4(al.z, n.x, n.y, n.z);
        s[3][i] = make_float4(C.k0, C.k1, C.k2, C.k3);
        s[4][i] = make_float4(C.k4, gA.x, gA.y, gA.z);
        s[5][i] = make_float4(hA, gB.x, gB.y, gB.z);
        shB[i] = hB;
    }
    __syncthreads();
    const int t = threadIdx.x & 255, grp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int lx = t & (SF_T - 1), ly = t / SF_T;
    const int qx = x0 + lx, qy = y0 + ly;
    const bool live = qx < W && qy < H;
    const int q0 = (ly + HALF) * E + lx + HALF;
    struct Px {
        float3 A, B, al, n;
    };
    auto image = [&](int k) {
        const float4 P0 = s[0][k], P1 = s[1][k], P2 = s[2][k];
        return Px{make_float3(P0.x, P0.y, P0.z), make_float3(P0.w, P1.x, P1.y), make_float3(P1.z, P1.w, P2.x),
                  make_float3(P2.y, P2.z, P2.w)};
    };
    struct Up {  // bands and upstream gradients
        float k0, k1, k2, k3, k4, hA, hB;
        float3 gA, gB;
    };
    auto upstream = [&](int k) {
        const float4 K = s[3][k], G = s[4][k], HG = s[5][k];
        return Up{K.x, K.y, K.z, K.w, G.x, HG.x, shB[k], make_float3(G.y, G.z, G.w), make_float3(HG.y, HG.z, HG.w)};
    };
    const Px Q = image(q0);
    const Up U = upstream(q0);
    const float3 zero = make_float3(0.f, 0.f, 0.f);
    float3 dA = zero, dB = zero, da = zero, dn = zero;  // sum of coefficient * (c_q - c_r)
    float3 eA = zero, eB = zero;                        // sum of w_rq g_r
    float g[5] = {0.f, 0.f, 0.f, 0.f, 0.f};             // BAND: sum of u_qr * distance
    // one pair (q, r) at the squared pixel distance r2: r's center term, and q's tap term where OWN
    auto pair = [&](int k, float r2, auto own) {
        constexpr bool OWN = decltype(own)::value;
        const Px R = image(k);
        const float3 xA = sub3(Q.A, R.A), xB = sub3(Q.B, R.B), xa = sub3(Q.al, R.al), xn = sub3(Q.n, R.n);
        const float DA = norm2(xA), DB = norm2(xB), Da = norm2(xa), Dn = norm2(xn);
        float cA = 0.f, cB = 0.f, ca = 0.f, cn = 0.f;
        if constexpr (OWN)
        {
            const float2 u2 = sf_grad_tap(g, make_float4(U.k0, U.k1, U.k2, U.k3), U.k4, DA, DB, Da, Dn, r2, U.gA, U.hA,
                                          R.A, U.gB, U.hB, R.B);
            const float u = u2.x + u2.y;
            cA = U.k0 * u2.x; cB = U.k1 * u2.y; ca = U.k2 * u; cn = U.k3 * u;
        }
        {
            const Up V = upstream(k);
            const float sh = V.k2 * Da + (V.k3 * Dn + V.k4 * r2);
            const float wA = fast_exp2(V.k0 * DA + sh), wB = fast_exp2(V.k1 * DB + sh);
            const float uA = wA * (V.gA.x * Q.A.x + V.gA.y * Q.A.y + V.gA.z * Q.A.z + V.hA);
            const float uB = wB * (V.gB.x * Q.B.x + V.gB.y * Q.B.y + V.gB.z * Q.B.z + V.hB);
            const float u = uA + uB;
            cA += V.k0 * uA; cB += V.k1 * uB; ca += V.k2 * u; cn += V.k3 * u;
            eA.x += wA * V.gA.x; eA.y += wA * V.gA.y; eA.z += wA * V.gA.z;
            eB.x += wB * V.gB.x; eB.y += wB * V.gB.y; eB.z += wB * V.gB.z;
        }
        dA.x += cA * xA.x; dA.y += cA * xA.y; dA.z += cA * xA.z;
        dB.x += cB * xB.x; dB.y += cB * xB.y; dB.z += cB * xB.z;
        da.x += ca * xa.x; da.y += ca * xa.y; da.z += ca * xa.z;
        dn.x += cn * xn.x; dn.y += cn * xn.y; dn.z += cn * xn.z;
    };
    // the row groups of sf_tile_split<GRAD>, for the same sums
    const int dy0 = grp ? 0 : -HALF, dy1 = grp ? HALF : -1, mid = sf_row0<HALF, 4>(2 * grp + 1);
    static_assert(P == 2 || P == 4, "row groups of the band gradient");
    float g0[5] = {0.f, 0.f, 0.f, 0.f, 0.f};  // BAND, P = 4: the first of the thread's two row groups
#pragma unroll 1
    for (int dy = dy0; dy <= dy1; ++dy)
    {
        if (BAND && P == 4 && dy == mid)
#pragma unroll
            for (int k = 0; k < 5; ++k) g0[k] = g[k], g[k] = 0.f;
        const int base = q0 + dy * E;
        const float y2 = (float)(dy * dy);
#pragma unroll
        for (int dx = -HALF; dx <= HALF; ++dx) pair(base + dx, y2 + (float)(dx * dx), Yes{});
    }
    // a pixel at most HALF from the first or last row or column is reached through the reflection
    if (live && (x0 <= HALF || y0 <= HALF || x0 + SF_T + HALF >= W || y0 + SF_T + HALF >= H))
    {
        // centers around the reflections of q (one or both axes reflected)
        const int vy[3] = {qy, qy > 0 ? -qy : INT_MIN, qy <= H - 2 ? 2 * H - 2 - qy : INT_MIN};
        const int vx[3] = {qx, qx > 0 ? -qx : INT_MIN, qx <= W - 2 ? 2 * W - 2 - qx : INT_MIN};
        for (int a = 0; a < 9; ++a)
        {
            const int ay = a / 3, ax = a - 3 * ay;
            if (a == 0 || vy[ay] == INT_MIN || vx[ax] == INT_MIN) continue;
            const int py0 = max(0, vy[ay] - HALF), py1 = min(H - 1, vy[ay] + HALF);
            const int px0 = max(0, vx[ax] - HALF), px1 = min(W - 1, vx[ax] + HALF);
            for (int py = py0 + grp; py <= py1; py += 2)
                for (int px = px0; px <= px1; ++px)
                {
                    const int ey = py - vy[ay], ex = px - vx[ax];
                    pair((py - y0 + HALF) * E + (px - x0 + HALF), (float)(ex * ex + ey * ey), No{});
                }
        }
    }
    // the second half of the rows joins through LDS (the tile is dead)
    __syncthreads();
    constexpr int NV = !BAND ? 18 : (P == 4 ? 28 : 23);
    float *red = reinterpret_cast<float *>(&s[0][0]);  // [NV][256]
    static_assert(sizeof(s) >= NV * 256 * sizeof(float), "reduction space");
    if (grp)
    {
        const float v[18] = {dA.x, dA.y, dA.z, dB.x, dB.y, dB.z, da.x, da.y, da.z,
                             dn.x, dn.y, dn.z, eA.x, eA.y, eA.z, eB.x, eB.y, eB.z};
#pragma unroll
        for (int k = 0; k < 18; ++k) red[k * 256 + t] = v[k];
        if constexpr (BAND)
#pragma unroll
            for (int k = 0; k < 5; ++k)
            {
                if (P == 4) red[(23 + k) * 256 + t] = g0[k];
                red[(18 + k) * 256 + t] = g[k];
            }
    }
    __syncthreads();
    if (grp || !live) return;
    {
        float3 *const v[6] = {&dA, &dB, &da, &dn, &eA, &eB};
#pragma unroll
        for (int k = 0; k < 6; ++k)
        {
            v[k]->x += red[(3 * k) * 256 + t];
            v[k]->y += red[(3 * k + 1) * 256 + t];
            v[k]->z += red[(3 * k + 2) * 256 + t];
        }
    }
    // the coefficients hold k = -log2e b for the bands: -2 b = 2 ln2 k
    constexpr float kScale = 2.f * 0.693147180559945309f;
    const size_t c = (size_t)qy * W + qx;
    if (F.gia) st3(F.gia, c, make_float3(eA.x + kScale * dA.x, eA.y + kScale * dA.y, eA.z + kScale * dA.z));
    if (F.gib) st3(F.gib, c, make_float3(eB.x + kScale * dB.x, eB.y + kScale * dB.y, eB.z + kScale * dB.z));
    if (F.galb) st3(F.galb, c, make_float3(kScale * da.x, kScale * da.y, kScale * da.z));
    if (F.gnrm) st3(F.gnrm, c, make_float3(kScale * dn.x, kScale * dn.y, kScale * dn.z));
    if constexpr (BAND)
    {
        float *o = F.gband + 5 * c;
#pragma unroll
        for (int k = 0; k < 5; ++k)
        {
            float v = g[k];
            if (P == 4) v = (g0[k] + v) + red[(23 + k) * 256 + t];
            o[k] = (k == 4 ? -inv_h2 : -1.f) * (v + red[(18 + k) * 256 + t]);
        }
    }
}

// ---------------------------------------------------------------------------------------------
static int div_up(int a, int b) { return (a + b - 1) / b; }

static SfBatch sf_batch(int n, const SfFrame *fr, int win)
{
    SfBatch b{};
    int tx[XDN_MAX_FRAMES], ty[XDN_MAX_FRAMES];
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        tx[i] = div_up(fr[i].W, SF_T);
        ty[i] = div_up(fr[i].H, SF_T);
    }
    b.map = make_tilemap(n, tx, ty);
    b.half = win / 2;
    return b;
}

template <int HALF, int MODE, int G, int P>
static void sf_launch_split(const SfBatch &b, hipStream_t st)
{
    hipLaunchKernelGGL((sf_tile_split<HALF, MODE, G, P>), dim3(b.map.total), dim3(256 * G), 0, st, b);
}

// Tiles of one image (a launch's images have one size).
static int sf_own_tiles(const SfBatch &b) { return div_up(b.f[0].W, SF_T) * div_up(b.f[0].H, SF_T); }

// Threads a pixel by the tiles of the launch, row groups by those of one image alone (an image's bits do not
// depend on its batch). Kernel alone in us with one, two, four threads, forward (band gradient):
//   256 tiles   win 3 3.8 4.0 4.2, win 7 8.3 7.0 6.7, win 11 15.2 11.8 10.9 (16.6 12.1 11.4), win 15 25.6 18.6 16.7
//   484 tiles   win 3 4.4 4.7 5.2, win 7 10.2 9.8 11.8, win 11 18.6 18.3 20.5 (20.5 20.1 21.1), win 15 31.9 29.7 31.3
//   1024 tiles  win 3 6.1 6.5 8.4, win 7 16.1 17.1 21.9, win 11 31.8 32.5 39.4 (36.1 35.3 40.8), win 15 58.0 54.5 60.6
// (win 3 loses 0.4 us to the split where a call takes 17 on the host). One thread with its rows in four groups
// instead of one: four images of 256 tiles at win 11 33.0 -> 34.0, sixteen 115 -> 118, at win 7 54.0 -> 55.7, at win
// 15 206 -> 211.
template <int HALF, int MODE>
static void sf_launch(const SfBatch &b, hipStream_t st)
{
    const int own = sf_own_tiles(b), total = b.map.total;
    if (total <= 256)
        sf_launch_split<HALF, MODE, 4, 4>(b, st);
    else if (MODE == SF_GRAD || total <= 512)
        own <= 256 ? sf_launch_split<HALF, MODE, 2, 4>(b, st) : sf_launch_split<HALF, MODE, 2, 2>(b, st);
    else if (own <= 256)
        sf_launch_split<HALF, SF_FWD, 1, 4>(b, st);
    else if (own <= 512)
        sf_launch_split<HALF, SF_FWD, 1, 2>(b, st);
    else
        hipLaunchKernelGGL((sf_tile<HALF>), dim3(b.map.total), dim3(256), 0, st, b);
}

// Windows up to 15x15 have tiled kernels; larger ones take direct loads (win 7, 512x512: forward 43 -> 19,
// band gradient 43 -> 19 us; 1920x1080: 294 -> 122, 271 -> 141).
template <int MODE>
static hipError_t sf_dispatch(const SfBatch &b, hipStream_t st)
{
    if (b.map.total == 0) return hipSuccess;
    switch (b.half)
    {
    case 1: sf_launch<1, MODE>(b, st); break;
    case 2: sf_launch<2, MODE>(b, st); break;
    case 3: sf_launch<3, MODE>(b, st); break;
    case 4: sf_launch<4, MODE>(b, st); break;
    case 5: sf_launch<5, MODE>(b, st); break;
    case 6: sf_launch<6, MODE>(b, st); break;
    case 7: sf_launch<7, MODE>(b, st); break;
    default: hipLaunchKernelGGL((sf_generic<MODE>), dim3(b.map.total), dim3(256), 0, st, b);
    }
    return hipGetLastError();
}

hipError_t launch_sf_forward(int n, const SfFrame *fr, int win, hipStream_t st)
{
    return sf_dispatch<SF_FWD>(sf_batch(n, fr, win), st);
}

hipError_t launch_sf_grad_band(int n, const SfFrame *fr, int win, hipStream_t st)
{
    return sf_dispatch<SF_GRAD>(sf_batch(n, fr, win), st);
}

// One launch computes both gradients where the band gradient takes the sums of two threads a pixel anyway;
// up to 256 tiles it takes four, and a second launch costs less than a chain twice as long.
static bool sf_grad_fused(const SfBatch &b) { return b.f[0].gband && b.map.total > 256; }

template <int HALF>
static void sf_grad_inputs_launch(const SfBatch &b, hipStream_t st)
{
    if (!sf_grad_fused(b))
        hipLaunchKernelGGL((sf_grad_inputs_tile<HALF, false, 2>), dim3(b.map.total), dim3(512), 0, st, b);
    else if (sf_own_tiles(b) <= 256)
        hipLaunchKernelGGL((sf_grad_inputs_tile<HALF, true, 4>), dim3(b.map.total), dim3(512), 0, st, b);
    else
        hipLaunchKernelGGL((sf_grad_inputs_tile<HALF, true, 2>), dim3(b.map.total), dim3(512), 0, st, b);
}

hipError_t launch_sf_grad_inputs(int n, const SfFrame *fr, int win, hipStream_t st)
{
    SfBatch b = sf_batch(n, fr, win);
    if (b.map.total == 0) return hipSuccess;
    if (b.f[0].gband && !sf_grad_fused(b))
        if (hipError_t e = launch_sf_grad_band(n, fr, win, st)) return e;
    switch (b.half)
    {
    case 1: sf_grad_inputs_launch<1>(b, st); break;
    case 2: sf_grad_inputs_launch<2>(b, st); break;
    case 3: sf_grad_inputs_launch<3>(b, st); break;
    case 4: sf_grad_inputs_launch<4>(b, st); break;
    case 5: sf_grad_inputs_launch<5>(b, st); break;
    case 6: sf_grad_inputs_launch<6>(b, st); break;
    case 7: sf_grad_inputs_launch<7>(b, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

int filter_train_tiles(int H, int W) { return div_up(W, SF_T) * div_up(H, SF_T); }

// A frame's results are the same bits whatever it is launched with: with `step` those of one thread a pixel at any
// size, else its own tiles decide. (A launch's frames have one size without `step`.)
hipError_t launch_filter_train(int n, const TrainFrame *fr, int win, bool step, hipStream_t st)
{
    if (win / 2 != 5) return hipErrorInvalidValue;
    TrBatch b{};
    int tx[XDN_MAX_FRAMES], ty[XDN_MAX_FRAMES];
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        tx[i] = div_up(fr[i].W, SF_T);
        ty[i] = div_up(fr[i].H, SF_T);
    }
    b.map = make_tilemap(n, tx, ty);
    if (b.map.total == 0) return hipSuccess;
    // operator call, one thread -> two: 64 tiles 28.4 -> 23.9 us (the host's launch rate), 256 30.8 -> 25.6; no
    // gain from 420 tiles on (39.4, 39.2; 1024: 66.1, 67.1; sixteen images of 256: 243, 244-249), and four threads
    // are no faster at any size
    if (!step && tx[0] * ty[0] <= 256)
        hipLaunchKernelGGL((sf_train_split<5>), dim3(b.map.total), dim3(512), 0, st, b);
    else
        hipLaunchKernelGGL((sf_train_tile<5>), dim3(b.map.total), dim3(256), 0, st, b);
    return hipGetLastError();
}

}  // namespace xdn
