// Cross-regression on gfx950: input variance, per-center weighted ridge regression and block
// reconstruction (the cross_regression op, regression.cu.cc:244-500).
//
// Data layout in HBM: images are NHWC float32 with 3 channels (12 B/px) exactly as the op
// boundary hands them over. The regression coefficients are an internal workspace laid out as
// [B][H/s][W/s][2 halves][6 coeffs][3 channels] float32 (144 B per center).
//
// Kernels
//   variance_kernel    3x3 clamped neighbourhood variance (EstInputVarianceKernel :244-276),
//                      HBM-bound, 1 px/thread. Optionally fuses log1p of the raw colour
//                      (scripts/main.py:207-212) and writes the log image.
//   regression_rows    fast path (win 17, sparsity 4): one workgroup = 64 centers of one center
//                      row, both halves; the 17 tap rows stream through a double-buffered LDS
//                      row (4 float4 planes per pixel) and each (center, half) is served by two
//                      lanes that split the 17 tap columns 9/8 and are reduced with a lane swap.
//                      61 FP32 accumulators per lane; 6x6 Cholesky per channel spread over the
//                      lane pair. VALU-bound.
//   regression_split   the same for launches of few blocks: the tap rows of 16 centers split over
//                      four waves.
//   recon_tile         fast path (win 17, sparsity 4, recon_scale 1): 16x16 pixels per
//                      workgroup; the <= 8x8 centers the tile touches are staged in LDS (both
//                      halves' coefficients and features), one pixel per lane, both halves; waves
//                      of pixels with equally many centers.
//   regression_generic / recon_generic: any win_size / sparsity / recon_scale, direct loads.
#include "xdn_common.h"
#include "xdn_kernels.h"
#include "xdn_regression.h"
#include "xdn_reproject.h"

namespace xdn {

// ---------------------------------------------------------------------------------------------
// Variance (and optional log1p prologue)
// ---------------------------------------------------------------------------------------------
struct VarFrame {
    const float *in;   // y (already log) or raw colour when log_in is set
    float *y_out;      // log1p(colour) when log_in is set, else unused
    float *var;        // [H][W]
    float *kept;       // a second copy for a later backward, or null
    int H, W;
};
struct VarBatch {
    TileMap map;
    VarFrame f[XDN_MAX_FRAMES];
    int log_in;
};

constexpr int VT_X = 32, VT_Y = 16;

// log1p(x) = ln(u) * x / (u - 1) with u = fl(1 + x) (Goldberg 1991, "What every computer scientist
// should know about floating-point arithmetic", Theorem 4): the rounding error of 1 + x cancels in
// the ratio, so a few-ulp ln(u) (v_log_f32 is log2 to ~1 ulp) gives a few-ulp log1p at ~10
// instructions instead of the libm polynomial.
__device__ __forceinline__ float log1p_acc(float x)
{
    const float u = 1.f + x;
    if (u == 1.f) return x;
    if (u == __builtin_inff()) return u;
    return (__builtin_amdgcn_logf(u) * 0.693147180559945309f) * (x * fast_rcp(u - 1.f));
}

// 32x16 pixels per workgroup, two per lane; the tile and its 1-px halo (zero outside the image)
// are loaded with every load of a lane in flight at once. The neighbour sum runs over all eight
// neighbours in the reference's order: the zeros of out-of-image taps leave it unchanged, and the
// count of in-image neighbours follows from the position.
__global__ __launch_bounds__(256) void variance_kernel(VarBatch b)
{
    constexpr int EX = VT_X + 2, EY = VT_Y + 2, NS = (EX * EY + 255) / 256;
    __shared__ float s[3][EY][EX];
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const VarFrame &F = b.f[L.f];
    const int H = F.H, W = F.W;
    const int x0 = L.tx * VT_X, y0 = L.ty * VT_Y;
    float3 v[NS];
#pragma unroll
    for (int u = 0; u < NS; ++u)
    {
        const int i = threadIdx.x + 256 * u;
        const int ly = i / EX, lx = i - ly * EX;
        const int gx = x0 + lx - 1, gy = y0 + ly - 1;
        v[u] = make_float3(0.f, 0.f, 0.f);
        if (i < EX * EY && gx >= 0 && gy >= 0 && gx < W && gy < H) v[u] = ld3(F.in, (size_t)gy * W + gx);
    }
#pragma unroll
    for (int u = 0; u < NS; ++u)
    {
        const int i = threadIdx.x + 256 * u;
        if (i >= EX * EY) continue;
        const int ly = i / EX, lx = i - ly * EX;
        const int gx = x0 + lx - 1, gy = y0 + ly - 1;
        float3 t = v[u];
        if (b.log_in && gx >= 0 && gy >= 0 && gx < W && gy < H)
        {
            t = make_float3(log1p_acc(t.x), log1p_acc(t.y), log1p_acc(t.z));
            if (lx >= 1 && ly >= 1 && lx <= VT_X && ly <= VT_Y) st3(F.y_out, (size_t)gy * W + gx, t);
        }
        s[0][ly][lx] = t.x;
        s[1][ly][lx] = t.y;
        s[2][ly][lx] = t.z;
    }
    __syncthreads();
    const int lx = threadIdx.x % VT_X;
#pragma unroll
    for (int r = 0; r < 2; ++r)
    {
        const int ly = threadIdx.x / VT_X + 8 * r;
        const int cx = x0 + lx, cy = y0 + ly;
        if (cx >= W || cy >= H) continue;
        const int n = (1 + (cx > 0) + (cx < W - 1)) * (1 + (cy > 0) + (cy < H - 1)) - 1;
        float acc[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for (int dy = -1; dy <= 1; ++dy)
#pragma unroll
            for (int dx = -1; dx <= 1; ++dx)
            {
                if ((dx | dy) == 0) continue;
#pragma unroll
                for (int k = 0; k < 3; ++k) acc[k] += s[k][ly + 1 + dy][lx + 1 + dx];
            }
        const float inv = 1.f / (float)n;
        float var = 0.f;
#pragma unroll
        for (int k = 0; k < 3; ++k)
        {
            const float d = acc[k] * inv - s[k][ly + 1][lx + 1];
            var += d * d;
        }
        F.var[(size_t)cy * W + cx] = var;
        if (F.kept) F.kept[(size_t)cy * W + cx] = var;
    }
}

// ---------------------------------------------------------------------------------------------
// Regression
// ---------------------------------------------------------------------------------------------
struct RegFrame {
    const float *y1, *y2, *var1, *var2, *alb, *nrm;
    float *beta;  // [Hs][Ws][2][18]
    float4 *fact; // Cholesky factors, see fact_at (FACT kernels)
    int H, W;
    int nfull;    // fast path with paired row tails: full 64-center blocks per center row, else 0
};
struct RegBatch {
    TileMap map;
    RegFrame f[XDN_MAX_FRAMES];
    int half_win, sparsity;  // generic kernel only
};

__device__ __forceinline__ float swap_add(float v) { return v + __shfl_xor(v, 1); }

__device__ __forceinline__ void reduce_pair(RegAcc &a)
{
    a.s00 = swap_add(a.s00); a.s03 = swap_add(a.s03); a.s04 = swap_add(a.s04); a.s05 = swap_add(a.s05);
    a.s33 = swap_add(a.s33); a.s34 = swap_add(a.s34); a.s35 = swap_add(a.s35); a.s44 = swap_add(a.s44);
    a.s45 = swap_add(a.s45); a.s55 = swap_add(a.s55);
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
        a.c01[c] = swap_add(a.c01[c]); a.c02[c] = swap_add(a.c02[c]); a.c11[c] = swap_add(a.c11[c]);
        a.c12[c] = swap_add(a.c12[c]); a.c22[c] = swap_add(a.c22[c]); a.c13[c] = swap_add(a.c13[c]);
        a.c14[c] = swap_add(a.c14[c]); a.c15[c] = swap_add(a.c15[c]); a.c23[c] = swap_add(a.c23[c]);
        a.c24[c] = swap_add(a.c24[c]); a.c25[c] = swap_add(a.c25[c]);
        a.x0[c] = swap_add(a.x0[c]); a.x1[c] = swap_add(a.x1[c]); a.x2[c] = swap_add(a.x2[c]);
        a.x3[c] = swap_add(a.x3[c]); a.x4[c] = swap_add(a.x4[c]); a.x5[c] = swap_add(a.x5[c]);
    }
}

constexpr int RG_CX = 64;       // centers per workgroup
constexpr int RG_S = 4;         // sparsity of the fast path
constexpr int RG_H = 8;         // half window of the fast path
constexpr int RG_ROW = RG_CX * RG_S + 2 * RG_H;

// Launch shape: one block per 64 centers of a center row; where a row's last block would hold at
// most 32 centers (1920 px: 480 centers = 7.5 blocks), the tails of two consecutive rows share one
// block instead (paired tail: wave w serves row 2p + (w & 1), half w >> 1, 32 centers each, over the
// 21 tap rows the two center rows span), so a 1080p frame is 2,025 blocks instead of 2,160: two
// rounds of the 1,024 resident at a time (four per CU) instead of three. Tile map per row pair p:
// nfull blocks of row 2p, nfull of row 2p + 1, then the paired tail. Each lane sums its taps in the
// same order either way. FACT: the centers' Cholesky factors are kept for the backward.
template <bool FACT>
__global__ __launch_bounds__(256) void regression_rows(RegBatch b)
{
    // [buffer][plane][pixel]; planes: (y1, var1), (y2, var2), (albedo, std1), (normal, std2)
    __shared__ float4 lds[2][4][RG_ROW];
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const RegFrame &F = b.f[L.f];
    const int H = F.H, W = F.W, Ws = W / RG_S, Hs = H / RG_S;
    const int t = threadIdx.x;
    int by, bx0;
    bool paired = false;
    if (F.nfull)
    {
        const int c = L.tx, nf = F.nfull;
        paired = c == 2 * nf;
        by = 2 * L.ty + (c >= nf && !paired);
        bx0 = (paired ? nf : (c >= nf ? c - nf : c)) * RG_CX;
        if (by >= Hs) return;  // odd row count: the last pair has no second row (whole block)
    }
    else
    {
        by = L.ty;
        bx0 = L.tx * RG_CX;
    }
    const int half = t >> 7;           // wave-uniform: waves 0-1 half A, waves 2-3 half B
    const int j = t & 127;
    const int o = paired ? (j >> 6) : 0;  // center row offset of this wave (paired tail only)
    const int ci = paired ? ((j & 63) >> 1) : (j >> 1), split = j & 1;
    const int row_c = by + o;          // this lane's center row
    const int bx = bx0 + ci;
    const bool active = bx < Ws && row_c < Hs;
    const int cx = (active ? bx : Ws - 1) * RG_S, cy = min(row_c, Hs - 1) * RG_S;
    const int px0 = bx0 * RG_S - RG_H;  // pixel x of LDS column 0

    const float *feat = half ? F.y2 : F.y1;
    const float *fvar = half ? F.var2 : F.var1;
    const size_t c = (size_t)cy * W + cx;
    const float3 cw = ld3(feat, c), ca = ld3(F.alb, c), cn = ld3(F.nrm, c);
    const float cvar = fvar[c];
    const float cvar_e = cvar + 1e-4f;
    const float cstd_e = sqrtf(cvar) + 1e-2f;

    RegAcc acc;
    acc.zero();

    const int ncols = min(RG_ROW, W + 2 * RG_H - bx0 * RG_S);  // columns actually needed
    // a wave whose centers all lie past the row end (or on a missing second row) only stages rows
    // and meets the barriers; its lanes' results are never stored
    const bool wave_busy = __builtin_amdgcn_readfirstlane(
        (bx0 + (paired ? 0 : (j & ~63) / 2)) < Ws && row_c < Hs);
    const int own = half, oth = 1 - half;
    // first tap column of this lane: split 0 covers dx in [-8, 0], split 1 covers [1, 8]
    const int col0 = ci * RG_S + (split ? RG_H + 1 : 0);
    const int ntap = split ? RG_H : RG_H + 1;
    const int nrows = 2 * RG_H + 1 + (paired ? RG_S : 0);

    for (int r = 0; r < nrows; ++r)
    {
        const int buf = r & 1;
        const int gy = mirror(by * RG_S + r - RG_H, H);
        const size_t row = (size_t)gy * W;
        for (int i = t; i < ncols; i += 256)
        {
            const size_t p = row + mirror(px0 + i, W);
            const float3 a = ld3(F.y1, p), bb = ld3(F.y2, p), al = ld3(F.alb, p), nr = ld3(F.nrm, p);
            const float v1 = F.var1[p], v2 = F.var2[p];
            lds[buf][0][i] = make_float4(a.x, a.y, a.z, v1);
            lds[buf][1][i] = make_float4(bb.x, bb.y, bb.z, v2);
            lds[buf][2][i] = make_float4(al.x, al.y, al.z, sqrtf(v1));
            lds[buf][3][i] = make_float4(nr.x, nr.y, nr.z, sqrtf(v2));
        }
        __syncthreads();
        if (!wave_busy || r < o * RG_S || r > o * RG_S + 2 * RG_H) continue;
#pragma unroll
        for (int k = 0; k < RG_H + 1; ++k)
        {
            if (k < ntap)
            {
                const int col = col0 + k;
                const float4 P = lds[buf][own][col];
                const float4 T = lds[buf][oth][col];
                const float4 A = lds[buf][2][col];
                const float4 N = lds[buf][3][col];
                const float istd = half ? N.w : A.w;
                const float3 dw = make_float3(P.x - cw.x, P.y - cw.y, P.z - cw.z);
                const float w = reg_weight(dw, cvar_e, P.w);
                const float inv = fast_rcp(cstd_e + istd);
                acc.add(w, inv, dw, make_float3(A.x - ca.x, A.y - ca.y, A.z - ca.z),
                        make_float3(N.x - cn.x, N.y - cn.y, N.z - cn.z), make_float3(T.x, T.y, T.z));
            }
        }
    }
    reduce_pair(acc);
    if (!active) return;
    // Lane pair solves the three channels: split 0 -> channels 0 and 1, split 1 -> channel 2.
    float *out = F.beta + (((size_t)row_c * Ws + bx) * 2 + half) * 18;
    const size_t centers = (size_t)Hs * Ws, center = (size_t)row_c * Ws + bx;
    {
        Sys6 s0, s2;
        acc.system(0, s0);
        acc.system(2, s2);
        Sys6 s;
#pragma unroll
        for (int k = 0; k < 21; ++k) s.a[k] = split ? s2.a[k] : s0.a[k];
#pragma unroll
        for (int k = 0; k < 6; ++k) s.x[k] = split ? s2.x[k] : s0.x[k];
        float be[6];
        const int ch = split ? 2 : 0;
        solve6(s, be, FACT ? F.fact + fact_at(centers, center, half, ch) : nullptr, centers);
#pragma unroll
        for (int k = 0; k < 6; ++k) out[k * 3 + ch] = be[k];
    }
    if (split == 0)
    {
        Sys6 s1;
        acc.system(1, s1);
        float be[6];
        solve6(s1, be, FACT ? F.fact + fact_at(centers, center, half, 1) : nullptr, centers);
#pragma unroll
        for (int k = 0; k < 6; ++k) out[k * 3 + 1] = be[k];
    }
}

// The same regression for launches that leave the chip idle: 16 centers of a center row per block, one
// wave (16 centers x 2 halves x 2 tap splits) for each quarter of the tap rows, which stages its own rows
// and loads the next one while it sums the current one. The four waves' sums meet in LDS, 21 accumulators
// at a time, and 96 lanes solve one channel's system each. FACT as in regression_rows. regression_rows has one wave per SIMD and 17
// rows in a chain at 512x512 (256 blocks); the same taps are summed in another order here. 164 registers,
// three waves per SIMD (at four waves it spills 160 B a lane and is slower at every size); three or
// six waves of six or three rows, nine of two: slower from 360x480 on.
constexpr int RS_CX = 16, RS_W = 4;  // centers, waves
constexpr int RS_ROW = RS_CX * RG_S + 2 * RG_H;
constexpr int RS_CHUNK = 21;                    // accumulators reduced at a time (3 x 21 >= 61)

// The accumulators in a fixed order: the 10 shared ones, then per channel c01 .. c25 and x0 .. x5.
constexpr int kAccShared = 10, kAccCh = 17, kAcc = kAccShared + 3 * kAccCh;
__device__ __forceinline__ void acc_list(const RegAcc &a, float v[kAcc])
{
    const float sh[kAccShared] = {a.s00, a.s03, a.s04, a.s05, a.s33, a.s34, a.s35, a.s44, a.s45, a.s55};
#pragma unroll
    for (int k = 0; k < kAccShared; ++k) v[k] = sh[k];
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
        const float w[kAccCh] = {a.c01[c], a.c02[c], a.c11[c], a.c12[c], a.c22[c], a.c13[c], a.c14[c], a.c15[c], a.c23[c],
                                 a.c24[c], a.c25[c], a.x0[c], a.x1[c], a.x2[c], a.x3[c], a.x4[c], a.x5[c]};
#pragma unroll
        for (int k = 0; k < kAccCh; ++k) v[kAccShared + c * kAccCh + k] = w[k];
    }
}

template <bool FACT>
__global__ __launch_bounds__(64 * RS_W, 3) void regression_split(RegBatch b)
{
    __shared__ float4 rows[RS_W][4][RS_ROW];       // one staged row per wave, planes as in regression_rows
    __shared__ float sums[kAcc][2 * RS_CX];        // [accumulator][half * 16 + center]
    static_assert(sizeof(rows) >= sizeof(float) * RS_W * RS_CHUNK * 2 * RS_CX, "reduction space");
    const TileLoc L = locate(b.map, xcd_tile(blockIdx.x, b.map.total));
    const RegFrame &F = b.f[L.f];
    const int H = F.H, W = F.W, Ws = W / RG_S;
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int by = L.ty, bx0 = L.tx * RS_CX;
    const int split = lane & 1, ci = (lane >> 1) & (RS_CX - 1), half = lane >> 5;
    const int cx = min(bx0 + ci, Ws - 1) * RG_S, cy = by * RG_S, px0 = bx0 * RG_S - RG_H;
    const float *feat = half ? F.y2 : F.y1;
    const size_t c = (size_t)cy * W + cx;
    const float3 cw = ld3(feat, c), ca = ld3(F.alb, c), cn = ld3(F.nrm, c);
    const float cvar = (half ? F.var2 : F.var1)[c];
    const float cvar_e = cvar + 1e-4f;
    const float cstd_e = sqrtf(cvar) + 1e-2f;
    RegAcc acc;
    acc.zero();
    const int ncols = min(RS_ROW, W + 2 * RG_H - bx0 * RG_S);
    constexpr int NS = (RS_ROW + 63) / 64;
    float3 va[NS], vb[NS], val[NS], vn[NS];
    float v1[NS], v2[NS];
    auto fetch = [&](int r) {
#pragma unroll
        for (int u = 0; u < NS; ++u)
        {
            // columns past the last one needed repeat it: no branch around the loads
            const int i = min(lane + 64 * u, ncols - 1);
            const size_t p = (size_t)mirror(cy + r - RG_H, H) * W + mirror(px0 + i, W);
            va[u] = ld3(F.y1, p); vb[u] = ld3(F.y2, p); val[u] = ld3(F.alb, p); vn[u] = ld3(F.nrm, p);
            v1[u] = F.var1[p];
            v2[u] = F.var2[p];
        }
    };
    float4(*const row)[RS_ROW] = rows[wv];
    auto commit = [&]() {
#pragma unroll
        for (int u = 0; u < NS; ++u)
        {
            const int i = lane + 64 * u;
            if (i >= RS_ROW) continue;
            row[0][i] = make_float4(va[u].x, va[u].y, va[u].z, v1[u]);
            row[1][i] = make_float4(vb[u].x, vb[u].y, vb[u].z, v2[u]);
            row[2][i] = make_float4(val[u].x, val[u].y, val[u].z, sqrtf(v1[u]));
            row[3][i] = make_float4(vn[u].x, vn[u].y, vn[u].z, sqrtf(v2[u]));
        }
    };
    const int col0 = ci * RG_S + (split ? RG_H + 1 : 0), ntap = split ? RG_H : RG_H + 1;
    constexpr int NR = 2 * RG_H + 1;
    const int r0 = NR * wv / RS_W, r1 = NR * (wv + 1) / RS_W;
    fetch(r0);
    for (int r = r0; r < r1; ++r)
    {
        commit();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the row is the wave's own
        fetch(min(r + 1, r1 - 1));
#pragma unroll
        for (int k = 0; k < RG_H + 1; ++k)
        {
            if (k < ntap)
            {
                const int col = col0 + k;
                const float4 P = row[half][col], T = row[1 - half][col], A = row[2][col], N = row[3][col];
                const float3 dw = make_float3(P.x - cw.x, P.y - cw.y, P.z - cw.z);
                const float w = reg_weight(dw, cvar_e, P.w);
                const float inv = fast_rcp(cstd_e + (half ? N.w : A.w));
                acc.add(w, inv, dw, make_float3(A.x - ca.x, A.y - ca.y, A.z - ca.z),
                        make_float3(N.x - cn.x, N.y - cn.y, N.z - cn.z), make_float3(T.x, T.y, T.z));
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    // [wave][accumulator of the chunk][lane], over the staged rows
    float *red = reinterpret_cast<float *>(&rows[0][0][0]);
    float v[kAcc];
    acc_list(acc, v);
#pragma unroll
    for (int k = 0; k < kAcc; ++k) v[k] = swap_add(v[k]);  // the two tap splits
    constexpr int PAIRS = 2 * RS_CX;
#pragma unroll
    for (int k0 = 0; k0 < kAcc; k0 += RS_CHUNK)
    {
        __syncthreads();
        if (!split)
#pragma unroll
            for (int k = 0; k < RS_CHUNK; ++k)
                if (k0 + k < kAcc) red[(wv * RS_CHUNK + k) * PAIRS + (lane >> 1)] = v[k0 + k];
        __syncthreads();
        const int n = (kAcc - k0 < RS_CHUNK ? kAcc - k0 : RS_CHUNK) * PAIRS;
        for (int e = t; e < n; e += 64 * RS_W)
        {
            float q[RS_W];
#pragma unroll
            for (int g = 0; g < RS_W; ++g) q[g] = red[g * RS_CHUNK * PAIRS + e];
            (&sums[k0][0])[e] = (q[0] + q[1]) + (q[2] + q[3]);
        }
    }
    __syncthreads();
    // lane t < 96: channel t / 32 of (half, center) t % 32
    const int pr = t & (PAIRS - 1), ch = t / PAIRS, sh = pr >> 4, sbx = bx0 + (pr & (RS_CX - 1));
    if (ch >= 3 || sbx >= Ws) return;
    Sys6 s;
    {
        auto g = [&](int k) { return sums[k][pr]; };
        auto gc = [&](int k) { return sums[kAccShared + ch * kAccCh + k][pr]; };
        const float a[21] = {g(0), gc(0), gc(1), g(1), g(2), g(3), gc(2), gc(3), gc(5), gc(6), gc(7),
                             gc(4), gc(8), gc(9), gc(10), g(4), g(5), g(6), g(7), g(8), g(9)};
#pragma unroll
        for (int k = 0; k < 21; ++k) s.a[k] = a[k];
#pragma unroll
        for (int k = 0; k < 6; ++k) s.x[k] = gc(11 + k);
    }
    const size_t centers = (size_t)(H / RG_S) * Ws, center = (size_t)by * Ws + sbx, rec = center * 2 + sh;
    float be[6];
    solve6(s, be, FACT ? F.fact + fact_at(centers, center, sh, ch) : nullptr, centers);
#pragma unroll
    for (int k = 0; k < 6; ++k) F.beta[rec * 18 + k * 3 + ch] = be[k];
}

// Any window / sparsity: one lane per (center, half), direct loads.
template <bool FACT>
__global__ __launch_bounds__(256) void regression_generic(RegBatch b)
{
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const RegFrame &F = b.f[L.f];
    const int S = b.sparsity, HW = b.half_win;
    const int H = F.H, W = F.W, Ws = W / S, Hs = H / S;
    const int half = threadIdx.x >> 7;
    const int bx = L.tx * 16 + (threadIdx.x & 15);
    const int by = L.ty * 8 + ((threadIdx.x & 127) >> 4);
    if (bx >= Ws || by >= Hs) return;
    const float *feat = half ? F.y2 : F.y1;
    const float *tgt = half ? F.y1 : F.y2;
    const float *fvar = half ? F.var2 : F.var1;
    const int cx = bx * S, cy = by * S;
    const size_t c = (size_t)cy * W + cx;
    const float3 cw = ld3(feat, c), ca = ld3(F.alb, c), cn = ld3(F.nrm, c);
    const float cvar = fvar[c], cvar_e = cvar + 1e-4f, cstd_e = sqrtf(cvar) + 1e-2f;
    RegAcc acc;
    acc.zero();
    for (int iy = cy - HW; iy <= cy + HW; ++iy)
        for (int ix = cx - HW; ix <= cx + HW; ++ix)
        {
            const size_t i = (size_t)mirror(iy, H) * W + mirror(ix, W);
            const float3 iw = ld3(feat, i), ia = ld3(F.alb, i), in = ld3(F.nrm, i), it = ld3(tgt, i);
            const float ivar = fvar[i];
            const float3 dw = make_float3(iw.x - cw.x, iw.y - cw.y, iw.z - cw.z);
            const float w = reg_weight(dw, cvar_e, ivar);
            const float inv = fast_rcp(cstd_e + sqrtf(ivar));
            acc.add(w, inv, dw, make_float3(ia.x - ca.x, ia.y - ca.y, ia.z - ca.z),
                    make_float3(in.x - cn.x, in.y - cn.y, in.z - cn.z), it);
        }
    const size_t centers = (size_t)Hs * Ws, center = (size_t)by * Ws + bx;
    float *out = F.beta + (center * 2 + half) * 18;
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
    {
        Sys6 s;
        acc.system(ch, s);
        float be[6];
        solve6(s, be, FACT ? F.fact + fact_at(centers, center, half, ch) : nullptr, centers);
#pragma unroll
        for (int k = 0; k < 6; ++k) out[k * 3 + ch] = be[k];
    }
}

// ---------------------------------------------------------------------------------------------
// Block reconstruction
// ---------------------------------------------------------------------------------------------
struct RecFrame {
    const float *beta;  // [Hs][Ws][2][18]
    const float *y1, *y2, *var1, *var2, *alb, *nrm;
    float *outa, *outb;  // [H/rs][W/rs][3]
    int H, W;
};
struct RecBatch {
    TileMap map;
    RecFrame f[XDN_MAX_FRAMES];
    int half_win, sparsity, recon_scale;  // generic kernel only
};

constexpr int RC_T = 16;                 // pixels per tile side
constexpr int RC_C = 8;                  // centers per tile side (fast path)
constexpr int RC_STRIDE = 13;            // float4 per staged center
constexpr int RC_ROW = RC_C * RC_STRIDE + 4;  // float4 per center row: rows half the banks apart

// Per-center contribution for one half: pred = beta . delta with delta = pixel - center.
__device__ __forceinline__ void recon_term(const float4 *cb, float3 dwv, float inv, float3 d2, float3 n,
                                           float w, float3 &acc)
{
    // cb: 18 floats of beta [k][ch] as 4.5 float4 starting at a 16-B boundary or at +8 B; we
    // read through a float pointer to keep it simple.
    const float *bt = reinterpret_cast<const float *>(cb);
    const float d1x = dwv.x * inv, d1y = dwv.y * inv, d1z = dwv.z * inv;
    const float px = bt[0] + bt[3] * d1x + bt[6] * d2.x + bt[9] * n.x + bt[12] * n.y + bt[15] * n.z;
    const float py = bt[1] + bt[4] * d1y + bt[7] * d2.y + bt[10] * n.x + bt[13] * n.y + bt[16] * n.z;
    const float pz = bt[2] + bt[5] * d1z + bt[8] * d2.z + bt[11] * n.x + bt[14] * n.y + bt[17] * n.z;
    acc.x += w * px;
    acc.y += w * py;
    acc.z += w * pz;
}

// The same prediction with the center's terms folded into the staged record: with
// K0 = beta0 - beta2 . a_c - beta3 . n_c (per channel), beta . delta = K0 + beta1 d1 + beta2 a_p +
// beta3 . n_p, so a (pixel, center) pair needs no albedo or normal difference. bt: K0 in place of
// beta0, then beta1..beta5 as in recon_term; ca, cn: the pixel's albedo and normal.
__device__ __forceinline__ void recon_term_k0(const float *bt, float3 dwv, float inv, float3 ca, float3 cn, float w,
                                              float3 &acc)
{
    const float d1x = dwv.x * inv, d1y = dwv.y * inv, d1z = dwv.z * inv;
    const float px = bt[0] + bt[3] * d1x + bt[6] * ca.x + bt[9] * cn.x + bt[12] * cn.y + bt[15] * cn.z;
    const float py = bt[1] + bt[4] * d1y + bt[7] * ca.y + bt[10] * cn.x + bt[13] * cn.y + bt[16] * cn.z;
    const float pz = bt[2] + bt[5] * d1z + bt[8] * ca.z + bt[11] * cn.x + bt[14] * cn.y + bt[17] * cn.z;
    acc.x += w * px;
    acc.y += w * py;
    acc.z += w * pz;
}

// cs: staged center records (13 float4): beta A (18) + beta B (18) = 9 float4, (y1, var1), (y2, var2),
// (alb, std1), (nrm, std2).
__device__ __forceinline__ void recon_block(const RecBatch &b, int bid, float4 *cs)
{
    const int tile = xcd_tile(bid, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const RecFrame &F = b.f[L.f];
    const int H = F.H, W = F.W, Ws = W / RG_S;
    const int x0 = L.tx * RC_T, y0 = L.ty * RC_T;
    // tile center window [clo, clo+RC_C) x [rlo, rlo+RC_C), a superset of every pixel's range
    const int clo = max(0, (x0 - RG_H + RG_S - 1 + 4 * RG_S) / RG_S - 4);
    const int rlo = max(0, (y0 - RG_H + RG_S - 1 + 4 * RG_S) / RG_S - 4);
    const int chi = min((W - 1) / RG_S, (x0 + RC_T - 1 + RG_H) / RG_S);
    const int rhi = min((H - 1) / RG_S, (y0 + RC_T - 1 + RG_H) / RG_S);
    const int ncx = chi - clo + 1, ncy = rhi - rlo + 1;
    for (int i = threadIdx.x; i < ncx * ncy * 9; i += 256)
    {
        const int cidx = i / 9, q = i - cidx * 9;
        const int ry = cidx / ncx, rx = cidx - ry * ncx;
        const float4 *src = reinterpret_cast<const float4 *>(F.beta + ((size_t)(rlo + ry) * Ws + (clo + rx)) * 36);
        cs[ry * RC_ROW + rx * RC_STRIDE + q] = src[q];
    }
    for (int i = threadIdx.x; i < ncx * ncy; i += 256)
    {
        const int ry = i / ncx, rx = i - ry * ncx;
        const size_t p = (size_t)((rlo + ry) * RG_S) * W + (size_t)((clo + rx) * RG_S);
        const float3 a = ld3(F.y1, p), bb = ld3(F.y2, p), al = ld3(F.alb, p), nr = ld3(F.nrm, p);
        const float v1 = F.var1[p], v2 = F.var2[p];
        float4 *d = cs + ry * RC_ROW + rx * RC_STRIDE;
        d[9] = make_float4(a.x, a.y, a.z, v1);
        d[10] = make_float4(bb.x, bb.y, bb.z, v2);
        d[11] = make_float4(al.x, al.y, al.z, sqrtf(v1));
        d[12] = make_float4(nr.x, nr.y, nr.z, sqrtf(v2));
    }
    __syncthreads();
    // fold each center's albedo and normal into its constant term, per half and channel
    for (int i = threadIdx.x; i < ncx * ncy * 2; i += 256)
    {
        const int cidx = i >> 1, hb = i & 1;
        const int ry = cidx / ncx, rx = cidx - ry * ncx;
        float4 *d = cs + ry * RC_ROW + rx * RC_STRIDE;
        float *bt = reinterpret_cast<float *>(d) + 18 * hb;
        const float4 A = d[11], N = d[12];
        const float av[3] = {A.x, A.y, A.z};
#pragma unroll
        for (int ch = 0; ch < 3; ++ch)
            bt[ch] = bt[ch] - bt[6 + ch] * av[ch] - (bt[9 + ch] * N.x + bt[12 + ch] * N.y + bt[15 + ch] * N.z);
    }
    __syncthreads();
    // Pixels with x = 0 mod 4 see five center columns, the others four, and so for rows. A wave takes four
    // of the 16 residue classes (16 pixels each): x = 0, then the rest by y, so the four waves walk
    // 25, 20, 16 and 16 centers where waves of four pixel rows walk 25 each. Lanes of one read phase
    // (0-3 with 20-23 and so on) are given the same center row, or rows four float4 apart in the banks.
    // At the VALU's issue rate: 1920x1080 110 -> 95 us, four 256x256 frames 19.8 -> 18.4, one 11.2 -> 10.9.
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = threadIdx.x >> 4 & 3;
    const int cls = 4 * (wv - 1) + j, pos = (threadIdx.x & 15) ^ (j & 1) << 2;
    const int cx = x0 + RG_S * (pos & 3) + (wv ? 1 + cls % 3 : 0);
    const int cy = y0 + RG_S * (pos >> 2) + (wv ? cls / 3 : j);
    if (cx >= W || cy >= H) return;
    const size_t c = (size_t)cy * W + cx;
    const float3 c1 = ld3(F.y1, c), c2 = ld3(F.y2, c), ca = ld3(F.alb, c), cn = ld3(F.nrm, c);
    const float v1 = F.var1[c], v2 = F.var2[c];
    const float v1e = v1 + 1e-4f, v2e = v2 + 1e-4f;
    const float s1e = sqrtf(v1) + 1e-2f, s2e = sqrtf(v2) + 1e-2f;
    const int sx = max(0, idivup(cx - RG_H, RG_S)), ex = min((W - 1) / RG_S, (cx + RG_H) / RG_S);
    const int sy = max(0, idivup(cy - RG_H, RG_S)), ey = min((H - 1) / RG_S, (cy + RG_H) / RG_S);
    float3 accA = make_float3(0.f, 0.f, 0.f), accB = accA;
    float sumA = 0.f, sumB = 0.f;
    for (int iy = sy; iy <= ey; ++iy)
        for (int ix = sx; ix <= ex; ++ix)
        {
            const float4 *rec = cs + (iy - rlo) * RC_ROW + (ix - clo) * RC_STRIDE;
            const float4 P1 = rec[9], P2 = rec[10];
            const float std1 = rec[11].w, std2 = rec[12].w;
            const float3 dwA = make_float3(c1.x - P1.x, c1.y - P1.y, c1.z - P1.z);
            const float3 dwB = make_float3(c2.x - P2.x, c2.y - P2.y, c2.z - P2.z);
            const float wA = reg_weight(dwA, v1e, P1.w), wB = reg_weight(dwB, v2e, P2.w);
            const float *bt = reinterpret_cast<const float *>(rec);
            recon_term_k0(bt, dwA, fast_rcp(s1e + std1), ca, cn, wA, accA);
            recon_term_k0(bt + 18, dwB, fast_rcp(s2e + std2), ca, cn, wB, accB);
            sumA += wA;
            sumB += wB;
        }
    const float iA = 1.f / fmaxf(sumA, 1e-7f), iB = 1.f / fmaxf(sumB, 1e-7f);
    st3(F.outa, c, make_float3(fmaxf(0.f, accA.x * iA), fmaxf(0.f, accA.y * iA), fmaxf(0.f, accA.z * iA)));
    st3(F.outb, c, make_float3(fmaxf(0.f, accB.x * iB), fmaxf(0.f, accB.y * iB), fmaxf(0.f, accB.z * iB)));
}

__global__ __launch_bounds__(256) void recon_tile(RecBatch b)
{
    __shared__ float4 cs[RC_C * RC_ROW];
    recon_block(b, blockIdx.x, cs);
}

struct RecRpBatch {
    RecBatch rec;
    RpBatch rp;
};
static_assert(sizeof(RecRpBatch) <= 4096, "kernel argument too large");

// The training step's reconstruction and its reprojection of the history, which do not depend on each other:
// the VALU-bound blocks first, the HBM-bound ones fill in behind them. Both use 62 registers and under
// 19 KB of LDS, eight waves per SIMD. A step, two launches -> one: 96x96 206 -> 198 us, four 256x256 U-Net
// streams 394 -> 387, 1280x720 809 -> 798, 1920x1080 1614 -> 1603; the reprojection first: 198, 390, 800,
// 1609; both in alternating groups of blocks: 198, 392, 801, 1603.
__global__ __launch_bounds__(256) void recon_reproject(RecRpBatch b)
{
    __shared__ union {
        float4 cs[RC_C * RC_ROW];
        RpShared<3, 3> rp;
    } sh;
    const int bid = blockIdx.x, n = b.rec.map.total;
    if (bid < n)
        recon_block(b.rec, bid, sh.cs);
    else
        reproject_block<3, 3, true>(b.rp, bid - n, sh.rp);
}

__global__ __launch_bounds__(256) void recon_generic(RecBatch b)
{
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const RecFrame &F = b.f[L.f];
    const int S = b.sparsity, HW = b.half_win, RS = b.recon_scale;
    const int H = F.H, W = F.W, Ws = W / S, Hr = H / RS, Wr = W / RS;
    const int rx = L.tx * 16 + (threadIdx.x & 15), ry = L.ty * 16 + (threadIdx.x >> 4);
    if (rx >= Wr || ry >= Hr) return;
    const int cx = rx * RS, cy = ry * RS;
    const size_t c = (size_t)cy * W + cx;
    const float3 c1 = ld3(F.y1, c), c2 = ld3(F.y2, c), ca = ld3(F.alb, c), cn = ld3(F.nrm, c);
    const float v1 = F.var1[c], v2 = F.var2[c];
    const float v1e = v1 + 1e-4f, v2e = v2 + 1e-4f;
    const float s1e = sqrtf(v1) + 1e-2f, s2e = sqrtf(v2) + 1e-2f;
    const int sx = max(0, idivup(cx - HW, S)), ex = min((W - 1) / S, (cx + HW) / S);
    const int sy = max(0, idivup(cy - HW, S)), ey = min((H - 1) / S, (cy + HW) / S);
    float3 accA = make_float3(0.f, 0.f, 0.f), accB = accA;
    float sumA = 0.f, sumB = 0.f;
    for (int iy = sy; iy <= ey; ++iy)
        for (int ix = sx; ix <= ex; ++ix)
        {
            const float *bt = F.beta + ((size_t)iy * Ws + ix) * 36;
            const size_t i = (size_t)(iy * S) * W + (size_t)(ix * S);
            const float3 p1 = ld3(F.y1, i), p2 = ld3(F.y2, i), ia = ld3(F.alb, i), in = ld3(F.nrm, i);
            const float iv1 = F.var1[i], iv2 = F.var2[i];
            const float3 d2 = make_float3(ca.x - ia.x, ca.y - ia.y, ca.z - ia.z);
            const float3 n = make_float3(cn.x - in.x, cn.y - in.y, cn.z - in.z);
            const float3 dwA = make_float3(c1.x - p1.x, c1.y - p1.y, c1.z - p1.z);
            const float3 dwB = make_float3(c2.x - p2.x, c2.y - p2.y, c2.z - p2.z);
            const float wA = reg_weight(dwA, v1e, iv1), wB = reg_weight(dwB, v2e, iv2);
            recon_term(reinterpret_cast<const float4 *>(bt), dwA, fast_rcp(s1e + sqrtf(iv1)), d2, n, wA, accA);
            recon_term(reinterpret_cast<const float4 *>(bt + 18), dwB, fast_rcp(s2e + sqrtf(iv2)), d2, n, wB, accB);
            sumA += wA;
            sumB += wB;
        }
    const size_t o = (size_t)ry * Wr + rx;
    const float iA = 1.f / fmaxf(sumA, 1e-7f), iB = 1.f / fmaxf(sumB, 1e-7f);
    st3(F.outa, o, make_float3(fmaxf(0.f, accA.x * iA), fmaxf(0.f, accA.y * iA), fmaxf(0.f, accA.z * iA)));
    st3(F.outb, o, make_float3(fmaxf(0.f, accB.x * iB), fmaxf(0.f, accB.y * iB), fmaxf(0.f, accB.z * iB)));
}

// ---------------------------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------------------------
static int div_up(int a, int b) { return (a + b - 1) / b; }

hipError_t launch_variance(int n, const CrFrame *fr, int which, bool log_in, hipStream_t st)
{
    // which: bit0 -> half A (y1/var1), bit1 -> half B (y2/var2); both halves share one launch
    VarBatch b{};
    int tx[XDN_MAX_FRAMES], ty[XDN_MAX_FRAMES];
    int m = 0;
    for (int i = 0; i < n; ++i)
        for (int h = 0; h < 2; ++h)
        {
            if (!(which & (1 << h))) continue;
            VarFrame &v = b.f[m];
            v.in = log_in ? (h ? fr[i].color2 : fr[i].color) : (h ? fr[i].y2 : fr[i].y1);
            v.y_out = h ? fr[i].y2 : fr[i].y1;
            v.var = h ? fr[i].var2 : fr[i].var1;
            v.kept = h ? fr[i].var2_kept : fr[i].var1_kept;
            v.H = fr[i].H;
            v.W = fr[i].W;
            tx[m] = div_up(v.W, VT_X);
            ty[m] = div_up(v.H, VT_Y);
            ++m;
        }
    b.map = make_tilemap(m, tx, ty);
    b.log_in = log_in ? 1 : 0;
    if (b.map.total == 0) return hipSuccess;
    hipLaunchKernelGGL(variance_kernel, dim3(b.map.total), dim3(256), 0, st, b);
    return hipGetLastError();
}

// Up to this many blocks of regression_rows regression_split is the faster one. Whole operator, rows ->
// split: 64 blocks (256x256) 62 -> 33 us, 256 (512x512) 70 -> 59, 540 (540x960) 118 -> 102, 900
// (720x1280) 161 -> 175. It is a frame's own blocks that count, so that its bits do not depend on its batch; in
// larger launches of such frames: 3 x 540x960 256 -> 252, 8 x 384x384 209 -> 200, 4 x 512x512 169 -> 179,
// 8 x 512x512 315 -> 338.
constexpr int kRowsFewBlocks = 640;

// A frame's coefficients are the same bits whatever it is launched with: regression_rows at any size with `step`
// (the training step, where another order in one layer would move the next frame's bf16 activations), else what its
// own size asks for, whether the factors are kept for a backward or not. (A launch's frames have one size without
// `step`.) Against 64 bits the split's shorter sums are the more accurate: 512x512, rows -> split, outputs 2.1e-7 ->
// 1.6e-7, gradients of the colors 3.3e-7 -> 1.9e-7, of the normals 1.3e-5 -> 5.7e-6 relative L2.
hipError_t launch_regression(int n, const CrFrame *fr, int win, int s, bool step, hipStream_t st)
{
    RegBatch b{};
    int tx[XDN_MAX_FRAMES], ty[XDN_MAX_FRAMES];
    const bool fast = (win / 2 == RG_H && s == RG_S);
    for (int i = 0; i < n; ++i)
    {
        RegFrame &r = b.f[i];
        r.y1 = fr[i].y1; r.y2 = fr[i].y2; r.var1 = fr[i].var1; r.var2 = fr[i].var2;
        r.alb = fr[i].alb; r.nrm = fr[i].nrm; r.beta = fr[i].beta; r.H = fr[i].H; r.W = fr[i].W;
        r.fact = fr[i].fact;
        const int Ws = r.W / s, Hs = r.H / s;
        // pair the rows' tail blocks where a tail holds at most half a block of centers
        const int rem = Ws % RG_CX;
        r.nfull = (fast && Ws >= RG_CX && rem > 0 && rem <= RG_CX / 2 && Hs >= 2) ? Ws / RG_CX : 0;
        if (r.nfull)
        {
            tx[i] = 2 * r.nfull + 1;
            ty[i] = div_up(Hs, 2);
        }
        else
        {
            tx[i] = fast ? div_up(Ws, RG_CX) : div_up(Ws, 16);
            ty[i] = fast ? Hs : div_up(Hs, 8);
        }
    }
    b.map = make_tilemap(n, tx, ty);
    b.half_win = win / 2;
    b.sparsity = s;
    if (b.map.total == 0) return hipSuccess;
    const bool fact = fr[0].fact != nullptr;  // all frames of a call or none
    if (fast && !step && tx[0] * ty[0] <= kRowsFewBlocks)
    {
        for (int i = 0; i < n; ++i)
        {
            tx[i] = div_up(fr[i].W / s, RS_CX);
            ty[i] = fr[i].H / s;
        }
        b.map = make_tilemap(n, tx, ty);
        hipLaunchKernelGGL((fact ? regression_split<true> : regression_split<false>), dim3(b.map.total), dim3(64 * RS_W), 0, st, b);
    }
    else if (fast)
        hipLaunchKernelGGL((fact ? regression_rows<true> : regression_rows<false>), dim3(b.map.total), dim3(256), 0, st, b);
    else
        hipLaunchKernelGGL((fact ? regression_generic<true> : regression_generic<false>), dim3(b.map.total), dim3(256), 0, st, b);
    return hipGetLastError();
}

static RecBatch rec_batch(int n, const CrFrame *fr, int win, int s, int rs)
{
    RecBatch b{};
    int tx[XDN_MAX_FRAMES], ty[XDN_MAX_FRAMES];
    for (int i = 0; i < n; ++i)
    {
        RecFrame &r = b.f[i];
        r.beta = fr[i].beta; r.y1 = fr[i].y1; r.y2 = fr[i].y2; r.var1 = fr[i].var1; r.var2 = fr[i].var2;
        r.alb = fr[i].alb; r.nrm = fr[i].nrm; r.outa = fr[i].outa; r.outb = fr[i].outb;
        r.H = fr[i].H; r.W = fr[i].W;
        tx[i] = div_up(r.W / rs, 16);
        ty[i] = div_up(r.H / rs, 16);
    }
    b.map = make_tilemap(n, tx, ty);
    b.half_win = win / 2;
    b.sparsity = s;
    b.recon_scale = rs;
    return b;
}

static bool rec_tiled(int win, int s, int rs) { return win / 2 == RG_H && s == RG_S && rs == 1; }

hipError_t launch_recon(int n, const CrFrame *fr, int win, int s, int rs, hipStream_t st)
{
    const RecBatch b = rec_batch(n, fr, win, s, rs);
    if (b.map.total == 0) return hipSuccess;
    if (rec_tiled(win, s, rs))
        hipLaunchKernelGGL(recon_tile, dim3(b.map.total), dim3(256), 0, st, b);
    else
        hipLaunchKernelGGL(recon_generic, dim3(b.map.total), dim3(256), 0, st, b);
    return hipGetLastError();
}

hipError_t launch_recon_reproject(int n, const CrFrame *fr, int win, int s, const RpFrame *rp, hipStream_t st)
{
    const int dims[3] = {3, 3, 3};
    bool three3;
    RecRpBatch b;
    b.rec = rec_batch(n, fr, win, s, 1);
    b.rp = rp_batch(n, rp, 3, dims, three3);
    if (b.rec.map.total + b.rp.map.total == 0) return hipSuccess;
    if (!rec_tiled(win, s, 1)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(recon_reproject, dim3(b.rec.map.total + b.rp.map.total), dim3(256), 0, st, b);
    return hipGetLastError();
}

}  // namespace xdn
