// Backward of cross_regression with respect to its four inputs (imga, imgb, albedo, normal),
// recon_scale 1. The reference registers no gradient for this op (regression.cc:25-103); this is
// the adjoint of the forward kernels of k_regression.hip, with every window weight recomputed.
//
// Notation for one half X (features f = own log colour, v = var(f), target t = other half):
//   regression at center c:  w = exp(-|f_i-f_c|^2/(v_c+v_i+1e-4)) + 1e-7,
//                            d = [1, (f_i-f_c)/(sqrt v_c + sqrt v_i + 1e-2), a_i-a_c, n_i-n_c],
//                            M = sum w d d^T + 1e-3 I,  b = sum w d t_i,  beta = M^-1 b
//   recon at pixel p:        out = max(0, sum_c w_pc (beta_c . delta_pc) / max(sum_c w_pc, 1e-7)),
//                            delta = x_p - x_c.
// Adjoint: u = M^-1 g_beta (the Cholesky clamp never binds: every pivot of M is >= 1e-3), and per
// tap  g_w = (u.d)(t_i - d.beta),  g_d = w (u (t_i - d.beta) - beta (u.d)),  g_t_i = w (u.d).
// Conventions at the kinks: max(0, .) passes the gradient where the value is > 0, the sumW guard
// where sumW > 1e-7, and d sqrt(v)/dv is 0 where v == 0.
//
// Kernels (all batched over frames like the forward), in launch order; the crg_*_tile forms take the
// windows that fit their LDS arrays (win 17 / sparsity 4 and smaller), the others any window with one
// thread per pixel or per (center, half) and direct loads:
//   crg_prep_tile, crg_recon_prep   per pixel: recompute the reconstruction sums, emit
//                        (g_acc, g_sumW)                                                  [H][W][2]
//   crg_center_tile, crg_center     per (center, half): gather g_beta over the pixels whose range holds
//                        the center (recon adjoint, center side), solve u, then the center side of
//                        the regression adjoint over the window                         [Hs][Ws][2]
//   crg_pixel_tile, crg_pixel       per pixel: recon adjoint (pixel side), regression adjoint (tap
//                        side, all mirrored positions of the pixel), center-side terms of grid
//                        pixels, variance adjoint (own term); writes grad albedo/normal and partial
//                        grad imga/imgb
//   crg_var_gather       per pixel: neighbour terms of the variance adjoint
#include "xdn_common.h"
#include "xdn_kernels.h"
#include "xdn_regression.h"

namespace xdn {

struct CrgBatch {
    TileMap map;
    CrgFrame f[XDN_MAX_FRAMES];
    int half_win, sparsity;
};

struct G10 {
    float3 f, a, n;
    float v;
    __device__ __forceinline__ void zero()
    {
        f = a = n = make_float3(0.f, 0.f, 0.f);
        v = 0.f;
    }
};

__device__ __forceinline__ float3 sub3(float3 a, float3 b) { return make_float3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ float comp(float3 a, int k) { return k == 0 ? a.x : (k == 1 ? a.y : a.z); }

// Adjoint of (w, delta) for the pair (P, Q), delta = x_P - x_Q, w = exp(-|df|^2 / S) + 1e-7 with
// S = v_P + v_Q + 1e-4, delta_1 = df * inv (inv = 1/(sqrt v_P + sqrt v_Q + 1e-2)).
// Adds the P side (sideP) or the Q side of the gradient to g.
__device__ __forceinline__ void pair_adj(float3 df, float S, float inv, float sP, float sQ, float gw,
                                         const float gd[3][6], bool sideP, G10 &g)
{
    const float D = df.x * df.x + df.y * df.y + df.z * df.z;
    const float rS = fast_rcp(S);
    const float E = fast_exp2(-kLog2e * D * rS);
    const float gD2 = -2.f * gw * E * rS;  // dL/dD * 2
    const float gS = gw * E * D * rS * rS;
    float3 gf, ga;
    gf.x = gD2 * df.x + gd[0][1] * inv;
    gf.y = gD2 * df.y + gd[1][1] * inv;
    gf.z = gD2 * df.z + gd[2][1] * inv;
    ga = make_float3(gd[0][2], gd[1][2], gd[2][2]);
    const float3 gn = make_float3(gd[0][3] + gd[1][3] + gd[2][3], gd[0][4] + gd[1][4] + gd[2][4],
                                  gd[0][5] + gd[1][5] + gd[2][5]);
    const float gden = -(gd[0][1] * df.x + gd[1][1] * df.y + gd[2][1] * df.z) * inv * inv;
    if (sideP)
    {
        g.f.x += gf.x; g.f.y += gf.y; g.f.z += gf.z;
        g.a.x += ga.x; g.a.y += ga.y; g.a.z += ga.z;
        g.n.x += gn.x; g.n.y += gn.y; g.n.z += gn.z;
        g.v += gS + (sP > 0.f ? 0.5f * gden / sP : 0.f);
    }
    else
    {
        g.f.x -= gf.x; g.f.y -= gf.y; g.f.z -= gf.z;
        g.a.x -= ga.x; g.a.y -= ga.y; g.a.z -= ga.z;
        g.n.x -= gn.x; g.n.y -= gn.y; g.n.z -= gn.z;
        g.v += gS + (sQ > 0.f ? 0.5f * gden / sQ : 0.f);
    }
}

// Reconstruction term of pixel p and center c for one half, as recon_generic computes it:
// delta = x_p - x_c; returns w, fills delta d[ch][k] and pred[ch].
__device__ __forceinline__ float recon_pair(float3 fp, float3 ap, float3 np, float vp, float sp, float3 fc, float3 ac,
                                            float3 nc, float vc, float sc, const float *bt, float d[3][6],
                                            float pred[3], float &inv)
{
    const float3 df = sub3(fp, fc), da = sub3(ap, ac), dn = sub3(np, nc);
    const float w = reg_weight(df, vp + 1e-4f, vc);
    inv = fast_rcp((sp + 1e-2f) + sc);
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
    {
        d[ch][0] = 1.f;
        d[ch][1] = comp(df, ch) * inv;
        d[ch][2] = comp(da, ch);
        d[ch][3] = dn.x;
        d[ch][4] = dn.y;
        d[ch][5] = dn.z;
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 6; ++k) s += bt[k * 3 + ch] * d[ch][k];
        pred[ch] = s;
    }
    return w;
}

// Regression tap i of center c for one half, as regression_generic computes it: d = x_i - x_c.
__device__ __forceinline__ float reg_pair(float3 fi, float3 ai, float3 ni, float vi, float si, float3 fc, float3 ac,
                                          float3 nc, float vc, float sc, float d[3][6], float &inv)
{
    const float3 df = sub3(fi, fc), da = sub3(ai, ac), dn = sub3(ni, nc);
    const float w = reg_weight(df, vc + 1e-4f, vi);
    inv = fast_rcp((sc + 1e-2f) + si);
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
    {
        d[ch][0] = 1.f;
        d[ch][1] = comp(df, ch) * inv;
        d[ch][2] = comp(da, ch);
        d[ch][3] = dn.x;
        d[ch][4] = dn.y;
        d[ch][5] = dn.z;
    }
    return w;
}

// Regression adjoint of one tap: g_w, g_d and the target gradient weight w (u.d) per channel.
__device__ __forceinline__ float reg_tap_adj(float w, const float d[3][6], const float *bt, const float *u, float3 t,
                                             float gd[3][6], float gt[3])
{
    float gw = 0.f;
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
    {
        float r = comp(t, ch), s = 0.f;
#pragma unroll
        for (int k = 0; k < 6; ++k)
        {
            r -= d[ch][k] * bt[k * 3 + ch];
            s += u[k * 3 + ch] * d[ch][k];
        }
        gw += s * r;
#pragma unroll
        for (int k = 0; k < 6; ++k) gd[ch][k] = w * (u[k * 3 + ch] * r - bt[k * 3 + ch] * s);
        gt[ch] = w * s;
    }
    return gw;
}

// ---------------------------------------------------------------------------------------------
// 1. per pixel: (g_acc, g_sumW) of the reconstruction, both halves
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void crg_recon_prep(CrgBatch b)
{
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const CrgFrame &F = b.f[L.f];
    const int S = b.sparsity, HW = b.half_win;
    const int H = F.H, W = F.W, Ws = W / S;
    const int px = L.tx * 16 + (threadIdx.x & 15), py = L.ty * 16 + (threadIdx.x >> 4);
    if (px >= W || py >= H) return;
    const size_t p = (size_t)py * W + px;
    const int sx = max(0, idivup(px - HW, S)), ex = min((W - 1) / S, (px + HW) / S);
    const int sy = max(0, idivup(py - HW, S)), ey = min((H - 1) / S, (py + HW) / S);
    const float3 ap = ld3(F.alb, p), np = ld3(F.nrm, p);
    for (int h = 0; h < 2; ++h)
    {
        const float *feat = h ? F.y2 : F.y1, *var = h ? F.var2 : F.var1;
        const float3 fp = ld3(feat, p);
        const float vp = var[p], sp = sqrtf(vp);
        float3 acc = make_float3(0.f, 0.f, 0.f);
        float sum = 0.f;
        for (int iy = sy; iy <= ey; ++iy)
            for (int ix = sx; ix <= ex; ++ix)
            {
                const size_t c = (size_t)(iy * S) * W + (size_t)(ix * S);
                const float *bt = F.beta + (((size_t)iy * Ws + ix) * 2 + h) * 18;
                float d[3][6], pred[3], inv;
                const float vc = var[c];
                const float w = recon_pair(fp, ap, np, vp, sp, ld3(feat, c), ld3(F.alb, c), ld3(F.nrm, c), vc,
                                           sqrtf(vc), bt, d, pred, inv);
                acc.x += w * pred[0];
                acc.y += w * pred[1];
                acc.z += w * pred[2];
                sum += w;
            }
        const float iv = 1.f / fmaxf(sum, 1e-7f);
        const float3 go = ld3(h ? F.goutb : F.gouta, p);
        float4 q;
        q.x = acc.x * iv > 0.f ? go.x * iv : 0.f;
        q.y = acc.y * iv > 0.f ? go.y * iv : 0.f;
        q.z = acc.z * iv > 0.f ? go.z * iv : 0.f;
        q.w = sum > 1e-7f ? -(q.x * acc.x + q.y * acc.y + q.z * acc.z) * iv : 0.f;
        F.gq[p * 2 + h] = q;
    }
}

// ---------------------------------------------------------------------------------------------
// 2. per (center, half): g_beta, u = M^-1 g_beta, center-side gradients
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void crg_center(CrgBatch b)
{
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const CrgFrame &F = b.f[L.f];
    const int S = b.sparsity, HW = b.half_win;
    const int H = F.H, W = F.W, Ws = W / S, Hs = H / S;
    const int h = threadIdx.x >> 7;
    const int bx = L.tx * 16 + (threadIdx.x & 15);
    const int by = L.ty * 8 + ((threadIdx.x & 127) >> 4);
    if (bx >= Ws || by >= Hs) return;
    const float *feat = h ? F.y2 : F.y1, *tgt = h ? F.y1 : F.y2, *var = h ? F.var2 : F.var1;
    const int cx = bx * S, cy = by * S;
    const size_t c = (size_t)cy * W + cx;
    const float3 fc = ld3(feat, c), ac = ld3(F.alb, c), nc = ld3(F.nrm, c);
    const float vc = var[c], sc = sqrtf(vc);
    const size_t crec = ((size_t)by * Ws + bx) * 2 + h;
    float bt[18];
#pragma unroll
    for (int k = 0; k < 18; ++k) bt[k] = F.beta[crec * 18 + k];
    G10 g;
    g.zero();
    float gb[18];
#pragma unroll
    for (int k = 0; k < 18; ++k) gb[k] = 0.f;

    // (a) reconstruction adjoint, gathered over the pixels whose center range holds (by, bx)
    const int py0 = max(0, cy - HW - S), py1 = min(H - 1, cy + HW + S);
    const int px0 = max(0, cx - HW - S), px1 = min(W - 1, cx + HW + S);
    for (int py = py0; py <= py1; ++py)
    {
        if (by < max(0, idivup(py - HW, S)) || by > min((H - 1) / S, (py + HW) / S)) continue;
        for (int px = px0; px <= px1; ++px)
        {
            if (bx < max(0, idivup(px - HW, S)) || bx > min((W - 1) / S, (px + HW) / S)) continue;
            const size_t p = (size_t)py * W + px;
            const float4 q = F.gq[p * 2 + h];
            if (q.x == 0.f && q.y == 0.f && q.z == 0.f && q.w == 0.f) continue;
            const float3 fp = ld3(feat, p);
            const float vp = var[p], sp = sqrtf(vp);
            float d[3][6], pred[3], inv, gd[3][6];
            const float w = recon_pair(fp, ld3(F.alb, p), ld3(F.nrm, p), vp, sp, fc, ac, nc, vc, sc, bt, d, pred, inv);
            const float ga[3] = {q.x, q.y, q.z};
            float gw = q.w;
#pragma unroll
            for (int ch = 0; ch < 3; ++ch)
            {
                gw += ga[ch] * pred[ch];
                const float wg = w * ga[ch];
#pragma unroll
                for (int k = 0; k < 6; ++k)
                {
                    gb[k * 3 + ch] += wg * d[ch][k];
                    gd[ch][k] = wg * bt[k * 3 + ch];
                }
            }
            pair_adj(sub3(fp, fc), (vp + 1e-4f) + vc, inv, sp, sc, gw, gd, false, g);
        }
    }

    // (b) u = M^-1 g_beta per channel, from the Cholesky factors of the forward (running the normal equations
    // again was a third pass over the window: 256x256, forward + backward, win 27 / sparsity 4 1626 -> 1406 us,
    // win 17 / sparsity 1 2453 -> 2327)
    float u[18];
#pragma unroll
    for (int ch = 0; ch < 3; ++ch)
    {
        float x[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) x[k] = gb[k * 3 + ch];
        fact6_solve(F.fact + fact_at((size_t)Hs * Ws, crec >> 1, h, ch), (size_t)Hs * Ws, x);
#pragma unroll
        for (int k = 0; k < 6; ++k) u[k * 3 + ch] = x[k];
    }

    // (c) regression adjoint, center side
    for (int iy = cy - HW; iy <= cy + HW; ++iy)
        for (int ix = cx - HW; ix <= cx + HW; ++ix)
        {
            const size_t i = (size_t)mirror(iy, H) * W + mirror(ix, W);
            const float3 fi = ld3(feat, i);
            const float vi = var[i], si = sqrtf(vi);
            float d[3][6], inv, gd[3][6], gt[3];
            const float w = reg_pair(fi, ld3(F.alb, i), ld3(F.nrm, i), vi, si, fc, ac, nc, vc, sc, d, inv);
            const float gw = reg_tap_adj(w, d, bt, u, ld3(tgt, i), gd, gt);
            pair_adj(sub3(fi, fc), (vc + 1e-4f) + vi, inv, si, sc, gw, gd, false, g);
        }

    float *uo = F.u + crec * 18;
#pragma unroll
    for (int k = 0; k < 18; ++k) uo[k] = u[k];
    float4 *go = reinterpret_cast<float4 *>(F.gcen + crec * 12);
    go[0] = make_float4(g.f.x, g.f.y, g.f.z, g.a.x);
    go[1] = make_float4(g.a.y, g.a.z, g.n.x, g.n.y);
    go[2] = make_float4(g.n.z, g.v, 0.f, 0.f);
}

// ---------------------------------------------------------------------------------------------
// 3. per pixel: pixel-side and tap-side adjoints, both halves
// ---------------------------------------------------------------------------------------------
// Tap positions j (along one axis of size n) that the reflect-101 index maps onto pixel i.
__device__ __forceinline__ int mirror_sources(int i, int n, int js[3])
{
    int m = 0;
    js[m++] = i;
    if (i >= 1) js[m++] = -i;
    if (i <= n - 2) js[m++] = 2 * (n - 1) - i;
    return m;
}

__device__ __forceinline__ int floor_div(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

__global__ __launch_bounds__(256) void crg_pixel(CrgBatch b)
{
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const CrgFrame &F = b.f[L.f];
    const int S = b.sparsity, HW = b.half_win;
    const int H = F.H, W = F.W, Ws = W / S, Hs = H / S;
    const int px = L.tx * 16 + (threadIdx.x & 15), py = L.ty * 16 + (threadIdx.x >> 4);
    if (px >= W || py >= H) return;
    const size_t p = (size_t)py * W + px;
    const float3 ap = ld3(F.alb, p), np = ld3(F.nrm, p);
    const int sx = max(0, idivup(px - HW, S)), ex = min((W - 1) / S, (px + HW) / S);
    const int sy = max(0, idivup(py - HW, S)), ey = min((H - 1) / S, (py + HW) / S);
    int jys[3], jxs[3];
    const int njy = mirror_sources(py, H, jys), njx = mirror_sources(px, W, jxs);
    const bool grid = (px % S == 0) && (py % S == 0);
    // 3x3 clamped neighbourhood (variance adjoint)
    const int nx0 = max(0, px - 1), nx1 = min(W - 1, px + 1), ny0 = max(0, py - 1), ny1 = min(H - 1, py + 1);
    const float ncount = (float)((nx1 - nx0 + 1) * (ny1 - ny0 + 1) - 1);

    float3 gy_own[2], gy_oth[2];
    float3 galb = make_float3(0.f, 0.f, 0.f), gnrm = galb;
    float3 ev[2];
    for (int h = 0; h < 2; ++h)
    {
        const float *feat = h ? F.y2 : F.y1, *tgt = h ? F.y1 : F.y2, *var = h ? F.var2 : F.var1;
        const float3 fp = ld3(feat, p), tp = ld3(tgt, p);
        const float vp = var[p], sp = sqrtf(vp);
        G10 g;
        g.zero();
        float3 gt = make_float3(0.f, 0.f, 0.f);

        // (a) reconstruction adjoint, pixel side
        const float4 q = F.gq[p * 2 + h];
        if (!(q.x == 0.f && q.y == 0.f && q.z == 0.f && q.w == 0.f))
        {
            const float ga[3] = {q.x, q.y, q.z};
            for (int iy = sy; iy <= ey; ++iy)
                for (int ix = sx; ix <= ex; ++ix)
                {
                    const size_t c = (size_t)(iy * S) * W + (size_t)(ix * S);
                    const float *bt = F.beta + (((size_t)iy * Ws + ix) * 2 + h) * 18;
                    const float3 fc = ld3(feat, c);
                    const float vc = var[c], sc = sqrtf(vc);
                    float d[3][6], pred[3], inv, gd[3][6];
                    const float w = recon_pair(fp, ap, np, vp, sp, fc, ld3(F.alb, c), ld3(F.nrm, c), vc, sc, bt, d,
                                               pred, inv);
                    float gw = q.w;
#pragma unroll
                    for (int ch = 0; ch < 3; ++ch)
                    {
                        gw += ga[ch] * pred[ch];
#pragma unroll
                        for (int k = 0; k < 6; ++k) gd[ch][k] = w * ga[ch] * bt[k * 3 + ch];
                    }
                    pair_adj(sub3(fp, fc), (vp + 1e-4f) + vc, inv, sp, sc, gw, gd, true, g);
                }
        }

        // (b) regression adjoint, tap side: every (center, tap position) whose tap maps onto p
        for (int a = 0; a < njy; ++a)
        {
            const int jy = jys[a];
            const int by0 = max(0, floor_div(jy - HW + S - 1, S)), by1 = min(Hs - 1, floor_div(jy + HW, S));
            for (int by = by0; by <= by1; ++by)
                for (int e = 0; e < njx; ++e)
                {
                    const int jx = jxs[e];
                    const int bx0 = max(0, floor_div(jx - HW + S - 1, S)), bx1 = min(Ws - 1, floor_div(jx + HW, S));
                    for (int bx = bx0; bx <= bx1; ++bx)
                    {
                        const size_t c = (size_t)(by * S) * W + (size_t)(bx * S);
                        const size_t crec = ((size_t)by * Ws + bx) * 2 + h;
                        const float *bt = F.beta + crec * 18;
                        const float *u = F.u + crec * 18;
                        const float3 fc = ld3(feat, c);
                        const float vc = var[c], sc = sqrtf(vc);
                        float d[3][6], inv, gd[3][6], gtt[3];
                        const float w = reg_pair(fp, ap, np, vp, sp, fc, ld3(F.alb, c), ld3(F.nrm, c), vc, sc, d, inv);
                        const float gw = reg_tap_adj(w, d, bt, u, tp, gd, gtt);
                        gt.x += gtt[0];
                        gt.y += gtt[1];
                        gt.z += gtt[2];
                        pair_adj(sub3(fp, fc), (vc + 1e-4f) + vp, inv, sp, sc, gw, gd, true, g);
                    }
                }
        }

        // (c) center-side terms when p is a regression center
        if (grid)
        {
            const float4 *gc =
                reinterpret_cast<const float4 *>(F.gcen + (((size_t)(py / S) * Ws + px / S) * 2 + h) * 12);
            const float4 g0 = gc[0], g1 = gc[1], g2 = gc[2];
            g.f.x += g0.x; g.f.y += g0.y; g.f.z += g0.z;
            g.a.x += g0.w; g.a.y += g1.x; g.a.z += g1.y;
            g.n.x += g1.z; g.n.y += g1.w; g.n.z += g2.x;
            g.v += g2.y;
        }

        // (d) variance adjoint, own term: e = g_v * 2 (mean_neighbours - f_p)
        const float *gvx = h ? F.gvarb : F.gvara;
        const float gv = g.v + (gvx ? gvx[p] : 0.f);
        float3 m = make_float3(0.f, 0.f, 0.f);
        for (int yy = ny0; yy <= ny1; ++yy)
            for (int xx = nx0; xx <= nx1; ++xx)
            {
                if (yy == py && xx == px) continue;
                const float3 f = ld3(feat, (size_t)yy * W + xx);
                m.x += f.x; m.y += f.y; m.z += f.z;
            }
        const float in = 1.f / ncount;
        const float3 e = make_float3(2.f * gv * (m.x * in - fp.x), 2.f * gv * (m.y * in - fp.y),
                                     2.f * gv * (m.z * in - fp.z));
        gy_own[h] = sub3(g.f, e);
        gy_oth[h] = gt;
        ev[h] = make_float3(e.x * in, e.y * in, e.z * in);
        galb.x += g.a.x; galb.y += g.a.y; galb.z += g.a.z;
        gnrm.x += g.n.x; gnrm.y += g.n.y; gnrm.z += g.n.z;
    }
    // half A: features imga, target imgb; half B: features imgb, target imga
    st3(F.gya, p, make_float3(gy_own[0].x + gy_oth[1].x, gy_own[0].y + gy_oth[1].y, gy_own[0].z + gy_oth[1].z));
    st3(F.gyb, p, make_float3(gy_own[1].x + gy_oth[0].x, gy_own[1].y + gy_oth[0].y, gy_own[1].z + gy_oth[0].z));
    st3(F.galb, p, galb);
    st3(F.gnrm, p, gnrm);
    float *eo = F.evar + p * 6;
    eo[0] = ev[0].x; eo[1] = ev[0].y; eo[2] = ev[0].z;
    eo[3] = ev[1].x; eo[4] = ev[1].y; eo[5] = ev[1].z;
}

// ---------------------------------------------------------------------------------------------
// Tiled forms of 1-3 for windows that fit LDS (win 17 / sparsity 4 and smaller)
// ---------------------------------------------------------------------------------------------
struct EdgeYes {
    static constexpr bool value = true;
};
struct EdgeNo {
    static constexpr bool value = false;
};

// Sum over the 16 lanes of a DPP row, the same bits in every lane (after each rotation the values
// repeat with half the period, so both partners add the same two numbers).
template <int R>
__device__ __forceinline__ float row_ror_add(float v)
{
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + R, 0xf, 0xf, true));
}
__device__ __forceinline__ float row_sum(float v)
{
    return row_ror_add<1>(row_ror_add<2>(row_ror_add<4>(row_ror_add<8>(v))));
}

// Staged center records of a 16x16-pixel tile, in float4: beta A, beta B (18 floats each), with U: u A,
// u B, then (y1, var1) (y2, var2) (albedo, std1) (normal, std2).
template <bool U, int MAXC>
struct CrgCenters {
    static constexpr int REC = U ? 22 : 13, IMG = REC - 4;
    int clo, rlo, ncx;
    __device__ __forceinline__ void stage(const CrgFrame &F, float4 (*cs)[REC], int x0, int y0, int S, int HW)
    {
        const int H = F.H, W = F.W, Ws = W / S, Hs = H / S;
        clo = max(0, (x0 - HW + S - 1) / S);
        rlo = max(0, (y0 - HW + S - 1) / S);
        if (x0 <= HW) clo = 0;
        if (y0 <= HW) rlo = 0;
        ncx = min(Ws - 1, (x0 + 15 + HW) / S) - clo + 1;
        const int ncy = min(Hs - 1, (y0 + 15 + HW) / S) - rlo + 1;
        for (int i = threadIdx.x; i < ncx * ncy * IMG; i += 256)
        {
            const int c = i / IMG, q = i - c * IMG, ry = c / ncx, rx = c - ry * ncx;
            const size_t crec = ((size_t)(rlo + ry) * Ws + (clo + rx)) * 9;  // float4 of beta or u
            const float4 *src = reinterpret_cast<const float4 *>(q < 9 ? F.beta : F.u);
            cs[c][q] = src[crec + (q < 9 ? q : q - 9)];
        }
        for (int i = threadIdx.x; i < ncx * ncy; i += 256)
        {
            const int ry = i / ncx, rx = i - ry * ncx;
            const size_t p = (size_t)((rlo + ry) * S) * W + (size_t)((clo + rx) * S);
            const float3 a = ld3(F.y1, p), bb = ld3(F.y2, p), al = ld3(F.alb, p), nr = ld3(F.nrm, p);
            const float v1 = F.var1[p], v2 = F.var2[p];
            cs[i][IMG] = make_float4(a.x, a.y, a.z, v1);
            cs[i][IMG + 1] = make_float4(bb.x, bb.y, bb.z, v2);
            cs[i][IMG + 2] = make_float4(al.x, al.y, al.z, sqrtf(v1));
            cs[i][IMG + 3] = make_float4(nr.x, nr.y, nr.z, sqrtf(v2));
        }
    }
};
// centers per tile axis
static int crg_axis_centers(int S, int HW) { return (15 + 2 * HW) / S + 1; }

// 1. (g_acc, g_sumW) of the reconstruction, both halves of a pixel per lane, its centers from LDS
// (512x512, win 17: 58 -> 23 us against a lane's own loads of every center record).
template <int MAXC>
__global__ __launch_bounds__(256) void crg_prep_tile(CrgBatch b)
{
    typedef CrgCenters<false, MAXC> Rec;
    __shared__ float4 cs[MAXC][Rec::REC];
    const TileLoc L = locate(b.map, xcd_tile(blockIdx.x, b.map.total));
    const CrgFrame &F = b.f[L.f];
    const int S = b.sparsity, HW = b.half_win, H = F.H, W = F.W;
    Rec rec;
    rec.stage(F, cs, L.tx * 16, L.ty * 16, S, HW);
    __syncthreads();
    const int px = L.tx * 16 + (threadIdx.x & 15), py = L.ty * 16 + (threadIdx.x >> 4);
    if (px >= W || py >= H) return;
    const size_t p = (size_t)py * W + px;
    const int sx = max(0, idivup(px - HW, S)), ex = min((W - 1) / S, (px + HW) / S);
    const int sy = max(0, idivup(py - HW, S)), ey = min((H - 1) / S, (py + HW) / S);
    const float3 ap = ld3(F.alb, p), np = ld3(F.nrm, p);
    float3 fp[2] = {ld3(F.y1, p), ld3(F.y2, p)};
    const float vp[2] = {F.var1[p], F.var2[p]};
    const float sp[2] = {sqrtf(vp[0]), sqrtf(vp[1])};
    float3 acc[2];
    float sum[2] = {0.f, 0.f};
    acc[0] = acc[1] = make_float3(0.f, 0.f, 0.f);
    for (int iy = sy; iy <= ey; ++iy)
        for (int ix = sx; ix <= ex; ++ix)
        {
            const float4 *c = cs[(iy - rec.rlo) * rec.ncx + (ix - rec.clo)];
            const float4 A = c[Rec::IMG + 2], N = c[Rec::IMG + 3];
#pragma unroll
            for (int h = 0; h < 2; ++h)
            {
                const float4 P = c[Rec::IMG + h];
                float d[3][6], pred[3], inv;
                const float w = recon_pair(fp[h], ap, np, vp[h], sp[h], make_float3(P.x, P.y, P.z),
                                           make_float3(A.x, A.y, A.z), make_float3(N.x, N.y, N.z), P.w, h ? N.w : A.w,
                                           reinterpret_cast<const float *>(c) + 18 * h, d, pred, inv);
                acc[h].x += w * pred[0];
                acc[h].y += w * pred[1];
                acc[h].z += w * pred[2];
                sum[h] += w;
            }
        }
#pragma unroll
    for (int h = 0; h < 2; ++h)
    {
        const float iv = 1.f / fmaxf(sum[h], 1e-7f);
        const float3 go = ld3(h ? F.goutb : F.gouta, p);
        float4 q;
        q.x = acc[h].x * iv > 0.f ? go.x * iv : 0.f;
        q.y = acc[h].y * iv > 0.f ? go.y * iv : 0.f;
        q.z = acc[h].z * iv > 0.f ? go.z * iv : 0.f;
        q.w = sum[h] > 1e-7f ? -(q.x * acc[h].x + q.y * acc[h].y + q.z * acc[h].z) * iv : 0.f;
        F.gq[p * 2 + h] = q;
    }
}

// 2. g_beta, u = M^-1 g_beta and the center-side gradients: a 4x4 block of centers per 512-lane
// workgroup, 16 lanes per (center, half) that split the window's taps and add up with DPP rotations;
// the pixels of the block's windows (image planes and the two g_acc planes, 29x29 px for win 17 /
// sparsity 4: 81 KB, two blocks per CU) in LDS; the Cholesky factor from the forward instead of a
// second accumulation of the normal equations. Every factor of a tap's adjoint that only depends on the
// center is taken out of the sum, e.g. sum gd_2 = beta_2 sum w g_acc: 28 sums for the reconstruction and
// 22 for the regression side instead of all of g_d. One lane per (center, half) had 512 waves for the
// whole chip at 512x512 and direct loads for every tap: 496 -> 63 us (VALU-bound now; at four waves per SIMD it
// spills five VGPRs, 24 B a lane).
constexpr int CC_T = 4, CC_MAXPX = 29 * 29;
__global__ __launch_bounds__(512, 4) void crg_center_tile(CrgBatch b)
{
    __shared__ float4 tl[6][CC_MAXPX];  // (y1, var1) (y2, var2) (albedo, std1) (normal, std2), g_acc A, B
    const TileLoc L = locate(b.map, xcd_tile(blockIdx.x, b.map.total));
    const CrgFrame &F = b.f[L.f];
    const int S = b.sparsity, HW = b.half_win, H = F.H, W = F.W, Ws = W / S, Hs = H / S;
    const int bx0 = L.tx * CC_T, by0 = L.ty * CC_T;
    const int RW = (CC_T - 1) * S + 1 + 2 * HW, NP = RW * RW;
    for (int i = threadIdx.x; i < NP; i += 512)
    {
        const int ly = i / RW, lx = i - ly * RW;
        const int ux = bx0 * S - HW + lx, uy = by0 * S - HW + ly;
        const size_t p = (size_t)mirror(min(uy, H - 1 + HW), H) * W + mirror(min(ux, W - 1 + HW), W);
        const float3 a = ld3(F.y1, p), bb = ld3(F.y2, p), al = ld3(F.alb, p), nr = ld3(F.nrm, p);
        const float v1 = F.var1[p], v2 = F.var2[p];
        // a position outside the image is a regression tap (of the mirrored pixel) but no pixel of the
        // reconstruction
        float4 qa = make_float4(0.f, 0.f, 0.f, 0.f), qb = qa;
        if (ux >= 0 && uy >= 0 && ux < W && uy < H) qa = F.gq[p * 2], qb = F.gq[p * 2 + 1];
        tl[0][i] = make_float4(a.x, a.y, a.z, v1);
        tl[1][i] = make_float4(bb.x, bb.y, bb.z, v2);
        tl[2][i] = make_float4(al.x, al.y, al.z, sqrtf(v1));
        tl[3][i] = make_float4(nr.x, nr.y, nr.z, sqrtf(v2));
        tl[4][i] = qa;
        tl[5][i] = qb;
    }
    __syncthreads();
    const int lane = threadIdx.x & 15, ch2 = threadIdx.x >> 4;
    const int h = __builtin_amdgcn_readfirstlane(ch2 >> 4), ci = ch2 & 15;
    const int bx = bx0 + (ci & 3), by = by0 + (ci >> 2);
    const bool active = bx < Ws && by < Hs;  // the others run along (their sums are not stored)
    const size_t crec = ((size_t)min(by, Hs - 1) * Ws + min(bx, Ws - 1)) * 2 + h;
    const int corner = (ci >> 2) * S * RW + (ci & 3) * S, mid = corner + HW * RW + HW;
    const float4 *own = tl[h], *oth = tl[1 - h], *alb = tl[2], *nrm = tl[3], *gq = tl[4 + h];
    float3 fc, ac, nc;
    float vc, sc;
    {
        const float4 P = own[mid], A = alb[mid], N = nrm[mid];
        fc = make_float3(P.x, P.y, P.z); ac = make_float3(A.x, A.y, A.z); nc = make_float3(N.x, N.y, N.z);
        vc = P.w;
        sc = h ? N.w : A.w;
    }
    float bt[18];
#pragma unroll
    for (int k = 0; k < 18; ++k) bt[k] = F.beta[crec * 18 + k];
    const float vce = vc + 1e-4f, sce = sc + 1e-2f;
    // a pixel whose lower center bound rounds up past center 0 (idivup of a negative value)
    const bool skx = bx == 0, sky = by == 0;
    const bool edge = bx0 == 0 || by0 == 0;  // wave-uniform

    const int W1 = 2 * HW + 1, n = W1 * W1;
    const uint32_t magic = ((1u << 20) + W1 - 1) / W1;
    struct Tap {
        float3 df, da, dn;
        float D, rS, E, inv, d1[3];
    };
    auto tap = [&](int i) {
        const float4 P = own[i], A = alb[i], N = nrm[i];
        Tap t;
        t.df = make_float3(P.x - fc.x, P.y - fc.y, P.z - fc.z);
        t.da = make_float3(A.x - ac.x, A.y - ac.y, A.z - ac.z);
        t.dn = make_float3(N.x - nc.x, N.y - nc.y, N.z - nc.z);
        t.D = t.df.x * t.df.x + t.df.y * t.df.y + t.df.z * t.df.z;
        t.rS = fast_rcp(vce + P.w);
        t.E = fast_exp2(-kLog2e * t.D * t.rS);
        t.inv = fast_rcp(sce + (h ? N.w : A.w));
        t.d1[0] = t.df.x * t.inv; t.d1[1] = t.df.y * t.inv; t.d1[2] = t.df.z * t.inv;
        return t;
    };
    auto dot6 = [](const float *v, int c, const Tap &t) {  // v . d of channel c (v [6][3])
        const float d2 = c == 0 ? t.da.x : (c == 1 ? t.da.y : t.da.z);
        return v[c] + v[3 + c] * t.d1[c] + v[6 + c] * d2 + v[9 + c] * t.dn.x + v[12 + c] * t.dn.y + v[15 + c] * t.dn.z;
    };

    // (a) reconstruction adjoint over the pixels of the window
    float gb[18], sD[3] = {0.f, 0.f, 0.f}, sT[3] = {0.f, 0.f, 0.f}, sG[3] = {0.f, 0.f, 0.f}, sV = 0.f;
#pragma unroll
    for (int k = 0; k < 18; ++k) gb[k] = 0.f;
    for (int j = lane; j < n; j += 16)
    {
        const int row = (int)((uint32_t)j * magic >> 20), col = j - row * W1, i = corner + row * RW + col;
        float4 q = gq[i];
        if (edge)
        {
            // pixel coordinates row - HW + cy, col - HW + cx; center 0 is skipped by the pixels
            // HW - S < p < HW, i.e. (center coordinate 0) window offsets 2 HW - S < row < 2 HW
            if ((sky && row > 2 * HW - S && row < 2 * HW) || (skx && col > 2 * HW - S && col < 2 * HW))
                q = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        const Tap t = tap(i);
        const float w = t.E + 1e-7f;
        const float ga[3] = {q.x, q.y, q.z};
        float gw = q.w;
#pragma unroll
        for (int c = 0; c < 3; ++c)
        {
            gw += ga[c] * dot6(bt, c, t);
            const float wg = w * ga[c], m = wg * t.inv;
            gb[c] += wg;
            gb[3 + c] += wg * t.d1[c];
            gb[6 + c] += wg * (c == 0 ? t.da.x : (c == 1 ? t.da.y : t.da.z));
            gb[9 + c] += wg * t.dn.x;
            gb[12 + c] += wg * t.dn.y;
            gb[15 + c] += wg * t.dn.z;
            sT[c] += m;
            sG[c] += m * t.d1[c];
        }
        const float g1 = gw * t.E * t.rS;
        sD[0] += g1 * t.df.x; sD[1] += g1 * t.df.y; sD[2] += g1 * t.df.z;
        sV += g1 * t.D * t.rS;
    }
#pragma unroll
    for (int k = 0; k < 18; ++k) gb[k] = row_sum(gb[k]);
#pragma unroll
    for (int c = 0; c < 3; ++c) sD[c] = row_sum(sD[c]), sT[c] = row_sum(sT[c]), sG[c] = row_sum(sG[c]);
    sV = row_sum(sV);
    // the center is the Q side of the pair: minus the sums (dL/d df = -2 g1 df + gd_1 inv)
    float gf[3], gal[3], gn[3] = {0.f, 0.f, 0.f}, gden = 0.f, gv = sV;
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
        gf[c] = 2.f * sD[c] - bt[3 + c] * sT[c];
        gal[c] = -bt[6 + c] * gb[c];
#pragma unroll
        for (int k = 0; k < 3; ++k) gn[k] -= bt[9 + 3 * k + c] * gb[c];
        gden -= bt[3 + c] * sG[c];
    }

    // (b) u = M^-1 g_beta
    float u[18];
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
        float x[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) x[k] = gb[k * 3 + c];
        fact6_solve(F.fact + fact_at((size_t)Hs * Ws, crec >> 1, h, c), (size_t)Hs * Ws, x);
#pragma unroll
        for (int k = 0; k < 6; ++k) u[k * 3 + c] = x[k];
    }

    // (c) regression adjoint, center side: with r = t - beta . d and s = u . d, gd_k = w (u_k r - beta_k s)
    float sR[3] = {0.f, 0.f, 0.f}, sS[3] = {0.f, 0.f, 0.f}, sRi[3] = {0.f, 0.f, 0.f}, sSi[3] = {0.f, 0.f, 0.f};
    float sRd[3] = {0.f, 0.f, 0.f}, sSd[3] = {0.f, 0.f, 0.f};
    sD[0] = sD[1] = sD[2] = sV = 0.f;
    for (int j = lane; j < n; j += 16)
    {
        const int row = (int)((uint32_t)j * magic >> 20), col = j - row * W1, i = corner + row * RW + col;
        const float4 T = oth[i];
        const Tap t = tap(i);
        const float w = t.E + 1e-7f;
        const float tv[3] = {T.x, T.y, T.z};
        float gw = 0.f;
#pragma unroll
        for (int c = 0; c < 3; ++c)
        {
            const float r = tv[c] - dot6(bt, c, t), s = dot6(u, c, t);
            gw += s * r;
            const float wr = w * r, ws = w * s, wri = wr * t.inv, wsi = ws * t.inv;
            sR[c] += wr;
            sS[c] += ws;
            sRi[c] += wri;
            sSi[c] += wsi;
            sRd[c] += wri * t.d1[c];
            sSd[c] += wsi * t.d1[c];
        }
        const float g1 = gw * t.E * t.rS;
        sD[0] += g1 * t.df.x; sD[1] += g1 * t.df.y; sD[2] += g1 * t.df.z;
        sV += g1 * t.D * t.rS;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
        sR[c] = row_sum(sR[c]); sS[c] = row_sum(sS[c]); sRi[c] = row_sum(sRi[c]); sSi[c] = row_sum(sSi[c]);
        sRd[c] = row_sum(sRd[c]); sSd[c] = row_sum(sSd[c]); sD[c] = row_sum(sD[c]);
    }
    gv += row_sum(sV);
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
        gf[c] += 2.f * sD[c] - (u[3 + c] * sRi[c] - bt[3 + c] * sSi[c]);
        gal[c] -= u[6 + c] * sR[c] - bt[6 + c] * sS[c];
#pragma unroll
        for (int k = 0; k < 3; ++k) gn[k] -= u[9 + 3 * k + c] * sR[c] - bt[9 + 3 * k + c] * sS[c];
        gden -= u[3 + c] * sRd[c] - bt[3 + c] * sSd[c];
    }
    if (sc > 0.f) gv += 0.5f * gden / sc;
    if (!active || lane != 0) return;
    float *uo = F.u + crec * 18;
#pragma unroll
    for (int k = 0; k < 18; ++k) uo[k] = u[k];
    float4 *go = reinterpret_cast<float4 *>(F.gcen + crec * 12);
    go[0] = make_float4(gf[0], gf[1], gf[2], gal[0]);
    go[1] = make_float4(gal[1], gal[2], gn[0], gn[1]);
    go[2] = make_float4(gn[2], gv, 0.f, 0.f);
}

// 3. pixel-side and tap-side adjoints: the pairs of both loops are the same (pixel, center) pairs at the
// same weight and delta, so one pass over the pixel's centers (records in LDS) serves both, with
// alpha = w (g_acc - s) and rho = w r per channel, gd_k = beta_k alpha + u_k rho, r = t - pred. A tap
// position reflected onto the pixel repeats the pair, so near an edge the regression terms are scaled
// by how many of the pixel's positions lie in the center's window; the reconstruction leaves center
// 0 out where its lower bound rounds up past it (EDGE tiles). 512x512, win 17: 202 -> 64 us.
template <int MAXC>
__global__ __launch_bounds__(256) void crg_pixel_tile(CrgBatch b)
{
    typedef CrgCenters<true, MAXC> Rec;
    __shared__ float4 cs[MAXC][Rec::REC];
    const TileLoc L = locate(b.map, xcd_tile(blockIdx.x, b.map.total));
    const CrgFrame &F = b.f[L.f];
    const int S = b.sparsity, HW = b.half_win, H = F.H, W = F.W, Ws = W / S, Hs = H / S;
    const int x0 = L.tx * 16, y0 = L.ty * 16;
    Rec rec;
    rec.stage(F, cs, x0, y0, S, HW);
    __syncthreads();
    const int px = x0 + (threadIdx.x & 15), py = y0 + (threadIdx.x >> 4);
    if (px >= W || py >= H) return;
    const size_t p = (size_t)py * W + px;
    const float3 ap = ld3(F.alb, p), np = ld3(F.nrm, p);
    const float3 fp[2] = {ld3(F.y1, p), ld3(F.y2, p)};
    const float vp[2] = {F.var1[p], F.var2[p]};
    const float sp[2] = {sqrtf(vp[0]), sqrtf(vp[1])};
    const float4 q[2] = {F.gq[p * 2], F.gq[p * 2 + 1]};
    float gf[2][3], gt[2][3], gv[2] = {0.f, 0.f}, gden[2] = {0.f, 0.f};
    float galb[3] = {0.f, 0.f, 0.f}, gnrm[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < 3; ++c) gf[h][c] = gt[h][c] = 0.f;
    // centers whose window holds the pixel
    const int cy0 = py <= HW ? 0 : (py - HW + S - 1) / S, cy1 = min(Hs - 1, (py + HW) / S);
    const int cx0 = px <= HW ? 0 : (px - HW + S - 1) / S, cx1 = min(Ws - 1, (px + HW) / S);
    auto run = [&](auto edge) {
        constexpr bool EDGE = decltype(edge)::value;
        const int sx = EDGE ? max(0, idivup(px - HW, S)) : cx0, sy = EDGE ? max(0, idivup(py - HW, S)) : cy0;
        for (int iy = cy0; iy <= cy1; ++iy)
            for (int ix = cx0; ix <= cx1; ++ix)
            {
                const float4 *rc = cs[(iy - rec.rlo) * rec.ncx + (ix - rec.clo)];
                const float4 A = rc[Rec::IMG + 2], N = rc[Rec::IMG + 3];
                const float da[3] = {ap.x - A.x, ap.y - A.y, ap.z - A.z};
                const float dn[3] = {np.x - N.x, np.y - N.y, np.z - N.z};
                float mult = 1.f;
                bool recon = true;
                if constexpr (EDGE)
                {
                    const int cy = iy * S, cx = ix * S;
                    const int my = 1 + (py >= 1 && py + cy <= HW) + (py <= H - 2 && 2 * (H - 1) - py - cy <= HW);
                    const int mx = 1 + (px >= 1 && px + cx <= HW) + (px <= W - 2 && 2 * (W - 1) - px - cx <= HW);
                    mult = (float)(my * mx);
                    recon = iy >= sy && ix >= sx;
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
                {
                    const float *bt = reinterpret_cast<const float *>(rc) + 18 * h, *u = bt + 36;
                    const float4 P = rc[Rec::IMG + h];
                    const float3 tp = fp[1 - h];
                    const float df[3] = {fp[h].x - P.x, fp[h].y - P.y, fp[h].z - P.z};
                    const float D = df[0] * df[0] + df[1] * df[1] + df[2] * df[2];
                    const float rS = fast_rcp((vp[h] + 1e-4f) + P.w);
                    const float E = fast_exp2(-kLog2e * D * rS), w = E + 1e-7f;
                    const float inv = fast_rcp((sp[h] + 1e-2f) + (h ? N.w : A.w));
                    const float ga[3] = {recon ? q[h].x : 0.f, recon ? q[h].y : 0.f, recon ? q[h].z : 0.f};
                    float gw = recon ? q[h].w : 0.f;
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                    {
                        const float d1 = df[c] * inv;
                        const float pred = bt[c] + bt[3 + c] * d1 + bt[6 + c] * da[c] + bt[9 + c] * dn[0] +
                                           bt[12 + c] * dn[1] + bt[15 + c] * dn[2];
                        float s = u[c] + u[3 + c] * d1 + u[6 + c] * da[c] + u[9 + c] * dn[0] + u[12 + c] * dn[1] +
                                  u[15 + c] * dn[2];
                        float r = (c == 0 ? tp.x : (c == 1 ? tp.y : tp.z)) - pred;
                        float wr = w * r;
                        if constexpr (EDGE)
                        {
                            s *= mult;
                            wr *= mult;
                        }
                        gw += ga[c] * pred + s * r;
                        const float al = w * (ga[c] - s);
                        const float g1 = (bt[3 + c] * al + u[3 + c] * wr) * inv;
                        gf[h][c] += g1;
                        gden[h] -= g1 * d1;
                        gt[h][c] += w * s;
                        galb[c] += bt[6 + c] * al + u[6 + c] * wr;
#pragma unroll
                        for (int k = 0; k < 3; ++k) gnrm[k] += bt[9 + 3 * k + c] * al + u[9 + 3 * k + c] * wr;
                    }
                    const float g2 = gw * E * rS;
#pragma unroll
                    for (int c = 0; c < 3; ++c) gf[h][c] -= 2.f * g2 * df[c];
                    gv[h] += g2 * D * rS;
                }
            }
    };
    if (x0 <= HW || y0 <= HW || x0 + 15 >= W - 1 - HW || y0 + 15 >= H - 1 - HW)
        run(EdgeYes{});
    else
        run(EdgeNo{});

    const bool grid = (px % S == 0) && (py % S == 0);
    // 3x3 clamped neighbourhood (variance adjoint)
    const int nx0 = max(0, px - 1), nx1 = min(W - 1, px + 1), ny0 = max(0, py - 1), ny1 = min(H - 1, py + 1);
    const float in = 1.f / (float)((nx1 - nx0 + 1) * (ny1 - ny0 + 1) - 1);
    float e[2][3];
#pragma unroll
    for (int h = 0; h < 2; ++h)
    {
        float g = gv[h];
        if (sp[h] > 0.f) g += 0.5f * gden[h] / sp[h];
        // center-side terms when p is a regression center
        if (grid)
        {
            const float4 *gc = reinterpret_cast<const float4 *>(F.gcen + (((size_t)(py / S) * Ws + px / S) * 2 + h) * 12);
            const float4 g0 = gc[0], g1 = gc[1], g2 = gc[2];
            gf[h][0] += g0.x; gf[h][1] += g0.y; gf[h][2] += g0.z;
            galb[0] += g0.w; galb[1] += g1.x; galb[2] += g1.y;
            gnrm[0] += g1.z; gnrm[1] += g1.w; gnrm[2] += g2.x;
            g += g2.y;
        }
        // variance adjoint, own term: e = g_v * 2 (mean_neighbours - f_p)
        const float *feat = h ? F.y2 : F.y1, *gvx = h ? F.gvarb : F.gvara;
        if (gvx) g += gvx[p];
        float m[3] = {0.f, 0.f, 0.f};
        for (int yy = ny0; yy <= ny1; ++yy)
            for (int xx = nx0; xx <= nx1; ++xx)
            {
                if (yy == py && xx == px) continue;
                const float3 f = ld3(feat, (size_t)yy * W + xx);
                m[0] += f.x; m[1] += f.y; m[2] += f.z;
            }
        const float fv[3] = {fp[h].x, fp[h].y, fp[h].z};
#pragma unroll
        for (int c = 0; c < 3; ++c)
        {
            e[h][c] = 2.f * g * (m[c] * in - fv[c]);
            gf[h][c] -= e[h][c];
        }
    }
    // half A: features imga, target imgb; half B: features imgb, target imga
    st3(F.gya, p, make_float3(gf[0][0] + gt[1][0], gf[0][1] + gt[1][1], gf[0][2] + gt[1][2]));
    st3(F.gyb, p, make_float3(gf[1][0] + gt[0][0], gf[1][1] + gt[0][1], gf[1][2] + gt[0][2]));
    st3(F.galb, p, make_float3(galb[0], galb[1], galb[2]));
    st3(F.gnrm, p, make_float3(gnrm[0], gnrm[1], gnrm[2]));
    float *eo = F.evar + p * 6;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < 3; ++c) eo[3 * h + c] = e[h][c] * in;
}

// ---------------------------------------------------------------------------------------------
// 4. per pixel: neighbour terms of the variance adjoint (the 3x3 relation is symmetric)
// ---------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void crg_var_gather(CrgBatch b)
{
    const int tile = xcd_tile(blockIdx.x, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const CrgFrame &F = b.f[L.f];
    const int H = F.H, W = F.W;
    const int px = L.tx * 16 + (threadIdx.x & 15), py = L.ty * 16 + (threadIdx.x >> 4);
    if (px >= W || py >= H) return;
    const size_t p = (size_t)py * W + px;
    float sa[3] = {0.f, 0.f, 0.f}, sb[3] = {0.f, 0.f, 0.f};
    for (int yy = max(0, py - 1); yy <= min(H - 1, py + 1); ++yy)
        for (int xx = max(0, px - 1); xx <= min(W - 1, px + 1); ++xx)
        {
            if (yy == py && xx == px) continue;
            const float *e = F.evar + ((size_t)yy * W + xx) * 6;
            sa[0] += e[0]; sa[1] += e[1]; sa[2] += e[2];
            sb[0] += e[3]; sb[1] += e[4]; sb[2] += e[5];
        }
    const float3 ga = ld3(F.gya, p), gb = ld3(F.gyb, p);
    st3(F.gya, p, make_float3(ga.x + sa[0], ga.y + sa[1], ga.z + sa[2]));
    st3(F.gyb, p, make_float3(gb.x + sb[0], gb.y + sb[1], gb.z + sb[2]));
}

// ---------------------------------------------------------------------------------------------
static int div_up_g(int a, int b) { return (a + b - 1) / b; }

hipError_t launch_cross_regression_grad(int n, const CrgFrame *fr, int win, int s, hipStream_t st)
{
    CrgBatch b{};
    int tx[XDN_MAX_FRAMES], ty[XDN_MAX_FRAMES], cx[XDN_MAX_FRAMES], cy[XDN_MAX_FRAMES];
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        tx[i] = div_up_g(fr[i].W, 16);
        ty[i] = div_up_g(fr[i].H, 16);
        cx[i] = div_up_g(fr[i].W / s, 16);
        cy[i] = div_up_g(fr[i].H / s, 8);
    }
    b.half_win = win / 2;
    b.sparsity = s;
    b.map = make_tilemap(n, tx, ty);
    if (b.map.total == 0) return hipSuccess;
    // tiled kernels where a tile's center records (at most 64, or 200: 70 KB) and the pixels of a 4x4
    // block of centers fit their LDS arrays: win 17 / sparsity 4 and smaller windows
    const int HW = win / 2, axis = crg_axis_centers(s, HW), rw = (CC_T - 1) * s + 1 + 2 * HW;
    const bool tiled = axis * axis <= 200 && rw * rw <= CC_MAXPX;
    const bool few = axis * axis <= 64;
    if (tiled)
        for (int i = 0; i < n; ++i)
        {
            cx[i] = div_up_g(fr[i].W / s, CC_T);
            cy[i] = div_up_g(fr[i].H / s, CC_T);
        }
    CrgBatch bc = b;
    bc.map = make_tilemap(n, cx, cy);
    if (tiled)
    {
        hipLaunchKernelGGL((few ? crg_prep_tile<64> : crg_prep_tile<200>), dim3(b.map.total), dim3(256), 0, st, b);
        hipLaunchKernelGGL(crg_center_tile, dim3(bc.map.total), dim3(512), 0, st, bc);
        hipLaunchKernelGGL((few ? crg_pixel_tile<64> : crg_pixel_tile<200>), dim3(b.map.total), dim3(256), 0, st, b);
    }
    else
    {
        hipLaunchKernelGGL(crg_recon_prep, dim3(b.map.total), dim3(256), 0, st, b);
        hipLaunchKernelGGL(crg_center, dim3(bc.map.total), dim3(256), 0, st, bc);
        hipLaunchKernelGGL(crg_pixel, dim3(b.map.total), dim3(256), 0, st, b);
    }
    hipLaunchKernelGGL(crg_var_gather, dim3(b.map.total), dim3(256), 0, st, b);
    return hipGetLastError();
}

}  // namespace xdn
