// Device code of the motion-vector reprojection (Reproject / isReprojValid, reproject.cu.cc:32-238), for the
// kernel of its own (k_reproject.hip) and the one that runs beside the reconstruction (k_regression.hip).
//
// One lane per pixel, 64x4 pixels per workgroup (full-wave rows for coalesced NHWC loads).
// HBM-bound gather. The validity mask and the tap indices must equal the reference bit for bit,
// so the decision path has a pinned FP32 operation order (no contraction in these functions):
//   posPrev   = fmaf(mvec, (float)dim, (float)pos)                      (:97, :103)
//   iposPrev  = trunc(posPrev + 0.5f), tap base = trunc(posPrev)          (cuda_utils.cuh:255-258)
//   depth     = |Zp - Z| / (fwZ + 1e-2f) > 10                             as a correctly rounded FP32 div
//   normal    = sqrtf(fmaf(dz,dz, fmaf(dx,dx, dy*dy))) / ((double)fwN + 1e-2) > 4   (FP64 divide)
//   bilinear  = fractions posPrev - floor(posPrev), sum of the valid weights in tap order >= 0.01f
// The two divisions are decided by exact products (see quotient_above_10 and quotient_above_4).
// The buffer list is passed by value (no pointer table in device memory, no host sync).
#pragma once
#include "xdn_common.h"
#include "xdn_kernels.h"

namespace xdn {

struct RpBatch {
    TileMap map;
    int n_list;
    int dims[XDN_MAX_LIST];
    RpFrame f[XDN_MAX_FRAMES];
};
static_assert(sizeof(RpBatch) <= 4096, "kernel argument too large");

constexpr int RP_TX = 64, RP_TY = 4;

// fl(a / b) > 10 for a >= 0 in FP32 without the division: the quotient rounds above 10 exactly when
// a / b > 10 + 2^-21 (half an ulp; the tie rounds to the even 10), and b (10 + 2^-21) has at most 49
// bits, so the FP64 product is exact. A negative b gives a quotient that is not above 10; infinities
// and NaN compare as their quotients do.
__device__ __forceinline__ bool quotient_above_10(float a, float b)
{
#pragma clang fp contract(off)
    return b >= 0.f && (double)a > (double)b * (10.0 + 0x1p-21);
}
// fl(d / x) > 4 for d >= 0 in FP64: exactly when d / x > 4 + 2^-51, i.e. d - 4x > 2^-51 x, where the
// fused difference is exact when d is within a factor of two of 4x and decides by far otherwise.
__device__ __forceinline__ bool quotient_above_4(double d, double x)
{
#pragma clang fp contract(off)
    return x > 0.0 && __builtin_fma(-4.0, x, d) > x * 0x1p-51;
}

__device__ __forceinline__ bool reproj_valid(int W, int H, int px, int py, float Z, float Zp, float fwZ, float3 n,
                                             float3 np, float fwN)
{
#pragma clang fp contract(off)
    if (px < 1 || py < 1 || px > W - 1 || py > H - 1) return false;
    const float dx = n.x - np.x, dy = n.y - np.y, dz = n.z - np.z;
    const float d = __builtin_sqrtf(__builtin_fmaf(dz, dz, __builtin_fmaf(dx, dx, dy * dy)));
    return !quotient_above_10(fabsf(Zp - Z), fwZ + 1e-2f) && !quotient_above_4((double)d, (double)fwN + 1e-2);
}

// A pixel whose bilinear taps all fail takes the mean of its valid 3x3 neighbours. With a tenth of the
// pixels disoccluded nearly every wave holds a few such pixels, and walking the nine neighbours in
// place ran nine dependent round trips for a handful of live lanes. The block queues them in LDS
// instead and gives every (pixel, neighbour) pair a lane: RP_ROUND pixels per round, all their
// validity inputs in flight together, then all their values; the values are summed in neighbour order
// from LDS, so the sums are those of the walk. HBM-bound gather: 3840x2160, three 3-channel buffers,
// 10% disoccluded: 363 -> 340 us (153 B/px, 3.7 TB/s). Where most of a block's pixels are queued (a scene cut, a
// disoccluded region) the rounds cost more than they hide: a lane then takes a queued pixel and walks its neighbours.
// 1920x1080, rounds alone -> with the walk, nothing valid: three 3-channel buffers 106 -> 55 us (every pixel walking in
// place: 53), one buffer 163 -> 58, four 4-channel ones 184 -> 111. The more floats a neighbour holds the longer the
// rounds stay the faster ones (pixels invalid at random, rounds and walk as fast: one buffer at about 85 queued of 256,
// three 3-channel ones at 115, four 4-channel ones at 140).
__device__ __forceinline__ int rp_walk_above(int floats) { return 80 + 4 * floats; }
constexpr int RP_ROUND = 28;               // queued pixels per round (28 x 9 = 252 of 256 lanes)
struct RpQueued {
    int ipx, ipy, c;                       // c: pixel of the block (thread index)
    float Z, fwZ, fwN, nx, ny, nz;
};

template <int FNL, int FD>
struct RpShared {
    static constexpr int ML = FNL > 0 ? FNL : XDN_MAX_LIST, MD = FNL > 0 ? FD : 4;
    RpQueued queue[256];
    float pair[9 * RP_ROUND][ML * MD];
    uint8_t pair_ok[9 * RP_ROUND];
    int queued;
};

// FNL > 0: the buffer list is FNL buffers of FD channels, known at compile time (the training
// step reprojects three 3-channel buffers); FNL == 0 reads the list shape from the batch.
// UNIT_OPAC: both opacities are one (the training step's case): their loads are skipped.
template <int FNL, int FD, bool UNIT_OPAC>
__device__ __forceinline__ void reproject_block(const RpBatch &b, int bid, RpShared<FNL, FD> &sh)
{
#pragma clang fp contract(off)
    constexpr int ML = FNL > 0 ? FNL : XDN_MAX_LIST, MD = FNL > 0 ? FD : 4;
    auto &queue = sh.queue;
    auto &pair = sh.pair;
    auto &pair_ok = sh.pair_ok;
    int &queued = sh.queued;
    const int tile = xcd_tile(bid, b.map.total);
    const TileLoc L = locate(b.map, tile);
    const RpFrame &F = b.f[L.f];
    const int H = F.H, W = F.W;
    const int bx0 = L.tx * RP_TX, by0 = L.ty * RP_TY;
    const int cx = bx0 + (threadIdx.x & (RP_TX - 1)), cy = by0 + threadIdx.x / RP_TX;
    const int nl = FNL > 0 ? FNL : b.n_list;
    if (threadIdx.x == 0) queued = 0;
    __syncthreads();
    if (cx < W && cy < H)
    {
        const size_t c = (size_t)cy * W + cx;
        float acc[ML][MD];
#pragma unroll
        for (int l = 0; l < ML; ++l)
#pragma unroll
            for (int k = 0; k < MD; ++k) acc[l][k] = 0.f;

        // Three round trips to memory: the pixel's own inputs; every bilinear tap's validity inputs,
        // loaded at coordinates clamped into the image and used only where the tap is in the image;
        // the list values of all four taps (compile-time lists; only the valid taps are summed).
        const float op = UNIT_OPAC ? 1.f : F.opac[c];
        const float mx = F.mvec[3 * c], my = F.mvec[3 * c + 1];
        const float fwN = F.pnFw[3 * c + 1];
        const float Z = F.linZ[3 * c], fwZ = F.linZ[3 * c + 1];
        const float3 n = ld3(F.nrm, c);
        bool valid = false, fallback = false;
        if (op != 0.f)
        {
            const float ppx = __builtin_fmaf(mx, (float)W, (float)cx);
            const float ppy = __builtin_fmaf(my, (float)H, (float)cy);
            const int ipx = (int)(ppx + 0.5f), ipy = (int)(ppy + 0.5f);
            const int bx = (int)ppx, by = (int)ppy;
            bool inb[4];
            size_t li[4];
            float po[4], pz[4];
            float3 pn[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
            {
                const int lx = bx + (t & 1), ly = by + (t >> 1);
                inb[t] = !(lx >= W || lx < 0 || ly >= H || ly < 0);
                li[t] = (size_t)min(max(ly, 0), H - 1) * W + min(max(lx, 0), W - 1);
                po[t] = UNIT_OPAC ? 1.f : F.prevOpac[li[t]];
                pz[t] = F.prevLinZ[3 * li[t]];
                pn[t] = ld3(F.prevNrm, li[t]);
            }
            bool v[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
            {
                v[t] = inb[t] && po[t] != 0.f && reproj_valid(W, H, ipx, ipy, Z, pz[t], fwZ, n, pn[t], fwN);
                valid = valid || v[t];
            }
            if (valid)
            {
                const float x = ppx - floorf(ppx), y = ppy - floorf(ppy);
                const float w[4] = {(1.f - x) * (1.f - y), x * (1.f - y), (1.f - x) * y, x * y};
                float sumw = 0.f;
                if constexpr (FNL > 0)
                {
                    // every tap's list values in flight at once (clamped in-image indices, so the
                    // loads are in bounds), then summed in tap order where the tap is valid
                    float val[4][ML][MD];
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int l = 0; l < ML; ++l)
#pragma unroll
                            for (int k = 0; k < MD; ++k) val[t][l][k] = F.in[l][li[t] * FD + k];
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                    {
#pragma unroll
                        for (int l = 0; l < ML; ++l)
#pragma unroll
                            for (int k = 0; k < MD; ++k)
                                acc[l][k] = v[t] ? __builtin_fmaf(w[t], val[t][l][k], acc[l][k]) : acc[l][k];
                        sumw = v[t] ? sumw + w[t] : sumw;
                    }
                }
                else
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                    {
                        if (!v[t]) continue;
#pragma unroll
                        for (int l = 0; l < ML; ++l)
                        {
                            if (l >= nl) break;
                            const int d = b.dims[l];
                            const float *src = F.in[l] + li[t] * d;
#pragma unroll
                            for (int k = 0; k < MD; ++k)
                                if (k < d) acc[l][k] = __builtin_fmaf(w[t], src[k], acc[l][k]);
                        }
                        sumw += w[t];
                    }
                valid = (sumw >= 0.01f);
                const float inv = 1.f / sumw;
#pragma unroll
                for (int l = 0; l < ML; ++l)
#pragma unroll
                    for (int k = 0; k < MD; ++k) acc[l][k] = valid ? acc[l][k] * inv : 0.f;
            }
            // a rounded position off the image has no valid neighbour either: nothing to look up
            fallback = !valid && ipx >= 1 && ipy >= 1 && ipx <= W - 1 && ipy <= H - 1;
            if (fallback)
                queue[atomicAdd(&queued, 1)] = RpQueued{ipx, ipy, (int)threadIdx.x, Z, fwZ, fwN, n.x, n.y, n.z};
        }
        if (!fallback)
        {
#pragma unroll
            for (int l = 0; l < ML; ++l)
            {
                if (l >= nl) break;
                const int d = FNL > 0 ? FD : b.dims[l];
                float *dst = F.out[l] + c * d;
#pragma unroll
                for (int k = 0; k < MD; ++k)
                    if (k < d) dst[k] = acc[l][k];
            }
            F.success[c] = valid ? 1 : 0;
        }
    }
    __syncthreads();
    const int nq = queued;
    int floats = FNL * FD;
    if (FNL == 0)
        for (int l = 0; l < nl; ++l) floats += b.dims[l];
    if (nq > rp_walk_above(floats))
    {
        if ((int)threadIdx.x >= nq) return;
        const RpQueued Q = queue[threadIdx.x];
        const float3 n = make_float3(Q.nx, Q.ny, Q.nz);
        float acc[ML][MD];
#pragma unroll
        for (int l = 0; l < ML; ++l)
#pragma unroll
            for (int k = 0; k < MD; ++k) acc[l][k] = 0.f;
        int nvalid = 0;
#pragma unroll 1
        for (int j = 0; j < 9; ++j)
        {
            const int qx = Q.ipx + j % 3 - 1, qy = Q.ipy + j / 3 - 1;
            if (qx >= W || qx < 0 || qy >= H || qy < 0) continue;
            const size_t qi = (size_t)qy * W + qx;
            if (!UNIT_OPAC && F.prevOpac[qi] == 0.f) continue;
            if (!reproj_valid(W, H, Q.ipx, Q.ipy, Q.Z, F.prevLinZ[3 * qi], Q.fwZ, n, ld3(F.prevNrm, qi), Q.fwN)) continue;
#pragma unroll
            for (int l = 0; l < ML; ++l)
            {
                if (l >= nl) break;
                const int d = FNL > 0 ? FD : b.dims[l];
                const float *src = F.in[l] + qi * d;
#pragma unroll
                for (int k = 0; k < MD; ++k)
                    if (k < d) acc[l][k] += src[k];
            }
            ++nvalid;
        }
        const float inv = nvalid > 0 ? 1.f / (float)nvalid : 0.f;
        const size_t c = (size_t)(by0 + Q.c / RP_TX) * W + bx0 + (Q.c & (RP_TX - 1));
#pragma unroll
        for (int l = 0; l < ML; ++l)
        {
            if (l >= nl) break;
            const int d = FNL > 0 ? FD : b.dims[l];
            float *dst = F.out[l] + c * d;
#pragma unroll
            for (int k = 0; k < MD; ++k)
                if (k < d) dst[k] = nvalid > 0 ? acc[l][k] * inv : 0.f;
        }
        F.success[c] = nvalid > 0 ? 1 : 0;
        return;
    }
    const int q = threadIdx.x / 9, nb = threadIdx.x - 9 * q;  // this lane's pixel of the round and neighbour
    for (int q0 = 0; q0 < nq; q0 += RP_ROUND)
    {
        if (q < RP_ROUND && q0 + q < nq)
        {
            const RpQueued Q = queue[q0 + q];
            const int qx = Q.ipx + nb % 3 - 1, qy = Q.ipy + nb / 3 - 1;
            bool ok = qx < W && qx >= 0 && qy < H && qy >= 0;
            const size_t qi = (size_t)min(max(qy, 0), H - 1) * W + min(max(qx, 0), W - 1);
            const float po = UNIT_OPAC ? 1.f : F.prevOpac[qi];
            const float pz = F.prevLinZ[3 * qi];
            const float3 pn = ld3(F.prevNrm, qi);
            ok = ok && po != 0.f &&
                 reproj_valid(W, H, Q.ipx, Q.ipy, Q.Z, pz, Q.fwZ, make_float3(Q.nx, Q.ny, Q.nz), pn, Q.fwN);
            pair_ok[threadIdx.x] = ok;
            if (ok)
#pragma unroll
                for (int l = 0; l < ML; ++l)
                {
                    if (l >= nl) break;
                    const int d = FNL > 0 ? FD : b.dims[l];
                    const float *src = F.in[l] + qi * d;
#pragma unroll
                    for (int k = 0; k < MD; ++k)
                        if (k < d) pair[threadIdx.x][l * MD + k] = src[k];
                }
        }
        __syncthreads();
        // one lane per (queued pixel, channel): the sum in neighbour order, over their count
        for (int i = threadIdx.x; i < RP_ROUND * ML * MD; i += 256)
        {
            const int qq = i / (ML * MD), ch = i - qq * (ML * MD), l = ch / MD, k = ch - l * MD;
            if (q0 + qq >= nq || l >= nl) continue;
            const int d = FNL > 0 ? FD : b.dims[l];
            int nvalid = 0;
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < 9; ++j)
                if (pair_ok[9 * qq + j])
                {
                    s += pair[9 * qq + j][ch];
                    ++nvalid;
                }
            const int t = queue[q0 + qq].c;
            const size_t c = (size_t)(by0 + t / RP_TX) * W + bx0 + (t & (RP_TX - 1));
            if (k < d) F.out[l][c * d + k] = nvalid > 0 ? s * (1.f / (float)nvalid) : 0.f;
        }
        // the masks, one lane per queued pixel (a list may be empty)
        if (threadIdx.x < RP_ROUND && q0 + (int)threadIdx.x < nq)
        {
            bool any = false;
#pragma unroll
            for (int j = 0; j < 9; ++j) any = any || pair_ok[9 * threadIdx.x + j];
            const int t = queue[q0 + threadIdx.x].c;
            F.success[(size_t)(by0 + t / RP_TX) * W + bx0 + (t & (RP_TX - 1))] = any ? 1 : 0;
        }
        __syncthreads();
    }
}

// Frames of one launch; three3: three buffers of three channels.
inline RpBatch rp_batch(int n, const RpFrame *fr, int n_list, const int *dims, bool &three3)
{
    RpBatch b{};
    int tx[XDN_MAX_FRAMES], ty[XDN_MAX_FRAMES];
    b.n_list = n_list;
    three3 = n_list == 3;
    for (int l = 0; l < n_list; ++l)
    {
        b.dims[l] = dims[l];
        three3 = three3 && dims[l] == 3;
    }
    for (int i = 0; i < n; ++i)
    {
        b.f[i] = fr[i];
        tx[i] = (fr[i].W + RP_TX - 1) / RP_TX;
        ty[i] = (fr[i].H + RP_TY - 1) / RP_TY;
    }
    b.map = make_tilemap(n, tx, ty);
    return b;
}

}  // namespace xdn
