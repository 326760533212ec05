// gfx950 kernels of the soft-shadow visibility path (one frame).
//
// Stage map (reference -> kernel):
//   sampleMaxZcal / triangleMaxZcal / sampleRectangleAABBcal /
//   verticesRectangleAABBcal + AABBReduce_kernel  -> k_reduce (one pass)
//   lightPlaneParamCal host part                 -> k_finalize
//   writeSampleAndBinPair + maxZpreBinReduce      -> k_rx_key
//   thrust::sort_by_key (receivers) + FindStart    -> k_scan + k_rx_scatter
//   triangleVertexSetup + countPairNumForPerTri    -> k_tri_count
//   exclusive_scan + writeTriBinPair + sort_by_key -> k_scan + k_tri_scatter
//   findTriangleStartEnd                           -> k_scan (block 0)
//   shadowCal_per_sample_kernel                    -> k_occlude
//
// Every kernel reads the frame status first, so the whole frame is one
// fixed launch sequence with no host round trip (graph-capturable).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>
#include "fd_device.h"
#include "fd_kernels.h"

using namespace fdk;

namespace {

constexpr int RED_BLOCK = 1024;
constexpr int RED_ITEMS = 2;           // receivers / vertices per thread in k_reduce
constexpr int SCAN_BLOCK = 1024;
constexpr int SCAN_ITEMS = 4;
constexpr int SCAN_CHUNK = SCAN_BLOCK * SCAN_ITEMS;
static_assert(SCAN_CHUNK % FD_TRB == 0, "a chunk of pair counts covers whole triangle blocks");

// Resets the frame state (by k_finalize's first thread: nothing reads the state
// before, and replays of a captured graph start from the same one).
__device__ __forceinline__ void init_state(FdState* s) {
    const uint32_t encMax = fenc(FD_F32_MAX), encNegMax = fenc(-FD_F32_MAX);
    s->rxZmaxAll = encNegMax;
    s->rxMin[0] = s->rxMin[1] = s->rxMin[2] = encMax;
    s->rxMaxA[0] = s->rxMaxA[1] = encNegMax;
    s->rxMaxZ = encNegMax;
    s->vxZmax = encNegMax;
    s->vxMin[0] = s->vxMin[1] = s->vxMin[2] = encMax;
    s->vxMaxA[0] = s->vxMaxA[1] = encNegMax;
    s->vxMaxZ = encNegMax;
    s->validRect = 0;
    s->status = FD_EXIT_OK;
    s->validSamples = 0;
    s->validTris = 0;
    s->keyOutOfRange = 0;
    s->capacityHit = 0;
    s->pairs = 0;
    s->rxTotal = 0;
    s->totalChunks = 0;
    s->triOrder = FD_TRI_ORDER_LIST;
}

// Resets the bin statistics (maxZ, minRange) and totals of this frame, dealt
// over k_reduce's blocks.
__device__ __forceinline__ void init_bins(const FdArgs& a, const int blk, const int blocks) {
    const int nb = 1 << (2 * a.gridLog2);
    const uint32_t encMax = fenc(FD_F32_MAX), encNegMax = fenc(-FD_F32_MAX);
    for (int b = blk * RED_BLOCK + threadIdx.x; b <= nb; b += blocks * RED_BLOCK) {
        a.rxTot[b] = 0;
        if (b == nb) break;
        a.triTot[b] = 0;
        a.binStat[5 * b + 0] = encNegMax;  // maxZ
        a.binStat[5 * b + 1] = encNegMax;  // max of rect min x
        a.binStat[5 * b + 2] = encNegMax;  // max of rect min y
        a.binStat[5 * b + 3] = encMax;     // min of rect max x
        a.binStat[5 * b + 4] = encMax;     // min of rect max y
    }
}

// Block-level reduction of NV uint32 values with op (0 = min, 1 = max,
// 2 = sum); the block's results go to part[k * P + blk] (no atomics: many
// blocks updating the few words of the frame state would serialise).
static_assert(RED_BLOCK / 64 == 16 && FD_FIN_THREADS / 64 == 16, "one 16-lane row holds a block's waves");
// op over a 16-lane row, in lane 15 of it (every lane of the row active)
__device__ __forceinline__ uint32_t row_reduce(uint32_t v, int op) {
    auto f = [&](uint32_t x) { v = op == 2 ? v + x : op ? max(v, x) : min(v, x); };
    const bool sum = op == 2;
    f((uint32_t)dpp_or<0x111, 0xf>(sum ? 0 : (int)v, (int)v));
    f((uint32_t)dpp_or<0x112, 0xf>(sum ? 0 : (int)v, (int)v));
    f((uint32_t)dpp_or<0x114, 0xf>(sum ? 0 : (int)v, (int)v));
    f((uint32_t)dpp_or<0x118, 0xf>(sum ? 0 : (int)v, (int)v));
    return v;
}
template <int NV>
__device__ void block_reduce_store(uint32_t (&v)[NV], const int (&op)[NV], uint32_t* part, int P, int blk) {
    __shared__ uint32_t sh[NV][RED_BLOCK / 64];
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const uint32_t r = op[k] == 2 ? (uint32_t)wave_sum_i32((int)v[k]) : op[k] ? wave_max_u32(v[k]) : wave_min_u32(v[k]);
        if (l == 0) sh[k][w] = r;
    }
    __syncthreads();
    // one 16-lane row per value: its waves' results
    if (threadIdx.x < NV * (RED_BLOCK / 64)) {
        const int k = threadIdx.x >> 4, j = threadIdx.x & 15;
        const uint32_t r = row_reduce(sh[k][j], op[k]);
        if (j == 15) part[(size_t)k * P + blk] = r;
    }
}

// --------------------------------------------------------------------------
// k_reduce: one pass over receivers (blocks [0, nbR)) and vertices (blocks
// [nbR, nbR + nbV)).  Receivers: z for the far plane
// (Step2_1_samplerRectangleAABB.inl:1-34), back-face test against the four
// light corners and the light-plane rectangle (:53-137).  1024 threads with two
// elements each: a thread's chain of loads is what small frames wait for (256
// threads with eight each: 7.8 us for 64 x 64 receivers, now 5.2).  The rectangle's max
// corner x' + F/z - S is reduced as max(x' + F/z) - S after the frame's S is
// known: rounding of (a - S) is monotone in a, so both give the same float.
// Vertices: Step2_2_modelRectangleAABB.inl:1-99.
// --------------------------------------------------------------------------
__device__ __forceinline__ void reduce_body(const FdArgs& a, const int blk) {
    const int nbR = a.nbR;
    const float* m = a.L.m;
    init_bins(a, blk, nbR + a.nbV);
    const uint32_t encMax = fenc(FD_F32_MAX), encNegMax = fenc(-FD_F32_MAX);
    if ((int)blk < nbR) {
        uint32_t v[7] = {encNegMax, encMax, encMax, encMax, encNegMax, encNegMax, encNegMax};
        int cnt = 0;
        const int base = blk * RED_BLOCK * RED_ITEMS + threadIdx.x;
#pragma unroll
        for (int it = 0; it < RED_ITEMS; ++it) {
            const int i = base + it * RED_BLOCK;
            if (i >= a.WH) break;
            const float4 p = a.pos[i];
            float4 out = make_float4(0.f, 0.f, 0.f, __uint_as_float(FD_TAG_NONE));
            if (!(p.x != p.x)) {
                const float z = getZ(m, p.x, p.y, p.z);
                if (!(z != z)) v[0] = max(v[0], fenc(z));
                const float4 n = a.nrm[i];
                const float* c[4] = {a.L.ur, a.L.ul, a.L.dl, a.L.dr};
                bool back = true;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    back = back && (dot3(c[k][0] - p.x, c[k][1] - p.y, c[k][2] - p.z, n.x, n.y, n.z) <= 0);
                if (back) {
                    out.w = __uint_as_float(FD_TAG_BACK);
                } else {
                    float rx, ry, rz;
                    makeRect(m, p.x, p.y, p.z, rx, ry, rz);
                    const float ax = rx + a.L.F[0] / rz;
                    const float ay = ry + a.L.F[1] / rz;
                    if (!(rx != rx)) v[1] = min(v[1], fenc(rx));
                    if (!(ry != ry)) v[2] = min(v[2], fenc(ry));
                    if (!(rz != rz)) { v[3] = min(v[3], fenc(rz)); v[6] = max(v[6], fenc(rz)); }
                    if (!(ax != ax)) v[4] = max(v[4], fenc(ax));
                    if (!(ay != ay)) v[5] = max(v[5], fenc(ay));
                    ++cnt;
                    out = make_float4(rx, ry, rz, __uint_as_float(FD_TAG_VALID));
                }
            }
            a.rec[i] = out;
        }
        uint32_t v8[8] = {v[0], v[1], v[2], v[3], v[4], v[5], v[6], (uint32_t)cnt};
        const int op[8] = {1, 0, 0, 0, 1, 1, 1, 2};
        block_reduce_store<8>(v8, op, a.part, nbR + a.nbV, blk);
    } else {
        uint32_t v[7] = {encNegMax, encMax, encMax, encMax, encNegMax, encNegMax, encNegMax};
        const int base = (blk - nbR) * RED_BLOCK * RED_ITEMS + threadIdx.x;
#pragma unroll
        for (int it = 0; it < RED_ITEMS; ++it) {
            const int vi = base + it * RED_BLOCK;
            if (vi >= a.nverts) break;
            const float* p = a.verts + (size_t)vi * a.vstride;
            const float px = p[0], py = p[1], pz = p[2];
            float rx, ry, rz;
            makeRect(m, px, py, pz, rx, ry, rz);
            const float ax = rx + a.L.F[0] / rz;
            const float ay = ry + a.L.F[1] / rz;
            if (!(rz != rz)) { v[0] = max(v[0], fenc(rz)); v[3] = min(v[3], fenc(rz)); v[6] = max(v[6], fenc(rz)); }
            if (!(rx != rx)) v[1] = min(v[1], fenc(rx));
            if (!(ry != ry)) v[2] = min(v[2], fenc(ry));
            if (!(ax != ax)) v[4] = max(v[4], fenc(ax));
            if (!(ay != ay)) v[5] = max(v[5], fenc(ay));
        }
        const int op[7] = {1, 0, 0, 0, 1, 1, 1};
        block_reduce_store<7>(v, op, a.part, nbR + a.nbV, blk);
    }
}

// --------------------------------------------------------------------------
// k_finalize: the host part of lightPlaneParamCal
// (Step2_3_defineFDbuffer.inl:5-111) on the device, with its early exits.
// Latency-bound: 16-lane rows reduce the waves' results (one thread that walked
// all 256 of them: 10.0 us, now 4.6).
// --------------------------------------------------------------------------
__device__ __forceinline__ void finalize_body(const FdArgs& a, const int blk) {
    if (blk != 0) return;
    FdState* s = a.st;
    {
        // the k_reduce block partials: receiver blocks [0, nbR), vertex
        // blocks [nbR, nbR + nbV); min/max of order-preserving encodings
        __shared__ uint32_t red[2][8][FD_FIN_THREADS / 64];
        const int nbR = a.nbR, P = a.nbR + a.nbV;
        const int op[8] = {1, 0, 0, 0, 1, 1, 1, 2};
        const uint32_t encMax = fenc(FD_F32_MAX), encNegMax = fenc(-FD_F32_MAX);
        uint32_t r[2][8];
#pragma unroll
        for (int k = 0; k < 8; ++k) r[0][k] = r[1][k] = op[k] == 2 ? 0u : op[k] ? encNegMax : encMax;
        for (int i = threadIdx.x; i < P; i += blockDim.x) {
            const int g = i < nbR ? 0 : 1;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (g == 1 && k == 7) continue;
                const uint32_t x = a.part[(size_t)k * P + i];
                r[g][k] = op[k] == 2 ? r[g][k] + x : op[k] ? max(r[g][k], x) : min(r[g][k], x);
            }
        }
        const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
        __shared__ uint32_t o[2][8];
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                uint32_t x = r[g][k];   // the start value where the wave has no partial
                if (w * 64 < P)
                    x = op[k] == 2 ? (uint32_t)wave_sum_i32((int)x) : op[k] ? wave_max_u32(x) : wave_min_u32(x);
                if (l == 0) red[g][k][w] = x;
            }
        __syncthreads();
        if (threadIdx.x < 256) {   // one 16-lane row per value
            const int g = threadIdx.x >> 7, k = (threadIdx.x >> 4) & 7, j = threadIdx.x & 15;
            const uint32_t x = row_reduce(red[g][k][j], k == 7 ? 2 : (k == 0 || k > 3) ? 1 : 0);
            if (j == 15) o[g][k] = x;
        }
        __syncthreads();
        if (threadIdx.x != 0) return;
        init_state(s);
        s->rxZmaxAll = o[0][0];
        s->rxMin[0] = o[0][1]; s->rxMin[1] = o[0][2]; s->rxMin[2] = o[0][3];
        s->rxMaxA[0] = o[0][4]; s->rxMaxA[1] = o[0][5];
        s->rxMaxZ = o[0][6];
        s->validRect = (int)o[0][7];
        s->vxZmax = o[1][0];
        s->vxMin[0] = o[1][1]; s->vxMin[1] = o[1][2]; s->vxMin[2] = o[1][3];
        s->vxMaxA[0] = o[1][4]; s->vxMaxA[1] = o[1][5];
        s->vxMaxZ = o[1][6];
    }
    // sampleMaxZcal / triangleMaxZcal: thrust::reduce(max) seeded with -1
    const float zs = fmax_(-1.0f, fdec(s->rxZmaxAll));
    const float zt = fmax_(-1.0f, fdec(s->vxZmax));
    s->sampleMaxZ = zs;
    s->triMaxZ = zt;
    if (zs < 0.0f) { s->status = FD_EXIT_SAMPLE_MAXZ; return; }
    if (zt < 0.0f) { s->status = FD_EXIT_TRI_MAXZ; return; }
    const float f = fmax_(zs, zt) + 0.1f;
    s->f = f;
    const float Sx = a.L.F[0] / f, Sy = a.L.F[1] / f;
    s->S[0] = Sx;
    s->S[1] = Sy;
    float sa[8] = {fdec(s->rxMin[0]), fdec(s->rxMin[1]), fdec(s->rxMin[2]), 0.0f,
                   fdec(s->rxMaxA[0]) - Sx, fdec(s->rxMaxA[1]) - Sy, fdec(s->rxMaxZ), 0.0f};
    float ma[8] = {fdec(s->vxMin[0]), fdec(s->vxMin[1]), fdec(s->vxMin[2]), 0.0f,
                   fdec(s->vxMaxA[0]) - Sx, fdec(s->vxMaxA[1]) - Sy, fdec(s->vxMaxZ), 0.0f};
    // the reductions started from +-FD_F32_MAX; (-MAX) - S rounds back to -MAX
    sa[4] = fmax_(sa[4], -FD_F32_MAX); sa[5] = fmax_(sa[5], -FD_F32_MAX);
    ma[4] = fmax_(ma[4], -FD_F32_MAX); ma[5] = fmax_(ma[5], -FD_F32_MAX);
    for (int k = 0; k < 8; ++k) { s->sAABB[k] = sa[k]; s->mAABB[k] = ma[k]; }
    if (s->validRect == 0) { s->status = FD_EXIT_NO_VALID_SAMPLE; return; }
    if (ma[0] > ma[4] || ma[1] > ma[5] || sa[0] > sa[4] || sa[1] > sa[5]) { s->status = FD_EXIT_EMPTY_AABB; return; }
    float B0 = fmax_(sa[0], ma[0]), B1 = fmax_(sa[1], ma[1]);
    float E0 = fmin_(sa[4], ma[4]), E1 = fmin_(sa[5], ma[5]);
    s->B[0] = B0; s->B[1] = B1; s->B[2] = ma[2];
    s->E[0] = E0; s->E[1] = E1; s->E[2] = sa[6];
    if (B0 >= E0 || B1 >= E1) { s->status = FD_EXIT_EMPTY_LP; return; }
    const int G = 1 << a.gridLog2;
    s->G = G;
    s->log2G = a.gridLog2;
    s->nb = G * G;
    s->factor[0] = (float)G / (E0 - B0);
    s->factor[1] = (float)G / (E1 - B1);
}

// --------------------------------------------------------------------------
// Receiver key (writeSampleAndBinPair, Step3_bindSampleToBin.inl:5-59) and
// the per-bin receiver statistics (maxZpreBinReduce_kernel, :61-104), which
// are min/max reductions and so are folded into the same pass with atomics.
// Each block owns RXB consecutive receivers, one per thread, and writes its key
// histogram (256 threads with four each: 15.8 us for 64 x 64 receivers, now 8.2).
// --------------------------------------------------------------------------
struct RxRect { float bx, by, ex, ey, z; };

__device__ __forceinline__ RxRect rx_rect(const float4 r, const FdState* s, const FdLight& L) {
    RxRect o;
    o.bx = r.x;
    o.by = r.y;
    o.ex = r.x + L.F[0] / r.z - s->S[0];
    o.ey = r.y + L.F[1] / r.z - s->S[1];
    o.z = r.z;
    return o;
}

// bin key of a valid receiver, or nb when outside the light plane
__device__ __forceinline__ int rx_key(const RxRect& q, const FdState* s, int nb, int log2G, bool& oor) {
    oor = false;
    const float B0 = s->B[0], B1 = s->B[1], E0 = s->E[0], E1 = s->E[1];
    if ((q.bx > q.ex || q.by > q.ey) || (q.bx < B0 || q.by < B1 || q.ex > E0 || q.ey > E1)) return nb;
    const float cx = (q.ex + q.bx) / 2.0f;
    const float cy = (q.ey + q.by) / 2.0f;
    const int bx = cvt_sat(floorf((cx - B0) * s->factor[0]));
    const int by = cvt_sat(floorf((cy - B1) * s->factor[1]));
    const int k = (int)(((unsigned)by << log2G) | (unsigned)bx);
    if (k < 0 || k >= nb) { oor = true; return nb; }
    return k;
}

// Receivers are traversed in pixel tiles of 64 (tile-major): TW x (64/TW)
// with TW = 1 << twl (8x8 by default), so that each 64-lane wave of the sort
// -- and later of the occlusion -- holds a compact tile rather than a
// 64-pixel strip.  The tile shape changes only the order of receivers within
// a bin, never a result.  Position p -> dense id, or -1 for padding outside
// the view.
__device__ __forceinline__ int tile_id(int p, int W, int H, int twl) {
    const int TW = 1 << twl;
    const int WT = (W + TW - 1) >> twl;
    const int t = p >> 6, j = p & 63;
    const int x = (t % WT) * TW + (j & (TW - 1));
    const int y = (t / WT) * (64 >> twl) + (j >> twl);
    return (x < W && y < H) ? y * W + x : -1;
}

__device__ __forceinline__ void rx_key_body(const FdArgs& a, const int blk) {
    extern __shared__ uint32_t hist[];  // nb + 1 counters, then (grids up to FD_LDS_BINS) 5 x nb bin statistics
    __shared__ uint32_t blkCount[2];    // valid receivers, keys out of range
    const FdState* s = a.st;
    if (s->status != FD_EXIT_OK) return;
    const int nb = s->nb, log2G = s->log2G;
    // bin statistics of the block in LDS, merged into the global ones once per
    // bin the block touched (else one set of global atomics per wave and key)
    const bool ldsStat = a.binLds && nb <= FD_LDS_BINS;
    uint32_t* bstat = hist + nb + 1;
    for (int k = threadIdx.x; k <= nb; k += blockDim.x) hist[k] = 0;
    if (ldsStat)
        for (int k = threadIdx.x; k < 5 * nb; k += blockDim.x) bstat[k] = (k % 5) < 3 ? 0u : 0xffffffffu;
    if (threadIdx.x < 2) blkCount[threadIdx.x] = 0;
    __syncthreads();
    int nvalid = 0, noor = 0;
    const int base = blk * FD_RXB;
    {
        const int p = base + threadIdx.x;
        const int i = p < a.npos ? tile_id(p, a.W, a.H, a.tileLog2) : -1;
        int key = nb;
        RxRect q{};
        const bool in = i >= 0;
        if (in) {
            const float4 r = a.rec[i];
            if (__float_as_uint(r.w) == FD_TAG_VALID) {
                q = rx_rect(r, s, a.L);
                bool oor;
                key = rx_key(q, s, nb, log2G, oor);
                if (key < nb || oor) ++nvalid;
                if (oor) ++noor;
            }
            a.rxKey[i] = (uint16_t)key;
        }
        // Segmented wave reduction: one pass per distinct key among the
        // wave's lanes (receivers of a wave are neighbours, so usually 1-3),
        // giving the key histogram and the per-bin receiver statistics with
        // one LDS add and five global atomics per (wave, key).
        const uint32_t v0 = (in && q.z == q.z) ? fenc(q.z) : 0u;
        const uint32_t v1 = (in && q.bx == q.bx) ? fenc(q.bx) : 0u;
        const uint32_t v2 = (in && q.by == q.by) ? fenc(q.by) : 0u;
        const uint32_t v3 = (in && q.ex == q.ex) ? fenc(q.ex) : 0xffffffffu;
        const uint32_t v4 = (in && q.ey == q.ey) ? fenc(q.ey) : 0xffffffffu;
        uint64_t pending = __ballot(in);
        while (pending) {
            const int lead = __ffsll((unsigned long long)pending) - 1;
            const int k0 = uniform(__shfl(key, lead, 64));
            const bool mine = in && key == k0;
            const uint64_t m = __ballot(mine);
            pending &= ~m;
            if (lane_id() == 0) atomicAdd(&hist[k0], (uint32_t)__popcll(m));
            if (k0 < nb) {
                const uint32_t r0 = wave_max_u32(mine ? v0 : 0u);
                const uint32_t r1 = wave_max_u32(mine ? v1 : 0u);
                const uint32_t r2 = wave_max_u32(mine ? v2 : 0u);
                const uint32_t r3 = wave_min_u32(mine ? v3 : 0xffffffffu);
                const uint32_t r4 = wave_min_u32(mine ? v4 : 0xffffffffu);
                if (lane_id() == 0) {
                    uint32_t* bs = (ldsStat ? bstat : a.binStat) + 5 * k0;
                    atomicMax(bs + 0, r0); atomicMax(bs + 1, r1); atomicMax(bs + 2, r2);
                    atomicMin(bs + 3, r3); atomicMin(bs + 4, r4);
                }
            }
        }
    }
    nvalid = wave_sum_i32(nvalid);
    noor = wave_sum_i32(noor);
    if (lane_id() == 0) {
        if (nvalid) atomicAdd(&blkCount[0], (uint32_t)nvalid);
        if (noor) atomicAdd(&blkCount[1], (uint32_t)noor);
    }
    __syncthreads();
    // valid receivers = binned ones (the scanned histogram) + out-of-range
    // keys, totalled in k_scan; only the rare out-of-range count is
    // accumulated here
    if (threadIdx.x == 0 && blkCount[1]) atomicAdd(&a.st->keyOutOfRange, (int)blkCount[1]);
    for (int k = threadIdx.x; k <= nb; k += blockDim.x) {
        const uint32_t h = hist[k];
        a.histR[(size_t)k * a.nblkR + blk] = h;
        if (h) atomicAdd(a.rxTot + k, h);
        if (ldsStat && k < nb && h) {
            const uint32_t* l = bstat + 5 * k;
            uint32_t* bs = a.binStat + 5 * k;
            atomicMax(bs + 0, l[0]); atomicMax(bs + 1, l[1]); atomicMax(bs + 2, l[2]);
            atomicMin(bs + 3, l[3]); atomicMin(bs + 4, l[4]);
        }
    }
}

// --------------------------------------------------------------------------
// Device-wide exclusive scans of uint32 counts (thrust::exclusive_scan / the
// offsets of a stable counting sort), one launch for all three of a frame:
// the blocks know what lies before them from sums that the counting passes
// leave behind (per bin, per triangle block), so no pass over the counts comes
// first.  Modulo 2^32; the number of pairs is totalled in 64 bits.
//
// Bound: latency.  Six launches (a pass of chunk sums and a pass of offsets
// for each array) of 4 to 8 us each before, and 9 us for the exits and tables;
// one of 7.5 us (64 x 64 receivers) to 10 us (1920 x 1080) now.
// --------------------------------------------------------------------------
// the frame got past k_finalize: receivers are binned (also where no triangle
// or no pair is found, or too many)
__device__ __forceinline__ bool binned(int status) {
    return status == FD_EXIT_OK || status == FD_EXIT_NO_VALID_TRI || status == FD_EXIT_NO_PAIRS ||
           status == FD_EXIT_CAPACITY;
}

// Exclusive prefix of v over the block's 1024 threads; total: over all of them.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t (&sh)[16], uint32_t& total) {
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t x = wave_incl_scan(v);
    __syncthreads();   // sh is free again
    if (l == 63) sh[w] = x;
    __syncthreads();
    uint32_t off = 0, all = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t t = sh[i];
        off += i < w ? t : 0u;
        all += t;
    }
    total = all;
    return off + x - v;
}

__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t (&sh)[16]) {
    const uint32_t x = (uint32_t)wave_sum_i32((int)v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = x;
    __syncthreads();
    uint32_t all = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) all += sh[i];
    return all;
}

// d[e0 .. e1), in place, by one block; base: the sum of what comes before
__device__ __forceinline__ void scan_range(uint32_t* __restrict__ d, long e0, long e1, uint32_t base, uint32_t (&sh)[16]) {
    for (long c = e0; c < e1; c += SCAN_CHUNK) {
        const long i0 = c + threadIdx.x * SCAN_ITEMS;
        uint32_t v[SCAN_ITEMS], sum = 0;
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k) v[k] = i0 + k < e1 ? d[i0 + k] : 0u;
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k) sum += v[k];
        uint32_t tot;
        uint32_t off = base + block_excl_scan(sum, sh, tot);
        base += tot;
#pragma unroll
        for (int k = 0; k < SCAN_ITEMS; ++k) {
            if (i0 + k < e1) d[i0 + k] = off;
            off += v[k];
        }
    }
}

// rows [r0, r1) of a histogram, nblk counts each; tot: the rows' sums
__device__ __forceinline__ void scan_rows(uint32_t* d, const uint32_t* __restrict__ tot, int r0, int r1, int nblk,
                                          uint32_t (&sh)[16]) {
    uint32_t pre = 0;
    for (int k = threadIdx.x; k < r0; k += SCAN_BLOCK) pre += tot[k];
    const uint32_t base = block_sum(pre, sh);
    scan_range(d, (long)r0 * nblk, (long)r1 * nblk, base, sh);
}

// --------------------------------------------------------------------------
// Stable receiver scatter: each of the block's 16 waves takes 64 of its
// receivers; lanes holding equal keys are matched with ballots over the key
// bits and ranked with mbcnt, and the counts of the waves before (16-bit, a row
// of 16 per key in LDS) place the wave within the block, so the result equals a
// stable sort_by_key (Step3_bindSampleToBin.inl:125-127).  Binned receivers
// also get their 32-byte occlusion record written in sorted order.
//
// Bound: latency for small views, then memory (134 MB at 1920 x 1080).  One
// wave that walked a block's receivers 64 at a time took 18 us for 64 x 64 and
// 27 us for 1920 x 1080 receivers; 16 waves take 4.5 and 21.6.
// --------------------------------------------------------------------------
__device__ __forceinline__ void rx_scatter_body(const FdArgs& a, const int blk) {
    extern __shared__ __align__(16) uint32_t rcnt[];  // (nb + 1) x 16 counts of 16 bits
    const FdState* s = a.st;
    if (!binned(s->status)) return;
    const int nb = s->nb;
    const int kbits = 2 * s->log2G + 1;   // keys 0 .. nb
    const int w = threadIdx.x >> 6;
    for (int k = threadIdx.x; k < (nb + 1) * 2; k += FD_RXB) ((uint4*)rcnt)[k] = make_uint4(0u, 0u, 0u, 0u);
    const int p = blk * FD_RXB + threadIdx.x;
    const int i = p < a.npos ? tile_id(p, a.W, a.H, a.tileLog2) : -1;
    const bool act = i >= 0;
    const int key = act ? (int)a.rxKey[i] : 0;
    const uint32_t base = act ? a.histR[(size_t)key * a.nblkR + blk] : 0u;
    float4 r = make_float4(0.f, 0.f, 0.f, 0.f), ps = r;
    if (act && key < nb) {
        r = a.rec[i];
        ps = a.pos[i];
    }
    uint64_t eq = __ballot(act);
    for (int b = 0; b < kbits; ++b) {
        const bool bit = (key >> b) & 1;
        const uint64_t bal = __ballot(act && bit);
        eq &= bit ? bal : ~bal;
    }
    const int rank = mbcnt(eq);
    __syncthreads();
    if (act && rank == 0) ((uint16_t*)rcnt)[16 * key + w] = (uint16_t)__popcll(eq);
    __syncthreads();
    if (!act) return;
    // counts of the waves before this one: two per word, at most 1024 in all
    uint32_t sum = 0;
    for (int j = 0; j < (w >> 1); ++j) sum += rcnt[8 * key + j];
    sum = (sum & 0xffffu) + (sum >> 16);
    if (w & 1) sum += rcnt[8 * key + (w >> 1)] & 0xffffu;
    const uint32_t d = base + sum + (uint32_t)rank;
    if (d >= (uint32_t)a.WH) return;
    a.sortedId[d] = i;
    if (key < nb) {
        const RxRect q = rx_rect(r, s, a.L);
        FdRxRec o;
        o.q[0] = ps.x; o.q[1] = ps.y; o.q[2] = ps.z;
        o.rminx = q.bx; o.rminy = q.by; o.rmaxx = q.ex; o.rmaxy = q.ey; o.z = q.z;
        a.sortedRec[d] = o;
    }
}

// --------------------------------------------------------------------------
// Triangle setup (triangleVertexSetup_kernel, Step0_triangleSetup.inl:56-191)
// fused with the pair count (countPairNumForPerTri_kernel,
// Step4_RasterizeTriangleToBin.inl:5-113).  The bin loop walks the union of
// the wave's bin rectangles with a wave-uniform bin index, so the bin
// statistics are scalar loads and the block histogram is updated once per
// (wave, bin).
// --------------------------------------------------------------------------
struct BinStat { float maxZ, mx, my, mz, mw; };

__device__ __forceinline__ BinStat load_bin(const uint32_t* bs) {
    BinStat b;
    b.maxZ = fdec(bs[0]); b.mx = fdec(bs[1]); b.my = fdec(bs[2]); b.mz = fdec(bs[3]); b.mw = fdec(bs[4]);
    return b;
}

// the bin test of the count pass (:94), on the LP-clamped AABB
__device__ __forceinline__ bool bin_test(const BinStat& b, float cbx, float cby, float cbz, float cex, float cey) {
    return b.maxZ >= cbz && cbx < b.mx && cby < b.my && b.mz < cex && b.mw < cey;
}

// Bin statistics staged in LDS by the pair passes (when the grid has at most
// FD_LDS_BINS bins): float4 (maxZ, mx, my, mz) and mw per bin, decoded once
// per block instead of five L2 loads per (triangle, bin) test.
__device__ __forceinline__ void stage_bins(const FdArgs& a, int nb, float4* q, float* w) {
    for (int k = threadIdx.x; k < nb; k += blockDim.x) {
        const uint32_t* bs = a.binStat + 5 * k;
        q[k] = make_float4(fdec(bs[0]), fdec(bs[1]), fdec(bs[2]), fdec(bs[3]));
        w[k] = fdec(bs[4]);
    }
}
__device__ __forceinline__ BinStat bin_at(const FdArgs& a, bool staged, const float4* q, const float* w, int bp) {
    if (staged) {
        const float4 v = q[bp];
        return BinStat{v.x, v.y, v.z, v.w, w[bp]};
    }
    return load_bin(a.binStat + 5 * bp);
}

struct TriClamp { float bx, by, bz, ex, ey; int sx, sy, ex_, ey_; bool ok; };

// the count pass's triangle rejection, LP clamp and bin range (:41-83)
__device__ __forceinline__ TriClamp tri_clamp(const float4 mn, const float4 mx, const FdState* s) {
    TriClamp c;
    const float B0 = s->B[0], B1 = s->B[1], E0 = s->E[0], E1 = s->E[1];
    c.ok = !(mn.x > mx.x || mn.y > mx.y || mn.z > mx.z || mn.x > E0 || mn.y > E1 || mx.x < B0 || mx.y < B1);
    c.bx = fmax_(mn.x, B0);
    c.by = fmax_(mn.y, B1);
    c.bz = mn.z;
    c.ex = fmin_(mx.x, E0);
    c.ey = fmin_(mx.y, E1);
    const float G = (float)s->G;
    c.sx = cvt_sat_u16(fmax_(floorf((c.bx - B0) * s->factor[0]), 0.0f));
    c.sy = cvt_sat_u16(fmax_(floorf((c.by - B1) * s->factor[1]), 0.0f));
    c.ex_ = cvt_sat_u16(fmin_(ceilf((c.ex - B0) * s->factor[0]), G));
    c.ey_ = cvt_sat_u16(fmin_(ceilf((c.ey - B1) * s->factor[1]), G));
    if (!c.ok) { c.sx = c.sy = 0; c.ex_ = c.ey_ = 0; }
    return c;
}

// Pair passes: a lane walks its own bin rectangle when it holds at most
// FD_BIG_AREA bins; larger rectangles (a triangle spanning much of the light
// plane) are walked by the whole wave, one rectangle at a time, so that one
// lane's long walk does not hold up its wave and block.
#define FD_BIG_AREA 64

// The bins of a wave-uniform rectangle [sx, ex) x [sy, ey), 64 per step:
// body(valid, i, j) on every lane.  Steps follow raster order and, within a
// step, lanes do too (rows of up to 64 bins share a step when narrower).
template <typename F>
__device__ __forceinline__ void walk_rect_wave(int sx, int sy, int ex, int ey, F&& body) {
    const int w = ex - sx;
    const int lane = lane_id();
    if (w <= 64) {
        int wl = 0;
        while ((1 << wl) < w) ++wl;
        const int rows = 64 >> wl;
        const int di = lane & ((1 << wl) - 1), dj = lane >> wl;
        for (int j0 = sy; j0 < ey; j0 += rows) body(di < w && j0 + dj < ey, sx + di, j0 + dj);
    } else {
        for (int j = sy; j < ey; ++j)
            for (int i0 = sx; i0 < ex; i0 += 64) body(i0 + lane < ex, i0 + lane, j);
    }
}

// Area class of a triangle projected on the light plane (its three
// makeRectangle points): 7 - floor(log2(area in bin cells)) clamped to
// [0, FD_TRI_CLASSES - 1]; 0 holds the largest triangles (128 cells and up,
// infinite areas too), the last class those under 1/128 of a cell and the
// degenerate ones (area zero or NaN).  The area is
// |(x1 - x0)(y2 - y0) - (y1 - y0)(x2 - x0)| / 2 in float, in that order.
__device__ __forceinline__ int area_class(const float (&px)[3], const float (&py)[3], const FdState* s) {
    const float twice = fabsf((px[1] - px[0]) * (py[2] - py[0]) - (py[1] - py[0]) * (px[2] - px[0]));
    const float cells = ((twice * 0.5f) * s->factor[0]) * s->factor[1];
    if (!(cells > 0.0f)) return FD_TRI_CLASSES - 1;
    const int e = (int)(__float_as_uint(cells) >> 23) - 127;   // floor(log2), -127 for denormals
    return min(max(7 - e, 0), FD_TRI_CLASSES - 1);
}

// Mesh order: the largest area class that comes last.  A class is
// 7 - floor(log2(area in bin cells)) and a bin cell is 1/4^log2G of the
// light plane, so 1/512 of the plane is class 16 - 2 log2G (8 at 16x16
// bins); classes up to it go last.
__device__ __forceinline__ int mesh_big_class(int log2G) { return 16 - 2 * log2G; }

// Walk key of an area class: the class itself (area order, big < 0), or
// for the mesh order the classes above big first (keys 0..14-big, larger
// triangles first) and the classes up to big last (one key, 15 - big).
__device__ __forceinline__ int walk_key(int cls, int big) {
    if (big < 0) return cls;
    return cls > big ? cls - big - 1 : FD_TRI_CLASSES - 1 - big;
}

__device__ __forceinline__ void tri_count_body(const FdArgs& a, const int blk) {
    // nb counters, then the staged bin statistics (float4 + float per bin);
    // 16-byte aligned behind the block's static counters, for the float4s
    extern __shared__ __align__(16) uint32_t thist[];
    __shared__ uint32_t blkStat, blkSum;   // valid | neighbours << 11 | overlaps << 21; pairs
    const FdState* s = a.st;
    if (s->status != FD_EXIT_OK) return;
    const int nb = s->nb, log2G = s->log2G;
    const bool staged = a.binLds && nb <= FD_LDS_BINS;
    float4* binQ = (float4*)(thist + nb);
    float* binW = (float*)(binQ + nb);
    for (int k = threadIdx.x; k < nb; k += blockDim.x) thist[k] = 0;
    if (threadIdx.x == 0) blkStat = blkSum = 0;
    if (staged) stage_bins(a, nb, binQ, binW);
    __syncthreads();
    const int t = blk * FD_TRB + threadIdx.x;
    const bool act = t < a.ntris;
    const float* m = a.L.m;
    float4 mn = make_float4(FD_F32_MAX, FD_F32_MAX, FD_F32_MAX, 1.0f);
    float4 mx = make_float4(-FD_F32_MAX, -FD_F32_MAX, -FD_F32_MAX, 1.0f);
    int valid = 0;
    if (act) {
        int i0 = a.idx[3 * t], i1 = a.idx[3 * t + 1], i2 = a.idx[3 * t + 2];
        // an index outside the vertex buffer makes the triangle unusable
        // (the reference reads out of bounds); it is treated as culled
        const bool badIdx = (unsigned)i0 >= (unsigned)a.nverts || (unsigned)i1 >= (unsigned)a.nverts ||
                            (unsigned)i2 >= (unsigned)a.nverts;
        if (badIdx) i0 = i1 = i2 = 0;
        const float* p0 = a.verts + (size_t)i0 * a.vstride;
        const float* p1 = a.verts + (size_t)i1 * a.vstride;
        const float* p2 = a.verts + (size_t)i2 * a.vstride;
        const float v0[3] = {p0[0], p0[1], p0[2]}, v1[3] = {p1[0], p1[1], p1[2]}, v2[3] = {p2[0], p2[1], p2[2]};
        // n = cross(v0 - v2, v1 - v0)   (:96-98)
        const float e0x = v1[0] - v0[0], e0y = v1[1] - v0[1], e0z = v1[2] - v0[2];
        const float e1x = v0[0] - v2[0], e1y = v0[1] - v2[1], e1z = v0[2] - v2[2];
        const float nx = e1y * e0z - e1z * e0y, ny = e1z * e0x - e1x * e0z, nz = e1x * e0y - e1y * e0x;
        bool culled = badIdx;
        if (a.cull && !badIdx) {
            const float* c[4] = {a.L.ur, a.L.ul, a.L.dr, a.L.dl};
            const float* vv[3] = {v0, v1, v2};
            culled = true;
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    culled = culled && (dot3(nx, ny, nz, c[k][0] - vv[j][0], c[k][1] - vv[j][1], c[k][2] - vv[j][2]) <= 0);
        }
        float px[3] = {0.0f, 0.0f, 0.0f}, py[3] = {0.0f, 0.0f, 0.0f};
        if (!culled) {
            const float* vv[3] = {v0, v1, v2};
#pragma unroll
            for (int k = 0; k < 3; ++k) {  // getTriAABB (:37-54)
                float rx, ry, rz;
                makeRect(m, vv[k][0], vv[k][1], vv[k][2], rx, ry, rz);
                px[k] = rx;
                py[k] = ry;
                mn.x = fmin_(mn.x, rx);
                mn.y = fmin_(mn.y, ry);
                mn.z = fmin_(mn.z, rz);
                mx.z = fmax_(mx.z, rz);
                mx.x = fmax_(mx.x, rx + a.L.F[0] / rz - s->S[0]);
                mx.y = fmax_(mx.y, ry + a.L.F[1] / rz - s->S[1]);
            }
            if (!(mn.x > s->E[0] || mn.y > s->E[1] || mx.x < s->B[0] || mx.y < s->B[1])) {
                valid = 1;
                FdTri d;
                for (int k = 0; k < 3; ++k) { d.v0[k] = v0[k]; d.v1[k] = v1[k]; d.v2[k] = v2[k]; }
                d.bminx = mn.x; d.bminy = mn.y; d.bmaxx = mx.x; d.bmaxy = mx.y;
                d.minz = mn.z; d.maxz = mx.z;
                // occlusion-side triangle constants, same expressions as
                // Step5_2_shadowCalPerSample.inl:130 and :7
                const float ax = v1[0] - v0[0], ay = v1[1] - v0[1], az = v1[2] - v0[2];
                const float bx = v2[0] - v1[0], by = v2[1] - v1[1], bz = v2[2] - v1[2];
                d.n[0] = ay * bz - az * by; d.n[1] = az * bx - ax * bz; d.n[2] = ax * by - ay * bx;
                for (int k = 0; k < 3; ++k) {
                    d.e01[k] = v0[k] - v1[k];
                    d.e12[k] = v1[k] - v2[k];
                    d.e20[k] = v2[k] - v0[k];
                }
                {   // light_window's edge term, e the largest edge (1-norm); 2^20 at most, or infinite
                    auto n1 = [](const float (&v)[3]) { return fabsf(v[0]) + fabsf(v[1]) + fabsf(v[2]); };
                    auto ni = [](const float (&v)[3]) { return fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fabsf(v[2])); };
                    const float e = fmaxf(fmaxf(n1(d.e01), n1(d.e12)), n1(d.e20));
                    const float rl = (float)a.L.res * (ni(a.L.xd) + ni(a.L.yd));
                    // 52u, 40u (u = 2^-24), 2^-60
                    d.we = fmaxf(fmaxf(3.0994415e-06f * e, 2.3841858e-06f * e * (e / rl)), 8.6736174e-19f);
                    if (!(d.we <= 1048576.0f)) d.we = INFINITY;
                }
                d.pad1[0] = d.pad1[1] = d.pad1[2] = d.pad1[3] = 0.0f;
                a.tri[t] = d;
            }
        }
        a.triAABB[2 * t] = mn;
        a.triAABB[2 * t + 1] = mx;
        a.triClass[t] = (uint8_t)(valid ? area_class(px, py, s) : FD_TRI_CLASSES - 1);
    }
    {
        const int nv = __popcll(__ballot(valid));
        // list coherence: how often a valid triangle's culling box overlaps
        // the next triangle's (the next lane's; the wave's last lane has none)
        const float nx0 = __shfl_down(mn.x, 1, 64), ny0 = __shfl_down(mn.y, 1, 64);
        const float nx1 = __shfl_down(mx.x, 1, 64), ny1 = __shfl_down(mx.y, 1, 64);
        const int nvld = __shfl_down(valid, 1, 64);
        const bool pair = valid && nvld && lane_id() < 63;
        const bool over = pair && mn.x <= nx1 && nx0 <= mx.x && mn.y <= ny1 && ny0 <= mx.y;
        const int np = __popcll(__ballot(pair)), no = __popcll(__ballot(over));
        if (lane_id() == 0 && nv) atomicAdd(&blkStat, (uint32_t)(nv | np << 11 | no << 21));
    }
    // count pass
    TriClamp c = tri_clamp(mn, mx, s);
    if (!act) { c.ok = false; c.sx = c.sy = c.ex_ = c.ey_ = 0; }
    int count = 0, tsx = 6000, tsy = 6000, tex = 0, tey = 0;
    const bool has = c.ok && c.sx < c.ex_ && c.sy < c.ey_;
    const bool big = has && (c.ex_ - c.sx) * (c.ey_ - c.sy) > FD_BIG_AREA;
    // small rectangles: every lane walks its own; per-block bin counts by
    // LDS atomics
    if (has && !big) {
        for (int j = c.sy; j < c.ey_; ++j)
            for (int i = c.sx; i < c.ex_; ++i) {
                const int bp = j << log2G | i;
                const BinStat b = bin_at(a, staged, binQ, binW, bp);
                if (bin_test(b, c.bx, c.by, c.bz, c.ex, c.ey)) {
                    ++count;
                    tsx = min(tsx, i); tsy = min(tsy, j);
                    tex = max(tex, i + 1); tey = max(tey, j + 1);
                    atomicAdd(&thist[bp], 1u);
                }
            }
    }
    // large rectangles: the wave walks them one by one
    for (uint64_t bigs = __ballot(big); bigs; bigs &= bigs - 1) {
        const int L = __ffsll((unsigned long long)bigs) - 1;
        const float bx = __shfl(c.bx, L, 64), by = __shfl(c.by, L, 64), bz = __shfl(c.bz, L, 64);
        const float ex = __shfl(c.ex, L, 64), ey = __shfl(c.ey, L, 64);
        const int sx = uniform(__shfl(c.sx, L, 64)), sy = uniform(__shfl(c.sy, L, 64));
        const int ex_ = uniform(__shfl(c.ex_, L, 64)), ey_ = uniform(__shfl(c.ey_, L, 64));
        int n = 0, mnx = 6000, mny = 6000, mxx = 0, mxy = 0;
        walk_rect_wave(sx, sy, ex_, ey_, [&](bool v, int i, int j) {
            const int bp = j << log2G | i;
            const bool pass = v && bin_test(bin_at(a, staged, binQ, binW, v ? bp : 0), bx, by, bz, ex, ey);
            if (pass) {
                atomicAdd(&thist[bp], 1u);
                mnx = min(mnx, i); mny = min(mny, j);
                mxx = max(mxx, i + 1); mxy = max(mxy, j + 1);
            }
            n += __popcll(__ballot(pass));
        });
        mnx = wave_min_i32(mnx); mny = wave_min_i32(mny);
        mxx = wave_max_i32(mxx); mxy = wave_max_i32(mxy);
        if (lane_id() == L) { count = n; tsx = mnx; tsy = mny; tex = mxx; tey = mxy; }
    }
    if (act) {
        a.triCount[t] = count;
        a.triOff[t] = (uint32_t)count;
        a.triRange[t] = make_uint2((uint32_t)tsx | ((uint32_t)tsy << 16), (uint32_t)tex | ((uint32_t)tey << 16));
    }
    const int sum = wave_sum_i32(count);
    if (lane_id() == 0 && sum) atomicAdd(&blkSum, (uint32_t)sum);
    __syncthreads();
    if (threadIdx.x == 0) {
        a.part[blk] = blkStat;
        a.part[a.nblkT + blk] = blkSum;
    }
    for (int k = threadIdx.x; k < nb; k += blockDim.x) {
        const uint32_t h = thist[k];
        a.histT[(size_t)k * a.nblkT + blk] = h;
        if (h) atomicAdd(a.triTot + k, h);
    }
}

// The large rectangles of the write pass, walked by the whole wave; a pair's
// place in its triangle's run is its rank among the passing bins in raster
// order, as in the per-lane walk.
__device__ __forceinline__ void tri_write_big(const FdArgs& a, int log2G, bool staged, const float4* binQ,
                                              const float* binW, bool big, int sx, int sy, int ex_, int ey_,
                                              const TriClamp& c, unsigned long long o0) {
    const unsigned long long cap = a.pairCap;
    for (uint64_t bigs = __ballot(big); bigs; bigs &= bigs - 1) {
        const int L = __ffsll((unsigned long long)bigs) - 1;
        const float bx = __shfl(c.bx, L, 64), by = __shfl(c.by, L, 64), bz = __shfl(c.bz, L, 64);
        const float ex = __shfl(c.ex, L, 64), ey = __shfl(c.ey, L, 64);
        const int rx0 = uniform(__shfl(sx, L, 64)), ry0 = uniform(__shfl(sy, L, 64));
        const int rx1 = uniform(__shfl(ex_, L, 64)), ry1 = uniform(__shfl(ey_, L, 64));
        unsigned long long o = __shfl(o0, L, 64);
        const uint32_t tag = (uint32_t)((threadIdx.x & ~63u) + (unsigned)L) << 16;
        walk_rect_wave(rx0, ry0, rx1, ry1, [&](bool v, int i, int j) {
            const int bp = j << log2G | i;
            const bool pass = v && bin_test(bin_at(a, staged, binQ, binW, v ? bp : 0), bx, by, bz, ex, ey);
            const uint64_t m = __ballot(pass);
            if (pass) {
                const unsigned long long d = o + (unsigned)mbcnt(m);
                if (d < cap) a.pairKT[d] = tag | (uint32_t)bp;
            }
            o += (unsigned)__popcll(m);
        });
    }
}

// Stable pair scatter (writeTriBinPair_kernel + sort_by_key,
// Step4_RasterizeTriangleToBin.inl:161-223): per bin, triangles ascending, one
// block of 1024 triangles at a time.
//
// First every triangle writes its (bin) pairs at its triangle-major offset
// (scanned pair counts), bins ascending within the triangle -- the order in
// which the reference's writeTriBinPair_kernel emits them (:161-204), with the
// count pass's test.  The block's pairs then are one stretch of that list, and
// its 16 waves sort equal slices of the stretch by bin: a pair of a bin means a
// triangle of its own, so a block has at most 1024 pairs of a bin and the 16
// per-wave counts of a bin fit 16-bit halves of LDS words (two waves per word,
// counted with 32-bit LDS adds).  After a barrier every bin's counts become
// exclusive prefixes over the waves, and each wave ranks its slice from base +
// prefix: lanes with equal bins are matched by ballots over the key bits and
// ranked with mbcnt, the last lane of a group advances the running offset.
// Result: bin-major, ascending triangle id within a bin.  LDS:
// FD_SCATTER_WIDE_LDS bytes per bin (bins <= 4096: grids up to 64 x 64), and
// before them the staged bin statistics.
//
// Bound: the ranking's chain of ballots, 64 pairs a step.  Slices of equal
// length keep the 16 waves alike: one slice per 64 triangles, in a launch of its
// own after the write, took 11 + 32 us for 512 x 512 receivers and 40 k
// triangles, and 29 + 69 us for 970 k; now 20 and 87 us.
__device__ __forceinline__ int wide_half(int w, int k, int nb) { return (((w >> 1) * nb + k) << 1) | (w & 1); }

__device__ __forceinline__ void tri_scatter_body(const FdArgs& a, const int blk) {
    extern __shared__ __align__(16) uint32_t wlds[];
    const FdState* s = a.st;
    if (s->status != FD_EXIT_OK) return;
    const int nb = s->nb, log2G = s->log2G;
    const bool staged = a.binLds && nb <= FD_LDS_BINS;
    float4* binQ = (float4*)wlds;
    float* binW = (float*)(binQ + nb);
    uint32_t* cnt32 = wlds + (staged ? nb * (FD_BIN_LDS_BYTES / 4) : 0);   // 8 * nb words
    uint16_t* cnt16 = (uint16_t*)cnt32;
    uint32_t* base = cnt32 + 8 * nb;                                       // nb block offsets
    if (staged) stage_bins(a, nb, binQ, binW);
    for (int k = threadIdx.x; k < 8 * nb; k += FD_TRB) cnt32[k] = 0u;
    for (int k = threadIdx.x; k < nb; k += FD_TRB) base[k] = a.histT[(size_t)k * a.nblkT + blk];
    const unsigned long long cap = a.pairCap;
    const int t0 = blk * FD_TRB;
    const int t = t0 + threadIdx.x;
    // the walk over the pair range (bins with pairs) of the count pass
    bool has = t < a.ntris;
    int sx = 0, sy = 0, ex = 0, ey = 0;
    TriClamp c{};
    unsigned long long o = 0;
    if (has) {
        const uint2 rg = a.triRange[t];
        const float4 mn = a.triAABB[2 * t], mx = a.triAABB[2 * t + 1];
        o = a.triOff[t];
        sx = rg.x & 0xffff; sy = rg.x >> 16; ex = rg.y & 0xffff; ey = rg.y >> 16;
        has = sx < ex && sy < ey;
        if (has) {
            c = tri_clamp(mn, mx, s);
            has = c.ok;
        }
    }
    __syncthreads();
    const bool big = has && (ex - sx) * (ey - sy) > FD_BIG_AREA;
    if (has && !big) {
        unsigned long long q = o;
        const uint32_t tag = (uint32_t)threadIdx.x << 16;
        for (int j = sy; j < ey; ++j)
            for (int i = sx; i < ex; ++i) {
                const int bp = j << log2G | i;
                if (bin_test(bin_at(a, staged, binQ, binW, bp), c.bx, c.by, c.bz, c.ex, c.ey)) {
                    if (q < cap) a.pairKT[q] = tag | (uint32_t)bp;
                    ++q;
                }
            }
    }
    tri_write_big(a, log2G, staged, binQ, binW, big, sx, sy, ex, ey, c, o);
    __syncthreads();   // the block's pairs are written
    // this wave's slice of them: whole steps of 64 pairs
    const int w = (int)(threadIdx.x >> 6);
    const unsigned long long b0 = a.triOff[t0];
    const unsigned long long b1 = t0 + FD_TRB < a.ntris ? (unsigned long long)a.triOff[t0 + FD_TRB] : s->pairs;
    const unsigned long long e1 = b1 < cap ? b1 : cap;
    const unsigned steps = b0 < e1 ? (unsigned)((e1 - b0 + 63) >> 6) : 0u;
    const unsigned per = (steps + 15) >> 4;
    const unsigned long long p0 = b0 + 64ull * per * w;
    const unsigned long long p1 = p0 + 64ull * per < e1 ? p0 + 64ull * per : e1;
    const uint32_t inc = (w & 1) ? 0x10000u : 1u;
#pragma unroll 4
    for (unsigned long long p = p0 + lane_id(); p < p1; p += 64)
        atomicAdd(&cnt32[(w >> 1) * nb + (int)(a.pairKT[p] & 0xffffu)], inc);
    __syncthreads();
    for (int k = threadIdx.x; k < nb; k += FD_TRB) {
        uint32_t run = 0;
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const uint32_t x = cnt32[v * nb + k], lo = x & 0xffffu;
            cnt32[v * nb + k] = run | (run + lo) << 16;
            run += lo + (x >> 16);
        }
    }
    __syncthreads();
    const int kbits = 2 * log2G;
    uint32_t nxt = p0 + lane_id() < p1 ? a.pairKT[p0 + lane_id()] : 0u;
    for (unsigned long long c0 = p0; c0 < p1; c0 += 64) {
        const unsigned long long p = c0 + lane_id();
        const bool act = p < p1;
        const uint32_t v = nxt;
        if (p + 64 < p1) nxt = a.pairKT[p + 64];
        const int key = (int)(v & 0xffffu);
        uint64_t eq = __ballot(act);
        for (int b = 0; b < kbits; ++b) {
            const bool bit = (key >> b) & 1;
            const uint64_t bal = __ballot(act && bit);
            eq &= bit ? bal : ~bal;
        }
        if (act) {
            const int rank = mbcnt(eq);
            const int gcount = __popcll(eq);
            const int h = wide_half(w, key, nb);
            const uint32_t r0 = cnt16[h];
            const unsigned long long dst = (unsigned long long)base[key] + r0 + (unsigned)rank;
            if (rank == gcount - 1) cnt16[h] = (uint16_t)(r0 + gcount);
            if (dst < cap) a.sortedTri[dst] = t0 + (int)(v >> 16);
        }
    }
}

// --------------------------------------------------------------------------
// Exit bookkeeping once the counts are known, the per-bin tables
// (FindStart_kernel, binRaster.inl:5-59) and the occlusion work list, by one
// block, from the bins' totals.
//
// Exits: setupTriangleVertex returns 1 when no triangle reached the light plane
// (Step0_triangleSetup.inl:224-225); FDLaunch skips the rest when there are no
// pairs (FD/api.cpp:522).
//
// Work list: one work item per 64 sorted receivers of a bin (the invalid key
// included, so every receiver's output is written exactly once).  Work items
// are issued bin by bin, longest triangle list first (by power-of-two class
// of the list length; the invalid key, with no list, last), so that the
// launch does not end on a few long-running waves.  The order only schedules
// work: every receiver's result is the same in any order.
// --------------------------------------------------------------------------
__device__ __forceinline__ void tables_body(const FdArgs& a, uint32_t (&sh)[16]) {
    __shared__ int classCount[33], classBase[33];
    __shared__ int waveCount[16][33];
    __shared__ uint16_t binAt[4097];     // per rank: the bin and its number of work items
    __shared__ uint32_t itemsAt[4097];
    FdState* s = a.st;
    const int nb = s->nb;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    // totals; the counting blocks' results (no count pass without triangles)
    unsigned long long pairs = 0;
    uint32_t nv = 0, np = 0, no = 0, rxIn = 0;
    for (int k = threadIdx.x; k < nb; k += SCAN_BLOCK) {
        pairs += a.triTot[k];
        rxIn += a.rxTot[k];
    }
    if (a.ntris > 0)
        for (int i = threadIdx.x; i < a.nblkT; i += SCAN_BLOCK) {
            const uint32_t x = a.part[i];
            nv += x & 0x7ffu;
            np += (x >> 11) & 0x3ffu;
            no += x >> 21;
        }
    nv = block_sum(nv, sh);
    np = block_sum(np, sh);
    no = block_sum(no, sh);
    rxIn = block_sum(rxIn, sh);
    // each bin has at most 2^31 pairs and a thread at most four bins
    const unsigned long long lo = block_sum((uint32_t)(pairs & 0xffffu), sh), mi = block_sum((uint32_t)(pairs >> 16) & 0xffffu, sh),
                             hi = block_sum((uint32_t)(pairs >> 32), sh);
    pairs = lo + (mi << 16) + (hi << 32);
    int status = FD_EXIT_OK;
    if (nv == 0) status = FD_EXIT_NO_VALID_TRI;
    else if (pairs == 0) status = FD_EXIT_NO_PAIRS;
    else if (pairs > a.pairCap || pairs >= 0x7fffffffull) status = FD_EXIT_CAPACITY;
    if (threadIdx.x == 0) {
        s->pairs = pairs;
        s->rxTotal = (unsigned long long)rxIn + a.rxTot[nb];
        s->validTris = (int)nv;
        // walk order of the bins' lists.  A triangle soup (neighbouring
        // triangles mostly apart): largest projected triangles first, big
        // occluders fill receivers early.  A connected mesh: the mesh order,
        // largest first except those covering 1/512 of the light plane or more,
        // which come last in list order (mostly triangles near the light; first,
        // they would scatter each object's triangles, which a receiver often
        // needs together) -- unless the lists are long (many objects overlap:
        // a receiver fills from whichever object comes first in the list, so
        // the list order, which keeps every object together, wins)
        const bool mesh = 2 * no >= np;
        const bool dense = pairs > (unsigned long long)FD_MESH_MAX_LIST16 * 256ull;
        s->triOrder = a.triOrder != FD_TRI_ORDER_AUTO ? a.triOrder
                      : !mesh ? FD_TRI_ORDER_AREA : dense ? FD_TRI_ORDER_LIST : FD_TRI_ORDER_MESH;
        // valid receivers: binned (keys < nb) plus keys out of range
        s->validSamples = (int)rxIn + s->keyOutOfRange;
        if (status == FD_EXIT_CAPACITY) s->capacityHit = 1;
        s->status = status;
    }
    // the receivers' start / end table exists once they are sorted: FDLaunch
    // binds the samples before it pairs the triangles (FD/api.cpp:505-522),
    // so a frame that ends without pairs (or over the pair arena) has it too
    if (status == FD_EXIT_NO_VALID_TRI) return;
    if (threadIdx.x < 33) classCount[threadIdx.x] = 0;
    __syncthreads();
    // the cost class of every bin (0 = longest lists): 31 - floor(log2(len + 1))
    for (int k = threadIdx.x; k <= nb; k += SCAN_BLOCK)
        atomicAdd(&classCount[k < nb ? __clz((int)a.triTot[k] + 1) : 32], 1);
    __syncthreads();
    if (w == 0) {
        const int c = lane < 33 ? classCount[lane] : 0;
        const int x = (int)wave_incl_scan((uint32_t)c);
        if (lane < 33) classBase[lane] = x - c;
    }
    __syncthreads();
    // stable within a class (ascending bin index, so that neighbouring bins,
    // which share triangles, stay close in the issue order): ranks from wave
    // ballots, then a prefix over the waves of each 1024-bin slice
    uint32_t rxCarry = 0, triCarry = 0;
    for (int k0 = 0; k0 <= nb; k0 += SCAN_BLOCK) {
        const int k = k0 + threadIdx.x;
        const bool in = k <= nb;
        const uint32_t rx = in ? a.rxTot[k] : 0u, tr = k < nb ? a.triTot[k] : 0u;
        uint32_t rxAll, trAll;
        const uint32_t rs = rxCarry + block_excl_scan(rx, sh, rxAll), ts = triCarry + block_excl_scan(tr, sh, trAll);
        rxCarry += rxAll;
        triCarry += trAll;
        if (in) {
            a.rxStart[k] = (int)rs;
            if (k == nb) a.rxStart[nb + 1] = a.WH;
            if (status == FD_EXIT_OK) {
                a.triStart[k] = (int)ts;   // triStart[nb]: the number of pairs
            }
        }
        if (status != FD_EXIT_OK) continue;
        const int cls = !in ? 0 : (k < nb) ? __clz((int)tr + 1) : 32;
        for (int i = lane; i < 33; i += 64) waveCount[w][i] = 0;
        int rankInWave = 0;
        for (uint64_t pending = __ballot(in); pending;) {
            const int lead = __ffsll((unsigned long long)pending) - 1;
            const int c = __shfl(cls, lead, 64);
            const uint64_t m = __ballot(in && cls == c);
            if (in && cls == c) rankInWave = mbcnt(m);
            if (lane == lead) waveCount[w][c] = __popcll(m);
            pending &= ~m;
        }
        __syncthreads();
        if (threadIdx.x < 33) {   // per class: exclusive prefix over the waves, then advance the class base
            int run = classBase[threadIdx.x];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int c = waveCount[j][threadIdx.x];
                waveCount[j][threadIdx.x] = run;
                run += c;
            }
            classBase[threadIdx.x] = run;
        }
        __syncthreads();
        if (in) {
            const int r = waveCount[w][cls] + rankInWave;
            binAt[r] = (uint16_t)k;
            itemsAt[r] = ((k == nb ? (uint32_t)a.WH - rs : rx) + 63) >> 6;
        }
        __syncthreads();
    }
    if (status != FD_EXIT_OK) return;
    // work-item prefix in rank order
    uint32_t carry = 0;
    for (int k0 = 0; k0 <= nb; k0 += SCAN_BLOCK) {
        const int r = k0 + threadIdx.x;
        uint32_t all;
        const uint32_t off = carry + block_excl_scan(r <= nb ? itemsAt[r] : 0u, sh, all);
        if (r <= nb) a.chunkStart[binAt[r]] = (int)off;
        carry += all;
    }
    if (threadIdx.x == 0) s->totalChunks = (int)carry;
}

// All that follows from the counts in one launch: block 0 the exits and tables,
// the others the scans of the receiver histogram, the pair histogram and the
// triangles' pair counts.  Nothing here depends on the status that block 0 sets.
__device__ __forceinline__ void scan_body(const FdArgs& a, int blk) {
    __shared__ uint32_t sh[16];
    const FdState* s = a.st;
    if (!binned(s->status)) return;
    if (blk == 0) {
        tables_body(a, sh);
        return;
    }
    --blk;
    const int nb = 1 << (2 * a.gridLog2);
    const int rr = fd_scan_rows(a.nblkR), nr = (nb + rr) / rr;   // rows per block; blocks of nb + 1 rows
    if (blk < nr) {
        scan_rows(a.histR, a.rxTot, blk * rr, min((blk + 1) * rr, nb + 1), a.nblkR, sh);
        return;
    }
    blk -= nr;
    const int rt = fd_scan_rows(a.nblkT), nt = (nb + rt - 1) / rt;
    if (blk < nt) {
        scan_rows(a.histT, a.triTot, blk * rt, min((blk + 1) * rt, nb), a.nblkT, sh);
        return;
    }
    blk -= nt;
    uint32_t pre = 0;
    for (int i = threadIdx.x; i < blk * (SCAN_CHUNK / FD_TRB); i += SCAN_BLOCK) pre += a.part[a.nblkT + i];
    const uint32_t base = block_sum(pre, sh);
    scan_range(a.triOff, (long)blk * SCAN_CHUNK, min((long)(blk + 1) * SCAN_CHUNK, (long)a.ntris), base, sh);
}

// Split lists only: zeroes the mask output before the occlusion merges into
// it (by blocks of k_tri_order, which waits for nothing of theirs; no memset, so
// that the sequence stays graph-capturable).  A launch of its own took 2.9 us.
constexpr int ZERO_WORDS = 4096;   // words per block
__device__ __forceinline__ void zero_masks_body(const FdArgs& a, const int blk) {
    const size_t n = (size_t)a.WH * a.L.res * a.L.wpr;
    const size_t base = (size_t)blk * ZERO_WORDS;
    for (int k = threadIdx.x; k < ZERO_WORDS; k += blockDim.x)
        if (base + k < n) a.masks[base + k] = 0u;
}

// Area order of one bin's triangle list (frames whose walk order is
// FD_TRI_ORDER_AREA): a stable counting sort of triStart..triEnd of the
// reference-order list by the triangles' area classes, into the same range
// of pairKT (free once the pairs are scattered).  One block of
// FD_ORDER_THREADS per bin.  A lane finds the lanes of its wave with its own key from one ballot per key
// bit (the AND of the matching ballots), its rank within them by mbcnt; the
// first such lane adds their number.  Pass 1 totals the keys (and keeps
// them in LDS for lists of up to FD_ORDER_CACHE entries), pass 2 ranks every
// entry and offsets it by an exclusive prefix over the waves of each slice.
__device__ __forceinline__ void tri_order_body(const FdArgs& a, const int bin) {
    constexpr int NWV = FD_ORDER_THREADS / 64, K = FD_TRI_CLASSES;
    __shared__ int waveCount[NWV][K];
    __shared__ int keyBase[K];
    __shared__ uint8_t keyCache[FD_ORDER_CACHE];
    const int nb = 1 << (2 * a.gridLog2);
    if (bin > nb) {
        zero_masks_body(a, bin - nb - 1);
        return;
    }
    const FdState* s = a.st;
    if (s->status != FD_EXIT_OK) return;
    const int ts = bin < s->nb ? a.triStart[bin] : 0, te = bin < s->nb ? a.triEnd[bin] : 0;
    {   // the bin's work items: one record each, so that the occlusion finds its own in one load
        const int c0 = a.chunkStart[bin], rs = a.rxStart[bin], re = a.rxEnd[bin];
        for (int i = threadIdx.x; rs + 64 * i < re; i += FD_ORDER_THREADS)
            a.chunks[c0 + i] = FdChunk{rs + 64 * i, min(64, re - rs - 64 * i) | bin << 8, ts, te};
    }
    if (s->triOrder == FD_TRI_ORDER_LIST || te <= ts) return;
    const int lane = lane_id(), w = threadIdx.x >> 6;
    int* out = (int*)a.pairKT;
    const int big = s->triOrder == FD_TRI_ORDER_MESH ? mesh_big_class(s->log2G) : -1;
    auto key_of = [&](int i, int& tri) -> int {
        tri = a.sortedTri[i];
        const int cls = ((unsigned)tri < (unsigned)a.ntris) ? (int)a.triClass[tri] : K - 1;
        return walk_key(cls, big);
    };
    // lanes of the wave with the same key (key K: no entry)
    auto same_key = [](int key) -> uint64_t {
        uint64_t m = ~0ull;
#pragma unroll
        for (int j = 0; j < FD_WALK_KEY_BITS; ++j) {
            const uint64_t b = __ballot((key >> j) & 1);
            m &= ((key >> j) & 1) ? b : ~b;
        }
        return m;
    };
    for (int k = threadIdx.x; k < K; k += FD_ORDER_THREADS) keyBase[k] = 0;
    __syncthreads();
    const bool cached = te - ts <= FD_ORDER_CACHE;
    // pass 1: key totals
    for (int i0 = ts; i0 < te; i0 += FD_ORDER_THREADS) {
        const int i = i0 + threadIdx.x;
        int tri = 0;
        const int key = i < te ? key_of(i, tri) : K;
        if (cached && i < te) keyCache[i - ts] = (uint8_t)key;
        const uint64_t m = same_key(key);
        if (key < K && mbcnt(m) == 0) atomicAdd(&keyBase[key], __popcll(m));
    }
    __syncthreads();
    if (threadIdx.x == 0) {   // exclusive prefix over the keys
        int run = 0;
        for (int k = 0; k < K; ++k) {
            const int x = keyBase[k];
            keyBase[k] = run;
            run += x;
        }
    }
    __syncthreads();
    // pass 2: stable scatter, one slice of FD_ORDER_THREADS entries at a time
    for (int i0 = ts; i0 < te; i0 += FD_ORDER_THREADS) {
        const int i = i0 + threadIdx.x;
        int tri = 0, key = K;
        if (i < te) {
            if (cached) {
                tri = a.sortedTri[i];
                key = keyCache[i - ts];
            } else {
                key = key_of(i, tri);
            }
        }
        for (int k = lane; k < K; k += 64) waveCount[w][k] = 0;
        const uint64_t m = same_key(key);
        const int rank = mbcnt(m);
        if (key < K && rank == 0) waveCount[w][key] = __popcll(m);
        __syncthreads();
        for (int k = threadIdx.x; k < K; k += FD_ORDER_THREADS) {   // per key: prefix over the waves
            int run = keyBase[k];
            for (int j = 0; j < NWV; ++j) {
                const int x = waveCount[j][k];
                waveCount[j][k] = run;
                run += x;
            }
            keyBase[k] = run;
        }
        __syncthreads();
        if (key < K) out[ts + waveCount[w][key] + rank] = tri;
        __syncthreads();
    }
}

// --------------------------------------------------------------------------
// Occlusion (shadowCal_per_sample_kernel, Step5_2_shadowCalPerSample.inl:37-234).
// A work item is 64 sorted receivers of one bin, one receiver per lane, run
// by several waves that take interleaved triangles of the bin's list.  Each
// wave walks its triangles with a wave-uniform index, so triangle records
// arrive through scalar loads; the receivers' light rows live in LDS
// (row-major by row, lane-minor: conflict-free), shared by the waves.
// --------------------------------------------------------------------------
template <typename T>
struct Bits;
template <>
struct Bits<uint32_t> {
    static constexpr int width = 32;
    __device__ static int ctz(uint32_t v) { return __builtin_ctz(v); }
    __device__ static int last(uint32_t v) { return 31 - __builtin_clz(v); }
    __device__ static int popc(uint32_t v) { return __popc(v); }
};
template <>
struct Bits<uint64_t> {
    static constexpr int width = 64;
    __device__ static int ctz(uint64_t v) { return __builtin_ctzll(v); }
    __device__ static int last(uint64_t v) { return 63 - __builtin_clzll(v); }
    __device__ static int popc(uint64_t v) { return __popcll(v); }
};

// getRowMaskForPlaneDiscriminant (:14-33): the mask of light samples along
// one row (or of rows) whose plane value D + B*c is non-negative, as
//   f1 = D >= 0, f2 = B*n + D >= 0;  f1 == f2 -> all / none,
//   else k = (int)ceil(-1*D/B), mask = (1 << k) - 1, complemented if !f1.
// Only min(k, R) is observable once the mask is clipped to the R-sample
// grid, and k outside [0, width) (shift to zero, then -1) is all ones, so k
// is reduced to kk in [0, R] with every out-of-grid value mapped to R.
//
// The division is the hot operation.  q' = -D * rcp(B) (v_rcp_f32, 1 ulp)
// is within |q| * 2^-22 of the correctly rounded quotient q, i.e. within
// 2e-5 for q <= 80.  Whenever q' is at least 2^-12 away from every integer,
// ceil(q') == ceil(q); q' >= R + 1 implies q > R.  Only the remaining cases
// (near an integer, near zero, negative, or |B| outside [2^-100, 2^100])
// take the IEEE division.
__device__ __forceinline__ int k_exact(float D, float B, int R) {
    const float c = ceilf(-1.0f * D / B);
    if (c != c) return 0;                       // cvt.rzi of NaN
    if (c < 0.0f || c > (float)R) return R;     // shift out of range / beyond the grid
    return (int)c;
}

// One edge plane A*row + B*col + C over the R x R sample grid, negated when
// the receiver sees the triangle's back (see the set-up in occlude_body).
struct Edge {
    float A, B, C;
    float nRowN;      // -(A * (R-1)):  f2 of the row-range mask is DN >= nRowN
    float nColN;      // -(B * (R-1)):  f2 of a row mask is D >= nColN
    float rA, rB;     // rcp(A), rcp(B); NaN when |A| / |B| is outside [2^-100, 2^100]
};

__device__ __forceinline__ bool rcp_ok(float x) {
    const float ax = fabsf(x);
    return ax >= 7.8886091e-31f && ax <= 1.2676506e+30f;
}
__device__ __forceinline__ float rcp_or_nan(float x) {
    return rcp_ok(x) ? __builtin_amdgcn_rcpf(x) : __builtin_nanf("");
}

// kk for one (D, divisor) in the division branch; sets slow when the exact
// quotient is needed.  With |divisor| in [2^-100, 2^100] the reciprocal
// quotient q is within 2e-5 of the exact one for q <= R + 1, and the exact
// quotient is >= 0 in this branch, so q > -2e-5: anything within 2^-12 of an
// integer (0 included) goes to the exact path.  q > R + 1 means all columns.
// A NaN reciprocal (divisor out of range) makes q NaN: always exact.
__device__ __forceinline__ int k_fast(float D, float r, float Rf, bool& slow) {
    const float q = (-D) * r;
    const float dist = fabsf(q - rintf(q));
    const bool fine = dist > 2.44140625e-4f || q > Rf + 1.0f;
    slow = !fine;
    return (int)__builtin_amdgcn_fmed3f(ceilf(q), 0.0f, Rf);   // NaN -> 0, then in [0, R]
}

template <typename T>
__device__ __forceinline__ T low_mask(int kk) {
    return (kk >= Bits<T>::width) ? ~(T)0 : (((T)1 << kk) - (T)1);
}

// AND of the three edge masks at plane offsets D[k] (row masks: divisor B,
// row-range masks: divisor A).  Each edge mask is all (f1 && f2), none
// (!f1 && !f2), a prefix [0, kk) (f1 && !f2) or a suffix [kk, R) (!f1 && f2);
// with v = (f1 != f2) ? kk : R the AND is the interval
// [max over !f1 edges of v, min over f1 edges of v).
// General form: valid for every input, including infinite limits B*(R-1).
template <typename T, bool ROWS>
__device__ __forceinline__ T three_edges(const Edge (&e)[3], const float (&D)[3], float Rf, int R) {
    bool f1[3], f2[3], slow[3];
    int kk[3];
    bool anySlow = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        f1[k] = D[k] >= 0.0f;
        f2[k] = (D[k] - (ROWS ? e[k].nRowN : e[k].nColN)) >= 0.0f;   // fl(B*n + D) >= 0
        kk[k] = k_fast(D[k], ROWS ? e[k].rA : e[k].rB, Rf, slow[k]);
        slow[k] = slow[k] && (f1[k] != f2[k]);
        anySlow |= slow[k];
    }
    if (anySlow) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (slow[k]) kk[k] = k_exact(D[k], ROWS ? e[k].A : e[k].B, R);
    }
    int v[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) v[k] = (f1[k] != f2[k]) ? kk[k] : R;
    const int hi = min(min(f1[0] ? v[0] : R, f1[1] ? v[1] : R), f1[2] ? v[2] : R);
    const int lo = max(max(f1[0] ? 0 : v[0], f1[1] ? 0 : v[1]), f1[2] ? 0 : v[2]);
    return low_mask<T>(hi) & ~low_mask<T>(lo);
}

// Bits [lo, lo + w) of a width-bit word, w + lo <= width.
template <typename T>
__device__ __forceinline__ T interval_bits(unsigned w, unsigned lo) {
    if (Bits<T>::width == 32) {
        unsigned m;
        asm("v_bfm_b32 %0, %1, %2" : "=v"(m) : "v"(w), "v"(lo));   // ((1 << w[4:0]) - 1) << lo[4:0]
        return (w >= 32u) ? ~(T)0 : (T)m;
    }
    return (w >= 64u) ? ~(T)0 : (T)((((uint64_t)1 << w) - 1ull) << (lo & 63u));
}

// Integer max3 / min3 as single instructions (kept opaque so that the
// selects feeding them are not folded into longer select chains).
__device__ __forceinline__ int max3i(int a, int b, int c) {
    int r;
    asm("v_max3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ int min3i(int a, int b, int c) {
    int r;
    asm("v_min3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Fast form of three_edges for limits nN = -(divisor * (R-1)) that are finite
// in every lane of the wave (the caller checks |A|, |B| <= 2^100).
//  * f2: for finite a and b, fl(a + b) >= 0 exactly when a + b >= 0 (a sum
//    of two floats is 0 or at least one denormal step away from it), so
//    fl(B*n + D) >= 0  <=>  D >= -fl(B*n)  -- also for infinite D.
//  * kk: only read when f1 != f2.  Then the exact quotient q lies in
//    [0, n + ulp] (f1 && !f2: D >= 0 > B; !f1 && f2: D < 0 < B, both with
//    |D| <= |B*n|).  X = D * rcp(B) + R is within |q| 2^-22 + 2^-19 < 2^-15
//    of Y = R - q.  The kernel forms x = fma(D, rcp(B), R + 2^-12) (Rs is
//    R + 2^-12, exact), which rounds X + 2^-12 by at most 2^-18.  When
//    fract(x) >= 2^-11, with k = floor(x):  X lies in
//    [k + 2^-12 - 2^-18, k + 1 - 2^-12 + 2^-18), so Y lies strictly inside
//    (k, k + 1) and kk = ceil(q) = R - floor(Y) = R - k, in [1, R-1] (no
//    clamp).  The lanes left (fract below 2^-11, or NaN from a NaN
//    reciprocal) divide exactly.
//  * with c = R - kk the AND is [R - min over suffix edges of c,
//    R - max over prefix edges of c), "none" edges giving the empty set.
template <typename T>
__device__ __forceinline__ T three_edges_fast(const float (&D)[3], const float (&nN)[3], const float (&r)[3],
                                              const float (&div)[3], float Rs, int R) {
    bool f1[3], f2[3], slow[3];
    int c[3];
    bool anySlow = false;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        f1[k] = D[k] >= 0.0f;
        f2[k] = D[k] >= nN[k];
        const float x = __builtin_fmaf(D[k], r[k], Rs);
        asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(c[k]) : "v"(x));   // floor(x), saturating, NaN -> 0
        slow[k] = !(__builtin_amdgcn_fractf(x) >= 4.8828125e-4f) && (f1[k] != f2[k]);
        anySlow |= slow[k];
    }
    if (anySlow) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (slow[k]) c[k] = R - k_exact(D[k], div[k], R);
    }
    const int hiC = max3i((f1[0] && !f2[0]) ? c[0] : 0, (f1[1] && !f2[1]) ? c[1] : 0, (f1[2] && !f2[2]) ? c[2] : 0);
    const int loC = min3i((!f1[0] && f2[0]) ? c[0] : R, (!f1[1] && f2[1]) ? c[1] : R, (!f1[2] && f2[2]) ? c[2] : R);
    const bool none = (!f1[0] && !f2[0]) || (!f1[1] && !f2[1]) || (!f1[2] && !f2[2]);
    const unsigned w = __builtin_elementwise_sub_sat((unsigned)loC, (unsigned)hiC);
    const T m = interval_bits<T>(w, (unsigned)(R - loC));
    return none ? (T)0 : m;
}

// Rows whose three-edge mask can be non-empty.  The reference visits every
// row of the row-range mask (each edge on its own); most of those rows end
// with an empty AND because a prefix edge (B < 0) and a suffix edge (B > 0)
// exclude each other.  Skipping a row whose AND is empty changes no output,
// so the window below only has to contain every row with a non-empty AND.
//
// Bound.  For a row r and column c in [0, R-1], a set bit of one edge's mask
// implies A r + B c + C >= -tau with tau = 4u (|A| R + |B| R + |C|)
// (u = 2^-24: the rounding of A*r, of + C, of the quotient and of B*(R-1);
// the set bit means c < q (prefix), c >= q (suffix) or both end columns
// pass).  The code uses one tau' = 2^-20 (2 M R + Mc) + 2^-126 for the three
// edges (M = max |A|, |B|; Mc = max |C|) and C' = fl(C + tau').
// A prefix edge m and a suffix edge p meet in some real column only if
//   |B_m| (A_p r + C'_p) + B_p (A_m r + C'_m) >= 0,
// which for a pair (i, j) of opposite-signed B is  s G(r) >= 0  with
// G(r) = (B_i A_j - B_j A_i) r + (B_i C'_j - B_j C'_i) = al r + be, s = sign(B_i).
// al and be are computed in float; their rounding is at most 3u (Sa R + Sb)
// (Sa, Sb: sums of the absolute products, Sa <= 2 M^2, Sb <= 2 M Mc'), and
// E = 2^-19 M (M R + Mc') + 2^-126 bounds it, so every row with a non-empty
// mask has  s (al r + be) + E >= 0, i.e.
//   r >= t0 - E/|al|  (s al > 0)   or   r <= t0 + E/|al|  (s al < 0),  t0 = -be/al.
// t0 and E/|al| come from v_rcp_f32 (2^-22 relative); a margin of 2^-10
// covers that while |t0| <= 2^11, and a pair is used only when
// E/|al| <= 2^10, so that beyond |t0| = 2^11 the window is far outside
// [0, R-1] either way.  The bounds t0 -/+ (E/|al| + 2^-10) are formed with
// one fma each (t0 - m = -(be * ra + m), t0 + m = -be * ra + m), which only
// rounds less than a product followed by a sum.  E is raised to at least
// 2^-30 (a larger E only widens the window), so m <= 2^10 also keeps
// |ra| <= 2^40, i.e. |al| >= 2^-40: al is a normal number, and a zero or
// denormal al (infinite or huge reciprocal) is never used.  Lanes with any
// |A|, |B|, |C| above 2^40 (where the products could overflow) are not
// used; every bound that is used is then finite.
template <typename T>
__device__ __forceinline__ T row_window(const Edge (&e)[3], float Rf, float mAB) {
    const float u20 = 9.5367431640625e-07f;   // 2^-20
    const float tiny = 1.17549435e-38f;       // 2^-126
    const float lim = 1.09951163e+12f;        // 2^40
    // mAB = max |A|, |B| (NaN-free maximum); a NaN coefficient makes the
    // lane's pair terms NaN, which fail the |al| test and are not used
    const float mC = fmaxf(fmaxf(fabsf(e[0].C), fabsf(e[1].C)), fabsf(e[2].C));
    const bool ok = fmaxf(mAB, mC) <= lim;
    const float tau = __builtin_fmaf(__builtin_fmaf(mAB, 2.0f * Rf, mC), u20, tiny);
    const float Cp[3] = {e[0].C + tau, e[1].C + tau, e[2].C + tau};
    const float E = fmaxf(__builtin_fmaf(__builtin_fmaf(mAB, Rf, mC + tau), mAB * 1.9073486328125e-06f, tiny),
                          9.31322575e-10f);   // >= 2^-30
    bool pos[3], neg[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) { pos[k] = e[k].B > 0.0f; neg[k] = e[k].B < 0.0f; }
    float lo[3], hi[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = k, j = (k + 1) % 3;
        const float pA = e[i].B * e[j].A, qA = e[j].B * e[i].A;
        const float pB = e[i].B * Cp[j], qB = e[j].B * Cp[i];
        const float al = pA - qA, be = pB - qB;
        const float ra = __builtin_amdgcn_rcpf(al);
        const float m = __builtin_fmaf(E, fabsf(ra), 9.765625e-4f);   // E/|al| + 2^-10
        const bool opp = (pos[i] && neg[j]) || (neg[i] && pos[j]);
        const bool use = ok && opp && m <= 1024.0f;
        const bool lower = pos[i] == (al > 0.0f);
        lo[k] = (use && lower) ? -__builtin_fmaf(be, ra, m) : 0.0f;
        hi[k] = (use && !lower) ? __builtin_fmaf(-be, ra, m) : Rf - 1.0f;
    }
    const float l = __builtin_amdgcn_fmed3f(fmaxf(fmaxf(lo[0], lo[1]), lo[2]), 0.0f, Rf);
    const float h = __builtin_amdgcn_fmed3f(fminf(fminf(hi[0], hi[1]), hi[2]), -1.0f, Rf - 1.0f);
    int nlc, hc;   // -ceil(l) = floor(-l), floor(h)
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(nlc) : "v"(-l));
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(hc) : "v"(h));
    const unsigned w = (unsigned)max(hc + 1 + nlc, 0);
    return interval_bits<T>(w, (unsigned)(-nlc));
}

// The light samples that one triangle can occlude from one receiver, bounded
// by projecting the triangle's three vertices from the receiver Q onto the
// light's sample grid -- before (and mostly instead of) the edge planes.
//
// With a_j = v_j - Q, N the light plane's normal, l = L0 - Q, h = l.N > 0 the
// light's height over Q and X, Y dual to the sample steps (xd.X = 1,
// yd.X = N.X = 0), vertex j projects to row r_j = (a_j.X) h / (a_j.N) - l.X
// and column c_j likewise with Y.
//
// Bound.  A set bit (r, c) has every edge value >= -tau in the float
// coefficients (tau = 4u (|A| R + |B| R + |C|), row_window above), whose own
// rounding is at most 8u |a|_1 |e|_1 (|l|_inf + R |xd|_inf + R |yd|_inf),
// u = 2^-24 (a, e: the largest vertex offset and triangle edge); so every
// exact edge value is >= -T with T = 12.5u a e Ld,
// Ld = |l|_1 + (R + 1) (|xd|_1 + |yd|_1) (2nd-order terms included).  The
// edge values of a sample P are |V| times the coordinates alpha_j of P - Q in
// the basis a_0, a_1, a_2 (V = det(a_0, a_1, a_2) = a_0.n), and the weights
// w_j = alpha_j (a_j.N) / h sum to 1 with r = sum w_j r_j.  For a_j.N > 0:
// w_j >= -eta, eta = wmax T / |V|, wmax = max a_j.N / h, so
//   min r_j - 2 eta (max r_j - min r_j) <= r <= max r_j + 2 eta (max - min).
// With d_j = projected vertex - Q, |a_j| = (a_j.N / h) |d_j| and |d_j|_1 <=
// t = Ld + |r_j|max |xd|_1 + |c_j|max |yd|_1 give a <= wmax t.  The record
// holds we >= max(52u e, 40u e^2 / (R (|xd|_inf + |yd|_inf))), so
//   q = we Ld t max(wmax, 1) >= 4 T  and  m = wmax q / |V| >= 4 wmax T / |V|
// (float V).
// m < 2 keeps the float V at 20u a e^2 or more (the second term of we), its
// rounding at 9u a e^2: the reference's sign of it is the exact one, the
// exact |V| at least half of it, and m >= 2 eta.  The projections are off by less
// than 64u t (1 + t / h) |X|_inf rows (axial lights: 11u (|r| + |l.X|), with
// |l.X| <= 2^12 under 2^-8), which with a constant makes the rest of the
// margin (vertices beyond |r| = 512 are off by a larger amount, but outside
// the grid by far more).  Vertices at or below Q,
// projections beyond 2^21 and NaN leave the window unknown: the caller then
// uses the exact row range and row_window.  (we <= 2^20, or infinite, and
// Ld t <= 2^40 keep the planes of the others finite, |A|, |B| < 2^78; q is at
// least 2^-100, which keeps underflow out of T.)  q is also at least
// 52u (|A| R + |B| R + |C|) of every edge.
//
// What bounds it: the VALU.  add, mul, fma and the bit operations on vector
// registers or literals issue at twice the rate of everything else (compares,
// selects, min/max, conversions, shifts, and any operation with a scalar
// register operand: 2.4 against 4.2 cycles per wave and SIMD measured), so
// rounding to integers goes through the addition of 1.5 * 2^23 and the tests
// are sign bits of integer differences, combined by and / or.
struct LightProj {   // uniform
    float kL, kr, kc;   // Ld^2, Ld |xd|_1, Ld |yd|_1 for the work item's largest Ld; infinite: no window
    float er, ec, iL;   // 64u |X|_inf, 64u |Y|_inf, 1 / Ld (lights that are not axial)
};

constexpr float WIN_MAGIC = 12582912.0f;       // 1.5 * 2^23: x + WIN_MAGIC holds the nearest integer of x in its low bits
constexpr int WIN_BASE = 0x4b400000;           // its bits: the integer is bits - WIN_BASE
constexpr float WIN_MARGIN = 0.0078125f;       // 2^-7 rows / columns
constexpr float WIN_MAX_OFFSET = 4096.0f;      // largest |l.X|, |l.Y| of axial lights (2^12)

// a: vertices in the light's frame (axial lights: the world's; else X, Y, N);
// h: light height; hr, hc: rows / columns per unit of a.x, a.y at that height;
// nr, nc: -l.X - 1/2, -l.Y - 1/2.  Returns whether a sample may be set: the
// rows are lo - WIN_BASE .. hi - WIN_BASE where known < 0, else unknown.
template <bool AXIAL>
__device__ __forceinline__ bool light_window(const LightProj& P, const float (&a)[3][3], float h, float hr, float hc,
                                             float nr, float nc, float V, float we, int nsubBits, int& lo, int& hi,
                                             int& known, float& q) {
    float r[3], c[3], ra[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        ra[j] = __builtin_amdgcn_rcpf(a[j][2]);
        r[j] = __builtin_fmaf(a[j][0] * ra[j], hr, nr);
        c[j] = __builtin_fmaf(a[j][1] * ra[j], hc, nc);
    }
    const float rwmin = fminf(fminf(ra[0], ra[1]), ra[2]) * h;   // 1 / wmax
    const float rmin = fminf(fminf(r[0], r[1]), r[2]), rmax = fmaxf(fmaxf(r[0], r[1]), r[2]);
    const float cmin = fminf(fminf(c[0], c[1]), c[2]), cmax = fmaxf(fmaxf(c[0], c[1]), c[2]);
    const float rs = fabsf(rmin) + fabsf(rmax), cs = fabsf(cmin) + fabsf(cmax);
    const float t = __builtin_fmaf(rs, P.kr, __builtin_fmaf(cs, P.kc, P.kL));   // Ld t
    const float den = fabsf(V) * rwmin;
    const float m = (we * t) * __builtin_amdgcn_rcpf(den * fminf(rwmin, 1.0f));
    q = m * den;
    float mr = WIN_MARGIN, mc = WIN_MARGIN;
    if (!AXIAL) {
        const float tt = t * P.iL;
        const float e = __builtin_fmaf(tt * __builtin_amdgcn_rcpf(h), tt, tt);
        mr = __builtin_fmaf(e, P.er, mr);
        mc = __builtin_fmaf(e, P.ec, mc);
    }
    mr = __builtin_fmaf(m, rmax - rmin, mr);
    mc = __builtin_fmaf(m, cmax - cmin, mc);
    // nearest integers of (bound - 1/2) + 1 and (bound - 1/2): the ceiling of
    // the lower, the floor of the upper bound
    lo = __float_as_int((rmin - mr) + (WIN_MAGIC + 1.0f));
    hi = __float_as_int((rmax + mr) + WIN_MAGIC);
    const int clo = __float_as_int((cmin - mc) + (WIN_MAGIC + 1.0f));
    const int chi = __float_as_int((cmax + mc) + WIN_MAGIC);
    // negative: no row or no column of the grid
    const int none = (hi - lo) | (hi - WIN_BASE) | (nsubBits - lo) | (chi - clo) | (chi - WIN_BASE) | (nsubBits - clo);
    // negative: m < 2 (a NaN is not, of either sign), rs + cs < 2^21, rwmin > 0
    known = ((__float_as_int(m) & 0x7fffffff) - 0x40000000) & (__float_as_int(rs + cs) - 0x4a000000) &
            __float_as_int(0.0f - rwmin);
    return (none & known) >= 0;
}

// The same for all receivers of a work item at once, one triangle per lane
// (the block prefilter): bounds of the rows and columns over the receivers'
// box.  In the light's frame relative to L0 (rows, columns, height; the
// light plane at height 0), the line from Q through v meets the light at
// row v.x + (v.x - Q.x) k, k = -v.z / (v.z - Q.z), so each vertex gives an
// interval over the box, and V = det / |xd x yd|^-1 is linear in Q.  The
// frame's coordinates, dz and k are off by at most 2^-18 S (1 + |k|)(1 + S / dz)
// of a row (times |X|_inf), S = the largest 1-norm of a vertex or receiver
// relative to L0.  m <= 1/2 here: V is 80u a e^2 or more and off by 29u a e^2
// (the frame's rounding adds 20u), so |V| is at least half of it.
struct TileBounds {
    float x0, x1, y0, y1, z0, z1;   // receivers in the light's frame relative to L0
    float iz;                       // 1 / -z1: the inverse of the least light height
};
struct TileBox {   // uniform
    TileBounds all;
    // without the receivers in the upper half of the heights, where these
    // spread: for triangles behind all of those (minz > zs), which the depth
    // cull then leaves out
    TileBounds low;
    float zs;
    float Ld, tr, tc;               // the largest Ld; |xd|_1, |yd|_1
    float sx, sy;                   // |X|_inf, |Y|_inf
    float A;                        // |xd x yd|
    float eps;                      // the frame's "Q on the triangle" bound of |V|
};

struct TileWindow {
    int lo, hi, clo, chi;   // rows and columns that bound every sample the triangle can set (clipped to the grid; lo > hi: none)
    bool known;             // else they are the whole grid
    // For every receiver of the work item, light_window would know its window,
    // |V| is above eps and has the sign of `side`; tol and mr are at least its
    // q / 16 and row margin.
    bool lanes;
    float side, tol, mr;
};

// v: vertices in the frame relative to L0, S0: their largest 1-norm in the
// world.
template <bool AXIAL>
__device__ __forceinline__ TileWindow tile_window(const TileBox& b, const TileBounds& r, const float (&v)[3][3], float S0, float we, int n) {
    TileWindow w;
    float rmin = 3.0e38f, rmax = -3.0e38f, cmin = 3.0e38f, cmax = -3.0e38f, kk = 0.0f, idz = 0.0f, g = 1.0f;   // g >= wmax, 1
    bool ok = true;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const float x = v[j][0], y = v[j][1], z = v[j][2];
        const float dz1 = z - r.z1, i1 = __builtin_amdgcn_rcpf(dz1);
        const float k0 = -z * __builtin_amdgcn_rcpf(z - r.z0), k1 = -z * i1;
        ok = ok && dz1 > 0.0f;
        const float dx0 = x - r.x1, dx1 = x - r.x0, dy0 = y - r.y1, dy1 = y - r.y0;
        const float xa = dx0 * k0, xb = dx0 * k1, xc = dx1 * k0, xd = dx1 * k1;
        const float ya = dy0 * k0, yb = dy0 * k1, yc = dy1 * k0, yd = dy1 * k1;
        rmin = fminf(rmin, x + fminf(fminf(xa, xb), fminf(xc, xd)));
        rmax = fmaxf(rmax, x + fmaxf(fmaxf(xa, xb), fmaxf(xc, xd)));
        cmin = fminf(cmin, y + fminf(fminf(ya, yb), fminf(yc, yd)));
        cmax = fmaxf(cmax, y + fmaxf(fmaxf(ya, yb), fmaxf(yc, yd)));
        kk = fmaxf(kk, fabsf(k1));
        g = fmaxf(g, (z - r.z0) * r.iz);
        idz = fmaxf(idz, i1);
    }
    const float e1[3] = {v[1][0] - v[0][0], v[1][1] - v[0][1], v[1][2] - v[0][2]};
    const float e2[3] = {v[2][0] - v[1][0], v[2][1] - v[1][1], v[2][2] - v[1][2]};
    const float n0 = e1[1] * e2[2] - e1[2] * e2[1], n1 = e1[2] * e2[0] - e1[0] * e2[2], n2 = e1[0] * e2[1] - e1[1] * e2[0];
    const float Vc = dot3(v[0][0] - 0.5f * (r.x0 + r.x1), v[0][1] - 0.5f * (r.y0 + r.y1), v[0][2] - 0.5f * (r.z0 + r.z1),
                          n0, n1, n2);
    const float Vh = dot3(0.5f * (r.x1 - r.x0), 0.5f * (r.y1 - r.y0), 0.5f * (r.z1 - r.z0), fabsf(n0), fabsf(n1), fabsf(n2));
    const float V = (fabsf(Vc) - Vh) * b.A;
    const float S = fmaxf(S0, b.Ld);
    const float rs = fabsf(rmin) + fabsf(rmax), cs = fabsf(cmin) + fabsf(cmax);
    const float t = b.Ld + rs * b.tr + cs * b.tc;
    const float q = we * b.Ld * t * g;
    const float m = q * g * __builtin_amdgcn_rcpf(V);
    const float E = 3.814697265625e-06f * S * (1.0f + kk) * (1.0f + S * idz), Ex = E * b.sx, Ey = E * b.sy;
    const float mr = m * (rmax - rmin) + (Ex + WIN_MARGIN), mc = m * (cmax - cmin) + (Ey + WIN_MARGIN);
    w.known = ok && V > 0.0f && m <= 0.5f && mr <= 4194304.0f && mc <= 4194304.0f;
    const float nf = (float)n;
    w.lo = (int)__builtin_amdgcn_fmed3f(ceilf(rmin - mr), 0.0f, nf + 1.0f);
    w.hi = (int)__builtin_amdgcn_fmed3f(floorf(rmax + mr), -1.0f, nf);
    w.clo = (int)__builtin_amdgcn_fmed3f(ceilf(cmin - mc), 0.0f, nf + 1.0f);
    w.chi = (int)__builtin_amdgcn_fmed3f(floorf(cmax + mc), -1.0f, nf);
    if (!w.known) { w.lo = w.clo = 0; w.hi = w.chi = n; }
    // no receiver's own t exceeds t by a hundredth (their rows and columns are
    // within Ex, Ey of these bounds); dz is far from 0 against its rounding;
    // |V| is at least half the V here
    w.lanes = w.known && 512.0f * (Ex * b.tr + Ey * b.tc) <= b.Ld && S * idz <= 65536.0f && rs + cs <= 1048576.0f &&
              0.5f * V > b.eps;
    w.side = Vc;
    w.tol = q * 0.0625f;
    // light_window's margin: its m and spread are below these
    w.mr = m * (rmax - rmin + 2.0f * Ex) + WIN_MARGIN;
    if (!AXIAL) w.mr += 3.814697265625e-06f * b.sx * (t + t * t * r.iz);
    return w;
}

// Which rows still lack samples of some receiver, per strip of columns: U[s]
// has bit r set when row r is not full in the columns [s << lsw, (s + 1) <<
// lsw) of every receiver of the work item.  Lane r ands the receivers' words
// of row r (FD_ROW_STRIDE keeps the lanes on different banks); the other waves
// may add bits meanwhile, which only makes the answer older.
template <typename T>
__device__ __forceinline__ void row_occupancy(const uint32_t* lds, int R, int lsw, T FULL, uint64_t (&U)[FD_OCC_STRIPS]) {
    const int lane = lane_id();
    T a = ~(T)0;
    if constexpr (Bits<T>::width == 32) {   // half the receivers per half wave
        const int r = min(lane & 31, R - 1);
        const uint32_t* p = lds + r * FD_ROW_STRIDE + (lane & 32);
        uint32_t x = ~0u;
#pragma unroll 8
        for (int l = 0; l < 32; ++l) x &= p[l];
        x &= (uint32_t)__shfl_xor((int)x, 32, 64);
        a = (T)x;
    } else {
        const int r = min(lane, R - 1);
        const uint32_t* p = lds + r * FD_ROW_STRIDE;
        const uint32_t* p1 = p + R * FD_ROW_STRIDE;
        uint32_t x = ~0u, y = ~0u;
#pragma unroll 8
        for (int l = 0; l < 64; ++l) {
            x &= p[l];
            y &= p1[l];
        }
        a = (T)(((uint64_t)y << 32) | x);
    }
    a = ~a & FULL;
    const uint64_t rows = R >= 64 ? ~0ull : (1ull << R) - 1ull;
    const T strip = (T)(((T)1 << (1 << lsw)) - (T)1);
#pragma unroll
    for (int s = 0; s < FD_OCC_STRIPS; ++s)
        U[s] = (s << lsw) < R ? __ballot((a & (T)(strip << (s << lsw))) != (T)0) & rows : 0ull;
}

// One row of a pair with finite planes without a division, where that decides
// it.  G = the least of the edges' largest values along the row,
// D + max(B (R-1), 0).  G < -tol: the mask is empty.  G > tol: the
// row is in the reference's row-range mask (its roundings
// and G's stay below 8u (|A| R + |B| R + |C|)) and every edge passes at its far end, so the
// edge's mask is the half line c >= -D/B (B > 0) or c < -D/B (B < 0)
// clipped to the grid; x = R - 1/2 + D rcp(B) rounds to
// R - ceil(-D/B) unless x is within 2^-15 of a tie (rcp, the fma and
// the reference's quotient are off by at most 2^-17 + 2^-19 + 2^-19
// while 0 <= -D/B <= R <= 64).  Edges
// of the other sign stand in with x = 0 (upper limits) and x = R
// (lower limits), the grid's own ends; planes through one vertex
// fan cannot all have one sign of B but by rounding, which goes the
// exact way, as do ties and |G| <= tol.  A zero B gives an infinite
// reciprocal: no limit, as every column then has the sign of G.
struct RowEdges {
    float rh[3], rl[3], Kh[3], Kl[3], bp[3];
    int tolBits;
};
// tolB: the bits of a tol >= 3u (|A| R + |B| R + |C|)
__device__ __forceinline__ RowEdges row_edges(const Edge (&e)[3], float Rf, float nsub, const int tolB) {
    RowEdges w;
    const int Rm = __float_as_int(Rf - 0.5f), RmR = Rm ^ __float_as_int(Rf);
    int sAnd = -1, sOr = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        int sB = __float_as_int(e[k].B) >> 31;
        asm("" : "+v"(sB));   // as a mask: selects run at half the rate
        const int rB = __float_as_int(__builtin_amdgcn_rcpf(e[k].B)), bn = __float_as_int(e[k].B * nsub);
        w.rh[k] = __int_as_float(rB & sB);
        w.rl[k] = __int_as_float(rB ^ (rB & sB));
        w.Kh[k] = __int_as_float(Rm & sB);
        w.Kl[k] = __int_as_float(Rm ^ (RmR & sB));
        w.bp[k] = __int_as_float(bn ^ (bn & sB));
        sAnd &= sB;
        sOr |= sB;
    }
    w.tolBits = tolB | ((sAnd | ~sOr) & 0x7f800000);
    return w;
}
// The rows where every edge is non-negative somewhere along the row: what is left
// of the projected rows of a triangle that reaches past the grid's columns (a
// diagonal sliver, a wall, any triangle larger than the light), where the window
// alone holds every row between its vertices.  A set bit has A r + B c + C >= -tau
// for every edge, tau = 4u (|A| R + |B| R + |C|), so A r + D >= 0 with D = C +
// max(B (R-1), 0) + 4 tol (13u at least: tau and the roundings of D); the bound
// -D/A is off by 2^-22 of itself, less than WIN_MARGIN up to 2^11 rows, and beyond
// the grid on its side past that.  A zero A gives an infinite bound (no limit, or
// no row) or, with D = 0, a NaN, which limits nothing.
// 30 instructions against 42 a row: taken where some lane's rows span more than
// FD_RANGE_ROWS.  1920 x 1080 receivers: 60 k slivers, 64 x 64 samples 24612 /
// 11588 us, tessellated boxes and ground of the receivers' own scene, 32 x 32,
// 1692 / 797; rows that span 4 or more (12): heightfield-1k 2348 (2249) against
// 2264 us, slivers with 16 x 16 samples 4126 (4666) against 4242.
template <typename T>
__device__ __forceinline__ T row_range(const Edge (&e)[3], const RowEdges& w, float tol, float Rf) {
    float lo = 0.0f, hi = Rf - 1.0f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float D = __builtin_fmaf(tol, 4.0f, e[k].C + w.bp[k]);
        const float t = -D * __builtin_amdgcn_rcpf(e[k].A);
        const bool neg = __float_as_int(e[k].A) < 0;
        lo = fmaxf(lo, neg ? 0.0f : t - WIN_MARGIN);
        hi = fminf(hi, neg ? t + WIN_MARGIN : hi);
    }
    const int l = (int)ceilf(fminf(lo, Rf)), h = (int)floorf(fmaxf(hi, -1.0f));
    return interval_bits<T>((unsigned)max(h + 1 - l, 0), (unsigned)l);
}
// row fr's mask where sure is all ones; sure 0: undecided
template <typename T>
__device__ __forceinline__ T row_fast(const Edge (&e)[3], const RowEdges& w, float fr, int R, T& sureT) {
    float D[3], xh[3], xl[3], g[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        D[k] = e[k].A * fr + e[k].C;
        xh[k] = __builtin_fmaf(D[k], w.rh[k], w.Kh[k]);
        xl[k] = __builtin_fmaf(D[k], w.rl[k], w.Kl[k]);
        g[k] = D[k] + w.bp[k];
    }
    const float xH = fmaxf(fmaxf(xh[0], xh[1]), xh[2]), xL = fminf(fminf(xl[0], xl[1]), xl[2]);
    const int G = __float_as_int(fminf(fminf(g[0], g[1]), g[2]));
    const float yH = -WIN_MAGIC - xH, yL = xL + WIN_MAGIC;
    const float zH = xH + (yH + WIN_MAGIC), zL = xL - (yL - WIN_MAGIC);
    // negative: decided (0x3efffc00 = 1/2 - 2^-15); a negative G needs no limits
    // (an edge along the rows that a row lies outside of has infinite ones)
    const int sure = ((((__float_as_int(zH) & 0x7fffffff) - 0x3efffc00) &
                       ((__float_as_int(zL) & 0x7fffffff) - 0x3efffc00)) | G) & (w.tolBits - (G & 0x7fffffff));
    // as unsigned integers: iH has the sign bit, iL gets it unless yL
    // (a limit far below the grid) or G (empty) is negative
    const unsigned iL = (unsigned)__float_as_int(yL), iH = (unsigned)__float_as_int(yH);
    const unsigned iS = (iL & 0x7fffffffu) | (~(iL | (unsigned)G) & 0x80000000u);
    const T M = interval_bits<T>(__builtin_elementwise_sub_sat(iS, iH), (unsigned)(WIN_BASE + R) - iL);
    int sm = sure >> 31;
    asm("" : "+v"(sm));
    sureT = (T)(int64_t)sm;
    return M;
}

// One row of a pair with finite planes, decided with exact quotients: the AND
// of the three edge masks, empty when the row is not in the reference's
// row-range mask (three_edges<T, true>).  The reference only visits rows of
// that mask.
template <typename T>
__device__ __forceinline__ T row_exact(const Edge (&e)[3], float fr, float nsub, int R) {
    const int r = (int)fr;
    T m = (R >= Bits<T>::width) ? ~(T)0 : (((T)1 << R) - (T)1);
    bool in = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float A = e[k].A, B = e[k].B;
        asm volatile("" : "+v"(A), "+v"(B));   // rare: keep the divisions out of the caller's set-up
        const float DN = (B > 0 ? B * nsub : 0.0f) + e[k].C;
        const bool f1 = DN >= 0.0f, f2 = (A * nsub + DN) >= 0.0f;
        in = in && (f1 == f2 ? f1 : f1 == (r < k_exact(DN, A, R)));
        const float D = A * fr + e[k].C;
        const bool g1 = D >= 0.0f, g2 = (B * nsub + D) >= 0.0f;
        const T low = low_mask<T>(k_exact(D, B, R));
        m &= g1 == g2 ? (g1 ? ~(T)0 : (T)0) : (g1 ? low : ~low);
    }
    return in ? m : (T)0;
}

// test3DPointInTriangle, Step5_2_shadowCal.inl:213-222
__device__ __forceinline__ bool point_in_tri(const float* A, const float* B, const float* C, float px, float py, float pz) {
    auto cross = [](float ax, float ay, float az, float bx, float by, float bz, float* o) {
        o[0] = ay * bz - az * by; o[1] = az * bx - ax * bz; o[2] = ax * by - ay * bx;
    };
    float N1[3], N2[3], N3[3];
    cross(B[0] - A[0], B[1] - A[1], B[2] - A[2], px - B[0], py - B[1], pz - B[2], N1);
    cross(C[0] - B[0], C[1] - B[1], C[2] - B[2], px - C[0], py - C[1], pz - C[2], N2);
    if (dot3(N1[0], N1[1], N1[2], N2[0], N2[1], N2[2]) < 0.0f) return false;
    cross(A[0] - C[0], A[1] - C[1], A[2] - C[2], px - A[0], py - A[1], pz - A[2], N3);
    if (dot3(N2[0], N2[1], N2[2], N3[0], N3[1], N3[2]) < 0.0f) return false;
    return true;
}

// Receiver of word j of a work item's masks, iper = 1 / (words per receiver):
// j / per, exact as j + 1/2 stays 1/2 word from a receiver's ends while the
// float product is off by less than 2^-16 (j < 2^13).
__device__ __forceinline__ int word_receiver(int j, float iper) { return (int)(((float)j + 0.5f) * iper); }

// The work item's rows go out; LDS holds row r's low words at [r][lane]
// (FD_ROW_STRIDE words per row), the high words (64-bit rows) R rows further.  The waves of the work item
// share the write-out.
__device__ __forceinline__ void store_masks(const FdArgs& a, const uint32_t* lds, int id, int n, int R, int wpr,
                                            int wave = 0, int waves = 1) {
    const float iper = 1.0f / (float)(R * wpr);
    // coalesced write-out: consecutive lanes write consecutive words of one
    // receiver's mask (rows x wpr words); the receiver id comes from its
    // lane by a cross-lane read with every lane active
    const int per = R * wpr;
    const int total = n * per;
    for (int j0 = wave * 64; j0 < total; j0 += 64 * waves) {
        const int j = j0 + lane_id();
        const int l = word_receiver(min(j, total - 1), iper), w = j - l * per;
        const int idl = __shfl(id, l, 64);
        if (j < total) {
            const int r = w >> (wpr - 1), h = w & (wpr - 1);
            a.masks[(size_t)idl * per + w] = lds[(h * R + r) * FD_ROW_STRIDE + l];
        }
    }
}

// Masks of n receivers (lane l holds the id of receiver l) set to all
// occluded (back) or none, written straight to the output.
__device__ __forceinline__ void fill_masks(const FdArgs& a, int id, bool back, int n, int R, int wpr, int wave, int waves) {
    const int per = R * wpr;
    const int total = n * per;
    const float iper = 1.0f / (float)per;
    const uint32_t w0 = (R >= 32) ? 0xffffffffu : ((1u << R) - 1u);
    const uint32_t w1 = (R >= 64) ? 0xffffffffu : (R > 32 ? (1u << (R - 32)) - 1u : 0u);
    for (int j0 = wave * 64; j0 < total; j0 += 64 * waves) {
        const int j = j0 + lane_id();
        const int l = word_receiver(min(j, total - 1), iper), w = j - l * per;
        const int idl = __shfl(id, l, 64);
        const bool bk = __shfl((int)back, l, 64) != 0;
        if (j < total) a.masks[(size_t)idl * per + w] = bk ? ((w & (wpr - 1)) == 0 ? w0 : w1) : 0u;
    }
}

// Merge of a segment's partial masks: atomic OR of the non-zero words into
// the (zeroed) output; same word order as store_masks.
__device__ __forceinline__ void or_masks(const FdArgs& a, const uint32_t* lds, int id, int n, int R, int wpr,
                                         int wave = 0, int waves = 1) {
    const float iper = 1.0f / (float)(R * wpr);
    const int per = R * wpr;
    const int total = n * per;
    for (int j0 = wave * 64; j0 < total; j0 += 64 * waves) {
        const int j = j0 + lane_id();
        const int l = word_receiver(min(j, total - 1), iper), w = j - l * per;
        const int idl = __shfl(id, l, 64);
        if (j < total) {
            const int r = w >> (wpr - 1), h = w & (wpr - 1);
            const uint32_t v = lds[(h * R + r) * FD_ROW_STRIDE + l];
            if (v) atomicOr(a.masks + (size_t)idl * per + w, v);
        }
    }
}

// --------------------------------------------------------------------------
// Bin-queue occlusion variant (shadowCal_CTA_kernel, Step5_2_shadowCal.inl:
// 408-1100, dead code in the reference).  Its arithmetic is not the
// per-sample kernel's: edge planes from dot(cross(edge, axis), S - v), a
// fourth plane (the triangle's own) in the row masks, other boundary tests,
// and mask rows along y_delt (bit j of row i: upRight + j x_delt + i y_delt).
// Not part of the per-sample bit-exact contract; selected per context.
//
// Work items and outputs are the per-sample kernel's (64 sorted receivers of
// a bin, the bin's triangle list or a stretch of it).  The lanes take 64
// consecutive triangles, two groups of 32 (the reference's warps: a group
// applies the triangle plane when any of its triangles reaches a row and is
// not entirely in front of the receiver, :876/:929), and the wave walks the
// receivers one by one, their data broadcast from the owning lane.  Row
// masks are merged with LDS atomic ORs into the receivers' rows; rows that
// become full are flagged and skipped (as the reference's flag word, :162-164).
// --------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T cta_shl(int k) { return (k >= 0 && k < Bits<T>::width) ? ((T)1 << k) : (T)0; }

// min(max(ceil(-D / div), 0), R) with the IEEE quotient (NaN -> R), from
// the reciprocal r = rcp_or_nan(div) where k_fast allows it (its bound holds
// for this clamp as well: beyond R + 1 both give R, below 0 both give 0).
__device__ __forceinline__ int cta_k(float D, float div, float r, float Rf) {
    bool slow;
    int k = k_fast(D, r, Rf, slow);
    if (slow) k = (int)fmaxf(0.0f, fminf(Rf, ceilf(-1.0f * D / div)));
    return k;
}

// calLightRowRange (:302-357); bits >= W are cleared by the caller.
// rB = rcp_or_nan(B).
template <typename T>
__device__ __forceinline__ T cta_row_range(float B, float D, int W, float rB) {
    if (B <= 0.0f && D <= 0.0f) return (T)0;
    if (B == 0.0f || D == 0.0f) return cta_shl<T>(W) - (T)1;
    const T m = cta_shl<T>(cta_k(D, B, rB, (float)W)) - (T)1;
    return B < 0.0f ? m : ~m;
}

// calLightHeightRange (:225-300), H = W = R; rA = rcp_or_nan(A)
template <typename T>
__device__ __forceinline__ T cta_height_range(float A, float B, float C, int R, T fullH, float rA) {
    const float D = fmaxf(B * (float)(R - 1) + C, C);
    if (A <= 0.0f && D <= 0.0f) return (T)0;
    if (A == 0.0f || D == 0.0f) return fullH;
    const T m = cta_shl<T>(cta_k(D, A, rA, (float)R)) - (T)1;
    return A < 0.0f ? m : (~m & fullH);
}

__device__ __forceinline__ float bcast(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The triangle loop of the variant for one work item: n receivers (lane s
// holds receiver s in q), triangle list entries [ts, te).  Rows go to lds
// (row r of receiver s at lds[r * FD_ROW_STRIDE + s], high words R rows further).
template <typename T>
__device__ __forceinline__ void cta_tris(const FdArgs& a, uint32_t* lds, T* fullRows, int ts, int te, int n,
                                         const FdRxRec& q, int R) {
    const int lane = lane_id();
    const T FULL = (R >= Bits<T>::width) ? ~(T)0 : (((T)1 << R) - (T)1);   // lightWidthFullBit
    // (T)(1 << H) - 1 with the int shift of the reference (:431): all ones of T from H = 32 on
    const T fullH = (R >= 32) ? ~(T)0 : (((T)1 << R) - (T)1);
    const float xd0 = a.L.xd[0], xd1 = a.L.xd[1], xd2 = a.L.xd[2];
    const float yd0 = a.L.yd[0], yd1 = a.L.yd[1], yd2 = a.L.yd[2];
    const float ur0 = a.L.ur[0], ur1 = a.L.ur[1], ur2 = a.L.ur[2];
    const float eps = a.eps;
    const uint64_t half = lane < 32 ? 0x00000000ffffffffull : 0xffffffff00000000ull;
    for (int tb = ts; tb < te; tb += 64) {
        const int ti = tb + lane;
        int tid = ti < te ? a.sortedTri[ti] : -1;
        const bool has = (unsigned)tid < (unsigned)a.ntris;
        float v[3][3] = {}, bminx = 3.402823466e+38f, bminy = 3.402823466e+38f, bmaxx = -3.402823466e+38f,
              bmaxy = -3.402823466e+38f, minz = 3.402823466e+38f, maxz = -3.402823466e+38f;
        if (has) {
            const FdTri& t = a.tri[tid];
            for (int k = 0; k < 3; ++k) { v[0][k] = t.v0[k]; v[1][k] = t.v1[k]; v[2][k] = t.v2[k]; }
            bminx = t.bminx; bminy = t.bminy; bmaxx = t.bmaxx; bmaxy = t.bmaxy;
            minz = t.minz; maxz = t.maxz;
        }
        // receiver-independent parts (:667-674, and the cross products of :720-742):
        // edge k runs from v_k to v_{k+1} (v0_v1, v1_v2, v2_v0), its plane is
        // dot(cross(edge, axis), S - v_{k+1})
        float cy[3][3], cx[3][3], cl[3][3];
        for (int k = 0; k < 3; ++k) {
            const int j = (k + 1) % 3;
            const float ex = v[k][0] - v[j][0], ey = v[k][1] - v[j][1], ez = v[k][2] - v[j][2];
            const float lx = ur0 - v[j][0], ly = ur1 - v[j][1], lz = ur2 - v[j][2];
            cy[k][0] = ey * yd2 - ez * yd1; cy[k][1] = ez * yd0 - ex * yd2; cy[k][2] = ex * yd1 - ey * yd0;
            cx[k][0] = ey * xd2 - ez * xd1; cx[k][1] = ez * xd0 - ex * xd2; cx[k][2] = ex * xd1 - ey * xd0;
            cl[k][0] = ey * lz - ez * ly;   cl[k][1] = ez * lx - ex * lz;   cl[k][2] = ex * ly - ey * lx;
        }
        // n = cross(v1 - v2, v2 - v0); A3, B3, C3 = n . y_delt, n . x_delt, n . (upRight - v0)
        float nn[3];
        {
            const float ax = v[1][0] - v[2][0], ay = v[1][1] - v[2][1], az = v[1][2] - v[2][2];
            const float bx = v[2][0] - v[0][0], by = v[2][1] - v[0][1], bz = v[2][2] - v[0][2];
            nn[0] = ay * bz - az * by; nn[1] = az * bx - ax * bz; nn[2] = ax * by - ay * bx;
        }
        const float A3o = dot3(nn[0], nn[1], nn[2], yd0, yd1, yd2);
        const float B3o = dot3(nn[0], nn[1], nn[2], xd0, xd1, xd2);
        const float C3o = dot3(nn[0], nn[1], nn[2], ur0 - v[0][0], ur1 - v[0][1], ur2 - v[0][2]);
        if (!__any(has)) break;
        for (int s = 0; s < n; ++s) {
            const T done = fullRows[s];
            if (done == FULL) continue;   // every row of this receiver is full
            const float rminx = bcast(q.rminx, s), rminy = bcast(q.rminy, s);
            const float rmaxx = bcast(q.rmaxx, s), rmaxy = bcast(q.rmaxy, s), rz = bcast(q.z, s);
            // :686-689
            const bool in = bminx <= rminx && bminy <= rminy && rmaxx <= bmaxx && rmaxy <= bmaxy && minz <= rz;
            if (!__any(in)) continue;
            const float S0 = bcast(q.q[0], s), S1 = bcast(q.q[1], s), S2 = bcast(q.q[2], s);
            T rows = 0;
            float A[4], B[4], C[4], rB[4];
            if (in) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const int j = (k + 1) % 3;
                    const float sx = S0 - v[j][0], sy = S1 - v[j][1], sz = S2 - v[j][2];
                    A[k] = dot3(cy[k][0], cy[k][1], cy[k][2], sx, sy, sz);
                    B[k] = dot3(cx[k][0], cx[k][1], cx[k][2], sx, sy, sz);
                    C[k] = dot3(cl[k][0], cl[k][1], cl[k][2], sx, sy, sz);
                }
                A[3] = A3o; B[3] = B3o; C[3] = C3o;
                const float temp = dot3(nn[0], nn[1], nn[2], S0 - v[0][0], S1 - v[0][1], S2 - v[0][2]);   // :772
                const bool skip = fabsf(temp) < eps && point_in_tri(v[0], v[1], v[2], S0, S1, S2);   // :783
                if (!skip) {
                    if (temp > 0.0f) {   // :785-802
#pragma unroll
                        for (int k = 0; k < 4; ++k) { A[k] = -A[k]; B[k] = -B[k]; C[k] = -C[k]; }
                    }
                    rows = fullH;   // :821-842
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        rows &= cta_height_range<T>(A[k], B[k], C[k], R, fullH, rcp_or_nan(A[k]));
                        rB[k] = rcp_or_nan(B[k]);
                    }
                }
            }
            // the group's triangle-plane decision (:876, :929), on the rows
            // before the removal of full rows
            const bool needDepth = rows != (T)0 && !(maxz < rz);
            const bool depth = (__ballot(needDepth) & half) != 0ull;
            rows &= FULL & ~done;   // rows >= H are not part of the grid
            while (rows) {
                const int i = Bits<T>::ctz(rows);
                const float fi = (float)i;
                T m = FULL;
#pragma unroll
                for (int k = 0; k < 3; ++k) m &= cta_row_range<T>(B[k], A[k] * fi + C[k], R, rB[k]);
                if (depth) m &= cta_row_range<T>(B[3], A[3] * fi + C[3], R, rB[3]);
                m &= FULL;
                if (m != (T)0) {
                    T cur;
                    if (Bits<T>::width == 32) {
                        cur = (T)(atomicOr(lds + i * FD_ROW_STRIDE + s, (uint32_t)m) | (uint32_t)m);
                    } else {
                        const uint64_t mm = (uint64_t)m;
                        const uint32_t lo = atomicOr(lds + i * FD_ROW_STRIDE + s, (uint32_t)mm) | (uint32_t)mm;
                        const uint32_t hi = atomicOr(lds + (R + i) * FD_ROW_STRIDE + s, (uint32_t)(mm >> 32)) | (uint32_t)(mm >> 32);
                        cur = (T)(((uint64_t)hi << 32) | lo);
                    }
                    if (cur == FULL) atomicOr(fullRows + s, (T)1 << i);
                }
                rows &= rows - (T)1;
            }
        }
    }
}

// NW waves per work item (2, 4 or 8; 1 in the counting and bin-queue variants):
// they share the work item's receivers and LDS rows and take interleaved
// triangles of the list (rows merged with LDS atomics), so a CU holds NW times
// the waves for the same LDS.
template <typename T, bool COUNT, bool CTA = false, int NW = 1>
__device__ __forceinline__ void occlude_body(const FdArgs& a, const int blkIn) {
    // per wave 64 tile windows (timed variants), then wpr * R rows of
    // FD_ROW_STRIDE words, then 64 full-row masks (T, 64-bit atomics for 64-bit
    // rows: the array is aligned for them)
    extern __shared__ __align__(16) uint32_t lds0[];
    uint32_t* const lds = lds0 + (COUNT || CTA ? 0 : NW * FD_TILE_WORDS);
    const FdState* s = a.st;
    const int status = s->status;
    const int R = a.L.res;                  // rows == columns
    const int wpr = a.L.wpr;
    const int lane = lane_id();
    const int wv = NW > 1 ? uniform((int)(threadIdx.x >> 6)) : 0;   // wave of the work item
    const T FULL = (R >= Bits<T>::width) ? ~(T)0 : (((T)1 << R) - (T)1);
    // work item = (triangle segment seg, chunk c); segment-major so that
    // neighbouring work items share a stretch of the same triangle list
    const int S = a.segs;
    const int seg = blkIn / a.chunkSlots;
    const int c = blkIn - seg * a.chunkSlots;

    if (status != FD_EXIT_OK) {
        if (seg != 0) return;
        // early exit of the frame: every receiver shadow 0, except back-facing
        // receivers once the back-face stage has run (FD/api.cpp:489,
        // Step2_1_samplerRectangleAABB.inl:97)
        const int i0 = c * 64;
        if (i0 >= a.WH) return;
        const int n = min(64, a.WH - i0);
        const bool backStage = status >= FD_EXIT_NO_VALID_SAMPLE;
        bool back = false;
        if (lane < n) {
            back = backStage && __float_as_uint(a.rec[i0 + lane].w) == FD_TAG_BACK;
            if (wv == 0) a.shadow[i0 + lane] = back ? 1.0f : 0.0f;
        }
        fill_masks(a, i0 + lane, back, n, R, wpr, wv, NW);
        return;
    }
    if (c >= s->totalChunks) return;
    const int nb = s->nb;
    const FdChunk ck = a.chunks[c];
    const int bin = ck.nbin >> 8, n = ck.nbin & 255;
    if (bin == nb && seg != 0) return;
    // this work item's stretch of the bin's triangle list (bins 0..nb-1)
    int ts = 0, te = 0;
    if (bin != nb) {
        ts = ck.ts;
        te = ck.te;
        if (S > 1) {
            int per = (te - ts + S - 1) / S;
            if (CTA) per = (per + 31) & ~31;   // stretches keep the groups of 32
            ts += seg * per;
            te = min(te, ts + per);
            if (ts >= te) return;   // nothing to add; the finishing pass counts the merged masks
        }
    }
    const int s0 = ck.s0;
    const bool act = lane < n;
    int id = 0;
    if (act) id = a.sortedId[s0 + lane];
    if ((unsigned)id >= (unsigned)a.WH) id = 0;   // defensive: ids form a permutation

    if (bin == nb) {
        // receivers outside the light plane, invalid or back-facing
        bool back = false;
        if (act) {
            back = __float_as_uint(a.rec[id].w) == FD_TAG_BACK;
            if (wv == 0) a.shadow[id] = back ? 1.0f : 0.0f;
        }
        fill_masks(a, id, back, n, R, wpr, wv, NW);
        return;
    }

    // The longest lists start first, and one of them may outlast all the
    // others (an overlap of many objects): its waves issue before their
    // neighbours.
    if (!COUNT) {
        const unsigned long long pairs = s->pairs, len = (unsigned long long)(te - ts) << (2 * a.gridLog2);
        if (len > 4 * pairs) __builtin_amdgcn_s_setprio(3);
        else if (len > 2 * pairs) __builtin_amdgcn_s_setprio(1);
    }

    FdRxRec q{};
    if (act) q = a.sortedRec[s0 + lane];
    // rows of lanes without a receiver start full (row_occupancy)
    for (int r = wv; r < R; r += NW) {
        lds[r * FD_ROW_STRIDE + lane] = act ? 0u : (uint32_t)FULL;
        if (wpr == 2) lds[(R + r) * FD_ROW_STRIDE + lane] = act ? 0u : (uint32_t)((uint64_t)FULL >> 32);
    }
    // rows shared by several waves: the rows each receiver has full, as any
    // wave found them (after the rows)
    constexpr bool SHARE_FULL = NW > 1 && !CTA;
    T* const fullSh = (T*)(lds + wpr * R * FD_ROW_STRIDE);
    // the receivers' rectangles and depths (after the full-row masks), for the
    // cull of the pairs: five registers more per lane spill
    float* const rectSh = (float*)(fullSh + 64);
    if (!CTA && wv == 0) {
        fullSh[lane] = (T)0;
        rectSh[lane] = q.rminx;
        rectSh[64 + lane] = q.rminy;
        rectSh[128 + lane] = q.rmaxx;
        rectSh[192 + lane] = q.rmaxy;
        rectSh[256 + lane] = q.z;
    }
    if (NW > 1) __syncthreads();
    if (CTA) {
        T* fullRows = (T*)(lds + wpr * R * FD_ROW_STRIDE);
        fullRows[lane] = (T)0;
        __syncthreads();
        cta_tris<T>(a, lds, fullRows, ts, te, n, q, R);
        __syncthreads();
        if (S == 1) {
            int cnt = 0;
            for (int r = 0; r < R; ++r) {
                cnt += __popc(lds[r * FD_ROW_STRIDE + lane]);
                if (wpr == 2) cnt += __popc(lds[(R + r) * FD_ROW_STRIDE + lane]);
            }
            if (act) a.shadow[id] = (float)cnt / (float)a.L.resNum;   // :1080-1088
            store_masks(a, lds, id, n, R, wpr);
        } else {
            or_masks(a, lds, id, n, R, wpr);
        }
        return;
    }
    const float Lx = a.L.ur[0] - q.q[0], Ly = a.L.ur[1] - q.q[1], Lz = a.L.ur[2] - q.q[2];  // L0 - Q
    // the same in the plane set-up: three subtractions cost less than holding or reloading them
    auto l0_q = [&](float (&l)[3]) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            float u = a.L.ur[k];
            asm volatile("" : "+s"(u));
            l[k] = u - q.q[k];
        }
    };
    const float xd0 = a.L.xd[0], xd1 = a.L.xd[1], xd2 = a.L.xd[2];
    const float yd0 = a.L.yd[0], yd1 = a.L.yd[1], yd2 = a.L.yd[2];
    // light axes along x and y (x_delt = (c, 0, 0), y_delt = (0, c', 0), zeros
    // of either sign): then dot(n, x_delt) = n.x * c exactly, up to the sign
    // of a zero result, whenever n is finite (the other two products are
    // zeros).  No later step can tell +0 from -0 (comparisons with 0, the
    // exact-division fallback maps both infinities of a zero divisor to R, and
    // the row window only uses magnitudes).
    const bool axial = xd1 == 0.0f && xd2 == 0.0f && yd0 == 0.0f && yd2 == 0.0f;
    const float nsub = (float)(unsigned)(R - 1);
    const float Rf = (float)R;
    const float Rs = Rf + 2.44140625e-4f;   // R + 2^-12, exact
    const float eps = a.eps;
    auto su = [](float v) { return __int_as_float(uniform(__float_as_int(v))); };   // into a scalar register
    // the projected sample window's constants.  Axial lights below their
    // receivers take the general form, whose normal can point either way.
    const bool axialW = axial && su(Lz) > 0.0f;
    LightProj P;
    TileBox tb{};
    uint32_t tileSide = 0;
    const bool tiles = !COUNT && te - ts >= FD_TILE_LIST * NW;   // the tile windows pay
    float hw, hr, hc, nr, nc;   // light_window's h, hr, hc, nr, nc
    float sgN = 1.0f;           // the light-plane normal's sign towards the light
    {
        auto n1 = [](const float (&v)[3]) { return fabsf(v[0]) + fabsf(v[1]) + fabsf(v[2]); };
        auto ni = [](const float (&v)[3]) { return fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fabsf(v[2])); };
        const float x1 = n1(a.L.xd), y1 = n1(a.L.yd);
        float off = 0.0f;   // |l.X|, |l.Y| of axial lights
        if (axialW) {
            hw = Lz;
            hr = Lz * a.L.X[0];
            hc = Lz * a.L.Y[1];
            nr = -__builtin_fmaf(Lx, a.L.X[0], 0.5f);
            nc = -__builtin_fmaf(Ly, a.L.Y[1], 0.5f);
            off = fmaxf(fabsf(nr), fabsf(nc));
        } else {
            hw = dot3(Lx, Ly, Lz, a.L.N[0], a.L.N[1], a.L.N[2]);
            if (su(hw) < 0.0f) sgN = -1.0f;
            hw *= sgN;
            hr = hc = hw;
            nr = -(dot3(Lx, Ly, Lz, a.L.X[0], a.L.X[1], a.L.X[2]) + 0.5f);
            nc = -(dot3(Lx, Ly, Lz, a.L.Y[0], a.L.Y[1], a.L.Y[2]) + 0.5f);
        }
        const float L1 = fabsf(Lx) + fabsf(Ly) + fabsf(Lz);
        float Ld = wave_max_f32(act ? L1 : 0.0f) + (Rf + 1.0f) * (x1 + y1);
        // Ld t is at most Ld (Ld + 2^21 (|xd|_1 + |yd|_1)); receivers at or above the light have no window
        if (!(Ld >= 9.5367431640625e-07f && Ld * (Ld + 2097152.0f * (x1 + y1)) <= 1.09951163e+12f) ||
            __any(act && !(L1 <= Ld && hw > 0.0f && off <= WIN_MAX_OFFSET)))
            Ld = INFINITY;
        P.kL = Ld * Ld;
        P.kr = Ld * x1;
        P.kc = Ld * y1;
        P.iL = 1.0f / Ld;
        P.er = 3.814697265625e-06f * ni(a.L.X);
        P.ec = 3.814697265625e-06f * ni(a.L.Y);
        if (tiles) {
            // receivers relative to L0: -l in the frame
            auto bounds = [&](bool in) {
                TileBounds b;
                b.x0 = wave_min_f32(in ? nr + 0.5f : INFINITY);
                b.x1 = wave_max_f32(in ? nr + 0.5f : -INFINITY);
                b.y0 = wave_min_f32(in ? nc + 0.5f : INFINITY);
                b.y1 = wave_max_f32(in ? nc + 0.5f : -INFINITY);
                b.z0 = wave_min_f32(in ? -hw : INFINITY);
                b.z1 = wave_max_f32(in ? -hw : -INFINITY);
                b.iz = 1.0f / -b.z1;
                return b;
            };
            tb.all = tb.low = bounds(act);
            tb.zs = INFINITY;
            if (tb.all.z1 - tb.all.z0 > -0.03125f * tb.all.z0) {
                const bool up = -hw > 0.5f * (tb.all.z0 + tb.all.z1);
                tb.low = bounds(act && !up);
                tb.zs = wave_max_f32(act && up ? q.z : -INFINITY);
            }
            tb.Ld = Ld;
            tb.tr = x1;
            tb.tc = y1;
            tb.sx = ni(a.L.X);
            tb.sy = ni(a.L.Y);
            const float cx = xd1 * yd2 - xd2 * yd1, cy = xd2 * yd0 - xd0 * yd2, cz = xd0 * yd1 - xd1 * yd0;
            tb.A = sqrtf(cx * cx + cy * cy + cz * cz);
            tb.eps = eps;
            // the frame's handedness: the sign of V there against the world's
            const float hx = a.L.X[1] * a.L.Y[2] - a.L.X[2] * a.L.Y[1], hy = a.L.X[2] * a.L.Y[0] - a.L.X[0] * a.L.Y[2],
                        hz = a.L.X[0] * a.L.Y[1] - a.L.X[1] * a.L.Y[0];
            const float hd = axialW ? a.L.X[0] * a.L.Y[1] : dot3(hx, hy, hz, a.L.N[0], a.L.N[1], a.L.N[2]) * sgN;
            tileSide = __float_as_uint(hd) & 0x80000000u;
        }
    }
    // strips of 1 << lsw columns: 8 cover the grid
    const int lsw = R <= 8 ? 0 : R <= 16 ? 1 : R <= 32 ? 2 : 3;
    const int nsubBits = WIN_BASE + R - 1;
    T full = act ? (T)0 : FULL;   // rows full; all: no receiver in this lane, or done
    unsigned long long nCand = 0, nPass = 0, nRows = 0, nWaveIt = 0, nWaveRows = 0, nRefRows = 0, nPlanes = 0;
    // read-only for this kernel: the constant address space lets the uniform
    // per-triangle loads go through the scalar unit (s_load)
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const __attribute__((address_space(4))) int* cint_p;
    typedef const __attribute__((address_space(4))) FdTri* ctri_p;
#else
    typedef const int* cint_p;   // host pass: the kernel body is never run
    typedef const FdTri* ctri_p;
#endif
    // the bin's list in the frame's walk order (the masks do not depend on it);
    // the order is read once into a scalar register, so the list address
    // stays scalar
    const int walkOrder = uniform(s->triOrder);
    const cint_p triList = (cint_p)(walkOrder != FD_TRI_ORDER_LIST ? (const int*)a.pairKT : a.sortedTri);
    const ctri_p tris = (ctri_p)(a.tri);
    // Prefilter (timed kernel): the wave reads its next 64 list entries and
    // their culling boxes with vector loads and keeps the triangles that pass
    // the containment + depth test against bounds of all its receivers (the
    // largest lower corner, the smallest upper corner, the largest depth).  A
    // triangle that fails them fails the test of every lane, which then skips
    // it: dropping it early changes nothing.  The counting kernel walks every
    // entry, as the reference does.
    const int* listV = walkOrder != FD_TRI_ORDER_LIST ? (const int*)a.pairKT : a.sortedTri;
    float gx0 = 0.0f, gy0 = 0.0f, gx1 = 0.0f, gy1 = 0.0f, gz = 0.0f;
    if (!COUNT) {
        gx0 = wave_max_f32(act ? q.rminx : -INFINITY);
        gy0 = wave_max_f32(act ? q.rminy : -INFINITY);
        gx1 = wave_min_f32(act ? q.rmaxx : INFINITY);
        gy1 = wave_min_f32(act ? q.rmaxy : INFINITY);
        gz = wave_max_f32(act ? q.z : -INFINITY);
    }
    // containment + depth cull (:120-127): all five bounds in one round trip
    auto culled = [&](const FdTri& t) {
        const float* rc = rectSh + lane;   // rminx, rminy, rmaxx, rmaxy, z
        const float x0 = rc[0], y0 = rc[64], x1 = rc[128], y1 = rc[192], z = rc[256];
        return !((t.bminx <= x0) & (t.bminy <= y0) & (x1 <= t.bmaxx) & (y1 <= t.bmaxy) & (t.minz <= z));
    };
    // row r's mask goes to the receiver's rows (bit: 1 << r); full rows are noted
    auto add_row = [&](uint32_t* w0, T bit, T M) {
        T cur;
        if (Bits<T>::width == 32) {
            if (NW > 1) {
                cur = (T)(atomicOr(w0, (uint32_t)M) | (uint32_t)M);
            } else {
                cur = (T)(*w0 | (uint32_t)M);
                *w0 = (uint32_t)cur;
            }
        } else {
            uint32_t* w1 = w0 + R * FD_ROW_STRIDE;
            const uint64_t mm = (uint64_t)M;
            uint32_t lo32, hi32;
            if (NW > 1) {
                lo32 = atomicOr(w0, (uint32_t)mm) | (uint32_t)mm;
                hi32 = atomicOr(w1, (uint32_t)(mm >> 32)) | (uint32_t)(mm >> 32);
            } else {
                lo32 = *w0 | (uint32_t)mm;
                hi32 = *w1 | (uint32_t)(mm >> 32);
                *w0 = lo32;
                *w1 = hi32;
            }
            cur = (T)(((uint64_t)hi32 << 32) | lo32);
        }
        if (cur == FULL) {
            full |= bit;
            if (SHARE_FULL) {
                if (Bits<T>::width == 32) atomicOr((uint32_t*)(fullSh + lane), (uint32_t)bit);
                else atomicOr((unsigned long long*)(fullSh + lane), (unsigned long long)bit);
            }
        }
    };
    // wave row iterations = max over lanes of this triangle's rows
    auto wave_rows = [&](int nr) {
        if (COUNT) {
            for (int o = 32; o >= 1; o >>= 1) nr = max(nr, __shfl_xor(nr, o, 64));
            if (lane == __ffsll((unsigned long long)__ballot(1)) - 1) nWaveRows += nr;
        }
    };
    // row by row from the first to the last row of the window that is not full
    auto rows_fast = [&](const Edge (&e)[3], T valid, const int tolB) {
        const RowEdges re = row_edges(e, Rf, nsub, tolB);
        if (__any(Bits<T>::last(valid) - Bits<T>::ctz(valid) >= FD_RANGE_ROWS)) {
            valid &= row_range<T>(e, re, __int_as_float(tolB), Rf);
            if (valid == (T)0) return;
        }
        const int r0 = Bits<T>::ctz(valid);
        const int r1 = Bits<T>::last(valid);
        wave_rows(r1 - r0 + 1);
        float fr = (float)r0;
        const float frEnd = (float)r1;
        uint32_t* w0 = lds + r0 * FD_ROW_STRIDE + lane;
        T bit = (T)1 << r0, redo = (T)0;
        do {
            if (COUNT) ++nRows;
            T sure;
            const T M = row_fast<T>(e, re, fr, R, sure);
            redo |= bit & ~sure;
            add_row(w0, bit, M & sure);
            fr += 1.0f;
            bit += bit;
            w0 += FD_ROW_STRIDE;
        } while (fr <= frEnd);
        // the rows left open (about one in a hundred row iterations of a
        // wave), out of the loop so that their divisions cost it no registers
        while (redo) {
            const int r = Bits<T>::ctz(redo);
            add_row(lds + r * FD_ROW_STRIDE + lane, (T)1 << r, row_exact<T>(e, (float)r, nsub, R));
            redo &= redo - (T)1;
        }
    };
    // planes and rows of a triangle whose window the block prefilter bounds for
    // every receiver (TileWindow::lanes): side, tolerance and margin are the
    // triangle's, and of the projections only the rows are left
    auto step_tile = [&](const int tid, const float4* slot, auto axialT) {
        constexpr bool AXIAL = decltype(axialT)::value;
        const FdTri t = tris[tid];
        const float4 sl = *slot;   // mr, tol, side, -
        asm volatile("" ::"s"(t.v0[0]), "s"(t.bminx), "s"(t.minz), "s"(t.e01[0]), "s"(t.e20[2]));
        const float* vb[3] = {t.v1, t.v2, t.v0};
        const float* ev[3] = {t.e01, t.e12, t.e20};
        float av[3][3], r[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            av[k][0] = vb[k][0] - q.q[0];
            av[k][1] = vb[k][1] - q.q[1];
            av[k][2] = vb[k][2] - q.q[2];
            float x = av[k][0], z = av[k][2];
            if constexpr (!AXIAL) {
                x = __builtin_fmaf(av[k][2], a.L.X[2], __builtin_fmaf(av[k][1], a.L.X[1], av[k][0] * a.L.X[0]));
                z = __builtin_fmaf(av[k][2], a.L.N[2], __builtin_fmaf(av[k][1], a.L.N[1], av[k][0] * a.L.N[0])) * sgN;
            }
            r[k] = __builtin_fmaf(x * __builtin_amdgcn_rcpf(z), hr, nr);
        }
        const float rmin = fminf(fminf(r[0], r[1]), r[2]), rmax = fmaxf(fmaxf(r[0], r[1]), r[2]);
        const int lo = __float_as_int((rmin - sl.x) + (WIN_MAGIC + 1.0f)), hi = __float_as_int((rmax + sl.x) + WIN_MAGIC);
        const int l0 = max(lo - WIN_BASE, 0), w = max(min(hi - WIN_BASE, R - 1) + 1 - l0, 0);
        if (SHARE_FULL) full |= (T)fullSh[lane];   // rows the other waves filled
        const T valid = interval_bits<T>((unsigned)w, (unsigned)l0) & (~full) & FULL;
        if (valid == (T)0 || culled(t)) return;
        const uint32_t sg = __float_as_uint(sl.z) & 0x80000000u;
        auto flip = [sg](float v) { return __uint_as_float(__float_as_uint(v) ^ sg); };
        float l[3];
        l0_q(l);
        const float Lxs = flip(l[0]), Lys = flip(l[1]), Lzs = flip(l[2]);
        const float x0 = flip(xd0), y1 = flip(yd1);
        Edge e[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float ax = av[k][0], ay = av[k][1], az = av[k][2];
            const float bx = ev[k][0], by = ev[k][1], bz = ev[k][2];
            const float n0 = ay * bz - az * by, n1 = az * bx - ax * bz, n2 = ax * by - ay * bx;
            e[k].C = dot3(n0, n1, n2, Lxs, Lys, Lzs);
            if (AXIAL) {
                e[k].A = n0 * x0;
                e[k].B = n1 * y1;
            } else {
                e[k].A = dot3(n0, n1, n2, x0, flip(xd1), flip(xd2));
                e[k].B = dot3(n0, n1, n2, flip(yd0), y1, flip(yd2));
            }
        }
        rows_fast(e, valid, __float_as_int(sl.y));
    };
    // one pair (triangle tid, this wave's receivers): cull, sample window,
    // planes, rows
    auto step = [&](const int tid, auto axialT) {
        constexpr bool AXIAL = decltype(axialT)::value;
        if ((unsigned)tid >= (unsigned)a.ntris) return;   // defensive: pair entries are triangle ids
        const FdTri t = tris[tid];
        // the whole record in one round trip
        if (!COUNT) asm volatile("" ::"s"(t.v0[0]), "s"(t.bminx), "s"(t.minz), "s"(t.n[0]), "s"(t.e20[2]));
        // the cull first: where the receivers' heights spread (boxes on a ground),
        // a third of these pairs pass the work item's bounds and no receiver's own
        // (1.2 M triangles of tessellated boxes and ground, 1920 x 1080 receivers,
        // tilted light, 16 x 16 samples: 8268 us after the window, 5966 before it)
        if (full == FULL || culled(t)) return;
        if (COUNT) ++nPass;
        // planes (Q,v0,v1), (Q,v1,v2), (Q,v2,v0) (:150-172) start from
        // a_k = v_{k+1} - Q; a_2 = v0 - Q also gives
        // dir = dot(Q - v0, n) (:130-132) = -dot(v0 - Q, n), exactly (every
        // rounding commutes with the negation)
        const float* vb[3] = {t.v1, t.v2, t.v0};
        const float* ev[3] = {t.e01, t.e12, t.e20};
        float av[3][3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            av[k][0] = vb[k][0] - q.q[0];
            av[k][1] = vb[k][1] - q.q[1];
            av[k][2] = vb[k][2] - q.q[2];
        }
        const float ndir = dot3(av[2][0], av[2][1], av[2][2], t.n[0], t.n[1], t.n[2]);   // -dir
        // Q on the triangle: the reference skips the pair (:134-135).  The
        // counting variant tests here, in the reference's order; the timed
        // variant tests below, only for pairs that can still set a bit (the
        // outcome is the same: a skipped pair sets nothing).
        const bool onTri = fabsf(ndir) < eps;
        if (COUNT && onTri && point_in_tri(t.v0, t.v1, t.v2, q.q[0], q.q[1], q.q[2])) return;
        // samples that can be set, from the projected vertices; most pairs of
        // small triangles end here
        int lo, hi, known;
        float tol;
        bool may;
        if constexpr (AXIAL) {
            may = light_window<true>(P, av, hw, hr, hc, nr, nc, ndir, t.we, nsubBits, lo, hi, known, tol);
        } else {
            float af[3][3];
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const float (&u)[3] = d == 0 ? a.L.X : d == 1 ? a.L.Y : a.L.N;
                    af[k][d] = __builtin_fmaf(av[k][2], u[2], __builtin_fmaf(av[k][1], u[1], av[k][0] * u[0]));
                    if (d == 2) af[k][d] *= sgN;
                }
            may = light_window<false>(P, af, hw, hr, hc, nr, nc, ndir, t.we, nsubBits, lo, hi, known, tol);
        }
        if (!COUNT && !may) return;
        if (SHARE_FULL) full |= (T)fullSh[lane];   // rows the other waves filled
        T valid = ~(T)0;
        if (known < 0) {
            const int l0 = max(lo - WIN_BASE, 0), w = max(min(hi - WIN_BASE, R - 1) + 1 - l0, 0);
            valid = may ? interval_bits<T>((unsigned)w, (unsigned)l0) : (T)0;
        }
        valid &= (~full) & FULL;
        if (!COUNT && valid == (T)0) return;
        // The reference negates t0, t1, L0_Q when dir < 0.  The sign is put
        // into L0 - Q and the light axes before the products (a sign flip
        // commutes with every rounding): A, B, C come out negated, identical
        // up to the sign of zero results, which no later step can observe.
        const uint32_t sg = __float_as_uint(0.0f - ndir) & 0x80000000u;   // dir < 0 (0 - (+-0) is +0)
        auto flip = [sg](float v) { return __uint_as_float(__float_as_uint(v) ^ sg); };
        float l[3];
        l0_q(l);
        const float Lxs = flip(l[0]), Lys = flip(l[1]), Lzs = flip(l[2]);
        Edge e[3];
        float nv[3][3];
        bool finiteC = true;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float ax = av[k][0], ay = av[k][1], az = av[k][2];
            const float bx = ev[k][0], by = ev[k][1], bz = ev[k][2];
            nv[k][0] = ay * bz - az * by;
            nv[k][1] = az * bx - ax * bz;
            nv[k][2] = ax * by - ay * bx;
            e[k].C = dot3(nv[k][0], nv[k][1], nv[k][2], Lxs, Lys, Lzs);
            finiteC = finiteC && __builtin_isfinite(e[k].C);
        }
        const bool allOk = !__any(known >= 0);   // then every plane is finite and small
        // a finite C = dot(n, L0 - Q) implies a finite n (an infinite
        // component makes a product infinite or NaN)
        const float x0 = flip(xd0), y1 = flip(yd1);
        if (AXIAL && (allOk || !__any(!finiteC))) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                e[k].A = nv[k][0] * x0;
                e[k].B = nv[k][1] * y1;
            }
        } else {
            // axial lights: the other components are zeros (of any sign)
            const float x1 = AXIAL ? 0.0f : flip(xd1), x2 = AXIAL ? 0.0f : flip(xd2);
            const float y0 = AXIAL ? 0.0f : flip(yd0), y2 = AXIAL ? 0.0f : flip(yd2);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                e[k].A = dot3(nv[k][0], nv[k][1], nv[k][2], x0, x1, x2);
                e[k].B = dot3(nv[k][0], nv[k][1], nv[k][2], y0, y1, y2);
            }
        }
        if (COUNT) {
            // the rows the reference visits for this pair: its row-range mask
            // minus the rows already full (general form, before any window)
            ++nPlanes;
            Edge g[3];
            float DNg[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                g[k] = e[k];
                g[k].nRowN = -(e[k].A * nsub);
                g[k].nColN = -(e[k].B * nsub);
                g[k].rA = rcp_or_nan(e[k].A);
                g[k].rB = rcp_or_nan(e[k].B);
                DNg[k] = (e[k].B > 0 ? -g[k].nColN : 0.0f) + e[k].C;
            }
            nRefRows += Bits<T>::popc((~full) & FULL & three_edges<T, true>(g, DNg, Rf, R));
            if (valid == (T)0) return;
        }
        if (!COUNT && onTri && point_in_tri(t.v0, t.v1, t.v2, q.q[0], q.q[1], q.q[2])) return;
        if (!allOk) {
            // the exact row range and the pairwise row window for every lane,
            // then row by row, lowest row first (:204-222)
            auto rows = [&](T valid, auto rowMask) {
                wave_rows(Bits<T>::popc(valid));
                while (valid) {
                    if (COUNT) ++nRows;
                    const int r = Bits<T>::ctz(valid);
                    const float fr = (float)r;
                    float D[3];
#pragma unroll
                    for (int k = 0; k < 3; ++k) D[k] = e[k].A * fr + e[k].C;
                    add_row(lds + r * FD_ROW_STRIDE + lane, (T)1 << r, rowMask(D));
                    valid &= valid - (T)1;
                }
            };
            // |A|, |B| <= 2^100 for the fast mask form (a NaN dropped by fmaxf is
            // harmless there: it makes both f1 and f2 false, as in the reference)
            const float mAB = fmaxf(fmaxf(fmaxf(fabsf(e[0].A), fabsf(e[1].A)), fabsf(e[2].A)),
                                    fmaxf(fmaxf(fabsf(e[0].B), fabsf(e[1].B)), fabsf(e[2].B)));
            if (__any(!(mAB <= 1.2676506e+30f))) {
                float DN[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    e[k].nRowN = -(e[k].A * nsub);
                    e[k].nColN = -(e[k].B * nsub);
                    e[k].rA = rcp_or_nan(e[k].A);
                    e[k].rB = rcp_or_nan(e[k].B);
                    DN[k] = (e[k].B > 0 ? -e[k].nColN : 0.0f) + e[k].C;
                }
                rows(valid & three_edges<T, true>(e, DN, Rf, R),
                     [&](const float (&D)[3]) { return (T)(FULL & three_edges<T, false>(e, D, Rf, R)); });
                return;
            }
            // |A|, |B| <= 2^100 here, so only the lower end of the reciprocal
            // range is checked (NaN coefficients fail it as well);
            // DN = C + max(B (R-1), 0) equals (B > 0 ? B (R-1) : 0) + C up to
            // the sign of a zero, B being finite or NaN
            float nR[3], rA[3], dA[3], bn[3], DN[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                dA[k] = e[k].A;
                nR[k] = -(e[k].A * nsub);
                bn[k] = e[k].B * nsub;
                rA[k] = fabsf(e[k].A) >= 7.8886091e-31f ? __builtin_amdgcn_rcpf(e[k].A) : __builtin_nanf("");
                DN[k] = e[k].C + fmaxf(bn[k], 0.0f);
            }
            valid &= three_edges_fast<T>(DN, nR, rA, dA, Rs, R);
            valid &= row_window<T>(e, Rf, mAB);
            if (!__any(valid != (T)0)) return;   // no lane can gain a bit from this triangle
            float nC[3], rB[3], dB[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                dB[k] = e[k].B;
                nC[k] = -bn[k];
                rB[k] = fabsf(e[k].B) >= 7.8886091e-31f ? __builtin_amdgcn_rcpf(e[k].B) : __builtin_nanf("");
                asm("" : "+v"(rB[k]));   // keep the select out of the row loop
            }
            rows(valid, [&](const float (&D)[3]) { return three_edges_fast<T>(D, nC, rB, dB, Rs, R); });
            return;
        }
        rows_fast(e, valid, __float_as_int(tol) - (4 << 23));   // tol / 16
    };
    // The block prefilter's second half: the windows of a block's triangles
    // (lane l holds the id of triangle l, cmask those that pass the boxes) for
    // all receivers at once, kept in LDS per wave.  Returns the triangles that
    // can set a sample; lanesM: those for step_tile.  All triangles at once,
    // it costs about a pair and a half; it saves a third of each pair that
    // step_tile takes (nine in ten on meshes), and the test against the rows
    // costs a quarter of what it did with the windows found anew each time.
    // Before / after: heightfield-1k 2644 / 2226 us, 968 k triangles of spheres
    // at 1280 x 720 6260 / 5045, 1080p soup with 32 x 32 samples 2090 / 1794.
    float4* const tileSh = (float4*)lds0 + wv * 64;   // per triangle: mr, tol, side, first / last row and column (bytes)
    auto tile_stage = [&](uint64_t cmask, const int tidv, const float minz, uint64_t& lanesM, auto axialT) -> uint64_t {
        bool keep = (cmask >> lane) & 1, lanes = false;
        if (keep) {
            const FdTri& tr = a.tri[tidv];
            float vf[3][3], S0 = 0.0f;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float* v = k == 0 ? tr.v0 : k == 1 ? tr.v1 : tr.v2;
                const float x = v[0] - a.L.ur[0], y = v[1] - a.L.ur[1], z = v[2] - a.L.ur[2];
                S0 = fmaxf(S0, fabsf(x) + fabsf(y) + fabsf(z));
                if constexpr (decltype(axialT)::value) {
                    vf[k][0] = x * a.L.X[0];
                    vf[k][1] = y * a.L.Y[1];
                    vf[k][2] = z;
                } else {
                    vf[k][0] = dot3(x, y, z, a.L.X[0], a.L.X[1], a.L.X[2]);
                    vf[k][1] = dot3(x, y, z, a.L.Y[0], a.L.Y[1], a.L.Y[2]);
                    vf[k][2] = dot3(x, y, z, a.L.N[0], a.L.N[1], a.L.N[2]) * sgN;
                }
            }
            const TileWindow w = tile_window<decltype(axialT)::value>(tb, minz > tb.zs ? tb.low : tb.all, vf, S0, tr.we, R - 1);
            lanes = w.lanes;
            keep = w.hi >= w.lo && w.chi >= w.clo;
            const uint32_t box = (uint32_t)(w.lo & 255) | (uint32_t)(w.hi & 255) << 8 | (uint32_t)(w.clo & 255) << 16 |
                                 (uint32_t)(w.chi & 255) << 24;
            // side: the sign of V in the world (negated: dir < 0 where V > 0)
            tileSh[lane] = make_float4(w.mr, w.tol, __uint_as_float(__float_as_uint(-w.side) ^ tileSide),
                                       __uint_as_float(box));
        }
        lanesM = __ballot(lanes);
        return __ballot(keep);
    };
    // Of the block's remaining triangles, those that can set a sample some
    // receiver lacks.  A receiver's rows fill early: on the 1080p soup 70-80%
    // of the pairs that pass the cull, on the sphere meshes a third, only meet
    // full rows.
    auto prune = [&](uint64_t cmask) -> uint64_t {
        uint64_t U[FD_OCC_STRIPS];
        row_occupancy<T>(lds, R, lsw, FULL, U);
        bool keep = (cmask >> lane) & 1;
        if (keep) {
            const uint32_t box = __float_as_uint(tileSh[lane].w);
            const int rlo = box & 255, rhi = (box >> 8) & 255, s0 = ((box >> 16) & 255) >> lsw, s1 = (box >> 24) >> lsw;
            T open = (T)0;
#pragma unroll
            for (int k = 0; k < FD_OCC_STRIPS; ++k) open |= (k >= s0 && k <= s1) ? (T)U[k] : (T)0;
            keep = (open & interval_bits<T>((unsigned)(rhi + 1 - rlo), (unsigned)rlo)) != (T)0;
        }
        return __ballot(keep);
    };
    // the list, once per light class: the axial one needs fewer registers
    auto walk = [&](auto axialT) {
        if (COUNT) {
            for (int ti = ts + wv; ti < te; ti += NW) {
                const uint64_t liveMask = __ballot(full != FULL);
                if (liveMask == 0) break;
                nCand += __popcll(liveMask);
                ++nWaveIt;
                step(triList[ti], axialT);
            }
            return;
        }
        // blocks of 64 of this wave's entries; the candidate loop reads the
        // block's ids from the lanes that loaded them (written once per
        // block, so any subset of lanes that runs an iteration reads the
        // same id).  The next block's ids load while this block's boxes are
        // tested and its pairs run; the box fields load unconditionally, in
        // one round trip.
        int tidNext = (ts + wv + lane * NW < te) ? listV[ts + wv + lane * NW] : -1;
        bool stepped = false;   // some pair has run: rows may be full
        for (int blk0 = ts + wv; blk0 < te; blk0 += 64 * NW) {
            // rows the other waves filled: else a wave whose blocks hold no pair
            // any more would walk its list to the end
            if (SHARE_FULL && stepped) full |= (T)fullSh[lane];
            if (__ballot(full != FULL) == 0) break;
            const int tidv = tidNext;
            bool keep = false;
            float4 bmn = make_float4(0.f, 0.f, 0.f, 0.f), bmx = bmn;
            const bool okv = (unsigned)tidv < (unsigned)a.ntris;
            if (okv) {
                bmn = a.triAABB[2 * tidv];
                bmx = a.triAABB[2 * tidv + 1];
            }
            const int tn = blk0 + (64 + lane) * NW;
            tidNext = tn < te ? listV[tn] : -1;
            if (okv) keep = bmn.x <= gx0 && bmn.y <= gy0 && gx1 <= bmx.x && gy1 <= bmx.y && bmn.z <= gz;
            uint64_t cmask = __ballot(keep);
            uint64_t lanesM = 0;
            const bool tile = tiles && __popcll(cmask) >= FD_TILE_MIN;
            if (tile) cmask = tile_stage(cmask, tidv, bmn.z, lanesM, axialT);
            while (cmask) {
                if (tile && stepped && __popcll(cmask) >= FD_PRUNE_LEFT) cmask = prune(cmask);
                for (int k = 0; k < FD_PRUNE_STEPS && cmask; ++k, cmask &= cmask - 1) {
                    if (__ballot(full != FULL) == 0) return;
                    const int l = uniform(__ffsll((unsigned long long)cmask) - 1);
                    const int tid = __builtin_amdgcn_readlane(tidv, l);
                    if ((lanesM >> l) & 1) step_tile(tid, tileSh + l, axialT);
                    else step(tid, axialT);
                    stepped = true;
                }
            }
        }
    };
    if (axialW) walk(std::true_type{});
    else walk(std::false_type{});
    if (COUNT) {
        // per-lane counts: nCand is wave-wide already
        unsigned long long p = nPass, r = nRows, rr = nRefRows, pl = nPlanes;
        for (int o = 32; o >= 1; o >>= 1) {
            p += __shfl_xor(p, o, 64);
            r += __shfl_xor(r, o, 64);
            rr += __shfl_xor(rr, o, 64);
            pl += __shfl_xor(pl, o, 64);
        }
        unsigned long long wr = nWaveRows;
        for (int o = 32; o >= 1; o >>= 1) wr += __shfl_xor(wr, o, 64);
        if (lane == 0) {
            atomicAdd(a.opCount + 0, nCand);
            atomicAdd(a.opCount + 1, p);
            atomicAdd(a.opCount + 2, r);
            if (wv == 0) atomicAdd(a.opCount + 3, 1ull);
            atomicAdd(a.opCount + 4, nWaveIt);
            atomicAdd(a.opCount + 5, wr);
            atomicAdd(a.opCount + 6, rr);
            atomicAdd(a.opCount + 7, pl);
        }
    }
    __syncthreads();
    // fraction = popcount / (W*H) (:226-231); split lists: after the merge.
    // The write-out is shared by the waves.
    if (wv == 0 && S == 1) {
        int cnt = 0;
        for (int r = 0; r < R; ++r) {
            cnt += __popc(lds[r * FD_ROW_STRIDE + lane]);
            if (wpr == 2) cnt += __popc(lds[(R + r) * FD_ROW_STRIDE + lane]);
        }
        if (act) a.shadow[id] = (float)cnt / (float)a.L.resNum;
    }
    if (S == 1) store_masks(a, lds, id, n, R, wpr, wv, NW);
    else or_masks(a, lds, id, n, R, wpr, wv, NW);
}

// Split lists: shadow value of every receiver of a
// real bin from its merged mask (popcount / samples, :226-231).
__device__ __forceinline__ void occlude_finish_body(const FdArgs& a, const int c) {
    __shared__ int cnt[64];
    const FdState* s = a.st;
    if (s->status != FD_EXIT_OK || c >= s->totalChunks) return;
    const int nb = s->nb;
    const FdChunk ck = a.chunks[c];
    if (ck.nbin >> 8 == nb) return;
    const int s0 = ck.s0, n = ck.nbin & 255;
    const int lane = lane_id();
    int id = lane < n ? a.sortedId[s0 + lane] : 0;
    if ((unsigned)id >= (unsigned)a.WH) id = 0;   // defensive: ids form a permutation
    cnt[lane] = 0;
    __syncthreads();
    // each receiver's words are contiguous: consecutive lanes read
    // consecutive words, and the counts gather per receiver in LDS
    const int per = a.L.res * a.L.wpr;
    const int total = n * per;
    for (int j0 = 0; j0 < total; j0 += 64) {
        const int j = j0 + lane;
        const int l = word_receiver(min(j, total - 1), 1.0f / (float)per), w = j - l * per;
        const int idl = __shfl(id, l, 64);
        if (j < total) {
            const int b = __popc(a.masks[(size_t)idl * per + w]);
            if (b) atomicAdd(&cnt[l], b);
        }
    }
    __syncthreads();
    if (lane < n) a.shadow[id] = (float)cnt[lane] / (float)a.L.resNum;
}

// ==========================================================================
// Kernel entry points.  Single frame: the FdArgs block travels as the kernel
// argument.  Batched: every stage is ONE launch over all instances; block b
// belongs to instance i with map[i] <= b < map[i+1] (host-built prefix), and
// the instance's FdArgs is read from the device-resident instance table.
// ==========================================================================
__global__ __launch_bounds__(RED_BLOCK) void k_reduce(FdArgs a) { reduce_body(a, blockIdx.x); }
__global__ __launch_bounds__(FD_FIN_THREADS) void k_finalize(FdArgs a) { finalize_body(a, blockIdx.x); }
__global__ __launch_bounds__(FD_RXB) void k_rx_key(FdArgs a) { rx_key_body(a, blockIdx.x); }
__global__ __launch_bounds__(FD_RXB) void k_rx_scatter(FdArgs a) { rx_scatter_body(a, blockIdx.x); }
__global__ __launch_bounds__(FD_TRB) void k_tri_count(FdArgs a) { tri_count_body(a, blockIdx.x); }
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan(FdArgs a) { scan_body(a, blockIdx.x); }
__global__ __launch_bounds__(FD_TRB) void k_tri_scatter(FdArgs a) { tri_scatter_body(a, blockIdx.x); }
__global__ __launch_bounds__(FD_ORDER_THREADS) void k_tri_order(FdArgs a) { tri_order_body(a, blockIdx.x); }
// Workgroups are dealt to the 8 XCDs round-robin (block b runs on XCD
// b % 8).  Work items of one bin share that bin's triangle list, so the
// occlusion kernels renumber blocks so that each XCD takes runs of 16
// consecutive work items (runs still alternate between XCDs, which keeps the
// load balanced): neighbouring chunks of a bin then read the list from the
// same L2.  A bijection of [0, n); the tail past the last full group of
// 8 x 16 blocks keeps its order.
__device__ __forceinline__ int xcd_block(int b, int n) {
    constexpr int G = 16;
    if (b >= n - n % (8 * G)) return b;
    const int j = b % (8 * G);
    return b - j + (j & 7) * G + (j >> 3);
}

__global__ __launch_bounds__(64) void k_occlude_finish(FdArgs a) { occlude_finish_body(a, blockIdx.x); }

// NW waves per occlusion work item (they share its receivers and LDS rows):
// 2, 4 or 8 per frame (FdArgs::occWaves; fd_default_waves).  The counting variant
// runs one wave per work item: each receiver then meets its triangles in
// list order with the full-row state of all earlier ones, as in the
// reference, so its work counters do not depend on the schedule.
// 6 waves per SIMD, 80 vector registers, of which 28 to 33 spill in the timed
// variants; at 8 (64) and 7 (72) more do (heightfield-1k 2944 / 2754 / 2739 us at
// 8 / 7 / 6 waves, 1080p soup with 32 x 32 samples 2510 / 2201 / 2100 us when the
// projected window came in), at 5 too few waves hide the record loads.
template <typename T, bool COUNT, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(6))) void k_occlude(FdArgs a) {
    occlude_body<T, COUNT, false, NW>(a, xcd_block(blockIdx.x, gridDim.x));
}
template <typename T>
__global__ __launch_bounds__(64) void k_occlude_cta(FdArgs a) {
    occlude_body<T, false, true>(a, xcd_block(blockIdx.x, gridDim.x));
}
// instance of block b: map[i] <= b < map[i+1] (wave-uniform binary search)
__device__ __forceinline__ int inst_of(const int* __restrict__ map, int n, int b) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (map[mid] <= b) lo = mid; else hi = mid;
    }
    return uniform(lo);
}

#define FD_BATCHED(NAME, BOUND, BODY)                                                          \
    __global__ __launch_bounds__(BOUND) void NAME(const FdArgs* __restrict__ inst,              \
                                                  const int* __restrict__ map, int n) {        \
        const int b = blockIdx.x;                                                              \
        const int i = inst_of(map, n, b);                                                      \
        const FdArgs a = inst[i];                                                              \
        BODY(a, b - map[i]);                                                                   \
    }
FD_BATCHED(kb_reduce, RED_BLOCK, reduce_body)
FD_BATCHED(kb_finalize, FD_FIN_THREADS, finalize_body)
FD_BATCHED(kb_rx_key, FD_RXB, rx_key_body)
FD_BATCHED(kb_tri_count, FD_TRB, tri_count_body)
FD_BATCHED(kb_scan, SCAN_BLOCK, scan_body)
FD_BATCHED(kb_rx_scatter, FD_RXB, rx_scatter_body)
FD_BATCHED(kb_tri_scatter, FD_TRB, tri_scatter_body)
FD_BATCHED(kb_tri_order, FD_ORDER_THREADS, tri_order_body)
#undef FD_BATCHED

// An instance's arguments where the scalar unit can read them again (its address
// in scalar registers, in the constant address space), as a single frame's are in
// its kernel arguments.  A copy of them was held in vector registers: 62 (64-bit
// rows 68) spilled, then 26 (35), and batches of 16 frames of 256 x 256 receivers
// and 16 x 16 samples over a soup of 300 k triangles took 2097 us, then 1942, over
// spheres of 200 k 3360, then 3128.
__device__ __forceinline__ const FdArgs& inst_args(const FdArgs* inst, int i) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const __attribute__((address_space(4))) FdArgs* cargs_p;
#else
    typedef const FdArgs* cargs_p;
#endif
    const uint64_t p = (uint64_t)(inst + i);
    const uint32_t lo = (uint32_t)uniform((int)p), hi = (uint32_t)uniform((int)(p >> 32));
    return *(const FdArgs*)(cargs_p)((uint64_t)lo | (uint64_t)hi << 32);
}

template <typename T, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(6))) void kb_occlude(const FdArgs* __restrict__ inst, const int* __restrict__ map, int n) {
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int i = inst_of(map, n, b);
    occlude_body<T, false, false, NW>(inst_args(inst, i), b - map[i]);
}
__global__ __launch_bounds__(64) void kb_occlude_finish(const FdArgs* __restrict__ inst, const int* __restrict__ map,
                                                        int n) {
    const int b = blockIdx.x;
    const int i = inst_of(map, n, b);
    occlude_finish_body(inst[i], b - map[i]);
}

// Verification of the row-mask primitive on given (D, B) pairs (n = R - 1),
// through the same fast / exact paths as the occlusion kernel.  mode 0: the
// general form for every pair; mode 1: the fast form wherever its
// precondition |B| <= 2^100 holds, the general form elsewhere.
__global__ void k_selftest_rowmask(const float* D, const float* B, int n, int R, int mode, unsigned long long* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    Edge e[3];
    float DD[3], nC[3], rB[3], dB[3];
    for (int k = 0; k < 3; ++k) {
        e[k].A = 0.0f; e[k].B = B[i]; e[k].C = 0.0f;
        e[k].nRowN = 0.0f;
        e[k].nColN = -(B[i] * (float)(unsigned)(R - 1));
        e[k].rA = __builtin_nanf("");
        e[k].rB = rcp_or_nan(B[i]);
        DD[k] = D[i];
        nC[k] = e[k].nColN; rB[k] = e[k].rB; dB[k] = B[i];
    }
    const bool fast = mode == 1 && fabsf(B[i]) <= 1.2676506e+30f;
    const float Rs = (float)R + 2.44140625e-4f;   // R + 2^-12
    const uint64_t FULL = (R >= 64) ? ~0ull : ((1ull << R) - 1ull);
    if (R <= 32) {
        out[i] = fast ? (uint64_t)three_edges_fast<uint32_t>(DD, nC, rB, dB, Rs, R)
                      : (uint64_t)(three_edges<uint32_t, false>(e, DD, (float)R, R)) & FULL;
    } else {
        out[i] = fast ? three_edges_fast<uint64_t>(DD, nC, rB, dB, Rs, R)
                      : three_edges<uint64_t, false>(e, DD, (float)R, R) & FULL;
    }
}

// Verification of the row window: for edge-plane triple i (coef[9i + 3k ..]
// = A_k, B_k, C_k) over an R x R grid, out[4i] = the rows whose three-edge
// AND (general form, clipped to the grid) is non-empty, out[4i + 1] = the
// same rows by the fast form, out[4i + 2] = row_window's rows, out[4i + 3] =
// the row-range mask (the rows the reference visits, general form).  Where
// the occlusion kernel would not take its fast branch (max |A|, |B| > 2^100,
// the only branch that applies the window) the fast rows repeat the general
// ones and the window is every row.
template <typename T>
__device__ __forceinline__ void selftest_rowwindow_one(const float* coef, int R, unsigned long long* out) {
    Edge e[3];
    float nC[3], rB[3], dB[3];
    const float nsub = (float)(unsigned)(R - 1);
    const float Rf = (float)R;
    const float Rs = Rf + 2.44140625e-4f;   // R + 2^-12
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        e[k].A = coef[3 * k];
        e[k].B = coef[3 * k + 1];
        e[k].C = coef[3 * k + 2];
        e[k].nRowN = -(e[k].A * nsub);
        e[k].nColN = -(e[k].B * nsub);
        e[k].rA = rcp_or_nan(e[k].A);
        e[k].rB = rcp_or_nan(e[k].B);
        nC[k] = e[k].nColN;
        dB[k] = e[k].B;
        rB[k] = fabsf(e[k].B) >= 7.8886091e-31f ? __builtin_amdgcn_rcpf(e[k].B) : __builtin_nanf("");
    }
    const float mAB = fmaxf(fmaxf(fmaxf(fabsf(e[0].A), fabsf(e[1].A)), fabsf(e[2].A)),
                            fmaxf(fmaxf(fabsf(e[0].B), fabsf(e[1].B)), fabsf(e[2].B)));
    const bool fast = mAB <= 1.2676506e+30f;
    const T FULL = (R >= Bits<T>::width) ? ~(T)0 : (((T)1 << R) - (T)1);
    uint64_t gen = 0, fst = 0;
    for (int r = 0; r < R; ++r) {
        float D[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) D[k] = e[k].A * (float)r + e[k].C;
        if ((FULL & three_edges<T, false>(e, D, Rf, R)) != (T)0) gen |= 1ull << r;
        if (fast && three_edges_fast<T>(D, nC, rB, dB, Rs, R) != (T)0) fst |= 1ull << r;
    }
    float DN[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) DN[k] = (e[k].B > 0 ? -e[k].nColN : 0.0f) + e[k].C;
    out[0] = gen;
    out[1] = fast ? fst : gen;
    out[2] = fast ? (uint64_t)(row_window<T>(e, Rf, mAB) & FULL) : (uint64_t)FULL;
    out[3] = (uint64_t)(FULL & three_edges<T, true>(e, DN, Rf, R));
}

__global__ void k_selftest_rowwindow(const float* coef, int n, int R, unsigned long long* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (R <= 32) selftest_rowwindow_one<uint32_t>(coef + 9 * (size_t)i, R, out + 4 * (size_t)i);
    else selftest_rowwindow_one<uint64_t>(coef + 9 * (size_t)i, R, out + 4 * (size_t)i);
}

// Verification of the row loop's decisions: for edge-plane triple i over an R x R
// grid, out[4i] = the rows that row_fast decides (none where a coefficient is not
// finite or above 2^78, where the kernel does not use it), out[4i + 1] = those
// decided otherwise than by the general form on the reference's row range,
// out[4i + 2] = the rows where row_exact is, out[4i + 3] = the rows with a sample
// that row_range leaves out.  tol is the least that the windows
// may give, 1/16 of max(52u (|A| R + |B| R + |C|), 2^-100).
template <typename T>
__device__ __forceinline__ void selftest_rows_one(const float* coef, int R, unsigned long long* out) {
    Edge e[3];
    const float nsub = (float)(unsigned)(R - 1);
    const float Rf = (float)R;
    float q = 7.8886091e-31f, DN[3];
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        e[k].A = coef[3 * k];
        e[k].B = coef[3 * k + 1];
        e[k].C = coef[3 * k + 2];
        e[k].nRowN = -(e[k].A * nsub);
        e[k].nColN = -(e[k].B * nsub);
        e[k].rA = rcp_or_nan(e[k].A);
        e[k].rB = rcp_or_nan(e[k].B);
        DN[k] = (e[k].B > 0 ? -e[k].nColN : 0.0f) + e[k].C;
        const float a = fabsf(e[k].A), b = fabsf(e[k].B), c = fabsf(e[k].C);
        ok = ok && a <= 3.0223145e+23f && b <= 3.0223145e+23f && c <= 3.0223145e+23f;   // 2^78; false for NaN
        q = fmaxf(q, 3.0994415e-06f * (a * Rf + b * Rf + c));   // 52u
    }
    uint64_t decided = 0, wrong = 0, wrongExact = 0, lost = 0;
    if (ok) {
        const T FULL = (R >= Bits<T>::width) ? ~(T)0 : (((T)1 << R) - (T)1);
        const T range = three_edges<T, true>(e, DN, Rf, R);
        const int tolB = __float_as_int(q) - (4 << 23);
        const RowEdges re = row_edges(e, Rf, nsub, tolB);
        const T keep = row_range<T>(e, re, __int_as_float(tolB), Rf);
        for (int r = 0; r < R; ++r) {
            float D[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) D[k] = e[k].A * (float)r + e[k].C;
            const T ref = ((range >> r) & (T)1) ? (T)(FULL & three_edges<T, false>(e, D, Rf, R)) : (T)0;
            T sure;
            const T M = row_fast<T>(e, re, (float)r, R, sure);
            if (sure) {
                decided |= 1ull << r;
                if (M != ref) wrong |= 1ull << r;
            }
            if ((row_exact<T>(e, (float)r, nsub, R) & FULL) != ref) wrongExact |= 1ull << r;
            if (ref != (T)0 && !((keep >> r) & (T)1)) lost |= 1ull << r;
        }
    }
    out[0] = decided;
    out[1] = wrong;
    out[2] = wrongExact;
    out[3] = lost;
}

__global__ void k_selftest_rows(const float* coef, int n, int R, unsigned long long* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (R <= 32) selftest_rows_one<uint32_t>(coef + 9 * (size_t)i, R, out + 4 * (size_t)i);
    else selftest_rows_one<uint64_t>(coef + 9 * (size_t)i, R, out + 4 * (size_t)i);
}

// Stage read-back of the receiver rectangles in the reference's 2-layer
// layout (Step2_1_samplerRectangleAABB.inl:122-123); verification only.
__global__ void k_debug_rect(FdArgs a, float* out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.WH) return;
    const float4 r = a.rec[i];
    float v[8] = {FD_F32_MAX, FD_F32_MAX, FD_F32_MAX, 1.0f, -FD_F32_MAX, -FD_F32_MAX, -FD_F32_MAX, 1.0f};
    if (__float_as_uint(r.w) == FD_TAG_VALID) {
        const RxRect q = rx_rect(r, a.st, a.L);
        v[0] = q.bx; v[1] = q.by; v[2] = q.z; v[4] = q.ex; v[5] = q.ey; v[6] = q.z;
    }
    for (int k = 0; k < 8; ++k) out[(size_t)i * 8 + k] = v[k];
}

}  // namespace

// ===========================================================================
// Host-side launch sequence of one frame.
// ===========================================================================
namespace fdk {

static inline int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

int reduce_blocks(long n) { return cdiv(n, RED_BLOCK * RED_ITEMS); }
int scan_blocks(const FdArgs& a) {
    const int nb = 1 << (2 * a.gridLog2);
    return 1 + cdiv(nb + 1, fd_scan_rows(a.nblkR)) +
           (a.ntris > 0 ? cdiv(nb, fd_scan_rows(a.nblkT)) + cdiv(a.ntris, SCAN_CHUNK) : 0);
}
int order_blocks(const FdArgs& a) {
    return (1 << (2 * a.gridLog2)) + 1 + (a.segs > 1 ? cdiv((long)a.WH * a.L.res * a.L.wpr, ZERO_WORDS) : 0);
}

hipError_t enqueue_batch(const FdBatchPlan& p, hipStream_t st) {
    const int n = p.n;
    auto L = [&](int m) { return dim3((unsigned)(p.total[m] > 0 ? p.total[m] : 1)); };
    const int nb = p.maxNb;
    const size_t binLds = nb <= FD_LDS_BINS ? (size_t)nb * FD_BIN_LDS_BYTES : 0;
    kb_reduce<<<L(FD_MAP_RED), RED_BLOCK, 0, st>>>(p.inst, p.map[FD_MAP_RED], n);
    kb_finalize<<<L(FD_MAP_ONE), FD_FIN_THREADS, 0, st>>>(p.inst, p.map[FD_MAP_ONE], n);
    kb_rx_key<<<L(FD_MAP_RX), FD_RXB, (nb + 1) * sizeof(uint32_t) + binLds, st>>>(p.inst, p.map[FD_MAP_RX], n);
    if (p.anyTris)
        kb_tri_count<<<L(FD_MAP_TRI), FD_TRB, nb * sizeof(uint32_t) + binLds, st>>>(p.inst, p.map[FD_MAP_TRI], n);
    kb_scan<<<L(FD_MAP_SCAN), SCAN_BLOCK, 0, st>>>(p.inst, p.map[FD_MAP_SCAN], n);
    kb_rx_scatter<<<L(FD_MAP_RX), FD_RXB, (size_t)(nb + 1) * FD_SCATTER_RX_LDS, st>>>(p.inst, p.map[FD_MAP_RX], n);
    if (p.anyTris) {
        kb_tri_scatter<<<L(FD_MAP_TRI), FD_TRB, (size_t)nb * FD_SCATTER_WIDE_LDS + binLds, st>>>(p.inst, p.map[FD_MAP_TRI], n);
        kb_tri_order<<<L(FD_MAP_NB), FD_ORDER_THREADS, 0, st>>>(p.inst, p.map[FD_MAP_NB], n);
    }
    for (int c = 0; c < FD_OCC_CLASSES; ++c) {   // fd_occ_class: 32 / 64-bit rows x 2 / 4 / 8 waves
        if (p.nocc[c] == 0) continue;
        const int wpr = c / 3 + 1, nw = 2 << (c % 3);
        const size_t shm = fd_occ_lds(wpr, p.maxRes[c], nw);
        const dim3 g = L(FD_MAP_OCC0 + c);
        const int* mp = p.map[FD_MAP_OCC0 + c];
        const FdArgs* in = p.occ[c];
        const int k = p.nocc[c];
        switch (c) {
            case 0: kb_occlude<uint32_t, 2><<<g, 64 * nw, shm, st>>>(in, mp, k); break;
            case 1: kb_occlude<uint32_t, 4><<<g, 64 * nw, shm, st>>>(in, mp, k); break;
            case 2: kb_occlude<uint32_t, 8><<<g, 64 * nw, shm, st>>>(in, mp, k); break;
            case 3: kb_occlude<uint64_t, 2><<<g, 64 * nw, shm, st>>>(in, mp, k); break;
            case 4: kb_occlude<uint64_t, 4><<<g, 64 * nw, shm, st>>>(in, mp, k); break;
            default: kb_occlude<uint64_t, 8><<<g, 64 * nw, shm, st>>>(in, mp, k); break;
        }
    }
    if (p.total[FD_MAP_FIN] > 0) kb_occlude_finish<<<L(FD_MAP_FIN), 64, 0, st>>>(p.occ[0], p.map[FD_MAP_FIN], n);
    return hipGetLastError();
}

// Number of differing 32-bit words of two device buffers (autotuner check).
__global__ __launch_bounds__(256) void k_count_diff(const uint32_t* __restrict__ a, const uint32_t* __restrict__ b,
                                                    size_t n, unsigned long long* out) {
    int c = 0;
    for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) c += a[i] != b[i];
    c = wave_sum_i32(c);
    if (lane_id() == 0 && c) atomicAdd(out, (unsigned long long)c);
}

hipError_t count_diff(const uint32_t* a, const uint32_t* b, size_t n, unsigned long long* out, hipStream_t st) {
    hipError_t e = hipMemsetAsync(out, 0, sizeof(unsigned long long), st);
    if (e != hipSuccess) return e;
    const size_t blocks = std::min<size_t>((n + 255) / 256, 8192);
    k_count_diff<<<(unsigned)std::max<size_t>(blocks, 1), 256, 0, st>>>(a, b, n, out);
    return hipGetLastError();
}

hipError_t selftest_rowmask(const float* D, const float* B, int n, int R, int mode, unsigned long long* out) {
    k_selftest_rowmask<<<cdiv(n, 256), 256>>>(D, B, n, R, mode, out);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipDeviceSynchronize();
    return e;
}

hipError_t selftest_rowwindow(const float* coef, int n, int R, unsigned long long* out) {
    k_selftest_rowwindow<<<cdiv(n, 256), 256>>>(coef, n, R, out);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipDeviceSynchronize();
    return e;
}

hipError_t selftest_rows(const float* coef, int n, int R, unsigned long long* out) {
    k_selftest_rows<<<cdiv(n, 256), 256>>>(coef, n, R, out);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipDeviceSynchronize();
    return e;
}

hipError_t debug_rect(const FdArgs& a, float* out8, hipStream_t st) {
    k_debug_rect<<<cdiv(a.WH, 256), 256, 0, st>>>(a, out8);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    return e;
}

hipError_t enqueue_frame(const FdArgs& a, hipStream_t st, hipEvent_t* ev) {
    const int nb = 1 << (2 * a.gridLog2);
    const size_t binLds = a.binLds ? (size_t)nb * FD_BIN_LDS_BYTES : 0;
    auto mark = [&](int i) { if (ev) (void)hipEventRecord(ev[i], st); };
    mark(0);
    k_reduce<<<a.nbR + a.nbV, RED_BLOCK, 0, st>>>(a);
    k_finalize<<<1, FD_FIN_THREADS, 0, st>>>(a);
    mark(1);
    // receivers: key + bin statistics; triangles: setup + pair count (needs the statistics)
    k_rx_key<<<a.nblkR, FD_RXB, (nb + 1) * sizeof(uint32_t) + binLds, st>>>(a);
    mark(2);
    if (a.ntris > 0) k_tri_count<<<a.nblkT, FD_TRB, nb * sizeof(uint32_t) + binLds, st>>>(a);
    // offsets and tables, then both stable scatters
    k_scan<<<scan_blocks(a), SCAN_BLOCK, 0, st>>>(a);
    k_rx_scatter<<<a.nblkR, FD_RXB, (size_t)(nb + 1) * FD_SCATTER_RX_LDS, st>>>(a);
    if (a.ntris > 0) k_tri_scatter<<<a.nblkT, FD_TRB, (size_t)nb * FD_SCATTER_WIDE_LDS + binLds, st>>>(a);
    mark(3);
    if (a.ntris > 0) k_tri_order<<<order_blocks(a), FD_ORDER_THREADS, 0, st>>>(a);
    mark(4);
    // occlusion (or the early-exit fill); split lists count the masks after the
    // merge
    const int wpr = a.L.wpr;
    if (a.occVariant == FD_OCC_BIN_QUEUE) {
        const int chunks = a.chunkSlots * a.segs;
        const size_t shmCta = (size_t)wpr * a.L.res * FD_ROW_STRIDE * sizeof(uint32_t) + 64 * sizeof(uint64_t);   // + full-row flags
        if (wpr == 1) k_occlude_cta<uint32_t><<<chunks, 64, shmCta, st>>>(a);
        else k_occlude_cta<uint64_t><<<chunks, 64, shmCta, st>>>(a);
    } else {
        const int chunks = a.chunkSlots * a.segs;
        if (a.opCount) {
            const size_t shm = fd_occ_lds(wpr, a.L.res, 0);
            if (wpr == 1) k_occlude<uint32_t, true, 1><<<chunks, 64, shm, st>>>(a);
            else k_occlude<uint64_t, true, 1><<<chunks, 64, shm, st>>>(a);
        } else {
            const int nw = fd_valid_waves(a.occWaves) ? a.occWaves : fd_default_waves(a.L.res, a.chunkSlots);
            const int c = fd_occ_class(wpr, nw);
            const size_t shm = fd_occ_lds(wpr, a.L.res, nw);
            switch (c) {
                case 0: k_occlude<uint32_t, false, 2><<<chunks, 64 * nw, shm, st>>>(a); break;
                case 1: k_occlude<uint32_t, false, 4><<<chunks, 64 * nw, shm, st>>>(a); break;
                case 2: k_occlude<uint32_t, false, 8><<<chunks, 64 * nw, shm, st>>>(a); break;
                case 3: k_occlude<uint64_t, false, 2><<<chunks, 64 * nw, shm, st>>>(a); break;
                case 4: k_occlude<uint64_t, false, 4><<<chunks, 64 * nw, shm, st>>>(a); break;
                default: k_occlude<uint64_t, false, 8><<<chunks, 64 * nw, shm, st>>>(a); break;
            }
        }
    }
    if (a.segs > 1) k_occlude_finish<<<a.chunkSlots, 64, 0, st>>>(a);
    mark(5);
    return hipGetLastError();
}

}  // namespace fdk
