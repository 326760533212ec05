// Launch interface of the gfx950 kernels (host side).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "fd_types.h"

#define FD_RXB 1024   // receivers per block in the key / scatter passes
#define FD_TRB 1024   // triangles per block in the count / scatter passes
#define FD_TRI_CLASSES 16      // area classes of the area walk order
// Automatic walk order of a connected mesh: the mesh order up to this many
// pairs per 256 bins (the mean list length in 16x16 bins: a small triangle
// touches about one bin at any grid), the list order above (dense scenes,
// where a receiver fills from whichever object comes first in the list)
#define FD_MESH_MAX_LIST16 7168
#define FD_WALK_KEY_BITS 5     // bits of an area class or of the no-entry value FD_TRI_CLASSES
#define FD_ORDER_CACHE 32768   // list entries whose walk keys the area-order pass keeps in LDS
#define FD_ORDER_THREADS 1024  // threads per bin in the area-order pass

// One occlusion work item: receivers s0 .. s0 + n - 1 of the sorted order and
// their bin's triangle list.
struct FdChunk {
    int s0;
    int nbin;    // n | bin << 8
    int ts, te;
};

// Everything one frame's kernels read, passed by value (kernarg segment).
struct FdArgs {
    FdLight L;
    float eps;
    int cull;
    int gridLog2;
    int tileLog2;         // receiver tiles of (1 << tileLog2) x (64 >> tileLog2) pixels, 3..6
    // occluders
    const float* verts;
    int vstride;          // floats between consecutive vertices
    int nverts;
    const int* idx;       // int3 per triangle
    int ntris;
    // receivers
    const float4* pos;
    const float4* nrm;
    int W, H, WH;
    int npos;             // receiver traversal positions: 8x8 tiles covering the view
    // outputs (dense y*W + x)
    float* shadow;
    uint32_t* masks;      // WH * res * wpr words
    // workspace
    FdState* st;
    float4* rec;          // WH: (x', y', z, tag)
    uint16_t* rxKey;      // WH
    uint32_t* histR;      // (nb + 1) * nblkR, scanned in place
    int nblkR;            // blocks of the receiver key / scatter passes
    int nblkT;            // blocks of the triangle count / scatter passes
    int nbR, nbV;         // k_reduce blocks over receivers / vertices
    long nR, nT;          // lengths of the receiver / pair histograms
    uint32_t* rxTot;      // nb + 1: receivers per key
    uint32_t* triTot;     // nb: pairs per bin
    int* sortedId;        // WH
    FdRxRec* sortedRec;   // WH
    uint32_t* binStat;    // nb * 5 (order-preserving encodings)
    float4* triAABB;      // 2 * ntris
    FdTri* tri;           // ntris
    int* triCount;        // ntris
    uint2* triRange;      // ntris: (sx | sy << 16, ex | ey << 16)
    uint32_t* histT;      // nb * nblkT, scanned in place
    uint32_t* triOff;     // ntris: pair counts, scanned in place into triangle-major offsets
    uint32_t* pairKT;     // pairCap: triangle-major pairs, (index in block << 16) | bin; after the
                          // scatter, the bins' lists in area-class order (when the frame uses it)
    uint8_t* triClass;    // ntris: area class of each light-plane triangle's culling box (0 = largest)
    int* sortedTri;       // pairCap
    unsigned long long pairCap;
    int* rxStart;         // nb + 1
    int* rxEnd;           // nb + 1 (rxStart + 1)
    int* triStart;        // nb
    int* triEnd;          // nb (triStart + 1)
    int* chunkStart;      // nb + 1: first work item of each bin (in occlusion order)
    FdChunk* chunks;      // chunkSlots: the work items (over histR / histT, done with by then)
    uint32_t* part;       // per-block partials: 8 per k_reduce block (value-major), then 2 per pair-count block
    unsigned long long* opCount;  // optional occlusion counters (FD_NOPS), or null
    // occlusion work split: chunkSlots = receiver chunk slots (64 each, an upper
    // bound of the work items); each bin's triangle list is cut into segs
    // segments, one work item per (chunk, segment); with segs > 1 the partial
    // masks merge by atomic OR into zeroed masks and a finishing pass counts them
    int chunkSlots;
    int segs;
    // pair passes: bin statistics staged in LDS (the launch allocates
    // FD_BIN_LDS_BYTES per bin besides the counters); set when nb <= FD_LDS_BINS
    int binLds;
    // occlusion kernel: FD_OCC_PER_SAMPLE (the contract) or FD_OCC_BIN_QUEUE
    int occVariant;
    // order of each bin's triangle list in the per-sample occlusion:
    // FD_TRI_ORDER_AUTO, FD_TRI_ORDER_LIST, FD_TRI_ORDER_AREA or FD_TRI_ORDER_MESH
    int triOrder;
    // waves per occlusion work item (per-sample kernel): 2, 4 or 8
    int occWaves;
    int wavesReq;         // asked for by the caller (0 = fd_default_waves, or a batch's own rule)
    // stretches per bin list asked for (fd_set_list_split; 0 = the automatic
    // rule, which a batch that fills the GPU overrides with no split)
    int splitReq;
};

// Stretches of a bin's triangle list (fd_set_list_split): 1 = whole lists,
// up to FD_LIST_SPLIT_MAX (fd4d.h).  The automatic rule: a frame of at
// most FD_SPLIT_ITEMS work items and fewer than FD_SPLIT_MIN_WAVES waves in
// all (work items x waves per item) splits its lists into about
// FD_SPLIT_WAVES waves, at most fd_split_max stretches; larger frames keep
// whole lists.  Each stretch merges its masks into the output by atomic OR,
// which only pays where the GPU would otherwise idle.
#define FD_SPLIT_ITEMS 2048
#define FD_SPLIT_MIN_WAVES 6144
#define FD_SPLIT_WAVES 49152
// Most stretches by the triangles per bin (the host does not know the lists):
// a stretch of a few entries costs more than it takes off.  Measured at 8 x 8
// and 16 x 16 bins, 16 x 16 to 200 x 200 receivers, 16 x 16 and 64 x 64
// samples, on soups, spheres and boxes: frames as at 64 x 64 receivers, us with
// 16 stretches / with this rule: 7 triangles per bin 115 / 96, 78 per bin 153 /
// 139 (evenly spread triangles); at 234 per bin and more single frames would
// take 16 rather than 8 (soup 196 / 226, 20 finely tessellated spheres 189 /
// 221).  Whole lists are up to 2.1 times faster where many objects overlap
// (968 k triangles of 500 spheres, 176 x 176 receivers: 2278 / 1068) and up to
// 4.3 times slower elsewhere (1 M triangles of 20 spheres 1674 / 7271, soup 1717
// / 2817), which the counts at hand do not tell apart: never chosen for dense
// lists.
inline int fd_split_max(long ntris, int nb) {
    const long e = ntris / nb;
    return e < 16 ? 4 : e < 512 ? 8 : 16;
}

// Waves per occlusion work item (per-sample kernel) unless a frame asks for
// another count (2, 4 or 8): the waves share a work item's receivers, LDS
// rows and full-row masks and split its triangle list.  8 for frames of up to
// FD_WAVES8_ITEMS work items (too few to fill the GPU with 4 waves each), 4 for
// larger frames: the fewer waves share a work item the less they walk past one
// another.  64-bit rows leave LDS for 5 work items of 4 waves per CU at 48 x 48
// samples and 4 at 64 x 64, where 3 of 8 fit either way: 4 waves then also leave
// fewer in flight, and the longest lists, which outlast the frame, to fewer:
// 4 only from FD_WAVES8_ITEMS64 items on (us, 8 / 4 waves, 48 x 48 samples: 1 M
// triangle soup 817 / 1252 at 720 x 720 receivers, 940 / 1106 at 960 x 960, 1697 /
// 1406 at 1920 x 1080; 300 k triangles of 20 spheres 2071 / 3275, 2865 / 3214 and
// 5421 / 5236; 500 spheres of 200 k triangles 1254 / 1147 and 3933 / 3315), and
// above 48 samples a side from FD_WAVES8_ITEMS_WIDE on (64 x 64 samples, occluders
// that the receivers lie on, at 1920 x 1080 and 2560 x 1440: 1.2 M triangles of
// tessellated boxes and ground 5949 / 7602 and 8299 / 8784, 216 k of boxes alone 2192
// / 2682 and 3329 / 3335, slivers 10655 / 11562 and 17904 / 19330, terrain 3677 /
// 3919 and 5814 / 5934; short and sparse lists go the other way: a canopy 1208 /
// 1014 and 2050 / 1718, the evenly spread boxes 3518 / 3392 and 5827 / 5487).
#define FD_WAVES8_ITEMS 8192
#define FD_WAVES8_ITEMS64 28672
#define FD_WAVES8_ITEMS_WIDE 45056
// In a batch of more than FD_BATCH_WAVES4_ITEMS work items in all, its small
// frames of 32-bit rows take 4 as well: the others fill the GPU beside them (us, 8
// / 4 waves: four of 700 x 700 receivers, 32 k items, 16 x 16 samples: spheres of
// 200 k triangles 3549 / 3052, soup of 300 k 1310 / 1340, 300 k triangles of 20
// spheres 7896 / 7938; 24 of 256 x 256, 31 k items: 4652 / 4143, 2889 / 2721 and
// 13704 / 13455).  Below, the longest lists outlast the batch (two of 512 x 512, 9
// k items, 8 x 8 samples: that soup 545 / 726, those 20 spheres 3065 / 3539; three
// of 700 x 700, 24 k items, 16 x 16: soup of 1 M 1702 / 1979), and 64-bit rows lose
// there and at 31 k items (0 to 11% with 64 x 64 samples).
#define FD_BATCH_WAVES4_ITEMS 28672
inline int fd_default_waves(int res, long items) {
    return items <= (res > 48 ? FD_WAVES8_ITEMS_WIDE : res > 32 ? FD_WAVES8_ITEMS64 : FD_WAVES8_ITEMS) ? 8 : 4;
}
inline bool fd_valid_waves(int w) { return w == 2 || w == 4 || w == 8; }

// LDS of an occlusion work item: the tile windows of each wave's block (64
// float4; nw = 0: none), its light rows ([row][receiver], a stride of
// 65 words, so that lanes that walk one receiver's rows, or one lane per row,
// use different banks: the write-out and the prefilter's occupancy pass), the
// full-row masks (one row word per receiver) and the receivers' rectangles and
// depths (5 floats).
#define FD_ROW_STRIDE 65
#define FD_TILE_WORDS 256
inline size_t fd_occ_lds(int wpr, int res, int nw) {
    return (size_t)nw * FD_TILE_WORDS * sizeof(uint32_t) + (size_t)wpr * res * FD_ROW_STRIDE * sizeof(uint32_t) + 64 * (wpr * sizeof(uint32_t) + 5 * sizeof(float));
}
// Column strips of the light grid in the occlusion prefilter
#define FD_OCC_STRIPS 8
// The prefilter's windows for all receivers at once: for lists of FD_TILE_LIST
// entries per wave and more, on blocks of FD_TILE_MIN triangles and more that
// pass the boxes.  Its test against the receivers' rows: on a block's remaining
// triangles (FD_PRUNE_LEFT or more) before every FD_PRUNE_STEPS pairs.
// Measured flat around these (16 / 4 / 4 and 32 / 6 / 6: within 1%; rows tested
// every 8 or 24 pairs: 1 to 3% slower on the soup or the meshes).
#define FD_TILE_LIST 32
#define FD_TILE_MIN 6
#define FD_PRUNE_LEFT 6
#define FD_PRUNE_STEPS 16
// Rows of a pair (last - first) from which the row loop takes row_range first
#define FD_RANGE_ROWS 6

// Occlusion classes of a batched launch: 32-bit / 64-bit rows x 2 / 4 / 8
// waves per work item (one launch each).
#define FD_OCC_CLASSES 6
inline int fd_occ_class(int wpr, int occWaves) { return (wpr - 1) * 3 + (occWaves == 2 ? 0 : occWaves == 4 ? 1 : 2); }


#define FD_LDS_BINS 1024
#define FD_BIN_LDS_BYTES 20

// Scatters with all 16 waves of a block: 16 x 16-bit per-wave counts, and for
// the pairs a 32-bit block offset, per bin in LDS (144 KiB at the largest
// grid, 64 x 64 = 4096 bins).
#define FD_SCATTER_RX_LDS 32
#define FD_SCATTER_WIDE_LDS 36

// Scans: rows of a histogram (nblk counts each) per block, about 4096 counts
__host__ __device__ inline int fd_scan_rows(int nblk) { return nblk >= 4096 ? 1 : 4096 / nblk; }

// Occlusion counters, in the order documented at fd_get_profile.
#define FD_NOPS FD_PROFILE_COUNTERS

// Stage boundaries recorded when profiling (events[0..FD_NSTAGES]).
#define FD_NSTAGES 5   // light plane, receiver keys, triangle pairing (and both scatters), list order, occlusion

#define FD_FIN_THREADS 1024   // k_finalize block size

// Block maps of a batched launch (prefix sums over instances, n + 1 each).
enum FdMap { FD_MAP_ONE, FD_MAP_RED, FD_MAP_RX, FD_MAP_TRI, FD_MAP_SCAN, FD_MAP_OCC0, FD_MAP_OCC1, FD_MAP_OCC2,
             FD_MAP_OCC3, FD_MAP_OCC4, FD_MAP_OCC5, FD_MAP_FIN, FD_MAP_NB, FD_NMAPS };
static_assert(FD_MAP_OCC0 + FD_OCC_CLASSES == FD_MAP_FIN, "one block map per occlusion class");
static_assert(FD_TRI_CLASSES < (1 << FD_WALK_KEY_BITS), "area classes and the no-entry value fit the key bits");

struct FdBatchPlan {
    const FdArgs* inst;       // device: instance table (n)
    const FdArgs* occ[FD_OCC_CLASSES];   // device: instances of each occlusion class (fd_occ_class), largest first
    int n, nocc[FD_OCC_CLASSES];
    const int* map[FD_NMAPS]; // device prefix arrays
    int total[FD_NMAPS];      // blocks per stage launch
    int maxNb;                // largest bin count (dynamic LDS sizes)
    int maxRes[FD_OCC_CLASSES];   // largest light grid per occlusion class
    bool anyTris;
};

namespace fdk {
hipError_t enqueue_frame(const FdArgs& a, hipStream_t st, hipEvent_t* stageEvents = nullptr);
hipError_t enqueue_batch(const FdBatchPlan& p, hipStream_t st);
int reduce_blocks(long n);
int scan_blocks(const FdArgs& a);
int order_blocks(const FdArgs& a);   // one per bin and the invalid key, and the mask-zeroing ones
}  // namespace fdk
