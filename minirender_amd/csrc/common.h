// common.h -- device-side tables of the rasterization pipeline (gfx950).
//
// A batch is a set of jobs (frames).  Every kernel works over the whole batch:
// the plain Renderer::render() path is a batch of one job.  All tables below
// live in device memory and are written by the host once per batch.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define MR_HD __host__ __device__
#else
#define MR_HD
#endif

namespace mr {

// One draw (Renderable + material) of a job.  The modelview and normal matrix
// rows 0..2 are what Renderer::paintMesh multiplies by (Renderer.cpp:336-348).
struct DrawDesc {
  float mv[12];  // modelview rows 0..2, row-major
  float nm[12];  // normal matrix rows 0..2
  float diffuse[3];
  float specular[3];
  float emissive[3];
  float shininess;
  const float* pos;    // positions, 3 floats each
  const float* nrm;    // normals, 3 floats each
  const float* uv;     // texcoords, 2 floats each (null: uv = 0)
  const int32_t* idx;  // 3 per triangle
  const int32_t* nidx;
  const int32_t* tidx;  // null when the mesh has no texcoords
  const void* tex;      // null unless texturing applies (Renderer.cpp:228)
  int32_t tex_format;
  int32_t tex_rows, tex_cols;
  int32_t ntri;
  int32_t job;
  int32_t tile_base;    // the job's first global tile and tiles per row
  int64_t tri_begin;    // first flat triangle index of this draw in the batch
  uint32_t order_base;  // 2 * triangles of earlier draws of the same job
  int32_t tiles_x;
  int64_t vbase;        // first projected-vertex record of this draw's mesh
  int32_t no_clip;      // 1: no near-plane test (paintTriangle, world = false)
  int32_t pad_;
};

// One frame of a batch.
struct JobDesc {
  float P[16];  // projection, row-major
  float znear;  // Renderer.cpp:324-326
  int32_t persp;
  int32_t W, H;
  int32_t tiles_x, tiles_y;
  int32_t tile_base;  // first global tile of this job
  int32_t draw_begin, draw_end;
  float bg[3];
  float light[3];
  int32_t light_is_point;
  float ambient;
  int32_t lighting;
  int32_t save_normals;
  int32_t shade_base;  // first shading block of this job
  int64_t tri_begin, tri_end;  // flat triangles of this job in the batch
  uint32_t* win;       // device scratch: draw-order id of each pixel's winner
  uint8_t* rgb8;       // device outputs (any may be null)
  float* depth;
  uint32_t* winner;
  float* rgb;
  float* normals;
  float* points;       // range image (Renderer.cpp:388-415)
};

// Projected-vertex record written once per vertex by the vertex kernel:
// {px, py, zv, ez}, the projection (Renderer.cpp:191-203) and eye depth
// (:344-345) of the vertex, all that triangle setup reads for a triangle in
// front of the near plane.  The eye x, y that the near-plane clip needs are
// transformed again from the positions where it runs.
constexpr int kVrecFloats = 4;

// A surviving (sub-)triangle as the binner sees it: its id (2 * flat
// triangle index + clip sub-index), its draw and clamped pixel bbox.
struct BinItem {
  uint32_t id;
  uint32_t draw;
  uint16_t bx0, bx1, by0, by1;
};
static_assert(sizeof(BinItem) == 16, "BinItem must be 16 bytes");

// Device counters of a batch (64-bit, cleared by the clear kernel).
enum Counter : int {
  kItems = 0,        // surviving (sub-)triangles (statistics)
  kBinOverflow = 2,  // set when the bin list was too small
  kError = 3,        // set when a bounded wait hit its limit
  kClipped = 4,      // input triangles that crossed the near plane
  kBinEntries = 6,   // total (tile, triangle) pairs (the scan's and the direct ones)
  kParts = 7,        // work items of split tiles (written by the scan)
  kHeavy = 8,        // tiles split over several work items
  kHeavyOverflow = 9,
  kListed = 10,      // tiles in the raster's tile list (written by the scan)
  kDirect = 11,      // direct items of all jobs, listed or (no room) binned after all
  kDirectPairs = 14, // (tile, direct item) pairs, at the end of the bin list
  kDirectTilesListed = 15,  // tiles with such pairs only, at the end of the tile list
  kWidePx = 12,      // bbox pixels of the items that want edge checkpoints ...
  kWideRows = 13,    // ... and their bbox rows (they choose the column spacing)
  kNumCounters = 16
};

// Raster work items of a batch, from its counters: parts and row bands of
// split tiles, and tiles rastered whole (those with bin entries, then those
// with direct entries only: `listed` in all).
struct TileItems {
  int64_t parts, whole, listed;
};
MR_HD inline TileItems tile_items(const unsigned long long* counters, uint32_t parts_cap,
                                  int32_t ntiles) {
  // After a bin-list overflow binning may have stored over the direct pairs
  // at the list's other end: a tile's range can hold pairs of another job,
  // whose setup with this tile's frame size and near plane gives boxes that
  // no checkpoints were taken for.  Nothing is drawn (nor shaded); the batch
  // runs again with a longer list.
  // After a merge-slot or part-list overflow the part list is incomplete:
  // split tiles are then skipped (the frame is re-run with larger buffers).
  // (All words are loaded before one is looked at: every raster workgroup
  // waits for them, also the many past the last item.)
  const unsigned long long over = counters[kBinOverflow], heavy = counters[kHeavyOverflow];
  const int64_t parts = (int64_t)counters[kParts], whole = (int64_t)counters[kListed],
                direct = (int64_t)counters[kDirectTilesListed];
  TileItems r;
  const int64_t listed = over ? 0 : ntiles, split = over | heavy ? 0 : parts_cap;
  r.parts = parts < split ? parts : split;
  r.whole = whole < listed ? whole : listed;
  r.listed = r.whole + direct < listed ? r.whole + direct : listed;
  return r;
}

// Row bands that each tile rastered whole is shared out in, in batches of few
// tiles.  A tile's direct entries (up to kDirectCap) are not among those that
// the scan splits tiles by, so one workgroup a tile would draw them all, however
// few tiles there are.  From kBandDirect items (a chunk of the raster) up to 8
// workgroups draw a tile while these are at most kBandGroups, about what the GPU
// holds, and the raster's grid (ntiles + parts_cap) holds them anyway.  With the shares of
// split tiles (direct_share), us a call: 8,000 triangles over a 96 x 64 frame
// 376 -> 310 (335 with all of them binned and split), 20,000 690 -> 404 (430);
// 20,000 over 320 x 240 885 -> 636.
constexpr int64_t kBandGroups = 1024;
constexpr unsigned long long kBandDirect = 256;
MR_HD inline bool few_tiles(int32_t ntiles) { return ntiles <= kBandGroups; }
MR_HD inline int whole_bands(const unsigned long long* counters, const TileItems& r,
                             uint32_t parts_cap, int32_t ntiles, int tile_h) {
  int n = 1;
  if (counters[kDirect] < kBandDirect) return n;
  while (n < 8 && 2 * n <= tile_h && 2 * n * r.listed <= kBandGroups &&
         r.parts + 2 * n * r.listed <= (int64_t)ntiles + parts_cap)
    n *= 2;
  return n;
}

// Entries [first, end) of a tile's n direct ones that part `part` of the tile
// draws.
struct DirectShare {
  uint32_t first, end;
};
MR_HD inline DirectShare direct_share(uint32_t n, uint32_t part, uint32_t nparts) {
  if (nparts == 1) return {0, n};
  const uint32_t q = n / nparts, rest = n % nparts;
  const uint32_t first = part * q + (part < rest ? part : rest);
  return {first, first + q + (part < rest ? 1u : 0u)};
}

// Workgroup index b in [0, n) -> work index, a bijection under which each of
// the 8 XCDs (which receive workgroups round-robin) gets one contiguous range
// of work: neighbouring tiles share vertices, and each XCD has its own L2.
// XCD x = b % 8 owns q + (x < n % 8) items starting at x * q + min(x, n % 8).
MR_HD inline int64_t xcd_remap(int64_t b, int64_t n) {
  constexpr int64_t kXcds = 8;
  const int64_t q = n / kXcds, rem = n % kXcds;
  const int64_t x = b % kXcds, k = b / kXcds;
  return x * q + (x < rem ? x : rem) + k;
}

// The same with each XCD owning every eighth chunk of `kChunk` consecutive
// items (the rest past the last whole round of chunks as it comes): chunks of
// neighbouring pixels still share an L2, and work that changes over the frame
// (sky above, ground below) is dealt to all XCDs alike.  kChunk a power of
// two: a division by a variable costs every workgroup more than it gains.
template <uint32_t kChunk>
MR_HD inline uint32_t xcd_chunks(uint32_t b, uint32_t n) {
  constexpr uint32_t kXcds = 8, kRound = kXcds * kChunk;
  if (b >= n / kRound * kRound) return b;
  const uint32_t x = b % kXcds, k = b / kXcds;
  return (k / kChunk * kXcds + x) * kChunk + k % kChunk;
}

// Chunk of the raster's and shading's work, tiles or blocks.  Measured against
// one range per XCD: raster 108 -> 67 us on the textured 1080p terrain, 140 ->
// 113 at 4K, shading 36 -> 31 and 121 -> 100 us, 339 -> 319 on a batch of 48
// mixed frames; 4 and 64 alike on single frames, 64 slower on batches.
constexpr uint32_t kXcdChunk = 16;

// Per-tile counters are spread one per 64-byte line: the atomics of the
// binner then spread over all memory channels instead of a few.
constexpr int kCtrStride = 16;
constexpr int kCtrStride64 = kCtrStride / 2;  // the same spacing in 64-bit words

// The first half of the edge-checkpoint buffer is cut into this many
// segments, each with its own allocation counter (kCtrStride words apart):
// one shared counter would serialize every wavefront's atomic.  The second
// half is one segment, for wavefronts that need more than an eighth of a
// small one (few: their triangles are large); its entries and row tasks are
// counted by two counters in the gaps between the segments'.
constexpr int kCkptSegs = 64;
constexpr int kCkptBigEntries = kCtrStride / 2;               // word of ckpt_ctr
constexpr int kCkptBigRows = kCtrStride + kCtrStride / 2;

// Items over kDirectTiles tiles or more are not binned with the others but
// listed per job (kDirectCap of them or as many as the batch's scratch has
// room for; further ones are binned), and the tiles test that list.
// Binning costs a wavefront a step per 64 pairs, so one of 64 such triangles
// keeps counting and scattering when the rest of the GPU is done (3,000
// triangles over a 1080p frame, 1 M pairs: geometry 700 us, binning 1,230);
// testing costs every tile the list.  From 16 tiles: textured 1080p terrain
// with loose triangles 270 us a frame, 263 from 32, 310 (launch of the scan
// alone 60 us) from 8, 336 without lists; 48 mixed frames in a batch 911, 957,
// 898 and 990; 8.4 M-triangle 4K terrain 516, 544, 529 and 635 us of kernels.
constexpr int kDirectTiles = 16;
constexpr uint32_t kDirectCap = 4096;
constexpr uint32_t kDirectMin = 16;  // lists shorter than this are not used
constexpr uint32_t kDirectFlag = 0x80000000u;  // in BinItem::draw: listed, not binned

constexpr int kRegion = 128;       // item slots per geometry wavefront (64 x 2)
constexpr int kShadeBlock = 256;   // pixels per deferred-shading workgroup
constexpr int kShadeW = 16;        // shading block: kShadeW x kShadeH pixels
constexpr int kShadeH = kShadeBlock / kShadeW;
constexpr int kMaxLdsDraws = 256;  // draw-table entries cached in LDS

constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;    // tiles per thread in the tile-count scan ...
constexpr int kScanWide = 16384; // ... of more tiles than this; one up to it
constexpr uint32_t kNoWinner = 0xFFFFFFFFu;
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;
constexpr uint32_t kEmptyTile = 0xFFFFFFFEu;  // tile_heavy of a tile with no bin entry
// A raster work item (parts list entry .y) that covers a band of the tile's
// rows with all of its entries: bit 31 set, band count in bits 8-15, band
// index in bits 0-7.  Other entries are entry-range parts (the part index).
constexpr uint32_t kBandPart = 0x80000000u;
constexpr float kClearDepth = 1e11f;  // Renderer.cpp:116
// Job lookup hints: one per kHintSpan consecutive tiles or shading blocks.
constexpr int kHintShift = 6;
constexpr int kHintSpan = 1 << kHintShift;
constexpr int kMaxDim = 16384;        // max width / height

}  // namespace mr
