// Differentiable attribute interpolation over a rasterized frame.
//
// Forward: for every pixel of a single-sample triangle-id surface (the
// per-sample index of the last triangle written, 0xFFFFFFFF where none),
// interpolate C float channels of the triangle's three vertices with
// perspective-correct barycentrics at the pixel centre.  Backward: given
// dL/dout, accumulate dL/dattr and dL/dpos (clip x, y, w) of those vertices,
// with visibility fixed by the forward triangle ids (interior barycentric
// gradients only; no edge or occlusion terms).
//
// Barycentrics from homogeneous 2D coordinates: with q = (qx, qy, 1) the
// pixel centre in NDC and v_k = (x_k, y_k, w_k), the point of the triangle
// that projects to q has barycentrics b_k = c_k / (c_0 + c_1 + c_2),
// c_k = (v_{k+1} x v_{k+2}) . q.  Shearing by x' = x - qx w, y' = y - qy w
// (determinant 1) moves q to (0, 0, 1) and leaves
// c_k = x'_{k+1} y'_{k+2} - y'_{k+1} x'_{k+2}.  All of it is evaluated in
// FP64 (cheap on CDNA4 and well conditioned for sub-pixel triangles); the
// backward sums each triangle's per-pixel gradient terms in FP64 and adds
// the sums to the FP32 outputs with atomics.
#include <algorithm>

#include "cr_device.h"

namespace crhip {

struct Bary {
  double b[3];
  double xs[3], ys[3];          // sheared vertex coordinates x', y'
  double sum;
  bool ok;                      // false for a degenerate projected triangle (sum == 0)
};

__device__ __forceinline__ void baryOf(const float4 p[3], double qx, double qy, Bary& B) {
#pragma unroll
  for (int k = 0; k < 3; k++) {
    B.xs[k] = (double)p[k].x - qx * (double)p[k].w;
    B.ys[k] = (double)p[k].y - qy * (double)p[k].w;
  }
  double c[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int k1 = (k + 1) % 3, k2 = (k + 2) % 3;
    c[k] = B.xs[k1] * B.ys[k2] - B.ys[k1] * B.xs[k2];
  }
  B.sum = c[0] + c[1] + c[2];
  B.ok = B.sum != 0.0;
  const double r = B.ok ? 1.0 / B.sum : 0.0;
#pragma unroll
  for (int k = 0; k < 3; k++) B.b[k] = c[k] * r;
}

__device__ __forceinline__ void baryAt(const float4* __restrict__ pos, const int32_t i[3], double qx, double qy,
                                       Bary& B) {
  const float4 p[3] = {pos[i[0]], pos[i[1]], pos[i[2]]};
  baryOf(p, qx, qy, B);
}

// Set bits of `mask` below this lane (v_mbcnt).
__device__ __forceinline__ uint32_t rankBelow(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// The views of one launch, in the kernel's arguments.
template <int N>
struct InterpTable {
  InterpView v[N];
};

// Looks up pixel (x, y) of the id surface; fills the vertex indices.
// Returns false for background or out-of-range ids / indices.
__device__ __forceinline__ bool pixelTriangle(const InterpGeom& G, const InterpView& V, int x, int y, uint32_t& t,
                                              int32_t i[3]) {
  t = V.ids[(size_t)y * G.texW + x];
  if (t >= (uint32_t)V.numTris) return false;
  const int3 v = reinterpret_cast<const int3*>(V.tris)[t];
  i[0] = v.x; i[1] = v.y; i[2] = v.z;
  for (int k = 0; k < 3; k++)
    if (i[k] < 0 || (int64_t)i[k] >= V.numVertices) return false;
  return true;
}

constexpr int kFwdThreads = 256;

// One lane per pixel, one W x (256 / W) pixel tile per workgroup, one grid layer
// per view.  Bound by the gathers of vertices where triangles are small: a
// tile's pixels share them in the CU's cache, a row's hardly do.  16 views of
// 200k triangles, 512x512, 8 channels: 97 us in rows of 256 pixels, 90 in 64 x 4,
// 83 in 32 x 8, 82 in 16 x 16.  Bound by the stores where they are large: a
// row's are longer runs.  1024x1024, 8k triangles, 24 channels: 46 us in rows, 56 in
// 64 x 4, 55 in 32 x 8, 62 in 16 x 16.
// vec4: C % 4 == 0 and attr / out 16-byte aligned, so channels move as
// float4.
template <int N, int W>
__global__ void __launch_bounds__(kFwdThreads) interpForwardKernel(const InterpGeom G, const InterpTable<N> T) {
  const InterpView& V = T.v[N == 1 ? 0 : blockIdx.z];
  const int x = (int)(blockIdx.x * W + threadIdx.x % W);
  const int y = (int)(blockIdx.y * (kFwdThreads / W) + threadIdx.x / W);
  if (x >= G.width || y >= G.height) return;
  const int64_t p = (int64_t)y * G.width + x;
  const int C = G.numChannels;
  const bool vec4 = V.vec4 != 0;
  float* __restrict__ o = V.out + p * C;
  int32_t* __restrict__ triImage = V.triImage;
  uint32_t t;
  int32_t i[3];
  if (!pixelTriangle(G, V, x, y, t, i)) {
    if (vec4) {
      for (int c = 0; c < C; c += 4) *reinterpret_cast<float4*>(o + c) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    } else {
      for (int c = 0; c < C; c++) o[c] = 0.0f;
    }
    if (triImage) triImage[p] = -1;
    return;
  }
  const double qx = (2.0 * x + 1.0) / G.width - 1.0, qy = (2.0 * y + 1.0) / G.height - 1.0;
  Bary B;
  baryAt(reinterpret_cast<const float4*>(V.pos), i, qx, qy, B);
  const float* __restrict__ a0 = V.attr + (int64_t)i[0] * C;
  const float* __restrict__ a1 = V.attr + (int64_t)i[1] * C;
  const float* __restrict__ a2 = V.attr + (int64_t)i[2] * C;
  if (vec4) {
    for (int c = 0; c < C; c += 4) {
      const float4 u = *reinterpret_cast<const float4*>(a0 + c), v = *reinterpret_cast<const float4*>(a1 + c),
                   w = *reinterpret_cast<const float4*>(a2 + c);
      *reinterpret_cast<float4*>(o + c) = make_float4((float)(B.b[0] * u.x + B.b[1] * v.x + B.b[2] * w.x),
                                                      (float)(B.b[0] * u.y + B.b[1] * v.y + B.b[2] * w.y),
                                                      (float)(B.b[0] * u.z + B.b[1] * v.z + B.b[2] * w.z),
                                                      (float)(B.b[0] * u.w + B.b[1] * v.w + B.b[2] * w.w));
    }
  } else {
    for (int c = 0; c < C; c++) o[c] = (float)(B.b[0] * a0[c] + B.b[1] * a1[c] + B.b[2] * a2[c]);
  }
  if (triImage) triImage[p] = (int32_t)t;
}

// Backward over 16x16-pixel tiles, one 256-lane workgroup each, one lane per
// pixel.  The lane evaluates its pixel's barycentrics, dL/db_k = sum_c g_c
// a_k,c, dL/dc_j = (dL/db_j - sum_k b_k dL/db_k) / (c_0 + c_1 + c_2), and from
// there through c_k = x'_{k+1} y'_{k+2} - y'_{k+1} x'_{k+2} and the shear
// x' = x - qx w, y' = y - qy w the gradient of each corner's clip x, y, w.
//
// The tile's terms are then summed per vertex:
//  - triangles: a hash table of triangle ids in LDS gives every pixel its
//    triangle's slot; a bit mask per (slot, wave) gives it its rank among the
//    triangle's pixels;
//  - vertices: the (triangle, corner) pairs go through a second table keyed by
//    vertex, which gives every pair a stretch of its vertex's list, as long as
//    the triangle has pixels; each pixel enters itself in its three lists;
//  - sums: one lane per (vertex, channel or x/y/w) sums the vertex's list in
//    FP64 and adds the total to the output gradient with one FP32 atomic.  The
//    tables keep consecutive ids in consecutive slots, so consecutive lanes
//    mostly reach consecutive addresses, which device-scope atomics serve
//    several times faster than scattered ones.
// A vertex receives one addition per tile that sees it, in whatever order the
// atomics land, so the last bits of a gradient can differ between runs.  All
// views of a call are one launch.
//
// What bounds it: for one view the chain of dependent loads (id, indices,
// positions and attributes: half of a workgroup's 40k cycles at 512x512) and
// of LDS steps; five workgroups fit a CU.  Measured against one that sorted
// the tile's pixels by triangle (36 barriers), loaded channel by channel and
// added per (triangle, corner): 512x512, 200k loose triangles, 8 channels
// 59.6 -> 28.2 us a view; 400x300 mesh, 40k triangles, 3 channels 18.7 ->
// 15.4 us; 640x480 mesh, 100k triangles, 12 channels, reproducible sums 167 ->
// 37.6 us (fewer and mostly single atomics).  One wave per 8x8 tile took 36 us
// for the first and rounds to FP32 more often.
constexpr int kBwdTile = 16;
constexpr int kBwdThreads = kBwdTile * kBwdTile;
constexpr int kBwdWaves = kBwdThreads / 64;
constexpr int kBwdChannels = 8;                // channels staged in LDS at a time
constexpr int kBwdPairs = 3 * kBwdThreads;     // (triangle, corner) pairs a tile can hold
constexpr int kTriSlots = 2 * kBwdThreads;     // hash tables: at most half and three quarters full
constexpr int kVertSlots = 4 * kBwdThreads;
constexpr uint32_t kNoKey = 0xFFFFFFFFu;       // (ids and vertex indices are below 2^31)

// Bit-reproducible accumulation: a value is a 128-bit two's-complement
// fixed-point number with 2^-64 resolution.  Each (tile, vertex) FP64 sum,
// whose terms are added in a fixed order, is converted once (magnitude
// truncated to the resolution, |x| < 2^63) and added to the vertex's two words
// (low, high) with integer atomics: the low word, then the high word with the
// low word's carry, only when that is not zero.  Integer addition is
// associative, so the total does not depend on the order the atomics land in.  The low word starts at 2^63 (kFixedBias): a small
// addition of either sign then rarely carries out of or borrows from it, so
// that most additions are one atomic.
constexpr unsigned long long kFixedBias = 1ull << 63;
__device__ __forceinline__ void fixedAdd(unsigned long long* __restrict__ acc, int64_t idx, double s) {
  const bool neg = s < 0.0;
  const double m = fmin(fabs(s) * 18446744073709551616.0, 1.7014118346046923e38);   // |s| 2^64, below 2^127
  const double mh = floor(m * 5.421010862427522e-20);                                // m / 2^64
  const double ml = m - mh * 18446744073709551616.0;                                 // exact
  uint64_t lo = (uint64_t)ml, hi = (uint64_t)mh;
  if (neg) {
    lo = ~lo + 1u;
    hi = ~hi + (lo == 0u ? 1u : 0u);
  }
  unsigned long long* w = acc + 2 * idx;
  const unsigned long long old = atomicAdd(w, (unsigned long long)lo);
  const uint64_t h = hi + ((old + lo) < old ? 1u : 0u);
  if (h != 0u) atomicAdd(w + 1, (unsigned long long)h);
}

// One lane's load of up to kBwdChannels floats; those at n and beyond are 0.
// vec4: n is a multiple of 4 and p 16-byte aligned.
__device__ __forceinline__ void loadChannels(const float* __restrict__ p, int n, bool vec4, float v[kBwdChannels]) {
  if (vec4) {
#pragma unroll
    for (int c = 0; c < kBwdChannels; c += 4) {
      const float4 f = c < n ? *reinterpret_cast<const float4*>(p + c) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      v[c] = f.x; v[c + 1] = f.y; v[c + 2] = f.z; v[c + 3] = f.w;
    }
  } else {
#pragma unroll
    for (int c = 0; c < kBwdChannels; c++) v[c] = c < n ? p[c] : 0.0f;
  }
}

// The slot of `key` in an open-addressing table of `slots` keys (a power of
// two) that starts out all kNoKey.  Consecutive keys start at consecutive
// slots; the multiple of the key's high part keeps keys that are a power of
// two apart (the rows of a grid) from starting at the same one.  Rows that do
// fall on one another are taken apart by jumps of 1, 3, 6, ... steps (which reach
// every slot when the step is odd), the step shared by 32 consecutive keys, so
// that they stay together (the high bits of a product with 2^32 over the golden
// ratio).  In steps of one the rows queued up behind each other, and with jumps of
// one step some pairs of rows still did: 512x512, meshes of 988x988, 1000x1000
// and 717x717 vertices, 3 channels 169, 145 and 55 us, 60, 63 and 35, now 59, 61 and
// 34; 256x256, 257x257 17, 26 and 18.
template <int SLOTS>
__device__ __forceinline__ uint32_t hashSlot(uint32_t* table, uint32_t key) {
  uint32_t h = (key + (key / SLOTS) * 37u) & (SLOTS - 1);
  const uint32_t step = ((key >> 5) * 0x9E3779B1u >> 20) | 1u;
  for (uint32_t jump = step;; jump += step) {
    const uint32_t old = atomicCAS(&table[h], kNoKey, key);
    if (old == kNoKey || old == key) return h;
    h = (h + jump) & (SLOTS - 1);
  }
}

// Exclusive sum over the workgroup (kBwdThreads lanes): one barrier, plus
// one before `sums` may be written again.
__device__ __forceinline__ uint32_t bwdScan(uint32_t v, uint32_t* sums, uint32_t& total) {
  const int wave = (int)(threadIdx.x >> 6);
  const uint32_t x = waveScan(v);
  if ((threadIdx.x & 63) == 63) sums[wave] = x;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kBwdWaves; w++) {
    const uint32_t n = sums[w];
    before += w < wave ? n : 0u;
    total += n;
  }
  return before + x - v;
}

// DET: accumulate into the view's fixed-point words (positions V*4 values,
// then attributes V*C) instead of FP32 atomics on the outputs.
template <bool DET, int N>
__global__ void __launch_bounds__(kBwdThreads) interpBackwardKernel(const InterpGeom G, const InterpTable<N> T,
                                                                    const int tilesX) {
  // Rows of the terms are one word longer than the tile has pixels, so that
  // lanes that differ in the corner or channel read different banks.
  constexpr int kRow = kBwdThreads + 1;
  // One area, several uses in turn: the triangle table (a pixel mask per slot
  // and wave, then the keys); the vertex table (keys, counts) and the pairs'
  // vertices; the barycentrics [corner] and dL/dout [channel] of the pixels;
  // dL/d(x, y, w) [corner * 3 + comp] of the pixels.
  constexpr size_t kTableBytes = kTriSlots * 4 + (size_t)kTriSlots * kBwdWaves * 8;
  constexpr size_t kTermBytes = 9 * kRow * sizeof(double);
  static_assert(kVertSlots * 12 + kBwdPairs * 4 <= (size_t)kTriSlots * kBwdWaves * 8 && 3 * kRow * 8 + kBwdChannels * kRow * 4 <= kTermBytes, "uses fit");
  __shared__ __attribute__((aligned(16))) uint8_t area[kTermBytes > kTableBytes ? kTermBytes : kTableBytes];
  uint64_t* const triMask = reinterpret_cast<uint64_t*>(area);
  uint32_t* const triKey = reinterpret_cast<uint32_t*>(area + (size_t)kTriSlots * kBwdWaves * 8);
  uint32_t* const vertKey = reinterpret_cast<uint32_t*>(area);
  uint32_t* const vertCount = vertKey + kVertSlots;
  uint32_t* const pairVertex = vertCount + kVertSlots;
  uint32_t* const vertPairs = pairVertex + kBwdPairs;   // DET: the slot's last entered pair (chained in sList)
  double* const sTerm = reinterpret_cast<double*>(area);
  double* const sB = sTerm;
  float* const sG = reinterpret_cast<float*>(sTerm + 3 * kRow);
  __shared__ uint16_t sLength[kBwdThreads];    // per triangle: its pixels in the tile
  __shared__ uint16_t sPair[kBwdPairs];        // per (triangle, corner): its place in the lists
  __shared__ uint16_t sList[kBwdPairs];        // the lists, vertex by vertex: pixel | corner << 8
  __shared__ int32_t sVertex[kBwdPairs];       // per listed vertex: its index
  __shared__ uint16_t sFirst[kBwdPairs + 1];   // and its list's start; then the end
  __shared__ uint32_t sums[2][kBwdWaves];

  const InterpView& V = T.v[N == 1 ? 0 : blockIdx.y];
  // Tiles in raster order: bands of tiles per XCD take the same time (16 views
  // 264 against 263 us), and a large triangle's partial sums, small at its ends,
  // then meet in an order that rounds worse (attribute gradients of 200k
  // triangles: 3.93e-8 off against 3.87e-8).
  const int tile = (int)blockIdx.x;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int C = G.numChannels;
  const bool vec4 = V.vec4 != 0;
  const int x = (tile % tilesX) * kBwdTile + (tid & (kBwdTile - 1));
  const int y = (tile / tilesX) * kBwdTile + tid / kBwdTile;
  const bool inside = x < G.width && y < G.height;
  const int64_t p = inside ? (int64_t)y * G.width + x : 0;

  // ---- the lane's pixel: every load that it can issue ---------------------------
  const int32_t t = inside ? V.triImage[p] : -1;
  float g[kBwdChannels];
  loadChannels(V.gradOut + p * C, min(C, kBwdChannels), vec4, g);
#pragma unroll
  for (int o = 0; o < (int)(kTableBytes / 16); o += kBwdThreads) {
    const int at = o + tid;
    const uint32_t f = at * 16 >= (int)((size_t)kTriSlots * kBwdWaves * 8) ? kNoKey : 0u;
    if (at < (int)(kTableBytes / 16)) reinterpret_cast<uint4*>(area)[at] = make_uint4(f, f, f, f);
  }
  bool ok = t >= 0 && t < V.numTris;
  int32_t i[3] = {0, 0, 0};
  if (ok) {
    const int3 v = reinterpret_cast<const int3*>(V.tris)[t];
    i[0] = v.x; i[1] = v.y; i[2] = v.z;
  }
#pragma unroll
  for (int k = 0; k < 3; k++) ok = ok && i[k] >= 0 && (int64_t)i[k] < V.numVertices;
  const float4* __restrict__ pos = reinterpret_cast<const float4*>(V.pos);
  float4 pv[3];
  double dB[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 3; k++) pv[k] = ok ? pos[i[k]] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int c0 = 0; c0 < C; c0 += kBwdChannels) {
    const int n = min(C - c0, kBwdChannels);
    float a[3][kBwdChannels], gc[kBwdChannels];
#pragma unroll
    for (int k = 0; k < 3; k++) loadChannels(V.attr + (int64_t)i[k] * C + c0, ok ? n : 0, vec4, a[k]);
    if (c0 > 0) loadChannels(V.gradOut + p * C + c0, n, vec4, gc);
#pragma unroll
    for (int c = 0; c < kBwdChannels; c++) {
      if (c < n) {
        const double d = (double)(c0 > 0 ? gc[c] : g[c]);
#pragma unroll
        for (int k = 0; k < 3; k++) dB[k] += d * (double)a[k][c];
      }
    }
  }
  const double qx = (2.0 * x + 1.0) / G.width - 1.0, qy = (2.0 * y + 1.0) / G.height - 1.0;
  double b[3], dxs[3] = {0.0, 0.0, 0.0}, dys[3] = {0.0, 0.0, 0.0};
  {
    Bary B;
    baryOf(pv, qx, qy, B);
    ok = ok && B.ok;
    const double mean = B.b[0] * dB[0] + B.b[1] * dB[1] + B.b[2] * dB[2];
    const double rs = 1.0 / B.sum;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const double dc = (dB[k] - mean) * rs;
      const int k1 = (k + 1) % 3, k2 = (k + 2) % 3;
      dxs[k1] += dc * B.ys[k2];
      dys[k1] -= dc * B.xs[k2];
      dxs[k2] -= dc * B.ys[k1];
      dys[k2] += dc * B.xs[k1];
      b[k] = B.b[k];
    }
  }

  // ---- triangles ---------------------------------------------------------------------
  __syncthreads();
  uint32_t slot = 0;
  if (ok) {
    slot = hashSlot<kTriSlots>(triKey, (uint32_t)t);
    atomicOr((unsigned long long*)&triMask[slot * kBwdWaves + wave], 1ull << lane);
  }
  __syncthreads();
  uint32_t rank = 0, length = 0;
  if (ok) {
#pragma unroll
    for (int w = 0; w < kBwdWaves; w++) {
      const uint64_t m = triMask[slot * kBwdWaves + w];
      const uint32_t n = (uint32_t)__popcll(m);
      rank += w < wave ? n : w == wave ? rankBelow(m) : 0u;
      length += n;
    }
  }
  // The first pixel of each triangle stands for it: triangles are numbered in
  // pixel order.
  const bool first = ok && rank == 0;
  const uint64_t fm = __ballot(first);
  if (lane == 0) sums[0][wave] = (uint32_t)__popcll(fm);
  __syncthreads();                             // (every lane has read its masks)
  int numTris = 0;
  uint32_t tri = rankBelow(fm);
#pragma unroll
  for (int w = 0; w < kBwdWaves; w++) {
    const uint32_t n = sums[0][w];
    tri += w < wave ? n : 0u;
    numTris += (int)n;
  }
  if (numTris == 0) return;
#pragma unroll
  for (int o = 0; o < 2 * kVertSlots / 4; o += kBwdThreads) {
    const uint32_t f = o < kVertSlots / 4 ? kNoKey : 0u;
    reinterpret_cast<uint4*>(area)[o + tid] = make_uint4(f, f, f, f);
  }
  if (DET) reinterpret_cast<uint4*>(vertPairs)[tid] = make_uint4(kNoKey, kNoKey, kNoKey, kNoKey);
  if (first) {
    triKey[slot] = tri;                        // the key's place takes the number
    sLength[tri] = (uint16_t)length;
    pairVertex[3 * tri] = (uint32_t)i[0];
    pairVertex[3 * tri + 1] = (uint32_t)i[1];
    pairVertex[3 * tri + 2] = (uint32_t)i[2];
  }
  __syncthreads();

  // ---- vertices ----------------------------------------------------------------------
  if (ok) tri = triKey[slot];
  const int numPairs = 3 * numTris;
  uint32_t pairSlot[3], pairAt[3];
#pragma unroll
  for (int o = 0; o < 3; o++) {
    const int e = o * kBwdThreads + tid;
    if (e < numPairs) {
      pairSlot[o] = hashSlot<kVertSlots>(vertKey, pairVertex[e]);
      pairAt[o] = atomicAdd(&vertCount[pairSlot[o]], (uint32_t)sLength[e / 3]);
      if (DET) sList[e] = (uint16_t)atomicExch(&vertPairs[pairSlot[o]], (uint32_t)e);
    }
  }
  __syncthreads();
  // The pairs of a vertex follow one another as their additions landed; for
  // sums in a fixed order, by number.
  if (DET) {
#pragma unroll
    for (int o = 0; o < 3; o++) {
      const int e = o * kBwdThreads + tid;
      if (e < numPairs) {
        pairAt[o] = 0;
        for (uint32_t c = vertPairs[pairSlot[o]]; c < (uint32_t)kBwdPairs; c = sList[c])   // (0xFFFF.. ends it)
          if ((int)c < e) pairAt[o] += sLength[c / 3];
      }
    }
  }
  // Four slots per lane: list entries, and vertices << 16.
  const uint4 cnt = reinterpret_cast<const uint4*>(vertCount)[tid];
  const uint4 key = reinterpret_cast<const uint4*>(vertKey)[tid];
  auto packed = [](uint32_t n) { return n | (n ? 1u << 16 : 0u); };
  uint32_t total;
  uint4 at;
  at.x = bwdScan(packed(cnt.x) + packed(cnt.y) + packed(cnt.z) + packed(cnt.w), sums[1], total);
  at.y = at.x + packed(cnt.x);
  at.z = at.y + packed(cnt.y);
  at.w = at.z + packed(cnt.z);
  const int numVerts = (int)(total >> 16);
  auto list = [&](uint32_t n, uint32_t k, uint32_t w) {
    if (n == 0) return;
    sVertex[w >> 16] = (int32_t)k;
    sFirst[w >> 16] = (uint16_t)(w & 0xFFFFu);
  };
  list(cnt.x, key.x, at.x);
  list(cnt.y, key.y, at.y);
  list(cnt.z, key.z, at.z);
  list(cnt.w, key.w, at.w);
  if (tid == 0) sFirst[numVerts] = (uint16_t)(total & 0xFFFFu);
  reinterpret_cast<uint4*>(vertCount)[tid] = at;
  __syncthreads();
#pragma unroll
  for (int o = 0; o < 3; o++) {
    const int e = o * kBwdThreads + tid;
    if (e < numPairs) sPair[e] = (uint16_t)((vertCount[pairSlot[o]] & 0xFFFFu) + pairAt[o]);
  }
  __syncthreads();
  if (ok) {
#pragma unroll
    for (int k = 0; k < 3; k++)
      sList[sPair[3 * tri + k] + rank] =
          (uint16_t)((uint32_t)tid | (uint32_t)k << 8);
  }

  // Calls f(vertex, column) for every (listed vertex, column) of `cols`,
  // stepped without a division.
  auto forEntries = [&](int cols, auto&& f) {
    const int stepV = kBwdThreads / cols, stepC = kBwdThreads - stepV * cols;
    int vi = tid / cols, col = tid - vi * cols;
    while (vi < numVerts) {
      f(vi, col);
      vi += stepV;
      col += stepC;
      if (col >= cols) {
        col -= cols;
        vi++;
      }
    }
  };
  // Sums term(corner, pixel) over vertex vi's list and adds the total to
  // value o (of the fixed-point words) or *out.  Four terms are fetched at a
  // time, and added in list order.
  auto sumVertex = [&](int vi, int64_t o, float* out, auto&& term) {
    const int end = sFirst[vi + 1];
    int e = sFirst[vi];
    double s = 0.0;
    for (; e + 4 <= end; e += 4) {
      uint32_t code[4];
      double v[4];
#pragma unroll
      for (int q = 0; q < 4; q++) code[q] = sList[e + q];
#pragma unroll
      for (int q = 0; q < 4; q++) v[q] = term(code[q] >> 8, code[q] & 255u);
#pragma unroll
      for (int q = 0; q < 4; q++) s += v[q];
    }
    for (; e < end; e++) {
      const uint32_t code = sList[e];
      s += term(code >> 8, code & 255u);
    }
    if (s != 0.0) {
      if (DET) fixedAdd(V.acc, o, s);
      else unsafeAtomicAdd(out, (float)s);
    }
  };

  // ---- attribute gradients sum_q b_k g_c, kBwdChannels channels at a time ------------
#pragma unroll
  for (int k = 0; k < 3; k++) sB[k * kRow + tid] = b[k];
  for (int c0 = 0; c0 < C; c0 += kBwdChannels) {
    const int n = min(C - c0, kBwdChannels);
    if (c0 > 0) {
      loadChannels(V.gradOut + p * C + c0, n, vec4, g);
      __syncthreads();                         // the last channels' sums are done
    }
#pragma unroll
    for (int c = 0; c < kBwdChannels; c++)
      if (c < n) sG[c * kRow + tid] = g[c];
    __syncthreads();
    forEntries(n, [&](int vi, int c) {
      const float* w = sG + c * kRow;
      const int64_t o = (int64_t)sVertex[vi] * C + c0 + c;
      sumVertex(vi, V.numVertices * 4 + o, V.gradAttr + o,
                [&](uint32_t k, uint32_t q) { return sB[k * kRow + q] * (double)w[q]; });
    });
  }

  // ---- position gradients ----------------------------------------------------------
  __syncthreads();                             // the attribute sums are done with the area
#pragma unroll
  for (int k = 0; k < 3; k++) {
    sTerm[(3 * k) * kRow + tid] = dxs[k];
    sTerm[(3 * k + 1) * kRow + tid] = dys[k];
    sTerm[(3 * k + 2) * kRow + tid] = -qx * dxs[k] - qy * dys[k];
  }
  __syncthreads();
  forEntries(3, [&](int vi, int comp) {
    const int64_t o = (int64_t)sVertex[vi] * 4 + (comp == 2 ? 3 : comp);
    sumVertex(vi, o, V.gradPos + o, [&](uint32_t k, uint32_t q) { return sTerm[(3 * k + comp) * kRow + q]; });
  });
}

// Zeroes [0, n) of p: up to three floats until a 16-byte boundary, then
// 16-byte stores, then the tail; `lane` and `lanes` stride the grid.
__device__ __forceinline__ void zeroFloats(float* __restrict__ p, int64_t n, int64_t lane, int64_t lanes) {
  const int64_t head = min<int64_t>(n, (int64_t)(((16u - ((uintptr_t)p & 15u)) & 15u) >> 2));
  if (lane < head) p[lane] = 0.0f;
  float4* __restrict__ q = reinterpret_cast<float4*>(p + head);
  const int64_t n4 = (n - head) >> 2;
  for (int64_t k = lane; k < n4; k += lanes) q[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const int64_t tail = head + (n4 << 2);
  if (lane < n - tail) p[tail + lane] = 0.0f;
}

// Zeroes every view's gradients (4-byte aligned).
template <int N>
__global__ void __launch_bounds__(256) zeroGradsKernel(const InterpTable<N> T, int numChannels) {
  const InterpView& V = T.v[N == 1 ? 0 : blockIdx.y];
  const int64_t lane = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, lanes = (int64_t)gridDim.x * blockDim.x;
  zeroFloats(V.gradPos, V.numVertices * 4, lane, lanes);
  zeroFloats(V.gradAttr, V.numVertices * numChannels, lane, lanes);
}

static int gridFor(int64_t n) { return (int)std::min<int64_t>((n + 255) / 256, 1 << 20); }

// Clears every view's fixed-point words: low words to kFixedBias, high to 0.
template <int N>
__global__ void __launch_bounds__(256) clearFixedKernel(const InterpTable<N> T, int numChannels) {
  const InterpView& V = T.v[N == 1 ? 0 : blockIdx.y];
  const int64_t n = V.numVertices * (4 + (int64_t)numChannels);
  ulonglong2* w = reinterpret_cast<ulonglong2*>(V.acc);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    w[k] = make_ulonglong2(kFixedBias, 0ull);
}

// Rounds the fixed-point totals to FP32: positions (V*4), then attributes.
template <int N>
__global__ void __launch_bounds__(256) fixedToFloatKernel(const InterpTable<N> T, int numChannels) {
  const InterpView& V = T.v[N == 1 ? 0 : blockIdx.y];
  const int64_t nPos = V.numVertices * 4, n = nPos + V.numVertices * numChannels;
  const ulonglong2* w = reinterpret_cast<const ulonglong2*>(V.acc);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
    const ulonglong2 q = w[k];
    const double v = (double)(int64_t)q.y + (double)(int64_t)(q.x - kFixedBias) * 5.421010862427522e-20;
    if (k < nPos) V.gradPos[k] = (float)v;
    else V.gradAttr[k - nPos] = (float)v;
  }
}

template <int W, int N>
static void forwardTiles(const InterpGeom& G, const InterpTable<N>& T, int n, hipStream_t stream) {
  constexpr int H = kFwdThreads / W;
  hipLaunchKernelGGL((interpForwardKernel<N, W>), dim3((unsigned)((G.width + W - 1) / W),
                     (unsigned)((G.height + H - 1) / H), (unsigned)n), dim3(kFwdThreads), 0, stream, G, T);
}

template <int N>
static void forwardViews(const InterpGeom& G, const InterpTable<N>& T, int n, hipStream_t stream) {
  // Tiles from one triangle in four pixels on.  1024x1024, rows against 32 x 8: a
  // mesh of 512x512 vertices (a triangle in two pixels), 1 channel 10.1 and 10.0
  // us, 16 34.8 and 29.9, 20 54.9 and 48.7; 300x300 (one in six), 24 channels 53.7 and
  // 59.3; 65x65, 1 channel 10.3 and 10.4, 16 25.3 and 26.2, 20 33.3 and 38.9.
  int64_t tris = 0;
  for (int v = 0; v < n; v++) tris += T.v[v].numTris;
  if (tris * 4 >= (int64_t)G.width * G.height * n) forwardTiles<32>(G, T, n, stream);
  else forwardTiles<256>(G, T, n, stream);
}

template <int N>
static void backwardViews(const InterpGeom& G, const InterpTable<N>& T, int n, hipStream_t stream) {
  const int C = G.numChannels;
  int64_t most = 0;
  bool work = false;
  for (int v = 0; v < n; v++) {
    most = std::max(most, T.v[v].numVertices);
    work = work || T.v[v].numTris > 0;
  }
  if (most == 0) return;                       // no view has a gradient to write
  const bool det = T.v[0].acc != nullptr;
  const int64_t values = most * (4 + (int64_t)C);
  const int tilesX = (G.width + kBwdTile - 1) / kBwdTile, tiles = tilesX * ((G.height + kBwdTile - 1) / kBwdTile);
  const dim3 grid((unsigned)tiles, (unsigned)n);
  if (!det) {
    hipLaunchKernelGGL((zeroGradsKernel<N>), dim3(gridFor((values + 3) / 4), (unsigned)n), dim3(256), 0, stream, T, C);
    if (work) hipLaunchKernelGGL((interpBackwardKernel<false, N>), grid, dim3(kBwdThreads), 0, stream, G, T, tilesX);
    return;
  }
  hipLaunchKernelGGL((clearFixedKernel<N>), dim3(gridFor(values), (unsigned)n), dim3(256), 0, stream, T, C);
  if (work) hipLaunchKernelGGL((interpBackwardKernel<true, N>), grid, dim3(kBwdThreads), 0, stream, G, T, tilesX);
  hipLaunchKernelGGL((fixedToFloatKernel<N>), dim3(gridFor(values), (unsigned)n), dim3(256), 0, stream, T, C);
}

// Runs `f` over the views, kInterpViews to a launch (one view: a table of one).
template <class F1, class FN>
static void overViews(const InterpView* views, int numViews, const void* (*moved)(const InterpView&), int numChannels,
                      F1&& one, FN&& many) {
  for (int v0 = 0; v0 < numViews; v0 += kInterpViews) {
    const int n = std::min(numViews - v0, kInterpViews);
    auto set = [&](InterpView& d, const InterpView& v) {
      d = v;
      d.vec4 = numChannels % 4 == 0 && ((uintptr_t)v.attr & 15) == 0 && ((uintptr_t)moved(v) & 15) == 0;
    };
    if (n == 1) {
      InterpTable<1> T;
      set(T.v[0], views[v0]);
      one(T);
    } else {
      InterpTable<kInterpViews> T = {};
      for (int v = 0; v < n; v++) set(T.v[v], views[v0 + v]);
      many(T, n);
    }
  }
}

void launchInterpForward(const InterpGeom& G, const InterpView* views, int numViews, hipStream_t stream) {
  if (G.width <= 0 || G.height <= 0) return;
  overViews(views, numViews, [](const InterpView& v) -> const void* { return v.out; }, G.numChannels,
            [&](const InterpTable<1>& T) { forwardViews(G, T, 1, stream); },
            [&](const InterpTable<kInterpViews>& T, int n) { forwardViews(G, T, n, stream); });
}

void launchInterpBackward(const InterpGeom& G, const InterpView* views, int numViews, hipStream_t stream) {
  if (G.width <= 0 || G.height <= 0) return;
  overViews(views, numViews, [](const InterpView& v) -> const void* { return v.gradOut; }, G.numChannels,
            [&](const InterpTable<1>& T) { backwardViews(G, T, 1, stream); },
            [&](const InterpTable<kInterpViews>& T, int n) { backwardViews(G, T, n, stream); });
}

}  // namespace crhip
