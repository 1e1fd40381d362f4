// Stage 1: triangle setup, one lane per input triangle.
//
// Follows triangleSetupImpl (cudaraster/cuda/TriangleSetup.inl:219-417):
// frustum cull, fast path (snap + guard band), or barycentric clip against
// the frustum fanned into subtriangles; backface and between-samples culls;
// plane equations for depth and perspective-correct barycentrics.  Output is
// the per-triangle subtriangle count, the 16-byte header and 64-byte data
// record per subtriangle slot.  Clipped triangles with >= 2 visible
// subtriangles take consecutive slots from a device counter (slots beyond
// numTris), their source index goes to subtriTri, and misc holds the base.
//
// The clip polygon lives in registers, one vertex per lane of the wave, or,
// where several of a wave's triangles are clipped, in scratch memory per lane,
// instead of the reference's per-thread shared-memory array.
#include "cr_device.h"

namespace crhip {

struct I2 { int32_t x, y; };

// Util.inl:65-91 (GPU plane-equation setup).
__device__ __forceinline__ void setupPleq(float vx, float vy, float vz, int32_t v0x, int32_t v0y,
                                          int32_t d1x, int32_t d1y, int32_t d2x, int32_t d2y,
                                          float areaRcp, int samplesLog2, uint32_t out[3]) {
  float mx = fmaxf(fmaxf(vx, vy), vz);
  int32_t sh = asr32((int32_t)__float_as_uint(mx), 23) - (127 + 22);
  sh = min(max(sh, 0), 8);
  int32_t t0 = (int32_t)(cvtRziSatU32(vx) >> sh);
  int32_t t1 = wsub((int32_t)(cvtRziSatU32(vy) >> sh), t0);
  int32_t t2 = wsub((int32_t)(cvtRziSatU32(vz) >> sh), t0);

  uint32_t rcpMant = (__float_as_uint(areaRcp) & 0x007FFFFFu) | 0x00800000u;
  int32_t rcpShift = (23 + 127) - asr32((int32_t)__float_as_uint(areaRcp), 23);

  int64_t xc = wmul64((int64_t)t1 * d2y - (int64_t)t2 * d1y, (int64_t)rcpMant);
  int64_t yc = wmul64((int64_t)t2 * d1x - (int64_t)t1 * d2x, (int64_t)rcpMant);
  int shp = rcpShift - (sh + kSubpixelLog2 - samplesLog2);
  out[0] = (uint32_t)asr64(xc, shp);
  out[1] = (uint32_t)asr64(yc, shp);

  int sc = kSubpixelLog2 - samplesLog2;
  int32_t minx = min(min(d1x, d2x), 0), maxx = max(max(d1x, d2x), 0);
  int32_t miny = min(min(d1y, d2y), 0), maxy = max(max(d1y, d2y), 0);
  int32_t centerX = asr32(wadd(wadd(wmul(v0x, 2), minx), maxx), sc + 1);
  int32_t centerY = asr32(wadd(wadd(wmul(v0y, 2), miny), maxy), sc + 1);
  int32_t vcx = wsub(v0x, (int32_t)((uint32_t)centerX << sc));
  int32_t vcy = wsub(v0y, (int32_t)((uint32_t)centerY << sc));

  uint32_t z = (uint32_t)t0 << sh;
  int64_t cross = (int64_t)((uint64_t)wmul64(asr64(xc, 13), vcx) + (uint64_t)wmul64(asr64(yc, 13), vcy));
  z -= (uint32_t)asr64(cross, rcpShift - (sh + 13));
  z -= out[0] * (uint32_t)centerX + out[1] * (uint32_t)centerY;
  out[2] = z;
}

// cover8x8_selectFlips (Util.hpp:207-217); kept in the header record.
__device__ __forceinline__ uint32_t selectFlips(int32_t dx, int32_t dy) {
  uint32_t f = 0;
  if (dy > 0 || (dy == 0 && dx <= 0)) f ^= (1u << 3) ^ (1u << 2) ^ (1u << 5);
  if (dx > 0) f ^= (1u << 3) ^ (1u << 2);
  if (wabs32(dx) < wabs32(dy)) f ^= (1u << 4) ^ (1u << 2);
  return f;
}

// The draw state the clip path reads, passed to it by value: a reference
// to the kernel's Params would make every wave copy the whole argument
// block to scratch memory.
struct ClipCtx {
  int32_t viewportWidth, viewportHeight, samplesLog2, flags, shader, numTris, maxSubtris, vertexStride;
  const uint8_t* vertices;
  const int32_t* indices;
  uint8_t* triSubtris;
  Header* triHeader;
  TriData* triData;
  uint32_t* subtriTri;
  Counters* counters;
};

// snapTriangle (TriangleSetup.inl:19-31)
template <class PP>
__device__ __forceinline__ void snap(const PP& P, const float4& v0, const float4& v1, const float4& v2,
                                     I2& p0, I2& p1, I2& p2, float rcpW[3], I2& lo, I2& hi) {
  float sx = (float)(P.viewportWidth << (kSubpixelLog2 - 1));
  float sy = (float)(P.viewportHeight << (kSubpixelLog2 - 1));
  rcpW[0] = 1.0f / v0.w;
  rcpW[1] = 1.0f / v1.w;
  rcpW[2] = 1.0f / v2.w;
  p0.x = cvtRniSatS32(v0.x * rcpW[0] * sx); p0.y = cvtRniSatS32(v0.y * rcpW[0] * sy);
  p1.x = cvtRniSatS32(v1.x * rcpW[1] * sx); p1.y = cvtRniSatS32(v1.y * rcpW[1] * sy);
  p2.x = cvtRniSatS32(v2.x * rcpW[2] * sx); p2.y = cvtRniSatS32(v2.y * rcpW[2] * sy);
  lo.x = min(min(p0.x, p1.x), p2.x); lo.y = min(min(p0.y, p1.y), p2.y);
  hi.x = max(max(p0.x, p1.x), p2.x); hi.y = max(max(p0.y, p1.y), p2.y);
}

// prepareTriangle (TriangleSetup.inl:38-100): 0 visible, 1 backfacing,
// 2 between samples.
template <class PP>
__device__ __forceinline__ int prepare(const PP& P, I2 p0, I2 p1, I2 p2, I2 lo, I2 hi,
                                       I2& d1, I2& d2, int32_t& area) {
  int s = P.samplesLog2;
  d1.x = wsub(p1.x, p0.x); d1.y = wsub(p1.y, p0.y);
  d2.x = wsub(p2.x, p0.x); d2.y = wsub(p2.y, p0.y);
  area = wsub(wmul(d1.x, d2.y), wmul(d1.y, d2.x));
  if (area <= 0) return 1;

  int32_t ss = 1 << (kSubpixelLog2 - s);
  int32_t biasX = (P.viewportWidth << (kSubpixelLog2 - 1)) - (ss >> 1);
  int32_t biasY = (P.viewportHeight << (kSubpixelLog2 - 1)) - (ss >> 1);
  int32_t lox = wadd(wadd(lo.x, ss - 1), biasX) & -ss;
  int32_t loy = wadd(wadd(lo.y, ss - 1), biasY) & -ss;
  int32_t hix = wadd(hi.x, biasX) & -ss;
  int32_t hiy = wadd(hi.y, biasY) & -ss;
  if (lox > hix || loy > hiy) return 2;

  int32_t diff = wsub(wadd(hix, hiy), wadd(lox, loy));
  if (diff <= ss) {
    I2 t0 = {wsub(wadd(p0.x, biasX), lox), wsub(wadd(p0.y, biasY), loy)};
    I2 t1 = {wsub(wadd(p1.x, biasX), lox), wsub(wadd(p1.y, biasY), loy)};
    I2 t2 = {wsub(wadd(p2.x, biasX), lox), wsub(wadd(p2.y, biasY), loy)};
    int32_t e0 = wsub(wmul(t0.x, t1.y), wmul(t0.y, t1.x));
    int32_t e1 = wsub(wmul(t1.x, t2.y), wmul(t1.y, t2.x));
    int32_t e2 = wsub(wmul(t2.x, t0.y), wmul(t2.y, t0.x));
    if (e0 < 0 || e1 < 0 || e2 < 0) {
      if (diff == 0) return 2;
      t0 = {wsub(wadd(p0.x, biasX), hix), wsub(wadd(p0.y, biasY), hiy)};
      t1 = {wsub(wadd(p1.x, biasX), hix), wsub(wadd(p1.y, biasY), hiy)};
      t2 = {wsub(wadd(p2.x, biasX), hix), wsub(wadd(p2.y, biasY), hiy)};
      e0 = wsub(wmul(t0.x, t1.y), wmul(t0.y, t1.x));
      e1 = wsub(wmul(t1.x, t2.y), wmul(t1.y, t2.x));
      e2 = wsub(wmul(t2.x, t0.y), wmul(t2.y, t0.x));
      if (e0 < 0 || e1 < 0 || e2 < 0) return 2;
    }
  }
  return 0;
}

// setupTriangle (TriangleSetup.inl:104-215)
template <class PP>
__device__ __forceinline__ void setupTriangle(const PP& P, Header* th, TriData* td, int3 vidx,
                                              const float4& v0, const float4& v1, const float4& v2,
                                              float2 b0, float2 b1, float2 b2, I2 p0, I2 p1, I2 p2,
                                              const float rcpW[3], I2 d1, I2 d2, int32_t area) {
  int s = P.samplesLog2;
  float areaRcp = 0.0f;
  I2 wv0 = {0, 0};
  if (P.flags & (kFlagDepth | kFlagLerp)) {
    areaRcp = 1.0f / (float)area;
    wv0.x = wadd(p0.x, P.viewportWidth << (kSubpixelLog2 - 1));
    wv0.y = wadd(p0.y, P.viewportHeight << (kSubpixelLog2 - 1));
  }

  uint32_t zmin = 0, zslope = 0;
  uint32_t zp[3] = {0u, 0u, 0u};
  if (P.flags & kFlagDepth) {
    const float zcoef = (float)(kDepthMax - kDepthMin) * 0.5f;
    const float zbias = (float)(kDepthMax + kDepthMin) * 0.5f;
    float z0 = fmaf(v0.z * zcoef, rcpW[0], zbias);
    float z1 = fmaf(v1.z * zcoef, rcpW[1], zbias);
    float z2 = fmaf(v2.z * zcoef, rcpW[2], zbias);
    int32_t zv0x = wv0.x - (1 << (kSubpixelLog2 - s - 1));
    int32_t zv0y = wv0.y - (1 << (kSubpixelLog2 - s - 1));
    setupPleq(z0, z1, z2, zv0x, zv0y, d1.x, d1.y, d2.x, d2.y, areaRcp, s, zp);
    zmin = cvtRniSatU32(fminf(fminf(z0, z1), z2) - (float)lerpError(s));
    if (s != 0) {
      uint32_t tmp = wabs32((int32_t)zp[0]) + wabs32(max((int32_t)zp[1], -INT32_MAX));
      int sh = max(s - 1, 0);
      zslope = tmp << sh;
      if ((zslope >> sh) != tmp) zslope = 0xFFFFFFFFu;
    }
  }
  uint32_t wp[3] = {0u, 0u, 0u}, up[3] = {0u, 0u, 0u}, vp[3] = {0u, 0u, 0u};
  if (P.flags & kFlagLerp) {
    float wcoef = fminf(fminf(v0.w, v1.w), v2.w) * (float)kBaryMax;
    float w0 = wcoef * rcpW[0], w1 = wcoef * rcpW[1], w2 = wcoef * rcpW[2];
    setupPleq(w0, w1, w2, wv0.x, wv0.y, d1.x, d1.y, d2.x, d2.y, areaRcp, s + 1, wp);
    setupPleq(b0.x * w0, b1.x * w1, b2.x * w2, wv0.x, wv0.y, d1.x, d1.y, d2.x, d2.y, areaRcp, s + 1, up);
    setupPleq(b0.y * w0, b1.y * w1, b2.y * w2, wv0.x, wv0.y, d1.x, d1.y, d2.x, d2.y, areaRcp, s + 1, vp);
  }
  uint4* tdv = reinterpret_cast<uint4*>(td);
  tdv[0] = make_uint4(zp[0], zp[1], zp[2], zslope);
  if (P.shader != kShaderConstant) {
    // Barycentric planes and vertex indices: read only by the shaders that
    // interpolate varyings (a constant-colour draw writes the depth plane
    // alone).
    tdv[1] = make_uint4(wp[0], wp[1], wp[2], up[0]);
    tdv[2] = make_uint4(up[1], up[2], vp[0], vp[1]);
    tdv[3] = make_uint4(vp[2], (uint32_t)vidx.x, (uint32_t)vidx.y, (uint32_t)vidx.z);
  }

  uint32_t f01 = selectFlips(d1.x, d1.y);
  uint32_t f12 = selectFlips(wsub(d2.x, d1.x), wsub(d2.y, d1.y));
  uint32_t f20 = selectFlips(-d2.x, -d2.y);
  *reinterpret_cast<uint4*>(th) = make_uint4(
      ((uint32_t)p0.x & 0xFFFFu) | ((uint32_t)p0.y << 16),
      ((uint32_t)p1.x & 0xFFFFu) | ((uint32_t)p1.y << 16),
      ((uint32_t)p2.x & 0xFFFFu) | ((uint32_t)p2.y << 16),
      (zmin & 0xFFFFF000u) | (f01 << 6) | (f12 << 2) | (f20 >> 2));
}

// ---- clipping -------------------------------------------------------------------
//
// A wave's only clipped triangle is clipped by the whole wave: lane i holds
// vertex i of the clip polygon (at most 9) as its barycentrics; vertices past
// the polygon's end take no part.  With more of them, every lane clips its own,
// in an array indexed at run time, and the wave takes all slots with one
// addition to the draw's counter.  One after another they would take as many
// times as long as there are: setup of 1024 triangles with 2 / 64 clipped of
// every 64 50 / 560 us, by lanes 50 / 55; of 100k, then bound by an addition per
// triangle, 73 / 1208 and 63 / 70.  A single one takes the 1024 triangles 30 us
// by the wave, 48 by its lane; 1M small triangles with 256 large clipped ones
// among them 66 and 98.
struct ClipVert { float b0, b1; };

// Vertex of lane `from`.
__device__ __forceinline__ ClipVert vertOf(const ClipVert& v, int from) {
  return {__shfl(v.b0, from, 64), __shfl(v.b1, from, 64)};
}

// clipPolygonWithPlane (Util.hpp:221-250): the polygon's part where
// v0 + v1 b0 + v2 b1 >= 0.  Per vertex, in order: the intersection on the edge
// that ends there, if any, then the vertex itself, if inside.
__device__ __forceinline__ void clipPolygon(ClipVert& v, int& num, float v0, float v1, float v2) {
  if (num < 3) {
    num = 0;
    return;
  }
  const int lane = (int)(threadIdx.x & 63);
  const ClipVert a = vertOf(v, lane == 0 ? num - 1 : lane - 1);
  const float av = fmaf(v2, a.b1, fmaf(v1, a.b0, v0));
  const float bv = fmaf(v2, v.b1, fmaf(v1, v.b0, v0));
  const bool in = lane < num;
  const bool cross = in && av * bv < 0.0f, keep = in && bv >= 0.0f;
  const float bc = av / (av - bv);
  const float ac = 1.0f - bc;
  const ClipVert x = {fmaf(a.b0, ac, v.b0 * bc), fmaf(a.b1, ac, v.b1 * bc)};
  const uint64_t cm = __ballot(cross), km = __ballot(keep);
  // Output j: the (j + 1)-th of the marks, two per lane (cross, then keep).
  // Each lane looks up the lane that its output comes from.
  num = (int)(__popcll(cm) + __popcll(km));
  int from = 0;
  bool fromCross = false;
  for (int q = 0, n = 0; q < 9; q++) {               // (at most 9 vertices: q is uniform)
    const int c = (int)((cm >> q) & 1u), k = (int)((km >> q) & 1u);
    if (c && n == lane) { from = q; fromCross = true; }
    n += c;
    if (k && n == lane) { from = q; fromCross = false; }
    n += k;
  }
  const ClipVert fx = vertOf(x, from), fv = vertOf(v, from);
  v = fromCross ? fx : fv;
}

__device__ __forceinline__ float comp(const float4& v, int a) { return a == 0 ? v.x : (a == 1 ? v.y : v.z); }

// clipTriangleWithFrustum (Util.hpp:260-286): returns the vertex count.
__device__ __forceinline__ int clipTriangle(ClipVert& v, const float4& v0, const float4& v1, const float4& v2,
                                            const float4& d1, const float4& d2) {
  const int lane = (int)(threadIdx.x & 63);
  int num = 3;
  v = {lane == 1 ? 1.0f : 0.0f, lane == 2 ? 1.0f : 0.0f};
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if ((v0.w < fabsf(comp(v0, a))) | (v1.w < fabsf(comp(v1, a))) | (v2.w < fabsf(comp(v2, a)))) {
      clipPolygon(v, num, v0.w + comp(v0, a), d1.w + comp(d1, a), d2.w + comp(d2, a));
      clipPolygon(v, num, v0.w - comp(v0, a), d1.w - comp(d1, a), d2.w - comp(d2, a));
    }
  }
  return num;
}

__device__ __forceinline__ float4 lerpClip(const float4& o, const float4& d1, const float4& d2, const ClipVert& b) {
  return make_float4(fmaf(d2.x, b.b1, fmaf(d1.x, b.b0, o.x)), fmaf(d2.y, b.b1, fmaf(d1.y, b.b0, o.y)),
                     fmaf(d2.z, b.b1, fmaf(d1.z, b.b0, o.z)), fmaf(d2.w, b.b1, fmaf(d1.w, b.b0, o.w)));
}

struct ClipResult { int numSub, base; };

// clipPolygon by one lane, its polygon in an array.
__device__ __forceinline__ int clipPolygonLane(float* out, const float* in, int numIn, float v0, float v1, float v2) {
  int numOut = 0;
  if (numIn >= 3) {
    int ai = (numIn - 1) * 2;
    float av = fmaf(v2, in[ai + 1], fmaf(v1, in[ai + 0], v0));
    for (int bi = 0; bi < numIn * 2; bi += 2) {
      const float bv = fmaf(v2, in[bi + 1], fmaf(v1, in[bi + 0], v0));
      if (av * bv < 0.0f && numOut < 18) {             // (at most 9 vertices)
        const float bc = av / (av - bv);
        const float ac = 1.0f - bc;
        out[numOut + 0] = fmaf(in[ai + 0], ac, in[bi + 0] * bc);
        out[numOut + 1] = fmaf(in[ai + 1], ac, in[bi + 1] * bc);
        numOut += 2;
      }
      if (bv >= 0.0f && numOut < 18) {
        out[numOut + 0] = in[bi + 0];
        out[numOut + 1] = in[bi + 1];
        numOut += 2;
      }
      ai = bi;
      av = bv;
    }
  }
  return numOut >> 1;
}

// The clip of the triangles of the lanes in `todo`, each by its own lane.
__device__ __forceinline__ ClipResult setupClippedLanes(const ClipCtx& P, uint64_t todo, int t) {
  const int lane = (int)(threadIdx.x & 63);
  const bool mine = ((todo >> lane) & 1u) != 0;
  float bary[18];
  int numVerts = 0, numSub = 0;
  int3 vidx = make_int3(0, 0, 0);
  float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f), od1 = o, od2 = o;
  auto vertex = [&](int i) { return lerpClip(o, od1, od2, {bary[2 * i], bary[2 * i + 1]}); };
  I2 p0, p1, p2, lo, hi, d1, d2;
  float rcpW[3];
  int32_t area;
  if (mine) {
    const int32_t* ip = P.indices + (int64_t)t * 3;
    vidx = make_int3(ip[0], ip[1], ip[2]);
    o = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.x * P.vertexStride);
    const float4 b = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.y * P.vertexStride);
    const float4 c = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.z * P.vertexStride);
    od1 = make_float4(b.x - o.x, b.y - o.y, b.z - o.z, b.w - o.w);
    od2 = make_float4(c.x - o.x, c.y - o.y, c.z - o.z, c.w - o.w);
    float temp[18];
    bary[0] = 0.0f; bary[1] = 0.0f;
    bary[2] = 1.0f; bary[3] = 0.0f;
    bary[4] = 0.0f; bary[5] = 1.0f;
    numVerts = 3;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      if ((o.w < fabsf(comp(o, a))) | (b.w < fabsf(comp(b, a))) | (c.w < fabsf(comp(c, a)))) {
        numVerts = clipPolygonLane(temp, bary, numVerts, o.w + comp(o, a), od1.w + comp(od1, a), od2.w + comp(od2, a));
        numVerts = clipPolygonLane(bary, temp, numVerts, o.w - comp(o, a), od1.w - comp(od1, a), od2.w - comp(od2, a));
      }
    }
    const float4 v0 = vertex(0);
    float4 v1 = vertex(1);
    for (int i = 2; i < numVerts; i++) {
      const float4 v2 = vertex(i);
      snap(P, v0, v1, v2, p0, p1, p2, rcpW, lo, hi);
      if (prepare(P, p0, p1, p2, lo, hi, d1, d2, area) == 0) numSub++;
      v1 = v2;
    }
  }
  // One addition to the slot counter for the wave.
  const uint32_t need = numSub > 1 ? (uint32_t)numSub : 0u;
  const uint32_t scan = waveScan(need);
  const uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)scan, 63);
  uint32_t at = 0;
  if (lane == 0 && all) at = atomicAdd(&P.counters->numSubtris, all);
  at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
  ClipResult out = {0, t};
  if (!mine) return out;
  if (numSub > 1) out.base = P.numTris + (int)(at + scan - need);
  const bool over = numSub > 1 && out.base + numSub > P.maxSubtris;
  P.triSubtris[t] = (uint8_t)numSub;
  if (numSub > 1) P.triHeader[t].misc = (uint32_t)out.base;
  if (over) {
    atomicOr(&P.counters->overflow, 1u);
    return out;
  }
  out.numSub = numSub;
  int slot = out.base;
  const float4 v0 = vertex(0);
  float4 v1 = vertex(1);
  for (int i = 2; i < numVerts; i++) {
    const float4 v2 = vertex(i);
    snap(P, v0, v1, v2, p0, p1, p2, rcpW, lo, hi);
    if (prepare(P, p0, p1, p2, lo, hi, d1, d2, area) == 0) {
      setupTriangle(P, &P.triHeader[slot], &P.triData[slot], vidx, v0, v1, v2, make_float2(bary[0], bary[1]),
                    make_float2(bary[2 * i - 2], bary[2 * i - 1]), make_float2(bary[2 * i], bary[2 * i + 1]), p0, p1,
                    p2, rcpW, d1, d2, area);
      if (slot >= P.numTris) P.subtriTri[slot - P.numTris] = (uint32_t)t;
      slot++;
    }
    v1 = v2;
  }
  return out;
}

// The clip of triangle t (uniform) by the whole wave; lane f sets up fan
// triangle f.
__device__ __forceinline__ ClipResult setupClippedWave(const ClipCtx& P, int t) {
  const int lane = (int)(threadIdx.x & 63);
  const int32_t* ip = P.indices + (int64_t)t * 3;
  const int3 vidx = make_int3(ip[0], ip[1], ip[2]);
  const float4 ov0 = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.x * P.vertexStride);
  const float4 ov1 = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.y * P.vertexStride);
  const float4 ov2 = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.z * P.vertexStride);
  const float4 od1 = make_float4(ov1.x - ov0.x, ov1.y - ov0.y, ov1.z - ov0.z, ov1.w - ov0.w);
  const float4 od2 = make_float4(ov2.x - ov0.x, ov2.y - ov0.y, ov2.z - ov0.z, ov2.w - ov0.w);
  ClipVert v;
  const int numVerts = clipTriangle(v, ov0, ov1, ov2, od1, od2);
  const ClipVert c0 = vertOf(v, 0), c1 = vertOf(v, (lane + 1) & 63), c2 = vertOf(v, (lane + 2) & 63);
  const float4 v0 = lerpClip(ov0, od1, od2, c0), v1 = lerpClip(ov0, od1, od2, c1), v2 = lerpClip(ov0, od1, od2, c2);
  I2 p0, p1, p2, lo, hi, d1, d2;
  float rcpW[3];
  int32_t area;
  snap(P, v0, v1, v2, p0, p1, p2, rcpW, lo, hi);
  const bool vis = lane + 2 < numVerts && prepare(P, p0, p1, p2, lo, hi, d1, d2, area) == 0;
  const uint64_t vm = __ballot(vis);
  const int numSub = (int)__popcll(vm);
  int base = t;
  if (numSub > 1) {
    int at = 0;
    if (lane == 0) at = P.numTris + (int)atomicAdd(&P.counters->numSubtris, (uint32_t)numSub);
    base = __builtin_amdgcn_readfirstlane(at);
  }
  const bool over = numSub > 1 && base + numSub > P.maxSubtris;
  if (lane == 0) {
    P.triSubtris[t] = (uint8_t)numSub;
    if (numSub > 1) P.triHeader[t].misc = (uint32_t)base;
    if (over) atomicOr(&P.counters->overflow, 1u);
  }
  if (vis && !over) {
    const int slot = base + (int)__popcll(vm & ((1ull << lane) - 1ull));
    setupTriangle(P, &P.triHeader[slot], &P.triData[slot], vidx, v0, v1, v2, make_float2(c0.b0, c0.b1),
                  make_float2(c1.b0, c1.b1), make_float2(c2.b0, c2.b1), p0, p1, p2, rcpW, d1, d2, area);
    if (slot >= P.numTris) P.subtriTri[slot - P.numTris] = (uint32_t)t;
  }
  return {over ? 0 : numSub, base};
}

// Slow path, kept out of line, called by whole waves: frustum clip and fan
// (TriangleSetup.inl:326-412) of the triangles of the lanes in `todo` (not
// empty).  Returns, per lane in todo, the number of subtriangles written (0
// when the slot allocation overflowed) and their first slot.
__device__ __noinline__ ClipResult setupClipped(const ClipCtx P, uint64_t todo, int t) {
  if (__popcll(todo) > 1) return setupClippedLanes(P, todo, t);
  return setupClippedWave(P, __builtin_amdgcn_readlane(t, (int)__builtin_ctzll(todo)));
}

// Outcome of one triangle's setup, as the reference's setup counters
// classify it (TriangleSetup.inl:255-330).
enum SetupOutcome : int { kSetupVisible = 0, kSetupFrustum, kSetupBackface, kSetupBetween, kSetupClipPath,
                          kSetupDropped };

// One triangle: returns its number of subtriangles (in slot t).  When the
// triangle is set up without clipping, *hv receives the header's vertex words
// (as written to P.triHeader[t]) and *hvOk is set.  *why receives the
// SetupOutcome; kSetupClipPath leaves the triangle to setupClipped, its
// vertices to be read again there (kept in registers, they would cost every
// wave).
__device__ __forceinline__ int setupOne(const Params& P, int t, uint4* hv, bool* hvOk, int* why) {
  *hvOk = false;
  *why = kSetupDropped;
  int3 vidx;
  const int32_t* ip = P.indices + (int64_t)t * 3;
  vidx.x = ip[0]; vidx.y = ip[1]; vidx.z = ip[2];
  // Indices outside the vertex buffer: the triangle is dropped (the
  // reference reads past the buffer; here the result is defined).
  if ((uint32_t)vidx.x >= (uint32_t)P.numVertices || (uint32_t)vidx.y >= (uint32_t)P.numVertices ||
      (uint32_t)vidx.z >= (uint32_t)P.numVertices) {
    P.triSubtris[t] = 0;
    return 0;
  }
  const float4 v0 = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.x * P.vertexStride);
  const float4 v1 = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.y * P.vertexStride);
  const float4 v2 = *reinterpret_cast<const float4*>(P.vertices + (int64_t)vidx.z * P.vertexStride);

  // Outside view frustum => cull (:262-281).
  if ((v0.w < fabsf(v0.x)) | (v0.w < fabsf(v0.y)) | (v0.w < fabsf(v0.z))) {
    bool out = ((v0.w < +v0.x) & (v1.w < +v1.x) & (v2.w < +v2.x)) |
               ((v0.w < -v0.x) & (v1.w < -v1.x) & (v2.w < -v2.x)) |
               ((v0.w < +v0.y) & (v1.w < +v1.y) & (v2.w < +v2.y)) |
               ((v0.w < -v0.y) & (v1.w < -v1.y) & (v2.w < -v2.y)) |
               ((v0.w < +v0.z) & (v1.w < +v1.z) & (v2.w < +v2.z)) |
               ((v0.w < -v0.z) & (v1.w < -v1.z) & (v2.w < -v2.z));
    if (out) {
      P.triSubtris[t] = 0;
      *why = kSetupFrustum;
      return 0;
    }
  }

  // Inside depth range => snap; inside the guard band => fast path (:285-322).
  if ((v0.w >= fabsf(v0.z)) & (v1.w >= fabsf(v1.z)) & (v2.w >= fabsf(v2.z))) {
    I2 p0, p1, p2, lo, hi, d1, d2;
    float rcpW[3];
    int32_t area;
    snap(P, v0, v1, v2, p0, p1, p2, rcpW, lo, hi);
    int32_t loxy = min(lo.x, lo.y);
    int32_t hixy = max(hi.x, hi.y);
    const int32_t aabbLimit = (1 << (11 + kSubpixelLog2)) - 1;
    if (loxy >= -32768 && hixy <= 32767 && hixy - loxy <= aabbLimit) {
      int res = prepare(P, p0, p1, p2, lo, hi, d1, d2, area);
      P.triSubtris[t] = (res == 0) ? 1 : 0;
      *why = res == 0 ? kSetupVisible : (res == 1 ? kSetupBackface : kSetupBetween);
      if (res == 0) {
        setupTriangle(P, &P.triHeader[t], &P.triData[t], vidx, v0, v1, v2, make_float2(0.0f, 0.0f),
                      make_float2(1.0f, 0.0f), make_float2(0.0f, 1.0f), p0, p1, p2, rcpW, d1, d2, area);
        *hv = make_uint4(((uint32_t)p0.x & 0xFFFFu) | ((uint32_t)p0.y << 16),
                         ((uint32_t)p1.x & 0xFFFFu) | ((uint32_t)p1.y << 16),
                         ((uint32_t)p2.x & 0xFFFFu) | ((uint32_t)p2.y << 16), 0u);
        *hvOk = true;
      }
      return res == 0 ? 1 : 0;
    }
  }
  *why = kSetupClipPath;
  return 0;
}

// ---------------------------------------------------------------------------
// Fused setup + bin stage.
//
// One block sets up a chunk of kSetupChunk consecutive triangles (one per
// thread) and immediately bins their subtriangles (128x128-pixel bins,
// bounding-box test).  The chunk's entries go to a region of the bin queue
// reserved with one atomic; inside the region the entries of each bin are
// contiguous and in (triangle, subtriangle) order -- ranks come from per-wave
// 64-bit emit masks and popcounts.  The coarse stage reads bin b as the
// concatenation of its per-chunk segments in chunk order, which is
// submission order, so no global scan is needed.  (The reference streams
// triangles into linked 512-entry segments per (bin, stream) and merges 16
// streams, BinRaster.inl:19-469, CoarseRaster.inl:170-257.)
// ---------------------------------------------------------------------------

constexpr int kSetupChunk = kSetupChunkTris;
constexpr int kSetupWaves = kSetupChunk / 64;

struct BinBox { int32_t x0, y0, x1, y1; };   // inclusive; empty when x0 > x1

__device__ __forceinline__ BinBox binBoxOf(const Params& P, uint4 h) {
  const int32_t ox = P.viewportWidth << (kSubpixelLog2 - 1), oy = P.viewportHeight << (kSubpixelLog2 - 1);
  const int32_t x0 = (int32_t)(int16_t)(h.x & 0xFFFFu), y0 = (int32_t)(int16_t)(h.x >> 16);
  const int32_t x1 = (int32_t)(int16_t)(h.y & 0xFFFFu), y1 = (int32_t)(int16_t)(h.y >> 16);
  const int32_t x2 = (int32_t)(int16_t)(h.z & 0xFFFFu), y2 = (int32_t)(int16_t)(h.z >> 16);
  const int32_t minx = min(min(x0, x1), x2) + ox, maxx = max(max(x0, x1), x2) + ox;
  const int32_t miny = min(min(y0, y1), y2) + oy, maxy = max(max(y0, y1), y2) + oy;
  BinBox b;
  const int sh = kSubpixelLog2 + kTileLog2 + P.binLog2;
  if (maxx < 0 || maxy < 0 || minx >= (P.widthPixels << kSubpixelLog2) || miny >= (P.heightPixels << kSubpixelLog2)) {
    b.x0 = 1; b.x1 = 0; b.y0 = 1; b.y1 = 0;
    return b;
  }
  b.x0 = max(minx >> sh, 0); b.x1 = min(maxx >> sh, P.widthBins - 1);
  b.y0 = max(miny >> sh, 0); b.y1 = min(maxy >> sh, P.heightBins - 1);
  return b;
}

// A wave's wide boxes are walked by the whole wave, 16 x 4 bins at a time, one
// box after another, instead of by their own lanes bin by bin, where the largest
// has more than kCoopBins bins for each of them.  A box takes the wave as long as
// three bins take the lanes if all waves of a workgroup have such boxes (their
// additions to the masks collide), nine if one has.  Setup of 1024 triangles, k
// of each 64 over 8 to 12 bins: lanes 2.6 us more than none for k = 4, 4 for 36,
// wave 0.65 k; over 64 to 81 bins: lanes 19 and 27, wave 1.2 k; over 256: lanes 62
// and 150, wave 2.7 k; 16 and 64 boxes of 230 bins in a single wave: lanes 34 and
// 26, wave 20 and 68.
constexpr int kCoopBins = 7;
__device__ __forceinline__ bool coopBoxes(const BinBox& b) {
  const int area = b.x0 <= b.x1 ? (b.x1 - b.x0 + 1) * (b.y1 - b.y0 + 1) : 0;
  const uint64_t wide = __ballot(area > kCoopBins);
  if (wide == 0) return false;
  const int most = waveReduce(area, 0, [](int a, int c) { return max(a, c); });
  return most > kCoopBins * (int)__popcll(wide) && area > kCoopBins;
}

// Calls f(bin, j) for every bin of lane j's box (j uniform).
template <class F>
__device__ __forceinline__ void forEachBinCoop(const Params& P, const BinBox& b, int j, F&& f) {
  const int lane = (int)(threadIdx.x & 63);
  const int x0 = __builtin_amdgcn_readlane(b.x0, j), x1 = __builtin_amdgcn_readlane(b.x1, j);
  const int y0 = __builtin_amdgcn_readlane(b.y0, j), y1 = __builtin_amdgcn_readlane(b.y1, j);
  for (int ys = y0; ys <= y1; ys += 4)
    for (int xs = x0; xs <= x1; xs += 16) {
      const int x = xs + (lane & 15), y = ys + (lane >> 4);
      if (x <= x1 && y <= y1) f(x + y * P.widthBins, j);
    }
}

__device__ __forceinline__ uint64_t laneLt() {
  const uint32_t lane = threadIdx.x & 63;
  return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Setup and binning of chunk `chunk` of one draw (one 1024-lane workgroup).
// load(): the draw's parameters; asked for once by the setup and once by the
// binning, so that a batch, which loads them from its table, need not hold
// the one's through the other.
template <class Load>
__device__ __forceinline__ void setupBinBody(Load&& load, const int chunk) {
  __shared__ uint32_t cnt[kMaxBins];
  __shared__ uint32_t run[kMaxBins];
  __shared__ uint64_t emitMask[kSetupWaves][kMaxBins];
  __shared__ uint32_t emitPre[kSetupWaves][kMaxBins];
  __shared__ uint32_t list[kSetupChunk];
  __shared__ uint32_t sums[2][kSetupWaves];
  __shared__ uint32_t sBase;
  __shared__ uint32_t sProf[8];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int t = chunk * kSetupChunk + threadIdx.x;
  // ---- setup ---------------------------------------------------------------
  int base = t, k = 0, why = kSetupDropped;
  uint4 hvOwn = make_uint4(0u, 0u, 0u, 0u);   // header vertex words kept from setup (no re-read)
  bool hvOwnOk = false;
  {
    auto&& P = load();
    if (chunk == 0) stampStage(P, kStampSetup);
    if (t < P.numTris) k = setupOne(P, t, &hvOwn, &hvOwnOk, &why);
    const uint64_t clip = __ballot(t < P.numTris && why == kSetupClipPath);
    if (__builtin_expect(clip != 0, 0)) {
      const ClipCtx C = {P.viewportWidth, P.viewportHeight, P.samplesLog2, (int32_t)P.flags, P.shader,
                         P.numTris, P.maxSubtris, P.vertexStride, P.vertices, P.indices, P.triSubtris, P.triHeader,
                         P.triData, P.subtriTri, P.counters};
      const ClipResult r = setupClipped(C, clip, t);
      if ((clip >> lane) & 1u) {
        k = r.numSub;
        base = r.base;
      }
    }
  }
  auto&& P = load();
  if (P.prof != nullptr) {
    // Profiling draws: per-outcome triangle counts of the chunk, then its
    // triangles with at least one subtriangle.
    if (threadIdx.x < 8) sProf[threadIdx.x] = 0;
    __syncthreads();
    const bool valid = t < P.numTris;
    const uint32_t nValid = (uint32_t)__popcll(__ballot(valid));
    const uint32_t nFr = (uint32_t)__popcll(__ballot(valid && why == kSetupFrustum));
    const uint32_t nBf = (uint32_t)__popcll(__ballot(valid && why == kSetupBackface));
    const uint32_t nBt = (uint32_t)__popcll(__ballot(valid && why == kSetupBetween));
    const uint32_t nCl = (uint32_t)__popcll(__ballot(valid && why == kSetupClipPath));
    const uint32_t nVis = (uint32_t)__popcll(__ballot(valid && k > 0));
    if (lane == 0) {
      atomicAdd(&sProf[0], nValid);
      atomicAdd(&sProf[1], nFr);
      atomicAdd(&sProf[2], nBf);
      atomicAdd(&sProf[3], nBt);
      atomicAdd(&sProf[4], nCl);
      atomicAdd(&sProf[5], nVis);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      profAdd(P.prof, kProfSetupViewportCull, 100ull * sProf[1], sProf[0]);
      profAdd(P.prof, kProfSetupBackfaceCull, 100ull * sProf[2], sProf[0]);
      profAdd(P.prof, kProfSetupBetweenPixelsCull, 100ull * sProf[3], sProf[0]);
      profAdd(P.prof, kProfSetupClipped, 100ull * sProf[4], sProf[0]);
      profAdd(P.prof, kProfSetupSamplesPerTri, 0, sProf[5]);
    }
  }

  for (int i = threadIdx.x; i < P.numBins; i += kSetupChunk) cnt[i] = 0;
  // Window = up to kSetupChunk consecutive subtriangles of the chunk in
  // submission order; a chunk without clipped triangles is a single window.
  const bool compact = __syncthreads_or(k > 1) != 0;
  uint32_t total;
  const uint32_t pos = blockScan<kSetupChunk>((uint32_t)k, sums[0], total);
  const uint32_t numWin = (total + kSetupChunk - 1) / kSetupChunk;
  if (P.chunkSubtris != nullptr && threadIdx.x == 0) P.chunkSubtris[chunk] = total;

  // Emit masks of one window: bit `lane` of emitMask[wave][bin] is set when
  // the window entry held by this thread touches the bin.
  auto buildMasks = [&](uint32_t w, uint32_t& slot, BinBox& bb, uint4& hv) -> bool {
    for (int i = threadIdx.x; i < kSetupWaves * P.numBins; i += kSetupChunk)
      emitMask[i / P.numBins][i % P.numBins] = 0ull;
    if (!compact) {
      // fast path: entry of this thread is its own subtriangle (k <= 1)
      slot = (uint32_t)base;
      bb.x0 = 1; bb.x1 = 0; bb.y0 = 1; bb.y1 = 0;
      __syncthreads();
      if (k == 1) {
        hv = hvOwnOk ? hvOwn : *reinterpret_cast<const uint4*>(&P.triHeader[slot]);
        bb = binBoxOf(P, hv);
      }
    } else {
      for (int s = 0; s < k; s++) {
        const uint32_t e = pos + (uint32_t)s;
        if (e >= w * kSetupChunk && e < (w + 1) * kSetupChunk) list[e - w * kSetupChunk] = (uint32_t)base + s;
      }
      __syncthreads();
      const uint32_t e = w * kSetupChunk + threadIdx.x;
      bb.x0 = 1; bb.x1 = 0; bb.y0 = 1; bb.y1 = 0;
      slot = 0;
      if (e < total) {
        slot = list[threadIdx.x];
        hv = *reinterpret_cast<const uint4*>(&P.triHeader[slot]);
        bb = binBoxOf(P, hv);
      }
    }
    const uint64_t bit = 1ull << lane;
    const bool big = coopBoxes(bb);
    if (!big) {
      for (int y = bb.y0; y <= bb.y1; y++)
        for (int x = bb.x0; x <= bb.x1; x++)
          atomicOr((unsigned long long*)&emitMask[wave][x + y * P.widthBins], (unsigned long long)bit);
    }
    for (uint64_t m = __ballot(big); m != 0; m &= m - 1)
      forEachBinCoop(P, bb, (int)__builtin_ctzll(m), [&](int bin, int j) {
        atomicOr((unsigned long long*)&emitMask[wave][bin], 1ull << j);
      });
    __syncthreads();
    return true;
  };

  // ---- pass 1: per-bin counts ---------------------------------------------
  uint32_t slot0 = 0;
  BinBox bb0;
  uint4 hv0 = make_uint4(0, 0, 0, 0);
  for (uint32_t w = 0; w < numWin; w++) {
    buildMasks(w, slot0, bb0, hv0);
    for (int i = threadIdx.x; i < P.numBins; i += kSetupChunk) {
      uint32_t acc = cnt[i];
#pragma unroll
      for (int q = 0; q < kSetupWaves; q++) acc += (uint32_t)__popcll(emitMask[q][i]);
      cnt[i] = acc;
    }
    if (P.prof != nullptr) {
      // Subtriangles whose box lies in a single bin.
      const uint32_t n1 = (uint32_t)__popcll(__ballot(bb0.x0 == bb0.x1 && bb0.y0 == bb0.y1));
      if (lane == 0 && n1) atomicAdd(&sProf[6], n1);
    }
    __syncthreads();
  }

  // ---- reserve the chunk's region; publish the bins' addresses --------------
  uint32_t tot2;
  const uint32_t c = (threadIdx.x < (unsigned)P.numBins) ? cnt[threadIdx.x] : 0u;
  const uint32_t off = blockScan<kSetupChunk>(c, sums[1], tot2);
  if (P.prof != nullptr && threadIdx.x == 0) {
    profAdd(P.prof, kProfBinTrisPerChunk, total, 1);
    profAdd(P.prof, kProfBinTriBBArea, tot2, total);
    profAdd(P.prof, kProfBinTriSingleBin, 100ull * sProf[6], total);
  }
  if (threadIdx.x == 0) {
    uint32_t b = tot2 ? atomicAdd(&P.counters->binEntries, tot2) : 0u;
    if (tot2 && (uint64_t)b + tot2 > (uint64_t)P.maxBinEntries) {
      atomicOr(&P.counters->overflow, 2u);
      b = 0xFFFFFFFFu;
    }
    sBase = b;
  }
  if (threadIdx.x < (unsigned)P.numBins) run[threadIdx.x] = off;
  __syncthreads();
  const uint32_t regionBase = sBase;
  // (Where the queue overflowed the row is never read.)
  uint32_t* row = P.binAddr + (size_t)chunk * (size_t)(P.numBins + 1);
  if (threadIdx.x < (unsigned)P.numBins) row[threadIdx.x] = regionBase + off;
  if (threadIdx.x == 0) row[P.numBins] = regionBase + tot2;
  if (regionBase == 0xFFFFFFFFu || tot2 == 0) return;

  // ---- pass 2: write the entries in order ------------------------------------
  for (uint32_t w = 0; w < numWin; w++) {
    uint32_t slot = slot0;
    BinBox bb = bb0;
    uint4 hv = hv0;
    if (numWin > 1) buildMasks(w, slot, bb, hv);
    for (int i = threadIdx.x; i < P.numBins; i += kSetupChunk) {
      uint32_t acc = run[i];
#pragma unroll
      for (int q = 0; q < kSetupWaves; q++) {
        emitPre[q][i] = acc;
        acc += (uint32_t)__popcll(emitMask[q][i]);
      }
      run[i] = acc;
    }
    __syncthreads();
    auto put = [&](int bin, uint64_t lt, const uint4& e) {
      const uint32_t p = regionBase + emitPre[wave][bin] + (uint32_t)__popcll(emitMask[wave][bin] & lt);
      if (p < (uint32_t)P.maxBinEntries) P.binList[p] = e;
    };
    const uint4 e = make_uint4(slot, hv.x, hv.y, hv.z);
    const bool big = coopBoxes(bb);
    if (!big) {
      const uint64_t lt = laneLt();
      for (int y = bb.y0; y <= bb.y1; y++)
        for (int x = bb.x0; x <= bb.x1; x++) put(x + y * P.widthBins, lt, e);
    }
    for (uint64_t m = __ballot(big); m != 0; m &= m - 1) {
      const int j = (int)__builtin_ctzll(m);
      const uint4 ej = make_uint4(__builtin_amdgcn_readlane(e.x, j), __builtin_amdgcn_readlane(e.y, j),
                                  __builtin_amdgcn_readlane(e.z, j), __builtin_amdgcn_readlane(e.w, j));
      forEachBinCoop(P, bb, j, [&](int bin, int l) { put(bin, (1ull << l) - 1ull, ej); });
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(kSetupChunk, 8) setupBinKernel(const Params P) {
  setupBinBody([&]() -> const Params& { return P; }, blockIdx.x);
}

// Batched draws: one workgroup per chunk of every view; blockStart[v] is the
// first workgroup of view v (numViews + 1 entries).
__global__ void __launch_bounds__(kSetupChunk, 8) setupBinBatchKernel(const Params* __restrict__ views,
                                                                   const int32_t* __restrict__ blockStart,
                                                                   const int32_t* __restrict__ order,
                                                                   int numViews) {
  const int k = findView(blockStart, numViews, (int)blockIdx.x);
  const Params* view = &views[order[k]];
  setupBinBody(
      [&]() {
        __asm__ volatile("" : "+s"(view));
        return loadParams(view);
      },
      (int)blockIdx.x - blockStart[k]);
}

void launchSetup(const Params& P, hipStream_t stream) {
  if (P.numTris <= 0) return;
  hipLaunchKernelGGL(setupBinKernel, dim3(P.numChunks), dim3(kSetupChunk), 0, stream, P);
}

void launchSetupBatch(const Params* views, const int32_t* blockStart, const int32_t* order, int numViews,
                      int totalBlocks, hipStream_t stream) {
  if (totalBlocks <= 0) return;
  hipLaunchKernelGGL(setupBinBatchKernel, dim3(totalBlocks), dim3(kSetupChunk), 0, stream, views, blockStart,
                     order, numViews);
}

}  // namespace crhip
