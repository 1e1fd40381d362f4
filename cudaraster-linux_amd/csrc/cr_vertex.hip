// The step before the path: the passthrough vertex shader.
//
// vertexShader_passthrough (test/shader/PassThrough.cu:16-35) writes each
// vertex's clip position posToClip * (modelPos, 1), with Mat4f * Vec4f as
// base/Math.hpp:990-1001 evaluates it: per row i, rr = 0, then
// rr += m(i, j) * v[j] for j = 0..3, which nvcc contracts to fused
// multiply-adds -- restated here as an explicit fmaf chain in the same
// order, so the clip positions are bit-identical.  Only the first 16 bytes
// of each output record are written (ShadedVertexBase::clipPos); the rest of
// the record (varyings) is left as it is, so the kernel can fill the
// position part of an interleaved vertex buffer that setup then reads.
//
// One lane per vertex: 12 bytes read, 16 bytes written, HBM-bound.  The
// matrix arrives as a kernel argument (scalar registers).
#include "cr_device.h"

namespace crhip {

struct Mat4 { float m[16]; };      // Mat4f memory order: m(r, c) = m[r + 4c]

// STREAM: the records are written past the caches (non-temporal).  Half a
// cache line each, they otherwise leave partial lines all over the caches.
template <bool STREAM>
__global__ void __launch_bounds__(256) vertexPassthroughKernel(const float* __restrict__ modelPos,
                                                               int64_t numVertices, const Mat4 M,
                                                               uint8_t* __restrict__ out, int64_t outStride) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= numVertices) return;
  const float in[4] = {modelPos[3 * v + 0], modelPos[3 * v + 1], modelPos[3 * v + 2], 1.0f};
  typedef float Floatx4 __attribute__((ext_vector_type(4)));
  Floatx4 r;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float rr = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) rr = fmaf(M.m[i + 4 * j], in[j], rr);
    r[i] = rr;
  }
  Floatx4* const o = reinterpret_cast<Floatx4*>(out + v * outStride);
  if (STREAM) __builtin_nontemporal_store(r, o);
  else *o = r;
}

void launchVertexPassthrough(const float* modelPos, int64_t numVertices, const float posToClip[16], void* out,
                             int64_t outStride, hipStream_t stream) {
  if (numVertices <= 0) return;
  Mat4 M;
  for (int k = 0; k < 16; k++) M.m[k] = posToClip[k];
  // Past what the 256 MB last-level cache holds beside a program's other
  // buffers: three sets in turn of 3M vertices in 32-byte records (132 MB a set)
  // 44 -> 38 us, in 64-byte records 81 -> 75, in 16-byte ones (84 MB) 13.3 ->
  // 12.8.  Below, the next reader finds the records there, and so does the next
  // write: 1M in 32-byte records (44 MB) 10.5 against 13.7.
  const bool past = numVertices * (12 + outStride) >= (int64_t)64 << 20;
  const auto kernel = past ? vertexPassthroughKernel<true> : vertexPassthroughKernel<false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((numVertices + 255) / 256)), dim3(256), 0, stream,
                     modelPos, numVertices, M, static_cast<uint8_t*>(out), outStride);
}

}  // namespace crhip
