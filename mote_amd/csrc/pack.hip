// The stacked projection weight of a layer, [w1; w2; wi] as bf16 rows back to back, from the fp32 master
// weights (mote/model/relation.py:204-207 concatenates them; autocast rounds the result). One launch
// reads each weight once and writes the stack once, rounding to nearest even as a cast does; as a
// concatenation and a cast it was two launches and the fp32 stack written and read again in between:
// 3 x 768 x 768 took 7.8 + 5.1 us.
#include "common.hpp"
#include "params.hpp"

namespace mote {

struct PackParams {
  const float* src[3];
  uint4* dst;
  int64_t chunks;  // 8-element chunks of one source
};

__global__ void __launch_bounds__(256) pack_weights_kernel(const PackParams p) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= p.chunks) return;
  const int s = blockIdx.y;
  const float4 a = reinterpret_cast<const float4*>(p.src[s])[2 * i], b = reinterpret_cast<const float4*>(p.src[s])[2 * i + 1];
  uint4 o;
  o.x = uint32_t(f2bf(a.x)) | (uint32_t(f2bf(a.y)) << 16);
  o.y = uint32_t(f2bf(a.z)) | (uint32_t(f2bf(a.w)) << 16);
  o.z = uint32_t(f2bf(b.x)) | (uint32_t(f2bf(b.y)) << 16);
  o.w = uint32_t(f2bf(b.z)) | (uint32_t(f2bf(b.w)) << 16);
  p.dst[s * p.chunks + i] = o;
}

}  // namespace mote

extern "C" int mote_pack_weights(const mote_pack_weights_args* a, void* stream) {
  using namespace mote;
  if (!a) return set_error(MOTE_ERR_ARGUMENT, "pack_weights: null args");
  if (a->n < 0 || a->n % 8) return set_error(MOTE_ERR_SHAPE, "pack_weights: %lld elements (a multiple of 8)", (long long)a->n);
  if (a->n == 0) return MOTE_OK;
  for (const void* ptr : {a->w0, a->w1, a->w2, (const void*)a->out})
    if (!ptr || reinterpret_cast<uintptr_t>(ptr) % 16)
      return set_error(MOTE_ERR_ARGUMENT, "pack_weights: pointers must be 16-byte aligned and not null");
  PackParams p;
  p.src[0] = static_cast<const float*>(a->w0);
  p.src[1] = static_cast<const float*>(a->w1);
  p.src[2] = static_cast<const float*>(a->w2);
  p.dst = static_cast<uint4*>(a->out);
  p.chunks = a->n / 8;
  const int64_t blocks = (p.chunks + 255) / 256;
  if (blocks > 0x7fffffff) return set_error(MOTE_ERR_SHAPE, "pack_weights: too many elements");
  hipLaunchKernelGGL(pack_weights_kernel, dim3(unsigned(blocks), 3), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), p);
  return check_launch("pack_weights");
}
