// Backward of the output gate z = y * s, s = sigmoid(x wg^T) (mote/model/relation.py:179-181), the
// elementwise half: dy = dz s and dg = dz y s (1 - s), in fp32 from bf16 and rounded once each (the
// products in the order of the eager expressions, so the bits are theirs). The products with wg and x
// that follow are the caller's.
//
// Bound by its bytes: three bf16 reads and two writes an element in one launch, 16 bytes a lane. As eager
// operations (three casts to fp32, four fp32 products, the difference, two casts back) it was ten
// launches and about five times the bytes: 4,966 x 768 elements 7.2 us here (5.3 TB/s) against 70 us.
#include "common.hpp"
#include "params.hpp"

namespace mote {

__global__ void __launch_bounds__(256) gate_bwd_kernel(const uint4* dz, const uint4* y, const uint4* s, uint4* dy,
                                                       uint4* dg, int64_t nchunks) {
#pragma clang fp contract(off)
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= nchunks) return;
  const uint4 a = dz[i], b = y[i], c = s[i];
  const uint32_t aw[4] = {a.x, a.y, a.z, a.w}, bw[4] = {b.x, b.y, b.z, b.w}, cw[4] = {c.x, c.y, c.z, c.w};
  uint32_t ow[4], gw[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    float o[2], g[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float dzf = __uint_as_float(h ? aw[w] & 0xffff0000u : aw[w] << 16);
      const float yf = __uint_as_float(h ? bw[w] & 0xffff0000u : bw[w] << 16);
      const float sf = __uint_as_float(h ? cw[w] & 0xffff0000u : cw[w] << 16);
      o[h] = dzf * sf;
      g[h] = dzf * yf * sf * (1.0f - sf);
    }
    ow[w] = uint32_t(f2bf(o[0])) | (uint32_t(f2bf(o[1])) << 16);
    gw[w] = uint32_t(f2bf(g[0])) | (uint32_t(f2bf(g[1])) << 16);
  }
  dy[i] = uint4{ow[0], ow[1], ow[2], ow[3]};
  dg[i] = uint4{gw[0], gw[1], gw[2], gw[3]};
}

}  // namespace mote

extern "C" int mote_gate_bwd(const mote_gate_bwd_args* a, void* stream) {
  using namespace mote;
  if (!a) return set_error(MOTE_ERR_ARGUMENT, "gate_bwd: null args");
  if (a->dtype != MOTE_BF16) return set_error(MOTE_ERR_ARGUMENT, "gate_bwd: dtype %d (bf16 only)", a->dtype);
  if (a->n < 0 || a->n % 8) return set_error(MOTE_ERR_SHAPE, "gate_bwd: %lld elements (a multiple of 8)", (long long)a->n);
  if (a->n == 0) return MOTE_OK;
  for (const void* ptr : {a->dz, a->y, a->s, (const void*)a->dy, (const void*)a->dg})
    if (!ptr || reinterpret_cast<uintptr_t>(ptr) % 16)
      return set_error(MOTE_ERR_ARGUMENT, "gate_bwd: pointers must be 16-byte aligned and not null");
  const int64_t nchunks = a->n / 8, blocks = (nchunks + 255) / 256;
  if (blocks > 0x7fffffff) return set_error(MOTE_ERR_SHAPE, "gate_bwd: too many elements");
  hipLaunchKernelGGL(gate_bwd_kernel, dim3(unsigned(blocks)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     static_cast<const uint4*>(a->dz), static_cast<const uint4*>(a->y), static_cast<const uint4*>(a->s),
                     static_cast<uint4*>(a->dy), static_cast<uint4*>(a->dg), nchunks);
  return check_launch("gate_bwd");
}
