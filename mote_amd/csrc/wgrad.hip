// Weight gradient of a projection: dW [N, K] = A^T X for A [M, N] (the output gradient, token rows)
// and X [M, K] (the projection's input rows), bf16 in and out, fp32 accumulation. This is the
// weight half of autograd through the projections of FullRelation (mote/model/relation.py:204-215:
// the stacked [w1; w2; wi] product, whose weight gradient is dqkv^T x), the product whose reduction
// runs over the M token rows.
//
// A workgroup (4 waves) owns a TN x TK tile of dW (128 x 128; 64 along a width that is no multiple of
// 128) and one contiguous range of token rows (a split of M); the k of the products is the token
// index. Stages of 64 token rows of both operands go global -> LDS by direct transfers into two slots
// ([token][columns], chunks swizzled as in tiles.hpp), and both MFMA operands are transposed LDS reads
// (ds_read_b64_tr_b16) of the staged tiles, so neither operand is transposed in memory. Wave (wr, wc)
// holds dW rows TN/2 wr .. and columns TK/2 wc .. as 16 x 16 accumulator tiles with the X columns in
// the accumulator rows, so a lane ends with 4 consecutive columns of one dW row (one 8-byte bf16 or
// 16-byte fp32 store).
//
// Splits: with few dW tiles (2304 x 768 is 108 of 128 x 128, 576 x 192 is 27 of 64 x 64) M is cut into S
// ranges of whole 64-row stages, S about two workgroups per CU over the tiles; each split writes its
// fp32 partial tile to the workspace and a second launch adds the S partials in a fixed order and
// rounds once to the output type (bitwise reproducible, independent of scheduling). One split writes
// the output directly. Rows past M in the last stage are zeroed in LDS in both operands.
//
// What bounds it: the two transposed fragment reads per pair of products (LDS), and for the narrow
// widths the bytes of the two operands. 576 x 192 over 19,856 rows (the 192-wide layer's stacked
// projections, 30 MB of operands): 17.8 us with the sum, against 110 us for the GEMM library's product;
// 2304 x 768 over 4964 rows 32.3 us (544 TFLOP/s; 36.1 over eight input sets in turn), library 50; over 79,424
// rows 336 us (837 TFLOP/s), library 524 (as graphs of ten calls).
#include "common.hpp"
#include "params.hpp"
#include "tiles.hpp"

namespace mote {

int device_cu_count();

constexpr int kWgTok = 64;    // token rows per stage (two 32-deep k steps)
constexpr int kWgWaves = 4;

struct WgradParams {
  const bf16_t* a; int64_t a_sr;  // [M, N]
  const bf16_t* x; int64_t x_sr;  // [M, K]
  void* dw; int64_t dw_sr;        // [N, K], bf16 or fp32 (dw_f32)
  int dw_f32;
  float* part;                    // [nsplit][N][K] fp32 partials, or null (one split: straight to dw)
  int M, N, K, nsplit, mper, ntn, ntk;
};

__device__ __forceinline__ void wgrad_store(const WgradParams& p, int n, int c, f32x4 v) {
  if (p.dw_f32) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.dw) + int64_t(n) * p.dw_sr + c) = v;
  } else {
    uint2 o;
    o.x = uint32_t(f2bf(v[0])) | (uint32_t(f2bf(v[1])) << 16);
    o.y = uint32_t(f2bf(v[2])) | (uint32_t(f2bf(v[3])) << 16);
    *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(p.dw) + int64_t(n) * p.dw_sr + c) = o;
  }
}

template <int TN, int TK>
__global__ void __launch_bounds__(64 * kWgWaves) __attribute__((amdgpu_waves_per_eu(2)))
wgrad_kernel(const WgradParams p) {
  using E = Elem<bf16_t>;
  using Frag = E::Frag;
  using StX = TileStager<TK, kWgWaves, 1>;
  using StA = TileStager<TN, kWgWaves, 1>;
  constexpr int XT = kWgTok * TK;          // elements of the staged X tile
  constexpr int STAGE = XT + kWgTok * TN;  // X tile | A tile
  constexpr int NI = TK / 32, NJ = TN / 32;
  __shared__ __align__(16) bf16_t smem[2 * STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lg = lane >> 4;
  // workgroup id -> (split, row tile, column tile): workgroups go round-robin over the 8 XCDs, so XCD
  // j takes the j-th contiguous run of that order, tiles of one split that share their operand rows
  const int per_split = p.ntn * p.ntk, nwg = per_split * p.nsplit, per = (nwg + 7) / 8;
  const int seq = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (seq >= nwg) return;
  const int split = seq / per_split, rem = seq - split * per_split;
  const int tn = rem / p.ntk, tk = rem - tn * p.ntk;
  const int m0 = split * p.mper, m1 = min(p.M, m0 + p.mper);
  const int nblk = (m1 - m0 + kWgTok - 1) / kWgTok;
  const bf16_t* const xsrc[1] = {p.x + int64_t(tk) * TK};
  const bf16_t* const asrc[1] = {p.a + int64_t(tn) * TN};
  const int64_t xstr[1] = {p.x_sr}, astr[1] = {p.a_sr};
  StX stx;
  StA sta;
  stx.init(wave, lane, xstr);
  sta.init(wave, lane, astr);
  auto issue = [&](bf16_t* dst, int r0) __attribute__((always_inline)) {
    stx.issue(dst, xsrc, xstr, r0, p.M - 1, wave, lane);
    sta.issue(dst + XT, asrc, astr, r0, p.M - 1, wave, lane);
  };
  const int wr = wave & 1, wc = wave >> 1;

  f32x4 acc[NI][NJ];  // [X column tile i][A column tile j]
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  issue(smem, m0);
  for (int b = 0; b < nblk; ++b) {
    bf16_t* cur = smem + (b & 1) * STAGE;
    __builtin_amdgcn_s_waitcnt(0);  // this wave's transfers of stage b
    lds_barrier();
    const int r0 = m0 + b * kWgTok;
    if (__builtin_expect(r0 + kWgTok > p.M, 0)) {
      // the last stage of the reduction: its rows past M hold copies of row M - 1; zero them in both
      // tiles (whole rows, so the chunk swizzle does not matter)
      // (one loop over both tiles, off the hot path, its bounds opaque: as two loops the compiler kept their
      // addresses in registers that every stage advanced between the products, 351 us at 79,424 rows)
      int z0 = p.M - r0;
      asm volatile("" : "+s"(z0));
      for (int q = threadIdx.x; q < (kWgTok - z0) * (TK + TN) / 8; q += 64 * kWgWaves) {
        const int row = z0 + q / ((TK + TN) / 8), c = q % ((TK + TN) / 8) * 8;
        *reinterpret_cast<bf16x8*>(cur + (c < TK ? row * TK + c : XT + row * TN + c - TK)) = bf16x8{};
      }
      lds_barrier();
    }
    // every fragment of the stage, then the next stage's transfers into the other slot, then the
    // products (the other slot's last reads were the previous stage's, before this barrier)
    Frag fx[2][NI], fa[2][NJ];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int i = 0; i < NI; ++i) fx[ks][i] = tile_tr_frag<TK>(cur, 32 * ks, NI * wc + i, li, lg);
#pragma unroll
      for (int j = 0; j < NJ; ++j) fa[ks][j] = tile_tr_frag<TN>(cur + XT, 32 * ks, NJ * wr + j, li, lg);
    }
    if (b + 1 < nblk) issue(smem + ((b + 1) & 1) * STAGE, r0 + kWgTok);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = E::mma(fx[ks][i], fa[ks][j], acc[i][j]);
  }

  // lane: dW row n = TN tn + TN/2 wr + 16 j + li, columns c = TK tk + TK/2 wc + 16 i + 4 lg .. +3
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int n = tn * TN + TN / 2 * wr + 16 * j + li;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int c = tk * TK + TK / 2 * wc + 16 * i + 4 * lg;
      if (p.part)
        *reinterpret_cast<f32x4*>(p.part + (int64_t(split) * p.N + n) * p.K + c) = acc[i][j];
      else
        wgrad_store(p, n, c, acc[i][j]);
    }
  }
}

// dW = the sum of the splits' partials, rounded once; no splits (M = 0): zeros. A thread owns four
// consecutive columns. NW = 1: it adds every split in order. NW = 4: the four waves of a workgroup own
// the same columns, wave w adds the splits w, w + 4, ..., and the waves' sums are added in wave order.
template <int NW>
__global__ void __launch_bounds__(256) wgrad_sum_kernel(const WgradParams p) {
  __shared__ f32x4 red[3][64];
  const int lane = threadIdx.x & 63, wave = NW == 1 ? 0 : threadIdx.x >> 6;
  const int64_t q = NW == 1 ? int64_t(blockIdx.x) * 256 + threadIdx.x : int64_t(blockIdx.x) * 64 + lane;
  const int64_t nq = int64_t(p.N) * (p.K / 4);  // float4s of one split
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  if (q < nq) {
    const f32x4* src = reinterpret_cast<const f32x4*>(p.part) + q;
    int k = wave;
    for (; k + 3 * NW < p.nsplit; k += 4 * NW) {  // four independent loads in flight
      const f32x4 a = src[k * nq], b = src[(k + NW) * nq], c = src[(k + 2 * NW) * nq], d = src[(k + 3 * NW) * nq];
      s += a; s += b; s += c; s += d;
    }
    for (; k < p.nsplit; k += NW) s += src[k * nq];
  }
  if (NW > 1) {
    if (wave) red[wave - 1][lane] = s;
    __syncthreads();
    if (wave) return;
#pragma unroll
    for (int w = 0; w < 3; ++w) s += red[w][lane];
  }
  if (q < nq) wgrad_store(p, int(q / (p.K / 4)), int(q % (p.K / 4)) * 4, s);
}

// The sum launch: four waves a column run from 16 splits (few, narrow tiles: 192 x 192 is 9 of them, so
// the splits are many and the elements few: product and sum over 19,856 rows 12.4 us with four waves
// in 56 splits), one below (768 x 768 over 4964 rows in 14 splits: 22.3 us with four, 21.6 with one).
static void launch_wgrad_sum(const WgradParams& p, hipStream_t stream) {
  const int64_t nq = int64_t(p.N) * (p.K / 4);
  if (p.nsplit >= 16)
    hipLaunchKernelGGL(wgrad_sum_kernel<4>, dim3(unsigned((nq + 63) / 64)), dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL(wgrad_sum_kernel<1>, dim3(unsigned((nq + 255) / 256)), dim3(256), 0, stream, p);
}

// The tile of dW along a width: 128 where it divides, else 64.
static int wgrad_tile(int width) { return width % 128 == 0 ? 128 : 64; }

// Splits of M: about two workgroups per CU over the dW tiles, at least four stages (256 rows) per
// split, every split a whole number of stages and none empty. Sets *mper (rows per split).
static int wgrad_splits(const mote_linear_wgrad_args* a, int* mper) {
  const int tiles = (a->N / wgrad_tile(a->N)) * (a->K / wgrad_tile(a->K));
  const int blocks = (a->M + kWgTok - 1) / kWgTok;
  int s = (2 * device_cu_count()) / (tiles > 0 ? tiles : 1);
  s = s < 1 ? 1 : s;
  const int cap = blocks / 4 < 1 ? 1 : blocks / 4;
  s = s < cap ? s : cap;
  const int per = (blocks + s - 1) / s;
  if (mper) *mper = per * kWgTok;
  return per > 0 ? (blocks + per - 1) / per : 1;
}

size_t linear_wgrad_workspace_bytes(const mote_linear_wgrad_args* a) {
  if (!a || a->M <= 0 || a->N <= 0 || a->K <= 0) return 0;
  const int s = wgrad_splits(a, nullptr);
  return s > 1 ? size_t(s) * size_t(a->N) * size_t(a->K) * sizeof(float) : 0;
}

// Arguments checked, launched (shared by both entry points; `what` names the one that was called).
static int wgrad_launch(const mote_linear_wgrad_args* a, const char* what, hipStream_t stream) {
  if (!a->dw || (a->M > 0 && (!a->a || !a->x))) return set_error(MOTE_ERR_ARGUMENT, "%s: null pointer", what);
  if (a->a_sr < a->N || a->x_sr < a->K || a->dw_sr < a->K || a->a_sr >= (int64_t(1) << 24) ||
      a->x_sr >= (int64_t(1) << 24) || a->dw_sr >= (int64_t(1) << 40))
    return set_error(MOTE_ERR_ARGUMENT, "%s: row strides (a_sr >= N, x_sr >= K, dw_sr >= K; below 2^24 elements)", what);
  auto al16 = [](const void* ptr, int64_t bytes) { return reinterpret_cast<uintptr_t>(ptr) % 16 == 0 && bytes % 16 == 0; };
  const bool f32 = a->dw_dtype == MOTE_F32;
  if ((a->M > 0 && (!al16(a->a, a->a_sr * 2) || !al16(a->x, a->x_sr * 2))) || !al16(a->dw, a->dw_sr * (f32 ? 4 : 2)))
    return set_error(MOTE_ERR_ARGUMENT, "%s: rows must start on 16-byte boundaries", what);
  const int tn = wgrad_tile(a->N), tk = wgrad_tile(a->K);
  WgradParams p;
  p.a = reinterpret_cast<const bf16_t*>(a->a); p.a_sr = a->a_sr;
  p.x = reinterpret_cast<const bf16_t*>(a->x); p.x_sr = a->x_sr;
  p.dw = a->dw; p.dw_sr = a->dw_sr; p.dw_f32 = f32;
  p.M = a->M; p.N = a->N; p.K = a->K;
  p.ntn = a->N / tn; p.ntk = a->K / tk;
  p.part = nullptr;
  if (a->M == 0) {  // an empty reduction: dW = 0
    p.nsplit = 0; p.mper = 0;
    launch_wgrad_sum(p, stream);
    return check_launch(what);
  }
  p.nsplit = wgrad_splits(a, &p.mper);
  if (p.nsplit > 1) {
    const size_t need = linear_wgrad_workspace_bytes(a);
    if (!a->workspace || a->workspace_bytes < need || reinterpret_cast<uintptr_t>(a->workspace) % 16)
      return set_error(MOTE_ERR_WORKSPACE, "%s: workspace too small or misaligned (%zu bytes needed)", what, need);
    p.part = reinterpret_cast<float*>(a->workspace);
  }
  const dim3 grid(unsigned((p.ntn * p.ntk * p.nsplit + 7) / 8 * 8)), block(64 * kWgWaves);
  if (tn == 128 && tk == 128) hipLaunchKernelGGL((wgrad_kernel<128, 128>), grid, block, 0, stream, p);
  else if (tn == 128) hipLaunchKernelGGL((wgrad_kernel<128, 64>), grid, block, 0, stream, p);
  else if (tk == 128) hipLaunchKernelGGL((wgrad_kernel<64, 128>), grid, block, 0, stream, p);
  else hipLaunchKernelGGL((wgrad_kernel<64, 64>), grid, block, 0, stream, p);
  int rc = check_launch(what);
  if (rc || p.nsplit == 1) return rc;
  launch_wgrad_sum(p, stream);
  return check_launch(what);
}

int launch_linear_wgrad(const mote_linear_wgrad_args* a, hipStream_t stream) {
  if (!a) return set_error(MOTE_ERR_ARGUMENT, "linear_wgrad: null args");
  if (a->dtype != MOTE_BF16 || (a->dw_dtype != MOTE_BF16 && a->dw_dtype != MOTE_F32))
    return set_error(MOTE_ERR_ARGUMENT, "linear_wgrad: dtype %d -> %d (bf16 operands, bf16 or fp32 dW)", a->dtype, a->dw_dtype);
  if (a->M < 0 || a->N <= 0 || a->K <= 0 || a->N % 64 || a->K % 64)
    return set_error(MOTE_ERR_SHAPE, "linear_wgrad: M = %d, N = %d, K = %d (N and K multiples of 64)", a->M, a->N, a->K);
  return wgrad_launch(a, "linear_wgrad", stream);
}

static mote_linear_wgrad_args linear_args(const mote_wgrad_args* a) {
  mote_linear_wgrad_args l{};
  l.dtype = l.dw_dtype = a->dtype;
  l.M = a->M; l.N = a->N; l.K = a->K;
  l.a = a->a; l.a_sr = a->a_sr; l.x = a->x; l.x_sr = a->x_sr; l.dw = a->dw; l.dw_sr = a->dw_sr;
  l.workspace = a->workspace; l.workspace_bytes = a->workspace_bytes;
  return l;
}

size_t wgrad_workspace_bytes(const mote_wgrad_args* a) {
  if (!a) return 0;
  const mote_linear_wgrad_args l = linear_args(a);
  return linear_wgrad_workspace_bytes(&l);
}

int launch_wgrad(const mote_wgrad_args* a, hipStream_t stream) {
  if (!a) return set_error(MOTE_ERR_ARGUMENT, "wgrad: null args");
  if (a->dtype != MOTE_BF16) return set_error(MOTE_ERR_ARGUMENT, "wgrad: dtype %d (bf16 only)", a->dtype);
  if (a->M < 0 || a->N <= 0 || a->K <= 0 || a->N % 128 || a->K % 128)
    return set_error(MOTE_ERR_SHAPE, "wgrad: M = %d, N = %d, K = %d (N and K multiples of 128)", a->M, a->N, a->K);
  const mote_linear_wgrad_args l = linear_args(a);
  return wgrad_launch(&l, "wgrad", stream);
}

}  // namespace mote
