// Key-block stage of the fp32 backward (the algebra at relation_bwd.hip's head), and the dP1 stage that
// reads the dU it stores.
//
// Keys: one workgroup of 2 NQ waves per 32 keys of one (batch, head), longest walk first; blocks of 16 NQ
// query rows (the rows stage's padded P1 and dI-bar copies) staged global -> LDS by direct transfers,
// double buffered, rows as they are with their 16-byte chunks XOR-swizzled by the row's low three bits.
// Wave w owns 16 keys (w % 2) and 16 queries (w / 2) of every block:
//   U = Q K^T, dW = dI-bar V^T   queries in the accumulator rows, the wave's keys in the columns; its P2 and
//                                I~ fragments stay in registers
//   dV += W^T dI-bar, dK += dU^T Q   A = w / dU straight from the accumulators, B = dI-bar / Q columns by
//                                single-dword LDS reads
// The query parts add dV and dK through LDS at the end; the Self terms join before the stores. dU:
//   kStore  to memory as 16 x 16 tiles, [key][query]: a wave's tile is one contiguous KB
//   kAtomic dQ = dU K over the 32 keys (dU through LDS) added to the fp32 accumulator with hardware float
//           atomics
//   kNone   nothing: the query-stationary kernel of relation_bwd.hip recomputes it
// dP1 (after kStore): one workgroup per 32 queries, 64-key P2 blocks staged as above, wave w owning 16
// queries and 32 keys of each, its dU columns loaded one block ahead.
//
// What bounds it: the fp32 matrix rate where the grid fills the chip, else key block 0's walk. The float
// atomics came to some 120 G adds a second over the device, more time than the products: B 4, H 8, T 620,
// dh 64: keys 117 us with them, 60 without; 4 bytes a visible pair written and read cost less.
// Whole backward there: 123 us register-staged with atomics, 87 here; B 2,
// H 4, T 256, dh 48: 49 and 30; B 2, H 8, T 1000, dh 96: 227 and 136; H 4, T 3000, dh 64: 405 and 201.
#include "bwd.hpp"
#include "common.hpp"
#include "tiles.hpp"

namespace mote {

enum DuMode { kNone, kAtomic, kStore };

__device__ __forceinline__ int f32_row_swz(int row) { return row & 7; }

// dU tile of (16-query tile q16, 16-key tile k16): [16 keys][16 queries]
__device__ __forceinline__ float* du_tile(const BwdParams& p, int bh, int q16, int k16) {
  const int64_t pair = int64_t(bh) * p.npairs + PairTable::offset(q16 / 4, p.q_start) + k16 / 4;
  return reinterpret_cast<float*>(p.dut) + (pair * 16 + (q16 % 4) * 4 + k16 % 4) * 256;
}

template <int DP, int NQ, DuMode MODE>
__global__ void __launch_bounds__(128 * NQ) __attribute__((amdgpu_waves_per_eu(2)))
bwd_keys_f32_kernel(const BwdParams p) {
  static_assert(MODE != kAtomic || NQ == 2);
  using E = Elem<float>;
  using Frag = E::Frag;
  constexpr int KS = DP / 32, DT = DP / 16, CPR = DP / 4, R = 16 * NQ, ULD = 36;
  constexpr int TILE = R * DP;               // floats of one staged tile
  constexpr int NINS = 2 * R * CPR / 64;     // wave transfers per stage: the P1 tile's, then the dI-bar tile's
  constexpr int PER = NINS / (2 * NQ);
  // vector-memory operations of a wave after a block's transfers, always issued, so the wait can count them
  constexpr int AFTER = MODE == kAtomic ? DT / 2 * 4 : MODE == kStore ? 1 : 0;
  constexpr bool WITH_DQ = MODE == kAtomic;
  __shared__ __align__(16) float smem[4 * TILE + (WITH_DQ ? 32 * DP + 32 * ULD : 0)];
  float* const Kt = smem + 4 * TILE;  // the workgroup's 32 P2 rows
  float* const dUs = Kt + 32 * DP;    // [32 queries][ULD]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int kt = wave & 1, qt = wave >> 1;
  const int BH = p.B * p.H;
  const int bh = blockIdx.x % BH, kb = blockIdx.x / BH;
  const int b = bh / p.H, h = bh % p.H;
  const int k0 = kb * 32, D = p.D;
  const float* kbase = reinterpret_cast<const float*>(p.p2) + b * p.k_sb + h * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.info) + b * p.v_sb + h * p.v_sh;
  const float* wq = reinterpret_cast<const float*>(p.wq) + int64_t(bh) * p.TQp * DP;
  const float* wd = reinterpret_cast<const float*>(p.wdib) + int64_t(bh) * p.TQp * DP;
  const float* lse2 = p.lse2 + int64_t(bh) * p.TQp;
  const float* cvec = p.cvec + int64_t(bh) * p.TQp;

  // the wave's 16 keys as B fragments (k = head dim, column = key); zero past the keys and past D
  const int jw = k0 + 16 * kt + li;
  Frag kf[KS], vf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = 32 * ks + 8 * lg;
    const bool ok = jw < p.TK && d0 < D;
    kf[ks] = ok ? E::load8(kbase + int64_t(jw) * p.k_sr + d0) : E::zero();
    vf[ks] = ok ? E::load8(vbase + int64_t(jw) * p.v_sr + d0) : E::zero();
  }
  // the P2 tile for dQ; zero past the keys and past D
  if constexpr (WITH_DQ) {
    for (int q = tid; q < 32 * CPR; q += 256) {
      const int row = q / CPR, c = q % CPR;
      const bool ok = k0 + row < p.TK && 4 * c < D;
      store_chunk(Kt + row * DP + (c ^ f32_row_swz(row)) * 4, ok ? load_chunk(kbase + int64_t(k0 + row) * p.k_sr + 4 * c) : zero_chunk());
    }
  }
  // query blocks that see a key of this block; none at all see keys from the last query's position on
  const int nqb = k0 < p.q_start + p.TQ - 1 ? (p.TQ + R - 1) / R : 0;
  const int qb_lo = max(0, k0 + 1 - p.q_start) / R;
  uint32_t voff[PER];  // bytes from the block's first row
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int n = wave + 2 * NQ * i;  // transfer n of the stage: its chunks 64 n .. 64 n + 63
    const int q = 64 * (n >= NINS / 2 ? n - NINS / 2 : n) + lane;
    const int row = q / CPR;
    voff[i] = uint32_t(row * DP + 4 * ((q % CPR) ^ f32_row_swz(row))) * 4;
  }
  auto issue = [&](int qb, int stage) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int n = wave + 2 * NQ * i;
      const float* base = (n >= NINS / 2 ? wd : wq) + int64_t(qb) * TILE;
      lds_dma16_s(base, voff[i], smem + stage * 2 * TILE + n * 256);
    }
  };
  f32x4 dvacc[DT], dkacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    dvacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    dkacc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const float c2 = p.scale * kLog2e;
  const int qr = 16 * qt;  // the wave's first query row in a block
  f32x4 lv = {0.f, 0.f, 0.f, 0.f}, cv = {0.f, 0.f, 0.f, 0.f};
  if (qb_lo < nqb) {
    lv = *reinterpret_cast<const f32x4*>(lse2 + qb_lo * R + qr + 4 * lg);
    cv = *reinterpret_cast<const f32x4*>(cvec + qb_lo * R + qr + 4 * lg);
    issue(qb_lo, 0);
  }
  __builtin_amdgcn_s_waitcnt(0);
  for (int qb = qb_lo; qb < nqb; ++qb) {
    const int n = qb - qb_lo;
    // everything older than the previous block's AFTER operations has completed: this block's transfers
    __builtin_amdgcn_s_waitcnt(kVmWaitStage<AFTER>());
    lds_barrier();  // every wave's part is in; every wave is done with the other stage and with dUs
    f32x4 lvn = lv, cvn = cv;
    if (qb + 1 < nqb) {
      lvn = *reinterpret_cast<const f32x4*>(lse2 + (qb + 1) * R + qr + 4 * lg);
      cvn = *reinterpret_cast<const f32x4*>(cvec + (qb + 1) * R + qr + 4 * lg);
      issue(qb + 1, (n + 1) & 1);
    }
    const float* Qs = smem + (n & 1) * 2 * TILE;
    const float* Ds = Qs + TILE;
    const int i0 = qb * R + qr;  // the wave's first query row
    f32x4 sacc = {0.f, 0.f, 0.f, 0.f}, wacc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int row = qr + li, c = 8 * ks + 2 * lg, sw = f32_row_swz(row);
      auto frag = [&](const float* t) {
        const float4 a = *reinterpret_cast<const float4*>(t + row * DP + (c ^ sw) * 4);
        const float4 e = *reinterpret_cast<const float4*>(t + row * DP + ((c + 1) ^ sw) * 4);
        Frag f;
        f.v[0] = a.x; f.v[1] = a.y; f.v[2] = a.z; f.v[3] = a.w;
        f.v[4] = e.x; f.v[5] = e.y; f.v[6] = e.z; f.v[7] = e.w;
        return f;
      };
      sacc = E::mma(frag(Qs), kf[ks], sacc);
      wacc = E::mma(frag(Ds), vf[ks], wacc);
    }
    // w and dU of query i0 + 4 lg + r, key jw
    float wv[4], uv[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float u2 = sacc[r] * c2;
      const float sg = frcp(1.0f + fexp2(-u2));
      float w = fexp2(u2 * sg - lv[r]);
      if (jw >= p.q_start + i0 + 4 * lg + r) w = 0.f;
      const float u = sacc[r] * p.scale;
      wv[r] = w;
      uv[r] = w * (wacc[r] + cv[r]) * (sg * (1.0f + u * (1.0f - sg)));
      if constexpr (WITH_DQ) dUs[(qr + 4 * lg + r) * ULD + 16 * kt + li] = uv[r];
    }
    if constexpr (MODE == kStore)
      *reinterpret_cast<f32x4*>(du_tile(p, bh, i0 / 16, k0 / 16 + kt) + li * 16 + 4 * lg) = f32x4{uv[0], uv[1], uv[2], uv[3]};
    // dV += W^T dI-bar, dK += dU^T Q over the wave's 16 queries, four an instruction
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = qr + 4 * lg + r, sw = f32_row_swz(row);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int off = row * DP + ((4 * dt + (li >> 2)) ^ sw) * 4 + (li & 3);
        dvacc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[r], Ds[off], dvacc[dt], 0, 0, 0);
        dkacc[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(uv[r], Qs[off], dkacc[dt], 0, 0, 0);
      }
    }
    if constexpr (WITH_DQ) {
      lds_barrier();  // the four waves' dU
      // dQ = dU K over the 32 keys: query tile w % 2, head-dim tiles w / 2, w / 2 + 2, ...; keys in the order
      // 4 lg + r, 16 + 4 lg + r of both operands
      const int dqt = wave & 1;
      const float* ur = dUs + (16 * dqt + li) * ULD + 4 * lg;
      const f32x4 ua = *reinterpret_cast<const f32x4*>(ur), ub = *reinterpret_cast<const f32x4*>(ur + 16);
#pragma unroll
      for (int i = 0; i < DT / 2; ++i) {
        const int dt = (wave >> 1) + 2 * i;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 4 * lg + r, sw = f32_row_swz(row);  // row + 16 has the same swizzle
          const int off = row * DP + ((4 * dt + (li >> 2)) ^ sw) * 4 + (li & 3);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ua[r], Kt[off], acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ub[r], Kt[off + 16 * DP], acc, 0, 0, 0);
        }
        // every block issues its AFTER adds: columns past D add zero to the row's own columns, each lane to
        // another one; rows past TQ are in the last block alone, whose adds nothing counts, and add nothing
        // (as zeros to one element, 4096 cached keys after one another took 170 us at T = 1)
        const int d = 16 * dt + li;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int qi = qb * 32 + 16 * dqt + 4 * lg + r;
          if (qi < p.TQ)
            unsafeAtomicAdd(&p.dp1acc[(int64_t(bh) * p.TQ + qi) * D + d % D], d < D ? acc[r] * p.scale : 0.f);
        }
      }
    }
    lv = lvn;
    cv = cvn;
  }

  // add the query parts through LDS, then the Self terms of key rows that are also queries and the
  // single store of dP2 and dI~
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  float* Rd = smem;  // [NQ - 1][2][32 keys][DP]
  if (qt > 0) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int o = (qt - 1) * 64 * DP + (16 * kt + 4 * lg + r) * DP + 16 * dt + li;
        Rd[o] = dvacc[dt][r];
        Rd[32 * DP + o] = dkacc[dt][r];
      }
  }
  __syncthreads();
  if (qt > 0) return;
  const float* q = reinterpret_cast<const float*>(p.p1) + b * p.q_sb + h * p.q_sh;
  const float* dy = reinterpret_cast<const float*>(p.dy) + b * p.y_sb + h * p.y_sh;
  float* dk = reinterpret_cast<float*>(p.dp2) + b * p.dk_sb + h * p.dk_sh;
  float* dv = reinterpret_cast<float*>(p.dinfo) + b * p.dv_sb + h * p.dv_sh;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 16 * kt + 4 * lg + r, j = k0 + row;
    if (j >= p.TK) continue;
    const int i = j - p.q_start;
    const float gs = i >= 0 ? p.g[int64_t(bh) * p.TQ + i] : 0.f;
    const float us = i >= 0 ? p.duii[int64_t(bh) * p.TQp + i] : 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d = 16 * dt + li;
      if (d >= D) continue;
      float vv = dvacc[dt][r], kk = dkacc[dt][r];
#pragma unroll
      for (int n = 0; n < NQ - 1; ++n) {
        vv += Rd[(64 * n + row) * DP + d];
        kk += Rd[(64 * n + 32 + row) * DP + d];
      }
      if (i >= 0) {
        vv += (1.0f - gs) * dy[int64_t(i) * p.y_sr + d];
        kk += us * q[int64_t(i) * p.q_sr + d];
      }
      dv[int64_t(j) * p.dv_sr + d] = vv;
      dk[int64_t(j) * p.dk_sr + d] = kk * p.scale;
    }
  }
}

template <int DP>
__global__ void __launch_bounds__(256) bwd_dq_f32_kernel(const BwdParams p) {
  constexpr int DT = DP / 16, CPR = DP / 4, TILE = 64 * DP;
  constexpr int PER = CPR / 4;  // 64 CPR chunks a stage, 64 a transfer, four waves
  __shared__ __align__(16) float smem[2 * TILE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int kh = wave & 1, qt = wave >> 1;
  const int BH = p.B * p.H;
  const int bh = blockIdx.x % BH;
  const int qb = (p.TQ + 31) / 32 - 1 - blockIdx.x / BH;
  const int b = bh / p.H, h = bh % p.H;
  const int D = p.D;
  if (blockIdx.x == gridDim.x - 1) {  // the shortest walk also sums dlam
    dlam_sum(p.dlam_part, BH * (p.TQp / kRowBlock), p.dlam, smem);
    __syncthreads();
  }
  const float* kbase = reinterpret_cast<const float*>(p.p2) + b * p.k_sb + h * p.k_sh;
  const int kend = p.q_start + min(p.TQ, 32 * qb + 32) - 1;  // keys j < kend
  const int nkb = (kend + 63) / 64;
  // rows past the keys copy the last one (their dU is zero), chunks past D the row's last (not stored)
  auto issue = [&](int kb, int stage) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int n = wave + 4 * i;
      const int q = 64 * n + lane, row = q / CPR, c = (q % CPR) ^ f32_row_swz(row);
      lds_dma16(kbase + int64_t(min(kb * 64 + row, p.TK - 1)) * p.k_sr + min(4 * c, D - 4), smem + stage * TILE + n * 256);
    }
  };
  // dU of query li, keys 16 t + 4 lg + r of the wave's 32; a half that no query sees was not written
  float u[2][4], un[2][4];
  auto load_u = [&](int kb, float (&v)[2][4]) {
    if (kb * 64 + 32 * kh >= kend) return;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const float* tile = du_tile(p, bh, 2 * qb + qt, 4 * kb + 2 * kh + t);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[t][r] = tile[(4 * lg + r) * 16 + li];
    }
  };
  f32x4 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (nkb > 0) {
    issue(0, 0);
    load_u(0, un);
  }
  for (int kb = 0; kb < nkb; ++kb) {
    __builtin_amdgcn_s_waitcnt(0);  // this wave's part of block kb
    lds_barrier();                  // every wave's; and every wave is done with block kb - 1's stage
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) u[t][r] = un[t][r];
    if (kb + 1 < nkb) {
      issue(kb + 1, (kb + 1) & 1);
      load_u(kb + 1, un);
    }
    if (kb * 64 + 32 * kh >= kend) continue;  // wave-uniform
    const float* Ks = smem + (kb & 1) * TILE + 32 * kh * DP;
    f32x4 blk[DT];  // the block's sum by itself, as the atomics add it: a chain over every key would round more
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) blk[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * t + 4 * lg + r, sw = f32_row_swz(row);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          blk[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(u[t][r], Ks[row * DP + ((4 * dt + (li >> 2)) ^ sw) * 4 + (li & 3)],
                                                        blk[dt], 0, 0, 0);
      }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] += blk[dt];
  }
  // add the key halves through LDS, then the Self term and the store
  __syncthreads();
  if (kh == 1) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) smem[(16 * qt + 4 * lg + r) * DP + 16 * dt + li] = acc[dt][r];
  }
  __syncthreads();
  if (kh == 1) return;
  float* out = reinterpret_cast<float*>(p.dp1) + b * p.dq_sb + h * p.dq_sh;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 16 * qt + 4 * lg + r, i = 32 * qb + row;
    if (i >= p.TQ) continue;
    const float us = p.duii[int64_t(bh) * p.TQp + i];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d = 16 * dt + li;
      if (d < D)
        out[int64_t(i) * p.dq_sr + d] =
            (acc[dt][r] + smem[row * DP + d] + us * kbase[int64_t(p.q_start + i) * p.k_sr + d]) * p.scale;
    }
  }
}

template <int DP>
static void launch_keys_t(const BwdParams& p, bool with_dq, hipStream_t stream) {
  const dim3 grid(unsigned((p.TK + 31) / 32 * p.B * p.H));
  // Eight waves and 64-query blocks halve the walk of a workgroup, four and 32 leave more workgroups on a CU
  // to cover each other's waits. Beyond two workgroups per CU the walk no longer bounds (whole backward,
  // eight and four waves): 376 workgroups (H 4, T 3000, dh 64) 202 and 249 us, 512 (B 2, H 8, T 1000, dh 96)
  // 135 and 146; 640 (B 4, H 8, T 620, dh 64) 90 and 87, 960 (B 16, H 6, T 300, dh 32) 46 and 42, 2016 (B 4,
  // H 8, T 2000, dh 96) 811 and 673.
  const bool wide = int(grid.x) <= 2 * device_cu_count();
  if (p.dut && wide) hipLaunchKernelGGL((bwd_keys_f32_kernel<DP, 4, kStore>), grid, dim3(512), 0, stream, p);
  else if (p.dut) hipLaunchKernelGGL((bwd_keys_f32_kernel<DP, 2, kStore>), grid, dim3(256), 0, stream, p);
  else if (with_dq) hipLaunchKernelGGL((bwd_keys_f32_kernel<DP, 2, kAtomic>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((bwd_keys_f32_kernel<DP, 2, kNone>), grid, dim3(256), 0, stream, p);
}

void launch_bwd_keys_f32(const BwdParams& p, int DP, bool with_dq, hipStream_t stream) {
  switch (DP) {
    case 32: launch_keys_t<32>(p, with_dq, stream); break;
    case 64: launch_keys_t<64>(p, with_dq, stream); break;
    case 96: launch_keys_t<96>(p, with_dq, stream); break;
    default: launch_keys_t<128>(p, with_dq, stream); break;
  }
}

void launch_bwd_dq_f32(const BwdParams& p, int DP, hipStream_t stream) {
  const dim3 grid(unsigned((p.TQ + 31) / 32 * p.B * p.H));
  switch (DP) {
    case 32: hipLaunchKernelGGL(bwd_dq_f32_kernel<32>, grid, dim3(256), 0, stream, p); break;
    case 64: hipLaunchKernelGGL(bwd_dq_f32_kernel<64>, grid, dim3(256), 0, stream, p); break;
    case 96: hipLaunchKernelGGL(bwd_dq_f32_kernel<96>, grid, dim3(256), 0, stream, p); break;
    default: hipLaunchKernelGGL(bwd_dq_f32_kernel<128>, grid, dim3(256), 0, stream, p); break;
  }
}

}  // namespace mote
