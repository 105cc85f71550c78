// Relation forward in fp32 on staged tiles (the algebra of relation_fwd.hip; mote/model/flash_relation.py:76-183).
//
// One workgroup of four waves per 64 query rows of one (sequence, head); blocks of BN key rows (P2 and
// I~) staged global -> LDS by direct transfers, double-buffered, rows as they are in memory with their
// 16-byte chunks XOR-swizzled by the row's low three bits. Wave w owns query half w / 2 and key half
// w % 2 of every block:
//   S^T = K Q^T       v_mfma_f32_16x16x4_f32, A = K rows (two ds_read_b128 a fragment), B = the queries
//                     (registers, loaded once)
//   online softmax per query against an upper bound of its exponents, in log2 units, rescaled only when
//   a block raises it by more than 2^8; row sums in fp32 registers
//   O^T += V^T P^T    A = I~ columns by single-dword LDS reads (lane (li, lg) reads column li of key
//                     4 lg + r: sixteen consecutive floats a lane group), B = P^T straight from the
//                     accumulators
// The two key halves merge through LDS; the epilogue is the other forward kernels'.
//
// What bounds it: the fp32 matrix rate (157 TFLOP/s) where the grid fills the chip, else one walk's
// latency. The register-staged kernel it replaces gave a wave 32 whole query rows, so half the waves,
// each twice the products a block, behind two barriers and a transpose through registers: H 8, B 4,
// T 620, dh 64 84.8 us, 42.6 here (47 TFLOP/s of visible pairs); B 2, H 4, T 256, dh 48 35 and 18; B 2, H 8,
// T 1000, dh 96 198 and 77. BN 64 up to dh 64 (64 KB of LDS, two workgroups a CU), 32 beyond.
#include "common.hpp"
#include "params.hpp"
#include "tiles.hpp"

namespace mote {

template <int DP>
struct F32Shape {
  static constexpr int BN = DP <= 64 ? 64 : 32;
  static constexpr int KT = BN / 32;           // 16-key tiles of a wave's half
  static constexpr int CPR = DP / 4;           // 16-byte chunks per row
  static constexpr int TILE = BN * DP;         // floats of one staged tile
  static constexpr int NINS = 2 * BN * CPR / 64;  // wave transfers per stage (P2 tile, then I~ tile)
  static constexpr int PER = NINS / 4;
  static constexpr int RLD = DP + 4;           // row stride of the merge buffer
  static constexpr int MERGE = 64 * RLD + 128;
  static constexpr int LDS = 4 * TILE > MERGE ? 4 * TILE : MERGE;
};

__device__ __forceinline__ int f32_swz(int row) { return row & 7; }

template <int DP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
relation_fwd_f32_kernel(const FwdParams p) {
  using S = F32Shape<DP>;
  using E = Elem<float>;
  using Frag = E::Frag;
  constexpr int KS = DP / 32, DT = DP / 16, BN = S::BN, KT = S::KT;
  __shared__ __align__(16) float smem[S::LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 15, lg = lane >> 4;
  const int kh = wave & 1, qh = wave >> 1;
  const int h = blockIdx.x % p.H;
  const int rest = blockIdx.x / p.H;
  const int seq = rest % p.nseq;
  const int qb = p.nqb - 1 - rest / p.nseq;
  const int D = p.D;

  int TQs, TKs, qs;
  int64_t qoff, koff, voff, yoff, soff;
  if (p.cu) {
    const int r0 = p.cu[seq];
    TQs = p.cu[seq + 1] - r0;
    TKs = TQs;
    qs = 0;
    qoff = int64_t(r0) * p.q_sr;
    koff = int64_t(r0) * p.k_sr;
    voff = int64_t(r0) * p.v_sr;
    yoff = int64_t(r0) * p.y_sr;
    soff = int64_t(h) * p.total_rows + r0;
  } else {
    TQs = p.TQ;
    TKs = p.TK;
    qs = p.q_start;
    qoff = int64_t(seq) * p.q_sb;
    koff = int64_t(seq) * p.k_sb;
    voff = int64_t(seq) * p.v_sb;
    yoff = int64_t(seq) * p.y_sb;
    soff = (int64_t(seq) * p.H + h) * p.TQ;
  }
  if (qb * 64 >= TQs) return;
  const float* qbase = reinterpret_cast<const float*>(p.p1) + qoff + int64_t(h) * p.q_sh;
  const float* kbase = reinterpret_cast<const float*>(p.p2) + koff + int64_t(h) * p.k_sh;
  const float* vbase = reinterpret_cast<const float*>(p.info) + voff + int64_t(h) * p.v_sh;
  float* ybase = reinterpret_cast<float*>(p.y) + yoff + int64_t(h) * p.y_sh;

  // queries: B fragments of Q^T; columns past D are zero, which keeps the staged copies there out of the scores
  const int q0 = qb * 64 + 32 * qh;
  Frag qf[2][KS];
  int qabs[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int qi = q0 + 16 * s + li;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int d0 = 32 * ks + 8 * lg;
      qf[s][ks] = qi < TQs && d0 < D ? E::load8(qbase + int64_t(qi) * p.q_sr + d0) : E::zero();
    }
    qabs[s] = qs + qi;
  }
  const int qlast = min(TQs, qb * 64 + 64) - 1;
  const int nkb = (qs + qlast + BN - 1) / BN;  // keys j < qs + qlast
  const int wq_last = min(q0 + 31, TQs - 1);
  const float c2 = p.scale * kLog2e;
  float m_run[2] = {0.f, 0.f}, l_run[2] = {0.f, 0.f};
  f32x4 oacc[DT][2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int s = 0; s < 2; ++s) oacc[dt][s] = f32x4{0.f, 0.f, 0.f, 0.f};

  // transfer n of a stage: chunks 64 n .. 64 n + 63 of the P2 tile, then of the I~ tile. Rows past the
  // keys copy the last one, chunks past D the row's last (masked / met by zeros / not stored).
  auto issue = [&](int kb, int stage) {
#pragma unroll
    for (int i = 0; i < S::PER; ++i) {
      const int n = wave + 4 * i;
      const bool isv = n >= S::NINS / 2;
      const int q = 64 * (isv ? n - S::NINS / 2 : n) + lane;
      const int row = q / S::CPR, c = (q % S::CPR) ^ f32_swz(row);
      const int j = min(kb * BN + row, TKs - 1);
      const float* src = (isv ? vbase + int64_t(j) * p.v_sr : kbase + int64_t(j) * p.k_sr) + min(4 * c, D - 4);
      lds_dma16(src, smem + stage * 2 * S::TILE + n * 256);
    }
  };
  if (nkb > 0) issue(0, 0);
  for (int kb = 0; kb < nkb; ++kb) {
    __builtin_amdgcn_s_waitcnt(0);  // this wave's part of block kb
    lds_barrier();                  // every wave's; and every wave is done with block kb - 1's stage
    if (kb + 1 < nkb) issue(kb + 1, (kb + 1) & 1);
    const float* Ks = smem + (kb & 1) * 2 * S::TILE;
    const float* Vs = Ks + S::TILE;
    const int kr = 16 * KT * kh, key0 = kb * BN + kr;  // the wave's first key in the block, and its position
    if (q0 >= TQs || key0 >= qs + wq_last) continue;   // wave-uniform: nothing visible
    f32x4 sacc[KT][2];
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int s = 0; s < 2; ++s) sacc[t][s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        const int row = kr + 16 * t + li, c = 8 * ks + 2 * lg, sw = f32_swz(row);
        const float4 a = *reinterpret_cast<const float4*>(Ks + row * DP + (c ^ sw) * 4);
        const float4 b = *reinterpret_cast<const float4*>(Ks + row * DP + ((c + 1) ^ sw) * 4);
        Frag kf;
        kf.v[0] = a.x; kf.v[1] = a.y; kf.v[2] = a.z; kf.v[3] = a.w;
        kf.v[4] = b.x; kf.v[5] = b.y; kf.v[6] = b.z; kf.v[7] = b.w;
#pragma unroll
        for (int s = 0; s < 2; ++s) sacc[t][s] = E::mma(kf, qf[s][ks], sacc[t][s]);
      }
    const bool masked = key0 + 16 * KT > qs + q0;
    // the block's bound of the exponents: SiLU(U) log2e never exceeds max(U log2e, 0)
    float bnd[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      float mx = kNegInf;
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool keep = !masked || key0 + 16 * t + 4 * lg + r < qabs[s];
          mx = fmaxf(mx, keep ? sacc[t][s][r] : kNegInf);
        }
      bnd[s] = mx;
    }
    const bool need = bnd[0] * c2 > m_run[0] + kRescale || bnd[1] * c2 > m_run[1] + kRescale;
    if (__ballot(need) != 0ull) {
      lanegroup_max2(bnd[0], bnd[1]);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const float b = fmaxf(bnd[s] * c2, 0.f);
        const float mn = b > m_run[s] + kRescale ? b : m_run[s];
        const float alpha = fexp2(m_run[s] - mn);
        l_run[s] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) oacc[dt][s] *= alpha;
        m_run[s] = mn;
      }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float u2 = sacc[t][s][r] * c2;
          const float sg = frcp(1.0f + fexp2(-u2));
          const float pr = fexp2(fmaf(u2, sg, -m_run[s]));
          const bool keep = !masked || key0 + 16 * t + 4 * lg + r < qabs[s];
          sacc[t][s][r] = keep ? pr : 0.f;
          l_run[s] += sacc[t][s][r];
        }
    // O^T += V^T P^T: key 16 t + 4 lg + r in the accumulators' order, four keys an instruction
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = kr + 16 * t + 4 * lg + r, sw = f32_swz(row);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const int c = 4 * dt + (li >> 2);
          const float v = Vs[row * DP + (c ^ sw) * 4 + (li & 3)];
#pragma unroll
          for (int s = 0; s < 2; ++s)
            oacc[dt][s] = __builtin_amdgcn_mfma_f32_16x16x4f32(v, sacc[t][s][r], oacc[dt][s], 0, 0, 0);
        }
      }
  }

  // merge the key halves: kh = 1 hands (m, l, O) to kh = 0 through LDS
#pragma unroll
  for (int s = 0; s < 2; ++s) l_run[s] = lanegroup_sum(l_run[s]);
  float* R = smem;
  float* RM = R + 64 * S::RLD;
  __syncthreads();  // every wave is done reading the stages (the last step waited for every transfer)
  if (kh == 1) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int row = 32 * qh + 16 * s + li;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(&R[row * S::RLD + 16 * dt + 4 * lg]) = oacc[dt][s];
      if (lg == 0) {
        RM[row] = m_run[s];
        RM[64 + row] = l_run[s];
      }
    }
  }
  __syncthreads();
  if (kh == 1) return;
  const float lam = *p.lam;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int row = 32 * qh + 16 * s + li;
    const float m1 = RM[row], l1 = RM[64 + row];
    const float mm = fmaxf(m_run[s], m1);
    const float a0 = fexp2(m_run[s] - mm), a1 = fexp2(m1 - mm);
    const float lt = l_run[s] * a0 + l1 * a1;
    const int qi = q0 + 16 * s + li;
    const bool qv = qi < TQs;
    const int qa = qs + qi;
    const bool has = lt > 0.f;
    // the running bound starts at 0, so the logarithm holds most of lse: its exponent is added exactly
    const float lse = has ? (mm + (float)__builtin_amdgcn_frexp_expf(lt) + __log2f(__builtin_amdgcn_frexp_mantf(lt))) * kLn2
                          : kNegInf;
    const float inv_l = has ? 1.0f / lt : 0.f;
    float ud = 0.f;
    if (qv) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int d0 = 32 * ks + 8 * lg;
        if (d0 < D) {
          const Frag kr8 = E::load8(kbase + int64_t(qa) * p.k_sr + d0);
#pragma unroll
          for (int j = 0; j < 8; ++j) ud = fmaf(qf[s][ks].v[j], kr8.v[j], ud);
        }
      }
    }
    ud += wave_xor(ud, 16);
    ud += wave_xor(ud, 32);
    const float sself = sigmoid_acc(ud * p.scale * p.tau_inv);
    const float gate = has ? sigmoid_acc(lse - lam * logf((float)qa + 1.0f) - sself) : 0.f;
    if (!qv) continue;
    const float* irow = vbase + int64_t(qa) * p.v_sr;
    float* yrow = ybase + int64_t(qi) * p.y_sr;
    float* brow = p.ibar + (soff + qi) * int64_t(D);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d0 = 16 * dt + 4 * lg;
      if (d0 >= D) continue;
      const f32x4 ib = (oacc[dt][s] * a0 + *reinterpret_cast<const f32x4*>(&R[row * S::RLD + d0]) * a1) * inv_l;
      const f32x4 iv = *reinterpret_cast<const f32x4*>(irow + d0);
      *reinterpret_cast<f32x4*>(yrow + d0) = (1.0f - gate) * iv + gate * ib;
      *reinterpret_cast<f32x4*>(brow + d0) = ib;
    }
    if (lg == 0) {
      p.lse[soff + qi] = lse;
      p.g[soff + qi] = gate;
    }
  }
}

// fp.nqb is set here: one workgroup per 64 query rows.
void launch_fwd_f32(FwdParams fp, int DP, hipStream_t stream) {
  fp.nqb = (fp.TQ + 63) / 64;
  const dim3 grid(unsigned(int64_t(fp.nseq) * fp.H * fp.nqb));
  switch (DP) {
    case 32: hipLaunchKernelGGL(relation_fwd_f32_kernel<32>, grid, dim3(256), 0, stream, fp); break;
    case 64: hipLaunchKernelGGL(relation_fwd_f32_kernel<64>, grid, dim3(256), 0, stream, fp); break;
    case 96: hipLaunchKernelGGL(relation_fwd_f32_kernel<96>, grid, dim3(256), 0, stream, fp); break;
    default: hipLaunchKernelGGL(relation_fwd_f32_kernel<128>, grid, dim3(256), 0, stream, fp); break;
  }
}

}  // namespace mote
