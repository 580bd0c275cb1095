// Edge-parallel backward at H = O = M = 256 (bf16, gfx950), equivariant and MPNN.
//
// Each wave runs the whole chain of its own 16 edges in registers, features on the MFMA rows, every stage's C-blocks
// the next stage's B operand:
//   S1 m1, SiLU'   S2 m, SiLU'   S3 q -> phi, g_q = g_phi w2_mov SiLU'(q)   S4 g_a2 = (gm_i + W1_mov g_q) SiLU'(pre2)
//   S5 g_a1 = (W_hl g_a2) SiLU'(pre1)   S6 dL/ddelta = phi gx_i + 2 (w_d . g_a1) delta
// No activation leaves the wave but the factors m1, m, g_q, g_a2 and Gh that the factor products and the node
// reduction read.  The four 256 x 256 operands (512 KB) go through two LDS buffers in the order of use, 64 rows
// (32 KB) at a time, shared by the block's eight waves: the next chunk's loads are in flight during the
// products of the current one and stored after them, one barrier per chunk, 16 chunks for 128 edges.  dw2_mov = sum g_phi p and
// dw_d = sum r^2 g_a1 are summed over the 16 edges by a halving exchange (16 values a lane -> one) and kept in
// registers over the passes: one partial row [M | H] per block.
// One block per CU, two waves per SIMD; vector and matrix issue (0.40 and 0.20 of the cycles) and the waits of LDS operand
// reads and barriers bound it.
// Measured against the kernel that shares a 32-edge tile over eight waves by feature rows (661k edges, F_E = 32):
// 990 -> 775 us; the weights' loads through generic pointers, whose waits join those of the LDS, cost 20 us of it.
// Every stage sums in the order of egnn_wide.hip (biases, P_i and Q_j onto the finished products, g_m as the first term), so
// the factors and Gh are bit for bit those of that kernel.
// A lane past the last edge computes that edge again and stores the same values, so no store is under a branch.
#include "egnn_device.h"
#include "egnn_internal.h"
#include "egnn_tile.h"

namespace egnn {
namespace {

using namespace tile;

constexpr int kWaves = 8, H = 256, O = 256, M = 256, KH = H / 32, kRB = 4, kST = H / (16 * kRB);   // kST chunks a stage
constexpr int kChunkElems = kRB * KH * kFragElems;

template <bool EQ, int NU>   // NU: 32-slot slices of the edge input (1 or 2)
__global__ __launch_bounds__(64 * kWaves, 2) void wide_bwd_ep_kernel(BwdArgs a) {
  constexpr int NCH = (EQ ? 4 : 2) * kST;
  __shared__ __attribute__((aligned(16))) bf16 s_w[2][kChunkElems];
  __shared__ __attribute__((aligned(16))) bf16 s_u[2 * KH * NU * kFragElems];
  __shared__ __attribute__((aligned(16))) float s_vec[O + 2 * M + H];   // b2 | bx1 | w2_mov | w_d
  __shared__ __attribute__((aligned(16))) bf16x4 s_d1[kWaves][H / 32][64];   // SiLU'(pre1) of the second half of the rows, to S5
  static_assert(sizeof(float) * kWaves * (M + H) <= sizeof(s_w[0]), "the final sums reuse a weight buffer");

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  const bf16* PQ = (const bf16*)a.PQ;
  const bf16* ef = (const bf16*)a.ef;
  const int64_t E = a.E;
  const int FE = a.FE;
  const int64_t npass = (E + 16 * kWaves - 1) / (16 * kWaves);

  for (int q = threadIdx.x; q < 2 * KH * NU * 64; q += 64 * kWaves)
    reinterpret_cast<bf16x8*>(s_u)[q] = reinterpret_cast<const bf16x8*>(a.fr.u)[q];
  for (int q = threadIdx.x; q < O; q += 64 * kWaves) {
    s_vec[q] = a.fr.b2f[q];
    if constexpr (EQ) {
      s_vec[O + q] = a.fr.bx1f[q];
      s_vec[O + M + q] = a.fr.w2mf[q];
      s_vec[O + 2 * M + q] = a.fr.wdf[q];
    }
  }
  bf16x8 st[4];
  // the lane's offset and the matrices' bases, made opaque once per pass: no chunk addresses hoisted out of the loop
  uint32_t so = threadIdx.x * 16;
  // (in the global address space: a generic load is counted with the LDS reads, whose waits would include it)
  typedef const __attribute__((address_space(1))) char* gptr;
  gptr f0 = (gptr)a.fr.hlT, f1 = (gptr)a.fr.movT, f2 = (gptr)a.fr.mov, f3 = (gptr)a.fr.hl;
  auto stream_load = [&](int ch) {   // W_hl^T (S2), W1_mov^T (S3), W1_mov (S4), W_hl (S5)
    const int s = EQ ? ch / kST : 3 * (ch / kST);
    gptr src = (s == 0 ? f0 : s == 1 ? f1 : s == 2 ? f2 : f3) + (ch % kST) * (kChunkElems * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) st[i] = *(const __attribute__((address_space(1))) bf16x8*)(src + i * (64 * kWaves * 16) + so);
  };
  auto stream_store = [&](int buf) {
    bf16* dst = s_w[buf] + threadIdx.x * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<bf16x8*>(dst + i * 64 * kWaves * 8) = st[i];
  };
  // 32 rows (half hh of chunk ch) of a product: acc[row block] += W . B.  After the second half the next chunk is
  // stored and the one after it requested, before the epilogue's stores, so that no wait for it includes those
  auto rows = [&](int ch, int hh, const bf16x8* B, f32x4* acc) {
    const bf16* W = s_w[ch & 1] + (2 * hh * KH * 64 + l) * 8;
    bf16x8 A0 = load_chunk(W), A1 = load_chunk(W + KH * kFragElems);
#pragma unroll
    for (int kc = 0; kc < KH; ++kc) {
      bf16x8 N0 = A0, N1 = A1;
      if (kc + 1 < KH) {
        N0 = load_chunk(W + (kc + 1) * kFragElems);
        N1 = load_chunk(W + (KH + kc + 1) * kFragElems);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma(acc[0], A0, B[kc]);
      mma(acc[1], A1, B[kc]);
      __builtin_amdgcn_sched_barrier(0);
      A0 = N0;
      A1 = N1;
    }
    if (hh == 1) {
      stream_store((ch + 1) & 1);
      stream_load((ch + 2) % NCH);
    }
  };
  stream_load(0);
  stream_store(0);
  stream_load(1);
  float sw2[EQ ? kST : 1] = {}, swd[EQ ? kST : 1] = {};   // the lane's sums of dw2_mov and dw_d: feature fsum of each 64
  const int fsum = 16 * (c >> 2) + 4 * g + (c & 3);
  __syncthreads();

  // the edge's row, source and edge id, one pass ahead (without edge ids a stand-in read, ignored)
  const int32_t* eidp = a.eids ? a.eids : a.erow;
  int n_ri, n_rj, n_eid;
  auto load_ids = [&](int64_t p) {
    const int64_t q = (p * kWaves + w) * 16 + c, e = q < E ? q : E - 1;
    n_ri = a.erow[e];
    n_rj = a.col[e];
    n_eid = eidp[e];
  };
  load_ids(blockIdx.x);
  for (int64_t ps = blockIdx.x; ps < npass; ps += gridDim.x) {
    __asm__ __volatile__("" : "+v"(so), "+s"(f0), "+s"(f1), "+s"(f2), "+s"(f3));
    const int64_t e0 = (ps * kWaves + w) * 16 + c;
    const bool valid = e0 < E;
    const int64_t e = valid ? e0 : E - 1;
    const int ri = clampi(n_ri, (int)a.N), rj = clampi(n_rj, (int)a.N);
    const int64_t fo = e * H + 4 * g;   // the lane's first element of the edge's rows
    auto store_rows = [&](void* D, int rb, const f32x4& v) { *reinterpret_cast<bf16x4*>((bf16*)D + fo + 16 * rb) = pack4(v); };
    f32x4 ga = zero4(), gb = zero4();   // r^2, g_phi, delta xy | delta z, grad x_i
    if constexpr (EQ) {
      ga = *reinterpret_cast<const f32x4*>(a.geo + e * 8);
      gb = *reinterpret_cast<const f32x4*>(a.geo + e * 8 + 4);
    }
    bf16x8 u[NU];
    {
      const int eid = a.eids ? clampi(n_eid, (int)E) : (int)e;
#pragma unroll
      for (int uc = 0; uc < NU; ++uc) {
        const int s0 = 32 * uc + 8 * g;
        u[uc] = zero_chunk<bf16>();
        if (s0 + 8 <= FE) u[uc] = load_chunk(ef + (int64_t)eid * a.se + s0);
        else if (EQ && s0 == FE) {   // r^2 as a bf16 hi + lo pair
          const bf16 hi = (bf16)ga[0];
          u[uc][0] = hi;
          u[uc][1] = (bf16)(ga[0] - (float)hi);
        }
      }
    }
    // ---- S1
    bf16x8 m1[KH];
    bf16x4 s1[H / 32];
#pragma unroll
    for (int k4 = 0; k4 < KH; k4 += 4) {
      bf16x8 p[4], q[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        p[k] = load_chunk(PQ + (int64_t)ri * 2 * H + 32 * (k4 + k) + 8 * g);
        q[k] = load_chunk(PQ + (int64_t)rj * 2 * H + H + 32 * (k4 + k) + 8 * g);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int kc = k4 + k;
        f32x4 y[2] = {zero4(), zero4()}, pv[2], qv[2];
        unpack_chunk(p[k], pv[0], pv[1]);
        unpack_chunk(q[k], qv[0], qv[1]);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
          for (int uc = 0; uc < NU; ++uc) mma(y[b], load_chunk(s_u + (((2 * kc + b) * NU + uc) * 64 + l) * 8), u[uc]);
          f32x4 d;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const YD r = silu_yd<bf16>(y[b][i] + pv[b][i] + qv[b][i]);
            y[b][i] = r.y;
            d[i] = r.d;
          }
          if (kc < KH / 2) s1[(2 * kc + b) % (H / 32)] = pack4(d);
          else s_d1[w][(2 * kc + b) % (H / 32)][l] = pack4(d);
          store_rows(a.Dm1, 2 * kc + b, y[b]);
        }
        m1[kc] = pack_chunk<bf16>(y[0], y[1]);
      }
    }
    // ---- S2
    bf16x8 mc[EQ ? O / 32 : 1];
    bf16x4 s2[O / 16];
#pragma unroll
    for (int k = 0; k < O / 32; ++k) {   // 32 rows at a time, chunk k / 2
      f32x4 acc[2] = {zero4(), zero4()};
      rows(k >> 1, k & 1, m1, acc);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const f32x4 b2 = *reinterpret_cast<const f32x4*>(s_vec + 32 * k + 16 * b + 4 * g);
        f32x4 d;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const YD r = silu_yd<bf16>(acc[b][i] + b2[i]);
          acc[b][i] = r.y;
          d[i] = r.d;
        }
        s2[2 * k + b] = pack4(d);
        if constexpr (EQ) store_rows(a.Dm, 2 * k + b, acc[b]);
      }
      if constexpr (EQ) mc[k] = pack_chunk<bf16>(acc[0], acc[1]);
      if (k & 1) __syncthreads();
    }
    // the gradient rows of S4, 32 features ahead of their use
    const bf16* gm = (const bf16*)a.gmsg + (int64_t)ri * a.sgm + 4 * g;
    bf16x4 gr0, gr1;
    if constexpr (!EQ) {
      gr0 = *reinterpret_cast<const bf16x4*>(gm);
      gr1 = *reinterpret_cast<const bf16x4*>(gm + 16);
    }
    // ---- S3: phi, g_q, dw2_mov
    float phi = 0.f;
    bf16x8 gq[EQ ? M / 32 : 1];
    if constexpr (EQ) {
      const float gphi = ga[1], gpm = valid ? gphi : 0.f;
      float pv[16];
#pragma unroll
      for (int k = 0; k < M / 32; ++k) {
        f32x4 acc[2] = {zero4(), zero4()};
        if (k + 1 == M / 32) {
          gr0 = *reinterpret_cast<const bf16x4*>(gm);
          gr1 = *reinterpret_cast<const bf16x4*>(gm + 16);
        }
        rows(kST + (k >> 1), k & 1, mc, acc);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const f32x4 bx = *reinterpret_cast<const f32x4*>(s_vec + O + 32 * k + 16 * b + 4 * g);
          const f32x4 w2 = *reinterpret_cast<const f32x4*>(s_vec + O + M + 32 * k + 16 * b + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const YD r = silu_yd<bf16>(acc[b][i] + bx[i]);
            phi += r.y * w2[i];
            pv[8 * (k & 1) + 4 * b + i] = gpm * r.y;
            acc[b][i] = gphi * w2[i] * r.d;
          }
          store_rows(a.Dgq, 2 * k + b, acc[b]);
        }
        gq[k] = pack_chunk<bf16>(acc[0], acc[1]);
        if (k & 1) {
          sw2[k >> 1] += edge_sum16(pv, c);
          __syncthreads();
        }
      }
      phi += shfl_xor(phi, 16);
      phi += shfl_xor(phi, 32);
    }
    // ---- S4: g_a2
    bf16x8 ga2[O / 32];
#pragma unroll
    for (int k = 0; k < O / 32; ++k) {
      const bf16x4 g0 = gr0, g1 = gr1;
      if (k + 1 < O / 32) {
        gr0 = *reinterpret_cast<const bf16x4*>(gm + 32 * (k + 1));
        gr1 = *reinterpret_cast<const bf16x4*>(gm + 32 * (k + 1) + 16);
      }
      f32x4 acc[2] = {unpack4(g0), unpack4(g1)};
      if constexpr (EQ) rows(2 * kST + (k >> 1), k & 1, gq, acc);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        acc[b] *= unpack4(s2[2 * k + b]);
        store_rows(a.Dga2, 2 * k + b, acc[b]);
      }
      ga2[k] = pack_chunk<bf16>(acc[0], acc[1]);
      if (EQ && (k & 1)) __syncthreads();
    }
    load_ids(ps + gridDim.x);
    // ---- S5: Gh, dw_d, S6
    float gr = 0.f, gv[16];
#pragma unroll
    for (int k = 0; k < H / 32; ++k) {
      f32x4 acc[2] = {zero4(), zero4()};
      rows((EQ ? 3 : 1) * kST + (k >> 1), k & 1, ga2, acc);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int rb = 2 * k + b;
        acc[b] *= unpack4(rb < H / 32 ? s1[rb % (H / 32)] : s_d1[w][rb % (H / 32)][l]);
        store_rows(a.Gh, rb, acc[b]);
        if constexpr (EQ) {
          const f32x4 wd = *reinterpret_cast<const f32x4*>(s_vec + O + 2 * M + 16 * rb + 4 * g);
          const float r2 = valid ? ga[0] : 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            gr += wd[i] * acc[b][i];
            gv[8 * (k & 1) + 4 * b + i] = r2 * acc[b][i];
          }
        }
      }
      if (k & 1) {
        if constexpr (EQ) swd[k >> 1] += edge_sum16(gv, c);
        __syncthreads();
      }
    }
    if constexpr (EQ) {
      gr += shfl_xor(gr, 16);
      gr += shfl_xor(gr, 32);
      const float k2 = 2.0f * gr;
      if (g == 0)
        *reinterpret_cast<f32x4*>(a.Gx + e * 4) =
            f32x4{phi * gb[1] + k2 * ga[2], phi * gb[2] + k2 * ga[3], phi * gb[3] + k2 * gb[0], ga[1]};
    }
    __asm__ __volatile__("" : "+v"(n_ri), "+v"(n_rj), "+v"(n_eid));   // complete before the next pass, whose waits stay exact
  }
  if constexpr (EQ) {   // the block's partial row: the waves' sums in wave order
    float* const s_sum = (float*)s_w[1];   // [wave][M | H]; buffer 0 holds the next pass's first chunk
#pragma unroll
    for (int h = 0; h < kST; ++h) {
      s_sum[w * (M + H) + 64 * h + fsum] = sw2[h];
      s_sum[w * (M + H) + M + 64 * h + fsum] = swd[h];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < M + H; q += 64 * kWaves) {
      float s = s_sum[q];
#pragma unroll
      for (int k = 1; k < kWaves; ++k) s += s_sum[k * (M + H) + q];
      a.dwpart[(int64_t)blockIdx.x * a.LW + q] = s;
    }
  }
}

template <bool EQ> void launch_nu(const BwdArgs& a, dim3 grid, hipStream_t st) {
  if (a.NUC == 1) hipLaunchKernelGGL((wide_bwd_ep_kernel<EQ, 1>), grid, dim3(64 * kWaves), 0, st, a);
  else hipLaunchKernelGGL((wide_bwd_ep_kernel<EQ, 2>), grid, dim3(64 * kWaves), 0, st, a);
}

}  // namespace

int wide_bwd_ep_blocks(int64_t E) { return (int)std::min<int64_t>(cdiv(E, 16 * kWaves), 256); }   // one block per CU

int launch_wide_bwd_ep(const LayerShape& s, const BwdArgs& a, int nblk, hipStream_t st) {
  if (a.E <= 0) return 0;
  if (nblk != wide_bwd_ep_blocks(a.E)) return (int)hipErrorInvalidValue;   // partial rows
  if (s.eq) launch_nu<true>(a, dim3(nblk), st);
  else launch_nu<false>(a, dim3(nblk), st);
  return (int)hipGetLastError();
}

}  // namespace egnn
