// Edge-parallel forward at H = O = M = 256 (bf16, gfx950), equivariant and MPNN, from 16,385 edges on (wide_fwd_ep).
//
// Each wave takes whole 32-edge schedule tiles and runs both 16-edge halves side by side in its own registers with the
// features on the MFMA rows, so every weight fragment read from LDS feeds two products:
//   S1  m1 = SiLU(W_u [e | r^2] + P_i + Q_j)
//   S2  m  = SiLU(W_hl^T m1 + b2), 32 rows at a time; their row sums right away
//   S3  phi = SiLU(W1_mov^T m + bx1) . w2_mov, 32 rows at a time
// P_i, Q_j and the biases are added to the finished products in fp32, in the order of egnn_wide.hip, so the messages are
// bit for bit those of the tile-sharing kernels (a P_i + Q_j by a product against a 0/1 operand saves 500 vector
// instructions a pass, but rounds differently and turns an infinite feature into 16 NaNs).
// The two 256 x 256 weights (256 KB) do not fit the LDS: 16 KB chunks of 32 rows go through two LDS buffers in the
// order of use, shared by the block's four waves, the next chunk loaded into registers before the products of the
// current one and stored after them, one barrier per chunk.  W_u's fragments stay in LDS.  75 KB leave two blocks per
// CU.  Row sums: the 32 features x 32 edges of a step go through the wave's 2 KB of LDS, are read back edge-major by
// transposing reads and multiplied by the 0/1 segment matrix of the schedule's rank table; whole rows are stored, the
// tile's partial rows go to its carry slots, as do the coordinate sums (delta phi as a bf16 hi + lo pair).
// Measured against the kernel whose eight waves share each tile by feature rows and exchange every stage through LDS
// (660k and 44k edges, F_E = 32): 564 -> 319 and 49 -> 38 us.
#include "egnn_device.h"
#include "egnn_internal.h"
#include "egnn_tile.h"

namespace egnn {
namespace {

using namespace tile;

constexpr int kWaves = 4, H = 256, O = 256, M = 256, KH = H / 32, KP = O / 32;
constexpr int kChunkElems = 2 * KH * kFragElems;   // 32 rows

template <bool EQ, int NU>   // NU: 32-slot slices of the edge input (1 or 2)
__global__ __launch_bounds__(64 * kWaves, 2) void wide_fwd_ep_kernel(FwdArgs a) {
  constexpr int SEGW = O + (EQ ? 4 : 0), NCH = EQ ? 2 * KP : KP, KG = 4;
  __shared__ __attribute__((aligned(16))) bf16 s_w[2][kChunkElems];
  __shared__ __attribute__((aligned(16))) bf16 s_u[2 * KH * NU * kFragElems];
  __shared__ __attribute__((aligned(16))) float s_vec[O + 2 * M];             // b2 | bx1 | w2_mov
  __shared__ __attribute__((aligned(16))) bf16 s_msg[kWaves][2 * kFragElems];
  __shared__ __attribute__((aligned(16))) f32x4 s_geo[kWaves][TE];
  __shared__ __attribute__((aligned(16))) float s_ph[kWaves][TE];

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  const bf16* PQ = (const bf16*)a.PQ;
  const bf16* ef = (const bf16*)a.ef;
  const int64_t E = a.E;
  const int FE = a.FE;
  const int64_t npass = (a.ntiles + kWaves - 1) / kWaves;

  for (int q = threadIdx.x; q < 2 * KH * NU * 64; q += 64 * kWaves)
    reinterpret_cast<bf16x8*>(s_u)[q] = reinterpret_cast<const bf16x8*>(a.fr.u)[q];
  for (int q = threadIdx.x; q < O; q += 64 * kWaves) {
    s_vec[q] = a.fr.b2f[q];
    if constexpr (EQ) {
      s_vec[O + q] = a.fr.bx1f[q];
      s_vec[O + M + q] = a.fr.w2mf[q];
    }
  }
  bf16x8 st[4];
  uint32_t so = threadIdx.x * 16;   // made opaque once per pass: a base in scalar registers + this, no hoisted addresses
  auto stream_load = [&](int ch) {
    const char* src = EQ && ch >= KP ? (const char*)a.fr.movT + (ch - KP) * (kChunkElems * 2) : (const char*)a.fr.hlT + ch * (kChunkElems * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) st[i] = *reinterpret_cast<const bf16x8*>(src + i * (64 * kWaves * 16) + so);
  };
  auto stream_store = [&](int buf) {
    bf16* dst = s_w[buf] + threadIdx.x * 8;
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<bf16x8*>(dst + i * 64 * kWaves * 8) = st[i];
  };
  // 32 rows (chunk ch) of a product with both edge blocks: acc[row block][edge block] += W . B
  auto rows = [&](int ch, const bf16x8 (*B)[2], f32x4 (*acc)[2]) {
    const bf16* W = s_w[ch & 1] + l * 8;
    stream_load((ch + 1) % NCH);
    bf16x8 A0 = load_chunk(W), A1 = load_chunk(W + KH * kFragElems);
#pragma unroll
    for (int kc = 0; kc < KH; ++kc) {
      bf16x8 N0 = A0, N1 = A1;
      if (kc + 1 < KH) {
        N0 = load_chunk(W + (kc + 1) * kFragElems);
        N1 = load_chunk(W + (KH + kc + 1) * kFragElems);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        mma(acc[0][nb], A0, B[kc][nb]);
        mma(acc[1][nb], A1, B[kc][nb]);
      }
      __builtin_amdgcn_sched_barrier(0);
      A0 = N0;
      A1 = N1;
    }
    stream_store((ch + 1) & 1);
  };
  stream_load(0);
  stream_store(0);
  __syncthreads();

  for (int64_t ps = blockIdx.x; ps < npass; ps += gridDim.x) {
    __asm__ __volatile__("" : "+v"(so));
    const int64_t T0 = ps * kWaves + w;
    const bool live_tile = T0 < a.ntiles;
    const int64_t T = live_tile ? T0 : a.ntiles - 1, base = T * TE;
    const int tabv = a.tile_tab[T * kTabInts + l];
    const int nrk = live_tile ? __builtin_amdgcn_readlane(tabv, kTabNrank) : 0;   // a wave past the end stores nothing
    int ri[2], rj[2];
    bf16x8 u[NU][2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int64_t e0 = base + 16 * nb + c, e = e0 < E ? e0 : E - 1;
      ri[nb] = clampi(a.erow[e], (int)a.N);
      rj[nb] = clampi(a.col[e], (int)a.N);
      const int eid = a.eids ? clampi(a.eids[e], (int)E) : (int)e;
      float r2 = 0.f;
      if constexpr (EQ) {
        const f32x4 geo = *reinterpret_cast<const f32x4*>(a.geo + e * 4);
        r2 = geo[3];
        if (g == 0) s_geo[w][16 * nb + c] = geo;
      }
#pragma unroll
      for (int uc = 0; uc < NU; ++uc) {
        const int s0 = 32 * uc + 8 * g;
        u[uc][nb] = zero_chunk<bf16>();
        if (s0 + 8 <= FE) u[uc][nb] = load_chunk(ef + (int64_t)eid * a.se + s0);
        else if (EQ && s0 == FE) {   // r^2 as a bf16 hi + lo pair
          const bf16 hi = (bf16)r2;
          u[uc][nb][0] = hi;
          u[uc][nb][1] = (bf16)(r2 - (float)hi);
        }
      }
    }
    // ---- S1
    bf16x8 m1[KH][2];
#pragma unroll
    for (int k4 = 0; k4 < KH; k4 += KG) {
      bf16x8 p[KG][2], q[KG][2];
#pragma unroll
      for (int k = 0; k < KG; ++k)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          p[k][nb] = load_chunk(PQ + (int64_t)ri[nb] * 2 * H + 32 * (k4 + k) + 8 * g);
          q[k][nb] = load_chunk(PQ + (int64_t)rj[nb] * 2 * H + H + 32 * (k4 + k) + 8 * g);
        }
#pragma unroll
      for (int k = 0; k < KG; ++k) {
        const int kc = k4 + k;
        f32x4 y[2][2];   // [row block][edge block]
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          y[b][0] = y[b][1] = zero4();
#pragma unroll
          for (int uc = 0; uc < NU; ++uc) {
            const bf16x8 A = load_chunk(s_u + (((2 * kc + b) * NU + uc) * 64 + l) * 8);
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) mma(y[b][nb], A, u[uc][nb]);
          }
        }
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
          f32x4 pv[2], qv[2];
          unpack_chunk(p[k][nb], pv[0], pv[1]);
          unpack_chunk(q[k][nb], qv[0], qv[1]);
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) y[b][nb][i] = y[b][nb][i] + pv[b][i] + qv[b][i];
        }
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
          for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int i = 0; i < 4; ++i) y[b][nb][i] = silu_t<bf16>(y[b][nb][i]);
          m1[kc][nb] = pack_chunk<bf16>(y[0][nb], y[1][nb]);
        }
      }
    }
    // ---- S2 and the row sums
    bf16x8 mc[EQ ? KP : 1][2];
#pragma unroll
    for (int kp = 0; kp < KP; ++kp) {
      f32x4 acc[2][2] = {{zero4(), zero4()}, {zero4(), zero4()}};
      rows(kp, m1, acc);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const f32x4 b2 = *reinterpret_cast<const f32x4*>(s_vec + 32 * kp + 16 * b + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[b][nb][i] = silu_t<bf16>(acc[b][nb][i] + b2[i]);
        }
        const bf16x8 v = pack_chunk<bf16>(acc[0][nb], acc[1][nb]);
        if constexpr (EQ) mc[kp][nb] = v;
        store_chunk(s_msg[w] + (nb * 64 + chain_slot<true>(l)) * 8, v);
      }
      wave_sync();
      const bf16x8 M0 = chain_edge_major<2, true>(s_msg[w], 0, c, g), M1 = chain_edge_major<2, true>(s_msg[w], 1, c, g);
      for (int rg = 0; 16 * rg < nrk; ++rg) {   // ranks 0..15, then 16..31 (a tile of short rows)
        const int r = 16 * rg + c;
        const int tg = __shfl(tabv, kTabTgt + r, 64), sp = __shfl(tabv, kTabSpan + (r >> 1), 64);
        const bool live = r < nrk;
        const bf16x8 S = seg_chunk_valu(live ? (sp >> (16 * (r & 1))) & 0xffff : 0, g);
        f32x4 D0 = zero4(), D1 = zero4();
        mma(D0, M0, S);
        mma(D1, M1, S);
        if (live && tg >= 0) {
          bf16* o = (bf16*)a.out_msg + (int64_t)tg * a.smsg + 32 * kp + 4 * g;
          *reinterpret_cast<bf16x4*>(o) = pack4(D0);
          *reinterpret_cast<bf16x4*>(o + 16) = pack4(D1);
        } else if (live) {
          float* o = a.carry + (T * 2 + (-1 - tg)) * SEGW + 32 * kp + 4 * g;
          *reinterpret_cast<f32x4*>(o) = D0;
          *reinterpret_cast<f32x4*>(o + 16) = D1;
        }
      }
      __syncthreads();
    }
    // ---- S3 and the coordinate sums
    if constexpr (EQ) {
      float phi[2] = {0.f, 0.f};
#pragma unroll
      for (int mp = 0; mp < M / 32; ++mp) {
        f32x4 acc[2][2] = {{zero4(), zero4()}, {zero4(), zero4()}};
        rows(KP + mp, mc, acc);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const f32x4 bx = *reinterpret_cast<const f32x4*>(s_vec + O + 32 * mp + 16 * b + 4 * g);
          const f32x4 w2 = *reinterpret_cast<const f32x4*>(s_vec + O + M + 32 * mp + 16 * b + 4 * g);
#pragma unroll
          for (int nb = 0; nb < 2; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) phi[nb] += silu_t<bf16>(acc[b][nb][i] + bx[i]) * w2[i];
        }
        __asm__ __volatile__("" : "+v"(phi[0]), "+v"(phi[1]));   // summed here: else the eight steps' sums are kept to the end
        __syncthreads();
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        phi[nb] += shfl_xor(phi[nb], 16);
        phi[nb] += shfl_xor(phi[nb], 32);
        if (g == 0) s_ph[w][16 * nb + c] = base + 16 * nb + c < E ? phi[nb] : 0.f;   // edges past E
      }
      wave_sync();
      // A operands: row c < 3 = component c of delta phi over edges kappa_chain(g, s), as a bf16 hi + lo pair
      bf16x8 ahi = zero_chunk<bf16>(), alo = zero_chunk<bf16>();
      if (c < 3) {
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          const int k = kappa_chain(g, s);
          const float v = s_geo[w][k][c] * s_ph[w][k];
          const bf16 hi = (bf16)v;
          ahi[s] = hi;
          alo[s] = (bf16)(v - (float)hi);
        }
      }
      for (int rg = 0; 16 * rg < nrk; ++rg) {
        const int r = 16 * rg + c;
        const int tg = __shfl(tabv, kTabTgt + r, 64), sp = __shfl(tabv, kTabSpan + (r >> 1), 64);
        const bool live = r < nrk;
        const int span = live ? (sp >> (16 * (r & 1))) & 0xffff : 0;
        const bf16x8 S = seg_chunk_valu(span, g);
        f32x4 D = zero4();
        mma(D, ahi, S);
        mma(D, alo, S);
        if (g == 0 && live) {
          float* o = tg >= 0 ? a.out_mov + (int64_t)tg * a.smov : a.carry + (T * 2 + (-1 - tg)) * SEGW + O;
          const float sc = a.mean && tg >= 0 ? 1.0f / (float)(span >> 8) : 1.0f;
          o[0] = D[0] * sc;
          o[1] = D[1] * sc;
          o[2] = D[2] * sc;
        }
      }
      wave_sync();
    }
  }
}

template <bool EQ>
void launch_nu(const FwdArgs& a, dim3 grid, hipStream_t st) {
  if (a.NUC == 1) hipLaunchKernelGGL((wide_fwd_ep_kernel<EQ, 1>), grid, dim3(64 * kWaves), 0, st, a);
  else hipLaunchKernelGGL((wide_fwd_ep_kernel<EQ, 2>), grid, dim3(64 * kWaves), 0, st, a);
}

}  // namespace

int launch_wide_fwd_ep(const LayerShape& s, const FwdArgs& a, hipStream_t st) {
  if (a.ntiles <= 0) return 0;
  const dim3 grid((unsigned)std::min<int64_t>(cdiv(a.ntiles, kWaves), 512));   // two blocks per CU
  if (s.eq) launch_nu<true>(a, grid, st);
  else launch_nu<false>(a, grid, st);
  return (int)hipGetLastError();
}

}  // namespace egnn
