// fp32 edge kernels of the layer at H = O = M = 128 on split bf16 operands (egnn_split.h): forward, backward and
// the weight-gradient products over the edges.
//
// Forward.  A block of four waves takes two 32-edge schedule tiles at a time, each wave one 16-edge half
// with the features on the MFMA rows, so a stage's two C-blocks are, split into parts, the next stage's
// B operand in the wave's own registers:
//   S1  m1 = SiLU(P_i + Q_j + W_u [e, r^2])
//   S2  m  = SiLU(W_hl^T m1 + b2), 32 rows at a time
//   S3  q += W1_mov^T m over those 32 rows, so no stage keeps all of m;  phi = SiLU(q + bx1) . w2_mov
// The weights in three parts are 2 x 96 KB, more than the LDS holds, so they are streamed: 24 KB chunks
// (two row blocks of S2, then one k slice of S3) go through two LDS buffers in the order of use, the next
// chunk loaded into registers before the products of the current one and stored after them, one barrier
// per chunk.  70 KB of LDS leave two blocks per CU, whose barriers and gathers overlap.
// Row sums: each wave adds up its half's rows from its own LDS rows, one feature per lane, in edge order;
// the first wave of a tile hands the sum of a row that goes on into the second half over through LDS.
// Measured against one wave per 32-edge tile on the fp32 instruction with the weights read from L2 (E = 394k,
// 46k and 0.7k edges of 9..29-atom molecules): 564 -> 236, 99 -> 36 and 51 -> 16 us.  What bounds it now is the
// issue of the 768 products and about 2,400 vector instructions per wave and pass.
#include "egnn_device.h"
#include "egnn_internal.h"
#include "egnn_split.h"

namespace egnn {
namespace {

using namespace split;

constexpr int kF32Waves = 4;

__device__ __forceinline__ Chunk3 lds_chunk3(const bf16* frag, int l) {
  const bf16* p = frag + l * 8;
  return Chunk3{load_chunk(p), load_chunk(p + kFragElems), load_chunk(p + 2 * kFragElems)};
}
// one address per lane; of(r): lane r's, wave-uniform
struct RowAddr {
  uint32_t lo, hi;
  __device__ __forceinline__ explicit RowAddr(float* p) : lo((uint32_t)(uintptr_t)p), hi((uint32_t)((uintptr_t)p >> 32)) {}
  // in the global address space: a generic (flat) store also waits for the LDS
  __device__ __forceinline__ __attribute__((address_space(1))) float* of(int r) const {
    return (__attribute__((address_space(1))) float*)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, r) << 32) |
                    (uint32_t)__builtin_amdgcn_readlane((int)lo, r));
  }
};
// fragments of two row blocks
struct Pair3 { Chunk3 a, b; };
__device__ __forceinline__ Pair3 pair3(const bf16* a, const bf16* b, int l) { return Pair3{lds_chunk3(a, l), lds_chunk3(b, l)}; }

template <bool EQ, bool FEAT>
__global__ __launch_bounds__(64 * kF32Waves, 2) void f32_fwd_kernel(FwdArgs a) {
  constexpr int H = 128, O = 128, M = 128, KH = H / 32, KP = O / 32, CH = EQ ? 2 : 1;
  constexpr int SEGW = O + (EQ ? 4 : 0), SP = 68;              // carry slot; row pitch of the message rows
  constexpr int CE = 24 * kFragElems;                          // one chunk of weight fragments
  __shared__ __attribute__((aligned(16))) bf16 s_w[2][CE];
  __shared__ __attribute__((aligned(16))) float s_msg[kF32Waves][16 * SP];
  __shared__ __attribute__((aligned(16))) float s_open[2][SEGW];   // a tile's row that goes on into its second half
  __shared__ __attribute__((aligned(16))) float s_vec[O + 2 * M + H];   // b2 | bx1 | w2_mov | w_d

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  const int h = w & 1, pr = w >> 1;
  const float sg = c & 1 ? -1.0f : 1.0f;   // the edge's sign in the chain
  const float* PQ = (const float*)a.PQ;
  const float* ef = (const float*)a.ef;
  const int64_t E = a.E;
  const int64_t npass = (a.ntiles + 1) / 2;

  for (int q = threadIdx.x; q < O; q += 64 * kF32Waves) {
    s_vec[q] = a.fr.b2f[q];
    s_vec[O + q] = a.fr.bx1f[q];
    s_vec[O + M + q] = a.fr.w2mf[q];
    s_vec[O + 2 * M + q] = a.fr.wdf[q];
  }

  // chunk ch of the weight stream: six 16-byte pieces per lane, to registers and then to LDS
  bf16x8 st[6];
  uint32_t so = threadIdx.x * 16;   // made opaque once per pass: a base in scalar registers + this, no hoisted addresses
  auto stream_load = [&](int ch) {
    const char* src = (const char*)a.fr.s_fwd + ch * (CE * 2);
#pragma unroll
    for (int i = 0; i < 6; ++i) st[i] = *reinterpret_cast<const bf16x8*>(src + i * (64 * kF32Waves * 16) + so);
  };
  auto stream_store = [&](int buf) {
    bf16* dst = s_w[buf] + threadIdx.x * 8;
#pragma unroll
    for (int i = 0; i < 6; ++i) *reinterpret_cast<bf16x8*>(dst + i * 64 * kF32Waves * 8) = st[i];
  };
  stream_load(0);
  stream_store(0);
  __syncthreads();

  for (int64_t ps = blockIdx.x; ps < npass; ps += gridDim.x) {
    __asm__ __volatile__("" : "+v"(so));
    const int64_t T = 2 * ps + pr, base = T * kTileEdges;
    const int64_t Tc = T < a.ntiles ? T : a.ntiles - 1;
    const int tabv = a.tile_tab[Tc * kTabInts + l];
    // lane r: where the sums of rank r of the tile go, its output row or a carry slot
    const bool whole = tabv >= 0;
    float* const cslot = a.carry + (Tc * 2 + (tabv == -2)) * SEGW;
    const RowAddr am(whole ? (float*)a.out_msg + (int64_t)tabv * a.smsg : cslot);
    const RowAddr ax(EQ && whole ? a.out_mov + (int64_t)tabv * a.smov : cslot + O);
    // last edge of each run of one row in the tile (none in a tile past the end)
    uint32_t ends;
    {
      const int64_t e = base + l;
      const int er = a.erow[e < E ? e : E - 1];
      const int en = __shfl(er, l + 1 < 64 ? l + 1 : 63, 64);
      ends = (uint32_t)__ballot(l < kTileEdges && e < E && (l == kTileEdges - 1 || e == E - 1 || er != en));
    }
    const int64_t e0 = base + 16 * h + c, ec = e0 < E ? e0 : E - 1;
    const int ri = clampi(a.erow[ec], (int)a.N), rj = clampi(a.col[ec], (int)a.N);
    float dx = 0.f, dy = 0.f, dz = 0.f, r2 = 0.f;
    if constexpr (EQ) {
      const float* xi = a.coord + (int64_t)ri * a.sc;
      const float* xj = a.coord + (int64_t)rj * a.sc;
      dx = xi[0] - xj[0];
      dy = xi[1] - xj[1];
      dz = xi[2] - xj[2];
      r2 = dx * dx + dy * dy + dz * dz;
    }
    // ---- S1
    Chunk3 m1[KH];
    {
      f32x4 y[KH][2];
#pragma unroll
      for (int kc = 0; kc < KH; ++kc) {
        const f32x8 p = load_chunk(PQ + (int64_t)ri * 2 * H + 32 * kc + 8 * g);
        const f32x8 q = load_chunk(PQ + (int64_t)rj * 2 * H + H + 32 * kc + 8 * g);
        y[kc][0] = p.lo + q.lo;
        y[kc][1] = p.hi + q.hi;
      }
      if constexpr (FEAT) {
        const int eid = a.eids ? clampi(a.eids[ec], (int)E) : (int)ec;
        for (int uc = 0; uc < a.NUC; ++uc) {
          const int s0 = 32 * uc + 8 * g;
          f32x8 u = zero_chunk<float>();
          if (s0 + 8 <= a.FE) u = load_chunk(ef + (int64_t)eid * a.se + s0);
          else if (EQ && s0 == a.FE) u.lo[0] = r2;
          const Chunk3 u3 = split_chunk(u.lo * sg, u.hi * sg);
#pragma unroll
          for (int rb = 0; rb < H / 16; ++rb) {
            const Chunk3 A = lds_chunk3((const bf16*)a.fr.s_u + ((int64_t)(rb >> 1) * 6 * a.NUC + ((rb & 1) * a.NUC + uc) * 3) * kFragElems, l);
            f32x4 lo = zero4(), hi = zero4();
            mma3(hi, lo, A, u3);
            y[rb >> 1][rb & 1] = add_signed(y[rb >> 1][rb & 1], joined(hi, lo), sg);
          }
        }
      } else if constexpr (EQ) {
#pragma unroll
        for (int rb = 0; rb < H / 16; ++rb) {
          const f32x4 wd = *reinterpret_cast<const f32x4*>(s_vec + O + 2 * M + 16 * rb + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) y[rb >> 1][rb & 1][i] = __builtin_fmaf(r2, wd[i], y[rb >> 1][rb & 1][i]);
        }
      }
#pragma unroll
      for (int kc = 0; kc < KH; ++kc) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) y[kc][b][i] = silu_f32(y[kc][b][i], sg);
        m1[kc] = split_chunk(y[kc][0], y[kc][1]);
      }
    }
    // loaded before the gathers, so complete by now: named here, not at each row's store, which would then wait for
    // every load under way
    __asm__ __volatile__("" ::"v"(tabv), "v"(am.lo), "v"(am.hi), "v"(ax.lo), "v"(ax.hi), "v"(dx), "v"(dy), "v"(dz));
    // ---- S2 and S3, 32 message features at a time
    f32x4 q[EQ ? M / 16 : 1];
    if constexpr (EQ) {
#pragma unroll
      for (int rb = 0; rb < M / 16; ++rb) q[rb] = zero4();
    }
    const uint32_t mine = (ends >> (16 * h)) & 0xffffu;
    const bool cont = !((ends >> 15) & 1u) && (ends >> 16) != 0u;   // a row goes on past edge 15
    float first[2] = {0.f, 0.f};   // second half: sums of the row that began in the first
    float* const mrow = s_msg[w];
#pragma unroll
    for (int kp = 0; kp < KP; ++kp) {
      {
        const bf16* W = s_w[(CH * kp) & 1];
        stream_load(EQ ? 2 * kp + 1 : (kp + 1) % KP);
        f32x4 hi[2], lo[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) hi[b] = lo[b] = zero4();
        Pair3 A = pair3(W, W + KH * 3 * kFragElems, l);
#pragma unroll
        for (int kc = 0; kc < KH; ++kc) {   // the next slice's fragments requested before this one's products
          Pair3 An = A;
          if (kc + 1 < KH) An = pair3(W + (kc + 1) * 3 * kFragElems, W + (KH + kc + 1) * 3 * kFragElems, l);
          __builtin_amdgcn_sched_barrier(0);
          mma3x2(hi, lo, A.a, A.b, m1[kc]);
          __builtin_amdgcn_sched_barrier(0);
          A = An;
        }
        f32x4 x[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const f32x4 b2 = *reinterpret_cast<const f32x4*>(s_vec + 32 * kp + 16 * b + 4 * g), p2 = joined(hi[b], lo[b]);
#pragma unroll
          for (int i = 0; i < 4; ++i) x[b][i] = silu_f32(__builtin_fmaf(p2[i], sg, b2[i]), sg);
          *reinterpret_cast<f32x4*>(mrow + c * SP + 32 * (kp & 1) + 16 * b + 4 * g) = x[b];
        }
        stream_store((CH * kp + 1) & 1);
        __syncthreads();
        if constexpr (EQ) {
          const Chunk3 mc = split_chunk(x[0], x[1]);
          const bf16* W3 = s_w[1];
          stream_load((2 * kp + 2) % (2 * KP));
          Pair3 A = pair3(W3, W3 + 3 * kFragElems, l);
#pragma unroll
          for (int rb = 0; rb < M / 16; rb += 2) {
            Pair3 An = A;
            if (rb + 2 < M / 16) An = pair3(W3 + (rb + 2) * 3 * kFragElems, W3 + (rb + 3) * 3 * kFragElems, l);
            __builtin_amdgcn_sched_barrier(0);
            f32x4 lo3[2] = {zero4(), zero4()};
            mma3x2(q + rb, lo3, A.a, A.b, mc);
            q[rb] += lo3[0];   // not joined: an infinite message makes phi NaN by its SiLU(-inf) too
            q[rb + 1] += lo3[1];
            __builtin_amdgcn_sched_barrier(0);
            A = An;
          }
          stream_store(0);
        }
      }
      if (kp & 1) {   // row sums of 64 features, one per lane
        wave_sync();
        float v[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = mrow[k * SP + l];
        const uint32_t f = 64 * (kp >> 1) + l;
        float acc = 0.f;
        int r = __builtin_amdgcn_readfirstlane(__popc(ends & ((1u << (16 * h)) - 1u)));   // rank of the half's first edge
        bool deferred = h && cont;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          acc += k & 1 ? -v[k] : v[k];   // the rows hold the signed messages
          if ((mine >> k) & 1u) {
            if (deferred) {
              first[kp >> 1] = acc;
              deferred = false;
            } else {
              am.of(r)[f] = acc;
            }
            acc = 0.f;
            ++r;
          }
        }
        if (!h && cont) s_open[pr][f] = acc;
        wave_sync();
      }
      if constexpr (EQ) __syncthreads();
    }
    // ---- phi and the coordinate sums
    float cfirst = 0.f;
    int cdeg = 0;
    if constexpr (EQ) {
      float phi = 0.f;
#pragma unroll
      for (int rb = 0; rb < M / 16; ++rb) {
        const f32x4 bx = *reinterpret_cast<const f32x4*>(s_vec + O + 16 * rb + 4 * g);
        const f32x4 w2 = *reinterpret_cast<const f32x4*>(s_vec + O + M + 16 * rb + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) phi += silu_f32(__builtin_fmaf(q[rb][i], sg, bx[i])) * w2[i];
      }
      phi += shfl_xor(phi, 16);
      phi += shfl_xor(phi, 32);
      if (g == 0) *reinterpret_cast<f32x4*>(mrow + 4 * c) = f32x4{dx * phi, dy * phi, dz * phi, 0.f};
      wave_sync();
      float v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = mrow[4 * k + (l & 3)];
      float acc = 0.f;
      int r = __popc(ends & ((1u << (16 * h)) - 1u)), n = 0;
      bool deferred = h && cont;
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        acc += v[k];
        ++n;
        if ((mine >> k) & 1u) {
          if (deferred) {
            cfirst = acc;
            cdeg = n;
            deferred = false;
          } else if (l < 3) {
            ax.of(r)[l] = a.mean && __builtin_amdgcn_readlane(tabv, r) >= 0 ? acc / (float)n : acc;
          }
          acc = 0.f;
          n = 0;
          ++r;
        }
      }
      if (!h && cont && l < 4) s_open[pr][O + l] = l < 3 ? acc : (float)n;
    }
    __syncthreads();
    if (h && cont) {   // the row that began in the first half
      const int r = __popc(ends & 0xffffu);
#pragma unroll
      for (int q = 0; q < 2; ++q) am.of(r)[64 * q + l] = s_open[pr][64 * q + l] + first[q];
      if (EQ && l < 3) {
        const float s = s_open[pr][O + l] + cfirst;
        ax.of(r)[l] = a.mean && __builtin_amdgcn_readlane(tabv, r) >= 0 ? s / ((float)cdeg + s_open[pr][O + 3]) : s;
      }
    }
  }
}

// Backward over 16 edges per wave, the chain of egnn_bwd.hip with every product on split operands:
//   S1 m1, SiLU'   S2 m, SiLU' (32 rows at a time)   S3 q += W1_mov^T m over those rows
//   g_q = g_phi w2_mov SiLU'(q)   S4 g_m = gm_i + W1_mov g_q, g_a2 = g_m SiLU' (32 rows at a time)
//   S5 g_a1 += W_hl g_a2 over those rows   S6 dL/ddelta = phi gx_i + 2 (w_d . g_a1) delta
// The weights go through LDS as in the forward, 16 chunks a pass.  Stores Gh, Gx and the factors m1, m, g_q, g_a2
// for atb_f32_kernel, all four with the edge's sign (odd edges negative: the products are the same); dw2_mov = sum g_phi p and dw_d = sum r^2 g_a1 are summed here (edge_sum16 over the wave's
// edges, then registers over the passes) into one partial row [M | H] per block.
// Measured against one wave per 32-edge tile on the fp32 instruction, which also stored p and r^2 for dw2_mov and
// dw_d: 989 -> 502 us at 384k edges (both in two chunks), 146 (two) -> 67 us (one) at 46k.  30 registers spill (38 with
// edge features): vector 0.35 and matrix issue 0.25 of the cycles, 0.48 of the wave cycles waiting.
template <bool EQ, bool FEAT>
__global__ __launch_bounds__(64 * kF32Waves, 2) void f32_bwd_kernel(BwdArgs a) {
  constexpr int H = 128, O = 128, M = 128, KH = H / 32, KP = O / 32, NCH = EQ ? 4 * KP : 2 * KP;
  constexpr int CE = 24 * kFragElems;
  __shared__ __attribute__((aligned(16))) bf16 s_w[2][CE];
  __shared__ __attribute__((aligned(16))) float s_vec[O + 2 * M + H];       // b2 | bx1 | w2_mov | w_d
  // SiLU'(pre1) of row blocks 0 .. 6, from S1 to the end of S5 (block 7 stays in registers: with it the LDS
  // would not hold two blocks)
  __shared__ __attribute__((aligned(16))) f32x4 s_d1[kF32Waves][7][64];
  static_assert(sizeof(float) * kF32Waves * (M + H) <= sizeof(s_w[0]), "the final sums reuse the weight buffer");

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  const float sg = c & 1 ? -1.0f : 1.0f;   // the edge's sign in the chain
  const float* PQ = (const float*)a.PQ;
  const float* ef = (const float*)a.ef;
  const float* gmsg = (const float*)a.gmsg;
  const int64_t E = a.E, ebeg = a.tile0 * kTileEdges;
  const int64_t eend = a.ntiles * kTileEdges < E ? a.ntiles * kTileEdges : E;
  const int64_t npass = (eend - ebeg + 16 * kF32Waves - 1) / (16 * kF32Waves);

  for (int q = threadIdx.x; q < O; q += 64 * kF32Waves) {
    s_vec[q] = a.fr.b2f[q];
    s_vec[O + q] = a.fr.bx1f[q];
    s_vec[O + M + q] = a.fr.w2mf[q];
    s_vec[O + 2 * M + q] = a.fr.wdf[q];
  }
  // Weight stream.  At the top of chunk ch (in buffer ch & 1): the first half of chunk ch + 1 is requested; in the
  // middle it is stored and the second half requested; at the end that is stored and a barrier follows.
  bf16x8 st[3];
  uint32_t so = threadIdx.x * 16;
  auto stream_load = [&](int ch, int half) {
    const char* src = (const char*)a.fr.s_fwd + (ch % NCH) * (CE * 2) + half * CE;
#pragma unroll
    for (int i = 0; i < 3; ++i) st[i] = *reinterpret_cast<const bf16x8*>(src + i * (64 * kF32Waves * 16) + so);
  };
  auto stream_store = [&](int ch, int half) {
    bf16* dst = s_w[ch & 1] + half * (CE / 2) + threadIdx.x * 8;
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(dst + i * 64 * kF32Waves * 8) = st[i];
  };
  // rows 32 kp .. + 31 of the first matrix of a chunk pair: out[b] = A[row block b] . B
  auto rows_chunk = [&](int ch, const Chunk3* B, f32x4* hi, f32x4* lo) {
    const bf16* W = s_w[ch & 1];
    stream_load(ch + 1, 0);
    Chunk3 A = lds_chunk3(W, l);
#pragma unroll
    for (int j = 0; j < 2 * KH; ++j) {
      const int kc = j >> 1, b = j & 1;
      Chunk3 An = A;
      if (j + 1 < 2 * KH) An = lds_chunk3(W + (((j + 1) & 1) * KH + ((j + 1) >> 1)) * 3 * kFragElems, l);
      __builtin_amdgcn_sched_barrier(0);
      mma3(hi[b], lo[b], A, B[kc]);
      __builtin_amdgcn_sched_barrier(0);
      A = An;
      if (j == KH - 1) {
        stream_store(ch + 1, 0);
        stream_load(ch + 1, 1);
      }
    }
    stream_store(ch + 1, 1);
    __syncthreads();
  };
  // one k slice of the second: acc[rb] += A[rb] . B; inf: infinities are kept (S5; in the recomputation an infinite
  // activation ends in SiLU' = NaN in any case)
  auto slice_chunk = [&](int ch, const Chunk3& B, f32x4* acc, auto inf) {
    const bf16* W = s_w[ch & 1];
    stream_load(ch + 1, 0);
    Chunk3 A = lds_chunk3(W, l);
#pragma unroll
    for (int rb = 0; rb < 8; ++rb) {
      Chunk3 An = A;
      if (rb + 1 < 8) An = lds_chunk3(W + (rb + 1) * 3 * kFragElems, l);
      __builtin_amdgcn_sched_barrier(0);
      f32x4 lo = zero4();
      mma3(acc[rb], lo, A, B);
      acc[rb] = inf ? joined(acc[rb], lo) : acc[rb] + lo;
      __builtin_amdgcn_sched_barrier(0);
      A = An;
      if (rb == 3) {
        stream_store(ch + 1, 0);
        stream_load(ch + 1, 1);
      }
    }
    stream_store(ch + 1, 1);
    __syncthreads();
  };

  stream_load(0, 0);
  stream_store(0, 0);
  stream_load(0, 1);
  stream_store(0, 1);
  float sw2[2] = {0.f, 0.f}, swd[2] = {0.f, 0.f};   // the lane's sums of dw2_mov and dw_d: feature fsum of each 64
  const int fsum = 16 * (c >> 2) + 4 * g + (c & 3);
  __syncthreads();

  for (int64_t ps = blockIdx.x; ps < npass; ps += gridDim.x) {
    __asm__ __volatile__("" : "+v"(so));
    const int64_t e0 = ebeg + (ps * kF32Waves + w) * 16 + c;
    const bool valid = e0 < eend;
    const int64_t ee = valid ? e0 : eend - 1;
    const int ri = clampi(a.erow[ee], (int)a.N), rj = clampi(a.col[ee], (int)a.N);
    const int64_t fo = (ee - a.fbase) * H + 4 * g;   // the lane's first element of the edge's factor rows
    float dx = 0.f, dy = 0.f, dz = 0.f, r2 = 0.f, gxx = 0.f, gxy = 0.f, gxz = 0.f, gphi = 0.f;
    if constexpr (EQ) {
      const float* xi = a.coord + (int64_t)ri * a.sc;
      const float* xj = a.coord + (int64_t)rj * a.sc;
      dx = xi[0] - xj[0];
      dy = xi[1] - xj[1];
      dz = xi[2] - xj[2];
      r2 = dx * dx + dy * dy + dz * dz;
      if (valid) {
        const float* gx = a.gmov + (int64_t)ri * a.sgx;
        float sc = 1.0f;
        if (a.mean) {
          const int deg = a.rowptr[ri + 1] - a.rowptr[ri];
          sc = 1.0f / (float)(deg > 1 ? deg : 1);
        }
        gxx = gx[0] * sc;
        gxy = gx[1] * sc;
        gxz = gx[2] * sc;
      }
      gphi = dx * gxx + dy * gxy + dz * gxz;
    }
    // ---- S1
    Chunk3 m1[KH];
    f32x4 s1last = zero4();
    {
      f32x4 y[KH][2];
#pragma unroll
      for (int kc = 0; kc < KH; ++kc) {
        const f32x8 p = load_chunk(PQ + (int64_t)ri * 2 * H + 32 * kc + 8 * g);
        const f32x8 q = load_chunk(PQ + (int64_t)rj * 2 * H + H + 32 * kc + 8 * g);
        y[kc][0] = p.lo + q.lo;
        y[kc][1] = p.hi + q.hi;
      }
      if constexpr (FEAT) {
        const int eid = a.eids ? clampi(a.eids[ee], (int)E) : (int)ee;
        for (int uc = 0; uc < a.NUC; ++uc) {
          const int s0 = 32 * uc + 8 * g;
          f32x8 u = zero_chunk<float>();
          if (s0 + 8 <= a.FE) u = load_chunk(ef + (int64_t)eid * a.se + s0);
          else if (EQ && s0 == a.FE) u.lo[0] = r2;
          const Chunk3 u3 = split_chunk(u.lo * sg, u.hi * sg);
#pragma unroll
          for (int rb = 0; rb < H / 16; ++rb) {
            const Chunk3 A = lds_chunk3((const bf16*)a.fr.s_u + ((int64_t)(rb >> 1) * 6 * a.NUC + ((rb & 1) * a.NUC + uc) * 3) * kFragElems, l);
            f32x4 lo = zero4(), hi = zero4();
            mma3(hi, lo, A, u3);
            y[rb >> 1][rb & 1] = add_signed(y[rb >> 1][rb & 1], hi + lo, sg);
          }
        }
      } else if constexpr (EQ) {
#pragma unroll
        for (int rb = 0; rb < H / 16; ++rb) {
          const f32x4 wd = *reinterpret_cast<const f32x4*>(s_vec + O + 2 * M + 16 * rb + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) y[rb >> 1][rb & 1][i] = __builtin_fmaf(r2, wd[i], y[rb >> 1][rb & 1][i]);
        }
      }
#pragma unroll
      for (int kc = 0; kc < KH; ++kc) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          f32x4 d;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const YD r = silu_yd_f32(y[kc][b][i], sg);
            y[kc][b][i] = r.y;
            d[i] = r.d;
          }
          if (2 * kc + b < 7) s_d1[w][2 * kc + b][l] = d;
          else s1last = d;
          if (valid) *reinterpret_cast<f32x4*>((float*)a.Dm1 + fo + 32 * kc + 16 * b) = y[kc][b];
        }
        m1[kc] = split_chunk(y[kc][0], y[kc][1]);
      }
    }
    // ---- S2, S3
    f32x4 q[EQ ? M / 16 : 1], s2[KP][2];
    if constexpr (EQ) {
#pragma unroll
      for (int rb = 0; rb < M / 16; ++rb) q[rb] = zero4();
    }
#pragma unroll
    for (int kp = 0; kp < KP; ++kp) {
      f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()};
      rows_chunk(EQ ? 2 * kp : kp, m1, hi, lo);
      f32x4 x[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const f32x4 b2 = *reinterpret_cast<const f32x4*>(s_vec + 32 * kp + 16 * b + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const YD r = silu_yd_f32(__builtin_fmaf(hi[b][i] + lo[b][i], sg, b2[i]), sg);
          x[b][i] = r.y;
          s2[kp][b][i] = r.d;
        }
        if (EQ && valid) *reinterpret_cast<f32x4*>((float*)a.Dm + fo + 32 * kp + 16 * b) = x[b];
      }
      if constexpr (EQ) slice_chunk(2 * kp + 1, split_chunk(x[0], x[1]), q, std::false_type());
    }
    // ---- phi, g_q, dw2_mov
    float phi = 0.f;
    Chunk3 gq[EQ ? M / 32 : 1];
    if constexpr (EQ) {
      float pv[16];
      const float gpsg = gphi * sg;
#pragma unroll
      for (int kc = 0; kc < M / 32; ++kc) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int rb = 2 * kc + b;
          const f32x4 bx = *reinterpret_cast<const f32x4*>(s_vec + O + 16 * rb + 4 * g);
          const f32x4 w2 = *reinterpret_cast<const f32x4*>(s_vec + O + M + 16 * rb + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const YD r = silu_yd_f32(__builtin_fmaf(q[rb][i], sg, bx[i]), sg);
            phi += r.y * w2[i];
            pv[4 * (rb & 3) + i] = gpsg * r.y;
            q[rb][i] = gphi * w2[i] * r.d;
          }
          if (valid) *reinterpret_cast<f32x4*>((float*)a.Dgq + fo + 16 * rb) = q[rb];
        }
        gq[kc] = split_chunk(q[2 * kc], q[2 * kc + 1]);
        if (kc & 1) sw2[kc >> 1] += edge_sum16(pv, c);
        __asm__ __volatile__("" : "+v"(phi));   // summed here, not at the end of all four
      }
      phi *= sg;
      phi += shfl_xor(phi, 16);
      phi += shfl_xor(phi, 32);
    }
    // ---- S4, S5
    f32x4 ga1[H / 16];
#pragma unroll
    for (int rb = 0; rb < H / 16; ++rb) ga1[rb] = zero4();
#pragma unroll
    for (int kp = 0; kp < KP; ++kp) {
      f32x4 x[2] = {zero4(), zero4()};
      if (valid) {
#pragma unroll
        for (int b = 0; b < 2; ++b) x[b] = load4_f32(gmsg + (int64_t)ri * a.sgm + 32 * kp + 16 * b + 4 * g);
      }
      if constexpr (EQ) {
        f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()};
        rows_chunk(2 * KP + 2 * kp, gq, hi, lo);
#pragma unroll
        for (int b = 0; b < 2; ++b) x[b] = add_signed(x[b], joined(hi[b], lo[b]), sg);
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        x[b] *= s2[kp][b];
        if (valid) *reinterpret_cast<f32x4*>((float*)a.Dga2 + fo + 32 * kp + 16 * b) = x[b];
      }
      slice_chunk(EQ ? 2 * KP + 2 * kp + 1 : KP + kp, split_chunk(x[0], x[1]), ga1, std::true_type());
    }
    // ---- Gh, S6, dw_d
    {
      float gr = 0.f, gv[16];
      const int64_t go = (ee - a.gbase) * H + 4 * g;
#pragma unroll
      for (int rb = 0; rb < H / 16; ++rb) {
        const f32x4 v = ga1[rb] * (rb < 7 ? s_d1[w][rb][l] : s1last);
        if (valid) *reinterpret_cast<f32x4*>((float*)a.Gh + go + 16 * rb) = v;
        if constexpr (EQ) {
          const f32x4 wd = *reinterpret_cast<const f32x4*>(s_vec + O + 2 * M + 16 * rb + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            gr += v[i] * wd[i];
            gv[4 * (rb & 3) + i] = r2 * v[i];
          }
          if ((rb & 3) == 3) swd[rb >> 2] += edge_sum16(gv, c);
          __asm__ __volatile__("" : "+v"(gr));
        }
      }
      if constexpr (EQ) {
        gr += shfl_xor(gr, 16);
        gr += shfl_xor(gr, 32);
        if (g == 0 && valid) {
          const float k2 = 2.0f * gr;
          *reinterpret_cast<f32x4*>(a.Gx + (ee - a.gbase) * 4) =
              f32x4{phi * gxx + k2 * dx, phi * gxy + k2 * dy, phi * gxz + k2 * dz, gphi};
        }
      }
    }
  }
  if constexpr (EQ) {   // the block's partial row: the waves' sums in wave order, added to an earlier chunk's
    float* const s_sum = (float*)s_w[0];   // [wave][M | H]; the passes ended with a barrier
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s_sum[w * (M + H) + 64 * h + fsum] = sw2[h];
      s_sum[w * (M + H) + M + 64 * h + fsum] = swd[h];
    }
    __syncthreads();
    float* row = a.dwpart + (int64_t)blockIdx.x * (M + H);
    for (int q = threadIdx.x; q < M + H; q += 64 * kF32Waves) {
      float s = s_sum[q];
#pragma unroll
      for (int k = 1; k < kF32Waves; ++k) s += s_sum[k * (M + H) + q];
      row[q] = a.fbase > 0 ? row[q] + s : s;
    }
  }
}

// [A | 1]^T B over the edges of a chunk, A and B edge-major fp32 rows of 128 (W_hl: m1, g_a2; W1_mov: m, g_q):
// blockIdx.y selects the product, blockIdx.x a range of len edges.  Bound by reading A and B once, so a block
// (eight waves, one per CU) computes the whole 128 x 128 result of its range: slices of 32 edges, split into
// parts on the way to LDS ([edge][column] rows of 288 bytes, which the transposing reads of 32 lanes cross
// without bank conflicts), two slices in flight in registers and two in LDS.  The ones row (bias gradient) is the
// sum of the B values each thread loads, in fp32, odd edges subtracted (their rows are stored negative).  Each block adds
// to its partial row of an earlier chunk.
// Measured (both products, two chunks, with the matrix-vector products the backward kernel now sums itself):
// 750 -> 222 us at 394k edges (3.6 TB/s), 123 -> 27 us at 46k (one chunk).
constexpr int kAtbPitch = 144, kAtbSlice = 32, kAtbThreads = 512;
constexpr int kAtbPlane = kAtbSlice * kAtbPitch;
__device__ __forceinline__ bf16x8 tr_chunk(const bf16* p) {   // rows p + 0..3 and + 16..19 of the lane's k group
  const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)p);
  const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(p + 16 * kAtbPitch));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
__global__ __launch_bounds__(kAtbThreads, 2) void atb_f32_kernel(AtbF32Args a) {
  __shared__ __attribute__((aligned(16))) bf16 s_ab[2 * 6 * kAtbPlane];   // [buffer][A parts, B parts][kAtbPlane]
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, c = l & 15, g = l >> 4;
  const float* A = blockIdx.y ? a.A1 : a.A0;
  const float* B = blockIdx.y ? a.B1 : a.B0;
  const int64_t kb = (int64_t)blockIdx.x * a.len;   // len: a multiple of 64
  const int64_t ke = kb + a.len < a.K ? kb + a.len : a.K;
  const uint32_t flip = (blockIdx.x & 1) << 31;   // every other range (flip_sign)
  const float sgn = flip ? -1.0f : 1.0f;
  const int row = tid >> 5, q4 = 4 * (tid & 31);   // the thread's rows row, row + 16 of a slice, columns q4 .. + 3

  struct Regs { f32x4 a[2], b[2]; };
  auto load = [&](int64_t k0, Regs& r) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t k = k0 + row + 16 * i;
      r.a[i] = r.b[i] = zero4();
      if (k < ke) {
        r.a[i] = load4_f32(A + k * 128 + q4);
        r.b[i] = load4_f32(B + k * 128 + q4);
      }
    }
  };
  f32x4 ones = zero4();
  auto store = [&](int buf, const Regs& r) {
    bf16* base = s_ab + buf * 6 * kAtbPlane + q4;
    const Chunk3 ca = split_chunk(r.a[0], r.a[1]), cb = split_chunk(flip_sign(r.b[0], flip), flip_sign(r.b[1], flip));
    auto put = [&](int plane, const bf16x8& v) {
      bf16* p = base + plane * kAtbPlane + row * kAtbPitch;
      *reinterpret_cast<bf16x4*>(p) = __builtin_shufflevector(v, v, 0, 1, 2, 3);
      *reinterpret_cast<bf16x4*>(p + 16 * kAtbPitch) = __builtin_shufflevector(v, v, 4, 5, 6, 7);
    };
    put(0, ca.p0); put(1, ca.p1); put(2, ca.p2);
    put(3, cb.p0); put(4, cb.p1); put(5, cb.p2);
    ones += r.b[0] + r.b[1];
  };
  const int wm = w >> 2, wn = w & 3;   // the wave's 64 x 32 part of the result
  f32x4 hi[4][2], lo[4][2];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) hi[i][j] = lo[i][j] = zero4();
  auto compute = [&](int buf) {
    // lane c addresses row kb + c / 4, columns 4 (c % 4) .. + 3 of its block, and receives column c
    const bf16* p = s_ab + buf * 6 * kAtbPlane + (4 * g + (c >> 2)) * kAtbPitch + 4 * (c & 3);
    const bf16* pa = p + 64 * wm;
    const bf16* pb = p + 3 * kAtbPlane + 32 * wn;
    Chunk3 b[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
      b[j] = Chunk3{tr_chunk(pb + 16 * j), tr_chunk(pb + kAtbPlane + 16 * j), tr_chunk(pb + 2 * kAtbPlane + 16 * j)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Chunk3 x{tr_chunk(pa + 16 * i), tr_chunk(pa + kAtbPlane + 16 * i), tr_chunk(pa + 2 * kAtbPlane + 16 * i)};
      mma3(hi[i][0], lo[i][0], x, b[0]);
      mma3(hi[i][1], lo[i][1], x, b[1]);
    }
  };
  Regs r0, r1;
  load(kb, r0);
  load(kb + kAtbSlice, r1);
  store(0, r0);
  __syncthreads();
  for (int64_t k0 = kb; k0 < ke; k0 += 2 * kAtbSlice) {   // rows past ke read as zeros
    load(k0 + 2 * kAtbSlice, r0);
    compute(0);
    store(1, r1);
    __syncthreads();
    load(k0 + 3 * kAtbSlice, r1);
    compute(1);
    store(0, r0);
    __syncthreads();
  }
  float* P = a.part + (int64_t)blockIdx.x * a.ldp + (blockIdx.y ? 129 * 128 : 0);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (r == 0) hi[i][j] = joined(hi[i][j], lo[i][j]);
        float* o = P + (64 * wm + 16 * i + 4 * g + r) * 128 + 32 * wn + 16 * j + c;
        const float v = sgn * hi[i][j][r];
        *o = a.add ? *o + v : v;
      }
  float* s = (float*)s_ab;   // [16][128] sums of the thread rows
  *reinterpret_cast<f32x4*>(s + row * 128 + q4) = row & 1 ? -ones : ones;
  __syncthreads();
  if (tid < 128) {
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) v += s[k * 128 + tid];
    float* o = P + 128 * 128 + tid;
    *o = a.add ? *o + v : v;
  }
}

}  // namespace

bool f32_split_supported(const LayerShape& s) { return !s.bf16 && s.H == 128; }

int launch_f32_fwd(const LayerShape& s, const FwdArgs& a, hipStream_t st) {
  if (a.ntiles <= 0) return 0;
  const int blocks = (int)std::min<int64_t>((a.ntiles + 1) / 2, 512);   // two blocks per CU
  const dim3 grid(blocks), blk(64 * kF32Waves);
  if (s.eq && s.FE > 0) hipLaunchKernelGGL((f32_fwd_kernel<true, true>), grid, blk, 0, st, a);
  else if (s.eq) hipLaunchKernelGGL((f32_fwd_kernel<true, false>), grid, blk, 0, st, a);
  else if (s.FE > 0) hipLaunchKernelGGL((f32_fwd_kernel<false, true>), grid, blk, 0, st, a);
  else hipLaunchKernelGGL((f32_fwd_kernel<false, false>), grid, blk, 0, st, a);
  return (int)hipGetLastError();
}

int f32_bwd_blocks(int64_t E) { return (int)std::max<int64_t>(1, std::min<int64_t>(cdiv(E, 16 * kF32Waves), 512)); }

int launch_f32_bwd(const LayerShape& s, const BwdArgs& a, hipStream_t st) {
  const int64_t n = std::min<int64_t>(a.ntiles * kTileEdges, a.E) - a.tile0 * kTileEdges;
  if (n <= 0) return 0;
  const dim3 grid(f32_bwd_blocks(n)), blk(64 * kF32Waves);
  if (s.eq && s.FE > 0) hipLaunchKernelGGL((f32_bwd_kernel<true, true>), grid, blk, 0, st, a);
  else if (s.eq) hipLaunchKernelGGL((f32_bwd_kernel<true, false>), grid, blk, 0, st, a);
  else if (s.FE > 0) hipLaunchKernelGGL((f32_bwd_kernel<false, true>), grid, blk, 0, st, a);
  else hipLaunchKernelGGL((f32_bwd_kernel<false, false>), grid, blk, 0, st, a);
  return (int)hipGetLastError();
}

// ranges of at least 128 edges, at most 128 of them (two products: one block per CU)
int64_t atb_f32_len(int64_t K) { return cdiv(cdiv(std::max<int64_t>(K, 1), std::min<int64_t>(128, cdiv(std::max<int64_t>(K, 1), 128))), 64) * 64; }

int launch_atb_f32(AtbF32Args a, int products, hipStream_t st) {
  if (a.K <= 0) return 0;
  hipLaunchKernelGGL(atb_f32_kernel, dim3((unsigned)cdiv(a.K, a.len), (unsigned)products), dim3(kAtbThreads), 0, st, a);
  return (int)hipGetLastError();
}

}  // namespace egnn
