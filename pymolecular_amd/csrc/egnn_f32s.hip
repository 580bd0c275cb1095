// fp32 edge kernels of the layer at the reference's widths (H = 64, O = M = 32, at most 32 edge-input slots), on
// split bf16 operands (egnn_split.h).
//
// All weights in three parts are 30 KB here, so they stay in LDS and the waves run free of barriers: each wave
// takes whole 32-edge schedule tiles (forward: two 16-edge column blocks side by side, so that each weight fragment
// read from LDS feeds twelve products) or 16 edges (backward), features on the MFMA rows, every stage's C-blocks the
// next stage's B operand.  Two blocks of four waves (forward: three) per CU; vector instructions (SiLU, the splits)
// bound both kernels.
// Measured against one wave per 32-edge tile on the fp32 instruction with the factors of the weight gradients in
// memory (E = 1.28M, F_E = 16): forward 306 -> 168 us; backward and its weight gradients 1,990 -> 444 us, 52 -> 2
// launches.
#include "egnn_device.h"
#include "egnn_internal.h"
#include "egnn_split.h"
#include "egnn_tile.h"

namespace egnn {
namespace {

using namespace split;

constexpr int kW = 4, H = 64, O = 32, M = 32, KH = H / 32;

// fp32 fragments (64 lanes x 8) -> three parts each, [fragment][part]
__device__ __forceinline__ void split_frags(bf16* dst, const float* src, int nfrag) {
  for (int q = threadIdx.x; q < nfrag * 64; q += 64 * kW) {
    const f32x8 v = load_chunk(src + q * 8);
    const Chunk3 s = split_chunk(v.lo, v.hi);
    bf16* d = dst + ((q >> 6) * 3 * 64 + (q & 63)) * 8;
    store_chunk(d, s.p0);
    store_chunk(d + kFragElems, s.p1);
    store_chunk(d + 2 * kFragElems, s.p2);
  }
}
__device__ __forceinline__ Chunk3 frag3(const bf16* f, int l) {
  const bf16* p = f + l * 8;
  return Chunk3{load_chunk(p), load_chunk(p + kFragElems), load_chunk(p + 2 * kFragElems)};
}
// r^2 and delta of an edge
struct Geo { float dx, dy, dz, r2; };
__device__ __forceinline__ Geo edge_delta(const float* coord, int64_t sc, int ri, int rj) {
  const float* xi = coord + (int64_t)ri * sc;
  const float* xj = coord + (int64_t)rj * sc;
  Geo d{xi[0] - xj[0], xi[1] - xj[1], xi[2] - xj[2], 0.f};
  d.r2 = d.dx * d.dx + d.dy * d.dy + d.dz * d.dz;
  return d;
}
// the lane's eight edge-input slots [e, r^2]
template <bool EQ, bool FEAT>
__device__ __forceinline__ f32x8 edge_slots(const float* ef, int64_t se, int eid, int FE, int g, float r2) {
  f32x8 u = zero_chunk<float>();
  if (FEAT && 8 * g + 8 <= FE) u = load_chunk(ef + (int64_t)eid * se + 8 * g);
  else if (EQ && 8 * g == FE) u.lo[0] = r2;
  return u;
}

template <bool EQ, bool FEAT>
__global__ __launch_bounds__(64 * kW, 3) void f32s_fwd_kernel(FwdArgs a) {
  constexpr int SEGW = O + (EQ ? 4 : 0), SP = SEGW + 4;
  constexpr bool U = EQ || FEAT;
  __shared__ __attribute__((aligned(16))) bf16 s_hlT[2 * KH * 3 * kFragElems];
  __shared__ __attribute__((aligned(16))) bf16 s_movT[EQ ? 2 * 3 * kFragElems : 8];
  __shared__ __attribute__((aligned(16))) bf16 s_u[U ? 4 * 3 * kFragElems : 8];
  __shared__ __attribute__((aligned(16))) float s_vec[O + 2 * M];   // b2 | bx1 | w2_mov
  __shared__ __attribute__((aligned(16))) float s_msg[kW][kTileEdges * SP];

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  const float sg = bitsf(0x3f800000u | (uint32_t)(c & 1) << 31);   // the edge's sign in the chain, 1 or -1
  const float* PQ = (const float*)a.PQ;
  const float* ef = (const float*)a.ef;
  const int64_t E = a.E;
  split_frags(s_hlT, (const float*)a.fr.hlT, 2 * KH);
  if constexpr (EQ) split_frags(s_movT, (const float*)a.fr.movT, 2);
  if constexpr (U) split_frags(s_u, (const float*)a.fr.u, 4);
  if (threadIdx.x < O) {
    s_vec[threadIdx.x] = a.fr.b2f[threadIdx.x];
    s_vec[O + threadIdx.x] = a.fr.bx1f[threadIdx.x];
    s_vec[O + M + threadIdx.x] = a.fr.w2mf[threadIdx.x];
  }
  __syncthreads();

  float* const msg = s_msg[w];
  const int64_t nw = (int64_t)gridDim.x * kW;
  for (int64_t T = (int64_t)blockIdx.x * kW + w; T < a.ntiles; T += nw) {
    const int64_t base = T * kTileEdges;
    const int tabv = a.tile_tab[T * kTabInts + l];
    const int64_t eo = base + (l & 31);
    int ri[2], rj[2];
    Geo d[2];
    f32x4 y[KH][2][2];   // [kc][column block][16-row half]
    f32x8 u[2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int64_t e0 = base + 16 * nb + c, e = e0 < E ? e0 : E - 1;
      ri[nb] = clampi(a.erow[e], (int)a.N);
      rj[nb] = clampi(a.col[e], (int)a.N);
      if constexpr (EQ) d[nb] = edge_delta(a.coord, a.sc, ri[nb], rj[nb]);
      const int eid = FEAT ? (a.eids ? clampi(a.eids[e], (int)E) : (int)e) : 0;
      if constexpr (U) u[nb] = edge_slots<EQ, FEAT>(ef, a.se, eid, a.FE, g, EQ ? d[nb].r2 : 0.f);
#pragma unroll
      for (int kc = 0; kc < KH; ++kc) {
        const f32x8 p = load_chunk(PQ + (int64_t)ri[nb] * 2 * H + 32 * kc + 8 * g);
        const f32x8 q = load_chunk(PQ + (int64_t)rj[nb] * 2 * H + H + 32 * kc + 8 * g);
        y[kc][nb][0] = p.lo + q.lo;
        y[kc][nb][1] = p.hi + q.hi;
      }
    }
    uint32_t ends;   // last edge of each run of one row in the tile
    {
      const int er = a.erow[eo < E ? eo : E - 1];
      const int en = __shfl(er, l + 1 < 64 ? l + 1 : 63, 64);
      ends = (uint32_t)__ballot(l < kTileEdges && eo < E && (l == kTileEdges - 1 || eo == E - 1 || er != en));
    }
    // ---- S1
    Chunk3 m1[KH][2];
    {
      Chunk3 u3[2];
      if constexpr (U) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) u3[nb] = split_chunk(u[nb].lo * sg, u[nb].hi * sg);
      }
#pragma unroll
      for (int rb = 0; rb < H / 16; ++rb) {
        if constexpr (U) {
          const Chunk3 A = frag3(s_u + rb * 3 * kFragElems, l);
          f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()};
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) mma3(hi[nb], lo[nb], A, u3[nb]);
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) y[rb >> 1][nb][rb & 1] = add_signed(y[rb >> 1][nb][rb & 1], joined(hi[nb], lo[nb]), sg);
        }
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int i = 0; i < 4; ++i) y[rb >> 1][nb][rb & 1][i] = silu_f32(y[rb >> 1][nb][rb & 1][i], sg);
        if (rb & 1) {
#pragma unroll
          for (int nb = 0; nb < 2; ++nb) m1[rb >> 1][nb] = split_chunk(y[rb >> 1][nb][0], y[rb >> 1][nb][1]);
        }
      }
    }
    // ---- S2; the messages to the wave's rows
    f32x4 x[2][2];   // [column block][row block]
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()};
#pragma unroll
      for (int kc = 0; kc < KH; ++kc) {
        const Chunk3 A = frag3(s_hlT + (b * KH + kc) * 3 * kFragElems, l);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) mma3(hi[nb], lo[nb], A, m1[kc][nb]);
      }
      const f32x4 b2 = *reinterpret_cast<const f32x4*>(s_vec + 16 * b + 4 * g);
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        const f32x4 p = joined(hi[nb], lo[nb]);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[nb][b][i] = silu_f32(__builtin_fmaf(p[i], sg, b2[i]), sg);
        *reinterpret_cast<f32x4*>(msg + (16 * nb + c) * SP + 16 * b + 4 * g) = x[nb][b];
      }
    }
    // ---- S3
    if constexpr (EQ) {
      float phi[2] = {0.f, 0.f};
      Chunk3 mc[2];
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) mc[nb] = split_chunk(x[nb][0], x[nb][1]);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()};
        const Chunk3 A = frag3(s_movT + b * 3 * kFragElems, l);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb) mma3(hi[nb], lo[nb], A, mc[nb]);
        const f32x4 bx = *reinterpret_cast<const f32x4*>(s_vec + O + 16 * b + 4 * g);
        const f32x4 w2 = *reinterpret_cast<const f32x4*>(s_vec + O + M + 16 * b + 4 * g);
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)   // not joined: an infinite message makes phi NaN by its SiLU(-inf) too
#pragma unroll
          for (int i = 0; i < 4; ++i) phi[nb] += silu_f32(__builtin_fmaf(hi[nb][i] + lo[nb][i], sg, bx[i])) * w2[i];
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) {
        phi[nb] *= sg;   // signed as the messages are
        phi[nb] += shfl_xor(phi[nb], 16);
        phi[nb] += shfl_xor(phi[nb], 32);
        if (g == 0)
          *reinterpret_cast<f32x4*>(msg + (16 * nb + c) * SP + O) = f32x4{d[nb].dx * phi[nb], d[nb].dy * phi[nb], d[nb].dz * phi[nb], 0.f};
      }
    }
    // ---- row sums in edge order: lane l < 32 message feature l, lanes 32 .. 34 the coordinates
    wave_sync();
    {
      const int col = l < SEGW ? l : 0;
      const bool whole = tabv >= 0;   // lane r: rank r of the tile
      float* const cslot = a.carry + (T * 2 + (tabv == -2)) * SEGW;
      float* const pm = whole ? (float*)a.out_msg + (int64_t)tabv * a.smsg : cslot;
      float* const px = EQ && whole ? a.out_mov + (int64_t)tabv * a.smov : cslot + O;
      const uint32_t mlo = (uint32_t)(uintptr_t)pm, mhi = (uint32_t)((uintptr_t)pm >> 32);
      const uint32_t xlo = (uint32_t)(uintptr_t)px, xhi = (uint32_t)((uintptr_t)px >> 32);
      float acc = 0.f;
      int r = 0, n = 0;
#pragma unroll
      for (int k0 = 0; k0 < kTileEdges; k0 += 8) {
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = msg[(k0 + k) * SP + col];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          acc += k & 1 ? -v[k] : v[k];   // the rows hold signed values
          ++n;
          if ((ends >> (k0 + k)) & 1u) {
            typedef __attribute__((address_space(1))) float gfloat;
            gfloat* const om = (gfloat*)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)mhi, r) << 32) |
                                       (uint32_t)__builtin_amdgcn_readlane((int)mlo, r));
            if (l < O) om[l] = acc;
            if constexpr (EQ) {
              gfloat* const ox = (gfloat*)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)xhi, r) << 32) |
                                         (uint32_t)__builtin_amdgcn_readlane((int)xlo, r));
              if (l >= O && l < O + 3) ox[l - O] = a.mean && __builtin_amdgcn_readlane(tabv, r) >= 0 ? acc / (float)n : acc;
            }
            acc = 0.f;
            n = 0;
            ++r;
          }
        }
      }
    }
    wave_sync();
  }
}

// ---- backward ---------------------------------------------------------------------------------------------------
// A weight of 32 columns in LDS, three planes of 64-byte rows whose 8-byte unit u of row r sits at u ^ swz(r): the
// row reads (16 rows at one unit) and the transposing reads (eight rows, four units) of 32 lanes then fall on all
// 64 banks.
__device__ __forceinline__ int swz(int r) { return (((r >> 2) & 1) << 2) | (((r >> 3) & 1) << 1); }
template <int R>
__device__ __forceinline__ Chunk3 w_rows3(const bf16* W, int blk, int c, int g) {   // A[r][k] = W[16 blk + r][kappa_chain]
  const int r = 16 * blk + c;
  const bf16* p = W + r * 32;
  auto one = [&](const bf16* q) {
    return __builtin_shufflevector(*reinterpret_cast<const bf16x4*>(q + 4 * (g ^ swz(r))),
                                   *reinterpret_cast<const bf16x4*>(q + 4 * ((4 + g) ^ swz(r))), 0, 1, 2, 3, 4, 5, 6, 7);
  };
  return Chunk3{one(p), one(p + R * 32), one(p + 2 * R * 32)};
}
template <int R>
__device__ __forceinline__ Chunk3 w_cols3(const bf16* W, int blk, int kc, int c, int g) {   // A[r][k] = W[32 kc + k][16 blk + r]
  const int r = 32 * kc + 4 * g + (c >> 2);
  const bf16* p = W + r * 32 + 4 * ((4 * blk + (c & 3)) ^ swz(r));   // swz(r + 16) = swz(r)
  auto one = [&](const bf16* q) {
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)q);
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(q + 16 * 32));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  return Chunk3{one(p), one(p + R * 32), one(p + 2 * R * 32)};
}
// W[r][k] (R x 32) from W row-major, or from its transpose (lin)
template <int R>
__device__ __forceinline__ void fill_w3(bf16* dst, const float* src, bool lin) {
  for (int q = threadIdx.x; q < R * 32; q += 64 * kW) {
    const int r = q >> 5, k = q & 31;
    bf16* p = dst + r * 32 + 4 * ((k >> 2) ^ swz(r)) + (k & 3);
    split1(lin ? src[k * R + r] : src[q], p[0], p[R * 32], p[2 * R * 32]);
  }
}

// v made opaque: what follows cannot reuse what was derived from it before (its parts would stay in registers)
__device__ __forceinline__ void opaque(f32x4& v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float t = v[i];
    __asm__ __volatile__("" : "+v"(t));
    v[i] = t;
  }
}

// an exchange slot: 32 features x 16 edges in three parts, [part][64 lanes][8]
constexpr int kSlot = 3 * kFragElems;
__device__ __forceinline__ void put_slot(bf16* s, int l, const Chunk3& v) {
  bf16* p = s + tile::chain_slot<true>(l) * 8;
  store_chunk(p, v.p0);
  store_chunk(p + kFragElems, v.p1);
  store_chunk(p + 2 * kFragElems, v.p2);
}
// block blk (16 features) of a slot edge-major: lane (c, g) holds edges 4g .. 4g + 3 of feature c
struct Quad3 { bf16x4 p0, p1, p2; };
__device__ __forceinline__ Quad3 get_slot(const bf16* s, int blk, int c, int g) {
  const bf16* p = s + tile::chain_slot<true>(16 * (c & 3) + 4 * g + (c >> 2)) * 8 + 4 * blk;
  auto one = [&](const bf16* q) { return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)q); };
  return Quad3{one(p), one(p + kFragElems), one(p + 2 * kFragElems)};
}
// acc += A^T B over the 16 edges: the corrections, then the large term (one accumulator, so an infinite operand gives NaN)
__device__ __forceinline__ void mma16(f32x4& acc, const bf16x4& a, const bf16x4& b) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), acc, 0, 0, 0);
}
// v with the sign bits of flip (0 or 0x80008000) changed
__device__ __forceinline__ bf16x4 flip4(const bf16x4& v, uint32_t flip) {
  const u32x2 x = __builtin_bit_cast(u32x2, v);
  return __builtin_bit_cast(bf16x4, u32x2{x[0] ^ flip, x[1] ^ flip});
}
__device__ __forceinline__ Quad3 flip3(const Quad3& v, uint32_t flip) { return Quad3{flip4(v.p0, flip), flip4(v.p1, flip), flip4(v.p2, flip)}; }
__device__ __forceinline__ void mma3e(f32x4& acc0, f32x4& acc1, const Quad3& a, const Quad3& b, const Quad3& d) {
  mma16(acc0, a.p2, b.p0);
  mma16(acc1, a.p2, d.p0);
  mma16(acc0, a.p0, b.p2);
  mma16(acc1, a.p0, d.p2);
  mma16(acc0, a.p1, b.p1);
  mma16(acc1, a.p1, d.p1);
  mma16(acc0, a.p1, b.p0);
  mma16(acc1, a.p1, d.p0);
  mma16(acc0, a.p0, b.p1);
  mma16(acc1, a.p0, d.p1);
  mma16(acc0, a.p0, b.p0);
  mma16(acc1, a.p0, d.p0);
}

// sums over the 16 edges (lanes c) of eight values that carry the edges' signs (odd lanes negative, so the exchanges with
// a lane of the other parity subtract); lane c ends with that of value c >> 1, odd lanes with its negative
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float edge_sums8(const f32x4& a, const f32x4& b, int c) {
  f32x4 v;
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = (c & 8 ? b[k] : a[k]) + dpp<0x128>(c & 8 ? a[k] : b[k]);       // row_ror:8
  const float p = (c & 4 ? v[2] : v[0]) - dpp<0x141>(c & 4 ? v[0] : v[2]);                           // row_half_mirror
  const float q = (c & 4 ? v[3] : v[1]) - dpp<0x141>(c & 4 ? v[1] : v[3]);
  const float r = (c & 2 ? q : p) + dpp<0x4E>(c & 2 ? p : q);                                        // quad_perm [2, 3, 0, 1]
  return r - dpp<0xB1>(r);                                                                           // quad_perm [1, 0, 3, 2]
}

// The whole backward of 16 edges per wave: the chain of egnn_bwd.hip, then every weight gradient from the wave's own
// operands, so nothing but Gh and Gx goes to memory.  m1, m, g_q, g_a2 and the edge inputs carry the edge's
// sign, Gh does not; a product of two signed operands is what it was.  The contractions over the edges (16-deep products) read both
// operands edge-major by transposing reads of the wave's 12 KB exchange buffer (m1, then g_a1; m, then g_a2; g_q,
// then the edge inputs) and accumulate in 80 registers over the wave's edges; 32 edges at a time would use the
// 32-deep products but not fit the registers.  The block's waves are added in wave order into one partial row in the
// layout of coop_dw_len.
template <bool EQ, bool FEAT>
__global__ __launch_bounds__(64 * kW, 2) void f32s_bwd_kernel(BwdArgs a) {
  constexpr bool U = EQ || FEAT;
  __shared__ __attribute__((aligned(16))) bf16 s_hl[3 * H * 32];               // W_hl[h][o]
  __shared__ __attribute__((aligned(16))) bf16 s_mov[EQ ? 3 * O * 32 : 8];     // W1_mov[o][m]
  __shared__ __attribute__((aligned(16))) bf16 s_u[U ? 4 * 3 * kFragElems : 8];
  __shared__ __attribute__((aligned(16))) float s_vec[O + 2 * M + H];          // b2 | bx1 | w2_mov | w_d
  __shared__ __attribute__((aligned(16))) bf16 s_x[kW][4 * kSlot];

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  const float sg = bitsf(0x3f800000u | (uint32_t)(c & 1) << 31);   // the edge's sign in the chain, 1 or -1
  const float* PQ = (const float*)a.PQ;
  const float* ef = (const float*)a.ef;
  const float* gmsg = (const float*)a.gmsg;
  const int64_t E = a.E;
  fill_w3<H>(s_hl, (const float*)a.w2, a.lin);
  if constexpr (EQ) fill_w3<O>(s_mov, (const float*)a.w1m, a.lin);
  if constexpr (U) split_frags(s_u, (const float*)a.fr.u, 4);
  if (threadIdx.x < O) {
    s_vec[threadIdx.x] = a.fr.b2f[threadIdx.x];
    s_vec[O + threadIdx.x] = a.fr.bx1f[threadIdx.x];
    s_vec[O + M + threadIdx.x] = a.fr.w2mf[threadIdx.x];
  }
  if (threadIdx.x < H) s_vec[O + 2 * M + threadIdx.x] = a.fr.wdf[threadIdx.x];
  __syncthreads();

  bf16* const sx = s_x[w];          // m1, then g_a1 (two slots)
  bf16* const sy = sx + 2 * kSlot;  // m, then g_a2
  bf16* const sz = sx + 3 * kSlot;  // g_q, then the edge inputs
  f32x4 gwh[4][2], gwm[2][2], gwu[4][2];   // dW_hl, dW1_mov, d[W_e | w_d] (columns: slots 8 (c / 4) + 4 b + c % 4)
  float sb2 = 0.f, sbx = 0.f, sw2 = 0.f;   // db2, dbx1, dw2_mov of feature 16 (n / 4) + 4 g + n % 4, n = c / 2
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      gwh[i][j] = gwu[i][j] = zero4();
      if (i < 2) gwm[i][j] = zero4();
    }

  const int64_t ebeg = a.tile0 * kTileEdges, eend = a.ntiles * kTileEdges < E ? a.ntiles * kTileEdges : E;
  const int64_t step = (int64_t)gridDim.x * kW * 16;
  // every other wave contracts with -B (flip_sign): at 1.9M edges dW1_mov is 2.6e-7 off float64, without it 1.05e-6
  const uint32_t flip = w & 1 ? 0x80008000u : 0u;
  for (int64_t base = ebeg + ((int64_t)blockIdx.x * kW + w) * 16; base < eend; base += step) {
    const bool valid = base + c < eend;
    const int64_t ee = valid ? base + c : eend - 1;
    const int ri = clampi(a.erow[ee], (int)a.N), rj = clampi(a.col[ee], (int)a.N);
    Geo d{0.f, 0.f, 0.f, 0.f};
    float gx0 = 0.f, gx1 = 0.f, gx2 = 0.f, gphi = 0.f;
    if constexpr (EQ) {
      d = edge_delta(a.coord, a.sc, ri, rj);
      if (valid) {
        const float* p = a.gmov + (int64_t)ri * a.sgx;
        float sc = 1.0f;
        if (a.mean) {
          const int deg = a.rowptr[ri + 1] - a.rowptr[ri];
          sc = 1.0f / (float)(deg > 1 ? deg : 1);
        }
        gx0 = p[0] * sc;
        gx1 = p[1] * sc;
        gx2 = p[2] * sc;
      }
      gphi = d.dx * gx0 + d.dy * gx1 + d.dz * gx2;
    }
    f32x8 u;
    if constexpr (U) {
      const int eid = FEAT ? (a.eids ? clampi(a.eids[ee], (int)E) : (int)ee) : 0;
      u = edge_slots<EQ, FEAT>(ef, a.se, eid, a.FE, g, FEAT ? d.r2 : sg * d.r2);
    }
    // ---- S1
    f32x4 s1[4];
    Chunk3 m1[KH];
    {
      f32x4 y[4];
#pragma unroll
      for (int kc = 0; kc < KH; ++kc) {
        const f32x8 p = load_chunk(PQ + (int64_t)ri * 2 * H + 32 * kc + 8 * g);
        const f32x8 q = load_chunk(PQ + (int64_t)rj * 2 * H + H + 32 * kc + 8 * g);
        y[2 * kc] = p.lo + q.lo;
        y[2 * kc + 1] = p.hi + q.hi;
      }
      if constexpr (U) {
        if constexpr (FEAT) {
          const uint32_t odd = c & 1 ? 1u << 31 : 0u;
          u.lo = flip_sign(u.lo, odd);
          u.hi = flip_sign(u.hi, odd);
        }
        const Chunk3 u3 = split_chunk(u.lo, u.hi);
#pragma unroll
        for (int rb = 0; rb < 4; rb += 2) {
          f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()};
          mma3x2(hi, lo, frag3(s_u + rb * 3 * kFragElems, l), frag3(s_u + (rb + 1) * 3 * kFragElems, l), u3);
          y[rb] = add_signed(y[rb], hi[0] + lo[0], sg);
          y[rb + 1] = add_signed(y[rb + 1], hi[1] + lo[1], sg);
        }
        opaque(u.lo);   // split again for d[W_e | w_d]
        opaque(u.hi);
      }
#pragma unroll
      for (int rb = 0; rb < 4; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const YD r = silu_yd_f32(y[rb][i], sg);
          y[rb][i] = r.y;
          s1[rb][i] = r.d;
        }
#pragma unroll
      for (int kc = 0; kc < KH; ++kc) {
        m1[kc] = split_chunk(y[2 * kc], y[2 * kc + 1]);
        put_slot(sx + kc * kSlot, l, m1[kc]);
      }
    }
    // ---- S2
    f32x4 x[2], s2[2];
    {
      f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()};
#pragma unroll
      for (int kc = 0; kc < KH; ++kc)   // W_hl^T
        mma3x2(hi, lo, w_cols3<H>(s_hl, 0, kc, c, g), w_cols3<H>(s_hl, 1, kc, c, g), m1[kc]);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const f32x4 b2 = *reinterpret_cast<const f32x4*>(s_vec + 16 * b + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const YD r = silu_yd_f32(__builtin_fmaf(hi[b][i] + lo[b][i], sg, b2[i]), sg);
          x[b][i] = r.y;
          s2[b][i] = r.d;
        }
      }
    }
    // ---- S3: phi, g_q, dw2_mov, dbx1, dW1_mov
    float phi = 0.f;
    Chunk3 gq;
    if constexpr (EQ) {
      const Chunk3 mc = split_chunk(x[0], x[1]);
      put_slot(sy, l, mc);
      f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()};
      mma3x2(hi, lo, w_cols3<O>(s_mov, 0, 0, c, g), w_cols3<O>(s_mov, 1, 0, c, g), mc);   // W1_mov^T
      f32x4 gv[2], pb[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const f32x4 bx = *reinterpret_cast<const f32x4*>(s_vec + O + 16 * b + 4 * g);
        const f32x4 w2 = *reinterpret_cast<const f32x4*>(s_vec + O + M + 16 * b + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const YD r = silu_yd_f32(__builtin_fmaf(hi[b][i] + lo[b][i], sg, bx[i]), sg);
          phi += r.y * w2[i];
          pb[b][i] = gphi * r.y;
          gv[b][i] = gphi * w2[i] * r.d;
        }
      }
      gq = split_chunk(gv[0], gv[1]);
      put_slot(sz, l, gq);
      phi *= sg;
      phi += shfl_xor(phi, 16);
      phi += shfl_xor(phi, 32);
      sw2 += edge_sums8(pb[0], pb[1], c);
      sbx += edge_sums8(gv[0], gv[1], c);
      wave_sync();
      const Quad3 B0 = flip3(get_slot(sz, 0, c, g), flip), B1 = flip3(get_slot(sz, 1, c, g), flip);
#pragma unroll
      for (int b = 0; b < 2; ++b) mma3e(gwm[b][0], gwm[b][1], get_slot(sy, b, c, g), B0, B1);
      wave_sync();
    }
    // ---- S4: g_a2, db2, dW_hl
    Chunk3 ga2;
    {
      f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()}, v[2];
      if constexpr (EQ) mma3x2(hi, lo, w_rows3<O>(s_mov, 0, c, g), w_rows3<O>(s_mov, 1, c, g), gq);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        f32x4 gm = zero4();
        if (valid) gm = load4_f32(gmsg + (int64_t)ri * a.sgm + 16 * b + 4 * g);
        v[b] = add_signed(gm, joined(hi[b], lo[b]), sg) * s2[b];
      }
      sb2 += edge_sums8(v[0], v[1], c);
      ga2 = split_chunk(v[0], v[1]);
      put_slot(sy, l, ga2);
      if constexpr (U) put_slot(sz, l, split_chunk(u.lo, u.hi));
      wave_sync();
      const Quad3 B0 = flip3(get_slot(sy, 0, c, g), flip), B1 = flip3(get_slot(sy, 1, c, g), flip);
#pragma unroll
      for (int hb = 0; hb < 4; ++hb) mma3e(gwh[hb][0], gwh[hb][1], get_slot(sx + (hb >> 1) * kSlot, hb & 1, c, g), B0, B1);
      wave_sync();
    }
    // ---- S5: g_a1 = dL/dpre1; S6; d[W_e | w_d]
    float gr = 0.f;
#pragma unroll
    for (int kc = 0; kc < KH; ++kc) {
      f32x4 hi[2] = {zero4(), zero4()}, lo[2] = {zero4(), zero4()}, v[2];
      mma3x2(hi, lo, w_rows3<H>(s_hl, 2 * kc, c, g), w_rows3<H>(s_hl, 2 * kc + 1, c, g), ga2);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        v[b] = joined(hi[b], lo[b]) * s1[2 * kc + b];
        if (valid) *reinterpret_cast<f32x4*>((float*)a.Gh + (ee - a.gbase) * H + 32 * kc + 16 * b + 4 * g) = v[b];
        if constexpr (EQ) {
          const f32x4 wd = *reinterpret_cast<const f32x4*>(s_vec + O + 2 * M + 32 * kc + 16 * b + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) gr += v[b][i] * wd[i];
        }
      }
      if constexpr (U) put_slot(sx + kc * kSlot, l, split_chunk(v[0], v[1]));
    }
    if constexpr (U) {
      wave_sync();
      const uint32_t fu = flip ^ 0x80000000u;   // g_a1 has no sign: the odd edges' inputs lose theirs
      const Quad3 B0 = flip3(get_slot(sz, 0, c, g), fu), B1 = flip3(get_slot(sz, 1, c, g), fu);
#pragma unroll
      for (int hb = 0; hb < 4; ++hb) mma3e(gwu[hb][0], gwu[hb][1], get_slot(sx + (hb >> 1) * kSlot, hb & 1, c, g), B0, B1);
      wave_sync();
    }
    if constexpr (EQ) {
      gr += shfl_xor(gr, 16);
      gr += shfl_xor(gr, 32);
      if (g == 0 && valid) {
        const float k2 = 2.0f * gr;
        *reinterpret_cast<f32x4*>(a.Gx + (ee - a.gbase) * 4) =
            f32x4{phi * gx0 + k2 * d.dx, phi * gx1 + k2 * d.dy, phi * gx2 + k2 * d.dz, gphi};
      }
    }
  }
  // the block's partial row, the waves added in wave order; with fbase > 0 on top of the earlier chunks'
  __syncthreads();
  float* const sum = (float*)s_x;   // [dW_hl | db2 | dW1_mov | dbx1 | dw2_mov | dW_e | dw_d]
  constexpr int oB2 = H * O, oM = oB2 + O, oBx = oM + (EQ ? O * M : 0), oW2 = oBx + (EQ ? M : 0), oE = oW2 + (EQ ? M : 0);
  const int FE = a.FE, LW = oE + H * FE + (EQ ? H : 0);   // at most 4,768 floats (EGNN, F_E = 24)
  static_assert((oE + H * 33) * sizeof(float) <= sizeof(s_x), "the partial row fits the exchange buffers");   // 32 slots and w_d
  for (int q = 0; q < kW; ++q) {
    if (w == q) {
      auto add = [&](int i, float v) { sum[i] = q ? sum[i] + v : v; };
      const float sgn = flip ? -1.0f : 1.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int row = 16 * i + 4 * g + r;
            add(row * O + 16 * j + c, sgn * gwh[i][j][r]);
            if (EQ && i < 2) add(oM + row * M + 16 * j + c, sgn * gwm[i < 2 ? i : 0][j][r]);
            if constexpr (U) {
              const int slot = 8 * (c >> 2) + 4 * j + (c & 3);
              if (slot < FE) add(oE + row * FE + slot, sgn * gwu[i][j][r]);
              else if (EQ && slot == FE) add(oE + H * FE + row, sgn * gwu[i][j][r]);
            }
          }
      if (!(c & 1)) {
        const int n = c >> 1, f = 16 * (n >> 2) + 4 * g + (n & 3);
        add(oB2 + f, sb2);
        if constexpr (EQ) {
          add(oBx + f, sbx);
          add(oW2 + f, sw2);
        }
      }
    }
    __syncthreads();
  }
  float* row = a.dwpart + (int64_t)blockIdx.x * a.LW;
  for (int q = threadIdx.x; q < LW; q += 64 * kW) row[q] = a.fbase > 0 ? row[q] + sum[q] : sum[q];
}

}  // namespace

bool f32_small_supported(const LayerShape& s) { return !s.bf16 && s.H == 64 && s.NUC <= 1; }

int launch_f32_small_fwd(const LayerShape& s, const FwdArgs& a, hipStream_t st) {
  if (a.ntiles <= 0) return 0;
  const dim3 grid((unsigned)std::min<int64_t>(cdiv(a.ntiles, kW), 256 * 3)), blk(64 * kW);   // three blocks per CU
  if (s.eq && s.FE > 0) hipLaunchKernelGGL((f32s_fwd_kernel<true, true>), grid, blk, 0, st, a);
  else if (s.eq) hipLaunchKernelGGL((f32s_fwd_kernel<true, false>), grid, blk, 0, st, a);
  else if (s.FE > 0) hipLaunchKernelGGL((f32s_fwd_kernel<false, true>), grid, blk, 0, st, a);
  else hipLaunchKernelGGL((f32s_fwd_kernel<false, false>), grid, blk, 0, st, a);
  return (int)hipGetLastError();
}

int f32_small_blocks(int64_t E) { return (int)std::max<int64_t>(1, std::min<int64_t>(cdiv(E, 16 * kW), 512)); }

int launch_f32_small_bwd(const LayerShape& s, const BwdArgs& a, hipStream_t st) {
  if (a.ntiles <= a.tile0) return 0;
  const dim3 grid(f32_small_blocks(std::min<int64_t>(a.ntiles * kTileEdges, a.E) - a.tile0 * kTileEdges)), blk(64 * kW);
  if (s.eq && s.FE > 0) hipLaunchKernelGGL((f32s_bwd_kernel<true, true>), grid, blk, 0, st, a);
  else if (s.eq) hipLaunchKernelGGL((f32s_bwd_kernel<true, false>), grid, blk, 0, st, a);
  else if (s.FE > 0) hipLaunchKernelGGL((f32s_bwd_kernel<false, true>), grid, blk, 0, st, a);
  else hipLaunchKernelGGL((f32s_bwd_kernel<false, false>), grid, blk, 0, st, a);
  return (int)hipGetLastError();
}

}  // namespace egnn
