// fp32 node products and split-K weight-gradient products on split bf16 operands (egnn_split.h).
//
// BM x 64 tile per block of four waves, 32-deep k slices: operand tiles are read in fp32 with 16-byte loads, split
// into three bf16 parts on the way to LDS and kept there in their global layout, so a k-contiguous tile gives an
// operand chunk in one 16-byte read and an m- or n-contiguous one in two transposing reads.  The products of a
// molecule batch are short (K = 128 or 256, tens to thousands of rows), so load latency bounds them: four slices
// are in flight in registers (a whole K of 128 at once) and LDS is double-buffered, one barrier per slice.
// The product is computed transposed, so a lane holds four consecutive columns of one row and every epilogue
// access is a 16-byte one.
// Measured against the fp32-instruction tiles it replaced, per launch: 27 x 256 -> 128 products 16.7 -> 7.1 us,
// 2,351 rows 20.9 -> 8.2 us, 19,623 rows 36 -> 23 us; [x | 1]^T dz over 2,351 rows 13.9 -> 11 us, over 19,623 rows
// 29 -> 21 us.
#include "egnn_device.h"
#include "egnn_internal.h"
#include "egnn_split.h"

namespace egnn {
namespace {

using namespace split;

constexpr int kBN = 64, kBK = 32, kRing = 4;

__device__ __forceinline__ int chain_pos4(int f) {   // chain position of features f .. f + 3 of a 32-group (f % 4 = 0)
  return f < 16 ? 2 * f : 2 * (f - 16) + 4;
}

// one operand's BR x 32 (rows x k) tile in LDS: [row][k], pitch 40 (KC), or [k][row], pitch BR + 16; each pitch
// spreads the 16 rows (the 8 k rows of 32 lanes) of one read over all banks
template <bool KC, int BR> struct Tile {
  static constexpr int pitch = KC ? kBK + 8 : BR + 16;
  static constexpr int plane = KC ? BR * pitch : kBK * pitch;
  static constexpr int nv = BR * kBK / 4 / 256;   // 16-byte vectors per thread and slice
  // (row, k) of vector i of the thread
  static __device__ __forceinline__ int row(int i) { const int x = threadIdx.x + 256 * i; return KC ? x / (kBK / 4) : 4 * (x % (BR / 4)); }
  static __device__ __forceinline__ int kk(int i) { const int x = threadIdx.x + 256 * i; return KC ? 4 * (x % (kBK / 4)) : x / (BR / 4); }
  static __device__ __forceinline__ void put(bf16* s, int i, const f32x4& v) {
    const Chunk3 p = split_chunk(v, v);   // the upper half is dead
    bf16* d = s + (KC ? row(i) * pitch + kk(i) : kk(i) * pitch + row(i));
    *reinterpret_cast<bf16x4*>(d) = __builtin_shufflevector(p.p0, p.p0, 0, 1, 2, 3);
    *reinterpret_cast<bf16x4*>(d + plane) = __builtin_shufflevector(p.p1, p.p1, 0, 1, 2, 3);
    *reinterpret_cast<bf16x4*>(d + 2 * plane) = __builtin_shufflevector(p.p2, p.p2, 0, 1, 2, 3);
  }
  static __device__ __forceinline__ bf16x8 get1(const bf16* s, int r0, int c, int g) {
    if constexpr (KC) {
      // k order of the transposing reads (4g .. 4g + 3, 16 + 4g ..): any order serves as long as both operands share it
      const bf16* p = s + (r0 + c) * pitch + 4 * g;
      return __builtin_shufflevector(*reinterpret_cast<const bf16x4*>(p), *reinterpret_cast<const bf16x4*>(p + 16), 0, 1, 2, 3, 4, 5, 6, 7);
    } else {
      const bf16* p = s + (4 * g + (c >> 2)) * pitch + r0 + 4 * (c & 3);
      const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)p);
      const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4*)(p + 16 * pitch));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    }
  }
  // k order 8g .. 8g + 7 (one read), when both operands are k-contiguous
  static __device__ __forceinline__ bf16x8 get1d(const bf16* s, int r0, int c, int g) { return load_chunk(s + (r0 + c) * pitch + 8 * g); }
  template <bool DIRECT>
  static __device__ __forceinline__ Chunk3 get(const bf16* s, int r0, int c, int g) {
    if constexpr (DIRECT) return Chunk3{get1d(s, r0, c, g), get1d(s + plane, r0, c, g), get1d(s + 2 * plane, r0, c, g)};
    else return Chunk3{get1(s, r0, c, g), get1(s + plane, r0, c, g), get1(s + 2 * plane, r0, c, g)};
  }
};

// FOLD: the last row of A is the ones row and lies past the last whole row tile; the blocks of the first row tile
// make it as the sum of the B values they load
template <bool A_KC, bool B_NC, int BM, bool FOLD>
__global__ __launch_bounds__(256, 2) void gemm_f32s_kernel(Gemm2Args g) {
  typedef Tile<A_KC, BM> TA;
  typedef Tile<!B_NC, kBN> TB;
  constexpr int MI = BM / 32, NJ = 2;   // the wave's 16 MI x 32 part of the tile
  constexpr bool DIRECT = A_KC && !B_NC;
  static_assert(!FOLD || (B_NC && !A_KC), "folded ones row: B by rows of k");
  __shared__ __attribute__((aligned(16))) bf16 s_a[2][3 * TA::plane];
  __shared__ __attribute__((aligned(16))) bf16 s_b[2][3 * TB::plane];
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, c = l & 15, gq = l >> 4;
  const int wm = w >> 1, wn = w & 1;
  const int64_t m0 = (int64_t)blockIdx.x * BM, n0 = (int64_t)blockIdx.y * kBN;
  const int64_t kbeg = g.ksplit > 0 ? (int64_t)blockIdx.z * g.ksplit : 0;
  const int64_t kend = g.ksplit > 0 && kbeg + g.ksplit < g.K ? kbeg + g.ksplit : g.K;
  const float* A = (const float*)g.A;
  const float* A2 = (const float*)g.A2;
  const float* B = (const float*)g.B;

  const uint32_t flip = g.partial ? (blockIdx.z & 1) << 31 : 0u;   // every other K range (flip_sign)
  const float sgn = flip ? -1.0f : 1.0f;
  const uint32_t odd = g.partial ? 0u : 1u << 31;   // without splits: every other row of A

  struct Regs { f32x4 a[TA::nv], b[TB::nv]; };
  auto load = [&](int64_t k0, Regs& r) {
    if (k0 >= kend) return;   // uniform
#pragma unroll
    for (int i = 0; i < TA::nv; ++i) {
      const int64_t m = m0 + TA::row(i), k = k0 + TA::kk(i);
      f32x4 v = zero4();
      if (m < g.M && k < kend) {
        if constexpr (A_KC) {   // A[m][k], columns from a_split of A2
          const float* p = (A2 && k >= g.a_split) ? A2 + m * g.lda2 - g.a_split + k : A + m * g.lda + k;
          if (m == g.a_ones_row) {
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = k + u < kend ? 1.0f : 0.0f;
          } else if (k + 4 <= kend) {
            v = load4_f32(p);
          } else {
            for (int u = 0; u < 4; ++u) if (k + u < kend) v[u] = p[u];
          }
        } else {                // A[k][m], rows from a_split of A2
          const float* p = (A2 && m >= g.a_split) ? A2 + k * g.lda2 - g.a_split + m : A + k * g.lda + m;
          if (m + 4 <= g.M && !(g.a_ones_row >= m && g.a_ones_row < m + 4)) {
            v = load4_f32(p);
          } else {
            for (int u = 0; u < 4; ++u) if (m + u < g.M) v[u] = m + u == g.a_ones_row ? 1.0f : p[u];
          }
        }
      }
      r.a[i] = v;
    }
#pragma unroll
    for (int i = 0; i < TB::nv; ++i) {
      const int64_t n = n0 + TB::row(i), k = k0 + TB::kk(i);
      f32x4 v = zero4();
      if (n < g.N && k < kend) {   // N % 4 == 0
        if constexpr (B_NC) {   // B[k][n], or B[b_kidx[k]][n]
          v = load4_f32(B + (g.b_kidx ? (int64_t)g.b_kidx[k] : k) * g.ldb + n);
        } else {                // B[n][k]
          const float* p = B + n * g.ldb + k;
          if (k + 4 <= kend) {
            v = load4_f32(p);
          } else {
            for (int u = 0; u < 4; ++u) if (k + u < kend) v[u] = p[u];
          }
        }
      }
      r.b[i] = v;
    }
  };
  f32x4 ones = zero4();
  f32x4 hi[MI][NJ], lo[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) hi[i][j] = lo[i][j] = zero4();
  Regs r[kRing];
#pragma unroll
  for (int u = 0; u < kRing; ++u) load(kbeg + u * kBK, r[u]);
  for (int64_t k0 = kbeg; k0 < kend; k0 += kRing * kBK) {
#pragma unroll
    for (int u = 0; u < kRing; ++u) {
      const int64_t k = k0 + u * kBK;
      if (k >= kend) break;   // uniform
      bf16* sa = s_a[u & 1];
      bf16* sb = s_b[u & 1];
#pragma unroll
      for (int i = 0; i < TA::nv; ++i) {
        f32x4 v = r[u].a[i];
        if constexpr (A_KC) {
          v = flip_sign(v, TA::row(i) & 1 ? odd : 0u);
        } else {   // rows 4 q .. 4 q + 3
          v[1] = bitsf(fbits(v[1]) ^ odd);
          v[3] = bitsf(fbits(v[3]) ^ odd);
        }
        TA::put(sa, i, v);
      }
#pragma unroll
      for (int i = 0; i < TB::nv; ++i) {
        TB::put(sb, i, flip_sign(r[u].b[i], flip));
        if constexpr (FOLD) ones += r[u].b[i];
      }
      load(k + kRing * kBK, r[u]);
      __syncthreads();
      Chunk3 b[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) b[j] = TB::template get<DIRECT>(sb, 32 * wn + 16 * j, c, gq);
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const Chunk3 a = TA::template get<DIRECT>(sa, 16 * MI * wm + 16 * i, c, gq);
#pragma unroll
        for (int j = 0; j < NJ; ++j) mma3(hi[i][j], lo[i][j], b[j], a);   // C rows: n, columns: m
      }
    }
  }
  // lane (c, gq): row m = c of its blocks, columns 4 gq .. + 3
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    const int64_t m = m0 + 16 * MI * wm + 16 * i + c;
    if (m >= g.M) continue;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int64_t n = n0 + 32 * wn + 16 * j + 4 * gq;
      if (n >= g.N) continue;
      f32x4 v = joined(hi[i][j], lo[i][j]);
      if (!g.partial && (c & 1)) v = -v;
      if (g.partial) {
        *reinterpret_cast<f32x4*>(g.partial + ((int64_t)blockIdx.z * g.M + m) * g.N + n) = sgn * v;
        continue;
      }
      if (g.bias) {
#pragma unroll
        for (int u = 0; u < 4; ++u) if (n + u < g.bias_len) v[u] += ((const float*)g.bias)[n + u];
      }
      if (g.zd) {   // * SiLU'(z)
        const f32x4 z = load4_f32((const float*)g.zd + m * g.ldz + n);
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] *= silu_yd_f32(z[u]).d;
      }
      if (g.act) {
        if (g.Cpre) *reinterpret_cast<f32x4*>((float*)g.Cpre + m * g.ldpre + n) = v;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = silu_f32(v[u]);
      }
      if (g.resid && n < g.resid_len) v += load4_f32((const float*)g.resid + m * g.ldr + n);   // resid_len % 4 == 0
      int64_t pn = n;
      if (g.perm_half > 0) {
        const int64_t f = n % g.perm_half;
        pn = n - f + (f & ~31) + chain_pos4((int)(f & 31));
      }
      *reinterpret_cast<f32x4*>((float*)g.C + m * g.ldc + pn) = v;
    }
  }
  if constexpr (FOLD) {
    if (blockIdx.x == 0) {   // the ones row (a split-K launch)
      __syncthreads();
      float* s = (float*)s_a;   // [16][64]
      *reinterpret_cast<f32x4*>(s + (tid >> 4) * kBN + 4 * (tid & 15)) = ones;
      __syncthreads();
      if (tid < kBN && n0 + tid < g.N) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < 16; ++k) v += s[k * kBN + tid];
        g.partial[((int64_t)blockIdx.z * g.M + g.M - 1) * g.N + n0 + tid] = v;
      }
    }
  }
}

template <int BM, bool FOLD>
void launch_bm(const Gemm2Args& g, dim3 grid, hipStream_t st) {
  if constexpr (FOLD) {
    hipLaunchKernelGGL((gemm_f32s_kernel<false, true, BM, true>), grid, dim3(256), 0, st, g);
  } else {
    if (g.a_kc && g.b_nc) hipLaunchKernelGGL((gemm_f32s_kernel<true, true, BM, false>), grid, dim3(256), 0, st, g);
    else if (g.a_kc) hipLaunchKernelGGL((gemm_f32s_kernel<true, false, BM, false>), grid, dim3(256), 0, st, g);
    else if (g.b_nc) hipLaunchKernelGGL((gemm_f32s_kernel<false, true, BM, false>), grid, dim3(256), 0, st, g);
    else hipLaunchKernelGGL((gemm_f32s_kernel<false, false, BM, false>), grid, dim3(256), 0, st, g);
  }
}

}  // namespace

// 16-byte rows of every operand, whole 4-column groups
bool gemm_f32s_ok(const Gemm2Args& g) {
  auto al = [](const void* p, int64_t ld) { return p == nullptr || ((((uintptr_t)p) & 15) == 0 && ld % 4 == 0); };
  return !g.a_bf16 && !g.b_bf16 && !g.a_silu && g.N % 4 == 0 && (!g.A2 || g.a_split % 4 == 0) && al(g.A, g.lda) &&
         al(g.A2, g.lda2) && al(g.B, g.ldb) &&
         (g.partial ? (((uintptr_t)g.partial) & 15) == 0
                    : !g.c_bf16 && !g.bias_bf16 && al(g.C, g.ldc) && al(g.Cpre, g.ldpre) && al(g.resid, g.ldr) &&
                          al(g.zd, g.ldz) && g.resid_len % 4 == 0 && (g.perm_half <= 0 || g.perm_half % 32 == 0));
}

int launch_gemm_f32s(const Gemm2Args& g, unsigned gz, hipStream_t st) {
  const unsigned gy = (unsigned)cdiv(g.N, kBN);
  if (g.partial && !g.a_kc && g.b_nc && g.a_ones_row == g.M - 1 && g.M > 1 && (g.M - 1) % 64 == 0) {
    launch_bm<64, true>(g, dim3((unsigned)((g.M - 1) / 64), gy, gz), st);
  } else {   // 32-row tiles at every size: three blocks per CU, at 19,623 rows 23 us against 26 us with 64-row tiles
    launch_bm<32, false>(g, dim3((unsigned)cdiv(g.M, 32), gy, gz), st);
  }
  return (int)hipGetLastError();
}

}  // namespace egnn
