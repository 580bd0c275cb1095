// fp32 edge kernels of the layer at H = O = M = 128 on split bf16 operands (egnn_split.h).
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
// 46k and 0.7k edges of 9..29-atom molecules): 564 -> 233, 99 -> 34 and 51 -> 16 us.  What bounds it now is the
// issue of the 768 products and about 2,400 vector instructions per wave and pass.
#include "egnn_device.h"
#include "egnn_internal.h"
#include "egnn_split.h"

namespace egnn {
namespace {

using namespace split;

constexpr int kF32Waves = 4;

__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }
__device__ __forceinline__ Chunk3 lds_chunk3(const bf16* frag, int l) {
  const bf16* p = frag + l * 8;
  return Chunk3{load_chunk(p), load_chunk(p + kFragElems), load_chunk(p + 2 * kFragElems)};
}
// one address per lane; of(r): lane r's, wave-uniform
struct RowAddr {
  uint32_t lo, hi;
  __device__ __forceinline__ explicit RowAddr(float* p) : lo((uint32_t)(uintptr_t)p), hi((uint32_t)((uintptr_t)p >> 32)) {}
  __device__ __forceinline__ float* of(int r) const {
    return (float*)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)hi, r) << 32) |
                    (uint32_t)__builtin_amdgcn_readlane((int)lo, r));
  }
};
// fragments of two row blocks
struct Pair3 { Chunk3 a, b; };
__device__ __forceinline__ Pair3 pair3(const bf16* a, const bf16* b, int l) { return Pair3{lds_chunk3(a, l), lds_chunk3(b, l)}; }
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

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
          const Chunk3 u3 = split_chunk(u.lo, u.hi);
#pragma unroll
          for (int rb = 0; rb < H / 16; ++rb) {
            const Chunk3 A = lds_chunk3((const bf16*)a.fr.s_u + ((int64_t)(rb >> 1) * 6 * a.NUC + ((rb & 1) * a.NUC + uc) * 3) * kFragElems, l);
            f32x4 lo = zero4(), hi = zero4();
            mma3(hi, lo, A, u3);
            y[rb >> 1][rb & 1] += hi + lo;
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
          for (int i = 0; i < 4; ++i) y[kc][b][i] = silu_f32(y[kc][b][i]);
        m1[kc] = split_chunk(y[kc][0], y[kc][1]);
      }
    }
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
          const f32x4 b2 = *reinterpret_cast<const f32x4*>(s_vec + 32 * kp + 16 * b + 4 * g);
#pragma unroll
          for (int i = 0; i < 4; ++i) x[b][i] = silu_f32(hi[b][i] + (lo[b][i] + b2[i]));
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
            q[rb] += lo3[0];
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
          acc += v[k];
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
        for (int i = 0; i < 4; ++i) phi += silu_f32(q[rb][i] + bx[i]) * w2[i];
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

}  // namespace egnn
