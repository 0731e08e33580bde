// fp32 products of the backward on operands as they are stored: the VJP of an
// fp32 layer (and of the fp16 layer with fp32 adapters, which runs it on x in
// fp32) and the orthogonality loss's gradient (moe.py:129-163).
//
//   first   S = x·A_e and G = dO·B_eᵀ for every expert (N x kx each), and the
//           selection counts f_e
//   last    dA_e = xᵀ·DSd_e, dB = SGdᵀ·dO, dW_gate = dℓᵀ·x,
//           dx = DSd·A_eᵀ + dℓ·W_gate
//   ortho   Gm = 2·d·(A_allᵀ·A_all) off the diagonal r x r blocks (fp32),
//           then dA = A_all·Gm
//
// These are 0.2-3 GFLOP each, too small for tiles that share operands through
// LDS: 128x64 tiles left S and G of 1024 tokens on 32 CUs (31 us each), and the
// transposes, paddings, split-K reductions and scatters around them took as
// long again.  Here a lane reads its own MFMA operand (v_mfma_f32_32x32x2f32:
// row or column l % 32, 8 k values from (l / 32)·8 of every 16) from wherever
// it lies: rows with k contiguous as two 16-byte loads, rows with k strided
// (tokens, adapters' (E, C, r)) as 8 loads that the wave's 32 lanes coalesce.
// Three chunks of 16 k are in flight ahead of the MFMAs.  The products of one
// stage share a launch, with their outputs written where the caller wants
// them: 4 launches where there were 11.  A workgroup is a 32x32 tile whose 4 or
// 16 waves split K (their sums added in wave order) or, where 64x64 tiles fill
// the chip twice, a 64x64 tile of four whole waves.
// The fine-tune layer's VJP (1024 tokens, D=768, E=8, r=32): 138 -> 69 us; its
// orthogonality gradient in 2 launches of 11 us where there were 6.
#include <algorithm>

#include "bwd.h"
#include "common.h"
#include "internal.h"

namespace rwkvmoe {
namespace {

// Where an operand's element (i, k) lies (i: the row or column a lane holds):
//   ROWK  p[i·ld + k]        KROW  p[k·ld + i]
//   ADA   lora_A (E,C,r), i an adapter column e·r + j, k a channel
//   ADK   lora_A, i a channel, k an adapter column
enum { ROWK = 0, KROW = 1, ADA = 2, ADK = 3 };
// Where output (m, n) goes: rows of ldo (columns past nv zero); dA (E,C,r) with
// m a channel and n an adapter column; Gm's masked, scaled Gram matrix.
enum { OUT_ROW = 0, OUT_DA = 1, OUT_GRAM = 2 };

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

struct SgProd {
  const void* a; long long lda;  // operand of the output's rows
  const void* b; long long ldb;  // operand of its columns
  int K;
  const float* a2; long long lda2;  // second segment (dx): ROWK, KROW
  const float* b2; long long ldb2;
  int K2;
  int M, N, nv;
  void* out; long long ldo;
  int tiles_n, tiles;  // tiles of the product (0: skipped)
};

struct SgArgs {
  SgProd p[4];
  int C, r;
  float inv_r;
  const float* d;  // OUT_GRAM's factor (null: 1)
  const int* inds; int nk, E; int* cnt;  // the selection counts (null: none)
};

// One lane's operand: 8 values of k from k0 on.
template <typename T, int MODE>
struct Lane {
  const T* q;
  long long ld;
  int r;
  float inv_r;
  RWKV_DEV Lane(const void* p, long long ld_, int i, const SgArgs& a) : ld(ld_), r(a.r), inv_r(a.inv_r) {
    const T* t = (const T*)p;
    if constexpr (MODE == ROWK) q = t + (size_t)i * ld;
    else if constexpr (MODE == KROW) q = t + i;
    else if constexpr (MODE == ADA) q = t + (size_t)(i / r) * a.C * r + i % r;
    else {
      q = t + (size_t)i * r;
      ld = (long long)a.C * r;
    }
  }
  RWKV_DEV void load(int k0, int K, float (&v)[8]) const {
    if constexpr (MODE == ROWK) {
      // (rows are padded to whole chunks)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const f32x4u f = *(const f32x4u*)(q + k0 + 4 * c);
#pragma unroll
        for (int u = 0; u < 4; ++u) v[4 * c + u] = f[u];
      }
    } else if (MODE == ADK && sizeof(T) == 4 && r % 8 == 0) {
      // 8 columns from a multiple of 8 lie in one expert, contiguous (K = E·r
      // here: a multiple of 8, so only whole groups are past the end)
      const int k = min(k0, K - 8), e = (int)(((float)k + 0.5f) * inv_r);
      const T* t = q + (size_t)e * ld + (k - e * r);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const f32x4u f = *(const f32x4u*)(t + 4 * c);
#pragma unroll
        for (int u = 0; u < 4; ++u) v[4 * c + u] = f[u];
      }
    } else {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int k = min(k0 + u, K - 1);
        if constexpr (MODE == KROW) v[u] = to_f(q[(size_t)k * ld]);
        else if constexpr (MODE == ADA) v[u] = to_f(q[(size_t)k * r]);
        else {
          const int e = (int)(((float)k + 0.5f) * inv_r);  // k / r (k < 2^11)
          v[u] = to_f(q[(size_t)e * ld + (k - e * r)]);
        }
      }
    }
  }
};

// acc += the product's chunks c0, c0 + step, ... of 16 k.
template <typename LA, typename LB>
RWKV_DEV void accumulate(const LA& la, const LB& lb, int K, int c0, int step, int h, f32x16& acc) {
  constexpr int D = 4;  // chunks in registers
  const int nc = (K + 15) / 16;
  float av[D][8], bv[D][8];
  auto fetch = [&](int s, int c) {
    const int k0 = min(c, nc - 1) * 16 + h * 8;
    la.load(k0, K, av[s]);
    lb.load(k0, K, bv[s]);
  };
#pragma unroll
  for (int s = 0; s < D - 1; ++s) fetch(s, c0 + s * step);
  for (int c = c0; c < nc; c += D * step) {
#pragma unroll
    for (int s = 0; s < D; ++s) {
      const int cc = c + s * step;
      fetch((s + D - 1) % D, cc + (D - 1) * step);
      if (cc < nc) {
        if (cc * 16 + 16 > K) {
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (cc * 16 + h * 8 + u >= K) av[s][u] = bv[s][u] = 0.f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = Mma32<float>::run(bv[s][u], av[s][u], acc);
      }
    }
  }
}

template <typename TA, int MA, typename TB, int MB, int OUT, bool SEG2, int TILE, int KS, typename TO>
RWKV_DEV void product(const SgArgs& g, const SgProd& p, int tile, float* red) {
  constexpr int SUB = (TILE / 32) * (TILE / 32);  // 32x32 blocks of the tile; wave w: block w % SUB, K group w / SUB
  constexpr bool KSPLIT = KS > 1;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5;
  const int sub = wave % SUB, kg = wave / SUB;
  const int tm = tile / p.tiles_n, tn = tile - tm * p.tiles_n;
  const int m0 = tm * TILE + (sub & 1) * 32, n0 = tn * TILE + (sub >> 1) * 32;
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.f;
  const int m = m0 + (lane & 31), nl = n0 + (lane & 31);
  if (m0 < p.M && n0 < p.N) {
    const int mi = min(m, p.M - 1), ni = min(nl, p.nv - 1);
    accumulate(Lane<TA, MA>(p.a, p.lda, mi, g), Lane<TB, MB>(p.b, p.ldb, ni, g), p.K, kg, KS, h, acc);
    if constexpr (SEG2)
      accumulate(Lane<float, ROWK>(p.a2, p.lda2, mi, g), Lane<float, KROW>(p.b2, p.ldb2, ni, g), p.K2, kg, KS, h, acc);
  }
  if constexpr (KSPLIT) {
    f32x4* r4 = (f32x4*)red;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      r4[(wave * 4 + q) * 64 + lane] = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    __syncthreads();
    if (kg >= 4) return;
  }
  const float d = OUT == OUT_GRAM ? 2.f * (g.d ? g.d[0] : 1.f) : 1.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (KSPLIT && q != kg) continue;
    f32x4 v;
    if constexpr (KSPLIT) {
      // K group q < 4 adds accumulators 4q..4q+3 of the block's KS waves, in order
      const f32x4* r4 = (const f32x4*)red;
      v = r4[(sub * 4 + q) * 64 + lane];
#pragma unroll
      for (int w = 1; w < KS; ++w) {
        const f32x4 o = r4[((w * SUB + sub) * 4 + q) * 64 + lane];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] += o[u];
      }
    } else {
      v = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    }
    const int n = n0 + acc_row(4 * q, lane);
    if (m >= p.M) continue;
    TO* out = (TO*)p.out;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int c = n + u;
      if (c >= p.N) break;
      if constexpr (OUT == OUT_ROW) out[(size_t)m * p.ldo + c] = from_f<TO>(c < p.nv ? v[u] : 0.f);
      else if constexpr (OUT == OUT_DA) out[((size_t)(c / g.r) * g.C + m) * g.r + c % g.r] = from_f<TO>(v[u]);
      else out[(size_t)m * p.ldo + c] = from_f<TO>(m / g.r != c / g.r ? d * v[u] : 0.f);
    }
  }
}

enum { SG_FIRST = 0, SG_DX = 1, SG_DW = 2, SG_GRAM = 3, SG_ORTHO = 4 };

template <typename T, int SET, int TILE, int KS>
__global__ __launch_bounds__(64 * KS * (TILE / 32) * (TILE / 32)) void bwd_f32_kernel(SgArgs g) {
  __shared__ __attribute__((aligned(16))) float red[KS > 1 ? KS * (TILE / 32) * (TILE / 32) * 16 * 64 : 64];
  int b = blockIdx.x;
  if constexpr (SET == SG_FIRST) {
    if (b == 0) {  // (dispatched first: it overlaps the rest)
      count_selections(g.inds, g.nk, g.E, (int*)red, g.cnt);
      return;
    }
    --b;
    if (b < g.p[0].tiles) product<float, ROWK, float, ADA, OUT_ROW, false, TILE, KS, float>(g, g.p[0], b, red);
    else product<float, ROWK, float, ROWK, OUT_ROW, false, TILE, KS, float>(g, g.p[1], b - g.p[0].tiles, red);
  } else if constexpr (SET == SG_DX) {
    product<float, ROWK, float, ADK, OUT_ROW, true, TILE, KS, float>(g, g.p[0], b, red);
  } else if constexpr (SET == SG_DW) {
    if (b < g.p[0].tiles) {
      product<float, KROW, float, KROW, OUT_DA, false, TILE, KS, float>(g, g.p[0], b, red);
      return;
    }
    b -= g.p[0].tiles;
    // dB and dW_gate: one form
    const int q = b < g.p[1].tiles ? 1 : 2;
    product<float, KROW, float, KROW, OUT_ROW, false, TILE, KS, float>(g, g.p[q], q == 1 ? b : b - g.p[1].tiles, red);
  } else if constexpr (SET == SG_GRAM) {
    product<T, ADA, T, ADA, OUT_GRAM, false, TILE, KS, float>(g, g.p[0], b, red);
  } else {
    product<T, ADK, float, ROWK, OUT_DA, false, TILE, KS, T>(g, g.p[0], b, red);
  }
}

template <typename T, int SET>
hipError_t run_set(SgArgs& g, int np, int extra, hipStream_t s) {
  auto tiles = [&](int t) {
    long long n = 0;
    for (int i = 0; i < np; ++i) n += (long long)((g.p[i].M + t - 1) / t) * ((g.p[i].N + t - 1) / t);
    return n;
  };
  // 64x64 tiles where they fill the chip twice; else 32x32 tiles, their K over
  // four waves, or over sixteen where there are too few to fill it and K is
  // long (K = 256 and 768: 11 us on four, 13-15 on sixteen; K = 1024: 33 and
  // 26).  Products that are not asked for count too: the sums' order is the
  // same without them.
  const int cus = num_cus();
  int kmax = 0;
  for (int i = 0; i < np; ++i) kmax = std::max(kmax, g.p[i].K);
  const int t = tiles(64) >= 2LL * cus ? 64 : 32;
  const int ks = t == 64 ? 1 : kmax < 1024 || tiles(32) >= 2LL * cus ? 4 : 16;
  long long total = extra;
  for (int i = 0; i < np; ++i) {
    SgProd& p = g.p[i];
    p.tiles_n = (p.N + t - 1) / t;
    p.tiles = p.out ? (p.M + t - 1) / t * p.tiles_n : 0;
    total += p.tiles;
  }
  if (total == extra && !extra) return hipSuccess;
  if (total >= (1ll << 31)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)total);
  if (ks == 1) launch_kernel((bwd_f32_kernel<T, SET, 64, 1>), grid, dim3(256), 0, s, g);
  else if (ks == 4) launch_kernel((bwd_f32_kernel<T, SET, 32, 4>), grid, dim3(256), 0, s, g);
  else launch_kernel((bwd_f32_kernel<T, SET, 32, 16>), grid, dim3(1024), 0, s, g);
  return hipGetLastError();
}

SgArgs blank_args(int E, int C, int r) {
  SgArgs g;
  __builtin_memset(&g, 0, sizeof(g));
  g.C = C;
  g.r = r;
  g.inv_r = 1.f / (float)r;
  g.E = E;
  return g;
}

SgProd prod(const void* a, long long lda, const void* b, long long ldb, int K, int M, int N, int nv, void* out,
            long long ldo) {
  SgProd p;
  __builtin_memset(&p, 0, sizeof(p));
  p.a = a; p.lda = lda; p.b = b; p.ldb = ldb; p.K = K;
  p.M = M; p.N = N; p.nv = nv; p.out = out; p.ldo = ldo;
  return p;
}

}  // namespace

// Where these products are ahead of the LDS-tiled ones with their layouts and
// transposes (whole VJP, us, against those): N·E·r·C up to about 0.8 G, where
// launches and half-empty grids count.  1024 tokens, C=768, E·r=256: 75 against
// 138; 4096, 768, 128: 108 / 156; 64, 768, 128: 42 / 103; 8192, 768, 128: 190 /
// 217; 4096, 1024, 256: 223 / 224; past that operands shared through LDS win:
// 3000, 768, 512: 262 / 229; 8192, 1024, 512: 723 / 551.
bool bwd_f32_direct(int dtype, int N, int C, int E, int r) {
  return dtype == 0 && (long long)N * E * r * C <= 3ll << 28;
}

// (fp32 MFMA runs at an eighth of the 16-bit rate: the two launches stay ahead
// of the 16-bit products' six up to about 2^29 multiply-adds each)
bool ortho_backward_direct(int dtype, int E, int C, int r) {
  return dtype == 0 || (long long)E * r * E * r * C <= 1ll << 29;
}

hipError_t launch_bwd_f32_first(const float* x, const float* dO, const float* A, const float* B, const int* inds, int N,
                                int C, int E, int k, int r, int kx, float* S, float* G, int* cnt, hipStream_t s) {
  SgArgs g = blank_args(E, C, r);
  const int er = E * r;
  g.inds = inds; g.nk = N * k; g.cnt = cnt;
  g.p[0] = prod(x, C, A, 0, C, N, kx, er, S, kx);
  g.p[1] = prod(dO, C, B, C, C, N, kx, er, G, kx);
  return mark(run_set<float, SG_FIRST>(g, 2, 1, s), "bwd_f32_first", s);
}

hipError_t launch_bwd_f32_last(const float* x, const float* dO, const float* A, const float* wg, const float* dsd,
                               const float* sgd, const float* dl, int N, int C, int E, int r, int kx, int ep, float* dx,
                               float* dA, float* dB, float* dwg, hipStream_t s) {
  const int er = E * r;
  SgArgs g = blank_args(E, C, r);
  g.p[0] = prod(x, C, dsd, kx, N, C, er, er, dA, 0);
  g.p[1] = prod(sgd, kx, dO, C, N, er, C, C, dB, C);
  g.p[2] = prod(dl, ep, x, C, N, E, C, C, dwg, C);
  const hipError_t e = mark(run_set<float, SG_DW>(g, 3, 0, s), "bwd_f32_dw", s);
  if (e != hipSuccess || !dx) return e;
  g.p[0] = prod(dsd, kx, A, 0, er, N, C, C, dx, C);
  g.p[0].a2 = dl; g.p[0].lda2 = ep; g.p[0].b2 = wg; g.p[0].ldb2 = C; g.p[0].K2 = E;
  return mark(run_set<float, SG_DX>(g, 1, 0, s), "bwd_f32_dx", s);
}

size_t ortho_gram_bytes(int E, int r) {
  const size_t ld = (size_t)(E * r + 15) / 16 * 16;
  return (size_t)E * r * ld * sizeof(float);
}

hipError_t launch_ortho_backward(int dtype, const void* A, int E, int C, int r, const float* d_ortho, float* gram,
                                 void* dA, hipStream_t s) {
  const int er = E * r, ld = (er + 15) / 16 * 16;
  RWKV_DISPATCH_DTYPE(dtype, T, {
    SgArgs g = blank_args(E, C, r);
    g.d = d_ortho;
    g.p[0] = prod(A, 0, A, 0, C, er, er, er, gram, ld);
    hipError_t e = mark(run_set<T, SG_GRAM>(g, 1, 0, s), "ortho_gram", s);
    if (e != hipSuccess) return e;
    g.p[0] = prod(A, 0, gram, ld, er, C, er, er, dA, 0);
    return mark(run_set<T, SG_ORTHO>(g, 1, 0, s), "ortho_da", s);
  });
  return hipErrorInvalidValue;
}

}  // namespace rwkvmoe
