// Pipelined 16-bit MFMA GEMM tiles for the layer's products (the key product
// with relu² and adapter columns, model.py:262 / moe.py:140-144; the value
// product with the adapter K-extension, model.py:263 / moe.py:139-147; the
// full-expert layer's grouped products, moe.py:228-229, and its weight
// gradients).  out(M,N) = A(M,K) · B(N,K)ᵀ, both operands K-contiguous.
//
// Eight waves, WGM x WGN over a BM x BN tile, v_mfma_f32_16x16x32.  K is walked
// in slices of 64 elements: an LDS row is one whole 128-byte cache line, so a
// line is fetched once (with 64-byte rows L1 fetched every line twice).
//   * buffer_load ... lds writes A and B slices straight into two LDS rings, of
//     L + 1 and L slots.  Slice d = g + L is requested while slice g is
//     multiplied: its A rows in the first half of slice g, into the slot that
//     A of slice g - 1 left, its B rows in the second half, into the slot that
//     B of slice g has just left.  A has one slot more, so 256x256 keeps two
//     slices ahead in 160 KB.
//   * A slice is two halves of 32 k.  A wave multiplies one half from
//     registers while it reads the next half's fragments; only one barrier per
//     slice, between its halves, where every fragment of the slice has been
//     read and the next slice has to have landed.  The second half and the
//     next slice's first reads run behind it.
//   * Fragment reads and requests are dealt between the MFMAs over the first
//     three quarters of a half: requests in a burst stall the wave that issues
//     them.
//   * Workgroups are persistent and the slices run on across tiles: the next
//     tile's first L slices land under the present tile's last MFMAs and its
//     epilogue.  The epilogue stages a wave's own rows through the A slot of
//     the tile's last slice, in the part that this wave itself requests next,
//     so it has no barrier; its stores stay in flight through the next tile's
//     first slices (every store is issued, with rows past the end dropped by
//     the buffer's bound, so their number is known to the vmcnt waits).
//
// What bounds it: the operands' way from L2 and the infinity cache, then power.
// The 256x256 loop at 16384 x 8192 x 2048 bf16 runs at 1.25 PFLOP/s as it is,
// 1.4 with every request an L2 hit, 1.6 without requests (random data; 1.8 on
// zeros).  Measured against the 32x32x16 ring kernel and the VGPR-staged kernel
// that these products ran before (us, whole launches, the same box):
//   16384 x 8192 x 2048 bf16, relu²   538 -> 464     2031 x 3840 x 1024 bf16  34 -> 25
//   16384 x 2048 x 8704 bf16          497 -> 423     2031 x 1024 x 3840 bf16  33 -> 25
//   8192 x 1024 x 4608 fp16            89 -> 75      4096 x 3072 x 768 fp16   26.7 -> 25.7
//   8 groups, 8192 x 3072 x 768 fp16   68 -> 57      8 groups, 8192 x 768 x 3072  72 -> 55
// Four waves of 128x128 over the same tile were slower (587 us: one wave a
// SIMD hides nothing), two half-rings of waves in turns no faster.
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gemm_tile.h"
#include "internal.h"

namespace rwkvmoe {
namespace {

// 16-byte chunk swizzle of a 128-byte LDS row: depends on row % 16 only, so
// the fragments of every 16-row block sit at one address plus an immediate;
// the 16 rows of a fragment read hit distinct 16-byte bank groups (rows of
// one parity share a half of the 256-byte sweep).
RWKV_DEV int swz16(int row) { return (row & 7) ^ ((row >> 3) & 1); }

RWKV_DEV void buffer_load_lds16s(__amdgpu_buffer_rsrc_t r, lds_ptr_t dst, unsigned voff, unsigned soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, dst, 16, voff, soff, 0, 0);
}

template <int N>
RWKV_DEV void wait_vm_lds_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <typename T, int BM, int BN, int WGM, int WGN, int L, int EPI, int MODE, bool SPLIT>
__global__ __launch_bounds__(512) void pipe_kernel(GemmParams<T> p) {
  static_assert(sizeof(T) == 2 && WGM * WGN == 8 && L >= 2, "eight waves, 16-bit");
  static_assert(EPI == EPI_STORE || EPI == EPI_KEYAD, "epilogues: store (+ residual), key (+ adapter columns)");
  static_assert(!SPLIT || MODE == PIPE_DENSE, "split K is dense");
  typedef Mma16<T> M;
  typedef typename M::frag frag;
  constexpr int BK = 64, RB = 128;
  constexpr int WM = BM / WGM, WN = BN / WGN, MI = WM / 16, NI = WN / 16;
  static_assert(MI * 16 * WGM == BM && NI * 16 * WGN == BN, "wave tile");
  constexpr int DA = BM / 64, DB = BN / 64;  // 1 KB requests of a wave per slice
  static_assert(DA * 64 == BM && DB * 64 == BN, "requests");
  constexpr int UA = BM * RB, UB = BN * RB;
  constexpr int LDS_BYTES = (L + 1) * UA + L * UB;  // (pipe_lds_bytes)
  static_assert(LDS_BYTES <= 163840, "LDS budget");
  constexpr int NT = 512;
  static_assert(256 + loss_scratch_bytes(NT) <= LDS_BYTES, "loss scratch");
  static_assert(256 + kDispScratchInts * 4 <= LDS_BYTES, "dispatch scratch");
  // epilogue staging: RCH rows of RS bytes in a wave's DA KB
  constexpr int CP = 2 * NI;  // 16-byte chunks of a wave's output row
  constexpr bool PAD = (NI & (NI - 1)) != 0;
  constexpr int RS = NI * 32 + (PAD ? 16 : 0);
  constexpr int RCH = DA * 1024 >= 32 * RS && MI % 2 == 0 ? 32 : 16;
  static_assert(RCH * RS <= DA * 1024, "staging rows");
  constexpr int RND = MI * 16 / RCH, SPR = (RCH * CP + 63) / 64;
  constexpr int NST = SPLIT ? MI * NI : RND * SPR;  // stores of one epilogue
  constexpr int WV = (L - 2) * (DA + DB) + DA;      // requests after the slice that a barrier waits for
  static_assert(WV + NST < 64, "vmcnt range");

  __shared__ __attribute__((aligned(1024))) unsigned char lds[LDS_BYTES];
  unsigned char* const ldsB = lds + (L + 1) * UA;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  // ---- this workgroup's items (tiles, or K ranges of tiles) ----
  const int ks = SPLIT ? p.ksplit : 1;
  const int tiles_n = p.n / BN;
  int tiles_m = (p.m + BM - 1) / BM;
  // grouped modes: lane e keeps group e's range, and for row groups the
  // inclusive sum of its tile rows (at most 64 groups)
  int g_lo = 0, g_hi = 0, g_sum = 0;
  if constexpr (MODE != PIPE_DENSE) {
    const int* off = MODE == PIPE_GRP ? p.grp_off : p.gk_off;
    const int ng = MODE == PIPE_GRP ? p.grp_n : p.gk_n;
    g_lo = off[min(lane, ng)];
    g_hi = off[min(lane + 1, ng)];
    if constexpr (MODE == PIPE_GRP) {
      g_sum = (g_hi - g_lo + BM - 1) / BM;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(g_sum, d);
        if (lane >= d) g_sum += v;
      }
      tiles_m = __builtin_amdgcn_readlane(g_sum, 63);
    }
  }
  const int total = (MODE == PIPE_GK ? p.gk_n : 1) * tiles_m * tiles_n * ks;
  // XCD x = w % 8 takes a contiguous run of the items
  const int G = gridDim.x, w = blockIdx.x, xcd = w & 7;
  const int step = (G - xcd + 7) >> 3;  // workgroups on this XCD
  const int run = total / 8 + (xcd < total % 8 ? 1 : 0);
  const int base = xcd * (total / 8) + min(xcd, total % 8) + (w >> 3);
  const int count = (w >> 3) < run ? (run - (w >> 3) + step - 1) / step : 0;

  constexpr bool JOBS = EPI == EPI_KEYAD;  // only key products are given any
  int ticket = 1;
  // Row groups with fewer tiles than workgroups: the last one, then without a
  // tile, runs the loss reduction beside the others' tiles, and those take no
  // ticket (an atomic each on one address: 0.8 us of the 7.8 that the key
  // product of 64 tokens and 4 experts of 512 x 2048 fp16 took).
  if constexpr (JOBS && MODE == PIPE_GRP) {
    if (total < G) ticket = w == G - 1 ? 0 : 2;
  }
  auto take_ticket = [&]() {
    if constexpr (!JOBS) return;
    if constexpr (MODE == PIPE_GRP) {
      if (ticket != 1) return;
    }
    if (p.loss.losses != nullptr && tid == 0) ticket = atomicAdd(p.loss.claim, 1);
  };
  // after the last tile (LDS is free then): the router's loss reduction in
  // the workgroup that took the first ticket, and the dispatch scatter's blocks
  auto run_jobs = [&]() {
    if constexpr (!JOBS) return;
    if (p.loss.losses != nullptr) {
      __syncthreads();
      int* flag = (int*)lds;
      if (tid == 0) flag[0] = ticket;
      __syncthreads();
      const bool mine = flag[0] == 0;
      __syncthreads();
      if (mine) {
        double* sp = (double*)(lds + 256);
        long long* sc = (long long*)(sp + NT);
        reduce_losses(p.loss, sp, sc, (double*)(sc + NT));
      }
    }
    dispatch_job_run(p.disp, (int*)lds + 1, (int*)(lds + 256));
  };
  if (count == 0) {
    take_ticket();
    run_jobs();
    return;
  }

  const int nk1 = p.k1 / BK, nkt = nk1 + p.k2 / BK;
  const int GROUP_M = p.group_m > 0 ? p.group_m : 8;
  struct Item {
    int m0, n0, mlim, e;  // first row and column, end of the rows, group
    int s0, s1;           // K slices
  };
  auto item_of = [&](int i) -> Item {
    int l = base + i * step;
    Item it;
    it.e = 0;
    it.mlim = p.m;
    it.s0 = 0;
    it.s1 = nkt;
    if constexpr (SPLIT) {
      const int sp = l % ks;
      l /= ks;
      it.s0 = nkt * sp / ks;
      it.s1 = nkt * (sp + 1) / ks;
    }
    if constexpr (MODE == PIPE_GK) {
      it.e = l / (tiles_m * tiles_n);
      l -= it.e * (tiles_m * tiles_n);
      it.s0 = __builtin_amdgcn_readlane(g_lo, it.e) / BK;
      it.s1 = __builtin_amdgcn_readlane(g_hi, it.e) / BK;
    }
    const int in_group = GROUP_M * tiles_n;
    const int first_m = (l / in_group) * GROUP_M;
    const int gsize = min(tiles_m - first_m, GROUP_M);
    const int mt = first_m + (l % in_group) % gsize;
    it.n0 = ((l % in_group) / gsize) * BN;
    it.m0 = mt * BM;
    if constexpr (MODE == PIPE_GRP) {
      // the group whose tile rows hold mt
      it.e = __popcll(__ballot(g_sum <= mt));
      const int before = it.e > 0 ? __builtin_amdgcn_readlane(g_sum, it.e - 1) : 0;
      it.m0 = __builtin_amdgcn_readlane(g_lo, it.e) + (mt - before) * BM;
      it.mlim = __builtin_amdgcn_readlane(g_hi, it.e);
    }
    return it;
  };

  // ---- requests: the slice d of item d_i, K slice d_k of [.., d_lim) in one segment ----
  __amdgpu_buffer_rsrc_t ra, rb;
  unsigned va[DA], vb[DB];
  unsigned soff = 0;
  int d_i = 0, d_k = 0, d_lim = 0, d_end = 0;
  auto segment = [&](const Item& it, int k) {
    int sl = lane;  // (as in the epilogue)
    asm volatile("" : "+v"(sl));
    const bool ad = EPI == EPI_KEYAD && it.n0 >= p.n_key;
    const bool s2 = k >= nk1 && MODE != PIPE_GK;
    const int lda = s2 ? p.lda2 : p.lda1, ldb = s2 ? p.ldb2 : p.ldb1;
    const T* A = s2 ? p.a2 : (ad ? p.a_ad : p.a1);
    const T* B = s2 ? p.b2 : (ad ? p.b_ad : p.b1);
    const int nb = ad ? it.n0 - p.n_key : it.n0;
    if constexpr (MODE == PIPE_GRP) B += (size_t)it.e * p.grp_bstride;
    // (offsets within a tile's rows stay below 4 GB: plan_pipe)
    ra = buf_rsrc(A + (size_t)it.m0 * lda, 0xFFFFFFF0u);
    rb = buf_rsrc(B + (size_t)nb * ldb, 0xFFFFFFF0u);
#pragma unroll
    for (int i = 0; i < DA; ++i) {
      const int row = (wave * DA + i) * 8 + (sl >> 3);
      // rows past the end read the last one
      va[i] = ((unsigned)(min(it.m0 + row, it.mlim - 1) - it.m0) * (unsigned)lda + ((sl & 7) ^ swz16(row)) * 8) * 2;
    }
#pragma unroll
    for (int i = 0; i < DB; ++i) {
      const int row = (wave * DB + i) * 8 + (sl >> 3);
      vb[i] = ((unsigned)row * (unsigned)ldb + ((sl & 7) ^ swz16(row)) * 8) * 2;
    }
    soff = (unsigned)(s2 ? k - nk1 : k) * (BK * 2);
    d_k = k;
    d_end = it.s1;
    d_lim = (MODE == PIPE_GK || s2) ? it.s1 : min(it.s1, nk1);
  };
  auto advance = [&]() {
    ++d_k;
    soff += BK * 2;
    if (d_k == d_lim) {
      if (d_k < d_end) {
        segment(item_of(d_i), d_k);
      } else if (d_i + 1 < count) {
        ++d_i;
        const Item it = item_of(d_i);
        segment(it, it.s0);
      } else {  // past the last slice: request it again (into slots that nothing reads any more)
        --d_k;
        soff -= BK * 2;
      }
    }
  };
  auto request_a = [&](int slot, int i) {
    buffer_load_lds16s(ra, (lds_ptr_t)(lds + slot * UA + (wave * DA + i) * 1024), va[i], soff);
  };
  auto request_b = [&](int slot, int i) {
    buffer_load_lds16s(rb, (lds_ptr_t)(ldsB + slot * UB + (wave * DB + i) * 1024), vb[i], soff);
  };

  // ---- fragments ----
  const int fsw = swz16(lane & 15), fch = lane >> 4;
  const int ao = (wm * WM + (lane & 15)) * RB + ((fch ^ fsw) << 4);
  const int bo = (wn * WN + (lane & 15)) * RB + ((fch ^ fsw) << 4);
  frag fa[MI], fb[NI], ga[MI], gb[NI];
  // fragment q of half h: B's blocks, then A's
  auto read_frag = [&](frag (&xa)[MI], frag (&xb)[NI], const unsigned char* a, const unsigned char* b, int q) {
    if (q < NI) xb[q] = *(const frag*)(b + q * 16 * RB);
    else xa[q - NI] = *(const frag*)(a + (q - NI) * 16 * RB);
  };
  f32x4 acc[MI][NI];
  auto zero_acc = [&]() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  // One half: MFMAs on (xa, xb), the next half's fragments into (ya, yb), and
  // ND requests, dealt between the first three quarters of the MFMAs in this
  // order (the compiler would gather the requests behind the reads, whose LDS
  // it cannot tell apart).
  auto half = [&](const frag (&xa)[MI], const frag (&xb)[NI], frag (&ya)[MI], frag (&yb)[NI], int slot_a, int slot_b,
                  int h, auto nd, auto request) {
    constexpr int ND = decltype(nd)::value, NR = MI + NI, NOPS = NR + ND, NMF = MI * NI, X = NMF * 3 / 4;
    const unsigned char* a = lds + slot_a * UA + (ao ^ (h << 6));
    const unsigned char* b = ldsB + slot_b * UB + (bo ^ (h << 6));
#pragma unroll
    for (int q = 0; q <= NOPS; ++q) {
      const int lo = q * X / NOPS, hi = q < NOPS ? (q + 1) * X / NOPS : NMF;
#pragma unroll
      for (int m = 0; m < NMF; ++m)
        if (m >= lo && m < hi) acc[m / NI][m % NI] = M::run(xb[m % NI], xa[m / NI], acc[m / NI][m % NI]);
      if (q < NOPS) {
        __builtin_amdgcn_sched_barrier(0);
        const int d = q * ND / NOPS;
        if ((q + 1) * ND / NOPS > d) request(d);
        else read_frag(ya, yb, a, b, q - d);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // ---- epilogue of the item ci; sa: the A slot of its last slice ----
  // Each block is computed transposed (A operand = B rows): accumulator v of a
  // lane is column 4·(lane / 16) + v of row lane % 16.
  auto epilogue = [&](int ci, int sa) {
    // (opaque here, or the addresses below, which depend on the lane alone, are
    // computed ahead of the main loop and take its registers)
    int el = lane;
    asm volatile("" : "+v"(el));
    const Item it = item_of(ci);
    const int valid = it.mlim - it.m0;  // rows of the tile inside the range
    if constexpr (SPLIT) {
      const int sp = (base + ci * step) % ks;
      const __amdgpu_buffer_rsrc_t ro =
          buf_rsrc(p.part + ((size_t)sp * p.m + it.m0) * p.n + it.n0, (unsigned)min(valid, BM) * (unsigned)p.n * 4u);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const int row = wm * WM + i * 16 + (el & 15), col = wn * WN + j * 16 + (el >> 4) * 4;
          const unsigned off = row < valid ? ((unsigned)row * (unsigned)p.n + col) * 4u : kOOB;
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), ro, off, 0, 0);
        }
      return;
    }
    const bool ad = EPI == EPI_KEYAD && it.n0 >= p.n_key;
    const int ldo = ad ? p.n - p.n_key : p.ldo;
    T* ob = ad ? p.out_ad + (size_t)it.m0 * ldo + (it.n0 - p.n_key)
               : p.out + (MODE == PIPE_GK ? (size_t)it.e * p.gk_ostride : 0) + (size_t)it.m0 * ldo + it.n0;
    const unsigned obytes = (unsigned)min(valid, BM) * (unsigned)ldo * 2u;
    const __amdgpu_buffer_rsrc_t ro = buf_rsrc(ob, obytes);
    const bool res = EPI == EPI_STORE && p.resid != nullptr;
    const __amdgpu_buffer_rsrc_t rr = buf_rsrc(res ? p.resid + (size_t)it.m0 * ldo + it.n0 : p.resid, res ? obytes : 0u);
    unsigned char* st = lds + sa * UA + wave * (DA * 1024);
    // chunk c of staged row r
    auto at = [&](int r, int c) { return r * RS + ((PAD ? c : c ^ ((NI == 4 ? r : r >> 1) & (CP - 1))) << 4); };
#pragma unroll
    for (int rd = 0; rd < RND; ++rd) {
#pragma unroll
      for (int ii = 0; ii < RCH / 16; ++ii)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const f32x4 v = acc[rd * (RCH / 16) + ii][j];
          const int row = ii * 16 + (el & 15), col = j * 16 + (el >> 4) * 4;
          unsigned char* dst = st + at(row, col >> 3) + ((col & 4) << 1);
          if constexpr (EPI == EPI_KEYAD && std::is_same<T, f16>::value) {
            if (!ad) {
              *(unsigned long long*)dst = relu2_f16x4(v[0], v[1], v[2], v[3]);
              continue;
            }
          }
          float r[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) r[q] = rnd<T>(v[q]);
          if constexpr (EPI == EPI_KEYAD) {
            if (!ad) {
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const float z = r[q] > 0.f ? r[q] : 0.f;
                r[q] = z * z;  // relu(key(k)) ** 2 (model.py:262)
              }
            } else {
              const int gm = it.m0 + wm * WM + rd * RCH + row;
              adapter_scale4(p, min(gm, it.mlim - 1), it.n0 - p.n_key + wn * WN + col, r);
            }
          }
          union { T e[4]; unsigned long long u; } pk;
#pragma unroll
          for (int q = 0; q < 4; ++q) pk.e[q] = from_f<T>(r[q]);
          *(unsigned long long*)dst = pk.u;
        }
      u32x4 o[SPR];
      unsigned off[SPR];
#pragma unroll
      for (int s = 0; s < SPR; ++s) {
        const int id = s * 64 + el, row = id / CP, c = id % CP;
        const int tr = wm * WM + rd * RCH + row;
        const bool in = (RCH * CP) % 64 == 0 || id < RCH * CP;
        o[s] = *(const u32x4*)(st + at(in ? row : 0, c));
        off[s] = in && tr < valid ? ((unsigned)tr * (unsigned)ldo + wn * WN + c * 8) * 2u : kOOB;
      }
      if (res) {
        Chunk<T> x[SPR];
#pragma unroll
        for (int s = 0; s < SPR; ++s) x[s].raw = buf_load16(rr, off[s]);
#pragma unroll
        for (int s = 0; s < SPR; ++s) {
          Chunk<T> y;
          y.raw = o[s];
#pragma unroll
          for (int e = 0; e < 8; ++e) y.e[e] = from_f<T>(to_f(x[s].e[e]) + to_f(y.e[e]));
          o[s] = y.raw;
        }
      }
#pragma unroll
      for (int s = 0; s < SPR; ++s) __builtin_amdgcn_raw_buffer_store_b128(o[s], ro, off[s], 0, 0);
    }
  };

  // ---- main loop ----
  {
    const Item it = item_of(0);
    segment(it, it.s0);
  }
#pragma unroll
  for (int s = 0; s < L; ++s) {
#pragma unroll
    for (int i = 0; i < DA; ++i) request_a(s, i);
#pragma unroll
    for (int i = 0; i < DB; ++i) request_b(s, i);
    if (s + 1 < L) advance();
  }
  zero_acc();
  wait_scalar_loads();
  wait_vm_barrier<(L - 1) * (DA + DB)>();
#pragma unroll
  for (int q = 0; q < MI + NI; ++q) read_frag(fa, fb, lds + ao, ldsB + bo, q);
  int sa = 0, sb = 0, ci = 0, kk = 0;
  int nk;
  {
    const Item it = item_of(0);
    nk = it.s1 - it.s0;
  }
  // slices of this item whose successors were requested before the last
  // epilogue's stores, which may then still be in flight
  int loose = 0;
  for (;;) {
    advance();
    const int na = sa == L ? 0 : sa + 1, nb = sb == L - 1 ? 0 : sb + 1;
    const int fr = sa == 0 ? L : sa - 1;  // the slot A of the previous slice left
    half(fa, fb, ga, gb, sa, sb, 1, std::integral_constant<int, DA>{}, [&](int i) { request_a(fr, i); });
    __builtin_amdgcn_sched_barrier(0);
    if (loose > 0) {
      --loose;
      wait_vm_lds_barrier<WV + NST>();
    } else {
      wait_vm_lds_barrier<WV>();
    }
    __builtin_amdgcn_sched_barrier(0);
    half(ga, gb, fa, fb, na, nb, 0, std::integral_constant<int, DB>{}, [&](int i) { request_b(sb, i); });
    __builtin_amdgcn_sched_barrier(0);
    if (++kk == nk) {
      const bool last = ci + 1 == count;
      if (last) take_ticket();
      epilogue(ci, sa);
      if (last) break;
      ++ci;
      zero_acc();
      kk = 0;
      // read again what the half above has read: the epilogue needs the registers
#pragma unroll
      for (int q = 0; q < MI + NI; ++q) read_frag(fa, fb, lds + na * UA + ao, ldsB + nb * UB + bo, q);
      if constexpr (SPLIT || MODE == PIPE_GK) {
        const Item it = item_of(ci);
        nk = it.s1 - it.s0;
      }
      loose = nk >= L ? L - 1 : 0;
    }
    sa = na;
    sb = nb;
  }
  // the trailing requests land before the workgroup's LDS is used again
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  run_jobs();
}

template <typename T, int CFG, int WGM, int WGN, int EPI, int MODE, bool SPLIT = false>
hipError_t run_pipe(const GemmParams<T>& p, hipStream_t s) {
  constexpr int BM = kPipeTiles[CFG].bm, BN = kPipeTiles[CFG].bn, L = kPipeTiles[CFG].depth;
  if (EPI != EPI_KEYAD && (p.loss.losses || p.disp.nblk > 0)) return hipErrorInvalidValue;
  if (p.k1 % 64 || p.k2 % 64 || p.n % BN || (EPI == EPI_KEYAD && p.n_key % BN)) return hipErrorInvalidValue;
  if (MODE == PIPE_GRP && (!p.grp_off || p.grp_n < 1 || p.grp_n > 64)) return hipErrorInvalidValue;
  if (MODE == PIPE_GK && (!p.gk_off || p.gk_n < 1 || p.gk_n > 64)) return hipErrorInvalidValue;
  const int ks = SPLIT ? p.ksplit : 1;
  if (SPLIT && (ks < 2 || !p.part || (p.k1 + p.k2) / 64 < ks)) return hipErrorInvalidValue;
  const int tiles = (MODE == PIPE_GK ? p.gk_n : 1) * ((p.m + BM - 1) / BM + (MODE == PIPE_GRP ? p.grp_n : 0)) *
                    (p.n / BN) * ks;
  if (tiles == 0) return hipSuccess;
  constexpr int per_cu = kPipeTiles[CFG].per_cu;
  GemmParams<T> q = p;
  q.group_m = walk_group_m((p.m + BM - 1) / BM, p.n / BN, BM, BN);
  launch_kernel((pipe_kernel<T, BM, BN, WGM, WGN, L, EPI, MODE, SPLIT>), dim3(std::min(tiles, num_cus() * per_cu)),
                dim3(512), 0, s, q);
  return hipGetLastError();
}

// Tile `cfg` of kPipeTiles.
template <typename T, int EPI, int MODE>
hipError_t run_pipe_cfg(const GemmParams<T>& p, int cfg, hipStream_t s) {
  if constexpr (MODE == PIPE_DENSE) {
    if (p.ksplit > 1) {
      switch (cfg) {
        case 4: return run_pipe<T, 4, 2, 4, EPI, MODE, true>(p, s);
        case 6: return run_pipe<T, 6, 4, 2, EPI, MODE, true>(p, s);
        case 7: return run_pipe<T, 7, 4, 2, EPI, MODE, true>(p, s);
      }
      return hipErrorInvalidValue;
    }
  }
  switch (cfg) {
    case 0: return run_pipe<T, 0, 2, 4, EPI, MODE>(p, s);
    case 1: return run_pipe<T, 1, 2, 4, EPI, MODE>(p, s);
    case 2: return run_pipe<T, 2, 4, 2, EPI, MODE>(p, s);
    case 3: return run_pipe<T, 3, 2, 4, EPI, MODE>(p, s);
    case 4: return run_pipe<T, 4, 2, 4, EPI, MODE>(p, s);
    case 5: return run_pipe<T, 5, 2, 4, EPI, MODE>(p, s);
    case 6: return run_pipe<T, 6, 4, 2, EPI, MODE>(p, s);
    case 7: return run_pipe<T, 7, 4, 2, EPI, MODE>(p, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

template <typename T>
hipError_t pipe_run(const GemmParams<T>& p, int cfg, int epi, int mode, hipStream_t s) {
  switch (mode) {
    case PIPE_DENSE:
      return epi == EPI_KEYAD ? run_pipe_cfg<T, EPI_KEYAD, PIPE_DENSE>(p, cfg, s)
                              : run_pipe_cfg<T, EPI_STORE, PIPE_DENSE>(p, cfg, s);
    case PIPE_GRP:
      return epi == EPI_KEYAD ? run_pipe_cfg<T, EPI_KEYAD, PIPE_GRP>(p, cfg, s)
                              : run_pipe_cfg<T, EPI_STORE, PIPE_GRP>(p, cfg, s);
    case PIPE_GK:
      return epi == EPI_STORE ? run_pipe_cfg<T, EPI_STORE, PIPE_GK>(p, cfg, s) : hipErrorInvalidValue;
  }
  return hipErrorInvalidValue;
}

}  // namespace rwkvmoe
