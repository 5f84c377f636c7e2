// Batched matrix products on CDNA4 MFMA for the Newton-Schulz / Polar Express
// iteration.
//
//  * SYRK mode ("NT": C(i, j) = alpha * sum_k A(i, k) A(j, k) + beta * Cin(i, j), both
//    operands K-contiguous rows, upper-triangle tiles only, mirrored store): the Gram
//    products X X^T and A A (A symmetric) of pe_loop_triton / ns_loop_triton
//    (polar_express.py:98-104, newton_schulz.py:105-112; Triton gram_nd,
//    gram.py:21-106). The polynomial combination B = b*A + c*A^2 rides in the
//    epilogue (beta*Cin with Cin = A).
//  * GEMM mode ("NN": C(i, j) = alpha * sum_k B(i, k) X(k, j) + beta * X(i, j)):
//    X' = a*X + B X (polar_express.py:109-110) with X in its own row-major layout
//    as the second operand; the epilogue writes X' row-major (into the other of two
//    ping-pong buffers) or, for the last iteration of a tall matrix, transposed.
//
// Operands live in workspaces whose extents are padded to the tile size and whose
// padding is rewritten as zeros by every producer, so the K loop and the stores
// need no masking (only the standalone gram_ path uses the masked variant). The one
// exception is the last 128 rows and columns of a SYRK output whose valid extent
// leaves them empty (packed tiles, below): what reads them lands only in output rows
// that are masked to zeros or not stored.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "common.h"

namespace {

enum { MODE_GEMM = 0, MODE_SYRK = 1 };

struct GemmArgs {
  const void* a;   // operand rows i, K contiguous
  const void* b;   // operand rows j, K contiguous
  const void* cin; // beta source, element (i, j) at cin[i * ldc + j]
  void* out;       // (i, j) at out[i * ldo + j]
  void* out_t;     // optional: (j, i) at out_t[j * ldt + i]
  int64_t lda, ldb, ldc, ldo, ldt;
  int64_t sa, sb, sc, so, st;  // batch strides in elements
  int64_t K;                   // multiple of BK (padded)
  int64_t Mv, Nv;              // valid extents; outside them zeros are stored
  int64_t Mt, Nt, Kt;          // masked variant only: true row counts of a / b and K
  float alpha, beta;
  const float* scale;          // per-batch prescale s (nullable)
  int scale_mode;              // 1: alpha *= s, beta *= s;  2: alpha *= s * s
  int tiles_m, tiles_n, tiles_per_batch;
  int tiles_total;             // tiles_per_batch * batch
  int store_out, store_out_t;
  int t0, nb;                  // tile_bx_kernel's apply: first tensor in the table, matrices per tensor
};

// One launch over the products of several buckets (GROUP_MAX at most): group i owns the tiles
// tile0[i] .. tile0[i + 1] - 1 of the launch. The buckets of a model share one side (its
// width), so their launches of one kind do the same work on different matrices, and each
// alone may leave most CUs idle.
constexpr int GROUP_MAX = 8;
struct GemmTab {
  int n;
  int tile0[GROUP_MAX + 1];
  GemmArgs g[GROUP_MAX];
};

// Workgroup L of a one-tile-per-workgroup launch of `total` -> tile index. Dispatch
// hands consecutive workgroups to the 8 XCDs round-robin (L on XCD L % 8). When a matrix
// has at least XCD_STRIPE tiles, XCD x takes stripes x, x + 8, x + 16, ... of XCD_STRIPE
// consecutive tiles while whole rounds of 8 stripes remain, so all XCDs work on the same
// matrices at a time (the operand panels their L2s miss on then come from one matrix's
// worth of data, which the Infinity Cache holds: X X^T on the 4096 x 14336 bucket 5%
// faster than contiguous ranges); the rest, or every tile of launches of smaller
// matrices, is dealt as one contiguous range per XCD, so each XCD works through
// neighbouring tiles with its own L2.
constexpr int XCD_STRIPE = 64;
MUON_DEVICE int64_t xcd_tile(int64_t L, int64_t total, int tiles_per_batch) {
  const int64_t x = L & 7, i = L >> 3;
  const int64_t nfull = tiles_per_batch >= XCD_STRIPE ? total / (8 * XCD_STRIPE) * XCD_STRIPE : 0;
  const int64_t rq = (total - 8 * nfull) >> 3, rr = (total - 8 * nfull) & 7;
  return i < nfull ? ((i / XCD_STRIPE) * 8 + x) * XCD_STRIPE + i % XCD_STRIPE
                   : 8 * nfull + x * rq + std::min<int64_t>(x, rr) + (i - nfull);
}

// Tile t of a group -> matrix, tile row and column.
MUON_DEVICE void tile_at(const GemmArgs& g, int mode, int64_t L, int& bidx, int& tm, int& tn) {
  bidx = (int)(L / g.tiles_per_batch);
  int t = (int)(L % g.tiles_per_batch);
  if (mode == MODE_SYRK) {
    int T = g.tiles_m, r = 0;
    while (t >= T - r) {
      t -= T - r;
      ++r;
    }
    tm = r;
    tn = r + t;
  } else {
    const int GM = 8;  // 8 tile rows per group: measured best for the GEMM stores (X^T rows stay adjacent)
    int TN = g.tiles_n, TM = g.tiles_m;
    int group = t / (GM * TN);
    int first = group * GM;
    int gsz = min(TM - first, GM);
    int local = t % (GM * TN);
    tm = first + local % gsz;
    tn = local / gsz;
  }
}

MUON_DEVICE void map_tile(const GemmArgs& g, int mode, int& bidx, int& tm, int& tn) {
  tile_at(g, mode, xcd_tile(blockIdx.x, (int64_t)gridDim.x, g.tiles_per_batch), bidx, tm, tn);
}

// This workgroup's arguments and tile. Of a launch over one bucket: its own; of several: the
// launch's tiles in one contiguous range per XCD.
MUON_DEVICE const GemmArgs& args_of(const GemmArgs& g, int mode, int& bidx, int& tm, int& tn) {
  map_tile(g, mode, bidx, tm, tn);
  return g;
}
MUON_DEVICE const GemmArgs& args_of(const GemmTab& tab, int mode, int& bidx, int& tm, int& tn) {
  const int64_t L = xcd_tile(blockIdx.x, (int64_t)gridDim.x, 1);
  int gi = 0;
  while (gi + 1 < tab.n && L >= tab.tile0[gi + 1]) ++gi;
  tile_at(tab.g[gi], mode, L - tab.tile0[gi], bidx, tm, tn);
  return tab.g[gi];
}

// The tiles left of a SYRK launch whose first `first` 256-row tiles another launch computes, each cut
// into split x split smaller ones (those below the diagonal have tm > tn: nothing to do).
struct GemmTail {
  GemmArgs g;  // in 256-row tiles
  int first, split;
};
MUON_DEVICE const GemmArgs& args_of(const GemmTail& t, int mode, int& bidx, int& tm, int& tn) {
  const int L = (int)xcd_tile(blockIdx.x, (int64_t)gridDim.x, 1);
  const int ss = t.split * t.split, sub = L % ss;
  tile_at(t.g, mode, t.first + L / ss, bidx, tm, tn);
  tm = tm * t.split + sub / t.split;
  tn = tn * t.split + sub % t.split;
  return t.g;
}

template <typename OutT>
MUON_DEVICE void store_elem(void* p, int64_t idx, float v);
template <>
MUON_DEVICE void store_elem<bf16_t>(void* p, int64_t idx, float v) {
  ((bf16_t*)p)[idx] = f32_to_bf16(v);
}
template <>
MUON_DEVICE void store_elem<float>(void* p, int64_t idx, float v) {
  ((float*)p)[idx] = v;
}
template <typename OutT>
MUON_DEVICE float load_elem(const void* p, int64_t idx);
template <>
MUON_DEVICE float load_elem<bf16_t>(const void* p, int64_t idx) {
  return bf16_to_f32(((const bf16_t*)p)[idx]);
}
template <>
MUON_DEVICE float load_elem<float>(const void* p, int64_t idx) {
  return ((const float*)p)[idx];
}

// Store 4 values at consecutive addresses (i0..i0+3 of row j in the transposed view).
template <typename OutT>
MUON_DEVICE void store4(void* p, int64_t idx, const float* v);
template <>
MUON_DEVICE void store4<bf16_t>(void* p, int64_t idx, const float* v) {
  uint2 w;
  w.x = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
  w.y = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
  *(uint2*)((bf16_t*)p + idx) = w;
}
template <>
MUON_DEVICE void store4<float>(void* p, int64_t idx, const float* v) {
  *(float4*)((float*)p + idx) = make_float4(v[0], v[1], v[2], v[3]);
}

// Epilogue over one wave's FM x FN grid of 32x32 MFMA accumulators.
// 32x32 accumulator layout: lane l, register r -> column j = l % 32,
// row i = 8 * (r / 4) + 4 * (l / 32) + r % 4.
// Unmasked (workspace) outputs are padded to the tile, and elements outside the
// valid Mv x Nv region are stored as zeros so the padding stays zero. Masked
// (caller-owned, unpadded) outputs skip every store outside the valid region and
// use element stores only, since their row pitch need not keep 4-element groups
// aligned.
template <typename OutT, int FM, int FN, bool MASKED>
MUON_DEVICE void epilogue(const GemmArgs& g, int mode, int bidx, int64_t row0, int64_t col0,
                          f32x16 (&acc)[FM][FN], int lane, bool diag) {
  float alpha = g.alpha, beta = g.beta;
  if (g.scale_mode != 0) {
    float s = g.scale[bidx];
    if (g.scale_mode == 1) {
      alpha *= s;
      beta *= s;
    } else {
      alpha *= s * s;
    }
  }
  const int64_t lc = lane & 31, lr = (lane >> 5) * 4;
  void* out = g.out ? (void*)((OutT*)g.out + (int64_t)bidx * g.so) : nullptr;
  void* out_t = g.out_t ? (void*)((OutT*)g.out_t + (int64_t)bidx * g.st) : nullptr;
  const void* cin = g.cin ? (const void*)((const OutT*)g.cin + (int64_t)bidx * g.sc) : nullptr;
#pragma unroll
  for (int fm = 0; fm < FM; ++fm) {
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      const int64_t j = col0 + fn * 32 + lc;
#pragma unroll
      for (int rb = 0; rb < 4; ++rb) {
        const int64_t i0 = row0 + fm * 32 + rb * 8 + lr;
        float v[4];
        bool ok[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int64_t i = i0 + q;
          ok[q] = i < g.Mv && j < g.Nv;
          float x = alpha * acc[fm][fn][rb * 4 + q];
          if (beta != 0.0f && ok[q]) x += beta * load_elem<OutT>(cin, i * g.ldc + j);
          if (!ok[q]) x = 0.0f;
          v[q] = x;
        }
        if (mode == MODE_SYRK) {
          if (!diag) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (!MASKED || ok[q]) store_elem<OutT>(out, (i0 + q) * g.ldo + j, v[q]);
            if (!MASKED) {
              store4<OutT>(out, j * g.ldo + i0, v);
            } else {
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (ok[q]) store_elem<OutT>(out, j * g.ldo + i0 + q, v[q]);
            }
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              const int64_t i = i0 + q;
              if (MASKED && !ok[q]) continue;
              if (i <= j) store_elem<OutT>(out, i * g.ldo + j, v[q]);
              if (i < j) store_elem<OutT>(out, j * g.ldo + i, v[q]);
            }
          }
        } else {
          if (g.store_out) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              if (!MASKED || ok[q]) store_elem<OutT>(out, (i0 + q) * g.ldo + j, v[q]);
          }
          if (g.store_out_t) {
            if (!MASKED) {
              store4<OutT>(out_t, j * g.ldt + i0, v);
            } else {
#pragma unroll
              for (int q = 0; q < 4; ++q)
                if (ok[q]) store_elem<OutT>(out_t, j * g.ldt + i0 + q, v[q]);
            }
          }
        }
      }
    }
  }
}

// ----------------------------------------------------------------------------------
// bf16: 256 x 256 x 64 tile over a WGM x WGN grid of wavefronts, each owning a
// (256/WGM) x (256/WGN) block of 32x32x16 MFMA accumulators. With 4 wavefronts
// (2 x 2) each holds 128 x 128 (256 fp32 accumulators per lane, one wave per SIMD);
// with 8 (2 x 4) each holds 128 x 64 and two waves share a SIMD, hiding each
// other's LDS and memory latency. LDS: double-buffered operand panels with an
// 8-element row pad (row pitch 144 B) so the 16-byte fragment reads of consecutive
// rows hit distinct banks. Global loads for tile k+1 are issued before the MFMAs of
// tile k and parked in registers until the LDS slot frees up.
constexpr int BF_BM = 256, BF_BN = 256, BF_BK = 64, BF_LDSP = BF_BK + 8;
constexpr int BF_SMEM = 2 * (BF_BM + BF_BN) * BF_LDSP * 2;

template <int MODE, bool MASKED, int WGM, int WGN>
__global__ __launch_bounds__(64 * WGM * WGN, 1) void gemm_bf16_kernel(GemmArgs g) {
  constexpr int NT = 64 * WGM * WGN;
  constexpr int WM = BF_BM / WGM, WN = BF_BN / WGN;
  constexpr int FM = WM / 32, FN = WN / 32;
  constexpr int CPT = (BF_BM * BF_BK / 8) / NT;  // 16-byte chunks per thread per operand
  constexpr int RPQ = NT / 8;                      // rows covered by one chunk pass
  extern __shared__ __align__(16) uint8_t smem[];
  bf16_t* As = (bf16_t*)smem;
  bf16_t* Bs = As + 2 * BF_BM * BF_LDSP;

  int bidx, tm, tn;
  map_tile(g, MODE, bidx, tm, tn);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WGN, wn = wave % WGN;

  const bf16_t* A = (const bf16_t*)g.a + (int64_t)bidx * g.sa;
  const bf16_t* B = (const bf16_t*)g.b + (int64_t)bidx * g.sb;
  const int64_t arow0 = (int64_t)tm * BF_BM, brow0 = (int64_t)tn * BF_BN;

  // Unmasked loads go through buffer descriptors (base in SGPRs, one VGPR offset per
  // thread, per-chunk offsets in SGPRs) to keep VGPR pressure off the main loop.
  const int64_t lda_b = g.lda * 2, ldb_b = g.ldb * 2;
  const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(A + arow0 * g.lda), 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(B + brow0 * g.ldb), 0, 0x7fffffff, 0x00020000);
  const int voa = (int)((tid >> 3) * lda_b + (tid & 7) * 16);
  const int vob = (int)((tid >> 3) * ldb_b + (tid & 7) * 16);
  uint4 ra[CPT], rb[CPT];
  auto gload = [&](int64_t k0) {
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
      if (!MASKED) {
        typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
        u32x4 va = __builtin_amdgcn_raw_buffer_load_b128(rsa, voa, (int)(q * RPQ * lda_b + k0 * 2), 0);
        u32x4 vb = __builtin_amdgcn_raw_buffer_load_b128(rsb, vob, (int)(q * RPQ * ldb_b + k0 * 2), 0);
        ra[q] = make_uint4(va.x, va.y, va.z, va.w);
        rb[q] = make_uint4(vb.x, vb.y, vb.z, vb.w);
      } else {
        const int c = q * NT + tid;
        const int r = c >> 3, cc = (c & 7) * 8;
        uint16_t ta[8], tb[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int64_t k = k0 + cc + e;
          const int64_t ia = arow0 + r, ib = brow0 + r;
          ta[e] = (ia < g.Mt && k < g.Kt) ? A[ia * g.lda + k] : (uint16_t)0;
          tb[e] = (ib < g.Nt && k < g.Kt) ? B[ib * g.ldb + k] : (uint16_t)0;
        }
        __builtin_memcpy(&ra[q], ta, 16);
        __builtin_memcpy(&rb[q], tb, 16);
      }
    }
  };
  auto sstore = [&](int buf) {
    bf16_t* as = As + buf * BF_BM * BF_LDSP;
    bf16_t* bs = Bs + buf * BF_BN * BF_LDSP;
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
      const int c = q * NT + tid;
      const int r = c >> 3, cc = (c & 7) * 8;
      *(uint4*)(as + r * BF_LDSP + cc) = ra[q];
      *(uint4*)(bs + r * BF_LDSP + cc) = rb[q];
    }
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int KT = (int)(g.K / BF_BK);
  gload(0);
  sstore(0);
  __syncthreads();
  const int frow = lane & 31, fk = (lane >> 5) * 8;
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < KT) gload((int64_t)(kt + 1) * BF_BK);
    const bf16_t* as = As + cur * BF_BM * BF_LDSP + (wm * WM + frow) * BF_LDSP + fk;
    const bf16_t* bs = Bs + cur * BF_BN * BF_LDSP + (wn * WN + frow) * BF_LDSP + fk;
#pragma unroll
    for (int ks = 0; ks < BF_BK / 16; ++ks) {
      bf16x8_mfma af[FM], bfr[FN];
#pragma unroll
      for (int f = 0; f < FM; ++f)
        af[f] = __builtin_bit_cast(bf16x8_mfma, *(const uint4*)(as + f * 32 * BF_LDSP + ks * 16));
#pragma unroll
      for (int f = 0; f < FN; ++f)
        bfr[f] = __builtin_bit_cast(bf16x8_mfma, *(const uint4*)(bs + f * 32 * BF_LDSP + ks * 16));
#pragma unroll
      for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
          acc[fm][fn] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[fm], bfr[fn], acc[fm][fn], 0, 0, 0);
    }
    if (kt + 1 < KT) sstore(cur ^ 1);
    __syncthreads();
  }

  epilogue<bf16_t, FM, FN, MASKED>(g, MODE, bidx, arow0 + wm * WM, brow0 + wn * WN, acc, lane,
                                   MODE == MODE_SYRK && tm == tn);
}

// ----------------------------------------------------------------------------------
// fp32 gram_ of caller-owned tensors (any extents, element loads with bounds): 128 x 128 x
// 16 tile, 4 wavefronts in 2 x 2, each 64 x 64 (2 x 2 MFMA 32x32x2 f32 blocks).
constexpr int F_BM = 128, F_BK = 16, F_LDSP = F_BK + 4;

__global__ __launch_bounds__(256, 2) void gemm_f32_masked_kernel(GemmArgs g) {
  __shared__ __align__(16) float As[2][F_BM * F_LDSP];
  __shared__ __align__(16) float Bs[2][F_BM * F_LDSP];

  int bidx, tm, tn;
  map_tile(g, MODE_SYRK, bidx, tm, tn);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  const float* A = (const float*)g.a + (int64_t)bidx * g.sa;
  const float* B = (const float*)g.b + (int64_t)bidx * g.sb;
  const int64_t arow0 = (int64_t)tm * F_BM, brow0 = (int64_t)tn * F_BM;

  float4 ra[2], rb[2];
  auto gload = [&](int64_t k0) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int c = q * 256 + tid;
      const int r = c >> 2, cc = (c & 3) * 4;
      float ta[4], tb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int64_t k = k0 + cc + e;
        const int64_t ia = arow0 + r, ib = brow0 + r;
        ta[e] = (ia < g.Mt && k < g.Kt) ? A[ia * g.lda + k] : 0.0f;
        tb[e] = (ib < g.Nt && k < g.Kt) ? B[ib * g.ldb + k] : 0.0f;
      }
      ra[q] = make_float4(ta[0], ta[1], ta[2], ta[3]);
      rb[q] = make_float4(tb[0], tb[1], tb[2], tb[3]);
    }
  };
  auto sstore = [&](int buf) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int c = q * 256 + tid;
      const int r = c >> 2, cc = (c & 3) * 4;
      *(float4*)(&As[buf][r * F_LDSP + cc]) = ra[q];
      *(float4*)(&Bs[buf][r * F_LDSP + cc]) = rb[q];
    }
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int KT = (int)(g.K / F_BK);
  gload(0);
  sstore(0);
  __syncthreads();
  const int frow = lane & 31, fk = lane >> 5;
  for (int kt = 0; kt < KT; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < KT) gload((int64_t)(kt + 1) * F_BK);
#pragma unroll
    for (int ks = 0; ks < F_BK / 2; ++ks) {
      float af[2], bfr[2];
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        af[f] = As[cur][(wm * 64 + f * 32 + frow) * F_LDSP + ks * 2 + fk];
        bfr[f] = Bs[cur][(wn * 64 + f * 32 + frow) * F_LDSP + ks * 2 + fk];
      }
#pragma unroll
      for (int fm = 0; fm < 2; ++fm)
#pragma unroll
        for (int fn = 0; fn < 2; ++fn)
          acc[fm][fn] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[fm], bfr[fn], acc[fm][fn], 0, 0, 0);
    }
    if (kt + 1 < KT) sstore(cur ^ 1);
    __syncthreads();
  }

  epilogue<float, 2, 2, true>(g, MODE_SYRK, bidx, arow0 + wm * 64, brow0 + wn * 64, acc, lane,
                              tm == tn);
}

// ----------------------------------------------------------------------------------
// bf16, direct-to-LDS: the unmasked workhorse of the iteration.
//
// Main loop. 256 x 256 x 64 tile, 8 wavefronts in 4 x 2 (each 64 x 128, two waves per
// SIMD). Operands stream HBM/L2 -> LDS with `buffer_load_dwordx4 ... lds` (no VGPR
// staging, no ds_write), double-buffered: the loads of K-tile k+2 go out in two
// halves during K-tile k (a panel) and k+1 (b panel) and land while their MFMAs run. Each load
// instruction fills 1 KB of LDS (64 lanes x 16 B), i.e. 8 rows of 128 B; the lane ->
// global-address map stores 16-byte chunk c of row r at chunk position c ^ kswz(r).
// The LDS has 64 four-byte banks (256 B per cycle) and serves a 16-byte read 16 lanes
// at a time; a fragment read puts 16 consecutive rows (at one logical chunk) in those
// 16 lanes. With a 128-byte row pitch even rows start at bank 0 and odd rows at bank
// 32, so the swizzle must give the 8 even (and the 8 odd) rows of a 16-row group 8
// distinct chunk positions: kswz(r) = (r >> 1) & 7. (c ^ (r & 7) repeats every 8 rows
// and costs a 2-way conflict on every fragment read.)
// The barrier is an LDS-only wait plus s_barrier: a full __syncthreads would also
// wait for the in-flight prefetch.
//
// Software pipeline. Each k-substep (16 of the 64 k) is one inline-asm block: the 8
// MFMAs of the current fragments interleaved with the 6 LDS reads of the next
// substep's fragments, ending with those reads complete, so LDS latency hides behind
// MFMAs instead of stalling them (the compiler otherwise reorders the MFMAs of the
// next substep up against their own loads). Per K-tile k:
//   DMA of K-tile k+1's b panel into the other stage, substeps 0-2 (reading substeps
//   1-3 of this K-tile), [beta term], wait for K-tile k+1's DMA, barrier, DMA of K-tile
//   k+2's a panel into this K-tile's stage, substep 3 (reading substep 0 of K-tile k+1).
// The loop body has no branch around the MFMAs, which keeps the accumulators in one
// register assignment (a branch there made the allocator copy and spill them); the
// last tile's extra fragment reads hit a stale stage and are discarded.
//
// The beta term. Both uses of beta read the transpose of the b operand:
//   GEMM  X' = a X + B X      with b = X^T   (cin = X   = b^T)
//   SYRK  B  = c A A + b A    with b = A     (cin = A   = A^T, A symmetric)
// so cin(i, j) = b(j, i), and during the K-tile whose k range covers a wave's output
// rows i the needed values sit in the b panel in LDS. The wave adds (beta/alpha) *
// cin into its accumulators there and never reads cin from memory.
//
// Epilogue. The finished tile is staged through LDS (the operand buffers are dead by
// then) so every global store is a coalesced 16-byte row chunk:
//   * transposed stores (GEMM out_t, the mirror half of an off-diagonal SYRK tile):
//     the accumulators hold 4 consecutive rows of one column per lane, written to a
//     transposed LDS tile with 8-byte ds_writes and read back as rows;
//   * row-major stores: written element-wise to a row-major LDS tile.
// Diagonal SYRK tiles store only their upper triangle, mirrored in place, so the
// output is exactly symmetric.
//
// Packed tiles (PK). When the valid extent m leaves the last 128 rows of the padded
// extent M empty (m <= M - 128), the last tile column holds one 128-wide unit of real
// output, columns c0 = M - 256 .. M - 129. A launch of 256 x 256 tiles would spend half
// of every tile of that column on padding, so the PK kernel's full tiles stop one tile
// column short and packed tiles cover the unit: 512 rows x 128 columns per workgroup
// (two 256-row sub-tiles of the a panel against one 128-row b panel), 8 wavefronts of
// 64 x 128 each, the same inner loop. A matrix's packed tiles follow its full tiles in
// one launch: in a launch of their own they re-read every row panel from HBM (the
// m = 1408 X X^T packed tiles ran 1.7x as long as a full tile each, memory-bound). The unit's own 128 x 128 diagonal block lies in
// one packed tile and is stored symmetric as a diagonal tile is; rows and columns from
// M - 128 on are neither computed into the output nor stored. Readers of the result
// never reach them: the products contract over K <= M - 128 and mask rows beyond m.
// Per matrix the packed layout takes T(T-1)/2 + ceil((2T - 1)/4) workgroups instead
// of T(T+1)/2 (T = M / 256): 18 instead of 21 at m = 1408.
constexpr int V2_BK = 64, V2_ROWB = V2_BK * 2, V2_TILEB = 256 * V2_ROWB;
constexpr int V2_STAGEB = 2 * V2_TILEB;
constexpr int V2_EP_PITCH = 256 + 8;  // staging row pitch (elements)
constexpr int V2_SMEM = (2 * V2_STAGEB > 256 * V2_EP_PITCH * 2) ? 2 * V2_STAGEB
                                                                   : 256 * V2_EP_PITCH * 2;
constexpr int V2P_TP = 512 + 8;  // packed: transposed staging, 128 rows of 512
constexpr int V2P_RP = 128 + 8;  // packed: row-major staging, 512 rows of 128
constexpr int v2_smem(bool pk) {
  return !pk ? V2_SMEM
             : std::max(2 * (512 + 128) * V2_ROWB, std::max(128 * V2P_TP * 2, 512 * V2P_RP * 2));
}
static_assert(v2_smem(true) <= 160 * 1024, "packed SYRK tile fits the LDS");

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Chunk swizzle of a K-contiguous operand panel row (rows of 128 B in LDS); a row offset
// by a multiple of 16 keeps its swizzle.
MUON_DEVICE int kswz(int row) { return (row >> 1) & 7; }

MUON_DEVICE void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

MUON_DEVICE void wait_vmcnt0() { __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8)); }

#define MUON_MFMA(C, A, B) "v_mfma_f32_32x32x16_bf16 %[" #C "], %[" #A "], %[" #B "], %[" #C "]\n\t"
// One k-substep of a 64 x 128 wave tile (2 x 4 accumulators of 32 x 32): 8 MFMAs on
// the current fragments (ca, cb), interleaved with the LDS reads of the next
// fragments (na from aa, aa + 4 KB; nb from ba + 0/4/8/12 KB), which are complete
// when the block ends.
MUON_DEVICE void mfma_substep(f32x16 (&acc)[2][4], const bf16x8_mfma (&ca)[2],
                              const bf16x8_mfma (&cb)[4], bf16x8_mfma (&na)[2],
                              bf16x8_mfma (&nb)[4], uint32_t aa, uint32_t ba) {
  asm volatile(
      "ds_read_b128 %[na0], %[aa]\n\t"
      MUON_MFMA(c00, ca0, cb0)
      "ds_read_b128 %[nb0], %[ba]\n\t"
      MUON_MFMA(c01, ca0, cb1)
      "ds_read_b128 %[na1], %[aa] offset:4096\n\t"
      MUON_MFMA(c02, ca0, cb2)
      "ds_read_b128 %[nb1], %[ba] offset:4096\n\t"
      MUON_MFMA(c03, ca0, cb3)
      "ds_read_b128 %[nb2], %[ba] offset:8192\n\t"
      MUON_MFMA(c10, ca1, cb0)
      "ds_read_b128 %[nb3], %[ba] offset:12288\n\t"
      MUON_MFMA(c11, ca1, cb1)
      MUON_MFMA(c12, ca1, cb2)
      MUON_MFMA(c13, ca1, cb3)
      "s_waitcnt lgkmcnt(0)"
      : [c00] "+v"(acc[0][0]), [c01] "+v"(acc[0][1]), [c02] "+v"(acc[0][2]),
        [c03] "+v"(acc[0][3]), [c10] "+v"(acc[1][0]), [c11] "+v"(acc[1][1]),
        [c12] "+v"(acc[1][2]), [c13] "+v"(acc[1][3]), [na0] "=&v"(na[0]), [na1] "=&v"(na[1]),
        [nb0] "=&v"(nb[0]), [nb1] "=&v"(nb[1]), [nb2] "=&v"(nb[2]), [nb3] "=&v"(nb[3])
      : [ca0] "v"(ca[0]), [ca1] "v"(ca[1]), [cb0] "v"(cb[0]), [cb1] "v"(cb[1]),
        [cb2] "v"(cb[2]), [cb3] "v"(cb[3]), [aa] "v"(aa), [ba] "v"(ba));
}
// The right half of mfma_substep (accumulator columns fn 2-3, a diagonal tile's wave
// block whose left half lies below the diagonal): 4 MFMAs, reading the next a fragments
// and b fragments 2-3.
MUON_DEVICE void mfma_substep_r(f32x16 (&acc)[2][4], const bf16x8_mfma (&ca)[2],
                                const bf16x8_mfma (&cb)[4], bf16x8_mfma (&na)[2],
                                bf16x8_mfma (&nb)[4], uint32_t aa, uint32_t ba) {
  asm volatile(
      "ds_read_b128 %[na0], %[aa]\n\t"
      MUON_MFMA(c02, ca0, cb2)
      "ds_read_b128 %[na1], %[aa] offset:4096\n\t"
      MUON_MFMA(c03, ca0, cb3)
      "ds_read_b128 %[nb2], %[ba] offset:8192\n\t"
      MUON_MFMA(c12, ca1, cb2)
      "ds_read_b128 %[nb3], %[ba] offset:12288\n\t"
      MUON_MFMA(c13, ca1, cb3)
      "s_waitcnt lgkmcnt(0)"
      : [c02] "+v"(acc[0][2]), [c03] "+v"(acc[0][3]), [c12] "+v"(acc[1][2]),
        [c13] "+v"(acc[1][3]), [na0] "=&v"(na[0]), [na1] "=&v"(na[1]), [nb2] "=&v"(nb[2]),
        [nb3] "=&v"(nb[3])
      : [ca0] "v"(ca[0]), [ca1] "v"(ca[1]), [cb2] "v"(cb[2]), [cb3] "v"(cb[3]), [aa] "v"(aa),
        [ba] "v"(ba));
}

MUON_DEVICE void frag_load_r(bf16x8_mfma (&na)[2], bf16x8_mfma (&nb)[4], uint32_t aa, uint32_t ba) {
  asm volatile(
      "ds_read_b128 %[na0], %[aa]\n\t"
      "ds_read_b128 %[na1], %[aa] offset:4096\n\t"
      "ds_read_b128 %[nb2], %[ba] offset:8192\n\t"
      "ds_read_b128 %[nb3], %[ba] offset:12288\n\t"
      "s_waitcnt lgkmcnt(0)"
      : [na0] "=&v"(na[0]), [na1] "=&v"(na[1]), [nb2] "=&v"(nb[2]), [nb3] "=&v"(nb[3])
      : [aa] "v"(aa), [ba] "v"(ba));
}

#undef MUON_MFMA

MUON_DEVICE void frag_load(bf16x8_mfma (&na)[2], bf16x8_mfma (&nb)[4], uint32_t aa, uint32_t ba) {
  asm volatile(
      "ds_read_b128 %[na0], %[aa]\n\t"
      "ds_read_b128 %[na1], %[aa] offset:4096\n\t"
      "ds_read_b128 %[nb0], %[ba]\n\t"
      "ds_read_b128 %[nb1], %[ba] offset:4096\n\t"
      "ds_read_b128 %[nb2], %[ba] offset:8192\n\t"
      "ds_read_b128 %[nb3], %[ba] offset:12288\n\t"
      "s_waitcnt lgkmcnt(0)"
      : [na0] "=&v"(na[0]), [na1] "=&v"(na[1]), [nb0] "=&v"(nb[0]), [nb1] "=&v"(nb[1]),
        [nb2] "=&v"(nb[2]), [nb3] "=&v"(nb[3])
      : [aa] "v"(aa), [ba] "v"(ba));
}

// The MFMAs run inside inline asm, which the compiler's hazard recognizer does not
// see: VALU access to their accumulators needs the XDL result latency (at most 19
// wait states on gfx950 for a 32x32 MFMA) in between, and an MFMA reading srcC
// written by VALU needs 2.
MUON_DEVICE void mfma_to_valu_wait() { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory"); }
MUON_DEVICE void valu_to_mfma_wait() { asm volatile("s_nop 4" ::: "memory"); }

typedef __attribute__((ext_vector_type(2))) float f2x;
typedef __attribute__((ext_vector_type(2))) __bf16 bf2x;  // v_cvt_pk_bf16_f32 (RNE)

// A finished 64 x 128 wave tile as bf16 pairs, converted once with the hardware RNE pair
// conversion: hv[fm][fn][2 rg + h] holds rows fm*32 + rg*8 + fh*4 + 2h and + 1 of the
// lane's column fn*32 + lane%32. Unless `full`, elements outside the valid extent are
// cleared to +0 (whatever they held): rem_i counts the valid rows from this lane's first
// row (fh*4 included), rem_j the valid columns from its column.
MUON_DEVICE void v2_pack(const f32x16 (&acc)[2][4], float alpha, bool full, int rem_i,
                         int rem_j, uint32_t (&hv)[2][4][8]) {
#pragma unroll
  for (int fm = 0; fm < 2; ++fm)
#pragma unroll
    for (int fn = 0; fn < 4; ++fn)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const f2x v = {alpha * acc[fm][fn][r], alpha * acc[fm][fn][r + 1]};
        hv[fm][fn][r >> 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf2x));
      }
  if (full) return;
#pragma unroll
  for (int fm = 0; fm < 2; ++fm)
#pragma unroll
    for (int fn = 0; fn < 4; ++fn)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const int il0 = fm * 32 + (r >> 2) * 8 + (r & 3);
        const bool vj = fn * 32 < rem_j;
        const uint32_t keep = (vj && il0 < rem_i ? 0x0000ffffu : 0u) |
                              (vj && il0 + 1 < rem_i ? 0xffff0000u : 0u);
        hv[fm][fn][r >> 1] &= keep;
      }
}

MUON_DEVICE int clamp_rem(int64_t v) { return (int)std::max<int64_t>(-1, std::min<int64_t>(v, 1 << 20)); }

template <int MODE, bool PK>
__global__ __launch_bounds__(512, 1) void gemm_bf16_v2_kernel(GemmArgs g) {
  // PK: the launch mixes the full tiles of the first T-1 tile columns' triangle with the
  // packed tiles of the last column; each matrix's packed tiles follow its full tiles in
  // the tile order, so the workgroups of one XCD share the matrix's row panels in L2
  constexpr int NW = 8, WM = 64, WN = 128, FM = 2, FN = 4;
  extern __shared__ __align__(16) uint8_t smem[];

  int bidx, tm = 0, tn = 0;
  bool pk = false;  // this workgroup's tile is a packed one
  // arow0: first output row; packed: rows arow0 .. arow0 + 511 (logical), the second
  // sub-tile's operand rows read from arow1, which differs from arow0 + 256 only when
  // that sub-tile lies wholly in the padding (it then re-reads valid rows, unstored)
  int64_t arow0, arow1, brow0;
  if constexpr (PK) {
    const int64_t L = xcd_tile(blockIdx.x, (int64_t)gridDim.x, g.tiles_per_batch);
    bidx = (int)(L / g.tiles_per_batch);
    int t = (int)(L % g.tiles_per_batch);
    const int T1 = g.tiles_m - 1;
    const int ntri = T1 * (T1 + 1) / 2;
    const int64_t mpad = (int64_t)g.tiles_m * 256;
    if (t < ntri) {
      int r = 0;
      while (t >= T1 - r) {
        t -= T1 - r;
        ++r;
      }
      tm = r;
      tn = r + t;
      arow0 = (int64_t)tm * 256;
      arow1 = arow0 + 256;
      brow0 = (int64_t)tn * 256;
    } else {
      pk = true;
      arow0 = (int64_t)(t - ntri) * 512;
      arow1 = std::min(arow0 + 256, mpad - 256);
      brow0 = mpad - 256;
    }
  } else {
    map_tile(g, MODE, bidx, tm, tn);
    arow0 = (int64_t)tm * 256;
    arow1 = arow0 + 256;
    brow0 = (int64_t)tn * 256;
  }
  // operand panels: full tiles 256 a rows and 256 b rows (waves 4 x 2), packed tiles
  // 512 a rows and 128 b rows (waves 8 x 1); each wave computes 64 x 128 either way
  const int arows = pk ? 512 : 256;
  const int stageb = (pk ? 640 : 512) * V2_ROWB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // A full diagonal tile (tm == tn) stores only its upper triangle, 10 of its 16 64 x 64
  // units. For B = b A + c A A, and for X X^T with K <= 4096, its waves take the 64 x 128
  // blocks in another order so that each SIMD's two waves (w and w + 4) carry 3, 3, 2 and 2
  // of those units: waves 0-3 compute blocks (0, 0), (0, 1), (1, 1), (2, 1) whole (mode 0),
  // waves 4 and 5 blocks (1, 0) and (3, 1) only in their right half, accumulator columns
  // fn 2-3 (mode 1), waves 6 and 7 blocks (2, 0) and (3, 0), wholly below the diagonal, not
  // at all (mode 2). Its a and b panels are the same rows: only the a panel is loaded.
  const bool dg = MODE == MODE_SYRK && !pk && tm == tn && (g.beta != 0.0f || g.K <= 4096);
  const int wm = pk ? wave : (dg ? (0x32312100 >> (4 * wave)) & 15 : wave >> 1);
  const int wn = pk ? 0 : (dg ? (0x00101110 >> (4 * wave)) & 15 : wave & 1);
  const int wmode = dg ? (0x22110000 >> (4 * wave)) & 15 : 0;
  const bf16_t* A = (const bf16_t*)g.a + (int64_t)bidx * g.sa;
  const bf16_t* B = (const bf16_t*)g.b + (int64_t)bidx * g.sb;
  const int lda_b = (int)(g.lda * 2), ldb_b = (int)(g.ldb * 2);
  const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(A + arow0 * g.lda), 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(B + brow0 * g.ldb), 0, 0x7fffffff, 0x00020000);
  // load slab q*NW + wave = rows (q*NW + wave)*8 .. +7; lane -> row lane/8, chunk
  // position lane%8, which holds logical chunk (lane%8) ^ kswz(row)
  const int r_in = wave * 8 + (lane >> 3);
  const int lch = (lane & 7) ^ kswz(r_in);
  const int voa = r_in * lda_b + lch * 16;
  const int vob = r_in * ldb_b + lch * 16;
  // PK: per-lane byte offsets of the a-panel slabs (slabs 4-7, packed tiles only, from
  // the second sub-tile's rows arow1)
  int voq[8];
#pragma unroll
  for (int q = 0; q < 8; ++q)
    voq[q] = voa + (int)((q >= 4 ? arow1 - arow0 + (q - 4) * NW * 8 : q * NW * 8) * lda_b);
  // A K-tile's DMA in two halves, issued in different substeps: the a panel of K-tile
  // k + 2 after the barrier of K-tile k, the b panel of K-tile k + 2 before the first
  // substep of K-tile k + 1 (all of a CU's loads of one K-tile issued together queue in
  // the load path and hold up the MFMAs behind them; in halves the products run 3-5%
  // faster)
  auto issue_a = [&](int kt, int st) {
    uint8_t* sa = smem + st * stageb;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int slab = q * NW + wave;
      if (q < 4 || pk) {
        const int vo = PK ? voq[q] : voa;
        const int so = PK ? kt * V2_ROWB : q * NW * 8 * lda_b + kt * V2_ROWB;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa, (lds_ptr_t)(sa + slab * 1024), 16, vo, so,
                                                 0, 0);
      }
    }
  };
  auto issue_b = [&](int kt, int st) {
    if (dg) return;
    uint8_t* sb = smem + st * stageb + arows * V2_ROWB;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int slab = q * NW + wave;
      if (q < 2 || !pk)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsb, (lds_ptr_t)(sb + slab * 1024), 16, vob,
                                                 q * NW * 8 * ldb_b + kt * V2_ROWB, 0, 0);
    }
  };

  // MFMA fragment read offsets: lane -> row lane%32 of the fragment, logical chunk
  // 2*ks + lane/32 for k-substep ks
  const int fr = lane & 31, fh = lane >> 5;
  int foff[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) foff[ks] = fr * V2_ROWB + (((ks * 2 + fh) ^ kswz(fr)) << 4);
  const int abase = wm * WM * V2_ROWB, bbase = (dg ? 0 : arows * V2_ROWB) + wn * WN * V2_ROWB;

  float alpha = g.alpha, beta = g.beta;
  if (g.scale_mode != 0) {
    const float s = g.scale[bidx];
    if (g.scale_mode == 1) {
      alpha *= s;
      beta *= s;
    } else {
      alpha *= s * s;
    }
  }
  const float ratio = beta != 0.0f ? beta / alpha : 0.0f;
  // K-tile whose k range equals this wave's output rows (WM == BK), as read
  const int64_t wrow = pk && wm >= 4 ? arow1 + (wm - 4) * WM : arow0 + wm * WM;
  const int kdiag = ratio != 0.0f ? (int)(wrow / V2_BK) : -1;

  const int KT = (int)(g.K / V2_BK);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  auto aaddr = [&](int st, int ks) -> uint32_t { return lds0 + st * stageb + abase + foff[ks]; };
  auto baddr = [&](int st, int ks) -> uint32_t { return lds0 + st * stageb + bbase + foff[ks]; };
  // one K loop and epilogue per MFMA mode, so no path merges into another's registers
  auto kloop = [&](auto mode_c) {
  constexpr int MC = decltype(mode_c)::value;
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  auto substep = [&](const bf16x8_mfma (&ca)[FM], const bf16x8_mfma (&cb)[FN],
                     bf16x8_mfma (&na)[FM], bf16x8_mfma (&nb)[FN], uint32_t aa, uint32_t ba) {
    if constexpr (MC == 0)
      mfma_substep(acc, ca, cb, na, nb, aa, ba);
    else if constexpr (MC == 1)
      mfma_substep_r(acc, ca, cb, na, nb, aa, ba);
  };
  bf16x8_mfma a0[FM], b0[FN], a1[FM], b1[FN];
  issue_a(0, 0);
  issue_b(0, 0);
  wait_vmcnt0();
  lds_barrier();
  if (KT > 1) issue_a(1, 1);
  if constexpr (MC == 0)
    frag_load(a0, b0, aaddr(0, 0), baddr(0, 0));
  else if constexpr (MC == 1)
    frag_load_r(a0, b0, aaddr(0, 0), baddr(0, 0));
  for (int kt = 0; kt < KT; ++kt) {
    const int cs = kt & 1;
    if (kt + 1 < KT) issue_b(kt + 1, cs ^ 1);
    substep(a0, b0, a1, b1, aaddr(cs, 1), baddr(cs, 1));
    substep(a1, b1, a0, b0, aaddr(cs, 2), baddr(cs, 2));
    if (MC != 2 && kt == kdiag) {
      // after the first 32 k, where the other SYRK kernels add it: same bits from each
      // cin(i, j) = b(j, i): row j of the b panel, k offset i - kt*BK (4 consecutive
      // rows i of one accumulator group are 8 contiguous bytes of that row)
      mfma_to_valu_wait();
      const uint8_t* sb = smem + cs * stageb + bbase;
#pragma unroll
      for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int rg = 0; rg < 4; ++rg) {
            const int jl = fn * 32 + fr;  // row within this wave's b rows
            const int kl = fm * 32 + rg * 8 + fh * 4;
            const uint2 w = *(const uint2*)(sb + jl * V2_ROWB +
                                            (((kl >> 3) ^ kswz(jl)) << 4) + (kl & 7) * 2);
            acc[fm][fn][rg * 4 + 0] += ratio * bf16_to_f32((bf16_t)(w.x & 0xffffu));
            acc[fm][fn][rg * 4 + 1] += ratio * bf16_to_f32((bf16_t)(w.x >> 16));
            acc[fm][fn][rg * 4 + 2] += ratio * bf16_to_f32((bf16_t)(w.y & 0xffffu));
            acc[fm][fn][rg * 4 + 3] += ratio * bf16_to_f32((bf16_t)(w.y >> 16));
          }
      valu_to_mfma_wait();
    }
    substep(a0, b0, a1, b1, aaddr(cs, 3), baddr(cs, 3));
    wait_vmcnt0();
    lds_barrier();
    if (kt + 2 < KT) issue_a(kt + 2, cs);
    substep(a1, b1, a0, b0, aaddr(cs ^ 1, 0), baddr(cs ^ 1, 0));
  }
  mfma_to_valu_wait();

  // ---- epilogue: stage through LDS, store 16-byte row chunks ----
  bf16_t* T = (bf16_t*)smem;
  if (PK && pk) {
    // Packed tile: logical rows arow0 + il (il < 512) against columns c0 + jl (jl <
    // 128), c0 = brow0. Rows below c0 are off-diagonal (stored, and mirrored into rows
    // c0 + jl); rows c0 .. c0 + 127 are the unit's diagonal block (upper triangle
    // stored, mirrored in place); later rows are padding, not stored.
    const int64_t c0 = brow0;
    bf16_t* out = (bf16_t*)g.out + (int64_t)bidx * g.so;
    uint32_t hv[FM][FN][8];
    v2_pack(acc, alpha, arow0 + 512 <= g.Mv && c0 + 128 <= g.Nv,
            clamp_rem(g.Mv - (arow0 + wm * WM + fh * 4)), clamp_rem(g.Nv - (c0 + fr)), hv);
    // mirror: T[jl][il], 4 consecutive il per lane -> one 8-byte write
    lds_barrier();
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const int jl = fn * 32 + fr;
          const int il = wm * WM + fm * 32 + rg * 8 + fh * 4;
          *(uint2*)(T + jl * V2P_TP + il) = make_uint2(hv[fm][fn][2 * rg], hv[fm][fn][2 * rg + 1]);
        }
    lds_barrier();
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
      const int id = it * 512 + tid;
      const int jl = id >> 6, c = (id & 63) * 8;
      if (arow0 + c < c0) {  // 8 rows of one off-diagonal unit
        const uint4 w = *(const uint4*)(T + jl * V2P_TP + c);
        *(uint4*)(out + (c0 + jl) * g.ldo + arow0 + c) = w;
      }
    }
    // row-major: T[il][jl]
    lds_barrier();
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int il = wm * WM + fm * 32 + (r >> 2) * 8 + fh * 4 + (r & 3);
          const int jl = fn * 32 + fr;
          T[il * V2P_RP + jl] = (bf16_t)(hv[fm][fn][r >> 1] >> (16 * (r & 1)));
        }
    lds_barrier();
    const int dl0 = (int)(c0 - arow0);  // staging row of the diagonal block's first row
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
      const int id = it * 512 + tid;
      const int il = id >> 4, c = (id & 15) * 8;
      const int dr = il - dl0;  // row within the diagonal block (< 0: off-diagonal)
      if (dr >= 128) continue;  // padding rows
      uint4 w;
      if (dr < 0 || c >= dr) {
        w = *(const uint4*)(T + il * V2P_RP + c);
      } else {
        // diagonal block, chunk reaching below the diagonal: those columns come from
        // the computed (upper) element of the mirror position
        uint16_t e[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
          e[q] = (c + q < dr) ? T[(dl0 + c + q) * V2P_RP + dr] : T[il * V2P_RP + c + q];
        __builtin_memcpy(&w, e, 16);
      }
      *(uint4*)(out + (arow0 + il) * g.ldo + c0 + c) = w;
    }
    return;
  }
  const bool diag = MODE == MODE_SYRK && tm == tn;
  const int row0w = wm * WM, col0w = wn * WN;  // wave origin within the tile
  uint32_t hv[FM][FN][8];
  v2_pack(acc, alpha, arow0 + 256 <= g.Mv && brow0 + 256 <= g.Nv,
          clamp_rem(g.Mv - (arow0 + row0w + fh * 4)), clamp_rem(g.Nv - (brow0 + col0w + fr)), hv);
  bf16_t* out = g.out ? (bf16_t*)g.out + (int64_t)bidx * g.so : nullptr;
  bf16_t* out_t = g.out_t ? (bf16_t*)g.out_t + (int64_t)bidx * g.st : nullptr;
  const int64_t ldt = MODE == MODE_SYRK ? g.ldo : g.ldt;
  if (MODE == MODE_SYRK && !diag) out_t = out;  // mirror half of the symmetric output
  const bool do_t = out_t != nullptr && !diag;
  const bool do_o = out != nullptr;

  if (do_t) {
    // transposed stage: T[j][i], 4 consecutive i per lane -> one 8-byte write
    lds_barrier();
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const int jl = col0w + fn * 32 + fr;
          const int il = row0w + fm * 32 + rg * 8 + fh * 4;
          *(uint2*)(T + jl * V2_EP_PITCH + il) = make_uint2(hv[fm][fn][2 * rg], hv[fm][fn][2 * rg + 1]);
        }
    lds_barrier();
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
      const int id = it * 512 + tid;
      const int jl = id >> 5, c = (id & 31) * 8;
      const uint4 w = *(const uint4*)(T + jl * V2_EP_PITCH + c);
      *(uint4*)(out_t + (brow0 + jl) * ldt + arow0 + c) = w;
    }
  }
  if (do_o) {
    // row-major stage: T[i][j]
    lds_barrier();
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int il = row0w + fm * 32 + (r >> 2) * 8 + fh * 4 + (r & 3);
          const int jl = col0w + fn * 32 + fr;
          T[il * V2_EP_PITCH + jl] = (bf16_t)(hv[fm][fn][r >> 1] >> (16 * (r & 1)));
        }
    lds_barrier();
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
      const int id = it * 512 + tid;
      const int il = id >> 5, c = (id & 31) * 8;
      uint4 w;
      if (!diag || c >= il) {
        w = *(const uint4*)(T + il * V2_EP_PITCH + c);
      } else {
        // diagonal tile, chunk reaching below the diagonal: those columns come from
        // the computed (upper) element of the mirror position
        uint16_t e[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
          e[q] = (c + q < il) ? T[(c + q) * V2_EP_PITCH + il] : T[il * V2_EP_PITCH + c + q];
        __builtin_memcpy(&w, e, 16);
      }
      *(uint4*)(out + (arow0 + il) * g.ldo + brow0 + c) = w;
    }
  }
  };
  if (wmode == 0)
    kloop(std::integral_constant<int, 0>{});
  else if (wmode == 1)
    kloop(std::integral_constant<int, 1>{});
  else
    kloop(std::integral_constant<int, 2>{});
}

// ----------------------------------------------------------------------------------
// bf16 X' = alpha * (B X + ratio * X) with X read in its own row-major layout.
//
// The a operand (B, rows i, k contiguous) is staged as in gemm_bf16_v2_kernel. The
// b operand is X itself, whose rows are k: each K-tile stages a 64 x 256 panel
// X[k][j] (rows of 512 B, 16-byte chunk c of row k stored at chunk c ^ ((k & 3) << 2))
// and the MFMA fragments, which need 8 consecutive k of one column j per lane, come
// from ds_read_b64_tr_b16: within a group of 16 lanes, lane r points at 4 consecutive
// elements of row kb + r/4, columns jb + 4 (r % 4) .. +3, and lane i receives column
// jb + i of rows kb .. kb+3. Two such reads (kb, kb + 4) fill one fragment. The
// swizzle puts the four rows of one read in four different 64-byte bank groups.
//
// The MFMA takes the X fragment as its first operand, so an accumulator holds X'
// transposed: lane l has row i = l % 32 and 4 consecutive columns j of a 32 x 32
// block. Stores of X' are then 8-byte row pieces straight from registers, and the
// beta term X(i, j .. j+3) is 8 contiguous bytes of row k = i of the X panel.
// No X^T is kept in memory; X ping-pongs between two buffers because every tile
// reads whole columns of X.
constexpr int NN_XROWB = 512;                        // X panel row: 256 bf16
constexpr int NN_ATILEB = 256 * V2_ROWB;             // B panel: 256 rows x 64 k
constexpr int NN_XTILEB = V2_BK * NN_XROWB;          // X panel: 64 k x 256 j
constexpr int NN_STAGEB = NN_ATILEB + NN_XTILEB;

typedef __attribute__((ext_vector_type(4))) short i16x4;

// ----------------------------------------------------------------------------------
// Persistent bf16 X' = alpha * (B X + ratio * X): 4 wavefronts (2 x 2), each owning a
// 128 x 128 block of the 256 x 256 tile, accumulators in AGPRs (256 per lane).
//
// Against 8 waves of 64 x 128 (measured 2-8% slower on the same box) a wave reads fewer LDS
// bytes per MFMA, and with one wave per SIMD the DMA of K-tile k + 2 is issued from inside the
// MFMA stream of K-tile k. The grid is one workgroup per CU; each walks a list of tiles with
// the operand pipeline running across tile boundaries: the last two K-tiles of a tile
// prefetch the first two of the next, so a tile's epilogue overlaps the next tile's loads.
//
// All CUs finish their tiles together, so each epilogue is a chip-wide burst of 32 MB
// (4 MB per XCD, the size of its L2). The epilogue therefore stages each wave's 32-row
// blocks through 8 KB of LDS and writes whole 256-byte rows with non-temporal stores:
// measured against stores straight from the accumulators (16-byte row pieces through
// L2), the burst no longer evicts the operand panels the XCD's CUs share, and the
// product runs 5-8% faster.
//
// Tiles are dealt to the 8 XCDs (workgroup b runs on XCD b % 8) in stripes of 64
// consecutive tiles: XCD x's list is stripes x, x + 8, x + 16, ... while whole rounds of 8
// stripes remain, then an equal share of the rest, and its workgroups take every gx-th
// tile of it. The workgroups of one XCD thus share its L2 across neighbouring tiles (GM = 8
// tile rows per column group, as map_tile), and all XCDs work on the same matrices at a
// time, so the operand panels their L2s miss on come from one matrix's worth of data (which
// the Infinity Cache holds) rather than from 8 matrices (contiguous ranges per XCD: 4%
// slower on the 4096 x 14336 bucket).
constexpr int N4_EPB = 32 * 256;                 // epilogue staging per wave: 32 rows
constexpr int N4_STRIPE = 64;                    // tiles per XCD stripe
constexpr int N4_SMEM = 2 * NN_STAGEB + 4 * N4_EPB;  // 160 KiB
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

// buffer descriptor words (raw, stride 0, 2^31 - 1 bytes; num_records 0 for `none`)
MUON_DEVICE u32x4 n4_rsrc(const void* base, bool none) {
  const uint64_t a = (uint64_t)base;
  return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, none ? 0u : 0x7fffffffu, 0x00020000u};
}

// Tile t of the launch -> (matrix, row origin, column origin); GM tile rows per column
// group, as map_tile.
MUON_DEVICE void nn4_tile(const GemmArgs& g, int t, int& bidx, int64_t& arow0, int64_t& bcol0) {
  bidx = t / g.tiles_per_batch;
  const int r = t - bidx * g.tiles_per_batch;
  const int GM = 8, TN = g.tiles_n, TM = g.tiles_m;
  const int group = r / (GM * TN);
  const int first = group * GM;
  const int gsz = min(TM - first, GM);
  const int local = r - group * (GM * TN);
  arow0 = (int64_t)(first + local % gsz) * 256;
  bcol0 = (int64_t)(local / gsz) * 256;
}

// The kernel: the wave's 128 x 128 block is 8 x 8 accumulators of 16 x 16 (AGPRs) and a K-tile
// is two 32-k substeps of 64 MFMAs. A single wave issues v_mfma_f32_32x32x16_bf16 at most
// every 32 cycles and each 16-byte fragment read between them costs it issue time; with
// v_mfma_f32_16x16x32_bf16 the same LDS bytes per FLOP ride along at almost no cost: a
// probe loop with this kernel's reads, DMA and barrier took 35.7 cycles per
// 32 x 32 x 16-equivalent against about 48 for the 32 x 32 x 16 loop. (On 32 x 32 x 16 MFMAs
// B X of 256 matrices of 512 x 1024 took 178 us against 167, of 200 of 640 x 2560 590 against
// 549, of 512 of 128 x 1024 96 against 93.)
//
// Fragments (lane l, r = l % 16, g = l / 16): srcA is X^T, 8 consecutive k (two tr reads)
// of column 16 fj + r; srcB is B, 8 consecutive k (one b128) of row 16 fi + r; the
// accumulator register q of block (fi, fj) is X'(16 fi + r, 16 fj + 4 g + q).
//
// The X panel's chunk swizzle has row bit 3 in it: chunk c of row k sits at c ^ ((k & 3) << 2) ^ (((k >> 3) & 1) << 1). A transposing read serves 32 lanes at a time,
// lanes 0-15 from rows 8 g' .. +3 and lanes 16-31 from rows 8 g' + 8 .. +11 (g' even); with
// the low-bit swizzle alone both groups hit the same 32 banks (35% of LDS-active cycles were
// bank conflicts), with bit 3 they use the other 32. The DMA takes the row parity of each X
// slab from one of two per-lane offsets (slab q holds rows 8 q .. 8 q + 7).
//
// The beta term is added during the two K-tiles whose k range is the wave's rows (no
// registers hold X values through the loop, which the double-buffered fragments need), by
// 32 more MFMAs per substep (n16_beta), so the accumulators never leave their AGPRs; those
// two K-tiles are peeled off the loop.
#define M16(C, X, B) "v_mfma_f32_16x16x32_bf16 %[" #C "], %[" #X "], %[" #B "], %[" #C "]\n\t"
#define N16_OUT(ACC)                                                                      \
  [c0] "+a"(ACC[0]), [c1] "+a"(ACC[1]), [c2] "+a"(ACC[2]), [c3] "+a"(ACC[3]),               \
  [c4] "+a"(ACC[4]), [c5] "+a"(ACC[5]), [c6] "+a"(ACC[6]), [c7] "+a"(ACC[7]),               \
  [nb] "=&v"(nb), [nl] "=&v"(nl), [nh] "=&v"(nh)
#define N16_IN                                                                            \
  [b] "v"(cb), [x0] "v"(cx[0]), [x1] "v"(cx[1]), [x2] "v"(cx[2]), [x3] "v"(cx[3]),          \
  [x4] "v"(cx[4]), [x5] "v"(cx[5]), [x6] "v"(cx[6]), [x7] "v"(cx[7]), [ba] "v"(ba),         \
  [xa] "v"(xa), [o0] "i"(XO), [o1] "i"(XO + 4 * NN_XROWB), [ob] "i"(FI * 16 * V2_ROWB)
// One block of a 32-k substep: the 8 MFMAs of row block FI (accumulators acc[0..7] hold
// X' rows 16 FI + lane%16, columns 16 fj + 4 (lane/16) .. +3) on the current fragments,
// with 3 reads of the next substep's fragments: both halves of X fragment FI (tr reads at
// xa + XO, + 2 KB) and B fragment FI (b128 at ba + 2 KB FI).
// SW (the last iteration of a tall matrix, whose update is applied in the parameter's
// layout): the operands swapped, srcA the B fragment and srcB the X fragments, so the
// accumulators hold X' columns 16 fj + lane%16, rows 16 FI + 4 (lane/16) .. +3, i.e. the
// transpose of the block within each 16 x 16 accumulator (the same products and sums).
#define M16S(C, X, B) "v_mfma_f32_16x16x32_bf16 %[" #C "], %[" #B "], %[" #X "], %[" #C "]\n\t"
#define N16_BLOCK(M)                                                                      \
  "ds_read_b64_tr_b16 %[nl], %[xa] offset:%[o0]\n\t" M(c0, x0, b)                          \
  M(c1, x1, b) M(c2, x2, b)                                                               \
  "ds_read_b64_tr_b16 %[nh], %[xa] offset:%[o1]\n\t" M(c3, x3, b)                          \
  M(c4, x4, b) M(c5, x5, b)                                                               \
  "ds_read_b128 %[nb], %[ba] offset:%[ob]\n\t" M(c6, x6, b)                                \
  M(c7, x7, b)
template <int FI, int XO, bool SW = false>
MUON_DEVICE void n16_block(f32x4 (&acc)[8], const bf16x8_mfma& cb, const bf16x8_mfma (&cx)[8],
                           bf16x8_mfma& nb, i16x4& nl, i16x4& nh, uint32_t ba, uint32_t xa) {
  if constexpr (SW)
    asm volatile(N16_BLOCK(M16S) : N16_OUT(acc) : N16_IN);
  else
    asm volatile(N16_BLOCK(M16) : N16_OUT(acc) : N16_IN);
}
// The same as the first block of a tile: the MFMAs start from zero (C = 0) and define the
// accumulators, so no instruction zeroes them between tiles.
#define M16Z(C, X, B) "v_mfma_f32_16x16x32_bf16 %[" #C "], %[" #X "], %[" #B "], 0\n\t"
#define M16SZ(C, X, B) "v_mfma_f32_16x16x32_bf16 %[" #C "], %[" #B "], %[" #X "], 0\n\t"
#define N16_OUTZ(ACC)                                                                     \
  [c0] "=a"(ACC[0]), [c1] "=a"(ACC[1]), [c2] "=a"(ACC[2]), [c3] "=a"(ACC[3]),               \
  [c4] "=a"(ACC[4]), [c5] "=a"(ACC[5]), [c6] "=a"(ACC[6]), [c7] "=a"(ACC[7]),               \
  [nb] "=&v"(nb), [nl] "=&v"(nl), [nh] "=&v"(nh)
template <int FI, int XO, bool SW = false>
MUON_DEVICE void n16_block_z(f32x4 (&acc)[8], const bf16x8_mfma& cb, const bf16x8_mfma (&cx)[8],
                             bf16x8_mfma& nb, i16x4& nl, i16x4& nh, uint32_t ba, uint32_t xa) {
  if constexpr (SW)
    asm volatile(N16_BLOCK(M16SZ) : N16_OUTZ(acc) : N16_IN);
  else
    asm volatile(N16_BLOCK(M16Z) : N16_OUTZ(acc) : N16_IN);
}
#undef M16Z
#undef M16SZ
#undef N16_OUTZ
// The same with two loads of the DMA of a K-tile (slabs 2 FI and 2 FI + 1 of the 16 this
// wave issues per K-tile: B panel slabs for FI < 4, X panel slabs for FI >= 4), each after an
// MFMA, with per-lane offsets vo0 and vo1. m0 and the scalar offsets of both loads come in
// precomputed.
#define N16_BLOCK_DMA(M)                                                                  \
  "s_mov_b32 m0, %[m00]\n\t"                                                              \
  "ds_read_b64_tr_b16 %[nl], %[xa] offset:%[o0]\n\t" M(c0, x0, b)                          \
  "buffer_load_dwordx4 %[vo0], %[rs], %[so0] offen lds\n\t"                               \
  M(c1, x1, b) "s_mov_b32 m0, %[m01]\n\t" M(c2, x2, b)                                    \
  "ds_read_b64_tr_b16 %[nh], %[xa] offset:%[o1]\n\t" M(c3, x3, b)                          \
  "buffer_load_dwordx4 %[vo1], %[rs], %[so1] offen lds\n\t"                               \
  M(c4, x4, b) M(c5, x5, b)                                                               \
  "ds_read_b128 %[nb], %[ba] offset:%[ob]\n\t" M(c6, x6, b)                                \
  M(c7, x7, b)
#define N16_DMA_IN                                                                        \
  N16_IN, [vo0] "v"(vo0), [vo1] "v"(vo1), [rs] "s"(rs), [so0] "s"(so0), [so1] "s"(so1),    \
      [m00] "s"(m00), [m01] "s"(m01)
template <int FI, int XO, bool SW = false>
MUON_DEVICE void n16_block_dma(f32x4 (&acc)[8], const bf16x8_mfma& cb, const bf16x8_mfma (&cx)[8],
                               bf16x8_mfma& nb, i16x4& nl, i16x4& nh, uint32_t ba, uint32_t xa,
                               int vo0, int vo1, u32x4 rs, int so0, int so1, uint32_t m00,
                               uint32_t m01) {
  if constexpr (SW)
    asm volatile(N16_BLOCK_DMA(M16S) : N16_OUT(acc) : N16_DMA_IN : "m0", "memory");
  else
    asm volatile(N16_BLOCK_DMA(M16) : N16_OUT(acc) : N16_DMA_IN : "m0", "memory");
}
#undef N16_BLOCK
#undef N16_BLOCK_DMA
#undef N16_DMA_IN
#undef N16_OUT
#undef N16_IN
#undef M16
#undef M16S

#define DA "buffer_load_dwordx4 %[voa], %[rsa], %[ta] offen lds\n\t"
#define DXE "buffer_load_dwordx4 %[voxe], %[rsx], %[tx] offen lds\n\t"
#define DXO "buffer_load_dwordx4 %[voxo], %[rsx], %[tx] offen lds\n\t"
#define NA "s_add_u32 m0, m0, 0x1000\n\ts_add_u32 %[ta], %[ta], %[sta]\n\ts_nop 0\n\t"
#define NX "s_add_u32 m0, m0, 0x1000\n\ts_add_u32 %[tx], %[tx], %[stx]\n\ts_nop 0\n\t"
// The DMA of one K-tile without MFMAs (pipeline start); X slab q takes the per-lane offsets
// of its row parity (voxe for even q, voxo for odd).
MUON_DEVICE void n16_dma(int voa, int voxe, int voxo, u32x4 rsa, u32x4 rsx, int soa, int sox,
                         int sta, int stx, uint32_t m0a, uint32_t m0x) {
  int ta, tx;
  asm volatile(
      "s_mov_b32 m0, %[m0a]\n\ts_mov_b32 %[ta], %[soa]\n\ts_nop 0\n\t"
      DA NA DA NA DA NA DA NA DA NA DA NA DA NA DA
      "s_mov_b32 m0, %[m0x]\n\ts_mov_b32 %[tx], %[sox]\n\ts_nop 0\n\t"
      DXE NX DXO NX DXE NX DXO NX DXE NX DXO NX DXE NX DXO
      : [ta] "=&s"(ta), [tx] "=&s"(tx)
      : [voa] "v"(voa), [voxe] "v"(voxe), [voxo] "v"(voxo), [rsa] "s"(rsa), [rsx] "s"(rsx),
        [soa] "s"(soa), [sox] "s"(sox), [sta] "s"(sta), [stx] "s"(stx), [m0a] "s"(m0a),
        [m0x] "s"(m0x)
      : "m0", "scc", "memory");
}
#undef DA
#undef DXE
#undef DXO
#undef NA
#undef NX

// All 24 fragment reads of one substep without MFMAs (pipeline start).
template <int XO>
MUON_DEVICE void n16_frag_load(bf16x8_mfma (&nb)[8], i16x4 (&nl)[8], i16x4 (&nh)[8], uint32_t ba,
                               const uint32_t (&xa)[8]) {
#pragma unroll
  for (int f = 0; f < 8; ++f) {
    asm volatile("ds_read_b64_tr_b16 %0, %3 offset:%4\n\t"
                 "ds_read_b64_tr_b16 %1, %3 offset:%5\n\t"
                 "ds_read_b128 %2, %6 offset:%7"
                 : "=&v"(nl[f]), "=&v"(nh[f]), "=&v"(nb[f])
                 : "v"(xa[f]), "i"(XO), "i"(XO + 4 * NN_XROWB), "v"(ba), "i"(0));
    ba += 16 * V2_ROWB;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

MUON_DEVICE void n16_join(bf16x8_mfma (&cx)[8], const i16x4 (&lo)[8], const i16x4 (&hi)[8]) {
#pragma unroll
  for (int f = 0; f < 8; ++f) {
    const __attribute__((ext_vector_type(8))) short v = __builtin_shufflevector(lo[f], hi[f], 0, 1, 2, 3, 4, 5, 6, 7);
    cx[f] = __builtin_bit_cast(bf16x8_mfma, v);
  }
}

// One 32-k substep: 8 blocks, then the wait for its 24 reads. The first of a tile (Z)
// starts the accumulators from zero.
template <int XO, bool SW = false, bool Z = false>
MUON_DEVICE void n16_substep(f32x4 (&acc)[8][8], const bf16x8_mfma (&cb)[8], const bf16x8_mfma (&cx)[8],
                             bf16x8_mfma (&nb)[8], i16x4 (&nl)[8], i16x4 (&nh)[8], uint32_t ba,
                             const uint32_t (&xa)[8]) {
  if constexpr (Z) {
    n16_block_z<0, XO, SW>(acc[0], cb[0], cx, nb[0], nl[0], nh[0], ba, xa[0]);
    n16_block_z<1, XO, SW>(acc[1], cb[1], cx, nb[1], nl[1], nh[1], ba, xa[1]);
    n16_block_z<2, XO, SW>(acc[2], cb[2], cx, nb[2], nl[2], nh[2], ba, xa[2]);
    n16_block_z<3, XO, SW>(acc[3], cb[3], cx, nb[3], nl[3], nh[3], ba, xa[3]);
    n16_block_z<4, XO, SW>(acc[4], cb[4], cx, nb[4], nl[4], nh[4], ba, xa[4]);
    n16_block_z<5, XO, SW>(acc[5], cb[5], cx, nb[5], nl[5], nh[5], ba, xa[5]);
    n16_block_z<6, XO, SW>(acc[6], cb[6], cx, nb[6], nl[6], nh[6], ba, xa[6]);
    n16_block_z<7, XO, SW>(acc[7], cb[7], cx, nb[7], nl[7], nh[7], ba, xa[7]);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    return;
  }
  n16_block<0, XO, SW>(acc[0], cb[0], cx, nb[0], nl[0], nh[0], ba, xa[0]);
  n16_block<1, XO, SW>(acc[1], cb[1], cx, nb[1], nl[1], nh[1], ba, xa[1]);
  n16_block<2, XO, SW>(acc[2], cb[2], cx, nb[2], nl[2], nh[2], ba, xa[2]);
  n16_block<3, XO, SW>(acc[3], cb[3], cx, nb[3], nl[3], nh[3], ba, xa[3]);
  n16_block<4, XO, SW>(acc[4], cb[4], cx, nb[4], nl[4], nh[4], ba, xa[4]);
  n16_block<5, XO, SW>(acc[5], cb[5], cx, nb[5], nl[5], nh[5], ba, xa[5]);
  n16_block<6, XO, SW>(acc[6], cb[6], cx, nb[6], nl[6], nh[6], ba, xa[6]);
  n16_block<7, XO, SW>(acc[7], cb[7], cx, nb[7], nl[7], nh[7], ba, xa[7]);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// The substep after the barrier, carrying the DMA of one whole K-tile into one stage: blocks
// 0-3 load the B panel slabs (rows 32 q + 8 wave .. +7, q = 0..7), blocks 4-7 the X panel
// slabs (rows 8 q + 2 wave, +1).
template <int XO, bool SW = false>
MUON_DEVICE void n16_substep_dma(f32x4 (&acc)[8][8], const bf16x8_mfma (&cb)[8],
                                 const bf16x8_mfma (&cx)[8], bf16x8_mfma (&nb)[8], i16x4 (&nl)[8],
                                 i16x4 (&nh)[8], uint32_t ba, const uint32_t (&xa)[8], int voa,
                                 int voxe, int voxo, u32x4 rsa, u32x4 rsx, int soa, int sox, int sta, int stx,
                                 uint32_t m0a, uint32_t m0x) {
  n16_block_dma<0, XO, SW>(acc[0], cb[0], cx, nb[0], nl[0], nh[0], ba, xa[0], voa, voa, rsa, soa, soa + sta, m0a, m0a + 0x1000);
  n16_block_dma<1, XO, SW>(acc[1], cb[1], cx, nb[1], nl[1], nh[1], ba, xa[1], voa, voa, rsa, soa + 2 * sta, soa + 3 * sta, m0a + 0x2000, m0a + 0x3000);
  n16_block_dma<2, XO, SW>(acc[2], cb[2], cx, nb[2], nl[2], nh[2], ba, xa[2], voa, voa, rsa, soa + 4 * sta, soa + 5 * sta, m0a + 0x4000, m0a + 0x5000);
  n16_block_dma<3, XO, SW>(acc[3], cb[3], cx, nb[3], nl[3], nh[3], ba, xa[3], voa, voa, rsa, soa + 6 * sta, soa + 7 * sta, m0a + 0x6000, m0a + 0x7000);
  n16_block_dma<4, XO, SW>(acc[4], cb[4], cx, nb[4], nl[4], nh[4], ba, xa[4], voxe, voxo, rsx, sox, sox + stx, m0x, m0x + 0x1000);
  n16_block_dma<5, XO, SW>(acc[5], cb[5], cx, nb[5], nl[5], nh[5], ba, xa[5], voxe, voxo, rsx, sox + 2 * stx, sox + 3 * stx, m0x + 0x2000, m0x + 0x3000);
  n16_block_dma<6, XO, SW>(acc[6], cb[6], cx, nb[6], nl[6], nh[6], ba, xa[6], voxe, voxo, rsx, sox + 4 * stx, sox + 5 * stx, m0x + 0x4000, m0x + 0x5000);
  n16_block_dma<7, XO, SW>(acc[7], cb[7], cx, nb[7], nl[7], nh[7], ba, xa[7], voxe, voxo, rsx, sox + 6 * stx, sox + 7 * stx, m0x + 0x6000, m0x + 0x7000);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// The beta term on the matrix cores: ratio * X(i, j) = sum_k X(k, j) (ratio delta(k, i)), so
// an MFMA with the substep's X fragment as srcA (k = the substep's 32 rows) and a diagonal
// fragment as srcB adds it to the accumulators of the two row blocks those rows are. ratio is
// split into two bf16 parts, hi = RNE(ratio) and lo = RNE(ratio - hi): hi + lo carries 16
// significant bits of the fp32 ratio, so the coefficient applied is a (1 + d) with
// |d| <= about 2^-17 (plus the fp32 rounding of beta / alpha), far below the bf16 output's
// resolution; each bf16 x bf16 product is exact in the fp32 accumulator. The accumulators
// never leave their AGPRs. (A read-modify-write
// through VGPRs made the compiler move accumulators between AGPRs next to the inline-asm
// MFMAs, whose latency it does not see, and the moves raced their results: B X then differed
// by an ulp from run to run.) db[par][part]: lane l (r = l%16, g = l/16) holds B(k, n) for
// k = 8 g .. 8 g + 7, n = r: part at k = 16 par + r, else zero.
MUON_DEVICE void n16_diag_frags(const uint32_t (&parts)[2], int lane, bf16x8_mfma (&db)[2][2]) {
  const int r = lane & 15, g = lane >> 4;
#pragma unroll
  for (int par = 0; par < 2; ++par)
#pragma unroll
    for (int pt = 0; pt < 2; ++pt) {
      const int e = 16 * par + r - 8 * g;  // element of this lane's 8 holding the diagonal
      uint32_t w[4];
#pragma unroll
      for (int d = 0; d < 4; ++d)
        w[d] = (e == 2 * d ? parts[pt] : 0u) | (e == 2 * d + 1 ? parts[pt] << 16 : 0u);
      db[par][pt] = __builtin_bit_cast(bf16x8_mfma, u32x4{w[0], w[1], w[2], w[3]});
    }
}
MUON_DEVICE void n16_beta_frags(float ratio, int lane, bf16x8_mfma (&db)[2][2]) {
  const float hi = bf16_to_f32(f32_to_bf16(ratio));
  const uint32_t parts[2] = {(uint32_t)f32_to_bf16(hi), (uint32_t)f32_to_bf16(ratio - hi)};
  n16_diag_frags(parts, lane, db);
}
// The third part of ratio (and zero): hi + lo + third is the fp32 value. Products of K below
// BETA3_K take it too: at two parts the coefficient's 2^-17 error changes the rounding of enough
// elements of X' that the update of a 256 x 512 matrix ends 9.1e-3 to 9.6e-3 from the iteration
// with the exact coefficient instead of 7.3e-3 to 8.2e-3 (768 x 2304: 7.1e-3 against 5.9e-3).
constexpr int BETA3_K = 768;
MUON_DEVICE void n16_beta_third(float ratio, int lane, bf16x8_mfma (&db)[2][2]) {
  const float hi = bf16_to_f32(f32_to_bf16(ratio));
  const float lo = bf16_to_f32(f32_to_bf16(ratio - hi));
  const uint32_t parts[2] = {(uint32_t)f32_to_bf16((ratio - hi) - lo), 0u};
  n16_diag_frags(parts, lane, db);
}

#define M16(C, X, B) "v_mfma_f32_16x16x32_bf16 %[" #C "], %[" #X "], %[" #B "], %[" #C "]\n\t"
#define M16S(C, X, B) "v_mfma_f32_16x16x32_bf16 %[" #C "], %[" #B "], %[" #X "], %[" #C "]\n\t"
#define NB_ROW(M, P, F, B)                                                                   \
  M(P##0, x0, B) M(P##1, x1, B) M(P##2, x2, B) M(P##3, x3, B)                                 \
  M(P##4, x4, B) M(P##5, x5, B) M(P##6, x6, B) M(P##7, x7, B)
#define NB_ALL(M) NB_ROW(M, a, FI, d0h) NB_ROW(M, b, FI + 1, d1h) NB_ROW(M, a, FI, d0l) NB_ROW(M, b, FI + 1, d1l)
#define NB_HI(M) NB_ROW(M, a, FI, d0h) NB_ROW(M, b, FI + 1, d1h)
#define NB_OUT                                                                               \
  [a0] "+a"(acc[FI][0]), [a1] "+a"(acc[FI][1]), [a2] "+a"(acc[FI][2]), [a3] "+a"(acc[FI][3]),   \
  [a4] "+a"(acc[FI][4]), [a5] "+a"(acc[FI][5]), [a6] "+a"(acc[FI][6]), [a7] "+a"(acc[FI][7]),   \
  [b0] "+a"(acc[FI + 1][0]), [b1] "+a"(acc[FI + 1][1]), [b2] "+a"(acc[FI + 1][2]),             \
  [b3] "+a"(acc[FI + 1][3]), [b4] "+a"(acc[FI + 1][4]), [b5] "+a"(acc[FI + 1][5]),             \
  [b6] "+a"(acc[FI + 1][6]), [b7] "+a"(acc[FI + 1][7])
#define NB_IN                                                                                \
  [x0] "v"(cx[0]), [x1] "v"(cx[1]), [x2] "v"(cx[2]), [x3] "v"(cx[3]), [x4] "v"(cx[4]),        \
  [x5] "v"(cx[5]), [x6] "v"(cx[6]), [x7] "v"(cx[7]), [d0h] "v"(db[0][0]), [d0l] "v"(db[0][1]), \
  [d1h] "v"(db[1][0]), [d1l] "v"(db[1][1])
// ratio * X added to row blocks FI and FI + 1 (rows 32 ks .. 32 ks + 31 of the K-tile whose
// X fragments cx are the substep's): 32 MFMAs, the hi parts of both row blocks first. The
// diagonal fragment serves as srcA as well (SW): its per-lane layout is the same. HI: db holds one
// part only (n16_beta_third), 16 MFMAs (B X of 100 x 512 x 2048 164 -> 156 us against 32 with a
// zero part).
template <int FI, bool SW = false, bool HI = false>
MUON_DEVICE void n16_beta(f32x4 (&acc)[8][8], const bf16x8_mfma (&cx)[8],
                          const bf16x8_mfma (&db)[2][2]) {
  if constexpr (HI && SW)
    asm volatile(NB_HI(M16S) : NB_OUT : NB_IN);
  else if constexpr (HI)
    asm volatile(NB_HI(M16) : NB_OUT : NB_IN);
  else if constexpr (SW)
    asm volatile(NB_ALL(M16S) : NB_OUT : NB_IN);
  else
    asm volatile(NB_ALL(M16) : NB_OUT : NB_IN);
}
#undef NB_ALL
#undef NB_HI
#undef NB_OUT
#undef NB_IN
#undef M16S
#undef NB_ROW
#undef M16

// APPLY 0: X' stored into the workspace. APPLY 1 / 2 (the last iteration, bf16 parameters):
// X' is not stored; each bf16 element of it is the update u of one parameter element, applied
// as the post-pass does (apply_elem: cautious weight decay and the shape-scaled step) and the
// parameter written back. 1: a wide matrix (parameter row i = X' row i); 2: a tall matrix
// (parameter row j = X' column j), computed with swapped MFMA operands so the accumulators
// hold parameter rows.
// MODE (APPLY 1, 2): the form of the apply, from the uniform wd and cautious (below).
// B3: K below BETA3_K, the beta term in three parts.
template <int APPLY, int MODE = 0, bool B3 = false>
__global__ __launch_bounds__(256, 1) void gemm_bf16_nn16_kernel(GemmArgs g, MuonApply ap) {
  constexpr int WM = 128, WN = 128;
  constexpr bool SW = APPLY == 2;
  extern __shared__ __align__(16) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  const int G = gridDim.x, T = g.tiles_total;
  const int x = blockIdx.x & 7, l = blockIdx.x >> 3;
  const int gx = (G >> 3) + (x < (G & 7) ? 1 : 0);
  const int nfull = T / (8 * N4_STRIPE) * N4_STRIPE;
  const int rq = (T - 8 * nfull) >> 3, rr = (T - 8 * nfull) & 7;
  const int tcount = nfull + rq + (x < rr ? 1 : 0);
  auto tile_of = [&](int i) {
    return i < nfull ? ((i / N4_STRIPE) * 8 + x) * N4_STRIPE + i % N4_STRIPE
                     : 8 * nfull + x * rq + min(x, rr) + (i - nfull);
  };
  int li = l;
  if (li >= tcount) return;

  const int lda_b = (int)(g.lda * 2), ldx_b = (int)(g.ldb * 2);
  const int ra_in = wave * 8 + (lane >> 3);
  const int voa = ra_in * lda_b + (((lane & 7) ^ kswz(ra_in)) << 4);
  const int rx_in = wave * 2 + (lane >> 5);
  const int vox = rx_in * ldx_b + (((lane & 31) ^ ((rx_in & 3) << 2)) << 4);
  const int voxo = rx_in * ldx_b + (((lane & 31) ^ ((rx_in & 3) << 2) ^ 2) << 4);
  const int sta = 32 * lda_b, stx = 8 * ldx_b;
  const bf16_t* const A0 = (const bf16_t*)g.a;
  const bf16_t* const X0 = (const bf16_t*)g.b;

  // fragment addresses. B (srcB): lane l -> panel row 128 wm + 16 fi + l%16, logical chunk
  // 4 ks + l/16 (8 consecutive k). X (srcA): tr reads, lane l -> panel row 32 ks + 8 (l/16) +
  // (l%16)/4 (+4 for the high half), columns 128 wn + 16 fj + 4 (l%4) .. +3.
  const int fr = lane & 15, fg = lane >> 4;
  int foff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) foff[ks] = fr * V2_ROWB + (((ks * 4 + fg) ^ kswz(fr)) << 4);
  const int abase = wm * WM * V2_ROWB;
  uint32_t xoff[8];
#pragma unroll
  for (int f = 0; f < 8; ++f) {
    const int chunk = (wn * 16 + f * 2 + ((fr & 3) >> 1)) ^ (((fr >> 2) & 3) << 2) ^ ((fg & 1) << 1);
    xoff[f] = NN_ATILEB + (8 * fg + (fr >> 2)) * NN_XROWB + chunk * 16 + (fr & 1) * 8;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  auto baddr = [&](int st, int ks) -> uint32_t { return lds0 + st * NN_STAGEB + abase + foff[ks]; };
  uint32_t xa[8];
  auto set_xa = [&](int st) {
#pragma unroll
    for (int f = 0; f < 8; ++f) xa[f] = lds0 + st * NN_STAGEB + xoff[f];
  };
  const uint32_t m0w = lds0 + wave * 1024;
  const int KT = (int)(g.K / V2_BK);

  int bidx;
  int64_t arow0, bcol0;
  nn4_tile(g, tile_of(li), bidx, arow0, bcol0);
  u32x4 rsa = n4_rsrc(A0 + (int64_t)bidx * g.sa + arow0 * g.lda, false);
  u32x4 rsx = n4_rsrc(X0 + (int64_t)bidx * g.sb + bcol0, false);

  bf16x8_mfma b0[8], b1[8], x0[8], x1[8];
  i16x4 xl[8], xh[8];
  // K-tiles 0 and 1 of the first tile
  n16_dma(voa, vox, voxo, rsa, rsx, 0, 0, sta, stx, m0w, m0w + NN_ATILEB);
  wait_vmcnt0();
  lds_barrier();
  n16_dma(voa, vox, voxo, rsa, rsx, V2_ROWB, V2_BK * ldx_b, sta, stx, m0w + NN_STAGEB,
          m0w + NN_STAGEB + NN_ATILEB);
  set_xa(0);
  n16_frag_load<0>(b0, xl, xh, baddr(0, 0), xa);
  n16_join(x0, xl, xh);

  f32x4 acc[8][8];
  for (;;) {
    const int lnext = li + gx;
    const bool has_next = lnext < tcount;
    int nbidx = 0;
    int64_t narow0 = 0, nbcol0 = 0;
    if (has_next) nn4_tile(g, tile_of(lnext), nbidx, narow0, nbcol0);
    const u32x4 rsa_n = n4_rsrc(A0 + (int64_t)nbidx * g.sa + narow0 * g.lda, !has_next);
    const u32x4 rsx_n = n4_rsrc(X0 + (int64_t)nbidx * g.sb + nbcol0, !has_next);

    float alpha = g.alpha, beta = g.beta;
    if (g.scale_mode == 1) {
      const float sc = g.scale[bidx];
      alpha *= sc;
      beta *= sc;
    }
    const float ratio = beta != 0.0f ? beta / alpha : 0.0f;
    // the wave's 128 output rows are the k rows of K-tiles kd0 and kd0 + 1; rows at or beyond
    // K are padding, whose X rows are zero
    const int kd = (int)((arow0 + wm * WM) / V2_BK);
    const int kd0 = ratio != 0.0f && kd < KT ? kd : -1;

    // one K-tile: substep 0 (reading substep 1's fragments), wait for K-tile kt + 1's DMA,
    // barrier, substep 1 (reading K-tile kt + 1's first fragments) with the DMA of K-tile
    // kt + 2 (this tile's or the next's) into this K-tile's stage. In the two K-tiles whose k
    // range is the wave's rows (peeled off the loops), each substep also adds ratio * X to
    // the two row blocks its 32 k rows are.
    // first: the tile's K-tile 0, whose first MFMAs start from zero (a compile-time true or
    // false, or a run-time test)
    auto kstep = [&](int kt, auto beta_fi0, auto first) {
      constexpr int FB = decltype(beta_fi0)::value;
      const int cs = kt & 1;
      set_xa(cs);
      if constexpr (std::is_same_v<decltype(first), bool>) {
        if (first)
          n16_substep<16 * NN_XROWB * 2, SW, true>(acc, b0, x0, b1, xl, xh, baddr(cs, 1), xa);
        else
          n16_substep<16 * NN_XROWB * 2, SW>(acc, b0, x0, b1, xl, xh, baddr(cs, 1), xa);
      } else {
        n16_substep<16 * NN_XROWB * 2, SW, decltype(first)::value>(acc, b0, x0, b1, xl, xh,
                                                                     baddr(cs, 1), xa);
      }
      if constexpr (FB >= 0) {
        bf16x8_mfma db[2][2];
        n16_beta_frags(ratio, lane, db);
        n16_beta<FB, SW>(acc, x0, db);
        if constexpr (B3) {
          n16_beta_third(ratio, lane, db);
          n16_beta<FB, SW, true>(acc, x0, db);
        }
      }
      n16_join(x1, xl, xh);
      wait_vmcnt0();
      lds_barrier();
      const bool c2 = kt + 2 < KT;
      const int k2 = c2 ? kt + 2 : kt + 2 - KT;
      set_xa(cs ^ 1);
      const uint32_t m0a = m0w + cs * NN_STAGEB;
      n16_substep_dma<0, SW>(acc, b1, x1, b0, xl, xh, baddr(cs ^ 1, 0), xa, voa, vox, voxo, c2 ? rsa : rsa_n,
                         c2 ? rsx : rsx_n, k2 * V2_ROWB, k2 * V2_BK * ldx_b, sta, stx, m0a,
                         m0a + NN_ATILEB);
      if constexpr (FB >= 0) {
        bf16x8_mfma db[2][2];
        n16_beta_frags(ratio, lane, db);
        n16_beta<FB + 2, SW>(acc, x1, db);
        if constexpr (B3) {
          n16_beta_third(ratio, lane, db);
          n16_beta<FB + 2, SW, true>(acc, x1, db);
        }
      }
      n16_join(x0, xl, xh);
    };
    using no_beta = std::integral_constant<int, -1>;
    using beta_lo = std::integral_constant<int, 0>;
    using beta_hi = std::integral_constant<int, 4>;
    const std::true_type first{};
    const std::false_type later{};
    // Leaving a loop that the peeled beta K-tiles follow, the compiler may copy accumulators
    // between registers before any asm that follows the loop; it does not see the MFMAs in
    // the asm, so the last K-tile of such a loop ends with their latency.
    if constexpr (APPLY == 0 && !B3) {
      // K-tile 0 peeled off every loop, so the loops carry no test for it (B X 1.6% faster on
      // the Llama set than with the test in the loops)
      int kt;
      if (kd0 == 0) {
        kstep(0, beta_lo{}, first);
        kstep(1, beta_hi{}, later);
        kt = 2;
      } else {
        kstep(0, no_beta{}, first);
        kt = 1;
        if (kd0 > 0) {
          for (; kt < kd0; ++kt) {
            kstep(kt, no_beta{}, later);
            if (kt + 1 == kd0) mfma_to_valu_wait();
          }
          kstep(kt++, beta_lo{}, later);
          kstep(kt++, beta_hi{}, later);
        }
      }
      for (; kt < KT; ++kt) kstep(kt, no_beta{}, later);
    } else {
      // the apply kernels test for K-tile 0 in the loops: peeled, their larger epilogue spilled
      // (their launches took 7% longer on the MoE experts), and so do those with the three-part
      // beta term, whose peeled K-tiles hold 64 more MFMAs each (80 bytes of scratch a lane and
      // 154 scalar registers spilled: 100 x 512 x 2048 154 -> 143 us, 200 x 640 x 640 223 -> 196,
      // 300 x 256 x 3072 235 -> 208)
      int kt = 0;
      if (kd0 >= 0) {
        for (; kt < kd0; ++kt) {
          kstep(kt, no_beta{}, kt == 0);
          if (kt + 1 == kd0) mfma_to_valu_wait();
        }
        kstep(kt, beta_lo{}, kt == 0);
        ++kt;
        kstep(kt++, beta_hi{}, later);
      }
      for (; kt < KT; ++kt) kstep(kt, no_beta{}, kt == 0);
    }
    mfma_to_valu_wait();

    // epilogue: accumulator (fi, fj) element q is X'(i, j + q) with i = 128 wm + 16 fi +
    // lane%16, j = 128 wn + 16 fj + 4 (lane/16) (SW: X'(i + q, j) with i = 128 wm + 16 fi +
    // 4 (lane/16), j = 128 wn + 16 fj + lane%16). Two row blocks (32 rows) at a time go through
    // the wave's LDS staging rows (16-byte chunk k of row r at chunk k ^ (r & 15)), then out as
    // 4 whole rows of 256 bytes per non-temporal store.
    const uint32_t ep = lds0 + 2 * NN_STAGEB + wave * N4_EPB;
    const uint32_t epr = ep + (lane >> 4) * 256;
    // staging rows 32 p .. 32 p + 31: X' rows (APPLY 0, 1) or X' columns (APPLY 2), packed bf16
    auto stage = [&](int p, auto masked, int rem_i, int rem_j) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          f32x4 av;
          if constexpr (SW)
            asm volatile("" : "=v"(av) : "0"(acc[k][2 * p + h]));
          else
            asm volatile("" : "=v"(av) : "0"(acc[2 * p + h][k]));
          f2x v01 = {alpha * av[0], alpha * av[1]};
          f2x v23 = {alpha * av[2], alpha * av[3]};
          if (decltype(masked)::value) {
            const int fi = 2 * p + h, jq = k * 16;
            const bool vi = fi * 16 < rem_i;
            v01.x = vi && jq + 0 < rem_j ? v01.x : 0.0f;
            v01.y = vi && jq + 1 < rem_j ? v01.y : 0.0f;
            v23.x = vi && jq + 2 < rem_j ? v23.x : 0.0f;
            v23.y = vi && jq + 3 < rem_j ? v23.y : 0.0f;
          }
          const u32x2 w = {__builtin_bit_cast(uint32_t, __builtin_convertvector(v01, bf2x)),
                           __builtin_bit_cast(uint32_t, __builtin_convertvector(v23, bf2x))};
          uint32_t ea = ep + (h * 16 + fr) * 256 + (fg & 1) * 8, fx = fr;
          asm volatile("" : "+v"(ea), "+v"(fx));
          *(u32x2 __attribute__((address_space(3)))*)(ea + (((2 * k + (fg >> 1)) ^ fx) << 4)) = w;
        }
      }
    };
    if constexpr (APPLY == 0) {
      bf16_t* outw = (bf16_t*)g.out + (int64_t)bidx * g.so + (arow0 + wm * WM) * g.ldo + bcol0 + wn * WN;
      const __amdgpu_buffer_rsrc_t rso =
          __builtin_amdgcn_make_buffer_rsrc((void*)outw, 0, 0x7fffffff, 0x00020000);
      const int ldo_b = (int)(g.ldo * 2);
      const int vor = (lane >> 4) * ldo_b + (lane & 15) * 16;
      const bool full = arow0 + 256 <= g.Mv && bcol0 + 256 <= g.Nv;
      const int rem_i = (int)g.Mv - (int)(arow0 + wm * WM + fr);
      const int rem_j = (int)g.Nv - (int)(bcol0 + wn * WN + 4 * fg);
      auto emit = [&](auto masked) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          stage(p, masked, rem_i, rem_j);
          uint32_t ra = epr, lc = lane & 15, lr = lane >> 4;
          int vs = vor;
          asm volatile("" : "+v"(ra), "+v"(vs), "+v"(lc), "+v"(lr));
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const uint32_t c = lc ^ ((4 * i + lr) & 15);
            const u32x4 q4 = *(const u32x4 __attribute__((address_space(3)))*)(ra + i * 1024 + (c << 4));
            __builtin_amdgcn_raw_buffer_store_b128(q4, rso, vs + i * 4 * ldo_b, p * 32 * ldo_b, 2);
          }
        }
      };
      if (full)
        emit(std::false_type{});
      else
        emit(std::true_type{});
    } else {
      // the parameter block of this wave: rows orow0 .., columns ocol0 .. of matrix mb of
      // tensor t; staging row r of round p is parameter row orow0 + 32 p + r, chunk c its
      // columns ocol0 + 8 c .. + 7
      const int t = (int)(bidx / ap.nb);
      const int64_t mb = bidx - (int64_t)t * ap.nb;
      const float adj = ap.adj[t];
      const int64_t orow0 = SW ? bcol0 + wn * WN : arow0 + wm * WM;
      const int64_t ocol0 = SW ? arow0 + wm * WM : bcol0 + wn * WN;
      bf16_t* pw = (bf16_t*)ap.params[t] + mb * ap.prows * ap.pcols + orow0 * ap.pcols + ocol0;
      const __amdgpu_buffer_rsrc_t rsp =
          __builtin_amdgcn_make_buffer_rsrc((void*)pw, 0, 0x7fffffff, 0x00020000);
      const int ldp_b = (int)(ap.pcols * 2);
      const int lr = lane >> 4, lc = lane & 15;
      const int vop = lr * ldp_b + lc * 16;
      const int vrows = (int)std::min<int64_t>(ap.prows - orow0, 1 << 20);  // valid rows from orow0
      const bool vcol = ocol0 + lc * 8 < ap.pcols;                          // whole 8-column chunks
      // Chunk i of round p is parameter row 32 p + 4 i + lane/16 of the block; its row offset is
      // the scalar offset of the access. A lane outside the parameter (padding rows or columns)
      // takes a per-lane offset past the descriptor's range instead of a branch: its loads
      // read zeros and its stores are dropped, so the code stays straight and the loads of
      // round p + 1 go out before round p is applied.
      const float adjr = bf16_to_f32(f32_to_bf16(adj));
      auto voff = [&](int p, int i) -> int {
        return vcol && lr < vrows - (p * 32 + 4 * i) ? vop : (int)0x80000000;
      };
      // apply_elem<bf16, bf16> in three straight forms (apply_bf16x8, one kernel each: MODE 1
      // cautious weight decay, 2 plain weight decay, 0 no weight decay)
      auto rounds = [&](auto mode_c) {
        constexpr int AM = decltype(mode_c)::value;
        u32x4 pv[2][8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          pv[0][i] = __builtin_amdgcn_raw_buffer_load_b128(rsp, voff(0, i), 4 * i * ldp_b, 2);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          if (p < 3) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
              pv[(p + 1) & 1][i] = __builtin_amdgcn_raw_buffer_load_b128(
                  rsp, voff(p + 1, i), ((p + 1) * 32 + 4 * i) * ldp_b, 2);
          }
          stage(p, std::false_type{}, 0, 0);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const uint32_t c = lc ^ ((4 * i + lr) & 15);
            const u32x4 q4 = *(const u32x4 __attribute__((address_space(3)))*)(epr + i * 1024 + (c << 4));
            const u32x4 o4 = apply_bf16x8<AM>(q4, pv[p & 1][i], adj, adjr, ap.wd);
            __builtin_amdgcn_raw_buffer_store_b128(o4, rsp, voff(p, i), (p * 32 + 4 * i) * ldp_b, 2);
          }
        }
      };
      rounds(std::integral_constant<int, MODE>{});
    }
    if (!has_next) break;
    li = lnext;
    bidx = nbidx;
    arow0 = narow0;
    bcol0 = nbcol0;
    rsa = rsa_n;
    rsx = rsx_n;
  }
}

// ----------------------------------------------------------------------------------
// The SYRK kernel (X X^T, A A) on 16 x 16 x 32 MFMAs.
//
// Tiles, tile order, waves (8, two per SIMD, 64 x 128 each), LDS stages and epilogue
// staging as gemm_bf16_v2_kernel; the wave's block is 4 x 8 accumulators of 16 x 16 and a
// K-tile is two 32-k substeps of 32 MFMAs, each substep reading the next one's 12 fragments
// (4 a, 8 b) between its MFMAs. The DMA of K-tile k + 2 is spread over the second substep
// of K-tile k (two loads per block of 8 MFMAs), right after the barrier that ends the reads
// of its stage. On the Llama shapes X X^T and A A run 6-7% faster than on 32 x 32 x 16
// MFMAs; launches with packed tiles measured 2-5% slower on X X^T (also with a K loop per
// tile kind) and stay on gemm_bf16_v2_kernel.
//
// Fragments (lane l, r = l % 16, g = l / 16): srcA is a-panel row 16 fi + r, srcB is
// b-panel row 16 fj + r, both 8 consecutive k (logical chunk 4 ks + g of the row); the
// accumulator register q of block (fi, fj) is C(16 fi + 4 g + q, 16 fj + r).
#define S16(C, B) "v_mfma_f32_16x16x32_bf16 %[" #C "], %[a], %[" #B "], %[" #C "]\n\t"
#define S16_OUT                                                                             \
  [c0] "+v"(acc[0]), [c1] "+v"(acc[1]), [c2] "+v"(acc[2]), [c3] "+v"(acc[3]),                \
  [c4] "+v"(acc[4]), [c5] "+v"(acc[5]), [c6] "+v"(acc[6]), [c7] "+v"(acc[7]),                \
  [na] "=&v"(na), [nb0] "=&v"(nb0), [nb1] "=&v"(nb1)
#define S16_IN                                                                              \
  [a] "v"(ca), [b0] "v"(cb[0]), [b1] "v"(cb[1]), [b2] "v"(cb[2]), [b3] "v"(cb[3]),           \
  [b4] "v"(cb[4]), [b5] "v"(cb[5]), [b6] "v"(cb[6]), [b7] "v"(cb[7]), [aa] "v"(aa),          \
  [ba] "v"(ba), [oa] "i"(FI * 16 * V2_ROWB), [ob0] "i"(2 * FI * 16 * V2_ROWB),                \
  [ob1] "i"((2 * FI + 1) * 16 * V2_ROWB)
#define S16_RA "ds_read_b128 %[na], %[aa] offset:%[oa]\n\t"
#define S16_RB0 "ds_read_b128 %[nb0], %[ba] offset:%[ob0]\n\t"
#define S16_RB1 "ds_read_b128 %[nb1], %[ba] offset:%[ob1]\n\t"
#define S16_M0(N) "s_mov_b32 m0, %[mz" #N "]\n\t"
#define S16_DL(N) "buffer_load_dwordx4 %[vo" #N "], %[rs" #N "], %[so" #N "] offen lds\n\t"
#define S16_LD(N)                                                                           \
  [vo##N] "v"(vo##N), [rs##N] "s"(rs##N), [so##N] "s"(so##N), [mz##N] "s"(mz##N)
// One block of a 32-k substep: the 8 MFMAs of a fragment FI (accumulators acc[0..7]) with
// the reads of the next substep's a fragment FI (aa + 2 KB FI) and b fragments 2 FI and
// 2 FI + 1 (ba + 2 KB (2 FI), + 2 KB (2 FI + 1)). MODE (diagonal tiles, below): 0 all 8
// column blocks; 1 column blocks 4-7 only (the same reads); 2 no MFMAs and no reads.
template <int FI, int MODE = 0>
MUON_DEVICE void s16_block(f32x4 (&acc)[8], const bf16x8_mfma& ca, const bf16x8_mfma (&cb)[8],
                           bf16x8_mfma& na, bf16x8_mfma& nb0, bf16x8_mfma& nb1, uint32_t aa,
                           uint32_t ba) {
  if constexpr (MODE == 0)
    asm volatile(S16_RA S16(c0, b0) S16(c1, b1) S16(c2, b2)
                 S16_RB0 S16(c3, b3) S16(c4, b4) S16(c5, b5)
                 S16_RB1 S16(c6, b6) S16(c7, b7)
                 : S16_OUT
                 : S16_IN);
  else if constexpr (MODE == 1)
    asm volatile(S16_RA S16(c4, b4) S16_RB0 S16(c5, b5) S16_RB1 S16(c6, b6) S16(c7, b7)
                 : S16_OUT
                 : S16_IN);
}
// The same with two loads of a K-tile's DMA, each after an MFMA that follows its M0 write
// (MODE 2: the loads alone, each one wait state after its M0 write).
template <int FI, int MODE = 0>
MUON_DEVICE void s16_block_dma(f32x4 (&acc)[8], const bf16x8_mfma& ca, const bf16x8_mfma (&cb)[8],
                               bf16x8_mfma& na, bf16x8_mfma& nb0, bf16x8_mfma& nb1, uint32_t aa,
                               uint32_t ba, int vo0, u32x4 rs0, int so0, uint32_t mz0, int vo1,
                               u32x4 rs1, int so1, uint32_t mz1) {
  if constexpr (MODE == 0)
    asm volatile(S16_M0(0) S16_RA S16(c0, b0) S16_DL(0) S16(c1, b1) S16_M0(1) S16(c2, b2)
                 S16_RB0 S16(c3, b3) S16_DL(1) S16(c4, b4) S16(c5, b5)
                 S16_RB1 S16(c6, b6) S16(c7, b7)
                 : S16_OUT
                 : S16_IN, S16_LD(0), S16_LD(1)
                 : "m0", "memory");
  else if constexpr (MODE == 1)
    asm volatile(S16_M0(0) S16_RA S16(c4, b4) S16_DL(0) S16_M0(1) S16_RB0 S16(c5, b5)
                 S16_DL(1) S16_RB1 S16(c6, b6) S16(c7, b7)
                 : S16_OUT
                 : S16_IN, S16_LD(0), S16_LD(1)
                 : "m0", "memory");
  else
    asm volatile(S16_M0(0) "s_nop 0\n\t" S16_DL(0) S16_M0(1) "s_nop 0\n\t" S16_DL(1)
                 :
                 : S16_LD(0), S16_LD(1)
                 : "m0", "memory");
}
#undef S16
#undef S16_OUT
#undef S16_IN
#undef S16_RA
#undef S16_RB0
#undef S16_RB1
#undef S16_M0
#undef S16_DL
#undef S16_LD

typedef bf16x8_mfma s16_frags[12];  // a fragments 0-3, b fragments 0-7

// One substep without DMA, then the wait for its 12 reads.
template <int MODE = 0>
MUON_DEVICE void s16_substep(f32x4 (&acc)[4][8], const s16_frags& c, s16_frags& n, uint32_t aa,
                             uint32_t ba) {
  const bf16x8_mfma(&cb)[8] = *(const bf16x8_mfma(*)[8]) & c[4];
  s16_block<0, MODE>(acc[0], c[0], cb, n[0], n[4], n[5], aa, ba);
  s16_block<1, MODE>(acc[1], c[1], cb, n[1], n[6], n[7], aa, ba);
  s16_block<2, MODE>(acc[2], c[2], cb, n[2], n[8], n[9], aa, ba);
  s16_block<3, MODE>(acc[3], c[3], cb, n[3], n[10], n[11], aa, ba);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// One substep with the DMA of one K-tile into one stage: this wave's slabs q = 0..3 of the a
// panel (scalar offsets soa + q sta, M0 ma + 8 KB q) and of the b panel (sob + q stb, mb +
// 8 KB q), two after each block. A slab is the wave's 1 KB of 8 panel rows. DIAG (a diagonal
// tile, whose b panel is its a panel): the a panel only.
template <int MODE = 0, bool DIAG = false>
MUON_DEVICE void s16_substep_dma(f32x4 (&acc)[4][8], const s16_frags& c, s16_frags& n, uint32_t aa,
                                 uint32_t ba, int voa, int vob, u32x4 rsa, u32x4 rsb, int soa,
                                 int sta, int sob, int stb, uint32_t ma, uint32_t mb) {
  const bf16x8_mfma(&cb)[8] = *(const bf16x8_mfma(*)[8]) & c[4];
  s16_block_dma<0, MODE>(acc[0], c[0], cb, n[0], n[4], n[5], aa, ba, voa, rsa, soa, ma, voa, rsa,
                         soa + sta, ma + 0x2000);
  s16_block_dma<1, MODE>(acc[1], c[1], cb, n[1], n[6], n[7], aa, ba, voa, rsa, soa + 2 * sta,
                         ma + 0x4000, voa, rsa, soa + 3 * sta, ma + 0x6000);
  if constexpr (DIAG) {
    s16_block<2, MODE>(acc[2], c[2], cb, n[2], n[8], n[9], aa, ba);
    s16_block<3, MODE>(acc[3], c[3], cb, n[3], n[10], n[11], aa, ba);
  } else {
    s16_block_dma<2, MODE>(acc[2], c[2], cb, n[2], n[8], n[9], aa, ba, vob, rsb, sob, mb, vob,
                           rsb, sob + stb, mb + 0x2000);
    s16_block_dma<3, MODE>(acc[3], c[3], cb, n[3], n[10], n[11], aa, ba, vob, rsb,
                           sob + 2 * stb, mb + 0x4000, vob, rsb, sob + 3 * stb, mb + 0x6000);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// All 12 fragment reads of one substep without MFMAs (pipeline start).
MUON_DEVICE void s16_frag_load(s16_frags& n, uint32_t aa, uint32_t ba) {
#pragma unroll
  for (int f = 0; f < 4; ++f)
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(n[f]) : "v"(aa), "i"(f * 16 * V2_ROWB));
#pragma unroll
  for (int f = 0; f < 8; ++f)
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(n[4 + f]) : "v"(ba), "i"(f * 16 * V2_ROWB));
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// A finished 64 x 128 wave tile as bf16 pairs (hardware RNE pair conversion): hv[fi][fj][h]
// holds rows 16 fi + 4 g + 2 h and + 1 of the lane's column 16 fj + r. Unless `full`,
// elements outside the valid extent are cleared to +0: rem_i counts the valid rows from the
// lane's first row (4 g included), rem_j the valid columns from its column.
template <int FJ>
MUON_DEVICE void s16_pack(const f32x4 (&acc)[4][FJ], float alpha, bool full, int rem_i, int rem_j,
                          uint32_t (&hv)[4][FJ][2]) {
#pragma unroll
  for (int fi = 0; fi < 4; ++fi)
#pragma unroll
    for (int fj = 0; fj < FJ; ++fj)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f2x v = {alpha * acc[fi][fj][2 * h], alpha * acc[fi][fj][2 * h + 1]};
        hv[fi][fj][h] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf2x));
      }
  if (full) return;
#pragma unroll
  for (int fi = 0; fi < 4; ++fi)
#pragma unroll
    for (int fj = 0; fj < FJ; ++fj)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int il0 = fi * 16 + 2 * h;
        const bool vj = fj * 16 < rem_j;
        const uint32_t keep = (vj && il0 < rem_i ? 0x0000ffffu : 0u) |
                              (vj && il0 + 1 < rem_i ? 0xffff0000u : 0u);
        hv[fi][fj][h] &= keep;
      }
}

__global__ __launch_bounds__(512, 1) void gemm_bf16_s16_kernel(GemmArgs g) {
  constexpr int NW = 8, WM = 64, WN = 128;
  extern __shared__ __align__(16) uint8_t smem[];

  int bidx, tm, tn;
  map_tile(g, MODE_SYRK, bidx, tm, tn);
  const int64_t arow0 = (int64_t)tm * 256, brow0 = (int64_t)tn * 256;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // A diagonal tile (tm == tn) stores only its upper triangle, 10 of its 16 64 x 64 units.
  // Its waves take the 64 x 128 blocks in another order, so that each SIMD's two waves
  // (waves w and w + 4 share a SIMD) carry 3, 3, 2 and 2 of those units instead of 2, 4, 1
  // and 3: waves 0-3 compute blocks (0, 0), (0, 1), (1, 1), (2, 1) whole (MFMA mode 0),
  // waves 4 and 5 blocks (1, 0) and (3, 1), of which only column blocks 4-7 reach the upper
  // triangle (mode 1), waves 6 and 7 blocks (2, 0) and (3, 0), wholly below it (mode 2: no
  // MFMAs). The a and b panels of a diagonal tile are the same rows: only the a panel is
  // loaded, and the b fragments are read from it. This applies to A A and to X X^T with
  // K <= 4096; X X^T over longer rows (K = 14336) ran 1 ms per Llama step slower in this form
  // and keeps whole 64 x 128 blocks and both panels (the epilogue treats its diagonal tiles
  // as diagonal either way).
  const bool dtile = tm == tn;
  const bool diag = dtile && (g.beta != 0.0f || g.K <= 4096);
  const int wm = diag ? (0x32312100 >> (4 * wave)) & 15 : wave >> 1;
  const int wn = diag ? (0x00101110 >> (4 * wave)) & 15 : wave & 1;
  const int wmode = diag ? (0x22110000 >> (4 * wave)) & 15 : 0;
  const bf16_t* A = (const bf16_t*)g.a + (int64_t)bidx * g.sa;
  const bf16_t* B = (const bf16_t*)g.b + (int64_t)bidx * g.sb;
  const int lda_b = (int)(g.lda * 2), ldb_b = (int)(g.ldb * 2);
  const u32x4 rsa = n4_rsrc(A + arow0 * g.lda, false);
  const u32x4 rsb = n4_rsrc(B + brow0 * g.ldb, false);
  const u32x4 rs_none = n4_rsrc(A, true);
  const __amdgpu_buffer_rsrc_t rsa_p =
      __builtin_amdgcn_make_buffer_rsrc((void*)(A + arow0 * g.lda), 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsb_p =
      __builtin_amdgcn_make_buffer_rsrc((void*)(B + brow0 * g.ldb), 0, 0x7fffffff, 0x00020000);
  // load slab q*NW + wave = panel rows (q*NW + wave)*8 .. +7; lane -> row lane/8, chunk
  // position lane%8, which holds logical chunk (lane%8) ^ kswz(row)
  const int r_in = wave * 8 + (lane >> 3);
  const int lch = (lane & 7) ^ kswz(r_in);
  const int voa = r_in * lda_b + lch * 16;
  const int vob = r_in * ldb_b + lch * 16;
  const int sta = NW * 8 * lda_b, stb = NW * 8 * ldb_b;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint32_t m0w = lds0 + wave * 1024;

  // fragment read offsets: lane -> row r of the fragment, logical chunk 4 ks + g
  const int fr = lane & 15, fg = lane >> 4;
  int foff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) foff[ks] = fr * V2_ROWB + (((ks * 4 + fg) ^ kswz(fr)) << 4);
  const int abase = wm * WM * V2_ROWB, bbase = (diag ? 0 : V2_TILEB) + wn * WN * V2_ROWB;

  float alpha = g.alpha, beta = g.beta;
  if (g.scale_mode != 0) {
    const float s = g.scale[bidx];
    if (g.scale_mode == 1) {
      alpha *= s;
      beta *= s;
    } else {
      alpha *= s * s;
    }
  }
  const float ratio = beta != 0.0f ? beta / alpha : 0.0f;
  // K-tile whose k range equals this wave's output rows (WM == BK)
  const int kdiag = ratio != 0.0f ? (int)((arow0 + wm * WM) / V2_BK) : -1;

  const int KT = (int)(g.K / V2_BK);
  auto aaddr = [&](int st, int ks) -> uint32_t { return lds0 + st * V2_STAGEB + abase + foff[ks]; };
  auto baddr = [&](int st, int ks) -> uint32_t { return lds0 + st * V2_STAGEB + bbase + foff[ks]; };
  // the DMA of K-tile kt into stage st (pipeline start; later K-tiles ride in the substeps)
  auto issue = [&](int kt, int st) {
    uint8_t* sa = smem + st * V2_STAGEB;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa_p, (lds_ptr_t)(sa + (q * NW + wave) * 1024), 16,
                                               voa, q * sta + kt * V2_ROWB, 0, 0);
      if (!diag)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsb_p, (lds_ptr_t)(sa + V2_TILEB + (q * NW + wave) * 1024), 16, vob,
            q * stb + kt * V2_ROWB, 0, 0);
    }
  };
  issue(0, 0);
  wait_vmcnt0();
  lds_barrier();
  if (KT > 1) issue(1, 1);
  // accumulators and fragments are declared per path: nothing of the K loop is live across
  // the branch on the mode
  auto kloop = [&](auto mode_c, auto diag_c) {
    constexpr int MODE = decltype(mode_c)::value;
    constexpr bool DIAG = decltype(diag_c)::value;
    f32x4 acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    s16_frags f0, f1;
    if (MODE != 2) s16_frag_load(f0, aaddr(0, 0), baddr(0, 0));
    for (int kt = 0; kt < KT; ++kt) {
      const int cs = kt & 1;
      s16_substep<MODE>(acc, f0, f1, aaddr(cs, 1), baddr(cs, 1));
      if (MODE != 2 && kt == kdiag) {
        // cin(i, j) = b(j, i): row j of the b panel, k offset i - kt*BK (the 4 rows of one
        // accumulator are 8 contiguous bytes of that row)
        mfma_to_valu_wait();
        const uint32_t sb = lds0 + cs * V2_STAGEB + bbase + fr * V2_ROWB + (fg & 1) * 8;
#pragma unroll
        for (int fi = 0; fi < 4; ++fi)
#pragma unroll
          for (int fj = 0; fj < 8; ++fj) {
            const u32x2 w = *(const u32x2 __attribute__((address_space(3)))*)(
                sb + fj * 16 * V2_ROWB + (((2 * fi + (fg >> 1)) ^ kswz(fr)) << 4));
            acc[fi][fj][0] += ratio * __uint_as_float(w.x << 16);
            acc[fi][fj][1] += ratio * __uint_as_float(w.x & 0xffff0000u);
            acc[fi][fj][2] += ratio * __uint_as_float(w.y << 16);
            acc[fi][fj][3] += ratio * __uint_as_float(w.y & 0xffff0000u);
          }
        valu_to_mfma_wait();
      }
      wait_vmcnt0();
      lds_barrier();
      // K-tile kt + 2 into this K-tile's stage; past the last K-tile the null descriptor
      // reads no memory
      const bool more = kt + 2 < KT;
      const int kb = (kt + 2) * V2_ROWB;
      const uint32_t ma = m0w + cs * V2_STAGEB;
      s16_substep_dma<MODE, DIAG>(acc, f1, f0, aaddr(cs ^ 1, 0), baddr(cs ^ 1, 0), voa, vob,
                                  more ? rsa : rs_none, more ? rsb : rs_none, kb, sta, kb, stb,
                                  ma, ma + V2_TILEB);
    }
    mfma_to_valu_wait();
    wait_vmcnt0();

    // ---- epilogue: stage through LDS, store 16-byte row chunks ----
    if (g.out == nullptr) return;
    bf16_t* T = (bf16_t*)smem;
    const int row0w = wm * WM, col0w = wn * WN;  // wave origin within the tile
    uint32_t hv[4][8][2];
    s16_pack(acc, alpha, arow0 + 256 <= g.Mv && brow0 + 256 <= g.Nv,
             clamp_rem(g.Mv - (arow0 + row0w + fg * 4)), clamp_rem(g.Nv - (brow0 + col0w + fr)), hv);
    bf16_t* out = (bf16_t*)g.out + (int64_t)bidx * g.so;
    if (!dtile) {
      // mirror half of the symmetric output: T[j][i], 4 consecutive i per lane -> one 8-byte
      // write
      lds_barrier();
#pragma unroll
      for (int fi = 0; fi < 4; ++fi)
#pragma unroll
        for (int fj = 0; fj < 8; ++fj) {
          const int jl = col0w + fj * 16 + fr;
          const int il = row0w + fi * 16 + fg * 4;
          *(uint2*)(T + jl * V2_EP_PITCH + il) = make_uint2(hv[fi][fj][0], hv[fi][fj][1]);
        }
      lds_barrier();
#pragma unroll 4
      for (int it = 0; it < 16; ++it) {
        const int id = it * 512 + tid;
        const int jl = id >> 5, c = (id & 31) * 8;
        const uint4 w = *(const uint4*)(T + jl * V2_EP_PITCH + c);
        *(uint4*)(out + (brow0 + jl) * g.ldo + arow0 + c) = w;
      }
    }
    // row-major stage: T[i][j]
    lds_barrier();
#pragma unroll
    for (int fi = 0; fi < 4; ++fi)
#pragma unroll
      for (int fj = 0; fj < 8; ++fj)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int il = row0w + fi * 16 + fg * 4 + q;
          const int jl = col0w + fj * 16 + fr;
          T[il * V2_EP_PITCH + jl] = (bf16_t)(hv[fi][fj][q >> 1] >> (16 * (q & 1)));
        }
    lds_barrier();
#pragma unroll 4
    for (int it = 0; it < 16; ++it) {
      const int id = it * 512 + tid;
      const int il = id >> 5, c = (id & 31) * 8;
      uint4 w;
      if (!dtile || c >= il) {
        w = *(const uint4*)(T + il * V2_EP_PITCH + c);
      } else {
        // diagonal tile, chunk reaching below the diagonal: those columns come from the
        // computed (upper) element of the mirror position
        uint16_t e[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
          e[q] = (c + q < il) ? T[(c + q) * V2_EP_PITCH + il] : T[il * V2_EP_PITCH + c + q];
        __builtin_memcpy(&w, e, 16);
      }
      *(uint4*)(out + (arow0 + il) * g.ldo + brow0 + c) = w;
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  // one K loop and epilogue per mode, so no path merges into another's registers
  if (!diag)
    kloop(I0{}, std::false_type{});
  else if (wmode == 0)
    kloop(I0{}, std::true_type{});
  else if (wmode == 1)
    kloop(I1{}, std::true_type{});
  else
    kloop(I2{}, std::true_type{});
}

// ----------------------------------------------------------------------------------
// The SYRK on 128 x 128 tiles, for launches of at most two rounds of 256-row tiles, which
// leave CUs idle (12 matrices of 768 rows: 72 workgroups of 256-row tiles, 252 of 128-row
// ones; 32 of 1024 rows: 320 = 256 + 64, against 1152 in two workgroups per CU). Four
// waves (2 x 2, 64 x 64 each: 4 x 4 accumulators of 16 x 16) and 64 KB of LDS per
// workgroup, so that two workgroups share a CU (two waves per SIMD, as in
// gemm_bf16_s16_kernel). The same K-tile pipeline: two 32-k substeps of 16 MFMAs, each
// reading the next substep's 8 fragments (4 a, 4 b) between its MFMAs, and the DMA of
// K-tile k + 2 spread over the second substep of K-tile k (two loads per block). Fragments
// and accumulator layout as gemm_bf16_s16_kernel's.
constexpr int H_TILEB = 128 * V2_ROWB;  // one 128-row K-panel
constexpr int H_STAGEB = 2 * H_TILEB;   // a and b panels
constexpr int H_EP_PITCH = 128 + 8;     // staging row pitch (elements)
constexpr int H_SMEM = 2 * H_STAGEB;
static_assert(128 * H_EP_PITCH * 2 <= H_SMEM, "the 128-row staging fits the stages");

#define H16(C, B) "v_mfma_f32_16x16x32_bf16 %[" #C "], %[a], %[" #B "], %[" #C "]\n\t"
#define H16_OUT                                                                              \
  [c0] "+v"(acc[0]), [c1] "+v"(acc[1]), [c2] "+v"(acc[2]), [c3] "+v"(acc[3]), [na] "=&v"(na), \
  [nb] "=&v"(nb)
#define H16_IN                                                                               \
  [a] "v"(ca), [b0] "v"(cb[0]), [b1] "v"(cb[1]), [b2] "v"(cb[2]), [b3] "v"(cb[3]), [aa] "v"(aa), \
  [ba] "v"(ba), [oa] "i"(FI * 16 * V2_ROWB)
#define H16_RA "ds_read_b128 %[na], %[aa] offset:%[oa]\n\t"
#define H16_RB "ds_read_b128 %[nb], %[ba] offset:%[oa]\n\t"
#define H16_M0(N) "s_mov_b32 m0, %[mz" #N "]\n\t"
#define H16_DL(N) "buffer_load_dwordx4 %[vo" #N "], %[rs" #N "], %[so" #N "] offen lds\n\t"
#define H16_LD(N) [vo##N] "v"(vo##N), [rs##N] "s"(rs##N), [so##N] "s"(so##N), [mz##N] "s"(mz##N)
// One block of a 32-k substep: the 4 MFMAs of row block FI with the reads of the next
// substep's a fragment FI (aa + 2 KB FI) and b fragment FI (ba + 2 KB FI). MODE 0: all of
// it; 2 (a wave wholly below a diagonal tile's diagonal): nothing.
template <int FI, int MODE = 0>
MUON_DEVICE void h16_block(f32x4 (&acc)[4], const bf16x8_mfma& ca, const bf16x8_mfma (&cb)[4],
                           bf16x8_mfma& na, bf16x8_mfma& nb, uint32_t aa, uint32_t ba) {
  if constexpr (MODE == 0)
    asm volatile(H16_RA H16(c0, b0) H16(c1, b1) H16_RB H16(c2, b2) H16(c3, b3)
                 : H16_OUT
                 : H16_IN);
}
// The same with two loads of a K-tile's DMA, each after an MFMA that follows its M0 write
// (MODE 2: the loads alone, each one wait state after its M0 write).
template <int FI, int MODE = 0>
MUON_DEVICE void h16_block_dma(f32x4 (&acc)[4], const bf16x8_mfma& ca, const bf16x8_mfma (&cb)[4],
                               bf16x8_mfma& na, bf16x8_mfma& nb, uint32_t aa, uint32_t ba,
                               int vo0, u32x4 rs0, int so0, uint32_t mz0, int vo1, u32x4 rs1,
                               int so1, uint32_t mz1) {
  if constexpr (MODE == 0)
    asm volatile(H16_M0(0) H16_RA H16(c0, b0) H16_DL(0) H16(c1, b1) H16_M0(1) H16_RB
                 H16(c2, b2) H16_DL(1) H16(c3, b3)
                 : H16_OUT
                 : H16_IN, H16_LD(0), H16_LD(1)
                 : "m0", "memory");
  else
    asm volatile(H16_M0(0) "s_nop 0\n\t" H16_DL(0) H16_M0(1) "s_nop 0\n\t" H16_DL(1)
                 :
                 : H16_LD(0), H16_LD(1)
                 : "m0", "memory");
}
#undef H16
#undef H16_OUT
#undef H16_IN
#undef H16_RA
#undef H16_RB
#undef H16_M0
#undef H16_DL
#undef H16_LD

typedef bf16x8_mfma h16_frags[8];  // a fragments 0-3, b fragments 0-3

template <int MODE = 0>
MUON_DEVICE void h16_substep(f32x4 (&acc)[4][4], const h16_frags& c, h16_frags& n, uint32_t aa,
                             uint32_t ba) {
  const bf16x8_mfma(&cb)[4] = *(const bf16x8_mfma(*)[4]) & c[4];
  h16_block<0, MODE>(acc[0], c[0], cb, n[0], n[4], aa, ba);
  h16_block<1, MODE>(acc[1], c[1], cb, n[1], n[5], aa, ba);
  h16_block<2, MODE>(acc[2], c[2], cb, n[2], n[6], aa, ba);
  h16_block<3, MODE>(acc[3], c[3], cb, n[3], n[7], aa, ba);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// One substep with the DMA of one K-tile into one stage: this wave's slabs q = 0..3 of the
// a panel (scalar offsets soa + q sta, M0 ma + 4 KB q) and of the b panel (sob + q stb,
// mb + 4 KB q), two after each block. DIAG (a diagonal tile): the a panel only.
template <int MODE = 0, bool DIAG = false>
MUON_DEVICE void h16_substep_dma(f32x4 (&acc)[4][4], const h16_frags& c, h16_frags& n, uint32_t aa,
                                 uint32_t ba, int voa, int vob, u32x4 rsa, u32x4 rsb, int soa,
                                 int sta, int sob, int stb, uint32_t ma, uint32_t mb) {
  const bf16x8_mfma(&cb)[4] = *(const bf16x8_mfma(*)[4]) & c[4];
  h16_block_dma<0, MODE>(acc[0], c[0], cb, n[0], n[4], aa, ba, voa, rsa, soa, ma, voa, rsa,
                         soa + sta, ma + 0x1000);
  h16_block_dma<1, MODE>(acc[1], c[1], cb, n[1], n[5], aa, ba, voa, rsa, soa + 2 * sta,
                         ma + 0x2000, voa, rsa, soa + 3 * sta, ma + 0x3000);
  if constexpr (DIAG) {
    h16_block<2, MODE>(acc[2], c[2], cb, n[2], n[6], aa, ba);
    h16_block<3, MODE>(acc[3], c[3], cb, n[3], n[7], aa, ba);
  } else {
    h16_block_dma<2, MODE>(acc[2], c[2], cb, n[2], n[6], aa, ba, vob, rsb, sob, mb, vob, rsb,
                           sob + stb, mb + 0x1000);
    h16_block_dma<3, MODE>(acc[3], c[3], cb, n[3], n[7], aa, ba, vob, rsb, sob + 2 * stb,
                           mb + 0x2000, vob, rsb, sob + 3 * stb, mb + 0x3000);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

MUON_DEVICE void h16_frag_load(h16_frags& n, uint32_t aa, uint32_t ba) {
#pragma unroll
  for (int f = 0; f < 4; ++f)
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(n[f]) : "v"(aa), "i"(f * 16 * V2_ROWB));
#pragma unroll
  for (int f = 0; f < 4; ++f)
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(n[4 + f]) : "v"(ba), "i"(f * 16 * V2_ROWB));
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

template <typename Args>
__global__ __launch_bounds__(256, 2) void gemm_bf16_s16h_kernel(Args args) {
  constexpr int NW = 4, WM = 64, WN = 64;
  extern __shared__ __align__(16) uint8_t smem[];

  int bidx, tm, tn;
  const GemmArgs& g = args_of(args, MODE_SYRK, bidx, tm, tn);
  if constexpr (std::is_same_v<Args, GemmTail>) {
    if (tm > tn) return;
  }
  const int64_t arow0 = (int64_t)tm * 128, brow0 = (int64_t)tn * 128;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  // A diagonal tile (tm == tn) stores its upper triangle: wave (1, 0) lies wholly below the
  // diagonal and runs no MFMAs, and since the a and b panels are the same rows only the a
  // panel is loaded, the b fragments read from it.
  const bool diag = tm == tn;
  const bool idle = diag && wm == 1 && wn == 0;
  const bf16_t* A = (const bf16_t*)g.a + (int64_t)bidx * g.sa;
  const bf16_t* B = (const bf16_t*)g.b + (int64_t)bidx * g.sb;
  const int lda_b = (int)(g.lda * 2), ldb_b = (int)(g.ldb * 2);
  const u32x4 rsa = n4_rsrc(A + arow0 * g.lda, false);
  const u32x4 rsb = n4_rsrc(B + brow0 * g.ldb, false);
  const u32x4 rs_none = n4_rsrc(A, true);
  const __amdgpu_buffer_rsrc_t rsa_p =
      __builtin_amdgcn_make_buffer_rsrc((void*)(A + arow0 * g.lda), 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsb_p =
      __builtin_amdgcn_make_buffer_rsrc((void*)(B + brow0 * g.ldb), 0, 0x7fffffff, 0x00020000);
  // load slab q*NW + wave = panel rows (q*NW + wave)*8 .. +7; lane -> row lane/8, chunk
  // position lane%8, which holds logical chunk (lane%8) ^ kswz(row)
  const int r_in = wave * 8 + (lane >> 3);
  const int lch = (lane & 7) ^ kswz(r_in);
  const int voa = r_in * lda_b + lch * 16;
  const int vob = r_in * ldb_b + lch * 16;
  const int sta = NW * 8 * lda_b, stb = NW * 8 * ldb_b;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const uint32_t m0w = lds0 + wave * 1024;

  const int fr = lane & 15, fg = lane >> 4;
  int foff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) foff[ks] = fr * V2_ROWB + (((ks * 4 + fg) ^ kswz(fr)) << 4);
  const int abase = wm * WM * V2_ROWB, bbase = (diag ? 0 : H_TILEB) + wn * WN * V2_ROWB;

  float alpha = g.alpha, beta = g.beta;
  if (g.scale_mode != 0) {
    const float s = g.scale[bidx];
    if (g.scale_mode == 1) {
      alpha *= s;
      beta *= s;
    } else {
      alpha *= s * s;
    }
  }
  const float ratio = beta != 0.0f ? beta / alpha : 0.0f;
  // K-tile whose k range equals this wave's output rows (WM == BK)
  const int kdiag = ratio != 0.0f ? (int)((arow0 + wm * WM) / V2_BK) : -1;

  const int KT = (int)(g.K / V2_BK);
  auto aaddr = [&](int st, int ks) -> uint32_t { return lds0 + st * H_STAGEB + abase + foff[ks]; };
  auto baddr = [&](int st, int ks) -> uint32_t { return lds0 + st * H_STAGEB + bbase + foff[ks]; };
  auto issue = [&](int kt, int st) {
    uint8_t* sa = smem + st * H_STAGEB;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsa_p, (lds_ptr_t)(sa + (q * NW + wave) * 1024), 16,
                                               voa, q * sta + kt * V2_ROWB, 0, 0);
      if (!diag)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsb_p, (lds_ptr_t)(sa + H_TILEB + (q * NW + wave) * 1024), 16, vob,
            q * stb + kt * V2_ROWB, 0, 0);
    }
  };
  issue(0, 0);
  wait_vmcnt0();
  lds_barrier();
  if (KT > 1) issue(1, 1);
  auto kloop = [&](auto mode_c, auto diag_c) {
    constexpr int MODE = decltype(mode_c)::value;
    constexpr bool DIAG = decltype(diag_c)::value;
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    h16_frags f0, f1;
    if (MODE != 2) h16_frag_load(f0, aaddr(0, 0), baddr(0, 0));
    for (int kt = 0; kt < KT; ++kt) {
      const int cs = kt & 1;
      h16_substep<MODE>(acc, f0, f1, aaddr(cs, 1), baddr(cs, 1));
      if (MODE != 2 && kt == kdiag) {
        // cin(i, j) = b(j, i): row j of the b panel, k offset i - kt*BK
        mfma_to_valu_wait();
        const uint32_t sb = lds0 + cs * H_STAGEB + bbase + fr * V2_ROWB + (fg & 1) * 8;
#pragma unroll
        for (int fi = 0; fi < 4; ++fi)
#pragma unroll
          for (int fj = 0; fj < 4; ++fj) {
            const u32x2 w = *(const u32x2 __attribute__((address_space(3)))*)(
                sb + fj * 16 * V2_ROWB + (((2 * fi + (fg >> 1)) ^ kswz(fr)) << 4));
            acc[fi][fj][0] += ratio * __uint_as_float(w.x << 16);
            acc[fi][fj][1] += ratio * __uint_as_float(w.x & 0xffff0000u);
            acc[fi][fj][2] += ratio * __uint_as_float(w.y << 16);
            acc[fi][fj][3] += ratio * __uint_as_float(w.y & 0xffff0000u);
          }
        valu_to_mfma_wait();
      }
      wait_vmcnt0();
      lds_barrier();
      // K-tile kt + 2 into this K-tile's stage; past the last K-tile the null descriptor
      // reads no memory
      const bool more = kt + 2 < KT;
      const int kb = (kt + 2) * V2_ROWB;
      const uint32_t ma = m0w + cs * H_STAGEB;
      h16_substep_dma<MODE, DIAG>(acc, f1, f0, aaddr(cs ^ 1, 0), baddr(cs ^ 1, 0), voa, vob,
                                  more ? rsa : rs_none, more ? rsb : rs_none, kb, sta, kb, stb,
                                  ma, ma + H_TILEB);
    }
    mfma_to_valu_wait();
    wait_vmcnt0();

    // ---- epilogue: stage through LDS, store 16-byte row chunks ----
    if (g.out == nullptr) return;
    bf16_t* T = (bf16_t*)smem;
    const int row0w = wm * WM, col0w = wn * WN;  // wave origin within the tile
    uint32_t hv[4][4][2];
    s16_pack<4>(acc, alpha, arow0 + 128 <= g.Mv && brow0 + 128 <= g.Nv,
                clamp_rem(g.Mv - (arow0 + row0w + fg * 4)),
                clamp_rem(g.Nv - (brow0 + col0w + fr)), hv);
    bf16_t* out = (bf16_t*)g.out + (int64_t)bidx * g.so;
    if (!diag) {
      // mirror half of the symmetric output: T[j][i], 4 consecutive i per lane
      lds_barrier();
#pragma unroll
      for (int fi = 0; fi < 4; ++fi)
#pragma unroll
        for (int fj = 0; fj < 4; ++fj) {
          const int jl = col0w + fj * 16 + fr;
          const int il = row0w + fi * 16 + fg * 4;
          *(uint2*)(T + jl * H_EP_PITCH + il) = make_uint2(hv[fi][fj][0], hv[fi][fj][1]);
        }
      lds_barrier();
#pragma unroll 4
      for (int it = 0; it < 8; ++it) {
        const int id = it * 256 + tid;
        const int jl = id >> 4, c = (id & 15) * 8;
        const uint4 w = *(const uint4*)(T + jl * H_EP_PITCH + c);
        *(uint4*)(out + (brow0 + jl) * g.ldo + arow0 + c) = w;
      }
    }
    // row-major stage: T[i][j]
    lds_barrier();
#pragma unroll
    for (int fi = 0; fi < 4; ++fi)
#pragma unroll
      for (int fj = 0; fj < 4; ++fj)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int il = row0w + fi * 16 + fg * 4 + q;
          const int jl = col0w + fj * 16 + fr;
          T[il * H_EP_PITCH + jl] = (bf16_t)(hv[fi][fj][q >> 1] >> (16 * (q & 1)));
        }
    lds_barrier();
#pragma unroll 4
    for (int it = 0; it < 8; ++it) {
      const int id = it * 256 + tid;
      const int il = id >> 4, c = (id & 15) * 8;
      uint4 w;
      if (!diag || c >= il) {
        w = *(const uint4*)(T + il * H_EP_PITCH + c);
      } else {
        // diagonal tile, chunk reaching below the diagonal: those columns come from the
        // computed (upper) element of the mirror position
        uint16_t e[8];
#pragma unroll
        for (int q = 0; q < 8; ++q)
          e[q] = (c + q < il) ? T[(c + q) * H_EP_PITCH + il] : T[il * H_EP_PITCH + c + q];
        __builtin_memcpy(&w, e, 16);
      }
      *(uint4*)(out + (arow0 + il) * g.ldo + brow0 + c) = w;
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I2 = std::integral_constant<int, 2>;
  if (!diag)
    kloop(I0{}, std::false_type{});
  else if (!idle)
    kloop(I0{}, std::true_type{});
  else
    kloop(I2{}, std::true_type{});
}

// ----------------------------------------------------------------------------------
// The fp32 iteration (padded workspaces) and fp32 gram_ of whole tiles: 64 x 64 output tiles,
// 8 waves: two groups of 2 x 2, each wave one 32 x 32 block of 32 x 32 x 2 MFMAs; group 0 sums
// k 0-15 of every 32, group 1 k 16-31, and group 0 adds the two sums at the end (half the
// length of the chains: 1.8e-6 from 64 bits after five iterations of 4 x 768 x 2304, 2.7e-6
// with one chain). Bound by the fp32 matrix rate (64 cycles for each 4 KFLOP MFMA), so the
// kernel has to keep an MFMA ready on every SIMD also where a launch has one workgroup per CU.
// Operands stream HBM/L2 -> LDS with `buffer_load_dwordx4 ... lds` into five stages of 32 k
// (80 KB: two workgroups per CU); a K-tile's fragments are read while the MFMAs of the one
// before run, and a lane reads 4 consecutive k of its row with one ds_read_b128: MFMA t of a
// group of 8 k takes k = 8 q + 4 (lane / 32) + t on both operands (a sum may take its k in
// any order). Panel rows of 32 floats are stored with the 16-byte chunk c of row r at
// c ^ kswz(r), so the 16 rows of a read phase fall in distinct banks. In GEMM (NN) mode the b
// panel is 32 rows k of X (one float per lane and MFMA, 32 consecutive columns; the rows of
// the two half waves are 4 apart, and the XOR of the column's bit 5 with row bit 2 keeps
// them in different banks).
// Four matrices of 768 x 2304, one iteration's three products (X X^T, A A, B X): 77, 33 and
// 106 us, against 265, 101 and 173 us on the 128-row tiles of a register-staged kernel before
// (84 workgroups for the Gram products on 256 CUs, one wave per SIMD, LDS bank conflicts). This
// kernel on 128-row tiles was slower at every size: 117 against 126 TFLOP/s over the whole loop
// on 2 x 4096 x 4096, 83 against 109 on 8 x 1024 x 4096, 54 against 64 on 64 x 256 x 1024.
constexpr int F_TM = 64, F_KT = 32, F_NS = 5;
constexpr int F_PANELB = F_TM * F_KT * 4, F_STAGEB = 2 * F_PANELB, F_SMEM = F_NS * F_STAGEB;

// 16 bytes per lane from memory to LDS (1 KB per wave from byte m0 on).
MUON_DEVICE void lds_dma(int vo, u32x4 rs, int so, uint32_t m0) {
  asm volatile("s_mov_b32 m0, %[mz]\n\ts_nop 0\n\tbuffer_load_dwordx4 %[vo], %[rs], %[so] offen lds\n\t"
               :
               : [vo] "v"(vo), [rs] "s"(rs), [so] "s"(so), [mz] "s"(m0)
               : "m0", "memory");
}

// OWN (SYRK): gram_ of caller-owned tensors with K a multiple of 4: rows past the last read the last
// one, chunks past a row's end its first one and count as zero, no stores outside the output.
template <int MODE, bool OWN = false>
__global__ __launch_bounds__(512, 4) void gemm_f32_kernel(GemmArgs g) {
  extern __shared__ __align__(16) uint8_t smem[];
  int bidx, tm, tn;
  map_tile(g, MODE, bidx, tm, tn);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  const int64_t row0 = (int64_t)tm * F_TM, col0 = (int64_t)tn * F_TM;
  const float* A = (const float*)g.a + (int64_t)bidx * g.sa + (OWN ? 0 : row0 * g.lda);
  const float* B = (const float*)g.b + (int64_t)bidx * g.sb +
                   (OWN ? 0 : MODE == MODE_GEMM ? col0 : col0 * g.ldb);
  const u32x4 rsa = n4_rsrc(A, false), rsb = n4_rsrc(B, false), rs_none = n4_rsrc(A, true);
  const int lda_b = (int)(g.lda * 4), ldb_b = (int)(g.ldb * 4);
  // this wave's load of a panel fills 1 KB: 8 rows of 8 chunks (K-contiguous panels), or 4
  // rows k of 16 chunks (X panel)
  const int ra = wave * 8 + (lane >> 3);
  const int lch = (lane & 7) ^ kswz(ra);
  const int voa = OWN ? min((int)row0 + ra, (int)g.Mt - 1) * lda_b : ra * lda_b + (lch << 4);
  int vob, kstep_b;
  if constexpr (MODE == MODE_GEMM) {
    const int rk = wave * 4 + (lane >> 4);
    vob = rk * ldb_b + (((lane & 15) ^ (((rk >> 2) & 1) << 3)) << 4);
    kstep_b = F_KT * ldb_b;
  } else {
    vob = OWN ? min((int)col0 + ra, (int)g.Mt - 1) * ldb_b : ra * ldb_b + (lch << 4);
    kstep_b = F_KT * 4;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  // (OWN: K-tiles up to a pair of them)
  const int KT = OWN ? (int)((g.Kt + 2 * F_KT - 1) / (2 * F_KT)) * 2 : (int)(g.K / F_KT);
  auto issue = [&](int kt, int st) {
    const bool on = kt < KT;  // past the last K-tile: the null descriptor reads no memory
    const int kk = on ? kt : 0;
    const uint32_t m0 = lds0 + st * F_STAGEB + wave * 1024;
    if constexpr (OWN) {
      const int co = kk * F_KT * 4 + lch * 16 < lda_b ? kk * F_KT * 4 + lch * 16 : 0;
      lds_dma(voa + co, on ? rsa : rs_none, 0, m0);
      lds_dma(vob + co, on ? rsb : rs_none, 0, m0 + F_PANELB);
      return;
    }
    lds_dma(voa, on ? rsa : rs_none, kk * F_KT * 4, m0);
    lds_dma(vob, on ? rsb : rs_none, kk * kstep_b, m0 + F_PANELB);
  };

  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
  const int fr = lane & 31, fh = lane >> 5;
  struct Frags {
    float4 a[2], b[2];  // this group's two groups of 8 k
  };
  auto load = [&](Frags& f, int kt, int st) {
    const uint8_t* pa = smem + st * F_STAGEB + (wm * 32 + fr) * (F_KT * 4);
    const uint8_t* pb = smem + st * F_STAGEB + F_PANELB;
#pragma unroll
    for (int q2 = 0; q2 < 2; ++q2) {
      const int q = 2 * grp + q2;
      const int cpos = ((2 * q + fh) ^ kswz(fr)) << 4;  // (a row offset by 32 keeps its swizzle)
      f.a[q2] = *(const float4*)(pa + cpos);
      if constexpr (MODE == MODE_GEMM) {
        const float* x = (const float*)pb + (8 * q + 4 * fh) * F_TM + ((wn * 32 + fr) ^ (fh << 5));
        f.b[q2] = make_float4(x[0], x[F_TM], x[2 * F_TM], x[3 * F_TM]);
      } else {
        f.b[q2] = *(const float4*)(pb + (wn * 32 + fr) * (F_KT * 4) + cpos);
      }
      if (OWN && kt * F_KT + 8 * q + 4 * fh >= g.Kt)
        f.a[q2] = f.b[q2] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
  };
  auto mma = [&](const Frags& f) {
#pragma unroll
    for (int q2 = 0; q2 < 2; ++q2)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(((const float*)&f.a[q2])[t],
                                                   ((const float*)&f.b[q2])[t], acc, 0, 0, 0);
  };
#pragma unroll
  for (int t = 0; t < F_NS - 1; ++t) issue(t, t);
  // K-tile kt: once K-tile kt + 1 has landed (those up to kt + F_NS - 2 may still be under way,
  // two loads each) and every wave has read K-tile kt, the load of K-tile kt + F_NS - 1, the
  // fragments of K-tile kt + 1, and the MFMAs of K-tile kt while those reads complete
  int st = 0;
  auto step = [&](int kt, const Frags& cur, Frags& next) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * (F_NS - 3)) : "memory");
    lds_barrier();
    issue(kt + F_NS - 1, st == 0 ? F_NS - 1 : st - 1);
    st = st + 1 == F_NS ? 0 : st + 1;
    load(next, kt + 1, st);
    mma(cur);
  };
  Frags f0, f1;
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * (F_NS - 2)) : "memory");
  lds_barrier();
  load(f0, 0, 0);
  for (int kt = 0; kt < KT; kt += 2) {  // (K is a multiple of 64)
    step(kt, f0, f1);
    step(kt + 1, f1, f0);
  }
  wait_vmcnt0();
  // group 1's sums through LDS (the stages are done with)
  float* sum = (float*)smem + (wave & 3) * 1024 + lane;
  lds_barrier();
  if (grp == 1) {
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[r * 64] = acc[r];
  }
  lds_barrier();
  if (grp == 1) return;
  f32x16 accs[1][1];
#pragma unroll
  for (int r = 0; r < 16; ++r) accs[0][0][r] = acc[r] + sum[r * 64];
  epilogue<float, 1, 1, OWN>(g, MODE, bidx, row0 + wm * 32, col0 + wn * 32, accs, lane,
                               MODE == MODE_SYRK && tm == tn);
}

// ----------------------------------------------------------------------------------
// Products of small and medium launches on TM x TM tiles (TM = 128 or 64), several buckets per
// launch (GemmTab): four waves of (TM / 2) x (TM / 2), 16 x 16 x 32 MFMAs. With 256-row tiles and
// one workgroup per CU such a launch fills a fraction of the CUs (a 256 x 512 matrix: one
// workgroup for X X^T, two for B X) and its time is that of one workgroup's K loop and
// epilogue: 9.7 us for X X^T and 14.6 us for B X of that matrix.
// A K-tile is 64 k. TM = 128: two stages of 32 KB, two workgroups per CU. TM = 64: four stages of
// 16 KB, two workgroups per CU: the loads of K-tiles k + 1 .. k + 3 are under way while K-tile k
// is multiplied, since a launch of one small workgroup per CU has nothing else to hide their
// latency with. Operands stream to LDS by `buffer_load_dwordx4 ... lds`, rows of K-contiguous
// panels swizzled with kswz.
// (A 128-row tile_syrk_kernel took 169 us against gemm_bf16_s16h_kernel's 155 for A A of two
// matrices of 4096 rows and 17 against 18 for a dozen of 768: the SYRK's 128-row tiles stay
// that kernel's.)
// Each output element sees the MFMAs of gemm_bf16_s16_kernel / gemm_bf16_nn16_kernel in the same
// order, the beta term at the same place, so its bits do not depend on the kernel that
// serves a launch.
template <int TM>
struct TileK {
  static constexpr int NS = TM == 64 ? 4 : 2;
  static constexpr int PANELB = TM * V2_ROWB;  // either operand's panel of one K-tile
  static constexpr int STAGEB = 2 * PANELB;
  static constexpr int SMEM = NS * STAGEB;
  static constexpr int F = TM / 32;            // 16-row blocks per wave and side
  static constexpr int LOADS = TM / 32;        // 1 KB loads per wave and panel
  static constexpr int PITCH = TM + 8;         // epilogue staging row (elements)
  static_assert(TM * PITCH * 2 <= SMEM, "the staging tile fits the stages");
};

// A = alpha X X^T (K = n) or B = alpha (A A + ratio A): upper-triangle tiles, mirrored.
// OWN: gram_ of caller-owned tensors, M and K any (rows a whole number of 16-byte chunks): rows past
// the last read the last one, the chunks past a row's end its first one and count as zero, and
// nothing is stored outside the M x M output. Eight matrices of 1000 x 1336 take 27 us, 166 on the
// register-staged masked kernel with its element loads (fp32, four of them: 84 and 181 us).
template <int TM, typename Args, bool OWN = false>
__global__ __launch_bounds__(256, 2) void tile_syrk_kernel(Args args) {
  typedef TileK<TM> C;
  constexpr int F = C::F, WM = TM / 2;
  extern __shared__ __align__(16) uint8_t smem[];
  int bidx, tm, tn;
  const GemmArgs& g = args_of(args, MODE_SYRK, bidx, tm, tn);
  if constexpr (std::is_same_v<Args, GemmTail>) {
    if (tm > tn) return;
  }
  const int row0 = tm * TM, col0 = tn * TM;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const bool diag = tm == tn;  // one panel serves both operands
  const bf16_t* A = (const bf16_t*)g.a + (int64_t)bidx * g.sa;
  const u32x4 rsa = n4_rsrc(OWN ? A : A + (int64_t)row0 * g.lda, false);
  const u32x4 rsb = n4_rsrc(OWN ? A : A + (int64_t)col0 * g.lda, diag);
  const u32x4 rs_none = n4_rsrc(A, true);
  const int lda_b = (int)(g.lda * 2);
  // load q of this wave: rows (4 q + wave) * 8 + lane / 8 of the panel, 16-byte chunk lane % 8
  const int r_in = wave * 8 + (lane >> 3);
  const int lch = (lane & 7) ^ kswz(r_in);
  const int vo = r_in * lda_b + (lch << 4);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const int KT = OWN ? (int)((g.Kt + V2_BK - 1) / V2_BK) : (int)(g.K / V2_BK);
  int voa[C::LOADS], vob[C::LOADS];  // (OWN) byte offsets of the rows from the matrix
  if constexpr (OWN) {
#pragma unroll
    for (int q = 0; q < C::LOADS; ++q) {
      voa[q] = min(row0 + q * 32 + r_in, (int)g.Mt - 1) * lda_b;
      vob[q] = min(col0 + q * 32 + r_in, (int)g.Mt - 1) * lda_b;
    }
  }
  auto issue = [&](int kt, int st) {
    const bool on = kt < KT;
    const int kb = on ? kt * V2_ROWB : 0;
    const uint32_t m0 = lds0 + st * C::STAGEB + wave * 1024;
    const u32x4 pa = on ? rsa : rs_none, pb = on ? rsb : rs_none;
#pragma unroll
    for (int q = 0; q < C::LOADS; ++q) {
      if constexpr (OWN) {
        const int co = kb + lch * 16 < lda_b ? kb + lch * 16 : 0;
        lds_dma(voa[q] + co, pa, 0, m0 + q * 4096);
        lds_dma(vob[q] + co, pb, 0, m0 + C::PANELB + q * 4096);
      } else {
        lds_dma(vo, pa, kb + q * 32 * lda_b, m0 + q * 4096);
        lds_dma(vo, pb, kb + q * 32 * lda_b, m0 + C::PANELB + q * 4096);
      }
    }
  };
  float alpha = g.alpha, beta = g.beta;
  if (g.scale_mode == 2) {
    const float s = g.scale[bidx];
    alpha *= s * s;
  }
  const float ratio = beta != 0.0f ? beta / alpha : 0.0f;
  // K-tile whose k range holds this wave's output rows (of a 64-row wave exactly, of a 32-row
  // one a half of it)
  const int kdiag = ratio != 0.0f ? (row0 + wm * WM) / V2_BK : -1;
  const int koff = (row0 + wm * WM) & 63;  // the rows' place in it

  f32x4 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int fr = lane & 15, fg = lane >> 4;
  const int abase = wm * WM * V2_ROWB, bbase = (diag ? 0 : C::PANELB) + wn * WM * V2_ROWB;
#pragma unroll
  for (int t = 0; t < C::NS - 1; ++t) issue(t, t);
  int st = 0;
  for (int kt = 0; kt < KT; ++kt) {
    // 2 LOADS loads per K-tile: those of K-tiles kt + 1 .. kt + NS - 2 may still be under way
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * C::LOADS * (C::NS - 2)) : "memory");
    lds_barrier();
    issue(kt + C::NS - 1, st == 0 ? C::NS - 1 : st - 1);
    const uint8_t* sp = smem + st * C::STAGEB;
    bf16x8_mfma a[2][F], b[2][F];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int off = fr * V2_ROWB + (((ks * 4 + fg) ^ kswz(fr)) << 4);
#pragma unroll
      for (int f = 0; f < F; ++f) {
        a[ks][f] = __builtin_bit_cast(bf16x8_mfma, *(const uint4*)(sp + abase + f * 16 * V2_ROWB + off));
        b[ks][f] = __builtin_bit_cast(bf16x8_mfma, *(const uint4*)(sp + bbase + f * 16 * V2_ROWB + off));
      }
    }
    if (OWN && (kt + 1) * V2_BK > g.Kt) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        if (kt * V2_BK + ks * 32 + fg * 8 >= g.Kt) {
#pragma unroll
          for (int f = 0; f < F; ++f) a[ks][f] = b[ks][f] = __builtin_bit_cast(bf16x8_mfma, u32x4{0, 0, 0, 0});
        }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ks][i], b[ks][j], acc[i][j], 0, 0, 0);
      if (ks == 0 && kt == kdiag) {
        // cin(i, j) = b(j, i): row j of the b panel, k offset of row i
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < F; ++j) {
            const int k = koff + i * 16 + fg * 4;
            const uint2 w = *(const uint2*)(sp + bbase + (j * 16 + fr) * V2_ROWB +
                                            (((k >> 3) ^ kswz(fr)) << 4) + (k & 7) * 2);
            acc[i][j][0] += ratio * __uint_as_float(w.x << 16);
            acc[i][j][1] += ratio * __uint_as_float(w.x & 0xffff0000u);
            acc[i][j][2] += ratio * __uint_as_float(w.y << 16);
            acc[i][j][3] += ratio * __uint_as_float(w.y & 0xffff0000u);
          }
      }
    }
    st = st + 1 == C::NS ? 0 : st + 1;
  }
  wait_vmcnt0();
  lds_barrier();

  // epilogue: accumulator (i, j) element q is C(16 i + 4 fg + q, 16 j + fr) of the wave's block.
  // The tile goes through LDS transposed (the mirror half, whole rows of the output; 4
  // consecutive rows of one column per lane) and then row-major.
  bf16_t* T = (bf16_t*)smem;
  bf16_t* out = (bf16_t*)g.out + (int64_t)bidx * g.so;
  const int mv = (int)g.Mv;
  uint32_t hv[F][F][2];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int r = row0 + wm * WM + i * 16 + fg * 4 + 2 * h, c = col0 + wn * WM + j * 16 + fr;
        const f2x v = {alpha * acc[i][j][2 * h], alpha * acc[i][j][2 * h + 1]};
        const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf2x));
        // zeros outside the valid extent, so that the padding stays zero
        hv[i][j][h] = w & ((c < mv && r < mv ? 0x0000ffffu : 0u) | (c < mv && r + 1 < mv ? 0xffff0000u : 0u));
      }
  constexpr int CH = TM / 8, ROWS = 256 / CH;  // 16-byte chunks per row, rows per store
  // eight elements of output row r from column c on (OWN: those inside it)
  const bool whole = !OWN || (g.ldo % 8 == 0 && !((uintptr_t)g.out & 15));
  auto put = [&](int r, int c, uint4 w) {
    bf16_t* o = out + (int64_t)r * g.ldo + c;
    if (!OWN || (whole && r < mv && c + 8 <= mv)) {
      *(uint4*)o = w;
    } else if (r < mv) {
      const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (c + e < mv) o[e] = (bf16_t)(u[e >> 1] >> (16 * (e & 1)));
    }
  };
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
      *(uint2*)(T + (wn * WM + j * 16 + fr) * C::PITCH + wm * WM + i * 16 + fg * 4) =
          make_uint2(hv[i][j][0], hv[i][j][1]);
  lds_barrier();
  if (!diag) {
#pragma unroll
    for (int it = 0; it < TM / ROWS; ++it) {
      const int jl = it * ROWS + tid / CH, c = tid % CH * 8;
      put(col0 + jl, row0 + c, *(const uint4*)(T + jl * C::PITCH + c));
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int j = 0; j < F; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          T[(wm * WM + i * 16 + fg * 4 + q) * C::PITCH + wn * WM + j * 16 + fr] =
              (bf16_t)(hv[i][j][q >> 1] >> (16 * (q & 1)));
    lds_barrier();
  }
  // (a diagonal tile stays transposed: row il of the output takes, at column c, the upper
  // element, (min, max) of its indices, which the stage holds at [max][min])
#pragma unroll
  for (int it = 0; it < TM / ROWS; ++it) {
    const int il = it * ROWS + tid / CH, c = tid % CH * 8;
    uint4 w;
    if (!diag) {
      w = *(const uint4*)(T + il * C::PITCH + c);
    } else {
      uint16_t e[8];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        e[q] = c + q > il ? T[(c + q) * C::PITCH + il] : T[il * C::PITCH + c + q];
      __builtin_memcpy(&w, e, 16);
    }
    put(row0 + il, col0 + c, w);
  }
}

// X' = alpha (B X + ratio X). PDT < 0: X' stored. PDT >= 0 (the last iteration): each element of
// X', rounded to bf16, is the update of one parameter element of type PDT, applied as the
// post-pass does (apply_elem) and the parameter written back; SW (tall parameters: their rows
// are columns of X') swaps the MFMA operands, so that the staged tile is the parameter's.
// Accumulator (i, j) element q is X'(16 i + fr, 16 j + 4 fg + q) of the wave's block, with SW
// X'(16 i + 4 fg + q, 16 j + fr).
template <int TM, int PDT, bool SW, typename Args>
__global__ __launch_bounds__(256, 2) void tile_bx_kernel(Args args, MuonApply ap) {
  typedef TileK<TM> C;
  constexpr int F = C::F, WM = TM / 2, XR = TM * 2, XCH = XR / 16;  // X panel: 64 rows of XR bytes
  extern __shared__ __align__(16) uint8_t smem[];
  int bidx, tm, tn;
  const GemmArgs& g = args_of(args, MODE_GEMM, bidx, tm, tn);
  const int row0 = tm * TM, col0 = tn * TM;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const bf16_t* A = (const bf16_t*)g.a + (int64_t)bidx * g.sa + (int64_t)row0 * g.lda;
  const bf16_t* X = (const bf16_t*)g.b + (int64_t)bidx * g.sb + col0;
  const u32x4 rsa = n4_rsrc(A, false), rsx = n4_rsrc(X, false), rs_none = n4_rsrc(A, true);
  const int lda_b = (int)(g.lda * 2), ldx_b = (int)(g.ldb * 2);
  const int r_in = wave * 8 + (lane >> 3);
  const int voa = r_in * lda_b + (((lane & 7) ^ kswz(r_in)) << 4);
  // X panel rows k: chunk c of row k at c ^ xsw(k). A transposing read takes 4 rows of 32 bytes for
  // 16 lanes, and the next 16 lanes 4 rows eight further: xsw puts the eight in different
  // 32-byte groups of the 64 banks.
  auto xsw = [](int k) {
    return TM == 128 ? ((k & 3) << 2) | (((k >> 3) & 1) << 1) : (((k >> 1) & 1) | (((k >> 3) & 1) << 1)) << 1;
  };
  const int x_in = wave * (1024 / XR) + lane / XCH;
  const int vox = x_in * ldx_b + (((lane % XCH) ^ xsw(x_in)) << 4);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  const int KT = (int)(g.K / V2_BK);
  auto issue = [&](int kt, int st) {
    const bool on = kt < KT;
    const int kk = on ? kt : 0;
    const uint32_t m0 = lds0 + st * C::STAGEB + wave * 1024;
    const u32x4 pa = on ? rsa : rs_none, px = on ? rsx : rs_none;
#pragma unroll
    for (int q = 0; q < C::LOADS; ++q) {
      lds_dma(voa, pa, kk * V2_ROWB + q * 32 * lda_b, m0 + q * 4096);
      lds_dma(vox, px, (kk * V2_BK + q * (4096 / XR)) * ldx_b, m0 + C::PANELB + q * 4096);
    }
  };
  float alpha = g.alpha, beta = g.beta;
  if (g.scale_mode == 1) {
    const float s = g.scale[bidx];
    alpha *= s;
    beta *= s;
  }
  const float ratio = beta != 0.0f ? beta / alpha : 0.0f;
  // 32-k step whose rows of X are this wave's output rows (F / 2 of them from here on)
  const int sdiag = ratio != 0.0f ? (row0 + wm * WM) / 32 : -2 * F;

  f32x4 acc[F][F];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int fr = lane & 15, fg = lane >> 4;
  auto mma = [&](const bf16x8_mfma& b, const bf16x8_mfma& x, f32x4& c) {
    c = SW ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, x, c, 0, 0, 0)
           : __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, b, c, 0, 0, 0);
  };
#pragma unroll
  for (int t = 0; t < C::NS - 1; ++t) issue(t, t);
  int st = 0;
  for (int kt = 0; kt < KT; ++kt) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(2 * C::LOADS * (C::NS - 2)) : "memory");
    lds_barrier();
    issue(kt + C::NS - 1, st == 0 ? C::NS - 1 : st - 1);
    const uint8_t* sp = smem + st * C::STAGEB;
    uint8_t* xp = smem + st * C::STAGEB + C::PANELB;
    bf16x8_mfma b[2][F], x[2][F];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int off = (wm * WM + fr) * V2_ROWB + (((ks * 4 + fg) ^ kswz(fr)) << 4);
      const int k = 32 * ks + 8 * fg + (fr >> 2);
#pragma unroll
      for (int f = 0; f < F; ++f) {
        b[ks][f] = __builtin_bit_cast(bf16x8_mfma, *(const uint4*)(sp + f * 16 * V2_ROWB + off));
        const int c = (wn * WM + f * 16) / 8 + ((fr & 3) >> 1);
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(xp + k * XR + ((c ^ xsw(k)) << 4) + (fr & 1) * 8));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) i16x4*)(xp + (k + 4) * XR + ((c ^ xsw(k + 4)) << 4) + (fr & 1) * 8));
        x[ks][f] = __builtin_bit_cast(bf16x8_mfma, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) mma(b[ks][i], x[ks][j], acc[i][j]);
      const int sd = 2 * kt + ks - sdiag;
      if (sd >= 0 && sd < F / 2) {
        bf16x8_mfma db[2][2], d3[2][2];
        n16_beta_frags(ratio, lane, db);
        n16_beta_third(ratio, lane, d3);
#pragma unroll
        for (int f = 0; f < F / 2; ++f)
          if (sd == f) {
#pragma unroll
            for (int part = 0; part < 2; ++part)
#pragma unroll
              for (int par = 0; par < 2; ++par)
#pragma unroll
                for (int j = 0; j < F; ++j) mma(db[par][part], x[ks][j], acc[2 * f + par][j]);
            if (g.K < BETA3_K) {
#pragma unroll
              for (int par = 0; par < 2; ++par)
#pragma unroll
                for (int j = 0; j < F; ++j) mma(d3[par][0], x[ks][j], acc[2 * f + par][j]);
            }
          }
      }
    }
    st = st + 1 == C::NS ? 0 : st + 1;
  }
  wait_vmcnt0();
  lds_barrier();

  // epilogue: rows of the staged tile are X' rows (SW: X' columns), 4 consecutive elements of
  // one row per lane
  bf16_t* T = (bf16_t*)smem;
  const int mv = (int)g.Mv, nv = (int)g.Nv;
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const f2x v01 = {alpha * acc[i][j][0], alpha * acc[i][j][1]};
      const f2x v23 = {alpha * acc[i][j][2], alpha * acc[i][j][3]};
      uint32_t w0 = __builtin_bit_cast(uint32_t, __builtin_convertvector(v01, bf2x));
      uint32_t w1 = __builtin_bit_cast(uint32_t, __builtin_convertvector(v23, bf2x));
      const int ri = wm * WM + i * 16, cj = wn * WM + j * 16;
      if constexpr (PDT < 0) {
        // zeros outside the valid extent, so that the padding stays zero
        const int r = row0 + ri + fr, c = col0 + cj + 4 * fg;
        w0 &= (r < mv && c < nv ? 0x0000ffffu : 0u) | (r < mv && c + 1 < nv ? 0xffff0000u : 0u);
        w1 &= (r < mv && c + 2 < nv ? 0x0000ffffu : 0u) | (r < mv && c + 3 < nv ? 0xffff0000u : 0u);
      }
      bf16_t* pos = SW ? T + (cj + fr) * C::PITCH + ri + 4 * fg : T + (ri + fr) * C::PITCH + cj + 4 * fg;
      *(uint2*)pos = make_uint2(w0, w1);
    }
  lds_barrier();
  constexpr int CH = TM / 8, ROWS = 256 / CH;
  if constexpr (PDT < 0) {
    bf16_t* out = (bf16_t*)g.out + (int64_t)bidx * g.so;
#pragma unroll
    for (int it = 0; it < TM / ROWS; ++it) {
      const int il = it * ROWS + tid / CH, c = tid % CH * 8;
      *(uint4*)(out + (int64_t)(row0 + il) * g.ldo + col0 + c) = *(const uint4*)(T + il * C::PITCH + c);
    }
  } else {
    // matrix bidx of the group is matrix bidx % nb of its tensor t0 + bidx / nb
    const int t = g.t0 + bidx / g.nb;
    const int64_t mb = bidx % g.nb;
    const float adj = ap.adj[t];
    const int prows = SW ? nv : mv, pcols = SW ? mv : nv;
    const int pr0 = SW ? col0 : row0, pc0 = SW ? row0 : col0;
    void* prm = ap.params[t];
    const int64_t base = mb * (int64_t)prows * pcols;
    Raw8<PDT> pv[TM / ROWS];
#pragma unroll
    for (int it = 0; it < TM / ROWS; ++it) {
      const int r = pr0 + it * ROWS + tid / CH, c = pc0 + tid % CH * 8;
      if (r < prows && c < pcols) pv[it].load(prm, base + (int64_t)r * pcols + c);
    }
#pragma unroll
    for (int it = 0; it < TM / ROWS; ++it) {
      const int il = it * ROWS + tid / CH, cl = tid % CH * 8;
      const int r = pr0 + il, c = pc0 + cl;
      if (r >= prows || c >= pcols) continue;
      float p[8], u[8];
      pv[it].unpack(p);
      Vec8<MUON_DT_BF16>::load(T + il * C::PITCH + cl, 0, u);
#pragma unroll
      for (int e = 0; e < 8; ++e) p[e] = apply_elem<PDT, MUON_DT_BF16>(p[e], u[e], ap.wd, ap.cautious, adj);
      pv[it].pack(p);
      pv[it].store(prm, base + (int64_t)r * pcols + c);
    }
  }
}

// Wave grid of the register-staged bf16 kernel (gemm_bf16_kernel), which serves the
// masked gram_ path and SYRKs whose beta term has no alpha to fold into: 4 x 2
// wavefronts, each 64 x 128, two waves per SIMD.
#ifndef MUON_BF16_WGM
#define MUON_BF16_WGM 4
#endif
#ifndef MUON_BF16_WGN
#define MUON_BF16_WGN 2
#endif
constexpr int BF_WGM = MUON_BF16_WGM, BF_WGN = MUON_BF16_WGN;
constexpr int BF_NT = 64 * BF_WGM * BF_WGN;

// The product kernels need more than the default 64 KiB of dynamic LDS; raise the
// per-kernel limit once per process for every instantiation.
int reserve_lds() {
  static int status = -1;
  static std::once_flag once;
  std::call_once(once, [] {
    const void* ks[2] = {(const void*)gemm_bf16_kernel<MODE_SYRK, false, BF_WGM, BF_WGN>,
                         (const void*)gemm_bf16_kernel<MODE_SYRK, true, BF_WGM, BF_WGN>};
    status = 0;
    for (const void* k : ks)
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, BF_SMEM) !=
          hipSuccess)
        status = -1;
    if (hipFuncSetAttribute((const void*)gemm_bf16_v2_kernel<MODE_SYRK, true>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, v2_smem(true)) !=
        hipSuccess)
      status = -1;
    if (hipFuncSetAttribute((const void*)gemm_bf16_s16_kernel,
                            hipFuncAttributeMaxDynamicSharedMemorySize, V2_SMEM) != hipSuccess)
      status = -1;
    if (hipFuncSetAttribute((const void*)gemm_bf16_s16h_kernel<GemmArgs>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, H_SMEM) != hipSuccess)
      status = -1;
    const void* n16[14] = {
#define N16_ALL(B3)                                                                           \
  (const void*)gemm_bf16_nn16_kernel<0, 0, B3>, (const void*)gemm_bf16_nn16_kernel<1, 0, B3>, \
      (const void*)gemm_bf16_nn16_kernel<1, 1, B3>, (const void*)gemm_bf16_nn16_kernel<1, 2, B3>, \
      (const void*)gemm_bf16_nn16_kernel<2, 0, B3>, (const void*)gemm_bf16_nn16_kernel<2, 1, B3>, \
      (const void*)gemm_bf16_nn16_kernel<2, 2, B3>
        N16_ALL(false), N16_ALL(true)
#undef N16_ALL
    };
    for (const void* k : n16)
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, N4_SMEM) !=
          hipSuccess)
        status = -1;
    const void* f32[3] = {(const void*)gemm_f32_kernel<MODE_SYRK>,
                          (const void*)gemm_f32_kernel<MODE_GEMM>,
                          (const void*)gemm_f32_kernel<MODE_SYRK, true>};
    for (const void* k : f32)
      if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, F_SMEM) !=
          hipSuccess)
        status = -1;
  });
  return status;
}

// Compute units of the current device (the persistent kernel's grid), cached per device.
int device_cus() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 256;
  if (dev < 64) {
    const int c = cache[dev].load(std::memory_order_relaxed);
    if (c > 0) return c;
  }
  int n = 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    n = 256;
  if (dev < 64) cache[dev].store(n, std::memory_order_relaxed);
  return n;
}

// Workgroups of a persistent launch over `blocks` tiles: as many rounds as one workgroup per
// CU needs, with the tiles spread evenly over them (a launch of a few hundred tiles leaves
// the CUs it does not need to kernels on other streams instead of idling them in its last
// round). Unchanged when the tile count is a multiple of the CU count.
static int persistent_wgs(int64_t blocks) {
  const int64_t cus = device_cus();
  if (blocks <= cus) return (int)blocks;
  const int64_t rounds = (blocks + cus - 1) / cus;
  return (int)((blocks + rounds - 1) / rounds);
}

// Tile size of a SYRK (256, 128 or 64 rows) and of a B X launch, by the time each would take: the
// kernels give the same bits. TileCost holds what a launch of one kernel takes in microseconds: up
// to one workgroup per CU `one` + `one_k` per k; beyond, `base` plus, for each round of
// workgroups over the CUs, `wave` + `wave_k` per k, where a last round that is partly filled counts
// the share `whole` as a full one (two workgroups share a CU on 128- and 64-row tiles, so there the
// others go on meanwhile). 256-row tiles have a long prologue and epilogue and the most reuse, 64-row
// tiles the shortest chain; the padding beyond round_up(m, 128) rows is only computed by 256-row tiles.
// Fitted to launches as they follow each other in 1178 iterations (1 to 300 matrices of 65 to 4096
// rows, up to 16384 columns) and 1978 Gram products (256 to 4096 rows, K from 128 to 8192), each on
// all three sizes; a launch is 5 to 11% from its cost (root mean square), and the size chosen
// is on average 0.6% (SYRK) and 0.4% (B X) slower than the best of the three.
// Measured (us, 256 / 128 / 64, between events): X X^T of 1 x 128 x 256 27 / 11 / 7, of 16 x 768 x 768 38 /
// 21 / 22, of 24 x 768 x 3072 82 / 53 / 88, of 4 x 4096 x 4096 276 / 294 / 587; B X of the same 15 / 8.9 / 7.4,
// 26 / 29 / 36, 93 / 111 / 183 and 386 / 538 / 896.
struct TileCost {
  double one, one_k, base, wave, wave_k, whole;
};
constexpr TileCost SYRK_256 = {22.4, 0.0162, 7.4, 13.0, 0.0220, 0.5};
constexpr TileCost SYRK_PACKED = {19.9, 0.0239, 20.0, 10.0, 0.0254, 0.5};  // gemm_bf16_v2_kernel
constexpr TileCost SYRK_128 = {6.8, 0.0081, 5.8, 2.35, 0.0068, 0.5};
constexpr TileCost SYRK_64 = {4.7, 0.0033, 3.5, 1.0, 0.0028, 0.7};
constexpr TileCost BX_256 = {16.7, 0.0213, 14.5, 6.0, 0.0216, 0.6};
constexpr TileCost BX_128 = {6.1, 0.0099, 3.1, 2.35, 0.0068, 0.8};
constexpr TileCost BX_64 = {4.9, 0.0046, 3.6, 1.1, 0.0029, 1.0};

static double tile_cost(const TileCost& c, int64_t tiles, double k) {
  const int64_t cus = device_cus(), rounds = (tiles + cus - 1) / cus;
  if (rounds <= 1) return c.one + c.one_k * k;
  const double w = c.whole * (double)rounds + (1.0 - c.whole) * (double)tiles / (double)cus;
  return c.base + w * (c.wave + c.wave_k * k);
}

// Tiles of k on average, kmax at most (several buckets in one launch): the longest takes its time.
static double tile_cost(const TileCost& c, int64_t tiles, double k, double kmax) {
  return std::max(c.one + c.one_k * kmax, tile_cost(c, tiles, k));
}

// Data beyond what the last cache (256 MB) keeps: the smaller tiles' further reads of their operands then
// compete with the result's way to memory. For a Gram product its operand and result count
// (32 x 2048 x 1024 takes 180 us on 256-row tiles and 198 on 128-row ones, 9 x 2048 x 2048 96 and 78), in
// an iteration X, X', A and B (24 x 2048 x 2048: 209 and 251).
static bool past_cache(int64_t bytes) { return bytes > ((int64_t)240 << 20); }

// B X on 256-row tiles is persistent: a workgroup count that is no multiple of the 8 XCDs spreads a
// round's tiles unevenly over their L2s (two rounds of 130 to 250 workgroups take 1.3 times those of
// a multiple of 8, three 1.2 times).
static double bx256_cost(int64_t tiles, double k) {
  const int64_t cus = device_cus(), rounds = (tiles + cus - 1) / cus;
  const bool uneven = rounds > 1 && persistent_wgs(tiles) % 8 != 0;
  return tile_cost(BX_256, tiles, k) * (uneven ? 1.0 + 0.6 / (double)rounds : 1.0);
}

// What a SYRK on 128- or 64-row tiles takes more where the L2s do not hold a matrix and its rows are
// read again from the last cache: 2240 rows, K 8108 (36 MB) takes 150 / 85 / 114 us on 256- / 128- /
// 64-row tiles, 4096 rows, K 4096 (32 MB) 78 / 93 / 159.
static double far_rows(int tm, int64_t tiles, double k, int64_t rows) {
  const double mb = (double)rows * k * 2.0 / (1 << 20);
  if (mb <= 2.0 || (tm == 64 && tiles <= device_cus())) return 1.0;
  return 1.0 + (tm == 64 ? 0.01 : 0.0025) * (mb - 2.0);
}
static double syrk_cost(int tm, int64_t tiles, double k, int64_t rows) {
  return tile_cost(tm == 64 ? SYRK_64 : SYRK_128, tiles, k) * far_rows(tm, tiles, k, rows);
}

// Costs within 5 or 6% of each other are ties and go to the larger tiles, which read less; a cut of
// long sums (K from 4096 on, where the two launches' ends weigh little) takes what it is thought to.
// beside: the launch shares the device with other streams' (a step's small buckets). The larger
// tiles then win over a wider range, since what the launch takes from its neighbours counts, not its
// own time (four matrices of 2048 x 2048 and two of 8192 x 2048, 128-row SYRK tiles for the former
// 2% shorter alone: 1.95 ms a step with them, 1.87 without; one fp32 matrix of 1022 x 1984 and one of
// 1022 x 1022 beside nine of 1984 x 1022: 780 us with B X of the two on 64-row tiles, 772 on 128).
//
// head > 0: the first `head` tiles (whole rounds) on 256-row tiles, the rest, which would leave most
// CUs idle for a round, cut into tm-row tiles in a second launch (8 us for its fill and the first
// one's drain). Eight matrices of 4096 rows are 4.25 rounds, four 2.125, two 1.06: the Gram launches
// of a step on four layers of a 4096-wide model (28 matrices) went from 23.7 to 21.0 ms, the step
// from 51.7 to 50.1 ms, on one layer from 13.5 to 12.5 ms. Over 936 products of more than a round
// the choice is 0.8% slower on average than the best form of each, and 1.4% if none is cut.
struct SyrkPlan {
  int tm;
  int64_t head;
};
static SyrkPlan syrk_plan(int64_t batch, int64_t m, int64_t K, int64_t blocks256, bool packed,
                          bool past, int beside) {
  const int64_t rows = round_up(m, 128), t1 = rows / 128, t2 = 2 * t1, cus = device_cus();
  const int64_t n128 = t1 * (t1 + 1) / 2 * batch, n64 = t2 * (t2 + 1) / 2 * batch;
  const double k = (double)K, far = past ? 1.07 : 1.0;
  const double c256 = tile_cost(packed ? SYRK_PACKED : SYRK_256, blocks256, k);
  const double c128 = far * syrk_cost(128, n128, k, rows), c64 = far * syrk_cost(64, n64, k, rows);
  SyrkPlan best = {256, 0};
  double cost = c256;
  const double tie = beside ? 0.65 : n64 > cus && K >= 2048 ? 0.95 : 1.0;
  if (c64 < tie * c128 && c64 < c256) best.tm = 64, cost = c64;
  else if (c128 < (beside ? 0.75 : 0.94) * c256) best.tm = 128, cost = c128;
  const int64_t head = blocks256 / cus * cus, rest = blocks256 - head;
  if (!packed && head > 0 && rest > 0) {
    const double r128 = tile_cost(SYRK_128, 4 * rest, k), r64 = tile_cost(SYRK_64, 16 * rest, k);
    if (tile_cost(SYRK_256, head, k) + 8.0 + std::min(r128, r64) <
        (K >= 4096 ? 0.98 : 0.94) * cost)
      best = {r64 < r128 ? 64 : 128, head};
  }
  return best;
}

static int bx_tile(int64_t batch, int64_t M, int64_t N, int64_t K, int64_t m, int beside) {
  const int64_t rows = round_up(m, 128);
  const int64_t n256 = (M / 256) * (N / 256) * batch, n128 = rows / 128 * (N / 128) * batch;
  const double k = (double)K, far = past_cache(batch * rows * (N + rows) * 4) ? 1.08 : 1.0;
  const double c256 = bx256_cost(n256, k), c128 = far * tile_cost(BX_128, n128, k),
               c64 = far * tile_cost(BX_64, 4 * n128, k);
  if (c64 < (beside ? 0.65 : 0.95) * c128 && c64 < c256) return 64;
  return c128 < (beside ? 0.5 : 1.0) * c256 ? 128 : 256;
}

// `g` on TM-row tiles covering round_up(m, 128) rows (of a SYRK, columns too).
static GemmArgs on_tiles(const GemmArgs& g, int mode, int TM, int64_t m, int64_t N, int64_t batch) {
  GemmArgs t = g;
  t.tiles_m = (int)(round_up(m, 128) / TM);
  t.tiles_n = (int)(mode == MODE_SYRK ? t.tiles_m : N / TM);
  t.tiles_per_batch = mode == MODE_SYRK ? t.tiles_m * (t.tiles_m + 1) / 2 : t.tiles_m * t.tiles_n;
  t.tiles_total = (int)(t.tiles_per_batch * batch);
  return t;
}

}  // namespace

// Launch one batched product. `dtype` selects bf16 (256-, 128- or 64-row tiles) or fp32 (64-row
// tiles; gram_ of rows that are no whole 16-byte chunks 128). M/N are the (padded) output extents;
// they must be multiples of 256 (fp32: 128) unless `masked`. SYRK: a and b are the same K-contiguous rows. GEMM (NN): b is the
// K x N row-major operand (row pitch ldb) and the beta term reads cin = b's first
// M rows (cin(i, j) = b(i, j), true of X' = a X + B X); the bf16 kernels take it from
// the staged operand panels. Masked (arbitrary-extent) launches exist for SYRK only.
int muon_launch_gemm(int dtype, int mode, bool masked, int64_t batch, int64_t M, int64_t N,
                     int64_t K, const void* a, int64_t lda, int64_t sa, const void* b,
                     int64_t ldb, int64_t sb, const void* cin, int64_t ldc, int64_t sc,
                     void* out, int64_t ldo, int64_t so, void* out_t, int64_t ldt, int64_t st,
                     int64_t Mv, int64_t Nv, float alpha, float beta, const float* scale,
                     int scale_mode, int beside, hipStream_t stream) {
  GemmArgs g;
  g.a = a;
  g.b = b;
  g.cin = cin;
  g.out = out;
  g.out_t = out_t;
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldc;
  g.ldo = ldo;
  g.ldt = ldt;
  g.sa = sa;
  g.sb = sb;
  g.sc = sc;
  g.so = so;
  g.st = st;
  g.Mv = Mv;
  g.Nv = Nv;
  g.Mt = M;
  g.Nt = N;
  g.Kt = K;
  g.alpha = alpha;
  g.beta = beta;
  g.scale = scale;
  g.scale_mode = scale_mode;
  g.store_out = out != nullptr;
  g.store_out_t = out_t != nullptr;
  const int bm = dtype == MUON_DT_BF16 ? BF_BM : F_BM;
  const int bk = dtype == MUON_DT_BF16 ? BF_BK : (masked ? F_BK : 64);
  g.tiles_m = (int)((M + bm - 1) / bm);
  g.tiles_n = (int)((N + bm - 1) / bm);
  g.K = masked ? round_up(K, bk) : K;
  if (!masked && (M % bm || N % bm || K % bk)) {
    muon_set_error("gemm: unmasked extents (%lld, %lld, %lld) not tile multiples", (long long)M,
                   (long long)N, (long long)K);
    return MUON_ERR_SHAPE;
  }
  if (masked && mode != MODE_SYRK) {
    muon_set_error("gemm: masked launches are SYRK only");
    return MUON_ERR_ARG;
  }
  // the bf16 kernels address one matrix's operands with 32-bit byte offsets
  const int64_t es = dtype == MUON_DT_BF16 ? 2 : 4;
  if (std::max(M * lda, (mode == MODE_SYRK ? M : K) * ldb) * es >= (int64_t)0x7fffffff) {
    muon_set_error("gemm: operand of %lld x %lld elements exceeds the 2 GiB per-matrix limit",
                   (long long)std::max(M, K), (long long)std::max(lda, ldb));
    return MUON_ERR_SHAPE;
  }
  if (mode == MODE_SYRK)
    g.tiles_per_batch = g.tiles_m * (g.tiles_m + 1) / 2;
  else
    g.tiles_per_batch = g.tiles_m * g.tiles_n;
  const int64_t blocks = (int64_t)g.tiles_per_batch * batch;
  if (blocks == 0) return MUON_OK;
  g.tiles_total = (int)std::min<int64_t>(blocks, 0x7fffffffLL);
  if (blocks > 0x7fffffffLL) {
    muon_set_error("gemm: grid too large (%lld workgroups)", (long long)blocks);
    return MUON_ERR_SHAPE;
  }
  dim3 grid((unsigned)blocks), block(256);
  if (reserve_lds() != 0) {
    muon_set_error("gemm: cannot reserve %d B of LDS", BF_SMEM);
    return MUON_ERR_LAUNCH;
  }
  if (dtype == MUON_DT_BF16) {
#define LAUNCH_BF(MODE_, MASK_)                                                        \
  do {                                                                                 \
    hipLaunchKernelGGL((gemm_bf16_kernel<MODE_, MASK_, BF_WGM, BF_WGN>), grid, dim3(BF_NT), \
                       BF_SMEM, stream, g);                                                \
  } while (0)
    if (mode == MODE_GEMM) {
      if (alpha == 0.0f) {
        muon_set_error("gemm: alpha must be nonzero");
        return MUON_ERR_ARG;
      }
      if (out_t != nullptr || K % 128 != 0) {
        muon_set_error("gemm: bf16 NN products take K a multiple of 128 and no transposed output");
        return MUON_ERR_ARG;
      }
      MuonApply none;
      none.nb = 1;
      const int TM = bx_tile(batch, M, N, K, Mv, beside);
      if (TM == 256) {
        // persistent: at most one workgroup per CU walks the tile list
        const dim3 pg((unsigned)persistent_wgs(blocks));
        if (K < BETA3_K)
          hipLaunchKernelGGL((gemm_bf16_nn16_kernel<0, 0, true>), pg, dim3(256), N4_SMEM, stream, g, none);
        else
          hipLaunchKernelGGL(gemm_bf16_nn16_kernel<0>, pg, dim3(256), N4_SMEM, stream, g, none);
      } else {
        const GemmArgs gt = on_tiles(g, mode, TM, Mv, N, batch);
        const dim3 tg((unsigned)gt.tiles_total);
        if (TM == 128)
          hipLaunchKernelGGL((tile_bx_kernel<128, -1, false, GemmArgs>), tg, dim3(256),
                             TileK<128>::SMEM, stream, gt, none);
        else
          hipLaunchKernelGGL((tile_bx_kernel<64, -1, false, GemmArgs>), tg, dim3(256),
                             TileK<64>::SMEM, stream, gt, none);
      }
    } else if (!masked && (alpha != 0.0f || beta == 0.0f)) {
      // the last 128 rows padding only: the last tile column's real unit in packed tiles,
      // in the same launch as the full tiles
      const int T = g.tiles_m;
      GemmArgs gp = g;
      const bool packed = T >= 2 && Mv <= M - 128 && Nv == Mv;
      if (packed) {
        gp.tiles_per_batch = (T - 1) * T / 2 + (2 * T - 1 + 3) / 4;
        gp.tiles_total = gp.tiles_per_batch * (int)batch;
      }
      // (A A's operands are a small part of an iteration's data)
      const bool past = beta == 0.0f && past_cache(batch * M * (K + M) * (scale ? 4 : 2));
      const SyrkPlan plan = syrk_plan(batch, Mv, K, gp.tiles_total, packed, past, beside);
      const int TM = plan.tm;
      if (plan.head > 0) {
        hipLaunchKernelGGL(gemm_bf16_s16_kernel, dim3((unsigned)plan.head), dim3(512), V2_SMEM,
                           stream, g);
        const int split = 256 / TM;
        const GemmTail tail = {g, (int)plan.head, split};
        const dim3 tg((unsigned)((blocks - plan.head) * split * split));
        if (TM == 128)
          hipLaunchKernelGGL((gemm_bf16_s16h_kernel<GemmTail>), tg, dim3(256), H_SMEM, stream, tail);
        else
          hipLaunchKernelGGL((tile_syrk_kernel<64, GemmTail>), tg, dim3(256), TileK<64>::SMEM, stream,
                             tail);
      } else if (TM != 256) {
        const GemmArgs gt = on_tiles(g, mode, TM, Mv, N, batch);
        const dim3 tg((unsigned)gt.tiles_total);
        if (TM == 128)
          hipLaunchKernelGGL((gemm_bf16_s16h_kernel<GemmArgs>), tg, dim3(256), H_SMEM, stream, gt);
        else
          hipLaunchKernelGGL((tile_syrk_kernel<64, GemmArgs>), tg, dim3(256), TileK<64>::SMEM, stream,
                             gt);
      } else if (packed) {
        hipLaunchKernelGGL((gemm_bf16_v2_kernel<MODE_SYRK, true>),
                           dim3((unsigned)gp.tiles_total), dim3(512), v2_smem(true), stream, gp);
      } else {
        // full tiles only: the 16 x 16 x 32 MFMA kernel
        hipLaunchKernelGGL(gemm_bf16_s16_kernel, grid, dim3(512), V2_SMEM, stream, g);
      }
    } else if (masked && K % 8 == 0 && !((uintptr_t)a & 15)) {
      // gram_ of any extents, rows of whole 16-byte chunks
      const int64_t t1 = (M + 127) / 128, t2 = (M + 63) / 64;
      const int TM = syrk_cost(64, t2 * (t2 + 1) / 2 * batch, (double)K, M) <
                             syrk_cost(128, t1 * (t1 + 1) / 2 * batch, (double)K, M) ? 64 : 128;
      GemmArgs gt = g;
      gt.tiles_m = gt.tiles_n = (int)((M + TM - 1) / TM);
      gt.tiles_per_batch = gt.tiles_m * (gt.tiles_m + 1) / 2;
      const int64_t bt = (int64_t)gt.tiles_per_batch * batch;
      if (bt > 0x7fffffffLL) {
        muon_set_error("gemm: grid too large (%lld workgroups)", (long long)bt);
        return MUON_ERR_SHAPE;
      }
      gt.tiles_total = (int)bt;
      if (TM == 64)
        hipLaunchKernelGGL((tile_syrk_kernel<64, GemmArgs, true>), dim3((unsigned)bt), dim3(256),
                           TileK<64>::SMEM, stream, gt);
      else
        hipLaunchKernelGGL((tile_syrk_kernel<128, GemmArgs, true>), dim3((unsigned)bt), dim3(256),
                           TileK<128>::SMEM, stream, gt);
    } else {
      if (masked) LAUNCH_BF(MODE_SYRK, true); else LAUNCH_BF(MODE_SYRK, false);
    }
#undef LAUNCH_BF
  } else if (dtype == MUON_DT_F32) {
    if (masked && (K % 4 || ((uintptr_t)a & 15))) {
      hipLaunchKernelGGL(gemm_f32_masked_kernel, grid, block, 0, stream, g);
    } else if (masked) {
      GemmArgs gh = g;
      gh.tiles_m = gh.tiles_n = (int)((M + F_TM - 1) / F_TM);
      gh.tiles_per_batch = gh.tiles_m * (gh.tiles_m + 1) / 2;
      const int64_t bh = (int64_t)gh.tiles_per_batch * batch;
      if (bh > 0x7fffffffLL) {
        muon_set_error("gemm: grid too large (%lld workgroups)", (long long)bh);
        return MUON_ERR_SHAPE;
      }
      hipLaunchKernelGGL((gemm_f32_kernel<MODE_SYRK, true>), dim3((unsigned)bh), dim3(512), F_SMEM,
                         stream, gh);
    } else {
      GemmArgs gh = g;  // 64-row tiles
      gh.tiles_m = (int)(M / F_TM);
      gh.tiles_n = (int)(N / F_TM);
      gh.tiles_per_batch = mode == MODE_SYRK ? gh.tiles_m * (gh.tiles_m + 1) / 2
                                             : gh.tiles_m * gh.tiles_n;
      const int64_t bh = (int64_t)gh.tiles_per_batch * batch;
      if (bh > 0x7fffffffLL) {
        muon_set_error("gemm: grid too large (%lld workgroups)", (long long)bh);
        return MUON_ERR_SHAPE;
      }
      if (mode == MODE_SYRK)
        hipLaunchKernelGGL((gemm_f32_kernel<MODE_SYRK>), dim3((unsigned)bh), dim3(512), F_SMEM,
                           stream, gh);
      else
        hipLaunchKernelGGL((gemm_f32_kernel<MODE_GEMM>), dim3((unsigned)bh), dim3(512), F_SMEM,
                           stream, gh);
    }
  } else {
    muon_set_error("gemm: unsupported dtype %d", dtype);
    return MUON_ERR_DTYPE;
  }
  MUON_CHECK_LAUNCH("gemm");
  return MUON_OK;
}

// Whether the apply of `batch` matrices' last B X is fused for parameters of type pdt: bf16 ones
// always (the 256-row kernel has the epilogue), others where the launch on 128- or 64-row
// tiles costs less than the 256-row one and a post-pass (which reads U and the parameters
// and writes the parameters, about 5 TB/s). Six fp32
// matrices of 768 x 3072: 26 us and 29 us of post-pass against 45 us.
int muon_apply_fuses(int64_t batch, int64_t M, int64_t N, int64_t K, int64_t m, int64_t n, int pdt,
                     int beside) {
  if (pdt == MUON_DT_BF16) return 1;
  const int pes = pdt == MUON_DT_F32 ? 4 : 2;
  const double post = 6.0 + (double)batch * m * n * (2 + 2 * pes) / 5.0e6;
  const int64_t n256 = (M / 256) * (N / 256) * batch, n128 = round_up(m, 128) / 128 * (N / 128) * batch;
  const double c256 = bx256_cost(n256, (double)K), c128 = tile_cost(BX_128, n128, (double)K);
  return bx_tile(batch, M, N, K, m, beside) != 256 || c128 < c256 + 0.5 * post;
}

// The last iteration's X' = a X + B X with the post-pass applied in its epilogue: extents and
// operands as muon_launch_gemm's GEMM mode, X' is not stored. tall: the parameter is the
// transpose of the iterate (its rows are the columns of X'). Parameter rows of whole 8-element
// chunks (pcols % 8 == 0), 16-byte aligned tensors and muon_apply_fuses are the caller's to
// check.
int muon_launch_gemm_apply(int64_t batch, int64_t M, int64_t N, int64_t K, const void* a,
                           int64_t lda, int64_t sa, const void* b, int64_t ldb, int64_t sb,
                           int64_t Mv, int64_t Nv, float alpha, float beta, const float* scale,
                           int scale_mode, const MuonApply& ap, int pdt, int tall, int beside,
                           hipStream_t stream) {
  if (K % 128 || M % BF_BM || N % BF_BM || alpha == 0.0f || ap.nb <= 0 ||
      (batch + ap.nb - 1) / ap.nb > MUON_APPLY_MAX || ap.pcols % 8 ||
      ap.prows != (tall ? Nv : Mv) || ap.pcols != (tall ? Mv : Nv)) {
    muon_set_error("gemm_apply: unsupported launch (K %lld, batch %lld)", (long long)K,
                   (long long)batch);
    return MUON_ERR_ARG;
  }
  if (std::max(M * lda, K * ldb) * 2 >= (int64_t)0x7fffffff ||
      ap.prows * ap.pcols * 2 >= (int64_t)0x7fffffff) {
    muon_set_error("gemm_apply: operand exceeds the 2 GiB per-matrix limit");
    return MUON_ERR_SHAPE;
  }
  GemmArgs g;
  memset(&g, 0, sizeof(g));
  g.a = a;
  g.b = b;
  g.cin = b;
  g.lda = lda;
  g.ldb = ldb;
  g.ldc = ldb;
  g.sa = sa;
  g.sb = sb;
  g.sc = sb;
  g.Mv = Mv;
  g.Nv = Nv;
  g.alpha = alpha;
  g.beta = beta;
  g.scale = scale;
  g.scale_mode = scale_mode;
  g.tiles_m = (int)(M / BF_BM);
  g.tiles_n = (int)(N / BF_BM);
  g.K = K;
  g.tiles_per_batch = g.tiles_m * g.tiles_n;
  const int64_t blocks = (int64_t)g.tiles_per_batch * batch;
  if (blocks == 0) return MUON_OK;
  if (blocks > 0x7fffffffLL / 16) {
    muon_set_error("gemm_apply: grid too large (%lld tiles)", (long long)blocks);
    return MUON_ERR_SHAPE;
  }
  g.tiles_total = (int)blocks;
  if (reserve_lds() != 0) {
    muon_set_error("gemm_apply: cannot reserve LDS");
    return MUON_ERR_LAUNCH;
  }
  int TM = bx_tile(batch, M, N, K, Mv, beside);
  if (TM == 256 && pdt != MUON_DT_BF16) TM = 128;
  if (TM == 256) {
    const int wgs = persistent_wgs(blocks);
    const int mode = ap.wd == 0.0f ? 0 : (ap.cautious ? 1 : 2);
#define LAUNCH_APPLY(A, M)                                                                         \
  do {                                                                                           \
    if (K < BETA3_K)                                                                             \
      hipLaunchKernelGGL((gemm_bf16_nn16_kernel<A, M, true>), dim3((unsigned)wgs), dim3(256), N4_SMEM, stream, g, ap); \
    else                                                                                         \
      hipLaunchKernelGGL((gemm_bf16_nn16_kernel<A, M>), dim3((unsigned)wgs), dim3(256), N4_SMEM, stream, g, ap); \
  } while (0)
    if (tall) {
      if (mode == 0) LAUNCH_APPLY(2, 0); else if (mode == 1) LAUNCH_APPLY(2, 1); else LAUNCH_APPLY(2, 2);
    } else {
      if (mode == 0) LAUNCH_APPLY(1, 0); else if (mode == 1) LAUNCH_APPLY(1, 1); else LAUNCH_APPLY(1, 2);
    }
#undef LAUNCH_APPLY
  } else {
    GemmArgs gt = on_tiles(g, MODE_GEMM, TM, Mv, N, batch);
    gt.t0 = 0;
    gt.nb = (int)ap.nb;
#define LAUNCH_TILE(TM_, P_, SW_)                                                               \
  hipLaunchKernelGGL((tile_bx_kernel<TM_, P_, SW_, GemmArgs>), dim3((unsigned)gt.tiles_total), \
                     dim3(256), TileK<TM_>::SMEM, stream, gt, ap)
#define LAUNCH_TILE_P(TM_, P_) \
  do { if (tall) LAUNCH_TILE(TM_, P_, true); else LAUNCH_TILE(TM_, P_, false); } while (0)
#define LAUNCH_TILE_T(TM_)                                              \
  do {                                                                  \
    if (pdt == MUON_DT_BF16) LAUNCH_TILE_P(TM_, MUON_DT_BF16);          \
    else if (pdt == MUON_DT_F16) LAUNCH_TILE_P(TM_, MUON_DT_F16);       \
    else LAUNCH_TILE_P(TM_, MUON_DT_F32);                               \
  } while (0)
    if (TM == 128) LAUNCH_TILE_T(128); else LAUNCH_TILE_T(64);
#undef LAUNCH_TILE_T
#undef LAUNCH_TILE_P
#undef LAUNCH_TILE
  }
  MUON_CHECK_LAUNCH("gemm_apply");
  return MUON_OK;
}

// A product of several buckets in launches of up to GROUP_MAX of them, on 128- or 64-row tiles
// (mode 1: SYRK, 0: B X, with `ap` the apply of parameters of type pdt, tall as
// muon_launch_gemm_apply's): the same bits as a launch per bucket. One launch per product
// instead of one per bucket, for buckets so small that the host's launches take longer than the
// kernels: 16 matrices of four shapes (512 x 512 to 512 x 2048) take 23 / 12 / 24 us for X X^T /
// A A / B X in one launch each, against four launches of 5 to 17 us for each product.
int muon_launch_products(int mode, int n, const MuonProduct* items, float alpha, float beta,
                         int scale_mode, const MuonApply* ap, int pdt, int tall,
                         hipStream_t stream) {
  if (reserve_lds() != 0) {
    muon_set_error("products: cannot reserve LDS");
    return MUON_ERR_LAUNCH;
  }
  if (alpha == 0.0f) {
    muon_set_error("products: alpha must be nonzero");
    return MUON_ERR_ARG;
  }
  for (int i0 = 0; i0 < n; i0 += GROUP_MAX) {
    const int cnt = std::min(GROUP_MAX, n - i0);
    // tile size by the whole launch: its tiles, their K on average and the longest
    int64_t n128 = 0;
    double work = 0.0, kmax = 0.0;
    for (int i = i0; i < i0 + cnt; ++i) {
      const MuonProduct& p = items[i];
      const int64_t t = round_up(p.m, 128) / 128;
      const int64_t tiles = (mode == MODE_SYRK ? t * (t + 1) / 2 : t * (p.N / 128)) * p.batch;
      if (p.K % 64 || p.N % 128 || p.lda * p.m * 2 >= (int64_t)0x7fffffff ||
          (mode == MODE_GEMM && p.ldb * p.K * 2 >= (int64_t)0x7fffffff)) {
        muon_set_error("products: unsupported extents (%lld, %lld, %lld)", (long long)p.m,
                       (long long)p.N, (long long)p.K);
        return MUON_ERR_SHAPE;
      }
      n128 += tiles;
      work += (double)tiles * p.K;
      kmax = std::max(kmax, (double)p.K);
    }
    if (n128 == 0) continue;
    if (n128 > (1 << 24)) {
      muon_set_error("products: grid too large (%lld tiles)", (long long)n128);
      return MUON_ERR_SHAPE;
    }
    const double kavg = work / (double)n128;
    const bool t64 = mode == MODE_SYRK ? tile_cost(SYRK_64, 4 * n128, kavg, kmax) <
                                             tile_cost(SYRK_128, n128, kavg, kmax)
                                       : tile_cost(BX_64, 4 * n128, kavg, kmax) <
                                             tile_cost(BX_128, n128, kavg, kmax);
    const int TM = t64 ? 64 : 128;
    GemmTab tab;
    memset(&tab, 0, sizeof(tab));
    tab.n = cnt;
    for (int i = 0; i < cnt; ++i) {
      const MuonProduct& p = items[i0 + i];
      GemmArgs g;
      memset(&g, 0, sizeof(g));
      g.a = p.a;
      g.lda = p.lda;
      g.sa = p.sa;
      g.b = mode == MODE_SYRK ? p.a : p.b;
      g.ldb = mode == MODE_SYRK ? p.lda : p.ldb;
      g.sb = mode == MODE_SYRK ? p.sa : p.sb;
      g.out = p.out;
      g.ldo = p.ldo;
      g.so = p.so;
      g.K = p.K;
      g.Mv = p.m;
      g.Nv = mode == MODE_SYRK ? p.m : p.nv;
      g.alpha = alpha;
      g.beta = beta;
      g.scale = p.scale;
      g.scale_mode = scale_mode;
      g.t0 = p.t0;
      g.nb = p.nb;
      tab.g[i] = on_tiles(g, mode, TM, p.m, p.N, p.batch);
      tab.tile0[i + 1] = tab.tile0[i] + tab.g[i].tiles_total;
    }
    const dim3 grid((unsigned)tab.tile0[cnt]), block(256);
    if (mode == MODE_SYRK) {
      if (t64)
        hipLaunchKernelGGL((tile_syrk_kernel<64, GemmTab>), grid, block, TileK<64>::SMEM, stream, tab);
      else
        hipLaunchKernelGGL((gemm_bf16_s16h_kernel<GemmTab>), grid, block, H_SMEM, stream, tab);
    } else {
      MuonApply none;
      none.nb = 1;
      const MuonApply& apv = ap ? *ap : none;
#define LAUNCH_GROUP(P_, SW_)                                                                     \
  do {                                                                                            \
    if (t64)                                                                                      \
      hipLaunchKernelGGL((tile_bx_kernel<64, P_, SW_, GemmTab>), grid, block, TileK<64>::SMEM,     \
                         stream, tab, apv);                                                       \
    else                                                                                          \
      hipLaunchKernelGGL((tile_bx_kernel<128, P_, SW_, GemmTab>), grid, block, TileK<128>::SMEM,   \
                         stream, tab, apv);                                                       \
  } while (0)
#define LAUNCH_GROUP_P(P_) \
  do { if (tall) LAUNCH_GROUP(P_, true); else LAUNCH_GROUP(P_, false); } while (0)
      if (!ap) LAUNCH_GROUP(-1, false);
      else if (pdt == MUON_DT_BF16) LAUNCH_GROUP_P(MUON_DT_BF16);
      else if (pdt == MUON_DT_F16) LAUNCH_GROUP_P(MUON_DT_F16);
      else LAUNCH_GROUP_P(MUON_DT_F32);
#undef LAUNCH_GROUP_P
#undef LAUNCH_GROUP
    }
  }
  MUON_CHECK_LAUNCH("products");
  return MUON_OK;
}
