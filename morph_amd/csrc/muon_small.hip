// Small Muon matrices for gfx950: one workgroup per matrix, the whole Newton-Schulz
// chain (streamtrain/optimizer.py:13-22) in one launch.
//
// A chain of general products is 15 dependent launches (muon.hip), each at least
// 3.7 us on one or two tiles: launch, first loads and a few K stages, all latency.
// Where X [m, n] (bf16, padded to 32) and A [m, m] fit one CU's 160 KiB of LDS, one
// workgroup of 8 waves keeps both there: per iteration A = X X^T, B' = b A + c A A +
// a I over A, X' = B' X over X, with a barrier between them.  Bound: LDS reads (a
// 32 x 32 x 16 MFMA takes two fragments of 1 KiB; X' shares its fragments over the
// wave's tiles).  One CU per matrix is enough up to m = 128, whatever the batch (one of 64
// matrices leaves the other CUs idle, and so do products of a tile or two).
//
// Measured, orthogonalize, us a call, the general products (on their 64 edge) -> this:
// one gradient of 200 x 96 80 -> 30, of 128 x 128 78 -> 31, and at the limits of the LDS of
// 128 x 480 80 -> 58, 96 x 736 82 -> 59, 64 x 1184 84 -> 63, 32 x 2496 107 -> 62; eight of
// 128 x 480 96 -> 60; sixty-four of them 220 -> 173, sixty-four of 32 x 32 217 -> 167, both
// then bound by the host.
//
// The bits are the general path's: 32x32x16 MFMAs over K in the same order (zero
// padding adds nothing), the same scaling, fused multiply-adds and roundings.  Only
// the FP64 sum of u^2 runs in another order (its last bits, before the FP32 root).
#include "muon_small.h"

namespace morph {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

constexpr int kPrep = 1024;  // lanes of the prepare kernel
constexpr int kChain = 512;  // lanes of the chain kernel: 8 waves
constexpr int kWaves = kChain / 64;

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// Row and column of the items i0, i0 + step, ... of rows of per_row items each: two
// divisions in all instead of one per item (about 40 instructions, which took longer than
// the rest of a pass over the matrix).
struct Walk {
  int r, c, dr, dc, per_row;
  __device__ Walk(int i0, int step, int per_row_) : per_row(per_row_) {
    r = i0 / per_row;
    c = i0 - r * per_row;
    dr = step / per_row;
    dc = step - dr * per_row;
  }
  __device__ void next() {
    r += dr;
    c += dc;
    if (c >= per_row) c -= per_row, ++r;
  }
};

// Four consecutive elements of one matrix: torch's lerp roundings, as momentum_one.
template <bool kMomentum>
__device__ __forceinline__ float blend(float g, float& m, float mom_w, float nest_w) {
  if constexpr (!kMomentum) return g;
  m = mom_w >= 0.5f ? __fmaf_rn(mom_w - 1.0f, g - m, g) : __fmaf_rn(mom_w, g - m, m);
  return nest_w >= 0.5f ? __fmaf_rn(nest_w - 1.0f, m - g, m) : __fmaf_rn(nest_w, m - g, g);
}

// One workgroup per matrix over its elements in stored order, 4 per lane and access
// when the rows and buffers allow 16-byte accesses, else one.  X0 keeps the stored
// layout (the chain transposes it on its way into the LDS).
template <bool kMomentum>
__global__ __launch_bounds__(kPrep) void small_prepare_kernel(const SmallBatch b, float mom_w,
                                                              float nest_w, uint32_t* found_inf) {
  __shared__ double lds[kPrep / 64];
  const int mat = blockIdx.x, tid = threadIdx.x;
  const bool tall = (b.tall >> mat) & 1;
  const int rows = tall ? b.n : b.m, cols = tall ? b.m : b.n, ld = (cols + 7) & ~7;
  const float* g = b.grad[mat];
  const float* mom = b.mom[mat];
  float* mom_out = b.mom_out[mat];
  uint16_t* x = b.x0 + mat * b.stride;
  const uintptr_t addr = reinterpret_cast<uintptr_t>(g) |
                         (kMomentum ? reinterpret_cast<uintptr_t>(mom) |
                                          reinterpret_cast<uintptr_t>(mom_out)
                                    : 0);
  double ss = 0.0;
  bool bad = false;
  if ((addr & 15) == 0 && (cols & 3) == 0) {
    const int quads = rows * cols / 4;
    Walk w(tid, kPrep, cols / 4);
#pragma unroll 4
    for (int i = tid; i < quads; i += kPrep, w.next()) {
      const f32x4 gv = reinterpret_cast<const f32x4*>(g)[i];
      f32x4 mv = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (kMomentum) mv = reinterpret_cast<const f32x4*>(mom)[i];
      uint32_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float gi = gv[e];  // a bit cast of the vector element itself reads element 0
        bad |= nonfinite_f32_bits(__builtin_bit_cast(uint32_t, gi));
        float m = mv[e];
        const float u = blend<kMomentum>(gi, m, mom_w, nest_w);
        mv[e] = m;
        h[e] = float_to_bf16_bits(u);
        ss += (double)u * (double)u;
      }
      if constexpr (kMomentum) reinterpret_cast<f32x4*>(mom_out)[i] = mv;
      *reinterpret_cast<u32x2*>(x + w.r * ld + w.c * 4) = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    }
  } else {
    Walk w(tid, kPrep, cols);
#pragma unroll 4
    for (int i = tid; i < rows * cols; i += kPrep, w.next()) {
      const float gi = g[i];
      bad |= nonfinite_f32_bits(__builtin_bit_cast(uint32_t, gi));
      float m = kMomentum ? mom[i] : 0.f;
      const float u = blend<kMomentum>(gi, m, mom_w, nest_w);
      if constexpr (kMomentum) mom_out[i] = m;
      x[w.r * ld + w.c] = (uint16_t)float_to_bf16_bits(u);
      ss += (double)u * (double)u;
    }
  }
  if (found_inf != nullptr && __any(bad) && (tid & 63) == 0)
    *reinterpret_cast<volatile uint32_t*>(found_inf) = 1u;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o);
  if ((tid & 63) == 0) lds[tid >> 6] = ss;
  __syncthreads();
  if (tid == 0) {
    double t = 0.0;
    for (int w = 0; w < kPrep / 64; ++w) t += lds[w];
    // as norm_kernel (muon.hip)
    const float den = (float)sqrt(t) + 1e-7f;
    b.scale[mat] = 1.0f / den;
    b.scale[b.count + mat] = (float)(1.0 / ((double)den * (double)den));
    b.scale[2 * b.count + mat] = den;
    b.form[mat] = tall ? 1u : 0u;
  }
}

// Column blocks of X (32 wide) per wave: what the LDS allows at MB row blocks.
template <int MB>
constexpr int column_blocks() {
  constexpr int mp = MB * 32;
  constexpr int np = ((kSmallLds / 2 - mp * (mp + 8)) / mp - 8) / 32 * 32;
  return (np / 32 + kWaves - 1) / kWaves;
}

// MB: 32-row blocks of X (m rounded up).  LDS: X [32 MB][np + 8], then A (and B' over
// it) [32 MB][32 MB + 8]; a row is an odd multiple of 16 bytes longer than a multiple of
// 64, so the 128-bit fragment reads of 16 consecutive rows hit distinct banks.
// Lane layouts as in gemm.hip: a fragment is a row of 8 consecutive k per lane, the
// [K, N] operand X comes through transposing reads, and with the Q fragment as the
// MFMA's first operand register r of lane (fr, fh) is C[fr][8 (r / 4) + 4 fh + r % 4].
template <int MB, SmallOut kOut>
__global__ __launch_bounds__(kChain, 1) void small_chain_kernel(const SmallBatch b,
                                                                const SmallChain ch) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[kSmallLds / 2];
  constexpr int mp = MB * 32, lda = mp + 8;
  constexpr int kCB = column_blocks<MB>();
  const int mat = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, fh = lane >> 5;
  const int m = b.m, n = b.n, np = (n + 31) & ~31, nb = np / 32, ldx = np + 8;
  const bool tall = __builtin_amdgcn_readfirstlane(b.form[mat]) != 0;
  uint16_t* X = lds;
  uint16_t* A = lds + mp * ldx;

  // X0 into the LDS, zero padding included
  for (int i = tid; i < mp * ldx / 8; i += kChain)
    reinterpret_cast<u32x4*>(X)[i] = u32x4{0u, 0u, 0u, 0u};
  __syncthreads();
  // A wave covers 16 rows x 4 pieces of a tall matrix at a time: its transposed LDS
  // accesses then fall on few banks twice, where whole rows of pieces would put 8 lanes on
  // one bank (470 x 128: 34 K cycles of loading).
  const int tile_r = lane >> 2, tile_c = lane & 3;
  {
    const int rows = tall ? n : m, cols = tall ? m : n, ld = (cols + 7) & ~7, per_row = ld / 8;
    const uint16_t* x0 = b.x0 + mat * b.stride;
    constexpr int kBatch = 8;  // loads in flight per lane
    // elements c .. c + 7 of a row, those past the row zero
    auto tail = [&](u32x4 v, int c) {
      const int left = cols - c;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[k] &= left >= 2 * k + 2 ? 0xFFFFFFFFu : left == 2 * k + 1 ? 0xFFFFu : 0u;
      return v;
    };
    if (!tall) {
      const int total = rows * per_row;
      Walk get(tid, kChain, per_row), put = get;
      for (int i0 = tid; i0 < total; i0 += kBatch * kChain) {
        u32x4 v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k, get.next())
          if (i0 + k * kChain < total)
            v[k] = *reinterpret_cast<const u32x4*>(x0 + get.r * ld + get.c * 8);
#pragma unroll
        for (int k = 0; k < kBatch; ++k, put.next())
          if (i0 + k * kChain < total)
            *reinterpret_cast<u32x4*>(X + put.r * ldx + put.c * 8) = tail(v[k], put.c * 8);
      }
    } else {
      const int tiles_c = (per_row + 3) / 4, tiles = (rows + 15) / 16 * tiles_c;
      Walk get(wave, kWaves, tiles_c), put = get;
      for (int t0 = wave; t0 < tiles; t0 += kBatch * kWaves) {
        u32x4 v[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k, get.next()) {
          const int r = get.r * 16 + tile_r, c = get.c * 4 + tile_c;
          if (t0 + k * kWaves < tiles && r < rows && c < per_row)
            v[k] = *reinterpret_cast<const u32x4*>(x0 + r * ld + c * 8);
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k, put.next()) {
          const int r = put.r * 16 + tile_r, c = put.c * 4 + tile_c;
          if (t0 + k * kWaves < tiles && r < rows && c < per_row) {
            const u32x4 w = tail(v[k], c * 8);  // X row c * 8 + e < round_up(m, 8) <= mp
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const uint32_t word = w[e >> 1];
              X[(c * 8 + e) * ldx + r] = (uint16_t)((e & 1) ? word >> 16 : word);
            }
          }
        }
      }
    }
  }
  __syncthreads();

  auto frag = [&](const uint16_t* at, int ld, int row0, int kk) {
    return *reinterpret_cast<const bf16x8*>(at + (row0 + fr) * ld + kk * 16 + fh * 8);
  };
  auto frag_kn = [&](int col0, int kk) {
    const int j = lane & 15;
    const uint16_t* at = X + (kk * 16 + 8 * fh + (j >> 2)) * ldx + col0 + 16 * ((lane >> 4) & 1) +
                         4 * (j & 3);
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
    auto half = [](const uint16_t* p) {
      return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
          (lds_bf16x4*)(__attribute__((address_space(3))) uint16_t*)p));
    };
    const u32x2 lo = half(at), hi = half(at + 4 * ldx);
    return __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y});
  };
  // a symmetric tile and its mirror into A
  auto store_sym = [&](int i, int j, const uint32_t (&w)[8]) {
    uint16_t* at = A + (i * 32 + fr) * lda + j * 32 + 4 * fh;
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<u32x2*>(at + 8 * q) = u32x2{w[2 * q], w[2 * q + 1]};
    if (i != j) {
      uint16_t* mt = A + (j * 32 + 4 * fh) * lda + i * 32 + fr;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        mt[(8 * (r >> 2) + (r & 3)) * lda] = (uint16_t)((r & 1) ? w[r >> 1] >> 16 : w[r >> 1]);
    }
  };

  // The symmetric products' upper triangle of tiles over the waves: wave w < MB has (w, w)
  // and the tile of rows w and w + 1 (mod MB), which share their two fragments (at MB = 2
  // wave 1 has its diagonal alone); at MB = 4 waves 4 and 5 have (0, 2) and (1, 3).  Half
  // the LDS reads of one tile per wave, and one round.
  // Tile 0 is (w, w), tile 1 the other, rows ri < rj of blocks.
  const bool has0 = wave < MB;
  const bool has1 = MB > 1 && (wave < (MB == 2 ? 1 : MB) || (MB == 4 && wave < 6));
  const bool wrap = has0 && wave == MB - 1;  // its tile 1 is (0, w)
  const int ri = wrap ? 0 : has0 ? wave : (has1 ? wave - MB : 0);
  const int rj = wrap ? MB - 1 : has0 ? wave + 1 : (has1 ? ri + 2 : 0);
  const int rd = has0 ? wave : 0;
  auto tile_i = [&](int p) { return p == 0 ? rd : ri; };
  auto tile_j = [&](int p) { return p == 0 ? rd : rj; };
  auto has = [&](int p) { return p == 0 ? has0 : has1; };
  // out[p]: tile p of S S^T over k columns (a multiple of 32); the next two steps'
  // fragments are read under the current two's MFMAs (the last round reads its own again,
  // unused).  The Q fragment, the MFMA's first operand, is the tile column's rows.
  auto product = [&](const uint16_t* S, int ld, int k, f32x16 (&out)[2]) {
    out[0] = f32x16{};
    out[1] = f32x16{};
    if (!has0 && !has1) return;
    bf16x8 a[2], c[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) a[u] = frag(S, ld, ri * 32, u), c[u] = frag(S, ld, rj * 32, u);
    for (int kk = 0; kk < k / 16; kk += 2) {
      const int nk = kk + 2 < k / 16 ? kk + 2 : kk;
      bf16x8 na[2], nc[2];
#pragma unroll
      for (int u = 0; u < 2; ++u)
        na[u] = frag(S, ld, ri * 32, nk + u), nc[u] = frag(S, ld, rj * 32, nk + u);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bf16x8 d = wrap ? c[u] : a[u];
        out[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(d, d, out[0], 0, 0, 0);
        out[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c[u], a[u], out[1], 0, 0, 0);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) a[u] = na[u], c[u] = nc[u];
    }
  };

  for (int it = 0; it < ch.steps; ++it) {
    const float s1 = it == 0 ? b.scale[mat] : 1.0f, s2 = it == 0 ? b.scale[b.count + mat] : 1.0f;
    // A = X X^T (times 1 / den^2 in the first iteration)
    f32x16 sym[2];
    product(X, ldx, np, sym);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if (has(p)) {
        uint32_t w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = pack2(s2 * sym[p][2 * k], s2 * sym[p][2 * k + 1]);
        store_sym(tile_i(p), tile_j(p), w);
      }
    }
    __syncthreads();
    // B' = c A A + b A + a I over A
    product(A, lda, mp, sym);
    uint32_t bw[2][8];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if (has(p)) {
        const int i = tile_i(p), j = tile_j(p);
        const uint16_t* at = A + (i * 32 + fr) * lda + j * 32 + 4 * fh;
        float x[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x2 d = *reinterpret_cast<const u32x2*>(at + 8 * q);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t w = e & 2 ? d.y : d.x;
            const float dv = bf16_bits_to_float(e & 1 ? w >> 16 : w & 0xFFFFu);
            x[4 * q + e] = __fmaf_rn(ch.b, dv, ch.c * sym[p][4 * q + e]);
            if (i == j && fr == 8 * q + 4 * fh + e) x[4 * q + e] = x[4 * q + e] + ch.a;
          }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) bw[p][k] = pack2(x[2 * k], x[2 * k + 1]);
      }
    }
    __syncthreads();  // every wave has read A
#pragma unroll
    for (int p = 0; p < 2; ++p)
      if (has(p)) store_sym(tile_i(p), tile_j(p), bw[p]);
    __syncthreads();
    // X' = B' X (times 1 / den in the first iteration) over X: wave w owns the column
    // blocks w, w + 8, ...
    f32x16 acc[kCB][MB];
#pragma unroll
    for (int c = 0; c < kCB; ++c)
#pragma unroll
      for (int i = 0; i < MB; ++i) acc[c][i] = f32x16{};
#pragma unroll
    for (int kk = 0; kk < mp / 16; ++kk) {
      bf16x8 fa[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[i] = frag(A, lda, i * 32, kk);
#pragma unroll
      for (int c = 0; c < kCB; ++c) {
        const int cb = wave + c * kWaves;
        if (cb < nb) {
          const bf16x8 fq = frag_kn(cb * 32, kk);
#pragma unroll
          for (int i = 0; i < MB; ++i)
            acc[c][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fq, fa[i], acc[c][i], 0, 0, 0);
        }
      }
    }
    __syncthreads();  // every wave has read X
#pragma unroll
    for (int c = 0; c < kCB; ++c) {
      const int cb = wave + c * kWaves;
      if (cb < nb) {
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          uint16_t* at = X + (i * 32 + fr) * ldx + cb * 32 + 4 * fh;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<u32x2*>(at + 8 * q) =
                u32x2{pack2(s1 * acc[c][i][4 * q], s1 * acc[c][i][4 * q + 1]),
                      pack2(s1 * acc[c][i][4 * q + 2], s1 * acc[c][i][4 * q + 3])};
        }
      }
    }
    __syncthreads();
  }

  if constexpr (kOut == SmallOut::kStore) {
    uint16_t* x = ch.x + mat * b.stride;
    const int per_row = (n + 7) / 8;
    Walk w(tid, kChain, per_row);
    for (int i = tid; i < m * per_row; i += kChain, w.next())
      *reinterpret_cast<u32x4*>(x + w.r * ch.ldx + w.c * 8) =
          *reinterpret_cast<const u32x4*>(X + w.r * ldx + w.c * 8);
    return;
  }
  // the parameter in its stored layout: 4 consecutive elements of a row per lane, or one
  // element per lane when a row or the buffer is not a whole number of 16 bytes
  float* p = b.param[mat];
  const int rows = tall ? n : m, cols = tall ? m : n;
  const float scale = ch.scale[mat];
  auto one = [&](float pv, uint32_t u) {
    if constexpr (kOut == SmallOut::kExtract) return bf16_bits_to_float(u);
    else return muon_update_element(pv, u, scale, ch.decay, ch.neg_lr);
  };
  auto value = [&](int r, int c) -> uint32_t { return tall ? X[c * ldx + r] : X[r * ldx + c]; };
  if ((reinterpret_cast<uintptr_t>(p) & 15) == 0 && (cols & 3) == 0) {
    // 4 consecutive elements per lane: along the rows, or 16 rows x 4 pieces (tile_r, tile_c)
    // of a tall matrix
    constexpr int kBatch = 4;
    const int per_row = cols / 4;
    const int tiles_c = tall ? (per_row + 3) / 4 : per_row;
    const int step = tall ? kWaves : kChain, first = tall ? wave : tid;
    const int total = tall ? (rows + 15) / 16 * tiles_c : rows * per_row;
    Walk get(first, step, tiles_c), put = get;
    auto row_of = [&](const Walk& w) { return tall ? w.r * 16 + tile_r : w.r; };
    auto col_of = [&](const Walk& w) { return tall ? w.c * 4 + tile_c : w.c; };
    for (int i0 = first; i0 < total; i0 += kBatch * step) {
      f32x4 v[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; ++k, get.next()) {
        const int r = row_of(get), c = col_of(get);
        v[k] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (kOut == SmallOut::kApply && i0 + k * step < total && r < rows && c < per_row)
          v[k] = reinterpret_cast<const f32x4*>(p)[r * per_row + c];
      }
#pragma unroll
      for (int k = 0; k < kBatch; ++k, put.next()) {
        const int r = row_of(put), c = col_of(put);
        if (i0 + k * step < total && r < rows && c < per_row) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[k][e] = one(v[k][e], value(r, c * 4 + e));
          reinterpret_cast<f32x4*>(p)[r * per_row + c] = v[k];
        }
      }
    }
  } else {
    constexpr int kBatch = 8;
    const int total = rows * cols;
    Walk w(tid, kChain, cols);
    for (int i0 = tid; i0 < total; i0 += kBatch * kChain) {
      float v[kBatch];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        v[k] = 0.f;
        if (kOut == SmallOut::kApply && i0 + k * kChain < total) v[k] = p[i0 + k * kChain];
      }
#pragma unroll
      for (int k = 0; k < kBatch; ++k, w.next())
        if (i0 + k * kChain < total) p[i0 + k * kChain] = one(v[k], value(w.r, w.c));
    }
  }
}

template <int MB>
void launch_chain(const SmallBatch& b, const SmallChain& c, SmallOut out, hipStream_t s) {
  const dim3 grid((unsigned)b.count), block(kChain);
  switch (out) {
    case SmallOut::kStore:
      hipLaunchKernelGGL((small_chain_kernel<MB, SmallOut::kStore>), grid, block, 0, s, b, c);
      break;
    case SmallOut::kApply:
      hipLaunchKernelGGL((small_chain_kernel<MB, SmallOut::kApply>), grid, block, 0, s, b, c);
      break;
    case SmallOut::kExtract:
      hipLaunchKernelGGL((small_chain_kernel<MB, SmallOut::kExtract>), grid, block, 0, s, b, c);
      break;
  }
}
static_assert(sizeof(SmallBatch) + sizeof(SmallChain) + 64 <= kMaxKernargBytes, "kernel arguments");

}  // namespace

int small_prepare(const SmallBatch& b, bool orth_only, float mom_w, float nest_w,
                  uint32_t* found_inf, hipStream_t s) {
  if (orth_only)
    hipLaunchKernelGGL(small_prepare_kernel<false>, dim3((unsigned)b.count), dim3(kPrep), 0, s, b,
                       mom_w, nest_w, found_inf);
  else
    hipLaunchKernelGGL(small_prepare_kernel<true>, dim3((unsigned)b.count), dim3(kPrep), 0, s, b,
                       mom_w, nest_w, found_inf);
  return launch_status();
}

int small_chain(const SmallBatch& b, const SmallChain& c, SmallOut out, hipStream_t s) {
  switch ((b.m + 31) / 32) {
    case 1: launch_chain<1>(b, c, out, s); break;
    case 2: launch_chain<2>(b, c, out, s); break;
    case 3: launch_chain<3>(b, c, out, s); break;
    case 4: launch_chain<4>(b, c, out, s); break;
    default: return MORPH_EINVAL;
  }
  return launch_status();
}

}  // namespace morph
