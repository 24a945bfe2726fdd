// Small Muon matrices for gfx950: one workgroup per matrix, the whole Newton-Schulz
// chain (streamtrain/optimizer.py:13-22) in one launch.
//
// A chain of general products is 15 dependent launches (muon.hip), each at least
// 3.7 us on one or two tiles: launch, first loads and a few K stages, all latency.
// Where X [m, n] (bf16, padded to 32) and A [m, m] fit one CU's 160 KiB of LDS, one
// workgroup of 8 waves keeps both there: per iteration A = X X^T, B' = b A + c A A +
// a I over A, X' = B' X over X, with a barrier between them.  Bound: LDS reads (a
// 32 x 32 x 16 MFMA takes two fragments of 1 KiB; X' shares its fragments over the
// wave's tiles).  One CU per matrix is enough up to m = 128: there an iteration costs
// about what three launches do.
//
// Measured, orthogonalize of one 200 x 96 gradient: 85 us a call (20 launches, 82 us of
// kernels) -> 30.6 us (2 launches).
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
    const int quads = rows * cols / 4, per_row = cols / 4;
#pragma unroll 4
    for (int i = tid; i < quads; i += kPrep) {
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
      const int r = i / per_row, c = (i - r * per_row) * 4;
      *reinterpret_cast<u32x2*>(x + r * ld + c) = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    }
  } else {
#pragma unroll 4
    for (int i = tid; i < rows * cols; i += kPrep) {
      const float gi = g[i];
      bad |= nonfinite_f32_bits(__builtin_bit_cast(uint32_t, gi));
      float m = kMomentum ? mom[i] : 0.f;
      const float u = blend<kMomentum>(gi, m, mom_w, nest_w);
      if constexpr (kMomentum) mom_out[i] = m;
      const int r = i / cols, c = i - r * cols;
      x[r * ld + c] = (uint16_t)float_to_bf16_bits(u);
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
  constexpr int kSym = MB * (MB + 1) / 2;                  // upper triangle of A's tiles
  constexpr int kSymPer = (kSym + kWaves - 1) / kWaves;    // of them per wave
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
  {
    const int rows = tall ? n : m, cols = tall ? m : n, ld = (cols + 7) & ~7, per_row = ld / 8;
    const uint16_t* x0 = b.x0 + mat * b.stride;
#pragma unroll 4
    for (int i = tid; i < rows * per_row; i += kChain) {
      const int r = i / per_row, c = (i - r * per_row) * 8;
      const u32x4 v = *reinterpret_cast<const u32x4*>(x0 + r * ld + c);
      if (!tall && c + 8 <= cols) {
        *reinterpret_cast<u32x4*>(X + r * ldx + c) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint16_t h = (uint16_t)((e & 1) ? v[e >> 1] >> 16 : v[e >> 1]);
          if (c + e < cols) {
            if (tall) X[(c + e) * ldx + r] = h;
            else X[r * ldx + c + e] = h;
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
  // tile t of the upper triangle, row by row
  auto tile_of = [](int t, int& i, int& j) {
    i = 0;
    while (t >= MB - i) t -= MB - i, ++i;
    j = i + t;
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

  for (int it = 0; it < ch.steps; ++it) {
    const float s1 = it == 0 ? b.scale[mat] : 1.0f, s2 = it == 0 ? b.scale[b.count + mat] : 1.0f;
    // A = X X^T (times 1 / den^2 in the first iteration)
#pragma unroll
    for (int p = 0; p < kSymPer; ++p) {
      const int t = wave + p * kWaves;
      if (t < kSym) {
        int i, j;
        tile_of(t, i, j);
        f32x16 acc = f32x16{};
#pragma unroll 4
        for (int kk = 0; kk < np / 16; ++kk)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(X, ldx, j * 32, kk),
                                                        frag(X, ldx, i * 32, kk), acc, 0, 0, 0);
        uint32_t w[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = pack2(s2 * acc[2 * k], s2 * acc[2 * k + 1]);
        store_sym(i, j, w);
      }
    }
    __syncthreads();
    // B' = c A A + b A + a I over A
    uint32_t bw[kSymPer][8];
#pragma unroll
    for (int p = 0; p < kSymPer; ++p) {
      const int t = wave + p * kWaves;
      if (t < kSym) {
        int i, j;
        tile_of(t, i, j);
        f32x16 acc = f32x16{};
#pragma unroll
        for (int kk = 0; kk < mp / 16; ++kk)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(frag(A, lda, j * 32, kk),
                                                        frag(A, lda, i * 32, kk), acc, 0, 0, 0);
        const uint16_t* at = A + (i * 32 + fr) * lda + j * 32 + 4 * fh;
        float x[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x2 d = *reinterpret_cast<const u32x2*>(at + 8 * q);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t w = e & 2 ? d.y : d.x;
            const float dv = bf16_bits_to_float(e & 1 ? w >> 16 : w & 0xFFFFu);
            x[4 * q + e] = __fmaf_rn(ch.b, dv, ch.c * acc[4 * q + e]);
            if (i == j && fr == 8 * q + 4 * fh + e) x[4 * q + e] = x[4 * q + e] + ch.a;
          }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) bw[p][k] = pack2(x[2 * k], x[2 * k + 1]);
      }
    }
    __syncthreads();  // every wave has read A
#pragma unroll
    for (int p = 0; p < kSymPer; ++p) {
      const int t = wave + p * kWaves;
      if (t < kSym) {
        int i, j;
        tile_of(t, i, j);
        store_sym(i, j, bw[p]);
      }
    }
    __syncthreads();
    // X' = B' X (times 1 / den in the first iteration) over X: wave w owns the column
    // blocks w, w + 8, ...
    f32x16 acc[kCB][MB];
#pragma unroll
    for (int c = 0; c < kCB; ++c)
#pragma unroll
      for (int i = 0; i < MB; ++i) acc[c][i] = f32x16{};
#pragma unroll 2
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
    for (int i = tid; i < m * per_row; i += kChain) {
      const int r = i / per_row, c = (i - r * per_row) * 8;
      *reinterpret_cast<u32x4*>(x + r * ch.ldx + c) = *reinterpret_cast<const u32x4*>(X + r * ldx + c);
    }
    return;
  }
  // the parameter in its stored layout: 4 elements of a row per lane
  float* p = b.param[mat];
  const int rows = tall ? n : m, cols = tall ? m : n, per_row = (cols + 3) / 4;
  const bool vec = (reinterpret_cast<uintptr_t>(p) & 15) == 0 && (cols & 3) == 0;
  const float scale = ch.scale[mat];
  auto one = [&](float pv, uint32_t u) {
    if constexpr (kOut == SmallOut::kExtract) return bf16_bits_to_float(u);
    else return muon_update_element(pv, u, scale, ch.decay, ch.neg_lr);
  };
#pragma unroll 4
  for (int i = tid; i < rows * per_row; i += kChain) {
    const int r = i / per_row, c = (i - r * per_row) * 4;
    float* at = p + (int64_t)r * cols + c;
    uint32_t u[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)  // past the row only inside X's padding
      u[e] = tall ? X[(c + e) * ldx + r] : X[r * ldx + c + e];
    if (vec) {
      f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (kOut == SmallOut::kApply) v = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = one(v[e], u[e]);
      *reinterpret_cast<f32x4*>(at) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (c + e < cols) at[e] = one(kOut == SmallOut::kApply ? at[e] : 0.f, u[e]);
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
