// Projections over a handful of rows: lin() (ming-dit.cc:1763-1771) at
// M <= kGemvMaxM with no live adapter. The forward runs these once per block
// and per forward at M = 1: the adaLN modulation of every modulated block
// (fill_mod, ming-dit.cc:2266-2273; quantized, [4H, adaln_dim]), the timestep
// MLP (2276-2281) and the final layer's adaLN (dense). A 256-row GEMM tile
// would spend 255 of its rows on nothing; this kernel instead streams each
// weight once, HBM-bound, with the rows' activations read wave-uniformly.
//
// The rows ride on the matrix cores: a wave takes 16 columns and walks K in
// the 64-wide groups with v_mfma_f32_16x16x32_bf16 (A: 16 weight rows x 32 k,
// B: 32 k x up to 16 rows of x, zero past M), so eight rows cost what one does,
// and lane (n, g) loads the group's k 16g..16g+15 of weight row n in one or two
// pieces: whole 128-byte rows a wave (dense), 512 bytes and up of codes. The
// kernel before gave a lane a column and multiplied row by row on the VALU:
// [3840, 3840] dense took 22.9 us at one row and 77.9 at eight (weights from
// HBM), every lane reading K * 2 bytes from its neighbour; this one 8.0 and 9.1,
// and [10240, 3840] 18.2 (4.3 TB/s).
//
// Products and sums are as precise as before: dense weights and activations
// enter as the bf16 they are, quantized weights as their integer codes (exact
// in bf16) in the affine form w = scale * q + bias the reference packs follow,
// per group scale * sum(q * x) + bias * sum(x) in f32 (the sum of x is the same
// MFMA against ones). One rounding to bf16 at the end.
//
// K <= 256 (the adaLN projections): four waves of 16 columns each, all of K.
// Longer K: eight waves share 16 columns, wave w the groups w, w + 8, ...; their
// sums meet in LDS and are added in wave order (the bits do not depend on
// timing).
//
// Weights are read in the resident general layout (kernels.h): codes
// [kt][n][w] with the w4 nibble order {0,2,4,6,1,3,5,7} and w8 bytes in k
// order, sb [kt][n] = bf16 scale | bf16 bias << 16; dense w [n][k].
#include "common.h"
#include "kernels.h"

namespace ming {
namespace {

__device__ __forceinline__ floatx4_t mfma16(const uint4& w, const uint4& x, floatx4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w),
                                                 __builtin_bit_cast(bf16x8_t, x), c, 0, 0, 0);
}

// Byte i as f32 (below 256: exact in bf16 too).
__device__ __forceinline__ float byte_f(uint32_t w, int i) { return (float)((w >> (8 * i)) & 0xffu); }

// One group's weights of a lane: 16 values, k 16g..16g+15, as the A operands
// of two MFMAs.
template <int BITS>
struct GroupRaw {
  uint4 v[BITS == 16 ? 2 : 1];   // w4: two words in x, y; w8: four words
};

template <int BITS>
__device__ __forceinline__ void load_group(const GemvArgs& a, int n, int kt, int g,
                                           GroupRaw<BITS>& r) {
  if constexpr (BITS == 4) {
    const uint2 c = *reinterpret_cast<const uint2*>(a.codes + ((long long)kt * a.N + n) * 8 + 2 * g);
    r.v[0] = make_uint4(c.x, c.y, 0, 0);
  } else if constexpr (BITS == 8) {
    r.v[0] = *reinterpret_cast<const uint4*>(a.codes + ((long long)kt * a.N + n) * 16 + 4 * g);
  } else {
    const uint4* p = reinterpret_cast<const uint4*>(a.w16 + (long long)n * a.K + 64 * kt + 16 * g);
    r.v[0] = p[0];
    r.v[1] = p[1];
  }
}

template <int BITS>
__device__ __forceinline__ void operands(const GroupRaw<BITS>& r, uint4& w0, uint4& w1) {
  if constexpr (BITS == 4) {
    // nibble i of a word holds k = {0,2,4,6,1,3,5,7}[i]: even nibbles are k 0,
    // 4, 1, 5 by byte, odd ones k 2, 6, 3, 7
    auto word = [](uint32_t c) {
      const uint32_t lo = c & 0x0F0F0F0Fu, hi = (c >> 4) & 0x0F0F0F0Fu;
      uint4 o;
      o.x = pack_bf16x2_rne(byte_f(lo, 0), byte_f(lo, 2));
      o.y = pack_bf16x2_rne(byte_f(hi, 0), byte_f(hi, 2));
      o.z = pack_bf16x2_rne(byte_f(lo, 1), byte_f(lo, 3));
      o.w = pack_bf16x2_rne(byte_f(hi, 1), byte_f(hi, 3));
      return o;
    };
    w0 = word(r.v[0].x);
    w1 = word(r.v[0].y);
  } else if constexpr (BITS == 8) {
    auto words = [](uint32_t c, uint32_t d) {
      uint4 o;
      o.x = pack_bf16x2_rne(byte_f(c, 0), byte_f(c, 1));
      o.y = pack_bf16x2_rne(byte_f(c, 2), byte_f(c, 3));
      o.z = pack_bf16x2_rne(byte_f(d, 0), byte_f(d, 1));
      o.w = pack_bf16x2_rne(byte_f(d, 2), byte_f(d, 3));
      return o;
    };
    w0 = words(r.v[0].x, r.v[0].y);
    w1 = words(r.v[0].z, r.v[0].w);
  } else {
    w0 = r.v[0];
    w1 = r.v[1];
  }
}

template <int BITS, int WK>
__device__ __forceinline__ void gemv_body(const GemvArgs& a) {
  constexpr int U = 4;                       // groups in flight a wave
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;    // weight row / row of x, and k part
  const int n0 = WK == 1 ? ((int)blockIdx.x * 4 + wave) * 16 : (int)blockIdx.x * 16;
  const int nw = n0 + c < a.N ? n0 + c : a.N - 1;   // rows past N compute, never store
  const int KT = a.K / 64;
  const bool row = c < a.M;
  const uint16_t* const xr = a.x + (long long)(row ? c : 0) * a.ldx + 16 * g;
  const uint32_t one2 = 0x3f803f80u;
  const uint4 ones = make_uint4(one2, one2, one2, one2);
  floatx4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int k0 = WK == 1 ? 0 : wave; k0 < KT; k0 += WK * U) {
    GroupRaw<BITS> w[U];
    uint4 x[U][2];
    uint32_t sb[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kt = k0 + WK * u;            // wave-uniform
      if (kt < KT) {
        load_group<BITS>(a, nw, kt, g, w[u]);
        const uint4* xp = reinterpret_cast<const uint4*>(xr + 64 * kt);
        x[u][0] = row ? xp[0] : make_uint4(0, 0, 0, 0);
        x[u][1] = row ? xp[1] : make_uint4(0, 0, 0, 0);
        if constexpr (BITS != 16) {
          // (s, b) of the four columns whose sums this lane holds
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int n = n0 + 4 * g + r;
            sb[u][r] = a.sb[(long long)kt * a.N + (n < a.N ? n : a.N - 1)];
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k0 + WK * u < KT) {
        uint4 w0, w1;
        operands<BITS>(w[u], w0, w1);
        if constexpr (BITS == 16) {
          acc = mfma16(w0, x[u][0], acc);
          acc = mfma16(w1, x[u][1], acc);
        } else {
          const floatx4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
          const floatx4_t d = mfma16(w1, x[u][1], mfma16(w0, x[u][0], zero));
          const floatx4_t s = mfma16(ones, x[u][1], mfma16(ones, x[u][0], zero));
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[r] += __builtin_fmaf(bf16_lo(sb[u][r]), d[r], bf16_hi(sb[u][r]) * s[r]);
        }
      }
    }
  }
  // lane (m = c, g): columns n0 + 4g + 0..3 of row m
  if constexpr (WK > 1) {
    __shared__ floatx4_t red[WK][64];
    red[wave][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
    acc = red[0][lane];
#pragma unroll
    for (int w = 1; w < WK; ++w)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[r] += red[w][lane][r];
  }
  if (!row) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = n0 + 4 * g + r;
    if (n < a.N) {
      float v = acc[r];
      if (a.bias) v += bf16_to_f32(a.bias[n]);
      a.y[(long long)c * a.ldy + n] = (uint16_t)f32_to_bf16_bits(v);
    }
  }
}

template <int BITS, int WK>
__global__ __launch_bounds__(WK == 1 ? 256 : 64 * WK) void gemv_kernel(const GemvArgs a) {
  gemv_body<BITS, WK>(a);
}

template <int BITS, int WK>
__global__ __launch_bounds__(WK == 1 ? 256 : 64 * WK) void gemv_batch_kernel(const GemvBatch b) {
  GemvArgs a = b.base;
  const GemvEntry& e = b.e[blockIdx.y];
  a.codes = e.codes;
  a.sb = e.sb;
  a.w16 = e.w16;
  a.y = e.y;
  gemv_body<BITS, WK>(a);
}

// K <= 256: one wave walks all of it. The same choice for the single and the
// batched launch, so an entry's bits are the single call's.
constexpr int kShortK = 256;

template <int BITS>
void launch_one(const GemvArgs& a, hipStream_t s) {
  if (a.K <= kShortK)
    hipLaunchKernelGGL((gemv_kernel<BITS, 1>), dim3((unsigned)((a.N + 63) / 64)), dim3(256), 0, s,
                       a);
  else
    hipLaunchKernelGGL((gemv_kernel<BITS, 8>), dim3((unsigned)((a.N + 15) / 16)), dim3(512), 0, s,
                       a);
}

template <int BITS>
void launch_many(const GemvBatch& b, hipStream_t s) {
  const unsigned n = (unsigned)b.base.N, count = (unsigned)b.count;
  if (b.base.K <= kShortK)
    hipLaunchKernelGGL((gemv_batch_kernel<BITS, 1>), dim3((n + 63) / 64, count), dim3(256), 0, s,
                       b);
  else
    hipLaunchKernelGGL((gemv_batch_kernel<BITS, 8>), dim3((n + 15) / 16, count), dim3(512), 0, s,
                       b);
}

}  // namespace

hipError_t launch_gemv_batch(int bits, const GemvBatch& b, hipStream_t s) {
  const GemvArgs& a = b.base;
  if (b.count <= 0 || a.M <= 0 || a.N <= 0) return hipSuccess;
  if (b.count > kGemvBatch || a.M > kGemvMaxM || a.K % 64 != 0) return hipErrorInvalidValue;
  switch (bits) {
    case 4: launch_many<4>(b, s); break;
    case 8: launch_many<8>(b, s); break;
    case 16: launch_many<16>(b, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_gemv(int bits, const GemvArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (a.M > kGemvMaxM || a.K % 64 != 0) return hipErrorInvalidValue;
  switch (bits) {
    case 4: launch_one<4>(a, s); break;
    case 8: launch_one<8>(a, s); break;
    case 16: launch_one<16>(a, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t validate_gemv_kernels() {
  hipFuncAttributes fa;
  const void* fns[] = {reinterpret_cast<const void*>(&gemv_kernel<4, 1>),
                       reinterpret_cast<const void*>(&gemv_kernel<4, 8>),
                       reinterpret_cast<const void*>(&gemv_kernel<8, 1>),
                       reinterpret_cast<const void*>(&gemv_kernel<8, 8>),
                       reinterpret_cast<const void*>(&gemv_kernel<16, 1>),
                       reinterpret_cast<const void*>(&gemv_kernel<16, 8>),
                       reinterpret_cast<const void*>(&gemv_batch_kernel<4, 1>),
                       reinterpret_cast<const void*>(&gemv_batch_kernel<4, 8>),
                       reinterpret_cast<const void*>(&gemv_batch_kernel<8, 1>),
                       reinterpret_cast<const void*>(&gemv_batch_kernel<8, 8>),
                       reinterpret_cast<const void*>(&gemv_batch_kernel<16, 1>),
                       reinterpret_cast<const void*>(&gemv_batch_kernel<16, 8>)};
  for (const void* f : fns) {
    const hipError_t e = hipFuncGetAttributes(&fa, f);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace ming
