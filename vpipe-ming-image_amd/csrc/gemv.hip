// Projections over a handful of rows: lin() (ming-dit.cc:1763-1771) at
// M <= kGemvMaxM with no live adapter. The forward runs these once per block
// and per forward at M = 1: the adaLN modulation of every modulated block
// (fill_mod, ming-dit.cc:2266-2273; quantized, [4H, adaln_dim]), the timestep
// MLP (2276-2281) and the final layer's adaLN (dense). A 256-row GEMM tile
// would spend 255 of its rows on nothing; this kernel streams each weight
// once. Bound by HBM where the weight is large, by the launch and one chain of
// load, product and reduction where it is small.
//
// The rows ride on the matrix cores: a wave takes 16 * CT columns and walks K
// in the 64-wide groups with v_mfma_f32_16x16x32_bf16 (A: 16 weight rows x 32
// k, B: 32 k x up to 16 rows of x), so eight rows cost what one does, and lane
// (n, g) loads the group's k 16g..16g+15 of weight row n in one or two pieces:
// whole 128-byte rows a wave (dense), 512 bytes and up of codes. The kernel
// before gave a lane a column and multiplied row by row on the VALU: [3840,
// 3840] dense took 22.9 us at one row and 77.9 at eight (weights from HBM),
// every lane reading K * 2 bytes from its neighbour; this one 8.0 and 9.1, and
// [10240, 3840] 18.2 (4.3 TB/s).
//
// Products and sums are as precise as before: dense weights and activations
// enter as the bf16 they are, quantized weights as their integer codes (exact
// in bf16) in the affine form w = scale * q + bias the reference packs follow,
// per group scale * sum(q * x) + bias * sum(x) in f32 (the sum of x is the same
// MFMA against ones). One rounding to bf16 at the end.
//
// The WK waves of a block share its columns. The groups fall into CL * WK
// residue classes, each summed by one wave; the sums meet in LDS and are added
// in class order, so the bits depend on the number of classes (on K alone, see
// kShortK) and not on timing, WK, CT, M or whether the call is batched.
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
      uint32_t lo = c & 0x0F0F0F0Fu, hi = (c >> 4) & 0x0F0F0F0Fu;
      // kept as the two masks: seen through, each nibble becomes a bit-field
      // extract and a conversion, not one conversion of a byte
      asm("" : "+v"(lo), "+v"(hi));
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

template <int BITS, int WK, int CT, int CL>
__device__ __forceinline__ void gemv_body(const GemvArgs& a) {
  constexpr int NC = WK * CL;                // residue classes of the groups
  constexpr int U = NC == 4 ? 1 : 4 / (CL * CT);   // groups of a class in flight
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;    // weight row / row of x, and k part
  const int n0 = (int)blockIdx.x * 16 * CT;
  const int KT = a.K / 64;
  const bool row = c < a.M;                  // lanes past M multiply row 0, never store
  const uint16_t* const xr = a.x + (long long)(row ? c : 0) * a.ldx + 16 * g;
  const uint32_t one2 = 0x3f803f80u;
  const uint4 ones = make_uint4(one2, one2, one2, one2);
  floatx4_t acc[CL][CT];
#pragma unroll
  for (int j = 0; j < CL; ++j)
#pragma unroll
    for (int t = 0; t < CT; ++t) acc[j][t] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
  for (int k0 = wave; k0 < KT; k0 += NC * U) {
    GroupRaw<BITS> w[U * CL][CT];
    uint4 x[U * CL][2], sb[U * CL][CT];
#pragma unroll
    for (int u = 0; u < U * CL; ++u) {
      const int kt = k0 + WK * u;            // wave-uniform
      if (kt < KT) {
        const uint4* xp = reinterpret_cast<const uint4*>(xr + 64 * kt);
        x[u][0] = xp[0];
        x[u][1] = xp[1];
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          // columns past N (a multiple of 8) compute the last ones, never store
          const int n = n0 + 16 * t + c;
          load_group<BITS>(a, n < a.N ? n : a.N - 1, kt, g, w[u][t]);
          if constexpr (BITS != 16) {
            // (s, b) of the four columns whose sums this lane holds
            const int ns = n0 + 16 * t + 4 * g;
            sb[u][t] = *reinterpret_cast<const uint4*>(a.sb + (long long)kt * a.N +
                                                       (ns < a.N ? ns : a.N - 4));
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < U * CL; ++u) {
      if (k0 + WK * u < KT) {
        [[maybe_unused]] floatx4_t s;
        const floatx4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (BITS != 16) s = mfma16(ones, x[u][1], mfma16(ones, x[u][0], zero));
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          floatx4_t& sum = acc[u % CL][t];
          uint4 w0, w1;
          operands<BITS>(w[u][t], w0, w1);
          if constexpr (BITS == 16) {
            sum = mfma16(w0, x[u][0], sum);
            sum = mfma16(w1, x[u][1], sum);
          } else {
            const floatx4_t d = mfma16(w1, x[u][1], mfma16(w0, x[u][0], zero));
            const uint32_t* sp = &sb[u][t].x;
#pragma unroll
            for (int r = 0; r < 4; ++r)
              sum[r] += __builtin_fmaf(bf16_lo(sp[r]), d[r], bf16_hi(sp[r]) * s[r]);
          }
        }
      }
    }
  }
  // Lane (m = c, g): columns 4g + 0..3 of each 16, row m. Wave t adds the
  // classes' sums of columns 16t.. in class order.
  __shared__ floatx4_t red[NC][CT][64];
#pragma unroll
  for (int j = 0; j < CL; ++j)
#pragma unroll
    for (int t = 0; t < CT; ++t) red[wave + WK * j][t][lane] = acc[j][t];
  __syncthreads();
  const int n = n0 + 16 * wave + 4 * g;
  if (wave >= CT || !row || n >= a.N) return;
  floatx4_t v = red[0][wave][lane];
#pragma unroll
  for (int j = 1; j < NC; ++j) v += red[j][wave][lane];
  if (a.bias) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] += bf16_to_f32(a.bias[n + r]);
  }
  *reinterpret_cast<uint2*>(a.y + (long long)c * a.ldy + n) =
      make_uint2(pack_bf16x2_rne(v[0], v[1]), pack_bf16x2_rne(v[2], v[3]));
}

template <int BITS, int WK, int CT>
__global__ __launch_bounds__(64 * WK) void gemv_kernel(const GemvArgs a) {
  gemv_body<BITS, WK, CT, 1>(a);
}

template <int BITS, int CL>
__global__ __launch_bounds__(256) void gemv_batch_kernel(const GemvBatch b) {
  GemvArgs a = b.base;
  const GemvEntry& e = b.e[blockIdx.y];
  a.codes = e.codes;
  a.sb = e.sb;
  a.w16 = e.w16;
  a.y = e.y;
  gemv_body<BITS, 4, 2, CL>(a);
}

template <int BITS, int WK, int CT>
void launch_shape(const GemvArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((gemv_kernel<BITS, WK, CT>), dim3((unsigned)((a.N + 16 * CT - 1) / (16 * CT))),
                     dim3(64 * WK), 0, s, a);
}
template <int BITS, int CL>
void launch_batch_shape(const GemvBatch& b, hipStream_t s) {
  hipLaunchKernelGGL((gemv_batch_kernel<BITS, CL>),
                     dim3((unsigned)((b.base.N + 31) / 32), (unsigned)b.count), dim3(256), 0, s, b);
}

// K <= 512: four classes of groups, a wave each (eight waves would only add
// waves to start: [15360, 512] w4 at one row 4.2 us, 3.3 with four). Longer K:
// eight, a wave each ([3840, 1024] w4 2.63 us, 2.73 with four; [3840, 3840] 5.1
// and 8.8). 16 columns a block; quantized weights 32 where that would be more
// than three blocks a CU: [10240, 3840] w4 10.0 us with 16, 11.0 with 32; [15360,
// 3840] 12.5 and 11.5 (dense 22.7 and 23.7). [15360, 256] w4 at one row takes
// 2.36 us; the VALU kernel took 2.53, one wave walking all four groups 3.13. A
// batch fills the chip with blocks: 32 columns each ([15360, 256] w4 x 32: 25.6
// us with 16, 21.3 with 32, 22.0 with 64, all before the bytes were converted as
// bytes: 19.8 now), past K = 512 four waves of two classes ([15360, 1024] w4 x
// 32: 77.6 us, with eight waves 96.7).
constexpr int kShortK = 512;

template <int BITS>
void launch_one(const GemvArgs& a, hipStream_t s) {
  if constexpr (BITS != 16) {
    if (a.N > 3 * 256 * 16) {
      a.K <= kShortK ? launch_shape<BITS, 4, 2>(a, s) : launch_shape<BITS, 8, 2>(a, s);
      return;
    }
  }
  a.K <= kShortK ? launch_shape<BITS, 4, 1>(a, s) : launch_shape<BITS, 8, 1>(a, s);
}

template <int BITS>
void launch_many(const GemvBatch& b, hipStream_t s) {
  if (b.base.K <= kShortK)
    launch_batch_shape<BITS, 1>(b, s);
  else
    launch_batch_shape<BITS, 2>(b, s);
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
  const void* fns[] = {
#define MING_GEMV_ALL(BITS)                                             \
  reinterpret_cast<const void*>(&gemv_kernel<BITS, 4, 1>),              \
      reinterpret_cast<const void*>(&gemv_kernel<BITS, 8, 1>),          \
      reinterpret_cast<const void*>(&gemv_batch_kernel<BITS, 1>),       \
      reinterpret_cast<const void*>(&gemv_batch_kernel<BITS, 2>)
      MING_GEMV_ALL(4), MING_GEMV_ALL(8), MING_GEMV_ALL(16),
#undef MING_GEMV_ALL
      reinterpret_cast<const void*>(&gemv_kernel<4, 4, 2>),
      reinterpret_cast<const void*>(&gemv_kernel<4, 8, 2>),
      reinterpret_cast<const void*>(&gemv_kernel<8, 4, 2>),
      reinterpret_cast<const void*>(&gemv_kernel<8, 8, 2>)};
  for (const void* f : fns) {
    const hipError_t e = hipFuncGetAttributes(&fa, f);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace ming
