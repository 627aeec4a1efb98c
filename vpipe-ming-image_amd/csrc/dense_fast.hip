// Dense bf16 projections (a dense checkpoint's blocks, the language
// encoder's linears) on MI355X: y = [x | T] . [W | B_live]^T with W the
// checkpoint's own bf16 [N][K], the contract of qproj_kernel<16> (qproj.hip).
//
// MFMA-bound. Block tile 64*RF rows x 256 columns, 8 wave64s in 2 x 4, each
// 32*RF rows x 64 columns (2 x RF tiles of v_mfma_f32_32x32x16_bf16, two waves
// a SIMD). K is walked in stages of 64 (whole 128-byte rows: with stages of 32
// the same kernel moved 26 B/clk a CU and took 107 us where it now takes 97,
// [4352, 3840] x [3840, 3840]) through an LDS ring filled by direct
// global->LDS DMA: three stages where they fit (RF <= 2), else five 32 KB
// slots (the CU's 160 KB) taken by x and W tiles in turn, so that x runs three
// stages ahead and W two. Two waves a SIMD hide each other's DMA issue,
// fragment reads and barrier: four waves of twice the columns took 274 us
// where these take 261, [4352, 3840] x [10240, 3840] (1313 TFLOP/s; the
// general kernel 386 us).
//
// One barrier a stage, before its last k16 step: each step's MFMAs run beside
// the next step's fragment reads, the last step's beside the next stage's
// first. After the barrier both tiles of stage t are free. The LoRA tail is
// the same ring over T and the gathered B rows, two chunks of 32 ranks a stage.
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "lds_ring.h"

namespace ming {
namespace {

constexpr int DBN = 256, DBK = 64, NW = 8;

// EPI: 0 plain; 1 a.bias added before the output's one rounding; 2 gated by
// a.g (the fused SwiGLU); 3 plain, a.nw projections over one x. One instance
// each: with the first three in one the 256-row tile's epilogue spilled
// registers.
template <int RF, int EPI>
__global__ __launch_bounds__(64 * NW, 1) void dense_fast_kernel(const QprojArgs a) {
  constexpr int BMT = 64 * RF;
  constexpr int XD = 8 * RF / NW, WD = 32 / NW;   // DMAs per wave per stage
  constexpr int JF = 16 / NW;              // column fragments per wave
  constexpr bool FIVE = RF >= 3;           // five slots of 32 KB, else three stages
  constexpr int XCH = BMT * 8, WCH = DBN * 8;   // 16-B chunks of the tiles
  constexpr int PERIOD = FIVE ? 5 : 3;
  __shared__ uint4 ring[FIVE ? 5 * WCH : 3 * (XCH + WCH)];
  // stage t's tiles, t given by its phase t % PERIOD
  auto xslot = [&](int ph) -> const uint4* {
    return FIVE ? ring + ((2 * ph) % 5) * WCH : ring + (ph % 3) * (XCH + WCH);
  };
  auto wslot = [&](int ph) -> const uint4* {
    return FIVE ? ring + ((2 * ph + 1) % 5) * WCH : ring + (ph % 3) * (XCH + WCH) + XCH;
  };
  // after stage t's barrier its two tiles are free: W of stage t + WAHEAD and
  // x of stage t + 3 go there
  constexpr int WAHEAD = FIVE ? 2 : 3;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, fk = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;

  const int tiles_m = (a.M + BMT - 1) / BMT;
  const int tiles_n = (a.N + DBN - 1) / DBN;
  int tm, tn;
  tile_of_block((int)blockIdx.x, tiles_m, EPI == 3 ? a.nw * tiles_n : tiles_n, &tm, &tn);
  int wsel = 0;                            // the tile's projection
  if constexpr (EPI == 3) {
    wsel = tn / tiles_n;
    tn -= wsel * tiles_n;
  }
  const uint16_t* const w16 = EPI == 3 && wsel > 0 ? a.more[wsel - 1].w16 : a.w16;
  uint16_t* const yout = EPI == 3 && wsel > 0 ? a.more[wsel - 1].y : a.y;
  const int m0 = tm * BMT, n0 = tn * DBN;
  const int mlast = a.M - 1, nlast = a.N - 1;
  const int KT = a.K / DBK;

  // LDS chunk p of a tile holds row p >> 3, logical chunk (p & 7) ^ swizzle.
  // Byte offsets from the stage's base; the host keeps both operands within
  // 2 GiB of theirs.
  auto row_of = [&](int p) { return p >> 3; };
  auto chunk_of = [&](int p) { return (p & 7) ^ (((p >> 3) >> 1) & 7); };
  uint32_t xoff[XD], woff[WD];
#pragma unroll
  for (int i = 0; i < XD; ++i) {
    const int p = 64 * (XD * wave + i) + lane;
    int mr = m0 + row_of(p);
    mr = mr < mlast ? mr : mlast;
    xoff[i] = (uint32_t)(((long long)mr * a.ldx + 8 * chunk_of(p)) * 2);
  }
#pragma unroll
  for (int i = 0; i < WD; ++i) {
    const int p = 64 * (WD * wave + i) + lane;
    int n = n0 + row_of(p);
    n = n < nlast ? n : nlast;
    woff[i] = (uint32_t)(((long long)n * a.K + 8 * chunk_of(p)) * 2);
  }

  floatx16_t acc[JF][RF];
#pragma unroll
  for (int j = 0; j < JF; ++j)
#pragma unroll
    for (int i = 0; i < RF; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.0f;

  uint4 wa[JF], xb[RF];
  auto read_frags = [&](const uint4* X, const uint4* W, int kk, uint4 (&av)[JF],
                        uint4 (&bv)[RF]) {
    const int c = 2 * kk + fk;
#pragma unroll
    for (int j = 0; j < JF; ++j) av[j] = W[swz8(32 * JF * wn + 32 * j + fr, c)];
#pragma unroll
    for (int i = 0; i < RF; ++i) bv[i] = X[swz8(32 * RF * wm + 32 * i + fr, c)];
  };
  // One stage of phase PH. iw(t, S) / ix(t, S, h) issue stage t's W DMAs and
  // half h of its x DMAs.
  auto body = [&](auto ph, int t, auto&& iw, auto&& ix) {
    constexpr int PH = decltype(ph)::value;
    const uint4 *const X = xslot(PH), *const W = wslot(PH);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      uint4 an[JF], bn[RF];
      if (kk < 2) ix(t + 2, xslot((PH + 2) % PERIOD), kk);   // freed by stage t - 1
      if (kk == 3) iw(t + WAHEAD, wslot((PH + WAHEAD) % PERIOD));
      if (kk < 3) {
        read_frags(X, W, kk + 1, an, bn);
      } else {
        read_frags(xslot((PH + 1) % PERIOD), wslot((PH + 1) % PERIOD), 0, an, bn);
      }
#pragma unroll
      for (int i = 0; i < RF; ++i)
#pragma unroll
        for (int j = 0; j < JF; ++j)
          acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8_t, wa[j]), __builtin_bit_cast(bf16x8_t, xb[i]),
              acc[j][i], 0, 0, 0);
      // the reads one per MFMA (two at RF 1, which has four MFMAs a step)
      constexpr int DPM = JF * RF >= JF + RF ? 1 : 2;
#pragma unroll
      for (int g = 0; g < (JF + RF + DPM - 1) / DPM; ++g) {
        __builtin_amdgcn_sched_group_barrier(0x100, DPM, 0);   // DS read
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // MFMA
      }
      __builtin_amdgcn_sched_barrier(0);
      if (kk == 2) {
        // stage t + 1 landed; newer: x of stage t + 2 (and W, three stages)
        ring_wait<XD + (FIVE ? 0 : WD)>();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < JF; ++j) wa[j] = an[j];
#pragma unroll
      for (int i = 0; i < RF; ++i) xb[i] = bn[i];
    }
  };
  // n stages through the ring. Past the last one the DMA re-reads it into a
  // tile nothing reads, so every stage issues and waits alike.
  auto walk = [&](int n, auto&& iw, auto&& ix) {
    const std::integral_constant<int, 0> p0{};
    const std::integral_constant<int, 1> p1{};
    const std::integral_constant<int, 2> p2{};
    iw(0, wslot(0));
    ix(0, xslot(0), 0);
    ix(0, xslot(0), 1);
    ix(1, xslot(1), 0);
    ix(1, xslot(1), 1);
    iw(1, wslot(1));
    if constexpr (!FIVE) iw(2, wslot(2));
    // stage 0 landed; newer: stage 1 (and W of stage 2)
    ring_wait<XD + (FIVE ? WD : 2 * WD)>();
    read_frags(xslot(0), wslot(0), 0, wa, xb);
    int t = 0;
    for (; t + PERIOD <= n; t += PERIOD) {
      body(p0, t, iw, ix);
      body(p1, t + 1, iw, ix);
      body(p2, t + 2, iw, ix);
      if constexpr (FIVE) {
        body(std::integral_constant<int, 3>{}, t + 3, iw, ix);
        body(std::integral_constant<int, 4>{}, t + 4, iw, ix);
      }
    }
    if (n - t >= 1) body(p0, t, iw, ix);
    if (n - t >= 2) body(p1, t + 1, iw, ix);
    if constexpr (FIVE) {
      if (n - t >= 3) body(p2, t + 2, iw, ix);
      if (n - t >= 4) body(std::integral_constant<int, 3>{}, t + 3, iw, ix);
    }
    ring_wait<0>();                        // drained; LDS free
  };

  walk(
      KT,
      [&](int t, const uint4* S) {
        const void* base = w16 + (long long)(t < KT ? t : KT - 1) * DBK;
#pragma unroll
        for (int i = 0; i < WD; ++i) dma16_sb(base, woff[i], lds_addr(S + 64 * (WD * wave + i)));
      },
      [&](int t, const uint4* S, int h) {
        const void* base = a.x + (long long)(t < KT ? t : KT - 1) * DBK;
#pragma unroll
        for (int i = h ? XD / 2 : 0; i < (h ? XD : XD / 2); ++i)
          dma16_sb(base, xoff[i], lds_addr(S + 64 * (XD * wave + i)));
      });

  // ---- LoRA tail: T and gathered B, two chunks of 32 ranks a stage ----
  int sg = 0;
  for (int i = 1; i < a.nseg; ++i)
    if (n0 >= a.seg[i].n_begin) sg = i;
  const QprojSeg& s = EPI == 3 && wsel > 0 ? a.more[wsel - 1].seg : a.seg[sg];
  const int chunks = s.chunks;
  if (chunks > 0) {
    const int grp0 = s.grp0;
    // a padding group's T columns are exactly 0: any finite B will do, the
    // first live group's
    const int g_safe = a.grp[grp0];
    uint32_t toff[XD], boff[WD];
#pragma unroll
    for (int i = 0; i < XD; ++i) {
      const int p = 64 * (XD * wave + i) + lane;
      int mr = m0 + row_of(p);
      mr = mr < mlast ? mr : mlast;
      toff[i] = (uint32_t)(((long long)mr * a.ldt + s.t_col0 + 8 * chunk_of(p)) * 2);
    }
#pragma unroll
    for (int i = 0; i < WD; ++i) {
      const int p = 64 * (WD * wave + i) + lane;
      int n = n0 + row_of(p);
      n = n < s.n_end - 1 ? n : s.n_end - 1;
      boff[i] = (uint32_t)((long long)(n - s.n_begin) * s.ldb * 2);
    }
    const int n2 = chunks / 2;
    // stage st of the tail; `half`: it holds one chunk, the second half of its
    // tiles (never multiplied) re-reads the first, in bounds
    auto issue_b = [&](int st, const uint4* S, bool half) {
      // the stage's eight groups: two aligned 8-byte words of the table
      const uint2* gp = reinterpret_cast<const uint2*>(a.grp) +
                        (__builtin_amdgcn_readfirstlane(grp0 + 8 * st) >> 2);
      const uint2 g0 = gp[0], g1 = gp[half ? 0 : 1];
#pragma unroll
      for (int i = 0; i < WD; ++i) {
        const int c = chunk_of(64 * (WD * wave + i) + lane);
        const uint2 gw = (c & 4) ? g1 : g0;
        const uint32_t w = (c & 2) ? gw.y : gw.x;
        int g = (int16_t)(w >> ((c & 1) << 4));
        g = g < 0 ? g_safe : g;
        dma16_sb(s.B, boff[i] + (uint32_t)g * 16u, lds_addr(S + 64 * (WD * wave + i)));
      }
    };
    auto issue_t = [&](int st, const uint4* S, int h, bool half) {
#pragma unroll
      for (int i = h ? XD / 2 : 0; i < (h ? XD : XD / 2); ++i) {
        const int c = chunk_of(64 * (XD * wave + i) + lane);
        dma16_sb(a.t + 64 * st, toff[i] - (half && (c & 4) ? 64u : 0u),
                 lds_addr(S + 64 * (XD * wave + i)));
      }
    };
    if (n2 > 0)
      walk(
          n2, [&](int t, const uint4* S) { issue_b(t < n2 ? t : n2 - 1, S, false); },
          [&](int t, const uint4* S, int h) { issue_t(t < n2 ? t : n2 - 1, S, h, false); });
    if (chunks & 1) {
      // the odd last chunk by itself: inside the pipelined walk its case
      // would double the accumulators' registers
      issue_b(n2, wslot(0), true);
      issue_t(n2, xslot(0), 0, true);
      issue_t(n2, xslot(0), 1, true);
      ring_wait<0>();
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        read_frags(xslot(0), wslot(0), kk, wa, xb);
#pragma unroll
        for (int i = 0; i < RF; ++i)
#pragma unroll
          for (int j = 0; j < JF; ++j)
            acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8_t, wa[j]), __builtin_bit_cast(bf16x8_t, xb[i]),
                acc[j][i], 0, 0, 0);
      }
      ring_wait<0>();                      // every wave's reads done: LDS free
    }
  }

  // Epilogue through LDS: each wave converts 64 columns x up to 128 rows at
  // a time to bf16 in its own region (rows of 128 B, chunks swizzled by
  // (row >> 1) & 7: conflict-free both ways), then stores whole 128-B row
  // segments. Only the wave itself touches its region and its LDS accesses
  // complete in order: no barrier.
  constexpr int RROWS = 32 * RF;
  uint4* const E = ring + (RROWS * 8) * wave;
  uint2* const E2 = reinterpret_cast<uint2*>(E);
  const bool st16 = (a.ldy & 7) == 0 && (reinterpret_cast<uintptr_t>(yout) & 15) == 0;
  const int cl = lane & 7;
#pragma unroll
  for (int h = 0; h < JF / 2; ++h) {
    const int nb = n0 + 32 * JF * wn + 64 * h;       // the half's first column
    const int n = nb + 8 * cl;
    // fused SwiGLU: the gate's rows are loaded first, their latency under the
    // conversion
    [[maybe_unused]] uint4 gv[4 * RF];
    if constexpr (EPI == 2) {
#pragma unroll
      for (int r = 0; r < 4 * RF; ++r) {
        int mr = m0 + RROWS * wm + 8 * r + (lane >> 3);
        mr = mr < a.M ? mr : mlast;
        const int nn = n < a.N ? n : a.N - 8;
        gv[r] = *reinterpret_cast<const uint4*>(a.g + (long long)mr * a.ldg + nn);
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        [[maybe_unused]] float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (EPI == 1) {
          const int nn = nb + 32 * j + 8 * q + 4 * fk;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (nn + e < a.N) b[e] = bf16_to_f32(a.bias[nn + e]);
        }
#pragma unroll
        for (int i = 0; i < RF; ++i) {
          const int ml = 32 * i + fr;
          const int c = 4 * j + q;
          const floatx16_t& v = acc[2 * h + j][i];
          uint2 o;
          if constexpr (EPI == 1) {
            o.x = pack_bf16x2_rne(v[4 * q + 0] + b[0], v[4 * q + 1] + b[1]);
            o.y = pack_bf16x2_rne(v[4 * q + 2] + b[2], v[4 * q + 3] + b[3]);
          } else {
            o.x = pack_bf16x2_rne(v[4 * q + 0], v[4 * q + 1]);
            o.y = pack_bf16x2_rne(v[4 * q + 2], v[4 * q + 3]);
          }
          E2[ml * 16 + 2 * (c ^ ((ml >> 1) & 7)) + fk] = o;
        }
      }
#pragma unroll
    for (int r = 0; r < 4 * RF; ++r) {
      const int ml = 8 * r + (lane >> 3);
      uint4 v = E[ml * 8 + (cl ^ ((ml >> 1) & 7))];
      const int mr = m0 + RROWS * wm + ml;
      if (mr < a.M && n < a.N) {
        if constexpr (EPI == 2) {
          const uint32_t* gp = &gv[r].x;
          uint32_t* vp = &v.x;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            vp[e] = pack_bf16x2_rne(silu_f(bf16_lo(gp[e])) * bf16_lo(vp[e]),
                                    silu_f(bf16_hi(gp[e])) * bf16_hi(vp[e]));
        }
        uint16_t* yp = yout + (long long)mr * a.ldy + n;
        if (st16) {
          *reinterpret_cast<uint4*>(yp) = v;
        } else {
          reinterpret_cast<uint2*>(yp)[0] = make_uint2(v.x, v.y);
          reinterpret_cast<uint2*>(yp)[1] = make_uint2(v.z, v.w);
        }
      }
    }
  }
}

}  // namespace

// Rounds of the chip, one block a CU, times a block's time: about 24 + 10 rf
// us for 60 K stages (one round, measured at [1280, 3840] x [3840, 3840]: rf 2
// 44, rf 3 54, rf 4 64 us), near the same ratio at other K: of the four heights
// at 300 to 16640 rows and K = 64 to 10240 it takes the fastest in 101 of 104
// shapes, one within 3% in the others.
static double dense_us(int M, int N, int nw, int rf) {
  const long long tiles =
      (long long)((M + 64 * rf - 1) / (64 * rf)) * ((N + DBN - 1) / DBN) * nw;
  const int cus = device_cus();
  return (double)((tiles + cus - 1) / cus) * (24 + 10 * rf);
}

int dense_fast_rf(int M, int N, int nw) {
  int best = 4;
  for (int rf = 3; rf >= 1; --rf)
    if (dense_us(M, N, nw, rf) < dense_us(M, N, nw, best)) best = rf;
  return best;
}

// Fewer rounds of the chip in one launch than in one each: three of [2560,
// 3840] x [3840, 3840] two of 256-row tiles for three of 192-row ones (a block
// 1101 us with three launches, 1059 with one).
bool dense_merge_pays(int M, int N, int nw) {
  return dense_us(M, N, nw, dense_fast_rf(M, N, nw)) <
         0.95 * nw * dense_us(M, N, 1, dense_fast_rf(M, N));
}

template <int RF>
static void launch_rf(const QprojArgs& a, hipStream_t s) {
  const int nw = a.nw > 1 ? a.nw : 1;
  const dim3 grid((unsigned)(((a.M + 64 * RF - 1) / (64 * RF)) * ((a.N + DBN - 1) / DBN) * nw));
  if (nw > 1)
    hipLaunchKernelGGL((dense_fast_kernel<RF, 3>), grid, dim3(64 * NW), 0, s, a);
  else if (a.bias)
    hipLaunchKernelGGL((dense_fast_kernel<RF, 1>), grid, dim3(64 * NW), 0, s, a);
  else if (a.g)
    hipLaunchKernelGGL((dense_fast_kernel<RF, 2>), grid, dim3(64 * NW), 0, s, a);
  else
    hipLaunchKernelGGL((dense_fast_kernel<RF, 0>), grid, dim3(64 * NW), 0, s, a);
}

hipError_t launch_dense_fast(const QprojArgs& a, int rf, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (a.N % 8 != 0 || a.K % 64 != 0 || a.kslices > 1 || a.yh || (a.bias && a.g) ||
      (a.nw > 1 && (a.nw > 3 || a.nseg != 1 || a.bias || a.g)))
    return hipErrorInvalidValue;
  switch (rf) {
    case 1: launch_rf<1>(a, s); break;
    case 2: launch_rf<2>(a, s); break;
    case 3: launch_rf<3>(a, s); break;
    case 4: launch_rf<4>(a, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <int RF>
static hipError_t validate_rf() {
  hipFuncAttributes fa;
  const void* fns[] = {reinterpret_cast<const void*>(&dense_fast_kernel<RF, 0>),
                       reinterpret_cast<const void*>(&dense_fast_kernel<RF, 1>),
                       reinterpret_cast<const void*>(&dense_fast_kernel<RF, 2>),
                       reinterpret_cast<const void*>(&dense_fast_kernel<RF, 3>)};
  for (const void* f : fns) {
    const hipError_t e = hipFuncGetAttributes(&fa, f);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t validate_dense_fast_kernels() {
  hipError_t e = validate_rf<1>();
  if (e == hipSuccess) e = validate_rf<2>();
  if (e == hipSuccess) e = validate_rf<3>();
  if (e == hipSuccess) e = validate_rf<4>();
  return e;
}

}  // namespace ming
