// The quantized projection's fast route on MI355X (gfx950): a three-stage
// LDS ring filled by direct global->LDS DMA (global_load_lds_dwordx4), raw
// int codes dequantized per MFMA fragment with packed-fp16 arithmetic,
// and the LoRA tail through the same ring.
//
// Same contract as qproj_kernel (y = [x | T] . [W_dq | B_live]^T, see
// qproj.hip), with two preconditions the host checks:
//   * x arrives as fp16 carrying bf16 values (exact inside fp16's range);
//   * every scale and bias of the weight is exact in fp16, so the weight
//     is dequantized as fp16(fma(code, s, b)) with ONE rounding by
//     v_pk_fma_f16 on the exact integer code (built with the 0x6400 magic:
//     (0x6400 | c) is 1024 + c in fp16, and 1024 is subtracted exactly).
//
// Per block: tile 32*RF(M) x 256(N) x 64(K). At 256 rows 4 wave64s split N,
// each owning 64 columns x all rows (2 x 8 tiles of v_mfma_f32_32x32x16_f16),
// so each weight is dequantized once; the lower tiles (kTiles) run 8 waves of
// 32 columns. Per stage the DMA moves the fp16 x tile (32 KB at 256 rows), the
// code tile (8 KB w4 / 16 KB w8) and 256 fp16 (scale, bias) pairs. No VGPR
// round trip, and each wave waits on its own vmcnt for the stage two behind
// the one in flight.
//
// The same body also runs as qproj_pair_kernel (a SwiGLU's gate and up
// projections in one tile, 128 columns of each), and split along K (few tiles).
//
// Resident code layout this kernel reads (built by repack_*_fast):
//   w4: codes[kt][n][fk][kk]   one u32 = the 8 codes of k = 16kk + 8fk + 0..7,
//       nibbles ordered {k0,k4,k1,k5,k2,k6,k3,k7} so w & 0x0F0F0F0F holds
//       k0..k3 one per byte and (w >> 4) & 0x0F0F0F0F holds k4..k7
//   w8: codes[kt][n][fk][kk][2] two u32 = those 8 codes, bytes in k order
//   sbf[kt][n] = fp16 scale | fp16 bias << 16
#include <atomic>

#include "common.h"
#include "kernels.h"
#include "lds_ring.h"

namespace ming {
namespace {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

constexpr int BM = 256, BN = 256, BK = 64;

// 8 codes (one w4 word) -> 8 fp16 dequantized values. The word's nibbles
// are ordered {k0,k4,k1,k5,k2,k6,k3,k7}, so lo = w & 0x0F0F0F0F holds
// k0..k3 one per byte and hi = (w >> 4) & 0x0F0F0F0F holds k4..k7; one
// v_perm per pair then lays a code under the 0x64 magic byte.
__device__ __forceinline__ uint4 deq_w4(uint32_t w, half2v s2, half2v b2) {
  const half2v k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
  const uint32_t lo = w & 0x0F0F0F0Fu;
  const uint32_t hi = (w >> 4) & 0x0F0F0F0Fu;
  uint32_t v[4];
  v[0] = __builtin_amdgcn_perm(0x64646464u, lo, 0x05010400u);
  v[1] = __builtin_amdgcn_perm(0x64646464u, lo, 0x05030402u);
  v[2] = __builtin_amdgcn_perm(0x64646464u, hi, 0x05010400u);
  v[3] = __builtin_amdgcn_perm(0x64646464u, hi, 0x05030402u);
  uint4 o;
  uint32_t* op = &o.x;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const half2v c = __builtin_bit_cast(half2v, v[p]) - k1024;
    op[p] = __builtin_bit_cast(uint32_t, c * s2 + b2);
  }
  return o;
}

// 8 codes (two w8 words, bytes in k order) -> 8 fp16.
__device__ __forceinline__ uint4 deq_w8(uint32_t w0, uint32_t w1, half2v s2,
                                        half2v b2) {
  const half2v k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
  uint32_t v[4];
  v[0] = __builtin_amdgcn_perm(0x64646464u, w0, 0x05010400u);
  v[1] = __builtin_amdgcn_perm(0x64646464u, w0, 0x05030402u);
  v[2] = __builtin_amdgcn_perm(0x64646464u, w1, 0x05010400u);
  v[3] = __builtin_amdgcn_perm(0x64646464u, w1, 0x05030402u);
  uint4 o;
  uint32_t* op = &o.x;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const half2v c = __builtin_bit_cast(half2v, v[p]) - k1024;
    op[p] = __builtin_bit_cast(uint32_t, c * s2 + b2);
  }
  return o;
}

// Code-chunk swizzle inside a row group: chunk h of row n sits at
// n*CPR + (h ^ sw(n)), so the 16 rows a fragment read serves per LDS cycle
// land on distinct banks (rows are 32 B (w4) / 64 B (w8) apart).
template <int CPR>
__device__ __forceinline__ int wswz(int n) {
  return CPR == 2 ? ((n >> 3) & 1) : ((n >> 2) & 3);
}
template <int CPR>
__device__ __forceinline__ int wchunk(int n, int h) {
  return n * CPR + (h ^ wswz<CPR>(n));
}

// SPLIT (a.kslices > 1, a projection of few tiles): block b is slice
// b / tiles of tile b % tiles. The slice runs its share of K (the last one
// also the LoRA tail) and writes f32 partials to a.part; the split reduce
// then sums the slices in order and finishes as the epilogue does.
//
// PAIR (launch_qproj_pair): the tile's 256 weight rows are 128 rows of the
// gate weight (the first half of the waves) and the same 128 rows of the up
// weight (the second half); the tail stages the gate's and the up projection's T chunks side by
// side; the epilogue meets the two in LDS and writes only the SwiGLU. MULTI
// (qproj_merged_kernel): a.nw projections over one x, their column tiles side
// by side in the tile grid.
template <int BITS, bool SPLIT, bool PAIR, int RF, int NW, bool MULTI = false>
__device__ __forceinline__ void qproj_fast_body(const QprojArgs& a) {
  constexpr int WCH = BITS == 4 ? 512 : 1024;    // 16-B code chunks per stage
  constexpr int CPR = BITS == 4 ? 2 : 4;         // code chunks per row
  constexpr int WDMA = WCH / (64 * NW);          // code DMAs per wave per stage
  constexpr int JT = 8 / NW;                     // 32-column tiles per wave
  constexpr int BMT = 32 * RF;                   // rows per tile: RF fragments of 32
  constexpr int XD = 4 * RF / NW;                // x DMAs per wave per stage
  static_assert(XD * NW == 4 * RF, "x DMAs divide among the waves");
  constexpr int TD = (2 * RF + NW - 1) / NW;     // T DMAs per wave per tail chunk
  constexpr int BD = 16 / NW;                    // B DMAs per wave per tail chunk
  constexpr int PER = XD + WDMA + 1;             // DMAs per wave per base stage
  constexpr int TPER = (PAIR ? 2 : 1) * TD + BD; // DMAs per wave per tail chunk
  constexpr int BNT = PAIR ? BN / 2 : BN;        // output columns per tile
  // A stage is [x tile | codes | (s, b)], a tail chunk [T | B (| the up
  // projection's T)]; the epilogue takes four 16 KB regions.
  constexpr int TRG = 64 * NW * TD;              // a tail chunk's T region
  constexpr int STG0 = BMT * 8 + WCH + BN / 4;
  constexpr int TSTG = (PAIR ? 2 : 1) * TRG + 1024;
  constexpr int STG = STG0 < TSTG ? TSTG : STG0;
  // One object a stage where each holds two epilogue regions: in one array the
  // compiler builds each address past 64 KB with a VALU op of its own (the w4
  // paired launch at 256 rows: 48 more in three stages, 574.8 us against 568).
  constexpr bool SEP = STG >= 2048;
  __shared__ uint4 ring0[SEP ? STG : 3 * STG < 4096 ? 4096 : 3 * STG];
  __shared__ uint4 ring1[SEP ? STG : 1], ring2[SEP ? STG : 1];
  static_assert(3 * STG <= 10240, "the CU's 160 KB");
  uint4* const st0 = ring0;
  uint4* const st1 = SEP ? ring1 : ring0 + STG;
  uint4* const st2 = SEP ? ring2 : ring0 + 2 * STG;
  auto region = [&](int r) { return SEP ? (r < 2 ? st0 : st1) + 1024 * (r & 1) : st0 + 1024 * r; };

  // Waves split N only: wave w owns the 32*JT output columns from 32*JT*w for
  // all of the tile's rows, so every weight fragment is dequantized by exactly
  // one wave.
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 31, fk = lane >> 5;
  // PAIR: the second half of the waves reads the up weight; their columns are
  // the gate's again
  const bool upw = PAIR && wave >= NW / 2;

  const int tiles_m = (a.M + BMT - 1) / BMT;
  const int tiles_n = (a.N + BNT - 1) / BNT;
  int tm, tn, blk = (int)blockIdx.x, ks = 0, kt0 = 0;
  int KT = a.K / BK;
  const int tiles_all = MULTI ? a.nw * tiles_n : tiles_n;
  if constexpr (SPLIT) {
    ks = blk / (tiles_m * tiles_all);
    blk -= ks * (tiles_m * tiles_all);
  }
  tile_of_block(blk, tiles_m, tiles_all, &tm, &tn);
  int wsel = 0;                                  // MULTI: the tile's projection
  if constexpr (MULTI) {
    wsel = tn / tiles_n;
    tn -= wsel * tiles_n;
  }
  const int m0 = tm * BMT, n0 = tn * BNT;
  const int mlast = a.M - 1, nlast = a.N - 1;
  int sg = 0;                                    // the tile's segment
  for (int i = 1; i < a.nseg; ++i)
    if (n0 >= a.seg[i].n_begin) sg = i;
  const QprojSeg& seg = MULTI && wsel > 0 ? a.more[wsel - 1].seg : a.seg[sg];
  uint16_t* const yout = MULTI && wsel > 0 ? a.more[wsel - 1].y : a.y;
  if constexpr (SPLIT) {
    // the last slice also runs the LoRA tail, a chunk of it about 5/8 of a
    // stage: it takes that much less of K (at least one stage each)
    const int total = KT + seg.chunks * 5 / 8;
    auto bound = [&](int i) {
      const int b = total * i / a.kslices, m = KT - (a.kslices - i);
      return b < m ? b : m;
    };
    kt0 = bound(ks);
    KT = bound(ks + 1) - kt0;
  }

  // stage 0 of this block's K range
  const _Float16* __restrict__ x16 = reinterpret_cast<const _Float16*>(a.x) + (long long)kt0 * BK;
  const uint4* __restrict__ codes =
      reinterpret_cast<const uint4*>(MULTI && wsel > 0 ? a.more[wsel - 1].codes
                                     : upw           ? a.codes_u
                                                     : a.codes) +
      (long long)kt0 * a.N * CPR;
  const uint32_t* __restrict__ sbp =
      (MULTI && wsel > 0 ? a.more[wsel - 1].sb : upw ? a.sb_u : a.sb) + (long long)kt0 * a.N;

  // DMA sources for this lane, per stage (advance by k).
  // x tile: wave issues chunks q = XD*wave + i; lane p = 64q + lane.
  // Byte offsets from the stage's base (the host keeps every operand
  // within 2 GiB of its base, so they fit 31 bits whether the hardware reads
  // the offset as signed or unsigned).
  uint32_t xoff[XD];
#pragma unroll
  for (int i = 0; i < XD; ++i) {
    const int p = 64 * (XD * wave + i) + lane;
    const int row = p >> 3;
    const int c = (p & 7) ^ ((row >> 1) & 7);
    int m = m0 + row;
    m = m < mlast ? m : mlast;
    xoff[i] = (uint32_t)(((long long)m * a.ldx + 8 * c) * 2);
  }
  // code tile: LDS chunk p holds row p / CPR, logical chunk (p % CPR) ^ sw
  uint32_t woff[WDMA];
#pragma unroll
  for (int i = 0; i < WDMA; ++i) {
    const int p = 64 * (WDMA * wave + i) + lane;
    const int r = p / CPR;
    const int h = (p % CPR) ^ wswz<CPR>(r);
    int n = n0 + (PAIR ? (r & 127) : r);
    n = n < nlast ? n : nlast;
    woff[i] = (uint32_t)((n * CPR + h) * 16);
  }
  // (s, b): 64 columns a wave from sst; with eight waves the runs overlap
  // (the same values), never across the tile's halves
  const int sst = NW == 4 ? 64 * wave : 128 * (wave >> 2) + (32 * (wave & 3) < 64 ? 32 * (wave & 3) : 64);
  int sn = n0 + (PAIR ? sst & 127 : sst) + lane;
  sn = sn < nlast ? sn : nlast;
  const uint32_t soff = (uint32_t)sn * 4u;

  // The stage's DMAs in three groups (the wave's x DMAs in two halves, codes +
  // (s, b)), issued one group per k16 step of the stage before.
  auto issue_grp = [&](int g, int kt, const uint4* B) {
    if (g < 2) {
      const void* base = x16 + (long long)kt * BK;
#pragma unroll
      for (int i = g ? XD / 2 : 0; i < (g ? XD : XD / 2); ++i)
        dma16_sb(base, xoff[i], lds_addr(B + 64 * (XD * wave + i)));
    } else {
      const void* wbase = codes + (long long)kt * a.N * CPR;
#pragma unroll
      for (int i = 0; i < WDMA; ++i)
        dma16_sb(wbase, woff[i], lds_addr(B + BMT * 8 + 64 * (WDMA * wave + i)));
      dma4_sb(sbp + (long long)kt * a.N, soff,
              lds_addr(reinterpret_cast<const uint32_t*>(B + BMT * 8 + WCH) + sst));
    }
  };

  floatx16_t acc[JT][RF];
#pragma unroll
  for (int j = 0; j < JT; ++j)
#pragma unroll
    for (int i = 0; i < RF; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[j][i][r] = 0.0f;

  // Stage state in registers: the code words and (s, b) of the wave's
  // n-tiles, and the current k16 step's operands.
  uint4 wc[JT][CPR / 2];
  half2v s2[JT], b2[JT];
  uint4 wa[JT], xb[RF];

  auto load_ws = [&](const uint4* B, uint4 (&wcv)[JT][CPR / 2], half2v (&s2v)[JT],
                     half2v (&b2v)[JT]) {
    const uint4* W = B + BMT * 8;
    const uint32_t* S = reinterpret_cast<const uint32_t*>(B + BMT * 8 + WCH);
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      const int n = 32 * JT * wave + 32 * j + fr;
#pragma unroll
      for (int h = 0; h < CPR / 2; ++h)
        wcv[j][h] = W[wchunk<CPR>(n, fk * (CPR / 2) + h)];
      const uint32_t sb = S[n];
      s2v[j] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(sb, sb, 0x01000100u));
      b2v[j] = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(sb, sb, 0x03020302u));
    }
  };
  auto deq = [&](const uint4 (&wcv)[JT][CPR / 2], const half2v (&s2v)[JT],
                 const half2v (&b2v)[JT], int j, int kk) -> uint4 {
    if constexpr (BITS == 4) {
      return deq_w4((&wcv[j][0].x)[kk], s2v[j], b2v[j]);
    } else {
      const uint32_t* w = &wcv[j][kk >> 1].x;
      return deq_w8(w[(kk & 1) * 2], w[(kk & 1) * 2 + 1], s2v[j], b2v[j]);
    }
  };

  // One stage, software-pipelined across the stage boundary. Steps 0-2
  // read and dequantize the next step's fragments beside the current
  // step's MFMAs and issue one DMA group of stage kt+2 into Pv (the
  // buffer stage kt-1 left). Between steps 2 and 3 the wave waits for its
  // stage kt+1 DMAs and the workgroup meets at the barrier: stage kt+1 is
  // in LDS and nobody reads stage kt's buffer again. Step 3's MFMAs then
  // carry the next stage's code / (s, b) reads, its first x fragments and
  // their dequantization, so no stage starts with an LDS round trip.
  // Interleave pinned with scheduling-group barriers (0x008 MFMA, 0x100 DS
  // read, 0x002 VALU). Past the last stage the DMA re-reads stage KT-1 into
  // a buffer nothing reads, so every stage issues and waits alike.
  auto body = [&](int kt, const uint4* C, const uint4* Nx, const uint4* Pv) {
    const int nk = kt + 2 < KT ? kt + 2 : KT - 1;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      uint4 wn_[JT], xn_[RF];
      uint4 wcn[JT][CPR / 2];
      half2v s2n[JT], b2n[JT];
      if (kk < 3) {
        issue_grp(kk, nk, Pv);
#pragma unroll
        for (int i = 0; i < RF; ++i) xn_[i] = C[swz8(32 * i + fr, 2 * (kk + 1) + fk)];
#pragma unroll
        for (int j = 0; j < JT; ++j) wn_[j] = deq(wc, s2, b2, j, kk + 1);
      } else {
        load_ws(Nx, wcn, s2n, b2n);
#pragma unroll
        for (int i = 0; i < RF; ++i) xn_[i] = Nx[swz8(32 * i + fr, fk)];
#pragma unroll
        for (int j = 0; j < JT; ++j) wn_[j] = deq(wcn, s2n, b2n, j, 0);
      }
#pragma unroll
      for (int i = 0; i < RF; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j)
          acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              __builtin_bit_cast(half8_t, wa[j]), __builtin_bit_cast(half8_t, xb[i]),
              acc[j][i], 0, 0, 0);
      if constexpr (NW == 8) {
        // two waves a SIMD: only the reads are pinned ahead of the MFMAs
#pragma unroll
        for (int g = 0; g < RF; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, 16 / RF, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
      } else if (kk < 3) {
#pragma unroll
        for (int g = 0; g < RF; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // DS read
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
        }
#pragma unroll
        for (int g = 0; g < RF; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x002, (32 + RF - 1) / RF, 0);   // VALU
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                    // MFMA
        }
      } else {
        // step 3: NDS reads over the DSM MFMAs left after the VG that carry
        // the next stage's first dequantization (w4 at 256 rows: spread
        // over 10 MFMAs, 4 VALU each, which measured ~0.5% faster launches
        // than 6 MFMAs of 6; the reads then go two per MFMA)
        constexpr int NDS = RF + JT * (CPR / 2) + JT;
        constexpr int VG = RF == 8 && CPR == 2 ? RF + 2 : 3 * RF / 4;
        constexpr int VPG = RF == 8 && CPR == 2 ? 4 : 6;   // VALU per group
        constexpr int DSM = 2 * RF - VG;
        constexpr int DPM = NDS / DSM, XTRA = NDS - DPM * DSM;   // reads per MFMA
#pragma unroll
        for (int g = 0; g < XTRA; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x100, DPM + 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
#pragma unroll
        for (int g = XTRA; g < DSM; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x100, DPM, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
#pragma unroll
        for (int g = 0; g < VG; ++g) {
          __builtin_amdgcn_sched_group_barrier(0x002, VPG, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (kk == 2) {
        ring_wait<PER>();                      // stage kt+1 landed, kt done
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < JT; ++j) wa[j] = wn_[j];
#pragma unroll
      for (int i = 0; i < RF; ++i) xb[i] = xn_[i];
      if (kk == 3) {
#pragma unroll
        for (int j = 0; j < JT; ++j) {
#pragma unroll
          for (int h = 0; h < CPR / 2; ++h) wc[j][h] = wcn[j][h];
          s2[j] = s2n[j];
          b2[j] = b2n[j];
        }
      }
    }
  };

  // Prologue: stages 0 and 1 in flight, wait for stage 0, load its state.
#pragma unroll
  for (int g = 0; g < 3; ++g) issue_grp(g, 0, st0);
#pragma unroll
  for (int g = 0; g < 3; ++g) issue_grp(g, KT > 1 ? 1 : 0, st1);
  ring_wait<PER>();
  load_ws(st0, wc, s2, b2);
#pragma unroll
  for (int i = 0; i < RF; ++i) xb[i] = st0[swz8(32 * i + fr, fk)];
#pragma unroll
  for (int j = 0; j < JT; ++j) wa[j] = deq(wc, s2, b2, j, 0);

  // Stage kt lives in buffer kt % 3; three stages per trip, the remainder
  // (KT % 3) after the loop, so the loop body has no branch.
  int kt = 0;
  for (; kt + 3 <= KT; kt += 3) {
    body(kt, st0, st1, st2);
    body(kt + 1, st1, st2, st0);
    body(kt + 2, st2, st0, st1);
  }
  if (KT - kt >= 1) body(kt, st0, st1, st2);
  if (KT - kt == 2) body(kt + 1, st1, st2, st0);
  ring_wait<0>();                               // drained; LDS free

  // ---- LoRA tail: T and gathered B chunks of 32 ranks, same ring ----
  const int chunks32 = (!SPLIT || ks == a.kslices - 1) ? seg.chunks : 0;
  if (chunks32 > 0) {
    // PAIR: the second half of the waves gathers the up projection's B (its segment, its
    // groups); both T chunks are staged for every wave
    const QprojSeg& sw = upw ? a.seg_u : seg;
    const int t_col0 = seg.t_col0;
    const int ldb = sw.ldb;
    const int grp0 = sw.grp0;
    const int seg_nb = sw.n_begin, seg_ne = sw.n_end;
    const uint16_t* __restrict__ Bp = sw.B;
    const uint16_t* const tu = a.t + (PAIR ? a.seg_u.t_col0 - t_col0 : 0);
    // the first live group of the segment: a finite source for padding
    // groups (their T columns are exactly 0)
    const int g_safe = a.grp[grp0];
    // T: BMT rows x 4 chunks (TD DMAs a wave, rounded up: rows past the tile
    // land in the region's end, unread); B: 256 rows x 4 chunks (BD)
    uint32_t toff[TD];
    uint32_t boff[BD];
    int bc[BD];
#pragma unroll
    for (int i = 0; i < TD; ++i) {
      const int p = 64 * (TD * wave + i) + lane;
      const int row = p >> 2;
      const int c = (p & 3) ^ ((row >> 2) & 3);
      int m = m0 + row;
      m = m < mlast ? m : mlast;
      toff[i] = (uint32_t)(((long long)m * a.ldt + t_col0 + 8 * c) * 2);
    }
#pragma unroll
    for (int i = 0; i < BD; ++i) {
      const int p = 64 * (BD * wave + i) + lane;
      const int row = p >> 2;
      const int c = (p & 3) ^ ((row >> 2) & 3);
      int n = n0 + (PAIR ? (row & 127) : row);
      n = n < seg_ne - 1 ? n : seg_ne - 1;
      boff[i] = (uint32_t)((long long)(n - seg_nb) * ldb * 2);
      bc[i] = c;
    }
    // A lane's 16 bytes are the 8 ranks of one group; the chunk's four groups
    // are wave-uniform (scalar loads).
    auto grp_word = [&](int ch) -> uint2 {
      const int gi = __builtin_amdgcn_readfirstlane(grp0 + 4 * ch);
      return reinterpret_cast<const uint2*>(a.grp)[gi >> 2];
    };
    uint2 gw_next = grp_word(0);
    auto issue_t = [&](int ch, const uint4* X) {
#pragma unroll
      for (int i = 0; i < TD; ++i)
        dma16_sb(a.t + 32 * ch, toff[i], lds_addr(X + 64 * (TD * wave + i)));
      if constexpr (PAIR) {
#pragma unroll
        for (int i = 0; i < TD; ++i)
          dma16_sb(tu + 32 * ch, toff[i], lds_addr(X + TRG + 1024 + 64 * (TD * wave + i)));
      }
      // The chunk's four groups are one aligned 8-byte word of the table (a
      // segment's groups start at a multiple of 4), read by a wave-uniform
      // scalar load one issue ahead, so no issue waits on it. A lane picks
      // its group's 16 bits with a select and a shift (no branch).
      const uint2 gw = gw_next;
      const int nx = ch + 1 < chunks32 ? ch + 1 : chunks32 - 1;
      gw_next = grp_word(nx);
#pragma unroll
      for (int i = 0; i < BD; ++i) {
        const uint32_t w = (bc[i] & 2) ? gw.y : gw.x;
        int g = (int16_t)(w >> ((bc[i] & 1) << 4));
        g = g < 0 ? g_safe : g;
        dma16_sb(Bp, boff[i] + (uint32_t)g * 16u, lds_addr(X + TRG + 64 * (BD * wave + i)));
      }
    };
    uint4 ta[JT], tb[RF];
    auto read_t = [&](const uint4* X, int kk, uint4 (&av)[JT], uint4 (&bv)[RF]) {
      const int c = 2 * kk + fk;
#pragma unroll
      for (int j = 0; j < JT; ++j) av[j] = X[TRG + swz4(32 * JT * wave + 32 * j + fr, c)];
      const uint4* const XT = upw ? X + TRG + 1024 : X;
#pragma unroll
      for (int i = 0; i < RF; ++i) bv[i] = XT[swz4(32 * i + fr, c)];
    };
    // Chunk ch: step 0 reads step 1's fragments and issues chunk ch+2 into
    // Pv; the wait + barrier sit between the steps; step 1 reads the next
    // chunk's step-0 fragments.
    auto body_t = [&](int ch, const uint4* C, const uint4* Nx, const uint4* Pv) {
      const int nc = ch + 2 < chunks32 ? ch + 2 : chunks32 - 1;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        uint4 an[JT], bn[RF];
        if (kk == 0) {
          issue_t(nc, Pv);
          read_t(C, 1, an, bn);
        } else {
          read_t(Nx, 0, an, bn);
        }
#pragma unroll
        for (int i = 0; i < RF; ++i)
#pragma unroll
          for (int j = 0; j < JT; ++j)
            acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8_t, ta[j]), __builtin_bit_cast(bf16x8_t, tb[i]),
                acc[j][i], 0, 0, 0);
#pragma unroll
        for (int g = 0; g < (JT + RF < JT * RF ? JT + RF : JT * RF); ++g) {
          __builtin_amdgcn_sched_group_barrier(0x100, JT + RF <= JT * RF ? 1 : 2, 0);   // DS read
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
        }
        __builtin_amdgcn_sched_barrier(0);
        if (kk == 0) {
          ring_wait<TPER>();                       // chunk ch+1 landed, ch done
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int j = 0; j < JT; ++j) ta[j] = an[j];
#pragma unroll
        for (int i = 0; i < RF; ++i) tb[i] = bn[i];
      }
    };
    issue_t(0, st0);
    issue_t(chunks32 > 1 ? 1 : 0, st1);
    ring_wait<TPER>();
    read_t(st0, 0, ta, tb);
    int ch = 0;
    for (; ch + 3 <= chunks32; ch += 3) {
      body_t(ch, st0, st1, st2);
      body_t(ch + 1, st1, st2, st0);
      body_t(ch + 2, st2, st0, st1);
    }
    if (chunks32 - ch >= 1) body_t(ch, st0, st1, st2);
    if (chunks32 - ch == 2) body_t(ch + 1, st1, st2, st0);
    ring_wait<0>();
  }

  if constexpr (SPLIT) {
    // f32 partials P[ks][m][n]: lane row 32i + fr, four columns per quad
#pragma unroll
    for (int i = 0; i < RF; ++i) {
      const int m = m0 + 32 * i + fr;
      if (m >= a.M) continue;
#pragma unroll
      for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = n0 + 32 * JT * wave + 32 * j + 8 * q + 4 * fk;
          if (n < a.N)
            *reinterpret_cast<float4*>(
                a.part + ((long long)(wsel * a.kslices + ks) * a.M + m) * a.N + n) =
                make_float4(acc[j][i][4 * q + 0], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2],
                            acc[j][i][4 * q + 3]);
        }
    }
    return;
  }

  if constexpr (PAIR) {
    // The gate's and the up projection's bf16 outputs meet in LDS, up to 128
    // rows at a time: regions 0 and 1 hold the gate's two column halves, 2 and 3
    // the up projection's (a wave a region, or two with eight waves), and after
    // the barrier wave w reads half w & 1 of both over its share of the rows and
    // writes y = bf16(silu(g) * u) and its fp16 copy: the bits of the gate's own
    // epilogue followed by the gated one.
    const int rg = wave * JT / 2;   // the 64-column region this wave writes
    uint2* const Ew = reinterpret_cast<uint2*>(region(rg));
    const uint4* const Eg = region(wave & 1);
    const uint4* const Eu = region(2 + (wave & 1));
    const int cl = lane & 7;
    const int n = n0 + 64 * (wave & 1) + 8 * cl;
    uint32_t seen = 0;
#pragma unroll
    for (int h = 0; h < (RF + 3) / 4; ++h) {
#pragma unroll
      for (int ii = 0; ii < (RF - 4 * h < 4 ? RF - 4 * h : 4); ++ii) {
        const int i = 4 * h + ii;
        const int ml = 32 * ii + fr;
#pragma unroll
        for (int j = 0; j < JT; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int c = 4 * (JT == 2 ? j : (wave & 1)) + q;
            uint2 v;
            v.x = pack_bf16x2_rne(acc[j][i][4 * q + 0], acc[j][i][4 * q + 1]);
            v.y = pack_bf16x2_rne(acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]);
            Ew[ml * 16 + 2 * (c ^ ((ml >> 1) & 7)) + fk] = v;
          }
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < JT * (RF - 4 * h < 4 ? RF - 4 * h : 4); ++r) {
        const int ml = 8 * JT * (RF - 4 * h < 4 ? RF - 4 * h : 4) * (wave >> 1) + 8 * r + (lane >> 3);
        const int e = ml * 8 + (cl ^ ((ml >> 1) & 7));
        const uint4 gv = Eg[e];
        uint4 v = Eu[e];
        const int m = m0 + 128 * h + ml;
        if (m < a.M && n < a.N) {
          const uint32_t* gp = &gv.x;
          uint32_t* vp = &v.x;
#pragma unroll
          for (int e2 = 0; e2 < 4; ++e2)
            vp[e2] = pack_bf16x2_rne(silu_f(bf16_lo(gp[e2])) * bf16_lo(vp[e2]),
                                     silu_f(bf16_hi(gp[e2])) * bf16_hi(vp[e2]));
          *reinterpret_cast<uint4*>(a.y + (long long)m * a.ldy + n) = v;
          if (a.yh) {
            seen = range_track4(seen, v);
            uint4 f;
            f.x = bf16x2_to_f16x2(v.x);
            f.y = bf16x2_to_f16x2(v.y);
            f.z = bf16x2_to_f16x2(v.z);
            f.w = bf16x2_to_f16x2(v.w);
            *reinterpret_cast<uint4*>(a.yh + (long long)m * a.ldyh + n) = f;
          }
        }
      }
      __syncthreads();   // the next half rewrites the regions
    }
    if (a.yh) range_report(a.range, seen);
    return;
  }

  // Epilogue through LDS: a 16 KB region holds 64 columns x up to 128 rows in
  // bf16 (rows of 128 B, chunks swizzled by (row >> 1) & 7 so both the 8-B
  // writes and the 16-B reads are conflict-free), stored as whole 128-B row
  // segments, 8 rows per instruction. With four waves only the wave itself
  // touches its region, and LDS accesses of one wave complete in order, so no
  // barrier is needed inside; with eight, two waves share one.
  const int rg = wave * JT / 2;   // the 64-column region this wave writes and stores from
  uint4* const E = region(rg);
  const bool st16 = (a.ldy & 7) == 0 && (reinterpret_cast<uintptr_t>(yout) & 15) == 0;
  const int cl = lane & 7;
  const int n = n0 + 64 * rg + 8 * cl;
  uint32_t seen = 0;   // magnitudes written to the fp16 copy (range_report)
#pragma unroll
  for (int h = 0; h < (RF + 3) / 4; ++h) {
    const int HF = RF - 4 * h < 4 ? RF - 4 * h : 4;   // fragments of this part
    // Fused SwiGLU: this half's gate rows are loaded first, so their memory
    // latency overlaps the conversion below instead of stalling each store.
    uint4 gv[16];
    if (a.g) {
#pragma unroll
      for (int r = 0; r < 2 * JT * HF; ++r) {
        int m = m0 + 128 * h + (JT == 2 ? 0 : 16 * HF * (wave & 1)) + 8 * r + (lane >> 3);
        m = m < a.M ? m : a.M - 1;
        const int nn = n < a.N ? n : a.N - 8;
        gv[r] = *reinterpret_cast<const uint4*>(a.g + (long long)m * a.ldg + nn);
      }
    }
    uint2* const E2 = reinterpret_cast<uint2*>(E);
#pragma unroll
    for (int ii = 0; ii < HF; ++ii) {
      const int i = 4 * h + ii;
      const int ml = 32 * ii + fr;
#pragma unroll
      for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int c = 4 * (JT == 2 ? j : (wave & 1)) + q;
          uint2 v;
          v.x = pack_bf16x2_rne(acc[j][i][4 * q + 0], acc[j][i][4 * q + 1]);
          v.y = pack_bf16x2_rne(acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]);
          E2[ml * 16 + 2 * (c ^ ((ml >> 1) & 7)) + fk] = v;
        }
    }
    // eight waves: two share a region, each writes its 32 columns and stores
    // half of the rows
    if constexpr (NW == 8) __syncthreads();
#pragma unroll
    for (int r = 0; r < 2 * JT * HF; ++r) {
      const int ml = (JT == 2 ? 0 : 16 * HF * (wave & 1)) + 8 * r + (lane >> 3);
      uint4 v = E[ml * 8 + (cl ^ ((ml >> 1) & 7))];
      const int m = m0 + 128 * h + ml;
      if (m < a.M && n < a.N) {
        if (a.g) {
          // the bf16 projection output is the "up" operand
          const uint32_t* gp = &gv[r].x;
          uint32_t* vp = &v.x;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            vp[e] = pack_bf16x2_rne(silu_f(bf16_lo(gp[e])) * bf16_lo(vp[e]),
                                    silu_f(bf16_hi(gp[e])) * bf16_hi(vp[e]));
        }
        uint16_t* yp = yout + (long long)m * a.ldy + n;
        if (st16) {
          *reinterpret_cast<uint4*>(yp) = v;
        } else {
          reinterpret_cast<uint2*>(yp)[0] = make_uint2(v.x, v.y);
          reinterpret_cast<uint2*>(yp)[1] = make_uint2(v.z, v.w);
        }
        if (a.yh) {
          seen = range_track4(seen, v);
          uint4 f;
          f.x = bf16x2_to_f16x2(v.x);
          f.y = bf16x2_to_f16x2(v.y);
          f.z = bf16x2_to_f16x2(v.z);
          f.w = bf16x2_to_f16x2(v.w);
          *reinterpret_cast<uint4*>(a.yh + (long long)m * a.ldyh + n) = f;
        }
      }
    }
    if constexpr (NW == 8 && RF > 4) __syncthreads();
  }
  if (a.yh) range_report(a.range, seen);
}

template <int BITS, bool SPLIT, int RF, int NW>
__global__ __launch_bounds__(64 * NW, 1) void qproj_fast_kernel(const QprojArgs a) {
  qproj_fast_body<BITS, SPLIT, false, RF, NW>(a);
}

template <int BITS, int RF, int NW>
__global__ __launch_bounds__(64 * NW, 1) void qproj_pair_kernel(const QprojArgs a) {
  qproj_fast_body<BITS, false, true, RF, NW>(a);
}

template <int BITS, bool SPLIT, int RF, int NW>
__global__ __launch_bounds__(64 * NW, 1) void qproj_merged_kernel(const QprojArgs a) {
  qproj_fast_body<BITS, SPLIT, false, RF, NW, true>(a);
}

// The split projection's end (grid y: the projection of a merged launch): y =
// bf16(sum of the slices in order), then as the epilogue: the fused SwiGLU
// bf16(silu(g) * y) and the fp16 copy.
// 32-bit indices: the host keeps M * N / 4 below 2^31.
__global__ void qproj_split_reduce_kernel(const QprojArgs a) {
  const unsigned n4 = (unsigned)a.N >> 2;
  const unsigned total = (unsigned)a.M * n4;
  const size_t plane = (size_t)a.M * (size_t)a.N;
  const unsigned w = blockIdx.y;
  const float* const part = a.part + w * a.kslices * plane;
  uint16_t* const y = w > 0 ? a.more[w - 1].y : a.y;
  uint32_t seen = 0;
  for (unsigned i = blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += gridDim.x * blockDim.x) {
    const unsigned m = i / n4;
    const unsigned n = (i - m * n4) * 4;
    const float* p = part + (size_t)m * a.N + n;
    float4 sum = *reinterpret_cast<const float4*>(p);
    for (int k = 1; k < a.kslices; ++k) {
      p += plane;
      const float4 v = *reinterpret_cast<const float4*>(p);
      sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
    }
    uint32_t vp[2] = {pack_bf16x2_rne(sum.x, sum.y), pack_bf16x2_rne(sum.z, sum.w)};
    if (a.g) {
      const uint2 gv = *reinterpret_cast<const uint2*>(a.g + (size_t)m * a.ldg + n);
      const uint32_t gp[2] = {gv.x, gv.y};
#pragma unroll
      for (int e = 0; e < 2; ++e)
        vp[e] = pack_bf16x2_rne(silu_f(bf16_lo(gp[e])) * bf16_lo(vp[e]),
                                silu_f(bf16_hi(gp[e])) * bf16_hi(vp[e]));
    }
    *reinterpret_cast<uint2*>(y + (size_t)m * a.ldy + n) = make_uint2(vp[0], vp[1]);
    if (a.yh) {
      seen = range_track(range_track(seen, vp[0]), vp[1]);
      *reinterpret_cast<uint2*>(a.yh + (size_t)m * a.ldyh + n) =
          make_uint2(bf16x2_to_f16x2(vp[0]), bf16x2_to_f16x2(vp[1]));
    }
  }
  range_report(a.range, seen);
}

// ---- T = x . A_live^T * coef: the adapters' stacked down-projection --------
// Block tile 64*MR rows x 64*CJ stacked ranks. Four MFMA waves in 2 x 2, each
// 32*MR rows x 32*CJ ranks (MR x CJ tiles of v_mfma_f32_32x32x16_bf16,
// D[rank][row], so a lane owns one row and 4 consecutive ranks per register
// quad), and a DMA-only wave beside each on its SIMD: a global_load_lds holds
// the wave that issues it for ~16 cycles its MFMAs do not hide, so no MFMA wave
// issues one. Split-K over kslices so the grid is about one round of the chip;
// slice s writes f32 partials P[s] and lora_xa_reduce_kernel sums the slices in
// a fixed order (no atomics: the bits do not depend on timing). With one slice
// the block writes T directly. A three-stage ring of [x | A] (48 KB a stage at
// 256 x 128) filled by inline-asm DMA, one barrier a stage, which every wave
// passes once: before it the DMA waves issue stage t + 2 into the buffer stage
// t - 1 left and wait until stage t + 1 has landed; the MFMA waves have then
// finished every read of stage t (steps 0-2 read it; step 3, after the barrier,
// reads stage t + 1's first fragments).
template <int MR, int CJ>
__global__ __launch_bounds__(512, 1) void lora_xa_fast_kernel(const LoraXaArgs a, float* part,
                                                              int kslices) {
  constexpr int XR = 64 * MR, XC = 64 * CJ;      // rows and ranks of the tile
  constexpr int XCH = XR * 8;                    // 16-B chunks of the x tile
  constexpr int STG = XCH + XC * 8;              // x tile + A tile
  constexpr int XD = 2 * MR, AD = 2 * CJ;        // DMAs per DMA wave per stage
  constexpr int PER = XD + AD;
  __shared__ uint4 st0[STG], st1[STG], st2[STG];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool dma_wave = wave >= 4;
  const int rw = wave & 3;                       // the role's wave index
  const int fr = lane & 31, fk = lane >> 5;
  const int wm = rw & 1, wc = rw >> 1;
  int m0, c0, ks;
  {
    const int tiles_m = (a.M + XR - 1) / XR, tiles_c = (a.n_cols + XC - 1) / XC;
    const int nb = (int)gridDim.x;
    const int q = nb / 8, rem = nb % 8;
    const int xcd = (int)blockIdx.x % 8, local = (int)blockIdx.x / 8;
    const int v = xcd * q + (xcd < rem ? xcd : rem) + local;
    const int tc = v % tiles_c, rest = v / tiles_c;
    m0 = (rest % tiles_m) * XR;
    c0 = tc * XC;
    ks = rest / tiles_m;
  }
  const int KT = a.K / 64;
  const int kt0 = (int)((long long)KT * ks / kslices);
  const int kt1 = (int)((long long)KT * (ks + 1) / kslices);
  const int NT = kt1 - kt0;
  const int mlast = a.M - 1;

  if (dma_wave) {
    uint32_t xoff[XD];
#pragma unroll
    for (int i = 0; i < XD; ++i) {
      const int p = 64 * (XD * rw + i) + lane;
      const int row = p >> 3;
      const int c = (p & 7) ^ ((row >> 1) & 7);
      int m = m0 + row;
      m = m < mlast ? m : mlast;
      xoff[i] = (uint32_t)(((long long)m * a.ldx + 8 * c) * 2);
    }
    const int g_safe = a.ident ? 0 : a.grp[0];
    uint32_t aoff[AD];
    int asrc[AD];
#pragma unroll
    for (int i = 0; i < AD; ++i) {
      const int p = 64 * (AD * rw + i) + lane;
      const int r = p >> 3;
      const int c = (p & 7) ^ ((r >> 1) & 7);
      const int col = c0 + r;
      int g, row;                                // stack (>> 12) and row of the column
      if (a.ident) {
        g = 0;
        row = col < a.n_cols ? col : a.n_cols - 1;
      } else {
        const int gc = col < a.n_cols ? a.grp[col >> 3] : -1;
        g = gc < 0 ? g_safe : gc;
        row = 8 * (g & 4095) + (gc < 0 ? 0 : (col & 7));
      }
      aoff[i] = (uint32_t)(((long long)row * a.K + 8 * c) * 2);
      asrc[i] = __builtin_amdgcn_readfirstlane(g >> 12);
    }
    auto issue = [&](int kt, const uint4* S) {
      const void* base = a.x + (long long)kt * 64;
#pragma unroll
      for (int i = 0; i < XD; ++i) dma16_sb(base, xoff[i], lds_addr(S + 64 * (XD * rw + i)));
#pragma unroll
      for (int i = 0; i < AD; ++i)
        dma16_sb(a.A[asrc[i]] + (long long)kt * 64, aoff[i],
                 lds_addr(S + XCH + 64 * (AD * rw + i)));
    };
    // The fp16 copy of x (a.xh): the column blocks of one row tile and K
    // slice split its rows, so each element is converted once. Stage t
    // is converted while it is in LDS (landed at the previous wait, its
    // buffer rewritten only after the next barrier): lane q takes chunk
    // q & 7 of rows r0 + q / 8 + 32 j.
    const int tiles_c = (a.n_cols + XC - 1) / XC, tc = c0 / XC;
    const int r0 = XR * tc / tiles_c, r1 = XR * (tc + 1) / tiles_c;
    const int q = 64 * rw + lane, qc = q & 7;
    uint32_t seen = 0;
    auto convert = [&](int t, const uint4* S) {
      if (!a.xh) return;
#pragma unroll 1
      for (int r = r0 + (q >> 3); r < r1; r += 32) {
        const uint4 v = S[r * 8 + (qc ^ ((r >> 1) & 7))];
        if (m0 + r < a.M) {
          seen = range_track4(seen, v);
          uint4 f;
          f.x = bf16x2_to_f16x2(v.x);
          f.y = bf16x2_to_f16x2(v.y);
          f.z = bf16x2_to_f16x2(v.z);
          f.w = bf16x2_to_f16x2(v.w);
          *reinterpret_cast<uint4*>(a.xh + (long long)(m0 + r) * a.ldxh +
                                    (long long)(kt0 + t) * 64 + 8 * qc) = f;
        }
      }
    };
    issue(kt0, st0);
    issue(kt0 + (NT > 1 ? 1 : 0), st1);
    ring_wait<PER>();                             // stage 0 landed
    // stage t: the copy of stage t, stage t + 2 (a re-read of the last past
    // the end) into the buffer of stage t - 1, then stage t + 1 landed, then
    // the barrier. The copy's stores go before the DMAs: vmcnt counts both
    // in issue order, so the wait for all but the newest PER (stage t + 2)
    // also covers the stores, whose latency the MFMA waves' stage hides.
    auto step = [&](int t, const uint4* C, const uint4* Pv) {
      convert(t, C);
      issue(kt0 + (t + 2 < NT ? t + 2 : NT - 1), Pv);
      ring_wait<PER>();
    };
    int t = 0;
    for (; t + 3 <= NT; t += 3) {
      step(t, st0, st2);
      step(t + 1, st1, st0);
      step(t + 2, st2, st1);
    }
    if (NT - t >= 1) step(t, st0, st2);
    if (NT - t == 2) step(t + 1, st1, st0);
    // no DMA outlives the block; no barrier: the MFMA waves meet no more
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (a.xh) range_report(a.range, seen);
    return;
  }

  floatx16_t acc[MR][CJ];
#pragma unroll
  for (int i = 0; i < MR; ++i)
#pragma unroll
    for (int j = 0; j < CJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  const bool live = c0 + 32 * CJ * wc < a.n_cols;
  uint4 xb[MR], ab[CJ];
  auto read_frags = [&](const uint4* S, int kk, uint4 (&xv)[MR], uint4 (&av)[CJ]) {
    const int c = 2 * kk + fk;
#pragma unroll
    for (int i = 0; i < MR; ++i) xv[i] = S[swz8(32 * MR * wm + 32 * i + fr, c)];
#pragma unroll
    for (int j = 0; j < CJ; ++j) av[j] = S[XCH + swz8(32 * CJ * wc + 32 * j + fr, c)];
  };
  auto body = [&](const uint4* C, const uint4* Nx) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      uint4 xn[MR], an[CJ];
      if (kk < 3) read_frags(C, kk + 1, xn, an);
      else read_frags(Nx, 0, xn, an);
      if (live) {
#pragma unroll
        for (int i = 0; i < MR; ++i)
#pragma unroll
          for (int j = 0; j < CJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf16x8_t, ab[j]), __builtin_bit_cast(bf16x8_t, xb[i]),
                acc[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int g = 0; g < (MR + CJ < MR * CJ ? MR + CJ : MR * CJ); ++g) {
        __builtin_amdgcn_sched_group_barrier(0x100, MR + CJ <= MR * CJ ? 1 : 2, 0);   // DS read
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
      }
      __builtin_amdgcn_sched_barrier(0);
      if (kk == 2) {
        ring_wait<0>();                          // (no DMAs of its own) reads done + barrier
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < MR; ++i) xb[i] = xn[i];
#pragma unroll
      for (int j = 0; j < CJ; ++j) ab[j] = an[j];
    }
  };
  ring_wait<0>();                                // stage 0 landed (the DMA waves' wait)
  read_frags(st0, 0, xb, ab);
  int t = 0;
  for (; t + 3 <= NT; t += 3) {
    body(st0, st1);
    body(st1, st2);
    body(st2, st0);
  }
  if (NT - t >= 1) body(st0, st1);
  if (NT - t == 2) body(st1, st2);

  if (!live) return;
  if (kslices > 1) {
    // The partials in the accumulators' own order: slice ks, tile (row tile,
    // column block), MFMA wave, fragment f = (CJ i + j) 4 + q, lane -- each store
    // instruction writes 64 lanes x 16 B contiguous (the row-major layout
    // scattered every instruction over 32 rows). lora_xa_reduce_kernel reads
    // the same order.
    const int tiles_c = (a.n_cols + XC - 1) / XC;
    const long long tile = (long long)(m0 / XR) * tiles_c + c0 / XC;
    const long long ntiles = (long long)((a.M + XR - 1) / XR) * tiles_c;
    float4* pw = reinterpret_cast<float4*>(part) +
                 (((ks * ntiles + tile) * 4 + rw) * (4 * MR * CJ)) * 64 + lane;
#pragma unroll
    for (int i = 0; i < MR; ++i)
#pragma unroll
      for (int j = 0; j < CJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          pw[(4 * (CJ * i + j) + q) * 64] =
              make_float4(acc[i][j][4 * q + 0], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                          acc[i][j][4 * q + 3]);
    return;
  }
  // D[c][m]: lane owns row m, four consecutive ranks per register quad.
#pragma unroll
  for (int i = 0; i < MR; ++i) {
    const int m = m0 + 32 * MR * wm + 32 * i + fr;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < CJ; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = c0 + 32 * CJ * wc + 32 * j + 8 * q + 4 * fk;
        const float f = a.ident ? 1.0f : a.coef[c >> 3];
        uint2 v;
        if (f == 0.0f) {
          v = make_uint2(0, 0);
        } else if (a.bias) {
          // the dense split-K GEMM with a bias (coef 1): one rounding
          float r[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] = f * acc[i][j][4 * q + e] + bf16_to_f32(a.bias[c + e]);
          v.x = pack_bf16x2_rne(r[0], r[1]);
          v.y = pack_bf16x2_rne(r[2], r[3]);
        } else {
          v.x = pack_bf16x2_rne(f * acc[i][j][4 * q + 0], f * acc[i][j][4 * q + 1]);
          v.y = pack_bf16x2_rne(f * acc[i][j][4 * q + 2], f * acc[i][j][4 * q + 3]);
        }
        *reinterpret_cast<uint2*>(a.t + (long long)m * a.ldt + c) = v;
      }
    }
  }
}

// T[m][c] = bf16(coef * sum_s P[s][m][c]), slices summed in order 0..S-1,
// over the partials in the order lora_xa_fast_kernel writes them. One thread
// per row and 8 consecutive ranks: the float4s of accumulator lanes fr and
// fr + 32 (ranks 8q + 0..3 and 8q + 4..7 of one row), read from every slice
// at the same positions (32 threads cover each 1-KB run, every load
// coalesced), one 16-byte store of T. Positions of row tiles past M or
// column blocks past n_cols are skipped. 32-bit indices (the host keeps a
// slice's float4 count below 2^31).
template <int MR, int CJ>
__global__ void lora_xa_reduce_kernel(const float* part, int kslices, int M,
                                      int n_cols, const LoraXaArgs a) {
  constexpr unsigned XR = 64 * MR, XC = 64 * CJ, FR = 4 * MR * CJ;
  const unsigned tiles_c = ((unsigned)n_cols + XC - 1) / XC;
  const unsigned ntiles = (((unsigned)M + XR - 1) / XR) * tiles_c;
  const unsigned total = ntiles * (256u * FR);       // float4s per slice
  const bool st16 = (reinterpret_cast<uintptr_t>(a.t) & 15) == 0 && (a.ldt & 7) == 0;
  const float4* p4 = reinterpret_cast<const float4*>(part);
  for (unsigned t = blockIdx.x * blockDim.x + threadIdx.x; t < total / 2;
       t += gridDim.x * blockDim.x) {
    // the float4 of accumulator lane fr: ((tile * 4 + wave) * FR + f) * 64 + fr,
    // f = (CJ fi + fj) 4 + fq; lane fr + 32 is 32 float4s on
    const unsigned fr = t & 31, g = t >> 5;
    const unsigned i = g * 64 + fr;
    const unsigned f = g % FR, wave = (g / FR) & 3, tile = g / (4 * FR);
    const unsigned fi = f / (4 * CJ), fj = (f >> 2) % CJ, fq = f & 3;
    const unsigned tm = tile / tiles_c, tc = tile - tm * tiles_c;
    const unsigned m = XR * tm + 32 * MR * (wave & 1) + 32 * fi + fr;
    const unsigned c = XC * tc + 32 * CJ * (wave >> 1) + 32 * fj + 8 * fq;
    if (m >= (unsigned)M || c >= (unsigned)n_cols) continue;
    float4 s0 = p4[i], s1 = p4[i + 32];
    for (int k = 1; k < kslices; ++k) {
      const float4 v0 = p4[(size_t)k * total + i];
      const float4 v1 = p4[(size_t)k * total + i + 32];
      s0.x += v0.x; s0.y += v0.y; s0.z += v0.z; s0.w += v0.w;
      s1.x += v1.x; s1.y += v1.y; s1.z += v1.z; s1.w += v1.w;
    }
    const float co = a.ident ? 1.0f : a.coef[c >> 3];
    uint4 o = make_uint4(0, 0, 0, 0);
    if (co != 0.0f && a.bias) {
      // the dense split-K GEMM with a bias (coef 1): one rounding
      float r[8] = {co * s0.x, co * s0.y, co * s0.z, co * s0.w,
                    co * s1.x, co * s1.y, co * s1.z, co * s1.w};
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] += bf16_to_f32(a.bias[c + e]);
      o.x = pack_bf16x2_rne(r[0], r[1]);
      o.y = pack_bf16x2_rne(r[2], r[3]);
      o.z = pack_bf16x2_rne(r[4], r[5]);
      o.w = pack_bf16x2_rne(r[6], r[7]);
    } else if (co != 0.0f) {
      o.x = pack_bf16x2_rne(co * s0.x, co * s0.y);
      o.y = pack_bf16x2_rne(co * s0.z, co * s0.w);
      o.z = pack_bf16x2_rne(co * s1.x, co * s1.y);
      o.w = pack_bf16x2_rne(co * s1.z, co * s1.w);
    }
    uint16_t* const tp = a.t + (size_t)m * a.ldt + c;
    if (st16) {
      *reinterpret_cast<uint4*>(tp) = o;
    } else {
      reinterpret_cast<uint2*>(tp)[0] = make_uint2(o.x, o.y);
      reinterpret_cast<uint2*>(tp)[1] = make_uint2(o.z, o.w);
    }
  }
}

// ---- resident layout for the fast route ------------------------------------
// codes: from the reference pack (LSB-first, [N][K*bits/32]) into
// [kt][n][fk][kk](w4) / [kt][n][fk][kk][2](w8); sbf: fp16 (s, b) pairs and
// a flag raised when any scale or bias is not exact in fp16.
__global__ void repack_fast_kernel(int bits, const uint32_t* codes, int N, int K,
                                   uint32_t* out) {
  const int wpr = bits == 4 ? 8 : 16;
  const long long total = (long long)(K / 64) * N * wpr;
  const long long words_row = (long long)K * bits / 32;
  for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x;
       idx < total; idx += (long long)gridDim.x * blockDim.x) {
    const int slot = (int)(idx % wpr);
    const long long rest = idx / wpr;
    const int n = (int)(rest % N);
    const int kt = (int)(rest / N);
    uint32_t o;
    if (bits == 4) {
      // slot = fk*4 + kk -> source word j = 2kk + fk (k = 8j .. 8j+7)
      const int fk = slot >> 2, kk = slot & 3;
      const uint32_t w = codes[(long long)n * words_row + (long long)kt * 8 + 2 * kk + fk];
      // new nibble i holds old nibble perm[i]: {k0,k4,k1,k5,k2,k6,k3,k7}
      const int perm[8] = {0, 4, 1, 5, 2, 6, 3, 7};
      o = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) o |= ((w >> (4 * perm[i])) & 15u) << (4 * i);
    } else {
      // slot = fk*8 + kk*2 + h -> k = 16kk + 8fk + 4h: source word (16kk+8fk+4h)/4
      const int fk = slot >> 3, kk = (slot >> 1) & 3, h = slot & 1;
      o = codes[(long long)n * words_row + (long long)kt * 16 + 4 * kk + 2 * fk + h];
    }
    out[idx] = o;
  }
}

__device__ __forceinline__ uint32_t bf16_to_f16_bits(uint16_t h, bool* exact) {
  const float f = __uint_as_float((uint32_t)h << 16);
  const _Float16 x = (_Float16)f;
  if ((float)x != f) *exact = false;
  return (uint32_t)__builtin_bit_cast(uint16_t, x);
}

__global__ void repack_sbf_kernel(const uint16_t* scales, const uint16_t* biases,
                                  int N, int G, uint32_t* sbf, int* inexact) {
  const long long total = (long long)G * N;
  bool exact = true;
  for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x;
       idx < total; idx += (long long)gridDim.x * blockDim.x) {
    const int n = (int)(idx % N);
    const int g = (int)(idx / N);
    const uint32_t s = bf16_to_f16_bits(scales[(long long)n * G + g], &exact);
    const uint32_t b = bf16_to_f16_bits(biases[(long long)n * G + g], &exact);
    sbf[idx] = s | (b << 16);
  }
  if (!exact) atomicOr(inexact, 1);
}

__global__ void bf16_to_f16_kernel(const uint16_t* x, long long ldx, uint16_t* y,
                                   long long ldy, int rows, int K, int* range) {
  const int k8 = K >> 3;
  const long long total = (long long)rows * k8;
  uint32_t seen = 0;
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    const long long r = i / k8;
    const int c = (int)(i % k8) * 8;
    const uint4 v = *reinterpret_cast<const uint4*>(x + r * ldx + c);
    seen = range_track4(seen, v);
    uint4 o;
    o.x = bf16x2_to_f16x2(v.x);
    o.y = bf16x2_to_f16x2(v.y);
    o.z = bf16x2_to_f16x2(v.z);
    o.w = bf16x2_to_f16x2(v.w);
    *reinterpret_cast<uint4*>(y + r * ldy + c) = o;
  }
  range_report(range, seen);
}

}  // namespace

int device_cus() {
  static std::atomic<int> cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        n <= 0)
      n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Rows per tile. A launch of `tiles` tiles of 32*rf rows takes a start, a full
// round's time for every whole round of the chip (one tile a CU), and for the
// last one less while it leaves CUs idle: the others then clock higher and
// share the memory with fewer. Per round a part of its own (prologue, epilogue,
// store) and a part a K stage, us, fitted to 600 launches at K = 64 to 10240
// and 60 to 1050 tiles, the paired launch's to 240; within 3% on the average
// (rf 2, two blocks a CU, 5%). Of w4: w8 takes 1.03 to 1.06 of it at every
// height. rf 8 is the best rate for a full chip, the lower tiles fill it where
// 256 rows leave it idle (1280 rows of [3840, 3840]: 75 tiles, 75.5 -> 49.8 us
// with 150 of rf 4). rf 2 to 6 run eight waves, two a SIMD, each 32 columns:
// 49.8 against 53.2 us with four waves at rf 4; at rf 8 their reads of x would
// fill the LDS.
struct TileCost {
  int rf;
  double full0, full, few0, few;   // a full round, one of at most half of the CUs
};
constexpr TileCost kTiles[4] = {{8, 8.2, 1.510, 7.6, 1.027},
                                {6, 5.7, 1.227, 4.1, 0.797},
                                {4, 4.7, 0.867, 2.5, 0.602},
                                {2, 2.3, 0.477, 1.3, 0.437}};
constexpr TileCost kPairTiles[3] = {{8, 8.5, 1.380, 8.5, 0.930},
                                    {6, 5.5, 1.110, 5.0, 0.680},
                                    {4, 4.4, 0.770, 3.0, 0.530}};

static double tiles_us(const TileCost& t, long long tiles, int stages) {
  const int cus = device_cus();
  const double full = t.full0 + t.full * stages, few = t.few0 + t.few * stages;
  const double fill = (double)(tiles % cus) / cus;
  double us = 5.0 + (double)(tiles / cus) * full;
  if (fill > 0.0) us += few + (fill > 0.5 ? (full - few) * (fill - 0.5) * 2.0 : 0.0);
  return us;
}

// One launch of one height, or the 256-row tile rows that fill some whole
// rounds and then a lower height in a second launch (4352 rows of a paired
// launch of 80 column tiles, K = 3840: 16 tile rows in five rounds, then 256
// rows as rf 4 in one). The model is good to a few percent, so what is not one
// launch of 256-row tiles has to gain by it: a lower height 3% of one or two
// rounds, 5% of more (16640 rows of [15360, 256], where both model alike: rf 6
// 321 us, rf 8 259), a second launch 5% of a round (2560 rows of [10240, 3840]:
// one launch 171.8 us, 240 tiles of rf 8 and then of rf 6 178.2). The paired
// launch's lower heights gain a little more than modelled (400 rows: rf 6 76.6
// us, rf 8 79.2) and its second launch starts inside the first one's end (a
// feed-forward at 2048 rows 407 us with two, 416 with one): none, and 5% less.
// With K in it 4096 rows of [10240, 64] take 28.5 us, by K = 3840's times 36.2.
RowPlan plan_rows(int M, int tiles_n, int stages, bool pair) {
  const int cus = device_cus();
  const TileCost* const tiles = pair ? kPairTiles : kTiles;
  const int nt = pair ? 3 : 4;
  const int tiles_m = (M + BM - 1) / BM;
  const long long all = ((long long)tiles_m * tiles_n + cus - 1) / cus;
  // the rows past the first m1 tile rows at the lower height that takes least
  auto rest = [&](int m1) {
    RowPlan best = {m1 * BM, 8, -1.0};
    for (int i = 1; i < nt; ++i) {
      const int rows = M - m1 * BM, h = 32 * tiles[i].rf;
      const double us = tiles_us(tiles[i], (long long)((rows + h - 1) / h) * tiles_n, stages);
      if (best.us < 0.0 || us < best.us) best = {m1 * BM, tiles[i].rf, us};
    }
    return best;
  };
  RowPlan best = {M, 8, tiles_us(tiles[0], (long long)tiles_m * tiles_n, stages)};
  const RowPlan low = rest(0);
  if (low.us < best.us * (all > 2 ? 0.95 : pair ? 1.0 : 0.97)) best = low;
  RowPlan two = {0, 0, -1.0};
  for (int k = 0; k < 3; ++k) {
    // the tile rows that fill all - 1 - k rounds
    const long long full = (all - 1 - k) * cus / tiles_n;
    const int m1 = full < tiles_m ? (int)full : tiles_m - 1;
    if (m1 <= 0) break;
    RowPlan p = rest(m1);
    p.us += tiles_us(tiles[0], (long long)m1 * tiles_n, stages);
    if (two.us < 0.0 || p.us < two.us) two = p;
  }
  const double round = tiles[0].full0 + tiles[0].full * stages;
  if (two.us >= 0.0 && two.us < best.us + (pair ? 0.05 : -0.05) * round) best = two;
  return best;
}

// K stages of a launch, its longest LoRA tail's chunks counted as 5/8 of one.
static int stages_of(const QprojArgs& a) {
  int chunks = 0;
  for (int i = 0; i < a.nseg; ++i) chunks = a.seg[i].chunks > chunks ? a.seg[i].chunks : chunks;
  return a.K / BK + chunks * 5 / 8;
}

// The K split of a projection of few 256 x 256 tiles (the context refiner's
// caption rows: 15 or 40): rows per tile and slices, by the time of a round
// (a stage of 64 about 0.45, 0.57 and 0.96 us at rf 2, 4 and 8) plus the f32
// partials, written and read at about 5 TB/s. Never more slices than 256-row
// tiles would take (one round, at least 6 stages each), so the partials stay
// within what they would take. [256, 3840] x [3840, 3840]: rf 2 in 4 slices, 24.6
// us, where rf 8 in 10 took 30.7; 16 rows 14.1 against 18.6. 0: no split.
struct StageCost {
  int rf;
  double us;
};
static constexpr StageCost kStages[3] = {{8, 0.96}, {4, 0.57}, {2, 0.45}};

static double split_us(const StageCost& t, int M, int N, int K, int ks, int nw) {
  const int cus = device_cus();
  const int grid = ((M + 32 * t.rf - 1) / (32 * t.rf)) * ((N + BN - 1) / BN) * nw;
  return (double)((grid * ks + cus - 1) / cus) * ((K / BK + ks - 1) / ks) * t.us +
         1.6e-6 * (double)M * N * nw * ks;
}

int qproj_split_plan(int M, int N, int K, int* rf) {
  *rf = 8;
  const int tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  if (tiles <= 0 || tiles >= 64 || N % 4 != 0) return 0;
  const int KT = K / BK;
  int kmax = device_cus() / tiles;
  if (kmax > KT / 6) kmax = KT / 6;
  if (kmax < 2) return 0;
  int best = 0;
  double cost = 0.0;
  for (const StageCost& t : kStages)
    for (int ks = 2; ks <= kmax; ++ks) {
      const double c = split_us(t, M, N, K, ks, 1);
      if (best == 0 || c < cost) {
        cost = c;
        best = ks;
        *rf = t.rf;
      }
    }
  return best;
}

int qproj_merged_split_rf(int M, int N, int K, int kslices, int nw) {
  int rf = 8;
  double cost = 0.0;
  for (const StageCost& t : kStages) {
    const double c = split_us(t, M, N, K, kslices, nw);
    if (cost == 0.0 || c < cost) {
      cost = c;
      rf = t.rf;
    }
  }
  return rf;
}

// One launch each against one for all. Split: the merged one fills its rounds
// of blocks, and is two launches where there were two each (a w4 block at 203
// rows 312 us with three, 288 with one). Unsplit: where the rounds of all are
// fewer (three of [1280, 3840] x [3840, 3840]: 135 against 73.5 by the model; a
// w8 block 577 us with three, 545 with one); equal rounds gain nothing (4352
// rows measured 0.3% slower a forward when merged).
bool qproj_merge_pays(int M, int N, int K, int nw) {
  int rf = 0;
  if (qproj_split_plan(M, N, K, &rf) > 0) return true;
  const int tiles_n = (N + BN - 1) / BN;
  return plan_rows(M, nw * tiles_n, K / BK, false).us <
         0.95 * nw * plan_rows(M, tiles_n, K / BK, false).us;
}

template <int BITS, bool SPLIT, int RF, int NW>
static void launch_tiles(const QprojArgs& a, hipStream_t s) {
  const int tiles = ((a.M + 32 * RF - 1) / (32 * RF)) * ((a.N + BN - 1) / BN);
  hipLaunchKernelGGL((qproj_fast_kernel<BITS, SPLIT, RF, NW>),
                     dim3((unsigned)(SPLIT ? tiles * a.kslices : tiles)), dim3(64 * NW), 0, s, a);
}
template <int BITS>
static void launch_rows(const QprojArgs& a, int rf, hipStream_t s) {
  switch (rf) {
    case 2: launch_tiles<BITS, false, 2, 8>(a, s); break;
    case 4: launch_tiles<BITS, false, 4, 8>(a, s); break;
    case 6: launch_tiles<BITS, false, 6, 8>(a, s); break;
    default: launch_tiles<BITS, false, 8, 4>(a, s); break;
  }
}
template <int BITS>
static void launch_split(const QprojArgs& a, hipStream_t s) {
  switch (a.split_rf) {
    case 2: launch_tiles<BITS, true, 2, 8>(a, s); break;
    case 4: launch_tiles<BITS, true, 4, 8>(a, s); break;
    default: launch_tiles<BITS, true, 8, 4>(a, s); break;
  }
}
template <int BITS, bool SPLIT, int RF, int NW>
static void launch_merged_tiles(const QprojArgs& a, hipStream_t s) {
  const int tiles = ((a.M + 32 * RF - 1) / (32 * RF)) * ((a.N + BN - 1) / BN) * a.nw;
  hipLaunchKernelGGL((qproj_merged_kernel<BITS, SPLIT, RF, NW>),
                     dim3((unsigned)(SPLIT ? tiles * a.kslices : tiles)), dim3(64 * NW), 0, s, a);
}
template <int BITS>
static void launch_merged_rows(const QprojArgs& a, int rf, hipStream_t s) {
  switch (rf) {
    case 2: launch_merged_tiles<BITS, false, 2, 8>(a, s); break;
    case 4: launch_merged_tiles<BITS, false, 4, 8>(a, s); break;
    case 6: launch_merged_tiles<BITS, false, 6, 8>(a, s); break;
    default: launch_merged_tiles<BITS, false, 8, 4>(a, s); break;
  }
}
template <int BITS>
static void launch_merged_split(const QprojArgs& a, hipStream_t s) {
  switch (a.split_rf) {
    case 2: launch_merged_tiles<BITS, true, 2, 8>(a, s); break;
    case 4: launch_merged_tiles<BITS, true, 4, 8>(a, s); break;
    default: launch_merged_tiles<BITS, true, 8, 4>(a, s); break;
  }
}
template <int BITS, int RF, int NW>
static void launch_pair_tiles(const QprojArgs& a, hipStream_t s) {
  const int tiles = ((a.M + 32 * RF - 1) / (32 * RF)) * ((a.N + BN / 2 - 1) / (BN / 2));
  hipLaunchKernelGGL((qproj_pair_kernel<BITS, RF, NW>), dim3((unsigned)tiles), dim3(64 * NW), 0,
                     s, a);
}
template <int BITS>
static void launch_pair_rows(const QprojArgs& a, int rf, hipStream_t s) {
  switch (rf) {
    case 4: launch_pair_tiles<BITS, 4, 8>(a, s); break;
    case 6: launch_pair_tiles<BITS, 6, 8>(a, s); break;
    default: launch_pair_tiles<BITS, 8, 4>(a, s); break;
  }
}

// `rows(args, rf)` over the plan's two row ranges (the second one's arguments
// shifted down by the first's rows).
template <class F>
static hipError_t launch_plan(const QprojArgs& a, const RowPlan& p, F&& rows) {
  if (p.rows_main > 0) {
    QprojArgs m = a;
    m.M = p.rows_main;
    rows(m, 8);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.rows_main == a.M) return e;
  }
  QprojArgs h = a;
  const long long r = p.rows_main;
  h.M = a.M - p.rows_main;
  h.x = a.x + r * a.ldx;
  h.y = a.y + r * a.ldy;
  if (a.g) h.g = a.g + r * a.ldg;
  if (a.yh) h.yh = a.yh + r * a.ldyh;
  if (a.t) h.t = a.t + r * a.ldt;
  for (int i = 0; i + 1 < a.nw; ++i) h.more[i].y = a.more[i].y + r * a.ldy;
  rows(h, p.rf_rest);
  return hipGetLastError();
}

hipError_t launch_qproj_fast(int bits, const QprojArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (bits != 4 && bits != 8) return hipErrorInvalidValue;
  if (a.kslices > 1) {
    if (!a.part || a.N % 4 != 0 || (long long)a.M * (a.N / 4) >= (1ll << 31) ||
        a.K / BK < a.kslices)
      return hipErrorInvalidValue;
    if (bits == 4)
      launch_split<4>(a, s);
    else
      launch_split<8>(a, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    long long blocks = ((long long)a.M * (a.N / 4) + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(qproj_split_reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, s, a);
    return hipGetLastError();
  }
  return launch_plan(a, plan_rows(a.M, (a.N + BN - 1) / BN, stages_of(a), false),
                     [&](const QprojArgs& m, int rf) {
                       if (bits == 4)
                         launch_rows<4>(m, rf, s);
                       else
                         launch_rows<8>(m, rf, s);
                     });
}

hipError_t launch_qproj_merged(int bits, const QprojArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if ((bits != 4 && bits != 8) || a.nw < 2 || a.nw > 3 || a.nseg != 1 || a.g || a.yh)
    return hipErrorInvalidValue;
  if (a.kslices > 1) {
    if (!a.part || a.N % 4 != 0 || (long long)a.M * (a.N / 4) >= (1ll << 31) ||
        a.K / BK < a.kslices)
      return hipErrorInvalidValue;
    QprojArgs m = a;
    m.split_rf = qproj_merged_split_rf(a.M, a.N, a.K, a.kslices, a.nw);
    if (bits == 4)
      launch_merged_split<4>(m, s);
    else
      launch_merged_split<8>(m, s);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    long long blocks = ((long long)a.M * (a.N / 4) + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(qproj_split_reduce_kernel, dim3((unsigned)blocks, (unsigned)a.nw), dim3(256),
                       0, s, a);
    return hipGetLastError();
  }
  return launch_plan(a, plan_rows(a.M, a.nw * ((a.N + BN - 1) / BN), stages_of(a), false),
                     [&](const QprojArgs& m, int rf) {
                       if (bits == 4)
                         launch_merged_rows<4>(m, rf, s);
                       else
                         launch_merged_rows<8>(m, rf, s);
                     });
}

hipError_t launch_qproj_pair(int bits, const QprojArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (a.kslices > 1 || a.g || !a.codes_u || !a.sb_u || a.nseg != 1 ||
      a.seg[0].chunks != a.seg_u.chunks || a.N % 8 != 0 || a.ldy % 8 != 0 ||
      (reinterpret_cast<uintptr_t>(a.y) & 15) != 0 || (bits != 4 && bits != 8))
    return hipErrorInvalidValue;
  return launch_plan(a, plan_rows(a.M, (a.N + BN / 2 - 1) / (BN / 2), stages_of(a), true),
                     [&](const QprojArgs& m, int rf) {
                       if (bits == 4)
                         launch_pair_rows<4>(m, rf, s);
                       else
                         launch_pair_rows<8>(m, rf, s);
                     });
}

// The K split depends on M and K only, never on how many columns are
// stacked: each T column is then summed in the same order, and so has the
// same bits, whether its projection's x.A runs alone or stacked with others
// over the same x. It is sized for an assumed number of 128-wide column
// blocks per launch, by K:
//  - K <= 4096 (the hidden-width inputs: q|k|v, o, w1|w3): 5 blocks, between
//    one projection's 2.5 and q|k|v's 7.5 at the config-2 adapter set. At
//    4352 rows that is 3 slices, measured best of 1, 2, 3, 5 and 8 over the
//    1024^2 forward's 136 launches (6.59 ms against 6.91 ms for 5).
//  - K > 4096 (the FFN-width input of w2, whose x.A always runs alone): 2
//    blocks (the config-2 set's 256 packed ranks), i.e. 7 slices at 4352
//    rows, one round of 238 blocks: w2's x.A 3.7 us faster than with 5
//    slices (3 blocks, 255 blocks of 32 K steps each).
int lora_xa_fast_slices(int M, int n_cols, int K) {
  (void)n_cols;
  const int tiles = ((M + 255) / 256) * (K > 4096 ? 2 : 5);
  const int KT = K / 64;
  int ks = 256 / (tiles > 0 ? tiles : 1);       // about one round of the chip
  const int kmax = KT / 8 > 1 ? KT / 8 : 1;      // keep >= 8 K steps per slice
  if (ks > kmax) ks = kmax;
  return ks < 1 ? 1 : ks;
}

// The tile of an adapters' x.A over its fixed slices (same bits in each): the
// 256 x 128 one stages the fewest bytes and is taken where its blocks fill
// half the chip; a narrow stack or a short x leaves it on a few CUs (one
// adapter of rank 16 at 4352 rows: 51 blocks, 42.3 us with its reduce) where
// 64-row tiles spread out (19.9). Measured over 64-1536 ranks, 300-16640 rows
// and K = 256 to 10240: up to 128 of its blocks the 64-row tiles take 0.4 to
// 0.9 of its time, from 132 it takes 0.75 to 1 of theirs (512 ranks at 8320
// rows, 132 blocks, K = 3840: 65.4 us against 73.8; at K = 256 1.1); at 130
// (256 ranks, 16640 rows) theirs are 8% faster at K = 3840, 2-6% slower at
// 10240, where a block stages more before it stores.
XaTile xa_tile(int M, int n_cols, int K, int kslices) {
  const long long blocks = (long long)((M + 255) / 256) * ((n_cols + 127) / 128) * kslices;
  if (blocks > (K > 4096 ? 128 : 130)) return {4, 2};
  return n_cols <= 64 ? XaTile{1, 1} : XaTile{1, 2};
}

size_t lora_xa_part_bytes(int M, int n_cols, int kslices, XaTile t) {
  if (kslices <= 1) return 0;
  const size_t xr = 64 * t.mr, xc = 64 * t.cj;
  return (size_t)kslices * (((size_t)M + xr - 1) / xr) * (((size_t)n_cols + xc - 1) / xc) *
         (xr * xc * 4);
}
size_t lora_xa_part_bytes(int M, int n_cols, int K, int kslices) {
  return lora_xa_part_bytes(M, n_cols, kslices, xa_tile(M, n_cols, K, kslices));
}

// A dense projection of fewer than 64 tiles of 256 x 256 through the x.A
// kernel: its tile and slices by a time model, and whether that beats one
// round of dense_fast.hip's 64-row tiles (about 4 us + 0.7 us a K stage). The
// model, us: a start, the larger of the staged bytes at the tile's rate and
// the stages of a block in its rounds, and for a split its reduce launch and
// the f32 partials, written and read at 5 TB/s; unsplit, at least the tile's
// own start (its scattered stores: the 256 x 128 one takes 10 us at one K
// stage, the 64 x 64 one 4, dense_fast 4.5), stages and a part a round of
// blocks. Measured with the weights rotated through more than the 256 MB
// cache, as a forward meets them, over 9-1024 rows of [64..15360] x [64..10240]
// in every tile and up to 12 slices; the plan against the best of those, us:
// 16 rows of [3840, 3840] 15.3 (128 x 128 in 8; 64 x 64 in 4 13.4), 231 of
// [3584, 2560] 17.7 (128 x 128 in 4, the best; 256 x 128 in 8 21.9), 1024 of
// [3840, 3840] 42.0 (256 x 128 in 2, the best; dense_fast 48.3), 203 of [10240,
// 256] 7.4 (dense_fast, the best; 256 x 128 unsplit 13.2). A gated call takes
// the same plan, though its SwiGLU is then a launch of its own: its bits are
// those of the plain call and ming_swiglu.
DensePlan dense_split_plan(int M, int N, int K) {
  const int KT = K / 64;
  DensePlan best = {{4, 2}, 0};
  double cost = 4.0 + 0.7 * KT;
  // the partials stay within what 256 x 128 tiles in one round would take
  const int cus = device_cus();
  const int tiles = ((M + 255) / 256) * ((N + 127) / 128);
  int kold = cus / (tiles > 0 ? tiles : 1);
  const int kmax = KT / 8 > 1 ? KT / 8 : 1;
  if (kold > kmax) kold = kmax;
  const size_t room = lora_xa_part_bytes(M, N, kold, {4, 2});
  const struct {
    XaTile t;
    int per_cu;                       // blocks a CU holds (LDS)
    double start_us, bytes_us, stage_us;
    double direct0, direct;           // unsplit, a short K: start and stage
  } cand[5] = {{{4, 2}, 1, 2.0, 14e6, 0.84, 8.8, 0.73},
               {{2, 2}, 1, 3.0, 11.5e6, 0.65, 5.0, 0.52},
               {{2, 1}, 2, 2.5, 10e6, 0.5, 3.9, 0.41},
               {{1, 2}, 2, 5.0, 10e6, 0.5, 4.0, 0.43},
               {{1, 1}, 3, 4.5, 10e6, 0.36, 3.1, 0.35}};
  for (const auto& c : cand) {
    const long long n = (long long)((M + 64 * c.t.mr - 1) / (64 * c.t.mr)) *
                        ((N + 64 * c.t.cj - 1) / (64 * c.t.cj));
    for (int ks = 1; ks == 1 || KT / ks >= 4; ++ks) {
      if (lora_xa_part_bytes(M, N, ks, c.t) > room) break;
      const double staged = (double)n * KT * (c.t.mr + c.t.cj) * 8192.0 / c.bytes_us;
      const double waits = (double)((n * ks + c.per_cu * cus - 1) / (c.per_cu * cus)) *
                           ((KT + ks - 1) / ks) * c.stage_us;
      double us = c.start_us + (staged > waits ? staged : waits);
      if (ks > 1) {
        us += 2.5 + 8.0 * ks * (double)M * N / 5e6;
      } else {
        const double own = c.direct0 + c.direct * KT + 1.2 * (double)n / cus;
        us = us > own ? us : own;
      }
      if (us < cost) {
        cost = us;
        best = {c.t, ks};
      }
    }
  }
  return best;
}

template <int MR, int CJ>
static hipError_t launch_xa_tiles(const LoraXaArgs& a, float* part, int kslices, hipStream_t s) {
  constexpr int XR = 64 * MR, XC = 64 * CJ;
  const long long tiles = (long long)((a.M + XR - 1) / XR) * ((a.n_cols + XC - 1) / XC);
  // the reduce's 32-bit indexing: one thread per two float4s of a slice
  const long long work = tiles * 1024 * MR * CJ;
  if (kslices > 1 && (a.n_cols % 8 != 0 || work >= (1ll << 31))) return hipErrorInvalidValue;
  hipLaunchKernelGGL((lora_xa_fast_kernel<MR, CJ>), dim3((unsigned)(tiles * kslices)), dim3(512),
                     0, s, a, part, kslices);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || kslices == 1) return e;
  long long blocks = (work / 2 + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL((lora_xa_reduce_kernel<MR, CJ>), dim3((unsigned)blocks), dim3(256), 0, s,
                     part, kslices, a.M, a.n_cols, a);
  return hipGetLastError();
}

hipError_t launch_lora_xa_fast(const LoraXaArgs& a, float* part, int kslices,
                               hipStream_t s) {
  if (a.M <= 0 || a.n_cols <= 0) return hipSuccess;
  const XaTile t = a.ident ? a.tile : xa_tile(a.M, a.n_cols, a.K, kslices);
  switch (10 * t.mr + t.cj) {
    case 11: return launch_xa_tiles<1, 1>(a, part, kslices, s);
    case 12: return launch_xa_tiles<1, 2>(a, part, kslices, s);
    case 21: return launch_xa_tiles<2, 1>(a, part, kslices, s);
    case 22: return launch_xa_tiles<2, 2>(a, part, kslices, s);
    case 42: return launch_xa_tiles<4, 2>(a, part, kslices, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_repack_fast(int bits, const uint32_t* codes,
                              const uint16_t* scales, const uint16_t* biases,
                              int N, int K, uint32_t* codes_f, uint32_t* sbf,
                              int* inexact, hipStream_t s) {
  hipLaunchKernelGGL(repack_fast_kernel, dim3(1024), dim3(256), 0, s, bits,
                     codes, N, K, codes_f);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(repack_sbf_kernel, dim3(256), dim3(256), 0, s, scales,
                     biases, N, K / 64, sbf, inexact);
  return hipGetLastError();
}

hipError_t launch_bf16_to_f16(const uint16_t* x, long long ldx, uint16_t* y,
                              long long ldy, int rows, int K, hipStream_t s, int* range) {
  long long work = (long long)rows * (K / 8);
  long long blocks = (work + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(bf16_to_f16_kernel, dim3((unsigned)blocks), dim3(256), 0,
                     s, x, ldx, y, ldy, rows, K, range);
  return hipGetLastError();
}

hipError_t validate_qproj_fast_kernels() {
  hipFuncAttributes fa;
  const void* fns[] = {reinterpret_cast<const void*>(&qproj_fast_kernel<4, false, 2, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<4, false, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<4, false, 6, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<4, false, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<4, true, 2, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<4, true, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<4, true, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<4, false, 2, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<4, false, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<4, false, 6, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<4, false, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<4, true, 2, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<4, true, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<4, true, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<8, false, 2, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<8, false, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<8, false, 6, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<8, false, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<8, true, 2, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<8, true, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_merged_kernel<8, true, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_pair_kernel<4, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_pair_kernel<4, 6, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<8, false, 2, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<8, false, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<8, false, 6, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<8, false, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<8, true, 2, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<8, true, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_fast_kernel<8, true, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_pair_kernel<8, 4, 8>),
                       reinterpret_cast<const void*>(&qproj_pair_kernel<8, 6, 8>),
                       reinterpret_cast<const void*>(&qproj_split_reduce_kernel),
                       reinterpret_cast<const void*>(&repack_fast_kernel),
                       reinterpret_cast<const void*>(&repack_sbf_kernel),
                       reinterpret_cast<const void*>(&bf16_to_f16_kernel),
                       reinterpret_cast<const void*>(&qproj_pair_kernel<4, 8, 4>),
                       reinterpret_cast<const void*>(&qproj_pair_kernel<8, 8, 4>),
                       reinterpret_cast<const void*>(&lora_xa_fast_kernel<1, 1>),
                       reinterpret_cast<const void*>(&lora_xa_reduce_kernel<1, 1>),
                       reinterpret_cast<const void*>(&lora_xa_fast_kernel<1, 2>),
                       reinterpret_cast<const void*>(&lora_xa_reduce_kernel<1, 2>),
                       reinterpret_cast<const void*>(&lora_xa_fast_kernel<2, 1>),
                       reinterpret_cast<const void*>(&lora_xa_reduce_kernel<2, 1>),
                       reinterpret_cast<const void*>(&lora_xa_fast_kernel<2, 2>),
                       reinterpret_cast<const void*>(&lora_xa_reduce_kernel<2, 2>),
                       reinterpret_cast<const void*>(&lora_xa_fast_kernel<4, 2>),
                       reinterpret_cast<const void*>(&lora_xa_reduce_kernel<4, 2>)};
  for (const void* f : fns) {
    const hipError_t e = hipFuncGetAttributes(&fa, f);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace ming
