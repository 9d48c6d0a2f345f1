// LM-head projection with a softmax-statistics epilogue: the logits producer
// of the sampling path (reference: models/qwen3/custom_builder.py:415 and
// models/qwen3_5/model.py:263, logits = lm_head(hidden), an nn.Linear without
// bias), fused with the per-row statistics a softmax of those logits needs.
//
//   out[m, n] = sum_k x[m, k] * w[n, k]          (fp32 accumulation, MFMA)
//   stats[m, b] = (max, sum exp(v - max))  over the 128 columns of block b,
//                 v = out[m, n] as stored (rounded to the output dtype)
//
// v_mfma_f32_32x32x16_{bf16,f16}: lane l holds A row l % 32 and B column l %
// 32, k = 8 (l / 32) .. +7; accumulator element i of lane l is row 8 (i / 4) +
// 4 (l / 32) + i % 4, column l % 32 (checked on gfx950).
//
// What bounds it: up to ~100 rows the weight's one pass over HBM, past ~250
// rows the matrix cores.  Both want the same thing, loads in flight that cost
// no registers and no waiting, so one kernel serves both.  A grid whose tiles
// all run at once takes the smallest tile of which that is true, others go by
// their rows (lmhead_shape):
//   rows <= 32    32 x 128, 4 waves, 3 stages of 128 columns (120 KB)
//   rows <= 64    64 x 128, 4 waves, 3 stages of 128 columns (144 KB)
//   rows <= 96    96 x 128, 4 waves, 5 stages of  64 columns (140 KB)
//   rows <= 128  128 x 128, 8 waves, 4 stages of  64 columns (128 KB)
//   257 .. 384   128 x 256, 4 waves, 2 stages of  64 columns (96 KB)
//   else         256 x 256, 8 waves, 2 stages of  64 columns (128 KB)
// Measured on rows x 4096 -> 151936 bf16 (us; before: 64 x 128 tiles staged
// through registers, one stage in flight): 1 row 260 -> 184 (6.8 TB/s of
// weight; a read of 2 GB reaches 7.1), 64 rows 262 -> 208, 96 rows 246, 128
// rows 274, 256 rows 370, 384 rows 554, 512 rows 627, 2048 rows 7570 -> 2319
// (1.10 PFLOP/s).  Other shapes at 64 rows: 6 stages of 64 columns 227 (as
// many bytes in flight, twice the barriers), 3 of 64 with two workgroups per
// CU 217, 64 x 256 tiles 227 (594 tiles are 2.3 rounds of 256 CUs); at 2048
// rows, in one process: 4 stages of 32 columns 2697 against 2451, 4 waves of
// 128 x 128 2521, 128 x 256 with two workgroups per CU 2942, without the
// priority hint 2531.
// Small grids (rows x 4096 -> V, us, by the rows' shape and as chosen; 64 x 128
// tiles through registers): 256 x 1000 99, 24 (46); 256 x 8192 99, 44 (50); 512 x
// 8192 100, 46 (95); 1024 x 8192 102, 73 (183); 256 x 32000 104, 77 (208).
#pragma once

#include "lps_common.h"
#include "lps_wave.h"

namespace lps {

constexpr int LMH_BN = 128;   // columns per statistics block
constexpr int LMH_MAX_ROWS = 65535 * 64;

struct LmHeadParams {
  const void* x;       // [M, H], row stride x_stride elements
  const void* w;       // [V, H], row stride w_stride elements
  void* out;           // [M, V], row stride out_stride elements
  float* stats;        // [M, G] pairs (max, sum), G = ceil(V / 128), or null
  int M, V, H;
  int64_t x_stride, w_stride, out_stride;
  int G;
  int mtiles, tiles;   // row tiles, all tiles
};

template <int DT> struct MfmaOps;
template <> struct MfmaOps<LPS_DTYPE_BF16> {
  typedef __bf16 v8 __attribute__((ext_vector_type(8)));
  typedef float acc __attribute__((ext_vector_type(16)));
  __device__ __forceinline__ static acc mma(u32x4 a, u32x4 b, acc c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
};
template <> struct MfmaOps<LPS_DTYPE_F16> {
  typedef _Float16 v8 __attribute__((ext_vector_type(8)));
  typedef float acc __attribute__((ext_vector_type(16)));
  __device__ __forceinline__ static acc mma(u32x4 a, u32x4 b, acc c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
};

// ---------------------------------------------------------------------------
// One workgroup of WM x WN waves computes a BM x BN tile; wave (i, j) owns rows
// i BM / WM and columns j BN / WN of it as 32 x 32 accumulators.  K is walked in
// stages of BK columns that stay in a ring of NS LDS buffers, filled by
// global_load_lds (16 bytes a lane, no registers): while a stage is multiplied
// the loads of the next NS - 1 are in flight.  The loads write LDS linearly
// (lane l at base + 16 l), so a row is BK * 2 bytes without padding; the
// 16-byte chunk c of row r sits at place c ^ f(r) of its row (the source
// address is permuted, not the destination), which spreads the fragment reads
// (one chunk from each of 32 rows) evenly over the banks.
// ---------------------------------------------------------------------------
template <int BM_, int BN_, int WM_, int WN_, int BK_, int NS_, int WPE_ = 1>
struct LmTile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, BK = BK_, NS = NS_, WPE = WPE_;
  static constexpr int NW = WM * WN, NT = 64 * NW;
  static constexpr int MT = BM / WM / 32, CT = BN / WN / 32;   // accumulators per wave: rows x columns
  static constexpr int CPR = BK / 8;                            // 16-byte chunks per row
  static constexpr int RPI = 64 / CPR;                          // rows one wave's load instruction covers
  static constexpr int ROWS = BM + BN;                          // X rows, then W rows
  static constexpr int LPW = ROWS / RPI / NW;                   // load instructions per wave and stage
  static constexpr int XPW = BM / RPI / NW;                     // ... of them X's
  static constexpr int STAGE = ROWS * BK * 2;                   // bytes
  static constexpr int KS = BK / 16;                            // matrix steps per stage
  static constexpr int WTN = 32 * CT;                           // columns per wave
  static_assert(ROWS % (RPI * NW) == 0 && BM % (RPI * NW) == 0, "whole load instructions per wave");
  static_assert(KS % 2 == 0 && BM % (32 * WM) == 0 && BN % (32 * WN) == 0 && BN % LMH_BN == 0, "tile shape");
  static_assert((NS - 1) * LPW < 64, "the load counter holds 63");
  // the permutation of a row's chunks: rows r and r + 1 of 64-byte rows share a
  // 128-byte bank line, wider rows fill one or more each
  __device__ __forceinline__ static int perm(int row) { return CPR >= 8 ? (row & 7) : ((row >> 1) & 3); }
};

// Epilogue rows in LDS: 32 rows of a wave's columns in the output type, padded by 16 bytes.
template <typename T, int ES>
constexpr int lmh_epi_bytes() {
  return T::NW * 32 * (T::WTN * ES + 16) + (T::WTN < LMH_BN ? T::BM * (T::BN / T::WTN) * 8 : 0);
}
template <typename T, int ES>
constexpr int lmh_lds_bytes() {
  return T::NS * T::STAGE > lmh_epi_bytes<T, ES>() ? T::NS * T::STAGE : lmh_epi_bytes<T, ES>();
}

#ifndef LPS_HOST_EMU
// 16 bytes per lane from g to LDS at (wave-uniform) base + 16 * lane.
template <bool NTL>
__device__ __forceinline__ void lmh_dma16(const char* g, char* base) {
  const uint32_t m0 = (uint32_t)__builtin_amdgcn_readfirstlane(
      (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)base);
  if constexpr (NTL)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(m0), "v"(g) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(m0), "v"(g) : "memory", "m0");
}
// All but the N youngest loads to LDS have landed, this wave's LDS reads are
// done; then every wave of the workgroup.
template <int N>
__device__ __forceinline__ void lmh_wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void lmh_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
#else
template <bool NTL>
inline void lmh_dma16(const char* g, char* base) { memcpy(base + 16 * ((int)threadIdx.x & 63), g, 16); }
template <int N>
inline void lmh_wait_barrier() { __syncthreads(); }
inline void lmh_wave_sync() { (void)__builtin_amdgcn_ballot_w64(true); }
#endif

// Stage s + 1 has landed when at most the `left` stages after it are in flight
// (NS - 2 of them until the last ones).
template <typename T>
__device__ __forceinline__ void lmh_wait_stage(int left) {
  constexpr int FULL = T::NS - 2;
  if (FULL > 0 && left >= FULL) lmh_wait_barrier<FULL * T::LPW>();
  else if (FULL > 2 && left == 2) lmh_wait_barrier<2 * T::LPW>();
  else if (FULL > 1 && left == 1) lmh_wait_barrier<T::LPW>();
  else lmh_wait_barrier<0>();
}

template <int DT, int ODT, typename T>
__device__ __forceinline__ void lmh_epilogue(const LmHeadParams& P, char* lds,
                                             const typename MfmaOps<DT>::acc (&acc)[T::MT][T::CT], int n0, int m0,
                                             int wv, int l) {
  constexpr int ES = ODT == LPS_DTYPE_F32 ? 4 : 2;
  constexpr int RS = T::WTN * ES + 16;             // LDS row (bytes)
  constexpr int PPR = T::WTN / 8, RPS = 64 / PPR;  // pieces per row, rows per step
  constexpr bool WHOLE = T::WTN == LMH_BN;         // the wave owns the block's columns
  constexpr int WPB = LMH_BN / T::WTN;             // waves per block
  static_assert(T::WTN <= LMH_BN && (PPR == 4 || PPR == 8 || PPR == 16), "epilogue shape");
  char* tile = lds + wv * 32 * RS;
  float* red = reinterpret_cast<float*>(lds + T::NW * 32 * RS);   // [BM][BN / WTN] pairs
  const int wm = wv / T::WN, wn = wv % T::WN;
  const int pr = l % PPR;
  const int c0 = n0 + wn * T::WTN + 8 * pr;        // this lane's columns c0 .. +7
  const bool aligned = ((reinterpret_cast<uintptr_t>(P.out) | (uintptr_t)(P.out_stride * ES)) & 15) == 0;
#pragma unroll
  for (int mt = 0; mt < T::MT; mt++) {
#pragma unroll
    for (int ct = 0; ct < T::CT; ct++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int row = 8 * (i >> 2) + 4 * (l >> 5) + (i & 3);
        char* d = tile + row * RS + (32 * ct + (l & 31)) * ES;
        const float v = acc[mt][ct][i];
        if constexpr (ODT == LPS_DTYPE_F32) *reinterpret_cast<float*>(d) = v;
        else if constexpr (ODT == LPS_DTYPE_BF16) *reinterpret_cast<unsigned short*>(d) = __builtin_bit_cast(unsigned short, (__bf16)v);
        else *reinterpret_cast<unsigned short*>(d) = __builtin_bit_cast(unsigned short, (_Float16)v);
      }
    lmh_wave_sync();
#pragma unroll
    for (int st = 0; st < 32 / RPS; st++) {
      const int r = st * RPS + l / PPR;            // row of the 32
      const int tr = wm * (T::MT * 32) + 32 * mt + r;   // row of the tile
      const int m = m0 + tr;
      const char* piece = tile + r * RS + 8 * pr * ES;
      u32x4 q[ES / 2];
#pragma unroll
      for (int e = 0; e < ES / 2; e++) q[e] = reinterpret_cast<const u32x4*>(piece)[e];
      if (P.stats) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          if constexpr (ODT == LPS_DTYPE_F32) {
            v[e] = __uint_as_float(q[e >> 2][e & 3]);
          } else {
            const uint32_t h = (q[0][e >> 1] >> (16 * (e & 1))) & 0xFFFFu;
            v[e] = ODT == LPS_DTYPE_BF16 ? bf16_to_f32(h) : f16_to_f32(h);
          }
          if (c0 + e >= P.V) v[e] = -INFINITY;
        }
        float mx = v[0];
#pragma unroll
        for (int e = 1; e < 8; e++) mx = fmaxf(mx, v[e]);
        mx = fmaxf(mx, dpp_t<0xB1>(mx, mx));    // quad_perm [1,0,3,2]
        mx = fmaxf(mx, dpp_t<0x4E>(mx, mx));    // quad_perm [2,3,0,1]
        if (PPR >= 8) mx = fmaxf(mx, dpp_t<0x141>(mx, mx));   // row_half_mirror
        if (PPR >= 16) mx = fmaxf(mx, dpp_t<0x140>(mx, mx));  // row_mirror
        // sum of exp2(v c - mx c), c = log2 e (a NaN or +inf value makes the sum NaN)
        // (a part whose values are all -inf counts 0: its block may hold others)
        const float mc = !WHOLE && mx == -INFINITY ? 0.0f : __fmul_rn(mx, 1.44269504088896340736f);
        float tsum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++)
          tsum += __builtin_amdgcn_exp2f(__builtin_fmaf(v[e], 1.44269504088896340736f, -mc));
        double s = (double)tsum;
        s += dpp_t<0xB1>(s, s);
        s += dpp_t<0x4E>(s, s);
        if (PPR >= 8) s += dpp_t<0x141>(s, s);
        if (PPR >= 16) s += dpp_t<0x140>(s, s);
        if (pr == 0) {
          if constexpr (WHOLE) {
            if (m < P.M && n0 + wn * T::WTN < P.V) {
              float* o = P.stats + ((int64_t)m * P.G + (n0 / LMH_BN + wn)) * 2;
              o[0] = mx;
              o[1] = (float)s;
            }
          } else {
            float* o = red + (tr * (T::BN / T::WTN) + wn) * 2;
            o[0] = mx;
            o[1] = (float)s;
          }
        }
      }
      if (aligned && m < P.M && c0 < P.V) {
        char* dst = reinterpret_cast<char*>(P.out) + ((int64_t)m * P.out_stride + c0) * ES;
        if (c0 + 8 <= P.V) {
#pragma unroll
          for (int e = 0; e < ES / 2; e++) reinterpret_cast<u32x4*>(dst)[e] = q[e];
        } else {
#pragma unroll
          for (int e = 0; e < 8; e++) {
            if (c0 + e < P.V) {
              if constexpr (ODT == LPS_DTYPE_F32) reinterpret_cast<uint32_t*>(dst)[e] = q[e >> 2][e & 3];
              else reinterpret_cast<unsigned short*>(dst)[e] = (unsigned short)(q[0][e >> 1] >> (16 * (e & 1)));
            }
          }
        }
      }
    }
    if (!aligned) {
      for (int i = l; i < 32 * T::WTN; i += 64) {
        const int r = i / T::WTN, c = i % T::WTN;
        const int m = m0 + wm * (T::MT * 32) + 32 * mt + r, n = n0 + wn * T::WTN + c;
        if (m < P.M && n < P.V) {
          const char* e = tile + r * RS + c * ES;
          char* dst = reinterpret_cast<char*>(P.out) + ((int64_t)m * P.out_stride + n) * ES;
          if constexpr (ODT == LPS_DTYPE_F32) *reinterpret_cast<uint32_t*>(dst) = *reinterpret_cast<const uint32_t*>(e);
          else *reinterpret_cast<unsigned short*>(dst) = *reinterpret_cast<const unsigned short*>(e);
        }
      }
    }
    lmh_wave_sync();
  }
  if constexpr (!WHOLE) {
    if (P.stats) {
      __syncthreads();
      // one thread per (row, block): the block's WPB pairs in column order
      constexpr int NB = T::BN / LMH_BN;
      for (int i = threadIdx.x; i < T::BM * NB; i += T::NT) {
        const int tr = i / NB, b = i % NB, m = m0 + tr;
        if (m >= P.M || n0 + b * LMH_BN >= P.V) continue;
        const float* p = red + (tr * (T::BN / T::WTN) + b * WPB) * 2;
        float mx = p[0];
#pragma unroll
        for (int w = 1; w < WPB; w++) mx = fmaxf(mx, p[2 * w]);
        const float mc = __fmul_rn(mx, 1.44269504088896340736f);
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < WPB; w++)   // a part of -inf or columns past V: 0 times 0
          s += (double)p[2 * w + 1] *
               (double)__builtin_amdgcn_exp2f(__fsub_rn(__fmul_rn(p[2 * w], 1.44269504088896340736f), mc));
        float* o = P.stats + ((int64_t)m * P.G + (n0 / LMH_BN + b)) * 2;
        o[0] = mx;
        o[1] = (float)s;
      }
    }
  }
}

// Accumulators Q0 .. Q1 - 1 (row-major) of a wave for one matrix step.
template <int DT, typename T, int Q0, int Q1>
__device__ __forceinline__ void lmh_mma(const u32x4 (&fx)[T::MT], const u32x4 (&fw)[T::CT],
                                        typename MfmaOps<DT>::acc (&acc)[T::MT][T::CT]) {
  __builtin_amdgcn_s_setprio(1);   // matrix instructions ahead of the other wave's address work
#pragma unroll
  for (int q = Q0; q < Q1; q++) acc[q / T::CT][q % T::CT] = MfmaOps<DT>::mma(fx[q / T::CT], fw[q % T::CT], acc[q / T::CT][q % T::CT]);
  __builtin_amdgcn_s_setprio(0);
}

template <int DT, int ODT, typename T, bool NTL>
__global__ __launch_bounds__(T::NT, T::WPE) void lmhead_kernel(LmHeadParams P) {
  constexpr int ES = ODT == LPS_DTYPE_F32 ? 4 : 2;
  constexpr int MT = T::MT, CT = T::CT, KS = T::KS;
  __shared__ __attribute__((aligned(1024))) char lds[lmh_lds_bytes<T, ES>()];
  // workgroup b runs on XCD b % 8: each XCD takes a contiguous run of tiles,
  // the row tiles of one column tile first, so a weight tile is fetched from
  // memory once and shared through the XCD's L2
  const int per = (P.tiles + 7) >> 3;
  const int t = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || t >= P.tiles) return;   // uniform over the workgroup
  const int m0 = (t % P.mtiles) * T::BM, n0 = (t / P.mtiles) * T::BN;
  const int wv = (int)threadIdx.x >> 6, l = (int)threadIdx.x & 63;
  const int wm = wv / T::WN, wn = wv % T::WN;

  // sources of this lane's chunks (rows clamped into range; their results are dropped)
  const char* src[T::LPW];
#pragma unroll
  for (int i = 0; i < T::LPW; i++) {
    const int row = (i * T::NW + wv) * T::RPI + l / T::CPR;
    const int c = (l % T::CPR) ^ T::perm(row);
    if (i < T::XPW) {
      const int m = m0 + row;
      src[i] = reinterpret_cast<const char*>(P.x) + ((int64_t)(m < P.M ? m : P.M - 1) * P.x_stride + c * 8) * 2;
    } else {
      const int n = n0 + row - T::BM;
      src[i] = reinterpret_cast<const char*>(P.w) + ((int64_t)(n < P.V ? n : P.V - 1) * P.w_stride + c * 8) * 2;
    }
  }
  const int ns = P.H / T::BK;   // whole stages; the rest of H follows them
  auto issue = [&](int buf) {   // the next stage into ring buffer buf
    char* base = lds + buf * T::STAGE + wv * 1024;
#pragma unroll
    for (int i = 0; i < T::LPW; i++) {
      if (i < T::XPW) lmh_dma16<false>(src[i], base + i * T::NW * 1024);
      else lmh_dma16<NTL>(src[i], base + i * T::NW * 1024);
      src[i] += T::BK * 2;
    }
  };

  typename MfmaOps<DT>::acc acc[MT][CT] = {};
  u32x4 fx[2][MT], fw[2][CT];
  // fragment rows of this lane: 32 t + l % 32 of the wave's rows / columns;
  // their chunk 2 j + l / 32 of matrix step j
  const int xr = wm * (MT * 32) + (l & 31), wr = T::BM + wn * T::WTN + (l & 31);
  const int px = T::perm(xr), pw = T::perm(wr);   // (rows 32 apart share it)
  auto frags = [&](const char* stage, int j, int b) {
    const int c = 2 * j + (l >> 5);
#pragma unroll
    for (int i = 0; i < MT; i++)
      fx[b][i] = *reinterpret_cast<const u32x4*>(stage + (xr + 32 * i) * (T::BK * 2) + ((c ^ px) * 16));
#pragma unroll
    for (int i = 0; i < CT; i++)
      fw[b][i] = *reinterpret_cast<const u32x4*>(stage + (wr + 32 * i) * (T::BK * 2) + ((c ^ pw) * 16));
  };
  if (ns > 0) {
#pragma unroll
    for (int s = 0; s < T::NS; s++)
      if (s < ns) issue(s);
    // stage 0 has landed once at most the stages after it are in flight
    if (ns >= T::NS) lmh_wait_barrier<(T::NS - 1) * T::LPW>();
    else lmh_wait_barrier<0>();
    frags(lds, 0, 0);
    int buf = 0;
    for (int s = 0; s < ns; s++) {
      const char* cur = lds + buf * T::STAGE;
      const int nb = buf + 1 == T::NS ? 0 : buf + 1;
#pragma unroll
      for (int j = 0; j < KS; j++) {
        constexpr int SP = MT * CT / 2, ALL = MT * CT;
        if (j + 1 < KS) {
          frags(cur, j + 1, (j + 1) & 1);
          lmh_mma<DT, T, 0, SP>(fx[j & 1], fw[j & 1], acc);
        } else {
          lmh_mma<DT, T, 0, SP>(fx[j & 1], fw[j & 1], acc);
          if (s + 1 < ns) {
            // every wave holds its last fragments of stage s, stage s + 1 has landed
            lmh_wait_stage<T>(ns - 2 - s);
            if (s + T::NS < ns) issue(buf);
            frags(lds + nb * T::STAGE, 0, 0);
          }
        }
        lmh_mma<DT, T, SP, ALL>(fx[j & 1], fw[j & 1], acc);
      }
      buf = nb;
    }
    __syncthreads();
  }
  if (ns * T::BK < P.H) {
    // the columns past the last whole stage, zero-filled up to one
    for (int i = threadIdx.x; i < T::ROWS * T::CPR; i += T::NT) {
      const int row = i / T::CPR, col = ns * T::BK + (((i % T::CPR) ^ T::perm(row)) * 8);
      u32x4 v = {0u, 0u, 0u, 0u};
      if (col < P.H) {
        const int m = m0 + row, n = n0 + row - T::BM;
        const char* p = row < T::BM
                            ? reinterpret_cast<const char*>(P.x) + ((int64_t)(m < P.M ? m : P.M - 1) * P.x_stride + col) * 2
                            : reinterpret_cast<const char*>(P.w) + ((int64_t)(n < P.V ? n : P.V - 1) * P.w_stride + col) * 2;
        v = *reinterpret_cast<const u32x4*>(p);
      }
      *reinterpret_cast<u32x4*>(lds + i * 16) = v;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < KS; j++) {
      if (ns * T::BK + j * 16 < P.H) {
        frags(lds, j, 0);
        lmh_mma<DT, T, 0, MT * CT>(fx[0], fw[0], acc);
      }
    }
    __syncthreads();
  }
  lmh_epilogue<DT, ODT, T>(P, lds, acc, n0, m0, wv, l);
}

}  // namespace lps
