// Matrix-core GEMM whose waves split K, C[M, N] = A[M, K] . B[N, K]^T (the
// kinds of gemm.hip, which includes this file).
//
// A workgroup owns a tile of 32 FN weight rows x 32 FM tokens; its W waves
// split K: wave w takes the 128-byte pieces w, w + W, ... of every operand row
// and accumulates the whole tile (v_mfma_f32_32x32x16_bf16 /
// v_mfma_i32_32x32x32_i8, weights as the A operand). No two waves need the
// same operand bytes, so each wave copies its own piece into its own part of
// the LDS (global_load_lds_dwordx4, the swizzled image of gemm_ring), waits
// for its own copies, reads the fragments once and requests its next piece
// under the MFMAs: no barrier until the W partial tiles are summed in LDS (in
// wave order, so the result does not depend on timing). Every operand byte is
// read from LDS once per workgroup, where waves arranged over the tile read
// it once per wave row or column.
//
// Bound: the copies. A workgroup moves (weight rows + tokens) x K bytes into
// LDS with at most its rings in flight, about 70 bytes per ns and CU (the L2
// answers in 1-2 us under this load), so the tile is the smallest that still
// covers the output with one workgroup per CU (the rule in gemm.hip). 2048x6144
// bf16 at 33 tokens: 31.4 us on 32 workgroups of the ring kernel, 10.1 us on
// 256 half tiles here (2.5 TB/s of weights); 2048x2048 13.5 -> 5.4 us;
// 12288x2048 SwiGLU at 64 tokens 25.5 -> 14.9 us. Loading the fragments from
// memory into registers without LDS was 1.5-4x slower: in the MFMA layout
// neighbouring lanes hold different rows, and each 1 KiB load then takes 61
// cycles of the texture unit in place of 16.
#pragma once
#include "q35_tile.hpp"

namespace {

enum { KIND_BF16 = 0, KIND_SWIGLU = 1, KIND_I32 = 2, KIND_DEQ = 3, KIND_DEQ_SWIGLU = 4, KIND_BIAS = 5, KIND_BIAS_GELU = 6 };
constexpr int kNumKinds = 5;  // kinds of q35_gemm; the bias kinds have their own entry

struct GemmArgs {
  const uint8_t* A;  // [M, K]
  const uint8_t* B;  // [N, K] (SwiGLU kinds: [2N, K])
  void* C;           // [M, N] bf16 or int32
  int M, N, K;       // K in elements
  const float* s_x;  // int8 kinds 3, 4: per-row scales of A
  const float* s_w;  // per-row scales of B; bias kinds: the bf16 bias [N]
  unsigned* cnt;     // split-K arrival counters, one per tile
  uint8_t* part;     // split-K partial tiles
  int splits, kps;   // splits per tile, stages per split
};

template <bool I8> struct GemmAcc { using T = q35_f32x16; using E = float; using Q = q35_f32x4; };
template <> struct GemmAcc<true> { using T = q35_i32x16; using E = int; using Q = q35_i32x4; };

constexpr bool kind_i8(int kind) { return kind >= KIND_I32 && kind <= KIND_DEQ_SWIGLU; }
constexpr bool kind_bias(int kind) { return kind == KIND_BIAS || kind == KIND_BIAS_GELU; }
// bf16 or int32 values straight from the accumulators
constexpr bool kind_direct(int kind) { return kind == KIND_BF16 || kind == KIND_I32 || kind_bias(kind); }
constexpr bool kind_swiglu(int kind) { return kind == KIND_SWIGLU || kind == KIND_DEQ_SWIGLU; }

Q35_DEV float bias_at(const GemmArgs& a, int n) { return bf2f(reinterpret_cast<const uint16_t*>(a.s_w)[n]); }

// Slot of 16-byte chunk c of tile row r in the swizzled LDS image.
template <int RB>
Q35_DEV int swz(int r) {
  return RB == 64 ? (r >> 2) & 3 : (r >> 1) & 7;
}

template <int FN, int FM, int W, int S, bool HALF, int KIND>
__global__ __launch_bounds__(W * 64) void gemm_ksplit(const GemmArgs a) {
  constexpr bool I8 = kind_i8(KIND);
  constexpr bool SWIGLU = kind_swiglu(KIND);
  constexpr int ES = I8 ? 1 : 2;
  constexpr int TM = 32 * FM;
  constexpr int NR = HALF ? 16 : 32 * FN;         // weight rows per tile
  constexpr int NC = SWIGLU ? NR / 2 : NR;        // output columns per tile
  constexpr int GB = NR / 8;                      // 1 KiB copies (8 rows) per piece of the weights
  constexpr int NG = GB + 4 * FM;                 // and of both operands
  constexpr int PIECE = NG * 1024;                // LDS bytes of a piece
  constexpr int RING = S * PIECE;                 // a wave's ring of S pieces
  constexpr int HV = FN * FM > 8 ? 2 : 1;  // a piece's fragments in registers at once, or half of them
  using AccT = typename GemmAcc<I8>::T;
  using QuadT = typename GemmAcc<I8>::Q;
  static_assert(S <= 3, "the waits count one or S - 1 pieces in flight");
  static_assert(!HALF || (FN == 1 && !SWIGLU), "a half tile is one block whose rows 16..31 repeat 0..15");
  static_assert(!SWIGLU || FN % 2 == 0, "SwiGLU tiles hold gate and up rows");
  // the sum: partial blocks (32 x 32, 4 KiB) of every wave, as many at a time as fit
  constexpr int UQ = SWIGLU ? 2 : 1;          // blocks of a unit: one, or gate and up
  constexpr int UNITS = FN * FM / UQ;
  constexpr int LIM = W * RING > 131072 ? W * RING : 131072;
  constexpr int UPP = LIM / (W * UQ * 4096) < UNITS ? LIM / (W * UQ * 4096) : UNITS;
  constexpr int PH = (UNITS + UPP - 1) / UPP;
  constexpr int LDSB = W * RING > W * UPP * UQ * 4096 ? W * RING : W * UPP * UQ * 4096;
  static_assert(UPP >= 1 && LDSB <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LDSB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, kh = lane >> 5;

  const int mt = (a.M + TM - 1) / TM;
  const int nt = (a.N + NC - 1) / NC;
  const int U = mt * nt;
  // consecutive units (the M tiles of one weight tile) on one XCD: workgroup b
  // (XCD b % 8) takes the b / 8-th of the XCD's eighth of the units
  const int xcd = (int)blockIdx.x & 7;
  const int u = xcd * (U >> 3) + min(xcd, U & 7) + ((int)blockIdx.x >> 3);
  const int m0 = (u % mt) * TM, n0 = (u / mt) * NC;
  const uint32_t rowb = (uint32_t)a.K * ES;
  const int np = (int)(rowb >> 7);                   // pieces of a row
  const int nw = w < np ? (np - 1 - w) / W + 1 : 0;  // pieces of this wave
  const int rot = (2 * (u & 15)) % np;

  // copy g: tile rows 8 g + lane / 8 (the 32 FN weight rows, then the tokens)
  uint32_t voff[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int r = 8 * g + (lane >> 3);
    int row;
    if (g >= GB) row = min(m0 + r - NR, a.M - 1);
    else if (SWIGLU) row = r < 16 * FN ? min(n0 + r, a.N - 1) : a.N + min(n0 + r - 16 * FN, a.N - 1);
    else row = min(n0 + r, a.N - 1);
    voff[g] = (uint32_t)row * rowb + 16u * (uint32_t)((lane & 7) ^ swz<128>(r));
  }
  uint8_t* mine = lds + w * RING;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_offset(lds) + (uint32_t)w * RING);
  auto copy = [&](int t, int slot) {
    int p = w + W * t + rot;
    if (p >= np) p -= np;
    const uint8_t* pb = a.B + (size_t)p * 128;
    const uint8_t* pa = a.A + (size_t)p * 128;
#pragma unroll
    for (int g = 0; g < NG; ++g) dma16(lds0 + (uint32_t)slot * PIECE + 1024u * g, g < GB ? pb : pa, voff[g]);
  };
  // fragment of k step s (16-byte chunk 2 s + kh) of 32-row block b
  uint32_t fo[4], fh[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    fo[s] = (uint32_t)l32 * 128 + 16u * (uint32_t)((2 * s + kh) ^ swz<128>(l32));
    fh[s] = (uint32_t)(l32 & 15) * 128 + 16u * (uint32_t)((2 * s + kh) ^ swz<128>(l32 & 15));
  }

  AccT acc[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

#pragma unroll
  for (int b = 0; b < S; ++b)
    if (b < nw) copy(b, b);
  int slot = 0;
  for (int t = 0; t < nw; ++t) {
    // this piece landed: at most the copies of the pieces after it are left
    if (S > 1 && t + S <= nw) wait_vm<(S - 1) * NG>();
    else if (S > 1 && t + 1 < nw) wait_vm<(S > 1 ? 1 : 0) * NG>();
    else wait_vm<0>();
    asm volatile("" ::: "memory");
    Q35_PIN();
    q35_u32x4 f[4 / HV][FN + FM];
#pragma unroll
    for (int h = 0; h < HV; ++h) {
#pragma unroll
      for (int s = 0; s < 4 / HV; ++s)
#pragma unroll
        for (int b = 0; b < FN + FM; ++b)
          f[s][b] = *reinterpret_cast<const q35_u32x4*>(
              mine + slot * PIECE + (b < FN ? 4096 * b : 128 * NR + 4096 * (b - FN)) +
              (HALF && b < FN ? fh : fo)[h * (4 / HV) + s]);
      if (h == HV - 1) {
        // the piece is in registers: its LDS may be overwritten
        wait_lds();
        asm volatile("" ::: "memory");
        Q35_PIN();
        if (t + S < nw) copy(t + S, slot);
        Q35_PIN();
      }
#pragma unroll
      for (int s = 0; s < 4 / HV; ++s)
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
          for (int j = 0; j < FM; ++j) acc[i][j] = mfma32(f[s][i], f[s][FN + j], acc[i][j]);
    }
    slot = slot + 1 == S ? 0 : slot + 1;
  }

  // ---- sum of the W partial tiles and the epilogue. Element 4 q + e of a
  // block: weight row 8 q + 4 kh + e, token l32. A partial block is staged as
  // [token][8 groups of 4 rows], group x of token t at slot (x + t) % 8, so the
  // writes (8 tokens of one group) and the reads (8 groups of one token) both
  // fall on distinct banks; a wave sums and stores 8 tokens x 32 rows at a time.
  const bool vec = (a.N & 3) == 0 && (((uintptr_t)a.C) & 15) == 0;
  const int grp = lane & 7;
#pragma unroll
  for (int ph = 0; ph < PH; ++ph) {
    __syncthreads();
#pragma unroll
    for (int x = 0; x < UPP; ++x) {
      const int unit = ph * UPP + x;
      if (unit >= UNITS) break;
#pragma unroll
      for (int g = 0; g < UQ; ++g) {
        const int i = unit / FM + g * (FN / 2), j = unit % FM;
        uint8_t* dst = lds + ((w * UPP + x) * UQ + g) * 4096 + l32 * 128;
#pragma unroll
        for (int q = 0; q < (HALF ? 2 : 4); ++q) {
          const QuadT v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
          *reinterpret_cast<QuadT*>(dst + 16 * ((2 * q + kh + l32) & 7)) = v;
        }
      }
    }
    __syncthreads();
    for (int y = w; y < UPP * 4; y += W) {
      const int x = y >> 2, unit = ph * UPP + x;
      if (unit >= UNITS) break;
      const int tok = 8 * (y & 3) + (lane >> 3);
      const uint8_t* src = lds + x * UQ * 4096 + tok * 128 + 16 * ((grp + tok) & 7);
      QuadT s[UQ];
#pragma unroll
      for (int g = 0; g < UQ; ++g) {
        s[g] = *reinterpret_cast<const QuadT*>(src + g * 4096);
#pragma unroll
        for (int v = 1; v < W; ++v) s[g] += *reinterpret_cast<const QuadT*>(src + (v * UPP * UQ + g) * 4096);
      }
      const int m = m0 + 32 * (unit % FM) + tok;
      const int n = n0 + 32 * (unit / FM) + 4 * grp;
      if (m >= a.M || n >= a.N || (HALF && grp >= 4)) continue;
      const size_t at = (size_t)m * a.N + n;
      if constexpr (KIND == KIND_I32) {
        int* C = reinterpret_cast<int*>(a.C) + at;
        if (vec) *reinterpret_cast<q35_i32x4*>(C) = s[0];
        else
          for (int e = 0; e < 4 && n + e < a.N; ++e) C[e] = s[0][e];
      } else {
        float v[UQ][4];
        const float sx = I8 ? a.s_x[m] : 0.f;
#pragma unroll
        for (int g = 0; g < UQ; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (I8) v[g][e] = (float)s[g][e] * sx * a.s_w[g * a.N + min(n + e, a.N - 1)];
            else v[g][e] = s[g][e];
            if constexpr (kind_bias(KIND)) v[g][e] += bias_at(a, min(n + e, a.N - 1));
            if constexpr (KIND == KIND_BIAS_GELU) v[g][e] = gelu_tanh_fast(v[g][e]);
          }
        if constexpr (SWIGLU) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[0][e] = round_bf(silu_fast(round_bf(v[0][e]))) * round_bf(v[1][e]);
        }
        uint16_t* C = reinterpret_cast<uint16_t*>(a.C) + at;
        if (vec) {
          *reinterpret_cast<uint2*>(C) = make_uint2(pack_bf2(v[0][0], v[0][1]), pack_bf2(v[0][2], v[0][3]));
        } else {
          for (int e = 0; e < 4 && n + e < a.N; ++e) C[e] = (uint16_t)f2bf(v[0][e]);
        }
      }
    }
  }
}

template <int FN, int FM, int W, int S, bool HALF, int KIND>
int launch_ksplit(const GemmArgs& a, hipStream_t stream) {
  constexpr int NC = HALF ? 16 : kind_swiglu(KIND) ? 16 * FN : 32 * FN;
  const long long units = (long long)((a.M + 32 * FM - 1) / (32 * FM)) * ((a.N + NC - 1) / NC);
  Q35_CHECK_ARG(units < (1ll << 31));
  gemm_ksplit<FN, FM, W, S, HALF, KIND><<<(unsigned)units, W * 64, 0, stream>>>(a);
  return q35_last_error();
}

}  // namespace
