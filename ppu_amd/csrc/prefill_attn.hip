// Causal GQA prefill attention over a bf16 K/V cache (heads of 256).
//
// q [B, QH, L, 256], K/V [B, KVH, cache_len, 256] (the prompt at cache offset
// kv_start), out [B, L, QH * 256]; query row i of a head attends to keys
// [0, kv_start + i]. Replaces the prefill attention interface call of
// reference integration.py:360-372.
#include "q35_tile.hpp"

namespace {

constexpr int kAD = 256;
constexpr int kFaKeys = 64;                 // keys per block
constexpr int kFaBlock = kFaKeys * kAD * 2; // bytes of a K or V block
constexpr int kFaWaves = 4;
constexpr int kFaRec = 32 * (kAD + 2);      // floats of a wave's split record
constexpr int kFaMaxSplits = 64;

Q35_DEV uint2 lds_read_tr16(const void* p) {
  typedef short q35_i16x4 __attribute__((ext_vector_type(4)));
  const q35_i16x4 v =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) q35_i16x4*)(p));
  return __builtin_bit_cast(uint2, v);
}
// 16-byte chunk c of a staged K or V row (32 chunks) sits at slot
// c ^ fa_swz(row): the 16 rows of a K fragment read and the 4 rows x 4 chunks
// of a transposed V read each fall on 16 distinct bank groups.
Q35_DEV uint32_t fa_swz(uint32_t r) { return ((r & 3) << 2) | ((r >> 2) & 3); }

template <bool V> struct FaTag { static constexpr bool value = V; };

// ------------------------------------------ causal prefill, 64-key blocks
// Flash attention on v_mfma_f32_32x32x16_bf16, transposed: a wave owns 32
// query rows of one head as the COLUMNS of every product,
//   S^T = K Q^T  (A = 32 keys x 16 dims from LDS, B = Q^T held in registers),
//   O^T += V^T P^T  (A = 32 dims x 16 keys from LDS, B = P^T),
// so a lane holds one query row: the softmax needs no cross-lane step but one
// exchange between lanes l and l ^ 32 per block, and the C layout of S^T is,
// with the 16 keys of a k step taken in the order {0-3, 8-11 | 4-7, 12-15},
// already the B operand of O^T: P never leaves the registers. P is kept as
// bf16 hi + lo (~16 mantissa bits, two MFMAs). V rows reach the A operand
// through the gfx950 transpose read ds_read_b64_tr_b16: within a 16-lane
// group, lane 4 e + q points at row e, column 4 q and lane i receives the 4
// rows of column i.
//
// A workgroup has 4 waves: HW = min(G, 4) query heads of one KV head x RT =
// 4 / HW row tiles, sharing the K and V blocks in LDS (two buffers each, rows
// copied straight into LDS a whole block ahead, one barrier per block). One
// wave runs per SIMD with up to 512 registers, so the vector work is
// interleaved by hand: the MFMAs of S for block j + 1 carry the copies of the
// following blocks and half of the exponentials of block j, the MFMAs of O the
// other half, the bf16 split of P and the scale and row maximum of block j + 1.
//
// The running maximum m (in units of log2) moves only when a row's block
// maximum passes it by 8: P stays below 2^8 and O is rescaled a few times per
// row instead of every block.
//
// Keys past the valid end are clamped to the last valid row on load (finite
// values) and masked to -inf in S, so they add exact zeros.
//
// Bound: per block and wave 96 MFMAs of 32 cycles (3072) against 256 KB of LDS
// reads per workgroup (2048 cycles); the 16-row form before it read the same
// 256 KB for half the rows and was bound by that. A block takes about 4640
// cycles (counters: MFMA 66 % of the wave's time) at 1.65-1.7 GHz, so the rest
// is near the power limit. 8 heads, 2 KV heads, with the merge, before and
// after: 1024 tokens 36 -> 28 us, 8192 tokens 827 -> 354 us (780 TFLOP/s of the
// causal products without the lo part). A workgroup has about 8 us of fixed
// cost (first copies, unoverlapped first and last block, record or row stores).
template <int G>
__global__ __launch_bounds__(kFaWaves * 64) void gqa_prefill_fa(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ Kc, const uint16_t* __restrict__ Vc,
    uint16_t* __restrict__ out, int B, int QH, int KVH, int L, int cache_len, int kv_start_host,
    const long long* __restrict__ valid_len, float scale, int sb, int smax, float* __restrict__ part) {
  constexpr int HW = G < 4 ? G : 4, RT = 4 / HW, QR = 32 * RT, HG = G / HW;
  // K buffers at 0 and 32 KiB, V buffers at 64 and 96 KiB
  __shared__ alignas(1024) uint8_t lds[4 * kFaBlock];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int l32 = lane & 31, kh = lane >> 5;
  // The last split of every tile, late tiles first, down to split 0: splits
  // 1 .. are whole ranges of sb blocks and split 0 the rest, so the longest
  // ranges start first, and every XCD (workgroup id % 8) gets all splits (with
  // the split as the fast index a power of two of them left XCDs idle: 213 us
  // in place of 110 at 4096 tokens).
  const int groups = KVH * HG, per = groups * B;
  const int ntiles = gridDim.x / (smax * per);
  const int grp = (int)blockIdx.x % groups, b = (int)blockIdx.x / groups % B;
  const int at = (int)blockIdx.x / per;
  const int tile = ntiles - 1 - at % ntiles;
  const int split = smax - 1 - at / ntiles;
  const int kvh = grp / HG;
  const int h = kvh * G + (grp % HG) * HW + w % HW;
  const int q0 = tile * QR, qw = q0 + 32 * (w / HW);
  // With a device length the prompt starts at valid_len - L + kv_start
  // (kv_start = 0 when the length already counts these L tokens, L when it
  // holds the start); the bound keeps reads in the cache.
  long long ks = valid_len ? valid_len[0] - L + kv_start_host : (long long)kv_start_host;
  if (ks < 0) ks = 0;
  if (ks + L > cache_len) ks = cache_len - L;
  const int kv_start = (int)ks;
  const int n_keys = min(kv_start + min(q0 + QR, L), cache_len);
  const int nblk = (n_keys + kFaKeys - 1) / kFaKeys;
  // This workgroup's key blocks [b0, b1) of the tile (sb blocks per split).
  const int nsplit = (nblk + sb - 1) / sb;
  if (split >= nsplit) return;  // whole workgroup: no barrier is skipped
  const int b1 = nblk - (nsplit - 1 - split) * sb, b0 = split ? b1 - sb : 0;
  const uint8_t* Kh = (const uint8_t*)(Kc + ((size_t)b * KVH + kvh) * cache_len * kAD);
  const uint8_t* Vh = (const uint8_t*)(Vc + ((size_t)b * KVH + kvh) * cache_len * kAD);

  // ---- copies: wave w takes row pairs g = w + 4 i (i < 8) of each block
  const uint32_t cr = 2u * w + kh;  // row of instruction i: cr + 8 i
  const uint32_t cc[2] = {16u * ((uint32_t)l32 ^ fa_swz(cr & 15)), 16u * ((uint32_t)l32 ^ fa_swz((cr + 8) & 15))};
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_offset(lds) + 1024u * (uint32_t)w);
  auto copy = [&](const uint8_t* base, uint32_t at, int blk, int i) {
    const uint32_t row = min(cr + 8u * i, (uint32_t)(n_keys - 1 - blk * kFaKeys));
    dma16(lds0 + at + 4096u * i, base + (size_t)blk * kFaBlock, row * (kAD * 2) + cc[i & 1]);
  };

  // ---- fragment addresses; the buffer is bit 15
  // K: row l32 of a 32-key half (the second half 16 KiB on), chunk 2 s + kh
  uint32_t ka[16];
#pragma unroll
  for (int s = 0; s < 16; ++s) ka[s] = (uint32_t)l32 * 512 + (16u * ((uint32_t)kh ^ fa_swz(l32 & 15)) ^ (32u * s));
  // V: rows 4 kh + e and 4 kh + 8 + e of a 16-key step (8 KiB each), dims
  // 32 d + 16 ((lane / 16) % 2) + 4 (lane % 4)
  uint32_t va[2][8];
  {
    const uint32_t e = (lane & 15) >> 2, cl = 2u * ((lane >> 4) & 1) + ((lane >> 1) & 1);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t row = 4u * kh + 8u * u + e;
      const uint32_t at = 2u * kFaBlock + row * 512 + 16u * (cl ^ fa_swz(row)) + 8u * (lane & 1);
#pragma unroll
      for (int d = 0; d < 8; ++d) va[u][d] = at ^ (64u * d);
    }
  }

  // ---- Q: column l32 of the B operand, dims 16 s + 8 kh ..
  q35_u32x4 qf[16];
  {
    const uint16_t* qp = q + (((size_t)b * QH + h) * L + min(qw + l32, L - 1)) * kAD + 8 * kh;
#pragma unroll
    for (int s = 0; s < 16; ++s) qf[s] = *reinterpret_cast<const q35_u32x4*>(qp + 16 * s);
  }
  const int row_abs = kv_start + min(qw + l32, L - 1);
  const int row_min = kv_start + min(qw, L - 1);
  const float c2 = scale * 1.4426950408889634f;

  q35_f32x16 o[8], sc[2], sn[2];
#pragma unroll
  for (int d = 0; d < 8; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
  float m = -INFINITY, l = 0.f, mx = -INFINITY;

  // ---- prologue: K and V of the first block, K of the second; S of the first
#pragma unroll
  for (int i = 0; i < 8; ++i) copy(Kh, 0, b0, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) copy(Vh, 2u * kFaBlock, b0, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) copy(Kh, kFaBlock, min(b0 + 1, b1 - 1), i);
  wait_vm<16>();
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) sn[t][r] = 0.f;
#pragma unroll
  for (int x = 0; x < 32; ++x)
    sn[x & 1] = mfma32(*reinterpret_cast<const q35_u32x4*>(lds + ka[x >> 1] + 16384 * (x & 1)), qf[x >> 1], sn[x & 1]);
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sc[t][r] = sn[t][r] * c2;
      mx = fmaxf(mx, sc[t][r]);
    }
#pragma unroll
  for (int s = 0; s < 16; ++s) ka[s] ^= (uint32_t)kFaBlock;
  wait_vm<0>();
  __syncthreads();

  // ---- one block: sc holds its scaled scores, mx their maximum over the
  // lane's keys; ka points at K of the next block, va at V of this one
  auto block = [&](int blk, auto next_tag) {
    constexpr bool NEXT = decltype(next_tag)::value;
    // O stays in AGPRs up to the rescale: without this the rescale's copies
    // out of them were made for every block, rescaled or not
#pragma unroll
    for (int d = 0; d < 8; ++d) asm volatile("" : "+a"(o[d]));
    q35_u32x4 kf[5], vf[2][8], ph[2], pl[2];
    auto readk = [&](int x) {
      kf[x % 5] = *reinterpret_cast<const q35_u32x4*>(lds + ka[x >> 1] + 16384 * (x & 1));
    };
    if constexpr (NEXT) {
#pragma unroll
      for (int x = 0; x < 4; ++x) readk(x);
      Q35_PIN();
    }
    if (blk * kFaKeys + kFaKeys - 1 > row_min || blk * kFaKeys + kFaKeys > n_keys) {
      mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = blk * kFaKeys + 32 * t + 8 * (r >> 2) + 4 * kh + (r & 3);
          if (key > row_abs || key >= n_keys) sc[t][r] = -INFINITY;
          mx = fmaxf(mx, sc[t][r]);
        }
    }
    mx = half_max(mx);
    if (__ballot(mx > m + 8.f)) {
#pragma unroll
      for (int d = 0; d < 8; ++d) asm volatile("" : "+a"(o[d]));
      const float mn = fmaxf(m, mx);
      const float corr = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
      l *= corr;
      if (__ballot(m != -INFINITY)) {  // else O is still zero
#pragma unroll
        for (int d = 0; d < 8; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[d][r] *= corr;
#pragma unroll
        for (int d = 0; d < 8; ++d) asm volatile("" : "+a"(o[d]));
      }
      m = mn;
    }
    // A row without any valid key so far keeps m = -inf: subtract 0 then.
    const float ms = m == -INFINITY ? 0.f : m;
    const uint32_t kbuf = (blk - b0) & 1 ? kFaBlock : 0;  // free: this block's K, the last one's V
    const uint32_t vbuf = 2u * kFaBlock + (kFaBlock - kbuf);

    float l1 = 0.f;
    auto ex = [&](int z) {  // exponential of element z
      const float p = __builtin_amdgcn_exp2f(sc[z >> 4][z & 15] - ms);
      sc[z >> 4][z & 15] = p;
      if (z & 1) l1 += p;
      else l += p;
    };
    auto split2 = [&](int kk, int e) {  // bf16 hi and lo of elements 2 e, 2 e + 1 of k step kk
      const float a = sc[kk >> 1][8 * (kk & 1) + 2 * e], c = sc[kk >> 1][8 * (kk & 1) + 2 * e + 1];
      const uint32_t hi = pack_bf2(a, c);
      ph[kk & 1][e] = hi;
      pl[kk & 1][e] = pack_bf2(a - bf_lo(hi), c - bf_hi(hi));
    };
    auto readv = [&](int kk, int d) {
      const uint2 a = lds_read_tr16(lds + va[0][d] + 8192 * kk), c = lds_read_tr16(lds + va[1][d] + 8192 * kk);
      vf[kk & 1][d] = q35_u32x4{a.x, a.y, c.x, c.y};
    };
    if constexpr (NEXT) {
#pragma unroll
      for (int x = 0; x < 32; ++x) {
        if (x < 2) {
          q35_f32x16 zero;
#pragma unroll
          for (int r = 0; r < 16; ++r) zero[r] = 0.f;
          sn[x] = mfma32(kf[x], qf[0], zero);
        } else {
          sn[x & 1] = mfma32(kf[x % 5], qf[x >> 1], sn[x & 1]);
        }
        if (x + 4 < 32) readk(x + 4);
        // every other slot: the texture unit takes a 1 KiB copy in 16 cycles
        if ((x & 1) == 0 && x < 16) copy(Kh, kbuf, min(blk + 2, b1 - 1), x >> 1);
        else if ((x & 1) == 0) copy(Vh, vbuf, blk + 1, (x >> 1) - 8);
        if (x >= 12 && x < 28) ex(x - 12);
        if (x >= 24) readv(0, x - 24);
        if (x >= 28) split2(0, x - 28);
        Q35_PIN();
      }
    } else {
#pragma unroll
      for (int d = 0; d < 8; ++d) readv(0, d);
#pragma unroll
      for (int z = 0; z < 16; ++z) ex(z);
#pragma unroll
      for (int e = 0; e < 4; ++e) split2(0, e);
      Q35_PIN();
    }
    if constexpr (NEXT) mx = -INFINITY;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
      for (int y = 0; y < 16; ++y) {
        const int d = y & 7;
        o[d] = mfma32(vf[kk & 1][d], y < 8 ? ph[kk & 1] : pl[kk & 1], o[d]);
        if (kk < 3) {
          if (y >= 6 && y < 14) readv(kk + 1, y - 6);
          if (kk < 2 && (y & 1) == 0) ex(16 + 8 * kk + (y >> 1));
          if ((y & 1) && y < 8) split2(kk + 1, y >> 1);
        } else if (NEXT) {
#pragma unroll
          for (int z = 2 * y; z < 2 * y + 2; ++z) {
            const float t = sn[z >> 4][z & 15] * c2;
            sc[z >> 4][z & 15] = t;
            mx = fmaxf(mx, t);
          }
        }
        Q35_PIN();
      }
    }
    l += l1;
    if constexpr (NEXT) {
#pragma unroll
      for (int s = 0; s < 16; ++s) ka[s] ^= (uint32_t)kFaBlock;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int d = 0; d < 8; ++d) va[u][d] ^= (uint32_t)kFaBlock;
      wait_vm<0>();
      __syncthreads();
    }
  };
  for (int blk = b0; blk + 1 < b1; ++blk) block(blk, FaTag<true>{});
  block(b1 - 1, FaTag<false>{});

  l = half_sum(l);
  if (nsplit > 1) {
    // This split's record: O relative to m, not yet divided by l, in register
    // order (quad q of dim tile d: 64 lanes x 16 bytes), then (m, l) per row.
    float* rec = part + (((((size_t)b * groups + grp) * ntiles + tile) * smax + split) * kFaWaves + w) * kFaRec;
#pragma unroll
    for (int d = 0; d < 8; ++d)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        *reinterpret_cast<float4*>(rec + ((d * 4 + u) * 64 + lane) * 4) =
            make_float4(o[d][4 * u], o[d][4 * u + 1], o[d][4 * u + 2], o[d][4 * u + 3]);
    if (kh == 0) *reinterpret_cast<float2*>(rec + 32 * kAD + 2 * l32) = make_float2(m, l);
    return;
  }
  // The final rows: bf16(O / l) through LDS (rows 528 bytes apart), stored as
  // whole 512-byte rows.
  __syncthreads();
  uint8_t* st = lds + w * (32 * 528);
  const float inv = 1.0f / l;
#pragma unroll
  for (int d = 0; d < 8; ++d)
#pragma unroll
    for (int u = 0; u < 4; ++u)
      *reinterpret_cast<uint2*>(st + l32 * 528 + 2 * (32 * d + 8 * u + 4 * kh)) =
          make_uint2(pack_bf2(o[d][4 * u] * inv, o[d][4 * u + 1] * inv),
                     pack_bf2(o[d][4 * u + 2] * inv, o[d][4 * u + 3] * inv));
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int r = 2 * i + kh;
    if (qw + r < L)
      *reinterpret_cast<q35_u32x4*>(out + ((size_t)b * L + qw + r) * QH * kAD + h * kAD + 8 * l32) =
          *reinterpret_cast<const q35_u32x4*>(st + r * 528 + 16 * l32);
  }
}

// Merge of the split records of the query tiles with more than one split: one
// workgroup per wave record (32 rows of one head), O = sum_s O_s 2^{m_s - M} /
// sum_s l_s 2^{m_s - M}, M = max_s m_s. Thread (lane, u) adds quads u + 4 i in
// the records' own order; the rows go out through LDS.
template <int G>
__global__ __launch_bounds__(256) void gqa_prefill_merge(
    const float* __restrict__ part, uint16_t* __restrict__ out, int B, int QH, int KVH, int L,
    int cache_len, int kv_start_host, const long long* __restrict__ valid_len, int sb, int smax) {
  constexpr int HW = G < 4 ? G : 4, RT = 4 / HW, QR = 32 * RT, HG = G / HW;
  __shared__ alignas(16) uint8_t st[32 * 528];
  __shared__ float f_s[kFaMaxSplits][32], inv_s[32];
  const int t = threadIdx.x, lane = t & 63, u = t >> 6;
  const int w = blockIdx.x & (kFaWaves - 1), tile = blockIdx.x / kFaWaves;
  const int ntiles = gridDim.x / kFaWaves;
  const int kvh = blockIdx.y / HG, b = blockIdx.z;
  const int h = kvh * G + (blockIdx.y % HG) * HW + w % HW;
  const int q0 = tile * QR, qw = q0 + 32 * (w / HW);
  long long ks = valid_len ? valid_len[0] - L + kv_start_host : (long long)kv_start_host;
  if (ks < 0) ks = 0;
  if (ks + L > cache_len) ks = cache_len - L;
  const int n_keys = min((int)ks + min(q0 + QR, L), cache_len);
  const int nblk = (n_keys + kFaKeys - 1) / kFaKeys;
  const int nsplit = (nblk + sb - 1) / sb;
  if (nsplit <= 1 || qw >= L) return;  // whole workgroup
  const size_t rs = (size_t)kFaWaves * kFaRec;
  const float* rec0 = part + ((((size_t)b * gridDim.y + blockIdx.y) * ntiles + tile) * smax * kFaWaves + w) * kFaRec;
  if (t < 32) {
    float mx = -INFINITY, lt = 0.f;
    for (int s = 0; s < nsplit; ++s) mx = fmaxf(mx, rec0[s * rs + 32 * kAD + 2 * t]);
    for (int s = 0; s < nsplit; ++s) {
      const float2 ml = *reinterpret_cast<const float2*>(rec0 + s * rs + 32 * kAD + 2 * t);
      const float f = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - mx);
      f_s[s][t] = f;
      lt += ml.y * f;
    }
    inv_s[t] = 1.0f / lt;
  }
  __syncthreads();
  const int l32 = lane & 31, kh = lane >> 5;
  float4 acc[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) acc[i] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s = 0; s < nsplit; ++s) {
    const float f = f_s[s][l32];
    const float* rec = rec0 + s * rs + ((size_t)u * 64 + lane) * 4;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float4 x = *reinterpret_cast<const float4*>(rec + i * 1024);
      acc[i].x = fmaf(x.x, f, acc[i].x);
      acc[i].y = fmaf(x.y, f, acc[i].y);
      acc[i].z = fmaf(x.z, f, acc[i].z);
      acc[i].w = fmaf(x.w, f, acc[i].w);
    }
  }
  const float inv = inv_s[l32];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    *reinterpret_cast<uint2*>(st + l32 * 528 + 2 * (32 * i + 8 * u + 4 * kh)) =
        make_uint2(pack_bf2(acc[i].x * inv, acc[i].y * inv), pack_bf2(acc[i].z * inv, acc[i].w * inv));
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 8 * i + (t >> 5);
    if (qw + r < L)
      *reinterpret_cast<q35_u32x4*>(out + ((size_t)b * L + qw + r) * QH * kAD + h * kAD + 8 * (t & 31)) =
          *reinterpret_cast<const q35_u32x4*>(st + r * 528 + 16 * (t & 31));
  }
}

// ---------------------------------------------------------- causal prefill
// q [B, QH, L, D], K/V [B, KVH, cache_len, D] (the prompt at cache offset
// kv_start), out [B, L, QH*D]. Query row i of a head attends to keys
// [0, kv_start + i]. One wave per (batch, head, query row); 4 keys per
// iteration, lane = (key kk = lane/16, 16-dim slice); online softmax in fp32.
__global__ __launch_bounds__(256) void gqa_prefill_rows(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ Kc, const uint16_t* __restrict__ Vc,
    uint16_t* __restrict__ out, int B, int QH, int KVH, int L, int cache_len, int kv_start_host,
    const long long* __restrict__ valid_len, float scale) {
  const int lane = threadIdx.x & 63;
  const long long wv = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wv >= (long long)B * QH * L) return;
  // With a device length the prompt starts at valid_len - L + kv_start
  // (kv_start = 0 when the length already counts these L tokens, L when it
  // holds the start); the bound keeps reads in the cache.
  long long ks = valid_len ? valid_len[0] - L + kv_start_host : (long long)kv_start_host;
  if (ks < 0) ks = 0;
  if (ks + L > cache_len) ks = cache_len - L;
  const int kv_start = (int)ks;
  // Heavy (late) rows first so that the tail of the grid is short.
  const int i = L - 1 - (int)(wv % L);
  const int h = (int)((wv / L) % QH);
  const int b = (int)(wv / ((long long)L * QH));
  const int kvh = h / (QH / KVH);
  const int ds = lane & 15;
  const uint16_t* qr = q + (((size_t)b * QH + h) * L + i) * kAD + ds * 16;
  float qf[16], t8[8];
  unpack8(*reinterpret_cast<const uint4*>(qr), t8);
  for (int j = 0; j < 8; ++j) qf[j] = t8[j] * scale;
  unpack8(*reinterpret_cast<const uint4*>(qr + 8), t8);
  for (int j = 0; j < 8; ++j) qf[8 + j] = t8[j] * scale;
  const uint16_t* Kh = Kc + ((size_t)b * KVH + kvh) * cache_len * kAD;
  const uint16_t* Vh = Vc + ((size_t)b * KVH + kvh) * cache_len * kAD;
  const int n = kv_start + i + 1;
  float m = -INFINITY, l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int t0 = 0; t0 < n; t0 += 4) {
    const int tok = t0 + (lane >> 4);
    const bool live = tok < n;
    float s = 0.f;
    if (live) {
      const uint16_t* kr = Kh + (size_t)tok * kAD + ds * 16;
      unpack8(*reinterpret_cast<const uint4*>(kr), t8);
      for (int j = 0; j < 8; ++j) s = fmaf(qf[j], t8[j], s);
      unpack8(*reinterpret_cast<const uint4*>(kr + 8), t8);
      for (int j = 0; j < 8; ++j) s = fmaf(qf[8 + j], t8[j], s);
    }
    uint2 vv[4];
    for (int k = 0; k < 4; ++k)
      vv[k] = t0 + k < n ? *reinterpret_cast<const uint2*>(Vh + (size_t)(t0 + k) * kAD + 4 * lane)
                         : make_uint2(0, 0);
    s = row16_sum(s);
    s = live ? s : -INFINITY;
    float sc[4];
    for (int k = 0; k < 4; ++k) sc[k] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 16 * k));
    const float m_new = fmaxf(m, fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3])));
    const float corr = expf(m - m_new);
    float p[4];
    for (int k = 0; k < 4; ++k) p[k] = expf(sc[k] - m_new);
    l = l * corr + ((p[0] + p[1]) + (p[2] + p[3]));
    for (int d = 0; d < 4; ++d) acc[d] *= corr;
    for (int k = 0; k < 4; ++k) {
      acc[0] = fmaf(p[k], bf_lo(vv[k].x), acc[0]);
      acc[1] = fmaf(p[k], bf_hi(vv[k].x), acc[1]);
      acc[2] = fmaf(p[k], bf_lo(vv[k].y), acc[2]);
      acc[3] = fmaf(p[k], bf_hi(vv[k].y), acc[3]);
    }
    m = m_new;
  }
  uint16_t* orow = out + ((size_t)b * L + i) * QH * kAD + h * kAD + 4 * lane;
  const float inv = 1.0f / l;
  *reinterpret_cast<uint2*>(orow) = make_uint2(pack_bf2(acc[0] * inv, acc[1] * inv),
                                               pack_bf2(acc[2] * inv, acc[3] * inv));
}

}  // namespace

extern "C" {

// Split plan: query tile t has nblk(t) key blocks and splits them into ranges
// of sb blocks, one workgroup each, late tiles first. sb minimises an estimate
// of the time in us over the prompt's tiles (it starts at key 0), one
// workgroup per CU (128 KB of LDS): 2.4 per block of the longest chain (the
// longest range while all run at once; beyond that the blocks over the CUs,
// plus what the dispatch order leaves uneven), 10 per round of workgroups, and
// the split records, 132 KB each, written at about 2.6 TB/s and read back.
// Measured with the merge (us, by sb): 1024 tokens 2: 35.5, 3: 31.5, 4: 28.4,
// 8: 29.7, unsplit 39.5; 2048 6: 58, 9: 54, 11: 45.1, 16: 47, unsplit 69; 3000
// 12: 83, 24: 69, 30: 75, unsplit 97; 4096 21: 123, 27: 136, 40: 108, unsplit
// 138; 6000 47: 237, unsplit 225; 8192 65: 372, unsplit 354. At most
// kFaMaxSplits ranges over the whole cache, which size the grid and the
// workspace. The plan depends only on (B, QH, KVH, L, cache_len), so
// q35_gqa_prefill_workspace sees the same one.
static int fa_device_cus() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
      cus = n;
    else
      cus = 256;
  }
  return cus;
}
struct FaPlan {
  int rows, groups, tiles, sb, smax;  // rows per tile, workgroups per tile and batch, tiles, blocks per split, splits
};
static FaPlan fa_plan(int B, int QH, int KVH, int L, int cache_len) {
  const int G = QH / KVH, hw = G < 4 ? G : 4;
  FaPlan p;
  p.rows = 32 * (4 / hw);
  p.groups = KVH * (G / hw);
  p.tiles = (L + p.rows - 1) / p.rows;
  const int nblk_max = (cache_len + kFaKeys - 1) / kFaKeys;
  // nblk takes each value 1 .. n about `rep` times over the tiles
  const int n = (L + kFaKeys - 1) / kFaKeys;
  const double rep = (double)kFaKeys / p.rows * p.groups * B, cus = fa_device_cus();
  const double share = rep * n * (n + 1) / 2 / cus;
  double best = 1e30;
  int sb = n;
  for (int c = n; c >= 2 || c == n; c = min(c - 1, c - c / 16)) {
    const double full = n / c, rest = n % c;
    const double wgs = rep * (c * full * (full + 1) / 2 + rest * (full + 1));  // sum of ceil(i / c)
    const double recs = wgs - rep * c;  // ranges of the split tiles (c == n: none)
    double span = c;
    if (wgs > cus && share + 0.25 * c > span) span = c == n ? (share > c ? share : c) : share + 0.25 * c;
    const double us = 2.4 * span + 10 * (wgs > cus ? wgs / cus : 1) + (c < n ? 3 + recs * (wgs > cus ? 0.04 : 0.06) : 0);
    // more ranges than CUs: the rests are dispatched in tile order, not by
    // size, which only tiles of at most two ranges of few tiles stand
    const bool uneven = wgs > cus && c < n && (2 * c <= n || rep * n > 1.25 * cus);
    if (!uneven && us < best) {
      best = us;
      sb = c;
    }
    if (c <= 2) break;
  }
  // unsplit: the whole cache in one range, unless it has room for a prompt
  // that starts late (a short one behind a long context still splits)
  if (sb == n) sb = nblk_max <= n + n / 4 ? nblk_max : max(n, 4);
  if (sb < (nblk_max + kFaMaxSplits - 1) / kFaMaxSplits) sb = (nblk_max + kFaMaxSplits - 1) / kFaMaxSplits;
  p.sb = sb;
  p.smax = (nblk_max + p.sb - 1) / p.sb;
  return p;
}
static bool fa_group(int QH, int KVH) {
  if (KVH <= 0 || QH <= 0 || QH % KVH) return false;
  const int G = QH / KVH;
  return G == 1 || G == 2 || G == 4 || G == 8;
}

long long q35_gqa_prefill_workspace(int B, int QH, int KVH, int L, int cache_len) {
  if (B <= 0 || L <= 0 || cache_len <= 0 || !fa_group(QH, KVH)) return 0;
  const FaPlan p = fa_plan(B, QH, KVH, L, cache_len);
  if (p.smax <= 1) return 0;
  return (long long)B * p.groups * p.tiles * p.smax * kFaWaves * kFaRec;
}

int q35_gqa_prefill(const void* q, const void* K, const void* V, void* out, int B, int QH, int KVH,
                    int D, int L, int cache_len, int kv_start, const void* valid_len, float scale,
                    void* workspace, long long workspace_floats, hipStream_t stream) {
  Q35_CHECK_ARG(D == kAD && KVH > 0 && QH % KVH == 0 && B >= 0 && L >= 0);
  Q35_CHECK_ARG(L <= cache_len && (valid_len || (kv_start >= 0 && kv_start + L <= cache_len)));
  Q35_CHECK_ARG(q35_aligned16(q) && q35_aligned16(K) && q35_aligned16(V) && q35_aligned16(out));
  if ((long long)B * QH * L == 0) return 0;
  if (fa_group(QH, KVH) && B < 65536 && KVH < 32768) {
    FaPlan p = fa_plan(B, QH, KVH, L, cache_len);
    if (p.smax <= 1 || !workspace || workspace_floats < q35_gqa_prefill_workspace(B, QH, KVH, L, cache_len)) {
      p.smax = 1;  // no room for the records: every tile in one range
      p.sb = (cache_len + kFaKeys - 1) / kFaKeys;
    }
    const long long wgs = (long long)p.tiles * p.smax * p.groups * B;
    Q35_CHECK_ARG(wgs < (1ll << 31));
    const unsigned grid = (unsigned)wgs;
    const dim3 mgrid((unsigned)(p.tiles * kFaWaves), (unsigned)p.groups, (unsigned)B);
#define Q35_FA(GG)                                                                               \
  do {                                                                                         \
    gqa_prefill_fa<GG><<<grid, kFaWaves * 64, 0, stream>>>(                                    \
        (const uint16_t*)q, (const uint16_t*)K, (const uint16_t*)V, (uint16_t*)out, B, QH, KVH,  \
        L, cache_len, kv_start, (const long long*)valid_len, scale, p.sb, p.smax,                \
        (float*)workspace);                                                                      \
    if (p.smax > 1)                                                                            \
      gqa_prefill_merge<GG><<<mgrid, 256, 0, stream>>>(                                        \
          (const float*)workspace, (uint16_t*)out, B, QH, KVH, L, cache_len, kv_start,           \
          (const long long*)valid_len, p.sb, p.smax);                                            \
  } while (0)
    switch (QH / KVH) {
      case 1: Q35_FA(1); break;
      case 2: Q35_FA(2); break;
      case 4: Q35_FA(4); break;
      default: Q35_FA(8); break;
    }
#undef Q35_FA
    return q35_last_error();
  }
  const long long waves = (long long)B * QH * L;
  Q35_CHECK_ARG(waves < (1ll << 31));
  gqa_prefill_rows<<<(unsigned)((waves + 3) / 4), 256, 0, stream>>>(
      (const uint16_t*)q, (const uint16_t*)K, (const uint16_t*)V, (uint16_t*)out, B, QH, KVH, L,
      cache_len, kv_start, (const long long*)valid_len, scale);
  return q35_last_error();
}

}  // extern "C"
