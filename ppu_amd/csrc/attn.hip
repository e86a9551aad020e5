// Full-attention layer kernels: Q/K RMSNorm + partial RoPE with the static
// KV-cache write, split-K GQA decode attention with a log-sum-exp combine
// (optionally fused with the sigmoid output gate), and causal GQA prefill
// attention.
//
// Layouts:
//   packed QGKV [B, L, 2*QH*D + 2*KVH*D] = per q head [q (D) | gate (D)], then k (KVH*D), v (KVH*D)
//   q           [B, QH, L, D] bf16
//   K/V cache   [B, KVH, cache_len, D] bf16; the valid length / write offset is
//               an int64 device scalar, so no launch depends on host state.
#include "q35_common.hpp"

namespace {

// ------------------------------------------------------------ QGKV norm + RoPE
// One wave per (token, q head); lane owns E = D/64 consecutive dims.
// Rounding points follow the reference kernel (kernels.py:419-573):
//   n = bf16(x * rsqrt(mean(x^2) + 1e-6) * (1 + w))
//   rot = bf16(bf16(n*cos) + bf16(bf16(+-n_partner) * sin)) for dims < rotary_dim
template <int E>
Q35_DEV void norm_head(const uint16_t* __restrict__ src, const void* w, int w_f32, int lane, int D,
                       float (&n)[E]) {
  float x[E];
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    x[e] = bf2f(src[lane * E + e]);
    ss += x[e] * x[e];
  }
  const float inv = rsqrt_cr(wave_sum(ss) / (float)D + 1.0e-6f);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int c = lane * E + e;
    const float wc = w_f32 ? reinterpret_cast<const float*>(w)[c] : bf2f(reinterpret_cast<const uint16_t*>(w)[c]);
    n[e] = round_bf(x[e] * inv * (1.0f + wc));
  }
}

template <int E>
Q35_DEV void rope_head(const float (&n)[E], const uint16_t* __restrict__ cos,
                       const uint16_t* __restrict__ sin, int lane, int rot, float (&o)[E]) {
  const int half = rot / 2;
  const int shift = half / E;  // partner lane distance (half is a multiple of E)
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int c = lane * E + e;
    const int partner_lane = c < half ? lane + shift : lane - shift;
    const float pn = __shfl(n[e], partner_lane & 63, 64);
    if (c < rot) {
      const float cs = bf2f(cos[c]), sn = bf2f(sin[c]);
      const float qc = round_bf(n[e] * cs);
      const float rh = c < half ? -pn : pn;
      const float qs = round_bf(rh * sn);
      o[e] = round_bf(qc + qs);
    } else {
      o[e] = n[e];
    }
  }
}

template <int E>
__global__ __launch_bounds__(256) void qgkv_norm_rope_k(
    const uint16_t* __restrict__ packed, const void* qw, const void* kw, int w_f32,
    const uint16_t* __restrict__ cos, const uint16_t* __restrict__ sin, uint16_t* __restrict__ q_out,
    uint16_t* __restrict__ k_out, uint16_t* __restrict__ v_out, const long long* cache_start,
    int B, int L, int QH, int KVH, int D, int rot, int cache_len) {
  const int lane = threadIdx.x & 63;
  const int pid = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (pid >= B * L * QH) return;
  const int head = pid % QH;
  const int tf = pid / QH;  // b*L + t
  const int t = tf % L, b = tf / L;
  const int P = 2 * QH * D + 2 * KVH * D;
  const uint16_t* row = packed + (size_t)tf * P;
  const uint16_t* cs = cos + (size_t)tf * rot;
  const uint16_t* sn = sin + (size_t)tf * rot;

  float n[E], o[E];
  norm_head<E>(row + head * 2 * D, qw, w_f32, lane, D, n);
  rope_head<E>(n, cs, sn, lane, rot, o);
  uint16_t* qo = q_out + (((size_t)b * QH + head) * L + t) * D;
#pragma unroll
  for (int e = 0; e < E; ++e) qo[lane * E + e] = (uint16_t)f2bf(o[e]);

  if (head < KVH) {
    const uint16_t* krow = row + 2 * QH * D + head * D;
    const uint16_t* vrow = row + 2 * QH * D + KVH * D + head * D;
    norm_head<E>(krow, kw, w_f32, lane, D, n);
    rope_head<E>(n, cs, sn, lane, rot, o);
    long long pos = t;
    int len = L;
    if (cache_start) {
      pos += cache_start[0];
      len = cache_len;
    }
    if (pos >= 0 && pos < len) {  // never write outside the cache
      const size_t off = (((size_t)b * KVH + head) * len + pos) * D;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        k_out[off + lane * E + e] = (uint16_t)f2bf(o[e]);
        v_out[off + lane * E + e] = vrow[lane * E + e];
      }
    }
  }
}

// ------------------------------------------------------- GQA split-K decode
// Grid (KVH, splits): a workgroup reads one contiguous chunk of one KV head
// once and serves all G = QH/KVH query heads of that head, so K/V bytes are
// read from HBM exactly once per step. D = 256. A workgroup of 4 waves covers
// 32 tokens per iteration, 8 per wave in two groups of 4 (8 waves, two per
// SIMD, measured no faster: the per-workgroup latency chain dominates):
//   QK: lane = (token row lane/16 of a group, dims 8*(lane%16) and
//       128 + 8*(lane%16)); bf16 pair dot products (v_dot2) reduced over the
//       16-lane DPP row, then times the softmax scale.
//   PV: lane owns dims 4*lane..4*lane+3; p values are broadcast by readlane.
// The loads that the Q/K norm + RoPE prologue needs are issued first and the
// K/V rows of the first iteration right after, so the prologue runs while
// K/V are in flight (loads retire in order); later iterations are prefetched
// one ahead. Each wave runs an online softmax over its tokens, the waves are
// merged in LDS and the workgroup writes (acc[D], m, l) per query head and
// split; gqa_decode_combine merges the splits.
constexpr int kAD = 256;
constexpr int kMaxG = 8;
constexpr int kSplitWaves = 4;                // waves per split workgroup
constexpr int kWaveTok = 32 / kSplitWaves;    // tokens per wave per iteration
constexpr int kWaveGroups = kWaveTok / 4;     // K row groups of 4 tokens per wave
static_assert(kWaveTok % 4 == 0 && kWaveGroups >= 1, "4-token K row groups per wave");
constexpr int kIterTok = kSplitWaves * kWaveTok;  // tokens per workgroup iteration
constexpr int kMaxSplits = 128;            // splits per KV head

// Extra inputs of the fused decode step: the packed QGKV row of the current
// token, the Q/K norm weights, the rotary frequencies and positions. The
// kernel then normalises and rotates q itself (every workgroup, its own G
// heads), and the workgroup whose chunk holds the new token also computes
// k, writes k and v into the cache and attends to the new token from LDS.
struct FusedQ {
  const uint16_t* packed;      // [2*QH*D + 2*KVH*D]
  const void* q_w;
  const void* k_w;
  int w_f32;
  const float* inv_freq;       // [rot/2] fp32
  const long long* pos_t;      // text/temporal position
  const long long* pos_h;      // multimodal rope rows (may equal pos_t)
  const long long* pos_w;
  int sec_h, sec_w;            // interleaved mrope: frequencies taken from H / W rows
  int rot;                     // rotary dims (64)
  uint16_t* k_cache;           // written at the new token's position
  uint16_t* v_cache;
};

// Global loads of one 256-wide head (lane: dims 4*lane..+3) and its norm
// weights (bf16 in w0, or fp32 in w0:w1).
struct HeadLoads {
  uint2 x, w0, w1;
};
Q35_DEV HeadLoads load_head(const uint16_t* __restrict__ src, const void* w, int w_f32, int lane) {
  HeadLoads h;
  h.x = *reinterpret_cast<const uint2*>(src + 4 * lane);
  const char* wb = reinterpret_cast<const char*>(w) + (w_f32 ? 16 * lane : 8 * lane);
  h.w0 = *reinterpret_cast<const uint2*>(wb);
  h.w1 = *reinterpret_cast<const uint2*>(wb + (w_f32 ? 8 : 0));
  return h;
}

// Rotary inputs: lane j owns frequency i = j mod rot/2 (rot/2 <= 64).
struct RopeLoads {
  float invf;
  long long pt, ph, pw;
};
Q35_DEV RopeLoads load_rope(const FusedQ& f, int lane) {
  // The positions are vector loads (nontemporal): issued in program order
  // with the other prologue loads, they return before the K/V stream instead
  // of waiting on the scalar cache.
  RopeLoads r;
  r.invf = f.inv_freq[lane % (f.rot / 2)];
  r.pt = __builtin_nontemporal_load(f.pos_t);
  r.ph = __builtin_nontemporal_load(f.pos_h);
  r.pw = __builtin_nontemporal_load(f.pos_w);
  return r;
}

// cos/sin of the lane's 4 dims (bf16-rounded), shared by every head of the
// token: freq_i = pos * inv_freq[i] in fp32, the position row of frequency i
// chosen by the interleaved multimodal sections, cos/sin in fp32 rounded to
// bf16, exactly as Transformers' rotary table; dims c and c + rot/2 share
// frequency c mod rot/2. Lane j computes frequency j mod rot/2 once and the
// lanes gather theirs by shuffle.
struct RopeTable {
  float cs[4], sn[4];
};
Q35_DEV RopeTable rope_table(const RopeLoads& r, const FusedQ& f, int lane) {
  const int half = f.rot / 2;
  const int i = lane % half;
  long long p = r.pt;
  if (i % 3 == 1 && i < 3 * f.sec_h) p = r.ph;
  if (i % 3 == 2 && i < 3 * f.sec_w) p = r.pw;
  float sn, cs;
  sincosf((float)p * r.invf, &sn, &cs);
  cs = round_bf(cs);
  sn = round_bf(sn);
  RopeTable t;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int src = (lane * 4 + e) % half;
    t.cs[e] = __shfl(cs, src, 64);
    t.sn[e] = __shfl(sn, src, 64);
  }
  return t;
}

// Q/K RMSNorm (1 + w) + partial RoPE of one head from its loads. Rounding
// points follow the reference kernel (kernels.py:419-573):
//   n = bf16(x * rsqrt(mean(x^2) + 1e-6) * (1 + w))
//   rot = bf16(bf16(n*cos) + bf16(bf16(+-n_partner) * sin)) for dims < rot
Q35_DEV void norm_rope(const HeadLoads& h, int w_f32, const RopeTable& t, int rot, int lane,
                       float (&o)[4]) {
  const float x[4] = {bf_lo(h.x.x), bf_hi(h.x.x), bf_lo(h.x.y), bf_hi(h.x.y)};
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) ss += x[e] * x[e];
  const float inv = rsqrt_cr(wave_sum(ss) / (float)kAD + 1.0e-6f);
  float wc[4];
  if (w_f32) {
    wc[0] = __uint_as_float(h.w0.x); wc[1] = __uint_as_float(h.w0.y);
    wc[2] = __uint_as_float(h.w1.x); wc[3] = __uint_as_float(h.w1.y);
  } else {
    wc[0] = bf_lo(h.w0.x); wc[1] = bf_hi(h.w0.x); wc[2] = bf_lo(h.w0.y); wc[3] = bf_hi(h.w0.y);
  }
  float n[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) n[e] = round_bf(x[e] * inv * (1.0f + wc[e]));
  const int half = rot / 2;
  const int shift = half / 4;
  // Partner of dim c is c + half (first half) or c - half: lane +- half/4.
  const bool first = lane * 4 < half;
  const int partner_lane = (first ? lane + shift : lane - shift) & 63;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float pn = __shfl(n[e], partner_lane, 64);
    const float qc = round_bf(n[e] * t.cs[e]);
    const float rh = first ? -pn : pn;
    const float r = round_bf(qc + round_bf(rh * t.sn[e]));
    o[e] = lane * 4 < rot ? r : n[e];
  }
}

// Prefill Q/K norm + RoPE for 256-wide heads (the qgkv_norm_rope_k contract,
// same arithmetic as norm_rope): one wave per (token, query head), lane dims
// 4*lane .. +3. Every load (the q head and its norm weights, the token's
// cos/sin, and the k and v heads with the k weights, read by every wave and
// used by waves of heads < KVH) is an 8-byte vector load issued before any
// arithmetic; the weight type is chosen by address, so no branch separates
// the loads. rot > 0, rot % 8 == 0 (checked on the host).
__global__ __launch_bounds__(256) void qgkv_norm_rope_256(
    const uint16_t* __restrict__ packed, const void* qw, const void* kw, int w_f32,
    const uint16_t* __restrict__ cos, const uint16_t* __restrict__ sin, uint16_t* __restrict__ q_out,
    uint16_t* __restrict__ k_out, uint16_t* __restrict__ v_out, const long long* cache_start,
    int B, int L, int QH, int KVH, int rot, int cache_len) {
  const int lane = threadIdx.x & 63;
  const int pid = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (pid >= B * L * QH) return;
  const int head = pid % QH;
  const int tf = pid / QH;  // b*L + t
  const int t = tf % L, b = tf / L;
  const uint16_t* row = packed + (size_t)tf * (2 * QH * kAD + 2 * KVH * kAD);
  const int kh = min(head, KVH - 1);
  const HeadLoads hq = load_head(row + head * 2 * kAD, qw, w_f32, lane);
  const HeadLoads hk = load_head(row + 2 * QH * kAD + kh * kAD, kw, w_f32, lane);
  const uint2 vv = *reinterpret_cast<const uint2*>(row + 2 * QH * kAD + KVH * kAD + kh * kAD + 4 * lane);
  const int rc = (4 * lane) % rot;  // lanes past rot/4 read valid, unused entries
  const uint2 cr = *reinterpret_cast<const uint2*>(cos + (size_t)tf * rot + rc);
  const uint2 sr = *reinterpret_cast<const uint2*>(sin + (size_t)tf * rot + rc);
  const long long start = cache_start ? cache_start[0] : 0;
  RopeTable tab;
  tab.cs[0] = bf_lo(cr.x); tab.cs[1] = bf_hi(cr.x); tab.cs[2] = bf_lo(cr.y); tab.cs[3] = bf_hi(cr.y);
  tab.sn[0] = bf_lo(sr.x); tab.sn[1] = bf_hi(sr.x); tab.sn[2] = bf_lo(sr.y); tab.sn[3] = bf_hi(sr.y);
  float o[4];
  norm_rope(hq, w_f32, tab, rot, lane, o);
  uint16_t* qo = q_out + (((size_t)b * QH + head) * L + t) * kAD + 4 * lane;
  *reinterpret_cast<uint2*>(qo) = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
  if (head < KVH) {
    norm_rope(hk, w_f32, tab, rot, lane, o);
    const long long pos = t + start;
    const int len = cache_start ? cache_len : L;
    if (pos >= 0 && pos < len) {  // never write outside the cache
      const size_t off = (((size_t)b * KVH + head) * len + pos) * kAD + 4 * lane;
      *reinterpret_cast<uint2*>(k_out + off) = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
      *reinterpret_cast<uint2*>(v_out + off) = vv;
    }
  }
}

// Max of a value that is uniform within each 16-lane row, over the 4 rows.
Q35_DEV float rows4_max(float v) {
  const float r0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
  const float r1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16));
  const float r2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
  const float r3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 48));
  return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

Q35_DEV float dot2_bf16(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(q35_bf16x2, a),
                                         __builtin_bit_cast(q35_bf16x2, b), c, false);
}

template <int G, bool FUSED>
__global__ __launch_bounds__(kSplitWaves * 64) void gqa_decode_split(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ Kc, const uint16_t* __restrict__ Vc,
    const long long* __restrict__ valid_len, float* __restrict__ acc_out, float* __restrict__ ml_out,
    int cache_len, int chunk, int splits, float scale, const FusedQ fq) {
  constexpr int NW = kSplitWaves;
  constexpr int HPW = (G + NW - 1) / NW;  // query heads per wave in the prologue
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int kvh = blockIdx.x;
  const int split = blockIdx.y;
  const int KVH = gridDim.x;
  const int QH = G * KVH;
  // FUSED: valid_len counts the tokens before this one; the new token sits at
  // index n_old and is attended from LDS by the workgroup that owns it.
  const long long n_old = FUSED ? valid_len[0] : 0;
  const int n_cached = FUSED ? (int)min((long long)cache_len, n_old)
                             : (int)min((long long)cache_len, valid_len[0]);
  const int start = split * chunk;
  const int end = min(start + chunk, n_cached);
  const bool owns_new = FUSED && n_old >= start && n_old < start + chunk;
  const int n_iter = end > start ? (end - start + kIterTok - 1) / kIterTok : 0;

  // 1. prologue loads: the wave's query heads, and (FUSED) the new token's k
  //    and v rows, the norm weights and the rotary inputs.
  HeadLoads hq[HPW], hk;
  uint2 vnew = make_uint2(0, 0);
  RopeLoads rl;
#pragma unroll
  for (int j = 0; j < HPW; ++j) {
    const int g = (wid + NW * j) % G;
    if (FUSED) {
      hq[j] = load_head(fq.packed + (size_t)(kvh * G + g) * 2 * kAD, fq.q_w, fq.w_f32, lane);
    } else {
      hq[j].x = *reinterpret_cast<const uint2*>(q + (size_t)(kvh * G + g) * kAD + 4 * lane);
    }
  }
  if (FUSED) {
    const uint16_t* krow = fq.packed + (size_t)2 * QH * kAD + (size_t)kvh * kAD;
    hk = load_head(krow, fq.k_w, fq.w_f32, lane);
    vnew = *reinterpret_cast<const uint2*>(krow + (size_t)KVH * kAD + 4 * lane);
    rl = load_rope(fq, lane);
  }

  // 2. K/V rows of the first iteration. Group gi of a wave holds tokens
  //    tb + 4*gi + row (K, the lane's 16 dims), V rows tb + i (dims 4*lane..).
  //    The row indices do not depend on the valid length (a device scalar
  //    whose load would otherwise delay every K/V request by a round trip):
  //    they are clamped to the chunk's last row inside the cache capacity,
  //    and rows at or past the valid end (whatever bits they hold) are
  //    masked out of the softmax and their V values replaced by zeros.
  const uint16_t* Kh = Kc + (size_t)kvh * cache_len * kAD;
  const uint16_t* Vh = Vc + (size_t)kvh * cache_len * kAD;
  const int rw = lane >> 4;
  const int ds = lane & 15;
  const int tmax = min(start + chunk, cache_len) - 1;
  uint4 kr[kWaveGroups][2];
  uint2 vr[kWaveTok];
  auto load_kv = [&](int it, uint4 (&kd)[kWaveGroups][2], uint2 (&vd)[kWaveTok]) {
    const int tb = start + it * kIterTok + wid * kWaveTok;
#pragma unroll
    for (int gi = 0; gi < kWaveGroups; ++gi) {
      const int t = min(tb + 4 * gi + rw, tmax);
      kd[gi][0] = *reinterpret_cast<const uint4*>(Kh + (size_t)t * kAD + ds * 8);
      kd[gi][1] = *reinterpret_cast<const uint4*>(Kh + (size_t)t * kAD + 128 + ds * 8);
    }
#pragma unroll
    for (int i = 0; i < kWaveTok; ++i) {
      const int t = min(tb + i, tmax);
      vd[i] = *reinterpret_cast<const uint2*>(Vh + (size_t)t * kAD + 4 * lane);
    }
  };
  load_kv(0, kr, vr);

  // 3. prologue: q heads (bf16 pairs, unscaled) into LDS; FUSED also the new
  //    token's k and v, written into the cache by the owning workgroup.
  __shared__ uint2 q_s[G][kAD / 4];
  __shared__ float kn_s[FUSED ? kAD : 1], vn_s[FUSED ? kAD : 1];
  RopeTable rt;
  if (FUSED) rt = rope_table(rl, fq, lane);
#pragma unroll
  for (int j = 0; j < HPW; ++j) {
    const int g = wid + NW * j;
    if (g < G) {
      if (FUSED) {
        float o[4];
        norm_rope(hq[j], fq.w_f32, rt, fq.rot, lane, o);
        q_s[g][lane] = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
      } else {
        q_s[g][lane] = hq[j].x;
      }
    }
  }
  // The new token's k is normalised by the first wave without a q head.
  constexpr int KW = G % NW;
  if (owns_new && wid == KW) {
    float o[4];
    norm_rope(hk, fq.w_f32, rt, fq.rot, lane, o);
    *reinterpret_cast<float4*>(&kn_s[4 * lane]) = make_float4(o[0], o[1], o[2], o[3]);
    *reinterpret_cast<float4*>(&vn_s[4 * lane]) =
        make_float4(bf_lo(vnew.x), bf_hi(vnew.x), bf_lo(vnew.y), bf_hi(vnew.y));
    if (n_old < cache_len) {
      const size_t off = ((size_t)kvh * cache_len + (size_t)n_old) * kAD + 4 * lane;
      *reinterpret_cast<uint2*>(fq.k_cache + off) = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
      *reinterpret_cast<uint2*>(fq.v_cache + off) = vnew;
    }
  }
  __syncthreads();

  // The lane's q slices as bf16 pairs: dims 8*ds.. and 128 + 8*ds...
  uint32_t qp[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint2 a = q_s[g][2 * ds], b = q_s[g][2 * ds + 1];
    const uint2 c = q_s[g][32 + 2 * ds], d = q_s[g][32 + 2 * ds + 1];
    qp[g][0] = a.x; qp[g][1] = a.y; qp[g][2] = b.x; qp[g][3] = b.y;
    qp[g][4] = c.x; qp[g][5] = c.y; qp[g][6] = d.x; qp[g][7] = d.y;
  }

  // 4. online softmax over the wave's tokens (m and l wave-uniform).
  float m[G], l[G], acc[G][4];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
    acc[g][0] = acc[g][1] = acc[g][2] = acc[g][3] = 0.f;
  }
  // One 32-token step of the workgroup from the registers KR / VR.
#define Q35_ATT_STEP(KR, VR, IT)                                                                \
  do {                                                                                          \
    const int tb = start + (IT) * kIterTok + wid * kWaveTok;                                    \
    float vf[kWaveTok][4];                                                                      \
    _Pragma("unroll") for (int i = 0; i < kWaveTok; ++i) {                                      \
      const bool in = tb + i < end;                                                             \
      vf[i][0] = in ? bf_lo(VR[i].x) : 0.f;                                                     \
      vf[i][1] = in ? bf_hi(VR[i].x) : 0.f;                                                     \
      vf[i][2] = in ? bf_lo(VR[i].y) : 0.f;                                                     \
      vf[i][3] = in ? bf_hi(VR[i].y) : 0.f;                                                     \
    }                                                                                           \
    _Pragma("unroll") for (int g = 0; g < G; ++g) {                                             \
      float s[kWaveGroups];                                                                     \
      _Pragma("unroll") for (int gi = 0; gi < kWaveGroups; ++gi) {                              \
        const uint4 k0 = KR[gi][0], k1 = KR[gi][1];                                             \
        float d = dot2_bf16(qp[g][0], k0.x, 0.f);                                               \
        d = dot2_bf16(qp[g][1], k0.y, d);                                                       \
        d = dot2_bf16(qp[g][2], k0.z, d);                                                       \
        d = dot2_bf16(qp[g][3], k0.w, d);                                                       \
        d = dot2_bf16(qp[g][4], k1.x, d);                                                       \
        d = dot2_bf16(qp[g][5], k1.y, d);                                                       \
        d = dot2_bf16(qp[g][6], k1.z, d);                                                       \
        d = dot2_bf16(qp[g][7], k1.w, d);                                                       \
        d = row16_sum(d) * scale;                                                               \
        s[gi] = tb + 4 * gi + rw < end ? d : -INFINITY;                                         \
      }                                                                                         \
      float smax = s[0];                                                                        \
      _Pragma("unroll") for (int gi = 1; gi < kWaveGroups; ++gi) smax = fmaxf(smax, s[gi]);     \
      const float m_new = fmaxf(m[g], rows4_max(smax));                                         \
      /* A wave whose tokens so far all lie past the valid end keeps m = -inf:              */  \
      /* subtract 0 then, so that corr and p are 0 instead of NaN.                          */  \
      const float m_sub = m_new == -INFINITY ? 0.f : m_new;                                     \
      const float corr = expf(m[g] - m_sub);                                                    \
      float pg[kWaveGroups];                                                                    \
      _Pragma("unroll") for (int gi = 0; gi < kWaveGroups; ++gi) pg[gi] = expf(s[gi] - m_sub);  \
      _Pragma("unroll") for (int e = 0; e < 4; ++e) acc[g][e] *= corr;                          \
      float psum = 0.f;                                                                         \
      _Pragma("unroll") for (int i = 0; i < kWaveTok; ++i) {                                    \
        const float pi = __int_as_float(                                                        \
            __builtin_amdgcn_readlane(__float_as_int(pg[i / 4]), 16 * (i & 3)));                \
        psum += pi;                                                                             \
        _Pragma("unroll") for (int e = 0; e < 4; ++e) acc[g][e] = fmaf(pi, vf[i][e], acc[g][e]); \
      }                                                                                         \
      l[g] = l[g] * corr + psum;                                                                \
      m[g] = m_new;                                                                             \
    }                                                                                           \
  } while (0)
  // Two register sets alternate over pairs of steps, the next step's rows
  // requested before the current one is reduced; nothing copies a set whose
  // loads are in flight, and a single step (the decode shape) issues no
  // prefetch at all.
  uint4 kb[kWaveGroups][2];
  uint2 vb[kWaveTok];
  int it = 0;
  for (; it + 1 < n_iter; it += 2) {
    load_kv(it + 1, kb, vb);
    Q35_ATT_STEP(kr, vr, it);
    if (it + 2 < n_iter) load_kv(it + 2, kr, vr);
    Q35_ATT_STEP(kb, vb, it + 1);
  }
  if (it < n_iter) Q35_ATT_STEP(kr, vr, it);
#undef Q35_ATT_STEP

  // The new token (FUSED): the owning workgroup folds it in, head g by wave
  // g % NW (into that wave's state), so the heads are folded in parallel.
  if (owns_new) {
    const float4 kv = *reinterpret_cast<const float4*>(&kn_s[4 * lane]);
    const float4 vv = *reinterpret_cast<const float4*>(&vn_s[4 * lane]);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g % NW != wid) continue;
      const uint2 qv = q_s[g][lane];
      float sdot = bf_lo(qv.x) * kv.x;
      sdot = fmaf(bf_hi(qv.x), kv.y, sdot);
      sdot = fmaf(bf_lo(qv.y), kv.z, sdot);
      sdot = fmaf(bf_hi(qv.y), kv.w, sdot);
      const float sc = wave_sum(sdot) * scale;
      const float m_new = fmaxf(m[g], sc);
      const float corr = expf(m[g] - m_new);
      const float p = expf(sc - m_new);
      l[g] = l[g] * corr + p;
      acc[g][0] = fmaf(p, vv.x, acc[g][0] * corr);
      acc[g][1] = fmaf(p, vv.y, acc[g][1] * corr);
      acc[g][2] = fmaf(p, vv.z, acc[g][2] * corr);
      acc[g][3] = fmaf(p, vv.w, acc[g][3] * corr);
      m[g] = m_new;
    }
  }

  // 5. merge the waves in LDS (one barrier: every thread derives the wave
  //    factors e^(m_w - max_w m_w), 0 for a wave without tokens, of its
  //    head itself); write this split's (acc, m, l) per head.
  __shared__ float m_s[NW][G], l_s[NW][G];
  __shared__ float a_s[NW][G][kAD];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    if (lane == 0) {
      m_s[wid][g] = m[g];
      l_s[wid][g] = l[g];
    }
    *reinterpret_cast<float4*>(&a_s[wid][g][4 * lane]) = make_float4(acc[g][0], acc[g][1], acc[g][2], acc[g][3]);
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < G * kAD / 4; idx += NW * 64) {
    const int g = idx / (kAD / 4), d = (idx % (kAD / 4)) * 4;
    float mm = -INFINITY;
#pragma unroll
    for (int v = 0; v < NW; ++v) mm = fmaxf(mm, m_s[v][g]);
    float f[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) f[w] = m_s[w][g] == -INFINITY ? 0.f : expf(m_s[w][g] - mm);
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float4 v = *reinterpret_cast<const float4*>(&a_s[w][g][d]);
      a.x += v.x * f[w];
      a.y += v.y * f[w];
      a.z += v.z * f[w];
      a.w += v.w * f[w];
    }
    const int slot = (kvh * G + g) * splits + split;
    *reinterpret_cast<float4*>(acc_out + (size_t)slot * kAD + d) = a;
    if (d == 0) {
      float ll = 0.f;
#pragma unroll
      for (int v = 0; v < NW; ++v) ll += l_s[v][g] * f[v];
      *reinterpret_cast<float2*>(ml_out + slot * 2) = make_float2(mm, ll);
    }
  }
}

// Log-sum-exp merge of the splits -> bf16, optionally times bf16(sigmoid(gate))
// [reference kernels.py:1007-1028 and 285-333]. Grid (query head, quarter of
// the 256 dims): thread (part = t/16, col = t%16) owns dims 64*quarter +
// 4*col .. +3 of splits part, part + 16, ... (up to 16*B splits). Every
// thread requests its partials (clamped indices) before wave 0 reads the
// (m, l) pairs and turns them into weights in LDS, so the merge is one
// memory round trip; the 16 parts are summed in LDS. Four workgroups per
// head keep each thread's share of a 128-split merge at 8 loads.
template <int B>
__global__ __launch_bounds__(256) void gqa_decode_combine(const float* __restrict__ acc,
                                                          const float* __restrict__ ml,
                                                          const uint16_t* __restrict__ packed_gate,
                                                          uint16_t* __restrict__ out, int splits,
                                                          long long* advance_len) {
  const int h = blockIdx.x >> 2, qd = blockIdx.x & 3;
  const int t = threadIdx.x;
  const int col = t & 15;
  const int part = t >> 4;
  const int d0 = 64 * qd + 4 * col;
  // The split kernel that read the length has completed (stream order).
  if (advance_len && blockIdx.x == 0 && t == 0) advance_len[0] += 1;
  const float* mlh = ml + (size_t)h * splits * 2;
  const float* acch = acc + (size_t)h * splits * kAD + d0;
  __shared__ float w_s[kMaxSplits];
  __shared__ float lt_s;
  __shared__ float4 red_s[16][16];
  const uint2 graw = packed_gate && part == 0
                         ? *reinterpret_cast<const uint2*>(packed_gate + h * 2 * kAD + kAD + d0)
                         : make_uint2(0, 0);
  float4 a[B];
#pragma unroll
  for (int j = 0; j < B; ++j)
    a[j] = *reinterpret_cast<const float4*>(acch + (size_t)min(part + 16 * j, splits - 1) * kAD);
  if (t < 64) {
    float mx = -INFINITY;
    for (int s = t; s < splits; s += 64) mx = fmaxf(mx, mlh[2 * s]);
    mx = wave_max(mx);
    float lt = 0.f;
    for (int s = t; s < splits; s += 64) {
      const float ms = mlh[2 * s];
      const float w = ms == -INFINITY ? 0.f : expf(ms - mx);
      w_s[s] = w;
      lt += mlh[2 * s + 1] * w;
    }
    lt = wave_sum(lt);
    if (t == 0) lt_s = lt;
  }
  __syncthreads();
  float4 tot = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int j = 0; j < B; ++j) {
    const int s = part + 16 * j;
    const float w = s < splits ? w_s[s] : 0.f;
    tot.x = fmaf(a[j].x, w, tot.x);
    tot.y = fmaf(a[j].y, w, tot.y);
    tot.z = fmaf(a[j].z, w, tot.z);
    tot.w = fmaf(a[j].w, w, tot.w);
  }
  red_s[part][col] = tot;
  __syncthreads();
  if (part == 0) {
    float4 r = red_s[0][col];
#pragma unroll
    for (int p = 1; p < 16; ++p) {
      const float4 v = red_s[p][col];
      r.x += v.x;
      r.y += v.y;
      r.z += v.z;
      r.w += v.w;
    }
    const float lt = lt_s;
    float o[4] = {round_bf(r.x / lt), round_bf(r.y / lt), round_bf(r.z / lt), round_bf(r.w / lt)};
    if (packed_gate) {
      o[0] *= round_bf(sigmoid_f(bf_lo(graw.x)));
      o[1] *= round_bf(sigmoid_f(bf_hi(graw.x)));
      o[2] *= round_bf(sigmoid_f(bf_lo(graw.y)));
      o[3] *= round_bf(sigmoid_f(bf_hi(graw.y)));
    }
    *reinterpret_cast<uint2*>(out + (size_t)h * kAD + d0) = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
  }
}

// Combine launch for a split count (partials per thread = ceil(splits / 16)).
void launch_combine(const float* acc, const float* ml, const uint16_t* gate, uint16_t* out, int QH,
                    int splits, long long* advance, hipStream_t stream) {
  const unsigned grid = (unsigned)(4 * QH);
  if (splits <= 32)
    gqa_decode_combine<2><<<grid, 256, 0, stream>>>(acc, ml, gate, out, splits, advance);
  else if (splits <= 64)
    gqa_decode_combine<4><<<grid, 256, 0, stream>>>(acc, ml, gate, out, splits, advance);
  else
    gqa_decode_combine<8><<<grid, 256, 0, stream>>>(acc, ml, gate, out, splits, advance);
}

}  // namespace

extern "C" {

int q35_qgkv_norm_rope(const void* packed, const void* q_w, const void* k_w, int w_f32,
                       const void* cos, const void* sin, void* q_out, void* k_out, void* v_out,
                       const void* cache_start, int B, int L, int QH, int KVH, int D,
                       int rotary_dim, int cache_len, hipStream_t stream) {
  Q35_CHECK_ARG(B >= 0 && L >= 0 && QH > 0 && KVH > 0 && KVH <= QH);
  Q35_CHECK_ARG(D == 64 || D == 128 || D == 256);
  const int E = D / 64;
  Q35_CHECK_ARG(rotary_dim >= 0 && rotary_dim <= D && rotary_dim % (2 * E) == 0);
  Q35_CHECK_ARG(!cache_start || cache_len > 0);
  const long long waves = (long long)B * L * QH;
  if (waves == 0) return 0;
  Q35_CHECK_ARG(waves < (1ll << 31));
  const unsigned grid = (unsigned)((waves + 3) / 4);
  const long long* cs = (const long long*)cache_start;
  if (D == kAD && rotary_dim > 0 && rotary_dim % 8 == 0 && q35_aligned8(packed) && q35_aligned8(q_w) &&
      q35_aligned8(k_w) && q35_aligned8(cos) && q35_aligned8(sin) && q35_aligned8(q_out) &&
      q35_aligned8(k_out) && q35_aligned8(v_out)) {
    qgkv_norm_rope_256<<<grid, 256, 0, stream>>>(
        (const uint16_t*)packed, q_w, k_w, w_f32, (const uint16_t*)cos, (const uint16_t*)sin,
        (uint16_t*)q_out, (uint16_t*)k_out, (uint16_t*)v_out, cs, B, L, QH, KVH, rotary_dim, cache_len);
    return q35_last_error();
  }
#define Q35_QGKV(EE)                                                                          \
  qgkv_norm_rope_k<EE><<<grid, 256, 0, stream>>>(                                             \
      (const uint16_t*)packed, q_w, k_w, w_f32, (const uint16_t*)cos, (const uint16_t*)sin,   \
      (uint16_t*)q_out, (uint16_t*)k_out, (uint16_t*)v_out, cs, B, L, QH, KVH, D, rotary_dim, \
      cache_len)
  if (E == 1) Q35_QGKV(1);
  else if (E == 2) Q35_QGKV(2);
  else Q35_QGKV(4);
#undef Q35_QGKV
  return q35_last_error();
}

// Split count and chunk length for a cache of cache_len tokens: chosen from
// the capacity only (never the valid length), so a captured graph stays valid.
// A chunk is a whole number of 32-token workgroup iterations and there are at
// most 128 splits per KV head (the combine requests them all at once).
int q35_gqa_decode_splits(int cache_len, int kv_heads, int* chunk_out) {
  if (cache_len <= 0 || kv_heads <= 0) return 0;
  long long chunk = ((long long)cache_len + kMaxSplits - 1) / kMaxSplits;
  chunk = (chunk + kIterTok - 1) / kIterTok * kIterTok;
  const int splits = (int)((cache_len + chunk - 1) / chunk);
  if (chunk_out) *chunk_out = (int)chunk;
  return splits;
}

// Workspace floats: acc[QH*splits*D] then ml[QH*splits*2].
long long q35_gqa_decode_workspace(int cache_len, int q_heads, int kv_heads, int D) {
  const int splits = q35_gqa_decode_splits(cache_len, kv_heads, nullptr);
  return (long long)q_heads * splits * (D + 2);
}

int q35_gqa_decode(const void* q, const void* K, const void* V, const void* valid_len, float scale,
                   const void* packed_gate, void* out, void* workspace, long long workspace_floats,
                   int QH, int KVH, int D, int cache_len, hipStream_t stream) {
  Q35_CHECK_ARG(D == kAD && KVH > 0 && QH % KVH == 0 && cache_len > 0);
  const int G = QH / KVH;
  Q35_CHECK_ARG(G == 1 || G == 2 || G == 4 || G == 8);
  int chunk = 0;
  const int splits = q35_gqa_decode_splits(cache_len, KVH, &chunk);
  Q35_CHECK_ARG(splits <= kMaxSplits);
  Q35_CHECK_ARG(workspace_floats >= q35_gqa_decode_workspace(cache_len, QH, KVH, D));
  Q35_CHECK_ARG(q35_aligned16(q) && q35_aligned16(K) && q35_aligned16(V) && q35_aligned16(workspace));
  Q35_CHECK_ARG(q35_aligned8(out) && q35_aligned8(packed_gate));
  float* acc = (float*)workspace;
  float* ml = acc + (size_t)QH * splits * D;
  dim3 grid(KVH, splits);
  const FusedQ none{};
#define Q35_GQA(GG)                                                                                    \
  gqa_decode_split<GG, false><<<grid, kSplitWaves * 64, 0, stream>>>((const uint16_t*)q, (const uint16_t*)K,       \
                                                        (const uint16_t*)V,                           \
                                                        (const long long*)valid_len, acc, ml,         \
                                                        cache_len, chunk, splits, scale, none)
  if (G == 1) Q35_GQA(1);
  else if (G == 2) Q35_GQA(2);
  else if (G == 4) Q35_GQA(4);
  else Q35_GQA(8);
#undef Q35_GQA
  int e = q35_last_error();
  if (e) return e;
  launch_combine(acc, ml, (const uint16_t*)packed_gate, (uint16_t*)out, QH, splits, nullptr, stream);
  return q35_last_error();
}

// One decode token of a full-attention layer after its packed projection:
// Q/K RMSNorm + RoPE (cos/sin from the device positions and inv_freq), K/V
// written into the static cache at index *cache_len_dev, split-K attention
// over the cache plus the new token, LSE combine, sigmoid gate, and
// *cache_len_dev += 1. Two launches; nothing is read on the host.
int q35_gqa_decode_fused(const void* packed, const void* q_w, const void* k_w, int w_f32,
                         const void* inv_freq, const void* pos_t, const void* pos_h,
                         const void* pos_w, int sec_h, int sec_w, int rotary_dim, void* K, void* V,
                         void* cache_len_dev, float scale, void* out, void* workspace,
                         long long workspace_floats, int QH, int KVH, int D, int cache_len,
                         hipStream_t stream) {
  Q35_CHECK_ARG(D == kAD && KVH > 0 && QH % KVH == 0 && cache_len > 0);
  Q35_CHECK_ARG(packed && q_w && k_w && inv_freq && pos_t && K && V && cache_len_dev && out);
  // The in-kernel rotary table holds rot/2 <= 64 frequencies, one per lane.
  Q35_CHECK_ARG(rotary_dim > 0 && rotary_dim <= 128 && rotary_dim % 8 == 0);
  Q35_CHECK_ARG(sec_h >= 0 && sec_w >= 0 && 3 * sec_h <= rotary_dim && 3 * sec_w <= rotary_dim);
  const int G = QH / KVH;
  Q35_CHECK_ARG(G == 1 || G == 2 || G == 4 || G == 8);
  int chunk = 0;
  const int splits = q35_gqa_decode_splits(cache_len, KVH, &chunk);
  Q35_CHECK_ARG(splits <= kMaxSplits);
  Q35_CHECK_ARG(workspace_floats >= q35_gqa_decode_workspace(cache_len, QH, KVH, D));
  Q35_CHECK_ARG(q35_aligned16(K) && q35_aligned16(V) && q35_aligned16(workspace));
  Q35_CHECK_ARG(q35_aligned4(inv_freq) && q35_aligned8(packed) && q35_aligned8(q_w) && q35_aligned8(k_w));
  Q35_CHECK_ARG(q35_aligned8(out));
  float* acc = (float*)workspace;
  float* ml = acc + (size_t)QH * splits * D;
  FusedQ f;
  f.packed = (const uint16_t*)packed;
  f.q_w = q_w;
  f.k_w = k_w;
  f.w_f32 = w_f32;
  f.inv_freq = (const float*)inv_freq;
  f.pos_t = (const long long*)pos_t;
  f.pos_h = (const long long*)(pos_h ? pos_h : pos_t);
  f.pos_w = (const long long*)(pos_w ? pos_w : pos_t);
  f.sec_h = sec_h;
  f.sec_w = sec_w;
  f.rot = rotary_dim;
  f.k_cache = (uint16_t*)K;
  f.v_cache = (uint16_t*)V;
  dim3 grid(KVH, splits);
#define Q35_GQA(GG)                                                                                 \
  gqa_decode_split<GG, true><<<grid, kSplitWaves * 64, 0, stream>>>(nullptr, (const uint16_t*)K,                \
                                                       (const uint16_t*)V,                         \
                                                       (const long long*)cache_len_dev, acc, ml,   \
                                                       cache_len, chunk, splits, scale, f)
  if (G == 1) Q35_GQA(1);
  else if (G == 2) Q35_GQA(2);
  else if (G == 4) Q35_GQA(4);
  else Q35_GQA(8);
#undef Q35_GQA
  int e = q35_last_error();
  if (e) return e;
  launch_combine(acc, ml, (const uint16_t*)packed, (uint16_t*)out, QH, splits,
                 (long long*)cache_len_dev, stream);
  return q35_last_error();
}

}  // extern "C"
