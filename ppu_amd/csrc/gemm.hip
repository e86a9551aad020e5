// Prefill GEMMs on the gfx950 matrix cores: C[M, N] = A[M, K] . B[N, K]^T
// with both operands K-contiguous (activations x weights^T, as F.linear).
//
//   kind 0  bf16 A, B -> bf16 C = bf16(acc)                        [F.linear, integration.py:183,245,298]
//   kind 1  bf16, B = [gate; up] (2N rows) -> C[m, n] = bf16(bf16(silu(bf16 g)) * bf16 u)
//                                                                   [integration.py:183-185 + kernels.py:158-180]
//   kind 2  int8 A, B -> int32 C = acc (exact)                     [the int8 GEMM of explore_runtime_quantization.py:173-180]
//   kind 3  int8 -> bf16 C = bf16(float(acc) * s_x[m] * s_w[n])    [the same with its dequant]
//   kind 4  int8, B = [gate; up] -> SwiGLU of the dequantised gate and up (kind 1's rounding points)
//   q35_gemm_bias  bf16 -> bf16(acc + bias[n]), or of its tanh GELU   [the vision tower's F.linear]
//
// bf16 runs on v_mfma_f32_32x32x16_bf16 (fp32 accumulators), int8 on
// v_mfma_i32_32x32x32_i8 (exact int32). Both take 16 bytes per lane and
// operand: lane l holds row l % 32 of its 32-row block and bytes
// [16 (l / 32), +16) of a 32-byte k window, so one LDS layout and one
// fragment read serve both.
//
// Workgroup: 4 waves as 2 x 2 over a TM x TN tile; each wave holds FM x FN
// accumulator blocks of 32 x 32 (tile 0: 256 x 192, the wave 128 x 96, 12
// blocks = 192 accumulator registers).
//
// Operand staging. K advances in stages of RB bytes per row. A stage of the
// A and B tiles goes straight from memory into LDS with
// global_load_lds_dwordx4 (each wave instruction writes 1 KiB of LDS: 1024 /
// RB rows, 16 bytes per lane) into a ring of NS stage buffers, so no register
// holds a fetched stage and NS - 1 stages are in flight. The loads are issued
// from inline asm, so the only waits on them are the ring's explicit vmcnt
// waits. Each lane's global source is chosen so that the LDS image is
// swizzled: 16-byte chunk c of tile row r sits at slot c ^ swz(r), which
// makes the fragment reads (16 consecutive rows, one logical chunk, per 16
// lanes) hit 16 distinct bank groups of the 256-byte LDS bank window.
// Measured on the 2B prefill shapes (timing copies with parts switched off):
//  * the operand stream is the bound; stages of 128-byte rows (every request
//    a whole L2 line) move twice the bytes per second of 64-byte rows, whose
//    requests each pull a 128-byte line for 64 useful bytes;
//  * workgroups that share operand rows (the M tiles of one weight tile, the
//    N tiles of one activation tile) run on one XCD; when they walk K in
//    lockstep every one of them waits for the same L2 misses, so each
//    workgroup starts its K walk at its own stage offset (K rotation) and the
//    later readers of a line find it in L2 (DMA-only time -15 to -30 %);
//  * a wave issues in order, so a run of fragment reads ahead of the MFMAs
//    stalls them behind the LDS queue; one read (and one DMA) per MFMA, in
//    the order the next k step consumes them, hides the reads completely.
//
// Ring schedule (one barrier per stage): in stage kt the fragments of k step
// t + 1 are read under the MFMAs of step t, and the buffer of stage kt - 1
// (free since the last barrier) is refilled with stage kt + NS - 1 under the
// MFMAs of the first steps; in the last step, after half of its MFMAs, each
// wave waits for its part of stage kt + 1 (vmcnt) and all waves meet at
// s_barrier, then the first fragments of stage kt + 1 are read under the
// second half.
//
// Split K (a caller's plan, or the default one for the dequant kind at K of
// 10240 and more): `splits` workgroups per tile each take kps stages. Each stores its partial tile (fp32 / int32 bit
// patterns, in accumulator-register order so every wave store is 512
// contiguous bytes) with agent-scope stores, every thread waits until its
// stores have completed (s_waitcnt vmcnt(0)), and one thread counts the
// workgroup's arrival on the tile's counter (agent-scope atomic add). The
// workgroup that arrives last resets the counter and sums the partials in
// split order, its own from registers, so the result does not depend on
// arrival order; it reads them with agent-scope loads issued only after it
// has seen the count. Agent-scope stores and loads (sc1) are coherent across
// the XCDs' L2s by themselves; completed stores before the count and loads
// after it give the ordering. (Agent-scope release / acquire fences would
// add an L2 write-back per arriving workgroup and an L2 invalidate per last
// one, which discards the operands the XCD's other workgroups are streaming:
// measured 2-3x slower on the split plans.) The counters (a fixed region of
// kMaxSplitTiles at the start of the workspace) and the partials live in the
// caller's workspace, which must be zero-filled once before its first use;
// every launch leaves the counters at zero again (a launch aborted part way
// can leave them non-zero: zero the workspace again after such an error).
// Two launches that overlap in time must not share a workspace.
//
// Tile order: units (tile, split) are grouped so that the units sharing B
// rows and a K range (consecutive M tiles) run on one XCD and read the
// weights into one L2: workgroup b (XCD b % 8) takes the b / 8-th of the XCD's
// eighth of the units. M runs fastest within bands of 8 M tiles, so the 32
// units that an XCD works on at a time are 8 M tiles x 4 N tiles and share both
// operands (with all M tiles fastest, each XCD of 2048x6144 at 8192 tokens
// streamed all 100 MB of activations for one N tile). Short of a whole round of
// CUs few M tiles are better off in one band (us, one band against bands of 8:
// 2048x6144 bf16 10 M tiles 64.8 / 65.6, 20 82.0 / 85.0, but 23 153.9 / 149.5, 32
// 166.9 / 160.1, and 16 with all 256 units 126.6 / 126.3).
#include "gemm_ksplit.hpp"

namespace {

constexpr int kMaxSplitTiles = 8192;  // counters at the start of a split-K workspace
constexpr int kCounterBytes = kMaxSplitTiles * 4;

// Workgroup barrier; the empty asm statements keep the compiler from moving
// memory accesses across it (the builtin barrier alone does not order them).
Q35_DEV void ring_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
Q35_DEV uint32_t acc_bits(float v) { return __float_as_uint(v); }
Q35_DEV uint32_t acc_bits(int v) { return (uint32_t)v; }
Q35_DEV float acc_from(uint32_t b, float) { return __uint_as_float(b); }
Q35_DEV int acc_from(uint32_t b, int) { return (int)b; }

constexpr int kBand = 8;

template <bool V> struct BoolTag { static constexpr bool value = V; };

template <int WM, int WN, int FM, int FN, int RB, int NSA, int NSB, bool ROT, int KIND, bool SPLIT, bool STAGED>
__global__ __launch_bounds__(256, 1) void gemm_ring(const GemmArgs a) {
  constexpr bool I8 = kind_i8(KIND);
  constexpr bool SWIGLU = kind_swiglu(KIND);
  constexpr int ES = I8 ? 1 : 2;
  constexpr int TM = WM * FM * 32, TN = WN * FN * 32;
  constexpr int NC = SWIGLU ? TN / 2 : TN;  // output columns per tile
  constexpr int RPG = 1024 / RB;             // tile rows per 1 KiB DMA group
  constexpr int CPR = RB / 16;               // 16-byte chunks per row and stage
  constexpr int GA = TM / RPG, GB = TN / RPG;
  constexpr int LA = GA / 4, LB = GB / 4;    // DMA instructions per wave and stage (A, B)
  constexpr int LPW = LA + LB;
  constexpr int ASTAGE = TM * RB, BSTAGE = TN * RB;  // LDS bytes per stage of A and of B
  constexpr int ABYTES = NSA * ASTAGE;       // the A ring, then the B ring
  constexpr int LDSB = ABYTES + NSB * BSTAGE;
  constexpr int T = RB / 32;                 // MFMA k steps per stage
  constexpr int NMF = FM * FN;               // MFMAs per k step
  constexpr int NR = FM + FN;                // fragment reads per k step
  constexpr int H = NMF / 2;                 // MFMAs of the last step before the barrier
  // MFMA slots that carry the DMA refills, spread evenly: four waves issuing
  // one 1 KiB copy per 32-cycle MFMA ask the texture unit for twice its 64
  // bytes per clock, and the MFMAs stall behind the copies (one copy per slot
  // from the first on: 8320x2048 bf16 at 1024 tokens 39.0 us, spread 35.8;
  // SwiGLU 12288x2048 at 4096 175 -> 168 us)
  constexpr int SLOTS = (T - 1) * NMF;
  static_assert(WM * WN == 4, "4 waves");
  static_assert(GA % 4 == 0 && GB % 4 == 0, "every wave issues the same DMA groups of A and B");
  static_assert(T % 2 == 0, "fragment register sets alternate between k steps");
  static_assert(!SWIGLU || WN == 2, "SwiGLU pairs the gate waves with the up waves");
  static_assert(NSA >= 2 && NSB >= NSA && LDSB <= 160 * 1024, "the stage rings fit the LDS");
  static_assert(LPW <= (T - 1) * NMF, "the refill fits the MFMA slots of the first steps");
  static_assert(STAGED || kind_direct(KIND), "direct stores: bf16 and int32 kinds");
  using AccT = typename GemmAcc<I8>::T;
  using EltT = typename GemmAcc<I8>::E;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LDSB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int wm = w % WM, wn = w / WM;

  // ---- unit of this workgroup: (tile, split)
  const int mt = (a.M + TM - 1) / TM;
  const int nt = (a.N + NC - 1) / NC;
  const int ntiles = mt * nt;
  const int S = SPLIT ? a.splits : 1;
  const int U = ntiles * S;
  const int xcd = (int)blockIdx.x & 7;
  int u = xcd * (U >> 3) + min(xcd, U & 7) + ((int)blockIdx.x >> 3);
  // bands of kBand M tiles (the last one smaller; up to 20 M tiles, with CUs to spare,
  // are one band): M tile fastest inside one
  const int kb = U <= 224 && mt <= 20 ? mt : kBand;
  const int band = u / (kb * nt * S);
  u -= band * (kb * nt * S);
  const int bm = min(kb, mt - band * kb);
  const int tm = band * kb + u % bm;
  const int rest = u / bm;
  const int ks = SPLIT ? rest % S : 0;
  const int tn = SPLIT ? rest / S : rest;
  const int tile = tn * mt + tm;
  const int m0 = tm * TM, n0 = tn * NC;
  const int nk = a.kps;  // stages of this workgroup
  // K rotation (ROT): the workgroups sharing rows start at different stages
  const int krot = ROT ? ((tm % 4) * nk / 4 + (tn & 7) * nk / 32) % nk : 0;
  const uint32_t rowb = (uint32_t)a.K * ES;
  // dequant kinds: the tile's row scales s_x[m0 ..] and column scales s_w[..]
  // (SwiGLU: gate then up columns), loaded now and published through LDS in
  // the epilogue (NSC <= 512: two per thread)
  constexpr bool DEQ = KIND == KIND_DEQ || KIND == KIND_DEQ_SWIGLU;
  constexpr int NSC = DEQ ? TM + (SWIGLU ? 2 * NC : NC) : 0;
  static_assert(NSC <= 512, "two scales per thread");
  float scl[2] = {0.f, 0.f};
  if constexpr (DEQ) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int x = tid + 256 * q;
      if (x < TM) {
        scl[q] = a.s_x[min(m0 + x, a.M - 1)];
      } else if (x < NSC) {
        const int y = x - TM;
        scl[q] = y < NC ? a.s_w[min(n0 + y, a.N - 1)] : a.s_w[a.N + min(n0 + y - NC, a.N - 1)];
      }
    }
  }

  // ---- DMA sources: wave w issues groups g = w + 4 i (A groups first)
  uint32_t voff[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int g = w + 4 * i;
    const bool isA = i < GA / 4;
    const int r = (isA ? g : g - GA) * RPG + lane / CPR;  // tile row
    const int c = (lane % CPR) ^ swz<RB>(r);
    int grow;
    if (isA) {
      grow = min(m0 + r, a.M - 1);
    } else if (SWIGLU) {
      grow = r < TN / 2 ? min(n0 + r, a.N - 1) : a.N + min(n0 + r - TN / 2, a.N - 1);
    } else {
      grow = min(n0 + r, a.N - 1);
    }
    voff[i] = (uint32_t)grow * rowb + (uint32_t)(ks * nk) * RB + 16u * c;
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_offset(lds) + (uint32_t)w * 1024u);
  // instruction i of the DMA of stage kt: A (i < LA) into A buffer abuf, B into B buffer bbuf
  auto dma = [&](int kt, int abuf, int bbuf, int i) {
    int ksr = kt + krot;
    if (ksr >= nk) ksr -= nk;
    if (i < LA)
      dma16(lds0 + (uint32_t)abuf * ASTAGE + 4096u * i, a.A + (size_t)ksr * RB, voff[i]);
    else
      dma16(lds0 + ABYTES + (uint32_t)bbuf * BSTAGE + 4096u * (i - LA), a.B + (size_t)ksr * RB, voff[i]);
  };

  // ---- fragment sources: row l32 of each 32-row block, logical chunk 2t + kh
  const int l32 = lane & 31, kh = lane >> 5;
  uint32_t fa[T], fb[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const uint32_t co = 16u * (uint32_t)((2 * t + kh) ^ swz<RB>(l32));
    fa[t] = (uint32_t)(wm * FM * 32 + l32) * RB + co;
    fb[t] = (uint32_t)(wn * FN * 32 + l32) * RB + co;
  }
  q35_u32x4 ra[2][FM], rb[2][FN];
  // fragment r of step t in the order the MFMAs consume them: A0, B0 .. B(FN-1), A1 ..
  auto read1 = [&](int abuf, int bbuf, int t, int set, int r) {
    const uint8_t* pa = lds + abuf * ASTAGE;
    const uint8_t* pb = lds + ABYTES + bbuf * BSTAGE;
    if (r == 0) {
      ra[set][0] = *reinterpret_cast<const q35_u32x4*>(pa + fa[t]);
    } else if (r <= FN) {
      rb[set][r - 1] = *reinterpret_cast<const q35_u32x4*>(pb + fb[t] + (r - 1) * 32 * RB);
    } else {
      ra[set][r - FN] = *reinterpret_cast<const q35_u32x4*>(pa + fa[t] + (r - FN) * 32 * RB);
    }
  };

  AccT acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;
  auto mfma = [&](int set, int q) {
    acc[q / FN][q % FN] = mfma32(ra[set][q / FN], rb[set][q % FN], acc[q / FN][q % FN]);
  };

  // ---- prologue: A stages 0 .. NSA-2 and B stages 0 .. NSB-2 in flight (A
  // before B of the same stage, as in the loop), stage 0 landed, its first
  // fragments read
#pragma unroll
  for (int s = 0; s < NSB - 1; ++s) {
    if (s < NSA - 1 && s < nk)
#pragma unroll
      for (int i = 0; i < LA; ++i) dma(s, s, 0, i);
    if (s < nk)
#pragma unroll
      for (int i = LA; i < LPW; ++i) dma(s, 0, s, i);
  }
  // issued after stage 0's B: (NSB - 2) later B stages and (NSA - 2) later A stages
  if (nk >= NSB - 1) wait_vm<(NSB - 2) * LB + (NSA - 2) * LA>();
  else wait_vm<0>();
  ring_barrier();
#pragma unroll
  for (int r = 0; r < NR; ++r) read1(0, 0, 0, 0, r);

  // One stage. RA / RB: the A / B buffer of stage kt - 1 is refilled with
  // stage kt + NSA - 1 / kt + NSB - 1 (A refills stop NSA - 1 stages before
  // the end, B refills NSB - 1).
  // Wait before the barrier, steady state: stage kt + 1's last load is its A
  // (issued at stage kt + 2 - NSA) when NSA < NSB, else its B; the loads
  // issued after it are then LB + (NSA - 2) (LA + LB), or (NSA - 2) (LA + LB).
  constexpr int WAITN = (NSA < NSB ? LB : 0) + (NSA - 2) * LPW;
  int abuf = 0, bbuf = 0;
  auto stage = [&](int kt, auto ra_tag, auto rb_tag) {
    constexpr bool RA = decltype(ra_tag)::value, RB_ = decltype(rb_tag)::value;
    const int rabuf = abuf == 0 ? NSA - 1 : abuf - 1;  // buffers of stage kt - 1
    const int rbbuf = bbuf == 0 ? NSB - 1 : bbuf - 1;
    // steps 0 .. T-2: one MFMA, one fragment read of the next step, and
    // (first steps) the DMA refills, per slot
#pragma unroll
    for (int t = 0; t < T - 1; ++t) {
#pragma unroll
      for (int q = 0; q < NMF; ++q) {
        mfma(t & 1, q);
        if constexpr (NR <= NMF) {
          if (q < NR) read1(abuf, bbuf, t + 1, (t + 1) & 1, q);
        } else {  // more fragments than MFMAs per step: spread them over the slots
#pragma unroll
          for (int r = q * NR / NMF; r < (q + 1) * NR / NMF; ++r) read1(abuf, bbuf, t + 1, (t + 1) & 1, r);
        }
        const int slot = t * NMF + q;
        const int i = (slot * LPW + SLOTS - 1) / SLOTS;  // the copy at slot i * SLOTS / LPW
        if (i < LPW && i * SLOTS / LPW == slot) {
          if (RA && i < LA) dma(kt + NSA - 1, rabuf, 0, i);
          if (RB_ && i >= LA) dma(kt + NSB - 1, 0, rbbuf, i);
        }
        Q35_PIN();
      }
    }
    // last step: half the MFMAs, the ring barrier, the other half with the
    // first fragments of stage kt + 1
    constexpr int cur = (T - 1) & 1;
#pragma unroll
    for (int q = 0; q < H; ++q) {
      mfma(cur, q);
      Q35_PIN();
    }
    const int nabuf = abuf + 1 == NSA ? 0 : abuf + 1;
    const int nbbuf = bbuf + 1 == NSB ? 0 : bbuf + 1;
    const bool more = kt + 1 < nk;
    wait_lds();  // on both paths, so the second half waits for nothing
    if (more) {
      // stage kt + 1 landed: this wave's part (vmcnt), then every wave's
      if (RA && RB_) wait_vm<WAITN>();
      else wait_vm<0>();
      ring_barrier();
    }
    Q35_PIN();
#pragma unroll
    for (int q = H; q < NMF; ++q) {
      mfma(cur, q);
      if (more) {
        const int s = q - H;
#pragma unroll
        for (int r = s * NR / (NMF - H); r < (s + 1) * NR / (NMF - H); ++r) read1(nabuf, nbbuf, 0, cur ^ 1, r);
      }
      Q35_PIN();
    }
    abuf = nabuf;
    bbuf = nbbuf;
  };
  int kt = 0;
  for (; kt + NSB - 1 < nk; ++kt) stage(kt, BoolTag<true>{}, BoolTag<true>{});
  for (; kt + NSA - 1 < nk; ++kt) stage(kt, BoolTag<true>{}, BoolTag<false>{});
  for (; kt < nk; ++kt) stage(kt, BoolTag<false>{}, BoolTag<false>{});

  // ---- split K: partial tiles, arrival count, the last workgroup sums
  if constexpr (SPLIT) {
    constexpr int NP = NMF * 8;  // 8-byte pairs per thread
    uint64_t* mine = reinterpret_cast<uint64_t*>(a.part) + ((size_t)ks * ntiles + tile) * NP * 256 + tid;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
          const uint64_t v = (uint64_t)acc_bits(acc[i][j][e]) | ((uint64_t)acc_bits(acc[i][j][e + 1]) << 32);
          __hip_atomic_store(mine + (size_t)(((i * FN + j) * 16 + e) / 2) * 256, v, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        }
    // Every thread waits for its own partial stores to complete (the
    // workgroup barrier does not wait for memory), then one arrival is counted.
    wait_vm<0>();
    // (the count is shared through the first word of the stage ring, which
    // no wave reads any more after this barrier)
    unsigned* arrived = reinterpret_cast<unsigned*>(lds);
    __syncthreads();
    if (tid == 0) {
      const unsigned n = __hip_atomic_fetch_add(a.cnt + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (n == (unsigned)S - 1)
        __hip_atomic_store(a.cnt + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *arrived = n;
    }
    __syncthreads();
    if (*arrived != (unsigned)S - 1) return;
    AccT own[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) own[i][j] = acc[i][j];
    for (int sp = 0; sp < S; ++sp) {
      const uint64_t* src = reinterpret_cast<const uint64_t*>(a.part) + ((size_t)sp * ntiles + tile) * NP * 256 + tid;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int e = 0; e < 16; e += 2) {
            EltT lo, hi;
            if (sp == ks) {
              lo = own[i][j][e];
              hi = own[i][j][e + 1];
            } else {
              const uint64_t v = __hip_atomic_load(
                  const_cast<uint64_t*>(src + (size_t)(((i * FN + j) * 16 + e) / 2) * 256),
                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              lo = acc_from((uint32_t)v, EltT{});
              hi = acc_from((uint32_t)(v >> 32), EltT{});
            }
            acc[i][j][e] = sp == 0 ? lo : acc[i][j][e] + lo;
            acc[i][j][e + 1] = sp == 0 ? hi : acc[i][j][e + 1] + hi;
          }
    }
  }

  // ---- epilogue. Element r of a 32x32 block sits at row 8 (r / 4) + 4 kh +
  // r % 4, column l32.
  if constexpr (!STAGED) {
    // Direct: each lane stores its elements (bf16: 64-byte row segments per
    // half wave; int32: 128-byte); tiles inside C store without checks.
    const int rbase = m0 + wm * FM * 32 + 4 * kh;
    const int cbase = n0 + wn * FN * 32 + l32;
    const bool full = m0 + TM <= a.M && n0 + TN <= a.N;
    float bias[FN];
    if constexpr (kind_bias(KIND)) {
#pragma unroll
      for (int j = 0; j < FN; ++j) bias[j] = bias_at(a, min(cbase + 32 * j, a.N - 1));
    }
    auto store = [&](int i, int r, int j, bool check) {
      const int row = rbase + 32 * i + 8 * (r >> 2) + (r & 3);
      const int col = cbase + 32 * j;
      if (check && (row >= a.M || col >= a.N)) return;
      const size_t at = (size_t)row * a.N + col;
      if constexpr (KIND == KIND_I32) {
        reinterpret_cast<int*>(a.C)[at] = acc[i][j][r];
      } else {
        float v = acc[i][j][r];
        if constexpr (kind_bias(KIND)) v += bias[j];
        if constexpr (KIND == KIND_BIAS_GELU) v = gelu_tanh_fast(v);
        reinterpret_cast<uint16_t*>(a.C)[at] = (uint16_t)f2bf(v);
      }
    };
    if (full) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
          for (int j = 0; j < FN; ++j) store(i, r, j, false);
    } else {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
          for (int j = 0; j < FN; ++j) store(i, r, j, true);
    }
    return;
  }
  // Staged through LDS. bf16 kinds and the int8 dequant kinds stage the
  // whole tile as bf16: the values they store, or the rounded gate / up; the
  // dequant kinds first publish the tile's scales in LDS and dequantise each
  // accumulator in registers, float(acc) * s_x * s_w rounded to bf16 (the
  // int32 tile would not fit the LDS in one pass, and staging it in two half
  // tiles left half the waves idle in each: the dequant epilogue of the
  // 256x192 tile took 11.2 us, now 5.9; with SwiGLU 11.6, now 8.5). The
  // int32 kind stages its accumulators one half tile (one wave row) at a
  // time. Rows are staged at a stride of TN elements + 16 bytes (the two
  // halves of each write instruction, rows r and r + 4, fall on different
  // banks). Then every thread takes ITER chunks of 16 staged bytes along the
  // rows, all read before any is converted, and stores each chunk's outputs
  // with one 16-byte store (a copy, or SwiGLU of the gate and up columns, the
  // two halves of a staged row).
  {
    constexpr bool W16 = !I8 || DEQ;           // staged as bf16
    constexpr int EB = W16 ? 2 : 4;            // staged bytes per element
    constexpr int PH = W16 ? 1 : WM;           // phases (half tiles for int8)
    constexpr int PR = TM / PH;                // staged rows per phase
    constexpr int SB = TN * EB + 16;           // staged row stride in bytes
    constexpr int VPC = 16 / EB;               // values per 16-byte chunk
    constexpr int CPRW = NC / VPC;             // output chunks per row
    constexpr int ITER = PR * CPRW / 256;      // chunks per thread and phase
    constexpr int SCO = PR * SB;               // LDS offset of the scales
    static_assert(PR * CPRW % 256 == 0, "the chunks divide over the workgroup");
    static_assert(!STAGED || SCO + NSC * 4 <= LDSB, "the staged tile and scales fit the rings");
    const bool vec = (a.N & 7) == 0;
    float* sc = reinterpret_cast<float*>(lds + SCO);
    wait_lds();
    __syncthreads();  // every wave is done with the stage ring
    if constexpr (DEQ) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
        if (tid + 256 * q < NSC) sc[tid + 256 * q] = scl[q];
      __syncthreads();  // the scales, before the dequant below reads them
    }
#pragma unroll
    for (int h = 0; h < PH; ++h) {
      if (PH == 1 || wm == h) {
        const int rb0 = PH == 1 ? wm * FM * 32 : 0;
        // dequant kinds: s_w of staged column c at sc[TM + c] (SwiGLU: the up
        // columns follow the gate columns), read once per column block; s_x
        // of the block row's 16 rows (4 runs of 4) as four 16-byte reads
        float swr[FN];
        if constexpr (DEQ) {
#pragma unroll
          for (int j = 0; j < FN; ++j) swr[j] = sc[TM + wn * FN * 32 + j * 32 + l32];
        } else if constexpr (kind_bias(KIND)) {
#pragma unroll
          for (int j = 0; j < FN; ++j) swr[j] = bias_at(a, min(n0 + wn * FN * 32 + j * 32 + l32, a.N - 1));
        }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          q35_f32x4 sxr[4];
          if constexpr (DEQ) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
              sxr[q] = *reinterpret_cast<const q35_f32x4*>(sc + rb0 + i * 32 + 8 * q + 4 * kh);
          }
#pragma unroll
          for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int off = (rb0 + i * 32 + 8 * (r >> 2) + 4 * kh + (r & 3)) * SB +
                              (wn * FN * 32 + j * 32 + l32) * EB;
              if constexpr (DEQ) {
                const float d = (float)acc[i][j][r] * sxr[r >> 2][r & 3] * swr[j];
                *reinterpret_cast<uint16_t*>(lds + off) = (uint16_t)f2bf(d);
              } else if constexpr (kind_bias(KIND)) {
                const float v = acc[i][j][r] + swr[j];
                *reinterpret_cast<uint16_t*>(lds + off) =
                    (uint16_t)f2bf(KIND == KIND_BIAS_GELU ? gelu_tanh_fast(v) : v);
              } else if constexpr (W16)
                *reinterpret_cast<uint16_t*>(lds + off) = (uint16_t)f2bf(acc[i][j][r]);
              else
                *reinterpret_cast<uint32_t*>(lds + off) = acc_bits(acc[i][j][r]);
            }
        }
      }
      __syncthreads();
      q35_u32x4 v[ITER], u[ITER];
#pragma unroll
      for (int it = 0; it < ITER; ++it) {
        const int c = tid + 256 * it;
        const uint8_t* src = lds + (c / CPRW) * SB + (c % CPRW) * 16;
        v[it] = *reinterpret_cast<const q35_u32x4*>(src);
        if constexpr (SWIGLU) u[it] = *reinterpret_cast<const q35_u32x4*>(src + TN / 2 * EB);
      }
#pragma unroll
      for (int it = 0; it < ITER; ++it) {
        const int c = tid + 256 * it;
        const int lrow = h * PR + c / CPRW, lcol = (c % CPRW) * VPC;
        const int grow = m0 + lrow;
        const int col = n0 + lcol;
        if (grow >= a.M || col >= a.N) continue;
        const int ncol = min(VPC, a.N - col);
        const size_t at = (size_t)grow * a.N + col;
        if constexpr (KIND == KIND_I32) {
          int* C = reinterpret_cast<int*>(a.C) + at;
          if (vec && ncol == VPC) *reinterpret_cast<q35_u32x4*>(C) = v[it];
          else for (int e = 0; e < ncol; ++e) C[e] = (int)v[it][e];
        } else if constexpr (!SWIGLU) {
          uint16_t* C = reinterpret_cast<uint16_t*>(a.C) + at;
          if (vec && ncol == VPC) *reinterpret_cast<q35_u32x4*>(C) = v[it];
          else for (int e = 0; e < ncol; ++e) C[e] = (uint16_t)(v[it][e >> 1] >> (16 * (e & 1)));
        } else {  // SwiGLU of the staged bf16 gate and up
          static_assert(VPC == 8, "SwiGLU kinds stage bf16");
          float o[VPC];
#pragma unroll
          for (int e = 0; e < VPC; ++e) {
            const uint32_t gw = v[it][e >> 1], uw = u[it][e >> 1];
            const float g = (e & 1) ? bf_hi(gw) : bf_lo(gw);
            const float uu = (e & 1) ? bf_hi(uw) : bf_lo(uw);
            o[e] = round_bf(silu_fast(g)) * uu;
          }
          uint16_t* C = reinterpret_cast<uint16_t*>(a.C) + at;
          if (vec && ncol == 8) *reinterpret_cast<uint4*>(C) = pack8(o);
          else for (int e = 0; e < ncol; ++e) C[e] = (uint16_t)f2bf(o[e]);
        }
      }
      if (h + 1 < PH) __syncthreads();
    }
  }
}

// ---------------------------------------------------------------- plans
// Tile shapes (waves 2 x 2; FM x FN blocks of 32 x 32 per wave; RB bytes per
// row and stage; NSA / NSB stages in the A / B rings; LDS = NSA TM RB + NSB
// TN RB; K rotation; epilogue staged through LDS, or direct stores for the
// bf16 / int32 kinds):
//   0: 256 x 192 (4 x 3), RB 128, NSA 2, NSB 4,       staged  (160 KiB)
//   1: 128 x 128 (2 x 2), RB 128, NSA 4, NSB 6, rot,  staged  (160 KiB)
//   2: 256 x 128 (4 x 2), RB 128, NSA 2, NSB 4,       staged  (128 KiB)
//   3: 128 x 192 (2 x 3), RB 128, NSA 4, NSB 4, rot,  staged  (160 KiB)
//   4: 256 x 192 (4 x 3), RB 128, NSA 2, NSB 2,       staged  (112 KiB)
//   5: tile 0 with direct stores; 6: tile 1 with direct stores; 7: tile 6
//   without K rotation
//   8: 128 x 64 (2 x 1), RB 128, NSA 6, NSB 8, rot, direct   (160 KiB)
//   9: 256 x 256 (4 x 4), RB 128, NSA 2, NSB 3, staged; 10: direct (160 KiB;
//   picked by the default plan only). 16 MFMAs for 8 fragment reads per k step
//   (12 for 7 in tile 0): the most work per LDS byte, for outputs that fill
//   their last round of CUs with it: 2048x6144 bf16 at 8192 tokens 222 -> 175
//   us (1180 TFLOP/s), 12288x2048 SwiGLU at 4096 204 -> 191 us, int8 2048x6144
//   at 8192 128 -> 99 us (2080 TOP/s)
#define Q35_GEMM_TILES(X)                     \
  X(0, 2, 2, 4, 3, 128, 2, 4, false, true)    \
  X(1, 2, 2, 2, 2, 128, 4, 6, true, true)     \
  X(2, 2, 2, 4, 2, 128, 2, 4, false, true)    \
  X(3, 2, 2, 2, 3, 128, 4, 4, true, true)     \
  X(4, 2, 2, 4, 3, 128, 2, 2, false, true)    \
  X(5, 2, 2, 4, 3, 128, 2, 4, false, false)   \
  X(6, 2, 2, 2, 2, 128, 4, 6, true, false)    \
  X(7, 2, 2, 2, 2, 128, 4, 6, false, false)   \
  X(8, 2, 2, 2, 1, 128, 6, 8, true, false)    \
  X(9, 2, 2, 4, 4, 128, 2, 3, false, true)    \
  X(10, 2, 2, 4, 4, 128, 2, 3, false, false)
constexpr int kTiles = 11;
constexpr int kPlanTiles = 9;  // tiles a caller's plan may name
constexpr int kRB = 128;
constexpr int kTM[kTiles] = {256, 128, 256, 128, 256, 256, 128, 128, 128, 256, 256};
constexpr int kTN[kTiles] = {192, 128, 128, 192, 192, 192, 128, 128, 64, 256, 256};
constexpr bool kStaged[kTiles] = {true, true, true, true, true, false, false, false, false, true, false};
constexpr bool kSplitOk[kTiles] = {false, true, true, true, false, false, true, true, true, false, false};  // up to 8 blocks per wave
constexpr int kMaxSplits = 8;

// Tiles of the K-splitting kernel, by operand rows (32 FN weight rows, 16 for
// a half tile, + 32 FM tokens): FN, FM, waves, ring pieces per wave, half tile;
// built for the SwiGLU kinds, for the others. Rings and waves from a sweep over
// the model's shapes at 17 to 1024 tokens.
#define Q35_GEMM_KS_TILES(X)                \
  X(0, 1, 1, 4, 3, true, false, true)       \
  X(1, 1, 1, 8, 2, false, false, true)      \
  X(2, 2, 1, 4, 3, false, true, true)       \
  X(3, 1, 2, 4, 3, false, false, true)      \
  X(4, 2, 2, 4, 2, false, true, true)       \
  X(5, 1, 3, 4, 2, false, false, true)      \
  X(6, 2, 3, 4, 1, false, true, true)       \
  X(7, 3, 2, 4, 1, false, false, true)      \
  X(8, 4, 2, 4, 1, false, false, true)      \
  X(9, 2, 4, 4, 1, false, true, true)       \
  X(10, 4, 3, 4, 1, false, true, false)     \
  X(11, 4, 4, 4, 1, false, true, false)
constexpr int kKsTiles = 12;
#define Q35_GEMM_KS_W(id, fn, fm, w, s, half, sg, pl) (half) ? 16 : 32 * fn,
#define Q35_GEMM_KS_T(id, fn, fm, w, s, half, sg, pl) 32 * fm,
#define Q35_GEMM_KS_SG(id, fn, fm, w, s, half, sg, pl) sg,
#define Q35_GEMM_KS_PL(id, fn, fm, w, s, half, sg, pl) pl,
constexpr int kKsWeights[kKsTiles] = {Q35_GEMM_KS_TILES(Q35_GEMM_KS_W)};
constexpr int kKsTokens[kKsTiles] = {Q35_GEMM_KS_TILES(Q35_GEMM_KS_T)};
constexpr bool kKsSwiglu[kKsTiles] = {Q35_GEMM_KS_TILES(Q35_GEMM_KS_SG)};
constexpr bool kKsPlain[kKsTiles] = {Q35_GEMM_KS_TILES(Q35_GEMM_KS_PL)};
#undef Q35_GEMM_KS_W
#undef Q35_GEMM_KS_T
#undef Q35_GEMM_KS_SG
#undef Q35_GEMM_KS_PL

long long tiles_of(int tile, int M, int N, int kind) {
  const int nc = kind_swiglu(kind) ? kTN[tile] / 2 : kTN[tile];
  return (long long)((M + kTM[tile] - 1) / kTM[tile]) * ((N + nc - 1) / nc);
}

long long workspace_bytes(int tile, int M, int N, int kind, int splits) {
  if (splits <= 1) return 0;
  return kCounterBytes + tiles_of(tile, M, N, kind) * splits * kTM[tile] * kTN[tile] * 4ll;
}

// Time of one workgroup of a ring tile with all CUs busy: kFixed + kStage per
// stage of 128 bytes, in us (fits of outputs 2048 to 12288 wide with K = 2048
// and 6144 bf16 or int8; by tile, 1 and 6, 0 and 5, 9 and 10 alike). kDequant:
// what the dequant epilogue adds (9 also with SwiGLU, about half; there it holds
// all 512 registers and 8-16 bytes per lane in scratch memory).
constexpr double kFixed[kTiles] = {11.6, 5.7, 7, 7.7, 11.6, 11.6, 5.7, 5.7, 4.8, 5.1, 5.1};
constexpr double kStage[kTiles] = {1.06, 0.51, 0.92, 0.667, 1.06, 1.06, 0.51, 0.51, 0.353, 1.7, 1.7};
constexpr double kDequant[kTiles] = {0, 1.3, 2, 0.5, 0, 0, 0, 0, 0, 10, 0};

// Estimated time of an output on a ring tile: whole rounds of 256 workgroups,
// and a last one that costs 0.7 of a round even if few CUs take part (0.45
// where earlier rounds have spread the workgroups' ends).
double ring_us(int tile, int M, int N, int nk, int kind) {
  const double r = (double)tiles_of(tile, M, N, kind) / 256;
  const double one = kFixed[tile] + kStage[tile] * nk +
                     kDequant[tile] * (kind == KIND_DEQ ? 1 : kind == KIND_DEQ_SWIGLU && tile == 9 ? 0.45 : 0);
  if (r <= 1) return one * (0.7 + 0.3 * r);
  const double whole = (double)(long long)r, rest = r - whole;
  return one * (whole + (rest > 0 ? (whole < 3 ? 0.7 + 0.3 * rest : 0.45 + 0.5 * rest) : 0));
}

// Operand rows (weights + tokens) up to which an output takes the K-splitting
// kernel; the figures stand at plan().
constexpr int ks_rows(int kind, int N) {
  return kind == KIND_SWIGLU ? 256 : kind == KIND_DEQ_SWIGLU ? 224 : kind == KIND_DEQ && N <= 4096 ? 192
         : kind == KIND_I32 && N > 4096 ? 128 : 160;
}

// Default plan. Large outputs: the ring tile with the least estimated time,
// direct stores for the bf16 / int32 kinds (tiles 2 and 3 are built staged only)
// and the staged epilogue for SwiGLU and dequant. What it decides is the last
// round of CUs: the down projection (2048x6144) at 4096 tokens has 176 tiles of
// 256x192 (116 us) but 256 of 256x128 (95 us), at 2003 tokens 66 us on 256x192 and
// 54 us on 128x128. The estimates hold from K = 2048 bytes up or so; over 238
// random shapes of 1 to 15 stages nine took 6-9 % longer than on the tile that
// the tile counts alone suggest. 128x128 tiles on at most half the CUs split K
// only when each split keeps at least 40 stages (the partial-tile exchange costs
// more than the idle CUs below that); that leaves the dequant kind, where no
// 128x64 tile takes such outputs.
//
// Outputs of few tokens or few columns run on the K-splitting kernel instead
// (tile kTiles + its index): the smallest of its tiles that covers the output
// with one workgroup per CU, as long as the tile's operand rows stay few
// enough. Measured at the edges (us, this kernel against the ring plans, cold
// weights): 2048x2048 bf16 M = 33 5.4 / 13.5, 340 9.9 / 13.8, 600 12.1 / 13.0,
// 1024 (192 rows) 14.8 / 13.8; 2048x6144 bf16 M = 33 10.1 / 31.4, 340 23.5 /
// 33.9, 600 30.2 / 35.0; int8 with the dequant M = 33 6.7 / 25.0, 340 13.4 /
// 25.0, 1024 (192 rows) 22.2 / 24.9, to int32 at 512 15.1 / 19.0, at 1024 20.2 /
// 20.1; 5120x2048 M = 256 13.8 / 15.9, 340 (192 rows) 16.0 / 15.4, to int32 (160
// rows) 14.6 / 14.2; 8320x2048 M = 96 16.4 / 17.1, 128 (192 rows) 18.6 / 17.5;
// 12288x2048 SwiGLU bf16 M = 64 14.9 / 25.5, 128 19.6 / 29.1, 230 (256 rows) 25.5 /
// 26.9, int8 180 (224 rows) 15.9 / 16.7, 230 (256 rows) 18.4 / 16.9. The row
// limits lie between the sides that these figures show.
void plan(int M, int N, int K, int kind, int* tile, int* splits) {
  const int es = kind_i8(kind) ? 1 : 2;
  const bool direct = kind_direct(kind);
  *splits = 1;
  const int rows = ks_rows(kind, N);
  for (int c = 0; c < kKsTiles; ++c) {
    if (kKsWeights[c] + kKsTokens[c] > rows) break;
    if (kind_swiglu(kind) ? !kKsSwiglu[c] : !kKsPlain[c]) continue;
    const int nc = kind_swiglu(kind) ? kKsWeights[c] / 2 : kKsWeights[c];
    if ((long long)((M + kKsTokens[c] - 1) / kKsTokens[c]) * ((N + nc - 1) / nc) <= 256) {
      *tile = kTiles + c;
      return;
    }
  }
  const int nk = (int)((long long)K * es / kRB);
  double best = 0;
  *tile = -1;
  for (int t = 0; t < kTiles; ++t) {
    // 4 and 7 are tiles 0 and 6 with another ring or walk: never faster
    if (t == 4 || t == 7 || (direct ? t == 0 || t == 1 || t == 9 : !kStaged[t])) continue;
    if (kind_swiglu(kind) && (t == 1 || t == 2)) continue;  // few columns per tile: the epilogue outweighs
    // 256x256 from 16 stages: the fit above does not hold for its prologue and
    // epilogue alone (us, against the next best tile: 441x9456 bf16 K = 128
    // 18.9 / 11.1, 1356x6784 K = 640 32.0 / 27.4, 554x15536 K = 768 35.1 / 31.9;
    // from 16 stages on never behind: 1141x12832 K = 1024 41.3 / 47.3)
    if (t >= 9 && nk < 16) continue;
    const double us = ring_us(t, M, N, nk, kind);
    if (*tile < 0 || us < best) {
      best = us;
      *tile = t;
    }
  }
  if ((*tile == 1 || *tile == 6) && !kind_bias(kind)) {
    const long long t = tiles_of(1, M, N, kind);
    while (*splits < kMaxSplits && t * *splits * 2 <= 256 && nk % (*splits * 2) == 0 &&
           nk / (*splits * 2) >= 40 && t <= kMaxSplitTiles)
      *splits *= 2;
  }
}

template <int WM, int WN, int FM, int FN, int RB, int NSA, int NSB, bool ROT, int KIND, bool STAGED>
int launch_one(const GemmArgs& a, hipStream_t stream) {
  constexpr int TM = WM * FM * 32, TN = WN * FN * 32;
  constexpr int NC = kind_swiglu(KIND) ? TN / 2 : TN;
  const long long units = (long long)((a.M + TM - 1) / TM) * ((a.N + NC - 1) / NC) * a.splits;
  Q35_CHECK_ARG(units < (1ll << 31));
  if (a.splits > 1) {
    if constexpr (kind_swiglu(KIND) || kind_bias(KIND) || FM * FN > 8) {
      return (int)hipErrorInvalidValue;  // split K: tiles of up to 8 blocks per wave, no SwiGLU
    } else {
      gemm_ring<WM, WN, FM, FN, RB, NSA, NSB, ROT, KIND, true, STAGED><<<(unsigned)units, 256, 0, stream>>>(a);
    }
  } else {
    gemm_ring<WM, WN, FM, FN, RB, NSA, NSB, ROT, KIND, false, STAGED><<<(unsigned)units, 256, 0, stream>>>(a);
  }
  return q35_last_error();
}

// Tiles that a kind can run on (the others are not built): what the default
// plan takes, and for the kinds of q35_gemm the ring tiles 0-8 of a caller's plan.
constexpr bool has_tile(int kind, int tile) {
  if (tile >= kTiles) {
    const int c = tile - kTiles;
    return (kind_swiglu(kind) ? kKsSwiglu[c] : kKsPlain[c]) && kKsWeights[c] + kKsTokens[c] <= ks_rows(kind, 1);
  }
  if (kind_bias(kind)) return tile != 0 && tile != 1 && tile != 4 && tile != 7 && tile != 9;
  return kind_direct(kind) ? tile != 9 : kStaged[tile];
}

template <int KIND>
int launch_tile(int tile, const GemmArgs& a, hipStream_t stream) {
  switch (tile) {
#define Q35_GEMM_KS_CASE(id, fn, fm, w, s, half, sg, pl) \
  case kTiles + id: \
    if constexpr (has_tile(KIND, kTiles + id)) return launch_ksplit<fn, fm, w, s, half, KIND>(a, stream); \
    break;
    Q35_GEMM_KS_TILES(Q35_GEMM_KS_CASE)
#undef Q35_GEMM_KS_CASE
#define Q35_GEMM_CASE(id, wm, wn, fm, fn, rb, nsa, nsb, rot, staged) \
  case id: \
    if constexpr (has_tile(KIND, id)) return launch_one<wm, wn, fm, fn, rb, nsa, nsb, rot, KIND, staged>(a, stream); \
    break;
    Q35_GEMM_TILES(Q35_GEMM_CASE)
#undef Q35_GEMM_CASE
    default: break;
  }
  return (int)hipErrorInvalidValue;
}

int gemm_run(const void* A, const void* B, void* C, int M, int N, int K, int kind, const float* s_x,
             const float* s_w, int tile, int splits, void* ws, long long ws_bytes, hipStream_t stream) {
  const int es = kind_i8(kind) ? 1 : 2;
  Q35_CHECK_ARG(A && B && C && M > 0 && N > 0 && K > 0 && tile < kPlanTiles);
  if (tile < 0) plan(M, N, K, kind, &tile, &splits);
  const bool ks = tile >= kTiles;
  Q35_CHECK_ARG(splits >= 1 && splits <= kMaxSplits);
  Q35_CHECK_ARG(ks || kStaged[tile] || kind_direct(kind));
  Q35_CHECK_ARG(q35_aligned16(A) && q35_aligned16(B) && ((long long)K * es) % kRB == 0);
  Q35_CHECK_ARG((kind != KIND_DEQ && kind != KIND_DEQ_SWIGLU) || (s_x && s_w));
  // 32-bit byte offsets of every operand row
  Q35_CHECK_ARG((long long)M * K * es < (1ll << 32) && (kind_swiglu(kind) ? 2ll : 1ll) * N * K * es < (1ll << 32));
  const int nk = (int)((long long)K * es / kRB);
  Q35_CHECK_ARG(nk % splits == 0);
  if (splits > 1) {
    Q35_CHECK_ARG(kSplitOk[tile] && !kind_swiglu(kind) && tiles_of(tile, M, N, kind) <= kMaxSplitTiles);
    Q35_CHECK_ARG(ws && q35_aligned16(ws) && ws_bytes >= workspace_bytes(tile, M, N, kind, splits));
  }
  GemmArgs a{(const uint8_t*)A, (const uint8_t*)B, C, M, N, K, s_x, s_w, nullptr, nullptr, splits, nk / splits};
  if (splits > 1) {
    a.cnt = (unsigned*)ws;
    a.part = (uint8_t*)ws + kCounterBytes;
  }
  switch (kind) {
    case KIND_BF16: return launch_tile<KIND_BF16>(tile, a, stream);
    case KIND_SWIGLU: return launch_tile<KIND_SWIGLU>(tile, a, stream);
    case KIND_I32: return launch_tile<KIND_I32>(tile, a, stream);
    case KIND_DEQ: return launch_tile<KIND_DEQ>(tile, a, stream);
    case KIND_BIAS: return launch_tile<KIND_BIAS>(tile, a, stream);
    case KIND_BIAS_GELU: return launch_tile<KIND_BIAS_GELU>(tile, a, stream);
    default: return launch_tile<KIND_DEQ_SWIGLU>(tile, a, stream);
  }
}

}  // namespace

extern "C" {

// Workspace bytes of q35_gemm for (M, N, K, kind) and a plan (tile < 0: the
// default plan); 0 when the plan does not split K, -1 for an invalid plan.
long long q35_gemm_workspace(int M, int N, int K, int kind, int tile, int splits) {
  if (M <= 0 || N <= 0 || K <= 0 || kind < 0 || kind >= kNumKinds) return -1;
  if (tile >= kPlanTiles) return -1;
  if (tile < 0) plan(M, N, K, kind, &tile, &splits);
  if (tile >= kTiles) return 0;
  if (splits < 1 || splits > kMaxSplits) return -1;
  if (!kStaged[tile] && kind != KIND_BF16 && kind != KIND_I32) return -1;
  if (splits > 1 && (!kSplitOk[tile] || kind_swiglu(kind) || tiles_of(tile, M, N, kind) > kMaxSplitTiles))
    return -1;
  return workspace_bytes(tile, M, N, kind, splits);
}

// Tile of the default plan (host only): 0-10 the ring kernel's, from 11 on the
// K-splitting kernel's, for the kinds of q35_gemm and 5 / 6 = q35_gemm_bias
// without / with gelu; -1 for sizes that the entries refuse.
int q35_gemm_plan(int M, int N, int K, int kind) {
  if (M <= 0 || N <= 0 || K <= 0 || kind < 0 || kind > KIND_BIAS_GELU) return -1;
  if (((long long)K * (kind_i8(kind) ? 1 : 2)) % kRB) return -1;
  int tile = -1, splits = 1;
  plan(M, N, K, kind, &tile, &splits);
  return tile;
}

// Prefill GEMM C = A . B^T of the given kind (0 bf16, 1 bf16 SwiGLU, 2 int8 ->
// int32, 3 int8 -> bf16 dequant, 4 int8 SwiGLU; see gemm.hip's header).
// K * element bytes a multiple of 128 (the stage width); A and B 16-byte
// aligned; every operand below 2^32 bytes. tile < 0 picks the default plan,
// otherwise tile 0-8 with `splits` K splits (the stage count divisible by
// splits). A split plan needs a workspace of q35_gemm_workspace bytes,
// zero-filled before its first use.
int q35_gemm(const void* A, const void* B, void* C, int M, int N, int K, int kind, const void* s_x,
             const void* s_w, int tile, int splits, void* workspace, long long workspace_bytes,
             hipStream_t stream) {
  Q35_CHECK_ARG(kind >= 0 && kind < kNumKinds);
  return gemm_run(A, B, C, M, N, K, kind, (const float*)s_x, (const float*)s_w, tile, splits,
                  workspace, workspace_bytes, stream);
}

// C[M, N] = bf16(A . B^T + bias), or with gelu bf16(GELU_tanh(A . B^T + bias)),
// bias [N] bf16, the sum and the GELU on the fp32 accumulators. K % 64 == 0; A
// and B 16-byte aligned; the default plan, no workspace.
int q35_gemm_bias(const void* A, const void* B, const void* bias, void* C, int M, int N, int K, int gelu,
                  hipStream_t stream) {
  Q35_CHECK_ARG(bias != nullptr);
  return gemm_run(A, B, C, M, N, K, gelu ? KIND_BIAS_GELU : KIND_BIAS, nullptr, (const float*)bias, -1, 1, nullptr,
                  0, stream);
}

}  // extern "C"
