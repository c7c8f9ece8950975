// Expert-grouped GEMM for calls with many routes per expert (long prefill).
//
// Covers the same projections as uqm_mfma.hip (the reference's prefill kernels,
// src/uma_qmoe/native/packed_q4_kernel.cu:560-776 for Q4, :781-1099 for Q8, and
// its BF16 grouped_mm path, src/uma_qmoe/native_backend.py:958-1005).
//
// What bounds uqm_mfma.hip there is its MMA waves' instruction stream: a route
// tile of 32 means that every 32 routes dequantise the expert's rows again, and
// an offset-binary weight needs the activation sums (one more MFMA per two).
// Here one workgroup of 4 waves takes 128 weight rows (gate/up: 64 of each) and
// up to 144 routes, each wave 32 rows and all the routes:
//   * weights go straight from global memory to the wave that uses them (no
//     row is shared between waves), one 128-element group ahead, and become
//     signed bf16 integers in registers: v_cvt_off_f32_i4 (q / 16) and
//     v_cvt_f32_i32 with a sign-extended byte are exact in bf16, so the MFMA
//     sums x * q directly and needs no activation sums; per 128-element group
//     acc += scale * sum in FP32. That is 104 conversions per group and 8 FMAs
//     per 16-route tile against 8 MFMAs per tile: at 9 tiles 2.4 VALU
//     instructions per MFMA, spread evenly between them (the next group is
//     converted while this one's MFMAs run, each tile's B operands are read
//     during the tile before, its sums folded during the one after);
//   * activations come through LDS (global_load_lds, 16 bytes per lane, one
//     128-element group of all routes per stage) in a ring of 2 to 6 stages,
//     and the group's scales with them, so that a lane reads the scales of its
//     4 rows as one vector;
//   * an expert's routes are split evenly (route_tile_step), and the loop is
//     compiled for every tile size from 1 to 9 sixteens, so that padding stays
//     below 16 routes per tile;
//   * one work item per workgroup and two workgroups per CU (at most 78 KB of
//     ring and 256 VGPRs): the hardware dispatcher balances items of different
//     sizes, and one workgroup's start and end run under the other's MFMAs.
// What bounds it (OLMoE shapes, 4095 tokens): without its loads the loop runs
// at ~1.5 PFLOP/s, the rate of a large library product on this card; the
// activation loads into LDS cost 17% of the call, the output writes (268 MB of
// FP32 rows for the down projection) 14%. BF16 is bound by its weights' 64-byte
// row segments: 3.8 TB/s.
// Measured (kernel trace, us, against uqm_mfma.hip's 32 routes): OLMoE shapes,
// 4095 tokens (512 routes per expert), Q4: gate/up 324 vs 859, down 214 vs 458;
// Qwen shapes, Q4 2048 tokens 155 + 93 (233 + 141 beside the shared expert),
// BF16 1535 tokens 183 + 96 (344 + 169).
// Loads that are not taken by four neighbouring lanes from one 64-byte segment
// cost 64 cache accesses instead of 16, and weight loads ahead of a stage's
// made the wait for that stage wait for HBM; with both as they are now the
// routed experts alone take (us per call, same box) BF16 1535 tokens 280 vs
// 301, Q8 999 185 vs 196 and 600 163 vs 183, Q4 1000 153 vs 159.
//
// MFMA operand layout (v_mfma_f32_16x16x32_bf16): A lane l holds row l%16 and
// K-slice 8*(l/16)..+7; B lane l holds token l%16, same K-slice; D lane l
// holds token l%16, rows 4*(l/16)+i. The K elements of a step follow the order
// of a lane's 16-byte weight loads, the same for A and B.
#include "uqm_prefill.h"

#include "uqm_stage.h"

#include <type_traits>

namespace uqm {
namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kRowBytes = 256;                  // one staged activation row: 128 bf16
constexpr int kTileBytes = 16 * kRowBytes;      // 16 routes of one stage
constexpr int kMaxTT = kPrefillTileTokens / 16;  // 16-route tiles per item
constexpr int kRingTiles = 18;                  // 72 KB of activations
constexpr int kMaxStages = 6;

// Stages of the ring for items of TT tiles: small items run through a stage
// in well under a microsecond and need more of them in flight.
constexpr int stages_for(int enc, int tt) {
  const int most = enc == kQ4 ? kMaxStages : 4;
  return kRingTiles / tt < most ? kRingTiles / tt : most;
}
// Weight groups in registers (in flight, or being converted), as many as the
// tile leaves registers for.
constexpr int raw_sets_for(int enc, int tt) { return enc == kQ4 && tt <= 6 ? 4 : 2; }

// LDS of one workgroup: ring of stages (activations, then the scales: 64
// floats per wave and stage), route ids, activation rows.
constexpr int kScaleBytes = 1024;  // per stage
constexpr int ring_bytes(int enc, int tt) { return stages_for(enc, tt) * (tt * kTileBytes + kScaleBytes); }
constexpr int max_ring_bytes(int tt) {
  return tt == 0 ? 0 : (ring_bytes(kQ4, tt) > max_ring_bytes(tt - 1) ? ring_bytes(kQ4, tt) : max_ring_bytes(tt - 1));
}
constexpr int kRouteOff = max_ring_bytes(kMaxTT);
constexpr int kSourceOff = kRouteOff + kPrefillTileTokens * 4;
constexpr int kLdsBytes = kSourceOff + kPrefillTileTokens * 4;
static_assert(2 * kLdsBytes <= 160 * 1024, "two workgroups per CU");

template <int ENC>
struct PEnc;
template <>
struct PEnc<kQ4> {
  static constexpr int kLoads = 1;         // 16-byte loads per lane, 16-row tile and 128-element group
  static constexpr int kGroupBytes = 64;   // bytes of one row's group
};
template <>
struct PEnc<kQ8> {
  static constexpr int kLoads = 2;
  static constexpr int kGroupBytes = 128;
};
template <>
struct PEnc<kBF16> {
  static constexpr int kLoads = 4;
  static constexpr int kGroupBytes = 256;
};

__device__ __forceinline__ uint32_t dword_of(const uint4& v, int i) {
  return i == 0 ? v.x : (i == 1 ? v.y : (i == 2 ? v.z : v.w));
}

// bf16 pair of two floats that are exact in bf16.
__device__ __forceinline__ uint32_t exact_pair(float lo, float hi) {
  return perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// Dword i (a bf16 pair) of the A operand (8 weights) of K-step S of a group
// from the lane's 16-byte loads:
//   Q4: dword S = elements 32q+8S .. +7, as q / 16
//   Q8: load S/2, dwords 2(S%2), 2(S%2)+1 = elements 64(S/2)+16q+8(S%2) .. +7
//   BF16: load S = elements 32S+8q .. +7
template <int ENC>
__device__ __forceinline__ uint32_t weight_pair(const uint4 (&v)[PEnc<ENC>::kLoads], int S, int i) {
  if constexpr (ENC == kQ4) {
    const uint32_t w = dword_of(v[0], S);
    uint32_t h = w >> 4;  // high nibble of byte i at bits 3:0 of its byte i
    asm("" : "+v"(h));    // (one shift per dword: the conversions select their byte)
    return exact_pair(__builtin_amdgcn_cvt_off_f32_i4((w >> (8 * i)) & 0xFFu),
                      __builtin_amdgcn_cvt_off_f32_i4((h >> (8 * i)) & 0xFFu));
  } else if constexpr (ENC == kQ8) {
    const uint32_t d = dword_of(v[S >> 1], 2 * (S & 1) + (i >> 1)) >> (16 * (i & 1));
    return exact_pair(static_cast<float>(static_cast<int8_t>(d)), static_cast<float>(static_cast<int8_t>(d >> 8)));
  } else {
    return dword_of(v[S], i);
  }
}

// 16-byte slot (8 elements, within a group) of the B operand of K-step S for
// lane quadrant q, matching weight_pair's order.
template <int ENC>
__device__ __forceinline__ int x_slot(int q, int S) {
  if constexpr (ENC == kQ4) return 4 * q + S;
  else if constexpr (ENC == kQ8) return 8 * (S >> 1) + 2 * q + (S & 1);
  else return 4 * S + q;
}

// LDS position of slot s of staged row r is s ^ row_swizzle(r). The LDS serves
// a 16-byte read of 64 lanes in four turns of 16; each turn holds 16 different
// rows of a tile, rows 0-3 and 12-15 from one lane quadrant and rows 4-11 from
// the next one (or the other way round), so their positions are distinct when
// {swizzle(rows 0-3, 12-15)} and {swizzle(rows 4-11) ^ (slot step from one
// quadrant to the next)} are: with the row itself for steps of 1 and 2 (BF16,
// Q8), with bit 2 of the row taken from bit 3 for steps of 4 (Q4). (The bank
// conflicts in the counters are the weights' reorder, 2 cycles per ds_bpermute.)
// An aligned group of four positions holds an
// aligned group of four slots, so that the four neighbouring lanes which the
// address unit takes together load 64 contiguous bytes: 16 cache accesses per
// load of 64 lanes, against 64 when the slots of a group are stored apart.
template <int ENC>
__device__ __forceinline__ int row_swizzle(int r) {
  return ENC == kQ4 ? ((r & 11) | ((r >> 1) & 4)) : (r & 15);
}

// g / (1 + exp(-g)) of four values: the reciprocal refined by one Newton step,
// as accurate as the divide at half its instructions. The reciprocal flushes
// subnormal results: from 1 + exp(-g) = 2^126 on (g below -87.3) it is taken of
// 2^-32 times that (where exp overflows it is 0 and the step's NaN becomes 1, so
// the result is -0, NaN for -inf). One comparison for the four and a branch that
// is hardly ever taken and short: with divides behind it the epilogue's code,
// unrolled for every tile size, cost 0.5% of a call, without the branch (the
// scale in every value) 0.4%.
__device__ __forceinline__ f32x4_t silu4(f32x4_t g) {
  f32x4_t d, s;
#pragma unroll
  for (int e = 0; e < 4; ++e) d[e] = 1.0f + __expf(-g[e]);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float r = __builtin_amdgcn_rcpf(d[e]);
    s[e] = g[e] * fmaf(fmaf(-d[e], r, 1.0f), r, r);
  }
  if (__builtin_expect(__any(fmaxf(fmaxf(d[0], d[1]), fmaxf(d[2], d[3])) > 0x1p126f), 0)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float k = 0x1p-32f * d[e];
      const float r = __builtin_amdgcn_rcpf(k);
      if (d[e] > 0x1p126f) s[e] = g[e] * fmaf(fminf(fmaf(-k, r, 1.0f), 1.0f), r, r) * 0x1p-32f;
    }
  }
  return s;
}

// One work item of TT 16-route tiles: rows of row block rb of `expert`, the
// nt <= 16 TT routes listed in LDS.
template <int ENC, int NMAT, int MODE, int TT>
__device__ __forceinline__ void run_item(const MfmaArgs& a, unsigned char* lds, int expert, int rb, int nt) {
  using E = PEnc<ENC>;
  constexpr bool kScaled = ENC != kBF16;
  constexpr int L = E::kLoads;
  constexpr int D = stages_for(ENC, TT);
  constexpr int NR = raw_sets_for(ENC, TT);
  constexpr int kStageBytes = TT * kTileBytes + kScaleBytes;
  constexpr int kPerStage = TT + (kScaled ? 1 : 0);  // loads into LDS per wave and stage
  static_assert((D - 2) * kPerStage + (D - 1) * 2 * L <= 63, "outstanding loads must fit vmcnt");
  static_assert(NR + 1 >= D - 1, "wait_next counts one weight group per stage from the first stage on");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int q = lane >> 4, t16 = lane & 15;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((stage_lds_t*)(lds)));
  const int S = static_cast<int>(a.K / 128);
  const int rows = static_cast<int>(a.rows);
  const uint32_t row_bytes = static_cast<uint32_t>(S) * E::kGroupBytes;
  const int* ids = reinterpret_cast<const int*>(lds + kRouteOff);
  const int* srcs = reinterpret_cast<const int*>(lds + kSourceOff);

  // ---- sources: weight rows, activation rows, scales ----
  const uint8_t* wbase[2];
  uint32_t woff[2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt) {
    // a load takes 64 bytes of 16 rows, four neighbouring lanes one row's (16
    // cache accesses; with the MFMA's own order, 16 rows in neighbouring lanes,
    // 64); to_operand then moves lane 4 r + c's bytes to lane r + 16 c
    int row = (lane >> 2) + (NMAT == 2 ? rb * 64 + 16 * wave : rb * 128 + 32 * wave + 16 * mt);
    row = min(row, rows - 1);  // padding rows of the last block repeat the last row
    wbase[mt] = a.w[NMAT == 2 ? mt : 0] + static_cast<int64_t>(expert) * rows * row_bytes;
    woff[mt] = static_cast<uint32_t>(row) * row_bytes + 16 * (lane & 3);
  }
  uint32_t xoff[TT];
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    const int r = 16 * j + 4 * wave + q;  // staged row this lane fills, at position t16
    xoff[j] = static_cast<uint32_t>(srcs[r]) * static_cast<uint32_t>(a.ldx * 2) + 16 * (t16 ^ row_swizzle<ENC>(r & 15));
  }
  const uint8_t* const x = reinterpret_cast<const uint8_t*>(a.x);
  const float* ssrc = nullptr;
  int gdiv = 1;
  if constexpr (kScaled) {
    const int G = static_cast<int>(a.K / a.group);
    gdiv = static_cast<int>(a.group / 128);
    // lanes 0-31: this wave's rows (16 of each matrix, or 32); the others
    // repeat lane 0's (one more cache access each 16)
    const int l = lane < 32 ? lane : 0;
    int row = NMAT == 2 ? rb * 64 + 16 * wave + (l & 15) : rb * 128 + 32 * wave + l;
    row = min(row, rows - 1);
    ssrc = a.s[NMAT == 2 ? l >> 4 : 0] + static_cast<int64_t>(expert) * a.scales_per_expert +
           static_cast<int64_t>(row) * G;
  }

  auto issue = [&](int g, int slot) {
    const uint32_t buf = __builtin_amdgcn_readfirstlane(lds_base + static_cast<uint32_t>(slot * kStageBytes));
    const uint8_t* xg = x + static_cast<int64_t>(g) * kRowBytes;
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      uint32_t o = xoff[j];
      asm("" : "+v"(o));  // (extended to 64 bits by the load itself, not kept extended)
      dma16_to(xg + o, buf + (16 * j + 4 * wave) * kRowBytes);
    }
    if constexpr (kScaled)
      dma4_to(ssrc + g / gdiv, __builtin_amdgcn_readfirstlane(buf + TT * kTileBytes + wave * 256));
  };
  auto load_weights = [&](int g, uint4 (&v)[2][L]) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int u = 0; u < L; ++u) v[mt][u] = ldg16(wbase[mt] + (woff[mt] + static_cast<uint32_t>(g * E::kGroupBytes + 64 * u)));
  };

  f32x4_t acc[2][TT];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) acc[mt][tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // bytes of lane 4 (lane % 16) + lane / 16
  const int from = 4 * (4 * t16 + q);
  auto to_operand = [&](uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from, static_cast<int>(v)));
  };

  uint32_t xo[4];  // LDS byte (within a 16-route tile) of this lane's B operand of each K-step
#pragma unroll
  for (int s = 0; s < 4; ++s) xo[s] = static_cast<uint32_t>(t16 * kRowBytes + ((x_slot<ENC>(q, s) ^ row_swizzle<ENC>(t16)) << 4));

  // Waits until the next stage is resident. Loads complete in issue order, and
  // after that stage's, its body's weight group and the loads of the D - 2
  // stages behind it with a weight group each were issued: those may be in
  // flight. Past the main loop the compiler may drop weight loads that nothing
  // uses, so only the loads into LDS are counted there.
  auto wait_next = [&](auto exact) {
    wait_loads<(D - 2) * kPerStage + (decltype(exact)::value ? (D - 1) * 2 * L : 0)>();
  };

  struct Weights {
    u32x4_t f[2][4];  // A operands of a group: [16-row tile][K-step]
  };
  struct Raw {
    uint4 v[2][L];
  };
  // Q4, Q8: the bytes in the operand's lane order
  auto reorder = [&](Raw& r) {
    if constexpr (kScaled) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int u = 0; u < L; ++u) {
          uint4& v = r.v[mt][u];
          v = make_uint4(to_operand(v.x), to_operand(v.y), to_operand(v.z), to_operand(v.w));
        }
    }
  };
  auto convert = [&](const Raw& r, Weights& w, int unit) {  // pair `unit` (0..31) of a group's operands
    const int mt = unit & 1, S_ = unit >> 3, i = (unit >> 1) & 3;
    if constexpr (kScaled)
      w.f[mt][S_][i] = weight_pair<ENC>(r.v[mt], S_, i);
    else
      w.f[mt][S_][i] = to_operand(dword_of(r.v[mt][S_], i));
  };
  int slot = 0;
  Weights w[2];
  Raw raw[NR];
  // Group g (a stage), u = g mod NR: its MFMAs from w[u % 2], while the next
  // group's bytes are converted into the other one and those of group g + NR
  // are loaded.
  auto group = [&](int g, auto u_tag, auto exact) {
    constexpr int U_ = decltype(u_tag)::value;
    const Weights& wc = w[U_ & 1];
    Weights& wn = w[(U_ + 1) & 1];
    Raw& r = raw[(U_ + 1) % NR];
    // (past the last stage the last one is loaded again, into a buffer nothing
    // reads: a branch here would split the group's code and let the compiler
    // move its arithmetic out of it)
    issue(min(g + D - 1, S - 1), slot == 0 ? D - 1 : slot - 1);
    __builtin_amdgcn_sched_barrier(0);
    // (behind the stage's loads, so that the wait for that stage does not
    // include these, which come from HBM)
    load_weights(min(g + NR, S - 1), raw[U_ % NR].v);
    __builtin_amdgcn_sched_barrier(0);
    const unsigned char* buf = lds + slot * kStageBytes;
    f32x4_t sc[2];
    if constexpr (kScaled) {
      const float* sl = reinterpret_cast<const float*>(buf + TT * kTileBytes + wave * 256) + 4 * q;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) sc[mt] = *reinterpret_cast<const f32x4_t*>(sl + 16 * mt);
    }
    bf16x8_t b[2][4];
    f32x4_t d[2][2];
    auto read = [&](int tt) {
#pragma unroll
      for (int s = 0; s < 4; ++s) b[tt & 1][s] = *reinterpret_cast<const bf16x8_t*>(buf + xo[s] + tt * kTileBytes);
    };
    auto fold = [&](int tt) {  // acc += scale * (sums over the group)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[mt][tt][e] = fmaf(sc[mt][e], d[tt & 1][mt][e], acc[mt][tt][e]);
    };
    read(0);
    reorder(r);
#pragma unroll
    for (int tt = 0; tt < TT; ++tt) {
      if (tt + 1 < TT) read(tt + 1);
      if constexpr (kScaled) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) d[tt & 1][mt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          f32x4_t& c = kScaled ? d[tt & 1][mt] : acc[mt][tt];
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wc.f[mt][s]), b[tt & 1][s], c, 0, 0, 0);
        }
      if constexpr (kScaled) {
        if (tt > 0) fold(tt - 1);
      }
#pragma unroll
      for (int unit = 32 * tt / TT; unit < 32 * (tt + 1) / TT; ++unit) convert(r, wn, unit);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kScaled) fold(TT - 1);
    wait_next(exact);
    stage_barrier();  // stage g consumed, stage g + 1 resident
    slot = slot + 1 == D ? 0 : slot + 1;
  };

#pragma unroll
  for (int g = 0; g < D - 1; ++g) issue(min(g, S - 1), g);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int g = 0; g < NR; ++g) load_weights(min(g, S - 1), raw[g].v);
  reorder(raw[0]);
#pragma unroll
  for (int unit = 0; unit < 32; ++unit) convert(raw[0], w[0], unit);
  wait_next(std::false_type{});
  stage_barrier();
  constexpr int U = NR;
  static_assert(NR % 2 == 0, "w alternates");
  constexpr std::true_type in_loop{};
  constexpr std::false_type last{};
  int g = 0;
  for (; g + U <= S; g += U) {
    group(g, std::integral_constant<int, 0>{}, in_loop);
    group(g + 1, std::integral_constant<int, 1>{}, in_loop);
    if constexpr (U > 2) {
      group(g + 2, std::integral_constant<int, 2>{}, in_loop);
      group(g + 3, std::integral_constant<int, 3>{}, in_loop);
    }
  }
  if (g < S) group(g, std::integral_constant<int, 0>{}, last);
  if constexpr (U > 2) {
    if (g + 1 < S) group(g + 1, std::integral_constant<int, 1>{}, last);
    if (g + 2 < S) group(g + 2, std::integral_constant<int, 2>{}, last);
  }
  wait_loads<0>();  // no load into LDS outlives the workgroup

  // ---- outputs ----
#pragma unroll
  for (int tt = 0; tt < TT; ++tt) {
    const int tok = 16 * tt + t16;
    if (tok >= nt) continue;
    const int64_t at = static_cast<int64_t>(ids[tok]) * a.ldo;
    constexpr float kUnit = ENC == kQ4 ? 16.f : 1.f;  // Q4 weights enter as q / 16
    if constexpr (MODE == kModeSilu) {
      const int r0 = rb * 64 + 16 * wave + 4 * q;
      if (r0 >= rows) continue;
      uint32_t g2[2], u2[2], h[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        g2[e] = pack_bf16x2(kUnit * acc[0][tt][2 * e], kUnit * acc[0][tt][2 * e + 1]);
        u2[e] = pack_bf16x2(kUnit * acc[1][tt][2 * e], kUnit * acc[1][tt][2 * e + 1]);
      }
      const f32x4_t s = silu4(f32x4_t{bf16lo(g2[0]), bf16hi(g2[0]), bf16lo(g2[1]), bf16hi(g2[1])});
#pragma unroll
      for (int e = 0; e < 2; ++e) h[e] = pack_bf16x2(s[2 * e] * bf16lo(u2[e]), s[2 * e + 1] * bf16hi(u2[e]));
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + at + r0) = make_uint2(h[0], h[1]);
    } else {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const int r0 = rb * 128 + 32 * wave + 16 * mt + 4 * q;
        if (r0 >= rows) continue;
        const f32x4_t v = acc[mt][tt] * kUnit;
        if constexpr (MODE == kModeF32)
          *reinterpret_cast<float4*>(static_cast<float*>(a.out) + at + r0) = make_float4(v[0], v[1], v[2], v[3]);
        else
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + at + r0) =
              make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
      }
    }
  }
}

}  // namespace

// One work item per workgroup. The items (row blocks of a tile next to each
// other, tiles in expert order) are split into 8 contiguous ranges, one per
// XCD (blockIdx % 8), so that a tile's row blocks share its activations and an
// expert's tiles share its rows in one XCD's L2.
template <int ENC, int NMAT, int MODE>
__global__ __launch_bounds__(kThreads, 2) void prefill_mfma_kernel(MfmaArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  const int n_tiles = a.tiles != nullptr ? *a.tile_count : a.tile_bound;
  const int64_t n_items = static_cast<int64_t>(n_tiles) * a.row_blocks;
  const int xcd = static_cast<int>(blockIdx.x & 7u);
  const int64_t item = n_items * xcd / 8 + (blockIdx.x >> 3);
  if (item >= n_items * (xcd + 1) / 8) return;  // uniform over the workgroup
  const int tile = __builtin_amdgcn_readfirstlane(static_cast<int>(item / a.row_blocks));
  const int rb = __builtin_amdgcn_readfirstlane(static_cast<int>(item % a.row_blocks));
  int expert = 0, first, nt;
  if (a.tiles != nullptr) {
    expert = __builtin_amdgcn_readfirstlane(a.tiles[2 * tile]);
    first = __builtin_amdgcn_readfirstlane(a.tiles[2 * tile + 1]);
    const int beg = __builtin_amdgcn_readfirstlane(a.expert_offsets[expert]);
    const int end = __builtin_amdgcn_readfirstlane(a.expert_offsets[expert + 1]);
    nt = min(route_tile_step(end - beg, kPrefillTileTokens), end - first);
  } else {
    const int step = even_step(a.n_routes, a.tile_bound);
    first = tile * step;
    nt = min(step, a.n_routes - first);
  }
  int* ids = reinterpret_cast<int*>(lds + kRouteOff);
  int* srcs = reinterpret_cast<int*>(lds + kSourceOff);
  for (int i = threadIdx.x; i < kPrefillTileTokens; i += kThreads) {
    int route = first + (i < nt ? i : 0);  // padding repeats the first route
    if (a.route_order != nullptr) route = a.route_order[route];
    ids[i] = route;
    srcs[i] = route / a.x_div;
  }
  __syncthreads();
  switch ((nt + 15) / 16) {
    case 1: run_item<ENC, NMAT, MODE, 1>(a, lds, expert, rb, nt); break;
    case 2: run_item<ENC, NMAT, MODE, 2>(a, lds, expert, rb, nt); break;
    case 3: run_item<ENC, NMAT, MODE, 3>(a, lds, expert, rb, nt); break;
    case 4: run_item<ENC, NMAT, MODE, 4>(a, lds, expert, rb, nt); break;
    case 5: run_item<ENC, NMAT, MODE, 5>(a, lds, expert, rb, nt); break;
    case 6: run_item<ENC, NMAT, MODE, 6>(a, lds, expert, rb, nt); break;
    case 7: run_item<ENC, NMAT, MODE, 7>(a, lds, expert, rb, nt); break;
    case 8: run_item<ENC, NMAT, MODE, 8>(a, lds, expert, rb, nt); break;
    default: run_item<ENC, NMAT, MODE, kMaxTT>(a, lds, expert, rb, nt); break;
  }
}

namespace {

template <int ENC, int NMAT, int MODE>
hipError_t launch_cfg(const MfmaArgs& args, hipStream_t stream) {
  MfmaArgs a = args;
  const int64_t block_rows = NMAT == 2 ? 64 : 128;
  a.row_blocks = static_cast<int32_t>((a.rows + block_rows - 1) / block_rows);
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_mfma_kernel<ENC, NMAT, MODE>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
  if (e != hipSuccess) return e;
  const int64_t items = static_cast<int64_t>(a.row_blocks) * a.tile_bound;
  const int64_t grid = (items + 7) / 8 * 8;  // every XCD's range rounded up
  if (grid > 0x7FFFFFFF) return hipErrorInvalidValue;
  hipLaunchKernelGGL((prefill_mfma_kernel<ENC, NMAT, MODE>), dim3(static_cast<unsigned>(grid)), dim3(kThreads),
                     kLdsBytes, stream, a);
  return hipGetLastError();
}

template <int ENC>
hipError_t launch_enc(int nmat, int mode, const MfmaArgs& a, hipStream_t stream) {
  if (nmat == 2 && mode == kModeSilu) return launch_cfg<ENC, 2, kModeSilu>(a, stream);
  if (nmat == 1 && mode == kModeF32) return launch_cfg<ENC, 1, kModeF32>(a, stream);
  if (nmat == 1 && mode == kModeBF16) return launch_cfg<ENC, 1, kModeBF16>(a, stream);
  return hipErrorInvalidValue;
}

}  // namespace

bool prefill_supported(int enc, int64_t rows, int64_t K, int64_t group, int64_t x_rows, int64_t ldx) {
  if (rows <= 0 || rows % 16 != 0 || K < 256 || K % 128 != 0) return false;
  // 32-bit byte offsets within one expert's matrix and within the activations
  if (rows * K * 2 >= (int64_t{1} << 31) || x_rows * ldx * 2 >= (int64_t{1} << 32)) return false;
  return enc == kBF16 || (group > 0 && group % 128 == 0 && K % group == 0);
}

hipError_t launch_prefill_mfma(int enc, int nmat, int mode, const MfmaArgs& args, hipStream_t stream) {
  MfmaArgs a = args;
  if (!prefill_supported(enc, a.rows, a.K, a.group, 0, a.ldx)) return hipErrorInvalidValue;
  if (a.tile_bound <= 0) return hipSuccess;
  if (enc != kBF16) a.scales_per_expert = a.rows * a.K / a.group;
  if (enc == kQ4) return launch_enc<kQ4>(nmat, mode, a, stream);
  if (enc == kQ8) return launch_enc<kQ8>(nmat, mode, a, stream);
  return launch_enc<kBF16>(nmat, mode, a, stream);
}

}  // namespace uqm
