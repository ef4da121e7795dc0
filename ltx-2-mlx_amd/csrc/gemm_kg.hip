// Mid-size projection GEMMs on CDNA4 matrix cores: the products of gemm.hip
// whose 256x256 tiles would leave most of the 256 CUs idle (a few hundred to
// ~1300 rows: text contexts, short or low-resolution clips, the connector).
//
//   C[m, n] = epilogue( sum_k A[m, k] * W[n, k] + bias[n] )
//
// Same operands, weight formats, epilogues and rounding points as gemm.hip.
//
// A workgroup computes a BM x 128 tile (BM = 64, 128 or 192) with 8 waves in
// two groups of four (2 x 2 wave tiles of BM/2 x 64).  The groups split K
// inside the workgroup: a unit of the K loop is one stage per group (64 k for
// 8-bit weights, 32 k for bf16), so each SIMD holds two waves that work on
// different stages of the same tile, and an LDS byte is read by two waves
// instead of the four that eight waves side by side on one stage would take
// (64 KB against 96 KB of fragment reads per 128 x 128 x 64 bf16 stage).
// The two fp32 accumulators meet once, through LDS, after the loop.
//
// Units reach LDS by direct buffer loads into rings several units deep; the
// fragments of the next k-step are read while the MFMAs of the current one
// run, also across the one barrier per unit.  Every row piece that a load
// moves is a whole 128-byte line: both groups' 64-byte halves lie in one LDS
// row.  (With a row of 64 bytes per group each line took two requests, and
// the requests bounded the bf16 tiles: 384 x 4096 -> 4096 36.5 -> 30.2 us,
// 384 x 4096 -> 16384 69.4 -> 59.3, 384 x 16384 -> 4096 105 -> 88, 1024 x
// 16384 -> 4096 164 -> 144; 8-bit weights, whose activations were whole
// lines already: 256 x 4096 -> 8192 MXFP8 27.1 -> 25.5, the rest within 3 %.)
// What bounds it: a CU's operand bytes, of which a 128 x 128 tile takes 384 (8-bit
// weights) or 512 (bf16) per k for 8 cycles of MFMA.  With all CUs busy each gets
// 47 bytes per ns, 12 TB/s together (384 x 4096 -> 16384 bf16 256 workgroups x
// 2.6 MB in 56 us, 1296 x 4096 -> 4096 MXFP8 224 x 2.1 MB in 44), while the MFMAs
// are busy 0.35-0.40 of the cycles, the LDS 0.17-0.19, and the L2 channels take
// 0.3 requests per cycle; a few CUs alone get no more from HBM (bf16 26 x 188160
// -> 2048, 16 workgroups: 43 bytes of weights per ns).  A deeper ring changed
// nothing.
#include "gemm_common.h"

namespace ltx {

constexpr int kKgThreads = 512;

template <int BKIND, int BM_>
struct KgCfg {
  static constexpr bool BF = BKIND == B_BF16, MXS = BKIND == B_MXFP8;
  static constexpr int BM = BM_, BN = 128;
  static constexpr int KU = BF ? 32 : 64;            // k per group and unit
  static constexpr int ES = BF ? 2 : 1;              // weight bytes per element
  static constexpr int KS = KU / 32;                 // MFMA k-steps per group and unit
  static constexpr int WM = BM / 2, WN = 64;         // wave tile
  static constexpr int AM = WM / 16, AN = WN / 16;   // its 16x16 accumulator blocks
  static constexpr int HM = AM / 2;                  // row blocks kept per group after the exchange
  static constexpr int A_ROWB = 128, B_ROWB = 128;   // LDS row bytes
  static constexpr int A_BYTES = BM * 2 * KU, B_BYTES = BN * KU * ES;  // one group's stage
  // ring depths in units.  192-row tiles of 8-bit weights: three whole units
  // exceed the LDS, so the activations (mostly L2 hits) run one unit ahead
  // and the weights (HBM) two.
  static constexpr int RA = BF ? (BM == 64 ? 6 : (BM == 128 ? 5 : 4)) : (BM == 64 ? 4 : (BM == 128 ? 3 : 2));
  static constexpr int RB = BF ? RA : (BM == 64 ? 4 : 3);
  // direct-load instructions (1 KiB) per wave and unit: both groups' stages
  static constexpr int A_DMA = 2 * A_BYTES / 1024 / 8, B_DMA = 2 * B_BYTES / 1024 / 8;
  // the wait at the barrier of unit u (h = u % 4): loads younger than those of
  // unit u + 1, the scale load of a unit with h == 0 among them
  static constexpr int in_flight(int h) {
    int n = (RA - 2) * (A_DMA + B_DMA) + (RB > RA ? B_DMA : 0);
    if (MXS)
      for (int t = 1; t <= RA - 2; ++t) n += (h - t + 8) % 4 == 0 ? 1 : 0;
    return n;
  }
  static constexpr int B_OFF = RA * 2 * A_BYTES;
  // E8M0 bytes of four units, [row][16], double buffered
  static constexpr int SC_OFF = B_OFF + RB * 2 * B_BYTES;
  static constexpr int RING = SC_OFF + (MXS ? 2 * BN * 16 : 0);
  // after the loop: the exchanged accumulator halves, the bf16 output tile,
  // the column values
  static constexpr int X_WAVE = HM * AN * 64 * 16, X_BYTES = 8 * X_WAVE;
  static constexpr int E_WAVE = HM * 16 * WN * 2;
  static constexpr int COL_OFF = X_BYTES + 8 * E_WAVE;
  static constexpr int EPI = COL_OFF + 2 * BN * 4;
  static constexpr int LDS_BYTES = RING > EPI ? RING : EPI;
  static_assert(AM % 2 == 0 && AN == 4, "accumulator row blocks split between the groups");
  static_assert((2 * A_BYTES) % 8192 == 0 && B_BYTES == 8192, "whole direct-load instructions per wave");
  static_assert(RB == RA || RB == RA + 1, "ring depths");
  static_assert(in_flight(0) < 60, "vmcnt range");
  static_assert(!MXS || RA <= 4, "a scale load lands within the four units before its use");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

// 4-byte direct load: one dword per lane to lds_dst + 4 * lane
__device__ __forceinline__ void kg_dma4(const void* base, int num_records, uint32_t voff, int soff, char* lds_dst) {
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, num_records, kBufferRsrcWord3);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)lds_dst, 4, voff, soff, 0, 0);
}

template <int BKIND, int EPI, int BM_>
__global__ __launch_bounds__(kKgThreads, 1) void gemm_kg_kernel(GemmArgs p) {
  using Cfg = KgCfg<BKIND, BM_>;
  constexpr bool BF = Cfg::BF, MXS = Cfg::MXS;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, WM = Cfg::WM, WN = Cfg::WN, AM = Cfg::AM, AN = Cfg::AN, HM = Cfg::HM;
  constexpr int A_ROWB = Cfg::A_ROWB, B_ROWB = Cfg::B_ROWB, A_BYTES = Cfg::A_BYTES, B_BYTES = Cfg::B_BYTES;
  constexpr int A_DMA = Cfg::A_DMA, B_DMA = Cfg::B_DMA, RA = Cfg::RA, RB = Cfg::RB, ES = Cfg::ES;
  constexpr bool RESID = EPI == LTX_GEMM_EPI_RESIDUAL || EPI == LTX_GEMM_EPI_RESIDUAL_ROUND;
  constexpr bool PARTIAL = EPI == kEpiPartial;
  __shared__ __attribute__((aligned(1024))) char lds[Cfg::LDS_BYTES];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2;  // waves w and w + 4 share a SIMD
  const int wm = wave & 1, wn = (wave >> 1) & 1;

  // split-K: block b works on split b / tiles of tile b % tiles, the split's
  // k range starting at kz * K
  const int tiles = p.tiles_m * p.tiles_n;
  const int kz = PARTIAL ? (int)blockIdx.x / tiles : 0;
  int tmi, tni;
  tile_coords(PARTIAL ? (int)blockIdx.x % tiles : (int)blockIdx.x, tiles, p.tiles_m, p.tiles_n, tmi, tni);
  const int m0 = tmi * BM, n0 = tni * BN;
  const int KT = p.K / (2 * Cfg::KU);  // units
  const int64_t k0 = (int64_t)kz * p.K;
  // a wave whose tile lies wholly past M or N moves its share of every unit
  // and meets every barrier, but reads no fragments and issues no MFMAs
  const int live = __builtin_amdgcn_readfirstlane((m0 + wm * WM < p.M && n0 + wn * WN < p.N) ? 1 : 0);

  // ---- direct-load sources: instruction d of wave w fills 1 KiB block
  // 8 d + w of the unit, 8 LDS rows of 128 bytes; lane j its 16-byte slot j,
  // which holds the logical chunk that the row's XOR swizzle puts there.
  // Rows of 64 bytes per group (weights; bf16 weights' activations) hold both
  // groups' halves, so every row of a load is a whole 128-byte line: half
  // lines cost the L2 as many requests each.  8-bit weights' activations, 128
  // bytes per group, are group 0's rows, then group 1's.  Rows past M / N
  // re-read the last row.  The record counts bound the lane offsets to their
  // operand; the scalar offset, which they do not cover, stays inside the row
  // because past the last unit that one is loaded again.
  const int a_records = (int)((int64_t)p.M * p.lda * 2), b_records = (int)((int64_t)p.N * p.ldb * ES);
  uint32_t a_src[A_DMA];
#pragma unroll
  for (int d = 0; d < A_DMA; ++d) {
    const int lr = 8 * (8 * d + wave) + (lane >> 3);  // LDS row
    const int r = BF ? lr : lr % BM, g = BF ? 0 : lr / BM;
    const int chunk = BF ? pair_chunk(lane) : (lane & 7) ^ g8_swz128(r, true);
    int gm = m0 + r;
    gm = gm < p.M ? gm : p.M - 1;
    a_src[d] = (uint32_t)(((int64_t)gm * p.lda + k0) * 2) + g * 128 + chunk * 16;
  }
  uint32_t b_src[B_DMA];
#pragma unroll
  for (int d = 0; d < B_DMA; ++d) {
    const int r = 8 * (8 * d + wave) + (lane >> 3);
    int gn = n0 + r;
    gn = gn < p.N ? gn : p.N - 1;
    b_src[d] = (uint32_t)(((int64_t)gn * p.ldb + k0) * ES) + pair_chunk(lane) * 16;
  }
  // MXFP8 scales, four units at a time: 16 bytes per weight row, a dword per
  // lane of 16 rows per wave (a dword per unit of 64 rows per wave would
  // touch 64 cache lines per instruction, as much address work as the whole
  // unit's data: 28.5 against ~20 us on 256 x 4096 -> 8192)
  uint32_t sc_src = 0;
  const int sc_records = MXS ? (int)((int64_t)p.N * p.ld_scale) : 0;
  if constexpr (MXS) {
    int gn = n0 + 16 * wave + (lane >> 2);
    gn = gn < p.N ? gn : p.N - 1;
    sc_src = (uint32_t)((int64_t)gn * p.ld_scale + k0 / 32) + (lane & 3) * 4;
  }
  auto load_scales = [&](int o) __attribute__((always_inline)) {  // of units 4 o .. 4 o + 3
    if constexpr (MXS)
      kg_dma4(p.bscale, sc_records, sc_src, (4 * o < KT ? o : KT / 4 - 1) * 16,
              lds + Cfg::SC_OFF + (o & 1) * BN * 16 + wave * 256);
  };
  // load instruction l of a unit: the activations', then the weights'; past
  // the last unit, data that nobody reads
  constexpr int NL = A_DMA + B_DMA;
  auto load = [&](int u, int sa, int sb, int l) __attribute__((always_inline)) {
    const int ua = clamp_unit(u + RA, KT), ub = clamp_unit(u + RB, KT);
    if (l < A_DMA)
      buffer_dma16(p.A, a_records, a_src[l < A_DMA ? l : 0], ua * 4 * Cfg::KU,
                   lds + sa * 2 * A_BYTES + (8 * l + wave) * 1024);
    else
      buffer_dma16(p.B, b_records, b_src[l >= A_DMA ? l - A_DMA : 0], ub * 2 * Cfg::KU * ES,
                   lds + Cfg::B_OFF + sb * 2 * B_BYTES + (8 * (l - A_DMA) + wave) * 1024);
  };

  // ---- fragment addresses of the lane (row r16 of a 16-row block, k-quarter
  // q) in unit slot 0.  8-bit codes: k-step s is k = 16 q + 8 s + [0, 8) in
  // both operands (codes: chunk q of the group's half row; activations: chunk
  // 2 q + s of the 128-byte row); bf16: k = 8 q + [0, 8).
  const int r16 = lane & 15, q = lane >> 4;
  int a_rd[Cfg::KS];
#pragma unroll
  for (int s = 0; s < Cfg::KS; ++s)
    a_rd[s] = (wm * WM + r16) * A_ROWB + (BF ? ((4 * grp + q) ^ swz_pair(r16)) * 16
                                             : grp * A_BYTES + ((2 * q + s) ^ g8_swz128(r16, true)) * 16);
  const int w_rd = Cfg::B_OFF + (wn * WN + r16) * B_ROWB + ((4 * grp + q) ^ swz_pair(r16)) * 16;
  const int s_rd = Cfg::SC_OFF + (wn * WN + r16) * 16 + 2 * grp + (q >> 1);  // the lane's k-block of 32

  float s_i8[AN];
#pragma unroll
  for (int j = 0; j < AN; ++j) {
    int gn = n0 + wn * WN + j * 16 + r16;
    gn = gn < p.N ? gn : p.N - 1;
    s_i8[j] = BKIND == B_INT8 ? ((const float*)p.bscale)[gn] : 0.0f;
  }

  f32x4 acc[AM][AN];
#pragma unroll
  for (int i = 0; i < AM; ++i)
#pragma unroll
    for (int j = 0; j < AN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0f;

  // row blocks [I0, I1) of the activation fragments of k-step s; weight
  // fragments (and their scale bytes) of the unit
  auto read_a = [&](bf16x8 (&x)[AM], int s, int slot, auto i0, auto i1) __attribute__((always_inline)) {
#pragma unroll
    for (int i = decltype(i0)::value; i < decltype(i1)::value; ++i)
      x[i] = *reinterpret_cast<const bf16x8*>(lds + a_rd[s] + slot * 2 * A_BYTES + i * 16 * A_ROWB);
  };
  auto read_w = [&](u32x4 (&w)[AN], uint32_t (&sc)[AN], int u, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < AN; ++j) {
      w[j] = *reinterpret_cast<const u32x4*>(lds + w_rd + slot * 2 * B_BYTES + j * 16 * B_ROWB);
      if constexpr (MXS)
        sc[j] = *reinterpret_cast<const uint8_t*>(lds + s_rd + ((u >> 2) & 1) * BN * 16 + (u & 3) * 4 + j * 256);
    }
  };
  auto dequant = [&](uint32_t w0, uint32_t w1, float sc) __attribute__((always_inline)) -> bf16x8 {
    uint32_t o[4];
    if constexpr (MXS) {
      o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, sc, false));
      o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, sc, true));
      o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, sc, false));
      o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, sc, true));
    } else {
      // bf16(fp32(q) * s): one fp32 product, a single rounding
      const uint32_t ws[2] = {w0, w1};
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        const uint32_t u = ws[d];
        bf16x2 p0, p1;
        p0[0] = (bf16)((float)(int8_t)u * sc);
        p0[1] = (bf16)((float)(int8_t)(u >> 8) * sc);
        p1[0] = (bf16)((float)(int8_t)(u >> 16) * sc);
        p1[1] = (bf16)((float)((int32_t)u >> 24) * sc);
        o[2 * d] = __builtin_bit_cast(uint32_t, p0);
        o[2 * d + 1] = __builtin_bit_cast(uint32_t, p1);
      }
    }
    return __builtin_bit_cast(bf16x8, u32x4{o[0], o[1], o[2], o[3]});
  };
  // the MFMAs of one weight fragment (weights as the MFMA "A" operand: a lane
  // then holds 4 consecutive output columns)
  auto multiply = [&](const bf16x8 (&x)[AM], bf16x8 wf, int j) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, x[i], acc[i][j], 0, 0, 0);
  };

  // ---- prologue: the loads that the turns of units -RB .. -1 would issue, in
  // the loop's order, so that its waits count the same loads from the first
  // unit on
  load_scales(0);
#pragma unroll
  for (int j = 0; j < RB; ++j) {
    const int u = j - RB;
#pragma unroll
    for (int l = 0; l < NL; ++l)
      if (l >= A_DMA || u + RA >= 0) load(u, u + RA, j, l);
  }
  wait_vmcnt<Cfg::in_flight(2)>();
  barrier_nofence();

  // ---- main loop.  Barrier of unit u: this wave's loads of unit u + 1 have
  // landed and its fragment reads of unit u are complete; after it the slots
  // of unit u take units u + RA / u + RB, and unit u + 1 is read.  The MFMAs
  // run in groups of one weight fragment; each group also issues a share of
  // the loads and fragment reads and converts the next weight fragment.  The
  // scheduling fences between groups keep the compiler from sinking the reads
  // to their first use.
  int sa = 0, sb = 0;  // slots of unit u
  // barrier of a unit u, h = u % 4; the scales of the next four units go out
  // first after it when h == 0
  auto turn_wait = [&](int u, auto hc) __attribute__((always_inline)) {
    constexpr int h = decltype(hc)::value;
    wait_lgkmcnt0();
    wait_vmcnt<Cfg::in_flight(h)>();
    barrier_nofence();
    if (MXS && h == 0) load_scales((u >> 2) + 1);
  };
  auto next_slots = [&]() __attribute__((always_inline)) {
    sa = sa + 1 < RA ? sa + 1 : 0;
    sb = sb + 1 < RB ? sb + 1 : 0;
  };
  using I0 = std::integral_constant<int, 0>;
  using IH = std::integral_constant<int, AM / 2>;
  using IA = std::integral_constant<int, AM>;
  constexpr int LQ = (NL + AN - 1) / AN;  // load instructions per group
  // f(u, u % 4) for every unit; MXFP8 has whole groups of four
  auto units = [&](auto f) __attribute__((always_inline)) {
    int u = 0;
    for (; u + 3 < KT; u += 4) static_for<0, 4>([&](auto hc) { f(u + decltype(hc)::value, hc); });
    if constexpr (!MXS)
      static_for<0, 3>([&](auto hc) {
        if (u + decltype(hc)::value < KT) f(u + decltype(hc)::value, hc);
      });
  };
  if (!live) {
    auto idle = [&](int u, auto hc) __attribute__((always_inline)) {
      turn_wait(u, hc);
#pragma unroll
      for (int l = 0; l < NL; ++l) load(u, sa, sb, l);
      next_slots();
    };
    units(idle);
  } else if constexpr (BF) {
    bf16x8 x[2][AM];
    u32x4 w[2][AN];
    uint32_t none[AN];
    read_a(x[0], 0, 0, I0{}, IA{});
    read_w(w[0], none, 0, 0);
    auto unit = [&](int u, auto hc) __attribute__((always_inline)) {
      constexpr int h = decltype(hc)::value & 1;
      turn_wait(u, hc);
      const int fa = sa, fb = sb;
      next_slots();
#pragma unroll
      for (int j = 0; j < AN; ++j) {
        if (j == 0) read_w(w[1 - h], none, u + 1, sb);
        if (j == 1) read_a(x[1 - h], 0, sa, I0{}, IH{});
        if (j == 2) read_a(x[1 - h], 0, sa, IH{}, IA{});
#pragma unroll
        for (int l = j * LQ; l < (j + 1) * LQ && l < NL; ++l) load(u, fa, fb, l);
        multiply(x[h], __builtin_bit_cast(bf16x8, w[h][j]), j);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    units(unit);
  } else {
    bf16x8 x[2][AM], wf[2];
    u32x4 w[2][AN];
    uint32_t sc[AN] = {};
    float sf[AN];
    auto scales = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < AN; ++j) sf[j] = MXS ? e8m0_to_f32_valu(sc[j]) : s_i8[j];
    };
    read_a(x[0], 0, 0, I0{}, IA{});
    read_w(w[0], sc, 0, 0);
    scales();
    wf[0] = dequant(w[0][0][0], w[0][0][1], sf[0]);
    auto unit = [&](int u, auto hc) __attribute__((always_inline)) {
      constexpr int h = decltype(hc)::value & 1;
      int fa = 0, fb = 0;
#pragma unroll
      for (int f = 0; f < 2 * AN; ++f) {
        if (f == AN) {
          turn_wait(u, hc);
          fa = sa;
          fb = sb;
          next_slots();
        }
        if (f == 0) read_a(x[1], 1, sa, I0{}, IH{});
        if (f == 1) read_a(x[1], 1, sa, IH{}, IA{});
        if (f == AN) read_w(w[1 - h], sc, u + 1, sb);
        if (f == AN + 1) read_a(x[0], 0, sa, I0{}, IH{});
        if (f == AN + 2) read_a(x[0], 0, sa, IH{}, IA{});
        if (f >= AN) {
#pragma unroll
          for (int l = (f - AN) * LQ; l < (f - AN + 1) * LQ && l < NL; ++l) load(u, fa, fb, l);
        }
        if (f + 1 < 2 * AN) {
          const int s = (f + 1) / AN, j = (f + 1) % AN;
          wf[(f + 1) & 1] = dequant(w[h][j][2 * s], w[h][j][2 * s + 1], sf[j]);
        } else {
          scales();
          wf[0] = dequant(w[1 - h][0][0], w[1 - h][0][1], sf[0]);
        }
        multiply(x[f / AN], wf[f & 1], f % AN);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    units(unit);
  }
  wait_vmcnt<0>();
  __syncthreads();

  // ---- the groups' accumulators: each wave keeps half of its row blocks
  // (group 0 the lower, group 1 the upper) and adds the other group's
  {
    char* X = lds + wave * Cfg::X_WAVE + lane * 16;
#pragma unroll
    for (int i = 0; i < HM; ++i)
#pragma unroll
      for (int j = 0; j < AN; ++j)
        *reinterpret_cast<f32x4*>(X + (i * AN + j) * 1024) = grp == 0 ? acc[HM + i][j] : acc[i][j];
  }
  float* col_lds = reinterpret_cast<float*>(lds + Cfg::COL_OFF);
  if (!PARTIAL && tid < BN) {
    float col_bias = 0.0f, col_gate = 0.0f;
    if (n0 + tid < p.N) {
      if (p.bias) col_bias = p.bias[n0 + tid];
      if (RESID) col_gate = p.gate[n0 + tid];
    }
    col_lds[tid] = col_bias;
    col_lds[BN + tid] = col_gate;
  }
  __syncthreads();
  f32x4 sum[HM][AN];
  {
    const char* X = lds + (wave ^ 4) * Cfg::X_WAVE + lane * 16;
#pragma unroll
    for (int i = 0; i < HM; ++i)
#pragma unroll
      for (int j = 0; j < AN; ++j) {
        const f32x4 o = *reinterpret_cast<const f32x4*>(X + (i * AN + j) * 1024);
        const f32x4 mine = grp == 0 ? acc[i][j] : acc[HM + i][j];
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[i][j][e] = mine[e] + o[e];
      }
  }
  const int row0 = m0 + wm * WM + grp * (HM * 16);  // the wave's first output row
  const int col0 = n0 + wn * WN;
  if constexpr (PARTIAL) {
    float* P = p.partial + (int64_t)kz * p.M * p.ldc;
#pragma unroll
    for (int i = 0; i < HM; ++i) {
      const int gm = row0 + i * 16 + r16;
#pragma unroll
      for (int j = 0; j < AN; ++j) {
        const int gn = col0 + j * 16 + 4 * q;  // N % 8 == 0: four columns inside or outside
        if (gm < p.M && gn < p.N) *reinterpret_cast<f32x4*>(P + (int64_t)gm * p.ldc + gn) = sum[i][j];
      }
    }
    return;
  } else {
    // ---- epilogue: bf16 tile through LDS (128-byte rows, 16-byte chunks
    // XORed by (row / 2) % 8), then whole 16-byte chunks of rows
    constexpr int ITS = HM * 2;  // 8 rows of 8 chunks per pass
    const int ch = lane & 7, rsub = lane >> 3;
    const int gn2 = col0 + ch * 8;
    const bool col_ok = gn2 < p.N;
    bf16x8 res[RESID ? ITS : 1];
    if constexpr (RESID) {
#pragma unroll
      for (int it = 0; it < ITS; ++it) {
        int gm = row0 + it * 8 + rsub;
        gm = gm < p.M ? gm : p.M - 1;
        res[it] = *reinterpret_cast<const bf16x8*>(p.R + (int64_t)gm * p.ldr + (col_ok ? gn2 : 0));
      }
    }
    char* E = lds + Cfg::X_BYTES + wave * Cfg::E_WAVE;
    auto phase1 = [&](auto sig_tag, auto rtb_tag) {
      constexpr bool SIG = decltype(sig_tag)::value, RTB = decltype(rtb_tag)::value;
#pragma unroll
      for (int j = 0; j < AN; ++j) {
        const int nl = j * 16 + 4 * q;
        const f32x4 bias4 = *reinterpret_cast<const f32x4*>(col_lds + wn * WN + nl);
#pragma unroll
        for (int i = 0; i < HM; ++i) {
          float y[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] = sum[i][j][e];
          if (RTB) {
            round_bf2(y[0], y[1]);
            round_bf2(y[2], y[3]);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) y[e] += bias4[e];
          if (EPI == LTX_GEMM_EPI_GELU || EPI == LTX_GEMM_EPI_SIGMOID2 || SIG) {
            float r[4] = {y[0], y[1], y[2], y[3]};
            round_bf2(r[0], r[1]);
            round_bf2(r[2], r[3]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              if (EPI == LTX_GEMM_EPI_GELU) y[e] = gelu_tanh(r[e]);
              if (EPI == LTX_GEMM_EPI_SIGMOID2) y[e] = sigmoid2_bf(r[e]);
              if (SIG && col0 + nl + e >= p.sig_from) y[e] = sigmoid2_bf(r[e]);
            }
          }
          bf16x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (bf16)y[e];
          const int row = i * 16 + r16;
          *reinterpret_cast<bf16x4*>(E + row * 128 + ((((nl >> 3) ^ (row >> 1)) & 7) << 4) + (nl & 7) * 2) = v;
        }
      }
    };
    const bool sig = EPI == LTX_GEMM_EPI_BIAS && col0 + WN > p.sig_from;
    if (p.round_then_bias) {
      if (sig) phase1(std::true_type{}, std::true_type{});
      else phase1(std::false_type{}, std::true_type{});
    } else {
      if (sig) phase1(std::true_type{}, std::false_type{});
      else phase1(std::false_type{}, std::false_type{});
    }
    // a wave reads back only what it wrote itself
    wait_lgkmcnt0();
    __builtin_amdgcn_wave_barrier();
    float g8[8];
    if constexpr (RESID) {
      const f32x4 ga = *reinterpret_cast<const f32x4*>(col_lds + BN + wn * WN + ch * 8);
      const f32x4 gb = *reinterpret_cast<const f32x4*>(col_lds + BN + wn * WN + ch * 8 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        g8[e] = ga[e];
        g8[4 + e] = gb[e];
      }
    }
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
      const int ml = it * 8 + rsub, gm = row0 + ml;
      bf16x8 v = *reinterpret_cast<const bf16x8*>(E + ml * 128 + ((ch ^ (ml >> 1)) & 7) * 16);
      if constexpr (RESID) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float y = (float)v[e];
          const float o = EPI == LTX_GEMM_EPI_RESIDUAL ? fmaf(g8[e], y, (float)res[it][e])
                                                       : round_bf(y * g8[e]) + (float)res[it][e];
          v[e] = (bf16)o;
        }
      }
      if (gm < p.M && col_ok) *reinterpret_cast<bf16x8*>(p.C + (int64_t)gm * p.ldc + gn2) = v;
      if constexpr (EPI == LTX_GEMM_EPI_BIAS) {
        // the row's sum of squares over this wave's 64 columns: eight per
        // lane, then over the row's eight lanes
        if (p.rowss != nullptr && col0 < p.ss_cols) {
          float t = 0.0f;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float f = (float)v[e];
            t = fmaf(f, f, t);
          }
          t += __shfl_xor(t, 1, 64);
          t += __shfl_xor(t, 2, 64);
          t += __shfl_xor(t, 4, 64);
          if (ch == 0 && gm < p.M) p.rowss[(int64_t)gm * p.ld_rowss + col0 / WN] = t;
        }
      }
    }
  }
}

template <int BKIND, int EPI>
static void kg_launch_bm(GemmArgs p, int bm, int splits, hipStream_t s) {
  p.tiles_m = (p.M + bm - 1) / bm;
  p.tiles_n = (p.N + 127) / 128;
  const int blocks = p.tiles_m * p.tiles_n * splits;
  if (bm == 64) gemm_kg_kernel<BKIND, EPI, 64><<<blocks, kKgThreads, 0, s>>>(p);
  else if (bm == 128) gemm_kg_kernel<BKIND, EPI, 128><<<blocks, kKgThreads, 0, s>>>(p);
  else gemm_kg_kernel<BKIND, EPI, 192><<<blocks, kKgThreads, 0, s>>>(p);
}

template <int BKIND>
static bool kg_launch_kind(const GemmArgs& p, int epi, int bm, int splits, hipStream_t s) {
  switch (epi) {
    case LTX_GEMM_EPI_BIAS: kg_launch_bm<BKIND, LTX_GEMM_EPI_BIAS>(p, bm, splits, s); return true;
    case LTX_GEMM_EPI_GELU: kg_launch_bm<BKIND, LTX_GEMM_EPI_GELU>(p, bm, splits, s); return true;
    case LTX_GEMM_EPI_RESIDUAL: kg_launch_bm<BKIND, LTX_GEMM_EPI_RESIDUAL>(p, bm, splits, s); return true;
    case LTX_GEMM_EPI_RESIDUAL_ROUND: kg_launch_bm<BKIND, LTX_GEMM_EPI_RESIDUAL_ROUND>(p, bm, splits, s); return true;
    case LTX_GEMM_EPI_SIGMOID2: kg_launch_bm<BKIND, LTX_GEMM_EPI_SIGMOID2>(p, bm, splits, s); return true;
    case kEpiPartial: kg_launch_bm<BKIND, kEpiPartial>(p, bm, splits, s); return true;
  }
  return false;
}

bool kg_launch(int bkind, const GemmArgs& p, int epi, int bm, int splits, hipStream_t s) {
  if (bkind == B_BF16) return kg_launch_kind<B_BF16>(p, epi, bm, splits, s);
  if (bkind == B_INT8) return kg_launch_kind<B_INT8>(p, epi, bm, splits, s);
  if (bkind == B_MXFP8) return kg_launch_kind<B_MXFP8>(p, epi, bm, splits, s);
  return false;
}

}  // namespace ltx
