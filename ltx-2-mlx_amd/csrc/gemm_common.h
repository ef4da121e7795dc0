// Device helpers shared by the projection GEMM kernels (gemm.hip: the 4- and
// 8-wave tile kernels; gemm_rows.hip: the few-row split-K kernel): epilogue
// arithmetic, E8M0 decoding, LDS-DMA / buffer-load helpers and wait counters.
#pragma once

#include <type_traits>

#include "gemm_addr.h"
#include "ltx_common.h"

namespace ltx {

// B_MX: MXFP8 weights and MXFP8 activations (E4M3 codes + E8M0 scale per 32
// along K on both operands), multiplied by the scaled fp8 MFMA -- an opt-in
// path with quantised activations, only on the 8-wave kernel.
enum BKind { B_BF16 = 0, B_INT8 = 1, B_MXFP8 = 2, B_MX = 3 };

// workgroups are dealt to the 8 XCDs round-robin (block b runs on XCD b % 8)
constexpr int kNumXcd = 8;

// bf16 rounding of two values with one conversion: the same bits as
// round_bf on each
__device__ __forceinline__ void round_bf2(float& x, float& y) {
  asm("" : "+v"(x), "+v"(y));
  const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){x, y}, bf16x2));
  x = __uint_as_float(u << 16);
  y = __uint_as_float(u & 0xffff0000u);
}

// GELU with the tanh approximation (feed_forward.py:8-14).  tanh(u) is
// evaluated as 1 - 2 / (exp(2u) + 1) with the hardware exp2 and reciprocal
// a few instructions instead of the libm tanh and an IEEE division, absolute
// error ~2e-7, far below the bf16 rounding of the result; saturates correctly
// at +-inf.
__device__ __forceinline__ float gelu_tanh(float x) {
  // 0.5 x (1 + tanh(u)) with u = sqrt(2/pi) (x + 0.044715 x^3) is
  // x sigmoid(2u) = x / (1 + 2^t), t = -2u log2(e) = x (A + B x^2):
  // five VALU instructions and two transcendentals per element
  constexpr float A = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
  constexpr float B = A * 0.044715f;
  const float t = x * fmaf(B, x * x, A);
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(t));
}

// 2 * bf16(sigmoid(y)) -- the head gate of attention.py:586-590 -- with the
// hardware exp2 and reciprocal (relative error ~2e-7 before the bf16 rounding).
__device__ __forceinline__ float sigmoid2_bf(float y) {
  const float e = __builtin_amdgcn_exp2f(-1.4426950408889634f * y);
  return 2.0f * round_bf(__builtin_amdgcn_rcpf(1.0f + e));
}

__device__ __forceinline__ float e8m0_to_f32(uint32_t s) {
  // 2^(s-127): s << 23 is the float for 1 <= s <= 254; s = 0 (2^-127) and
  // s = 255 (NaN) set the top mantissa bit as well.  Branch-free: s differs
  // per lane.
  const uint32_t special = (s == 0u || s == 0xffu) ? 0x00400000u : 0u;
  return __uint_as_float((s << 23) | special);
}

// The same value in vector instructions only (no lane-mask round trip):
// 2^-127 * 2^s by ldexp -- exact, 2^-127 itself a denormal (denormals are
// kept) -- and s = 255 (+inf from ldexp) turned into NaN by x + (x - x).
__device__ __forceinline__ float e8m0_to_f32_valu(uint32_t s) {
  const float x = __builtin_amdgcn_ldexpf(__uint_as_float(0x00400000u), (int)s);
  return x + (x - x);
}


// LDS-DMA helpers: each lane of a wave writes the 16 bytes it loads to
// `lds_wave_base + 16 * lane`; the per-lane source address implements the
// swizzle (the data a lane fetches is the data its LDS slot must hold).
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) const void* gbl_ptr_t;

__device__ __forceinline__ void dma16(const void* src, char* lds_wave_base) {
  __builtin_amdgcn_global_load_lds((gbl_ptr_t)src, (lds_ptr_t)lds_wave_base, 16, 0, 0);
}

// s_waitcnt through the builtin (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] |
// lgkmcnt[11:8] | vmcnt_hi[15:14]) so the compiler's own wait insertion
// sees it.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | 0x70 | 0xF00);
}
__device__ __forceinline__ void wait_lgkmcnt0() { __builtin_amdgcn_s_waitcnt(0xC07F); }


// dword 3 of a raw buffer descriptor on gfx9-class GPUs (untyped, 32-bit
// data format so that dwordx4 loads are not format-converted)
constexpr int kBufferRsrcWord3 = 0x00020000;

// 16 bytes per lane from base + voff + soff (bounded by num_records bytes) to
// LDS at lds_dst + 16 * lane: a buffer load with the lds modifier.  The
// descriptor is built from wave-uniform values (scalar registers; the
// compiler hoists it out of loops).  Kept out of the kernel bodies, whose
// host-side launch stubs are not emitted when they name the descriptor type.
__device__ __forceinline__ void buffer_dma16(const void* base, int num_records, uint32_t voff, int soff,
                                             char* lds_dst) {
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, num_records, kBufferRsrcWord3);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)lds_dst, 16, voff, soff, 0, 0);
}

// Workgroup barrier without the memory fence of __syncthreads(): the fence
// would wait for every outstanding global->LDS load of the wave (they count as
// LDS writes), including the ones meant to stay in flight across the barrier.
// Callers wait for exactly what the barrier has to publish.
__device__ __forceinline__ void barrier_nofence() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

struct GemmArgs {
  const bf16* A;
  int64_t lda;
  const void* B;
  int64_t ldb;
  const void* bscale;  // int8: fp32 (N); mxfp8: uint8 (N, K/32)
  int64_t ld_scale;    // mxfp8 scale row stride (bytes)
  const float* bias;   // fp32 (N) or null
  bf16* C;
  int64_t ldc;
  const bf16* R;       // residual (gated epilogues), may alias C
  int64_t ldr;
  const float* gate;   // fp32 (N)
  int sig_from;        // columns n >= sig_from get the 2*sigmoid head-gate epilogue
  int round_then_bias; // bias added to the bf16-rounded product (quantised-linear form)
  float* partial;      // split-K: fp32 partial products [split][M][ldc], no epilogue
  const uint8_t* ascale;  // B_MX: activation E8M0 scales (M, K/32)
  int64_t ld_ascale;      // B_MX: their row stride (bytes)
  uint8_t* cscale;        // kEpiGeluMx: output E8M0 scales (M, N/32); C holds the codes
  int64_t ld_cscale;
  int M, N, K;         // split-K: K is the per-split depth
  int tiles_m, tiles_n;
  // 8-wave and mid-size bias epilogue: per-row sums of squares of the bf16 outputs of
  // columns [0, ss_cols), one fp32 partial per 64-column slice at
  // rowss[row * ld_rowss + col / 64] (null: none)
  float* rowss = nullptr;
  int64_t ld_rowss = 0;
  int ss_cols = 0;
};

// EPI value of the split-K pass: the accumulators go to the fp32 partial
// buffer as they are, the epilogue runs in splitk_epilogue_kernel.
constexpr int kEpiPartial = 16;
// EPI value of the MX kernel's FF up-projection: the GELU epilogue whose
// bf16 result leaves as MXFP8 rows (codes in C, E8M0 scales in cscale) --
// the next product's quantised activations, written by this one.
constexpr int kEpiGeluMx = 5;
constexpr int kGroupM = 4;

__device__ __forceinline__ void tile_coords(int bid, int nblocks, int tiles_m, int tiles_n, int& tm,
                                            int& tn) {
  // XCD-contiguous renumbering: hardware sends block b to XCD b % 8.
  const int q = nblocks / kNumXcd, r = nblocks % kNumXcd;
  const int xcd = bid % kNumXcd, idx = bid / kNumXcd;
  const int logical = xcd * q + (xcd < r ? xcd : r) + idx;
  // grouped ordering: kGroupM tile-rows sweep the tile-columns together
  const int per_group = kGroupM * tiles_n;
  const int group = logical / per_group;
  const int first_m = group * kGroupM;
  const int gsize = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
  const int in_group = logical % per_group;
  tm = first_m + in_group % gsize;
  tn = in_group / gsize;
}

// f(integral_constant<int, I>) for I = I0 .. N-1, in order
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

// 16-byte chunk XOR of row r in the 8-wave kernels' stages, 64-byte rows (4
// chunks) and 128-byte rows (8 chunks).  ds_read_b128 services a wave's lanes
// 16 at a time, in the lane-octet pairs (0, 3), (1, 2), (4, 7), (5, 6)
// (probed: two octets reading the same banks at other addresses conflict only
// in those pairs), and its conflicts were probed per read pattern (rocprofv3
// SQ_LDS_BANK_CONFLICT of a one-read kernel over 290 lane -> address tables):
// the 32x32 fragment reads (lane = row 0-31, lane / 32 = chunk half) are
// conflict-free under chunk ^ ((r / 4) % 4) and chunk ^ ((r / 2) % 8), but the
// 16x16 reads (lane % 16 = row, lane / 16 = chunk quarter) conflict under
// those (the FF up-projection: 36-39 M conflict cycles per launch) and not
// under chunk ^ (r bit 0 | r bit 2 << 1) and chunk ^ (r bit 1 | r bit 0 << 1
// | r bit 2 << 2).
__device__ __forceinline__ int g8_swz64(int r, bool s16) { return s16 ? ((r & 1) | ((r >> 1) & 2)) : ((r >> 2) & 3); }
__device__ __forceinline__ int g8_swz128(int r, bool s16) {
  return s16 ? (((r >> 1) & 1) | ((r & 1) << 1) | (r & 4)) : ((r >> 1) & 7);
}

// gemm_kg.hip: launch the mid-size kernel with BM-row tiles (64, 128 or 192)
// and `splits` K ranges (epi kEpiPartial; p.K is then the depth of one).
// The caller has checked kg_ok.  False: no such kernel.
bool kg_launch(int bkind, const GemmArgs& p, int epi, int bm, int splits, hipStream_t s);

}  // namespace ltx
