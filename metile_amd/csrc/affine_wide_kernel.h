// Wide affine GEMM (gfx950): y[M, N] = x[M, K] @ dequantize(w_q)[N, K]^T (+ residual), or the
// fused silu(x Wg^T) * (x Wu^T), for more rows than a small-row dispatch takes: prompts, large
// batches and the prefill matmul (reference: lower_affine_matmul,
// metile/compiler/affine_quantized.py:7-99, and the row loop of kernels/affine_qmv.py:4-322). The
// weights are read once per row tile instead of once per 32 rows.
//
// A workgroup of WN waves computes TM x 32 rows by 32 WN code columns; every wave owns 32 columns
// over all of the tile's rows (TM accumulators of v_mfma_f32_32x32x16), so each code is unpacked
// once per workgroup. What bounds it is issue slots: an MFMA of 32 x 32 x 16 takes the matrix
// cores 32 clocks, which leaves room for about six other vector instructions. So everything that
// need not be done per output and group is kept out of the loop:
//  * Codes become exact 16-bit floats without an offset: a nibble q in a byte is the fp8 (e4m3)
//    number q 2^-9 for all of 0..15, and v_cvt_scalef32_pk_*_fp8 with scale 2^9 turns two of them
//    into q exactly (9 instructions per 8 codes in K order, the price of unpacking alone). A chain
//    of four MFMAs then sums x q over a group from zero, with no correction for an offset.
//  * Per output and group one FMA remains, acc += s (x q).
//  * The bias term sum_g b_g X_g (X_g: the row's activation sum over group g) is a product of
//    depth K / G on the matrix cores, every 16 groups: X_g comes from MFMAs of the activations
//    against a one-hot column of ones (two per 16 rows and step, shared out over the waves; result
//    column = group), and enters as three bf16 parts (8 + 8 + 8 bits hold an fp32 sum exactly), so
//    the products are exact and the sum stays fp32. f16 biases enter as two bf16 parts (11 bits).
//
// Activations reach LDS through buffer_load...lds into four or eight stages of one K step (64),
// each stage its own array (the compiler then sees that reads do not touch the stage being filled);
// codes go straight to registers. One barrier per step: placed before the last row tile's MFMAs,
// when every wave holds the step's remaining operands in registers; behind it the stage is refilled
// and the next step's first operands are read, whose latency that row tile hides. The scales and
// biases of 16 groups are staged in LDS a chunk ahead.
//
// Measured (MI355X, 4-bit groups of 64, weights from memory; before: the ring GEMM for one projection,
// 32-row dispatches for the others): 2048 x 14336 x 4096 f16 437 -> 277 us, bf16 404 -> 262 (868 and 918
// TFLOP/s; torch's dense products 223 and 214 us), 512 x 1536 x 8960 bf16 30.9 -> 27.0 us, SwiGLU
// 1536 -> 8960 of 333 rows 148 -> 33.4 us over MLX rows and 106 -> 32.2 repacked, of 48 rows 27.2 -> 16.7
// and 18.5 -> 15.9. At 2048 rows the matrix cores are busy 55% of a SIMD's clocks and vector
// instructions are issued in 54% (131 per wave and step, 64 FMAs and 36 for codes, beside 20 MFMAs); a
// wave waits 35% of its life. Tried at that size in f16 (259 us with inputs that
// let the clocks run higher): waves of 64 columns, one a SIMD with 512 registers (348 us: nothing hides a
// wait); waves of 64 x 64 (317 us, spills); a barrier every second step (267 us); codes through LDS (260
// us, the same, and 8 KiB a stage).
// Groups of 32 keep two chains and two scales a step and spill: 4 to 66 registers, at most 180 bytes a
// lane, in the 64-row instances and in those of 96 and 128 rows whose registers two waves a SIMD share;
// 8-bit groups of 64 spill 2 to 5 in three of the 64 x 64 instances. The planner's costs were fitted with
// that in.
#pragma once

#include "affine_wide.h"
#include "common.h"

namespace mt {

namespace {

constexpr int kSbDwords = 9;   // 16 groups of 2 bytes, one more dword for an odd first group
constexpr int kXsStride = 144;  // bytes per row of the staged row sums: 16 groups x 4 parts x 2 + pad

// The 16-byte chunk c of LDS row r sits in slot c ^ swz(r): reads of one chunk of 16 consecutive
// rows hit distinct banks, and rows 32 apart swizzle alike.
__device__ __forceinline__ int swz(int r) { return (r ^ ((r >> 3) & 1)) & 7; }

// A pointer's bits in scalar registers, opaque to the optimizer: a choice between two of them stays
// a scalar select (of pointers in the argument block it became an indexed load from scratch, and
// the buffer descriptor made from it was read lane by lane).
__device__ __forceinline__ uint64_t uniform_bits(const void* q) {
  const uint64_t v = reinterpret_cast<uint64_t>(q);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

typedef const unsigned char __attribute__((address_space(1))) * global_ptr_t;

// silu(gate) * up of two accumulator registers x0, x1 of a tile whose rows of 16 lanes hold gate, up,
// gate, up columns: swapping the odd rows of 16 lanes of x0 with the even ones of x1 leaves the gate
// values of both in one register (lane rows x0, x1, x0, x1) and their up values in the other.
__device__ __forceinline__ float swiglu_pair(float x0, float x1) {
  const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(x0), __float_as_uint(x1), false,
                                                   false);
  const uint32_t gate = sw[0], up = sw[1];
  return silu_mul(__uint_as_float(gate), __uint_as_float(up));
}

// A value that must be computed by here (opaque to the optimizer).
__device__ __forceinline__ void pin(f32x16& v) { __asm__ volatile("" : "+v"(v)); }

// Two nibble bytes (the low or high half of w) as exact 16-bit floats.
template <int DT, bool HI>
__device__ __forceinline__ uint32_t nibble_pair(uint32_t w) {
  if constexpr (DT == kBF16)
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 512.0f, HI));
  else
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 512.0f, HI));
}

// 8 codes of one word (4 bits) as exact 16-bit floats in K order.
template <int DT>
__device__ __forceinline__ u32x4 exact_u4(uint32_t w) {
  const uint32_t a = w & 0x0F0F0F0Fu;         // codes 0 2 4 6
  const uint32_t b = (w >> 4) & 0x0F0F0F0Fu;  // codes 1 3 5 7
  const uint32_t lo = __builtin_amdgcn_perm(b, a, 0x05010400u);  // codes 0 1 2 3
  const uint32_t hi = __builtin_amdgcn_perm(b, a, 0x07030602u);  // codes 4 5 6 7
  return (u32x4){nibble_pair<DT, false>(lo), nibble_pair<DT, true>(lo), nibble_pair<DT, false>(hi),
                 nibble_pair<DT, true>(hi)};
}

// 8 codes of two words (8 bits).
template <int DT>
__device__ __forceinline__ u32x4 exact_u8(uint32_t w0, uint32_t w1) {
  const u32x2 lo = unpack_u8<DT>(w0), hi = unpack_u8<DT>(w1);
  return codes_for_sum<DT>((u32x4){lo.x, lo.y, hi.x, hi.y});
}

template <int BITS, int DT, bool HALF, int TM, int WN, int NPROJ>
__global__ __launch_bounds__(64 * WN) __attribute__((amdgpu_waves_per_eu(2))) void
affine_wide_kernel(const WideParams args) {
  const WideParams p = preload_args(args);
  constexpr int BM = 32 * TM, BN = 32 * WN;
  constexpr int kABytes = BM * 128;
  constexpr int kALoads = kABytes / 1024;                 // 1 KiB each
  constexpr int kAPer = (kALoads + WN - 1) / WN;
  constexpr int kCodeWords = BITS;                        // a lane's codes of a column and step
  constexpr int kCodeLoads = HALF ? 4 : BITS / 4;         // and the loads that bring them
  constexpr int kPer = kAPer + kCodeLoads;                // loads per wave and step
  constexpr int kRows = BN / NPROJ;                       // code columns of one projection
  constexpr int kSecLoads = (kRows * kSbDwords + 63) / 64;  // 256-byte loads per scale section
  constexpr int kSecBytes = kSecLoads * 256;
  constexpr int kSbLoads = 2 * NPROJ * kSecLoads;         // s of each projection, then b
  constexpr int kSbPer = (kSbLoads + WN - 1) / WN;
  constexpr int kBlocks = BM / 16;                        // 16-row blocks of the row sums
  constexpr int kBlocksPer = (kBlocks + WN - 1) / WN;
  constexpr int kGroupsPerStep = HALF ? 2 : 1;
  // Steps in flight: stages of activations (LDS) and of codes (registers), four, or eight where few
  // rows leave room: there the time is memory latency.
  constexpr int DA = TM == 1 ? 8 : 4, DC = TM <= 2 ? 8 : 4;
  constexpr int kUnroll = DC;

  __shared__ __attribute__((aligned(1024))) unsigned char A0[kABytes], A1[kABytes], A2[kABytes],
      A3[kABytes];
  constexpr int kMore = DA == 8 ? kABytes : 1024;
  __shared__ __attribute__((aligned(1024))) unsigned char A4[kMore], A5[kMore], A6[kMore], A7[kMore];
  __shared__ __attribute__((aligned(256))) unsigned char SB0[2 * NPROJ * kSecBytes],
      SB1[2 * NPROJ * kSecBytes];
  __shared__ __attribute__((aligned(16))) unsigned char XS[BM * kXsStride];
  __shared__ __attribute__((aligned(1024))) unsigned char spare[1024];  // surplus loads
  auto a_stage = [&](auto sc) -> unsigned char* {
    constexpr int S = decltype(sc)::value % DA;
    if constexpr (S == 0) return A0;
    else if constexpr (S == 1) return A1;
    else if constexpr (S == 2) return A2;
    else if constexpr (S == 3) return A3;
    else if constexpr (S == 4) return A4;
    else if constexpr (S == 5) return A5;
    else if constexpr (S == 6) return A6;
    else return A7;
  };
  auto sb_stage = [&](auto pc) -> unsigned char* {
    if constexpr (decltype(pc)::value == 0) return SB0;
    else return SB1;
  };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;    // MFMA 32x32x16: column (or row) and K half
  const int i16 = lane & 15, g4 = lane >> 4;  // MFMA 16x16x32
  const int M = p.M, K = p.K, N = p.N;

  // Workgroup -> (column tile, row tile, split). Workgroups go to the 8 XCDs in turn; each XCD
  // takes a contiguous run of the tiles, which lie in bands of 8 row tiles with the rows fastest,
  // so that an L2 serves a compact block of rows and columns.
  const int tiles_n = (N * NPROJ + BN - 1) / BN, tiles_m = (M + BM - 1) / BM;
  const int tiles = tiles_n * tiles_m;
  int bx, by, bz, tile;
  {
    const int total = gridDim.x, lin = blockIdx.x, k = lin & 7;
    const int item = k * (total >> 3) + min(k, total & 7) + (lin >> 3);
    bz = item / tiles;
    tile = item - bz * tiles;
    const int band = tile / (8 * tiles_n), rem = tile - band * 8 * tiles_n;
    const int rb = min(8, tiles_m - 8 * band);
    bx = rem / rb;
    by = 8 * band + rem - bx * rb;
  }
  const int m0 = by * BM, n0 = bx * kRows;
  const int gshift = p.group_shift;
  const int gpr = K >> gshift;
  const int s_beg = bz * p.steps_per_split;
  const int s_end = min(K >> 6, s_beg + p.steps_per_split);
  const int g_beg = (s_beg << 6) >> gshift;
  const uint32_t sbbytes = (uint32_t)N * (uint32_t)gpr * 2u;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, (uint32_t)M * (uint32_t)K * 2u);
  const uint64_t s0 = uniform_bits(p.s[0]), b0 = uniform_bits(p.b[0]);
  const uint64_t s1 = NPROJ == 2 ? uniform_bits(p.s[1]) : s0;
  const uint64_t b1 = NPROJ == 2 ? uniform_bits(p.b[1]) : b0;

  // ---- load addresses. Activation load d fills LDS rows 8 d .. 8 d + 7, lane l slot l % 8 of
  // row l / 8. Rows past M (and surplus loads) read zero.
  uint32_t a_src[kAPer];
#pragma unroll
  for (int i = 0; i < kAPer; ++i) {
    const int d = wave + WN * i;
    const int r = 8 * d + (lane >> 3);
    const int c = (lane & 7) ^ swz(r);
    a_src[i] = oob_unless(d < kALoads && m0 + r < M,
                          ((uint32_t)(m0 + r) * (uint32_t)K + 8u * c) * 2u);
  }
  // This lane's column: one of 32 of a projection, or (SwiGLU) 16 of each projection in the wave's
  // rows of 16 lanes. Its codes go straight to the registers of the two lanes that multiply them (no
  // other wave reads them): lane half h takes K 32 h .. of a step. Columns past N and steps past the
  // end read another column's or step's codes, which meet no output and no scale.
  const int proj = NPROJ == 2 ? j >> 4 : 0;
  const int srow = NPROJ == 2 ? 16 * wave + i16 : 32 * wave + j;
  const uint32_t c_src =
      (uint32_t)min(n0 + srow, N - 1) * p.col_stride + (HALF ? 8u : 4u * BITS) * h;
  const unsigned char* const c_base =  // SwiGLU: its own projection
      reinterpret_cast<const unsigned char*>(proj ? p.w[1] : p.w[0]) + c_src;
  uint32_t cw[DC][kCodeWords];  // codes of the steps in flight, by stage
  const uint32_t wbytes = wide_code_bytes(N, K, BITS);
  // Steps past the end load the last one again (unused).
  auto issue_a = [&](int st, auto sc) {
    const uint32_t at = (uint32_t)min(st, s_end - 1);
    unsigned char* as = a_stage(sc);
#pragma unroll
    for (int i = 0; i < kAPer; ++i) {
      const int d = wave + WN * i;
      unsigned char* to = kALoads % WN == 0 || d < kALoads ? as + d * 1024 : spare;
      load_lds16(rx, to, a_src[i], at * 128u);
    }
  };
  auto issue_codes = [&](int st, auto sc) {
    const uint32_t step_off = (uint32_t)min(st, s_end - 1) * p.step_stride;
    uint32_t(&to)[kCodeWords] = cw[decltype(sc)::value % DC];
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w[0], wbytes);
    constexpr int kWords = kCodeWords / kCodeLoads;  // 4, or 2 for groups of 32
#pragma unroll
    for (int e = 0; e < kCodeLoads; ++e) {
      if constexpr (kWords == 2) {
        u32x2 v;
        if constexpr (NPROJ == 2)
          v = *(const __attribute__((address_space(1))) u32x2*)((global_ptr_t)c_base + step_off +
                                                                16 * e);
        else
          v = __builtin_amdgcn_raw_buffer_load_b64(rw, c_src + 16u * e, step_off, 0);
        to[2 * e] = v.x; to[2 * e + 1] = v.y;
      } else {
        u32x4 v;
        if constexpr (NPROJ == 2)
          v = *(const __attribute__((address_space(1))) u32x4*)((global_ptr_t)c_base + step_off +
                                                                16 * e);
        else
          v = __builtin_amdgcn_raw_buffer_load_b128(rw, c_src + 16u * e, step_off, 0);
        to[4 * e] = v.x; to[4 * e + 1] = v.y; to[4 * e + 2] = v.z; to[4 * e + 3] = v.w;
      }
    }
  };
  // The scales and biases of a chunk: sections s0, [s1,] b0, [b1], each kRows columns of 9 dwords,
  // from the even element at or below the column's first group. Dword q of a section is dword q % 9
  // of column q / 9; a wave's next load is 64 WN dwords on.
  auto issue_sb = [&](int chunk, auto pc) {
    unsigned char* to = sb_stage(pc);
    int l = lane;
    __asm__ volatile("" : "+v"(l));  // addresses made here each time: kept, they cost 18 registers
    const uint32_t g0 = (uint32_t)g_beg + 16u * (uint32_t)chunk;
#pragma unroll
    for (int i = 0; i < kSbPer; ++i) {
      const int d = wave + WN * i;
      const int sec = d / kSecLoads;
      const uint64_t base = NPROJ == 1 ? (sec == 0 ? s0 : b0)
                                       : sec == 0 ? s0 : sec == 1 ? s1 : sec == 2 ? b0 : b1;
      const __amdgpu_buffer_rsrc_t r = make_rsrc(reinterpret_cast<const void*>(base), sbbytes);
      const int q = (d - sec * kSecLoads) * 64 + l;
      const int row = (q * 7282) >> 16;  // q / 9 for q < 4096
      const int n = n0 + row;
      const uint32_t first = ((uint32_t)n * (uint32_t)gpr + g0) & ~1u;
      const uint32_t off = oob_unless(d < kSbLoads && row < kRows && n < N,
                                      (first + 2u * (uint32_t)(q - 9 * row)) * 2u);
      unsigned char* dst = kSbLoads % WN == 0 || d < kSbLoads ? to + d * 256 : spare;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)dst, 4, off, 0, 0, 0);
    }
  };

  // Its first group in the staged scales; the bias sections follow the scales'.
  const uint32_t s_off = (uint32_t)(proj * kSecBytes + srow * (4 * kSbDwords)) +
                         2u * (((uint32_t)(n0 + srow) * (uint32_t)gpr + (uint32_t)g_beg) & 1u);
  constexpr uint32_t kBiasOff = (uint32_t)(NPROJ * kSecBytes);
  constexpr uint32_t kOnes = DT == kBF16 ? 0x3F803F80u : 0x3C003C00u;

  f32x16 acc[TM], t[2], th[2];  // t: two row tiles' chains; th: groups of 32, the second group's
  f32x16 zero16;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero16[r] = 0.0f;
#pragma unroll
  for (int a = 0; a < TM; ++a) acc[a] = zero16;
  t[0] = t[1] = th[0] = th[1] = zero16;
  f32x4 xsum[kBlocksPer];
#pragma unroll
  for (int i = 0; i < kBlocksPer; ++i) xsum[i] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // MFMA e of a chain takes K chunk kc(e) of the step (8 K) in lane half h: 4 h + e, or with groups
  // of 32 2 e + h (MFMAs 0, 1 the first group, 2, 3 the second).
  uint32_t a_off[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    a_off[e] = (uint32_t)(j * 128 + 16 * ((HALF ? 2 * e + h : 4 * h + e) ^ swz(j)));
  auto read_a = [&](auto sc, int a, u32x4 (&f)[4]) {
    const unsigned char* as = a_stage(sc) + 4096 * a;
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = *reinterpret_cast<const u32x4*>(as + a_off[e]);
  };
  // MFMA operand e (8 K) of a column's codes.
  auto unpack = [&](const uint32_t (&w)[kCodeWords], int e) -> u32x4 {
    if constexpr (BITS == 4) return exact_u4<DT>(w[e]);
    else return exact_u8<DT>(w[2 * e], w[2 * e + 1]);
  };
  auto sync = [&]() {
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- prologue: the first scales and four steps in flight, then the first operands ------------
  issue_sb(0, IntConst<0>{});
  auto each = [&](auto&& self, auto ic, auto&& f) {
    constexpr int I = decltype(ic)::value;
    f(ic);
    if constexpr (I + 1 < kUnroll) self(self, IntConst<I + 1>{}, f);
  };
  each(each, IntConst<0>{}, [&](auto ic) {
    if constexpr (decltype(ic)::value < DC - DA) issue_codes(s_beg + decltype(ic)::value, ic);
  });
  each(each, IntConst<0>{}, [&](auto ic) {
    constexpr int I = decltype(ic)::value;
    if constexpr (I < DA) {
      __builtin_amdgcn_sched_barrier(0);
      issue_a(s_beg + I, ic);
      issue_codes(s_beg + I + DC - DA, IntConst<I + DC - DA>{});
    }
  });
  // In flight behind the first step's loads: the other stages'. Within a step the scheduler orders
  // loads as it likes (they write different memory), so a wait counts whole steps only.
  wait_vmcnt<(DA - 1) * kPer>();
  sync();
  u32x4 af[2][4], bf[2][4];
  read_a(IntConst<0>{}, 0, af[0]);
#pragma unroll
  for (int e = 0; e < 4; ++e) bf[0][e] = unpack(cw[0], e);

  float sc_cur[kGroupsPerStep], sc_prev[kGroupsPerStep];
#pragma unroll
  for (int q = 0; q < kGroupsPerStep; ++q) sc_cur[q] = sc_prev[q] = 0.0f;

  // acc of row tile a gets the scaled sums that lie in buffer u.
  auto fix = [&](int a, int u, const float (&sc)[kGroupsPerStep]) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[a][r] = __builtin_fmaf(sc[0], t[u][r], acc[a][r]);
      if constexpr (HALF) acc[a][r] = __builtin_fmaf(sc[kGroupsPerStep - 1], th[u][r], acc[a][r]);
    }
    pin(acc[a]);  // left free, these sums sink past the next branch and keep every chain alive
  };

  // Step st (stage S, its position `i` in the chunk); `burst`: the next chunk's scales were
  // requested at the chunk's first step.
  auto step = [&](auto sc, auto pc, int st, int i, bool burst, int chunk) {
    constexpr int S = decltype(sc)::value;
    const unsigned char* sb = sb_stage(pc);
    const int gl = HALF ? 2 * i : (i << 6) >> gshift;  // the step's group within the chunk
#pragma unroll
    for (int q = 0; q < kGroupsPerStep; ++q) {
      sc_prev[q] = sc_cur[q];
      const float v = act_to_f32<DT>(*reinterpret_cast<const uint16_t*>(sb + s_off + 2 * (gl + q)));
      sc_cur[q] = st < s_end ? v : 0.0f;  // a step past the end has no scale of its own
    }
    // Row sums of this wave's 16-row blocks, into result column gl.
#pragma unroll
    for (int i2 = 0; i2 < kBlocksPer; ++i2) {
      const int rb = wave + WN * i2;
      if (kBlocks % WN == 0 || rb < kBlocks) {
        const int row = 16 * rb + i16;
        const unsigned char* as = a_stage(sc) + row * 128;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const u32x4 f = *reinterpret_cast<const u32x4*>(as + 16 * ((4 * kk + g4) ^ swz(row)));
          const uint32_t one = i16 == (st < s_end ? gl + (HALF ? kk : 0) : -1) ? kOnes : 0u;
          xsum[i2] = mfma16<DT>(f, (u32x4){one, one, one, one}, xsum[i2]);
        }
      }
    }
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      const int fa = (S * TM + a) & 1;  // buffers of this row tile's operands and chain
      if (a + 1 < TM) {
        read_a(sc, a + 1, af[fa ^ 1]);
      } else {
        // Every operand of this step is in registers (or arrives at the wait below): the stage may
        // be refilled behind the barrier, and the next step's stage is complete there.
        constexpr int kBehind = (DA - 2) * kPer;  // issued in the steps since the next one's
        if (S > 0 && S < DA - 1 && burst) wait_vmcnt<kBehind + kSbPer>();
        else wait_vmcnt<kBehind>();
        sync();
        if (S == 0 && burst) issue_sb(chunk + 1, IntConst<1 - decltype(pc)::value>{});
        issue_a(st + DA, sc);
        issue_codes(st + DC, sc);
        read_a(IntConst<S + 1>{}, 0, af[fa ^ 1]);
      }
      // The chain of row tile a, beside it the scaled sums of the tile before and a share of the next
      // step's codes.
      const int u = fa;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (HALF && e >= 2)
          th[u] = mfma32<DT>(af[fa][e], bf[S & 1][e], e == 2 ? zero16 : th[u]);
        else
          t[u] = mfma32<DT>(af[fa][e], bf[S & 1][e], e == 0 ? zero16 : t[u]);
      }
      if (a > 0) fix(a - 1, u ^ 1, sc_cur);
      else fix(TM - 1, u ^ 1, sc_prev);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e * TM / 4 == a) bf[(S & 1) ^ 1][e] = unpack(cw[(S + 1) % DC], e);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);  // the next operands' reads,
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA,
        __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);  // then seven VALU
      }
    }
  };

  // acc += sum over the chunk's groups of b X: the row sums as three bf16 parts through LDS.
  auto bias = [&](auto pc, int groups) {
    const unsigned char* sb = sb_stage(pc);
#pragma unroll
    for (int i2 = 0; i2 < kBlocksPer; ++i2) {
      const int rb = wave + WN * i2;
      if (kBlocks % WN == 0 || rb < kBlocks) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = xsum[i2][r];
          const uint32_t hi = f32_to_act<kBF16>(v);
          const float r1 = v - act_to_f32<kBF16>(hi);
          const uint32_t mid = f32_to_act<kBF16>(r1);
          const uint32_t lo = f32_to_act<kBF16>(r1 - act_to_f32<kBF16>(mid));
          *reinterpret_cast<u32x2*>(XS + (16 * rb + 4 * g4 + r) * kXsStride + 8 * i16) =
              (u32x2){hi | (mid << 16), lo};
        }
      }
      xsum[i2] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    sync();
    constexpr int kParts = DT == kBF16 ? 1 : 2;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (4 * q >= groups) break;
      u32x4 bb[kParts];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int gi = 4 * q + 2 * h + e;
        uint32_t v = *reinterpret_cast<const uint16_t*>(sb + s_off + kBiasOff + 2 * gi);
        v = gi < groups ? v : 0u;  // past the chunk's groups another column's
        if constexpr (DT == kBF16) {
          bb[0][2 * e] = v | (v << 16);
          bb[0][2 * e + 1] = v;
        } else {
          const float f = act_to_f32<kF16>(v);
          const uint32_t bh = f32_to_act<kBF16>(f);
          const uint32_t bl = f32_to_act<kBF16>(f - act_to_f32<kBF16>(bh));
          bb[0][2 * e] = bh | (bh << 16);
          bb[0][2 * e + 1] = bh;
          bb[kParts - 1][2 * e] = bl | (bl << 16);
          bb[kParts - 1][2 * e + 1] = bl;
        }
      }
#pragma unroll
      for (int a = 0; a < TM; ++a) {
        const u32x4 xa = *reinterpret_cast<const u32x4*>(XS + (32 * a + j) * kXsStride +
                                                         16 * (2 * q + h));
#pragma unroll
        for (int k = 0; k < kParts; ++k) acc[a] = mfma32<kBF16>(xa, bb[k], acc[a]);
      }
    }
  };

  // ---- K loop: chunks of 16 groups, four steps an iteration -------------------------------------
  const int nsteps = s_end - s_beg;
  const int chunk_steps = HALF ? 8 : 1 << (gshift - 2);  // 16 G / 64
  const int chunks = (nsteps + chunk_steps - 1) / chunk_steps;
  auto run_chunk = [&](int chunk, auto pc) {
    const int first = chunk * chunk_steps;
    const int count = min(chunk_steps, nsteps - first);
#pragma clang loop unroll(disable)
    for (int i = 0; i < count; i += kUnroll) {
      const bool burst = i == 0 && chunk + 1 < chunks;
      const int st = s_beg + first + i;
      each(each, IntConst<0>{}, [&](auto ic) {
        constexpr int I = decltype(ic)::value;
        // Half an iteration may be the last (only where K ends).
        if (I < 4 || i + 4 < count) step(ic, pc, st + I, i + I, burst, chunk);
      });
    }
    bias(pc, min(16, HALF ? 2 * count : ((count << 6) + (1 << gshift) - 1) >> gshift));
  };
  for (int chunk = 0; chunk < chunks; chunk += 2) {
    run_chunk(chunk, IntConst<0>{});
    if (chunk + 1 < chunks) run_chunk(chunk + 1, IntConst<1>{});
  }
  fix(TM - 1, 1, sc_cur);

  // ---- split K: a wave leaves its accumulators as they lie in its registers (16-byte
  // device-coherent stores, 1 KiB contiguous each); of a tile's and wave's splits the last to
  // arrive adds all in split order, so the sum does not depend on the order of arrival. -----------
  if (p.ksplit > 1) {
    constexpr uint32_t kWaveBytes = BM * 32 * 4;
    const uint32_t slot = (uint32_t)tile * WN + (uint32_t)wave;
    const uint32_t split_bytes = (uint32_t)tiles * WN * kWaveBytes;
    const __amdgpu_buffer_rsrc_t rp = make_rsrc(p.partial, (uint32_t)p.ksplit * split_bytes);
    auto part = [&](int sp, int a, int q) {
      return (uint32_t)sp * split_bytes + slot * kWaveBytes + (uint32_t)(a * 4 + q) * 1024u +
             (uint32_t)lane * 16u;
    };
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = (f32x4){acc[a][4 * q], acc[a][4 * q + 1], acc[a][4 * q + 2],
                                acc[a][4 * q + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rp, part(bz, a, q), 0,
                                               kDeviceScope);
      }
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    unsigned prev = 0;
    if (lane == 0)
      prev = __hip_atomic_fetch_add(&p.counters[slot], 1u, __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
    prev = __builtin_amdgcn_readfirstlane(prev);
    if (prev != (unsigned)(p.ksplit - 1)) return;
    if (lane == 0)
      __hip_atomic_store(&p.counters[slot], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __asm__ volatile("" ::: "memory");
    // One row tile's parts of two splits requested at a time (its own part too: it is in the cache
    // hierarchy).
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      u32x4 v[2][4];
      auto fetch = [&](int sp, u32x4 (&d)[4]) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          d[q] = load16_device(rp, oob_unless(sp < p.ksplit, part(sp, a, q)));
      };
      auto add = [&](int sp, const u32x4 (&d)[4]) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 x = __builtin_bit_cast(f32x4, d[q]);
#pragma unroll
          for (int r = 0; r < 4; ++r)
            acc[a][4 * q + r] = sp == 0 ? x[r] : acc[a][4 * q + r] + x[r];
        }
      };
      fetch(0, v[0]);
      for (int sp = 0; sp < p.ksplit; sp += 2) {
        fetch(sp + 1, v[1]);
        add(sp, v[0]);
        fetch(sp + 2, v[0]);
        if (sp + 1 < p.ksplit) add(sp + 1, v[1]);
      }
    }
  }

  // ---- output: neighbouring lanes exchange a value, so that a lane holds two adjacent columns of
  // one row and stores 4 bytes --------------------------------------------------------------------
  const __amdgpu_buffer_rsrc_t ry = make_rsrc(p.y, (uint32_t)M * (uint32_t)N * 2u);
  const __amdgpu_buffer_rsrc_t rr =
      make_rsrc(p.residual ? p.residual : p.y, p.residual ? (uint32_t)M * (uint32_t)N * 2u : 0u);
  const bool odd = lane & 1;
  constexpr int kPuts = NPROJ == 1 ? 8 : 4;  // stores of a row tile
#pragma unroll
  for (int a = 0; a < TM; ++a) {
    uint32_t off[kPuts], res[kPuts];
#pragma unroll
    for (int q = 0; q < kPuts; ++q) {
      const int row = m0 + 32 * a + (NPROJ == 1 ? mfma32_row(2 * q, h) + (odd ? 1 : 0)
                                                : mfma32_row(4 * q, h) + ((lane >> 4) & 1) +
                                                      (odd ? 2 : 0));
      const int col = n0 + (NPROJ == 1 ? 32 * wave + (j & ~1) : 16 * wave + (i16 & ~1));
      off[q] = oob_unless(row < M && col < N,
                          ((uint32_t)row * (uint32_t)N + (uint32_t)col) * 2u);
    }
    if (p.residual) {
#pragma unroll
      for (int q = 0; q < kPuts; ++q) res[q] = load4(rr, off[q]);
    }
#pragma unroll
    for (int q = 0; q < kPuts; ++q) {
      // This lane's values for the row that even lanes store and for the one that odd lanes store.
      float even_v, odd_v;
      if constexpr (NPROJ == 1) {
        even_v = acc[a][2 * q];
        odd_v = acc[a][2 * q + 1];
      } else {
        even_v = swiglu_pair(acc[a][4 * q], acc[a][4 * q + 1]);
        odd_v = swiglu_pair(acc[a][4 * q + 2], acc[a][4 * q + 3]);
      }
      const float recv = dpp_read<kDppXor1>(odd ? even_v : odd_v);
      float lo = odd ? recv : even_v, hi = odd ? odd_v : recv;
      if (p.residual) {
        lo += lo16<DT>(res[q]);
        hi += hi16<DT>(res[q]);
      }
      __builtin_amdgcn_raw_buffer_store_b32(
          (uint32_t)f32_to_act<DT>(lo) | ((uint32_t)f32_to_act<DT>(hi) << 16), ry, off[q], 0, 0);
    }
  }
}

template <int BITS, int DT, bool HALF, int TM, int WN, int NPROJ>
hipError_t launch_one(const WideParams& p, hipStream_t stream) {
  constexpr int BM = 32 * TM, BN = 32 * WN;
  const int tiles = ((p.M + BM - 1) / BM) * ((p.N * NPROJ + BN - 1) / BN);
  affine_wide_kernel<BITS, DT, HALF, TM, WN, NPROJ><<<tiles * p.ksplit, 64 * WN, 0, stream>>>(p);
  return hipGetLastError();
}

template <int BITS, int DT, bool HALF, int TM, int NPROJ>
hipError_t launch_wn(const WideParams& p, hipStream_t stream) {
  switch (p.tile_n) {
    case 64: return launch_one<BITS, DT, HALF, TM, 2, NPROJ>(p, stream);
    case 128: return launch_one<BITS, DT, HALF, TM, 4, NPROJ>(p, stream);
    case 256: return launch_one<BITS, DT, HALF, TM, 8, NPROJ>(p, stream);
  }
  return hipErrorInvalidValue;
}

template <int BITS, int DT, bool HALF, int NPROJ>
hipError_t launch_tm(const WideParams& p, hipStream_t stream) {
  switch (p.tile_m) {
    case 32: return launch_wn<BITS, DT, HALF, 1, NPROJ>(p, stream);
    case 64: return launch_wn<BITS, DT, HALF, 2, NPROJ>(p, stream);
    case 96: return launch_wn<BITS, DT, HALF, 3, NPROJ>(p, stream);
    case 128: return launch_wn<BITS, DT, HALF, 4, NPROJ>(p, stream);
  }
  return hipErrorInvalidValue;
}

template <int BITS, int DT, bool HALF>
hipError_t launch_proj(const WideParams& p, int nproj, hipStream_t stream) {
  return nproj == 2 ? launch_tm<BITS, DT, HALF, 2>(p, stream)
                    : launch_tm<BITS, DT, HALF, 1>(p, stream);
}

}  // namespace

}  // namespace mt
