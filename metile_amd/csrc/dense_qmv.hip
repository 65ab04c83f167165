// Dense 16-bit small-batch projections for gfx950: the gate/up SwiGLU and the down projection
// with a residual epilogue (reference: metile/compiler/dense.py:193-381 with the typed
// epilogues of metile/codegen/msl_emitter.py:1098-1120,1218-1252).
//
// Weights are the native output-major [N, K] matrices. The kernel streams them exactly like
// the affine kernel (32-column strips, 64-wide K steps split over four waves, a register
// pipeline of whole K steps, 16-byte buffer loads), but the codes are already 16-bit floats,
// so each step is four MFMAs chained into the same accumulator and there is no per-step
// fix-up.
//
// Row invariance: the value of every output depends only on its own activation row and on an
// accumulation order fixed by (K, N): the K partition among splits and waves comes from
// (K, N) alone, every wave accumulates its steps in order through one MFMA chain, and the
// cross-wave and split-K sums run in a fixed order. Running a row alone or inside a batch
// therefore gives the same bits. The host dispatches up to 128 rows at a time: up to 32 rows run on
// the kernel with a K quarter a wave, more on the one with shared tiles (dense_tile_kernel).
#include "common.h"
#include "dense_qmv.h"

namespace mt {

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;

template <int NPROJ, int MT>
struct DStage {
  u32x4 w[NPROJ][4];  // 4 x 8 K of column j for each projection
  u32x4 x[MT][4];     // 4 x 8 K of row j of each 32-row tile
};

// The reference's typed SwiGLU epilogue: gate and up rounded to the activation type, then
// y = 1/(1+exp(|g|)), sig = g < 0 ? y : 1 - y, act = g*sig, out = act*u, each operation
// computed in fp32 and rounded to the activation type.
template <int DT>
__device__ __forceinline__ float round_act(float v) {
  return act_to_f32<DT>(f32_to_act<DT>(v));
}

template <int DT>
__device__ __forceinline__ uint16_t typed_swiglu(float g, float u) {
  const float left = round_act<DT>(g);
  const float right = round_act<DT>(u);
  const float e = round_act<DT>(expf(fabsf(left)));
  const float y = round_act<DT>(1.0f / round_act<DT>(1.0f + e));
  const float sig = left < 0.0f ? y : round_act<DT>(1.0f - y);
  const float act = round_act<DT>(left * sig);
  return f32_to_act<DT>(act * right);
}

// Activation tiles above 8 rows go through LDS (XLDS): lane j of an MFMA operand needs row
// j, so loading the operand directly touches 32 rows (32 cache lines, 32 bytes of each) per
// instruction; loaded 8 lanes per row instead, every instruction reads 8 whole 128-byte lines.
// Each wave stages its own tile of the step (wave-private, no barrier) and reads it back in the
// MFMA layout; the 16-byte chunk c of staged row r sits at slot c ^ (r % 8), so that the eight
// lanes of a read phase (rows r..r+7, one chunk) hit distinct banks. The operands, and so every
// MFMA and sum, are the same as with direct loads.

// LDS of one workgroup, 16-byte units: during the K loop each wave's staged activation tile
// (XLDS) and weight tile ([NPROJ][32 columns][8 chunks], the same swizzle); after it the
// cross-wave reduction buffer [kWaves][NPROJ][32][33] (fp32), in the same space.
template <int MT, int NPROJ, bool XLDS>
constexpr int dense_lds_units() {
  constexpr int per_wave = (XLDS ? MT * 32 * 8 : 0) + NPROJ * 32 * 8;
  constexpr int loop = kWaves * per_wave;
  constexpr int red = (kWaves * NPROJ * 32 * 33 + 3) / 4;
  return loop > red ? loop : red;
}

// Weights are read once, with the non-temporal hint (M = 1 MLP 25.0 -> 22.5 us).
template <int DT, int NPROJ, int STAGES, bool XLDS>
__global__ __launch_bounds__(kThreads, 2) void dense_qmv_kernel(const DenseParams args) {
  constexpr int MT = 1;  // 32-row tiles
  const DenseParams p = preload_args(args);  // all arguments in one batch of scalar loads
  constexpr int kXUnits = XLDS ? MT * 32 * 8 : 0;  // per wave
  constexpr int kWUnits = NPROJ * 32 * 8;          // per wave
  __shared__ __attribute__((aligned(16))) u32x4 smem[dense_lds_units<MT, NPROJ, XLDS>()];
  __shared__ int last_flag;
  auto red = reinterpret_cast<float (*)[NPROJ][32][33]>(smem);  // [kWaves][NPROJ][32][33]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31;
  const int h = lane >> 5;
  const int strip = blockIdx.x;
  const int split = blockIdx.y;
  const int K = p.K, N = p.N;
  const int M = p.M;
  const int steps_total = K >> 6;
  const int s_beg = split * p.steps_per_split;
  const int s_end = min(steps_total, s_beg + p.steps_per_split);
  const int per_wave = (s_end - s_beg + kWaves - 1) / kWaves;
  const int w_beg = s_beg + wave * per_wave;
  const int w_end = min(s_end, w_beg + per_wave);

  const uint32_t row_bytes = (uint32_t)K * 2u;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, (uint32_t)M * K * 2u);
  __amdgpu_buffer_rsrc_t rw[NPROJ];
#pragma unroll
  for (int pr = 0; pr < NPROJ; ++pr) rw[pr] = make_rsrc(p.w[pr], (uint32_t)N * row_bytes);
  // Weights are loaded 8 lanes per column like the staged activations: instruction e of a
  // projection reads columns 8 e + lane / 8 of the strip, chunk lane % 8 of each step, and the
  // wave reads them back from LDS as the MFMA B operand (column j, chunks 4 h + e).
  const uint32_t w_row = (uint32_t)(strip * 32 + (lane >> 3)) * row_bytes + 16u * (lane & 7);
  const uint32_t w_step8 = 8u * row_bytes;
  u32x4* const xs = smem + wave * (kXUnits + kWUnits);  // [MT * 32 rows][8]
  u32x4* const ws = xs + kXUnits;                        // [NPROJ][32 columns][8]
  // Direct operand loads: lane (j, h) reads row 32 rt + j, K [32 h, 32 h + 32) of each step.
  // Staged loads (XLDS): instruction e of row tile rt reads rows 32 rt + 8 e + lane / 8, chunk
  // lane % 8 (K [8 (lane % 8), +8)) of each step.
  uint32_t x_row[MT];
#pragma unroll
  for (int rt = 0; rt < MT; ++rt) {
    const int row = XLDS ? 32 * rt + (lane >> 3) : 32 * rt + j;
    x_row[rt] = row < M ? (XLDS ? ((uint32_t)row * K + 8u * (lane & 7)) * 2u
                                : ((uint32_t)row * K + 32u * h) * 2u)
                        : kOOB;
  }
  // XLDS: rows 8 e + lane / 8 of a tile are 8 apart per instruction, whatever M is.
  const uint32_t x_step8 = 8u * (uint32_t)K * 2u;

  DStage<NPROJ, MT> ring[STAGES];
  // Out-of-range offsets are set with oob_unless (x_row of a row past M already is), not
  // with selects: with selects the compiler could no longer count the ring's loads and waited
  // for nearly all of them before every step.
  auto load_stage = [&](DStage<NPROJ, MT>& S, int st) {
    const bool ok = st < w_end;
    const uint32_t woff = w_row + (uint32_t)st * 128u;
#pragma unroll
    for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t off = oob_unless(ok, woff + e * w_step8);
        S.w[pr][e] = load16_nt(rw[pr], off);
      }
#pragma unroll
    for (int rt = 0; rt < MT; ++rt) {
      const uint32_t xoff = x_row[rt] + (uint32_t)st * 128u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (XLDS) {
          // rows past M read zero: their offset is already out of range, and rows 8 e apart
          // past the end of x stay beyond the buffer's range
          const bool row_ok = 32 * rt + 8 * e + (lane >> 3) < M;
          S.x[rt][e] = load16(rx, oob_unless(ok && row_ok, xoff + (uint32_t)e * x_step8));
        } else {
          S.x[rt][e] = load16(rx, oob_unless(ok, xoff + 16u * e));
        }
      }
    }
  };
  // The ring is filled in stage order: the scheduler may not issue a later stage's loads
  // first, or the first step would wait for all of them (and the loop, whose wait counts also
  // cover its entry, for nearly every load in flight).
#pragma unroll
  for (int d = 0; d < STAGES; ++d) {
    load_stage(ring[d], w_beg + d);
    __builtin_amdgcn_sched_barrier(0);
  }

  f32x16 acc[NPROJ][MT];
#pragma unroll
  for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
    for (int rt = 0; rt < MT; ++rt) acc[pr][rt] = (f32x16){0};

  for (int s0 = w_beg; s0 < w_end; s0 += STAGES) {
#pragma unroll
    for (int d = 0; d < STAGES; ++d) {
      DStage<NPROJ, MT>& S = ring[d];
      if (s0 + d < w_end) {
        // Stage the step's tiles (slot of chunk c of row or column r: c ^ (r % 8)), then read
        // row or column j, chunks 4 h + e, back; the waits keep this step's reads after its
        // writes and ahead of the next step's writes.
        const int wr = lane >> 3, wc = lane & 7;
#pragma unroll
        for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
          for (int e = 0; e < 4; ++e) ws[(pr * 32 + 8 * e + wr) * 8 + (wc ^ wr)] = S.w[pr][e];
        if constexpr (XLDS) {
#pragma unroll
          for (int rt = 0; rt < MT; ++rt)
#pragma unroll
            for (int e = 0; e < 4; ++e) xs[(32 * rt + 8 * e + wr) * 8 + (wc ^ wr)] = S.x[rt][e];
        }
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        u32x4 b[NPROJ][4];
#pragma unroll
        for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
          for (int e = 0; e < 4; ++e) b[pr][e] = ws[(pr * 32 + j) * 8 + ((4 * h + e) ^ (j & 7))];
#pragma unroll
        for (int rt = 0; rt < MT; ++rt) {
          u32x4 a[4];
#pragma unroll
          for (int e = 0; e < 4; ++e)
            a[e] = XLDS ? xs[(32 * rt + j) * 8 + ((4 * h + e) ^ (j & 7))] : S.x[rt][e];
#pragma unroll
          for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[pr][rt] = mfma32<DT>(a[e], b[pr][e], acc[pr][rt]);
        }
        __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      load_stage(S, s0 + d + STAGES);
    }
  }

  // ---- per row tile: cross-wave reduction (fixed order), then epilogue or split-K -------
  const size_t plane = (size_t)M * N;
  __syncthreads();  // the reduction buffer reuses the other waves' staging space
#pragma unroll
  for (int rt = 0; rt < MT; ++rt) {
    if (rt > 0) __syncthreads();
#pragma unroll
    for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
      for (int r = 0; r < 16; ++r) red[wave][pr][mfma32_row(r, h)][j] = acc[pr][rt][r];
    __syncthreads();
    const int rows = min(32, M - 32 * rt);
    for (int o = tid; o < rows * 32; o += kThreads) {
      const int i = o >> 5, c = o & 31;
      const size_t oi = (size_t)(32 * rt + i) * N + strip * 32 + c;
#pragma unroll
      for (int pr = 0; pr < NPROJ; ++pr) {
        const float v = ((red[0][pr][i][c] + red[1][pr][i][c]) + red[2][pr][i][c]) +
                        red[3][pr][i][c];
        if (p.ksplit == 1) {
          // stash the full sum for the epilogue below
          red[0][pr][i][c] = v;
        } else {
          __hip_atomic_store(&p.partial[(size_t)(split * NPROJ + pr) * plane + oi], v,
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      if (p.ksplit == 1) {
        if constexpr (NPROJ == 2) {
          p.y[oi] = typed_swiglu<DT>(red[0][0][i][c], red[0][1][i][c]);
        } else {
          float out = round_act<DT>(red[0][0][i][c]);
          if (p.residual) out = out + act_to_f32<DT>(p.residual[oi]);
          p.y[oi] = f32_to_act<DT>(out);
        }
      }
    }
  }
  if (p.ksplit == 1) return;

  // ---- split-K handoff: see the affine kernel; partials and counter are agent-coherent ----
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const unsigned prev =
        __hip_atomic_fetch_add(&p.counters[strip], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_flag = (prev == (unsigned)(p.ksplit - 1));
  }
  __syncthreads();
  if (!last_flag) return;
  // A thread's outputs over every split, their loads requested in batches (sum_partials_multi)
  // rather than one round trip per output: one output at up to 8 rows (the instances without
  // staged activations), else up to 32 MT rows x 32 columns over the workgroup's threads.
  constexpr int kOuts = XLDS ? 32 * 32 * MT / kThreads : 1;
  const float* src[kOuts * NPROJ];
  float sum[kOuts * NPROJ];
#pragma unroll
  for (int u = 0; u < kOuts; ++u) {
    const int o = tid + u * kThreads;
    const size_t oi = (size_t)(o >> 5) * N + strip * 32 + (o & 31);
#pragma unroll
    for (int pr = 0; pr < NPROJ; ++pr)
      src[u * NPROJ + pr] = o < M * 32 ? p.partial + (size_t)pr * plane + oi : nullptr;
  }
  sum_partials_multi<kOuts * NPROJ>(src, (size_t)NPROJ * plane, p.ksplit, sum);
#pragma unroll
  for (int u = 0; u < kOuts; ++u) {
    const int o = tid + u * kThreads;
    if (o >= M * 32) break;
    const size_t oi = (size_t)(o >> 5) * N + strip * 32 + (o & 31);
    const float* v = sum + u * NPROJ;
    if constexpr (NPROJ == 2) {
      p.y[oi] = typed_swiglu<DT>(v[0], v[1]);
    } else {
      float out = round_act<DT>(v[0]);
      if (p.residual) out = out + act_to_f32<DT>(p.residual[oi]);
      p.y[oi] = f32_to_act<DT>(out);
    }
  }
  if (tid == 0)
    __hip_atomic_store(&p.counters[strip], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---- more than 32 rows: shared tiles ------------------------------------------------------
// A workgroup of four waves computes MT x 32 rows by a 32-column strip (of both projections), the
// whole K range of its split: every step's activations (MT x 4 KiB) and weights (4 KiB a projection)
// go from memory straight to LDS, once for all waves, in a ring of D steps with one barrier each. Wave
// w owns row tile w (MT = 2 with two projections: tile w % 2 of projection w / 2). With one K quarter
// a wave, as in the kernel above, every wave would need its own activations and weights staged, which
// left one step in flight a wave at 64 rows, and more rows had to read the weights again.
//
// The sums are those of the kernel above to the bit: each K quarter of the split is one MFMA chain
// from zero, in the same operand order, and the quarters are added in order.
//
// What bounds it: 2048 -> 8192 runs at the weights' rate from memory; more strips and rows, one
// workgroup a CU, at what that workgroup receives: about 20 bytes a clock, activations and weights
// together (a ring of six steps instead of three, or reading operands a step ahead, changed nothing; two
// workgroups a CU, the down projection's four splits, receive 31). Measured (MI355X, bf16, weights from
// memory, gate and up / down, us; before: a K quarter a wave, over 64 rows in two chunks): 2048 -> 8192 at
// 64 rows 18.6 / 14.4 -> 18.3 / 13.9, at 128 26.6 / 21.5 -> 21.6 / 21.8; 4096 -> 14336 at 100 rows 102 /
// 55 -> 72 / 45; 5120 -> 17408 at 100 rows 181 / 88 -> 113 / 79. The kernel before was the faster one for
// gate and up of 2048 -> 8192 at 33 rows (17.4 -> 18.9) and of 1536 -> 8960 at 128 (28.5 -> 29.7), and
// with 178 MB of weights left in the caches (5120 -> 17408, down, 100 rows: 70.9 -> 78.6).
// NT: weights read once, with the non-temporal hint; not where a second row chunk or a later launch of
// the call reads them again (5120 -> 17408 at 160 rows, 128 and 32, with the hint 201 / 133, without 186 /
// 125 us).
template <int DT, int MT, int NPROJ, int D, bool NT>
__global__ __launch_bounds__(kThreads, 2) void dense_tile_kernel(const DenseParams args) {
  const DenseParams p = preload_args(args);
  constexpr int kLoads = MT + NPROJ;  // per wave and step: 8 rows of every row tile and projection
  constexpr int kStage = kLoads * 4096;
  constexpr bool kPair = MT == 2 && NPROJ == 2;  // a wave has one projection of its tile
  constexpr int kOwn = kPair ? 1 : NPROJ;
  __shared__ __attribute__((aligned(1024))) unsigned char S0[kStage], S1[kStage], S2[kStage],
      S3[D > 3 ? kStage : 1024], S4[D > 4 ? kStage : 1024], S5[D > 5 ? kStage : 1024];
  auto stage = [&](auto sc) -> unsigned char* {
    constexpr int S = decltype(sc)::value % D;
    if constexpr (S == 0) return S0;
    else if constexpr (S == 1) return S1;
    else if constexpr (S == 2) return S2;
    else if constexpr (S == 3) return S3;
    else if constexpr (S == 4) return S4;
    else return S5;
  };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;
  const int K = p.K, N = p.N;
  // Workgroup -> (row chunk, strip, split). Workgroups go to the 8 XCDs in turn; each takes a
  // contiguous run with the chunks fastest, so that a strip's chunks meet its weights in one L2. (Dealt
  // out strip by strip, two projections 8192 -> 8192 at 64 rows took 74 us instead of 67.) Before a row
  // kernel's launch over the same weights the strips of one chunk are dealt out as there, and it finds
  // them in its XCD's L2: 1536 -> 8960 gate and up at 160 rows 44.7 -> 42.7 us.
  const int rc = p.row_chunk, chunks = rc ? (p.M + rc - 1) / rc : 1;
  int strip, split, chunk;
  {
    const int total = gridDim.x, lin = blockIdx.x, k = lin & 7, strips = N / 32;
    const int item = p.dealt ? lin : k * (total >> 3) + min(k, total & 7) + (lin >> 3);
    const int rest = item / chunks;
    chunk = item - rest * chunks;
    split = rest / strips;
    strip = rest - split * strips;
  }
  const int r0 = chunk * rc;
  const int M = rc ? min(rc, p.M - r0) : p.M;
  uint16_t* const y = p.y + (size_t)r0 * N;
  const uint16_t* const residual = p.residual ? p.residual + (size_t)r0 * N : nullptr;
  const int s_beg = split * p.steps_per_split;
  const int s_end = min(K >> 6, s_beg + p.steps_per_split);
  const int quarter = (s_end - s_beg + kWaves - 1) / kWaves;
  const int tile = kPair ? wave & 1 : wave;
  const int proj = kPair ? wave >> 1 : 0;

  // Load i of a wave brings rows 8 wave .. of row tile i, or columns 8 wave .. of projection i - MT:
  // lane l slot l % 8 of row l / 8, the slot of the 16-byte chunk c of row r being c ^ (r % 8).
  const int lr = 8 * wave + (lane >> 3), lc = (lane & 7) ^ (lane >> 3);
  const uint32_t row_bytes = (uint32_t)K * 2u;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x + (size_t)r0 * K, (uint32_t)M * row_bytes);
  uint32_t x_src[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
    x_src[i] = oob_unless(32 * i + lr < M, (uint32_t)(32 * i + lr) * row_bytes + 16u * lc);
  const uint32_t w_src = (uint32_t)(strip * 32 + lr) * row_bytes + 16u * lc;
  auto issue = [&](int st, auto sc) {  // steps past the end load the last one again (unused)
    const uint32_t at = (uint32_t)min(st, s_end - 1) * 128u;
    unsigned char* to = stage(sc) + 1024 * wave;
#pragma unroll
    for (int i = 0; i < MT; ++i) load_lds16(rx, to + 4096 * i, x_src[i], at);
#pragma unroll
    for (int pr = 0; pr < NPROJ; ++pr)
      load_lds16<NT ? kCachePolicyNt : 0>(make_rsrc(p.w[pr], (uint32_t)N * row_bytes),
                                          to + 4096 * (MT + pr), w_src, at);
  };

  f32x16 zero16;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero16[r] = 0.0f;
  f32x16 acc[kOwn], sum[kOwn];  // this quarter's chain, the quarters before it
#pragma unroll
  for (int q = 0; q < kOwn; ++q) acc[q] = sum[q] = zero16;
  uint32_t f_off[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) f_off[e] = (uint32_t)(j * 128 + 16 * ((4 * h + e) ^ (j & 7)));
  int boundary = s_beg + quarter;

  auto step = [&](auto sc, int st) {
    constexpr int S = decltype(sc)::value;
    // This step's loads done (behind them the D - 2 younger steps'), and every wave past its reads of
    // the stage that is refilled.
    wait_vmcnt<(D - 2) * kLoads>();
    __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    issue(st + D - 1, IntConst<(S + D - 1) % D>{});
    __builtin_amdgcn_sched_barrier(0);
    if (st >= s_beg && (MT == 4 || kPair || tile < MT)) {
      const unsigned char* xs = stage(sc) + 4096 * tile;
      const unsigned char* ws = stage(sc) + 4096 * (MT + proj);
      u32x4 a[4], b[kOwn][4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[e] = *reinterpret_cast<const u32x4*>(xs + f_off[e]);
#pragma unroll
        for (int q = 0; q < kOwn; ++q)
          b[q][e] = *reinterpret_cast<const u32x4*>(ws + 4096 * q + f_off[e]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int q = 0; q < kOwn; ++q) acc[q] = mfma32<DT>(a[e], b[q][e], acc[q]);
      __builtin_amdgcn_sched_group_barrier(0x100, 4 + 4 * kOwn, 0);  // every operand's read,
      __builtin_amdgcn_sched_group_barrier(0x008, 4 * kOwn, 0);      // then the MFMAs
    }
    if (st + 1 == boundary) {
#pragma unroll
      for (int q = 0; q < kOwn; ++q) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[q][r] += acc[q][r];
        acc[q] = zero16;
      }
      boundary += quarter;
    }
  };
  // The first D - 1 positions only fill the ring (loads issued outside the loop made the compiler wait
  // for all of them at its head). Left as soon as the steps end: were later positions skipped instead,
  // the compiler would have to assume a stage refilled one step before it is read.
  for (int st = s_beg - (D - 1);;) {
    step(IntConst<0>{}, st);
    if (++st == s_end) break;
    step(IntConst<1>{}, st);
    if (++st == s_end) break;
    step(IntConst<2>{}, st);
    if (++st == s_end) break;
    if constexpr (D > 3) {
      step(IntConst<3>{}, st);
      if (++st == s_end) break;
    }
    if constexpr (D > 4) {
      step(IntConst<4>{}, st);
      if (++st == s_end) break;
    }
    if constexpr (D > 5) {
      step(IntConst<5>{}, st);
      if (++st == s_end) break;
    }
  }
#pragma unroll
  for (int q = 0; q < kOwn; ++q)
#pragma unroll
    for (int r = 0; r < 16; ++r) sum[q][r] += acc[q][r];
  // No load may still be on its way to LDS when it changes hands (to the exchange below, or, behind
  // the last wave's end, to another workgroup).
  wait_vmcnt<0>();

  const int row0 = 32 * tile;
  if (p.ksplit > 1) {
    // [split][projection][M][N] partial sums, device-coherent.
    const uint32_t plane = (uint32_t)M * (uint32_t)N * 4u;
    const char* const parts = reinterpret_cast<const char*>(p.partial) +
                              (size_t)chunk * p.ksplit * NPROJ * rc * N * 4;
    uint32_t* const counter = p.counters + (size_t)chunk * (N / 32) + strip;
    auto part = [&](int sp) {
      return make_rsrc(parts + (size_t)sp * NPROJ * plane, NPROJ * plane);
    };
    if (MT == 4 || kPair || tile < MT) {
      const __amdgpu_buffer_rsrc_t to = part(split);
#pragma unroll
      for (int q = 0; q < kOwn; ++q)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = row0 + mfma32_row(r, h);
          const float v = sum[q][r];
          __builtin_amdgcn_raw_buffer_store_b32(
              __float_as_uint(v), to,
              oob_unless(row < M, (uint32_t)(proj + q) * plane +
                                      ((uint32_t)row * (uint32_t)N + strip * 32 + j) * 4u),
              0, kDeviceScope);
        }
    }
    // ---- split-K handoff: as in the kernel above (its flag in the first stage) ----
    int& last_flag = *reinterpret_cast<int*>(S0);
    __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const unsigned prev = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
      last_flag = (prev == (unsigned)(p.ksplit - 1));
    }
    __syncthreads();
    if (!last_flag) return;
    // Thread: four columns of one row of every row tile, two splits requested at a time (past the last
    // split zeros are read: the sums, which start from +0, stay as they are).
    const int row = tid >> 3, col = strip * 32 + 4 * (tid & 7);
    f32x4 v[NPROJ][MT];
#pragma unroll
    for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
      for (int i = 0; i < MT; ++i) v[pr][i] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int sp = 0; sp < p.ksplit; sp += 2) {
      u32x4 q[2][NPROJ][MT];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const __amdgpu_buffer_rsrc_t from = part(min(sp + u, p.ksplit - 1));
#pragma unroll
        for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
          for (int i = 0; i < MT; ++i)
            q[u][pr][i] = load16_device(
                from, oob_unless(sp + u < p.ksplit && 32 * i + row < M,
                                 pr * plane + ((uint32_t)(32 * i + row) * N + col) * 4u));
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int pr = 0; pr < NPROJ; ++pr)
#pragma unroll
          for (int i = 0; i < MT; ++i) v[pr][i] += __builtin_bit_cast(f32x4, q[u][pr][i]);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      if (32 * i + row >= M) break;
      const size_t oi = (size_t)(32 * i + row) * N + col;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if constexpr (NPROJ == 2) {
          y[oi + c] = typed_swiglu<DT>(v[0][i][c], v[1][i][c]);
        } else {
          float out = round_act<DT>(v[0][i][c]);
          if (residual) out = out + act_to_f32<DT>(residual[oi + c]);
          y[oi + c] = f32_to_act<DT>(out);
        }
      }
    }
    if (tid == 0)
      __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }

  // ---- output: neighbouring lanes exchange a value, so that a lane holds two adjacent columns of one
  // row and stores 4 bytes ----
  f32x16 up = zero16;
  if constexpr (NPROJ == 2 && !kPair) up = sum[kOwn - 1];
  if constexpr (kPair) {  // the up projection's wave hands its sums over (16 KiB, the first stage)
    f32x4* const ex = reinterpret_cast<f32x4*>(S0) + tile * 256 + lane;
    __syncthreads();
    if (proj == 1) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        ex[64 * q] = (f32x4){sum[0][4 * q], sum[0][4 * q + 1], sum[0][4 * q + 2],
                             sum[0][4 * q + 3]};
    }
    __syncthreads();
    if (proj == 1) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 v = ex[64 * q];
#pragma unroll
      for (int r = 0; r < 4; ++r) up[4 * q + r] = v[r];
    }
  }
  if (!kPair && MT < 4 && tile >= MT) return;
  const bool odd = lane & 1;
  const __amdgpu_buffer_rsrc_t ry = make_rsrc(y, (uint32_t)M * (uint32_t)N * 2u);
  const __amdgpu_buffer_rsrc_t rr =
      make_rsrc(residual ? residual : y, residual ? (uint32_t)M * (uint32_t)N * 2u : 0u);
  uint32_t off[8], res[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int row = row0 + mfma32_row(2 * q, h) + (odd ? 1 : 0);
    off[q] = oob_unless(row < M,
                        ((uint32_t)row * (uint32_t)N + (uint32_t)(strip * 32 + (j & ~1))) * 2u);
  }
  if (residual) {
#pragma unroll
    for (int q = 0; q < 8; ++q) res[q] = load4(rr, off[q]);
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    float even_v, odd_v;  // this lane's values for the row even lanes store and the one odd lanes do
    if constexpr (NPROJ == 2) {
      even_v = act_to_f32<DT>(typed_swiglu<DT>(sum[0][2 * q], up[2 * q]));
      odd_v = act_to_f32<DT>(typed_swiglu<DT>(sum[0][2 * q + 1], up[2 * q + 1]));
    } else {
      even_v = round_act<DT>(sum[0][2 * q]);
      odd_v = round_act<DT>(sum[0][2 * q + 1]);
    }
    const float recv = dpp_read<kDppXor1>(odd ? even_v : odd_v);
    float lo = odd ? recv : even_v, hi = odd ? odd_v : recv;
    if (residual) {
      lo += lo16<DT>(res[q]);
      hi += hi16<DT>(res[q]);
    }
    __builtin_amdgcn_raw_buffer_store_b32(
        (uint32_t)f32_to_act<DT>(lo) | ((uint32_t)f32_to_act<DT>(hi) << 16), ry, off[q], 0, 0);
  }
}

// Register ring depth: the stages that fit beside the accumulators in the registers of one
// wave (256 at two workgroups per CU), with at most 60 loads in flight: the
// hardware counts at most 63 outstanding loads per wave, and a ring deeper than that count
// makes the compiler wait for almost every load before each step.
template <int NPROJ, int MT>
constexpr int dense_stages() {
  constexpr int per_stage = 16 * NPROJ + 16 * MT;
  constexpr int loads = 4 * NPROJ + 4 * MT;
  constexpr int budget = 112;  // ring registers beside the accumulators at two workgroups per CU
  constexpr int s = budget / per_stage < 60 / loads ? budget / per_stage : 60 / loads;
  return s < 1 ? 1 : (s > 4 ? 4 : s);
}

template <int DT, int NPROJ>
hipError_t launch_dense_rows(const DenseParams& p, dim3 grid, hipStream_t stream) {
  // Activations staged through LDS above 8 rows (at fewer rows most operand lanes read zero
  // and the direct loads touch few lines).
  constexpr int kStages = dense_stages<NPROJ, 1>();
  if (p.M <= 8)
    dense_qmv_kernel<DT, NPROJ, kStages, false><<<grid, kThreads, 0, stream>>>(p);
  else
    dense_qmv_kernel<DT, NPROJ, kStages, true><<<grid, kThreads, 0, stream>>>(p);
  return hipGetLastError();
}

// A ring of as many steps as leave room for two workgroups a CU, at most six.
constexpr int dense_ring(int mt, int nproj) {
  const int d = 80 / (4 * (mt + nproj));
  return d < 6 ? d : 6;
}

template <int DT, int NPROJ, int MT, bool NT>
hipError_t launch_dense_tile(const DenseParams& p, dim3 grid, hipStream_t stream) {
  dense_tile_kernel<DT, MT, NPROJ, dense_ring(MT, NPROJ), NT><<<grid, kThreads, 0, stream>>>(p);
  return hipGetLastError();
}

template <int DT, int NPROJ>
hipError_t launch_dense_dt(const DenseParams& p, hipStream_t stream) {
  const int tiles = p.N / 32 * p.ksplit;
  if (p.row_chunk)
    return launch_dense_tile<DT, NPROJ, 2, false>(
        p, dim3(tiles * ((p.M + p.row_chunk - 1) / p.row_chunk)), stream);
  switch ((p.M + 31) / 32) {
    case 1: return launch_dense_rows<DT, NPROJ>(p, dim3(p.N / 32, p.ksplit), stream);
    case 2: return launch_dense_tile<DT, NPROJ, 2, true>(p, dim3(tiles), stream);
    case 3: return launch_dense_tile<DT, NPROJ, 3, true>(p, dim3(tiles), stream);
    case 4:  // the only one that others follow
      return p.reread ? launch_dense_tile<DT, NPROJ, 4, false>(p, dim3(tiles), stream)
                      : launch_dense_tile<DT, NPROJ, 4, true>(p, dim3(tiles), stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_dense_qmv(const DenseParams& p, int dtype, int nproj, hipStream_t stream) {
  if (dtype == kBF16)
    return nproj == 2 ? launch_dense_dt<kBF16, 2>(p, stream) : launch_dense_dt<kBF16, 1>(p, stream);
  return nproj == 2 ? launch_dense_dt<kF16, 2>(p, stream) : launch_dense_dt<kF16, 1>(p, stream);
}

}  // namespace mt
