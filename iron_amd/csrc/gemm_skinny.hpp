// GEMM of few rows (M <= 48): C = epi(A . B^T) as a stream over the weights.
//
// At these M the weights are the traffic (13 x 2048 -> 3072: 12.6 MB against
// 0.13 MB of A and C). A workgroup owns 16 * NT output columns and all rows;
// its 8 waves split K into ranges of whole 128-deep units. Each wave streams
// the rows of A and B of its range through a ring of its own in LDS
// (load_lds16: 8 rows x 128 contiguous bytes per instruction), waits for its own
// loads only and reads the fragments of v_mfma_f32_16x16x32_bf16 from there: no
// barrier until the waves' fp32 sums meet in LDS, added in wave order. One or two
// stages are in flight per wave (launch_skinny_tile): with one, a stage is loaded
// once the LDS reads of the one before are done and waited for in full, which the
// other workgroups of the CU cover. (Fragments loaded straight into registers
// were limited by the address unit: four adjacent lanes then touch four rows,
// ~64 clocks per load instead of 16.)
//
// The tiled kernel pads M to 64 rows and needs a K split with a second (merge)
// launch to use the CUs; this one reads each weight once in one launch.
//
// The int4 form brings the codes (16 rows x 64 bytes per unit) and scales the
// same way and dequantizes in registers (dequant8: the tiled kernel's values).
// The form for a row-major B (K, N) stages 64 k-rows of 32 columns and reads
// its fragments with ds_read_b64_tr_b16, as the NN tiles do.
// The split of K and the order of the MFMAs and of the final sums depend on K
// only, so the int4 form, the plain form on the dequantized weights, the
// row-major form and the SwiGLU pair agree bit for bit, as the tiled kernels do.
#pragma once

namespace iron {
namespace {

constexpr int kSkinnyM = 48;      // rows this form takes
constexpr int kSkinnyWaves = 8;   // K ranges, one wave each
constexpr int kSkinnyUnit = 128;  // K granularity of the ranges

typedef float f32x4v __attribute__((ext_vector_type(4)));

enum SkinnyKind : int { SK_BF16 = 0, SK_I4 = 1, SK_PAIR = 2, SK_NN = 3 };

// One 64-deep (bf16) or 128-deep (int4) stage of a wave: MT blocks of 16 A
// rows, then the B rows. bf16 rows of 64 k: 128 bytes, chunk c at slot
// c ^ ((row / 2) % 8) (swz). int4: A as two such halves, then per 16 B rows
// 1 KiB of codes (64 bytes a row, chunk g at slot g ^ ((row / 4) % 4): the
// 4-byte reads of 16 rows hit distinct banks) and 256 bytes of scales.
// Row-major B: 64 k-rows of 64 bytes, chunk c at slot c ^ 2 ((row / 8) % 2): a
// transposing read serves 32 lanes per pass, 4 k-rows and the 4 that lie 8
// further on, 32 bytes each; rows r, r + 1, .. take a quarter of the banks in
// turn and the swizzle puts the two groups on its two halves.
template <int MT, int NT, int KIND>
struct SkinnyStage {
  static constexpr bool I4 = KIND == SK_I4;
  static constexpr int kDepth = I4 ? 128 : 64;
  static constexpr int kABytes = MT * 16 * kDepth * 2;
  static constexpr int kBytes = kABytes + (I4 ? NT * 1280 : NT * 16 * 128);
  static constexpr int kLoads = I4 ? 4 * MT + 2 * NT : 2 * (MT + NT);
};

template <int N>
__device__ __forceinline__ void wait_own_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// MT: 16-row tiles of M. NT: 16-column tiles (SK_PAIR: tile 0 gate, tile 1 up
// of the same 16 features; B rows alternate 64-row blocks of gate and up).
// D: stages in flight per wave (1 or 2). TR: traced instance (points 0 start, 5 stored).
template <int MT, int NT, int KIND, int D, bool TR>
__global__ __launch_bounds__(64 * kSkinnyWaves) void gemm_skinny_kernel(GemmArgs a) {
  using S = SkinnyStage<MT, NT, KIND>;
  constexpr int W = kSkinnyWaves;
  static_assert((KIND != SK_PAIR && KIND != SK_NN) || NT == 2, "a gate and an up tile; 64-byte k-rows");
  static_assert(D == 1 || D == 2, "the waits of the last stages");
  constexpr int COLS = 16 * NT, ROWS = 16 * MT;
  constexpr int LD = COLS + 1;  // padded row of the reduction buffer
  constexpr int kRing = D * S::kBytes, kRed = W * ROWS * LD * 4;
  constexpr int kLds = W * kRing > kRed ? W * kRing : kRed;
  static_assert(kLds <= 160 * 1024, "LDS budget");
  __shared__ u32x4v smem[kLds / 16];
  void* const trace = TR ? a.trace : nullptr;
  unsigned long long t_start = 0;
  if constexpr (TR) t_start = trace_clock();
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, q = lane >> 4;
  const int tile = xcd_tile(gridDim.x);
  const int c0 = tile * (KIND == SK_PAIR ? 16 : COLS);  // first output column
  unsigned char* const ring = reinterpret_cast<unsigned char*>(smem) + wave * kRing;

  const int units = (a.K + kSkinnyUnit - 1) / kSkinnyUnit;
  const int groups = a.K / 32;  // 32-deep MFMA steps, int4 groups of a row (an even number: K % 64 == 0)
  const int u0 = units * wave / W, u1 = units * (wave + 1) / W;
  // this wave's stages [s0, s1) of kDepth
  const int s0 = S::I4 ? u0 : 2 * u0, s1 = S::I4 ? u1 : min(2 * u1, a.K / 64);

  // Byte offsets of this lane's chunk of each load, from uniform bases (A, and
  // the tile's first row of B); rows past M or N repeat the last one (their
  // outputs are never stored).
  const int row0 = KIND == SK_PAIR ? (c0 >> 6) * 128 + (c0 & 63) : c0;  // F % 64 == 0: 16 features share a block
  const i32x4v rsrc_a = buffer_rsrc(a.A);
  const i32x4v rsrc_b = KIND == SK_NN ? buffer_rsrc(a.B)
                        : S::I4       ? buffer_rsrc(a.codes + static_cast<size_t>(row0) * (a.K / 2))
                                      : buffer_rsrc(a.B + static_cast<size_t>(row0) * a.K);
  const i32x4v rsrc_s = S::I4 ? buffer_rsrc(a.scales + static_cast<size_t>(row0) * groups) : rsrc_b;
  // 8 rows x 128 bytes per load: lane -> row lane / 8, slot lane % 8
  unsigned aoff[2 * MT], boff[2 * NT], soff[NT];
#pragma unroll
  for (int b = 0; b < 2 * MT; ++b) {
    const int r = b * 8 + (lane >> 3);
    aoff[b] = static_cast<unsigned>(min(r, a.M - 1)) * a.K * 2 + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
  }
#pragma unroll
  for (int b = 0; b < 2 * NT; ++b) {
    const int r = b * 8 + (lane >> 3);
    // a pair's second 16 rows are its up rows, 64 further on
    const int br = KIND == SK_PAIR ? (r & 15) + 64 * (r >> 4) : min(c0 + r, a.N - 1) - c0;
    boff[b] = static_cast<unsigned>(br) * a.K * 2 + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
    if (KIND == SK_NN) {  // 16 k-rows x 64 bytes; columns past N load the row's last 8 (N % 8 == 0)
      const int kr = b * 16 + (lane >> 2);
      boff[b] = (static_cast<unsigned>(kr) * a.N + min(c0 + ((lane & 3) ^ (((kr >> 3) & 1) << 1)) * 8, a.N - 8)) * 2u;
    }
  }
  const unsigned step_b = KIND == SK_NN ? static_cast<unsigned>(a.N) * 128u : 128u;  // bytes from stage to stage
  unsigned coff[NT], cg[NT];  // int4: lane -> row lane / 4, slot lane % 4
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int r = lane >> 2;
    coff[j] = static_cast<unsigned>(min(c0 + j * 16 + r, a.N - 1) - c0) * (a.K / 2);
    cg[j] = (lane & 3) ^ ((r >> 2) & 3);
    // scales: lane -> row (lane / 2) % 16, pair lane % 2 (lanes 32-63 repeat)
    soff[j] = static_cast<unsigned>(min(c0 + j * 16 + ((lane >> 1) & 15), a.N - 1) - c0) * groups * 2;
  }

  // Stage s into ring slot s % D. An int4 stage that holds half a unit (the
  // end of K) loads its first half twice; those MFMAs are skipped.
  auto issue = [&](int s) {
    unsigned char* st = ring + (s - s0) % D * S::kBytes;
    if constexpr (S::I4) {
      const bool half = s * 4 + 2 >= groups;  // uniform
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int b = 0; b < 2 * MT; ++b)
          load_lds16(rsrc_a, aoff[b] + s * 256 + (h && !half ? 128 : 0), st + h * (MT * 2048) + b * 1024);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        load_lds16(rsrc_b, coff[j] + s * 64 + (half ? cg[j] & 1 : cg[j]) * 16, st + S::kABytes + j * 1024);
        load_lds4(rsrc_s, soff[j] + s * 8 + (half ? 0 : (lane & 1) * 4), st + S::kABytes + NT * 1024 + j * 256);
      }
    } else {
#pragma unroll
      for (int b = 0; b < 2 * MT; ++b) load_lds16(rsrc_a, aoff[b] + s * 128, st + b * 1024);
#pragma unroll
      for (int b = 0; b < 2 * NT; ++b) load_lds16(rsrc_b, boff[b] + s * step_b, st + S::kABytes + b * 1024);
    }
  };

  f32x4v acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4v{0.f, 0.f, 0.f, 0.f};

  // The MFMAs of the resident stage s; ends with its LDS reads done.
  auto compute = [&](int s) {
    const unsigned char* st = ring + (s - s0) % D * S::kBytes;
    auto frag = [&](const unsigned char* base, int blk, int step) {  // 16 rows, 32-deep step of a 64-deep half
      const int r = blk * 16 + n;
      return __builtin_bit_cast(bf16x8_t, reinterpret_cast<const u32x4v*>(base)[swz(r, step * 4 + q)]);
    };
    constexpr int STEPS = S::kDepth / 32;
    bf16x8_t fa[STEPS][MT], fb[STEPS][NT];
#pragma unroll
    for (int t = 0; t < STEPS; ++t)
#pragma unroll
      for (int i = 0; i < MT; ++i) fa[t][i] = frag(st + (t >> 1) * (MT * 2048), i, t & 1);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if constexpr (S::I4) {
        const unsigned char* cb = st + S::kABytes + j * 1024 + n * 64;
        const u32x2v sc = *reinterpret_cast<const u32x2v*>(st + S::kABytes + NT * 1024 + j * 256 + n * 8);
        unsigned cw[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) cw[t] = *reinterpret_cast<const unsigned*>(cb + ((t ^ ((n >> 2) & 3)) * 16 + q * 4));
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const unsigned sw = t < 2 ? sc.x : sc.y;
          fb[t][j] = __builtin_bit_cast(
              bf16x8_t, dequant8(cw[t], __builtin_bit_cast(float, (t & 1) ? sw & 0xffff0000u : sw << 16), a.is_signed));
        }
      } else if constexpr (KIND == SK_NN) {
        // 16-lane group q: lane 4r + c addresses columns 4c.. of k-row 8 q + r, lane i receives column i of the four rows
        const int kr = q * 8 + (n >> 2), col = j * 16 + (n & 3) * 4;
        const unsigned char* p =
            st + S::kABytes + kr * 64 + ((col >> 3) ^ (((kr >> 3) & 1) << 1)) * 16 + (col & 7) * 2;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const u32x2v lo = __builtin_bit_cast(u32x2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                           (__attribute__((address_space(3))) i16x4v*)(p + t * 2048)));
          const u32x2v hi = __builtin_bit_cast(u32x2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16((
                                                           __attribute__((address_space(3))) i16x4v*)(p + t * 2048 + 256)));
          fb[t][j] = __builtin_bit_cast(bf16x8_t, (u32x4v){lo.x, lo.y, hi.x, hi.y});
        }
      } else {
#pragma unroll
        for (int t = 0; t < 2; ++t) fb[t][j] = frag(st + S::kABytes, j, t);
      }
    }
#pragma unroll
    for (int t = 0; t < STEPS; ++t) {
      if (t == 2 && s * 4 + 2 >= groups) break;  // int4: half a unit at the end of K (uniform)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[t][i], fb[t][j], acc[i][j], 0, 0, 0);
    }
    // every LDS read of this stage has returned: its slot may be refilled
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

#pragma unroll
  for (int d = 0; d < D; ++d)
    if (s0 + d < s1) issue(s0 + d);
  trace_write(trace, kTraceGemm, blockIdx.x, 0, t_start);
  int s = s0;
  for (; s + D < s1; ++s) {
    wait_own_loads<(D - 1) * S::kLoads>();
    compute(s);
    issue(s + D);
  }
  // the last D stages
  for (; s < s1; ++s) {
    const int left = s1 - s - 1;
    if (D == 2 && left == 1)
      wait_own_loads<S::kLoads>();
    else
      wait_own_loads<0>();
    compute(s);
  }
  __syncthreads();  // every wave is done with its ring

  float* const red = reinterpret_cast<float*>(smem);
  // lane l holds rows 4 q + v, column n of each 16 x 16 tile
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) red[(wave * ROWS + i * 16 + q * 4 + v) * LD + j * 16 + n] = acc[i][j][v];
  __syncthreads();
  auto total = [&](int row, int col) {
    float x = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) x += red[(w * ROWS + row) * LD + col];
    return x;
  };
  constexpr int OC = KIND == SK_PAIR ? 16 : COLS;  // output columns
  const int n_out = KIND == SK_PAIR ? a.N / 2 : a.N;
  for (int e = tid; e < ROWS * OC; e += 64 * W) {
    const int row = e / OC, col = e % OC;
    if (row >= a.M || c0 + col >= n_out) continue;
    uint16_t* dst = a.C + static_cast<size_t>(row) * a.ldc + c0 + col;
    if constexpr (KIND == SK_PAIR) {
      const float g = bf16_to_f32(f32_to_bf16(total(row, col))), u = bf16_to_f32(f32_to_bf16(total(row, 16 + col)));
      *dst = f32_to_bf16(silu_f32(g) * u);
    } else {
      float x = total(row, col);
      if (a.epi != EPI_NONE || a.clamp) {
        x = bf16_to_f32(out_bf16(x, a.toward_zero));
        x = apply_epilogue(x, a.epi);
        if (a.clamp) x = fminf(fmaxf(x, a.lo), a.hi);
      }
      *dst = out_bf16(x, a.toward_zero);
    }
  }
  trace_stamp(trace, kTraceGemm, blockIdx.x, 5);
}

}  // namespace
}  // namespace iron
