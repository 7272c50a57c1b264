// Float-input GEMM (the products of lab_gemm_q8 / lab_gemm_q4 mode 0,
// lab_native.c:489-501 and :1013-1023, for many tokens) on gfx950 bf16 MFMA:
//   y[m][r] = sum_b sw[r][b] * D_b[m][r],   D_b[m][r] = sum_{k in b} x[m][k] * w[r][k]
// with w the Q8 value or q - 8 for Q4, x fp32 as the caller gives it.
//
// Exact operands. Every weight value is an integer of at most 8 significant
// bits (|w| <= 127), exact in bf16. x is split into three bf16 pieces that
// sum to it exactly (split3_bf16: 8 + 8 + 8 significant bits), so every
// product piece * w is exact in fp32 and D_b is the fp32 sum of exact
// products, in the matrix core's order instead of the CPU's fma chain: the
// outputs agree with the CPU kernel to fp32 rounding (the tolerance bar, as
// the reference's own float GPU kernels, lab_metal.m:79-144, :174-258, sum
// in yet another order).
//
// The weight scale sw is the same for all 16 outputs a lane holds (they are
// one weight row r = the lane's column), so the per-block epilogue is one
// fma per output: acc = fma(D_b, sw, acc), blocks in order, as the CPU's
// acc = fmadd(s, sw, acc).
//
// Per 32 x 32 tile and block: six v_mfma_f32_32x32x16_bf16 (three pieces x
// two halves of the block's K, 192 clocks) and 16 fma. x is split and the
// weights are converted to bf16 once per workgroup, on their way into LDS:
// a wave that splits its own 32 tokens beside 64 or 128 rows spends more on
// the VALU (about 220 instructions per block) than on the matrix cores.
//
// Workgroup: 512 threads; a wave holds 64 tokens x 64 weight rows (32 x 64 in
// the smallest tile), so a block's fragments, 16 KB of LDS reads, feed 24
// MFMAs. Three tiles: 128 tokens x 256 rows, 64 x 256 in two block parities
// and 32 x 128 in four (groups of waves that take the blocks of a stage in
// turn and add their sums through LDS at the end, in order). One stage (1, 2
// or 4 blocks) is converted into one LDS buffer while the other is
// multiplied, its loads in flight a stage ahead. The two waves of a SIMD
// take the two parts of a stage in opposite order, the multiplying one at
// higher priority, so that the matrix cores and the VALU work side by side
// (4320 x 1152 at 1024 tokens: 60 us in the same order, 48 so).
//
// What bounds it: the MFMAs of three pieces (25.8 GFLOP, 16 us at the 1.6
// PFLOP/s a large bf16 product reaches here, for 4096 x 4096 at 256 tokens),
// the conversions the matrix cores do not cover, and where K is split the
// partials' round trip. Measured (us, graph-timed, against four waves of 32
// tokens that each split their own x): 4096 x 4096 at 256 tokens 63.6 ->
// 35-38, 4320 x 1152 and 1152 x 4320 at 1024 70.5 / 73.8 -> 48-52 / 47,
// 6144 x 2048 Q4 at 512 / 64 95.9 / 28.1 -> 50-56 / 16, 1024 x 1024 at 1024
// 24.2 -> 14.1, 8192 x 4096 at 16 48.0 -> 15.9, 3072 x 1024 at 12 11.3 -> 7.3.
//
// When the tiles alone would leave CUs idle, K is split over blockIdx.y and
// a second kernel adds the partials in split order (deterministic).

#include "common.h"
#include "dnx_kernels.h"

using namespace dnx;

namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kThreads = 512;
constexpr int kWaves = 8;

struct FParams {
  const void* qs;       // Q8 int8 [rows][cols] or Q4 nibbles [rows][cols/2]
  const void* scales;   // Q8 fp32 / Q4 fp16 bits [rows][cols/32]
  const float* x;       // [n][cols]
  float* y;             // [n][rows]
  float* part;          // split partials [splits][n][rows], or null
  int rows, cols, n;
  int tiles_m, tiles;
  int split_blocks;     // blocks per K split, a multiple of the tile's parities
};

// The top halves of two dwords as one (a in the low half).
DNX_DEV uint32_t hi16x2(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// Two small integers as a pair of bf16 (exact: at most 8 significant bits).
DNX_DEV uint32_t bf16x2(int a, int b) {
  return hi16x2(__float_as_uint((float)a), __float_as_uint((float)b));
}

// 8 weights of a block (k = 8c .. 8c + 7 of one K half) as one 16-byte bf16
// fragment, from their integer values in w[0..7].
DNX_DEV uint4 weight_frag(const int* w) {
  return make_uint4(bf16x2(w[0], w[1]), bf16x2(w[2], w[3]), bf16x2(w[4], w[5]),
                    bf16x2(w[6], w[7]));
}

// Eight floats -> the three bf16 pieces of each (p0 + p1 + p2 == x), each
// piece as one 16-byte fragment (element j of the fragment = value j).
// split_any: an infinity or NaN is carried whole by p0 (a quiet NaN for
// every NaN) with zero pieces after it, so it meets the weights as the CPU's
// x does. It is called only for the eight values that hold one.
DNX_DEV void split_any(const float* x, uint4* p) {
  uint32_t q[3][8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    const uint32_t bits = __float_as_uint(x[j]);
    const float r = x[j] - __uint_as_float(bits & 0xffff0000u);
    const uint32_t b1 = __float_as_uint(r);
    const float r2 = r - __uint_as_float(b1 & 0xffff0000u);
    const bool inf_nan = (bits & 0x7f800000u) == 0x7f800000u;
    q[0][j] = inf_nan && (bits & 0x007fffffu) ? 0x7fc00000u : bits;
    q[1][j] = inf_nan ? 0u : b1;
    q[2][j] = inf_nan ? 0u : __float_as_uint(r2);
  }
#pragma unroll
  for (int i = 0; i < 3; i++) {
    p[i] = make_uint4(hi16x2(q[i][0], q[i][1]), hi16x2(q[i][2], q[i][3]),
                      hi16x2(q[i][4], q[i][5]), hi16x2(q[i][6], q[i][7]));
  }
}

DNX_DEV void split_frags(const float* x, uint4* p) {
  float rest = 0.0f;   // of the first pieces: NaN when a value is infinite or NaN
  uint32_t w[3][4];
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    const uint32_t a = __float_as_uint(x[j]), b = __float_as_uint(x[j + 1]);
    const float ra = x[j] - __uint_as_float(a & 0xffff0000u);
    const float rb = x[j + 1] - __uint_as_float(b & 0xffff0000u);
    const uint32_t a1 = __float_as_uint(ra), b1 = __float_as_uint(rb);
    const float ra2 = ra - __uint_as_float(a1 & 0xffff0000u);
    const float rb2 = rb - __uint_as_float(b1 & 0xffff0000u);
    w[0][j / 2] = hi16x2(a, b);
    w[1][j / 2] = hi16x2(a1, b1);
    w[2][j / 2] = hi16x2(__float_as_uint(ra2), __float_as_uint(rb2));
    rest += ra + rb;
  }
#pragma unroll
  for (int i = 0; i < 3; i++) p[i] = make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]);
  if (__builtin_expect(rest != rest, 0)) split_any(x, p);
}

// Shape of a workgroup's tile: WM x WN waves of TM * 32 tokens x 64 weight
// rows, and PAR groups of them that take the blocks of a stage in turn.
template <int WM_, int WN_, int PAR_, int TM_>
struct Tile {
  static constexpr int WM = WM_, WN = WN_, PAR = PAR_, TM = TM_;
  static constexpr int BM = WM * TM * 32, BN = WN * 64;
  static_assert(WM * WN * PAR == kWaves, "eight waves");
  // LDS strides of one fragment row set (tokens or weight rows x 16 bytes):
  // the pads put the four threads that write one 32-value block, and the two
  // rows beside them, in different banks.
  static constexpr int kFA = BM * 16 + 32, kFB = BN * 16 + 16;
  static constexpr int kA = PAR * 12 * kFA;             // [par][piece][4 k-groups]
  static constexpr int kB = PAR * 4 * kFB;              // [par][4 k-groups]
  static constexpr int kStage = kA + kB + PAR * BN * 4; // + fp32 weight scales
  static constexpr int kLds = 2 * kStage;
  static_assert(PAR == 1 || kLds >= (PAR - 1) * BM * BN * 4, "the parities' sums reuse the stages");
};

template <bool kQ4, class T>
__global__ void __launch_bounds__(kThreads) gemm_float_kernel(FParams p) {
  constexpr int WM = T::WM, WN = T::WN, PAR = T::PAR, TM = T::TM, BM = T::BM, BN = T::BN;
  constexpr int UA = BM * 4 * PAR, PA = (UA + kThreads - 1) / kThreads;   // 8 x values each
  constexpr int UB = BN * 2 * PAR, PB = (UB + kThreads - 1) / kThreads;   // 16 weights each
  constexpr int US = BN * PAR, PS = (US + kThreads - 1) / kThreads;       // weight scales
  __shared__ __align__(16) uint8_t lds[T::kLds];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int par = wave / (WM * WN), wm = wave % (WM * WN) / WN, wn = wave % WN;
  const int K = p.cols, B = K / kBlock, M = p.n, N = p.rows;
  // XCD-aware order (workgroups are dealt round-robin to the 8 XCDs): each
  // XCD walks a contiguous run of tiles, all token tiles of its weight rows.
  const int i0 = blockIdx.x;
  const int t = (p.tiles % 8 == 0) ? (i0 % 8) * (p.tiles / 8) + i0 / 8 : i0;
  const int m0 = t % p.tiles_m * BM, n0 = t / p.tiles_m * BN;
  const int b_begin = blockIdx.y * p.split_blocks;
  const int nb = min(B, b_begin + p.split_blocks) - b_begin;   // this split's blocks
  const int steps = (nb + PAR - 1) / PAR;

  constexpr int wbytes = kQ4 ? 16 : 32, sbytes = kQ4 ? 2 : 4;
  constexpr int kFar = -(1 << 20);   // past every operand: reads zeros
  const i32x4 rq = buffer_rsrc(p.qs, (uint32_t)((size_t)N * B * wbytes));
  const i32x4 rs = buffer_rsrc(p.scales, (uint32_t)((size_t)N * B * sbytes));
  const i32x4 rx = buffer_rsrc(p.x, (uint32_t)((size_t)M * K * 4));

  // ---- staging: what each thread carries from memory to LDS in a step.
  // x: (token, block, group of 8 values), four threads to a token's 128-byte
  // block; weights: (row, block, half of 16 values); scales: (row, block).
  i32x4 xr[PA][2], wr[PB];
  int sr[PS];
  auto load_step = [&](int s) {
    const int b0 = b_begin + s * PAR, left = nb - s * PAR;   // blocks from b0 on
#pragma unroll
    for (int e = 0; e < PA; e++) {
      const int u = e * kThreads + tid, f = u & 3, tok = (u >> 2) % BM, blk = (u >> 2) / BM;
      const bool ok = u < UA && m0 + tok < M && blk < left;
      const int off = ok ? ((m0 + tok) * K + (b0 + blk) * kBlock + 8 * f) * 4 : kFar;
      xr[e][0] = dnx_raw_buffer_load_v4i32(rx, off, 0, 0);
      xr[e][1] = dnx_raw_buffer_load_v4i32(rx, off + 16, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < PB; e++) {
      const int u = e * kThreads + tid, h = u & 1, blk = (u >> 1) % PAR, row = u / (2 * PAR);
      const bool ok = u < UB && n0 + row < N && blk < left;
      // A Q4 block's 16 bytes hold both halves (low and high nibbles).
      const int off = ((n0 + row) * B + b0 + blk) * wbytes + (kQ4 ? 0 : 16 * h);
      wr[e] = dnx_raw_buffer_load_v4i32(rq, ok ? off : kFar, 0, 0);
    }
#pragma unroll
    for (int e = 0; e < PS; e++) {
      const int u = e * kThreads + tid, blk = u % PAR, row = u / PAR;
      const bool ok = u < US && n0 + row < N && blk < left;
      const int off = ok ? ((n0 + row) * B + b0 + blk) * sbytes : kFar;
      // Q4: the raw 16 bits (an operation on them here would wait for them).
      sr[e] = kQ4 ? (int)dnx_raw_buffer_load_i16(rs, off, 0, 0)
                  : dnx_raw_buffer_load_i32(rs, off, 0, 0);
    }
  };
  auto store_step = [&](int buf) {
    uint8_t* base = lds + buf * T::kStage;
#pragma unroll
    for (int e = 0; e < PA; e++) {
      const int u = e * kThreads + tid, f = u & 3, tok = (u >> 2) % BM, blk = (u >> 2) / BM;
      if (UA % kThreads != 0 && u >= UA) break;
      float xv[8];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        xv[j] = __int_as_float(xr[e][0][j]);
        xv[4 + j] = __int_as_float(xr[e][1][j]);
      }
      uint4 q[3];
      split_frags(xv, q);
#pragma unroll
      for (int pc = 0; pc < 3; pc++)
        *(uint4*)(base + ((blk * 3 + pc) * 4 + f) * T::kFA + tok * 16) = q[pc];
    }
#pragma unroll
    for (int e = 0; e < PB; e++) {
      const int u = e * kThreads + tid, h = u & 1, blk = (u >> 1) % PAR, row = u / (2 * PAR);
      if (UB % kThreads != 0 && u >= UB) break;
      int w[16];
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const uint32_t v = (uint32_t)wr[e][k >> 2];
        w[k] = kQ4 ? (int)((v >> (8 * (k & 3) + 4 * h)) & 15u) - 8
                   : (int)(int8_t)(v >> (8 * (k & 3)));
      }
      uint8_t* d = base + T::kA + (blk * 4 + 2 * h) * T::kFB + row * 16;
      *(uint4*)d = weight_frag(w);
      *(uint4*)(d + T::kFB) = weight_frag(w + 8);
    }
#pragma unroll
    for (int e = 0; e < PS; e++) {
      const int u = e * kThreads + tid, blk = u % PAR, row = u / PAR;
      if (US % kThreads != 0 && u >= US) break;
      const float sw = kQ4 ? half_bits_to_float((uint16_t)sr[e]) : __int_as_float(sr[e]);
      *(float*)(base + T::kA + T::kB + (blk * BN + row) * 4) = sw;
    }
  };

  v16f acc[TM][2];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;

  const int l32 = lane & 31, c = lane >> 5;
  load_step(0);
  store_step(0);
  if (steps > 1) load_step(1);
  __syncthreads();
  // The two waves of a SIMD (waves w and w + 4) take a step's parts in
  // opposite order, so that one's matrix work runs beside the other's
  // conversions: in the same order both wait for the same unit at once.
  const bool stage_first = wave < kWaves / 2;
  auto stage_next = [&](int s) {
    if (s + 1 < steps) {
      store_step((s + 1) & 1);
      if (s + 2 < steps) load_step(s + 2);
    }
  };
  for (int s = 0; s < steps; s++) {
    const uint8_t* base = lds + (s & 1) * T::kStage;
    if (stage_first) stage_next(s);
    if (s * PAR + par < nb) {   // the wave's block of this stage exists
      const uint8_t* ab = base + par * 12 * T::kFA + (wm * TM * 32 + l32) * 16;
      const uint8_t* bb = base + T::kA + par * 4 * T::kFB + (wn * 64 + l32) * 16;
      __builtin_amdgcn_s_setprio(1);   // before the other wave's conversions
      v16f d[TM][2];
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int v = 0; v < 16; v++) d[i][j][v] = 0.0f;
      // The smallest pieces first: each MFMA rounds its sum, and only the last
      // two then do so at its full size.
      bf8 w[2][2];
#pragma unroll
      for (int h = 0; h < 2; h++)
#pragma unroll
        for (int j = 0; j < 2; j++)
          w[h][j] = __builtin_bit_cast(bf8, *(const uint4*)(bb + (2 * h + c) * T::kFB + j * 512));
#pragma unroll
      for (int pc = 2; pc >= 0; pc--)
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
          for (int i = 0; i < TM; i++) {
            const bf8 a = __builtin_bit_cast(
                bf8, *(const uint4*)(ab + (pc * 4 + 2 * h + c) * T::kFA + i * 512));
#pragma unroll
            for (int j = 0; j < 2; j++)
              d[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, w[h][j], d[i][j], 0, 0, 0);
          }
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const float sw =
            *(const float*)(base + T::kA + T::kB + (par * BN + wn * 64 + j * 32 + l32) * 4);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int v = 0; v < 16; v++) acc[i][j][v] = fmaf(d[i][j][v], sw, acc[i][j][v]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
    if (!stage_first) stage_next(s);
    __syncthreads();
  }

  // The parities' sums, added in parity order by parity 0's waves.
  if constexpr (PAR > 1) {
    float* red = (float*)lds + wave % (WM * WN) * (TM * 2 * 16 * 64) + lane;
#pragma unroll
    for (int q = 1; q < PAR; q++) {
      float* mine = red + (q - 1) * BM * BN;
      if (par == q) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
          for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) mine[((i * 2 + j) * 16 + v) * 64] = acc[i][j][v];
      }
    }
    __syncthreads();
    if (par != 0) return;
#pragma unroll
    for (int q = 1; q < PAR; q++) {
      const float* theirs = red + (q - 1) * BM * BN;
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
          for (int v = 0; v < 16; v++) acc[i][j][v] += theirs[((i * 2 + j) * 16 + v) * 64];
    }
  }
  float* out = p.part ? p.part + (size_t)blockIdx.y * M * N : p.y;
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int r = n0 + wn * 64 + j * 32 + l32;
      if (r >= N) continue;
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const int m = m0 + (wm * TM + i) * 32 + (v >> 2) * 8 + c * 4 + (v & 3);
        if (m < M) store_wt(out + (size_t)m * N + r, acc[i][j][v]);
      }
    }
}

// y = the split partials summed in split order (deterministic), four
// outputs to a thread where they are whole 16-byte pieces.
template <bool kVec>
__global__ void __launch_bounds__(256) float_splitk_reduce_kernel(
    const float* __restrict__ part, float* __restrict__ y, int64_t count, int splits) {
  const int64_t items = kVec ? count / 4 : count;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < items;
       i += (int64_t)gridDim.x * 256) {
    if constexpr (kVec) {
      f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int z0 = 0; z0 < splits; z0 += 4) {   // four splits' loads together
        f32x4 t[4];
#pragma unroll
        for (int u = 0; u < 4; u++)
          t[u] = ((const f32x4*)part)[(size_t)min(z0 + u, splits - 1) * items + i];
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (z0 + u < splits) v = z0 + u == 0 ? t[u] : v + t[u];
      }
      store_wt4(y + 4 * i, make_float4(v.x, v.y, v.z, v.w));
    } else {
      store_wt(y + i, split_sum(part, count, i, splits));
    }
  }
}

// Library-owned split partials, grown on demand (a call at a larger shape
// than any before allocates: not the first call inside a graph capture).
float* gPart = nullptr;
size_t gPartBytes = 0;

float* part_workspace(size_t bytes) {
  if (bytes <= gPartBytes) return gPart;
  if (gPart != nullptr) {
    if (hipDeviceSynchronize() != hipSuccess) return nullptr;
    (void)hipFree(gPart);
    gPart = nullptr;
    gPartBytes = 0;
  }
  if (hipMalloc(&gPart, bytes) != hipSuccess) {
    gPart = nullptr;
    return nullptr;
  }
  gPartBytes = bytes;
  return gPart;
}

template <bool kQ4, class T>
int launch(const void* qs, const void* scales, const float* x, float* y, int64_t rows,
           int64_t cols, int64_t n, int splits, hipStream_t stream) {
  FParams p{};
  p.qs = qs;
  p.scales = scales;
  p.x = x;
  p.y = y;
  p.rows = (int)rows;
  p.cols = (int)cols;
  p.n = (int)n;
  p.tiles_m = (int)((n + T::BM - 1) / T::BM);
  p.tiles = p.tiles_m * (int)((rows + T::BN - 1) / T::BN);
  const int B = (int)(cols / kBlock);
  p.split_blocks = (B + splits - 1) / splits;
  p.split_blocks = (p.split_blocks + T::PAR - 1) / T::PAR * T::PAR;
  splits = (B + p.split_blocks - 1) / p.split_blocks;
  const int64_t count = n * rows;
  p.part = nullptr;
  if (splits > 1) {
    p.part = part_workspace((size_t)splits * count * 4);
    if (p.part == nullptr) return DNX_ENOMEM;
  }
  hipLaunchKernelGGL((gemm_float_kernel<kQ4, T>), dim3((unsigned)p.tiles, (unsigned)splits),
                     dim3(kThreads), 0, stream, p);
  if (hipGetLastError() != hipSuccess) return DNX_ELAUNCH;
  if (splits > 1) {
    const bool vec = count % 4 == 0 && ((uintptr_t)y & 15) == 0;
    const int64_t blocks = ((vec ? count / 4 : count) + 255) / 256;
    hipLaunchKernelGGL(vec ? float_splitk_reduce_kernel<true> : float_splitk_reduce_kernel<false>,
                       dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, stream,
                       p.part, y, count, splits);
    if (hipGetLastError() != hipSuccess) return DNX_ELAUNCH;
  }
  return DNX_OK;
}

// What a tile and K split cost, in us: rounds of 256 workgroups (a tile's
// LDS holds a CU to one) times a fixed part and the stages of a split, and
// the partials' round trip. The constants are a fit to 1500 runs (40 shapes
// of 512..8192 rows, 512..4096 columns, 5..1024 tokens, Q4 and Q8): it picks
// within 1% of the fastest of them on average, 8% at worst.
struct FloatCost {
  double us;
  int splits;
};

template <class T>
FloatCost float_cost(int64_t rows, int64_t cols, int64_t n, double round_us, double stage_us,
                     bool may_split) {
  const int64_t tiles = ((n + T::BM - 1) / T::BM) * ((rows + T::BN - 1) / T::BN);
  const int64_t B = cols / kBlock;
  FloatCost best{1e30, 1};
  for (int want : {1, 2, 3, 4, 6, 8, 12, 16}) {
    if (want > B || (want > 1 && !may_split)) break;
    const int64_t run = ((B + want - 1) / want + T::PAR - 1) / T::PAR * T::PAR;
    const int64_t splits = (B + run - 1) / run;
    const double rounds = (double)((tiles * splits + 255) / 256);
    const double us = rounds * (round_us + stage_us * (double)(run / T::PAR)) +
                      (splits > 1 ? 1.8 + 1.5e-6 * (double)(splits * n * rows) : 0.0);
    if (us < best.us) best = {us, want};
  }
  return best;
}

template <bool kQ4>
int launch_float(const void* qs, const void* scales, const float* x, float* y, int64_t rows,
                 int64_t cols, int64_t n, hipStream_t stream) {
  if (rows <= 0 || cols <= 0 || n <= 0 || cols % kBlock != 0) return DNX_EINVAL;
  // 32-bit buffer offsets: each operand below 2 GB.
  if (rows * (kQ4 ? cols / 2 : cols) >= (1ll << 31) || n * cols * 4 >= (1ll << 31) ||
      n * rows >= (1ll << 31)) {
    return DNX_EINVAL;
  }
  if (((uintptr_t)qs & 15) || ((uintptr_t)x & 3) || ((uintptr_t)y & 3) ||
      ((uintptr_t)scales & (kQ4 ? 1 : 3))) {
    return DNX_EINVAL;
  }
  // The tile and K split the measured costs put lowest. With 256 tiles of
  // 128 tokens x 64 rows or more K stays whole: such calls need no memory of
  // the library's own (a split would gain at most 9% on them).
  const bool may_split = ((n + 127) / 128) * ((rows + 63) / 64) < 256;
  const FloatCost costs[] = {float_cost<Tile<2, 4, 1, 2>>(rows, cols, n, 3.1, 1.13, may_split),
                             float_cost<Tile<1, 4, 2, 2>>(rows, cols, n, 3.4, 1.28, may_split),
                             float_cost<Tile<1, 2, 4, 1>>(rows, cols, n, 2.4, 1.01, may_split)};
  const FloatCost& a = costs[0];
  const FloatCost& b = costs[1];
  const FloatCost& c = costs[2];
  if (c.us <= a.us && c.us <= b.us)
    return launch<kQ4, Tile<1, 2, 4, 1>>(qs, scales, x, y, rows, cols, n, c.splits, stream);
  if (b.us <= a.us)
    return launch<kQ4, Tile<1, 4, 2, 2>>(qs, scales, x, y, rows, cols, n, b.splits, stream);
  return launch<kQ4, Tile<2, 4, 1, 2>>(qs, scales, x, y, rows, cols, n, a.splits, stream);
}

}  // namespace

extern "C" {

int dnx_gemm_q8_float(const int8_t* qs, const float* scales, const float* x, float* y,
                      int64_t rows, int64_t cols, int64_t n, dnx_stream_t stream) {
  return launch_float<false>(qs, scales, x, y, rows, cols, n, (hipStream_t)stream);
}

int dnx_gemm_q4_float(const uint8_t* qs, const uint16_t* scales, const float* x, float* y,
                      int64_t rows, int64_t cols, int64_t n, dnx_stream_t stream) {
  return launch_float<true>(qs, scales, x, y, rows, cols, n, (hipStream_t)stream);
}

}  // extern "C"
