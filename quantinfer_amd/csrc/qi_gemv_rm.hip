// Row-major (blocks along N) GEMV and GEMM, F32 mode: y[m, n] = sum_k x[m, k]
// w(k, n) for QuantInfer-layout weights (backends/cpu/src/backend.rs:62-140 ->
// matmul.rs:14-90; element values matmul.rs:162-280). On a tiled image with K
// a multiple of 4 calls of 5 rows and more (Q6_K and small weights: 3, see
// rm_gemm_min_rows in qi_abi.hip) take the f16 matrix-core GEMM
// (qi_gemm_rm.hip) or, where the scales are outside its range (f32 block
// scales), rm_gemm_kernel below: the records dequantized into LDS for the f32
// matrix cores. Two GEMV kernels by image:
//
// Tiled image (N a multiple of 256; gemv_rmd_kernel, 1 to 4 rows): record
// (t, u) holds rows k = 16t + c (c = 0..15) of outputs n = 256u + [0, 256), in
// the arrangement of the output-rows records. Along N the scales change with
// k, the index that is summed, so they go on the activations' side and the
// codes to the int8 matrix cores: per 64 k and sub-block (outputs that share a
// scale), F = rint(x a 2^s), 30 bits below the largest |x a|, is cut into four
// signed 8-bit digits and v_mfma_i32_16x16x64_i8 multiplies the digits of up
// to four (row, level) slots (16 rows of A) by the codes of 16 outputs,
// exactly. What F leaves of x a makes the next level, times 2^31, until nothing
// is left: two levels ride one instruction at one or two rows, more (in
// practice at 3 and 4 rows, or past activations 2^37 times the others) repeat
// it. So an activation far above the others takes no bits from them. (With the
// first level alone, outputs with zero codes at an activation 1e6 times the
// others had errors of 1.3e-4; now as without it.) Codes are
// centred, Q4_K/Q5_K on a zero point per (k, window), whose small offset
// b - a z is summed in f32 beside them. Both operands need 64 k of one output in
// a lane, the records hold 64 outputs of one k: a wavefront writes its codes
// and digits to its own LDS area in row order and reads them back with
// transposing reads (ds_read_b64_tr_b8); row strides of 144 bytes keep both
// sides free of bank conflicts. A workgroup of four wavefronts takes one unit
// and one K split, each wavefront every fourth chunk of 64 k, at most two, all
// loaded before the first is used (two wavefronts share a chunk, 128 outputs
// each, where there are few: gemv_rm_splits); the wavefronts' sums are added
// through LDS, the splits by rm_sum_kernel.
// MI355X, us per call (one launch of 1 row, 2-row launches or from 3 rows the
// f32 GEMM, f32 multiply-adds per code, before -> now): Q4_K 4096 x 14336 1 row
// 16.1 -> 14.6, 2 27.7 -> 16.0, 4 34.8 -> 21.2; Q5_K 1 row 17.4 -> 16.7; Q6_K
// 14336 x 4096 1 row 21.0 -> 19.8, 4 35.6 -> 31.1; Q4_0 4096 x 12288 2 rows 20.5
// -> 14.3; Q8_0 4096 x 4096 4 rows 15.9 -> 12.2. (One level, 30 bits: Q4_K 14.0,
// 15.1, 17.5.) Error against 64-bit sums 1.0e-7 at K = 4096 (1.4e-7 before). Of
// the 14.6 us the split sum's launch and round trip take 4.
//
// Planar image (gemv_rm_kernel): flat block index k * (N / bs) + nb, so at
// one k the code bytes of consecutive output blocks are contiguous. A lane
// owns one column unit: the outputs one 4-byte code word decodes to
// (Q8_0: 4 outputs; Q4_0 and Q4_K/Q5_K: 8, low and high nibbles; Q6_K: 16 from
// two ql words and one qh word). 64 consecutive column units per workgroup
// column, the four wavefronts split the workgroup's K range, and the grid's
// y dimension splits K further; every k a lane loads its code word(s) and its
// block's scales (the activations are wavefront-uniform loads), forms the
// weights in f32 and accumulates x * w for up to MT activation rows.
// Partials of the K parts are summed in a fixed order: the four wavefronts
// through LDS, the K splits by rm_sum_kernel. Results are deterministic; the
// summation order differs from the reference's sequential k, so the mode is
// judged by tolerance like the output-rows F32 GEMV.
#include "qi_device.h"
#include "qi_internal.h"
#include "qi_unit.h"

#include <type_traits>

namespace qi {

namespace {

template <int QT>
struct RmGeo {
  static constexpr uint32_t kBs = (QT == kQ8_0 || QT == kQ4_0) ? 32 : 256;   // outputs per block
  static constexpr int kOut = QT == kQ8_0 ? 4 : QT == kQ6_K ? 16 : 8;        // outputs per lane
  static constexpr uint32_t kCus = kBs / kOut;                              // column units per block
};

__device__ __forceinline__ uint32_t load_u32(const uint8_t* p) { return *reinterpret_cast<const uint32_t*>(p); }

// Weights of column unit c of flat block blk: w[j] for the lane's outputs
// (their positions within the block: rm_offset).
template <int QT, bool WIDE>
__device__ __forceinline__ void rm_weights(const View& v, uint64_t blk, uint32_t c, float w[RmGeo<QT>::kOut]) {
  const float d = load_scale<WIDE>(v.d, blk);
  if constexpr (QT == kQ8_0) {
    const uint32_t q = load_u32(v.qs + blk * 32 + 4 * c);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = d * static_cast<float>(static_cast<int8_t>(q >> (8 * j)));
  } else if constexpr (QT == kQ4_0) {
    const uint32_t q = load_u32(v.qs + blk * 16 + 4 * c);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      w[j] = d * (static_cast<float>((q >> (8 * j)) & 15u) - 8.0f);
      w[4 + j] = d * (static_cast<float>((q >> (8 * j + 4)) & 15u) - 8.0f);
    }
  } else if constexpr (QT == kQ4_K || QT == kQ5_K) {
    const uint32_t g = c / 8, i = c % 8;
    const uint32_t q = load_u32(v.qs + blk * 128 + 32 * g + 4 * i);
    const uint8_t* s = v.sc + blk * 12;
    uint32_t sc0, m0, sc1, m1;
    const uint32_t w0 = load_u32(s), w1 = load_u32(s + 4), w2 = load_u32(s + 8);
    kquant_sc_m(w0, w1, w2, static_cast<int>(2 * g), sc0, m0);
    kquant_sc_m(w0, w1, w2, static_cast<int>(2 * g + 1), sc1, m1);
    const float dmin = load_scale<WIDE>(v.dmin, blk);
    const float a0 = d * static_cast<float>(sc0), b0 = dmin * static_cast<float>(m0);
    const float a1 = d * static_cast<float>(sc1), b1 = dmin * static_cast<float>(m1);
    [[maybe_unused]] uint32_t h = 0;
    if constexpr (QT == kQ5_K) h = load_u32(v.qh + blk * 32 + 4 * i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t lo = (q >> (8 * j)) & 15u, hi = (q >> (8 * j + 4)) & 15u;
      if constexpr (QT == kQ5_K) {
        lo += ((h >> (8 * j + 2 * g)) & 1u) << 4;
        hi += ((h >> (8 * j + 2 * g + 1)) & 1u) << 4;
      }
      w[j] = a0 * static_cast<float>(lo) - b0;
      w[4 + j] = a1 * static_cast<float>(hi) - b1;
    }
  } else {  // kQ6_K
    const uint32_t ip = c / 8, i = c % 8;
    const uint32_t A = load_u32(v.qs + blk * 128 + 64 * ip + 4 * i);
    const uint32_t B = load_u32(v.qs + blk * 128 + 64 * ip + 32 + 4 * i);
    const uint32_t H = load_u32(v.qh + blk * 64 + 32 * ip + 4 * i);
    const int8_t* s = reinterpret_cast<const int8_t*>(v.sc + blk * 16) + 8 * ip + i / 4;
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) {
      const uint32_t src = (ch & 1) ? B : A;
      const int sh = ch < 2 ? 0 : 4;
      const float a = d * static_cast<float>(s[2 * ch]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t low = (src >> (8 * j + sh)) & 15u;
        const uint32_t high = (H >> (8 * j + 2 * ch)) & 3u;
        w[4 * ch + j] = a * static_cast<float>(static_cast<int>(low | (high << 4)) - 32);
      }
    }
  }
}

// output offset within the block of the lane's output j
template <int QT>
__device__ __forceinline__ uint32_t rm_offset(uint32_t c, int j) {
  if constexpr (QT == kQ8_0) return 4 * c + j;
  else if constexpr (QT == kQ4_0) return j < 4 ? 4 * c + j : 16 + 4 * c + (j - 4);
  else if constexpr (QT == kQ4_K || QT == kQ5_K) return 64 * (c / 8) + 4 * (c % 8) + (j < 4 ? j : 32 + j - 4);
  else return 128 * (c / 8) + 32 * (j / 4) + 4 * (c % 8) + (j % 4);
}

template <int QT, bool WIDE, int MT>
__global__ __launch_bounds__(256) void gemv_rm_kernel(View v, const float* __restrict__ x, uint32_t m,
                                                      uint32_t ksplit, float* __restrict__ out) {
  using G = RmGeo<QT>;
  constexpr int OUT = G::kOut;
  __shared__ float red[3][MT][OUT][64];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t nb_count = static_cast<uint32_t>(v.n / G::kBs);
  const uint32_t cu = blockIdx.x * 64 + lane;  // global column unit
  const uint32_t nb = cu / G::kCus, c = cu % G::kCus;
  const bool live = nb < nb_count;
  const uint32_t K = static_cast<uint32_t>(v.k);
  // this workgroup's K range, then this wavefront's quarter of it
  const uint32_t kb = static_cast<uint32_t>((static_cast<uint64_t>(blockIdx.y) * K) / ksplit);
  const uint32_t ke = static_cast<uint32_t>((static_cast<uint64_t>(blockIdx.y + 1) * K) / ksplit);
  const uint32_t k0 = kb + (ke - kb) * wave / 4, k1 = kb + (ke - kb) * (wave + 1) / 4;

  float acc[MT][OUT];
#pragma unroll
  for (int r = 0; r < MT; ++r)
#pragma unroll
    for (int j = 0; j < OUT; ++j) acc[r][j] = 0.0f;
  const uint64_t blk_nb = live ? nb : 0;  // lanes past N read block 0 and store nothing
#pragma unroll 4
  for (uint32_t k = k0; k < k1; ++k) {
    float w[OUT];
    rm_weights<QT, WIDE>(v, static_cast<uint64_t>(k) * nb_count + blk_nb, c, w);
#pragma unroll
    for (int r = 0; r < MT; ++r) {
      const float xv = static_cast<uint32_t>(r) < m ? x[static_cast<uint64_t>(r) * K + k] : 0.0f;
#pragma unroll
      for (int j = 0; j < OUT; ++j) acc[r][j] = fmaf(xv, w[j], acc[r][j]);
    }
  }
  // the four K quarters, in order
  if (wave > 0) {
#pragma unroll
    for (int r = 0; r < MT; ++r)
#pragma unroll
      for (int j = 0; j < OUT; ++j) red[wave - 1][r][j][lane] = acc[r][j];
  }
  __syncthreads();
  if (wave != 0 || !live) return;
  float* dst = out + static_cast<uint64_t>(blockIdx.y) * m * v.n;
#pragma unroll
  for (int r = 0; r < MT; ++r) {
    if (static_cast<uint32_t>(r) >= m) break;
#pragma unroll
    for (int j = 0; j < OUT; ++j) {
      float s = ((acc[r][j] + red[0][r][j][lane]) + red[1][r][j][lane]) + red[2][r][j][lane];
      const uint64_t col = static_cast<uint64_t>(nb) * G::kBs + rm_offset<QT>(c, j);
      // a NaN or infinite activation: the reference's order decides NaN or
      // +-Inf (with a K split, rm_sum_kernel checks the sum instead)
      if (ksplit == 1 && !__builtin_isfinite(s)) s = exact_row_major_col<QT, WIDE>(v, x + static_cast<uint64_t>(r) * K, col);
      dst[static_cast<uint64_t>(r) * v.n + col] = s;
    }
  }
}

// y = sum of the K-split partials in a fixed order; a sum that is not finite
// is recomputed in the reference's order
// (PAIRS: each eight in pairs, for the GEMM's up to 32 parts: the sums of 28,
// Q6_K 14336 x 4096, added one by one left 1.7e-7 of the result, in pairs 1.4e-7)
template <int QT, bool WIDE, bool PAIRS = false>
__global__ __launch_bounds__(256) void rm_sum_kernel(const float* __restrict__ part, uint32_t splits,
                                                     uint64_t count, float* __restrict__ y, View v,
                                                     const float* __restrict__ x) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= count) return;
  // loads issued 8 at a time with no condition (past the last split the last
  // one is read again and not added), ahead of the adds
  float s = 0.0f;
  for (uint32_t p0 = 0; p0 < splits; p0 += 8) {
    float t[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t pj = p0 + j < splits ? p0 + j : splits - 1;
      t[j] = part[static_cast<uint64_t>(pj) * count + i];
    }
    if constexpr (PAIRS) {
#pragma unroll
      for (int j = 0; j < 8; ++j) t[j] = p0 + j < splits ? t[j] : 0.0f;
      s += ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) s = p0 + j == 0 ? t[j] : p0 + j < splits ? s + t[j] : s;
    }
  }
  if (!__builtin_isfinite(s)) s = exact_row_major_col<QT, WIDE>(v, x + (i / v.n) * v.k, i % v.n);
  y[i] = s;
}

// ------------------------------------------------------------ tiled image

constexpr int kRmtRows = 4;  // activation rows per launch

typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kRmdChunk = 64;          // weight rows of a chunk: one matrix-instruction step
constexpr uint32_t kRmdWs = 128 + 16;       // LDS row stride of a chunk's codes (bytes)
constexpr uint32_t kRmdCodes = kRmdChunk * kRmdWs;
constexpr int kRmdMaxShift = 144;           // 2^-144 / code_scale is an f32 number

// Sub-blocks (one scale each) of a lane group's 32 outputs in a phase, and
// LDS bytes of one wavefront: codes, digits [sub-block][k][16] and factors.
template <int QT>
constexpr uint32_t rmd_subs() {
  return QT == kQ6_K ? 2 : 1;
}
template <int QT>
struct RmdLds {
  static constexpr uint32_t kDig = kRmdChunk * 16 + 8;  // digits of one sub-block, padded against conflicts
  static constexpr uint32_t kSubs = 4 * rmd_subs<QT>();
  static constexpr uint32_t kFac = kRmdCodes + kSubs * kDig;
  static constexpr uint32_t kWave = kFac + kSubs * 4 * 8;
  static_assert(kWave % 16 == 0, "aligned wavefront areas");
};

__device__ __forceinline__ uint32_t rmd_max(uint32_t v) {
  auto step = [&](auto ctrl) {
    const int moved = __builtin_amdgcn_update_dpp(0, static_cast<int>(v), decltype(ctrl)::value, 0xF, 0xF, false);
    const uint32_t o = static_cast<uint32_t>(moved);
    v = o > v ? o : v;
  };
  step(std::integral_constant<int, 0x121>{});
  step(std::integral_constant<int, 0x122>{});
  step(std::integral_constant<int, kDppRor4>{});
  step(std::integral_constant<int, kDppRor8>{});
  return v;
}

// The 8 codes of step st as signed bytes s (q - z): Q4_K / Q5_K with the
// zero point of their sub-block (t = (128 - z) in every byte, s = 1), the
// other formats on the middle of their range (code_scale, code_centre).
template <int QT>
__device__ __forceinline__ uint64_t rmd_codes(const typename Unit<QT>::Raw& r, uint32_t g, int st, uint32_t t) {
  if constexpr (window_centered<QT>()) {
    const uint64_t q = static_cast<uint64_t>(Unit<QT>::codes(r, g, st));
    const uint32_t lo = (static_cast<uint32_t>(q) + t) ^ 0x80808080u;
    const uint32_t hi = (static_cast<uint32_t>(q >> 32) + t) ^ 0x80808080u;
    return (static_cast<uint64_t>(hi) << 32) | lo;
  } else {
    return static_cast<uint64_t>(gemv_codes<QT>(r, g, st));
  }
}

template <int QT, bool WIDE, int MT, int C>
__global__ __launch_bounds__(256, 2) void gemv_rmd_kernel(View v, const float* __restrict__ x, uint32_t m,
                                                          uint32_t ksplit, float* __restrict__ out) {
  using U = Unit<QT>;
  using L = RmdLds<QT>;
  constexpr int SW = rmd_subs<QT>(), NT = 2 / SW;  // sub-blocks per lane group and phase, 16-output tiles of each
  constexpr int LV = MT <= 2 ? 2 : 1, Slots = MT * LV;  // levels in one matrix instruction (4 slots of 4 digits)
  constexpr bool kHalf = C == 0;           // two chunks a workgroup, a phase of one for each wavefront
  constexpr int R = kHalf ? 1 : C;
  constexpr int SI = MT == 4 ? 1 : SW;  // sub-blocks at a time
  constexpr int X = MT == 4 ? 1 : R;  // chunks of x loaded ahead: 256 registers hold no more
  constexpr bool kOff = window_centered<QT>();
  constexpr float kInv = kOff ? 1.0f : 1.0f / static_cast<float>(code_scale<QT>());
  extern __shared__ __align__(16) uint8_t lds[];
  const uint32_t lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t K = static_cast<uint32_t>(v.k), T = v.tiles, chunks = (T + 3) / 4;
  const uint32_t cb = static_cast<uint32_t>((static_cast<uint64_t>(blockIdx.y) * chunks) / ksplit);
  const uint32_t ce = static_cast<uint32_t>((static_cast<uint64_t>(blockIdx.y + 1) * chunks) / ksplit);
  const uint8_t* base = v.qs + static_cast<uint64_t>(blockIdx.x) * v.rec.bytes;
  const uint64_t tile_bytes = static_cast<uint64_t>(v.units) * v.rec.bytes;
  uint8_t* const wl = lds + wave * L::kWave;

  float acc[2][4][2];
#pragma unroll
  for (int j = 0; j < 16; ++j) acc[j >> 3][(j >> 1) & 3][j & 1] = 0.0f;

  // this wavefront's chunks: cb + wave, cb + wave + 4, ... (at most R), the
  // records of all of them loaded before the first is used, with no condition
  // (chunks and tiles past the end load the last one again; their activations
  // are zero)
  const uint32_t c0 = cb + (kHalf ? wave >> 1 : wave), n = c0 < ce ? (ce - c0 + 3) / 4 : 0;
  if (n > 0) {
    typename U::Raw r[R][4];
    float xs[X][4][MT];
    auto load_x = [&](uint32_t tile, float (&o)[MT]) {
      const uint32_t k = min(16 * tile + c, K - 1);
#pragma unroll
      for (int row = 0; row < MT; ++row)
        o[row] = x[static_cast<uint64_t>(min(static_cast<uint32_t>(row), m - 1)) * K + k];
    };
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint32_t tile = min(4 * (c0 + 4 * (static_cast<uint32_t>(j) < n ? j : n - 1)) + t, T - 1);
        if (j < X) load_x(tile, xs[j][t]);
        U::template load<WIDE, true>(base + tile * tile_bytes, lane, r[j][t]);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int j = 0; j < R; ++j) {
      if (static_cast<uint32_t>(j) >= n) break;
      if (j >= X) {
#pragma unroll
        for (int t = 0; t < 4; ++t) load_x(min(4 * (c0 + 4 * j) + t, T - 1), xs[0][t]);
      }
      const uint32_t k0 = kRmdChunk * (c0 + 4 * j) + c;  // record t: row k0 + 16 t
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (kHalf && (wave & 1) != static_cast<uint32_t>(h)) continue;
        // scales of the phase's sub-blocks, their zero points and offsets
        float a[4][SW], b[4][SW];
        uint32_t zt[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          float aa[U::kWindows], bb[U::kWindows];
          U::template scales<WIDE>(g, r[j][t], aa, bb);
#pragma unroll
          for (int i = 0; i < SW; ++i) a[t][i] = aa[h * SW + i];
          if constexpr (kOff) {
            // q - z stays a signed byte for codes up to 31
            const float z = fmaxf(window_zero_point(aa[h], bb[h]), -96.0f);
            b[t][0] = fmaf(-z, aa[h], bb[h]);
            zt[t] = static_cast<uint32_t>(128 - static_cast<int>(z)) * 0x01010101u;
          } else {
            zt[t] = 0;
          }
        }
        // codes [k][128 outputs of the phase]
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          uint64_t q[4];
#pragma unroll
          for (int st = 0; st < 4; ++st) q[st] = rmd_codes<QT>(r[j][t], g, 4 * h + st, zt[t]);
          ulonglong2* dst = reinterpret_cast<ulonglong2*>(wl + (16 * t + c) * kRmdWs + 32 * g);
          dst[0] = make_ulonglong2(q[0], q[1]);
          dst[1] = make_ulonglong2(q[2], q[3]);
        }
#pragma unroll
        for (int i0 = 0; i0 < SW; i0 += SI) {
          // x a as fixed point: digits of level l are those of rint(t) for t = x a
          // 2^sh, |t| < 2^30 at the first level and the remainder times 2^31 at
          // each next one, until nothing is left of any product
          float tt[MT][SI][4], ff[MT][SI];  // t of record t; the level's factor, NaN for a non-finite chunk
          int sh[MT][SI];
          float off[MT];
#pragma unroll
          for (int row = 0; row < MT; ++row) {
            float xv[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) xv[t] = k0 + 16 * t < K ? xs[j % X][t][row] : 0.0f;
#pragma unroll
            for (int i = 0; i < SI; ++i) {
              float p[4];
              uint32_t mx = 0;
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                p[t] = xv[t] * a[t][i0 + i];
                const uint32_t bits = __builtin_bit_cast(uint32_t, p[t]) & 0x7FFFFFFFu;
                mx = bits > mx ? bits : mx;
              }
              mx = rmd_max(mx);
              const bool finite = mx < 0x7F800000u;
              const int e = finite && mx != 0 ? __builtin_amdgcn_frexp_expf(__builtin_bit_cast(float, mx)) : 0;
              sh[row][i] = min(30 - e, kRmdMaxShift);
              // NaN: every output of the row comes out non-finite and is
              // recomputed in the reference's order
              ff[row][i] = finite ? kInv : __builtin_nanf("");
#pragma unroll
              for (int t = 0; t < 4; ++t) tt[row][i][t] = finite ? ldexpf(p[t], sh[row][i]) : 0.0f;
            }
            off[row] = 0.0f;
            if constexpr (kOff) {
#pragma unroll
              for (int t = 0; t < 4; ++t) off[row] = fmaf(xv[t], b[t][0], off[row]);
              off[row] += dpp_move<0x121>(off[row]);
              off[row] += dpp_move<0x122>(off[row]);
              off[row] += dpp_move<kDppRor4>(off[row]);
              off[row] += dpp_move<kDppRor8>(off[row]);
            }
          }
          for (bool more = true; more;) {
            bool left = false;
#pragma unroll
            for (int l = 0; l < LV; ++l)
#pragma unroll
              for (int row = 0; row < MT; ++row)
#pragma unroll
                for (int i = 0; i < SI; ++i) {
                  const int slot = l * MT + row, step = min(31, kRmdMaxShift - sh[row][i]);
                  uint8_t* const dig = wl + kRmdCodes + (g * SI + i) * L::kDig + 4 * slot;
                  float f[4];
#pragma unroll
                  for (int t = 0; t < 4; ++t) {
                    f[t] = rintf(tt[row][i][t]);
                    const uint32_t d = (static_cast<uint32_t>(static_cast<int>(f[t])) + 0x00808080u) ^ 0x00808080u;
                    *reinterpret_cast<uint32_t*>(dig + (16 * t + c) * 16) = d;
                  }
                  if (c == 0)
                    *reinterpret_cast<float2*>(wl + L::kFac + ((g * SI + i) * 4 + slot) * 8) =
                        make_float2(ldexpf(ff[row][i], -sh[row][i]), off[row]);
                  if constexpr (kOff) off[row] = 0.0f;
#pragma unroll
                  for (int t = 0; t < 4; ++t) {
                    tt[row][i][t] = ldexpf(tt[row][i][t] - f[t], step);
                    if (l == LV - 1) left |= tt[row][i][t] != 0.0f && step > 0;
                  }
                  sh[row][i] += step;
                }
            more = __any(left);
            // the wavefront's own LDS accesses complete in order: no wait beyond
            // the reads' own
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            // k slots of both operands: lane group g, 8 g + [0, 8) and 32 + 8 g + [0, 8)
            typedef __attribute__((address_space(3))) i32x2* lds_t;
            auto tr = [&](const uint8_t* p0, uint32_t stride) {
              const i32x2 lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_t)(p0));
              const i32x2 hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_t)(p0 + 32 * stride));
              return i32x4{lo[0], lo[1], hi[0], hi[1]};
            };
#pragma unroll
            for (int w = 0; w < 4; ++w)
#pragma unroll
              for (int i = 0; i < SI; ++i) {
                const uint32_t at = (8 * g + (c >> 1)) * 16 + 8 * (c & 1);
                const i32x4 av = tr(wl + kRmdCodes + (w * SI + i) * L::kDig + at, 16);
                const float2 f = *reinterpret_cast<const float2*>(wl + L::kFac + ((w * SI + i) * 4 + g) * 8);
#pragma unroll
                for (int q = 0; q < NT; ++q) {
                  const int tile = SW == 2 ? i0 + i : q;
                  const i32x4 bv = tr(wl + (8 * g + (c >> 1)) * kRmdWs + 32 * w + 16 * tile + 8 * (c & 1), kRmdWs);
                  // lane 16 g + c: the four digit sums of slot g, output c of the tile
                  const i32x4 d = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, i32x4{0, 0, 0, 0}, 0, 0, 0);
                  const float low = static_cast<float>(d[0] + 256 * d[1]), high = static_cast<float>(d[2] + 256 * d[3]);
                  const float comb = fmaf(high, 65536.0f, low);
                  acc[h][w][tile] += kOff ? fmaf(comb, f.x, -f.y) : comb * f.x;
                }
              }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
          }
        }
      }
    }
  }

  // the four wavefronts' sums [wave][level, row][256], the last level first, in
  // wave order
  __syncthreads();
  float* const red = reinterpret_cast<float*>(lds);
  if (g < static_cast<uint32_t>(Slots)) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int w = 0; w < 4; ++w)
#pragma unroll
        for (int q = 0; q < 2; ++q)
          red[(wave * Slots + g) * 256 + window_first<QT>(w, h) + 16 * q + c] = acc[h][w][q];
  }
  __syncthreads();
  const uint64_t col = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
#pragma unroll
  for (int row = 0; row < MT; ++row) {
    if (static_cast<uint32_t>(row) >= m) break;
    float y = 0.0f;
#pragma unroll
    for (int l = LV - 1; l >= 0; --l)
#pragma unroll
      for (int wv = 0; wv < 4; ++wv) y += red[(wv * Slots + l * MT + row) * 256 + threadIdx.x];
    // a NaN or infinite activation: the reference's order decides NaN or
    // +-Inf (with a K split, rm_sum_kernel checks the sum instead)
    if (ksplit == 1 && !__builtin_isfinite(y))
      y = exact_row_major_col<QT, WIDE>(v, x + static_cast<uint64_t>(row) * K, col);
    out[(static_cast<uint64_t>(blockIdx.y) * m + row) * v.n + col] = y;
  }
}

// Chunks of a wavefront, all loaded before the first is used.
constexpr uint32_t kRmdChunks = 2;

template <int QT, bool WIDE, int MT>
hipError_t launch_rmt_rows(const View& v, const float* x, uint32_t m, float* out, uint32_t splits, hipStream_t st) {
  // chunks per wavefront: ceil(ceil(C / splits) / 4)
  const uint32_t chunks = (v.tiles + 3) / 4, per = ((chunks + splits - 1) / splits + 3) / 4;
  constexpr uint32_t bytes = 4 * RmdLds<QT>::kWave;
  auto go = [&](auto kern) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(v.units, splits), dim3(256), bytes, st, v, x, m, splits, out);
    return hipGetLastError();
  };
  if constexpr (MT <= 2) {  // at most two chunks a workgroup: two wavefronts for each
    if ((chunks + splits - 1) / splits <= 2) return go(gemv_rmd_kernel<QT, WIDE, MT, 0>);
  }
  if (per <= 1) return go(gemv_rmd_kernel<QT, WIDE, MT, 1>);
  if (per <= kRmdChunks) return go(gemv_rmd_kernel<QT, WIDE, MT, kRmdChunks>);
  return hipErrorInvalidValue;
}

template <int QT, bool WIDE>
hipError_t launch_rmt_q(const View& v, const float* x, uint32_t m, float* y, float* part, uint32_t splits,
                        hipStream_t st) {
  float* out = splits > 1 ? part : y;
  if (m < 1 || m > kRmtRows) return hipErrorInvalidValue;
  hipError_t e = m == 1   ? launch_rmt_rows<QT, WIDE, 1>(v, x, m, out, splits, st)
                 : m == 2 ? launch_rmt_rows<QT, WIDE, 2>(v, x, m, out, splits, st)
                          : launch_rmt_rows<QT, WIDE, 4>(v, x, m, out, splits, st);
  if (e != hipSuccess || splits == 1) return e;
  const uint64_t count = static_cast<uint64_t>(m) * v.n;
  hipLaunchKernelGGL((rm_sum_kernel<QT, WIDE>), dim3(static_cast<uint32_t>((count + 255) / 256)), dim3(256), 0,
                     st, part, splits, count, y, v, x);
  return hipGetLastError();
}

template <int QT, bool WIDE>
hipError_t launch_rm_q(const View& v, const float* x, uint32_t m, float* y, float* part, uint32_t splits,
                       hipStream_t st) {
  const uint64_t cus = (v.n / RmGeo<QT>::kBs) * RmGeo<QT>::kCus;
  float* out = splits > 1 ? part : y;
  const dim3 grid(static_cast<uint32_t>((cus + 63) / 64), splits);
  if (m == 1)
    hipLaunchKernelGGL((gemv_rm_kernel<QT, WIDE, 1>), grid, dim3(256), 0, st, v, x, m, splits, out);
  else
    hipLaunchKernelGGL((gemv_rm_kernel<QT, WIDE, 4>), grid, dim3(256), 0, st, v, x, m, splits, out);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || splits == 1) return e;
  const uint64_t count = static_cast<uint64_t>(m) * v.n;
  hipLaunchKernelGGL((rm_sum_kernel<QT, WIDE>), dim3(static_cast<uint32_t>((count + 255) / 256)), dim3(256), 0,
                     st, part, splits, count, y, v, x);
  return hipGetLastError();
}

}  // namespace

namespace {

// Row-major GEMM of images that the f16 one (qi_gemm_rm.hip) leaves, f32 block
// scales and Q8_0 / Q4_0 scales outside f16's range, from 3 or 5 rows
// (rm_gemm_min_rows, qi_abi.hip): y[m, n] = sum_k x[m, k] w(k, n) with the
// weights dequantized in LDS, never stored to HBM. Workgroup (u, mb, z) takes
// unit u (outputs 256u .. 256u + 255), rows 16 TM mb .. of x and K part z
// (tiles [z T / P, (z + 1) T / P)). A stage is 64 weight rows: wavefront w
// loads the record of the stage's tile w (Unit<QT>, lane 16g + c row c's lane
// group g) and writes its 64 weights per lane to LDS as f32, each by the
// reference's operation sequence, so bit-identical to dequantize
// (matmul.rs:162-280): Q8_0 d q; Q4_0 d (q - 8); Q4_K/Q5_K (d sc) q - dmin m,
// no fused multiply-add (the file is compiled with -ffp-contract=off); Q6_K
// (d sc) (q - 32). The stage's activations go to LDS beside it. The
// next stage's record and activations are loaded into registers while the
// matrix cores (v_mfma_f32_16x16x4f32, f32 products) take the current one:
// wavefront w owns outputs 64w .. 64w + 63 for all 16 TM rows. Each 32-row
// half of a stage is summed apart and then added to the running sums (one
// chain over K missed the 1e-5 bar at K = 4096). One part stores y, recomputing a
// non-finite sum in the reference's order; more store partial sums, which
// rm_sum_kernel adds in part order.
constexpr uint32_t kRmgStageK = 64;       // weight rows per stage: one record per wavefront
constexpr uint32_t kRmgWs = 256 + 4;      // LDS row stride of the stage's weights (floats)
constexpr uint32_t kRmgXs = kRmgStageK + 4;  // LDS row stride of the stage's activations

typedef float rmg_f32x4 __attribute__((ext_vector_type(4)));

template <int QT, bool WIDE, int TM>
__global__ __launch_bounds__(256) void rm_gemm_kernel(View v, const float* __restrict__ x, uint32_t M,
                                                      uint32_t parts, float* __restrict__ out) {
  using U = Unit<QT>;
  constexpr int kW = U::kWindows, kS = U::kSteps;
  __shared__ __align__(16) float ws[kRmgStageK * kRmgWs];
  __shared__ __align__(16) float xs[TM * 16 * kRmgXs];
  const uint32_t lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t u = blockIdx.x, m0 = blockIdx.y * TM * 16, z = blockIdx.z;
  const uint32_t K = static_cast<uint32_t>(v.k), T = v.tiles;
  const uint32_t tb = static_cast<uint32_t>((static_cast<uint64_t>(z) * T) / parts);
  const uint32_t te = static_cast<uint32_t>((static_cast<uint64_t>(z + 1) * T) / parts);
  const uint32_t kend = 16 * te < K ? 16 * te : K;  // activations past it are zero
  const uint32_t stages = (te - tb + 3) / 4;
  const uint8_t* base = v.qs + static_cast<uint64_t>(u) * v.rec.bytes;
  const uint64_t tile_bytes = static_cast<uint64_t>(v.units) * v.rec.bytes;

  // two stages in flight: stage s's record and activations in registers
  // r[s % 2], xr[s % 2] (s + 1 loads while s is multiplied)
  typename U::Raw r[2];
  rmg_f32x4 xr[2][TM];
  // stage s: tile tb + 4s + wave (if below te) and activation columns
  // 16 tb + 64 s .. + 63 of rows m0 .. m0 + 16 TM - 1
  auto fetch = [&](uint32_t s, typename U::Raw& rr, rmg_f32x4 (&xx)[TM]) {
    const uint32_t t = tb + 4 * s + wave;
    if (t < te) U::template load<WIDE>(base + t * tile_bytes, lane, rr);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const uint32_t e = threadIdx.x + 256 * i, row = e / 16, k = 16 * tb + kRmgStageK * s + (e % 16) * 4;
      xx[i] = (m0 + row < M && k < kend)
                  ? *reinterpret_cast<const rmg_f32x4*>(x + static_cast<uint64_t>(m0 + row) * K + k)
                  : rmg_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  auto put = [&](uint32_t s, const typename U::Raw& rr, const rmg_f32x4 (&xx)[TM]) {
    const uint32_t t = tb + 4 * s + wave;
    float* wrow = ws + (16 * wave + c) * kRmgWs;
    if (t < te) {
      float a[kW], b[kW];
      U::template scales<WIDE>(g, rr, a, b);
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        const uint64_t q = static_cast<uint64_t>(U::codes(rr, g, st));
        const int w = st / kS;
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t byte = static_cast<uint32_t>(q >> (8 * e)) & 0xFFu;
          if constexpr (QT == kQ8_0) {
            o[e] = a[w] * static_cast<float>(static_cast<int8_t>(byte));
          } else if constexpr (QT == kQ4_0) {
            o[e] = a[w] * (static_cast<float>(byte) - 8.0f);
          } else if constexpr (QT == kQ6_K) {
            o[e] = a[w] * static_cast<float>(static_cast<int32_t>(byte) - 32);
          } else {
            o[e] = a[w] * static_cast<float>(byte) - b[w];
          }
        }
        float4* dst = reinterpret_cast<float4*>(wrow + window_first<QT>(g, st / 4) + 8 * (st % 4));
        dst[0] = make_float4(o[0], o[1], o[2], o[3]);
        dst[1] = make_float4(o[4], o[5], o[6], o[7]);
      }
    } else {
#pragma unroll
      for (int st = 0; st < 8; ++st) {
        float4* dst = reinterpret_cast<float4*>(wrow + window_first<QT>(g, st / 4) + 8 * (st % 4));
        dst[0] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        dst[1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const uint32_t e = threadIdx.x + 256 * i;
      *reinterpret_cast<rmg_f32x4*>(xs + (e / 16) * kRmgXs + (e % 16) * 4) = xx[i];
    }
  };

  rmg_f32x4 acc[TM][4];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = rmg_f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // lane (c, g) supplies A[c][g] = x[row c][k] and B[g][c] = w(k, column c)
  // of each 16 x 16 x 4 product, k = 16 kk + 4 g + step
  const float* xb = xs + c * kRmgXs + 4 * g;
  const float* wb = ws + (4 * g) * kRmgWs + wave * 64 + c;
  auto multiply = [&]() {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      rmg_f32x4 part[TM][4];
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const int kk = 2 * h + k2;
        rmg_f32x4 a[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = *reinterpret_cast<const rmg_f32x4*>(xb + i * 16 * kRmgXs + kk * 16);
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          float bv[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) bv[j] = wb[(kk * 16 + st) * kRmgWs + j * 16];
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
              part[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                  a[i][st], bv[j], k2 == 0 && st == 0 ? rmg_f32x4{0.0f, 0.0f, 0.0f, 0.0f} : part[i][j], 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += part[i][j];
    }
  };
  if (stages > 0) fetch(0, r[0], xr[0]);
  if (stages > 1) fetch(1, r[1], xr[1]);
  for (uint32_t s = 0; s < stages; s += 2) {
    put(s, r[0], xr[0]);
    __syncthreads();
    if (s + 2 < stages) fetch(s + 2, r[0], xr[0]);
    multiply();
    __syncthreads();
    if (s + 1 < stages) {
      put(s + 1, r[1], xr[1]);
      __syncthreads();
      if (s + 3 < stages) fetch(s + 3, r[1], xr[1]);
      multiply();
      __syncthreads();
    }
  }

  // lane (c, g) holds rows 4g .. 4g + 3 of each 16 x 16 block, column c
  float* const dst = out + (parts == 1 ? 0 : static_cast<uint64_t>(z) * M * v.n);
  bool bad = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint64_t n = static_cast<uint64_t>(u) * 256 + wave * 64 + j * 16 + c;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t m = m0 + i * 16 + 4 * g + q;
        if (m >= M) continue;
        bad |= !__builtin_isfinite(acc[i][j][q]);
        dst[static_cast<uint64_t>(m) * v.n + n] = acc[i][j][q];
      }
    }
  // with one part, a non-finite sum (NaN or infinite activations) is
  // recomputed in the reference's order, which decides NaN or +-Inf; this
  // lane's own stores are read back (a loop of its own, so that the
  // accumulator tile above stays in registers)
  if (parts == 1 && bad) {
#pragma unroll 1
    for (int e = 0; e < TM * 16; ++e) {
      const uint32_t i = e / 16, j = (e / 4) % 4, q = e % 4, m = m0 + i * 16 + 4 * g + q;
      const uint64_t n = static_cast<uint64_t>(u) * 256 + wave * 64 + j * 16 + c;
      float* p = dst + static_cast<uint64_t>(m) * v.n + n;
      if (m < M && !__builtin_isfinite(*p)) *p = exact_row_major_col<QT, WIDE>(v, x + static_cast<uint64_t>(m) * K, n);
    }
  }
}

template <int QT, bool WIDE>
hipError_t launch_rm_gemm_q(const View& v, const float* x, uint32_t m, float* y, float* part, uint32_t parts,
                            hipStream_t st) {
  const uint32_t tm = rm_gemm_tile_rows(m) / 16;
  const dim3 grid(v.units, (m + 16 * tm - 1) / (16 * tm), parts);
  float* out = parts > 1 ? part : y;
  if (tm == 1)
    hipLaunchKernelGGL((rm_gemm_kernel<QT, WIDE, 1>), grid, dim3(256), 0, st, v, x, m, parts, out);
  else
    hipLaunchKernelGGL((rm_gemm_kernel<QT, WIDE, 2>), grid, dim3(256), 0, st, v, x, m, parts, out);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || parts == 1) return e;
  const uint64_t count = static_cast<uint64_t>(m) * v.n;
  hipLaunchKernelGGL((rm_sum_kernel<QT, WIDE>), dim3(static_cast<uint32_t>((count + 255) / 256)), dim3(256), 0,
                     st, part, parts, count, y, v, x);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_rm_sum(const Image& im, const View& v, const float* part, uint32_t splits, uint64_t count,
                         float* y, const float* x, hipStream_t st) {
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(static_cast<uint32_t>((count + 255) / 256)), dim3(256), 0, st, part, splits, count,
                       y, v, x);
    return hipGetLastError();
  };
  const bool w = im.wide != 0;
  switch (im.qtype) {
    case kQ8_0: return w ? hipErrorInvalidValue : go(rm_sum_kernel<kQ8_0, false, true>);
    case kQ4_0: return w ? hipErrorInvalidValue : go(rm_sum_kernel<kQ4_0, false, true>);
    case kQ4_K: return w ? hipErrorInvalidValue : go(rm_sum_kernel<kQ4_K, false, true>);
    case kQ5_K: return w ? hipErrorInvalidValue : go(rm_sum_kernel<kQ5_K, false, true>);
    case kQ6_K: return w ? hipErrorInvalidValue : go(rm_sum_kernel<kQ6_K, false, true>);
    default: return hipErrorInvalidValue;
  }
}

// 16-row tiles up to 16 rows, 32 above: 64-row tiles (one wavefront per
// SIMD) ran 2-5% slower from 64 rows on (MI355X, Q4_K 4096 x 14336 M=512
// 684 against 660 us, M=2048 2388 against 2272; Q8_0 4096 x 4096 M=2048 682
// against 642)
uint32_t rm_gemm_tile_rows(uint64_t m) { return m <= 16 ? 16 : 32; }

uint32_t rm_gemm_parts(const Image& im, uint64_t m, uint64_t max_part_floats) {
  // The part count with the fewest rounds of resident workgroups per part
  // (two per CU, 256 CUs), the smaller count on a tie; each part at least two
  // stages (8 tiles), the partial sums within max_part_floats.
  const uint64_t rows = rm_gemm_tile_rows(m), slots = 512;
  const uint64_t groups = static_cast<uint64_t>(im.units) * ((m + rows - 1) / rows);
  uint64_t pmax = im.tiles / 8;
  const uint64_t by_space = max_part_floats / (m * im.n);
  if (pmax > by_space) pmax = by_space;
  if (pmax > 64) pmax = 64;
  uint64_t best = 1;
  for (uint64_t p = 2; p <= pmax; ++p) {
    // rounds(p) / p < rounds(best) / best
    const uint64_t rp = (groups * p + slots - 1) / slots, rb = (groups * best + slots - 1) / slots;
    if (rp * best < rb * p) best = p;
  }
  return static_cast<uint32_t>(best);
}

bool rm_gemm_supported(const Image& im) {
  return gemv_rm_supported(im) && im.tiled && im.k % 4 == 0 && im.k <= 0xFFFFFFF0ull;
}

hipError_t launch_rm_gemm(const Image& im, const View& v, const float* x, uint64_t m, float* y, float* part,
                          uint32_t parts, hipStream_t st) {
  // grid: units x row blocks (at most 0xFFFF) x parts; each part at least one tile
  if (!rm_gemm_supported(im) || m < 1 || (m + 31) / 32 > 0xFFFFu || parts < 1 || parts > 0xFFFFu ||
      parts > im.tiles || (parts > 1 && part == nullptr) || v.units != im.n / 256 || v.tiles != (im.k + 15) / 16 ||
      (m * im.n + 255) / 256 > 0x7fffffffull)
    return hipErrorInvalidValue;
  const uint32_t mm = static_cast<uint32_t>(m);
  const bool w = im.wide != 0;
  switch (im.qtype) {
    case kQ8_0: return w ? launch_rm_gemm_q<kQ8_0, true>(v, x, mm, y, part, parts, st)
                         : launch_rm_gemm_q<kQ8_0, false>(v, x, mm, y, part, parts, st);
    case kQ4_0: return w ? launch_rm_gemm_q<kQ4_0, true>(v, x, mm, y, part, parts, st)
                         : launch_rm_gemm_q<kQ4_0, false>(v, x, mm, y, part, parts, st);
    // K-quants with f16 scales always take the f16 GEMM (gemm_rm_supported)
    case kQ4_K: return w ? launch_rm_gemm_q<kQ4_K, true>(v, x, mm, y, part, parts, st) : hipErrorInvalidValue;
    case kQ5_K: return w ? launch_rm_gemm_q<kQ5_K, true>(v, x, mm, y, part, parts, st) : hipErrorInvalidValue;
    case kQ6_K: return w ? launch_rm_gemm_q<kQ6_K, true>(v, x, mm, y, part, parts, st) : hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

bool gemv_rm_supported(const Image& im) {
  // tiled: grid x = units, grid y = splits of at most 4 * 4 records per workgroup
  return im.layout == kRowMajor && im.qtype >= kQ8_0 && im.qtype <= kQ6_K && im.n % block_elems(im.qtype) == 0 &&
         im.k > 0 && (!im.tiled || (im.units <= 0xFFFFu && im.tiles <= 16ull * 0xFFFFu));
}

uint32_t gemv_rm_rows(const Image& im) { return im.tiled ? kRmtRows : 4; }

uint32_t gemv_rm_fewest_splits(const Image& im) {
  return im.tiled ? static_cast<uint32_t>(((im.tiles + 3) / 4 + 4 * kRmdChunks - 1) / (4 * kRmdChunks))
                  : gemv_rm_splits(im, 1);
}

uint32_t gemv_rm_splits(const Image& im, uint32_t rows) {
  const uint32_t be = block_elems(im.qtype);
  if (im.tiled) {
    // One chunk of 64 k for each wavefront, or two. Two workgroups share a
    // compute unit; time by the workgroups of the busiest of 256 (a pair, and an
    // odd one at the end), with two chunks 39 a pair and 21 an odd one, with one
    // 20 and 12: fits to graphs of 17 shapes in every format. MI355X, us per
    // call, two chunks / one: Q6_K 2048 x 22528 (352 / 704 workgroups) 17.3 / 14.5
    // (f32 multiply-adds 15.3), 4096 x 10240 (320 / 640) 17.2 / 14.4, 4096 x 14336
    // (448 / 896) 17.4 / 17.3; Q8_0 4096 x 24576 (768 / 1536) 21.6 / 23.0, 14336 x
    // 4096 (448 / 896) 16.0 / 17.3.
    const uint64_t chunks = (im.tiles + 3) / 4, s1 = (chunks + 3) / 4, s2 = gemv_rm_fewest_splits(im);
    // Two wavefronts a chunk where that takes no second workgroup on a compute
    // unit (1 and 2 rows). A wavefront each / two, 1 row: Q6_K 1024 x 8192 8.3 /
    // 7.2 (f32 multiply-adds 7.5), 2048 x 2048 8.1 / 7.1 (7.1), Q4_K 512 x 4096
    // 6.7 / 5.9 (6.4); 512 workgroups, Q4_0 2048 x 8192, 7.2 / 7.2.
    const uint64_t s0 = (chunks + 1) / 2;
    if (rows <= 2 && s0 <= 16 && im.units * s0 <= 256) return static_cast<uint32_t>(s0);
    auto cost = [&](uint64_t s, uint64_t pair, uint64_t odd) {
      const uint64_t busiest = (im.units * s + 255) / 256;
      return busiest / 2 * pair + busiest % 2 * odd;
    };
    const bool one = s1 * rows * im.n <= kRmPartFloats && cost(s1, 20, 12) < cost(s2, 39, 21);
    return static_cast<uint32_t>(one ? s1 : s2);
  }
  // enough K splits for about 1024 workgroups, keeping at least 16 k per
  // wavefront (4 wavefronts per workgroup) and at most 256 splits
  const uint64_t out = im.qtype == kQ8_0 ? 4 : im.qtype == kQ6_K ? 16 : 8;
  const uint64_t col_groups = ((im.n / be) * (be / out) + 63) / 64;
  uint64_t s = col_groups >= 1024 ? 1 : 1024 / col_groups;
  const uint64_t cap = im.k / 64 < 256 ? im.k / 64 : 256;
  if (s > cap) s = cap;
  return static_cast<uint32_t>(s < 1 ? 1 : s);
}

hipError_t launch_gemv_rm(const Image& im, const View& v, const float* x, uint32_t m, float* y, float* part,
                          uint32_t splits, hipStream_t st) {
  if (m < 1 || m > gemv_rm_rows(im) || splits < 1 || (splits > 1 && part == nullptr)) return hipErrorInvalidValue;
  const bool wide = im.wide != 0;
  if (im.tiled) {
    if (v.units != im.n / 256 || v.tiles != (im.k + 15) / 16 || !gemv_rm_supported(im)) return hipErrorInvalidValue;
    switch (im.qtype) {
      case kQ8_0: return wide ? launch_rmt_q<kQ8_0, true>(v, x, m, y, part, splits, st)
                              : launch_rmt_q<kQ8_0, false>(v, x, m, y, part, splits, st);
      case kQ4_0: return wide ? launch_rmt_q<kQ4_0, true>(v, x, m, y, part, splits, st)
                              : launch_rmt_q<kQ4_0, false>(v, x, m, y, part, splits, st);
      case kQ4_K: return wide ? launch_rmt_q<kQ4_K, true>(v, x, m, y, part, splits, st)
                              : launch_rmt_q<kQ4_K, false>(v, x, m, y, part, splits, st);
      case kQ5_K: return wide ? launch_rmt_q<kQ5_K, true>(v, x, m, y, part, splits, st)
                              : launch_rmt_q<kQ5_K, false>(v, x, m, y, part, splits, st);
      case kQ6_K: return wide ? launch_rmt_q<kQ6_K, true>(v, x, m, y, part, splits, st)
                              : launch_rmt_q<kQ6_K, false>(v, x, m, y, part, splits, st);
      default: return hipErrorInvalidValue;
    }
  }
  switch (im.qtype) {
    case kQ8_0: return wide ? launch_rm_q<kQ8_0, true>(v, x, m, y, part, splits, st)
                            : launch_rm_q<kQ8_0, false>(v, x, m, y, part, splits, st);
    case kQ4_0: return wide ? launch_rm_q<kQ4_0, true>(v, x, m, y, part, splits, st)
                            : launch_rm_q<kQ4_0, false>(v, x, m, y, part, splits, st);
    case kQ4_K: return wide ? launch_rm_q<kQ4_K, true>(v, x, m, y, part, splits, st)
                            : launch_rm_q<kQ4_K, false>(v, x, m, y, part, splits, st);
    case kQ5_K: return wide ? launch_rm_q<kQ5_K, true>(v, x, m, y, part, splits, st)
                            : launch_rm_q<kQ5_K, false>(v, x, m, y, part, splits, st);
    case kQ6_K: return wide ? launch_rm_q<kQ6_K, true>(v, x, m, y, part, splits, st)
                            : launch_rm_q<kQ6_K, false>(v, x, m, y, part, splits, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace qi
