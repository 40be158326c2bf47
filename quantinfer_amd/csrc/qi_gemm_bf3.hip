// GEMM of F32 weights with f32 accuracy on the bf16 matrix cores: the
// reference's dense `matmul` (backends/cpu/src/matmul.rs:92-117), y[m, n] =
// sum_k x[m, k] W[k, n], row-major W, K and N multiples of 4.
//
// Arithmetic. Every f32 number times 2^23, the smallest subnormal too, is
// exactly the sum of three bf16 ones (bf3_pair, qi_half.h: 8 + 8 + 8 bits). Of
// the nine products of two such sums the six down to 2^-16 of the largest run on
// v_mfma_f32_16x16x32_bf16 (the other three are below 2^-24 of it), smallest
// first from a zero accumulator for each step of 32 k, whose sum joins the
// running one in one f32 fused multiply-add with 2^-46. Numbers from 2^105, or
// sums of a step from 2^82, overflow: such outputs are recomputed in the
// reference's order, correct and slow. Error against 64-bit sums,
// 2-norm, N(0, 1) x N(0, 0.02^2): 1.0e-7 at K = 2048, 1.2e-7 at K = 4096 (300
// rows), the same with weights of 2^-126 or activations of 2^-130 (without the
// factor numbers below 2^-110 lost bits: 1.8e-3 and 3.6e-2 there, for 1-3% less
// time); the f32 matrix cores (v_mfma_f32_16x16x4f32, one sixteenth of the bf16
// rate, six products here) left 1.8e-7 and 2.3e-7.
//
// Tiling. A workgroup takes 256 columns, 16 TM rows with 4 wavefronts or 32 TM
// with 8 (two groups that share the stage's weights), and one K part; wavefront
// wn its columns 64 wn .. + 63. A stage is 32 weight rows: loaded two stages
// ahead into registers as f32, split into three bf16 planes in LDS in their
// row order, and read as the matrix operand (8 k of one column per lane) by
// transposing LDS reads (ds_read_b64_tr_b16), so no lane moves are needed; a
// row stride of 544 bytes spreads the 4 rows of each read over the banks.
// With 4 wavefronts one stage is in LDS and two workgroups share a compute
// unit; with 8 the next stage is split into a second slot between the matrix
// instructions of this one.
// K parts write partial sums that launch_f32w_sum adds in order.
//
// What bounds it: the matrix cores from about 128 rows. 2048 x 4096 x 14336
// runs at 1107 TFLOP/s of bf16 products (185 TFLOP/s of the call's own), the
// rate a large bf16 library product reaches here (1105). Below, the weights'
// conversion and the start of short K parts. MI355X, us per call, the f32
// matrix-core kernel before -> now: 2048 x 8192, 16 rows 110.4 -> 25.7, 64 97.2
// -> 36.5, 128 97.8 -> 43.5, 300 158.1 -> 82, 512 171.3 -> 103; 4096 x 4096, 300
// rows 191.9 -> 85.5.
#include "qi_device.h"
#include "qi_half.h"
#include "qi_internal.h"
#include "qi_unit.h"

namespace qi {

namespace {

using namespace half;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kBStageK = 32;           // weight rows of a stage: one matrix-instruction step
constexpr uint32_t kBCols = 256;            // outputs of a workgroup, 64 per wavefront
constexpr uint32_t kBWs = 2 * kBCols + 32;  // bytes of a weight row in LDS
constexpr uint32_t kBWPlane = kBStageK * kBWs;

// A wavefront's share of a stage's weights, from memory to three bf16 planes
// in LDS.
template <int WM>
struct Weights {
  static constexpr int kLoads = 8 / WM;
  f32x4 w[kLoads];
  // rows 32s + wave + 4 WM i, columns 256u + 4 lane .. + 3 (N a multiple of 4)
  __device__ __forceinline__ void fetch(const View& v, uint32_t s, uint32_t u, uint32_t wave, uint32_t lane) {
    const float* W = reinterpret_cast<const float*>(v.qs);
    const uint64_t n = min(static_cast<uint64_t>(u) * kBCols + 4 * lane, v.n - 4);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const uint64_t k = min(static_cast<uint64_t>(s) * kBStageK + wave + 4 * WM * i, v.k - 1);
      w[i] = *reinterpret_cast<const f32x4*>(W + k * v.n + n);
    }
  }
  __device__ __forceinline__ void put_load(uint8_t* ws, uint32_t wave, uint32_t lane, int i) const {
    uint32_t p[2][3];
    bf3_pair(w[i][0], w[i][1], p[0]);
    bf3_pair(w[i][2], w[i][3], p[1]);
    uint8_t* const at = ws + (wave + 4 * WM * i) * kBWs + 8 * lane;
#pragma unroll
    for (int j = 0; j < 3; ++j) *reinterpret_cast<uint2*>(at + j * kBWPlane) = make_uint2(p[0][j], p[1][j]);
  }
  __device__ __forceinline__ void put(uint8_t* ws, uint32_t wave, uint32_t lane) const {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) put_load(ws, wave, lane, i);
  }
};

__device__ __forceinline__ float f32w_col(const View& v, const float* x, uint64_t n) {
  const float* W = reinterpret_cast<const float*>(v.qs);
  float s = 0.0f;
  for (uint64_t k = 0; k < v.k; ++k) s += x[k] * W[k * v.n + n];
  return s;
}

// Workgroup shapes: 4 wavefronts, 16 TM rows (WM = 1), or 8 wavefronts, 32 TM
// rows (WM = 2, F32 weights: two groups of 4 wavefronts share the stage's
// weights).
template <int TM, int WM>
struct Bf3Lds {
  static constexpr uint32_t kXTiles = (TM + 1) / 2 * 2 * WM;  // whole loads of the workgroup's threads
  static constexpr uint32_t kXPlane = kXTiles * 1024;
  static constexpr uint32_t kStage = 3 * kBWPlane + 3 * kXPlane;
  static constexpr uint32_t kSlots = WM;  // stages in LDS
  static constexpr uint32_t kBytes = kSlots * kStage;
  static_assert(kBytes <= 160 * 1024, "fits a compute unit");
};

template <int TM, int WM>
__global__ __launch_bounds__(256 * WM, 2) void gemm_bf3_kernel(View v, const float* __restrict__ x, uint32_t M,
                                                            uint32_t parts, float* __restrict__ out) {
  using L = Bf3Lds<TM, WM>;
  constexpr int D = TM > 3 && WM == 1 ? 1 : 2;  // stages in flight
  constexpr uint32_t XPlane = L::kXPlane;
  constexpr uint32_t MT = 16 * TM * WM;
  extern __shared__ __align__(16) uint8_t lds[];
  const uint32_t tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave & 3, wm = wave >> 2;
  const uint32_t u = blockIdx.x, m0 = blockIdx.y * MT, z = blockIdx.z;
  const uint32_t K = static_cast<uint32_t>(v.k), S = (K + kBStageK - 1) / kBStageK;
  const uint32_t sb = static_cast<uint32_t>((static_cast<uint64_t>(z) * S) / parts);
  const uint32_t se = static_cast<uint32_t>((static_cast<uint64_t>(z + 1) * S) / parts);

  // Loads past the weights or past x's rows repeat the last ones, with no
  // branch; k past K is zero in x, rows and columns past M and N are never
  // stored.
  Weights<WM> wr[D];
  constexpr int XI = L::kXTiles / (2 * WM);  // 16-byte loads of x per thread
  f32x4 xr[D][XI];
  auto fetch = [&](uint32_t s, Weights<WM>& w, f32x4 (&xx)[XI]) {
    w.fetch(v, s, u, wave, lane);
#pragma unroll
    for (int i = 0; i < XI; ++i) {
      const uint32_t e = tid + 256 * WM * i, row = min(m0 + e / 8, M - 1), k = min(s * kBStageK + 4 * (e % 8), K - 4);
      xx[i] = *reinterpret_cast<const f32x4*>(x + static_cast<uint64_t>(row) * K + k);
    }
  };
  // x in operand order: lane 16 g + r of row tile i holds row 16 i + r, k = 4 g
  // + [0, 4) and 16 + 4 g + [0, 4)
  auto put_x = [&](uint32_t s, uint8_t* st, const f32x4& xx, int i) {
    const uint32_t e = tid + 256 * WM * i, row = e / 8, q = e % 8;
    const bool live = s * kBStageK + 4 * q < K;
    uint32_t p[2][3];
    bf3_pair(live ? xx[0] : 0.0f, live ? xx[1] : 0.0f, p[0]);
    bf3_pair(live ? xx[2] : 0.0f, live ? xx[3] : 0.0f, p[1]);
    uint8_t* const at = st + 3 * kBWPlane + (row / 16) * 1024 + (16 * (q & 3) + row % 16) * 16 + 8 * (q >> 2);
#pragma unroll
    for (int j = 0; j < 3; ++j) *reinterpret_cast<uint2*>(at + j * XPlane) = make_uint2(p[0][j], p[1][j]);
  };
  auto put = [&](uint32_t s, uint8_t* st, const Weights<WM>& w, const f32x4 (&xx)[XI]) {
    w.put(st, wave, lane);
#pragma unroll
    for (int i = 0; i < XI; ++i) put_x(s, st, xx[i], i);
  };

  f32x4 acc[TM][4];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  // transposing reads: lane 16 g + c addresses row 4 g + c / 4, columns 4 (c % 4)
  // of a 16-column tile and receives column c of rows 4 g .. 4 g + 3
  const uint32_t wo = (4 * g + (c >> 2)) * kBWs + 2 * (wn * 64 + 4 * (c & 3));
  const uint32_t xo = 3 * kBWPlane + wm * TM * 1024 + lane * 16;
  // stage `st`'s products; between the matrix instructions of column tile j,
  // `beside(j)`
  auto multiply = [&](const uint8_t* st, auto beside) {
    auto read_w = [&](int j, bf16x8 (&b)[3]) {
      typedef __attribute__((address_space(3))) i16x4* lds_t;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const uint8_t* p = st + wo + i * kBWPlane + 32 * j;
        const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p));
        const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p + 16 * kBWs));
        b[i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      }
    };
    bf16x8 a[3][TM], b[2][3];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int p = 0; p < 3; ++p) a[p][i] = *reinterpret_cast<const bf16x8*>(st + xo + p * XPlane + i * 1024);
    read_w(0, b[0]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j < 3) read_w(j + 1, b[(j + 1) & 1]);
      f32x4 sum[TM];
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int i = 0; i < TM; ++i)
          sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kBf3X[q]][i], b[j & 1][kBf3W[q]],
                                                           q == 0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : sum[i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[i][j][q] = fmaf(sum[i][q], kBf3Down, acc[i][j][q]);
      beside(j);
    }
  };
  auto nothing = [](int) {};

#pragma unroll
  for (int d = 0; d < D; ++d)
    if (WM == 2 || sb + d < se) fetch(sb + d, wr[d], xr[d]);
  if constexpr (WM == 1) {
    for (uint32_t s = sb; s < se; s += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        if (s + d >= se) break;
        put(s + d, lds, wr[d], xr[d]);
        __syncthreads();
        if (s + d + D < se) fetch(s + d + D, wr[d], xr[d]);
        multiply(lds, nothing);
        __syncthreads();
      }
    }
  } else {
    // stage s + 1 goes into the other slot while stage s is multiplied; past
    // the last stage both the loads (in bounds: rows past K are zero) and the
    // slot they fill are unused, so that the loop body has no branch and the
    // conversion can run between the matrix instructions
    put(sb, lds, wr[0], xr[0]);
    fetch(sb + 2, wr[0], xr[0]);
    __syncthreads();
    auto stage = [&](uint32_t s, uint32_t slot, Weights<WM>& w, f32x4 (&xx)[XI]) {
      uint8_t* const next = lds + (1 - slot) * L::kStage;
      multiply(lds + slot * L::kStage, [&](int j) {
        if (j < Weights<WM>::kLoads) w.put_load(next, wave, lane, j);
        if (j < XI) put_x(s + 1, next, xx[j], j);
        if (j == 3) fetch(s + 3, w, xx);
#pragma unroll
        for (int i = 0; i < 6 * TM; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one matrix instruction,
          __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // three vector ones
        }
        __builtin_amdgcn_sched_barrier(0);
      });
      __syncthreads();
    };
    uint32_t s = sb;
    for (; s + 1 < se; s += 2) {
      stage(s, 0, wr[1], xr[1]);
      stage(s + 1, 1, wr[0], xr[0]);
    }
    if (s < se) multiply(lds, nothing);
  }

  // lane 16 g + c holds rows 4 g .. 4 g + 3 of each 16 x 16 block, column c
  float* const dst = out + (parts == 1 ? 0 : static_cast<uint64_t>(z) * M * v.n);
  bool bad = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint64_t col = static_cast<uint64_t>(u) * kBCols + wn * 64 + j * 16 + c;
      if (col >= v.n) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t m = m0 + (wm * TM + i) * 16 + 4 * g + q;
        if (m >= M) continue;
        bad |= !__builtin_isfinite(acc[i][j][q]);
        dst[static_cast<uint64_t>(m) * v.n + col] = acc[i][j][q];
      }
    }
  // with one part, a non-finite sum (NaN or infinite activations, or an
  // overflow) is recomputed in the reference's order, which decides NaN or
  // +-Inf; this lane's own stores are read back (a loop of its own, so that
  // the accumulators above stay in registers)
  if (parts == 1 && bad) {
#pragma unroll 1
    for (int e = 0; e < TM * 16; ++e) {
      const uint32_t i = e / 16, j = (e / 4) % 4, q = e % 4, m = m0 + (wm * TM + i) * 16 + 4 * g + q;
      const uint64_t col = static_cast<uint64_t>(u) * kBCols + wn * 64 + j * 16 + c;
      if (m >= M || col >= v.n) continue;
      float* p = dst + static_cast<uint64_t>(m) * v.n + col;
      const float* xm = x + static_cast<uint64_t>(m) * K;
      if (!__builtin_isfinite(*p)) *p = f32w_col(v, xm, col);
    }
  }
}

uint64_t units_of(const Image& im) { return (im.n + kBCols - 1) / kBCols; }
uint64_t stages_of(const Image& im) { return (im.k + kBStageK - 1) / kBStageK; }

template <int TM, int WM>
hipError_t launch_bf3(const Image& im, const View& v, const float* x, uint32_t m, float* out, uint32_t parts,
                      hipStream_t st) {
  constexpr uint32_t rows = 16 * TM * WM;
  auto kern = gemm_bf3_kernel<TM, WM>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           static_cast<int>(Bf3Lds<TM, WM>::kBytes));
  if (e != hipSuccess) return e;
  const dim3 grid(static_cast<uint32_t>(units_of(im)), (m + rows - 1) / rows, parts);
  hipLaunchKernelGGL(kern, grid, dim3(256 * WM), (Bf3Lds<TM, WM>::kBytes), st, v, x, m, parts, out);
  return hipGetLastError();
}

}  // namespace

bool gemm_bf3_supported(const Image& im) {
  return im.qtype == kF32 && im.layout == kRowMajor && im.n % 4 == 0 && im.k % 4 == 0 && im.k > 0 &&
         im.k <= 0x7fffffe0ull;
}

Bf3Plan gemm_bf3_plan(const Image& im, uint64_t m, uint64_t max_part_floats) {
  // The tile and part count with the least modelled time: the stages of a
  // part, each at the tile's time with one workgroup on a compute unit or with
  // two (4-wavefront tiles: two fit), for every round of resident workgroups;
  // and with parts the sum launch and the partial sums' trip. The stage times
  // are fits to every tile and part counts 1 to 16 at 2048 x 8192, 16 to 512
  // rows. Of 17 calls at K 512 to 14336 and N 1024 to 24576 the model is within
  // 15% at 12 (from 40 rows) and 24% high at 12 us; it is 17-30% low at 16 and 20
  // rows of large weights, whose bytes, the same for every tile and part count,
  // it does not count (MI355X).
  struct Tile {
    uint32_t tm, wm;
    double one_us, two_us;
  };
  constexpr Tile kTiles[] = {{1, 1, 1.5, 1.9}, {2, 1, 1.75, 2.3}, {3, 1, 2.0, 2.9},
                             {4, 1, 2.2, 3.3}, {3, 2, 2.1, 0.0}, {4, 2, 2.4, 0.0}};
  constexpr uint32_t kParts[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32};
  constexpr double kFixedUs = 8.0, kSumUs = 3.0, kPartUsPerByte = 0.25e-6;
  constexpr uint64_t kCUs = 256;
  const uint64_t units = units_of(im), stages = stages_of(im);
  Bf3Plan best;
  double best_us = 0.0;
  for (const Tile& t : kTiles) {
    const uint64_t rows = 16 * t.tm * t.wm, blocks = units * ((m + rows - 1) / rows);
    // no taller than the call needs, but for its last row tile
    if (best.tm != 0 && rows >= m + 16 * t.wm) continue;
    for (const uint32_t p : kParts) {
      const uint64_t bytes = p > 1 ? p * m * im.n * 4 : 0;
      if (p > 1 && (2 * p > stages || bytes > 4 * max_part_floats)) break;
      const uint64_t n = blocks * p, per = kCUs * (t.wm == 1 ? 2 : 1);
      const uint64_t full = n / per, rest = n % per;
      const double round_us = t.wm == 1 ? t.two_us : t.one_us;
      const double rest_us = rest == 0 ? 0.0 : rest <= kCUs ? t.one_us : t.two_us;
      const double us = static_cast<double>((stages + p - 1) / p) * (static_cast<double>(full) * round_us + rest_us) +
                        kFixedUs + (p > 1 ? kSumUs + static_cast<double>(bytes) * kPartUsPerByte : 0.0);
      if (best.tm == 0 || us < best_us) {
        best = Bf3Plan{t.tm, t.wm, p};
        best_us = us;
      }
    }
  }
  return best;
}

hipError_t launch_gemm_bf3(const Image& im, const View& v, const float* x, uint64_t m, float* y, float* part,
                           const Bf3Plan& plan, hipStream_t st) {
  const uint32_t parts = plan.parts;
  if (!gemm_bf3_supported(im) || m < 1 || m > 0xFFFFull * 16 || parts < 1 || parts > 0xFFFFu ||
      parts > stages_of(im) || (parts > 1 && part == nullptr) || units_of(im) > 0x7fffffffull ||
      (m * im.n + 255) / 256 > 0x7fffffffull)
    return hipErrorInvalidValue;
  const uint32_t mm = static_cast<uint32_t>(m);
  float* const out = parts > 1 ? part : y;
  hipError_t e = hipErrorInvalidValue;
  switch (4 * plan.wm + plan.tm) {
    case 5: e = launch_bf3<1, 1>(im, v, x, mm, out, parts, st); break;
    case 6: e = launch_bf3<2, 1>(im, v, x, mm, out, parts, st); break;
    case 7: e = launch_bf3<3, 1>(im, v, x, mm, out, parts, st); break;
    case 8: e = launch_bf3<4, 1>(im, v, x, mm, out, parts, st); break;
    case 11: e = launch_bf3<3, 2>(im, v, x, mm, out, parts, st); break;
    case 12: e = launch_bf3<4, 2>(im, v, x, mm, out, parts, st); break;
    default: break;
  }
  if (e != hipSuccess || parts == 1) return e;
  return launch_f32w_sum(v, part, parts, m * im.n, y, x, st);
}

}  // namespace qi
