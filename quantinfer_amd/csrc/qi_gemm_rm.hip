// Row-major (blocks along N) GEMM on the f16 matrix cores with f32 accuracy:
// y[m, n] = sum_k x[m, k] w(k, n) for QuantInfer-layout weights
// (backends/cpu/src/backend.rs:62-140 -> matmul.rs:14-90; element values
// matmul.rs:162-280), from 3 or 5 rows (rm_gemm_min_rows, qi_abi.hip), tiled
// images with f16 scales.
//
// Arithmetic (the split halves of qi_half.h, with the scales that change along
// k on the activations' side). A weight is d s (q - z) - b', with d the scale
// of its (k, 256 outputs) block for the K-quants:
//   Q4_K/Q5_K  x' = x d; sc (q - z) is an exact f16 integer, z the integer
//              nearest the window's offset over its scale, at most the largest
//              code; the offsets left, |b'| <= d sc / 2 (more only past the
//              largest code, where every weight of the window has their sign),
//              one per (k, window of 32 outputs), are a product of their own
//              with x, both as three exact bf16 pieces;
//   Q6_K       x' = x d; sc (q - 32) has up to 12 bits: two exact f16 planes;
//   Q8_0/Q4_0  x' = x; d q has up to 19 bits: two exact f16 planes (scales in
//              the range plan_image calls f16_gemm).
// Per row and 64 k, x' is scaled by a power of two that brings the largest
// under 2^15 and held as two f16 halves, 23 bits. v_mfma_f32_16x16x32_f16 then
// sums the exact products of all parts, smallest first (without that of the two
// low parts, 2^-22 of the product, 4 x 256 missed the 1e-5 bar), and each 64 k
// join the running sum in one f32 fused multiply-add with the scale. The low
// half ends at f16's last bit, 2^-39 of the largest: where a wavefront finds an
// activation under 2^-18 of its row's largest, what the halves leave makes two
// further pieces, and the row tiles concerned run a product with each
// (multiply_rest; the second one only where an activation is under 2^-24). So
// every activation keeps 22 bits down to 2^-53 of the largest of its 64 k;
// without them, outputs with zero codes at an activation 1e8 times the others
// had errors of 3e-5 to 6e-5, now as without it, to 1e15 times. (x d below 2^-126, x near 2^-113, has the bits of f32's subnormals.)
// N(0, 1) activations need the first in 4% of a 64-row tile's chunks: 1-2%
// of the time, finding them 2%.
// Error against 64-bit sums, 2-norm, N(0, 1) activations, before (f32 matrix
// cores) -> now: Q8_0 4096 x 4096 130 rows 1.4e-7 -> 1.2e-7, Q4_K 4096 x 14336
// 512 rows 2.3e-7 -> 1.8e-7, Q6_K 14336 x 4096 16 rows 1.6e-7 -> 1.4e-7. One-hot
// activations give the dequantized weights bit for bit, as before.
//
// Tiling. A workgroup of 4 wavefronts takes one unit (256 outputs), 16 TM rows
// and one K part; wavefront w its outputs 64 w .. + 63. A stage is 32 weight
// rows (two record tiles; each wavefront converts half of one tile's record)
// loaded two stages ahead into registers. The codes go to LDS as f16 in row
// order and are read as the matrix operand (8 k of one output per lane) by
// transposing LDS reads (ds_read_b64_tr_b16); a row stride of 544 bytes
// spreads the 4 rows of each read over the banks. The activations of 64 k are
// converted once per workgroup. Two workgroups share a compute unit. K parts
// write partial sums that rm_sum_kernel adds in order.
//
// What bounds it: the conversions' vector instructions (Q4_K about 110 per
// wavefront and stage for the weights, 90 for 64 rows of activations, against
// 38 matrix instructions of 16 cycles), which slow down from 5 to 8-11 cycles
// each while the other wavefront of a SIMD runs matrix instructions. MI355X, us
// per call, the f32 matrix-core kernel (wide scales still take it) -> this one:
// Q8_0 4096 x 4096 5 rows 16.3 -> 14.8, 16 17.0 -> 15.6, 130 65.4 -> 42, 512 170
// -> 92; Q4_K 4096 x 14336 16 rows 38 -> 29.3, 130 235 -> 102, 512 655 -> 314;
// Q6_K 14336 x 4096 512 rows 619 -> 272; Q4_0 4096 x 12288 64 rows 79 -> 50.5, 512
// rows 504 -> 283.
#include "qi_device.h"
#include "qi_half.h"
#include "qi_internal.h"
#include "qi_unit.h"

#include <type_traits>

namespace qi {

namespace {

using namespace half;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kRChunk = 64;      // k of one activation scale: two stages
constexpr uint32_t kRStage = 32;      // weight rows of a stage: one matrix-instruction step
constexpr uint32_t kRWs = 512 + 32;   // bytes of a weight row in LDS (256 f16 and padding)
constexpr uint32_t kRWPlane = kRStage * kRWs;

template <int QT>
struct RmFmt {
  static constexpr bool kK45 = QT == kQ4_K || QT == kQ5_K;
  static constexpr bool kD = kK45 || QT == kQ6_K;  // the activations carry the block scale d
  static constexpr int kPlanes = kK45 ? 1 : 2;
};

template <int QT, int TM>
struct RmLds {
  using F = RmFmt<QT>;
  static constexpr uint32_t kW = 0;
  static constexpr uint32_t kOff = F::kPlanes * kRWPlane;            // offsets [piece][k][16] bf16 (K45)
  static constexpr uint32_t kX = kOff + (F::kK45 ? 3 * kRStage * 32 : 0);
  static constexpr uint32_t kXHalf = 2 * TM * 1024;                  // one half [stage][row tile][lane] x 16 B
  static constexpr uint32_t kXP = kX + 2 * kXHalf;                   // x's bf16 pieces, likewise (K45)
  static constexpr uint32_t kXRest = kXP + (F::kK45 ? 3 * kXHalf : 0);  // what the halves leave: two pieces, likewise
  static constexpr uint32_t kUnsc = kXRest + 2 * kXHalf;
  static constexpr uint32_t kFlag = kUnsc + TM * 16 * 4;             // [row tile][wavefront]: 2 (chunk + 1) + second piece
  static constexpr uint32_t kBytes = kFlag + TM * 4 * 4;
  static_assert(2 * kBytes <= 160 * 1024, "two workgroups on a compute unit");
};

// The half of a record that one wavefront of a stage converts: of each lane's
// 64 outputs, the 32 of code chunk `half` (K-quants: steps 2 half, 2 half + 1
// of both windows; Q8_0 / Q4_0: window `half`). The chunk takes the first
// slots of Raw, so step j (0..3) of the half is step half_step(j) of Raw.
template <int QT>
__device__ __forceinline__ void load_half(const uint8_t* rec, uint32_t lane, uint32_t half,
                                          typename Unit<QT>::Raw& r) {
  constexpr Record R = record_geometry(QT, false);
  const uint32_t col = lane & 15, g = lane >> 4;
  const uint4* p = reinterpret_cast<const uint4*>(rec + R.qs) + lane;
  if constexpr (QT == kQ8_0 || QT == kQ4_0) {
    if constexpr (QT == kQ8_0) {
      r.q[0] = p[128 * half];
      r.q[1] = p[128 * half + 64];
    } else {
      r.q[0] = p[64 * half];
    }
    r.s0 = reinterpret_cast<const uint16_t*>(rec + R.d)[col * 8 + 2 * g + half];
  } else if constexpr (QT == kQ6_K) {
    r.q[0] = p[64 * half];
    r.h[0] = (reinterpret_cast<const uint4*>(rec + R.qh) + 32 * (lane >> 5) + col)[16 * half];
    r.sc = *reinterpret_cast<const uint32_t*>(rec + R.sc + col * 16 + 4 * g);
  } else {
    r.q[0] = p[64 * half];
    if constexpr (QT == kQ5_K) r.h[0] = (reinterpret_cast<const uint4*>(rec + R.qh) + col)[16 * half];
    const uint32_t* s = reinterpret_cast<const uint32_t*>(rec + R.sc + col * 12);
    r.sc[0] = s[0];
    r.sc[1] = s[1];
    r.sc[2] = s[2];
    r.s0 = reinterpret_cast<const uint16_t*>(rec + R.d)[col];
    r.s1 = reinterpret_cast<const uint16_t*>(rec + R.dmin)[col];
  }
}

template <int QT>
constexpr int half_step(int j) {
  return QT == kQ8_0 || QT == kQ4_0 ? j : (j & 1) + 4 * (j >> 1);
}
template <int QT>
__device__ __forceinline__ uint32_t half_first(uint32_t g, uint32_t half, int j) {
  if constexpr (QT == kQ8_0 || QT == kQ4_0) return window_first<QT>(g, half) + 8 * j;
  else return window_first<QT>(g, j >> 1) + 8 * (2 * half + (j & 1));
}

// Factors of a lane's half record for split_codes, and (K45) the offset
// -(b - a z) of window 2g + half.
template <int QT>
__device__ __forceinline__ float half_scales(const typename Unit<QT>::Raw& r, uint32_t g, uint32_t half,
                                             SplitScales& o) {
  if constexpr (QT == kQ8_0 || QT == kQ4_0) {
    o.sc[0] = splat(f16_bits(r.s0));
    return 0.0f;
  } else if constexpr (QT == kQ6_K) {
    // sub-scales half and 2 + half of the lane group's four
    const uint32_t s = r.sc >> (8 * half);
    o.sc[0] = splat(static_cast<float>(static_cast<int32_t>(s << 24) >> 24));
    o.sc[2] = splat(static_cast<float>(static_cast<int32_t>(s << 8) >> 24));
    return 0.0f;
  } else {
    constexpr float kQMax = QT == kQ5_K ? 31.0f : 15.0f;
    float d, dmin, off[2];
    Unit<QT>::template dmins<false>(r, d, dmin);
    const uint32_t f = Unit<QT>::field(g, r);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float sc = static_cast<float>((f >> (12 * h)) & 63u), mn = static_cast<float>((f >> (12 * h + 6)) & 63u);
      const float a = d * sc, b = dmin * mn;  // both exact in f32
      const float z = fminf(fmaxf(rintf(b * __builtin_amdgcn_rcpf(a)), 0.0f), kQMax);
      off[h] = fmaf(a, z, -b);
      o.sc[h] = splat(sc);
      o.c[h] = splat(h == 0 ? -(1024.0f + z) : -(64.0f + z));
    }
    return half ? off[1] : off[0];
  }
}

template <int QT, int TM>
__global__ __launch_bounds__(256, 2) void gemm_rm_kernel(View v, const float* __restrict__ x, uint32_t M,
                                                         uint32_t parts, float* __restrict__ out) {
  using F = RmFmt<QT>;
  using L = RmLds<QT, TM>;
  constexpr int NP = F::kPlanes;
  constexpr Record R = record_geometry(QT, false);
  extern __shared__ __align__(16) uint8_t lds[];
  const uint32_t tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t u = blockIdx.x, m0 = blockIdx.y * TM * 16, z = blockIdx.z;
  const uint32_t K = static_cast<uint32_t>(v.k), C = (K + kRChunk - 1) / kRChunk;
  const uint32_t cb = static_cast<uint32_t>((static_cast<uint64_t>(z) * C) / parts);
  const uint32_t ce = static_cast<uint32_t>((static_cast<uint64_t>(z + 1) * C) / parts);
  const uint8_t* const base = v.qs + static_cast<uint64_t>(u) * R.bytes;
  const uint64_t tile_bytes = static_cast<uint64_t>(v.units) * R.bytes;

  // Loads past the weights or past x's rows repeat the last ones; k past K is
  // zero in x, rows past M are never stored.
  typename Unit<QT>::Raw wr[2];
  v4f xr[TM];
  uint2 dr[TM];
  auto fetch_w = [&](uint32_t s, typename Unit<QT>::Raw& r) {
    const uint32_t t = min(2 * s + (wave >> 1), v.tiles - 1);
    load_half<QT>(base + t * tile_bytes, lane, wave & 1, r);
  };
  auto fetch_x = [&](uint32_t chunk) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const uint32_t e = tid + 256 * i, row = min(m0 + e / 16, M - 1), k = min(chunk * kRChunk + 4 * (e % 16), K - 4);
      xr[i] = *reinterpret_cast<const v4f*>(x + static_cast<uint64_t>(row) * K + k);
      if constexpr (F::kD) dr[i] = *reinterpret_cast<const uint2*>(base + (k / 16) * tile_bytes + R.d + 2 * (k % 16));
    }
  };
  // the chunk's activations (times d): one power of two per row that brings
  // the largest under 2^15, hi = f16(x') and lo = f16(x' - hi) in operand
  // order (lane 16 g + r of a row tile: k = 4 g + [0, 4) and 16 + 4 g +
  // [0, 4) of a stage); K45: x's bf16 pieces beside them
  auto put_x = [&](uint32_t chunk) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const uint32_t e = tid + 256 * i, row = e / 16, q = e % 16;
      const bool live = chunk * kRChunk + 4 * q < K;
      float xv[4], v4[4], mx = 0.0f;
      uint32_t least = ~0u;  // bits of the smallest magnitude above zero, doubled, less 1
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        xv[j] = live ? xr[i][j] : 0.0f;
        v4[j] = F::kD ? xv[j] * f16_bits((j < 2 ? dr[i].x : dr[i].y) >> (16 * (j & 1))) : xv[j];
        mx = fmaxf(mx, fabsf(v4[j]));
        least = min(least, (__builtin_bit_cast(uint32_t, v4[j]) << 1) - 1);
      }
      mx = fmaxf(mx, dpp_move<0x121>(mx));
      mx = fmaxf(mx, dpp_move<0x122>(mx));
      mx = fmaxf(mx, dpp_move<kDppRor4>(mx));
      mx = fmaxf(mx, dpp_move<kDppRor8>(mx));
      // (a NaN or infinite activation stays non-finite through the halves:
      // its row's outputs are recomputed in the reference's order)
      const int ex = __builtin_isfinite(mx) && mx > 0.0f ? __builtin_amdgcn_frexp_expf(mx) : 0;
      const int sh = min(15 - ex, 125);
      const float scale = __builtin_bit_cast(float, static_cast<uint32_t>(127 + sh) << 23);
      const float unscale = __builtin_bit_cast(float, static_cast<uint32_t>(127 - sh) << 23);  // 2^-sh
      uint32_t hi[2], lo[2];
      f32x2 r[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        // both halves rounded to nearest: 23 bits together
        const f32x2 s = {v4[2 * j] * scale, v4[2 * j + 1] * scale};
        const h2 h = __builtin_convertvector(s, h2);
        r[j] = f32x2{s[0] - static_cast<float>(h[0]), s[1] - static_cast<float>(h[1])};
        hi[j] = h2u(h);
        lo[j] = h2u(__builtin_convertvector(r[j], h2));
      }
      const uint32_t at = (q / 8) * TM * 1024 + (row / 16) * 1024 + (16 * (q & 3) + row % 16) * 16 + 8 * ((q >> 2) & 1);
      *reinterpret_cast<uint2*>(lds + L::kX + at) = make_uint2(hi[0], hi[1]);
      *reinterpret_cast<uint2*>(lds + L::kX + L::kXHalf + at) = make_uint2(lo[0], lo[1]);
      if (q == 0) *reinterpret_cast<float*>(lds + L::kUnsc + 4 * row) = unscale;
      // a number under 2^-18 of the row's largest, of which the low half, ending
      // at f16's last bit, keeps fewer than 22 bits: the rest of this
      // wavefront's rows, times 2^24, as two halves 2^12 apart. Numbers under
      // 2^-24 of it go there whole: beside the largest, a matrix instruction
      // drops bits of products near 2^-42.
      auto under = [&](float bound) { return __any(least < (__builtin_bit_cast(uint32_t, unscale * bound) << 1) - 1); };
      if (under(0x1p-3f)) {
        uint32_t rest[2][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const h2 l = __builtin_bit_cast(h2, lo[j]);
          f32x2 t, t2;
          uint32_t keep = 0;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float s = v4[2 * j + e] * scale;
            const bool halves = fabsf(s) >= 0x1p-9f;
            t[e] = (halves ? r[j][e] - static_cast<float>(l[e]) : s) * 0x1p24f;
            keep |= halves ? 0xFFFFu << (16 * e) : 0u;
          }
          const h2 h = __builtin_convertvector(t, h2);
#pragma unroll
          for (int e = 0; e < 2; ++e) t2[e] = (t[e] - static_cast<float>(h[e])) * 0x1p12f;
          rest[0][j] = h2u(h);
          rest[1][j] = h2u(__builtin_convertvector(t2, h2));
          hi[j] &= keep;
          lo[j] &= keep;
        }
        *reinterpret_cast<uint2*>(lds + L::kX + at) = make_uint2(hi[0], hi[1]);
        *reinterpret_cast<uint2*>(lds + L::kX + L::kXHalf + at) = make_uint2(lo[0], lo[1]);
#pragma unroll
        for (int p = 0; p < 2; ++p)
          *reinterpret_cast<uint2*>(lds + L::kXRest + p * L::kXHalf + at) = make_uint2(rest[p][0], rest[p][1]);
        const uint32_t second = under(0x1p-9f) ? 1 : 0;  // numbers above it end with the first piece
        if (lane == 0) *reinterpret_cast<uint32_t*>(lds + L::kFlag + 16 * i + 4 * wave) = 2 * (chunk + 1) + second;
      }
      if constexpr (F::kK45) {
        uint32_t p[2][3];
        bf3_pair(xv[0], xv[1], p[0]);
        bf3_pair(xv[2], xv[3], p[1]);
#pragma unroll
        for (int j = 0; j < 3; ++j)
          *reinterpret_cast<uint2*>(lds + L::kXP + j * L::kXHalf + at) = make_uint2(p[0][j], p[1][j]);
      }
    }
  };
  // a stage's weight codes [plane][k][256 outputs, each 8 in the order 0 2 1 3
  // 4 6 5 7] and offsets
  auto put_w = [&](const typename Unit<QT>::Raw& r) {
    const uint32_t half = wave & 1, k = 16 * (wave >> 1) + c;
    SplitScales sc;
    const float off = half_scales<QT>(r, g, half, sc);
    uint8_t* const row = lds + k * kRWs;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t b[NP][4];
      split_codes<QT>(r, g, half_step<QT>(j), sc, b);
#pragma unroll
      for (int p = 0; p < NP; ++p)
        *reinterpret_cast<uint4*>(row + p * kRWPlane + 2 * half_first<QT>(g, half, j)) =
            make_uint4(b[p][0], b[p][1], b[p][2], b[p][3]);
    }
    if constexpr (F::kK45) {
      uint32_t p[3];
      bf3_pair(off, 0.0f, p);
#pragma unroll
      for (int j = 0; j < 3; ++j)
        *reinterpret_cast<uint16_t*>(lds + L::kOff + j * kRStage * 32 + k * 32 + 2 * (2 * g + half)) =
            static_cast<uint16_t>(p[j]);
    }
  };

  v4f acc[TM][4], part[TM][4], aoff = {0.0f, 0.0f, 0.0f, 0.0f};
  const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zero;

  // transposing reads: lane 16 g + c addresses row 4 g + c / 4, columns 4 (c % 4)
  // of a 16-column tile and receives column c of rows 4 g .. 4 g + 3
  typedef __attribute__((address_space(3))) i16x4* lds_t;
  auto read_t = [&](const uint8_t* p, uint32_t stride) {
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p + 16 * stride));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  const uint8_t* const wb = lds + (4 * g + (c >> 2)) * kRWs + 2 * (wave * 64 + 4 * (c & 3));
  auto multiply = [&](auto sub) {
    constexpr int kSub = decltype(sub)::value;
    h8 ahi[TM], alo[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const uint8_t* const p = lds + L::kX + (kSub * TM + i) * 1024 + lane * 16;
      ahi[i] = *reinterpret_cast<const h8*>(p);
      alo[i] = *reinterpret_cast<const h8*>(p + L::kXHalf);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h8 b[NP];
#pragma unroll
      for (int p = 0; p < NP; ++p) b[p] = __builtin_bit_cast(h8, read_t(wb + p * kRWPlane + 32 * j, kRWs));
#pragma unroll
      for (int i = 0; i < TM; ++i)
        part[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[i], b[NP - 1], kSub == 0 ? zero : part[i][j], 0, 0, 0);
      if constexpr (NP == 2) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
          part[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(alo[i], b[0], part[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
          part[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[i], b[NP - 1], part[i][j], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
        part[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ahi[i], b[0], part[i][j], 0, 0, 0);
    }
    if constexpr (F::kK45) {
      // offsets of row tile `wave`: x's pieces times the offsets', eight
      // windows in a 16-column tile, the smallest products first
      if (wave < static_cast<uint32_t>(TM)) {
        bf16x8 a[3], b[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
          a[p] = *reinterpret_cast<const bf16x8*>(lds + L::kXP + p * L::kXHalf + (kSub * TM + wave) * 1024 + lane * 16);
          b[p] = __builtin_bit_cast(
              bf16x8, read_t(lds + L::kOff + p * kRStage * 32 + (4 * g + (c >> 2)) * 32 + 8 * (c & 3), 32));
        }
        v4f s = zero;
#pragma unroll
        for (int q = 0; q < 6; ++q) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kBf3X[q]], b[kBf3W[q]], s, 0, 0, 0);
#pragma unroll
        for (int q = 0; q < 4; ++q) aoff[q] = fmaf(s[q], kBf3Down, aoff[q]);
      }
    }
  };

  // a stage's products with what the halves left of the activations, in the
  // row tiles of the chunk where put_x found such rows (the others' are zero)
  auto multiply_rest = [&](auto sub, uint32_t chunk) {
    constexpr int kSub = decltype(sub)::value;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const uint32_t flag = *reinterpret_cast<const uint32_t*>(lds + L::kFlag + 16 * i + 4 * (c >> 2));
      const bool mine = flag / 2 == chunk + 1;
      if (!__any(mine)) continue;
      const bool second = __any(mine && flag % 2 != 0);
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if (p == 1 && !second) break;
        h8 a = *reinterpret_cast<const h8*>(lds + L::kXRest + p * L::kXHalf + (kSub * TM + i) * 1024 + lane * 16);
        if (!mine) a = h8{};
        const float4 us = *reinterpret_cast<const float4*>(lds + L::kUnsc + 4 * (16 * i + 4 * g));
        const float uu[4] = {us.x, us.y, us.z, us.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v4f s = zero;
#pragma unroll
          for (int n = NP - 1; n >= 0; --n)
            s = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                a, __builtin_bit_cast(h8, read_t(wb + n * kRWPlane + 32 * j, kRWs)), s, 0, 0, 0);
#pragma unroll
          for (int q = 0; q < 4; ++q)
            acc[i][j][q] = fmaf(uu[q] * (p == 0 ? 0x1p-24f : 0x1p-36f), s[q], acc[i][j][q]);
          __builtin_amdgcn_sched_barrier(0);  // one tile at a time: its registers are few
        }
      }
    }
  };

  constexpr bool kLate = TM == 4;  // the next chunk's activations a stage later: 256 registers hold no more
  const uint32_t sb = 2 * cb;
  // a wavefront's flags are its own writes: no barrier before put_x
  if (lane < static_cast<uint32_t>(TM)) *reinterpret_cast<uint32_t*>(lds + L::kFlag + 16 * lane + 4 * wave) = 0;
  fetch_x(cb);
  fetch_w(sb, wr[0]);
  fetch_w(sb + 1, wr[1]);
  for (uint32_t ch = cb; ch < ce; ++ch) {
    put_x(ch);
    put_w(wr[0]);
    __syncthreads();
    const bool rest =
        __any(*reinterpret_cast<const uint32_t*>(lds + L::kFlag + 4 * (lane % (4 * TM))) / 2 == ch + 1);
    if constexpr (!kLate) fetch_x(ch + 1);
    fetch_w(2 * ch + 2, wr[0]);
    multiply(std::integral_constant<int, 0>{});
    if (rest) multiply_rest(std::integral_constant<int, 0>{}, ch);
    __syncthreads();
    put_w(wr[1]);
    __syncthreads();
    if constexpr (kLate) fetch_x(ch + 1);
    fetch_w(2 * ch + 3, wr[1]);
    multiply(std::integral_constant<int, 1>{});
    if (rest) multiply_rest(std::integral_constant<int, 1>{}, ch);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const float4 us = *reinterpret_cast<const float4*>(lds + L::kUnsc + 4 * (16 * i + 4 * g));
      const float uu[4] = {us.x, us.y, us.z, us.w};
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[i][j][q] = fmaf(uu[q], part[i][j][q], acc[i][j][q]);
    }
    __syncthreads();
  }

  // offsets [row][16] through LDS
  if constexpr (F::kK45) {
    float* const o = reinterpret_cast<float*>(lds);
    if (wave < static_cast<uint32_t>(TM)) {
#pragma unroll
      for (int q = 0; q < 4; ++q) o[(16 * wave + 4 * g + q) * 16 + c] = aoff[q];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float2 f = *reinterpret_cast<const float2*>(o + (16 * i + 4 * g + q) * 16 + 2 * wave);
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j][q] += j < 2 ? f.x : f.y;
      }
  }

  // lane 16 g + c holds rows 4 g .. 4 g + 3 of each 16 x 16 block, memory column c
  const uint32_t cc = 8 * (c >> 3) + ((0x75643120u >> (4 * (c & 7))) & 7u);
  float* const dst = out + (parts == 1 ? 0 : static_cast<uint64_t>(z) * M * v.n);
  bool bad = false;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint64_t n = static_cast<uint64_t>(u) * 256 + wave * 64 + j * 16 + cc;
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
      const uint64_t n = static_cast<uint64_t>(u) * 256 + wave * 64 + j * 16 + cc;
      float* p = dst + static_cast<uint64_t>(m) * v.n + n;
      if (m < M && !__builtin_isfinite(*p)) *p = exact_row_major_col<QT, false>(v, x + static_cast<uint64_t>(m) * K, n);
    }
  }
}

template <int QT, int TM>
hipError_t launch_rm_t(const View& v, const float* x, uint32_t m, float* out, uint32_t parts, hipStream_t st) {
  constexpr uint32_t bytes = RmLds<QT, TM>::kBytes;
  auto kern = gemm_rm_kernel<QT, TM>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(v.units, (m + 16 * TM - 1) / (16 * TM), parts), dim3(256), bytes, st, v, x, m, parts,
                     out);
  return hipGetLastError();
}

// Q5_K's 64-row tile does not fit 256 registers.
constexpr uint32_t rm_max_tm(int32_t qtype) { return qtype == kQ5_K ? 3 : 4; }

template <int QT>
hipError_t launch_rm_q(const View& v, const float* x, uint32_t m, float* out, const RmPlan& p, hipStream_t st) {
  switch (p.tm) {
    case 1: return launch_rm_t<QT, 1>(v, x, m, out, p.parts, st);
    case 2: return launch_rm_t<QT, 2>(v, x, m, out, p.parts, st);
    case 3: return launch_rm_t<QT, 3>(v, x, m, out, p.parts, st);
    case 4:
      if constexpr (rm_max_tm(QT) >= 4) return launch_rm_t<QT, 4>(v, x, m, out, p.parts, st);
      break;
    default: break;
  }
  return hipErrorInvalidValue;
}

}  // namespace

bool gemm_rm_supported(const Image& im) {
  if (im.layout != kRowMajor || !im.tiled || im.wide || im.k % 4 != 0 || im.k > 0x7fffffc0ull || im.units > 0xFFFFu)
    return false;
  switch (im.qtype) {
    case kQ8_0:
    case kQ4_0: return im.f16_gemm != 0;  // code times scale is exact as two f16 halves
    case kQ4_K:
    case kQ5_K:
    case kQ6_K: return true;
    default: return false;
  }
}

RmPlan gemm_rm_plan(const Image& im, uint64_t m, uint64_t max_part_floats) {
  // The tile and part count with the least modelled time: the 64-row chunks of
  // a part, each at the tile's time with one workgroup on a compute unit or
  // with two, for every round of resident workgroups; and with parts the sum
  // launch and the partial sums' trip. The chunk times are fits to every tile
  // and part counts 1 to 24 at Q8_0 4096 x 4096, Q4_K 4096 x 14336 and Q6_K
  // 14336 x 4096, 16 to 512 rows (MI355X, model mostly within 10%).
  constexpr double kOne[] = {1.55, 1.95, 2.3, 2.7}, kTwo[] = {2.1, 2.85, 3.6, 4.3};
  constexpr uint32_t kParts[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32};
  constexpr double kFixedUs = 5.0, kSumUs = 2.0, kPartUsPerByte = 0.25e-6;
  constexpr uint64_t kCUs = 256;
  const uint64_t chunks = (im.k + kRChunk - 1) / kRChunk, row_tiles = (m + 15) / 16;
  RmPlan best;
  double best_us = 0.0;
  for (uint32_t tm = 1; tm <= rm_max_tm(im.qtype) && tm <= row_tiles; ++tm) {
    const uint64_t blocks = im.units * ((row_tiles + tm - 1) / tm);
    for (const uint32_t p : kParts) {
      const uint64_t bytes = p > 1 ? p * m * im.n * 4 : 0;
      if (p > chunks || bytes > 4 * max_part_floats) break;
      const uint64_t n = blocks * p, full = n / (2 * kCUs), rest = n % (2 * kCUs);
      const double us = static_cast<double>((chunks + p - 1) / p) *
                            (static_cast<double>(full) * kTwo[tm - 1] +
                             (rest == 0 ? 0.0 : rest <= kCUs ? kOne[tm - 1] : kTwo[tm - 1])) +
                        kFixedUs + (p > 1 ? kSumUs + static_cast<double>(bytes) * kPartUsPerByte : 0.0);
      if (best.tm == 0 || us < best_us) {
        best = RmPlan{tm, p};
        best_us = us;
      }
    }
  }
  return best;
}

hipError_t launch_gemm_rm(const Image& im, const View& v, const float* x, uint64_t m, float* y, float* part,
                          const RmPlan& plan, hipStream_t st) {
  const uint32_t parts = plan.parts;
  if (!gemm_rm_supported(im) || m < 1 || m > 0xFFFFull * 16 || parts < 1 || parts > 0xFFFFu ||
      parts > (im.k + kRChunk - 1) / kRChunk || (parts > 1 && part == nullptr) || v.units != im.n / 256 ||
      v.tiles != (im.k + 15) / 16 || (m * im.n + 255) / 256 > 0x7fffffffull)
    return hipErrorInvalidValue;
  const uint32_t mm = static_cast<uint32_t>(m);
  float* const out = parts > 1 ? part : y;
  hipError_t e = hipErrorInvalidValue;
  switch (im.qtype) {
    case kQ8_0: e = launch_rm_q<kQ8_0>(v, x, mm, out, plan, st); break;
    case kQ4_0: e = launch_rm_q<kQ4_0>(v, x, mm, out, plan, st); break;
    case kQ4_K: e = launch_rm_q<kQ4_K>(v, x, mm, out, plan, st); break;
    case kQ5_K: e = launch_rm_q<kQ5_K>(v, x, mm, out, plan, st); break;
    case kQ6_K: e = launch_rm_q<kQ6_K>(v, x, mm, out, plan, st); break;
    default: break;
  }
  if (e != hipSuccess || parts == 1) return e;
  return launch_rm_sum(im, v, part, parts, m * im.n, y, x, st);
}

}  // namespace qi
