// Group-wise W4 products of more than 16 rows, fp16 and bf16 activations: the
// formats, the exact centred nibbles and the affine form are w4g.hip's.
//
// A 256-lane workgroup computes 16 MT rows x 256 columns over a K range; wave
// w owns all rows x columns 64 w .. +63 (four groups of 16).  K advances 128
// inputs a block (one scale per column):
//  * x: global -> registers a block ahead -> LDS, two stages, as fp16 in the
//    nibbles' order [0,4,1,5,2,6,3,7].  bf16 values become fp16 there (exact
//    between 2^-14 and 65504).  The 16-byte chunk 4 kg + s of a row lies in
//    half s / 2 at position (2 kg + s % 2) ^ key(row) of a 128-byte row, the
//    order whose 16-byte reads are free of bank conflicts on gfx950;
//  * weights: a lane reads 16 bytes (32 inputs) of its column per group, the
//    four operands of its MFMA steps, dequantised once for all rows;
//  * the block's four MFMAs accumulate from zero and the column's scale is
//    applied in fp32.  W is the A operand, so a lane holds one row and, across
//    a pair of groups, 8 consecutive columns (columns permuted as
//    32 p + 8 (n / 4) + 4 (g % 2) + n % 4): its four scales are one 16-byte
//    LDS read and the outputs 16-byte stores;
//  * affine: the block's row sums of x from one more MFMA against ones.
// Where the tiles do not fill the chip K is split over workgroups and a second
// launch adds the fp32 partials.
//
// Two workgroups a CU, so one's MFMAs cover the other's dequantisation and
// barriers; bound by instruction issue (per wave and block 64 MFMAs, 144
// dequantising and 64 scaling VALU).  Measured against w4g_kernel's 64-row
// launches (kernel time): 384 rows 4096 -> 16384, 409 -> 76 us (677 TFLOP/s),
// affine 431 -> 100; 1000 rows 4096 -> 4096 bf16, 581 -> 61; 16384 -> 4096
// affine, 1000 rows 1890 -> 219, 200 rows (symmetric) 373 -> 53, 40 rows 104
// -> 29.
#include "w4_common.h"

namespace rwkv7mi {

namespace {

struct W4mArgs {
  const void* x;
  const uint8_t* w;
  const void *scales, *gbias, *bias, *residual;
  void* y;
  float* part;  // S > 1: [split][row][ldp]
  int rows, O, I, G, gsh;  // G scales per column, gsh = log2(group / 128)
  int nt;                  // column tiles
  int S, bps;              // K splits, blocks of 128 inputs of each
  int ldp, epilogue, vec;  // vec: O % 8 == 0, y and residual 16-byte aligned
};

__device__ __forceinline__ int w4m_key(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// 8 consecutive 16-bit inputs -> fp16 in the order [0,4,1,5,2,6,3,7]
template <typename TA>
__device__ __forceinline__ u32x4 w4m_perm(u32x4 v) {
  if constexpr (std::is_same<TA, __hip_bfloat16>::value) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t d = v[q];
      const _Float16 lo = (_Float16)__uint_as_float(d << 16), hi = (_Float16)__uint_as_float(d & 0xffff0000u);
      v[q] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
    }
  }
  const uint32_t d0 = v[0], d1 = v[1], d2 = v[2], d3 = v[3];
  return (u32x4){__builtin_amdgcn_perm(d2, d0, 0x05040100u), __builtin_amdgcn_perm(d2, d0, 0x07060302u),
                 __builtin_amdgcn_perm(d3, d1, 0x05040100u), __builtin_amdgcn_perm(d3, d1, 0x07060302u)};
}

template <typename TA, typename TS>
__device__ __forceinline__ void w4m_store8(const W4mArgs& A, int row, int c0, float (&v)[8]) {
  const int64_t oi = (int64_t)row * A.O + c0;
  const TS* bp = static_cast<const TS*>(A.bias);
  TA* y = static_cast<TA*>(A.y) + oi;
  const bool whole = A.vec && c0 + 8 <= A.O;
  float r[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = 0.f;
  if (A.epilogue == RWKV7MI_EPI_RESIDUAL) {
    const TA* rp = static_cast<const TA*>(A.residual) + oi;
    if (whole) {
      ld8(rp, r);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) r[e] = c0 + e < A.O ? to_f32(rp[e]) : 0.f;
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (bp && c0 + e < A.O) v[e] += to_f32(bp[c0 + e]);
    if (A.epilogue == RWKV7MI_EPI_RELU2) {
      v[e] = fmaxf(v[e], 0.f);
      v[e] *= v[e];
    }
    v[e] += r[e];
  }
  if (whole) {
    st8(y, v);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (c0 + e < A.O) y[e] = from_f32<TA>(v[e]);
  }
}

}  // namespace

template <int MT, bool AFF, typename TA, typename TS>
__global__ __launch_bounds__(256, 2) void w4m_kernel(const W4mArgs A) {
  __shared__ __align__(16) _Float16 xs[2][2][16 * MT][64];  // [stage][half][row][64 inputs]
  __shared__ __align__(16) float ss[2][256], zs[AFF ? 2 : 1][AFF ? 256 : 4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, kg = lane >> 4;
  const int tn = blockIdx.x % A.nt, tm = blockIdx.x / A.nt;
  const int o0 = 256 * tn, row0 = 16 * MT * tm;
  const int nrow = min(16 * MT, A.rows - row0), ncol = min(256, A.O - o0);
  const int I = A.I;
  const int b0 = blockIdx.z * A.bps, b1 = min(I / 128, b0 + A.bps);

  // descriptors end at the tile's last row / column: past them zeros
  const __amdgpu_buffer_rsrc_t xr =
      make_rsrc(static_cast<const char*>(A.x) + (int64_t)row0 * I * 2, (uint32_t)(nrow * I * 2));
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(A.w + (int64_t)o0 * (I / 2), (uint32_t)(ncol * (I / 2)));
  const __amdgpu_buffer_rsrc_t sr =
      make_rsrc(static_cast<const TS*>(A.scales) + (int64_t)o0 * A.G, (uint32_t)(ncol * A.G * sizeof(TS)));
  const __amdgpu_buffer_rsrc_t br = make_rsrc(
      AFF ? static_cast<const TS*>(A.gbias) + (int64_t)o0 * A.G : nullptr, AFF ? (uint32_t)(ncol * A.G * sizeof(TS)) : 0u);

  u32x4 xg[MT], wg[4];  // the next block's x chunks and weights
  float sg, zg = 0.f;
  auto load = [&](int b) {
    const bool ok = b < b1;
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      const int row = 16 * u + (tid >> 4), c = tid & 15;
      xg[u] = buf_ld16(xr, ok ? (uint32_t)((row * I + 128 * b + 8 * c) * 2) : BUF_OOB);
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int col = 64 * wave + 32 * (g >> 1) + 8 * (n >> 2) + 4 * (g & 1) + (n & 3);
      wg[g] = buf_ld16(wr, ok ? (uint32_t)(col * (I / 2) + 64 * b + 16 * kg) : BUF_OOB);
    }
    sg = buf_ld1<TS>(sr, (uint32_t)(tid * A.G + (b >> A.gsh)), ok);
    if constexpr (AFF) zg = buf_ld1<TS>(br, (uint32_t)(tid * A.G + (b >> A.gsh)), ok);
  };
  auto stage = [&](int st) {
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      const int row = 16 * u + (tid >> 4), c = tid & 15;
      const int pos = (2 * (c >> 2) + (c & 1)) ^ w4m_key(row);
      *reinterpret_cast<u32x4*>(&xs[st][(c >> 1) & 1][row][8 * pos]) = w4m_perm<TA>(xg[u]);
    }
    ss[st][tid] = sg;
    if constexpr (AFF) zs[st][tid] = 8.f * sg + zg;
  };

  f32x4 acc[MT][4];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int g = 0; g < 4; ++g) acc[m][g] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (_Float16)1.0f;
  const int key = w4m_key(n);

  load(b0);
  f16x8 wb[4][4];
  auto dequant = [&]() {
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const uint32_t d = wg[g][s];
        wb[g][s] = w4_nibbles_to_f16(d);
      }
  };
  stage(0);
  dequant();
  __syncthreads();
  for (int b = b0; b < b1; ++b) {
    const int st = (b - b0) & 1;
    load(b + 1);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 sc[4], zc[AFF ? 4 : 1];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int c = 64 * wave + 32 * (g >> 1) + 8 * kg + 4 * (g & 1);
      sc[g] = *reinterpret_cast<const f32x4*>(&ss[st][c]);
      if constexpr (AFF) zc[g] = *reinterpret_cast<const f32x4*>(&zs[st][c]);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      f16x8 xa[4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
        xa[s] = *reinterpret_cast<const f16x8*>(&xs[st][s >> 1][16 * m + n][8 * ((2 * kg + (s & 1)) ^ key)]);
      f32x4 t[4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int g = 0; g < 4; ++g) t[g] = mfma16x16x32(wb[g][s], xa[s], s ? t[g] : zero);
#pragma unroll
      for (int g = 0; g < 4; ++g) acc[m][g] += sc[g] * t[g];
      if constexpr (AFF) {
        f32x4 r = zero;
#pragma unroll
        for (int s = 0; s < 4; ++s) r = mfma16x16x32(ones, xa[s], r);
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[m][g] += zc[g] * r;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    stage(st ^ 1);  // (last read during block b - 1, before the previous barrier)
    dequant();
    __syncthreads();
  }

  // lane: row 16 m + n and, in groups 2 p and 2 p + 1, 8 columns from c0
  float* part = A.S > 1 ? A.part + (int64_t)blockIdx.z * A.rows * A.ldp : nullptr;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int c0 = o0 + 64 * wave + 32 * p + 8 * kg;
    if (c0 >= A.O) continue;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int row = row0 + 16 * m + n;
      if (row >= A.rows) continue;
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = acc[m][2 * p][e];
        v[4 + e] = acc[m][2 * p + 1][e];
      }
      if (part)
        st8(part + (int64_t)row * A.ldp + c0, v);
      else
        w4m_store8<TA, TS>(A, row, c0, v);
    }
  }
}

// One thread: 8 columns of a row, the S partials in split order
template <typename TA, typename TS>
__global__ __launch_bounds__(256) void w4m_reduce_kernel(const W4mArgs A) {
  const int cols = A.ldp / 8;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (int64_t)A.rows * cols) return;
  const int row = (int)(t / cols), c0 = 8 * (int)(t % cols);
  if (c0 >= A.O) return;
  const float* p = A.part + (int64_t)row * A.ldp + c0;
  float v[8];
  ld8(p, v);
  for (int z = 1; z < A.S; ++z) {
    float a[8];
    ld8(p + (int64_t)z * A.rows * A.ldp, a);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += a[e];
  }
  w4m_store8<TA, TS>(A, row, c0, v);
}

// row tiles of a workgroup: 32 or 64 rows
static int w4m_mt(int64_t rows) { return rows <= 32 ? 2 : 4; }

// K splits: a tile alone runs a serial chain of its blocks, with up to 256
// workgroups 1.4 us each (64 rows; 1.2 for 32), with two on a CU 1.9 to 2.2 (1.4), the
// affine form with its row sums and converted bf16 inputs more (measured unsplit,
// 64 rows: fp16 768 -> 768 13.8 us, 1024 -> 1024 16.5, affine 19.0, bf16 17.6, both
// 24.4; 96 rows 2048 -> 8192, 64 workgroups, 28.1; 4096 -> 16384 at 200 rows, 256,
// 55.8, at 300, 320, 68.0).  A split adds the reduce, 0.4 us a partial, and the
// partials' traffic, and an eager call then takes the host 15 us for the scratch
// and the second launch.  Priced at 0.9 a block, 1024 -> 1024 ran unsplit at 64
// rows and more (now 10.5-12 us) and 2048 -> 8192 at 96 (now 20.1).
static int w4m_splits(int64_t rows, int64_t O, int64_t I, int act_dtype, bool aff) {
  const int mt = w4m_mt(rows);
  const int64_t tiles = (rows + 16 * mt - 1) / (16 * mt) * ((O + 255) / 256);
  const int64_t nblk = I / 128;
  const double pb = 4.0 * rows * ((O + 7) / 8 * 8);
  const bool bf = act_dtype == RWKV7MI_BF16;
  const double block = mt == 2 ? 1.2 : 1.4 * (aff && bf ? 1.75 : aff ? 1.15 : bf ? 1.06 : 1.0);
  int best = 1;
  double cost = 1e30;
  for (int S = 1; S <= 32 && (S == 1 || tiles * S <= 512); ++S) {
    const int64_t bps = (nblk + S - 1) / S, wgs = tiles * S;
    if (S > 1 && (bps < 2 || (nblk + bps - 1) / bps != S)) continue;
    const double two = (mt == 2 ? 0.25 : 1.0) * (0.5 + 0.3 * (std::min<int64_t>(wgs, 512) - 256) / 256.0);
    const double per = block + (wgs > 256 ? two : 0.0);
    const double k = (bps + 4) * per * ((wgs + 511) / 512);
    const double t = S > 1 ? std::max(15.0, k + 3.0 + 0.4 * S + pb * S / 4e6) : k;
    if (t < cost) cost = t, best = S;
  }
  return best;
}

bool w4m_supported(int64_t rows, int64_t O, int64_t I, int64_t group, int act_dtype) {
  if (act_dtype != RWKV7MI_F16 && act_dtype != RWKV7MI_BF16) return false;
  // 32-bit offsets: 64 rows of x, 256 columns of weights and (fp32) scales
  if ((int64_t)64 * I * 2 >= (int64_t)BUF_OOB || 256 * (I / 2) >= (int64_t)BUF_OOB) return false;
  const int64_t tiles = (rows + 31) / 32 * ((O + 255) / 256);
  return rows > 0 && rows <= INT32_MAX / 2 && O <= INT32_MAX / 2 && tiles <= INT32_MAX / 2;
}

int64_t w4m_workspace_bytes(int64_t rows, int64_t O, int64_t I, int act_dtype, bool aff) {
  const int S = w4m_splits(rows, O, I, act_dtype, aff);
  return S > 1 ? S * rows * ((O + 7) / 8 * 8) * 4 : 0;
}

template <bool AFF, typename TA, typename TS>
static int w4m_go(const W4mArgs& a, int mt, hipStream_t s) {
  const dim3 grid((unsigned)((a.rows + 16 * mt - 1) / (16 * mt) * a.nt), 1, (unsigned)a.S);
  if (mt == 2)
    hipLaunchKernelGGL((w4m_kernel<2, AFF, TA, TS>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((w4m_kernel<4, AFF, TA, TS>), grid, dim3(256), 0, s, a);
  if (int rc = check_launch("w4m_kernel")) return rc;
  if (a.S == 1) return RWKV7MI_OK;
  const int64_t nthr = (int64_t)a.rows * (a.ldp / 8);
  hipLaunchKernelGGL((w4m_reduce_kernel<TA, TS>), dim3((unsigned)((nthr + 255) / 256)), dim3(256), 0, s, a);
  return check_launch("w4m_reduce_kernel");
}

int w4m_run(const void* x, const uint8_t* packed, const void* scales, const void* gbias, const void* bias,
            const void* residual, void* y, int64_t rows, int64_t O, int64_t I, int64_t group, int epilogue,
            int act_dtype, int scale_dtype, void* ws, int64_t ws_bytes, void* stream) {
  W4mArgs a{x, packed, scales, gbias, bias, residual, y, static_cast<float*>(ws)};
  a.rows = (int)rows;
  a.O = (int)O;
  a.I = (int)I;
  a.G = (int)(I / group);
  a.gsh = group == 256 ? 1 : 0;
  a.nt = (int)((O + 255) / 256);
  a.ldp = (int)((O + 7) / 8 * 8);
  const bool aff = gbias != nullptr;
  a.S = w4m_splits(rows, O, I, act_dtype, aff);
  if (!ws || (reinterpret_cast<uintptr_t>(ws) & 15) || ws_bytes < w4m_workspace_bytes(rows, O, I, act_dtype, aff)) a.S = 1;
  a.bps = (int)((I / 128 + a.S - 1) / a.S);
  a.epilogue = epilogue;
  a.vec = O % 8 == 0 && !(reinterpret_cast<uintptr_t>(y) & 15) &&
          !(epilogue == RWKV7MI_EPI_RESIDUAL && (reinterpret_cast<uintptr_t>(residual) & 15));
  const int mt = w4m_mt(rows);
  const auto go = [&](auto ta, auto ts) {
    using TA = decltype(ta);
    using TS = decltype(ts);
    return aff ? w4m_go<true, TA, TS>(a, mt, as_stream(stream)) : w4m_go<false, TA, TS>(a, mt, as_stream(stream));
  };
  return dispatch_dtype(scale_dtype, [&](auto ts) {
    return act_dtype == RWKV7MI_BF16 ? go(__hip_bfloat16{}, ts) : go(__half{}, ts);
  });
}

}  // namespace rwkv7mi
