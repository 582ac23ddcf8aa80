// W/A/G/V LoRA projections of more than LORA_PAIR_MIN rows, fp16 and bf16
// (rwkv7_hf/fused_lora.py:559 fused_wag_lora, :706 fused_wavg_lora), as two
// launches over all rows and problems:
//
//   lora_mid_kernel  mid_p = round(act_down_p(x_p Wd_p^T))    [rows, r_p]
//   lora_out_kernel  y_p   = act_up_p(mid_p Wu_p^T + b_p)     [rows, A]
//
// mid (the reference's own tensor, in the activation dtype) goes through the
// workspace: rows x 288 values against rows x 4 x 4096 of x and y.
//
// Measured (D = A = 4096, ranks 64/64/128/32, both launches, before -> after):
//   fp16  700 rows  233 -> 35 us (the one-launch kernel put 12 workgroups on
//         the chip), 2000 rows 235 -> 63, 4000 rows 238 -> 115; 250 rows at
//         2048: 68 -> 16 (four 64-row split-K pairs)
//   bf16  700 rows  475 -> 35 us, 16000 rows 1250 -> 371 (bf16 MFMAs on the
//         values themselves instead of three fp16 ones on a split)
// Against lora_seq_kernel: lora_seq_faster in lora.hip.
// Against the split-K pair of lora.hip, us: 33 rows at 4096 18.7 -> 15.4, 64 rows
// 22.2 -> 15.9, at 768 12.6 -> 9.3 and 16.4 -> 9.5; 16 rows at 4096 take 13.5 there,
// and up to 32 rows keep it.
#include <algorithm>

#include "lora_common.h"

namespace rwkv7mi {

namespace {

template <typename TA> struct LpVec { typedef f16x8 V; typedef _Float16 E; };
template <> struct LpVec<__hip_bfloat16> { typedef bf16x8 V; typedef __bf16 E; };

constexpr int LP_NW = 4;       // mid: waves per workgroup, each a share of K
constexpr int LP_RT = 4;       // mid: rank tiles of 16 per workgroup (64 rank columns)
constexpr int LP_RS = 68;      // mid: LDS row (floats): 64 rank columns, 16-byte aligned, bank-skewed
constexpr int LP_MAXUNITS = 8; // 4 problems x ceil(128 / 64)

struct LpProb {
  const void *x, *wd, *wu, *bu;
  void *y, *mid;
  int r, act_d, act_u;
  int vec;  // A % 8 == 0 and y 16-byte aligned: 16-byte output rows
};
struct LpBatch {
  LpProb p[4];
  uint8_t unit_p[LP_MAXUNITS], unit_t[LP_MAXUNITS];  // problem and first 64-column rank block of each unit
  int rows, D, A;
  int ncb;  // out: column blocks of 256
  int rb;   // out: rows per workgroup (a multiple of 16)
};

}  // namespace

// A workgroup takes 16 MT rows x 64 rank columns of one problem over all of K;
// the 128-column G problem is two units, and the rows are cut finely enough (MT)
// to give every CU a workgroup.  Bound by what one CU pulls: in the MFMA operand
// order neighbouring lanes read different rows, 16 bytes of a line at a time,
// and a CU's L1 then gave about 33 GB/s (the two launches at 4096: 65 rows 28 us
// against 16 now, 250 rows 33 and 21, 700 rows 44 and 35, 8000 215 and 184; 65
// rows at 768 14 and 10).  So each of the four waves brings its own
// 64-input steps (w, w + 4, ..) in by LDS DMA, 128 contiguous bytes per eight
// lanes, into a ring of R stages of its own: no barrier in the loop, only the
// wave's own counters.  The 16-byte chunk c of a row lies at position c ^ (r % 8)
// ^ (r / 8 % 2), which leaves the operand reads free of bank conflicts on gfx950.
// The waves' sums meet in LDS, one 16-row tile at a time, added in wave order.
template <int MT>
struct LpMid {
  static constexpr int R = MT == 4 ? 2 : 3;       // stages of a wave
  static constexpr int NL = 2 * MT + 2 * LP_RT;   // DMA instructions (KB) of a step: 8 rows each
  static constexpr int LDS = LP_NW * R * NL * 1024;
  // vmcnt: the steps after the oldest one may be in flight
  static constexpr int LEFT = (R - 1) * NL;
  static constexpr int WAIT = (LEFT & 15) | 0x0F70 | ((LEFT >> 4) << 14);
  static_assert(LDS <= 160 * 1024 && LDS >= LP_NW * 16 * LP_RS * 4 && LEFT < 64, "ring of a workgroup");
};

template <typename TA, int MT>
__global__ __launch_bounds__(64 * LP_NW, 1) void lora_mid_kernel(const LpBatch B) {
  using V = typename LpVec<TA>::V;
  typedef __attribute__((address_space(3))) void* lds_ptr;
  using M = LpMid<MT>;
  extern __shared__ __align__(16) char smem[];
  const LpProb& P = B.p[B.unit_p[blockIdx.y]];
  const int D = B.D, r = P.r;
  const int c0 = 64 * B.unit_t[blockIdx.y];
  const int row0 = blockIdx.x * 16 * MT;
  const int nrow = min(16 * MT, B.rows - row0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, kg = lane >> 4;
  // descriptors end at the tile's last row / the problem's last rank: rows and
  // ranks past them read zeros
  const __amdgpu_buffer_rsrc_t xr =
      make_rsrc(static_cast<const char*>(P.x) + (int64_t)row0 * D * 2, (uint32_t)(nrow * D * 2));
  const __amdgpu_buffer_rsrc_t wr =
      make_rsrc(static_cast<const char*>(P.wd) + (int64_t)c0 * D * 2, (uint32_t)(min(64, r - c0) * D * 2));

  f32x4 acc[MT][LP_RT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < LP_RT; ++t) acc[m][t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  char* ring = smem + wave * M::R * M::NL * 1024;
  // instruction u: rows 8 u + lane / 8, the chunk of position lane % 8
  const int ch = (lane & 7) ^ (lane >> 3);
  auto issue = [&](int s, int st) {
    char* d = ring + st * M::NL * 1024;
#pragma unroll
    for (int u = 0; u < M::NL; ++u) {
      const int uu = u < 2 * MT ? u : u - 2 * MT;
      const int kk = 64 * s + 8 * (ch ^ (uu & 1));
      const int off = kk < D ? ((8 * uu + (lane >> 3)) * D + kk) * 2 : (int)BUF_OOB;  // D % 8 == 0
      __builtin_amdgcn_raw_ptr_buffer_load_lds(u < 2 * MT ? xr : wr, (lds_ptr)(d + 1024 * u), 16, off, 0, 0, 0);
    }
  };
  const int key = (n & 7) ^ (n >> 3);
  auto read = [&](int st, int tile, int h) {  // 16-row tile, inputs 16 kg + 8 h of the step
    return *reinterpret_cast<const V*>(ring + st * M::NL * 1024 + (16 * tile + n) * 128 + 16 * ((2 * kg + h) ^ key));
  };
  const int nst = ((D + 63) / 64 + LP_NW - 1) / LP_NW;  // steps per wave (past the end: zeros)
#pragma unroll
  for (int j = 0; j < M::R; ++j) issue(wave + LP_NW * j, j);
  for (int i = 0; i < nst; i += M::R) {
#pragma unroll
    for (int j = 0; j < M::R; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(M::WAIT);  // the oldest step has landed
      __builtin_amdgcn_sched_barrier(0);
      V xa[MT][2], wb[LP_RT][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int m = 0; m < MT; ++m) xa[m][h] = read(j, m, h);
#pragma unroll
        for (int t = 0; t < LP_RT; ++t) wb[t][h] = read(j, MT + t, h);
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage is read and may be overwritten
      __builtin_amdgcn_sched_barrier(0);
      issue(wave + LP_NW * (i + j + M::R), j);
      __builtin_amdgcn_sched_barrier(0);
      // Wd as the A operand, x as B: a lane holds one row and four consecutive ranks
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int t = 0; t < LP_RT; ++t) acc[m][t] = mfma16x16x32(wb[t][h], xa[m][h], acc[m][t]);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the trailing loads have landed, the ring is free
  __syncthreads();

  float(*red)[16][LP_RS] = reinterpret_cast<float(*)[16][LP_RS]>(smem);
  TA* mid = static_cast<TA*>(P.mid);
  const int er = tid >> 4, ec = 4 * (tid & 15);  // 16 rows x 16 runs of four rank columns
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m) __syncthreads();
#pragma unroll
    for (int t = 0; t < LP_RT; ++t) *reinterpret_cast<f32x4*>(&red[wave][n][16 * t + 4 * kg]) = acc[m][t];
    __syncthreads();
    f32x4 v = *reinterpret_cast<const f32x4*>(&red[0][er][ec]);
#pragma unroll
    for (int w = 1; w < LP_NW; ++w) v += *reinterpret_cast<const f32x4*>(&red[w][er][ec]);
    if (16 * m + er < nrow && c0 + ec < r) {  // r % 8 == 0
      uint16_t o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = __builtin_bit_cast(uint16_t, from_f32<TA>(lora_act_fast(v[e], P.act_d)));
      *reinterpret_cast<uint2*>(mid + (int64_t)(row0 + 16 * m + er) * r + c0 + ec) =
          make_uint2((uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16));
    }
  }
}

// One workgroup: B.rb rows x 256 output columns of one problem; each of its
// four waves keeps the up weights of its own 64 columns in registers (4 tiles
// x KU rank steps) and walks the rows 16 at a time, the next tile's mid rows
// loaded before this tile's MFMAs.  Bound by the output stream: Wu's tiles are
// taken in the column order 32 p + 8 (n / 4) + 4 (j % 2) + n % 4, which leaves
// a lane with 8 consecutive outputs of one row per pair of tiles (16-byte
// stores, 64 contiguous bytes per row).
template <typename TA, int KU>
__device__ __forceinline__ void lora_out_body(const LpBatch& B, const LpProb& P) {
  using V = typename LpVec<TA>::V;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int n = lane & 15, kg = lane >> 4;
  const int A = B.A, r = P.r;
  const int c0 = 256 * (int)(blockIdx.x % B.ncb) + 64 * wave;
  const int row0 = (int)(blockIdx.x / B.ncb) * B.rb;
  const int nrow = min(B.rb, B.rows - row0);
  if (c0 >= A) return;  // whole waves; no barrier below
  const __amdgpu_buffer_rsrc_t ur = make_rsrc(P.wu, (uint32_t)((int64_t)A * r * 2));
  const __amdgpu_buffer_rsrc_t mr =
      make_rsrc(static_cast<const char*>(P.mid) + (int64_t)row0 * r * 2, (uint32_t)(nrow * r * 2));
  V u[4][KU];
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int q = 0; q < KU; ++q) {
      const int o = c0 + 32 * (j >> 1) + 8 * (n >> 2) + 4 * (j & 1) + (n & 3), kk = 32 * q + 8 * kg;
      u[j][q] = __builtin_bit_cast(V, buf_ld16(ur, o < A && kk < r ? (uint32_t)((o * r + kk) * 2) : BUF_OOB));
    }
  const TA* bp = static_cast<const TA*>(P.bu);
  float bo[2][8];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int o = c0 + 32 * p + 8 * kg + e;
      bo[p][e] = bp && o < A ? to_f32(bp[o]) : 0.f;
    }
  auto load = [&](int i, V (&md)[KU]) {
#pragma unroll
    for (int q = 0; q < KU; ++q) {
      const int kk = 32 * q + 8 * kg;
      md[q] = __builtin_bit_cast(V, buf_ld16(mr, kk < r ? (uint32_t)(((16 * i + n) * r + kk) * 2) : BUF_OOB));
    }
  };
  TA* y = static_cast<TA*>(P.y);
  const int nt = (nrow + 15) / 16;
  auto tile = [&](int i, const V (&md)[KU]) {
    f32x4 c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      c[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < KU; ++q) c[j] = mfma16x16x32(u[j][q], md[q], c[j]);
    }
    const int row = 16 * i + n;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int o = c0 + 32 * p + 8 * kg;
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = lora_act_fast(c[2 * p][e] + bo[p][e], P.act_u);
        v[4 + e] = lora_act_fast(c[2 * p + 1][e] + bo[p][4 + e], P.act_u);
      }
      if (row < nrow) {
        TA* d = y + (int64_t)(row0 + row) * A + o;
        if (P.vec && o + 8 <= A) {
          st8(d, v);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (o + e < A) d[e] = from_f32<TA>(v[e]);
        }
      }
    }
  };
  V m0[KU], m1[KU];
  load(0, m0);
  for (int i = 0; i < nt; i += 2) {
    load(i + 1, m1);
    __builtin_amdgcn_sched_barrier(0);
    tile(i, m0);
    if (i + 1 >= nt) break;
    load(i + 2, m0);
    __builtin_amdgcn_sched_barrier(0);
    tile(i + 1, m1);
  }
}

template <typename TA>
__global__ __launch_bounds__(256) void lora_out_kernel(const LpBatch B) {
  const LpProb& P = B.p[blockIdx.y];
  switch ((P.r + 31) / 32) {  // uniform over the workgroup
    case 1: lora_out_body<TA, 1>(B, P); break;
    case 2: lora_out_body<TA, 2>(B, P); break;
    case 3: lora_out_body<TA, 3>(B, P); break;
    default: lora_out_body<TA, 4>(B, P); break;
  }
}

bool lora_pair_supported(const LoraBatch& b, int64_t rows, int act_dtype, const void* ws, size_t ws_bytes) {
  if (act_dtype != RWKV7MI_F16 && act_dtype != RWKV7MI_BF16) return false;
  if (rows <= 0 || rows > (int64_t)INT32_MAX / 64) return false;
  int64_t mid = 0;
  for (int i = 0; i < b.nprob; ++i) {
    if (b.p[i].r > 128) return false;
    mid += rows * b.p[i].r * 2;
  }
  // 32-bit offsets inside one descriptor: 64 rows of x or of Wd, all of Wu
  if ((int64_t)64 * b.D * 2 >= (int64_t)BUF_OOB || (int64_t)b.A * 128 * 2 >= (int64_t)BUF_OOB) return false;
  if ((int64_t)((b.A + 255) / 256) * ((rows + 15) / 16) > INT32_MAX / 2) return false;
  return ws && !(reinterpret_cast<uintptr_t>(ws) & 15) && (int64_t)ws_bytes >= mid;
}

template <typename TA>
static int lora_pair_go(LpBatch& b, int nprob, int units, hipStream_t s) {
  const int64_t t16 = ((int64_t)b.rows + 15) / 16;
  auto mid = [&](auto kern, int mt, int lds, std::atomic<uint64_t>& raised) {
    if (int rc = raise_dynamic_lds(reinterpret_cast<const void*>(kern), lds, raised, "lora_mid_kernel")) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)((t16 + mt - 1) / mt), (unsigned)units), dim3(64 * LP_NW), (size_t)lds, s, b);
    return check_launch("lora_mid_kernel");
  };
  static std::atomic<uint64_t> raised[3];  // devices whose dynamic LDS limit is raised for each instance
  // rows per workgroup (16 mt): the least time at a fixed rate per CU, i.e.
  // rounds of 256 workgroups x the 64 rank and 16 mt input rows each one reads
  int mt = 1;
  int64_t best = INT64_MAX;
  for (int c = 1; c <= 4; c *= 2) {
    const int64_t cost = ((t16 + c - 1) / c * units + 255) / 256 * (64 + 16 * c);
    if (cost < best) best = cost, mt = c;
  }
  const int rc = mt == 4   ? mid(&lora_mid_kernel<TA, 4>, 4, LpMid<4>::LDS, raised[2])
                 : mt == 2 ? mid(&lora_mid_kernel<TA, 2>, 2, LpMid<2>::LDS, raised[1])
                           : mid(&lora_mid_kernel<TA, 1>, 1, LpMid<1>::LDS, raised[0]);
  if (rc) return rc;
  b.ncb = (b.A + 255) / 256;
  // rows per workgroup, 16..256: about 512 workgroups (each re-reads its 256
  // columns of Wu: 16 rows a workgroup cost 26 us where 64 take 18, 700 rows)
  const int64_t per = t16 * b.ncb * nprob / 512;
  b.rb = 16 * (int)std::max<int64_t>(1, std::min<int64_t>(16, per));
  const int64_t nrb = ((int64_t)b.rows + b.rb - 1) / b.rb;
  hipLaunchKernelGGL(lora_out_kernel<TA>, dim3((unsigned)(nrb * b.ncb), (unsigned)nprob), dim3(256), 0, s, b);
  return check_launch("lora_out_kernel");
}

int lora_pair_run(const LoraBatch& b0, int64_t rows, int act_dtype, void* ws, void* stream) {
  LpBatch b{};
  b.rows = (int)rows;
  b.D = b0.D;
  b.A = b0.A;
  int units = 0;
  char* mid = static_cast<char*>(ws);
  for (int i = 0; i < b0.nprob; ++i) {
    const LoraProb& q = b0.p[i];
    const int vec = b.A % 8 == 0 && !(reinterpret_cast<uintptr_t>(q.y) & 15);
    b.p[i] = LpProb{q.x, q.wd, q.wu, q.bu, q.y, mid, q.r, q.act_d, q.act_u, vec};
    mid += rows * q.r * 2;  // r % 8 == 0: the next problem's rows stay 16-byte aligned
    for (int t = 0; t < (q.r + 63) / 64; ++t, ++units) {
      b.unit_p[units] = (uint8_t)i;
      b.unit_t[units] = (uint8_t)t;
    }
  }
  if (act_dtype == RWKV7MI_BF16) return lora_pair_go<__hip_bfloat16>(b, b0.nprob, units, as_stream(stream));
  return lora_pair_go<__half>(b, b0.nprob, units, as_stream(stream));
}

}  // namespace rwkv7mi
