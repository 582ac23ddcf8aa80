// Dense products y = act(x W^T + b) (+ residual) of 5 rows and more, fp16 and
// bf16, W in nn.Linear layout [N, K]: small and middle sizes, where 256 x 256
// tiles would leave most CUs idle and copying W into operand order would cost
// as much as the product.
//
// A 256-lane workgroup computes 16 MT rows x 16 NT columns of one problem; its
// four waves take the 64-input steps of its K range in turn and each holds the
// whole tile.  Both operands go straight from global memory to MFMA registers:
// lane n + 16 kg reads inputs 16 kg .. +15 of a step of row / column n (two
// 16-byte loads, whole 128-byte lines over the four kg), the next steps' loads
// in flight in a ring.  Bound by what a CU pulls through its L1, so MT and NT
// are chosen for the least (MT + NT) x rounds of workgroups.  The waves' sums
// meet in LDS 16 rows at a time, added in wave order.
//
// Measured (fp16, kernel time): 512 rows, three 768 -> 768 in one launch 21 us
// (3 x 21 for 6 tiles of 256 x 256 and 3 x 5 for the copies of W before), 768 ->
// 3072 22 us (28 + 10), 3072 -> 768 in K splits 24 (91 + 10); 8 rows 768 -> 768
// three at once 4.7 us (3 x 7), 8 rows 3072 -> 768 8 us (12).
#include <algorithm>

#include "dense_common.h"

namespace rwkv7mi {

namespace {

template <typename TA> struct DtVec { typedef f16x8 V; };
template <> struct DtVec<__hip_bfloat16> { typedef bf16x8 V; };

struct DtArgs {
  DenseBatch b;
  int rows, S;
  float* part;
  int64_t ldp;
};

}  // namespace

template <int MT, int NT, typename TA>
__global__ __launch_bounds__(256) void dense_tile_kernel(const DtArgs G) {
  using V = typename DtVec<TA>::V;
  constexpr int RS = 16 * NT + 4;
  __shared__ __align__(16) float red[4][16][RS];
  int pi = 0;
#pragma unroll
  for (int q = 1; q < 4; ++q)
    if (q < G.b.nprob && (int)blockIdx.x >= G.b.p[q].tile0) pi = q;
  const DenseProb& P = G.b.p[pi];
  const int N = P.N, K = P.K;
  const int nt = (N + 16 * NT - 1) / (16 * NT);
  const int t = (int)blockIdx.x - P.tile0;
  const int n0 = 16 * NT * (t % nt), row0 = 16 * MT * (t / nt);
  const int nrow = min(16 * MT, G.rows - row0), ncol = min(16 * NT, N - n0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, kg = lane >> 4;
  const int steps = (K + 63) / 64, sps = (steps + G.S - 1) / G.S;
  const int s0 = (int)blockIdx.z * sps, s1 = min(steps, s0 + sps);

  // descriptors end at the tile's last row / column: past them zeros
  const __amdgpu_buffer_rsrc_t xr =
      make_rsrc(static_cast<const char*>(P.x) + (int64_t)row0 * K * 2, (uint32_t)(nrow * K * 2));
  const __amdgpu_buffer_rsrc_t wr =
      make_rsrc(static_cast<const char*>(P.W) + (int64_t)n0 * K * 2, (uint32_t)(ncol * K * 2));

  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[m][c] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto load = [&](int s, V (&xa)[MT][2], V (&wa)[NT][2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int kk = 64 * s + 16 * kg + 8 * h;
      const bool ok = s < s1 && kk < K;  // K % 8 == 0
#pragma unroll
      for (int c = 0; c < NT; ++c)
        wa[c][h] = __builtin_bit_cast(V, buf_ld16(wr, ok ? (uint32_t)(((16 * c + n) * K + kk) * 2) : BUF_OOB));
#pragma unroll
      for (int m = 0; m < MT; ++m)
        xa[m][h] = __builtin_bit_cast(V, buf_ld16(xr, ok ? (uint32_t)(((16 * m + n) * K + kk) * 2) : BUF_OOB));
    }
  };
  constexpr int R = MT + NT <= 3 ? 4 : MT + NT <= 6 ? 3 : 2;
  V xa[R][MT][2], wa[R][NT][2];
#pragma unroll
  for (int j = 0; j < R; ++j) load(s0 + wave + 4 * j, xa[j], wa[j]);
  __builtin_amdgcn_sched_barrier(0);
  for (int s = s0; s < s1; s += 4 * R) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      // W as the A operand: a lane holds row n and columns 16 c + 4 kg .. +3
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int c = 0; c < NT; ++c) acc[m][c] = mfma16x16x32(wa[j][c][h], xa[j][m][h], acc[m][c]);
      __builtin_amdgcn_sched_barrier(0);
      load(s + wave + 4 * (j + R), xa[j], wa[j]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  const TA* bias = static_cast<const TA*>(P.bias);
  const TA* res = static_cast<const TA*>(P.residual);
  TA* y = static_cast<TA*>(P.y);
  const int er = tid >> 4, ec = NT * (tid & 15);  // 16 rows x 16 runs of NT columns
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m) __syncthreads();
#pragma unroll
    for (int c = 0; c < NT; ++c) *reinterpret_cast<f32x4*>(&red[wave][n][16 * c + 4 * kg]) = acc[m][c];
    __syncthreads();
    if (16 * m + er >= nrow) continue;  // (every lane reaches the barriers above)
    const int64_t row = row0 + 16 * m + er;
    float v[NT];
#pragma unroll
    for (int e = 0; e < NT; ++e)
      v[e] = ((red[0][er][ec + e] + red[1][er][ec + e]) + red[2][er][ec + e]) + red[3][er][ec + e];
#pragma unroll
    for (int e = 0; e < NT; ++e) {
      const int o = n0 + ec + e;
      if (o >= N) continue;
      if (G.part) {
        G.part[((int64_t)(pi * G.S + (int)blockIdx.z) * G.rows + row) * G.ldp + o] = v[e];
      } else {
        const float r = res ? to_f32(res[row * N + o]) : 0.f;
        y[row * N + o] = from_f32<TA>(apply_act(v[e] + (bias ? to_f32(bias[o]) : 0.f), P.act) + r);
      }
    }
  }
}

// workgroups of a launch with 16 mt x 16 nt tiles
static int64_t dt_wgs(const DenseBatch& b, int64_t rows, int mt, int nt) {
  int64_t w = 0;
  for (int i = 0; i < b.nprob; ++i) w += (rows + 16 * mt - 1) / (16 * mt) * ((b.p[i].N + 16 * nt - 1) / (16 * nt));
  return w;
}

// The tile with the least time, and that time: rounds of 256 workgroups x the
// bytes each pulls (its rows and columns over its K range) at 45 GB/s, plus a
// launch.
static double dt_pick(const DenseBatch& b, int64_t rows, int S, int* mt_out, int* nt_out) {
  int64_t kmax = 0;
  for (int i = 0; i < b.nprob; ++i) kmax = std::max<int64_t>(kmax, b.p[i].K);
  double best = 1e30;
  for (int mt = 1; mt <= 4; mt *= 2) {
    if (mt > 1 && rows <= 8 * mt) break;
    for (int nt = 1; nt <= 4; nt *= 2) {
      const int64_t rounds = (dt_wgs(b, rows, mt, nt) * S + 255) / 256;
      const double us = 6.0 + rounds * (1.0 + (double)(mt + nt) * 16 * 2 * kmax / S / 45e3);
      if (us < best) best = us, *mt_out = mt, *nt_out = nt;
    }
  }
  return best;
}

bool dense_tile_supported(const DenseBatch& b, int64_t rows, int act_dtype) {
  if (act_dtype != RWKV7MI_F16 && act_dtype != RWKV7MI_BF16) return false;
  if (rows <= 0 || rows > INT32_MAX / 2) return false;
  for (int i = 0; i < b.nprob; ++i)
    if ((int64_t)64 * b.p[i].K * 2 >= (int64_t)BUF_OOB) return false;  // 32-bit offsets inside a tile
  return dt_wgs(b, rows, 1, 1) <= INT32_MAX / 2;
}

double dense_tile_us(const DenseBatch& b, int64_t rows, int S) {
  int mt, nt;
  return dt_pick(b, rows, S, &mt, &nt);
}

int dense_tile_run(const DenseBatch& b0, int64_t rows, int act_dtype, int S, float* part, int64_t ldp, void* stream) {
  DtArgs g{b0, (int)rows, S, part, ldp};
  int mt = 1, nt = 1, tiles = 0;
  dt_pick(b0, rows, S, &mt, &nt);
  for (int i = 0; i < b0.nprob; ++i) {
    g.b.p[i].tile0 = tiles;
    tiles += (int)((rows + 16 * mt - 1) / (16 * mt) * ((b0.p[i].N + 16 * nt - 1) / (16 * nt)));
  }
  const dim3 grid((unsigned)tiles, 1, (unsigned)S);
  auto go = [&](auto ta) {
    using TA = decltype(ta);
    hipStream_t s = as_stream(stream);
#define DT_GO(M_, N_) \
  if (mt == M_ && nt == N_) hipLaunchKernelGGL((dense_tile_kernel<M_, N_, TA>), grid, dim3(256), 0, s, g)
    DT_GO(1, 1); DT_GO(1, 2); DT_GO(1, 4);
    DT_GO(2, 1); DT_GO(2, 2); DT_GO(2, 4);
    DT_GO(4, 1); DT_GO(4, 2); DT_GO(4, 4);
#undef DT_GO
    return check_launch("dense_tile_kernel");
  };
  return act_dtype == RWKV7MI_BF16 ? go(__hip_bfloat16{}) : go(__half{});
}

}  // namespace rwkv7mi
