// Dense products y = act(x W^T + b) (+ residual) of 5 rows and more, fp16 and
// bf16, W in nn.Linear layout [N, K]: small and middle sizes, where 256 x 256
// tiles would leave most CUs idle and copying W into operand order would cost
// as much as the product.
//
// A 256-lane workgroup computes 16 MT rows x 16 NT columns of one problem; its
// four waves take the 64-input steps of its K range in turn and each holds the
// whole tile.  Bound by what a CU pulls, so MT and NT are chosen for the least
// (MT + NT) x rounds of workgroups.  Read straight into the MFMA operands,
// neighbouring lanes take 16 bytes of different rows and the L1 gives 33-45 GB/s
// a CU; so each wave brings its own steps in by LDS DMA, 128 contiguous bytes per
// eight lanes, into a ring of its own: no barrier in the loop, only the wave's
// own counters.  The 16-byte chunk c of a row lies at position c ^ (r % 8) ^ (r /
// 8 % 2), which leaves the operand reads free of bank conflicts on gfx950.  The
// waves' sums meet in LDS 16 rows at a time, added in wave order.
//
// Measured (fp16, time a call in a graph; operands straight into registers ->
// the ring): 512 rows, three 768 -> 768 in one launch 20.0 -> 17.4 us, 768 ->
// 3072 19.9 -> 17.1, 3072 -> 768 (unsplit) 21.8 -> 11.8; 64 rows, three 2048 ->
// 2048 16.3 -> 10.6; 8 rows 3072 -> 768 7.3 -> 4.9; 1000 rows 8192 -> 2048 (also
// unsplit) 127 -> 68.  (The 256 x 256 form and its copy of W took 38 us for 512 rows 768 -> 3072
// and 101 for 3072 -> 768.)
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

template <int MT, int NT>
struct DtRing {
  static constexpr int NL = 2 * (MT + NT);  // DMA instructions (KB) of a step: 8 rows each
  static constexpr int R = NL <= 4 ? 4 : NL <= 6 ? 3 : NL <= 8 ? 4 : NL <= 12 ? 3 : 2;  // stages of a wave
  static constexpr int LDS = 4 * R * NL * 1024;
  // vmcnt: the steps after the oldest one may be in flight
  static constexpr int LEFT = (R - 1) * NL;
  static constexpr int WAIT = (LEFT & 15) | 0x0F70 | ((LEFT >> 4) << 14);
  static_assert(LDS <= 160 * 1024 && LDS >= 4 * 16 * (16 * NT + 4) * 4 && LEFT < 64, "ring of a workgroup");
};

template <int MT, int NT, typename TA>
__global__ __launch_bounds__(256) void dense_tile_kernel(const DtArgs G) {
  using V = typename DtVec<TA>::V;
  typedef __attribute__((address_space(3))) void* lds_ptr;
  using Q = DtRing<MT, NT>;
  constexpr int RS = 16 * NT + 4, R = Q::R;
  extern __shared__ __align__(16) char smem[];
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
  char* ring = smem + wave * R * Q::NL * 1024;
  // instruction u: rows 8 u + lane / 8 of x, then columns of W; the chunk of position lane % 8
  const int ch = (lane & 7) ^ (lane >> 3);
  auto issue = [&](int s, int st) {
    char* d = ring + st * Q::NL * 1024;
#pragma unroll
    for (int u = 0; u < Q::NL; ++u) {
      const int uu = u < 2 * MT ? u : u - 2 * MT;
      const int kk = 64 * s + 8 * (ch ^ (uu & 1));
      const int off = s < s1 && kk < K ? ((8 * uu + (lane >> 3)) * K + kk) * 2 : (int)BUF_OOB;  // K % 8 == 0
      __builtin_amdgcn_raw_ptr_buffer_load_lds(u < 2 * MT ? xr : wr, (lds_ptr)(d + 1024 * u), 16, off, 0, 0, 0);
    }
  };
  const int key = (n & 7) ^ (n >> 3);
  auto read = [&](int st, int tile, int h) {  // 16-row tile, inputs 16 kg + 8 h of the step
    return *reinterpret_cast<const V*>(ring + st * Q::NL * 1024 + (16 * tile + n) * 128 + 16 * ((2 * kg + h) ^ key));
  };
  // this thread's outputs: row er of every 16-row tile, NT columns; their bias and
  // residual are read ahead of all stores (a load behind a store that may alias it
  // waits for the store: with 16 outputs a thread that chain was half of the kernel)
  const TA* bias = static_cast<const TA*>(P.bias);
  const TA* res = static_cast<const TA*>(P.residual);
  TA* y = static_cast<TA*>(P.y);
  const int er = tid >> 4, ec = NT * (tid & 15), oc = n0 + ec;
  const bool vec = N % NT == 0 && !(reinterpret_cast<uintptr_t>(y) & (2 * NT - 1));
  const __amdgpu_buffer_rsrc_t br = make_rsrc(bias, bias ? (uint32_t)(N * 2) : 0u);
  const __amdgpu_buffer_rsrc_t rr = make_rsrc(res ? res + (int64_t)row0 * N : nullptr, res ? (uint32_t)(nrow * N * 2) : 0u);
  float bv[NT], rv[MT][NT];
#pragma unroll
  for (int e = 0; e < NT; ++e) {
    bv[e] = buf_ld1<TA>(br, (uint32_t)(oc + e), oc + e < N);
#pragma unroll
    for (int m = 0; m < MT; ++m)
      rv[m][e] = buf_ld1<TA>(rr, (uint32_t)((16 * m + er) * N + oc + e), oc + e < N);
  }
#pragma unroll
  for (int j = 0; j < R; ++j) issue(s0 + wave + 4 * j, j);
  for (int s = s0; s < s1; s += 4 * R) {
#pragma unroll
    for (int j = 0; j < R; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(Q::WAIT);  // the oldest step has landed
      __builtin_amdgcn_sched_barrier(0);
      V xa[MT][2], wa[NT][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int m = 0; m < MT; ++m) xa[m][h] = read(j, m, h);
#pragma unroll
        for (int c = 0; c < NT; ++c) wa[c][h] = read(j, MT + c, h);
      }
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage is read and may be overwritten
      __builtin_amdgcn_sched_barrier(0);
      issue(s + wave + 4 * (j + R), j);
      __builtin_amdgcn_sched_barrier(0);
      // W as the A operand: a lane holds row n and columns 16 c + 4 kg .. +3
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int c = 0; c < NT; ++c) acc[m][c] = mfma16x16x32(wa[c][h], xa[m][h], acc[m][c]);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the trailing loads have landed, the ring is free
  __syncthreads();

  float(*red)[16][RS] = reinterpret_cast<float(*)[16][RS]>(smem);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m) __syncthreads();
#pragma unroll
    for (int c = 0; c < NT; ++c) *reinterpret_cast<f32x4*>(&red[wave][n][16 * c + 4 * kg]) = acc[m][c];
    __syncthreads();
    if (16 * m + er >= nrow || oc >= N) continue;  // (every lane reaches the barriers above)
    const int64_t row = row0 + 16 * m + er;
    float v[NT];
#pragma unroll
    for (int e = 0; e < NT; ++e)
      v[e] = ((red[0][er][ec + e] + red[1][er][ec + e]) + red[2][er][ec + e]) + red[3][er][ec + e];
    if (G.part) {
      float* d = G.part + ((int64_t)(pi * G.S + (int)blockIdx.z) * G.rows + row) * G.ldp + oc;
#pragma unroll
      for (int e = 0; e < NT; ++e)
        if (oc + e < N) d[e] = v[e];
      continue;
    }
    TA o[NT];
#pragma unroll
    for (int e = 0; e < NT; ++e) o[e] = from_f32<TA>(apply_act(v[e] + bv[e], P.act) + rv[m][e]);
    TA* d = y + row * N + oc;
    if (NT == 4 && vec) {
      uint32_t q[2] = {0u, 0u};
#pragma unroll
      for (int e = 0; e < NT; ++e) q[e >> 1] |= (uint32_t)__builtin_bit_cast(uint16_t, o[e]) << (16 * (e & 1));
      *reinterpret_cast<uint2*>(d) = make_uint2(q[0], q[1]);
    } else {
#pragma unroll
      for (int e = 0; e < NT; ++e)
        if (oc + e < N) d[e] = o[e];
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
// launch.  (The ring reaches about 65: between tiles only the ratios count, and
// against the 256 x 256 form the estimate errs towards that one.)
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
    if ((int64_t)64 * std::max(b.p[i].K, b.p[i].N) * 2 >= (int64_t)BUF_OOB) return false;  // 32-bit offsets inside a tile
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
    static std::atomic<uint64_t> raised[9];  // devices whose dynamic LDS limit is raised for each instance
    auto launch = [&](auto kern, int lds, std::atomic<uint64_t>& done) {
      if (int rc = raise_dynamic_lds(reinterpret_cast<const void*>(kern), lds, done, "dense_tile_kernel")) return rc;
      hipLaunchKernelGGL(kern, grid, dim3(256), (size_t)lds, s, g);
      return check_launch("dense_tile_kernel");
    };
#define DT_GO(M_, N_) \
  if (mt == M_ && nt == N_) \
    return launch(&dense_tile_kernel<M_, N_, TA>, DtRing<M_, N_>::LDS, raised[3 * (M_ / 2) + N_ / 2])
    DT_GO(1, 1); DT_GO(1, 2); DT_GO(1, 4);
    DT_GO(2, 1); DT_GO(2, 2); DT_GO(2, 4);
    DT_GO(4, 1); DT_GO(4, 2); DT_GO(4, 4);
#undef DT_GO
    return fail(RWKV7MI_EINVAL, "dense_tile: no such tile");
  };
  return act_dtype == RWKV7MI_BF16 ? go(__hip_bfloat16{}) : go(__half{});
}

}  // namespace rwkv7mi
