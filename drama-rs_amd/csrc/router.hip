// Router: logits, softmax and top-k (reference: kernels/drama.cu:317-468, src/ffi.rs:41,55-59)
// plus the bf16 GEMM dr_gemm that the prefill router uses (src/engine.rs:554).
//
// These kernels follow the canonical fp32 operation order of canon.hpp (RMSNorm, row dot,
// softmax, top-k), so the CPU oracle reproduces the logits, the softmax probabilities and
// hence the selected experts bit for bit.
#include "router_rows.hpp"

#include <algorithm>

#pragma clang fp contract(off)

using namespace drm;

namespace {

// Decode router of a few rows in one launch: sets of two rows (LAST in the last one; ONE: a single
// set), each with its own router blocks (router_rows.hpp) and its own byte of the counter.  A block's time is its staging, norms
// and LDS reads per row: 8 rows on one set of blocks took 12.8 us, on two sets 8.9, on four 8.1; 4 rows 8.6
// on one set, 8.0 on two.
template <int LAST, bool ONE>
__global__ void __launch_bounds__(RT_WPB * 64)
    k_router_topk_rows(const uint16_t* __restrict__ W, const float* __restrict__ x, const float* __restrict__ nw,
                       float eps, float* __restrict__ logits, int E, int topk, int* __restrict__ idx,
                       float* __restrict__ wts, float* __restrict__ sgate, uint32_t* __restrict__ counter) {
  __shared__ float4 xs[ONE ? LAST : 2][2048 / 4];
  const int set = ONE ? 0 : blockIdx.y, r = 2 * set;  // r: first row of the set
  x += (size_t)r * 2048, logits += (size_t)r * (E + 1), idx += r * topk, wts += r * topk, sgate += r;
  if constexpr (!ONE && LAST == 1) {
    if (blockIdx.y + 1 < gridDim.y) {
      router_rows_block<2, false>(blockIdx.x, gridDim.x, W, x, nw, eps, logits, E, topk, idx, wts, sgate, counter,
                                  nullptr, 0u, xs, 8 * set);
      return;
    }
  }
  router_rows_block<LAST, ONE>(blockIdx.x, gridDim.x, W, x, nw, eps, logits, E, topk, idx, wts, sgate, counter, nullptr,
                               0u, xs, 8 * set);
}

// One row per block.  topk <= 8: waves 0..3 each pick the top 8 of 64 experts and wave 4
// computes the softmax denominator, then wave 0 ranks the 32 candidates (the same selection
// and weights as canon_softmax_topk, in less than half the time); topk > 8: wave 0 alone.
__global__ void __launch_bounds__(320)
    k_moe_topk(const float* __restrict__ logits, int E, int topk, int stride, int* __restrict__ idx,
               float* __restrict__ wts, float* __restrict__ sgate) {
  const int r = blockIdx.x, lane = lane_id(), wave = wave_id();
  const float* l = logits + (size_t)r * stride;
  __shared__ float lg[257];
  __shared__ uint64_t s_cand[32];
  __shared__ int s_sel[8];
  __shared__ float s_mz[2];
  if ((int)threadIdx.x <= E) lg[threadIdx.x] = l[threadIdx.x];
  __syncthreads();
  if (wave == 0 && lane == 0) sgate[r] = lg[E];
  if (topk <= 8) {
    if (wave < 4) {
      int ck, ce;
      canon_select_group8(lg, E, wave, &ck, &ce);
      if (lane < 8) s_cand[wave * 8 + lane] = canon_cand64(ck, ce);
    } else {
      float m;
      const float z = canon_softmax_z(lg, E, &m);
      if (lane == 0) s_mz[0] = m, s_mz[1] = z;
    }
    __syncthreads();
    if (wave != 0) return;
    const int id = merge_picks(s_cand, s_sel, topk);
    const float w = canon_topk_weight(lg[lane < topk ? id : 0], s_mz[0], s_mz[1], topk);
    if (lane < topk) idx[(size_t)r * topk + lane] = id, wts[(size_t)r * topk + lane] = w;
  } else {
    if (wave != 0) return;
    int my_idx;
    float my_w;
    canon_softmax_topk(lg, E, topk, &my_idx, &my_w);
    if (lane < topk) idx[(size_t)r * topk + lane] = my_idx, wts[(size_t)r * topk + lane] = my_w;
  }
}

// The canonical GEMM for up to 4 rows of A (decode batches): one wave per W row, which it loads once and
// dots with every A row (all loads issued first); 8 waves per block.  3.8 us at 4 x 257 x 2048 against
// 5.1 for k_gemm_mfma, whose 16-row tiles would be mostly empty (5 rows: 5.3 against 4.9).
constexpr int GR_MAXM = 4;
template <int NCH>
__global__ void __launch_bounds__(512)
    k_gemm_rows(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W, float* __restrict__ C, int M,
                int N, int K, float beta) {
  const int lane = lane_id();
  const int n = blockIdx.x * 8 + wave_id();
  if (n >= N) return;
  const int KC = K / 8;
  uint4 w[NCH];
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int c = lane + WAVE * j;
    w[j] = c < KC ? ld16(W + (size_t)n * K + (size_t)c * 8) : make_uint4(0, 0, 0, 0);
  }
  static_assert(GR_MAXM == 4, "all rows at once");
  uint4 av[4][NCH];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = r < M ? r : M - 1;
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      const int c = lane + WAVE * j;
      av[r][j] = c < KC ? ld16(A + (size_t)m * K + (size_t)c * 8) : make_uint4(0, 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < NCH; ++j) {
      if (lane + WAVE * j < KC) {
        const uint4 a = av[r][j], b = w[j];
        acc = __builtin_fmaf(bf16_lo(b.x), bf16_lo(a.x), acc);
        acc = __builtin_fmaf(bf16_hi(b.x), bf16_hi(a.x), acc);
        acc = __builtin_fmaf(bf16_lo(b.y), bf16_lo(a.y), acc);
        acc = __builtin_fmaf(bf16_hi(b.y), bf16_hi(a.y), acc);
        acc = __builtin_fmaf(bf16_lo(b.z), bf16_lo(a.z), acc);
        acc = __builtin_fmaf(bf16_hi(b.z), bf16_hi(a.z), acc);
        acc = __builtin_fmaf(bf16_lo(b.w), bf16_lo(a.w), acc);
        acc = __builtin_fmaf(bf16_hi(b.w), bf16_hi(a.w), acc);
      }
    }
    acc = wave_sum(acc);
    if (lane == 0 && r < M) {
      float* c = C + (size_t)r * N + n;
      *c = beta == 0.f ? acc : acc + beta * *c;
    }
  }
}

// one chunk of -0 and one of +0 (k_gemm_mfma)
__device__ const uint4 k_pad[2] = {{0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u}, {0u, 0u, 0u, 0u}};

// The same canonical GEMM on the fp32 matrix unit.  v_mfma_f32_16x16x1_4b_f32 is four independent 16 x 16
// rank-1 updates whose every element is one fp32 fma (rounded to nearest even, subnormals kept, checked
// against fmaf), so block b of an instruction can carry the running sum of one canonical lane: set s
// of a wave holds lanes 4 s .. 4 s + 3 of the 64 as the four blocks, and inputs enter in the canonical
// order (chunk lane + 64 j, then element).  An MFMA lane (b, i) reads whole 16-byte chunks of row i, 8
// MFMAs per chunk pair, straight from global memory.  The four blocks of an output lie in one
// lane's registers, so the canonical xor tree is (b0 + b1) + (b2 + b3) there, then over the wave's
// sets, then over the NW waves through LDS (a + b = b + a, so the same bits as the butterfly).
// The matrix unit does 32 of these fmas per clock and SIMD where the vector unit does 16, and
// the bf16 -> fp32 conversions fall from one per 8 / 5 fmas to one per 16 and matrix row.
// Block: 16 BM x 16 BN outputs, NW waves of 64 / NW canonical lanes each, four waves per SIMD (at most 128
// registers: two blocks of 8 waves per CU).  Consecutive tiles of
// one XCD share their W rows.
// What bounds it: large shapes the loads (16 rows x 64 bytes per instruction, ~8 TB/s of L2 reads; 32 x 32
// tiles run at 65% of the fp32 matrix rate), small ones the MFMAs of one tile (K = 2048, 32 x 32: 128 per wave, four
// waves per SIMD, 33 clocks each: 7 us).
typedef float f32x16 __attribute__((ext_vector_type(16)));
template <int NCH, int BM, int BN, int NW, bool FULL>
__global__ void __launch_bounds__(NW * 64, 4)
    k_gemm_mfma(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W, float* __restrict__ C, int M, int N,
                int K, float beta) {
  constexpr int S = 16 / NW;               // sets of four canonical lanes per wave
  constexpr int D = NCH < 2 ? NCH : 2;     // chunk rounds in flight
  __shared__ float red[NW][BM * BN * 4][64];
  const int lane = lane_id(), wave = wave_id(), i16 = lane & 15;
  const int tm = (M + 16 * BM - 1) / (16 * BM), tiles = tm * ((N + 16 * BN - 1) / (16 * BN));
  const int per = (tiles + 7) / 8, tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (tile >= tiles) return;
  const int m0 = tile % tm * 16 * BM, n0 = tile / tm * 16 * BN;
  const int KC = K / 8, c0 = 64 / NW * wave + (lane >> 4);  // this lane's first chunk
  const uint16_t *ap[BM], *wp[BN];  // rows past the end repeat the last one; their outputs are not stored
#pragma unroll
  for (int x = 0; x < BM; ++x) ap[x] = A + (size_t)min(m0 + 16 * x + i16, M - 1) * K;
#pragma unroll
  for (int y = 0; y < BN; ++y) wp[y] = W + (size_t)min(n0 + 16 * y + i16, N - 1) * K;
  f32x16 acc[S][BM][BN];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int x = 0; x < BM; ++x)
#pragma unroll
      for (int y = 0; y < BN; ++y) acc[s][x][y] = (f32x16)(0.f);
  uint4 av[D][S][BM], wv[D][S][BN];
  // FULL: every chunk exists (K = 512 NCH); otherwise chunks past K / 8 are -0 in A and +0 in W
  // (fma(-0, +0, sum) = sum for every sum; a product of +0 would turn a sum of -0 into +0).  With more than one
  // round they are loaded from k_pad: a select on the loaded words would wait for them where they are requested
  auto chunk = [&](const uint16_t* row, int c, int pad) {
    const uint16_t* p = row + (size_t)c * 8;
    if (FULL) return ld16(p);
    if (NCH > 1) return ld16(c < KC ? p : reinterpret_cast<const uint16_t*>(k_pad + pad));
    const uint32_t z = pad == 0 ? 0x80008000u : 0u;
    const uint4 v = ld16(row + (size_t)min(c, KC - 1) * 8);
    return c < KC ? v : make_uint4(z, z, z, z);
  };
  // round j has a chunk: without asking up to NCH / 2, since K > 256 NCH for NCH > 1 (NCH = 8: asked from the
  // second round on, which keeps the unrolled rounds apart and the 8-wave tile at 125 registers, not 136)
  auto round_in = [&](int j) { return FULL || j <= (NCH < 8 ? NCH / 2 : 0) || 64 * j < KC; };
  auto load = [&](int j) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
#pragma unroll
      for (int x = 0; x < BM; ++x) av[j % D][s][x] = chunk(ap[x], c0 + 4 * s + 64 * j, 0);
#pragma unroll
      for (int y = 0; y < BN; ++y) wv[j % D][s][y] = chunk(wp[y], c0 + 4 * s + 64 * j, 1);
    }
  };
#pragma unroll
  for (int j = 0; j < D; ++j)
    if (round_in(j)) load(j);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    if (!round_in(j)) break;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        auto element = [&](const uint4& v) {
          const uint32_t q = e < 2 ? v.x : e < 4 ? v.y : e < 6 ? v.z : v.w;
          return (e & 1) ? bf16_hi(q) : bf16_lo(q);
        };
        float a[BM], w[BN];
#pragma unroll
        for (int x = 0; x < BM; ++x) a[x] = element(av[j % D][s][x]);
#pragma unroll
        for (int y = 0; y < BN; ++y) w[y] = element(wv[j % D][s][y]);
#pragma unroll
        for (int x = 0; x < BM; ++x)
#pragma unroll
          for (int y = 0; y < BN; ++y)
            acc[s][x][y] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[x], w[y], acc[s][x][y], 0, 0, 0);
      }
    if (j + D < NCH && round_in(j + D)) load(j + D);
    __builtin_amdgcn_sched_barrier(0);
  }
  // D layout: register 4 b + r of lane l is row 4 (l / 16) + r, column l % 16 of block b
#pragma unroll
  for (int x = 0; x < BM; ++x)
#pragma unroll
    for (int y = 0; y < BN; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float p[S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const f32x16& v = acc[s][x][y];
          p[s] = (v[r] + v[4 + r]) + (v[8 + r] + v[12 + r]);
        }
#pragma unroll
        for (int d = 1; d < S; d *= 2)
#pragma unroll
          for (int s = 0; s + d < S; s += 2 * d) p[s] = p[s] + p[s + d];
        red[wave][(x * BN + y) * 4 + r][lane] = p[0];
      }
  __syncthreads();
  for (int o = wave; o < BM * BN * 4; o += NW) {
    float p[NW];
#pragma unroll
    for (int q = 0; q < NW; ++q) p[q] = red[q][o][lane];
#pragma unroll
    for (int d = 1; d < NW; d *= 2)
#pragma unroll
      for (int q = 0; q + d < NW; q += 2 * d) p[q] = p[q] + p[q + d];
    const int m = m0 + 16 * (o / (4 * BN)) + 4 * (lane >> 4) + (o & 3), n = n0 + 16 * (o / 4 % BN) + i16;
    if (m < M && n < N) {
      float* c = C + (size_t)m * N + n;
      *c = beta == 0.f ? p[0] : p[0] + beta * *c;
    }
  }
}

template <int NCH, int BM, int BN, int NW>
void launch_gemm_mfma(const uint16_t* A, const uint16_t* W, float* C, int M, int N, int K, float beta, hipStream_t st) {
  const int tiles = ((M + 16 * BM - 1) / (16 * BM)) * ((N + 16 * BN - 1) / (16 * BN));
  const dim3 grid((tiles + 7) / 8 * 8), block(NW * 64);
  // K = 4096, 8 waves: always the instance with chunk bounds, since the other would need 135 registers
  // (one block per CU: 300 x 1024 x 4096 40.6 us against 38.1, 1024 x 1024 108 against 97)
  if constexpr (NW != 8 || NCH != 8) {
    if (K == NCH * 512) {
      hipLaunchKernelGGL((k_gemm_mfma<NCH, BM, BN, NW, true>), grid, block, 0, st, A, W, C, M, N, K, beta);
      return;
    }
  }
  hipLaunchKernelGGL((k_gemm_mfma<NCH, BM, BN, NW, false>), grid, block, 0, st, A, W, C, M, N, K, beta);
}

// The tile with the least cost a + b r, r the rounds of 256 tiles: fitted to the times of every tile over 5 to
// 1024 rows, 33 to 16384 columns and K = 504 to 4096 (units of 10 ns at K = 512 and at K = 2048, where the order is that
// of every larger K but for the 8-wave tile).  Few tiles: the smallest, whose waves have the fewest products; many: the large
// ones, which load less per product, as long as their last round and their rows past M cost less than that saves.
// us at K = 2048 for 16 x 16, 32 x 16 or 16 x 32, 32 x 32, 32 x 16 tiles of 8 waves: 100 x 257 5.8 / 8.1 / 12.0 / 8.7,
// 300 x 257 9.4 / 8.1 / 12.2 / 8.8, 512 x 257 13.0 / 14.6 / 12.2 / 14.3, 1024 x 257 20.0 / 21 / 23.5 / 19.9, 5 x 4104 7.3 /
// 7.6 (16 x 32) / 11.2 / 12.3.  The vector kernel this replaces: 6.9, 8.5, 15.3, 28.0 and 9.5; it was the faster one (by up
// to 15%, K <= 1024) only where 17 to 32 rows meet a little over 4096 columns: 257 tiles or more at every size but 32 x 32.
template <int NCH>
void launch_gemm(const uint16_t* A, const uint16_t* W, float* C, int M, int N, int K, float beta, hipStream_t st) {
  if (M <= GR_MAXM) {
    hipLaunchKernelGGL(k_gemm_rows<NCH>, dim3((N + 7) / 8), dim3(512), 0, st, A, W, C, M, N, K, beta);
    return;
  }
  const long long m16 = (M + 15ll) / 16, m32 = (M + 31ll) / 32, n16 = (N + 15ll) / 16, n32 = (N + 31ll) / 32;
  auto cost = [](long long tiles, int a1, int b1, int a, int b) {
    const long long r = (tiles + 255) / 256;
    return NCH == 1 ? a1 + b1 * r : a + b * r;
  };
  const long long c11 = cost(m16 * n16, 240, 120, 230, 350), c21 = cost(m32 * n16, 200, 175, 150, 655);
  const long long c12 = cost(m16 * n32, 200, 176, 150, 660), c22 = cost(m32 * n32, 100, 390, 90, 1120);
  // 8 waves: K = 4096 runs with chunk bounds (above) and costs more (700 x 2048 130 us against 123 for 32 x 32).
  // K = 2048 at three rounds: 1024 x 257 takes 19.8 us, level with 16 x 16 tiles (20.0), but beside other kernels, which
  // the 16-wave blocks of those leave no room, it is the shorter one: a prefill layer of 1024 rows with its shared
  // expert on a second stream 237 us against 250
  const long long c8 = K == 4096   ? cost(m32 * n16, 220, 164, 200, 630)
                       : K == 2048 ? cost(m32 * n16, 220, 164, 315, 550)
                                   : cost(m32 * n16, 220, 164, 345, 550);
  const long long c = std::min({c11, c21, c12, c22, c8});
  if (c == c11) launch_gemm_mfma<NCH, 1, 1, 16>(A, W, C, M, N, K, beta, st);
  else if (c == c21) launch_gemm_mfma<NCH, 2, 1, 16>(A, W, C, M, N, K, beta, st);
  else if (c == c12) launch_gemm_mfma<NCH, 1, 2, 16>(A, W, C, M, N, K, beta, st);
  else if (c == c22) launch_gemm_mfma<NCH, 2, 2, 16>(A, W, C, M, N, K, beta, st);
  else launch_gemm_mfma<NCH, 2, 1, 8>(A, W, C, M, N, K, beta, st);
}

}  // namespace

hipStream_t gemm_handle_stream(void* h);

API int dr_router_topk(const uint16_t* W, const float* x, const float* nw, float eps, float* logits, int E, int topk,
                       int K, int* idx, float* wts, float* sgate, uint32_t* counter, const char*, const char*,
                       const char*, const char*, size_t, size_t, size_t, size_t, hipStream_t st) {
  if (K != 2048 || E > 256 || E < 1 || topk > 32 || topk < 1 || topk > E) return -1;
  // the one-row case of the small-batch router (its one-wave top-k measured 0.3 us shorter per
  // call than four group selections and a rank merge, with the same picks)
  hipLaunchKernelGGL((k_router_topk_rows<1, true>), dim3((E + RT_WPB) / RT_WPB), dim3(RT_WPB * 64), 0, st, W, x, nw, eps, logits,
                     E, topk, idx, wts, sgate, counter);
  return 0;
}

API int dr_router_topk_rows(const uint16_t* W, const float* x, const float* nw, float eps, float* logits, int E,
                            int topk, int K, int rows, int* idx, float* wts, float* sgate, uint32_t* counter,
                            hipStream_t st) {
  if (K != 2048 || E > 256 || E < 1 || topk > 32 || topk < 1 || topk > E || rows < 1 || rows > 8) return -1;
  const dim3 g((E + RT_WPB) / RT_WPB, (rows + 1) / 2), b(RT_WPB * 64);
  static_assert((256 + RT_WPB) / RT_WPB < 256, "a set's block count fits its byte of the counter");
  // one set alone on the counter needs no set offsets and clears it with a store: 2 rows, 256 experts, the same
  // time as before there were sets (6.60 us against 6.61); as one of several sets 2% more (6.63 against 6.49)
  auto kern = rows == 1 ? k_router_topk_rows<1, true> : rows == 2 ? k_router_topk_rows<2, true>
              : rows % 2 ? k_router_topk_rows<1, false> : k_router_topk_rows<2, false>;
  hipLaunchKernelGGL(kern, g, b, 0, st, W, x, nw, eps, logits, E, topk, idx, wts, sgate, counter);
  return 0;
}

API int dr_moe_topk(const float* logits, int rows, int E, int topk, int stride, int* idx, float* wts, float* sgate,
                    hipStream_t st) {
  if (E > 256 || E < 1 || topk > 32 || topk < 1 || topk > E || stride < E + 1) return -1;
  if (rows <= 0) return 0;
  hipLaunchKernelGGL(k_moe_topk, dim3(rows), dim3(320), 0, st, logits, E, topk, stride, idx, wts, sgate);
  return 0;
}

API int dr_gemm(void* h, const uint16_t* A, const uint16_t* W, float* C, int M, int N, int K, float beta) {
  if (K % 8 != 0 || K <= 0 || M < 0 || N < 0) return -1;
  if (M == 0 || N == 0) return 0;
  hipStream_t st = gemm_handle_stream(h);
  const int kc = K / 8;
  if (kc <= 64) launch_gemm<1>(A, W, C, M, N, K, beta, st);
  else if (kc <= 128) launch_gemm<2>(A, W, C, M, N, K, beta, st);
  else if (kc <= 256) launch_gemm<4>(A, W, C, M, N, K, beta, st);
  else if (kc <= 512) launch_gemm<8>(A, W, C, M, N, K, beta, st);
  else return -1;
  return 0;
}
