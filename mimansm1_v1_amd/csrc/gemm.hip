// Plain bf16 products on the GEMM core for gfx950: the products around the
// SwiGLU and LM-head kernels and the projections' weight gradients, which the
// reference leaves to torch's GEMMs (CODE/mimans/model/swiglu_tilelang.py:284-301,
// lm_head_tilelang.py:226-243, attention_tilelang.py:470-472).
//
//   out[m][n] = sum_k X(m, k) W(n, k), fp32 accumulation, bf16 or fp32 output
//
// with either operand ROW (k contiguous) or COL (k-major).  W may be two
// matrices joined along k, and the output two matrices joined along n.
//
// Tiles are 256 x 256 or 256 x 320, one workgroup per CU.  Where the tile count leaves a
// last round mostly empty and the reduction is long, the leftover tiles are
// split along k over all workgroups (SplitTiles): each workgroup writes its
// fp32 partial tiles (at most two, 256 or 320 KiB each) and split_sum_kernel adds
// them in a fixed order and rounds once, so results are deterministic.
#include <hip/hip_runtime.h>

#include "gemm.h"
#include "gemm_core.h"

namespace mm1 {

namespace {

struct Output {
  void* p0;      // columns [0, n_cut)
  void* p1;      // columns [n_cut, N)
  long ld;
  int M, N, n_cut;
};

// Address of (row, col) or nullptr outside the tensor; the 64 columns a wave
// stores lie on one side of n_cut (a multiple of 64).
template <class T>
__device__ __forceinline__ T* out_at(const Output& o, long row, int col) {
  if (row >= o.M || col >= o.N) return nullptr;
  return col < o.n_cut ? static_cast<T*>(o.p0) + row * o.ld + col
                       : static_cast<T*>(o.p1) + row * o.ld + (col - o.n_cut);
}

// Rows row0 .. +31 of a wave's TJ column blocks from val(b, q), the f32x4 of
// columns 32b + 8q + 4(lane/32) .. +3 of row lane & 31.
template <class S, bool F32, bool NT, class Val>
__device__ __forceinline__ void store_rows32(const Output& o, char* lds, int lane, long row0, int col0, Val&& val) {
  auto bf16_quad = [&](int b, int q) {
    const f32x4 x = val(b, q);
    bf16x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (__bf16)x[e];
    return v;
  };
  if constexpr (F32) {
#pragma unroll
    for (int b = 0; b < S::TJ; ++b)
      gemm::store_block_f32<S::STAGE_BYTES / 128, NT>(
          lds, lane, [&](int q) { return val(b, q); },
          [&](int r) { return out_at<float>(o, row0 + r, col0 + 32 * b); },
          [&](int c) { return col0 + 32 * b + 4 * c < o.N; });
  } else if constexpr (S::TJ == 2) {
    gemm::store_block128<NT>(
        lds, lane, bf16_quad, [&](int r) { return out_at<__bf16>(o, row0 + r, col0); },
        [&](int c) { return col0 + 8 * c < o.N; });
  } else {
#pragma unroll
    for (int b = 0; b < S::TJ; ++b)
      gemm::store_block64<NT>(
          lds, lane, [&](int q) { return bf16_quad(b, q); },
          [&](int r) { return out_at<__bf16>(o, row0 + r, col0 + 32 * b); },
          [&](int c) { return col0 + 32 * b + 8 * c < o.N; });
  }
}

// One 32 x 32 block from val(q), the f32x4 of columns 8q + 4(lane/32) .. +3 of
// row lane & 31.
template <bool F32, class Val>
__device__ __forceinline__ void store_block32(const Output& o, char* lds, int lane, long row0, int col0, Val&& val) {
  if constexpr (F32) {
    gemm::store_block_f32<16, false>(
        lds, lane, val, [&](int r) { return out_at<float>(o, row0 + r, col0); },
        [&](int c) { return col0 + 4 * c < o.N; });
  } else {
    gemm::store_block64<false>(
        lds, lane,
        [&](int q) {
          const f32x4 x = val(q);
          bf16x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = (__bf16)x[e];
          return v;
        },
        [&](int r) { return out_at<__bf16>(o, row0 + r, col0); }, [&](int c) { return col0 + 8 * c < o.N; });
  }
}

__device__ __forceinline__ f32x4 quad(const f32x16& a, int q) {
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = a[4 * q + e];
  return v;
}

// Partial tile of a slot: [wave][column block][row block][q][lane] x 4 floats,
// so every instruction of a wave moves 1 KiB.
template <class S>
__device__ __forceinline__ long part_index(int slot, int wave, int b, int i, int q, int lane) {
  return ((((((long)slot * gemm::WAVES + wave) * S::TJ + b) * S::TI + i) * 4 + q) * 64 + lane) * 4;
}

}  // namespace

template <gemm::Layout LX, gemm::Layout LW, class S, bool F32, bool NT, class Tiles>
__global__ __launch_bounds__(512, 1) void gemm_kernel(const gemm::Problem p, const Output o, float* part) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = w % S::WM, wn = w / S::WM;
  char* stage = smem + S::RING + S::STAGE_BYTES * w;
  gemm::run<LX, LW, false, S, Tiles>(p, smem, [](int, int) MM1_INLINE {},
                                     [&](int mb, int nb, f32x16 (&acc)[S::TJ][S::TI], int slot) MM1_INLINE {
    if (slot >= 0) {
#pragma unroll
      for (int b = 0; b < S::TJ; ++b) {
#pragma unroll
        for (int i = 0; i < S::TI; ++i) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(part + part_index<S>(slot, w, b, i, q, lane)) = quad(acc[b][i], q);
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < S::TI; ++i)
      store_rows32<S, F32, NT>(o, stage, lane, (long)mb * gemm::BM + 32 * (S::TI * wm + i),
                               nb * S::BN + 32 * S::TJ * wn, [&](int b, int q) { return quad(acc[b][i], q); });
  });
}

// Leftover tile blockIdx.x / 8, wave blockIdx.x % 8 of it, row block = wave of
// this workgroup: the sum of its partial tiles in workgroup order.
template <class S, bool F32>
__global__ __launch_bounds__(64 * S::TI) void split_sum_kernel(const float* __restrict__ part, const Output o,
                                                               int n_mblk, int n_nblk, int left0, int left, int upt,
                                                               int n_g) {
  __shared__ __attribute__((aligned(1024))) char smem[S::TI * S::STAGE_BYTES];
  const int lane = threadIdx.x & 63, i = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = blockIdx.x >> 3, w = blockIdx.x & 7;
  const int wm = w % S::WM, wn = w / S::WM;
  // workgroups whose run [unit(g), unit(g + 1)) meets [l upt, (l + 1) upt)
  auto unit = [&](int g) { return gemm::SplitTiles::unit(g, left, upt, n_g); };
  int g = (int)((long)l * n_g / left);
  while (g > 0 && unit(g) > (long)l * upt) --g;
  while (unit(g + 1) <= (long)l * upt) ++g;
  f32x4 sum[S::TJ][4];
#pragma unroll
  for (int b = 0; b < S::TJ; ++b) {
#pragma unroll
    for (int q = 0; q < 4; ++q) sum[b][q] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (; g < n_g && unit(g) < (long)(l + 1) * upt; ++g) {
    if (unit(g + 1) == unit(g)) continue;   // fewer units than workgroups: an empty run wrote nothing
#pragma unroll
    for (int b = 0; b < S::TJ; ++b) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        sum[b][q] += *reinterpret_cast<const f32x4*>(part + part_index<S>(g + l, w, b, i, q, lane));
    }
  }
  int mb, nb;
  gemm::tile_coords(left0 + l, n_mblk, n_nblk, mb, nb);
  store_rows32<S, F32, false>(o, smem + S::STAGE_BYTES * i, lane, (long)mb * gemm::BM + 32 * (S::TI * wm + i),
                              nb * S::BN + 32 * S::TJ * wn, [&](int b, int q) { return sum[b][q]; });
}

// Small tiles (gemm_core.h): workgroup item = split * tiles + tile, an XCD's
// workgroups on consecutive items; with several splits of k each writes its
// fp32 partial tile ([wave][q][lane] x 4 floats) to slot tile * splits + split
// and small_sum_kernel adds them in split order.  Bound by the latency of one
// tile's k walk (0.35 us a window): 77 x 3328 x 1280 10.6 us a call, 300 x 1280 x
// 1280 10.5, 77 x 1280 x 6656 (6 splits) 14.9, where torch's GEMM takes 20.6 to 23
// (its host work).
template <gemm::Layout LX, gemm::Layout LW, bool F32>
__global__ __launch_bounds__(256) void gemm_small_kernel(const gemm::Problem p, const Output o, float* part,
                                                         int splits) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tiles = p.n_mblk * p.n_nblk, total = tiles * splits, per = (total + 7) / 8;
  const int j = (int)(blockIdx.x >> 3), item = (int)(blockIdx.x & 7) * per + j;
  if (j >= per || item >= total) return;
  const int split = item / tiles, t = item - split * tiles;
  const int nb = t / p.n_mblk, mb = t - nb * p.n_mblk;
  const int n_win = (p.K + gemm::BK - 1) / gemm::BK;
  const int w0 = (int)((long)split * n_win / splits), w1 = (int)((long)(split + 1) * n_win / splits);
  f32x16 acc[1];
  gemm::run_small<LX, LW, false>(p, smem, mb, nb, w0, w1 - w0, acc);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (splits > 1) {
    float* dst = part + ((((long)t * splits + split) * 4 + w) * 4 * 64 + lane) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<f32x4*>(dst + q * 256) = quad(acc[0], q);
    return;
  }
  store_block32<F32>(o, smem + 2048 * w, lane, (long)mb * gemm::SMALL + 32 * (w & 1), nb * gemm::SMALL + 32 * (w >> 1),
                     [&](int q) { return quad(acc[0], q); });
}

template <bool F32>
__global__ __launch_bounds__(256) void small_sum_kernel(const float* __restrict__ part, const Output o, int n_mblk,
                                                        int splits) {
  __shared__ __attribute__((aligned(1024))) char smem[4 * 2048];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t = blockIdx.x, nb = t / n_mblk, mb = t - nb * n_mblk;
  f32x4 sum[4] = {};
  for (int s = 0; s < splits; ++s) {
    const float* src = part + ((((long)t * splits + s) * 4 + w) * 4 * 64 + lane) * 4;
#pragma unroll
    for (int q = 0; q < 4; ++q) sum[q] += *reinterpret_cast<const f32x4*>(src + q * 256);
  }
  store_block32<F32>(o, smem + 2048 * w, lane, (long)mb * gemm::SMALL + 32 * (w & 1), nb * gemm::SMALL + 32 * (w >> 1),
                     [&](int q) { return sum[q]; });
}

namespace {

// Cost of a plan in windows of a 256-column tile (~1.4 us each).
constexpr double SPLIT_COST = 28;   // writing the partial sums and adding them: ~40 us, measured at 65 to 320 tiles
constexpr double FILL_COST = 7;     // launch, first window and epilogue, 10 us
constexpr double HALF_COST = 0.85;  // a half tile (WholeTiles), whose copies are a whole tile's, or a whole tile of
                                    // a k-contiguous x with half of the CUs idle (plan_of)

// Small tiles, in us: the launch and the ring's first fill, each round of
// workgroups, each of its windows, and the sum of the splits.
constexpr double SMALL_FILL = 3, SMALL_ROUND = 1.5, SMALL_WINDOW = 0.35, SMALL_SUM = 4, WINDOW_US = 1.4;

struct Plan {
  bool wide320;
  int splits;                       // small tiles: splits of k (0: large tiles)
  int n_mblk, n_nblk, grid, left;   // left: tiles split along k (0: none)
  double cost;
  size_t part_bytes;
};

// A last round of tiles for at most half of the CUs: half tiles after full
// rounds; alone, whole tiles, which run faster than in a full round with x
// k-contiguous (5662 x 1280 x 3328, 115 tiles: 63 us whole, 79 split along k; 3584 x
// 2048 x 4096, 112 tiles: 86, 96) but not with both operands k-major (4096 x 2048
// x 4937, 128 tiles: 122, 93; x 4096 100, 85).
Plan plan_of(int bn, int M, int N, int K, bool k_major, int n_g) {
  Plan p{};
  p.wide320 = bn == 320;
  p.n_mblk = (M + gemm::BM - 1) / gemm::BM;
  p.n_nblk = (N + bn - 1) / bn;
  const long total = (long)p.n_mblk * p.n_nblk;
  const int left = (int)(total % n_g);
  const double tile = (double)gemm::windows_of(K) * bn / 256, full = (double)(total / n_g);
  const double last = left == 0 ? 0 : 2 * left <= n_g && (total > n_g || !k_major) ? HALF_COST : 1;
  p.cost = FILL_COST + (full + last) * tile;
  p.grid = gemm::persistent_grid(n_g, (int)total);
  const double split = FILL_COST + (full + (double)left / n_g) * tile + SPLIT_COST;
  if (left > 0 && split < p.cost) {
    p.cost = split;
    p.left = left;
    p.grid = n_g;
    p.part_bytes = (size_t)(n_g + left) * gemm::BM * bn * 4;
  }
  return p;
}

Plan small_plan(int M, int N, int K, int n_g) {
  Plan p{};
  p.n_mblk = (M + gemm::SMALL - 1) / gemm::SMALL;
  p.n_nblk = (N + gemm::SMALL - 1) / gemm::SMALL;
  const long tiles = (long)p.n_mblk * p.n_nblk;
  const int n_win = (K + gemm::BK - 1) / gemm::BK;
  auto us = [&](int splits) {
    const double rounds = (double)((tiles * splits + n_g - 1) / n_g);
    return SMALL_FILL + rounds * (SMALL_ROUND + SMALL_WINDOW * ((n_win + splits - 1) / splits)) +
           (splits > 1 ? SMALL_SUM : 0);
  };
  p.splits = 1;
  double best = us(1);
  for (int s = 2; s <= 16 && s * 4 <= n_win && s * tiles <= 2 * n_g; ++s) {
    if (us(s) < best) {
      best = us(s);
      p.splits = s;
    }
  }
  p.cost = best / WINDOW_US;
  p.grid = (int)((tiles * p.splits + 7) / 8 * 8);
  p.part_bytes = p.splits > 1 ? (size_t)tiles * p.splits * gemm::SMALL * gemm::SMALL * 4 : 0;
  return p;
}

// The tile size, and the split of the leftover tiles or of k, by modelled cost.
// k_major: both operands are.
Plan make_plan(int M, int N, int K, bool k_major, int cus, bool joined) {
  const int n_g = ((cus > 0 ? cus : 256) + 7) & ~7;
  const Plan a = plan_of(256, M, N, K, k_major, n_g), b = plan_of(320, M, N, K, k_major, n_g);
  const Plan c = small_plan(M, N, K, n_g);
  const Plan& large = b.cost < a.cost ? b : a;
  return c.cost < large.cost && !joined ? c : large;      // the small tiles take one W only
}

hipError_t cu_count(int& cus) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  return e;
}

struct Launch {
  const GemmArgs& a;
  const Plan& plan;
  const gemm::Problem& p;
  const Output& o;
  hipStream_t stream;
};

template <gemm::Layout LX, gemm::Layout LW, class S, bool F32, bool NT, class Tiles>
hipError_t launch_t(const Launch& l) {
  auto kern = gemm_kernel<LX, LW, S, F32, NT, Tiles>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::LDS_BYTES);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3(l.plan.grid), dim3(512), S::LDS_BYTES, l.stream, l.p, l.o,
                     static_cast<float*>(l.a.workspace));
  return hipGetLastError();
}

template <class S, bool F32, bool NT, class Tiles>
hipError_t launch_l(const Launch& l) {
  if (l.a.x_layout == gemm::ROW)
    return l.a.w_layout == gemm::ROW ? launch_t<gemm::ROW, gemm::ROW, S, F32, NT, Tiles>(l)
                                     : launch_t<gemm::ROW, gemm::COL, S, F32, NT, Tiles>(l);
  return launch_t<gemm::COL, gemm::COL, S, F32, NT, Tiles>(l);
}

template <class S, bool F32, bool NT>
hipError_t launch_s(const Launch& l) {
  if (l.plan.left == 0) return launch_l<S, F32, NT, gemm::WholeTiles>(l);
  hipError_t e = launch_l<S, F32, NT, gemm::SplitTiles>(l);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((split_sum_kernel<S, F32>), dim3(l.plan.left * 8), dim3(64 * S::TI), 0, l.stream,
                     static_cast<const float*>(l.a.workspace), l.o, l.plan.n_mblk, l.plan.n_nblk,
                     l.plan.n_mblk * l.plan.n_nblk - l.plan.left, l.plan.left, gemm::windows_of(l.a.K) / 2, l.plan.grid);
  return hipGetLastError();
}

template <gemm::Layout LX, gemm::Layout LW, bool F32>
hipError_t launch_small_t(const Launch& l) {
  auto kern = gemm_small_kernel<LX, LW, F32>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, gemm::SMALL_LDS);
  if (e != hipSuccess) return e;
  auto part = static_cast<float*>(l.a.workspace);
  hipLaunchKernelGGL(kern, dim3(l.plan.grid), dim3(256), gemm::SMALL_LDS, l.stream, l.p, l.o, part, l.plan.splits);
  if (l.plan.splits > 1)
    hipLaunchKernelGGL((small_sum_kernel<F32>), dim3(l.plan.n_mblk * l.plan.n_nblk), dim3(256), 0, l.stream,
                       static_cast<const float*>(part), l.o, l.plan.n_mblk, l.plan.splits);
  return hipGetLastError();
}

template <bool F32>
hipError_t launch_small(const Launch& l) {
  if (l.a.x_layout == gemm::ROW)
    return l.a.w_layout == gemm::ROW ? launch_small_t<gemm::ROW, gemm::ROW, F32>(l)
                                     : launch_small_t<gemm::ROW, gemm::COL, F32>(l);
  return launch_small_t<gemm::COL, gemm::COL, F32>(l);
}

template <class S>
hipError_t launch_o(const Launch& l) {
  const bool nt = (long)l.a.M * l.a.N * (l.a.f32 ? 4 : 2) > gemm::CACHED_BYTES;
  if (l.a.f32) return nt ? launch_s<S, true, true>(l) : launch_s<S, true, false>(l);
  return nt ? launch_s<S, false, true>(l) : launch_s<S, false, false>(l);
}

}  // namespace

bool gemm_operand_fits(int layout, long ld, int n, int K) {
  return gemm::offsets_fit(static_cast<gemm::Layout>(layout), ld, n, K);
}

size_t gemm_workspace_bytes(int M, int N, int K, bool k_major, bool joined) {
  int cus = 0;
  if (cu_count(cus) != hipSuccess) cus = 256;
  return make_plan(M, N, K, k_major, cus, joined).part_bytes;
}

double gemm_estimate_us(int M, int N, int K) {
  int cus = 0;
  if (cu_count(cus) != hipSuccess) cus = 256;
  return make_plan(M, N, K, false, cus, false).cost * WINDOW_US;
}

hipError_t launch_gemm(const GemmArgs& a, hipStream_t stream) {
  int cus = 0;
  hipError_t e = cu_count(cus);
  if (e != hipSuccess) return e;
  const Plan plan = make_plan(a.M, a.N, a.K, a.x_layout == gemm::COL, cus, a.w1 != nullptr);
  const gemm::Problem p{{static_cast<const __bf16*>(a.x), a.ldx, a.M}, {static_cast<const __bf16*>(a.w), a.ldw, a.N},
                        static_cast<const __bf16*>(a.w1), a.k_cut, a.K, plan.n_mblk, plan.n_nblk};
  const Output o{a.out, a.out1, a.ldo, a.M, a.N, a.out1 ? a.n_cut : a.N};
  const Launch l{a, plan, p, o, stream};
  if (plan.splits > 0) return a.f32 ? launch_small<true>(l) : launch_small<false>(l);
  return plan.wide320 ? launch_o<gemm::Wide320>(l) : launch_o<gemm::Wide256>(l);
}

}  // namespace mm1
