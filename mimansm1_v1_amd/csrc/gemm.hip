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
// Tiles are 256 x 256, one workgroup per CU.  Where the tile count leaves a
// last round mostly empty and the reduction is long, the leftover tiles are
// split along k over all workgroups (SplitTiles): each workgroup writes its
// fp32 partial tiles (at most two, 256 KiB each) and split_sum_kernel adds
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
    for (int b = 0; b < S::TJ; ++b) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float* p = out_at<float>(o, row0 + (lane & 31), col0 + 32 * b + 8 * q + 4 * (lane >> 5));
        if (p) *reinterpret_cast<f32x4*>(p) = val(b, q);
      }
    }
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

namespace {

// Cost of a plan in windows of a 256-column tile (~1.4 us each).
constexpr double SPLIT_COST = 28;   // writing the partial sums and adding them: ~40 us, measured at 65 to 320 tiles
constexpr double HALF_COST = 0.85;  // a half tile (WholeTiles): its copies are a whole tile's

struct Plan {
  bool wide320;
  int n_mblk, n_nblk, grid, left;   // left: tiles split along k (0: none)
  double cost;
  size_t part_bytes;
};

Plan plan_of(int bn, int M, int N, int K, int n_g) {
  Plan p{};
  p.wide320 = bn == 320;
  p.n_mblk = (M + gemm::BM - 1) / gemm::BM;
  p.n_nblk = (N + bn - 1) / bn;
  const long total = (long)p.n_mblk * p.n_nblk;
  const int left = (int)(total % n_g);
  const double tile = (double)gemm::windows_of(K) * bn / 256, full = (double)(total / n_g);
  const double last = left == 0 ? 0 : 2 * left <= n_g ? HALF_COST : 1;
  p.cost = (full + last) * tile;
  p.grid = gemm::persistent_grid(n_g, (int)total);
  const double split = (full + (double)left / n_g) * tile + SPLIT_COST;
  if (left > 0 && split < p.cost) {
    p.cost = split;
    p.left = left;
    p.grid = n_g;
    p.part_bytes = (size_t)(n_g + left) * gemm::BM * bn * 4;
  }
  return p;
}

// The tile width and the split of the leftover tiles, by modelled cost.
Plan make_plan(int M, int N, int K, int cus) {
  const int n_g = ((cus > 0 ? cus : 256) + 7) & ~7;
  const Plan a = plan_of(256, M, N, K, n_g), b = plan_of(320, M, N, K, n_g);
  return b.cost < a.cost ? b : a;
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

template <class S>
hipError_t launch_o(const Launch& l) {
  if (l.a.f32) return launch_s<S, true, false>(l);
  return (long)l.a.M * l.a.N * 2 > gemm::CACHED_BYTES ? launch_s<S, false, true>(l) : launch_s<S, false, false>(l);
}

}  // namespace

bool gemm_operand_fits(int layout, long ld, int n, int K) {
  return gemm::offsets_fit(static_cast<gemm::Layout>(layout), ld, n, K);
}

size_t gemm_workspace_bytes(int M, int N, int K) {
  int cus = 0;
  if (cu_count(cus) != hipSuccess) cus = 256;
  return make_plan(M, N, K, cus).part_bytes;
}

hipError_t launch_gemm(const GemmArgs& a, hipStream_t stream) {
  int cus = 0;
  hipError_t e = cu_count(cus);
  if (e != hipSuccess) return e;
  const Plan plan = make_plan(a.M, a.N, a.K, cus);
  const gemm::Problem p{{static_cast<const __bf16*>(a.x), a.ldx, a.M}, {static_cast<const __bf16*>(a.w), a.ldw, a.N},
                        static_cast<const __bf16*>(a.w1), a.k_cut, a.K, plan.n_mblk, plan.n_nblk};
  const Output o{a.out, a.out1, a.ldo, a.M, a.N, a.out1 ? a.n_cut : a.N};
  const Launch l{a, plan, p, o, stream};
  return plan.wide320 ? launch_o<gemm::Wide320>(l) : launch_o<gemm::Wide256>(l);
}

}  // namespace mm1
