// Host interface of the plain bf16 products (gemm.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace mm1 {

struct GemmArgs {
  const void* x;
  long ldx;
  int x_layout;         // 0: [M, K] rows, 1: [K, M] rows
  const void* w;
  long ldw;
  int w_layout;         // 0: [N, K] rows, 1: [K, N] rows
  const void* w1;       // W from k = k_cut on, or nullptr (k_cut 0)
  int k_cut;
  void* out;
  void* out1;           // columns from n_cut on, or nullptr
  int n_cut;
  long ldo;
  bool f32;
  void* workspace;
  int M, N, K;
};

bool gemm_operand_fits(int layout, long ld, int n, int K);
size_t gemm_workspace_bytes(int M, int N, int K, bool k_major, bool joined);
double gemm_estimate_us(int M, int N, int K);
hipError_t launch_gemm(const GemmArgs& a, hipStream_t stream);

}  // namespace mm1
