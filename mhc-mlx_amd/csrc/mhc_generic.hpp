// Arguments of the kernels with runtime n (generic.hip, lf32_*, lv_*), and the entry points of generic.hip (16 < n <= 64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mhc {

struct GenArgs {
  const void* x;
  const void* y;
  const void* g;
  void* out;  // fused fwd: out; bwd: dx
  void* dy;
  const float* M;
  const float* hpre;
  const float* hpost;
  const float* w;
  float* inv_rms;
  float* part;
  float* scratch;  // bwd: 2*C floats per workgroup
  float* dM_tok;
  float* dpre_tok;
  float* dpost_tok;
  int64_t T;
  int64_t M_ts;
  int64_t h_ts;
  int n;
  int C;
  int Cp;
  int P;
  int h_mode;
  float eps;
};

// What a forward kernel reads of GenArgs: the runtime's launch costs 0.65 us
// more of host time above 112 bytes of kernel arguments, which a small
// forward, bound by its launches, would pay on every call.
struct GenFwdArgs {
  const void* x;
  void* out;
  const float* M;
  const float* hpre;
  const float* hpost;
  const float* w;
  float* inv_rms;
  int64_t T;
  int M_ts;  // n * n and n, or 0
  int h_ts;
  int n;
  int C;
  int h_mode;
  float eps;

  explicit GenFwdArgs(const GenArgs& A)
      : x(A.x), out(A.out), M(A.M), hpre(A.hpre), hpost(A.hpost), w(A.w), inv_rms(A.inv_rms), T(A.T),
        M_ts((int)A.M_ts), h_ts((int)A.h_ts), n(A.n), C(A.C), h_mode(A.h_mode), eps(A.eps) {}
};
static_assert(sizeof(GenFwdArgs) + sizeof(int) <= 112, "beyond the runtime's fast kernel-argument size");

int64_t gen_grid(int64_t T);
int gen_fused_fwd(const GenArgs& A, int x_dtype, int out_dtype, hipStream_t s);
int gen_fused_bwd(const GenArgs& A, int x_dtype, int g_dtype, hipStream_t s, int64_t* num_partials);
int gen_mix_fwd(const GenArgs& A, int x_dtype, int y_dtype, int out_dtype, hipStream_t s);
int gen_mix_bwd(const GenArgs& A, int x_dtype, int y_dtype, int g_dtype, hipStream_t s, int64_t blocks);

}  // namespace mhc
