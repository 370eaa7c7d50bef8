// Internal interface of the small-batch quantised matmul (k_matmul_small.hip),
// used by the GpuMatMulQuant entry points (k_matmul.hip).
#ifndef RPG_AMD_MATMUL_SMALL_H_
#define RPG_AMD_MATMUL_SMALL_H_

#include <cstdint>

namespace rpg {

// One matrix of a launch and its output [n_tokens][rows].
struct SmallMat {
  const uint8_t* w;
  float* out;
  int64_t rows;  // at most 2^31 - 1
  bool q6;       // Q6_K, else Q4_K
};
constexpr int kSmallMaxMats = 4;  // of one kernel launch (a longer group takes several)

// OUT_i[t][r] = sum_e W_i[r][e] x[t][e] for matrices that share x (16-byte aligned,
// cols = 256 nb; Q4_K matrices 16-byte aligned, Q6_K 2-byte). Each output's
// arithmetic depends on its own matrix's size and data, x and n_tokens alone, so a
// group gives the same bits as one call per matrix.
void LaunchMatMulSmall(const SmallMat* mats, int32_t n_mats, int32_t nb, const float* x, int64_t n_tokens);

// Whether that is faster than the tiled kernel (k_matmul.hip, below 32 tokens) or
// the prefill GEMM (matmul_mfma.h). A rule on the matrix's own size.
bool MatMulSmallWins(const SmallMat& m, int32_t nb, int64_t n_tokens);

// up.out <- x . W_up^T, gate.out <- silu(x . W_gate^T) * up.out for two matrices of one type and
// shape: the bits of LaunchMatMulSmall followed by GpuSiluMulInPlace.
void LaunchMatMulSmallSwiGLU(const SmallMat& gate, const SmallMat& up, int32_t nb, const float* x, int64_t n_tokens);

}  // namespace rpg

#endif  // RPG_AMD_MATMUL_SMALL_H_
