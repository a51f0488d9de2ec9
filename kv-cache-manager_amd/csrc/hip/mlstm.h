// What both forms of the matrix memory (mlstm.hip, mlstm_chunks.hip) begin with.
#pragma once
#include <hip/hip_runtime.h>

namespace kvcm {

// every row's three factors, coef[row, head] = (exp(lf + m before - m), exp(li - m), exp(-m), .), and the slots' new maxima; `stretches`: a long run's by
// several waves
void mlstm_factors(const float* ig, int ldi, const float* fg, int ldf, const float* i_bias, const float* f_bias, float cap, float4* coef,
                   float* m_state, const int* run_start, const int* seq_start, const int* state_slots, int S, int heads, int T, int max_run,
                   int one_order, bool stretches, hipStream_t s);

}  // namespace kvcm
