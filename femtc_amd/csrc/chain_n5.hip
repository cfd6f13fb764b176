// Chain-kernel instances for N = 5 dofs per direction (degree 4),
// Q in {N, N+1, N+2}, FP64 and FP32.
#include "apply_chain.hpp"

namespace femtc
{
int launch_chain_n5(const ApplyReq& r) { return chain_q<5>(r); }
} // namespace femtc
