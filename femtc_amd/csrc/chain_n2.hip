// Chain-kernel instances for N = 2 dofs per direction (degree 1),
// Q in {N, N+1, N+2}, FP64 and FP32.
#include "apply_chain.hpp"

namespace femtc
{
int launch_chain_n2(const ApplyReq& r) { return chain_q<2>(r); }
} // namespace femtc
