// Chain-kernel instances for N = 4 dofs per direction (degree 3),
// Q in {N, N+1, N+2}, FP64 and FP32.
#include "apply_chain.hpp"

namespace femtc
{
int launch_chain_n4(const ApplyReq& r) { return chain_q<4>(r); }
} // namespace femtc
