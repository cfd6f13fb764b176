// Chain-kernel instances for N = 3 dofs per direction (degree 2),
// Q in {N, N+1, N+2}, FP64 and FP32.
#include "apply_chain.hpp"

namespace femtc
{
int launch_chain_n3(const ApplyReq& r) { return chain_q<3>(r); }
} // namespace femtc
