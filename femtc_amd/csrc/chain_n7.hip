// Chain-kernel instances for N = 7 dofs per direction (degree 6),
// Q in {N, N+1, N+2}, FP64 and FP32.
#include "apply_chain.hpp"

namespace femtc
{
int launch_chain_n7(const ApplyReq& r) { return chain_q<7>(r); }
} // namespace femtc
