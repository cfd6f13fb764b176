// Chain-kernel instances for N = 6 dofs per direction (degree 5),
// Q in {N, N+1, N+2}, FP64 and FP32.
#include "apply_chain.hpp"

namespace femtc
{
int launch_chain_n6(const ApplyReq& r) { return chain_q<6>(r); }
} // namespace femtc
