// Chain-kernel instances for N = 9 dofs per direction (degree 8),
// Q in {N, N+1, N+2}, FP64 and FP32.
#include "apply_chain.hpp"

namespace femtc
{
int launch_chain_n9(const ApplyReq& r) { return chain_q<9>(r); }
} // namespace femtc
