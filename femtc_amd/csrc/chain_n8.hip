// Chain-kernel instances for N = 8 dofs per direction (degree 7),
// Q in {N, N+1, N+2}, FP64 and FP32.
#include "apply_chain.hpp"

namespace femtc
{
int launch_chain_n8(const ApplyReq& r) { return chain_q<8>(r); }
} // namespace femtc
