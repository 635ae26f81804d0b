// The wide context-encoding GEMM for e4m3 weights (gemm_wide.h).
#include "gemm_wide.h"

namespace mi {
template int launch_gemm_wide_wd<MI_W_F8E4M3>(const LinearW&, int, const uint16_t*, int, int, const EpiArgs&, hipStream_t, int, int, int, float*, SlabSum*);
}
