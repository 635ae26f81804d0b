// Token-generation weight stream, F8E4M3 weights (templates: linear_device.h).
#define MI_TRACE_EXPORT 1
#include "gemv_regs.h"

namespace mi {
template int launch_gemv_wd<MI_W_F8E4M3>(const LinearW&, int, int, const ProArgs&, int, const EpiArgs&, hipStream_t);
template int launch_gemv_regs_wd<MI_W_F8E4M3>(const LinearW&, int, const uint16_t*, int, int, const EpiArgs&, hipStream_t, float*, size_t, SlabSum*, bool);
template bool gemv_regs_fits_wd<MI_W_F8E4M3>(int, int, int, size_t);
template bool gemv_regs_whole_wd<MI_W_F8E4M3>(int, int, int, size_t);
template double gemv_regs_us_wd<MI_W_F8E4M3>(int, int, int, size_t, bool);
}
