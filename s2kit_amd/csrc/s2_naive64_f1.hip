// K-chunked dense FP64 forward, bw <= 256, 64 columns per block (a file of its own: its
// K-loop instances compile beside the others').
#include "s2_naive64_kc.h"

namespace s2 {
template void n64_fwd_kc_launch<1, 4>(const DevConsts&, const GemmTables&, const double2*, double*, double*, int, Fmt,
                                      hipStream_t);
}
