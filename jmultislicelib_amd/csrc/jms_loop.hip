// jms_loop.hip -- instantiates the one-launch slice loops of one row length,
// selected at compile time with -DJMS_N=<length>.
#include "jms_loop_impl.hpp"

#ifndef JMS_N
#error "compile with -DJMS_N=<row length>"
#endif

namespace jms {
template hipError_t launch_loop_n<JMS_N, 64>(int, const LoopArgs&, bool, hipStream_t);
template hipError_t launch_loop_n<JMS_N, 96>(int, const LoopArgs&, bool, hipStream_t);
template hipError_t launch_loop_n<JMS_N, 128>(int, const LoopArgs&, bool, hipStream_t);
}  // namespace jms
