// A unit of the library for the CPU (UNIT), with its dynamic LDS (LDS 1: the DP consumers',
// 2: the Rietkerk consumers').
#include UNIT

#if LDS == 1
namespace tmk { namespace {
thread_local double s_lds[20480];
} }
#elif LDS == 2
namespace {
thread_local __align__(16) double s_move[20480];
}
namespace tmk { namespace {
thread_local __align__(16) double s_move[20480];
} }
#endif
