// int4_staged_mm_kernel (e2h_int4_staged_kernel.h) at group size 64.
#include "e2h_int4_staged_kernel.h"

template int e2h::staged::launch_group<64>(int, const e2h::staged::StagedArgs &, const e2h::staged::Geometry &, hipStream_t);
