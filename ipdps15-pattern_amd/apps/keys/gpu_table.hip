// The functors of keys.h compiled for the device (pat_app_gr_table()).
#include "keys.h"

#include "gpu/regular_table.hpp"

PAT_GR_TABLE(FFGPU::map_function_table, FFGPU::reduce_function_table)
