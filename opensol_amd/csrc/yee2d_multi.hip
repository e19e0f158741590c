// Several 2D steps per launch of one instance (yee2d_multi.h).
#include "yee2d_multi_kernel.h"

YEE_MULTI_KERNELS(YEE_EZ, false)
YEE_MULTI_KERNELS(YEE_HZ, false)
