// RK4 stages in row form, FP32 state (lee_rk_row.h).
#define LEE_RK_T float
#include "lee_rk_row.h"
