// RK4 stages in row form, FP64 state (lee_rk_row.h).
#define LEE_RK_T double
#include "lee_rk_row.h"
