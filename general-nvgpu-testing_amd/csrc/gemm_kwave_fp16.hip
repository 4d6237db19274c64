#define KW_T _Float16
#include "gemm_kwave_inst.h"
