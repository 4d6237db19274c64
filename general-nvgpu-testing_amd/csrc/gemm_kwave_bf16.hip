#define KW_T __bf16
#include "gemm_kwave_inst.h"
