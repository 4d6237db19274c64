#define BEAM_T __bf16
#include "gemm_lines_inst.h"
