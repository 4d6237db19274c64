#define BEAM_T _Float16
#include "gemm_lines_inst.h"
