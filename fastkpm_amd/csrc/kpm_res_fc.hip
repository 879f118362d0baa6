#define FKD_S float
#define FKD_CX true
#define FKD_FIND find_res_fc
#include "kpm_res_inst.inc"
