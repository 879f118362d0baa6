#define FKD_S float
#define FKD_CX false
#define FKD_FIND find_res_fr
#include "kpm_res_inst.inc"
