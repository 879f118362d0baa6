#define FKD_S double
#define FKD_CX true
#define FKD_FIND find_res_dc
#include "kpm_res_inst.inc"
