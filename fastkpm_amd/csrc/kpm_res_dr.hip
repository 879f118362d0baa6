#define FKD_S double
#define FKD_CX false
#define FKD_FIND find_res_dr
#include "kpm_res_inst.inc"
