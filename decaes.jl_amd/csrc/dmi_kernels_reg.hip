// The register-resident voxel kernel of one size class: compiled once per class with -DDMI_REG_S=<rows in registers>
// (see dmi_nnls_reg.h).
#include "dmi_kernels.hip"
