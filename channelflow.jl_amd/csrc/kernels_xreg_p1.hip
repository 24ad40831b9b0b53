// one form of the register x pass (list at the end of kernels_xreg.hip)
#define CF_X_PART 1
#include "kernels_xreg.hip"
