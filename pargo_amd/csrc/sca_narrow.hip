// sca_narrow.hip -- the kernels of sca.hip for rasters of at most 32 columns
// or 16 rows, whose working memory is laid out by the cells they have.
#define PARGO_SCA_NARROW
#include "sca.hip"
