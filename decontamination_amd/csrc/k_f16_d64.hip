// The 16-bit BMU search over FP32 rows of up to 64 dimensions.
#include "bmu_f16.hpp"

template int somhip_search_f16<64, float>(somhip_model *, const float *, int64_t, int, int, int, int32_t *, int32_t *, double *,
                                       float *, int64_t *, unsigned int *, const int32_t *);
