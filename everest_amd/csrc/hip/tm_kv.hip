// One instantiation of the mining kernel (tm_variants.h): TMV_VARIANT is its
// node map, enumerate, instrumented, register cap and multi-query numbers.
#include "tm_variants.cuh"
#define TMV_ONE(...) TMV_DEF(__VA_ARGS__)
TMV_ONE(TMV_VARIANT)
