// Umbrella translation unit: all kernels + torch bindings compiled together
// (template instantiation happens at the launch sites in bindings.cpp).
#include "elementwise.hip"
#include "kvcache.hip"
#include "attention.hip"
#include "paged_decode.hip"
#include "flash_prefill.hip"
#include "skinny_gemm.hip"
#include "stream_gemm.hip"
#include "slab_gemm.hip"
#include "ring_gemm.hip"
#include "tile_gemm.hip"
#include "sampling.hip"
#include "bindings.cpp"
