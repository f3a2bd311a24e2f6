// Internal (NOT part of the C ABI): the outlier-column mask of LLM.int8 products that follow each other.
//
// A product's rows OR their outlier columns into a mask that must be zero before (csrc/int8_gemm.hip): a launch of 4 us in front of each of the 9 products of a
// two-layer prompt.  In a chain of products on one stream and workspace the mask has a place of its own, and each product clears it for the next one behind its use.
#pragma once
#include "common.h"

struct mi355_i8_chain {
    unsigned* mask;  // in the last mi355_i8_chain_bytes() of a workspace, which no product's own part reaches
    int words;       // of the longest row
    bool clear;      // the mask is zero once the launches so far are done
};
// how a launch is cut: waves of a block, K-slices
extern "C" void mi355_linear_int8_gemm_plan(int M, int N, int K, int R, int* waves, int* ksplit);
size_t mi355_i8_chain_bytes(int K);
int mi355_linear_int8_gemm_chained(const mi355_int8_args* a, mi355_i8_chain* chain, void* workspace, size_t workspace_bytes, mi355_stream_t stream);
