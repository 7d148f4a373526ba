// Source generator for the FP32 MFMA matrix-product kernel (see gemm.cpp).
#pragma once
#include <string>

namespace adhip {

struct GemmConfig {
    bool a_kcontig = true;  // A[m,k]: k has unit stride (else m has)
    bool b_kcontig = false; // B[k,n]: k has unit stride (else n has)
    bool edge = false;      // bounds-checked accesses (odd sizes or unaligned operands)
    bool edge_vec = false;  // with edge: both operands' contiguous extents are at least 4, so threads load 128 bits where all four exist
    int bm = 128;           // block tile: 256 (256x128, 8 waves), 128 (128x128, 4 waves) or 64 (64x64, 4 waves); k depth 16
    int bn = 0;             // block tile columns; 0 = the default for bm (128, or 64 for bm 64).  128x64 is the only other shape
    bool split_k = false;   // blockIdx.y picks a range of k (extra argument k_chunk); slice y of the product goes to C + y*M*N
    bool bf16_parts = false;  // the kernel on the bf16 matrix cores (gemm_split.cpp); needs K >= bk
    int bk = 16;            // k depth of its tiles (16, 32 or 64)
    int k_waves = 1;        // of that kernel: 2 = a tile's k is shared between two sets of wavefronts, whose sums are added at the end
    bool grouped = false;   // blockIdx.y picks one of kGemmGroupSlots products of the same shape (parameters c<i>, a<i>, b<i>)
};

// Problem slots of the grouped kernel; a launch may use fewer (gridDim.y) and fills the rest with any valid pointer.
constexpr int kGemmGroupSlots = 16;

// Element-wise work done on every finished element before it leaves the registers (generated by
// gen_dot_epilogue): extra kernel parameters (", float* e0, const float* b0 ..."), statements that may use
// `row`, `col` and `sum_value`, and whether the product itself is still written to C.
struct GemmEpilogue {
    std::string prelude;  // helper definitions the statements rely on
    std::string params;
    std::string code;
    bool store_c = true;
};

// What both kernels of a configuration share: the epilogue as a macro, the switches, the choice among grouped problems.
std::string gemm_kernel_head(const GemmConfig& cfg, const GemmEpilogue* epilogue);
std::string gemm_tile_head(const GemmConfig& cfg, const std::string& entry);
int gemm_tile_columns(const GemmConfig& cfg);
unsigned gemm_threads(const GemmConfig& cfg);

std::string gemm_kernel_source(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue = nullptr);
// The same product on the bf16 matrix cores, every operand split into three bf16 parts (gemm_split.cpp).
std::string gemm_split_kernel_source(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue = nullptr);

// Products too small for the matrix cores, and operands of any strides (takes the product kernels' arguments, then `int lanes`).
std::string dot_small_source(const std::string& entry, const GemmEpilogue* epilogue = nullptr, bool grouped = false);

}  // namespace adhip
