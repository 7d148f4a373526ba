// Source generators for the matrix-product kernels: on the bf16 matrix cores (gemm_split.cpp), on the FP32 ones and for small
// products (gemm.cpp).
#pragma once
#include <string>

namespace adhip {

struct GemmConfig {
    bool a_kcontig = true;  // A[m,k]: k has unit stride (else m has)
    bool b_kcontig = false; // B[k,n]: k has unit stride (else n has)
    bool edge = false;      // bounds-checked accesses (odd sizes or unaligned operands)
    bool edge_vec = false;  // with edge: both operands' contiguous extents are at least 4, so threads load 128 bits where all four exist
    // block tile: on the bf16 matrix cores 256x256, 128x128, 128x64, 64x64, and without a staging buffer 64x32, 32x64 and 32x32; on the FP32 ones 256x128, 128x128, 128x64 or 64x64
    int bm = 128;
    int bn = 0;             // its columns; 0 = the FP32 kernel's for bm (128, or 64 for bm 64)
    bool bf16_parts = false;  // the kernel on the bf16 matrix cores (gemm_split.cpp); needs K >= bk
    bool split_k = false;   // of that kernel: blockIdx.y picks a range of k (extra argument k_chunk); slice y of the product goes to C + y*M*N
    int bk = 16;            // k depth of a tile: 16, 32 or 64, on the FP32 matrix cores 16
    // of that kernel: 2 = a tile's k is shared between two sets of wavefronts, whose sums are added at the end; kDirectWaves =
    // the kernel without a staging buffer (gemm_direct.cpp), whose eight wavefronts share k in steps of 32
    int k_waves = 1;
    bool narrow_m = false, narrow_n = false;  // of the latter: fewer rows / columns than a tile's
    bool wide_lines = false;                  // of the latter: lines of 2^22 elements and more
    bool grouped = false;   // blockIdx.y picks one of kGemmGroupSlots products of the same shape (parameters c<i>, a<i>, b<i>)
};

constexpr int kDirectWaves = 8;

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
std::string gemm_tile_head(const GemmConfig& cfg);
// The entry's name and parameters, in plain text (a launch that runs several kernels reads them from the source), the
// test of its guard and the choice among grouped problems; `more` are further parameters behind the strides.
std::string gemm_entry(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue, unsigned threads, const char* more = "");
int gemm_tile_columns(const GemmConfig& cfg);
unsigned gemm_threads(const GemmConfig& cfg);
// LDS of a block: on the bf16 matrix cores one array `lds`
size_t gemm_lds_bytes(const GemmConfig& cfg);

std::string gemm_kernel_source(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue = nullptr);
// The same product on the bf16 matrix cores, every operand split into three bf16 parts (gemm_split.cpp).
std::string gemm_split_kernel_source(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue = nullptr);

// The same for small outputs, with operands that go from memory to the matrix cores' registers (gemm_direct.cpp).
std::string gemm_direct_kernel_source(const GemmConfig& cfg, const std::string& entry, const GemmEpilogue* epilogue = nullptr);
// What both have in common: types and the splitting of operands; the product once more where it is not finite, and the stores.
std::string split_types();
std::string split_tail();

// Products too small for the matrix cores, and operands of any strides (takes the product kernels' arguments, then `int lanes`).
std::string dot_small_source(const std::string& entry, const GemmEpilogue* epilogue = nullptr, bool grouped = false);

}  // namespace adhip
