// Source generator for the fused attention kernel (see attention.cpp).
#pragma once
#include <cstddef>
#include <cstdint>
#include <string>

namespace adhip {

struct AttentionConfig {
    int d = 128;   // features of a query / key row (multiple of 4, at most 256)
    int dv = 128;  // features of a value / result row (multiple of 16, at most 256)
    int bn = 64;   // keys per tile (64 or 32)
    int wg = 2;    // key groups: 1 (a block is 4 wavefronts) or 2 (8 wavefronts, each group takes half of every tile)
    bool parts = false; // on the bf16 matrix cores, every operand split into three bf16 parts (the FP32 ones where that does not come out finite)
    bool mask = false;  // the scaled scores are multiplied by a [Sq, Sk] mask before the softmax
};

// bytes of LDS a block of this configuration needs (two stages of K and V tiles and a patch per wavefront)
size_t attention_lds_bytes(const AttentionConfig& cfg);

// Widths of heads that the kernel on the bf16 matrix cores takes: query rows in chunks of 32 features, results in registers.
inline bool attention_takes_parts(int d, int dv) { return d % 32 == 0 && d <= 128 && (dv == 32 || dv == 64 || dv == 128); }

// Problem slots of one launch (the heads of multi-head attention; a block's number picks problem and row block); a launch may use
// fewer and fills the rest with any valid pointers.
constexpr int kAttentionSlots = 16;

// With `parts`: floats of a problem's keys and values in parts, and the kernel that writes them before the attention kernel
// runs (arguments k0, v0, k1 ... , parts, Sk, k_ld, v_ld; a block per tile of 32 keys and problem).
int64_t attention_parts_floats(const AttentionConfig& cfg, int64_t sk);
std::string attention_split_source(const AttentionConfig& cfg, const std::string& entry);

std::string attention_kernel_source(const AttentionConfig& cfg, const std::string& entry);

}  // namespace adhip
