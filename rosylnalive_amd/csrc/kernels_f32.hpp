// The float32 contractions of the reference catalog on the f32 matrix cores (kernels_f32.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace lrm {
namespace f32k {

// y[i][m, n[i]] = x[m, k] . w[i][n[i], k]^T (bf16 w) for i < count, every output one ascending fused chain over k.
struct MatmulGroup {
    const uint16_t* w[3];
    float* y[3];
    uint32_t n[3];
    uint32_t count;
};
void matmul_bf16w(const float* x, const MatmulGroup& group, uint32_t m, uint32_t k, hipStream_t s);

// attention_gqa_causal on the matrix cores; false (nothing launched) where the general kernel takes the call: a shape or an
// alignment that is not covered, or too few keys to be worth it. A
// decode row spreads over the chip when `workspace` (kWorkspaceBytes, written by each call, its contents not kept; null:
// none) holds its blocks: of the 0.6B's 16 heads, up to 21,500 keys.
constexpr uint64_t kWorkspaceBytes = uint64_t(4) << 20;
bool attention(const float* q, const float* kc, const float* vc, float* y, uint32_t rows, uint32_t q_row0, uint32_t past,
               uint32_t qh, uint32_t kvh, uint32_t hd, float scale, void* workspace, hipStream_t s);

}  // namespace f32k
}  // namespace lrm
