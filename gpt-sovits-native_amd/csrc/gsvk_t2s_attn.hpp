// gsvk_t2s_attn.hpp — a T2S decode layer's QKV projection and attention in one launch (internal).
#ifndef GSVK_T2S_ATTN_HPP
#define GSVK_T2S_ATTN_HPP

#include <cstddef>
#include <cstdint>

namespace gsvk {

// fp16 activations and caches, head width 32.
struct T2sAttnArgs {
  const void* z;         // [B, D]: x (no LayerNorm) or the rows to normalise
  const float* ln_g;     // [D] or nullptr (ones)
  const float* ln_b;     // [D] or nullptr (zeros)
  void* x;               // [B, D]: LN(z), stored; unused without LayerNorm
  const uint16_t* wqkv;  // [3D, D]
  const float* bqkv;     // [3D] or nullptr
  void* kc;              // [B, max_len, D]
  void* vc;
  const int64_t* pos;    // [B]
  void* out;             // [B, D]
  int32_t* err;          // or nullptr
  long max_len;
  int heads;
  float eps, scale;
  double inv_n;          // 1 / D
};

// Whether the launch can take these operands (shapes, alignment, nothing overlapping); x is nullptr
// without LayerNorm.
bool t2s_qkv_attention_ok(const T2sAttnArgs& a, size_t batch, size_t D);
int t2s_qkv_attention(const T2sAttnArgs& a, size_t batch, size_t D, bool ln, void* stream);

}  // namespace gsvk

#endif
