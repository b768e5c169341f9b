// gsvk_conv_group.hpp — several same-shape convolutions in one launch (internal to the library).
#ifndef GSVK_CONV_GROUP_HPP
#define GSVK_CONV_GROUP_HPP

#include <cstddef>
#include <cstdint>

namespace gsvk {

constexpr int kConvGroupMax = 3;

// One convolution of a group: gsvk_conv1d's operands of that name (rows of stride ld).
struct ConvItem {
  const void* x;
  const uint16_t* w_packed;
  const float* bias;
  void* cur;
  const void* res;
  void* y;
  size_t k, dilation;
};

// Whether running a decoder stage's three convolutions as one launch beats three concurrent
// branches: up to 200 tiles of 64 columns x 32 rows each, i.e. while the three fit the chip in about
// one round. Measured on the whole decoder (fp16 storage / exact fp32): 20 frames 434 -> 368 and
// 495 -> 459 us; every stage grouped at 150 frames 834 -> 935 and 1086 -> 1194, since a branch runs
// into the next convolution while another's last workgroups drain and a group cannot.
bool conv1d_group_pays(size_t C, size_t T);

// n (1 .. kConvGroupMax) convolutions C -> C over T columns, each as gsvk_conv1d(dtype, round_x, x,
// ld, w_packed, bias, epi, slope, cur, res, ld, y, ld, C, C, T, k, dilation, stream), in one launch
// where the kernel for few tiles can run them all, otherwise one after another.
// No convolution may read what another of the group writes. List the longest (largest k) first: its
// workgroups start first.
int conv1d_group(int dtype, int round_x, const ConvItem* items, int n, int epi, float slope,
                 size_t ld, size_t C, size_t T, void* stream);

// n ResBlock pairs, c2[j].cur = c2[j].res + conv2(lrelu(conv1(lrelu(c1[j].x)))) (c1.y, c1.cur, c2.x,
// c2.y not used), in one launch, for shapes conv1d_pair_fits takes (both convolutions of a pair of one
// k, the second of dilation 1; rows of stride T at most 2^31 bytes in all). c2.cur must not overlap
// c1.x or c2.res: other workgroups still read their columns. List the longest first.
bool conv1d_pair_fits(size_t C, size_t T, size_t k, size_t dilation, size_t esz);
int conv1d_pairs(int dtype, int round_x, const ConvItem* c1, const ConvItem* c2, int n, float slope,
                 size_t ld, size_t C, size_t T, void* stream);

}  // namespace gsvk

#endif
