// The gather convolution of conv_group.hip, shared with the dispatch in conv.hip.
#pragma once

#include "common.h"

namespace hi3d {

struct GroupConv {
  const char* in;
  int64_t n_in;
  int32_t cin;
  const char* weight;   // 16-bit: [cout][kvol][cin]
  const char* packed;   // fp32: [kvol][cin / 16][col_blocks][3 parts][64 lanes][16 bytes]
  int32_t col_blocks;   // 32-channel blocks of the packed weights (the last may be padding)
  const char* bias;
  int32_t cout;
  int32_t kvol;
  const int32_t* rows;
  const int32_t* gidx;
  int64_t n_out;
  int32_t ny;           // column tiles
  const char* residual;
  int32_t act;
  char* out;
  // the row norm of conv_wide_kernel<.., kLN> (fp16, cout 128); null: none
  const int32_t* ln_coords;
  const void* ln_scale;
  const void* ln_shift;
  int32_t ln_batches;
  float ln_eps;
};

// Whether a 16-bit convolution is one of few tiles that group_conv16 takes.
bool group_conv16_takes(int64_t n_out, int cin, int cout, int kvol);
int group_conv16(const GroupConv& c, bool bf16, hipStream_t stream);

}  // namespace hi3d
