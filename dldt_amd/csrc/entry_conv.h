// A FakeQuantize on a graph input and the convolution behind it, whose f32 values are the graph's result, as one launch
// (entry_conv.hip).
#pragma once
#include <memory>

#include "common.h"

struct hipie_fq;
struct hipie_conv;

namespace hipie {

// the convolution's weights in the kernel's order, and its shape for these tensors
struct EntryConv;
// null: the kernel does not take the layers.  `mid`: the tensor of levels between them (its data is not touched), `fill`: the stored
// byte of its padding
std::shared_ptr<EntryConv> make_entry_conv(int device, const hipie_fq* fq, bool u8_in, const hipie_conv* conv, const hipie_tensor& mid, const hipie_tensor& out, int fill);
// in: dense [N, C, H, W], f32 or u8 as made; the levels into `mid`, the values into `planes`, dense [N, OC, H, W], which has no byte
// in common with `in`: values are stored while other workgroups still have input to read.  With `out` the values go into that tensor
// as well
void run_entry_conv(const EntryConv& e, const void* in, const hipie_tensor& mid, const hipie_tensor* out, void* planes, hipStream_t s);

}  // namespace hipie
