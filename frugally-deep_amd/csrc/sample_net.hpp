// A small network as one launch: a workgroup takes a sample from the first layer to the last (sample_net.hip, sample_plan.cpp).
#pragma once
#include <cstdint>
#include <memory>
#include <vector>

namespace fdx {

// One step of the program that a workgroup runs (read through the scalar cache, three lines each).  Positions (base, tab, weights, bias, ...) count floats
// from the start of LDS; tensors are rows of pixels of channels with strides of their own.
struct alignas(64) SampleStep {
    enum Kind { Load, Conv, Row, Pool, GlobalPool, Softmax, Activation };
    int kind;
    int out_base, out_row, out_pix, out_h, out_w, out_c; // out_base < 0: the sample's row of the result
    int frame_base, frame_h, frame_w, frame_top, frame_left; // output with its frame of zeros, frame_h = 0: none
    int in_base, in_row, in_pix, in_h, in_w, in_c; // Conv: base of tap (0, 0) of output pixel (0, 0), inside the frame
    int kh, kw, sy, sx, pad_top, pad_left, mode;   // Pool: window; mode as in fdx_pool2d_nhwc_f32
    int form, tab, tab_stride, chunks, whole, vec, weights, bias, n_tiles; // Conv: offsets of its K elements (vec: of fours) from tap (0, 0);
                                                    // chunks of 16 K, the first `whole` of them without padding
    int res_base, res_row, res_pix;                // Conv: residual operand, res_base < 0: none
    int scratch;                                   // GlobalPool: 1024 floats
    uint32_t by_out_w, by_out_c, by_in_w, by_frame_w; // ceil(2^32 / x): quotients of values below 2^16
    int act_kind;
    float act_max, act_slope, act_threshold;
};
static_assert(sizeof(SampleStep) == 192, "three lines");
// forms of a convolution: tiles of 16 pixels and of 16 channels that a wave takes at once, by SampleStep::form
struct SampleForm {
    bool vec;
    int mt, nt;
};
constexpr SampleForm kSampleForms[] = { { false, 1, 1 }, { false, 4, 1 }, { true, 1, 1 }, { true, 4, 1 }, { true, 1, 2 }, { true, 2, 2 } };
constexpr int kSampleLdsFloats = 40960; // a CU's LDS
constexpr int kSampleThreads = 1024, kSampleInput = kSampleThreads * 16; // most floats of an input

// A program for one input shape: offset tables and weights as they lie in LDS, then the steps; in host memory until a plan runs it.
struct SampleProgram {
    std::vector<float> host;
    size_t step_at = 0; // floats in front of the steps
    float* image = nullptr;
    const SampleStep* program = nullptr;
    int image_floats = 0, lds_floats = 0, steps = 0, in_volume = 0, out_volume = 0;
    double us_per_sample = 0, flops = 0; // predicted: one sample on a CU
    ~SampleProgram();
};

} // namespace fdx
