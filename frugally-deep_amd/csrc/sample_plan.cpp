// Programs for small networks as one launch (sample_net.hip): which models and shapes have one, and when it is taken.
#include <algorithm>
#include <cstring>
#include <map>

#include "model.hpp"
#include "sample_net.hpp"

namespace fdx {

static bool g_fail_sample_memory = false; // test hooks
static int g_sample_loads = 0;

namespace {

    // a tensor in LDS: h x w pixels of c channels inside a frame of zeros
    struct Tensor {
        int h = 1, w = 1, c = 1;
        int top = 0, left = 0, bottom = 0, right = 0;
        bool compact = false; // read under another shape: one run of floats
        int row = 0, pix = 0, floats = 0, start = -1;
        int first = 0, last = 0; // steps between which it is held
        int base() const { return start + top * row + left * pix; }
    };

    bool hwc_of(const Shape& s, int* d)
    {
        if (s.empty() || s.size() > 3 || volume(s) >= (1 << 16)) // (quotients of positions below 2^16)
            return false;
        d[0] = s.size() > 2 ? (int)s[0] : 1;
        d[1] = s.size() > 1 ? (int)s[s.size() - 2] : 1;
        d[2] = (int)s.back();
        return true;
    }

    bool window_of(const Op& o, const Tensor& x, int* g)
    {
        return fdx_window_geometry(x.h + o.zp[0] + o.zp[1], x.w + o.zp[2] + o.zp[3], o.kind == OpKind::Conv2D ? (o.kh - 1) * o.dy + 1 : o.kh,
                   o.kind == OpKind::Conv2D ? (o.kw - 1) * o.dx + 1 : o.kw, o.sy, o.sx, o.padding, g)
            == FDX_OK;
    }

    bool epilogue_kind(const Act& a) { return a.kind == FDX_ACT_NONE || a.kind == FDX_ACT_RELU || a.kind == FDX_ACT_GELU; }

    // Cycles of a CU.  A convolution: the matrix pipes', or the chain of a wave's own items where there are few, longer where pixels are
    // read one float at a time, and an epilogue a tile.  These and the other steps' constants below, of 100 timed models with 300
    // convolutions, predict 100 others to 9 % rms (1 to 5 convolutions of 4 to 64 channels on maps of 6 to 40, or Dense layers).
    double conv_cycles(int pixels, int n_tiles, int chunks, bool vec)
    {
        const double tiles = (pixels + 15) / 16 * (double)n_tiles, chain = std::max(tiles * chunks * 32, std::ceil(tiles / 16) * chunks * 350);
        return (vec ? 1450 + 0.93 * chain : 1750 + 1.14 * chain) + 110 * tiles;
    }

} // namespace

// A model whose weights are small enough that a workgroup could hold them beside its tensors: they stay in host memory for the
// programs' images.  Everything else that a program needs is looked at when a plan is made.
bool sample_net_keeps_weights(const fdx_model& m)
{
    if (m.inputs.size() != 1 || m.outputs.size() != 1 || !m.host_layers.empty())
        return false;
    size_t floats = 0;
    for (const Op& o : m.ops) {
        if (o.dead)
            continue;
        switch (o.kind) {
        case OpKind::Input: case OpKind::View: case OpKind::Pool: case OpKind::GlobalPool: case OpKind::Softmax: case OpKind::Act: break;
        case OpKind::Conv2D: case OpKind::Dense:
            if (o.hw.size() < 2 || o.dual_cin > 0 || o.ln_src >= 0 || o.chain >= 0 || o.chained_from >= 0)
                return false;
            floats += o.hw[0].size() + o.hw[1].size();
            break;
        default: return false;
        }
    }
    return floats > 0 && floats <= (size_t)kSampleLdsFloats;
}

// The program for these shapes, in host memory, or none where an operation, a layout or the size of LDS speaks against it.
std::shared_ptr<SampleProgram> sample_net_build(const fdx_model& m, const std::vector<int>& order, const std::vector<Shape>& shapes)
{
    std::vector<Tensor> tensors;
    std::vector<int> of(m.ops.size(), -1);  // tensor that holds an op's result
    std::vector<Tensor> seen(m.ops.size()); // the shape under which its readers see it
    struct Pending {
        int op;
        bool behind; // the fused softmax or GELU of `op`, a step of its own
    };
    std::vector<Pending> run;
    int input_op = -1, tail = m.outputs[0];
    while (m.ops[(size_t)tail].kind == OpKind::View)
        tail = m.ops[(size_t)tail].in[0];
    // a result that something else reads as well would have to be kept twice
    for (int i = m.outputs[0];; i = m.ops[(size_t)i].in[0]) {
        if (m.ops[(size_t)i].consumers != 1)
            return nullptr;
        if (i == tail)
            break;
    }
    auto add_tensor = [&](const Tensor& like, int first) {
        Tensor t;
        t.h = like.h;
        t.w = like.w;
        t.c = like.c;
        t.first = t.last = first;
        tensors.push_back(t);
        return (int)tensors.size() - 1;
    };
    std::vector<int> in_front(m.ops.size(), -1); // tensor in front of an op's fused softmax or GELU
    std::vector<int> scratch_of(m.ops.size(), -1);
    for (int idx : order) {
        const Op& o = m.ops[(size_t)idx];
        if (o.dead)
            continue;
        int d[3];
        if (!hwc_of(shapes[(size_t)idx], d))
            return nullptr;
        Tensor me;
        me.h = d[0];
        me.w = d[1];
        me.c = d[2];
        seen[(size_t)idx] = me;
        if (o.kind == OpKind::View) {
            const int src = o.in[0];
            of[(size_t)idx] = of[(size_t)src];
            const Tensor& s = seen[(size_t)src];
            if (of[(size_t)src] >= 0 && (s.h != me.h || s.w != me.w || s.c != me.c))
                tensors[(size_t)of[(size_t)src]].compact = true;
            continue;
        }
        const int step = (int)run.size();
        run.push_back({ idx, false });
        const Tensor* x = nullptr;
        if (o.kind == OpKind::Input) {
            if (input_op >= 0 || volume(shapes[(size_t)idx]) > kSampleInput)
                return nullptr;
            input_op = idx;
        } else {
            if (o.in.size() != 1 || of[(size_t)o.in[0]] < 0)
                return nullptr;
            Tensor& held = tensors[(size_t)of[(size_t)o.in[0]]];
            held.last = step;
            x = &seen[(size_t)o.in[0]];
            if (o.kind == OpKind::Conv2D || o.kind == OpKind::Dense) {
                if (!epilogue_kind(o.act) || o.sample_w.empty() || o.sample_bias.empty())
                    return nullptr;
                if (o.residual >= 0) {
                    const Tensor& r = seen[(size_t)o.residual];
                    if (of[(size_t)o.residual] < 0 || r.h != me.h || r.w != me.w || r.c != me.c)
                        return nullptr;
                    tensors[(size_t)of[(size_t)o.residual]].last = step;
                }
            }
            int g[6];
            if (o.kind == OpKind::Conv2D) {
                if (o.n_in != x->c || o.cout != me.c || !window_of(o, *x, g) || g[4] != me.h || g[5] != me.w
                    || (int64_t)o.sample_w.size() != (int64_t)o.cout * o.kh * o.kw * o.n_in)
                    return nullptr;
                const int top = g[0] + o.zp[0], left = g[2] + o.zp[2];
                held.top = std::max(held.top, top);
                held.left = std::max(held.left, left);
                held.bottom = std::max(held.bottom, (g[4] - 1) * o.sy + (o.kh - 1) * o.dy + 1 - top - x->h);
                held.right = std::max(held.right, (g[5] - 1) * o.sx + (o.kw - 1) * o.dx + 1 - left - x->w);
            } else if (o.kind == OpKind::Dense) {
                if (o.n_in != x->c || o.units != me.c || (int64_t)o.sample_w.size() != (int64_t)o.units * o.n_in)
                    return nullptr;
            } else if (o.kind == OpKind::Pool) {
                if (o.zp[0] || o.zp[1] || o.zp[2] || o.zp[3] || !window_of(o, *x, g) || g[4] != me.h || g[5] != me.w)
                    return nullptr;
            } else if (o.kind == OpKind::Softmax) {
                if (o.log_after)
                    return nullptr;
            } else if (o.kind == OpKind::GlobalPool) {
                Tensor s;
                s.c = kSampleThreads;
                scratch_of[(size_t)idx] = add_tensor(s, step);
            } else if (o.kind != OpKind::Act)
                return nullptr;
        }
        if (o.softmax || (o.kind != OpKind::Act && o.act.kind == FDX_ACT_GELU)) {
            if ((o.kind != OpKind::Conv2D && o.kind != OpKind::Dense) || (o.softmax && o.act.kind != FDX_ACT_NONE))
                return nullptr;
            in_front[(size_t)idx] = add_tensor(me, step);
            tensors.back().last = step + 1;
            run.push_back({ idx, true });
        }
        if (idx != tail)
            of[(size_t)idx] = add_tensor(me, (int)run.size() - 1);
    }
    if (input_op < 0 || tail == input_op)
        return nullptr;

    // strides, then places: first fit among the tensors held at the same time
    for (Tensor& t : tensors) {
        if (t.compact) {
            if (t.top || t.left || t.bottom > 0 || t.right > 0)
                return nullptr;
            t.pix = t.c;
        } else
            t.pix = t.c % 4 == 0 ? ((t.c / 4) | 1) * 4 : t.c;
        t.bottom = std::max(t.bottom, 0);
        t.right = std::max(t.right, 0);
        t.row = (t.left + t.w + t.right) * t.pix;
        t.floats = ((t.top + t.h + t.bottom) * t.row + 3) / 4 * 4;
    }

    std::vector<float> image;
    auto words = [&](size_t n) {
        const size_t at = image.size();
        image.resize((at + n + 3) / 4 * 4, 0.f);
        return (int)at;
    };
    std::vector<SampleStep> steps;
    double cycles = 0;
    for (const Pending& r : run) {
        const Op& o = m.ops[(size_t)r.op];
        SampleStep s;
        std::memset(&s, 0, sizeof s);
        s.act_kind = FDX_ACT_NONE;
        s.act_max = 3.402823466e+38f;
        s.res_base = -1;
        const Tensor& me = seen[(size_t)r.op];
        if ((r.behind && o.softmax) || o.kind == OpKind::Softmax) {
            s.kind = SampleStep::Softmax;
            cycles += 900 + std::ceil(me.h * me.w / 16.0) * (1270 + me.c * 3.8);
        } else if (o.kind == OpKind::Input) {
            s.kind = SampleStep::Load;
            cycles += 1600 + volume(shapes[(size_t)r.op]) * 0.42;
        } else if (r.behind || o.kind == OpKind::Act) {
            s.kind = SampleStep::Activation;
            s.act_kind = o.act.kind;
            s.act_max = o.act.max_value;
            s.act_slope = o.act.negative_slope;
            s.act_threshold = o.act.threshold;
            cycles += 900 + (double)me.h * me.w * me.c * 0.64;
        } else if (o.kind == OpKind::Pool) {
            const Tensor& x = seen[(size_t)o.in[0]];
            int g[6];
            if (!window_of(o, x, g))
                return nullptr;
            s.kind = SampleStep::Pool;
            s.kh = o.kh;
            s.kw = o.kw;
            s.sy = o.sy;
            s.sx = o.sx;
            s.pad_top = g[0];
            s.pad_left = g[2];
            s.mode = o.pool_mode;
            cycles += 1900 + (double)me.h * me.w * me.c * o.kh * o.kw * 0.13;
        } else if (o.kind == OpKind::GlobalPool) {
            const Tensor& x = seen[(size_t)o.in[0]];
            s.kind = SampleStep::GlobalPool;
            s.mode = o.pool_mode;
            cycles += 2500 + (double)x.h * x.w * x.c * 0.19;
        } else { // convolution; a Dense layer is one of 1 x 1
            const bool conv = o.kind == OpKind::Conv2D;
            const Tensor& x = seen[(size_t)o.in[0]];
            const Tensor& held = tensors[(size_t)of[(size_t)o.in[0]]];
            // (where a shape of its own is read, the run of floats has the strides of that shape)
            const int pix = held.compact ? x.c : held.pix, row = held.compact ? x.w * x.c : held.row;
            const int kh = conv ? o.kh : 1, kw = conv ? o.kw : 1, cin = x.c, cout = me.c, k_all = kh * kw * cin;
            int g[6] = { 0, 0, 0, 0, 0, 0 };
            if (conv && !window_of(o, x, g))
                return nullptr;
            s.kind = SampleStep::Conv;
            s.kh = kh;
            s.kw = kw;
            s.sy = conv ? o.sy : 1;
            s.sx = conv ? o.sx : 1;
            s.pad_top = conv ? g[0] + o.zp[0] : 0;
            s.pad_left = conv ? g[2] + o.zp[2] : 0;
            s.chunks = (k_all + 15) / 16;
            s.whole = k_all / 16;
            s.vec = cin % 4 == 0 && pix % 4 == 0 && row % 4 == 0;
            s.n_tiles = (cout + 15) / 16;
            // the form whose busiest wave has the least to do; of equal ones the one with the longer items, which wait less often
            int least = 1 << 30;
            for (int f = 0; f < (int)(sizeof kSampleForms / sizeof kSampleForms[0]); ++f) {
                const SampleForm& q = kSampleForms[f];
                if (q.vec != (s.vec != 0) || s.n_tiles % q.nt != 0)
                    continue;
                const int items = (me.h * me.w + 16 * q.mt - 1) / (16 * q.mt) * (s.n_tiles / q.nt), waves = kSampleThreads / 64;
                const int tiles = (items + waves - 1) / waves * q.mt * q.nt;
                if (tiles <= least) {
                    least = tiles;
                    s.form = f;
                }
            }
            if (o.act.kind == FDX_ACT_RELU) {
                s.act_kind = o.act.kind;
                s.act_max = o.act.max_value;
                s.act_slope = o.act.negative_slope;
                s.act_threshold = o.act.threshold;
            }
            if (kh * kw == 1 && x.h * x.w == 1 && me.h * me.w == 1 && !s.pad_top && !s.pad_left) { // one pixel: weights as rows
                s.kind = SampleStep::Row;
                const int stride = (cin + 3) / 4 * 4;
                s.weights = words((size_t)cout * stride);
                for (int n = 0; n < cout; ++n)
                    std::memcpy(&image[(size_t)s.weights + (size_t)n * stride], &o.sample_w[(size_t)n * cin], (size_t)cin * 4);
            } else {
                const int dy = conv ? o.dy : 1, dx = conv ? o.dx : 1;
                auto offset = [&](int k) {
                    const int tap = k / cin, fy = tap / kw, fx = tap - fy * kw;
                    return k < k_all ? fy * dy * row + fx * dx * pix + (k - tap * cin) : -1;
                };
                // a lane group's offsets side by side, a chunk's four groups one after the other
                const int per = s.vec ? 4 : 1;
                s.tab_stride = s.vec ? (s.chunks + 3) / 4 * 4 : s.chunks * 4;
                s.tab = words((size_t)s.tab_stride * 4);
                for (int kc = 0; kc < s.chunks; ++kc)
                    for (int fg = 0; fg < 4; ++fg)
                        for (int e = 0; e < 4; e += per) {
                            const int v = offset(kc * 16 + fg * 4 + e);
                            std::memcpy(&image[(size_t)(s.tab + fg * s.tab_stride + (s.vec ? kc : kc * 4 + e))], &v, 4);
                        }
                s.weights = words((size_t)s.n_tiles * s.chunks * 256);
                for (int nt = 0; nt < s.n_tiles; ++nt)
                    for (int kc = 0; kc < s.chunks; ++kc)
                        for (int lane = 0; lane < 64; ++lane)
                            for (int e = 0; e < 4; ++e) {
                                const int n = nt * 16 + (lane & 15), k = kc * 16 + (lane >> 4) * 4 + e;
                                if (n < cout && k < k_all)
                                    image[(size_t)s.weights + ((size_t)(nt * s.chunks + kc) * 64 + lane) * 4 + e] = o.sample_w[(size_t)n * k_all + k];
                            }
            }
            s.bias = words((size_t)s.n_tiles * 16);
            for (int n = 0; n < cout && n < (int)o.sample_bias.size(); ++n)
                image[(size_t)(s.bias + n)] = o.sample_bias[(size_t)n];
            cycles += s.kind == SampleStep::Row ? 1400 + std::ceil(cout / 128.0) * (210 + cin * 2.8) : conv_cycles(me.h * me.w, s.n_tiles, s.chunks, s.vec);
        }
        if (image.size() > (size_t)kSampleLdsFloats)
            return nullptr;
        steps.push_back(s);
    }

    const int image_floats = (int)image.size();
    int lds = image_floats;
    for (size_t i = 0; i < tensors.size(); ++i) {
        Tensor& t = tensors[i];
        int at = image_floats;
        for (bool moved = true; moved;) {
            moved = false;
            for (size_t k = 0; k < i; ++k) {
                const Tensor& u = tensors[k];
                if (u.first <= t.last && t.first <= u.last && at < u.start + u.floats && u.start < at + t.floats) {
                    at = u.start + u.floats;
                    moved = true;
                }
            }
        }
        t.start = at;
        lds = std::max(lds, at + t.floats);
    }
    if (lds > kSampleLdsFloats)
        return nullptr;

    const int p_in_volume = (int)volume(shapes[(size_t)input_op]);
    for (size_t i = 0; i < steps.size(); ++i) {
        SampleStep& s = steps[i];
        const int idx = run[i].op;
        const Op& o = m.ops[(size_t)idx];
        const Tensor& me = seen[(size_t)idx];
        // where a step reads (under which shape) and writes
        const bool ahead = !run[i].behind && in_front[(size_t)idx] >= 0; // its activation comes behind it
        const int to = ahead ? in_front[(size_t)idx] : of[(size_t)idx];
        s.out_h = me.h;
        s.out_w = me.w;
        s.out_c = me.c;
        s.out_base = -1;
        if (to >= 0) {
            const Tensor& t = tensors[(size_t)to];
            s.out_base = t.base();
            s.out_row = t.row;
            s.out_pix = t.pix;
            if (t.top || t.left || t.bottom || t.right) {
                s.frame_base = t.start;
                s.frame_h = t.top + t.h + t.bottom;
                s.frame_w = t.left + t.w + t.right;
                s.frame_top = t.top;
                s.frame_left = t.left;
            }
        }
        auto by = [](int d) { return d > 1 ? (uint32_t)((0x100000000ull + (uint64_t)d - 1) / (uint64_t)d) : 0u; };
        s.by_out_w = by(s.out_w);
        s.by_out_c = by(s.out_c);
        s.by_frame_w = by(s.frame_w);
        if (s.kind == SampleStep::Load) {
            s.vec = (s.out_c | s.out_base | s.out_row | s.out_pix | p_in_volume) % 4 == 0;
            continue;
        }
        const int from = run[i].behind ? in_front[(size_t)idx] : of[(size_t)o.in[0]];
        const Tensor& held = tensors[(size_t)from];
        const Tensor& x = run[i].behind ? me : seen[(size_t)o.in[0]];
        s.in_h = x.h;
        s.in_w = x.w;
        s.in_c = x.c;
        s.in_row = held.compact ? x.w * x.c : held.row;
        s.in_pix = held.compact ? x.c : held.pix;
        s.in_base = held.base();
        s.by_in_w = by(s.in_w);
        if (s.kind == SampleStep::Pool) {
            s.vec = s.out_base >= 0 && (s.in_c | s.in_base | s.in_row | s.in_pix | s.out_base | s.out_row | s.out_pix) % 4 == 0;
            s.by_out_c = by(s.vec ? s.out_c / 4 : s.out_c);
            s.whole = s.kh == 2 && s.kw == 2 && !s.pad_top && !s.pad_left && (s.out_h - 1) * s.sy + 2 <= s.in_h && (s.out_w - 1) * s.sx + 2 <= s.in_w;
        }
        if (s.kind == SampleStep::Row)
            s.vec = (s.in_c | s.in_base) % 4 == 0;
        if (s.kind == SampleStep::Conv || s.kind == SampleStep::Row) {
            s.in_base -= s.pad_top * s.in_row + s.pad_left * s.in_pix;
            if (o.residual >= 0) {
                const Tensor& r = tensors[(size_t)of[(size_t)o.residual]];
                const Tensor& rs = seen[(size_t)o.residual];
                s.res_base = r.base();
                s.res_row = r.compact ? rs.w * rs.c : r.row;
                s.res_pix = r.compact ? rs.c : r.pix;
            }
        }
        if (s.kind == SampleStep::GlobalPool) {
            s.scratch = tensors[(size_t)scratch_of[(size_t)idx]].start;
            s.vec = (s.in_c | s.in_base | s.in_pix) % 4 == 0 && s.in_row == s.in_w * s.in_pix;
        }
    }

    auto p = std::make_shared<SampleProgram>();
    p->image_floats = image_floats;
    p->lds_floats = lds;
    p->steps = (int)steps.size();
    p->in_volume = p_in_volume;
    p->out_volume = (int)volume(shapes[(size_t)m.outputs[0]]);
    p->us_per_sample = (cycles + 0.68 * p->out_volume) / 2400.0; // (a result's way out)
    const size_t step_floats = steps.size() * sizeof(SampleStep) / 4;
    p->step_at = (image.size() + 15) / 16 * 16;
    image.resize(p->step_at + step_floats);
    std::memcpy(&image[p->step_at], steps.data(), step_floats * 4);
    p->host = std::move(image);
    return p;
}

// The program into device memory, at the first plan that runs it; false where the memory is refused.
bool sample_net_load(SampleProgram& p)
{
    if (p.image)
        return true;
    ++g_sample_loads;
    float* d = nullptr;
    const size_t bytes = p.host.size() * sizeof(float);
    // (the model then runs as launches, whose checks must not find this call's error)
    if (hipMalloc(reinterpret_cast<void**>(&d), g_fail_sample_memory ? (size_t)1 << 60 : bytes) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    if (hipMemcpyAsync(d, p.host.data(), bytes, hipMemcpyHostToDevice, stream()) != hipSuccess || hipStreamSynchronize(stream()) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipFree(d);
        return false;
    }
    p.image = d;
    p.program = reinterpret_cast<const SampleStep*>(d + p.step_at);
    p.host = std::vector<float>();
    return true;
}

// One launch or one per operation, by predicted times: a convolution or Dense layer's own launch as layer_cost has it, any other by its traffic,
// 3.7 us at least.  Over 1200 timed calls (200 models of 1 to 5 convolutions of 4 to 64 channels or 1 to 4 Dense layers, 1 to 8192 samples) the
// choice takes 0.4 % longer than the faster form, at worst 32 %; with one rate for all convolutions it took 10 %, and 2.1 times as
// long where 8192 samples of two convolutions to 24 and 64 channels went into one launch.  Measured, us of a call, launches / one: the small
// CNN (two 3x3 convolutions of 16 and 32 channels on 32 x 32 x 3) at batch 1 / 256 / 8192 24 / 17.0, 59 / 17.8, 903 / 485; 28 x 28 with 5x5
// convolutions of 6 and 16 channels and two Dense layers 44 / 15.3, 62 / 16.1, 717 / 411; four 3x3 convolutions of 16 channels on 16 x 16 25 /
// 20.6, 65 / 21.5, 1059 / 597; strided 3x3 of 32 and 64 channels on 32 x 32 x 3 22 / 15.6, 34 / 16.6, 335 / 427 (the last left to the
// launches); three Dense layers, 64 -> 128 -> 128 -> 4, at batch 1 / 256 / 2048 13.2 / 6.7, 13.6 / 7.0, 13.5 / 28 (left); one 3x3 convolution 8 -> 32 on
// 24 x 24 at batch 1 / 256 / 8192 8.1 / 13.0, 19.3 / 16.4, 385 / 396 (all left, the second wrongly).
bool sample_net_by_rule(const SampleProgram& p, const fdx_model& m, const std::vector<int>& order, const std::vector<Shape>& shapes, int batch)
{
    double launches = 0;
    for (int idx : order) {
        const Op& o = m.ops[(size_t)idx];
        if (o.dead || o.kind == OpKind::Input || o.kind == OpKind::View)
            continue;
        const Shape &is = shapes[(size_t)o.in[0]], &os = shapes[(size_t)idx];
        const double in = (double)batch * volume(is), out = (double)batch * volume(os);
        double us = std::max(3.7, (in + out) * 4 / 3e6);
        if (o.kind == OpKind::Conv2D || o.kind == OpKind::Dense) {
            const int n = (int)os.back();
            const int64_t rows = (int64_t)batch * (volume(os) / n), a_floats = (int64_t)in;
            int d[3], e[3];
            (void)hwc_of(is, d);
            (void)hwc_of(os, e);
            const bool same = o.kind == OpKind::Conv2D && o.sy == 1 && o.sx == 1 && d[0] == e[0] && d[1] == e[1];
            const bool pointwise = o.kind == OpKind::Dense || (same && o.kh == 1 && o.kw == 1);
            const int taps = o.kind == OpKind::Dense ? 1 : o.kh * o.kw;
            us = layer_cost(!pointwise, rows, o.n_in, taps, n, a_floats, o.residual >= 0, same && taps >= 6 && o.n_in % 32 == 0 && d[1] <= 63);
            if (same && o.kh == 3 && o.kw == 3 && fdx_conv2d_winograd_supported(o.n_in, n))
                us = std::min(us, (double)conv2d_winograd_cost(batch, o.n_in, n, e[0], e[1]));
        }
        launches += us + (o.softmax ? 3.0 : 0.0);
    }
    return 3.0 + std::ceil((double)batch / sample_net_cus()) * p.us_per_sample < launches;
}

} // namespace fdx

extern "C" fdx_status fdx_debug_fail_sample_memory(int on)
{
    fdx::g_fail_sample_memory = on != 0;
    return FDX_OK;
}
extern "C" int fdx_debug_sample_loads(void) { return fdx::g_sample_loads; }
