// Host side of the Python package: argument checks, output and workspace allocation, and the calls into
// libprime_moe_hip.so.  Registers the CUDA-key implementations of the prime_moe:: ops (their schemas are defined in
// prime_moe/__init__.py) and exposes what is not an op (route, quantize_mx, the checks) as Python functions.
//
// Replaces the stubs of the reference's prime_moe/csrc/torch_interface.cpp:82-268; the conditions are those of its
// TORCH_CHECKs (:85-87, :132-155, :208-241) and the ones the kernels need on top.  No device code.
//
// In C++ because the calls a decode step makes are short: checks, allocations and ctypes in Python cost 25 - 30 us a
// call, which the device spends less than on a single token.
#include <limits>

#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "../../include/prime_moe_hip.h"

namespace {

using at::Tensor;

#define REQUIRE(cond, ...)                                            \
    do {                                                              \
        if (C10_UNLIKELY(!(cond))) fail(c10::str(__VA_ARGS__));       \
    } while (0)

[[noreturn]] void fail(const std::string &msg) { throw std::runtime_error(msg); }

void check_status(int rc) {
    if (C10_UNLIKELY(rc != PMOE_OK)) {
        const char *msg = pmoe_last_error();
        fail(msg != nullptr && *msg ? msg : c10::str("prime_moe native error ", rc));
    }
}

void *stream_of(const c10::Device &dev) {
    return c10::hip::getCurrentHIPStream(dev.index()).stream();
}

Tensor empty(at::IntArrayRef size, at::ScalarType dtype, const c10::Device &dev) {
    return at::empty(size, at::TensorOptions().dtype(dtype).device(dev));
}
// Scratch of one call, from torch's caching allocator: stream ordered, no hipMalloc in steady state, capturable.
Tensor workspace(size_t bytes, const c10::Device &dev) {
    return empty({(int64_t)std::max<size_t>(bytes, 256)}, at::kByte, dev);
}

struct Arg {
    const char *name;
    const Tensor *t;
};

// Every tensor must live on the GPU of the first one: the kernels take raw device pointers, so a CPU tensor (or one on
// another GPU) would be a memory fault on the device, not an exception.
void require_same_device(const char *op, std::initializer_list<Arg> args) {
    const Arg &anchor = *args.begin();
    const c10::Device dev = anchor.t->device();
    REQUIRE(dev.is_cuda(), op, ": ", anchor.name, " must be a GPU tensor, got device ", dev);
    for (const Arg &a : args)
        REQUIRE(a.t->device() == dev, op, ": ", a.name, " is on ", a.t->device(), ", expected ", dev, " (the device of ",
                anchor.name, ")");
}
// The kernels read these with `align`-byte vector loads from the start of the tensor.
void require_aligned(const char *op, std::initializer_list<Arg> args, uintptr_t align) {
    for (const Arg &a : args)
        REQUIRE(reinterpret_cast<uintptr_t>(a.t->const_data_ptr()) % align == 0, op, ": ", a.name, " must start at a ", align,
                "-byte aligned address");
}
void require_contiguous(const char *op, std::initializer_list<Arg> args) {
    for (const Arg &a : args) REQUIRE(a.t->is_contiguous(), op, ": ", a.name, " must be contiguous");
}
void require_dtype(const char *op, std::initializer_list<Arg> args, at::ScalarType dtype, const char *dtype_name) {
    for (const Arg &a : args) REQUIRE(a.t->scalar_type() == dtype, op, ": ", a.name, " must be ", dtype_name);
}

void check_tuning(const char *what, int64_t block_m, int64_t block_n, int64_t warp_n, int64_t stages, int64_t max_stages) {
    REQUIRE((block_n == 64 && warp_n == 4) || (block_n == 32 && warp_n == 8), what,
            ": (block_n, warp_n) must be (64, 4) or (32, 8), got (", block_n, ", ", warp_n, ")");
    REQUIRE(stages > 0 && stages <= max_stages, what, " supports stages in 1..", max_stages, ", got ", stages);
    REQUIRE(block_m == 128, what, " requires block_m=128, got ", block_m);
}

// ------------------------------------------------------------------------------- moe_align

// (pad_to, max_padded, max_blocks) as torch_interface.cpp:88-91 computes them.  Ids, positions and sizes are int32 in the
// kernels and the C ABI: what does not fit is an error here (block_m, bpc > 0, num_experts <= 1024: no step overflows).
struct AlignSizes {
    int64_t pad_to, max_padded, max_blocks;
    AlignSizes(int64_t n, int64_t num_experts, int64_t block_m, int64_t bpc) {
        constexpr int64_t kMax = std::numeric_limits<int32_t>::max();
        REQUIRE(n <= kMax, "moe_align: ", n, " ids do not fit 32 bits");
        REQUIRE(block_m <= kMax && bpc <= kMax / block_m, "moe_align: block_m * bpc does not fit 32 bits (", block_m, " * ", bpc, ")");
        pad_to = block_m * bpc;
        max_padded = (n + num_experts * (pad_to - 1) + pad_to - 1) / pad_to * pad_to;
        REQUIRE(max_padded <= kMax, "moe_align: a schedule of ", max_padded, " rows does not fit 32 bits");
        max_blocks = max_padded / block_m;
    }
};

// `placement`: false leaves out the device check (what is left can then be exercised with CPU tensors).
void validate_align(const Tensor &topk_ids, int64_t num_experts, int64_t block_m, int64_t bpc, bool placement) {
    REQUIRE(topk_ids.is_cuda() || !placement, "moe_align: topk_ids must be a GPU tensor, got device ", topk_ids.device());
    REQUIRE(topk_ids.is_contiguous(), "moe_align: topk_ids must be contiguous");
    REQUIRE(topk_ids.scalar_type() == at::kInt, "moe_align: topk_ids must be int32");
    REQUIRE(block_m > 0 && bpc > 0 && num_experts > 0, "moe_align: block_m, bpc and num_experts must be positive");
    REQUIRE(num_experts <= 1024, "moe_align supports at most 1024 experts, got ", num_experts);
    AlignSizes(topk_ids.numel(), num_experts, block_m, bpc);
}

struct Schedule {
    Tensor sorted_token_ids, expert_ids, num_tokens_post_padded, ws;
    size_t ws_bytes;
    Schedule(const AlignSizes &sz, int64_t n, int64_t num_experts, const c10::Device &dev)
        : sorted_token_ids(empty({sz.max_padded}, at::kInt, dev)),
          expert_ids(empty({sz.max_blocks}, at::kInt, dev)),
          num_tokens_post_padded(empty({1}, at::kInt, dev)) {
        // many ids: scratch for the multi-workgroup sort (0 bytes when one workgroup does it)
        ws_bytes = pmoe_moe_align_workspace_bytes_fast((int)n, (int)num_experts);
        if (ws_bytes > 0) ws = workspace(ws_bytes, dev);
    }
    void *ws_ptr() const { return ws_bytes > 0 ? ws.data_ptr() : nullptr; }
};

std::tuple<Tensor, Tensor, Tensor> moe_align(const Tensor &topk_ids, int64_t num_experts, int64_t block_m, int64_t bpc) {
    validate_align(topk_ids, num_experts, block_m, bpc, true);
    const c10::Device dev = topk_ids.device();
    const c10::DeviceGuard guard(dev);
    const int64_t n = topk_ids.numel();
    const AlignSizes sz(n, num_experts, block_m, bpc);
    Schedule s(sz, n, num_experts, dev);
    check_status(pmoe_moe_align_ws(topk_ids.const_data_ptr<int32_t>(), s.sorted_token_ids.data_ptr<int32_t>(),
                                   s.expert_ids.data_ptr<int32_t>(), s.num_tokens_post_padded.data_ptr<int32_t>(), (int)n,
                                   (int)num_experts, (int)block_m, (int)sz.pad_to, (int)sz.max_padded, (int)sz.max_blocks,
                                   s.ws_ptr(), s.ws_bytes, stream_of(dev)));
    return {s.sorted_token_ids, s.expert_ids, s.num_tokens_post_padded};
}

// ------------------------------------------------------------------------------- fused_moe_bf16

void validate_bf16(const Tensor &x, const Tensor &w, const Tensor &w2, const Tensor &sorted_token_ids, const Tensor &expert_ids,
                   const Tensor &num_tokens_post_padded, const Tensor &topk_weights, const Tensor &out, int64_t top_k,
                   int64_t block_m, int64_t block_n, int64_t warp_n, int64_t stages, int64_t bpc, int64_t cpc, bool split,
                   bool placement) {
    const char *op = "fused_moe_bf16";
    REQUIRE(x.dim() == 2 && w.dim() == 3 && w2.dim() == 3, op, ": x must be 2-D, w and w2 3-D");
    REQUIRE(x.size(0) > 0, op, ": x has no rows");
    REQUIRE(x.size(1) == w.size(2), op, ": x.size(1) must equal w.size(2)");
    REQUIRE(x.size(1) % 128 == 0, "K dimension must be a multiple of 128");
    REQUIRE(w.size(1) % 256 == 0, op, ": N must be a multiple of 256, got ", w.size(1));
    REQUIRE(w2.size(0) == w.size(0) && w2.size(1) == x.size(1) && w2.size(2) == w.size(1) / 2, op,
            ": w2 must have shape (E, K, N/2)");
    check_tuning(op, block_m, block_n, warp_n, stages, 5);
    REQUIRE(bpc == 1 && cpc == 1, "bpc=cpc=1 is the only supported configuration");
    REQUIRE(!split || stages <= 4, "split=True requires stages<=4, got stages=", stages);
    REQUIRE(top_k > 0, op, ": top_k must be positive");
    const Arg ax{"x", &x}, aw{"w", &w}, aw2{"w2", &w2}, as{"sorted_token_ids", &sorted_token_ids}, ae{"expert_ids", &expert_ids},
        an{"num_tokens_post_padded", &num_tokens_post_padded}, at_{"topk_weights", &topk_weights}, ao{"out", &out};
    if (placement) {
        require_same_device(op, {ax, aw, aw2, as, ae, an, at_, ao});
        require_aligned(op, {ax, aw, aw2, ao}, 16);
        require_aligned(op, {as, ae, an, at_}, 4);
    }
    require_contiguous(op, {ax, aw, aw2, as, ae, an, at_, ao});
    require_dtype(op, {ax, aw, aw2, ao}, at::kBFloat16, "bfloat16");
    require_dtype(op, {at_}, at::kFloat, "float32");
    require_dtype(op, {as, ae, an}, at::kInt, "int32");
    REQUIRE(out.sizes() == x.sizes(), op, ": out must have the shape of x");
    REQUIRE(num_tokens_post_padded.numel() >= 1, op, ": num_tokens_post_padded is empty");
    REQUIRE(expert_ids.numel() * block_m >= sorted_token_ids.numel(), op,
            ": expert_ids is shorter than sorted_token_ids / block_m");
}

void fused_moe_bf16(const Tensor &x, const Tensor &w, const Tensor &w2, const Tensor &sorted_token_ids, const Tensor &expert_ids,
                    const Tensor &num_tokens_post_padded, const Tensor &topk_weights, Tensor &out, int64_t top_k, int64_t block_m,
                    int64_t block_n, int64_t warp_n, int64_t stages, int64_t bpc, int64_t cpc, bool split) {
    validate_bf16(x, w, w2, sorted_token_ids, expert_ids, num_tokens_post_padded, topk_weights, out, top_k, block_m, block_n,
                  warp_n, stages, bpc, cpc, split, true);
    const c10::Device dev = x.device();
    const c10::DeviceGuard guard(dev);
    const int M = (int)x.size(0), K = (int)x.size(1), E = (int)w.size(0), N = (int)w.size(1), S = (int)sorted_token_ids.size(0);
    const Tensor ws = workspace(pmoe_fused_moe_bf16_workspace_bytes(M, K, N, E, S, (int)top_k, split), dev);
    check_status(pmoe_fused_moe_bf16(
        x.const_data_ptr(), w.const_data_ptr(), w2.const_data_ptr(), out.data_ptr(), sorted_token_ids.const_data_ptr<int32_t>(),
        expert_ids.const_data_ptr<int32_t>(), num_tokens_post_padded.const_data_ptr<int32_t>(),
        topk_weights.const_data_ptr<float>(), (int)top_k, M, K, N, E, S, (int)block_m, (int)block_n, (int)warp_n, (int)stages,
        (int)bpc, (int)cpc, split, ws.data_ptr(), (size_t)ws.numel(), stream_of(dev)));
}

// ------------------------------------------------------------------------------- fused_moe_mxfp8

void validate_mxfp8(const Tensor &x, const Tensor &x_scales, const Tensor &w, const Tensor &w_scales, const Tensor &w2,
                    const Tensor &w2_scales, const Tensor &sorted_token_ids, const Tensor &expert_ids,
                    const Tensor &num_tokens_post_padded, const Tensor &topk_weights, const Tensor &out, int64_t top_k,
                    int64_t block_m, int64_t block_n, int64_t warp_n, int64_t stages, int64_t bpc, bool split, bool placement) {
    const char *op = "fused_moe_mxfp8";
    REQUIRE(x.dim() == 2 && w.dim() == 3 && w2.dim() == 3, op, ": x must be 2-D, w and w2 3-D");
    const int64_t M = x.size(0), K = x.size(1), E = w.size(0), N = w.size(1);
    REQUIRE(M > 0, op, ": x has no rows");
    REQUIRE(K == w.size(2), op, ": x.size(1) must equal w.size(2)");
    REQUIRE(K % 256 == 0, "K dimension must be a multiple of 256 on the mxfp8 path");
    REQUIRE(N % 256 == 0, "N dimension must be a multiple of 256 on the mxfp8 path");
    REQUIRE(w2.size(0) == E && w2.size(1) == K && w2.size(2) == N / 2, op, ": w2 must have shape (E, K, N/2)");
    check_tuning("mxfp8", block_m, block_n, warp_n, stages, 4);
    REQUIRE(bpc == 1, "mxfp8 supports bpc=1 only");
    REQUIRE(top_k > 0, op, ": top_k must be positive");
    REQUIRE(x_scales.numel() == M * (K / 32), "x_scales must be a row major (M, K/32) e8m0 tensor");
    REQUIRE(w_scales.numel() == E * N * (K / 32), "w_scales must hold E*N*K/32 e8m0 values in the blocked layout");
    REQUIRE(w2_scales.numel() == E * K * ((N / 2) / 32), "w2_scales must hold E*K*(N/2)/32 e8m0 values in the blocked layout");
    const Arg ax{"x", &x}, axs{"x_scales", &x_scales}, aw{"w", &w}, aws{"w_scales", &w_scales}, aw2{"w2", &w2},
        aw2s{"w2_scales", &w2_scales}, as{"sorted_token_ids", &sorted_token_ids}, ae{"expert_ids", &expert_ids},
        an{"num_tokens_post_padded", &num_tokens_post_padded}, at_{"topk_weights", &topk_weights}, ao{"out", &out};
    if (placement) {
        require_same_device(op, {ax, axs, aw, aws, aw2, aw2s, as, ae, an, at_, ao});
        require_aligned(op, {ax, aw, aw2, ao}, 16);
        require_aligned(op, {axs, aws, aw2s, as, ae, an, at_}, 4);
    }
    require_contiguous(op, {ax, axs, aw, aws, aw2, aw2s, as, ae, an, at_, ao});
    require_dtype(op, {ax, aw, aw2}, at::kFloat8_e4m3fn, "float8_e4m3fn");
    require_dtype(op, {axs, aws, aw2s}, at::kFloat8_e8m0fnu, "float8_e8m0fnu");
    require_dtype(op, {at_}, at::kFloat, "float32");
    require_dtype(op, {as, ae, an}, at::kInt, "int32");
    require_dtype(op, {ao}, at::kBFloat16, "bfloat16");
    REQUIRE(out.dim() == 2 && out.size(0) == M && out.size(1) == K, op, ": out must have shape (M, K)");
    REQUIRE(num_tokens_post_padded.numel() >= 1, op, ": num_tokens_post_padded is empty");
    REQUIRE(expert_ids.numel() * block_m >= sorted_token_ids.numel(), op,
            ": expert_ids is shorter than sorted_token_ids / block_m");
}

void fused_moe_mxfp8(const Tensor &x, const Tensor &x_scales, const Tensor &w, const Tensor &w_scales, const Tensor &w2,
                     const Tensor &w2_scales, const Tensor &sorted_token_ids, const Tensor &expert_ids,
                     const Tensor &num_tokens_post_padded, const Tensor &topk_weights, Tensor &out, int64_t top_k,
                     int64_t block_m, int64_t block_n, int64_t warp_n, int64_t stages, int64_t bpc, bool split) {
    validate_mxfp8(x, x_scales, w, w_scales, w2, w2_scales, sorted_token_ids, expert_ids, num_tokens_post_padded, topk_weights,
                   out, top_k, block_m, block_n, warp_n, stages, bpc, split, true);
    const c10::Device dev = x.device();
    const c10::DeviceGuard guard(dev);
    const int M = (int)x.size(0), K = (int)x.size(1), E = (int)w.size(0), N = (int)w.size(1), S = (int)sorted_token_ids.size(0);
    const Tensor ws = workspace(pmoe_fused_moe_mxfp8_workspace_bytes(M, K, N, E, S, (int)top_k, split), dev);
    check_status(pmoe_fused_moe_mxfp8(
        x.const_data_ptr(), x_scales.const_data_ptr(), w.const_data_ptr(), w_scales.const_data_ptr(), w2.const_data_ptr(),
        w2_scales.const_data_ptr(), out.data_ptr(), sorted_token_ids.const_data_ptr<int32_t>(),
        expert_ids.const_data_ptr<int32_t>(), num_tokens_post_padded.const_data_ptr<int32_t>(),
        topk_weights.const_data_ptr<float>(), (int)top_k, M, K, N, E, S, (int)block_m, (int)block_n, (int)warp_n, (int)stages,
        (int)bpc, split, ws.data_ptr(), (size_t)ws.numel(), stream_of(dev)));
}

// ------------------------------------------------------------------------------- helpers that are not ops

std::tuple<Tensor, Tensor> quantize_mx(const Tensor &t) {
    REQUIRE(t.is_cuda(), "quantize_mx: a GPU tensor is required");
    REQUIRE(t.scalar_type() == at::kBFloat16, "quantize_mx: bfloat16 input required");
    REQUIRE(t.is_contiguous(), "quantize_mx: input must be contiguous");
    REQUIRE(t.dim() > 0, "quantize_mx: input must have a dimension");
    const int64_t cols = t.size(-1);
    REQUIRE(cols > 0 && cols % 32 == 0, "quantize_mx: last dim ", cols, " must be a multiple of 32");
    const c10::Device dev = t.device();
    const c10::DeviceGuard guard(dev);
    Tensor q = empty(t.sizes(), at::kFloat8_e4m3fn, dev);
    std::vector<int64_t> size = t.sizes().vec();
    size.back() = cols / 32;
    Tensor s = empty(size, at::kFloat8_e8m0fnu, dev);
    check_status(pmoe_quantize_mx(t.const_data_ptr(), q.data_ptr(), s.data_ptr(), t.numel() / cols, (int)cols, stream_of(dev)));
    return {q, s};
}

std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> route(const Tensor &logits, int64_t top_k, int64_t block_m, int64_t bpc,
                                                         const std::optional<Tensor> &bias) {
    REQUIRE(logits.is_cuda(), "route: logits must be a GPU tensor, got device ", logits.device());
    REQUIRE(logits.dim() == 2 && logits.is_contiguous(), "route: logits must be a contiguous (T, E) tensor");
    REQUIRE(logits.scalar_type() == at::kFloat || logits.scalar_type() == at::kBFloat16, "route: logits must be float32 or bfloat16");
    const int64_t T = logits.size(0), E = logits.size(1);
    REQUIRE(E > 0 && E <= 1024, "route supports 1..1024 experts, got ", E);
    REQUIRE(top_k > 0 && top_k <= std::min<int64_t>(32, E), "route: top_k must be in 1..min(32, E), got ", top_k);
    REQUIRE(block_m > 0 && bpc > 0, "route: block_m and bpc must be positive");
    const c10::Device dev = logits.device();
    if (bias.has_value())
        REQUIRE(bias->device() == dev && bias->scalar_type() == at::kFloat && bias->is_contiguous() && bias->numel() == E,
                "route: bias must be a contiguous float32 (E,) tensor on the device of logits");
    const c10::DeviceGuard guard(dev);
    const int64_t n = T * top_k;
    const AlignSizes sz(n, E, block_m, bpc);
    Tensor topk_ids = empty({T, top_k}, at::kInt, dev), topk_weights = empty({T, top_k}, at::kFloat, dev);
    Schedule s(sz, n, E, dev);
    check_status(pmoe_route(logits.const_data_ptr(), logits.scalar_type() == at::kFloat ? PMOE_DTYPE_F32 : PMOE_DTYPE_BF16,
                            bias.has_value() ? bias->const_data_ptr<float>() : nullptr, topk_ids.data_ptr<int32_t>(),
                            topk_weights.data_ptr<float>(), s.sorted_token_ids.data_ptr<int32_t>(),
                            s.expert_ids.data_ptr<int32_t>(), s.num_tokens_post_padded.data_ptr<int32_t>(), (int)T, (int)E,
                            (int)top_k, (int)block_m, (int)sz.pad_to, (int)sz.max_padded, (int)sz.max_blocks, s.ws_ptr(),
                            s.ws_bytes, stream_of(dev)));
    return {topk_ids, topk_weights, s.sorted_token_ids, s.expert_ids, s.num_tokens_post_padded};
}

}  // namespace

TORCH_LIBRARY_IMPL(prime_moe, CUDA, m) {
    m.impl("moe_align", &moe_align);
    m.impl("fused_moe_bf16", &fused_moe_bf16);
    m.impl("fused_moe_mxfp8", &fused_moe_mxfp8);
}

PYBIND11_MODULE(_torch_ops, m) {
    namespace py = pybind11;
    const auto nogil = py::call_guard<py::gil_scoped_release>();
    m.def("validate_align", &validate_align, nogil);
    m.def("validate_bf16", &validate_bf16, nogil);
    m.def("validate_mxfp8", &validate_mxfp8, nogil);
    m.def("quantize_mx", &quantize_mx, nogil);
    m.def("route", &route, nogil);
}
