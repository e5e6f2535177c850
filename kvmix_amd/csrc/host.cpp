// The host side of the operators that run once per layer and step: argument checks, strides, outputs and workspaces, and
// the call into the C ABI, on torch tensors.  In Python the descriptor of one attention step took longer to fill than its
// kernels took to run: a GEMV call 12 us of interpreter for 7 us of GPU, an append or a step on the 9-tuple three to
// five times its launches.  The kernels are reached through the addresses that bind() is given, so that the library in use
// stays the one the loader chose.
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <stdexcept>
#include <string>
#include <tuple>
#include <unordered_map>
#include <vector>

#include "../../include/kvmix_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using Triple = std::tuple<Tensor, Tensor, Tensor>;
using OptTriple = std::optional<std::tuple<OptTensor, OptTensor, OptTensor>>;

struct Api {
    decltype(&kvmix_strerror) strerror;
    decltype(&kvmix_quant_pack_last_dim) quant_pack_last_dim;
    decltype(&kvmix_quant_pack_kv_flush) quant_pack_kv_flush;
    decltype(&kvmix_gemv_workspace_bytes) gemv_workspace_bytes;
    decltype(&kvmix_quantized_gemv) quantized_gemv;
    decltype(&kvmix_decode_attention_workspace_bytes) decode_attention_workspace_bytes;
    decltype(&kvmix_decode_attention) decode_attention;
    decltype(&kvmix_decode_attention_fused_supported) decode_attention_fused_supported;
    decltype(&kvmix_decode_attention_fused_workspace_bytes) decode_attention_fused_workspace_bytes;
    decltype(&kvmix_decode_attention_fused) decode_attention_fused;
    decltype(&kvmix_decode_attention_fused_plan) decode_attention_fused_plan;
    decltype(&kvmix_decode_attention_fused_weights_workspace_bytes) decode_attention_fused_weights_workspace_bytes;
    decltype(&kvmix_decode_attention_fused_weights_recommended) decode_attention_fused_weights_recommended;
    decltype(&kvmix_decode_attention_fused_weights) decode_attention_fused_weights;
    decltype(&kvmix_copy_rows) copy_rows;
    decltype(&kvmix_grow) grow;
    decltype(&kvmix_linear_rows) linear_rows;
} api;

void bind(const std::unordered_map<std::string, uintptr_t> &at)
{
#define KVMIX_BIND(name) api.name = reinterpret_cast<decltype(api.name)>(at.at("kvmix_" #name))
    KVMIX_BIND(strerror);
    KVMIX_BIND(quant_pack_last_dim);
    KVMIX_BIND(quant_pack_kv_flush);
    KVMIX_BIND(gemv_workspace_bytes);
    KVMIX_BIND(quantized_gemv);
    KVMIX_BIND(decode_attention_workspace_bytes);
    KVMIX_BIND(decode_attention);
    KVMIX_BIND(decode_attention_fused_supported);
    KVMIX_BIND(decode_attention_fused_workspace_bytes);
    KVMIX_BIND(decode_attention_fused);
    KVMIX_BIND(decode_attention_fused_plan);
    KVMIX_BIND(decode_attention_fused_weights_workspace_bytes);
    KVMIX_BIND(decode_attention_fused_weights_recommended);
    KVMIX_BIND(decode_attention_fused_weights);
    KVMIX_BIND(copy_rows);
    KVMIX_BIND(grow);
    KVMIX_BIND(linear_rows);
#undef KVMIX_BIND
}

[[noreturn]] void fail(const std::string &what) { throw std::runtime_error(what); }

void check(int rc)
{
    if (rc != KVMIX_OK) fail(api.strerror(rc));
}

std::string dtype_name(const Tensor &t)
{
    const py::gil_scoped_acquire gil;
    return py::str(py::reinterpret_borrow<py::object>((PyObject *)torch::getTHPDtype(t.scalar_type())));
}

void need_gpu(std::initializer_list<const Tensor *> ts)
{
    for (const Tensor *t : ts)
        if (!t->is_cuda()) fail("KVmix operators run on the GPU only: got a tensor on " + t->device().str());
}

void need_half(std::initializer_list<const Tensor *> ts)
{
    for (const Tensor *t : ts)
        if (t->scalar_type() != at::kHalf) fail("expected scalar type Half but found " + dtype_name(*t));
}

// what a kernel reads or writes beside `ref` lies where `ref` does
void need_with(const Tensor &ref, std::initializer_list<const Tensor *> ts)
{
    for (const Tensor *t : ts)
        if (t->device() != ref.device()) fail("expected all tensors on " + ref.device().str() + ", but one is on " + t->device().str());
}

void check_bits(int64_t bits)
{
    if (bits < 1 || bits > 4) fail("Supported quantization bits: 1, 2, 3, 4");
}

kvmix_stream_t stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

int dtype_tag(const Tensor &t) { return t.scalar_type() == at::kHalf ? KVMIX_F16 : KVMIX_F32; }

// Whether a call on this tensor is an ordinary one, which a kernel without an autograd formula may serve: nothing records
// it (gradients of either mode, a trace) and nothing interprets it (transforms, tensor subclasses and modes).
bool plain(const Tensor &t)
{
    using c10::DispatchKey;
    static const c10::DispatchKeySet wrapped({DispatchKey::Python, DispatchKey::FuncTorchGradWrapper, DispatchKey::FuncTorchBatched,
                                              DispatchKey::Batched, DispatchKey::Functionalize});
    return !(at::GradMode::is_enabled() && t.requires_grad()) && !t.key_set().has_any(wrapped) && !t._fw_grad(0).defined() &&
           c10::impl::TorchDispatchModeTLS::stack_len() == 0 && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           !torch::jit::tracer::isTracing();
}

// [B, H, R, S] as [B*H, R, S] without copying when its strides allow it (unit stride along S)
struct Rows {
    Tensor t;
    int64_t outer, inner;  // strides in elements
};

Rows rows3(const Tensor &x)
{
    const int64_t B = x.size(0), H = x.size(1), R = x.size(2), S = x.size(3);
    const bool ok = (S <= 1 || x.stride(3) == 1) && (B <= 1 || x.stride(0) == H * x.stride(1)) && (R <= 1 || x.stride(2) >= S) &&
                    (H <= 1 || x.stride(1) >= x.stride(2));
    Tensor t = ok ? x : x.contiguous();
    const int64_t outer = B * H > 1 ? t.stride(1) : std::max<int64_t>(R * std::max(t.stride(2), S), 1);
    const int64_t inner = R > 1 ? t.stride(2) : std::max<int64_t>(S, 1);
    return {std::move(t), outer, inner};
}

Tensor empty(std::initializer_list<int64_t> sizes, c10::ScalarType type, const Tensor &like)
{
    return at::empty(c10::IntArrayRef(sizes.begin(), sizes.size()), like.options().dtype(type).requires_grad(false));
}

Tensor scratch(size_t bytes, const Tensor &like) { return bytes ? empty({(int64_t)bytes}, at::kByte, like) : Tensor(); }

// ---------------------------------------------------------------------------------------------------------------------
// quantizers

int64_t codes_per_word(int64_t bits) { return bits == 3 ? 11 : 32 / bits; }

void quantize_into(const Tensor &x, int64_t group, int64_t bits, int fmt, int scale_mode, const Tensor &code, const Tensor &scale, const Tensor &mn)
{
    const Rows r = rows3(x);
    const c10::DeviceGuard guard(x.device());
    check(api.quant_pack_last_dim(r.t.data_ptr(), dtype_tag(x), x.size(0) * x.size(1), x.size(2), x.size(3), r.outer, r.inner, (int)group,
                                  (int)bits, fmt, scale_mode, (uint32_t *)code.data_ptr(), code.stride(1), code.stride(2), scale.data_ptr(),
                                  mn.data_ptr(), scale.stride(1), scale.stride(2), stream_of(x)));
}

void check_input(const Tensor &x)
{
    if (x.scalar_type() != at::kHalf && x.scalar_type() != at::kFloat) fail("expected scalar type Float or Half but found " + dtype_name(x));
    if (x.dim() != 4) fail("input_tensor must be a 4D tensor");
}

Triple quantize(const Tensor &x, int64_t group, int64_t bits, int fmt, int64_t words)
{
    need_gpu({&x});
    Tensor code = empty({x.size(0), x.size(1), x.size(2), words}, at::kInt, x);
    Tensor scale = empty({x.size(0), x.size(1), x.size(2), x.size(3) / group}, x.scalar_type(), x);
    Tensor mn = at::empty_like(scale);
    quantize_into(x, group, bits, fmt, KVMIX_SCALE_RECIPROCAL, code, scale, mn);
    return {code, scale, mn};
}

Triple quantize_pack_last_dim(const Tensor &x, int64_t group, int64_t bits)
{
    if (bits == 3 && group != 11) fail("For 3-bit quantization, group_length must be 11");
    check_input(x);
    check_bits(bits);
    const int64_t S = x.size(3);
    if (bits == 3) {
        if (S % 11 != 0) fail("For 3-bit quantization, steps must be divisible by 11");
    } else {
        if (group <= 0 || S % group != 0) fail("steps must be divisible by group_length");
        if (S % (32 / bits) != 0) fail("steps must be divisible by (32 / quant_bits)");
    }
    return quantize(x, group, bits, KVMIX_FMT_REF, S / codes_per_word(bits));
}

Triple quantize_pack_dense3(const Tensor &x, int64_t group)
{
    check_input(x);
    if (group <= 0 || group % 32 != 0) fail("dense 3-bit needs a group_length that is a multiple of 32");
    if (x.size(3) % group != 0) fail("steps must be divisible by group_length");
    return quantize(x, group, 3, KVMIX_FMT_DENSE3, x.size(3) * 3 / 32);
}

// ---------------------------------------------------------------------------------------------------------------------
// copies

struct Copies {
    std::vector<kvmix_copy_rows_t> items;
    std::vector<Tensor> keep;
    Tensor first;

    // whether a copy of this tensor is within the 16-byte pieces that one launch counts (whatever its rows join to)
    static bool fits(const Tensor &t)
    {
        const int64_t row = t.dim() == 4 ? t.size(3) : 1;
        return row == 0 || t.numel() / row * ((row * (int64_t)t.element_size() + 15) / 16) < (1ll << 31) - 4096;
    }

    void add(const Tensor &dst, const Tensor &from)
    {
        if (from.sizes() != dst.sizes() || from.scalar_type() != dst.scalar_type() || from.dim() != 4)
            fail("copy_rows: source and destination must be 4-D and of equal shape and type");
        if (from.numel() == 0) return;
        need_gpu({&from, &dst});
        if (!first.defined()) first = dst;
        if (from.device() != first.device() || dst.device() != first.device()) fail("the copies of one launch must be on one device");
        const int64_t B = dst.size(0), H = dst.size(1), R = dst.size(2), S = dst.size(3), es = dst.element_size();
        // unit stride along the last dimension, (B, H) collapsible
        auto ok = [&](const Tensor &t) { return (S <= 1 || t.stride(3) == 1) && (B <= 1 || H <= 1 || t.stride(0) == H * t.stride(1)); };
        if (!ok(dst)) fail("copy_rows: destinations must be unit-stride along the last dimension, (B, H) collapsible");
        const Tensor src = ok(from) ? from : from.contiguous();
        keep.push_back(src);
        kvmix_copy_rows_t it;
        it.src = src.data_ptr();
        it.dst = dst.data_ptr();
        it.outer = B * H, it.inner = R, it.row_bytes = S * es;
        it.src_outer_stride = es * src.stride(H > 1 ? 1 : 0), it.src_inner_stride = es * src.stride(2);
        it.dst_outer_stride = es * dst.stride(H > 1 ? 1 : 0), it.dst_inner_stride = es * dst.stride(2);
        items.push_back(it);
    }

    // rows [from_row, from_row + rows) of `from` (its last dimension `cols`) to rows [row, ..) of `out`, a fresh [B, H, ., .]
    // tensor, from column 0 on; the caller has seen that their sizes and types match
    void add_rows(const Tensor &out, int64_t row, const Tensor &from, int64_t from_row, int64_t rows, int64_t cols)
    {
        if (rows == 0 || cols == 0) return;
        if (!first.defined()) first = out;
        const int64_t B = from.size(0), H = from.size(1), es = from.element_size();
        const bool ok = (cols <= 1 || from.stride(3) == 1) && (B <= 1 || H <= 1 || from.stride(0) == H * from.stride(1));
        Tensor copied;
        if (!ok) copied = from.narrow(2, from_row, rows).contiguous();
        const Tensor &src = ok ? from : copied;
        if (!ok) from_row = 0;
        kvmix_copy_rows_t it;
        it.src = (const char *)src.data_ptr() + from_row * src.stride(2) * es;
        it.dst = (char *)out.data_ptr() + row * out.stride(2) * es;
        it.outer = B * H, it.inner = rows, it.row_bytes = cols * es;
        it.src_outer_stride = es * src.stride(H > 1 ? 1 : 0), it.src_inner_stride = es * src.stride(2);
        it.dst_outer_stride = es * out.stride(1), it.dst_inner_stride = es * out.stride(2);
        items.push_back(it);
        if (!ok) keep.push_back(std::move(copied));
    }

    void run()
    {
        if (items.empty()) return;
        const c10::DeviceGuard guard(first.device());
        check(api.copy_rows(items.data(), (int)items.size(), stream_of(first)));
    }
};

void copy_rows(const std::vector<std::pair<Tensor, Tensor>> &pairs)
{
    Copies c;
    for (const auto &p : pairs) c.add(p.first, p.second);
    c.run();
}

// the cache so far to the front of its grown copy: one launch, or torch's copies for what that does not take (previous
// codes of another integer type, tensors on another device, calls that something records)
void copy_previous(const std::vector<std::pair<Tensor, Tensor>> &pairs)
{
    Copies c;
    for (const auto &p : pairs) {
        const Tensor src = p.second.reshape(p.first.sizes());
        if (src.scalar_type() == p.first.scalar_type() && src.device() == p.first.device() && plain(src) && Copies::fits(p.first))
            c.add(p.first, src);
        else
            p.first.copy_(src);
    }
    c.run();
}

// Previous parts of a grown cache that one launch moves, quantizing x to behind them (rows of 16-bit values): of the
// expected shape and type, on x's device, in a call that nothing records.
bool grows_in_one(const Tensor &x, const Tensor &code0, const Tensor &scale0, const Tensor &mn0, int64_t R, int64_t words, int64_t groups)
{
    auto takes = [&](const Tensor &t, c10::ScalarType type, int64_t cols) {
        return t.scalar_type() == type && t.device() == x.device() && t.dim() == 4 && t.size(0) == x.size(0) && t.size(1) == x.size(1) &&
               t.size(2) == R && t.size(3) == cols && plain(t) && Copies::fits(t);
    };
    return x.scalar_type() == at::kHalf && x.numel() > 0 && takes(code0, at::kInt, words) && takes(scale0, at::kHalf, groups) &&
           takes(mn0, at::kHalf, groups);
}

// the launch: code, scale and mn are fresh; x's results go to behind `words` / `groups` columns (dim 3) or `rows` rows (dim 2)
void grow_rows(const Tensor &x, const Tensor &code0, const Tensor &scale0, const Tensor &mn0, const Tensor &code, const Tensor &scale, const Tensor &mn,
               int64_t group, int64_t bits, int fmt, int64_t code_at, int64_t scale_at)
{
    Copies c;
    c.items.reserve(3);
    c.add_rows(code, 0, code0, 0, code0.size(2), code0.size(3));
    c.add_rows(scale, 0, scale0, 0, scale0.size(2), scale0.size(3));
    c.add_rows(mn, 0, mn0, 0, mn0.size(2), mn0.size(3));
    const Rows r = rows3(x);
    kvmix_value_flush_t vf{};
    vf.x = r.t.data_ptr(), vf.outer = x.size(0) * x.size(1), vf.inner = x.size(2), vf.steps = x.size(3);
    vf.x_outer_stride = r.outer, vf.x_inner_stride = r.inner;
    vf.group = (int)group, vf.bits = (int)bits, vf.fmt = fmt, vf.scale_mode = KVMIX_SCALE_DIVIDE;
    vf.code = (uint32_t *)code.data_ptr() + code_at, vf.code_outer_stride = code.stride(1), vf.code_inner_stride = code.stride(2);
    vf.scale = (char *)scale.data_ptr() + 2 * scale_at, vf.zero = (char *)mn.data_ptr() + 2 * scale_at;
    vf.sz_outer_stride = scale.stride(1), vf.sz_inner_stride = scale.stride(2);
    const c10::DeviceGuard guard(x.device());
    check(api.grow(c.items.data(), (int)c.items.size(), nullptr, &vf, stream_of(x)));
}

void append_checks(const Tensor &x, const Tensor &scale, const Tensor &mn, int64_t bits)
{
    if (x.dim() != 4) fail("input_tensor must be a 4D tensor");
    if (x.scalar_type() != at::kHalf && x.scalar_type() != at::kFloat) fail("expected scalar type Float or Half but found " + dtype_name(x));
    if (scale.scalar_type() != x.scalar_type() || mn.scalar_type() != x.scalar_type()) fail("previous_scale / previous_min must have the input's dtype");
    check_bits(bits);
}

Triple append_keys(const Tensor &x, const Tensor &code0, const Tensor &scale0, const Tensor &mn0, int64_t group, int64_t bits)
{
    append_checks(x, scale0, mn0, bits);
    const int64_t B = x.size(0), H = x.size(1), D = x.size(2), n = x.size(3);
    if (bits == 3) {
        if (group != 11) fail("For 3-bit quantization, group_length must be 11");
        if (n % 11 != 0) fail("new_steps must be divisible by 11 for 3-bit quantization");
    } else if (group <= 0 || n % group != 0) {
        fail("new_steps must be divisible by group_length");
    }
    need_gpu({&x, &code0, &scale0, &mn0});
    const int64_t vpw = codes_per_word(bits);
    if (bits != 3 && (group % vpw != 0 || n % vpw != 0)) check(KVMIX_ERR_UNSUPPORTED);
    const int64_t ow = code0.size(3), og = scale0.size(3);
    Tensor code = empty({B, H, D, ow + n / vpw}, at::kInt, x), scale = empty({B, H, D, og + n / group}, x.scalar_type(), x);
    Tensor mn = at::empty_like(scale);
    if (grows_in_one(x, code0, scale0, mn0, D, ow, og)) {
        grow_rows(x, code0, scale0, mn0, code, scale, mn, group, bits, KVMIX_FMT_REF, ow, og);
        return {code, scale, mn};
    }
    copy_previous({{code.narrow(3, 0, ow), code0}, {scale.narrow(3, 0, og), scale0}, {mn.narrow(3, 0, og), mn0}});
    if (n > 0)
        quantize_into(x, group, bits, KVMIX_FMT_REF, KVMIX_SCALE_DIVIDE, code.narrow(3, ow, n / vpw), scale.narrow(3, og, n / group),
                      mn.narrow(3, og, n / group));
    return {code, scale, mn};
}

Triple append_values(const Tensor &x, const Tensor &code0, const Tensor &scale0, const Tensor &mn0, int64_t group, int64_t bits)
{
    append_checks(x, scale0, mn0, bits);
    const int64_t B = x.size(0), H = x.size(1), n = x.size(2), D = x.size(3);
    if (bits == 3) {
        if (group != 11) fail("For 3-bit quantization, group_length must be 11");
        if (D % 11 != 0) fail("head_dim must be divisible by 11 for 3-bit quantization");
    } else if (group <= 0 || D % group != 0) {
        fail("head_dim must be divisible by group_length");
    }
    need_gpu({&x, &code0, &scale0, &mn0});
    const int64_t vpw = codes_per_word(bits);
    if (bits != 3 && (group % vpw != 0 || D % vpw != 0)) check(KVMIX_ERR_UNSUPPORTED);
    const int64_t old = code0.size(2);
    Tensor code = empty({B, H, old + n, D / vpw}, at::kInt, x), scale = empty({B, H, old + n, D / group}, x.scalar_type(), x);
    Tensor mn = at::empty_like(scale);
    if (grows_in_one(x, code0, scale0, mn0, old, D / vpw, D / group)) {
        grow_rows(x, code0, scale0, mn0, code, scale, mn, group, bits, bits == 3 ? KVMIX_FMT_REF3_WRAP : KVMIX_FMT_REF, old * (D / vpw),
                  old * (D / group));
        return {code, scale, mn};
    }
    copy_previous({{code.narrow(2, 0, old), code0}, {scale.narrow(2, 0, old), scale0}, {mn.narrow(2, 0, old), mn0}});
    if (n > 0)
        quantize_into(x, group, bits, bits == 3 ? KVMIX_FMT_REF3_WRAP : KVMIX_FMT_REF, KVMIX_SCALE_DIVIDE, code.narrow(2, old, n),
                      scale.narrow(2, old, n), mn.narrow(2, old, n));
    return {code, scale, mn};
}

// The 9-tuple after one call's tokens: everything moved into new tensors, and what the policy flushes (nk, nv tokens of the
// OLD tails) quantized from the old tails to behind the old packed part, in one launch (kvmix_grow; two or three where the
// value half streams or the formats are not the fused kernel's).  The caller has checked
// that nk and nv fit the old tails and that the flush kernels take the groups and widths.  None: torch's composition.
using Grown = std::tuple<OptTensor, Tensor, OptTensor, OptTensor, OptTensor, Tensor, OptTensor, OptTensor>;
std::optional<Grown> grow_tuple(const OptTensor &kc, const Tensor &k_tail, const OptTensor &ks, const OptTensor &km, const OptTensor &vc,
                                const Tensor &v_tail, const OptTensor &vs, const OptTensor &vm, const Tensor &key, const Tensor &value,
                                int64_t nk, int64_t nv, int64_t k_bits, int64_t k_group, int64_t v_bits)
{
    auto takes = [&](const Tensor &t, c10::ScalarType type) {
        return t.scalar_type() == type && t.dim() == 4 && t.is_cuda() && t.device() == key.device() && plain(t) && Copies::fits(t);
    };
    for (const Tensor *t : {&k_tail, &v_tail, &key, &value})
        if (!takes(*t, at::kHalf)) return std::nullopt;
    for (const OptTensor *t : {&ks, &km, &vs, &vm})
        if (*t && !takes(**t, at::kHalf)) return std::nullopt;
    for (const OptTensor *t : {&kc, &vc})
        if (*t && !takes(**t, at::kInt)) return std::nullopt;
    const int64_t B = key.size(0), H = key.size(1), n = key.size(2), D = key.size(3);
    if (value.sizes() != key.sizes() || D % 32 != 0) return std::nullopt;
    for (const Tensor *t : {&k_tail, &v_tail})
        if (t->size(0) != B || t->size(1) != H || t->size(3) != D || (t->size(2) > 1 && t->stride(2) < D)) return std::nullopt;
    if (kc.has_value() != ks.has_value() || kc.has_value() != km.has_value() || vc.has_value() != vs.has_value() ||
        vc.has_value() != vm.has_value())
        return std::nullopt;
    // the previous packed parts must be what their new tensors continue
    auto shaped = [&](const OptTensor &t, int64_t rows, int64_t cols) {
        return !t || (t->size(0) == B && t->size(1) == H && (rows < 0 || t->size(2) == rows) && (cols < 0 || t->size(3) == cols));
    };
    const bool even_k = shaped(kc, D, -1) && shaped(ks, D, -1) && shaped(km, D, -1);
    const bool even_v = shaped(vc, -1, D * v_bits / 32) && shaped(vs, -1, D / 32) && shaped(vm, -1, D / 32);
    if ((nk > 0 && !even_k) || (nv > 0 && !even_v)) fail("copy_rows: source and destination must be 4-D and of equal shape and type");
    Copies c;
    c.items.reserve(10);
    auto tail = [&](const Tensor &old, const Tensor &fresh, int64_t drop) {
        const int64_t keep = old.size(2) - drop;
        Tensor out = empty({B, H, keep + n, D}, at::kHalf, key);
        c.add_rows(out, 0, old, drop, keep, D);
        c.add_rows(out, keep, fresh, 0, n, D);
        return out;
    };
    const Tensor new_k = tail(k_tail, key, nk), new_v = tail(v_tail, value, nv);
    // (behind: where the flush writes, the columns or rows past the old part)
    auto grown = [&](const OptTensor &old, c10::ScalarType type, int64_t rows, int64_t cols, int64_t dim, void *&behind) {
        const int64_t have = old ? old->size(dim) : 0;
        Tensor out = dim == 3 ? empty({B, H, rows, have + cols}, type, key) : empty({B, H, have + rows, cols}, type, key);
        if (have) c.add_rows(out, 0, *old, 0, dim == 3 ? rows : have, dim == 3 ? have : cols);
        behind = (char *)out.data_ptr() + have * (dim == 3 ? 1 : cols) * (int64_t)out.element_size();
        return OptTensor(std::move(out));
    };
    Grown g(kc, new_k, ks, km, vc, new_v, vs, vm);
    kvmix_key_flush_t kf{};
    kvmix_value_flush_t vf{};
    kf.group = (int)k_group, kf.bits = (int)k_bits, kf.fmt = KVMIX_FMT_REF, kf.scale_mode = KVMIX_SCALE_RECIPROCAL;
    vf.group = 32, vf.bits = (int)v_bits, vf.fmt = KVMIX_FMT_REF, vf.scale_mode = KVMIX_SCALE_RECIPROCAL;
    Tensor from_k;
    Rows from_v;
    void *behind = nullptr;
    if (nk > 0) {
        std::get<0>(g) = grown(kc, at::kInt, D, nk / codes_per_word(k_bits), 3, behind);
        kf.code = (uint32_t *)behind;
        std::get<2>(g) = grown(ks, at::kHalf, D, nk / k_group, 3, kf.scale);
        std::get<3>(g) = grown(km, at::kHalf, D, nk / k_group, 3, kf.zero);
        const Tensor &code = *std::get<0>(g), &scale = *std::get<2>(g);
        from_k = k_tail.narrow(2, 0, nk);
        if (from_k.stride(3) != 1 || (B > 1 && from_k.stride(0) != H * from_k.stride(1))) from_k = from_k.contiguous();
        kf.k = from_k.data_ptr(), kf.outer = B * H, kf.n = nk, kf.D = D;
        kf.k_outer_stride = from_k.stride(1), kf.k_token_stride = from_k.stride(2);
        kf.code_outer_stride = code.stride(1), kf.code_inner_stride = code.stride(2);
        kf.sz_outer_stride = scale.stride(1), kf.sz_inner_stride = scale.stride(2);
    }
    if (nv > 0) {
        std::get<4>(g) = grown(vc, at::kInt, nv, D * v_bits / 32, 2, behind);
        vf.code = (uint32_t *)behind;
        std::get<6>(g) = grown(vs, at::kHalf, nv, D / 32, 2, vf.scale);
        std::get<7>(g) = grown(vm, at::kHalf, nv, D / 32, 2, vf.zero);
        const Tensor &vcode = *std::get<4>(g), &vscale = *std::get<6>(g);
        from_v = rows3(v_tail.narrow(2, 0, nv));
        vf.x = from_v.t.data_ptr(), vf.outer = B * H, vf.inner = nv, vf.steps = D;
        vf.x_outer_stride = from_v.outer, vf.x_inner_stride = from_v.inner;
        vf.code_outer_stride = vcode.stride(1), vf.code_inner_stride = vcode.stride(2);
        vf.sz_outer_stride = vscale.stride(1), vf.sz_inner_stride = vscale.stride(2);
    }
    const c10::DeviceGuard guard(key.device());
    check(api.grow(c.items.data(), (int)c.items.size(), nk > 0 ? &kf : nullptr, nv > 0 ? &vf : nullptr, stream_of(key)));
    return g;
}

// ---------------------------------------------------------------------------------------------------------------------
// products and the attention step

// scales and zeros in one pair of strides
std::pair<Rows, Rows> scale_rows(const Tensor &scale, const Tensor &zero)
{
    Rows s = rows3(scale), z = rows3(zero);
    if (s.outer != z.outer || s.inner != z.inner) {
        s = rows3(scale.contiguous());
        z = rows3(zero.contiguous());
    }
    return {s, z};
}

Tensor quantized_gemm(int64_t group, const Tensor &fA, const Tensor &qB, const Tensor &scales, const Tensor &zeros, int64_t bits, int64_t fmt)
{
    if (fA.dim() != 4 || qB.dim() != 4) fail("Input tensors must be 4-dimensional");
    check_bits(bits);
    const int64_t B = fA.size(0), nh = fA.size(1), M = fA.size(2), K = fA.size(3), nkv = qB.size(1);
    if (nkv == 0 || nh % nkv != 0) fail("Total heads must be divisible by KV heads");
    if (bits == 3 && fmt == KVMIX_FMT_REF && group != 11) fail("For 3-bit quantization, group size must be 11");
    if (fA.scalar_type() != at::kHalf || scales.scalar_type() != at::kHalf || zeros.scalar_type() != at::kHalf)
        fail("expected scalar type Half for fA, scales and zeros");
    if (qB.scalar_type() != at::kInt) fail("expected scalar type Int for qB");
    need_gpu({&fA, &qB, &scales, &zeros});
    if (scales.dim() != 4 || zeros.dim() != 4 || scales.sizes() != zeros.sizes()) fail("scales and zeros must be 4-dimensional and of equal shape");
    if (qB.size(0) != B || qB.size(2) != K || scales.size(0) != B || scales.size(1) != nkv || scales.size(2) != K)
        fail("shape mismatch between fA, qB and scales");
    const int64_t N = zeros.size(3) * group;  // dequantization_gemv_cuda.cu:184
    const Rows x = rows3(fA), c = rows3(qB);
    const auto [s, z] = scale_rows(scales, zeros);
    Tensor out = empty({B, nh, M, N}, at::kHalf, fA);
    const size_t ws_bytes = api.gemv_workspace_bytes(B * nh, M, K, N);
    const Tensor ws = scratch(ws_bytes, fA);
    const c10::DeviceGuard guard(fA.device());
    check(api.quantized_gemv((int)group, x.t.data_ptr(), x.outer, x.inner, (const uint32_t *)c.t.data_ptr(), c.outer, c.inner, s.t.data_ptr(),
                             z.t.data_ptr(), s.outer, s.inner, (int)bits, (int)fmt, B * nh, (int)(nh / nkv), M, K, N, out.data_ptr(), M * N, N,
                             ws.defined() ? ws.data_ptr() : nullptr, ws_bytes, stream_of(fA)));
    return out;
}

bool prefer_single_pass(int64_t batch, int64_t heads, int64_t kv_heads, int64_t D, int64_t width, int64_t k_bits, int64_t k_fmt, int64_t k_group,
                        int64_t v_bits, int64_t v_fmt, int64_t v_group, int64_t k_tokens, int64_t v_tokens, bool weights)
{
    kvmix_decode_attn_t st{};
    const bool ref3 = k_bits == 3 && k_fmt == KVMIX_FMT_REF;
    st.samples = batch * heads, st.heads = (int)heads, st.heads_per_kv = (int)(heads / kv_heads), st.D = D;
    st.q_stride = st.out_stride = D;
    st.k_bits = (int)k_bits, st.k_fmt = (int)k_fmt, st.k_group = (int)k_group, st.k_tokens = k_tokens;
    st.k_code_row_stride = ref3 ? k_tokens / 11 : k_tokens * k_bits / 32;
    st.k_code_batch_stride = D * st.k_code_row_stride;
    st.k_sz_row_stride = k_tokens / (ref3 ? 11 : std::max<int64_t>(k_group, 1));
    st.k_sz_batch_stride = D * st.k_sz_row_stride;
    st.v_bits = (int)v_bits, st.v_fmt = (int)v_fmt, st.v_group = (int)v_group, st.v_tokens = v_tokens;
    st.v_code_row_stride = D * v_bits / 32;
    st.v_code_batch_stride = v_tokens * st.v_code_row_stride;
    st.v_sz_row_stride = D / std::max<int64_t>(v_group, 1);
    st.v_sz_batch_stride = v_tokens * st.v_sz_row_stride;
    st.k_tail_slots = st.k_tail_len = width - k_tokens, st.v_tail_slots = st.v_tail_len = width - v_tokens;
    st.k_tail_token_stride = st.v_tail_token_stride = D;
    st.k_tail_batch_stride = st.k_tail_slots * D, st.v_tail_batch_stride = st.v_tail_slots * D;
    if (weights) return api.decode_attention_fused_weights_recommended(&st);
    kvmix_attn_plan_t plan;
    return api.decode_attention_fused_plan(&st, &plan) == KVMIX_OK && plan.recommended;
}

// k_len / v_len: live tail slots (none: all); *_len_dev: where the kernels read them instead
std::pair<Tensor, OptTensor> decode_attention(const Tensor &q_in, const OptTriple &k_packed, const OptTriple &v_packed, const Tensor &k_tail,
                                              const Tensor &v_tail, int64_t k_group, int64_t k_bits, int64_t v_group, int64_t v_bits,
                                              int64_t k_fmt, int64_t v_fmt, const OptTensor &mask_in, std::optional<int64_t> k_len,
                                              const OptTensor &k_len_dev, std::optional<int64_t> v_len, const OptTensor &v_len_dev, bool single_pass,
                                              bool weights)
{
    if (q_in.dim() != 4 || q_in.size(2) != 1) fail("decode_attention takes one query position: q must be [B, nh, 1, D]");
    need_half({&q_in, &k_tail, &v_tail});
    need_gpu({&q_in, &k_tail, &v_tail});
    check_bits(k_bits);
    check_bits(v_bits);
    const int64_t B = q_in.size(0), nh = q_in.size(1), D = q_in.size(3), nkv = k_tail.size(1);
    if (nkv == 0 || nh % nkv != 0) fail("Total heads must be divisible by KV heads");
    kvmix_decode_attn_t st{};
    const Rows q = rows3(q_in);
    st.q = q.t.data_ptr(), st.q_stride = q.outer;
    Rows kc, vc;
    std::pair<Rows, Rows> ksz, vsz;
    if (k_packed && std::get<0>(*k_packed)) {
        kc = rows3(*std::get<0>(*k_packed));
        ksz = scale_rows(std::get<1>(*k_packed).value(), std::get<2>(*k_packed).value());
        st.k_code = (const uint32_t *)kc.t.data_ptr(), st.k_code_batch_stride = kc.outer, st.k_code_row_stride = kc.inner;
        st.k_scale = ksz.first.t.data_ptr(), st.k_zero = ksz.second.t.data_ptr();
        st.k_sz_batch_stride = ksz.first.outer, st.k_sz_row_stride = ksz.first.inner;
        st.k_tokens = ksz.second.t.size(3) * k_group;
    }
    if (v_packed && std::get<0>(*v_packed)) {
        vc = rows3(*std::get<0>(*v_packed));
        vsz = scale_rows(std::get<1>(*v_packed).value(), std::get<2>(*v_packed).value());
        st.v_code = (const uint32_t *)vc.t.data_ptr(), st.v_code_batch_stride = vc.outer, st.v_code_row_stride = vc.inner;
        st.v_scale = vsz.first.t.data_ptr(), st.v_zero = vsz.second.t.data_ptr();
        st.v_sz_batch_stride = vsz.first.outer, st.v_sz_row_stride = vsz.first.inner;
        st.v_tokens = vc.t.size(2);
    }
    st.k_bits = (int)k_bits, st.k_fmt = (int)k_fmt, st.k_group = (int)k_group;
    st.v_bits = (int)v_bits, st.v_fmt = (int)v_fmt, st.v_group = (int)v_group;
    const Rows kt = rows3(k_tail), vt = rows3(v_tail);
    st.k_tail = kt.t.data_ptr(), st.k_tail_batch_stride = kt.outer, st.k_tail_token_stride = kt.inner, st.k_tail_slots = kt.t.size(2);
    st.v_tail = vt.t.data_ptr(), st.v_tail_batch_stride = vt.outer, st.v_tail_token_stride = vt.inner, st.v_tail_slots = vt.t.size(2);
    for (const OptTensor *t : {&k_len_dev, &v_len_dev})
        if (*t && ((*t)->scalar_type() != at::kLong || (*t)->numel() != 1 || !(*t)->is_cuda()))
            fail("a device-side tail length must be one int64 element on the GPU");
    if (k_len_dev) st.k_tail_len_dev = k_len_dev->data_ptr<int64_t>();
    else st.k_tail_len = k_len.value_or(st.k_tail_slots);
    if (v_len_dev) st.v_tail_len_dev = v_len_dev->data_ptr<int64_t>();
    else st.v_tail_len = v_len.value_or(st.v_tail_slots);
    const int64_t width = std::max(st.k_tokens + st.k_tail_slots, st.v_tokens + st.v_tail_slots);
    Tensor mask;
    if (mask_in) {
        mask = *mask_in;
        if (mask.scalar_type() != at::kFloat || mask.sizes() != c10::IntArrayRef({B, 1, 1, width}))
            fail("attention_mask must be fp32 of shape (" + std::to_string(B) + ", 1, 1, " + std::to_string(width) + ")");
        if (mask.stride(3) != 1) mask = mask.contiguous();
        st.mask = mask.data_ptr<float>(), st.mask_stride = B > 1 ? mask.stride(0) : width;
    }
    st.samples = B * nh, st.heads = (int)nh, st.heads_per_kv = (int)(nh / nkv), st.D = D;
    Tensor out = empty({B, nh, 1, D}, at::kHalf, q_in);
    st.out = out.data_ptr(), st.out_stride = D;
    if (single_pass) {
        if (!api.decode_attention_fused_supported(&st))
            fail("the single-pass attention step does not take this layout (head_dim 128, keys 1/2/4-bit or dense 3-bit group 32 or "
                 "reference 3-bit, values 1/2/4-bit or dense 3-bit group 32)");
        if (weights) {
            Tensor probs = empty({B, nh, 1, width}, at::kHalf, q_in);
            st.probs = probs.data_ptr(), st.probs_stride = width;
            const size_t bytes = api.decode_attention_fused_weights_workspace_bytes(&st);
            const Tensor ws = empty({(int64_t)bytes}, at::kByte, q_in);
            const c10::DeviceGuard guard(q_in.device());
            check(api.decode_attention_fused_weights(&st, ws.data_ptr(), bytes, stream_of(q_in)));
            return {out, probs};
        }
        const size_t bytes = api.decode_attention_fused_workspace_bytes(&st);
        const Tensor ws = empty({(int64_t)bytes}, at::kByte, q_in);
        const c10::DeviceGuard guard(q_in.device());
        check(api.decode_attention_fused(&st, ws.data_ptr(), bytes, stream_of(q_in)));
        return {out, std::nullopt};
    }
    Tensor probs = empty({B, nh, 1, width}, at::kHalf, q_in);
    st.probs = probs.data_ptr(), st.probs_stride = width;
    const size_t bytes = api.decode_attention_workspace_bytes(&st);
    const Tensor ws = scratch(bytes, q_in);
    const c10::DeviceGuard guard(q_in.device());
    check(api.decode_attention(&st, ws.defined() ? ws.data_ptr() : nullptr, bytes, stream_of(q_in)));
    return {out, probs};
}

// ---------------------------------------------------------------------------------------------------------------------
// projections of a decode step

// [..., n] fp16 as [rows, n] with unit-stride rows
Tensor rows2(const Tensor &t, const char *what)
{
    if (t.scalar_type() != at::kHalf) fail(std::string("expected scalar type Half for ") + what + " but found " + dtype_name(t));
    const Tensor r = t.reshape({-1, t.size(-1)});
    return r.stride(1) == 1 && r.stride(0) >= r.size(1) ? r : r.contiguous();
}

// ws: one stacked weight, cut into parts of `split` rows, or one weight per part
Tensor linear_operands(kvmix_linear_rows_t &st, const Tensor &x_in, const std::vector<Tensor> &ws, const std::vector<int64_t> &split, int epilogue,
                       const OptTensor &norm, double eps)
{
    const Tensor x = rows2(x_in, "x");
    need_gpu({&x});
    st.x = x.data_ptr(), st.m = x.size(0), st.k = x.size(1);
    st.x_stride = x.size(0) > 1 ? x.stride(0) : x.size(1);
    st.epilogue = epilogue;
    if (ws.empty() || ws.size() > 3) fail("a projection has one to three weights");
    auto row_stride = [](const Tensor &w) { return w.size(0) > 1 ? w.stride(0) : w.size(1); };  // (of one row: whatever the view left)
    for (const Tensor &w : ws) {
        need_with(x, {&w});
        if (w.scalar_type() != at::kHalf || w.dim() != 2 || w.size(1) != x.size(1) || w.stride(1) != 1 || row_stride(w) != row_stride(ws[0]))
            fail("weights must be fp16 [rows, k] with unit-stride rows and one row stride");
    }
    st.w_stride = row_stride(ws[0]);
    if (ws.size() == 1) {
        int64_t sum = 0;
        for (int64_t n : split) sum += n;
        if (sum != ws[0].size(0)) fail("the stacked weight must hold the rows of all its parts");
        const char *at = (const char *)ws[0].data_ptr();
        for (size_t j = 0; j < split.size(); j++) {
            st.w[j] = at, st.rows[j] = split[j];
            at += 2 * split[j] * st.w_stride;
        }
    } else {
        // (the epilogues place their outputs by `split`: rows beyond it would be written where no output was made for them)
        if (ws.size() != split.size()) fail("a projection in parts has one weight per part");
        for (size_t j = 0; j < ws.size(); j++) {
            if (ws[j].size(0) != split[j]) fail("each part's weight must hold the rows of that part");
            st.w[j] = ws[j].data_ptr(), st.rows[j] = split[j];
        }
    }
    if (norm) {
        need_with(x, {&*norm});
        if (norm->scalar_type() != at::kHalf || norm->numel() != x.size(1) || !norm->is_contiguous())
            fail("norm_weight must be k contiguous fp16 values");
        st.norm_weight = norm->data_ptr(), st.norm_eps = (float)eps;
    }
    return x;
}

void linear_launch(const kvmix_linear_rows_t &st, const Tensor &x)
{
    const c10::DeviceGuard guard(x.device());
    check(api.linear_rows(&st, stream_of(x)));
}

Tensor linear_output(const Tensor &x, int64_t n, c10::ScalarType type)
{
    std::vector<int64_t> sizes = x.sizes().vec();
    sizes.back() = n;
    return at::empty(sizes, x.options().dtype(type).requires_grad(false));
}

Tensor linear_rows(const Tensor &x_in, const Tensor &w, const OptTensor &norm, double eps, const OptTensor &residual_in, bool fp32)
{
    kvmix_linear_rows_t st{};
    if (w.dim() != 2) fail("weights must be fp16 [rows, k] with unit-stride rows and one row stride");
    if (residual_in && fp32) fail("a product with a residual is fp16: fp32 cannot be asked for with it");
    const int64_t n = w.size(0);
    const Tensor x = linear_operands(st, x_in, {w}, {n}, residual_in ? KVMIX_LINEAR_RESIDUAL : fp32 ? KVMIX_LINEAR_FLOAT : KVMIX_LINEAR_PLAIN, norm, eps);
    Tensor residual;
    if (residual_in) {
        residual = rows2(*residual_in, "residual");
        need_with(x, {&residual});
        if (residual.size(0) != x.size(0) || residual.size(1) != n) fail("residual must have the shape of the product");
        st.residual = residual.data_ptr(), st.residual_stride = residual.size(0) > 1 ? residual.stride(0) : n;
    }
    Tensor out = linear_output(x_in, n, fp32 ? at::kFloat : at::kHalf);
    st.out = out.data_ptr(), st.out_stride = n;
    linear_launch(st, x);
    return out;
}

Tensor swiglu_rows(const Tensor &x_in, const std::vector<Tensor> &ws, const OptTensor &norm, double eps)
{
    kvmix_linear_rows_t st{};
    if (ws.empty() || ws[0].dim() != 2) fail("weights must be fp16 [rows, k] with unit-stride rows and one row stride");
    const int64_t n = ws.size() > 1 ? ws[0].size(0) : ws[0].size(0) / 2;
    const Tensor x = linear_operands(st, x_in, ws, {n, n}, KVMIX_LINEAR_SWIGLU, norm, eps);
    Tensor out = linear_output(x_in, n, at::kHalf);
    st.out = out.data_ptr(), st.out_stride = n;
    linear_launch(st, x);
    return out;
}

Tensor qkv_rope_append(const Tensor &x_in, const std::vector<Tensor> &ws, int64_t heads, int64_t kv_heads, const Tensor &cos_in, const Tensor &sin_in,
                       const Tensor &k_tail, const Tensor &v_tail, int64_t k_slot, const OptTensor &k_slot_dev, int64_t v_slot,
                       const OptTensor &v_slot_dev, const OptTensor &norm, double eps)
{
    kvmix_linear_rows_t st{};
    const int64_t D = k_tail.size(-1);
    const Tensor x = linear_operands(st, x_in, ws, {heads * D, kv_heads * D, kv_heads * D}, KVMIX_LINEAR_ROPE_APPEND, norm, eps);
    const int64_t B = x.size(0);
    need_with(x, {&cos_in, &sin_in, &k_tail, &v_tail});
    for (const Tensor *t : {&cos_in, &sin_in})
        if (t->scalar_type() != at::kHalf || (t->numel() != D && t->numel() != B * D))
            fail("qkv_rope_append: cos and sin must hold head_dim fp16 values, shared or per sequence");
    const Tensor cos = cos_in.reshape({-1, D}).contiguous(), sin = sin_in.reshape({-1, D}).contiguous();
    if (cos.size(0) != sin.size(0)) fail("qkv_rope_append: cos and sin must have the same shape");
    st.cos = cos.data_ptr(), st.sin = sin.data_ptr(), st.cos_sin_batch_stride = cos.size(0) > 1 ? D : 0, st.head_dim = D;
    for (const Tensor *t : {&k_tail, &v_tail})
        if (t->scalar_type() != at::kHalf || t->dim() != 4 || t->size(0) != B || t->size(1) != kv_heads || t->size(3) != D || t->stride(3) != 1)
            fail("qkv_rope_append: tails must be fp16 [B, kv_heads, slots, D] with unit stride along D");
    for (const OptTensor *t : {&k_slot_dev, &v_slot_dev})
        if (*t && ((*t)->scalar_type() != at::kLong || (*t)->numel() != 1 || (*t)->device() != x.device()))
            fail("a device-side slot must be one int64 element on the GPU");
    // (strides of one-element dimensions are whatever the view left there)
    st.k_tail = k_tail.data_ptr(), st.k_tail_batch_stride = k_tail.stride(0), st.k_tail_head_stride = k_tail.stride(1);
    st.k_tail_token_stride = std::max(k_tail.stride(2), k_tail.size(2) > 1 ? 0 : D), st.k_tail_slots = k_tail.size(2);
    st.v_tail = v_tail.data_ptr(), st.v_tail_batch_stride = v_tail.stride(0), st.v_tail_head_stride = v_tail.stride(1);
    st.v_tail_token_stride = std::max(v_tail.stride(2), v_tail.size(2) > 1 ? 0 : D), st.v_tail_slots = v_tail.size(2);
    st.k_slot = k_slot, st.v_slot = v_slot;
    if (k_slot_dev) st.k_slot_dev = k_slot_dev->data_ptr<int64_t>();
    if (v_slot_dev) st.v_slot_dev = v_slot_dev->data_ptr<int64_t>();
    Tensor q = empty({B, heads, 1, D}, at::kHalf, x);
    st.out = q.data_ptr(), st.out_stride = heads * D;
    linear_launch(st, x);
    return q;
}

}  // namespace

PYBIND11_MODULE(_host, m)
{
    // Allocation and launch run without the interpreter's lock: a launch into a full queue waits, and other Python threads
    // go on meanwhile.
    using NoGil = py::call_guard<py::gil_scoped_release>;
    m.def("bind", &bind);
    m.def("quantize_pack_last_dim", &quantize_pack_last_dim, NoGil());
    m.def("quantize_pack_dense3", &quantize_pack_dense3, NoGil());
    m.def("append_keys", &append_keys, NoGil());
    m.def("append_values", &append_values, NoGil());
    m.def("copy_rows", &copy_rows, NoGil());
    m.def("grow_tuple", &grow_tuple, NoGil());
    m.def("quantized_gemm", &quantized_gemm, NoGil());
    m.def("prefer_single_pass", &prefer_single_pass, NoGil());
    m.def("decode_attention", &decode_attention, NoGil());
    m.def("linear_rows", &linear_rows, NoGil());
    m.def("swiglu_rows", &swiglu_rows, NoGil());
    m.def("qkv_rope_append", &qkv_rope_append, NoGil());
}
