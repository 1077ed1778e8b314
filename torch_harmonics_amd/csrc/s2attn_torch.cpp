// Thin libtorch binding of libs2attn.so: registers the attention operators under the reference's own names and schemas
//   attention_kernels::forward, backward, permute_to_nhwc, permute_to_nchw      (attention_interface.cpp:85-119)
// for the CUDA dispatch key (ROCm tensors dispatch there), plus the two entry points that hand the forward's output and
// softmax normaliser to the backward (s2attn_kernels::forward_lse, backward_saved; the reference recomputes both,
// attention_cuda_bwd.cu:856-956).  Everything here is host code: argument checks (the conditions of attention_cuda_fwd.cu:
// 553-570 and attention_cuda_bwd.cu:874-893), output allocation, the plan cache, and one call into the C ABI on torch's
// current stream.  There is no CPU implementation: CPU tensors are refused with a clear error.
//
// s2attn_kernels::module_attention is the whole NeighborhoodAttentionS2 layer (projections, q/k norm, attention, output projection)
// as ONE autograd node: twelve launches per training step (self-attention without q/k norm) and no Python between them, where the operator-by-operator form
// needs about forty and spends 0.8 ms of host time on them.
//
// Built by the Makefile next to it into torch_harmonics_amd/_C.so and loaded with torch.ops.load_library; the fake (meta)
// kernels and the autograd rules are registered from Python (torch_harmonics_amd/ops.py), as the reference does.

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/custom_class.h>
#include <torch/library.h>

#include <array>
#include <list>
#include <mutex>
#include <string>
#include <utility>
#include <tuple>
#include <vector>

#include "../../include/s2attn.h"

namespace {

using at::Tensor;

void check_rc(int64_t rc, const char *what)
{
    if (rc < 0) {
        const char *msg = s2attn_last_error();
        TORCH_CHECK(false, what, ": ", (msg && *msg) ? msg : "error");
    }
}

int dtype_code(at::ScalarType t)
{
    switch (t) {
    case at::kFloat: return S2ATTN_F32;
    case at::kBFloat16: return S2ATTN_BF16;
    case at::kHalf: return S2ATTN_F16;
    default: TORCH_CHECK(false, "unsupported dtype ", t); return -1;
    }
}

void require_gpu(const Tensor &t, const char *name, const c10::Device &dev)
{
    TORCH_CHECK(t.is_cuda(), name, " is on ", t.device(), "; the s2attn operators only run on a ROCm GPU (no CPU implementation is shipped)");
    TORCH_CHECK(t.device() == dev, name, " is on ", t.device(), " but the other operands are on ", dev);
}

// Activations are contiguous NHWC (the reference's contract) or a COLUMN BLOCK of a contiguous row-major buffer: unit
// channel stride, one point stride ld >= channels for the longitude axis, latitude and batch strides that follow from it.
// That is what a slice buf[..., c0:c1] of a fused q | k | v projection is; the library reads it in place.
// Returns 0 for a packed tensor, else ld; raises for anything else.
int64_t point_stride(const Tensor &t, const char *name)
{
    if (t.is_contiguous()) return 0;
    const int64_t ld = t.stride(2);
    const bool ok = t.stride(3) == 1 && ld >= t.size(3) && ld % 4 == 0 && t.stride(1) == t.size(2) * ld && t.stride(0) == t.size(1) * t.size(2) * ld
                    && t.storage_offset() % 4 == 0;
    TORCH_CHECK(ok, name, " must be contiguous, or a column block of a contiguous (B, nlat, nlon, width) buffer with width and offset multiples of 4");
    return ld;
}

// Same conditions the reference entry points enforce (attention_cuda_fwd.cu:553-570, attention_cuda_bwd.cu:874-893).
void validate(const Tensor &kx, const Tensor &vx, const Tensor &qy, const Tensor *dy, const Tensor &quad_weights, const Tensor &col_idx,
              const Tensor &row_off, int64_t num_heads, int64_t nlon_in, int64_t nlat_out, int64_t nlon_out)
{
    TORCH_CHECK(nlon_in > 0 && nlon_out > 0 && (nlon_in % nlon_out == 0 || nlon_out % nlon_in == 0), "either nlon_in (", nlon_in,
                ") must be an integer multiple of nlon_out (", nlon_out, "), or vice versa");
    TORCH_CHECK(num_heads >= 1, "num_heads must be positive, got ", num_heads);
    const Tensor *ts[] = {&kx, &vx, &qy, dy};
    const char *names[] = {"kx", "vx", "qy", "dy"};
    for (int i = 0; i < 4; i++) {
        if (!ts[i]) continue;
        TORCH_CHECK(ts[i]->dim() == 4, names[i], " must be a 4-dimensional (B, nlat, nlon, heads*channels) tensor, got ", ts[i]->dim(), " dimensions");
        (void)point_stride(*ts[i], names[i]);
    }
    TORCH_CHECK(qy.size(3) % num_heads == 0, "q/k channel count (", qy.size(3), ") must be divisible by num_heads (", num_heads, ")");
    TORCH_CHECK(vx.size(3) % num_heads == 0, "v channel count (", vx.size(3), ") must be divisible by num_heads (", num_heads, ")");
    TORCH_CHECK(kx.scalar_type() == qy.scalar_type(), "k dtype (", kx.scalar_type(), ") must match q dtype (", qy.scalar_type(), ")");
    TORCH_CHECK(vx.scalar_type() == qy.scalar_type(), "v dtype (", vx.scalar_type(), ") must match q dtype (", qy.scalar_type(), ")");
    if (dy) TORCH_CHECK(dy->scalar_type() == qy.scalar_type(), "dy dtype (", dy->scalar_type(), ") must match q dtype (", qy.scalar_type(), ")");
    TORCH_CHECK(kx.size(3) == qy.size(3), "k and q must have the same channel count, got ", kx.size(3), " and ", qy.size(3));
    TORCH_CHECK(kx.size(0) == vx.size(0) && kx.size(1) == vx.size(1) && kx.size(2) == vx.size(2) && kx.size(0) == qy.size(0),
                "k and v must share (B, nlat_in, nlon_in) and q must share B");
    TORCH_CHECK(kx.size(2) == nlon_in && qy.size(1) == nlat_out && qy.size(2) == nlon_out, "tensor extents do not match nlon_in=", nlon_in,
                ", nlat_out=", nlat_out, ", nlon_out=", nlon_out);
    if (dy)
        TORCH_CHECK(dy->size(0) == qy.size(0) && dy->size(1) == qy.size(1) && dy->size(2) == qy.size(2) && dy->size(3) == vx.size(3),
                    "dy must have the shape of the forward output");
    TORCH_CHECK(quad_weights.numel() == kx.size(1), "quad_weights must have nlat_in = ", kx.size(1), " entries, got ", quad_weights.numel());
    TORCH_CHECK(col_idx.scalar_type() == at::kLong && row_off.scalar_type() == at::kLong, "col_idx and row_off must be int64");
    const auto t = qy.scalar_type();
    TORCH_CHECK(t == at::kFloat || t == at::kBFloat16 || t == at::kHalf || t == at::kDouble, "unsupported dtype ", t);
    const auto dev = kx.device();
    require_gpu(kx, "kx", dev), require_gpu(vx, "vx", dev), require_gpu(qy, "qy", dev);
    if (dy) require_gpu(*dy, "dy", dev);
    require_gpu(quad_weights, "quad_weights", dev), require_gpu(col_idx, "col_idx", dev), require_gpu(row_off, "row_off", dev);
}

// ---- plans ------------------------------------------------------------------------------------------------------------
// The reference re-sorts the CSR rows on the device in every call (attention_cuda_utils.cu:74-113).  Here psi is turned into
// the library's run-length plan once, on the host, the first time a (col_idx, row_off) pair is seen (one device-to-host
// copy), and the device copy of the plan is kept.  An entry holds its index tensors, so their addresses cannot be recycled
// for another psi while it lives, and an in-place edit of either bumps its version counter and misses the cache.  A caller
// that built the plan ahead of time (the module does, in its constructor) passes it in and nothing is copied at all.
struct PlanEntry {
    const void *col = nullptr, *row = nullptr, *blob_ptr = nullptr;
    int64_t ncol = 0, nrow = 0;
    uint32_t vcol = 0, vrow = 0, vblob = 0;
    c10::Device device = c10::Device(c10::kCPU);
    int64_t ext[4] = {0, 0, 0, 0};
    Tensor blob, keep_col, keep_row;
    s2attn_plan plan = {};
};

std::mutex g_plan_mutex;
std::list<PlanEntry> g_plans; // most recently used first
constexpr size_t MAX_PLANS = 32;

uint32_t version_of(const Tensor &t) { return t.is_inference() ? 0u : t._version(); }

s2attn_plan plan_for(const Tensor &col_idx, const Tensor &row_off, int64_t nlat_in, int64_t nlon_in, int64_t nlat_out, int64_t nlon_out,
                     const c10::optional<Tensor> &blob, const c10::OptionalArrayRef<int64_t> &header)
{
    std::lock_guard<std::mutex> lock(g_plan_mutex);
    const bool given = blob.has_value() && blob->defined() && header.has_value();
    for (auto it = g_plans.begin(); it != g_plans.end(); ++it) {
        const bool hit = given ? (it->blob_ptr == blob->data_ptr() && it->vblob == version_of(*blob) && it->device == blob->device())
                               : (it->blob_ptr == nullptr && it->col == col_idx.data_ptr() && it->row == row_off.data_ptr() && it->ncol == col_idx.numel()
                                  && it->nrow == row_off.numel() && it->vcol == version_of(col_idx) && it->vrow == version_of(row_off)
                                  && it->device == col_idx.device());
        if (hit && it->ext[0] == nlat_in && it->ext[1] == nlon_in && it->ext[2] == nlat_out && it->ext[3] == nlon_out) {
            g_plans.splice(g_plans.begin(), g_plans, it);
            return g_plans.front().plan;
        }
    }
    PlanEntry e;
    e.ext[0] = nlat_in, e.ext[1] = nlon_in, e.ext[2] = nlat_out, e.ext[3] = nlon_out;
    if (given) {
        TORCH_CHECK(blob->scalar_type() == at::kInt && blob->is_contiguous() && (int64_t)header->size() == S2ATTN_PLAN_HEADER_INTS
                        && (*header)[S2ATTN_PH_MAGIC] == S2ATTN_PLAN_MAGIC && (*header)[S2ATTN_PH_TOTAL] == blob->numel(),
                    "plan header does not describe this plan tensor");
        TORCH_CHECK(blob->is_cuda() && blob->device() == col_idx.device(), "plan is on ", blob->device(), " but psi is on ", col_idx.device());
        e.blob = *blob;
        e.blob_ptr = blob->data_ptr();
        e.vblob = version_of(*blob);
        e.device = blob->device();
        for (int i = 0; i < S2ATTN_PLAN_HEADER_INTS; i++) e.plan.header[i] = (int32_t)(*header)[i];
    } else {
        const bool up = nlon_out % nlon_in == 0 && nlon_out != nlon_in;
        const int64_t want = (up ? nlat_in : nlat_out) + 1;
        TORCH_CHECK(row_off.numel() == want, "row_off must have ", up ? "nlat_in" : "nlat_out", " + 1 = ", want, " entries, got ", row_off.numel());
        const Tensor ci = col_idx.detach().to(at::kCPU).contiguous(), ro = row_off.detach().to(at::kCPU).contiguous();
        const int64_t n = s2attn_plan_size(ci.data_ptr<int64_t>(), ro.data_ptr<int64_t>(), ci.numel(), (int)nlat_in, (int)nlon_in, (int)nlat_out, (int)nlon_out);
        check_rc(n, "s2attn_plan_size");
        Tensor host = at::empty({n}, at::TensorOptions().dtype(at::kInt));
        check_rc(s2attn_plan_build(ci.data_ptr<int64_t>(), ro.data_ptr<int64_t>(), ci.numel(), (int)nlat_in, (int)nlon_in, (int)nlat_out, (int)nlon_out,
                                   host.data_ptr<int32_t>(), n),
                 "s2attn_plan_build");
        std::copy(host.data_ptr<int32_t>(), host.data_ptr<int32_t>() + S2ATTN_PLAN_HEADER_INTS, e.plan.header);
        e.blob = host.to(col_idx.device());
        e.col = col_idx.data_ptr(), e.row = row_off.data_ptr(), e.ncol = col_idx.numel(), e.nrow = row_off.numel();
        e.vcol = version_of(col_idx), e.vrow = version_of(row_off), e.device = col_idx.device();
        e.keep_col = col_idx, e.keep_row = row_off;
    }
    e.plan.data = e.blob.data_ptr<int32_t>();
    g_plans.push_front(std::move(e));
    while (g_plans.size() > MAX_PLANS) g_plans.pop_back();
    return g_plans.front().plan;
}

s2attn_shape shape_of(const Tensor &kx, const Tensor &vx, const Tensor &qy, int64_t num_heads)
{
    s2attn_shape sh = {};
    sh.ld_k = (int)point_stride(kx, "kx"), sh.ld_v = (int)point_stride(vx, "vx"), sh.ld_q = (int)point_stride(qy, "qy");
    sh.batch = (int)kx.size(0), sh.num_heads = (int)num_heads;
    sh.nlat_in = (int)kx.size(1), sh.nlon_in = (int)kx.size(2), sh.nlat_out = (int)qy.size(1), sh.nlon_out = (int)qy.size(2);
    sh.ck = (int)(kx.size(3) / num_heads), sh.cv = (int)(vx.size(3) / num_heads);
    sh.dtype = dtype_code(qy.scalar_type());
    return sh;
}

void *current_stream(const c10::Device &dev) { return static_cast<void *>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream()); }

// ---- forward ------------------------------------------------------------------------------------------------------------
std::tuple<Tensor, Tensor> forward_impl(const Tensor &kx, const Tensor &vx, const Tensor &qy, const Tensor &quad_weights, const Tensor &col_idx,
                                        const Tensor &row_off, int64_t num_heads, int64_t nlon_in, int64_t nlat_out, int64_t nlon_out, bool with_lse,
                                        const c10::optional<Tensor> &plan_blob, const c10::OptionalArrayRef<int64_t> &plan_header)
{
    validate(kx, vx, qy, nullptr, quad_weights, col_idx, row_off, num_heads, nlon_in, nlat_out, nlon_out);
    if (qy.scalar_type() == at::kDouble) { // stored as fp64, computed in fp32 like the reference (attention_cuda_utils.cuh:185-190)
        auto r = forward_impl(kx.to(at::kFloat), vx.to(at::kFloat), qy.to(at::kFloat), quad_weights, col_idx, row_off, num_heads, nlon_in, nlat_out,
                              nlon_out, with_lse, plan_blob, plan_header);
        return {std::get<0>(r).to(at::kDouble), std::get<1>(r)};
    }
    Tensor y = at::empty({kx.size(0), nlat_out, nlon_out, vx.size(3)}, kx.options());
    Tensor lse = with_lse ? at::empty({kx.size(0), num_heads, nlat_out, nlon_out}, kx.options().dtype(at::kFloat)) : at::empty({0}, kx.options().dtype(at::kFloat));
    if (y.numel() == 0) return {y, lse};
    const s2attn_plan plan = plan_for(col_idx, row_off, kx.size(1), nlon_in, nlat_out, nlon_out, plan_blob, plan_header);
    const s2attn_shape sh = shape_of(kx, vx, qy, num_heads);
    const Tensor qw = quad_weights.to(at::kFloat).contiguous();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(kx.device());
    check_rc(s2attn_forward_lse(kx.data_ptr(), vx.data_ptr(), qy.data_ptr(), qw.data_ptr<float>(), y.data_ptr(), with_lse ? lse.data_ptr<float>() : nullptr,
                                &plan, &sh, current_stream(kx.device())),
             "s2attn_forward_lse");
    return {y, lse};
}

Tensor forward(const Tensor &kx, const Tensor &vx, const Tensor &qy, const Tensor &quad_weights, const Tensor &col_idx, const Tensor &row_off,
               int64_t num_heads, int64_t nlon_in, int64_t nlat_out, int64_t nlon_out)
{
    return std::get<0>(forward_impl(kx, vx, qy, quad_weights, col_idx, row_off, num_heads, nlon_in, nlat_out, nlon_out, false, c10::nullopt, c10::nullopt));
}

std::tuple<Tensor, Tensor> forward_lse(const Tensor &kx, const Tensor &vx, const Tensor &qy, const Tensor &quad_weights, const Tensor &col_idx,
                                       const Tensor &row_off, int64_t num_heads, int64_t nlon_in, int64_t nlat_out, int64_t nlon_out,
                                       const c10::optional<Tensor> &plan, c10::OptionalArrayRef<int64_t> plan_header)
{
    return forward_impl(kx, vx, qy, quad_weights, col_idx, row_off, num_heads, nlon_in, nlat_out, nlon_out, true, plan, plan_header);
}

// ---- backward -----------------------------------------------------------------------------------------------------------
std::tuple<Tensor, Tensor, Tensor> backward_impl(const Tensor &kx, const Tensor &vx, const Tensor &qy, const Tensor &dy, const Tensor *y, const Tensor *lse,
                                                 const Tensor &quad_weights, const Tensor &col_idx, const Tensor &row_off, int64_t num_heads,
                                                 int64_t nlon_in, int64_t nlat_out, int64_t nlon_out, const c10::optional<Tensor> &plan_blob,
                                                 const c10::OptionalArrayRef<int64_t> &plan_header)
{
    validate(kx, vx, qy, &dy, quad_weights, col_idx, row_off, num_heads, nlon_in, nlat_out, nlon_out);
    const bool saved = y != nullptr;
    if (saved) {
        require_gpu(*y, "y", kx.device()), require_gpu(*lse, "lse", kx.device());
        TORCH_CHECK(y->sizes() == dy.sizes() && y->scalar_type() == dy.scalar_type(), "y must be the forward output (shape and dtype of dy)");
        (void)point_stride(*y, "y");
        TORCH_CHECK(lse->dim() == 4 && lse->size(0) == kx.size(0) && lse->size(1) == num_heads && lse->size(2) == nlat_out && lse->size(3) == nlon_out
                        && lse->scalar_type() == at::kFloat && lse->is_contiguous(),
                    "lse must be the contiguous fp32 (B, num_heads, nlat_out, nlon_out) tensor returned by forward_lse");
    }
    if (qy.scalar_type() == at::kDouble) {
        const Tensor yf = saved ? y->to(at::kFloat) : Tensor();
        auto r = backward_impl(kx.to(at::kFloat), vx.to(at::kFloat), qy.to(at::kFloat), dy.to(at::kFloat), saved ? &yf : nullptr, lse, quad_weights, col_idx,
                               row_off, num_heads, nlon_in, nlat_out, nlon_out, plan_blob, plan_header);
        return {std::get<0>(r).to(at::kDouble), std::get<1>(r).to(at::kDouble), std::get<2>(r).to(at::kDouble)};
    }
    // Gradients mirror the layout of their tensors: k | v (| q) that are column blocks of ONE buffer get their gradients as the
    // same column blocks of ONE new buffer, so that the caller's input gradient is a single GEMM over it.
    Tensor dk, dv, dq;
    const int64_t ldk = point_stride(kx, "kx"), ldv = point_stride(vx, "vx"), ldq = point_stride(qy, "qy");
    // (the column ranges must lie inside one row of the buffer and be pairwise disjoint: k and v given as the same or overlapping
    // slices would otherwise have their gradients written to the same addresses)
    auto cols = [](const Tensor &t, int64_t ld) { return std::pair<int64_t, int64_t>(t.storage_offset() % ld, t.storage_offset() % ld + t.size(3)); };
    auto disjoint = [](std::pair<int64_t, int64_t> a, std::pair<int64_t, int64_t> b) { return a.second <= b.first || b.second <= a.first; };
    bool kv_fused = ldk > 0 && ldk == ldv && kx.storage().is_alias_of(vx.storage()) && kx.storage_offset() / ldk == vx.storage_offset() / ldk;
    if (kv_fused) kv_fused = cols(kx, ldk).second <= ldk && cols(vx, ldk).second <= ldk && disjoint(cols(kx, ldk), cols(vx, ldk));
    bool all_fused = kv_fused && ldq == ldk && qy.storage().is_alias_of(kx.storage()) && qy.sizes().slice(0, 3) == kx.sizes().slice(0, 3)
                     && qy.storage_offset() / ldk == kx.storage_offset() / ldk;
    if (all_fused) all_fused = cols(qy, ldk).second <= ldk && disjoint(cols(qy, ldk), cols(kx, ldk)) && disjoint(cols(qy, ldk), cols(vx, ldk));
    if (kv_fused) {
        Tensor buf = at::empty({kx.size(0), kx.size(1), kx.size(2), ldk}, kx.options());
        const int64_t used = kx.size(3) + vx.size(3) + (all_fused ? qy.size(3) : 0);
        if (used != ldk) buf.zero_(); // columns of the buffer that belong to none of the three
        dk = buf.narrow(3, kx.storage_offset() % ldk, kx.size(3));
        dv = buf.narrow(3, vx.storage_offset() % ldk, vx.size(3));
        dq = all_fused ? buf.narrow(3, qy.storage_offset() % ldk, qy.size(3)) : at::empty(qy.sizes(), qy.options());
    } else {
        dk = at::empty(kx.sizes(), kx.options()), dv = at::empty(vx.sizes(), vx.options()), dq = at::empty(qy.sizes(), qy.options());
    }
    if (qy.numel() == 0 || kx.numel() == 0) return {dk.zero_(), dv.zero_(), dq.zero_()};
    const s2attn_plan plan = plan_for(col_idx, row_off, kx.size(1), nlon_in, nlat_out, nlon_out, plan_blob, plan_header);
    s2attn_shape sh = shape_of(kx, vx, qy, num_heads);
    sh.ld_dy = (int)point_stride(dy, "dy"), sh.ld_y = saved ? (int)point_stride(*y, "y") : 0;
    sh.ld_dk = (int)point_stride(dk, "dk"), sh.ld_dv = (int)point_stride(dv, "dv"), sh.ld_dq = (int)point_stride(dq, "dq");
    // the backward that is handed y and lse needs the two statistics per point only; the other one also recomputes y and lse
    const int64_t nbytes = saved ? s2attn_backward_saved_workspace_bytes(&sh) : s2attn_backward_workspace_bytes(&sh);
    check_rc(nbytes, "s2attn_backward_workspace_bytes");
    Tensor ws = at::empty({(nbytes + 3) / 4}, kx.options().dtype(at::kFloat));
    const Tensor qw = quad_weights.to(at::kFloat).contiguous();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(kx.device());
    void *stream = current_stream(kx.device());
    if (saved)
        check_rc(s2attn_backward_saved(kx.data_ptr(), vx.data_ptr(), qy.data_ptr(), dy.data_ptr(), y->data_ptr(), lse->data_ptr<float>(), qw.data_ptr<float>(),
                                       dk.data_ptr(), dv.data_ptr(), dq.data_ptr(), ws.data_ptr(), &plan, &sh, stream),
                 "s2attn_backward_saved");
    else
        check_rc(s2attn_backward(kx.data_ptr(), vx.data_ptr(), qy.data_ptr(), dy.data_ptr(), qw.data_ptr<float>(), dk.data_ptr(), dv.data_ptr(), dq.data_ptr(),
                                 ws.data_ptr(), &plan, &sh, stream),
                 "s2attn_backward");
    return {dk, dv, dq};
}

std::tuple<Tensor, Tensor, Tensor> backward(const Tensor &kx, const Tensor &vx, const Tensor &qy, const Tensor &dy, const Tensor &quad_weights,
                                            const Tensor &col_idx, const Tensor &row_off, int64_t num_heads, int64_t nlon_in, int64_t nlat_out,
                                            int64_t nlon_out)
{
    return backward_impl(kx, vx, qy, dy, nullptr, nullptr, quad_weights, col_idx, row_off, num_heads, nlon_in, nlat_out, nlon_out, c10::nullopt, c10::nullopt);
}

std::tuple<Tensor, Tensor, Tensor> backward_saved(const Tensor &kx, const Tensor &vx, const Tensor &qy, const Tensor &dy, const Tensor &y, const Tensor &lse,
                                                  const Tensor &quad_weights, const Tensor &col_idx, const Tensor &row_off, int64_t num_heads,
                                                  int64_t nlon_in, int64_t nlat_out, int64_t nlon_out, const c10::optional<Tensor> &plan,
                                                  c10::OptionalArrayRef<int64_t> plan_header)
{
    return backward_impl(kx, vx, qy, dy, &y, &lse, quad_weights, col_idx, row_off, num_heads, nlon_in, nlat_out, nlon_out, plan, plan_header);
}

// ---- the module as one autograd node ----------------------------------------------------------------------------------------
struct LayerConfig {
    int64_t num_heads = 1, nlat_in = 0, nlon_in = 0, nlat_out = 0, nlon_out = 0;
    double scale = 1.0;
    at::ScalarType compute = at::kFloat; // element type of q, k, v, y and of the result
    std::vector<int64_t> plan_header;
};

constexpr float RMS_EPS = 1.1920928955078125e-7f; // F.rms_norm's default: the fp32 machine epsilon, for 16-bit inputs too

int blocks64(int64_t c) { return (int)((c + 63) / 64); }
void *at_byte(const Tensor &t, int64_t ofs) { return static_cast<char *>(t.data_ptr()) + ofs; }

// Packed weights of several matrices in one allocation (see include/s2attn.h).
struct Packer {
    int compute;
    std::vector<s2attn_pack_job> jobs;
    std::vector<int64_t> at; // byte offsets of weights and bias inside the allocation, per job
    int64_t bytes = 0;
    explicit Packer(int c) : compute(c) {}
    int k16(int64_t cols) const { return s2attn_pack_k16((int)cols, compute); }
    int64_t reserve(int blocks, int k16s)
    {
        const int64_t o = bytes;
        bytes += (s2attn_pack_bytes(blocks, k16s, compute) + 255) / 256 * 256;
        return o;
    }
    int64_t reserve_bias(int blocks)
    {
        const int64_t o = bytes;
        bytes += (int64_t)blocks * 256;
        return o;
    }
    // w: [rows, cols] or, transposed, [cols, rows]
    void add(const Tensor &w, const Tensor &bias, int64_t rows, int64_t cols, bool transposed, double scale, int64_t ofs, int64_t bias_ofs, int block, int first_k16, int total_k16)
    {
        s2attn_pack_job j = {};
        j.w = w.data_ptr(), j.bias = bias.defined() ? bias.data_ptr() : nullptr;
        j.rows = (int)rows, j.cols = (int)cols, j.dtype = dtype_code(w.scalar_type());
        j.row_stride = transposed ? 1 : cols, j.col_stride = transposed ? rows : 1;
        j.first_block = block, j.first_k16 = first_k16, j.total_k16 = total_k16, j.scale = (float)scale;
        jobs.push_back(j), at.push_back(ofs), at.push_back(bias_ofs);
    }
    Tensor run(const Tensor &like, void *stream)
    {
        Tensor buf = at::empty({bytes}, like.options().dtype(at::kByte));
        for (size_t i = 0; i < jobs.size(); i++) {
            jobs[i].dst = at_byte(buf, at[2 * i]);
            jobs[i].dst_bias = at[2 * i + 1] >= 0 ? static_cast<float *>(at_byte(buf, at[2 * i + 1])) : nullptr;
        }
        check_rc(s2attn_pack_weights(jobs.data(), (int)jobs.size(), compute, stream), "s2attn_pack_weights");
        return buf;
    }
};

struct Part {
    const Tensor *t;
    int64_t channels;
};

// One projection launch: NCHW source -> NHWC destinations (to_nhwc) or NHWC sources -> NCHW destination.
void project(bool to_nhwc, const std::vector<Part> &src, const std::vector<Part> &dst, int64_t batch, int64_t points, int compute, const void *packed,
             const void *bias, void *stream)
{
    s2attn_proj p = {};
    p.batch = (int)batch, p.points = points, p.nsrc = (int)src.size(), p.ndst = (int)dst.size();
    p.src_dtype = dtype_code(src[0].t->scalar_type()), p.dst_dtype = dtype_code(dst[0].t->scalar_type()), p.compute = compute;
    for (size_t i = 0; i < src.size(); i++) p.src[i] = src[i].t->data_ptr(), p.src_channels[i] = (int)src[i].channels;
    for (size_t i = 0; i < dst.size(); i++) p.dst[i] = dst[i].t->data_ptr(), p.dst_channels[i] = (int)dst[i].channels;
    p.packed = packed, p.bias = static_cast<const float *>(bias);
    check_rc(to_nhwc ? s2attn_proj_nchw_to_nhwc(&p, stream) : s2attn_proj_nhwc_to_nchw(&p, stream), "s2attn_proj");
}

// Weight and bias gradients: partial sums now, all final sums of the backward in one launch at its end.
struct Gradients {
    void *stream;
    std::vector<s2attn_finish_job> jobs;
    std::vector<Tensor> keep;
    void job(const float *part, Tensor &out, int64_t slices, int64_t slice_stride, int64_t rows, int64_t cols, int64_t rs, int64_t cs, double scale)
    {
        s2attn_finish_job j = {};
        j.part = part, j.out = out.data_ptr(), j.slice_stride = slice_stride, j.row_stride = rs, j.col_stride = cs;
        j.slices = (int)slices, j.rows = (int)rows, j.cols = (int)cols, j.dtype = dtype_code(out.scalar_type()), j.scale = (float)scale;
        jobs.push_back(j);
    }
    // cm [B, ci, points], pm_p [B, points, c_p]; returns the partials of pm x cm, pm and cm (the latter two undefined if not wanted)
    std::tuple<Tensor, Tensor, Tensor, int64_t> partials(const Tensor &cm, int64_t ci, const std::vector<Part> &pm, int64_t batch, int64_t points, int compute, bool want_cm, bool want_pm)
    {
        s2attn_grad g = {};
        g.batch = (int)batch, g.points = points, g.npm = (int)pm.size(), g.compute = compute;
        g.cm = cm.data_ptr(), g.cm_channels = (int)ci, g.cm_dtype = dtype_code(cm.scalar_type()), g.pm_dtype = dtype_code(pm[0].t->scalar_type());
        int64_t cj = 0;
        for (size_t i = 0; i < pm.size(); i++) g.pm[i] = pm[i].t->data_ptr(), g.pm_channels[i] = (int)pm[i].channels, cj += pm[i].channels;
        const int64_t slices = s2attn_grad_slices(&g);
        check_rc(slices, "s2attn_grad_slices");
        const auto opt = cm.options().dtype(at::kFloat);
        Tensor part = at::empty({slices * cj * ci}, opt), sc, sp;
        if (want_cm) sc = at::empty({slices * ci}, opt);
        if (want_pm) sp = at::empty({slices * cj}, opt);
        g.part = part.data_ptr<float>(), g.part_cm = want_cm ? sc.data_ptr<float>() : nullptr, g.part_pm = want_pm ? sp.data_ptr<float>() : nullptr;
        check_rc(s2attn_grad_partials(&g, stream), "s2attn_grad_partials");
        keep.push_back(part), keep.push_back(sc), keep.push_back(sp);
        return {part, sc, sp, slices};
    }
    void finish()
    {
        if (!jobs.empty()) check_rc(s2attn_finish(jobs.data(), (int)jobs.size(), stream), "s2attn_finish");
    }
};

Tensor dense(const Tensor &t) { return t.defined() ? t.contiguous() : t; }

// Tensor arguments of the layer
enum { XQ, XK, XV, WQ, WK, WV, WP, BQ, BK, BV, BP, NQ, NK, QUAD, COL, ROW, PLAN, NTENSORS };

struct LayerState : torch::CustomClassHolder {
    LayerConfig cfg;
    int slot[NTENSORS]; // position among the tensors given to the node, -1: absent
};

// Which of q, k, v are made from an input: query (B, C, nlat_out, nlon_out), key and value (B, C, nlat_in, nlon_in); an absent
// key is the query, an absent value the key.
struct Source {
    int x;             // XQ, XK or XV
    int first, count;  // of q (0), k (1), v (2)
};
std::vector<Source> sources(bool has_key, bool has_value)
{
    if (!has_key) return has_value ? std::vector<Source>{{XQ, 0, 2}, {XV, 2, 1}} : std::vector<Source>{{XQ, 0, 3}};
    return has_value ? std::vector<Source>{{XQ, 0, 1}, {XK, 1, 1}, {XV, 2, 1}} : std::vector<Source>{{XQ, 0, 1}, {XK, 1, 2}};
}

// Kept for the backward: the inputs (NCHW, as they came), q, k, v (and q, k before their norm), y and the softmax normaliser.
enum { S_Q = NTENSORS, S_K, S_V, S_QRAW, S_KRAW, S_Y, S_LSE, NSAVED };

constexpr int NKEPT = NSAVED - NTENSORS;
constexpr int NGRADS = NK + 1; // tensor arguments that may need a gradient

// The result, and in kept[] what S_Q ... S_LSE name (undefined where there is none; nothing without `keep`).
Tensor layer_forward(const Tensor (&given)[NTENSORS], const LayerConfig &cfg, bool keep, Tensor (&kept)[NKEPT])
{
    Tensor t[NTENSORS];
    for (int i = 0; i < NTENSORS; i++)
        if (given[i].defined()) t[i] = given[i].contiguous();
    const int64_t B = t[XQ].size(0), C = t[XQ].size(1), nh = cfg.num_heads, Ck = t[WQ].size(0), Cv = t[WV].size(0);
    const int64_t Po = cfg.nlat_out * cfg.nlon_out, Pi = cfg.nlat_in * cfg.nlon_in;
    const bool normed = t[NQ].defined();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(t[XQ].device());
    void *stream = current_stream(t[XQ].device());
    const auto opt = t[XQ].options().dtype(cfg.compute);
    const int comp = dtype_code(cfg.compute);

    // weights in operand order: q | k | v below each other, and the output projection
    Packer pk(comp);
    const int64_t ch[3] = {Ck, Ck, Cv};
    const int kin = pk.k16(C), first[4] = {0, blocks64(Ck), 2 * blocks64(Ck), 2 * blocks64(Ck) + blocks64(Cv)};
    const int64_t w_ofs = pk.reserve(first[3], kin), b_ofs = t[BQ].defined() ? pk.reserve_bias(first[3]) : -1;
    for (int i = 0; i < 3; i++) pk.add(t[WQ + i], t[BQ + i], ch[i], C, false, i == 0 && !normed ? cfg.scale : 1.0, w_ofs, b_ofs, first[i], 0, kin);
    const int64_t p_ofs = pk.reserve(blocks64(Cv), pk.k16(Cv)), pb_ofs = t[BP].defined() ? pk.reserve_bias(blocks64(Cv)) : -1;
    pk.add(t[WP], t[BP], Cv, Cv, false, 1.0, p_ofs, pb_ofs, 0, 0, pk.k16(Cv));
    const Tensor packed = pk.run(t[XQ], stream);

    Tensor qkv[3] = {at::empty({B, cfg.nlat_out, cfg.nlon_out, Ck}, opt), at::empty({B, cfg.nlat_in, cfg.nlon_in, Ck}, opt),
                     at::empty({B, cfg.nlat_in, cfg.nlon_in, Cv}, opt)};
    const int64_t block_bytes = s2attn_pack_bytes(1, kin, comp);
    for (const Source &s : sources(t[XK].defined(), t[XV].defined())) {
        std::vector<Part> dst;
        for (int i = s.first; i < s.first + s.count; i++) dst.push_back({&qkv[i], ch[i]});
        project(true, {{&t[s.x], C}}, dst, B, s.x == XQ ? Po : Pi, comp, at_byte(packed, w_ofs + first[s.first] * block_bytes),
                b_ofs >= 0 ? at_byte(packed, b_ofs + first[s.first] * 256) : nullptr, stream);
    }
    Tensor raw[2];
    if (normed) {
        s2attn_norm n = {};
        n.ntensors = 2, n.head_channels = (int)(Ck / nh), n.dtype = comp, n.gain_dtype = dtype_code(t[NQ].scalar_type()), n.eps = RMS_EPS;
        n.blocks = 2048;
        for (int i = 0; i < 2; i++) {
            raw[i] = qkv[i];
            if (keep) qkv[i] = at::empty_like(raw[i]); // else in place
            n.x[i] = raw[i].data_ptr(), n.y[i] = qkv[i].data_ptr(), n.gain[i] = t[NQ + i].data_ptr(), n.mult[i] = i ? 1.f : (float)cfg.scale;
            n.rows[i] = B * (i ? Pi : Po) * nh;
        }
        check_rc(s2attn_head_norm(&n, stream), "s2attn_head_norm");
    }

    auto [y, lse] = forward_impl(qkv[1], qkv[2], qkv[0], t[QUAD], t[COL], t[ROW], nh, cfg.nlon_in, cfg.nlat_out, cfg.nlon_out, keep, t[PLAN],
                                 c10::OptionalArrayRef<int64_t>(cfg.plan_header));
    Tensor out = at::empty({B, Cv, cfg.nlat_out, cfg.nlon_out}, opt);
    project(false, {{&y, Cv}}, {{&out, Cv}}, B, Po, comp, at_byte(packed, p_ofs), pb_ofs >= 0 ? at_byte(packed, pb_ofs) : nullptr, stream);

    if (keep) {
        for (int i = 0; i < 3; i++) kept[S_Q - NTENSORS + i] = qkv[i];
        kept[S_QRAW - NTENSORS] = raw[0], kept[S_KRAW - NTENSORS] = raw[1], kept[S_Y - NTENSORS] = y, kept[S_LSE - NTENSORS] = lse;
    }
    return out;
}

// Gradients of the arguments that need one; t: the contiguous arguments (biases are not looked at) followed by what was kept.
void layer_backward(const Tensor &grad, const Tensor *t, const LayerConfig &cfg, const std::array<bool, NGRADS> &needed, Tensor (&result)[NGRADS])
{
    auto need = [&](int i) { return needed[i]; };
    auto give = [&](int i, const Tensor &g) { result[i] = g; };
    const int64_t B = t[XQ].size(0), C = t[XQ].size(1), nh = cfg.num_heads, Ck = t[WQ].size(0), Cv = t[WV].size(0);
    const int64_t Po = cfg.nlat_out * cfg.nlon_out, Pi = cfg.nlat_in * cfg.nlon_in;
    const bool normed = t[NQ].defined();
    c10::hip::HIPGuardMasqueradingAsCUDA guard(t[XQ].device());
    void *stream = current_stream(t[XQ].device());
    const auto opt = t[XQ].options().dtype(cfg.compute);
    const int comp = dtype_code(cfg.compute);
    const Tensor g = grad.contiguous();
    const auto srcs = sources(t[XK].defined(), t[XV].defined());
    const int64_t ch[3] = {Ck, Ck, Cv};
    bool through = false; // does anything ahead of the output projection need a gradient?
    for (int i : {XQ, XK, XV, WQ, WK, WV, BQ, BK, BV, NQ, NK}) through |= need(i);

    // transposed weights: of the output projection; of each input's projections, next to each other along the columns
    Packer pk(comp);
    int64_t p_ofs = 0, x_ofs[3] = {0, 0, 0};
    if (through) {
        p_ofs = pk.reserve(blocks64(Cv), pk.k16(Cv));
        pk.add(t[WP], Tensor(), Cv, Cv, true, 1.0, p_ofs, -1, 0, 0, pk.k16(Cv));
        for (size_t j = 0; j < srcs.size(); j++) {
            if (!need(srcs[j].x)) continue;
            int total = 0, at = 0;
            for (int i = srcs[j].first; i < srcs[j].first + srcs[j].count; i++) total += pk.k16(ch[i]);
            x_ofs[j] = pk.reserve(blocks64(C), total);
            for (int i = srcs[j].first; i < srcs[j].first + srcs[j].count; i++) {
                pk.add(t[WQ + i], Tensor(), C, ch[i], true, i == 0 && !normed ? cfg.scale : 1.0, x_ofs[j], -1, 0, at, total);
                at += pk.k16(ch[i]);
            }
        }
    }
    const Tensor packed = through ? pk.run(t[XQ], stream) : Tensor();

    Gradients gr{stream, {}, {}};
    if (need(WP) || need(BP)) { // rows of the partial sums are y's channels, columns the gradient's
        auto [part, sums, none, slices] = gr.partials(g, Cv, {{&t[S_Y], Cv}}, B, Po, comp, need(BP), false);
        if (need(WP)) {
            Tensor w = at::empty(t[WP].sizes(), t[WP].options());
            gr.job(part.data_ptr<float>(), w, slices, Cv * Cv, Cv, Cv, 1, Cv, 1.0);
            give(WP, w);
        }
        if (need(BP)) {
            Tensor b = at::empty({Cv}, t[WP].options());
            gr.job(sums.data_ptr<float>(), b, slices, Cv, 1, Cv, 0, 1, 1.0);
            give(BP, b);
        }
    }
    if (through) {
        Tensor gy = at::empty(t[S_Y].sizes(), opt);
        project(true, {{&g, Cv}}, {{&gy, Cv}}, B, Po, comp, at_byte(packed, p_ofs), nullptr, stream);
        const auto [dk, dv, dq] = backward_impl(t[S_K], t[S_V], t[S_Q], gy, &t[S_Y], &t[S_LSE], t[QUAD], t[COL], t[ROW], nh, cfg.nlon_in, cfg.nlat_out,
                                                cfg.nlon_out, t[PLAN], c10::OptionalArrayRef<int64_t>(cfg.plan_header));
        const Tensor *d[3] = {&dq, &dk, &dv};
        if (normed) { // the gradients of the normed q and k become those of the projected ones, in place
            s2attn_norm n = {};
            n.ntensors = 2, n.head_channels = (int)(Ck / nh), n.dtype = comp, n.gain_dtype = dtype_code(t[NQ].scalar_type()), n.eps = RMS_EPS;
            n.blocks = 1024;
            for (int i = 0; i < 2; i++) {
                const Tensor part = at::empty({n.blocks * n.head_channels}, opt.dtype(at::kFloat));
                gr.keep.push_back(part);
                n.x[i] = t[S_QRAW + i].data_ptr(), n.y[i] = d[i]->data_ptr(), n.gain[i] = t[NQ + i].data_ptr(), n.mult[i] = i ? 1.f : (float)cfg.scale;
                n.dgain[i] = part.data_ptr<float>(), n.rows[i] = B * (i ? Pi : Po) * nh;
                if (need(NQ + i)) {
                    Tensor w = at::empty(t[NQ + i].sizes(), t[NQ + i].options());
                    gr.job(part.data_ptr<float>(), w, n.blocks, n.head_channels, 1, n.head_channels, 0, 1, n.mult[i]);
                    give(NQ + i, w);
                }
            }
            check_rc(s2attn_head_norm_backward(&n, stream), "s2attn_head_norm_backward");
        }
        for (size_t j = 0; j < srcs.size(); j++) {
            const Source &s = srcs[j];
            const int64_t points = s.x == XQ ? Po : Pi;
            std::vector<Part> parts;
            bool want_w = false, want_b = false;
            int64_t cj = 0;
            for (int i = s.first; i < s.first + s.count; i++) {
                parts.push_back({d[i], ch[i]});
                want_w |= need(WQ + i), want_b |= need(BQ + i), cj += ch[i];
            }
            if (need(s.x)) {
                Tensor dx = at::empty_like(t[s.x]);
                project(false, parts, {{&dx, C}}, B, points, comp, at_byte(packed, x_ofs[j]), nullptr, stream);
                give(s.x, dx);
            }
            if (!want_w && !want_b) continue;
            auto [part, none, sums, slices] = gr.partials(t[s.x], C, parts, B, points, comp, false, want_b);
            int64_t at = 0;
            for (int i = s.first; i < s.first + s.count; i++) {
                const double scale = i == 0 && !normed ? cfg.scale : 1.0;
                if (need(WQ + i)) {
                    Tensor w = at::empty(t[WQ + i].sizes(), t[WQ + i].options());
                    gr.job(part.data_ptr<float>() + at * C, w, slices, cj * C, ch[i], C, C, 1, scale);
                    give(WQ + i, w);
                }
                if (need(BQ + i)) {
                    Tensor b = at::empty({ch[i]}, t[WQ + i].options());
                    gr.job(sums.data_ptr<float>() + at, b, slices, cj, 1, ch[i], 0, 1, scale);
                    give(BQ + i, b);
                }
                at += ch[i];
            }
        }
    }
    gr.finish();
}

#define LAYER_ARGS                                                                                                                                             \
    const Tensor &query, const c10::optional<Tensor> &key, const c10::optional<Tensor> &value, const Tensor &wq, const Tensor &wk, const Tensor &wv,            \
        const Tensor &wp, const c10::optional<Tensor> &bq, const c10::optional<Tensor> &bk, const c10::optional<Tensor> &bv, const c10::optional<Tensor> &bp,  \
        const c10::optional<Tensor> &nq, const c10::optional<Tensor> &nk, double scale, const Tensor &quad_weights, const Tensor &col_idx,                     \
        const Tensor &row_off, const Tensor &plan, c10::ArrayRef<int64_t> plan_header, int64_t num_heads, int64_t nlat_in, int64_t nlon_in,                    \
        int64_t nlat_out, int64_t nlon_out, at::ScalarType compute
#define LAYER_TENSORS                                                                                                                                          \
    {query, key.value_or(Tensor()), value.value_or(Tensor()), wq, wk, wv, wp, bq.value_or(Tensor()), bk.value_or(Tensor()), bv.value_or(Tensor()),             \
     bp.value_or(Tensor()), nq.value_or(Tensor()), nk.value_or(Tensor()), quad_weights, col_idx, row_off, plan}
#define LAYER_CONFIG LayerConfig{num_heads, nlat_in, nlon_in, nlat_out, nlon_out, scale, compute, plan_header.vec()}

// (thirteen tensors and no list: an operator that batching transforms can loop over)
using Tensors13 = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>;
std::vector<Tensor> layer_forward_op(LAYER_ARGS, bool keep);
Tensors13 layer_backward_op(const Tensor &grad, LAYER_ARGS, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &qraw, const Tensor &kraw,
                            const Tensor &y, const Tensor &lse, std::array<bool, NGRADS> need);
Tensors13 as_tuple(const Tensor (&g)[NGRADS])
{
    return {g[0], g[1], g[2], g[3], g[4], g[5], g[6], g[7], g[8], g[9], g[10], g[11], g[12]};
}

// Where a dispatch mode (a tracer, a counter, a policy of what is recomputed) is active or a tensor is a wrapper, the layer's two steps
// go through the dispatcher, as the operators layer_forward and layer_backward: what the node launches by itself nobody would see.
bool observed(const Tensor &t) { return c10::impl::dispatch_mode_enabled() || (t.defined() && at::isTensorSubclassLike(t)); }

c10::optional<Tensor> given_or_none(const Tensor &t) { return t.defined() ? c10::optional<Tensor>(t) : c10::nullopt; }

struct LayerFunction : public torch::autograd::Function<LayerFunction> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, at::TensorList given, const c10::intrusive_ptr<LayerState> &state, bool need_backward)
    {
        Tensor t[NTENSORS], kept[NKEPT];
        for (int i = 0; i < NTENSORS; i++)
            if (state->slot[i] >= 0) t[i] = given[state->slot[i]];
        Tensor out = layer_forward(t, state->cfg, need_backward, kept);
        if (need_backward) {
            torch::autograd::variable_list saved(NSAVED);
            for (int i = 0; i < NTENSORS; i++)
                if (i < BQ || i > BP) saved[i] = t[i];
            for (int i = 0; i < NKEPT; i++) saved[NTENSORS + i] = kept[i];
            ctx->save_for_backward(std::move(saved));
            ctx->saved_data["state"] = c10::IValue::make_capsule(state);
        }
        return out;
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads)
    {
        const auto held = ctx->saved_data["state"].toCapsule();
        const LayerState &state = *static_cast<const LayerState *>(held.get());
        int ngiven = 0;
        for (int s : state.slot) ngiven += s >= 0;
        torch::autograd::variable_list result(ngiven + 2); // + the two arguments that are no tensors
        if (!grads[0].defined()) return result;
        Tensor g[NGRADS];
        std::array<bool, NGRADS> need;
        for (int i = 0; i < NGRADS; i++) need[i] = state.slot[i] >= 0 && ctx->needs_input_grad(state.slot[i]);
        const auto t = ctx->get_saved_variables();
        // (create_graph=True: the operator ties the gradients to what they depend on, and refuses to be differentiated)
        if (observed(grads[0]) || c10::GradMode::is_enabled()) {
            static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("s2attn_kernels::layer_backward", "").typed<decltype(layer_backward_op)>();
            const LayerConfig &c = state.cfg;
            const c10::optional<Tensor> none;
            auto kept = [&](int i) { return t[i].defined() ? t[i] : at::empty({0}, t[S_Q].options()); };
            const Tensors13 r = op.call(grads[0], t[XQ], given_or_none(t[XK]), given_or_none(t[XV]), t[WQ], t[WK], t[WV], t[WP], none, none, none, none,
                                   given_or_none(t[NQ]), given_or_none(t[NK]), c.scale, t[QUAD], t[COL], t[ROW], t[PLAN], c.plan_header, c.num_heads, c.nlat_in,
                                   c.nlon_in, c.nlat_out, c.nlon_out, c.compute, kept(S_Q), kept(S_K), kept(S_V), kept(S_QRAW), kept(S_KRAW), kept(S_Y), kept(S_LSE), need);
            std::apply([&](const auto &...x) {
                int i = 0;
                ((need[i] ? (void)(g[i] = x) : (void)0, i++), ...);
            }, r);
        } else {
            layer_backward(grads[0], t.data(), state.cfg, need, g);
        }
        for (int i = 0; i < NGRADS; i++)
            if (g[i].defined()) result[state.slot[i]] = g[i];
        return result;
    }
};

void check_layer(const Tensor (&t)[NTENSORS], const LayerConfig &cfg)
{
    for (const Tensor &x : t)
        if (x.defined()) require_gpu(x, "a tensor of the layer", t[XQ].device());
    const int64_t B = t[XQ].size(0), C = t[XQ].size(1), Ck = t[WQ].size(0), Cv = t[WV].size(0);
    auto image = [&](const Tensor &x, int64_t h, int64_t w) {
        return x.dim() == 4 && x.size(0) == B && x.size(1) == C && x.size(2) == h && x.size(3) == w && x.scalar_type() == t[XQ].scalar_type();
    };
    const Tensor &xk = t[XK].defined() ? t[XK] : t[XQ], &xv = t[XV].defined() ? t[XV] : xk;
    TORCH_CHECK(B > 0 && C > 0 && image(t[XQ], cfg.nlat_out, cfg.nlon_out) && image(xk, cfg.nlat_in, cfg.nlon_in) && image(xv, cfg.nlat_in, cfg.nlon_in),
                "query, key and value must be non-empty (B, channels, nlat, nlon) tensors of one dtype on the layer's grids");
    TORCH_CHECK(t[WQ].numel() == Ck * C && t[WK].numel() == Ck * C && t[WK].size(0) == Ck && t[WV].numel() == Cv * C && t[WP].numel() == Cv * Cv && t[WP].size(0) == Cv,
                "projection weights do not fit the channels");
    TORCH_CHECK(cfg.num_heads > 0 && Ck % cfg.num_heads == 0 && Cv % cfg.num_heads == 0, "num_heads must divide the channels");
    TORCH_CHECK(t[BQ].defined() == t[BK].defined() && t[BQ].defined() == t[BV].defined() && t[NQ].defined() == t[NK].defined(), "q, k and v have a bias, q and k a norm, all or none");
    const int64_t want[] = {Ck, Ck, Cv, Cv, Ck / cfg.num_heads, Ck / cfg.num_heads};
    for (int i = BQ; i <= NK; i++)
        TORCH_CHECK(!t[i].defined() || (t[i].numel() == want[i - BQ] && t[i].scalar_type() == t[i <= BP ? i - (BQ - WQ) : (int)NQ].scalar_type()), "bias or norm weight of a wrong length or dtype");
}

bool wants_gradient(const Tensor (&t)[NTENSORS])
{
    bool any = false;
    for (const Tensor &x : t) any |= x.defined() && x.requires_grad();
    return any && c10::GradMode::is_enabled();
}

// eager mode: one C++ autograd node
Tensor module_attention(LAYER_ARGS)
{
    const Tensor t[NTENSORS] = LAYER_TENSORS;
    if (at::areAnyTensorSubclassLike(at::ArrayRef<Tensor>(t, NTENSORS))) {
        static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("s2attn_kernels::layer_forward", "").typed<decltype(layer_forward_op)>();
        return op.call(query, key, value, wq, wk, wv, wp, bq, bk, bv, bp, nq, nk, scale, quad_weights, col_idx, row_off, plan, plan_header, num_heads, nlat_in,
                       nlon_in, nlat_out, nlon_out, compute, wants_gradient(t))[0];
    }
    auto state = c10::make_intrusive<LayerState>();
    state->cfg = LAYER_CONFIG;
    check_layer(t, state->cfg);
    std::vector<Tensor> given;
    given.reserve(NTENSORS);
    for (int i = 0; i < NTENSORS; i++) {
        state->slot[i] = t[i].defined() ? (int)given.size() : -1;
        if (!t[i].defined()) continue;
        given.push_back(t[i].contiguous()); // (a copy belongs to the graph, so it is made ahead of the node)
    }
    return LayerFunction::apply(at::TensorList(given), state, wants_gradient(t));
}

// the same two steps as operators without an autograd node of their own: what a compiled graph records (fake kernels and the autograd
// rule in ops.py).  keep: also return what the backward needs.  An absent tensor is returned as an empty one.
std::vector<Tensor> layer_forward_op(LAYER_ARGS, bool keep)
{
    const Tensor t[NTENSORS] = LAYER_TENSORS;
    const LayerConfig cfg = LAYER_CONFIG;
    check_layer(t, cfg);
    Tensor kept[NKEPT];
    std::vector<Tensor> r{layer_forward(t, cfg, keep, kept)};
    for (const Tensor &x : kept) r.push_back(x.defined() ? x : at::empty({0}, query.options().dtype(compute)));
    return r;
}

Tensors13 layer_backward_op(const Tensor &grad, LAYER_ARGS, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &qraw, const Tensor &kraw,
                            const Tensor &y, const Tensor &lse, std::array<bool, NGRADS> need)
{
    Tensor given[NTENSORS] = LAYER_TENSORS;
    const LayerConfig cfg = LAYER_CONFIG;
    check_layer(given, cfg);
    std::vector<Tensor> t(NSAVED);
    for (int i = 0; i < NTENSORS; i++)
        if (given[i].defined()) t[i] = given[i].contiguous();
    t[S_Q] = q, t[S_K] = k, t[S_V] = v, t[S_QRAW] = qraw, t[S_KRAW] = kraw, t[S_Y] = y, t[S_LSE] = lse;
    Tensor g[NGRADS];
    for (int i = 0; i < NGRADS; i++) need[i] = need[i] && (given[i].defined() || (i >= BQ && i <= BP)); // (a bias is not looked at)
    layer_backward(grad, t.data(), cfg, need, g);
    for (Tensor &x : g)
        if (!x.defined()) x = at::empty({0}, query.options());
    return as_tuple(g);
}

// ---- layout ---------------------------------------------------------------------------------------------------------------
Tensor permute(const Tensor &x, bool to_nhwc)
{
    TORCH_CHECK(x.dim() == 4, "expected a 4-dimensional tensor, got ", x.dim(), " dimensions");
    TORCH_CHECK(x.is_contiguous(), "layout conversion expects a contiguous tensor");
    TORCH_CHECK(x.is_cuda(), "x is on ", x.device(), "; the s2attn operators only run on a ROCm GPU (no CPU implementation is shipped)");
    const int64_t d0 = x.size(0), d1 = x.size(1), d2 = x.size(2), d3 = x.size(3);
    Tensor out = to_nhwc ? at::empty({d0, d2, d3, d1}, x.options()) : at::empty({d0, d3, d1, d2}, x.options());
    if (x.numel() == 0) return out;
    const int es = (int)x.element_size();
    TORCH_CHECK(es == 2 || es == 4 || es == 8, "layout conversion supports 2-, 4- and 8-byte elements, got ", x.scalar_type());
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    void *stream = current_stream(x.device());
    check_rc(to_nhwc ? s2attn_permute_to_nhwc(x.data_ptr(), out.data_ptr(), d0, d1, d2, d3, es, stream)
                     : s2attn_permute_to_nchw(x.data_ptr(), out.data_ptr(), d0, d1, d2, d3, es, stream),
             "s2attn_permute");
    return out;
}
Tensor permute_to_nhwc(const Tensor &x) { return permute(x, true); }
Tensor permute_to_nchw(const Tensor &x) { return permute(x, false); }

} // namespace

// Schema strings as in the reference (attention_interface.cpp:85-86, 114-119).
TORCH_LIBRARY(attention_kernels, m)
{
    m.def("permute_to_nhwc(Tensor x) -> Tensor", {at::Tag::pt2_compliant_tag});
    m.def("permute_to_nchw(Tensor x) -> Tensor", {at::Tag::pt2_compliant_tag});
    m.def("forward(Tensor kx, Tensor vx, Tensor qy, Tensor quad_weights, Tensor col_idx, Tensor row_off, int "
          "num_heads, int nlon_in, int nlat_out, int nlon_out) -> Tensor",
          {at::Tag::pt2_compliant_tag});
    m.def("backward(Tensor kx, Tensor vx, Tensor qy, Tensor dy, Tensor quad_weights, Tensor col_idx, Tensor "
          "row_off, int num_heads, int nlon_in, int nlat_out, int nlon_out) -> (Tensor, Tensor, Tensor)",
          {at::Tag::pt2_compliant_tag});
}

TORCH_LIBRARY_IMPL(attention_kernels, CUDA, m)
{
    m.impl("permute_to_nhwc", &permute_to_nhwc);
    m.impl("permute_to_nchw", &permute_to_nchw);
    m.impl("forward", &forward);
    m.impl("backward", &backward);
}

// CPU tensors reach the same entry points, whose device check fails with this package's own message ("only run on a ROCm
// GPU"): there is no CPU implementation, and the dispatcher's "could not run with arguments from the CPU backend" says less.
TORCH_LIBRARY_IMPL(attention_kernels, CPU, m)
{
    m.impl("permute_to_nhwc", &permute_to_nhwc);
    m.impl("permute_to_nchw", &permute_to_nchw);
    m.impl("forward", &forward);
    m.impl("backward", &backward);
}

// The same pair with the forward's output and normaliser handed to the backward, and an optional plan built ahead of time.
TORCH_LIBRARY(s2attn_kernels, m)
{
    m.def("forward_lse(Tensor kx, Tensor vx, Tensor qy, Tensor quad_weights, Tensor col_idx, Tensor row_off, int num_heads, int nlon_in, int "
          "nlat_out, int nlon_out, Tensor? plan=None, int[]? plan_header=None) -> (Tensor, Tensor)",
          {at::Tag::pt2_compliant_tag});
    m.def("backward_saved(Tensor kx, Tensor vx, Tensor qy, Tensor dy, Tensor y, Tensor lse, Tensor quad_weights, Tensor col_idx, Tensor row_off, int "
          "num_heads, int nlon_in, int nlat_out, int nlon_out, Tensor? plan=None, int[]? plan_header=None) -> (Tensor, Tensor, Tensor)",
          {at::Tag::pt2_compliant_tag});
    // the layer: module_attention makes its autograd node inside, so it is a composite operator
    const std::string layer =
        "Tensor query, Tensor? key, Tensor? value, Tensor q_weights, Tensor k_weights, Tensor v_weights, Tensor proj_weights, Tensor? q_bias, Tensor? k_bias, "
        "Tensor? v_bias, Tensor? proj_bias, Tensor? q_norm, Tensor? k_norm, float scale, Tensor quad_weights, Tensor col_idx, Tensor row_off, Tensor plan, "
        "int[] plan_header, int num_heads, int nlat_in, int nlon_in, int nlat_out, int nlon_out, ScalarType compute";
    m.def(("module_attention(" + layer + ") -> Tensor").c_str(), &module_attention);
    m.def(("layer_forward(" + layer + ", bool keep=True) -> Tensor[]").c_str(), {at::Tag::pt2_compliant_tag});
    std::string thirteen = "Tensor";
    for (int i = 1; i < NGRADS; i++) thirteen += ", Tensor";
    m.def(("layer_backward(Tensor grad, " + layer + ", Tensor q, Tensor k, Tensor v, Tensor q_raw, Tensor k_raw, Tensor y, Tensor lse, bool[13] need) -> (" + thirteen + ")").c_str(), {at::Tag::pt2_compliant_tag});
}

TORCH_LIBRARY_IMPL(s2attn_kernels, CUDA, m)
{
    m.impl("forward_lse", &forward_lse);
    m.impl("backward_saved", &backward_saved);
    m.impl("layer_forward", &layer_forward_op);
    m.impl("layer_backward", &layer_backward_op);
}

TORCH_LIBRARY_IMPL(s2attn_kernels, CPU, m) // fails with the same message as above
{
    m.impl("forward_lse", &forward_lse);
    m.impl("backward_saved", &backward_saved);
    m.impl("layer_forward", &layer_forward_op);
    m.impl("layer_backward", &layer_backward_op);
}
